"""The per-op attention kernels for 16-byte aligned rows and the general ones,
against float64: every rows-per-wave split (head_dim 32 to 256), groups of q
heads that do not divide, sequence lengths around the kernels' blocks, and
caches that start 2 bytes off a 16-byte boundary.  Float32 sums of at most 5000
terms in [0, 1] of either order stay within 1e-5 of float64 (n eps / 2 at
worst 3e-4, sqrt(n) eps = 4e-6 in practice; 1e-4 is asserted, as in
test_gpu_ops); 16-bit outputs within one unit in the last place."""
import numpy as np
import pytest
import torch

from tests.test_gpu_ops import KINDS, _assert_16, _call, _p, _to_host

pytestmark = pytest.mark.gpu

SHAPES = [  # heads, kv heads, head_dim, seq
    (4, 2, 32, 1), (20, 5, 128, 63), (8, 1, 64, 511), (7, 3, 128, 513), (16, 16, 64, 1025),
    (3, 1, 256, 2049), (20, 5, 128, 5000), (5, 2, 80, 700), (2, 2, 20, 130), (9, 1, 8, 300),
    # groups over several blocks, the
    # last lengths of the general output kernel and the first of 1, 2 and 4 heads a block
    (64, 1, 128, 1300), (8, 1, 64, 4500), (64, 1, 64, 24), (64, 1, 64, 25), (64, 1, 128, 400),
    (64, 1, 256, 512), (20, 5, 128, 13), (20, 5, 128, 14), (20, 5, 128, 512),
]


@pytest.mark.parametrize("kind", ["f16", "bf16"])
@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("nh,nkv,hd,seq", SHAPES)
def test_attention_ops(gpu, kind, off, nh, nkv, hd, seq):
    max_seq = seq + 3
    g = torch.Generator().manual_seed(nh * hd + seq)

    def rand(n):  # `off` elements into a buffer
        return torch.randn(n + off, generator=g).to(KINDS[kind]).cuda()[off:]

    q, K, V = rand(nh * hd), rand(nkv * max_seq * hd), rand(nkv * max_seq * hd)
    sc = torch.full((nh, max_seq), 7.0, dtype=torch.float32, device="cuda")
    out = torch.empty(nh * hd, dtype=KINDS[kind], device="cuda")
    scale = 1.0 / np.sqrt(hd)
    _call(f"spb_attention_scores_{kind}", _p(q), _p(K), _p(sc), nh, nkv, hd, max_seq, seq,
          float(scale), None)
    kv = np.arange(nh) * nkv // nh
    k64 = _to_host(K).reshape(nkv, max_seq, hd)[kv][:, :seq]
    v64 = _to_host(V).reshape(nkv, max_seq, hd)[kv][:, :seq]
    want = np.einsum("hd,hjd->hj", _to_host(q).reshape(nh, hd), k64) * scale
    got = _to_host(sc)
    assert np.abs(got[:, :seq] - want).max() <= 1e-4
    assert (got[:, seq:] == 7.0).all()
    _call("spb_softmax", _p(sc), nh, max_seq, seq, None)
    p = np.exp(got[:, :seq] - got[:, :seq].max(1, keepdims=True))
    p /= p.sum(1, keepdims=True)
    got = _to_host(sc)
    assert np.abs(got[:, :seq] - p).max() <= 5e-6
    assert (got[:, seq:] == 7.0).all()
    _call(f"spb_attention_output_{kind}", _p(sc), _p(V), _p(out), nh, nkv, hd, max_seq, seq, None)
    want = np.einsum("hj,hjd->hd", got[:, :seq], v64)
    err = np.abs(_to_host(out).reshape(nh, hd) - want)
    # half a unit of the rounding to 16 bits, and the float32 sum's error
    unit = 2.0 ** -10 if kind == "f16" else 2.0 ** -7
    assert (err <= 0.51 * unit * np.abs(want) + 1e-5).all()
