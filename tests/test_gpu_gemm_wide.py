"""The wide sparse GEMM (256 rows x 128 tokens per block) behind
sparse_ternary_gemm_gpu and CuSparseLtGemm, exact against float64 (int32 sums
far below 2^53): rows and tokens that end inside a tile or a lane's four rows,
every remainder of the four-step loop, an output that is not 16-byte aligned,
and CuSparseLtGemm at column counts that end inside a step and at the sizes
where its smaller tiles change."""
import numpy as np
import pytest
import torch

from spbitnet_amd import kernels as K
from spbitnet_amd import weights as W

pytestmark = pytest.mark.gpu


def _ternary(rows, cols, seed):
    L = W.random_layer(rows, cols, seed)
    meta = torch.from_numpy(L.meta.view(np.int32)).cuda()
    values = torch.from_numpy(L.values.view(np.int32)).cuda()
    dense = torch.empty((rows, cols), dtype=torch.int8, device="cuda")
    K.sparse_ternary_unpack_gpu(meta, values, dense, rows, cols, L.meta_stride, L.values_stride)
    return L, meta, values, dense


@pytest.mark.parametrize("nh,nkv,ffn", [(26, 13, 3200), (48, 12, 1024)])
def test_wide_stacks_in_an_engine(gpu, nh, nkv, ffn):
    """Passes of 2048 prompt tokens whose projections take the wide kernel, against
    one decode step per token, bit for bit: 26 heads: q | k | v (boundaries at rows
    3328 and 4992, the latter inside a 256-row block) and gate | up (3200, inside a
    block) with the bf16 sink; 48 heads: o and down with the bf16 and residual sinks."""
    from spbitnet_amd.model import Model, ModelConfig
    from tests.test_gpu_engine import _prompt
    from tests.test_gpu_prefill_attention import _both
    cfg = ModelConfig(hidden_size=128 * nh, num_hidden_layers=1, num_attention_heads=nh,
                      num_key_value_heads=nkv, intermediate_size=ffn, vocab_size=512,
                      max_position_embeddings=2100, head_dim=128)
    model = Model.random(cfg, seed=nh)
    print(f"hidden {cfg.hidden_size}", flush=True)
    batched, stepwise = _both(model, 2100, _prompt(2049, cfg.vocab_size, nh))
    assert torch.isfinite(stepwise).all()
    assert torch.equal(batched.view(torch.int32), stepwise.view(torch.int32))


def _tokens(n, cols, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randint(-128, 128, (n, cols), dtype=torch.int8, device="cuda", generator=g)


# at least 384 blocks each (1.5 per CU); cols / 128 = 2, 4, 6, 10 steps
@pytest.mark.parametrize("rows,cols,n", [(4096, 256, 3072), (4001, 512, 3073), (8190, 768, 1601),
                                         (257, 1280, 25000), (100000, 256, 1), (13825, 1280, 1000),
                                         # beside the lines to the staged tiles
                                         (100000, 256, 16), (100000, 256, 17), (100000, 256, 32),
                                         (100000, 256, 33), (8193, 256, 2047), (9217, 256, 2047)])
def test_ternary_wide(gpu, rows, cols, n):
    L, meta, values, dense = _ternary(rows, cols, rows + n)
    X = _tokens(n, cols, n)
    Y = torch.full((n * rows + 5,), -7, dtype=torch.int32, device="cuda")
    for off in (0, 1):
        print(f"rows={rows} cols={cols} n={n} off={off}", flush=True)
        K.sparse_ternary_gemm_gpu(meta, values, X, Y[off:], rows, cols, n, L.meta_stride,
                                  L.values_stride)
        want = X.double() @ dense.double().T
        assert torch.equal(Y[off:off + n * rows].view(n, rows).double(), want)
        assert (Y[off + n * rows:] == -7).all()
        Y.fill_(-7)


@pytest.mark.parametrize("m,k,n", [
    (4097, 144, 1600), (6000, 272, 1025), (49200, 64, 33),    # wide: 160 blocks or more
    (49200, 64, 3), (40970, 272, 17), (49170, 64, 32),        # as many, up to 32 tokens
    (6912, 400, 230), (97, 2560, 5500),                       # 96 x 32: 512 blocks or more
    (2560, 4112, 201), (129, 6912, 2100),                     # long rows: 128 x 32
    (640, 48, 17), (33, 2560, 40), (2560, 4096, 33), (50, 6912, 64),  # 64 x 32
    (31, 272, 16), (2560, 6912, 1),                           # up to 16 tokens
])
def test_sparse_i8_tiles(gpu, m, k, n):
    print(f"m={m} k={k} n={n}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(m + n)
    A = torch.randint(-128, 128, (m, k), dtype=torch.int8, device="cuda", generator=g)
    B = _tokens(n, k, n)
    op = K.CuSparseLtGemm(m, k, n)
    op.prepare(A)
    P = torch.empty((m, k), dtype=torch.int8, device="cuda")
    op.get_pruned_weights(P)
    D = torch.full((n * m + 4,), -7, dtype=torch.int32, device="cuda")
    op.execute(B, D)
    assert torch.equal(D[:n * m].view(n, m).double(), B.double() @ P.double().T)
    assert (D[n * m:] == -7).all()
