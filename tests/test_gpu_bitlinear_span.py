"""The one-launch BitLinear against the reference's pair of calls (absmax, then
the fused layer), bit for bit: one to two units per thread, rows of one block
up to the last that the one launch takes and past it, activations with NaN,
infinities, zeros and denormals, and an output written over its input."""
import numpy as np
import pytest
import torch

from spbitnet_amd import kernels as K
from spbitnet_amd import weights as W

pytestmark = pytest.mark.gpu
HALF = {"f16": torch.float16, "bf16": torch.bfloat16}


def _layer(rows, cols):
    L = W.random_layer(rows, cols, rows + cols)
    return (torch.from_numpy(L.meta.view(np.int32)).cuda(),
            torch.from_numpy(L.values.view(np.int32)).cuda(), L)


def _pair(meta, values, L, x, rows, cols):
    amax = torch.empty(1, dtype=torch.float32, device="cuda")
    out = torch.empty(rows, dtype=x.dtype, device="cuda")
    K.absmax_reduce_gpu(x, amax, cols)
    K.fused_sparse_bitlinear_gpu(meta, values, x, out, amax, L.gamma, rows, cols, L.meta_stride,
                                 L.values_stride)
    return out


def _one(meta, values, L, x, out, rows, cols):
    ws = torch.full((K.bitlinear_workspace_size(cols),), 0xA5, dtype=torch.uint8, device="cuda")
    K.bitlinear_gpu(meta, values, x, out, L.gamma, rows, cols, L.meta_stride, L.values_stride, ws)
    return out


@pytest.mark.parametrize("kind", ["f16", "bf16"])
@pytest.mark.parametrize("rows,cols", [(1, 128), (257, 384), (25600, 2560), (25601, 2560),
                                       (300, 4096), (513, 4224), (100, 8192), (70, 8320)])
def test_one_launch_equals_the_pair(gpu, kind, rows, cols):
    meta, values, L = _layer(rows, cols)
    g = torch.Generator(device="cuda").manual_seed(cols)
    x = torch.randn(cols, device="cuda", generator=g).to(HALF[kind])
    specials = {"plain": [], "zeros": None, "nan": [(3, float("nan"))],
                "inf": [(5, float("inf")), (cols - 1, -float("inf"))],
                "tiny": "tiny"}
    for name, sp in specials.items():
        y = x.clone()
        if sp is None:
            y.zero_()
        elif sp == "tiny":
            y = (x.float() * (1e-7 if kind == "f16" else 1e-39)).to(HALF[kind])
        else:
            for i, v in sp:
                y[i] = v
        want = _pair(meta, values, L, y, rows, cols)
        got = _one(meta, values, L, y, torch.zeros_like(want), rows, cols)
        same = got.view(torch.int16) == want.view(torch.int16)
        assert (same | (got.isnan() & want.isnan())).all(), name


@pytest.mark.parametrize("kind", ["f16", "bf16"])
@pytest.mark.parametrize("rows,cols", [(1, 128), (257, 384), (25600, 2560), (513, 4224),
                                       (100, 8192), (70, 8320), (25601, 2560), (33, 1000)])
def test_workspace_holds_absmax_and_planes(gpu, kind, rows, cols):
    """The workspace afterwards: the absmax, and from byte 256 on the planes of
    absmax_quantize_planes_gpu, in one launch (to 8192 columns) as in two."""
    meta, values, L = _layer(rows, cols // 64 * 64 + (64 if cols % 64 else 0))
    x = torch.randn(cols, device="cuda").to(HALF[kind])
    planes = torch.empty(8 * -(-cols // 32), dtype=torch.int32, device="cuda")
    amax = torch.empty(1, dtype=torch.float32, device="cuda")
    K.absmax_quantize_planes_gpu(x, planes, amax, cols)
    ws = torch.full((K.bitlinear_workspace_size(cols),), 0xA5, dtype=torch.uint8, device="cuda")
    out = torch.empty(rows, dtype=x.dtype, device="cuda")
    K.bitlinear_gpu(meta, values, x, out, L.gamma, rows, cols, L.meta_stride, L.values_stride, ws)
    assert torch.equal(ws[:4].view(torch.float32), amax)
    assert torch.equal(ws[256:].view(torch.int32), planes)


def test_output_over_input(gpu):
    meta, values, L = _layer(2560, 2560)
    x = torch.randn(2560, device="cuda").to(torch.bfloat16)
    want = _pair(meta, values, L, x, 2560, 2560)
    _one(meta, values, L, x, x, 2560, 2560)
    assert torch.equal(x.view(torch.int16), want.view(torch.int16))
