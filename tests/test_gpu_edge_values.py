"""
Operands at the edge of their range - quadrature weights of zero - on every kernel family of the attention, against float64.

Bounds: fp32 rtol = atol = 1e-5, the suite's bound for fp32; 16-bit storage as in test_gpu_widths._bounds.
"""

import pytest
import torch

from oracle import cpu_attention as oracle
from oracle import geometry as ogeo
from tests.test_gpu_widths import BF16, F16, F32, _bounds
from tests.util import assert_close, randn_inputs

pytestmark = pytest.mark.gpu

# storage, ck, cv, grid (input and output), batch copies, heads.  Copies of one batch entry: the fp32 dispatch goes by the number of
# workgroups (heads of up to 16 channels: 1024, heads of 32: 4096), the oracle by one entry.
SHAPES = {
    "f32_c3c5": (F32, 3, 5, (9, 48), 1, 2),  # vector kernels
    "f32_c8": (F32, 8, 8, (9, 48), 1, 2),  # 16-longitude fp32 tiles, few workgroups
    "f32_c8_many": (F32, 8, 8, (9, 48), 60, 2),  # split products
    "f32_c4c12_many": (F32, 4, 12, (9, 48), 60, 2),
    "f32_c16_many": (F32, 16, 16, (9, 48), 60, 2),
    "f32_c20c12": (F32, 20, 12, (9, 48), 1, 2),
    "f32_c32": (F32, 32, 32, (9, 64), 1, 2),
    "f32_c32_many": (F32, 32, 32, (16, 64), 128, 2),  # hybrid kernels over short runs
    "f32_c40": (F32, 40, 40, (9, 48), 1, 2),
    "f32_c64": (F32, 64, 64, (9, 48), 1, 2),
    "f32_c68c20": (F32, 68, 20, (9, 48), 1, 2),  # fp32 tiles of 128 channels
    "f32_c160": (F32, 160, 160, (9, 48), 1, 1),  # two channel groups
    "bf16_c32": (BF16, 32, 32, (9, 48), 1, 2),  # 16-bit tiles
    "bf16_c20c12": (BF16, 20, 12, (9, 48), 1, 2),  # split products
    "bf16_c12": (BF16, 12, 12, (9, 48), 1, 2),
    "f16_c64": (F16, 64, 64, (9, 48), 1, 2),
    "f16_c36c44": (F16, 36, 44, (9, 48), 1, 2),
}


def _problem(shape, theta):
    dtype, ck, cv, (H, W), copies, nh = SHAPES[shape]
    col, roff = ogeo.neighborhood_csr((H, W), (H, W), "equiangular", "equiangular", theta)
    quad = ogeo.attention_quad_weights(H, W, "equiangular")
    k, v, q, dy = [t.to(dtype) for t in randn_inputs(1, H, W, H, W, nh, ck, cv, scale=1.0 if dtype == F32 else 0.5)]
    return dtype, (k, v, q, dy), quad, col, roff, nh, copies


def _run(tensors, quad, col, roff, nh, copies):
    """(y, dk, dv, dq) of the first batch entry; the others are the same entry and have to give the same bits."""
    from torch_harmonics_amd import ops

    k, v, q, dy = [t.cuda().repeat(copies, 1, 1, 1) for t in tensors]
    geo = (quad.cuda(), col.cuda(), roff.cuda(), nh, k.shape[2], q.shape[1], q.shape[2])
    y, lse = ops.forward_lse(k, v, q, *geo)
    out = (y, *ops.backward_saved(k, v, q, dy, y, lse, *geo))
    bits = {2: torch.int16, 4: torch.int32}[y.element_size()]
    for t in out:
        assert torch.equal(t.view(bits), t[:1].view(bits).expand(t.shape)), "copies of one batch entry differ"
    return [t[:1].cpu() for t in out]


@pytest.mark.parametrize("zero", ["first", "middle", "first_two", "all_but_one"])
@pytest.mark.parametrize("shape", SHAPES)
def test_quadrature_weight_zero(shape, zero):
    """A latitude of quadrature weight zero takes no part in the softmax, wherever it stands in a query's neighborhood (the reference
    multiplies by the weight, attention_torch.py:97-125).  all_but_one: with a disk that holds the whole sphere."""
    theta = 4.0 if zero == "all_but_one" else 0.9
    dtype, tensors, quad, col, roff, nh, copies = _problem(shape, theta)
    H = quad.numel()
    quad = quad.clone()
    quad[{"first": slice(0, 1), "middle": slice(H // 2, H // 2 + 1), "first_two": slice(0, 2), "all_but_one": slice(0, H - 2)}[zero]] = 0.0
    if zero == "all_but_one":
        quad[H - 1] = 0.0
    k, v, q, dy = tensors
    kr, vr, qr = [t.double().requires_grad_(True) for t in (k, v, q)]
    y64 = oracle.dense_attention_f64(kr, vr, qr, quad, col, roff, nh)
    assert torch.isfinite(y64).all(), "every query is left a neighbor"
    y64.backward(dy.double())
    want = [y64.detach(), kr.grad, vr.grad, qr.grad]
    got = _run(tensors, quad, col, roff, nh, copies)
    if dtype == F32:
        for name, a, b in zip(("y", "dk", "dv", "dq"), got, want):
            assert_close(name, a, b, rtol=1e-5, atol=1e-5)
        return
    mask = oracle.dense_mask(col, roff, H, k.shape[2], H, k.shape[2])
    for name, a, b, bound in zip(("y", "dk", "dv", "dq"), got, want, _bounds(k, v, q, dy, quad, mask, nh, 2.0**-8 if dtype == BF16 else 2.0**-11)):
        worst = ((a.double() - b).abs() - bound).max().item()
        assert torch.isfinite(a).all() and worst <= 0, f"{name}: {worst:.3e} beyond the bound"
