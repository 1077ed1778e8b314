"""
Head widths of the matrix-core kernels: q / k and v of different widths, widths that are no multiple of 8 or of the tile, and grids
around the sizes their staged band depends on (32 columns, a band of 80 rows, a workgroup of 64 columns, several turns of a
band around a narrow circle), against the float64 oracle fed the stored values.

Bounds: fp32 storage rtol = atol = 1e-5, the suite's bound for fp32.  16-bit storage (_bounds): inputs are exact; with u the storage
type's unit roundoff, the backward's scaled query (key) moves a score by at most u sum |q k|, P, dS and every result are rounded
once each, and I = <dy, y> is formed from the stored y.  First order in u, absolute values throughout, 10 % for second order and
1e-5 for the fp32 arithmetic.
"""

import pytest
import torch

from oracle import cpu_attention as oracle
from oracle import geometry as ogeo
from tests.families import families
from tests.util import assert_close, randn_inputs

pytestmark = pytest.mark.gpu
F32, BF16, F16 = torch.float32, torch.bfloat16, torch.float16

WIDTHS = [(4, 4), (8, 12), (16, 16), (20, 12), (12, 32), (32, 32), (40, 40), (48, 28), (36, 64), (64, 4), (64, 64), (68, 20), (20, 132)]
GRIDS = [  # in_shape, out_shape, theta
    ((7, 32), (7, 32), 0.5), ((6, 33), (6, 33), 0.9), ((9, 79), (9, 79), 0.45), ((5, 80), (5, 80), 4.0), ((8, 130), (8, 130), 0.3),
    ((9, 160), (5, 80), 0.5), ((5, 34), (9, 102), 0.6),
]  # fmt: skip


def _bounds(k, v, q, dy, quad, mask, nh, u):
    """Bounds on the error of (y, dk, dv, dq), shaped like them; mask [points of the output grid, points of the input grid]."""
    heads = lambda t: t.double().reshape(t.shape[0], -1, nh, t.shape[3] // nh).transpose(1, 2)  # noqa: E731
    K, V, Q, G = heads(k), heads(v), heads(q), heads(dy)
    w = quad.double().repeat_interleave(k.shape[2])
    a = torch.where(mask, (Q @ K.transpose(2, 3)) + w.log(), torch.tensor(float("-inf"), dtype=torch.float64))
    p = torch.softmax(a, -1)
    y, g = p @ V, G @ V.transpose(2, 3)
    ds = p * (g - (G * y).sum(-1, keepdim=True))
    e = torch.where(mask, u * (Q.abs() @ K.abs().transpose(2, 3)), torch.zeros((), dtype=torch.float64))  # of a score of the backward
    ey = u * (p @ V.abs()) + u * y.abs()
    eds = ds.abs() * (e + u) + p * (G.abs() * ey).sum(-1, keepdim=True)
    eq = eds @ K.abs() + u * (ds @ K).abs()
    ek = eds.transpose(2, 3) @ Q.abs() + u * (ds.transpose(2, 3) @ Q).abs()
    ev = (p * (e + u)).transpose(2, 3) @ G.abs() + u * (p.transpose(2, 3) @ G).abs()
    flat = lambda t, like: t.transpose(1, 2).reshape(like.shape[0], like.shape[1], like.shape[2], -1)  # noqa: E731
    return [1.1 * flat(t, like) + 1e-5 for t, like in ((ey, q), (ek, k), (ev, v), (eq, q))]


@pytest.mark.parametrize("grid", GRIDS, ids=lambda g: f"{g[0][0]}x{g[0][1]}to{g[1][0]}x{g[1][1]}")
@pytest.mark.parametrize("widths", WIDTHS, ids=lambda w: f"ck{w[0]}cv{w[1]}")
@pytest.mark.parametrize("dtype", [F32, BF16, F16], ids=["f32", "bf16", "f16"])
def test_head_widths(widths, grid, dtype):
    from torch_harmonics_amd import ops

    (ck, cv), (ins, outs, theta), nh = widths, grid, 3
    up = oracle.is_upsample(ins[1], outs[1])
    gi = go = "equiangular"
    col, roff = ogeo.neighborhood_csr(outs, ins, go, gi, theta) if up else ogeo.neighborhood_csr(ins, outs, gi, go, theta)
    quad = ogeo.attention_quad_weights(ins[0], ins[1], gi)
    k, v, q, dy = [t.to(dtype) for t in randn_inputs(1, ins[0], ins[1], outs[0], outs[1], nh, ck, cv, scale=1.0 if dtype == F32 else 0.5)]
    kr, vr, qr = [t.double().requires_grad_(True) for t in (k, v, q)]
    y64 = oracle.dense_attention_f64(kr, vr, qr, quad, col, roff, nh)
    y64.backward(dy.double())
    geo = (quad.cuda(), col.cuda(), roff.cuda(), nh, ins[1], outs[0], outs[1])
    kd, vd, qd, gd = [t.cuda() for t in (k, v, q, dy)]
    y, lse = ops.forward_lse(kd, vd, qd, *geo)
    grads = ops.backward_saved(kd, vd, qd, gd, y, lse, *geo)
    plain = ops.backward(kd, vd, qd, gd, *geo)
    results = [("y", y, y64.detach())] + list(zip(("dk", "dv", "dq"), grads, (kr.grad, vr.grad, qr.grad)))
    if dtype == F32:
        for name, got, want in results:
            assert_close(name, got, want, rtol=1e-5, atol=1e-5)
    else:
        mask = (oracle.dense_mask_upsample if up else oracle.dense_mask)(col, roff, ins[0], ins[1], outs[0], outs[1])
        for (name, got, want), bound in zip(results, _bounds(k, v, q, dy, quad, mask, nh, 2.0**-8 if dtype == BF16 else 2.0**-11)):
            worst = ((got.double().cpu() - want).abs() - bound).max().item()
            assert torch.isfinite(got).all() and worst <= 0, f"{name}: {worst:.3e} beyond the bound"
    for a, b in zip(grads, plain):  # the backward that recomputes y and its normaliser runs the same kernels on them
        assert torch.equal(a, b)


# fp32 heads of up to 16 channels: which kernels run goes by the number of workgroups (1024, and for dk/dv over short runs 4096) and by
# the share of latitudes with long runs.  widths, grid, theta, batch, families of the three passes
NARROW = [
    ((4, 4), (7, 32), 0.5, 60, ("fp32", "split", "split")),
    ((4, 4), (7, 32), 1.2, 60, ("split", "split", "split")),
    ((8, 12), (6, 33), 2.0, 60, ("split", "split", "split")),
    ((16, 16), (9, 79), 0.45, 30, ("split", "split", "split")),
    ((12, 16), (5, 80), 4.0, 60, ("split", "split", "split")),
    ((16, 4), (8, 130), 0.3, 20, ("split", "split", "split")),
    ((16, 16), (16, 64), 0.2, 30, ("fp32", "split", "split")),
    ((8, 8), (16, 64), 0.2, 90, ("fp32", "split", "fp32")),
    ((4, 12), (16, 64), 0.2, 30, ("fp32", "split", "split")),
    ((16, 16), (16, 64), 0.2, 1, ("fp32", "fp32", "fp32")),
]


def _against_float64(results, k, v, q, dy, quad, col, roff, nh):
    kr, vr, qr = [t.double().requires_grad_(True) for t in (k, v, q)]
    y = oracle.dense_attention_f64(kr, vr, qr, quad, col, roff, nh)
    y.backward(dy.double())
    for name, got, want in zip(("y", "dk", "dv", "dq"), results, (y.detach(), kr.grad, vr.grad, qr.grad)):
        assert_close(name, got, want, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("case", NARROW, ids=lambda c: f"ck{c[0][0]}cv{c[0][1]}_{c[1][0]}x{c[1][1]}_{c[2]}_b{c[3]}")
def test_narrow_fp32_heads_on_every_family(case):
    from torch_harmonics_amd import ops

    (ck, cv), grid, theta, batch, want = case
    nh = 3
    col, roff = ogeo.neighborhood_csr(grid, grid, "equiangular", "equiangular", theta)
    assert families(F32, batch, nh, ck, cv, grid, grid, col, roff) == want
    quad = ogeo.attention_quad_weights(*grid, "equiangular")
    tensors = randn_inputs(2, *grid, *grid, nh, ck, cv)
    kd, vd, qd, gd = [t.cuda()[torch.arange(batch) % 2] for t in tensors]  # two entries, repeated
    geo = (quad.cuda(), col.cuda(), roff.cuda(), nh, grid[1], *grid)
    y, lse = ops.forward_lse(kd, vd, qd, *geo)
    results = [y, *ops.backward_saved(kd, vd, qd, gd, y, lse, *geo)]
    for t in results:
        for i in range(2):
            assert torch.equal(t[i::2], t[i : i + 1].expand(t[i::2].shape)) if i < batch else True
    if batch > 1:
        _against_float64([t[:2] for t in results], *tensors, quad, col, roff, nh)
    else:
        _against_float64(results, *[t[:1] for t in tensors], quad, col, roff, nh)


@pytest.mark.parametrize("offset", [1, 2])
@pytest.mark.parametrize("widths", [(4, 4), (8, 8), (16, 12), (20, 12), (32, 32), (48, 48), (64, 64), (68, 20)], ids=lambda w: f"ck{w[0]}cv{w[1]}")
def test_fp32_tensors_at_any_element(widths, offset):
    """Tensors that start at any multiple of four bytes: the split products take them as they are (up to 64 channels), wider heads go to
    the vector kernels."""
    from torch_harmonics_amd import ops

    (ck, cv), grid, nh = widths, (9, 66), 2
    col, roff = ogeo.neighborhood_csr(grid, grid, "equiangular", "equiangular", 0.5)
    assert set(families(F32, 1, nh, ck, cv, grid, grid, col, roff, alignment=4 * offset)) == {"split" if ck <= 64 else "vector"}
    quad = ogeo.attention_quad_weights(*grid, "equiangular")
    tensors = randn_inputs(1, *grid, *grid, nh, ck, cv)

    def shifted(t):
        room = torch.empty(t.numel() + offset, device="cuda")
        room[offset:] = t.flatten()
        return room[offset:].view(t.shape)

    kd, vd, qd, gd = [shifted(t) for t in tensors]
    assert all(t.is_contiguous() and t.data_ptr() % 16 == 4 * offset for t in (kd, vd, qd, gd))
    geo = (quad.cuda(), col.cuda(), roff.cuda(), nh, grid[1], *grid)
    y, lse = ops.forward_lse(kd, vd, qd, *geo)
    results = [y, *ops.backward_saved(kd, vd, qd, gd, y, lse, *geo)]
    _against_float64(results, *tensors, quad, col, roff, nh)
    for a, b in zip(results[1:], ops.backward(kd, vd, qd, gd, *geo)):
        assert_close("recomputed", a, b, rtol=1e-5, atol=1e-5)
