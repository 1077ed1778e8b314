"""
Operands at the edge of their range - quadrature weights of zero and below, NaN, infinities, the largest magnitudes - on every
kernel family of the attention, against float64.

Bounds: fp32 rtol = atol = 1e-5, the suite's bound for fp32; 16-bit storage as in test_gpu_widths._bounds, or 2e-2 of the tensor's scale.
"""

import pytest
import torch

from oracle import cpu_attention as oracle
from oracle import geometry as ogeo
from tests.families import families
from tests.test_gpu_widths import BF16, F16, F32, _bounds
from tests.util import assert_close, randn_inputs

pytestmark = pytest.mark.gpu

# storage, ck, cv, grid (one, or input and output grid), batch copies, heads, family of kernels of all three passes.  Copies of one batch entry: the fp32 dispatch goes by the
# number of workgroups (heads of up to 16 channels: 1024, heads of 32: 4096), the oracle by one entry.
SHAPES = {
    "f32_c3c5": (F32, 3, 5, (9, 48), 1, 2, "vector"),
    "f32_c8": (F32, 8, 8, (9, 48), 1, 2, "fp32"),
    "f32_c4_w96": (F32, 4, 4, (9, 96), 1, 2, "fp32"),
    "f32_c8_w96": (F32, 8, 8, (9, 96), 1, 2, "fp32"),
    "f32_c12_w96_many": (F32, 12, 12, (9, 96), 30, 2, "split"),
    "f32_c8_many": (F32, 8, 8, (9, 48), 60, 2, "split"),
    "f32_c4c12_many": (F32, 4, 12, (9, 48), 60, 2, "split"),
    "f32_c16_many": (F32, 16, 16, (9, 48), 60, 2, "split"),
    "f32_c20c12": (F32, 20, 12, (9, 48), 1, 2, "split"),
    "f32_c20c12_down": (F32, 20, 12, ((9, 96), (5, 48)), 1, 2, "split"),
    "f32_c20c12_up": (F32, 20, 12, ((5, 34), (9, 102)), 1, 2, "split"),
    "f32_c32": (F32, 32, 32, (9, 64), 1, 2, "split"),
    "f32_c32_many": (F32, 32, 32, (16, 64), 128, 2, "hybrid"),
    "f32_c40": (F32, 40, 40, (9, 48), 1, 2, "split"),
    "f32_c64": (F32, 64, 64, (9, 48), 1, 2, "split"),
    "f32_c68c20": (F32, 68, 20, (9, 48), 1, 2, "fp32"),
    "f32_c68c20_down": (F32, 68, 20, ((9, 96), (5, 48)), 1, 2, "fp32"),
    "f32_c68c20_up": (F32, 68, 20, ((5, 34), (9, 102)), 1, 2, "fp32"),
    "f32_c160": (F32, 160, 160, (9, 48), 1, 1, "fp32"),  # two channel groups
    "f32_c20c132": (F32, 20, 132, (9, 48), 1, 1, "fp32"),
    "bf16_c32": (BF16, 32, 32, (9, 48), 1, 2, "16bit"),
    "bf16_c20c12": (BF16, 20, 12, (9, 48), 1, 2, "split"),
    "bf16_c12": (BF16, 12, 12, (9, 48), 1, 2, "split"),
    "f16_c64": (F16, 64, 64, (9, 48), 1, 2, "16bit"),
    "f16_c36c44": (F16, 36, 44, (9, 48), 1, 2, "split"),
    "f16_c36c44_up": (F16, 36, 44, ((5, 34), (9, 102)), 1, 2, "split"),
}
TILES = {"f32_c32", "f32_c32_many", "bf16_c32", "f16_c64"}  # what is not finite may reach the columns of a whole tile


def _theta(shape, fine, coarse):
    """Disk radius for the shape's input grid; the hybrid kernels take mostly short runs."""
    grid = SHAPES[shape][3]
    if SHAPES[shape][6] == "hybrid":
        return 0.3
    return coarse if isinstance(grid[0], tuple) and grid[0][0] == 5 else fine


def _problem(shape, theta):
    dtype, ck, cv, grid, copies, nh, family = SHAPES[shape]
    ins, outs = grid if isinstance(grid[0], tuple) else (grid, grid)
    up = oracle.is_upsample(ins[1], outs[1])
    col, roff = ogeo.neighborhood_csr(*((outs, ins) if up else (ins, outs)), "equiangular", "equiangular", theta)
    assert set(families(dtype, copies, nh, ck, cv, ins, outs, col, roff)) == {family}
    quad = ogeo.attention_quad_weights(*ins, "equiangular")
    mask = (oracle.dense_mask_upsample if up else oracle.dense_mask)(col, roff, *ins, *outs)
    tensors = [t.to(dtype) for t in randn_inputs(1, *ins, *outs, nh, ck, cv, scale=1.0 if dtype == F32 else 0.5)]
    return dtype, tensors, quad, (col, roff, nh, copies), mask


def _run(tensors, quad, geometry):
    """(y, dk, dv, dq) of the first batch entry; the others are the same entry and have to give the same bits."""
    from torch_harmonics_amd import ops

    col, roff, nh, copies = geometry
    k, v, q, dy = [t.cuda().repeat(copies, 1, 1, 1) for t in tensors]
    geo = (quad.cuda(), col.cuda(), roff.cuda(), nh, k.shape[2], q.shape[1], q.shape[2])
    y, lse = ops.forward_lse(k, v, q, *geo)
    out = (y, *ops.backward_saved(k, v, q, dy, y, lse, *geo))
    bits = {2: torch.int16, 4: torch.int32}[y.element_size()]
    for t in out:
        assert torch.equal(t.view(bits), t[:1].view(bits).expand(t.shape)), "copies of one batch entry differ"
    return [t[:1].cpu() for t in out]


def _true_neighbors(tensors, quad, mask, nh):
    """(y, dk, dv, dq) in float64 from each query's true neighbors and nothing else (attention_torch.py:97-125), differentiated by torch."""
    idx = torch.zeros(mask.shape[0], int(mask.sum(1).max()), dtype=torch.int64)
    there = torch.zeros(idx.shape, dtype=torch.bool)
    for i, row in enumerate(mask):
        n = row.nonzero().flatten()
        idx[i], idx[i, : len(n)], there[i, : len(n)] = n[0], n, True  # (padded with a true neighbor, which then counts once)
    k, v, q, dy = tensors
    leaves = [t.double().requires_grad_(True) for t in (k, v, q)]
    K, V, Q = [t.reshape(-1, nh, t.shape[3] // nh) for t in leaves]
    w = quad.double().repeat_interleave(k.shape[2])[idx]
    s = (Q[:, None] * K[idx]).sum(-1)
    s = torch.where(there[..., None], s, -torch.inf)
    p = torch.where(there[..., None], torch.exp(s - torch.nan_to_num(s.detach(), nan=-torch.inf, posinf=torch.inf).amax(1, keepdim=True)) * w[..., None], 0.0)
    y = sum(torch.where(there[:, i, None, None], p[:, i, :, None] * V[idx[:, i]], 0.0) for i in range(idx.shape[1])) / p.sum(1)[..., None]
    y = y.reshape(1, q.shape[1], q.shape[2], -1)
    y.backward(dy.double())
    return [y.detach()] + [t.grad for t in leaves]


@pytest.mark.parametrize("zero", ["first", "middle", "first_two", "all_but_one"])
@pytest.mark.parametrize("shape", SHAPES)
def test_quadrature_weight_zero(shape, zero):
    """A latitude of quadrature weight zero takes no part in the softmax, wherever it stands in a query's neighborhood (the reference
    multiplies by the weight, attention_torch.py:97-125).  all_but_one: with a disk that holds the whole sphere."""
    if zero in ("first_two", "all_but_one") and SHAPES[shape][6] == "hybrid":
        pytest.skip("needs a disk of a radius that has long runs only")
    dtype, tensors, quad, geometry, mask = _problem(shape, 4.0 if zero == "all_but_one" else _theta(shape, 0.9, 1.7))
    H = quad.numel()
    quad = quad.clone()
    quad[{"first": slice(0, 1), "middle": slice(H // 2, H // 2 + 1), "first_two": slice(0, 2), "all_but_one": slice(0, H - 2)}[zero]] = 0.0
    if zero == "all_but_one":
        quad[H - 1] = 0.0
    k, v, q, dy = tensors
    kr, vr, qr = [t.double().requires_grad_(True) for t in (k, v, q)]
    y64 = oracle.dense_attention_f64(kr, vr, qr, quad, *geometry[:3])
    assert torch.isfinite(y64).all(), "every query is left a neighbor"
    y64.backward(dy.double())
    want = [y64.detach(), kr.grad, vr.grad, qr.grad]
    got = _run(tensors, quad, geometry)
    if dtype == F32:
        for name, a, b in zip(("y", "dk", "dv", "dq"), got, want):
            assert_close(name, a, b, rtol=1e-5, atol=1e-5)
        return
    for name, a, b, bound in zip(("y", "dk", "dv", "dq"), got, want, _bounds(k, v, q, dy, quad, mask, geometry[2], 2.0**-8 if dtype == BF16 else 2.0**-11)):
        worst = ((a.double() - b).abs() - bound).max().item()
        assert torch.isfinite(a).all() and worst <= 0, f"{name}: {worst:.3e} beyond the bound"


@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan"), 3.4e38])
def test_heads_of_32_channels_keep_an_infinity_where_it_is_seen(value):
    """Split products of heads of 32 channels: a query that sees the value gets what arithmetic on its neighbors gives; what stays finite
    has the bits it has without the value."""
    dtype, tensors, quad, geometry, mask = _problem("f32_c32", 0.6)
    clean = _run(tensors, quad, geometry)[0]
    H, W = tensors[1].shape[1:3]
    tensors[1][0, H // 2, W // 3, 1] = value
    got, want = _run(tensors, quad, geometry)[0], _true_neighbors(tensors, quad, mask, geometry[2])[0]
    sees = mask[:, (H // 2) * W + W // 3].reshape(1, H, W)
    a, b = got[sees].double(), want[sees]
    special = torch.isnan(b) | torch.isinf(b)
    assert torch.equal(torch.isfinite(a), ~special)
    assert torch.equal(torch.isnan(a), torch.isnan(b)) and torch.equal(a[torch.isinf(b)], b[torch.isinf(b)])
    big = b.abs() > 1e30
    assert_close("seen", a[~special & ~big], b[~special & ~big], rtol=1e-5, atol=1e-5)
    assert_close("seen, near the end of the range", a[~special & big] / 1e38, b[~special & big] / 1e38, rtol=1e-5, atol=0)
    unseen = got[~sees]
    assert torch.equal(unseen[torch.isfinite(unseen)], clean[~sees][torch.isfinite(unseen)])


NAN, INF = float("nan"), float("inf")
POISON = {"k_nan": (0, NAN), "v_nan": (1, NAN), "q_nan": (2, NAN), "dy_nan": (3, NAN), "k_minus_inf": (0, -INF), "v_inf": (1, INF), "dy_inf": (3, -INF), "v_huge": (1, 3.4e38)}


@pytest.mark.parametrize("poison", [*POISON, "weight_below_zero"])
@pytest.mark.parametrize("shape", [s for s in SHAPES if s not in TILES])
def test_what_is_not_finite_reaches_true_neighbors_only(shape, poison):
    """One channel of one point is NaN, infinite or of a magnitude that only fp32 holds: what sees the point gets what float64
    arithmetic on its neighbors gives, and everything else the result it has without it."""
    dtype, tensors, quad, geometry, mask = _problem(shape, _theta(shape, 0.6, 0.9))
    if poison == "weight_below_zero":
        quad = quad.clone()
        quad[quad.numel() // 2] *= -0.01  # (the sums must not cancel)
    else:
        which, value = POISON[poison]
        if dtype != F32 and poison == "v_huge":
            pytest.skip("fp32's range")
        t = tensors[which]
        t[0, t.shape[1] // 2, t.shape[2] // 3, 1] = value
    got, want = _run(tensors, quad, geometry), _true_neighbors(tensors, quad, mask, geometry[2])
    clean = (poison == "weight_below_zero") or None
    for name, a, b in zip(("y", "dk", "dv", "dq"), got, want):
        if poison == "v_huge" and name != "y":  # (<dy, v> leaves fp32's range)
            continue
        a = a.double()
        finite = torch.isfinite(b)
        assert bool(finite.all()) if clean else True
        assert torch.equal(torch.isfinite(a), finite), f"{name}: {int((torch.isfinite(a) != finite).sum())} of {finite.numel()} values are finite on one side only"
        if name == "y":
            special = lambda x: torch.nan_to_num(x, nan=7.0, posinf=8.0, neginf=9.0)  # noqa: E731
            assert torch.equal(special(a)[~finite], special(b)[~finite])
        if name == "y" and poison == "v_huge":
            big = b.abs() > 1e30
            assert_close(name, a[big] / 1e38, b[big] / 1e38, rtol=1e-5, atol=0)
            finite &= ~big
        x, y = a[finite], b[finite]
        if dtype == F32:
            assert_close(name, x, y, rtol=1e-5, atol=1e-5)
        else:
            assert_close(name, x, y, rtol=2e-2, atol=2e-2 * y.square().mean().sqrt().item())


def _layer(dtype, channels, k_channels, out_channels, **kw):
    from torch_harmonics_amd import NeighborhoodAttentionS2

    torch.manual_seed(11)
    m = NeighborhoodAttentionS2(channels, (10, 66), (10, 66), num_heads=2, k_channels=k_channels, out_channels=out_channels, theta_cutoff=0.5, **kw).cuda()
    return m.to(dtype) if dtype != F32 else m


@pytest.mark.parametrize("value", [NAN, INF, -3.4e38])
@pytest.mark.parametrize("channels", [(17, 8, 40), (64, 40, 24)], ids=lambda c: f"c{c[0]}k{c[1]}o{c[2]}")
def test_layer_keeps_what_is_not_finite_to_the_points_that_see_it(channels, value):
    """The projections contract channels, never points, and the attention touches true neighbors: the layer's result is untouched
    elsewhere, and not finite at every point whose neighborhood holds the value (an infinity may come out as NaN)."""
    m = _layer(F32, *channels)
    x = torch.randn(2, channels[0], 10, 66, device="cuda")
    mask = oracle.dense_mask(m.psi_col_idx.cpu(), m.psi_roff_idx.cpu(), 10, 66, 10, 66).reshape(10, 66, 10, 66)[:, :, 4, 30].cuda()
    for channel in (0, channels[0] - 1):
        bad = x.clone()
        bad[1, channel, 4, 30] = value
        with torch.no_grad():
            a, b = m(bad), m(x)
        assert torch.equal(a[0], b[0])
        assert not torch.isfinite(a[1][:, mask]).any() and torch.isfinite(a[1][:, ~mask]).all()
        assert_close("elsewhere", a[1][:, ~mask], b[1][:, ~mask], rtol=1e-5, atol=1e-5)


def test_small_magnitudes_keep_their_precision():
    """Three bf16 terms hold a value to 2^-24 down to 2^-110, and to 2^-133 absolutely below: the layer is linear in its value input (three
    products with sums of at most 40, 120 and 40 terms of magnitude below 4)."""
    m = _layer(F32, 40, 40, 40, bias=False)
    x, v = torch.randn(1, 40, 10, 66, device="cuda"), torch.randn(1, 40, 10, 66, device="cuda")
    with torch.no_grad():
        want = m(x, x, v).double()
        for k in (60, 90, 105, 115, 120):
            got = m(x, x, v * 2.0**-k).double() * 2.0**k
            worst = ((got - want).abs() - 2.0**-22 * want.abs().max() - 200 * 2.0 ** (k - 133)).max().item()
            assert worst <= 0, f"2^-{k}: {worst:.3e} beyond the bound"
