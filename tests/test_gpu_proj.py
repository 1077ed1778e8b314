"""
The module's projections, their gradients and the q/k norm (csrc/s2attn_proj.hip) through the C ABI, against float64, and the
layer as one native node against the same layer composed of separate operators.

Bounds: with u the unit roundoff of fp32 (2^-24), a sum of K products accumulated 16 at a time is off by at most
(K / 16 + c) u sum |x| |w|; c = 8 covers the operands' own splitting (three bf16 terms: 2 * 2^-25 per product), the omitted
third-order products (below 2^-26) and the final addition.  A 16-bit result adds its own rounding (2^-8 |y| for bf16, 2^-11 |y| for
fp16); 16-bit operands are exact.
"""

import ctypes

import pytest
import torch

from tests.util import SEED, assert_close

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
F32, BF16, F16 = torch.float32, torch.bfloat16, torch.float16
U = 2.0**-24
ROUND = {F32: 0.0, BF16: 2.0**-8, F16: 2.0**-11}


def _code(dtype):
    from torch_harmonics_amd import _lib

    return {F32: _lib.S2ATTN_F32, BF16: _lib.S2ATTN_BF16, F16: _lib.S2ATTN_F16}[dtype]


def _stream():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


def _pack(lib, weights, biases, scales, compute, stacked):
    """Packed weights: matrices below each other (stacked: several destinations) or next to each other (several sources)."""
    from torch_harmonics_amd import _lib

    k16 = [lib.s2attn_pack_k16(w.shape[1], compute) for w in weights]
    blocks = [(w.shape[0] + 63) // 64 for w in weights]
    nblk, total = (sum(blocks), k16[0]) if stacked else (blocks[0], sum(k16))
    buf = torch.empty(lib.s2attn_pack_bytes(nblk, total, compute), dtype=torch.uint8, device=DEV)
    bias = None if biases is None else torch.empty(nblk * 64, device=DEV)
    jobs = (_lib.PackJobStruct * len(weights))()
    blk = col = 0
    for j, w, s, i in zip(jobs, weights, scales, range(len(weights))):
        j.w, j.dst = w.data_ptr(), buf.data_ptr()
        if bias is not None:
            j.bias, j.dst_bias = biases[i].data_ptr(), bias.data_ptr()
        j.row_stride, j.col_stride = w.stride()
        j.rows, j.cols, j.dtype, j.scale = w.shape[0], w.shape[1], _code(w.dtype), s
        j.first_block, j.first_k16, j.total_k16 = blk, col, total
        blk, col = (blk + blocks[i], col) if stacked else (blk, col + k16[i])
    _lib.check(lib.s2attn_pack_weights(jobs, len(weights), compute, _stream()), "pack")
    return buf, bias


def _project(lib, src, dst, src_c, dst_c, batch, points, packed, bias, compute, to_nhwc):
    from torch_harmonics_amd import _lib

    p = _lib.ProjStruct(batch=batch, nsrc=len(src), ndst=len(dst), src_dtype=_code(src[0].dtype), dst_dtype=_code(dst[0].dtype), compute=compute, points=points)
    for i, t in enumerate(src):
        p.src[i], p.src_channels[i] = t.data_ptr(), src_c[i]
    for i, t in enumerate(dst):
        p.dst[i], p.dst_channels[i] = t.data_ptr(), dst_c[i]
    p.packed, p.bias = packed.data_ptr(), None if bias is None else bias.data_ptr()
    _lib.check((lib.s2attn_proj_nchw_to_nhwc if to_nhwc else lib.s2attn_proj_nhwc_to_nchw)(ctypes.byref(p), _stream()), "proj")


def _grad(lib, cm, pms, batch, points, compute):
    from torch_harmonics_amd import _lib

    g = _lib.GradStruct(batch=batch, npm=len(pms), cm_dtype=_code(cm.dtype), pm_dtype=_code(pms[0].dtype), compute=compute, cm_channels=cm.shape[1], points=points, cm=cm.data_ptr())
    for i, t in enumerate(pms):
        g.pm[i], g.pm_channels[i] = t.data_ptr(), t.shape[-1]
    slices, ci, cj = lib.s2attn_grad_slices(ctypes.byref(g)), cm.shape[1], sum(t.shape[-1] for t in pms)
    part, pc, pp = (torch.full(s, float("nan"), device=DEV) for s in ((slices, cj, ci), (slices, ci), (slices, cj)))
    g.part, g.part_cm, g.part_pm = part.data_ptr(), pc.data_ptr(), pp.data_ptr()
    _lib.check(lib.s2attn_grad_partials(ctypes.byref(g), _stream()), "grad")
    outs = [torch.empty(s, device=DEV) for s in ((ci, cj), (ci,), (cj,))]  # the matrix transposed: both strides of a job are used
    jobs = (_lib.FinishJobStruct * 3)()
    for j, t, o, r, c, rs, cs in zip(jobs, (part, pc, pp), outs, (cj, 1, 1), (ci, ci, cj), (1, 0, 0), (cj, 1, 1)):
        j.part, j.out, j.slice_stride, j.row_stride, j.col_stride, j.slices, j.rows, j.cols, j.dtype, j.scale = t.data_ptr(), o.data_ptr(), r * c, rs, cs, slices, r, c, 0, 2.0
    _lib.check(lib.s2attn_finish(jobs, 3, _stream()), "finish")
    return [o / 2 for o in outs], slices


def _within(name, got, want, bound):
    worst = ((got.double() - want).abs() - bound).max().item()
    assert torch.isfinite(got).all() and worst <= 0, f"{name}: {worst:.3e} beyond the bound"


# batch, points, input channels, output channels: one, either side of a block of 64 channels / a chunk of 32 or 64 / a tile of 64,
# 128 or 256 points, odd and single points, and enough points and channels for every size of tile
PROJ_CASES = [
    (2, 1, 5, [3]), (3, 2, 1, [1, 1, 2]), (1, 63, 31, [64, 33, 65]), (2, 127, 32, [63]), (1, 129, 33, [130]), (2, 257, 64, [20, 20, 36]),
    (1, 1023, 73, [21, 21, 129]), (1, 4099, 96, [64] * 3), (2, 20011, 130, [128, 128, 66]), (1, 70000, 256, [256]), (1, 140001, 200, [256, 256, 257]),
]  # fmt: skip


@pytest.mark.parametrize("case", PROJ_CASES, ids=lambda c: f"b{c[0]}_p{c[1]}_c{c[2]}_o{'_'.join(map(str, c[3]))}")
@pytest.mark.parametrize("x_dtype,dtype", [(F32, F32), (BF16, BF16), (F16, F16), (F32, BF16), (F32, F16)], ids=["f32", "bf16", "f16", "f32_as_bf16", "f32_as_f16"])
def test_projections_and_their_gradients(case, x_dtype, dtype):
    from torch_harmonics_amd import _lib

    lib, compute = _lib.load(), _code(dtype)
    B, P, C, outs = case
    gen = torch.Generator(device=DEV).manual_seed(SEED)
    rnd = lambda *s: torch.randn(*s, device=DEV, generator=gen)  # noqa: E731
    x, ws, bs = rnd(B, C, P).to(x_dtype), [rnd(o, C) for o in outs], [rnd(o) for o in outs]
    gs = [rnd(B, P, o).to(dtype) for o in outs]
    scales = [0.5] + [1.0] * (len(outs) - 1)
    xd, wd = x.to(dtype).double(), [(w * s).to(dtype).double() for w, s in zip(ws, scales)]
    r = ROUND[dtype]

    ys = [torch.full((B, P, o), float("nan"), device=DEV, dtype=dtype) for o in outs]
    packed, bias = _pack(lib, ws, bs, scales, compute, True)
    _project(lib, [x], ys, [C], outs, B, P, packed, bias, compute, True)
    for y, w, b, s in zip(ys, wd, bs, scales):
        b = (b * s).to(dtype).double()
        want, size = xd.transpose(1, 2) @ w.t() + b, xd.abs().transpose(1, 2) @ w.abs().t() + b.abs()
        _within("NCHW -> NHWC", y, want, (C / 16 + 8) * U * size + r * want.abs() + 1e-7 * (r > 0))

    dx = torch.full((B, C, P), float("nan"), device=DEV, dtype=x_dtype)
    packed, _ = _pack(lib, [w.t() for w in ws], None, scales, compute, False)
    _project(lib, gs, [dx], outs, [C], B, P, packed, None, compute, False)
    want = sum(w.t() @ g.double().transpose(1, 2) for w, g in zip(wd, gs))
    size = sum(w.abs().t() @ g.double().abs().transpose(1, 2) for w, g in zip(wd, gs))
    _within("NHWC -> NCHW", dx, want, (sum(outs) / 16 + 8 + 3) * U * size + ROUND[x_dtype] * want.abs() + 1e-7 * (ROUND[x_dtype] > 0))

    (dw, sx, sg), slices = _grad(lib, x, gs, B, P, compute)
    g = torch.cat(gs, 2).double()
    want, size = (sum(xd[b] @ g[b] for b in range(B)), sum(xd[b].abs() @ g[b].abs() for b in range(B)))
    terms = B * (P / 16 / slices + 5) + slices / 8 + 16
    _within("weight gradient", dw, want, terms * U * size)
    # bias gradients add up eight values at a time
    for name, got, t, dims in (("sum of x", sx, x.double(), (0, 2)), ("sum of g", sg, g, (0, 1))):
        _within(name, got, t.sum(dims), (B * (P / 8 / slices + 5) + slices / 8 + 24) * U * t.abs().sum(dims))


@pytest.mark.parametrize("d", [1, 3, 4, 16, 20, 33, 64, 130, 132, 512])
@pytest.mark.parametrize("dtype", [F32, BF16], ids=["f32", "bf16"])
def test_head_norm_and_its_gradients(d, dtype):
    """Head widths on both sides of every lane-group size; forward and both gradients against torch's rms_norm in float64."""
    from torch_harmonics_amd import _lib

    lib, eps = _lib.load(), torch.finfo(F32).eps
    gen = torch.Generator(device=DEV).manual_seed(SEED)
    rows, mult, blocks = (1037, 3), (0.25, 1.0), 7
    x = [torch.randn(n, d, device=DEV, generator=gen).to(dtype) for n in rows]
    w = [0.3 * torch.randn(d, device=DEV, generator=gen) for _ in rows]
    dy = [torch.randn(n, d, device=DEV, generator=gen).to(dtype) for n in rows]
    y, dx, part = [torch.empty_like(t) for t in x], [t.clone() for t in dy], [torch.full((blocks, d), float("nan"), device=DEV) for _ in rows]
    n = _lib.NormStruct(ntensors=2, head_channels=d, dtype=_code(dtype), gain_dtype=_lib.S2ATTN_F32, blocks=blocks, eps=eps)
    for i in range(2):
        n.x[i], n.y[i], n.gain[i], n.dgain[i], n.rows[i], n.mult[i] = x[i].data_ptr(), y[i].data_ptr(), w[i].data_ptr(), part[i].data_ptr(), rows[i], mult[i]
    _lib.check(lib.s2attn_head_norm(ctypes.byref(n), _stream()), "norm")
    for i in range(2):
        n.y[i] = dx[i].data_ptr()
    _lib.check(lib.s2attn_head_norm_backward(ctypes.byref(n), _stream()), "norm backward")
    tol = dict(rtol=2e-6 + 2 * ROUND[dtype], atol=2e-6 * d**0.5 + 1e-2 * ROUND[dtype])
    for i in range(2):
        xd, wd = x[i].double().requires_grad_(True), w[i].double().requires_grad_(True)
        out = torch.nn.functional.rms_norm(xd, (d,), eps=eps) * (1 + wd) * mult[i]
        out.backward(dy[i].double())
        assert_close("norm", y[i], out, **tol)
        assert_close("d x", dx[i], xd.grad, rtol=tol["rtol"], atol=tol["atol"] * (xd.grad.abs().max().item() + 1))
        assert_close("d gain", part[i].sum(0) * mult[i], wd.grad, rtol=1e-5, atol=1e-5 * rows[i] ** 0.5)


LAYERS = [  # channels, k_channels, out_channels, heads, in_shape, out_shape, which inputs are given
    (24, 24, 24, 2, (9, 36), (9, 36), "q"),
    (24, 48, 12, 3, (9, 36), (9, 36), "qk"),
    (24, 24, 24, 2, (9, 36), (9, 36), "qqv"),
    (64, 64, 64, 2, (12, 128), (7, 64), "qkk"),
    (17, 16, 40, 2, (6, 30), (11, 60), "qkv"),
]


@pytest.mark.parametrize("layer", LAYERS, ids=lambda c: f"c{c[0]}k{c[1]}o{c[2]}h{c[3]}_{c[6]}")
@pytest.mark.parametrize("qknorm,bias", [(False, True), (True, False), (True, True)])
@pytest.mark.parametrize("autocast", [None, BF16], ids=["f32", "autocast_bf16"])
def test_layer_as_one_node_equals_its_separate_operators(layer, qknorm, bias, autocast):
    """Every way to pass query, key and value, all gradients, with one parameter and (cross attention) one input frozen."""
    from torch_harmonics_amd import NeighborhoodAttentionS2, ops

    C, ck, cv, nh, ins, outs, given = layer
    torch.manual_seed(SEED)
    m = NeighborhoodAttentionS2(C, ins, outs, num_heads=nh, k_channels=ck, out_channels=cv, use_qknorm=qknorm, bias=bias).to(DEV)
    with torch.no_grad():
        for n, p in m.named_parameters():
            if "bias" in n or "norm" in n:
                p.uniform_(-0.2, 0.2)
    m.v_weights.requires_grad_(False)
    xq, xk, xv = torch.randn(2, C, *outs, device=DEV), torch.randn(2, C, *ins, device=DEV), torch.randn(2, C, *ins, device=DEV)
    frozen = given == "qkv"
    gout = torch.randn(2, cv, *outs, device=DEV)

    def run():
        q, k, v = xq.clone().requires_grad_(True), xk.clone().requires_grad_(True), xv.clone().requires_grad_(not frozen)
        args = {"q": (q,), "qk": (q, k), "qqv": (q, q, v), "qkk": (q, k, k), "qkv": (q, k, v)}[given]
        m.zero_grad(set_to_none=True)
        with torch.autocast("cuda", dtype=autocast or F32, enabled=autocast is not None):
            out = m(*args)
        out.backward(gout.to(out.dtype))
        grads = {"query": q.grad, "key": k.grad, "value": v.grad}
        # k's bias shifts every score of a query alike unless k is normalised: its gradient is rounding alone
        return out, {**grads, **{n: p.grad for n, p in m.named_parameters() if qknorm or n != "k_bias"}}

    calls = []
    native, composed = run(), None
    m.attention_handle = lambda *a: calls.append(1) or ops.neighborhood_s2_attention(*a)
    composed = run()
    assert calls, "the composed route did not run"
    tol = 1e-5 if autocast is None else 4e-2
    assert native[0].dtype == composed[0].dtype
    for name, a, b in [("output", native[0], composed[0])] + [(n, native[1][n], composed[1][n]) for n in composed[1]]:
        assert (a is None) == (b is None), name
        if a is not None:
            assert a.dtype == b.dtype and a.shape == b.shape, name
            scale = b.float().abs().max().item()
            assert_close(name, a.float(), b.float(), rtol=tol, atol=tol * scale)
    assert native[1]["v_weights"] is None and (native[1]["value"] is None) == (frozen or given in ("q", "qk", "qkk"))
