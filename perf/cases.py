"""
The work a user of this package has it do, as cases that can be timed and compared: the attention module in training and in
inference, in fp32, in 16-bit storage and under autocast, in all three directions (self-attention, down-sampling, up-sampling),
the autograd operator on its own, and the ring steps of one rank of a longitude-sharded layer.

A case is a dict of plain values:

  kind        "train" (module forward + backward), "infer" (module forward without autograd), "op" (the autograd operator on
              NHWC q, k, v, forward + backward), "ring" (one rank's forward fold, backward pass 1 and pass 2)
  nlat_in, nlon_in, nlat_out, nlon_out, grid_in, grid_out, theta (disk radius, radians)
  batch, channels (module input), k_channels, out_channels, heads
  storage     element type of the activations (and of the module's parameters): "fp32", "bf16", "fp16"
  autocast    "none", "bf16", "fp16"
  qknorm, bias    options of the module
  chunks      "ring": number of longitude chunks (= ranks)
"""

import contextlib
import math

import numpy as np
import torch

DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}


def _case(name, kind, ins, outs, batch, channels, heads, theta, **more):
    c = dict(
        name=name, kind=kind, nlat_in=ins[0], nlon_in=ins[1], nlat_out=outs[0], nlon_out=outs[1], grid_in="equiangular", grid_out="equiangular",
        theta=theta, batch=batch, channels=channels, k_channels=channels, out_channels=channels, heads=heads, storage="fp32", autocast="none",
        qknorm=False, bias=True, chunks=1,
    )  # fmt: skip
    c.update(more)
    return c


def listed():
    return [
        # a layer on a coarse grid, one head, default radius: every kernel is a few microseconds, so launches and host time count
        _case("train_32x64_c16", "train", (32, 64), (32, 64), 1, 16, 1, math.pi / 31),
        # inference on a 2-degree grid with one wide head
        _case("infer_91x180_c256_1head", "infer", (91, 180), (91, 180), 1, 256, 1, math.pi / 90),
        # a small training batch, four heads of 16 channels, neighborhoods of about a hundred points
        _case("train_128x256_c64_b4", "train", (128, 256), (128, 256), 4, 64, 4, 4 * math.pi / 127),
        # 0.5-degree grid, one head of 64 channels (the head width the package's users publish timings for)
        _case("train_360x720_c64_1head", "train", (360, 720), (360, 720), 1, 64, 1, 0.03),
        # the decoder of a U-shaped model: coarse keys and values, fine queries
        _case("train_up_180x360_to_360x720", "train", (180, 360), (360, 720), 1, 64, 1, 0.03),
        # its encoder on the 0.25-degree grid: equiangular input, Gaussian output of half the resolution
        _case("train_down_721x1440_to_lg360x720", "train", (721, 1440), (360, 720), 2, 128, 4, 2 * math.pi / 359, grid_out="legendre-gauss"),
        # a layer of a 0.25-degree weather model in fp32: 256 channels, eight heads of 32
        _case("train_721x1440_c256", "train", (721, 1440), (721, 1440), 1, 256, 8, 3 * math.pi / 720),
        # the same layer used for a forecast under bf16 autocast
        _case("infer_autocast_721x1440_c256", "infer", (721, 1440), (721, 1440), 1, 256, 8, 3 * math.pi / 720, autocast="bf16"),
        # mixed-precision training with q/k normalisation on an odd number of latitudes
        _case("train_autocast_qknorm_181x360", "train", (181, 360), (181, 360), 2, 192, 6, 3 * math.pi / 180, autocast="bf16", qknorm=True),
        # a wide 16-bit layer with a large radius: thousands of neighbors per point near the poles
        _case("train_bf16_lg361x720_c1024", "train", (361, 720), (361, 720), 4, 1024, 16, 8 * math.pi / 360, grid_in="legendre-gauss", grid_out="legendre-gauss", storage="bf16"),
        # the operator inside a model of the user's own: head widths of q/k and v that differ and are no power of two
        _case("op_lobatto_145x288_ck20_cv12", "op", (145, 288), (145, 288), 2, 60, 3, 2 * math.pi / 144, out_channels=36, grid_in="lobatto", grid_out="lobatto"),
        # one of four ranks of the 0.25-degree layer with its longitudes sharded: its own queries against four rotating chunks
        _case("ring_721x1440_4ranks", "ring", (721, 1440), (721, 1440), 1, 256, 8, 3 * math.pi / 720, chunks=4),
    ]


# ---- sizes ------------------------------------------------------------------------------------------------------------------
def _colatitudes(n, grid):
    """Roughly where the rings lie: enough to count neighbors."""
    return np.pi * np.arange(n) / (n - 1) if grid != "legendre-gauss" else np.pi * (np.arange(n) + 0.5) / n


def _pairs(c):
    """Query-key pairs of one forward over all heads, from the arc that a disk of radius theta cuts out of every ring (within a
    few per cent of the exact count)."""
    a, b = _colatitudes(c["nlat_out"], c["grid_out"])[:, None], _colatitudes(c["nlat_in"], c["grid_in"])[None, :]
    num, den = math.cos(c["theta"]) - np.cos(a) * np.cos(b), np.sin(a) * np.sin(b)
    ratio = np.where(den > 1e-9, num / np.maximum(den, 1e-9), np.where(num <= 1e-9, -2.0, 2.0))
    arc = np.where(ratio <= -1.0, 1.0, np.where(ratio > 1.0, 0.0, np.arccos(np.clip(ratio, -1.0, 1.0)) / np.pi))
    per_column = float(np.where(arc > 0, np.maximum(1.0, arc * c["nlon_in"]), 0.0).sum())
    return c["batch"] * c["heads"] * (c["nlon_out"] // c["chunks"] if c["kind"] == "ring" else c["nlon_out"]) * per_column


def _is_self(c):
    return (c["nlat_in"], c["nlon_in"], c["grid_in"]) == (c["nlat_out"], c["nlon_out"], c["grid_out"])


def work(case):
    """Bytes: inputs and upstream gradients read once, results and gradients written once, nothing in between.  Flops: two per
    multiply-add of the projections (forward, input gradient, weight gradient) and of the attention (q.k and p.v forward; those
    two again and dq, dk, dv backward; the ring's two passes each recompute both products)."""
    c = case
    es = 4 if c["storage"] == "fp32" else 2
    B, nin, nout = c["batch"], c["nlat_in"] * c["nlon_in"], c["nlat_out"] * c["nlon_out"]
    C, Ck, Cv, nh = c["channels"], c["k_channels"], c["out_channels"], c["heads"]
    ck, cv, pairs = Ck / nh, Cv / nh, _pairs(c)
    fwd_att, bwd_att = 2 * pairs * (ck + cv), 2 * pairs * (3 * ck + 2 * cv)
    if c["kind"] == "op":
        t = B * (nin * (Ck + Cv) + nout * Ck) * es
        return {"bytes": 2 * t + 2 * B * nout * Cv * es, "flops": fwd_att + bwd_att}
    if c["kind"] == "ring":
        nloc = c["nlat_out"] * (c["nlon_out"] // c["chunks"])
        read = B * (nin * (Ck + Cv) + nloc * (Ck + Cv)) * es
        write = B * (nin * (Ck + Cv) + nloc * (Ck + Cv)) * 4 + 3 * B * nh * nloc * 4
        return {"bytes": read + write, "flops": fwd_att + 2 * pairs * (3 * ck + cv) + 2 * pairs * (2 * ck + 2 * cv)}
    weights = C * (2 * Ck + Cv) + Cv * Cv
    xs = B * C * (nout if _is_self(c) else nout + nin)
    proj = 2 * B * (nout * C * Ck + nin * C * (Ck + Cv) + nout * Cv * Cv)
    out = B * nout * Cv
    ws = 4 if c["storage"] == "fp32" else 2
    os_ = 2 if c["autocast"] != "none" else es
    if c["kind"] == "infer":
        return {"bytes": xs * es + weights * ws + out * os_, "flops": proj + fwd_att}
    return {"bytes": 2 * xs * es + 2 * weights * ws + 2 * out * os_, "flops": 3 * proj + fwd_att + bwd_att}


def tolerance(case):
    """32-bit sums in another order; 16-bit: results, probabilities and activations rounded to the storage type."""
    low = {case["storage"], case["autocast"]}
    if "bf16" in low:
        return {"rel": 1e-2, "max": 0.5}
    if "fp16" in low:
        return {"rel": 3e-3, "max": 0.1}
    return {"rel": 1e-5, "max": 1e-3}


# ---- one more case of the same ranges -----------------------------------------------------------------------------------------
def _draw_once(rng):
    kind = rng.choice(["train", "train", "train", "infer", "infer", "op", "ring"])
    direction = rng.choice(["self", "self", "down", "up"])
    nlat = int(round(math.exp(rng.uniform(math.log(32), math.log(721)))))
    nlon = 2 * nlat + rng.choice([0, 0, -2, 2, 6])
    chunks = 1
    if kind == "ring":
        chunks = rng.choice([2, 3, 4, 8])
        nlon -= nlon % (2 * chunks)
    ratio = 1 if direction == "self" else rng.choice([2, 2, 3])
    fine, coarse = (nlat, nlon - nlon % ratio), (max(16, (nlat + 1) // ratio), nlon // ratio)
    if kind == "ring" and ratio > 1:
        coarse = (coarse[0], coarse[1] - coarse[1] % chunks)
        fine = (nlat, ratio * coarse[1])
    ins, outs = {"self": (fine, fine), "down": (fine, coarse), "up": (coarse, fine)}[direction]
    gi, go = rng.choice([("equiangular", "equiangular"), ("equiangular", "equiangular"), ("legendre-gauss", "legendre-gauss"), ("equiangular", "legendre-gauss"), ("lobatto", "lobatto")])
    if direction == "self":
        go = gi
    d = rng.choice([16, 16, 32, 32, 32, 64, 64, 128, 8, 20, 24, 40])
    heads = rng.choice([1, 2, 3, 4, 6, 8, 12, 16])
    channels = min(1024, d * heads)
    heads = channels // d
    channels = d * heads
    c = _case("", kind, ins, outs, rng.choice([1, 1, 2, 3, 4]), channels, heads, 0.0, grid_in=gi, grid_out=go, chunks=chunks)
    del c["name"]
    spacings = rng.uniform(1.0, 4.0)
    c["storage"], c["autocast"] = rng.choice([("fp32", "none")] * 4 + [("fp32", "bf16")] * 2 + [("fp32", "fp16"), ("bf16", "none"), ("fp16", "none")])
    if kind in ("op", "ring"):
        c["autocast"] = "none"
    if kind != "ring" and rng.random() < 0.2:
        c["out_channels"] = heads * rng.choice([8, 12, 16, 32, 64])
    if kind in ("train", "infer"):
        c["qknorm"], c["bias"] = rng.random() < 0.25, rng.random() < 0.8
        if rng.random() < 0.2:
            c["channels"] = rng.choice([24, 48, 73, 96, 128, 200, 256])
    if c["storage"] != "fp32" or c["autocast"] != "none":
        spacings = rng.uniform(1.0, 8.0)
    c["theta"] = spacings * math.pi / (min(c["nlat_in"], c["nlat_out"]) - 1)
    return c


def draw(rng):
    """A case between the listed ones: sizes over the logarithm of their range, odd ones among them, every option.  Kept below the
    largest listed case (fp32 and head widths the matrix cores do not take count for more than 16-bit work)."""
    largest = max(work(c)["flops"] for c in listed())
    while True:
        c = _draw_once(rng)
        narrow = c["storage"] != "fp32" or c["autocast"] != "none"
        slow = c["k_channels"] != c["out_channels"] or (c["k_channels"] // c["heads"]) % (8 if narrow else 4) or c["k_channels"] // c["heads"] < 16
        w = work(c)
        if w["flops"] * (64 if slow else 1 if narrow else 16) <= largest and w["bytes"] <= 1.2e10:
            return c


# ---- inputs -------------------------------------------------------------------------------------------------------------------
def _fields(shape, gen, dtype):
    """(B, C, nlat, nlon): per channel a smooth field (a coarse random one, interpolated) plus noise, of about unit variance, as
    the activations of a model on physical fields have it."""
    B, C, H, W = shape
    coarse = torch.randn(B, C, max(2, H // 16), max(2, W // 16), generator=gen, device="cuda")
    x = torch.nn.functional.interpolate(coarse, size=(H, W), mode="bilinear", align_corners=True)
    x.mul_(1.2).add_(torch.randn(shape, generator=gen, device="cuda"), alpha=0.6)
    return x.to(dtype)


def _geometry(c):
    """psi and the quadrature weights of the input rings, as the module's constructor makes them."""
    from torch_harmonics_amd import precompute_latitudes, precompute_neighborhood_s2

    ins, outs = (c["nlat_in"], c["nlon_in"]), (c["nlat_out"], c["nlon_out"])
    up = outs[1] % ins[1] == 0 and outs[1] != ins[1]
    args = (outs, ins, c["grid_out"], c["grid_in"]) if up else (ins, outs, c["grid_in"], c["grid_out"])
    col, roff, _ = precompute_neighborhood_s2(*args, theta_cutoff=c["theta"])
    quad = (2.0 * torch.pi * precompute_latitudes(ins[0], grid=c["grid_in"])[1].float() / ins[1]).contiguous()
    return col, roff, quad, up


def _prepare_module(c, gen, seed):
    from torch_harmonics_amd import NeighborhoodAttentionS2

    torch.manual_seed(seed)
    dtype = DTYPES[c["storage"]]
    m = NeighborhoodAttentionS2(
        c["channels"], (c["nlat_in"], c["nlon_in"]), (c["nlat_out"], c["nlon_out"]), grid_in=c["grid_in"], grid_out=c["grid_out"], num_heads=c["heads"],
        use_qknorm=c["qknorm"], bias=c["bias"], theta_cutoff=c["theta"], k_channels=c["k_channels"], out_channels=c["out_channels"],
    ).cuda()  # fmt: skip
    with torch.no_grad():  # parameters as they are some way into a training, not the zeros of the first step
        for n, p in m.named_parameters():
            if "bias" in n or "norm" in n:
                p.uniform_(-0.2, 0.2, generator=gen)
    quad = m.quad_weights
    m = m.to(dtype)
    m.quad_weights = quad  # 16-bit storage is for activations and parameters, the quadrature stays fp32
    train = c["kind"] == "train"
    xq = _fields((c["batch"], c["channels"], c["nlat_out"], c["nlon_out"]), gen, dtype).requires_grad_(train)
    xk = xq if _is_self(c) else _fields((c["batch"], c["channels"], c["nlat_in"], c["nlon_in"]), gen, dtype).requires_grad_(train)
    state = dict(case=c, module=m.train(train), inputs=(xq,) if xk is xq else (xq, xk, xk), leaves=[xq] if xk is xq else [xq, xk])
    if train:
        out_dtype = dtype if c["autocast"] == "none" else DTYPES[c["autocast"]]
        state["dy"] = torch.randn(c["batch"], c["out_channels"], c["nlat_out"], c["nlon_out"], generator=gen, device="cuda").to(out_dtype)
        # without q/k normalisation the softmax does not see k's bias (it adds the same to every score of a query): its gradient is
        # zero in exact arithmetic, and what a program returns for it is rounding alone
        state["params"] = [(n, p) for n, p in m.named_parameters() if c["qknorm"] or n != "k_bias"]
    return state


def _prepare_op(c, gen):
    dtype = DTYPES[c["storage"]]
    col, roff, quad, _ = _geometry(c)
    ck = c["k_channels"] // c["heads"]
    r = lambda h, w, n: torch.randn(c["batch"], h, w, n, generator=gen, device="cuda")  # noqa: E731
    k = r(c["nlat_in"], c["nlon_in"], c["k_channels"]).to(dtype).requires_grad_(True)
    v = r(c["nlat_in"], c["nlon_in"], c["out_channels"]).to(dtype).requires_grad_(True)
    q = (r(c["nlat_out"], c["nlon_out"], c["k_channels"]) / math.sqrt(ck)).to(dtype).requires_grad_(True)
    dy = r(c["nlat_out"], c["nlon_out"], c["out_channels"]).to(dtype)
    return dict(case=c, leaves=[k, v, q], dy=dy, geo=(quad.cuda(), col.cuda(), roff.cuda(), c["heads"], c["nlon_in"], c["nlat_out"], c["nlon_out"]))


def _prepare_ring(c, gen):
    """Rank 1 of `chunks`: all latitudes, its share of the output longitudes, heads folded into the batch."""
    from torch_harmonics_amd import ops

    dtype = DTYPES[c["storage"]]
    col, roff, quad, up = _geometry(c)
    Hi, Wi, Ho, Wo, n = c["nlat_in"], c["nlon_in"], c["nlat_out"], c["nlon_out"], c["chunks"]
    BB, d, dv, wloc, wchunk = c["batch"] * c["heads"], c["k_channels"] // c["heads"], c["out_channels"] // c["heads"], Wo // n, Wi // n
    lo = wloc
    if up:  # keyed by input latitude: keep the columns as output longitudes counted from the window's first one
        lat = torch.div(col, Wo, rounding_mode="floor")
        col = lat * Wo + (col - lat * Wo - lo) % Wo
        tail = [(Wi, Wo, Wo // Wi, i * wchunk, 0, Ho, wloc) for i in range(n)]
        row_idx = None
    else:
        lat = torch.div(col, Wi, rounding_mode="floor")
        col = lat * Wi + (col - lat * Wi + (Wi // Wo) * lo) % Wi
        row_idx = torch.argsort(roff[1:] - roff[:-1], descending=True, stable=True).to(torch.int32)
        tail = [(Wi, Wi // Wo, i * wchunk, 0, Ho, wloc, *ops.split_csr_rows(row_idx, roff, Ho)) for i in range(n)]
        row_idx = row_idx.cuda()
    r = lambda h, w, ch: torch.randn(BB, h, w, ch, generator=gen, device="cuda")  # noqa: E731
    kv = [(r(Hi, wchunk, d).to(dtype), r(Hi, wchunk, dv).to(dtype)) for _ in range(n)]
    q, dy = (r(Ho, wloc, d) / math.sqrt(d)).to(dtype), r(Ho, wloc, dv).to(dtype)
    return dict(case=c, up=up, kv=kv, q=q, dy=dy, quad=quad.cuda(), psi=(col.cuda(), roff.cuda()) + (() if up else (row_idx,)), tail=tail, dv=dv)


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    if case["kind"] == "op":
        return _prepare_op(case, gen)
    if case["kind"] == "ring":
        return _prepare_ring(case, gen)
    return _prepare_module(case, gen, seed)


# ---- one pass -----------------------------------------------------------------------------------------------------------------
def _run_module(s):
    c, m = s["case"], s["module"]
    cast = contextlib.nullcontext() if c["autocast"] == "none" else torch.autocast("cuda", dtype=DTYPES[c["autocast"]])
    if c["kind"] == "infer":
        with torch.no_grad(), cast:
            return m(*s["inputs"])
    for x in s["leaves"]:
        x.grad = None
    m.zero_grad(set_to_none=True)
    with cast:
        y = m(*s["inputs"])
    y.backward(s["dy"])
    return {"y": y.detach(), "inputs": [x.grad for x in s["leaves"]], "params": {n: p.grad for n, p in s["params"]}}


def _run_op(s):
    from torch_harmonics_amd import _neighborhood_s2_attention_optimized

    k, v, q = s["leaves"]
    for x in s["leaves"]:
        x.grad = None
    y = _neighborhood_s2_attention_optimized(k, v, q, *s["geo"])
    y.backward(s["dy"])
    return {"y": y.detach(), "dk": k.grad, "dv": v.grad, "dq": q.grad}


def _run_ring(s):
    from torch_harmonics_amd import ops

    q, dy, quad, psi = s["q"], s["dy"], s["quad"], s["psi"]
    B, H, W, d = q.shape
    z = lambda *ch: torch.zeros(B, H, W, *ch, device="cuda")  # noqa: E731
    y_acc, asum, qmax = z(s["dv"]), z(), torch.full((B, H, W), float("-inf"), device="cuda")
    fwd = ops.forward_ring_step_upsample if s["up"] else ops.forward_ring_step
    for (k, v), tail in zip(s["kv"], s["tail"]):
        fwd(k, v, q, y_acc, asum, qmax, quad, *psi, *tail)
    y = y_acc / asum[..., None]
    integral, ak, akvw = z(), z(d), z(d)
    if not s["up"]:
        asum2, qmax2 = z(), torch.full((B, H, W), float("-inf"), device="cuda")
    for (k, v), tail in zip(s["kv"], s["tail"]):
        if s["up"]:
            ops.backward_ring_step_upsample_pass1(k, v, q, dy, qmax, integral, ak, akvw, quad, *psi, *tail)
        else:
            ops.backward_ring_step_pass1(k, v, q, dy, asum2, qmax2, integral, ak, akvw, quad, *psi, *tail)
    norm = integral / asum
    dq = (akvw - norm[..., None] * ak) / asum[..., None]
    second = ops.backward_ring_step_upsample_pass2 if s["up"] else ops.backward_ring_step_pass2
    grads = []
    for (k, v), tail in zip(s["kv"], s["tail"]):
        dk, dv = torch.zeros(k.shape, device="cuda"), torch.zeros(v.shape, device="cuda")
        second(k, v, q, dy, asum, qmax, norm, dk, dv, quad, *psi, *tail)
        grads.append((dk, dv))
    return {"y": y, "dq": dq, "grads": grads}


def run(state):
    kind = state["case"]["kind"]
    return _run_op(state) if kind == "op" else _run_ring(state) if kind == "ring" else _run_module(state)
