"""
The layer where something looks at the operators it runs - tracers, FLOP counters, selective checkpoints, batched gradients - against
the layer on its own: the same kernels on the same operands, so the same bits.
"""

import pytest
import torch
from torch.fx.experimental.proxy_tensor import make_fx

pytestmark = pytest.mark.gpu

OPTIONS = {
    "c64h2": {},
    "c64h2_norm": dict(use_qknorm=True),
    "c24h2_nobias": dict(channels=24, bias=False),
    "bf16": dict(dtype=torch.bfloat16),
    "cross": dict(cross=True),
    "channels_last": dict(layout=torch.channels_last),
}


@pytest.fixture(params=OPTIONS)
def layer(request):
    """(f, leaves, y shape): f(*leaves) is the layer on the inputs and parameters in `leaves`."""
    from torch_harmonics_amd import NeighborhoodAttentionS2

    o = dict(channels=64, dtype=torch.float32, cross=False, layout=torch.contiguous_format)
    o.update({k: v for k, v in OPTIONS[request.param].items() if k in o})
    torch.manual_seed(5)
    kw = {k: v for k, v in OPTIONS[request.param].items() if k not in o}
    ins, outs = ((16, 64), (8, 32)) if o["cross"] else ((12, 64), (12, 64))
    m = NeighborhoodAttentionS2(o["channels"], ins, outs, num_heads=2, theta_cutoff=0.6, **kw).cuda()
    with torch.no_grad():
        for n, p in m.named_parameters():
            if "bias" in n or "norm" in n:
                p.uniform_(-0.2, 0.2)
    m = m.to(o["dtype"])
    shapes = [(2, o["channels"], *outs)] + ([(2, o["channels"], *ins)] if o["cross"] else [])
    return m, [torch.randn(s, device="cuda").to(o["dtype"]).contiguous(memory_format=o["layout"]) for s in shapes]


def _call(m, xs):
    return m(xs[0]) if len(xs) == 1 else m(xs[0], xs[1], xs[1])


def _fresh(xs):
    return [torch.randn_like(x) for x in xs]


def test_graph_traced_from_the_layer(layer):
    m, xs = layer
    with torch.no_grad():
        g = make_fx(lambda *t: _call(m, t))(*xs)
        new = _fresh(xs)
        assert torch.equal(g(*new), _call(m, new))


def test_graph_traced_from_the_layer_and_its_gradients(layer):
    m, xs = layer

    def step(dy, *t):
        y = _call(m, t)
        return (y, *torch.autograd.grad(y, [*t, *m.parameters()], dy))

    leaves = [x.requires_grad_() for x in xs]
    dy = torch.randn_like(_call(m, leaves))
    g = make_fx(step)(dy, *leaves)
    new = [x.requires_grad_() for x in _fresh(xs)]
    dy = torch.randn_like(dy)
    for a, b in zip(g(dy, *new), step(dy, *new)):
        assert torch.equal(a, b)


def test_graph_traced_from_the_gradients_of_a_layer_that_ran_before(layer):
    m, xs = layer
    leaves = [x.requires_grad_() for x in xs]
    y = _call(m, leaves)
    grads = lambda dy: torch.autograd.grad(y, [*leaves, *m.parameters()], dy, retain_graph=True)  # noqa: E731
    g = make_fx(grads)(torch.ones_like(y))
    dy = torch.randn_like(y)
    for a, b in zip(g(dy), grads(dy)):
        assert torch.equal(a, b)


def test_batched_gradients(layer):
    m, xs = layer
    leaves = [x.requires_grad_() for x in xs]
    y = _call(m, leaves)
    wrt = [*leaves, *m.parameters()]
    dy = torch.randn(3, *y.shape, device="cuda").to(y.dtype)
    batched = torch.autograd.grad(y, wrt, dy, is_grads_batched=True, retain_graph=True)
    for i in range(3):
        for a, b in zip(batched, torch.autograd.grad(y, wrt, dy[i], retain_graph=True)):
            assert torch.equal(a[i], b)


def test_flop_counter_and_selective_checkpoint_see_the_layer(layer):
    from functools import partial

    from torch.utils.checkpoint import CheckpointPolicy, checkpoint, create_selective_checkpoint_contexts
    from torch.utils.flop_counter import FlopCounterMode

    m, xs = layer
    leaves = [x.requires_grad_() for x in xs]
    points = [x.shape[0] * x.shape[2] * x.shape[3] for x in (xs[0], xs[-1])]  # of the output grid and of the input grid
    c = xs[0].shape[1]
    products = 2 * c * c * (2 * points[0] + 2 * points[1])
    with FlopCounterMode(display=False) as forward:
        y = _call(m, leaves)
    with FlopCounterMode(display=False) as backward:
        y.backward(torch.ones_like(y))
    assert forward.get_total_flops() == products and backward.get_total_flops() == 2 * products
    want = [t.grad.clone() for t in (*leaves, *m.parameters())]
    m.zero_grad()
    for x in leaves:
        x.grad = None
    y = _call(m, leaves)
    with FlopCounterMode(display=False) as backward:  # (of a layer that ran before the counter)
        y.backward(torch.ones_like(y))
    assert backward.get_total_flops() == 2 * products

    seen = set()

    def policy(ctx, op, *args, **kwargs):
        seen.add(str(op))
        return CheckpointPolicy.MUST_SAVE if "layer_forward" in str(op) else CheckpointPolicy.PREFER_RECOMPUTE

    y = checkpoint(lambda *t: _call(m, t), *leaves, use_reentrant=False, context_fn=partial(create_selective_checkpoint_contexts, policy))
    got = torch.autograd.grad(y, [*leaves, *m.parameters()], torch.ones_like(y))
    assert "s2attn_kernels.layer_forward.default" in seen
    for a, b in zip(got, want):
        assert torch.equal(a, b)


def test_functorch_transforms_are_refused(layer):
    """autograd functions of this kind take no functorch transform: an error, never a result without its derivative."""
    m, xs = layer
    with pytest.raises(RuntimeError, match="functorch"):
        torch.func.vmap(lambda *t: _call(m, t))(*[torch.stack([x, x]) for x in xs])
    with pytest.raises(RuntimeError, match="functorch"):
        torch.func.grad(lambda *t: _call(m, t).float().sum())(*xs)


@pytest.mark.parametrize("traced", [False, True], ids=["node", "operators"])
def test_gradients_of_the_gradients_are_refused(layer, traced):
    """create_graph=True is taken, and gives the same gradients; differentiating them is an error, with respect to anything they
    depend on (a penalty on the layer's gradient must not drop out of a loss)."""
    from torch_harmonics_amd import ops

    m, xs = layer
    leaves = [x.requires_grad_() for x in xs]
    if traced:  # as under torch.compile
        import torch_harmonics_amd.attention as attention

        mp = pytest.MonkeyPatch()
        mp.setattr(attention, "module_attention", ops.module_attention_traced)
    try:
        y = _call(m, leaves)
    finally:
        if traced:
            mp.undo()
    wrt = [*leaves, *m.parameters()]
    dy = torch.randn_like(y).requires_grad_()
    plain = torch.autograd.grad(y, wrt, dy, retain_graph=True)
    graph = torch.autograd.grad(y, wrt, dy, create_graph=True)
    for a, b in zip(graph, plain):
        assert torch.equal(a, b)
    assert all(g.requires_grad for g in graph)
    penalty = sum(g.float().square().sum() for g in graph)
    for x in (leaves[0], m.q_weights, dy):
        with pytest.raises(RuntimeError, match="cannot be differentiated"):
            torch.autograd.grad(penalty, x, retain_graph=True)


def _layer_args(m, xs, compute):
    key = None if len(xs) == 1 else xs[1]
    return (
        xs[0], key, None, m.q_weights, m.k_weights, m.v_weights, m.proj_weights, m.q_bias, m.k_bias, m.v_bias, m.proj_bias, m.q_norm_weights, m.k_norm_weights, float(m.scale),
        m.quad_weights, m.psi_col_idx, m.psi_roff_idx, m.psi_plan, m._psi_plan_header, m.num_heads, m.nlat_in, m.nlon_in, m.nlat_out, m.nlon_out, compute,
    )  # fmt: skip


def test_opcheck_of_the_layer(layer):
    """Schema, fake kernels and autograd registration of both operators, with and without what the backward needs."""
    from torch_harmonics_amd import ops

    m, xs = layer
    args = _layer_args(m, [x.requires_grad_() for x in xs], xs[0].dtype)
    torch.library.opcheck(ops.layer_forward, (*args, True))
    torch.library.opcheck(ops.layer_forward, args)  # (the flag's default)
    plain = tuple(a.detach() if isinstance(a, torch.Tensor) else a for a in args)
    torch.library.opcheck(ops.layer_forward, (*plain, False))
    out, *kept = ops.layer_forward(*plain, True)
    torch.library.opcheck(ops.layer_backward, (torch.randn_like(out), *plain, *kept, [a is not None for a in plain[:13]]))


@pytest.mark.parametrize("autocast", [None, torch.bfloat16], ids=["", "autocast"])
def test_compiled_layer(layer, autocast):
    m, xs = layer
    torch._dynamo.reset()
    compiled = torch.compile(m, backend="aot_eager", fullgraph=True)
    cast = lambda: torch.autocast("cuda", dtype=autocast or torch.bfloat16, enabled=autocast is not None)  # noqa: E731
    dy = None
    results = []
    for f in (m, compiled):
        leaves = [x.detach().clone().requires_grad_() for x in xs]
        with cast():
            y = _call(f, leaves)
        dy = torch.randn_like(y) if dy is None else dy
        results.append((y, *torch.autograd.grad(y, [*leaves, *m.parameters()], dy)))
    for a, b in zip(*results):
        assert torch.equal(a, b)
    with torch.no_grad(), cast():
        assert torch.equal(_call(compiled, xs), _call(m, xs))


@pytest.mark.parametrize("options", [{}, dict(use_qknorm=True)], ids=["plain", "qknorm"])
def test_compiled_inference_keeps_nothing_for_a_backward(options):
    from torch_harmonics_amd import NeighborhoodAttentionS2

    torch._dynamo.reset()
    m = NeighborhoodAttentionS2(64, (32, 64), (32, 64), num_heads=16, theta_cutoff=0.3, **options).cuda().eval()
    compiled = torch.compile(m, backend="aot_eager", fullgraph=True)
    x = torch.randn(8, 64, 32, 64, device="cuda")
    peak = []
    with torch.no_grad():
        for f in (m, compiled):
            f(x)
            torch.cuda.synchronize()
            base = torch.cuda.memory_allocated()
            torch.cuda.reset_peak_memory_stats()
            f(x)
            peak.append(torch.cuda.max_memory_allocated() - base)
    assert peak[1] <= peak[0] + 65536, peak  # (the normaliser alone is 1 MB)
