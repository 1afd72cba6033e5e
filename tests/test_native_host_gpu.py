"""The native host path against the general Python route: same kernels, same operands, so the same bits -- outputs, tangents,
gradients -- in every way an operator is differentiated; and the cases it hands back to the general route."""
import contextlib

import pytest
import torch
import torch.autograd.forward_ad as fwAD
from torch.utils._python_dispatch import TorchDispatchMode

import dmf_amd
from dmf_amd import _lib, block_ops, harness
from dmf_amd.dmft import DMFT
from dmf_amd.flash_attention_hip_jvp import flash_attn_projection
from dmf_amd.layers import Attention, DiTBlock, FinalLayer, Linear, Mlp, TimestepEmbedder, frozen_low_precision_params, stacked_modulations

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _general(fn):
    """``fn()`` with the native path switched off."""
    native, _lib.native = _lib.native, lambda *t: False
    try:
        return fn()
    finally:
        _lib.native = native


def _attn_case(kind, dtype):
    g = torch.Generator().manual_seed(9)
    B, L, H, D = 2, 40, 3, 64
    rnd = lambda *s: torch.randn(*s, generator=g).to(dtype).to(DEV)
    if kind == "separate":
        return dmf_amd.flash_attn_func, [rnd(B, L, H, D) for _ in range(3)]
    if kind == "views":
        return dmf_amd.flash_attn_func, list(rnd(B, L, 3, H, D).unbind(2))
    if kind == "packed":
        return dmf_amd.flash_attn_qkvpacked_func, [rnd(B, L, 3, H, D)]
    gains = [torch.rand(D, generator=g).to(DEV) + 0.5 for _ in range(2)]
    return dmf_amd.flash_attn_qknorm_qkvpacked_func, [rnd(B, L, 3, H, D), *gains]


def _all_modes(fn, args, moving):
    """Plain, no-grad, torch.func.jvp and dual-level calls, the last two with a gradient through the primal output; the first
    ``moving`` arguments carry tangents."""
    outs = []
    with torch.no_grad():
        outs.append(fn(*args))
    leaves = [a.detach().clone().requires_grad_() for a in args]
    o = fn(*leaves)
    gy = torch.linspace(-1, 1, o.numel(), device=DEV).reshape(o.shape).to(o.dtype)
    outs += [o.detach(), *torch.autograd.grad(o, leaves, gy)]
    tangents = [a.detach().flip(0) for a in args[:moving]]
    o, to = torch.func.jvp(lambda *m: fn(*m, *leaves[moving:]), tuple(leaves[:moving]), tuple(tangents))
    outs += [o.detach(), to.detach(), *torch.autograd.grad(o, leaves, gy)]
    with fwAD.dual_level():
        o, to = fwAD.unpack_dual(fn(*(fwAD.make_dual(a, t) for a, t in zip(leaves, tangents)), *leaves[moving:]))
    outs += [o.detach(), to.detach(), *torch.autograd.grad(o, leaves, gy)]
    # only one operand moves: the others' tangents are zeros
    o, to = torch.func.jvp(lambda m: fn(m, *args[1:]), (args[0],), (tangents[0],))
    return outs + [o, to]


@pytest.mark.parametrize("kind,dtype", [("separate", torch.float32), ("separate", torch.float16), ("views", torch.bfloat16),
                                        ("packed", torch.bfloat16), ("packed", torch.float32), ("qknorm", torch.bfloat16)])
def test_attention_operators_give_the_same_bits(kind, dtype):
    fn, args = _attn_case(kind, dtype)
    moving = len(args) if kind in ("separate", "views") else 1
    if kind in ("separate", "views"):
        assert _lib.host().attention(*args, None) is not None
    new, old = _all_modes(fn, args, moving), _general(lambda: _all_modes(fn, args, moving))
    assert len(new) == len(old)
    for i, (a, b) in enumerate(zip(new, old)):
        assert a.dtype == b.dtype and a.shape == b.shape and torch.equal(a, b), i


@pytest.mark.parametrize("qk_norm", [False, True])
@pytest.mark.parametrize("functorch", [True, False])
@pytest.mark.parametrize("autocast", [True, False])
def test_training_step_gives_the_same_bits(autocast, functorch, qk_norm):
    """Every block operator, forward-mode and backward, through a small model."""
    torch.manual_seed(3)
    model = DMFT(input_size=16, hidden_size=256, depth=3, num_heads=4, dmf_depth=2, qk_norm=qk_norm, attn_func="hip", block_ops="hip")
    model = model.to(DEV).init_trunc_normal_()
    batch = harness.synthetic_batch(3, DEV, input_size=16)

    def step():
        model.zero_grad(set_to_none=True)
        loss = harness.train_step(model, batch, autocast=autocast, functorch=functorch)
        return [loss.detach()] + [p.grad for p in model.parameters() if p.requires_grad]

    for i, (a, b) in enumerate(zip(step(), _general(step))):
        assert torch.equal(a, b), i


def test_what_the_native_path_hands_back():
    q = torch.randn(2, 16, 2, 64, device=DEV)
    host = _lib.host()
    assert host.attention(q, q, q, None) is not None
    assert host.attention(q.cpu(), q.cpu(), q.cpu(), None) is None                      # not on the GPU
    assert host.attention(q[..., :40], q[..., :40], q[..., :40], None) is None           # head dim without a kernel
    assert host.attention(q.transpose(2, 3), q.transpose(2, 3), q.transpose(2, 3), None) is None
    assert host.attention(q.double(), q.double(), q.double(), None) is None
    seen = []
    torch.func.jvp(lambda x: torch.func.jvp(lambda y: (seen.append(host.attention(y, y, y, None)), y)[1], (x,), (x,))[0], (q,), (q,))
    assert seen == [None]                                                                # two levels
    x = torch.randn(2, 8, 64, device=DEV)
    m = torch.randn(2, 64, device=DEV)
    with torch.enable_grad():   # saved tensors are freed with the first backward, as for any node
        y = block_ops.ln_modulate(x.requires_grad_(), m, m)
        y.sum().backward()
        with pytest.raises(RuntimeError, match="second time"):
            y.sum().backward()
        z = x * 1.0
        y = block_ops.ln_modulate(z, m, m)
        z.mul_(2.0)             # and modifying one in place is caught
        with pytest.raises(RuntimeError, match="inplace"):
            y.sum().backward()


def test_qknorm_backward_of_far_apart_gradient_rows():
    """Rows of the output gradient 2 GiB / (L + 256) or more apart (time-major, a very large batch): no kernel has the norms' backward in its
    epilogue there, so attention and norms run one after the other, as on the general route, whose bits these are."""
    fn, (qkv, qg, kg) = _attn_case("qknorm", torch.bfloat16)
    B, L, _, H, D = qkv.shape
    row = (1 << 31) // (2 * (L + 256)) // 8 * 8 + 8
    gy = torch.empty(L * row, device=DEV, dtype=torch.bfloat16).as_strided((B, L, H, D), (H * D, row, D, 1))
    gy.copy_(torch.linspace(-1, 1, B * L * H * D, device=DEV).view(B, L, H, D))

    def grads():
        leaves = [t.detach().clone().requires_grad_() for t in (qkv, qg, kg)]
        return torch.autograd.grad(fn(*leaves), leaves, gy)

    for got, exp in zip(grads(), _general(grads)):
        assert got.dtype == exp.dtype and torch.equal(got, exp)


def test_gradients_at_tangent_outputs():
    """Attention drops them, the block operators refuse them -- attached to a loss together with the primal output or alone."""
    q, t = torch.randn(2, 16, 2, 64, device=DEV, requires_grad=True), torch.randn(2, 16, 2, 64, device=DEV)
    o, to = torch.func.jvp(lambda x: dmf_amd.flash_attn_func(x, x, x), (q,), (t,))
    assert to.requires_grad
    both, alone = torch.autograd.grad((o.sum() + to.sum()), q, retain_graph=True)[0], torch.autograd.grad(o.sum(), q)[0]
    assert torch.equal(both, alone)
    x, tx = torch.randn(2, 8, 64, device=DEV, requires_grad=True), torch.randn(2, 8, 64, device=DEV)
    m, w = torch.randn(2, 64, device=DEV), torch.randn(128, 64, device=DEV)
    for fn in (lambda x: block_ops.ln_modulate(x, m, m), lambda x: block_ops.gate_residual(x, m, x), block_ops.gelu_tanh, block_ops.silu,
               lambda x: block_ops.residual_ln_modulate(x, m, x, m, m)[0], lambda x: block_ops.residual_ln_modulate(x, m, x, m, m)[1],
               lambda x: block_ops.dual_linear(x, w), lambda x: block_ops.chunk_last(x, 2)[1]):
        y, ty = torch.func.jvp(fn, (x,), (tx,))
        torch.autograd.grad(y.sum(), x, retain_graph=True)
        with pytest.raises(NotImplementedError, match="primal output only"):
            (y.sum() + ty.sum()).backward()
        # only the tangent asks for a gradient: none, and no error, as on the general route
        _, ty = torch.func.jvp(fn, (x.detach(),), (tx.clone().requires_grad_(),))
        assert ty.requires_grad


@pytest.mark.parametrize("op", ["packed", "qknorm", "linear"])
def test_in_place_changes_of_reshaped_operands_are_noticed(op):
    gains = torch.ones(64, device=DEV)
    x = torch.randn(2, 16, 3 * 128, device=DEV, requires_grad=True)
    z = (x * 1.0).to(torch.bfloat16)
    if op == "linear":
        y = block_ops.dual_linear(z, torch.randn(64, 384, device=DEV, dtype=torch.bfloat16, requires_grad=True))
    else:
        y = flash_attn_projection(z, 2, *((gains, gains) if op == "qknorm" else ()))
    z.mul_(2.0)
    with pytest.raises(RuntimeError, match="inplace"):
        y.sum().backward()


def test_chunks_are_views():
    """In-place writes to a chunk: refused where the chunk has history, a change of the whole tensor elsewhere."""
    x = torch.randn(2, 1, 192, device=DEV, requires_grad=True)
    z = x * 1.0
    part = block_ops.chunk_last(z, 3)[1]
    assert part._is_view() and part._base is z
    with pytest.raises(RuntimeError, match="view"):
        part.mul_(2.0)
    y = z.square()   # saves z
    with torch.no_grad():
        block_ops.chunk_last(z, 3)[0].zero_()
    assert z._version == 1
    with pytest.raises(RuntimeError, match="inplace"):
        y.sum().backward()


def test_linear_and_chunk_stay_twice_differentiable():
    torch.manual_seed(1)
    x = torch.randn(3, 5, 64, device=DEV, requires_grad=True)
    w, b = torch.randn(32, 64, device=DEV, requires_grad=True), torch.randn(32, device=DEV, requires_grad=True)

    def second(linear, chunk):
        a, c = chunk(linear(x, w, b), 2)
        gx, gw, gb = torch.autograd.grad((a * c).sum(), (x, w, b), create_graph=True)
        return torch.autograd.grad(gx.square().sum() + gw.square().sum() + gb.square().sum(), (x, w))

    for got, exp in zip(second(block_ops.dual_linear, block_ops.chunk_last), second(torch.nn.functional.linear, lambda t, n: t.chunk(n, -1))):
        # two library products of 64 to 480 terms in fp32, in another order
        assert (got - exp).norm() <= 1e-5 * exp.norm()
    g = torch.randn(4, 3, 5, 32, device=DEV)
    batched = torch.autograd.grad(block_ops.dual_linear(x, w), (x, w), g, is_grads_batched=True)
    for i in range(4):
        for got, exp in zip(batched, torch.autograd.grad(block_ops.dual_linear(x, w), (x, w), g[i])):
            assert (got[i] - exp).norm() <= 1e-5 * exp.norm()


@pytest.mark.parametrize("route", [lambda f: f(), _general], ids=["native", "python"])
@pytest.mark.parametrize("case", ["second", "over_reverse"])
@pytest.mark.parametrize("op", ["gelu_tanh", "silu", "dual_linear"])
def test_operators_differentiated_again(op, case, route):
    """Gradients of create_graph=True differentiated once more, and gradients that carry a tangent (forward over reverse), against torch's operators in
    fp64: elementwise in fp32 and products of up to 64 terms.  The layer has the size from which its input gradient is the package's own (M 3072, bf16):
    2^-9 of each of the at most three factors that are rounded."""
    bf16 = op == "dual_linear"
    g = torch.Generator(device=DEV).manual_seed(12)
    r = lambda *s: torch.randn(*s, generator=g, device=DEV).to(torch.bfloat16 if bf16 else torch.float32)
    args = [r(3072, 192), r(64, 192)] if bf16 else [2 * r(24, 64)]
    gy, tgy = r(3072, 64) if bf16 else r(24, 64), r(3072, 64) if bf16 else r(24, 64)
    probes = [r(*a.shape) for a in args]
    assert not bf16 or _lib.load().dmf_linear_dgrad_plan(3072, 64, 192) == 1

    def run(fn, dt):
        leaves, up = [a.to(dt).requires_grad_() for a in args], gy.to(dt)
        if case == "over_reverse":
            with fwAD.dual_level():
                return [fwAD.unpack_dual(t).tangent for t in torch.autograd.grad(fn(*leaves), leaves, fwAD.make_dual(up, tgy.to(dt)))]
        up.requires_grad_()
        grads = torch.autograd.grad(fn(*leaves), leaves, up, create_graph=True)
        return torch.autograd.grad(sum((a * p.to(dt)).sum(dtype=torch.float32 if bf16 and dt != torch.float64 else dt) for a, p in zip(grads, probes)), [*leaves, up])

    ref = {"gelu_tanh": lambda x: torch.nn.functional.gelu(x, approximate="tanh"), "silu": lambda x: x * torch.sigmoid(x), "dual_linear": torch.nn.functional.linear}[op]
    got, exp = route(lambda: run(getattr(block_ops, op), args[0].dtype)), run(ref, torch.float64)
    for a, e in zip(got, exp):
        assert a is not None and (a.double() - e).norm() <= (3 * 2 ** -9 if bf16 else 1e-5) * e.norm()


def test_graphs_that_never_run_backward_are_freed():
    """A gradient-enabled call whose results are dropped without a backward pass leaves nothing behind: a node that holds its own output
    would keep the graph above it."""
    torch.manual_seed(6)
    model = DMFT(input_size=16, hidden_size=256, depth=2, num_heads=4, dmf_depth=1, attn_func="hip", block_ops="hip").to(DEV).init_trunc_normal_()
    x, c = torch.randn(2, 4, 16, 16, device=DEV), torch.randn(2, 1, 3 * 64, device=DEV, requires_grad=True)
    t, y = torch.rand(2, device=DEV), torch.zeros(2, dtype=torch.long, device=DEV)
    calls = (lambda: block_ops.chunk_last(c * 1.0, 3), lambda: model(x, t, t, y), lambda: block_ops.dual_linear(c * 1.0, torch.randn(64, 192, device=DEV)),
             lambda: torch.func.jvp(lambda v: block_ops.chunk_last(v * 1.0, 3)[0], (c,), (c.detach(),)),
             lambda: dmf_amd.flash_attn_qkvpacked_func((c * torch.ones(2, 40, 1, device=DEV)).view(2, 40, 3, 1, 64)))
    for i, call in enumerate(calls):
        call()
        held = []
        for _ in range(3):
            call()
            held.append(torch.cuda.memory_allocated())
        assert held[0] == held[-1], (i, held)


@pytest.mark.parametrize("autocast", [False, True])
def test_linear_under_two_jvp_levels(autocast):
    """The second directional derivative of linear(x * x) and the mixed parts, against the same nesting of torch's own linear: bf16 operands
    in the sizes that the package's product kernel takes (the values of x are small integers, so x * x and its derivatives are exact in bf16
    and both sides round the same fp32 sums once: 2^-8 of an element apart at most)."""
    M, N, K = 64, 128, 64
    assert _lib.load().dmf_linear_plan(M, N, K, 1, 0) == 1
    g = torch.Generator(device=DEV).manual_seed(2)
    x, t = (torch.randint(-4, 5, (M, K), generator=g, device=DEV).to(torch.float32 if autocast else torch.bfloat16) for _ in range(2))
    w, b = torch.randn(N, K, generator=g, device=DEV).bfloat16(), torch.randn(N, generator=g, device=DEV).bfloat16()
    if autocast:
        w, b = w.float(), b.float()

    def twice(linear):
        inner = lambda x: torch.func.jvp(lambda y: linear(y * y, w, b), (x,), (t,))
        with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16, enabled=autocast):
            (o, to), (o2, to2) = torch.func.jvp(inner, (x,), (t,))
        return o, to, o2, to2

    for got, exp in zip(twice(block_ops.dual_linear), twice(torch.nn.functional.linear)):
        assert float(exp.float().norm()) > 0 and float((got.float() - exp.float()).norm()) <= 2 ** -8 * float(exp.float().norm())


def test_tangents_of_incoming_gradients():
    """Forward over reverse: a gradient that carries a tangent at a dual level gives input gradients that carry theirs."""
    torch.manual_seed(5)
    x, w, b = torch.randn(6, 64, device=DEV, requires_grad=True), torch.randn(32, 64, device=DEV, requires_grad=True), torch.randn(32, device=DEV, requires_grad=True)
    g, tg = torch.randn(6, 32, device=DEV), torch.randn(6, 32, device=DEV)
    with fwAD.dual_level():
        grads = torch.autograd.grad(block_ops.dual_linear(x, w, b), (x, w, b), fwAD.make_dual(g, tg))
        for got, exp in zip(grads, (tg @ w, tg.t() @ x, tg.sum(0))):
            tangent = fwAD.unpack_dual(got).tangent
            assert tangent is not None and (tangent - exp).norm() <= 1e-5 * exp.norm()   # up to 64 terms in fp32
        parts = block_ops.chunk_last(x, 2)
        gx, = torch.autograd.grad(parts[1], x, fwAD.make_dual(g, tg))
        assert torch.equal(fwAD.unpack_dual(gx).tangent, torch.cat([torch.zeros_like(tg), tg], -1))


def test_traced_linear_gelu_computes():
    """torch.jit.trace records operators, not the buffers that a launch of the package's own filled while it was recorded.  Both sides round
    fp32 values once to bf16 (the library's after rounding the pre-activation as well)."""
    x, x2, w, b = (torch.randn(*s, device=DEV).bfloat16() for s in ((64, 64), (64, 64), (128, 64), (128,)))
    with torch.no_grad():
        traced = torch.jit.trace(lambda x: block_ops.linear_gelu_tanh(x, w, b), (x,), check_trace=False)
        got, exp = traced(x2).float(), block_ops.linear_gelu_tanh(x2, w, b).float()
    assert (got - exp).norm() <= 2 ** -7 * exp.norm()


def test_watched_calls_take_the_general_route():
    class Watch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    class Tagged(torch.Tensor):
        pass

    q = torch.randn(2, 16, 2, 64, device=DEV)
    host = _lib.host()
    with Watch():
        assert host.attention(q, q, q, None) is None
    assert _lib.native(q, None) and not _lib.native(q, q.as_subclass(Tagged)) and host.attention(q, q, q, None) is not None


@pytest.mark.parametrize("dual", [False, True])
@pytest.mark.parametrize("B,C,depth", [(1, 128, 1), (2, 384, 3), (31, 768, 2), (32, 640, 2), (33, 1152, 2), (64, 768, 2), (65, 1024, 1), (128, 384, 2)])
def test_stacked_modulations_against_the_blocks_own(B, C, depth, dual):
    """All adaLN projections in one launch: batches around the 32-row tiles, widths around the 128-column work-groups, one and two
    conditioning vectors, weights in bf16 and as low-precision copies under autocast.  Both sides round the same fp32 sums of products
    of bf16 numbers to bf16, so elements differ by one unit in the last place (2^-8) where the sums straddle a boundary: few."""
    torch.manual_seed(B + C)
    blocks = [DiTBlock(C, C // 64, attn_func="hip", block_ops="hip").to(DEV) for _ in range(depth)]
    final = FinalLayer(C, 2, 4, block_ops="hip").to(DEV)
    stack = torch.nn.ModuleList([*blocks, final]).requires_grad_(False)
    for p in stack.parameters():
        torch.nn.init.normal_(p, std=0.05)
    cs = [torch.randn(B, 1, C, device=DEV) for _ in range(2)]
    ts = [torch.randn(B, 1, C, device=DEV) for _ in range(2)]

    def call(c, c2):
        mods, last = stacked_modulations(blocks, [c] + [c2] * (depth - 1), final, c2)
        return [m for group in (*mods, last) for m in group]

    def run(c, c2):
        if not dual:
            return call(c, c2)
        o, to = torch.func.jvp(lambda a, b: tuple(call(a, b)), (c, c2), (ts[0].to(c.dtype), ts[1].to(c.dtype)))
        return [*o, *to]

    seen = []
    native = _lib.host().modulations
    for low in (False, True):
        if low:
            stack.bfloat16()
        args = [c.bfloat16() if low else c for c in cs]
        with contextlib.ExitStack() as ctx:
            if not low:
                ctx.enter_context(torch.autocast("cuda", dtype=torch.bfloat16))
                ctx.enter_context(frozen_low_precision_params(stack))
            new, old = run(*args), _general(lambda: run(*args))
            seen.append(native([args[0]], [0, 0], [blocks[0].adaLN_modulation[1].weight, final.adaLN_modulation[1].weight], [None, None],
                               *([m.adaLN_modulation[1].lp_weight for m in (blocks[0], final)], [None, None]), 6, 2) is not None)
        assert len(new) == len(old) == (6 * depth + 2) * (2 if dual else 1)
        for a, b in zip(new, old):
            assert a.dtype == b.dtype == torch.bfloat16 and a.shape == b.shape and a.stride() == b.stride()
            assert (a.float() - b.float()).abs().max() <= 2 ** -7 * b.float().abs().max() and (a != b).float().mean() <= 0.02
    assert seen == [True, True]


def test_stacked_modulations_leave_to_the_blocks():
    C = 256
    blk, final = DiTBlock(C, 4, attn_func="hip", block_ops="hip").to(DEV).bfloat16(), FinalLayer(C, 2, 4, block_ops="hip").to(DEV).bfloat16()
    host, taken = _lib.host(), []

    class Spy:
        def __getattr__(self, name):
            return getattr(host, name)

        def modulations(self, *a):
            taken.append(host.modulations(*a) is not None)
            return host.modulations(*a)

    def tries(c):
        taken.clear()
        real, _lib.host = _lib.host, Spy
        try:
            stacked_modulations([blk], [c], final, c)
        finally:
            _lib.host = real
        return list(taken)

    c = torch.randn(4, 1, C, device=DEV, dtype=torch.bfloat16)
    assert tries(c) == []                       # parameters ask for gradients
    with torch.no_grad():
        assert tries(c) == [True]
        with pytest.raises(RuntimeError, match="dtype"):   # fp32 outside of autocast is refused as ever
            tries(c.float())
        assert taken == [False]
        assert tries(torch.randn(129, 1, C, device=DEV, dtype=torch.bfloat16)) == [False]
        calls = []
        handle = blk.adaLN_modulation[0].register_forward_hook(lambda *a: calls.append(1))
        assert tries(c) == [] and calls == [1]  # hooks see their module's call
        handle.remove()
    blk.requires_grad_(False), final.requires_grad_(False)
    assert tries(c) == [True] and tries(c.requires_grad_()) == [False]


@pytest.mark.parametrize("C,H,L", [(128, 2, 24), (1152, 16, 40), (384, 6, 333)])
@pytest.mark.parametrize("dtype,qk_norm,autocast", [(torch.float32, False, True), (torch.float32, True, True), (torch.float32, True, False),
                                                   (torch.bfloat16, False, False)])
def test_block_in_one_call(dtype, qk_norm, autocast, C, H, L):
    """A block as one native call and as its modules one by one: the same bits in every way it is differentiated, with frozen weights too."""
    torch.manual_seed(3)
    blk = DiTBlock(C, H, qk_norm=qk_norm, attn_func="hip", block_ops="hip").to(DEV, dtype)
    rnd = lambda *s: torch.randn(*s, device=DEV).to(dtype)
    x, z, mods, nxt = rnd(2, L, C), rnd(2, L, C), [rnd(2, 1, C) for _ in range(6)], [rnd(2, 1, C) for _ in range(2)]
    params = list(blk.parameters())[:-2]   # (the modulation's own layer is not part of it)

    def every_mode():
        call = lambda x, z, *m: blk.forward_chained(x, z, m, *nxt, 1e-6)
        with torch.autocast("cuda", dtype=torch.bfloat16, enabled=autocast):
            with torch.no_grad():
                outs = [*call(x, z, *mods)]
            leaves = [t.clone().requires_grad_() for t in (x, z, *mods)]
            y = call(*leaves)
            for weights in (True, False):
                blk.requires_grad_(weights)
                y, ty = torch.func.jvp(call, tuple(leaves), tuple(t.detach().flip(-1) for t in leaves))
                outs += [*y, *ty]
                grads = torch.autograd.grad([t.float().square().sum() for t in y], leaves + (params if weights else []), allow_unused=True)
                outs += [g for g in grads if g is not None]
            blk.requires_grad_(True)
        return outs

    layers, one_call = [], DiTBlock._one_call
    try:
        DiTBlock._one_call = lambda self, *a: layers.append(one_call(self, *a)) or layers[-1]
        got = every_mode()
        assert len(layers) == 4 and all(l is not None for l in layers)
        DiTBlock._one_call = lambda self, *a: None
        ref = every_mode()
    finally:
        DiTBlock._one_call = one_call
    assert len(got) == len(ref) and all(torch.equal(a, b) for a, b in zip(got, ref))


def test_block_with_hooks_or_replaced_parts_is_not_one_call():
    blk = DiTBlock(128, 2, attn_func="hip", block_ops="hip").to(DEV)
    x = torch.randn(2, 24, 128, device=DEV)
    assert blk._one_call(x, x) is not None
    for module in (blk.attn, blk.attn.qkv, blk.attn.proj, blk.mlp, blk.mlp.fc1, blk.mlp.fc2):
        for hook in (module.register_forward_hook, module.register_forward_pre_hook, module.register_full_backward_hook):
            handle = hook(lambda *a: None)
            assert blk._one_call(x, x) is None
            handle.remove()
        module.forward = type(module).forward.__get__(module)
        assert blk._one_call(x, x) is None
        del module.forward
        module.compile()   # (nothing is compiled before the first call)
        assert blk._one_call(x, x) is None
        module._compiled_call_impl = None
    assert blk._one_call(x, x) is not None


def test_block_with_modulations_of_a_class_of_their_own_is_not_one_call():
    """Gates, shifts and scales whose class has a __torch_function__: it sees the operators, as it did one by one."""
    class Watching(torch.Tensor):
        seen = []

        @classmethod
        def __torch_function__(cls, func, types, args=(), kwargs=None):
            cls.seen.append(func)
            return super().__torch_function__(func, types, args, kwargs or {})

    blk = DiTBlock(128, 2, attn_func="hip", block_ops="hip").to(DEV).requires_grad_(False)
    x, mods = torch.randn(2, 24, 128, device=DEV), [torch.randn(2, 1, 128, device=DEV) for _ in range(8)]
    ref = blk.forward_chained(x, x, mods[:6], *mods[6:], 1e-6)
    assert blk._one_call(x, x, *mods[2:]) is not None
    for i in range(2, 8):
        own = [m.as_subclass(Watching) if k == i else m for k, m in enumerate(mods)]
        assert blk._one_call(x, x, *own[2:]) is None
        Watching.seen.clear()
        got = blk.forward_chained(x, x, own[:6], *own[6:], 1e-6)
        assert Watching.seen and all(torch.equal(g.as_subclass(torch.Tensor), r) for g, r in zip(got, ref))


@pytest.mark.parametrize("cls", [Attention, Mlp, Linear])
def test_block_honours_a_forward_replaced_on_a_class(cls, monkeypatch):
    blk = DiTBlock(128, 2, attn_func="hip", block_ops="hip").to(DEV).requires_grad_(False)
    x, mods = torch.randn(2, 24, 128, device=DEV), [torch.randn(2, 1, 128, device=DEV) for _ in range(8)]
    call, calls, forward = lambda: blk.forward_chained(x, x, mods[:6], *mods[6:], 1e-6), [], cls.forward
    ref = call()
    monkeypatch.setattr(cls, "forward", lambda self, *a: calls.append(self) or forward(self, *a))
    got = call()
    assert calls and all(torch.equal(g, r) for g, r in zip(got, ref))


def test_stacked_modulations_honour_replaced_and_compiled_parts(monkeypatch):
    blk, final = DiTBlock(128, 2, attn_func="hip", block_ops="hip").to(DEV, torch.bfloat16), FinalLayer(128, 2, 4, block_ops="hip").to(DEV, torch.bfloat16)
    blk.requires_grad_(False), final.requires_grad_(False)
    c = torch.randn(2, 1, 128, device=DEV).bfloat16()
    ref, calls = stacked_modulations([blk], [c], final, c), []
    flat = lambda out: [*out[0][0], *out[1]]
    for owner, name in ((Linear, "forward"), (DiTBlock, "modulation"), (FinalLayer, "modulation")):
        method = getattr(owner, name)
        with monkeypatch.context() as m:
            m.setattr(owner, name, lambda self, *a: calls.append(owner) or method(self, *a))
            got = stacked_modulations([blk], [c], final, c)
        # (bf16 results of sums in another order: a rounding each, 2^-8 of the value; sums near zero differ by 128 terms' fp32 roundings)
        assert owner in calls and all(torch.allclose(g, r, rtol=2 ** -7, atol=1e-3) for g, r in zip(flat(got), flat(ref)))


@pytest.mark.parametrize("view", [lambda t: t[:, 1:], lambda t: t.transpose(0, 1), lambda t: t[..., :128]])
@pytest.mark.parametrize("both", [True, False])
def test_linear_under_autocast_on_rows_that_have_to_be_copied(view, both):
    """fp32 tokens that are no rows in memory, primal and tangent (or the primal alone): the bits of the dense call, with the weights
    cast per call or kept."""
    width = view(torch.empty(3, 9, 192)).shape[-1]
    x, tx = (view(torch.randn(3, 9, 192, device=DEV)) for _ in range(2))
    if not both:
        tx = tx.contiguous()
    layer = Linear(width, 256, block_ops="hip").to(DEV).requires_grad_(False)
    fns = [layer, lambda t: block_ops.linear_gelu_tanh(t, layer.weight, layer.bias, layer.lp_weight, layer.lp_bias)]
    with torch.autocast("cuda", dtype=torch.bfloat16):
        for kept in (contextlib.nullcontext(), frozen_low_precision_params(layer)):
            with kept:
                for fn in fns:
                    got, ref = (torch.func.jvp(fn, (a,), (b,)) for a, b in ((x, tx), (x.contiguous(), tx.contiguous())))
                    assert all(torch.equal(g, r) for g, r in zip(got, ref))
                    assert torch.equal(fn(x), ref[0])


def test_views_that_stand_for_the_negative_of_their_buffer():
    """torch._neg_view of fp32 operands: the values of the negated tensor, under autocast (one cast for all operands) and without."""
    x, t = torch.randn(3, 8, 128, device=DEV), torch.rand(16, device=DEV)
    layer, emb = Linear(128, 256, block_ops="hip").to(DEV), TimestepEmbedder(128, block_ops="hip").to(DEV)
    fns = [(layer, x), (lambda a: block_ops.linear_gelu_tanh(a, layer.weight, layer.bias), x), (emb, t), (block_ops.gelu_tanh, x),
           (lambda a: block_ops.chunk_last(a, 2)[1], x)]
    for autocast in (True, False):
        with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16, enabled=autocast):
            for fn, a in fns:
                neg = torch._neg_view(a)
                assert neg.is_neg() and torch.equal(fn(neg), fn(-a))
                assert all(torch.equal(g, r) for g, r in zip(torch.func.jvp(fn, (neg,), (neg,)), torch.func.jvp(fn, (-a,), (-a,))))
    part = block_ops.chunk_last(torch._neg_view(x), 2)[0]
    x[0, 0, 0] = 5.0
    assert part[0, 0, 0] == -5.0


def test_gradients_that_stand_for_the_negative_of_their_buffer():
    """A torch._neg_view as an incoming gradient, and zeros without storage: the gradients of the ordinary tensors, on the native and on the Python
    route of every operator."""
    r = lambda *s: torch.randn(*s, device=DEV)
    cases = [_attn_case(k, torch.bfloat16) for k in ("separate", "packed", "qknorm")]
    cases += [(block_ops.ln_modulate, [r(2, 16, 64), r(2, 64), r(2, 64)]), (block_ops.gate_residual, [r(2, 16, 64), r(2, 64), r(2, 16, 64)]),
              (block_ops.gelu_tanh, [r(3, 64)]), (block_ops.silu, [r(3, 64)]), (block_ops.rms_norm, [r(2, 16, 2, 64), r(64)]),
              (lambda *a: torch.cat(block_ops.residual_ln_modulate(*a)), [r(2, 16, 64), r(2, 64), r(2, 16, 64), r(2, 64), r(2, 64)])]
    for fn, args in cases:
        def grads(gy):
            leaves = [a.detach().clone().requires_grad_() for a in args]
            return torch.autograd.grad(fn(*leaves), leaves, gy)
        gy = torch.randn_like(fn(*args))
        zero = torch._efficientzerotensor(gy.shape, dtype=gy.dtype, device=DEV)
        for route in (lambda f: f(), _general):
            plain = route(lambda: grads(gy))
            assert all(torch.equal(g, e) for g, e in zip(route(lambda: grads(torch._neg_view(-gy))), plain))
            assert not any(bool(g.any()) for g in route(lambda: grads(zero)))


def test_what_saved_tensor_hooks_hand_back():
    """Other strides are read (or copied) and another type is cast; what is not of the saved tensor's device and sizes is refused: nothing is read past its
    end, or through a host address."""
    r = lambda *s: torch.randn(*s, device=DEV)
    cases = [_attn_case(k, torch.bfloat16) for k in ("separate", "packed", "qknorm")]
    cases += [(block_ops.ln_modulate, [r(2, 16, 64), r(2, 64), r(2, 64)]), (block_ops.gate_residual, [r(2, 16, 64), r(2, 64), r(2, 16, 64)]),
              (block_ops.gelu_tanh, [r(3, 64)]), (block_ops.silu, [r(3, 64)]), (block_ops.dual_linear, [r(3, 64), r(32, 64), r(32)])]
    for fn, args in cases:
        def grads(pack, unpack):
            leaves = [a.detach().clone().requires_grad_() for a in args]
            with torch.autograd.graph.saved_tensors_hooks(pack, unpack):
                y = fn(*leaves)
            return torch.autograd.grad(y, leaves, torch.linspace(-1, 1, y.numel(), device=DEV).reshape(y.shape).to(y.dtype))
        same = lambda t: t
        plain = grads(same, same)
        for got, exp in zip(grads(lambda t: t.mT.contiguous() if t.dim() > 1 else t, lambda t: t.mT if t.dim() > 1 else t), plain):
            assert (got - exp).norm() <= 2 ** -8 * exp.norm()   # (the same kernels; a layer's products in another layout)
        assert all(torch.equal(g, e) for g, e in zip(grads(lambda t: t.cpu(), lambda t: t.to(DEV)), plain))
        if fn not in (block_ops.gelu_tanh, block_ops.silu, block_ops.dual_linear):   # (these compute in the type that they get)
            assert all(torch.equal(g, e) for g, e in zip(grads(same, lambda t: t.double()), plain))
        for unpack in (lambda t: t.cpu(), lambda t: t[:1] if t.dim() > 1 else t[:-8]):
            with pytest.raises(RuntimeError, match="hook handed back"):
                grads(same, unpack)
            with pytest.raises((RuntimeError, ValueError)):
                _general(lambda: grads(same, unpack))
        assert all(torch.equal(g, e) for g, e in zip(_general(lambda: grads(lambda t: t.cpu(), lambda t: t.to(DEV))), _general(lambda: grads(same, same))))
