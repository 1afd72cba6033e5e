"""The package's own product kernel (dmf_linear_fwd) against fp32 products of the same bf16 operands."""
import ctypes

import pytest
import torch

from dmf_amd import _lib, block_ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
# operands are exact and sums in fp32 (up to 4608 terms: below 1e-5); what is left is the rounding of the result to bf16, at most 2^-9 of
# an element, and for gelu an exp2 and a reciprocal good to 2^-21
TOL = 2 ** -9 * 1.05


def _operands(M, N, K, seed=0):
    g = torch.Generator(device=DEV).manual_seed(seed + M + N + K)
    r = lambda *s: torch.randn(*s, generator=g, device=DEV)
    return r(M, K).bfloat16(), r(M, K).bfloat16(), (r(N, K) * K ** -0.5).bfloat16(), r(N).bfloat16()


def _call(x, tx, w, b, gelu):
    lib, (M, K), N = _lib.load(), x.shape, w.shape[0]
    # (one row more than the result: what is written past it shows)
    y = torch.full((M + 1, N), 7.0, device=DEV, dtype=torch.bfloat16)
    ty = torch.full_like(y, 7.0) if tx is not None else None
    p = lambda t: None if t is None else t.data_ptr()
    rc = lib.dmf_linear_fwd(p(x), p(tx), p(w), p(b), p(y), p(ty), M, N, K, gelu, torch.cuda.current_stream().cuda_stream)
    assert rc == 0, rc
    for t in (y, ty):
        assert t is None or (t[M] == 7.0).all()
    return y[:M], None if ty is None else ty[:M]


def _check(got, ref):
    assert (got.float() - ref).norm() <= TOL * ref.norm()
    assert ((got.float() - ref).abs() <= 2 ** -8 * ref.abs() + 1e-5 * ref.abs().max()).all()


# edges of whatever tile is taken: one row, a row past a tile, columns that fill none, one step (which kernel runs: REACHED, below)
SIZES = [(1, 8, 64), (63, 64, 64), (65, 72, 128), (129, 200, 192), (333, 1152, 384), (4096, 768, 768), (4097, 712, 640), (2048, 2304, 768),
         (2000, 3456, 128), (8192, 2304, 768), (16384, 2304, 64), (16389, 2296, 320), (256, 768, 3072)]


@pytest.mark.parametrize("M,N,K", SIZES)
def test_products(M, N, K):
    x, tx, w, b = _operands(M, N, K)
    ref, tref = torch.nn.functional.linear(x.float(), w.float(), b.float()), tx.float() @ w.float().t()
    _check(_call(x, None, w, b, 0)[0], ref)
    _check(_call(x, None, w, None, 0)[0], ref - b.float())
    y, ty = _call(x, tx, w, b, 0)
    _check(y, ref)
    _check(ty, tref)
    gelu = lambda t: torch.nn.functional.gelu(t, approximate="tanh")
    act, tact = torch.func.jvp(gelu, (ref.double(),), (tref.double(),))
    for tangent in (None, tx):
        y, ty = _call(x, tangent, w, b, 1)
        assert (y.float() - act).norm() <= TOL * act.norm()
        if tangent is not None:
            assert (ty.float() - tact).norm() <= TOL * tact.norm()


def test_what_the_entry_refuses():
    x, tx, w, b = _operands(64, 64, 64)
    lib, p = _lib.load(), lambda t: t.data_ptr()
    y = torch.empty(64, 64, device=DEV, dtype=torch.bfloat16)
    for (M, N, K), rc in (((64, 64, 32), -3), ((64, 60, 64), -3), ((0, 64, 64), -3)):
        assert lib.dmf_linear_fwd(p(x), None, p(w), p(b), p(y), None, M, N, K, 0, None) == rc
    assert lib.dmf_linear_fwd(p(x), p(tx), p(w), p(b), p(y), None, 64, 64, 64, 0, None) == -5
    assert lib.dmf_linear_fwd(p(x) + 2, None, p(w), p(b), p(y), None, 64, 64, 64, 0, None) == -6


@pytest.mark.parametrize("dual", [False, True])
def test_layers_take_it_for_what_it_covers(dual):
    """dual_linear and linear_gelu_tanh on dense, strided, misaligned and other-typed operands: the same values as library products (two
    roundings apart at most: their pre-activation is rounded, the fused one's is not)."""
    x, tx, w, b = _operands(130, 256, 128)
    wide = torch.randn(130, 256, device=DEV).bfloat16()
    cases = [(x, tx), (wide[:, ::2], tx), (wide[:, 1:129], tx), (x.float(), tx.float()), (x.reshape(2, 65, 128), tx.reshape(2, 65, 128))]
    for i, (a, ta) in enumerate(cases):
        wt, bias = (w.float(), b.float()) if a.dtype == torch.float32 else (w, b)
        for fn, ref in ((block_ops.dual_linear, torch.nn.functional.linear),
                        (block_ops.linear_gelu_tanh, lambda t, w, b: torch.nn.functional.gelu(torch.nn.functional.linear(t, w, b), approximate="tanh"))):
            if dual:
                got = torch.func.jvp(lambda t: fn(t, wt, bias), (a,), (ta,))
                exp = torch.func.jvp(lambda t: ref(t, wt.float(), bias.float()), (a.float(),), (ta.float(),))
            else:
                with torch.no_grad():
                    got, exp = (fn(a, wt, bias),), (ref(a.float(), wt.float(), bias.float()),)
            for g, e in zip(got, exp):
                assert g.shape == e.shape and (g.float() - e).norm() <= 2 * TOL * e.norm(), (i, fn)


# ---- input gradient (dmf_linear_dgrad), N -> K: one row, rows and columns that fill no tile, one step per tile and fewer than stages, whole rounds with
# half tiles behind them, only half tiles, either tile width; exact operands and fp32 sums, so that the bound is the result's rounding
DGRAD = {"4, 2, 2, 3, 3": [(1, 64, 8), (63, 64, 64), (129, 192, 200), (4097, 640, 712), (12345, 192, 1016), (16389, 64, 2304), (2300, 448, 3064), (256, 3072, 768)],
         "4, 3, 2, 3, 2": [(2049, 768, 2296), (8193, 1152, 1152), (4100, 1024, 1016), (8192, 4608, 1152)]}


@pytest.mark.parametrize("M,N,K,tile", [(*size, tile) for tile, sizes in DGRAD.items() for size in sizes])
def test_input_gradient(M, N, K, tile):
    assert trained(1, M, N, K) == f"dmf::linear_dgrad_kernel<dmf::WalkTile<{tile}> >"
    gen = torch.Generator(device=DEV).manual_seed(M + N + K)
    # (what lies behind the last row of either operand would show if it were summed)
    g, w = torch.randn(M + 64, N, generator=gen, device=DEV).bfloat16(), (torch.randn(N + 64, K, generator=gen, device=DEV) * N ** -0.5).bfloat16()
    g[M:], w[N:] = 1e4, 1e4
    ref, lib = g[:M].float() @ w[:N].float(), _lib.load()
    for _ in range(2):
        gx = torch.full((M + 1, K), 7.0, device=DEV, dtype=torch.bfloat16)
        assert lib.dmf_linear_dgrad(g.data_ptr(), w.data_ptr(), gx.data_ptr(), M, N, K, torch.cuda.current_stream().cuda_stream) == 0
        _check(gx[:M], ref)
        assert (gx[M] == 7.0).all()


def test_input_gradient_routes():
    """A layer's input gradient, native and Python route, for dense, strided and negated gradients and with a saved weight that a hook hands back
    in another layout: the product of the bf16 operands; the general form where it is differentiated again."""
    M, N, K = 3072, 384, 768
    gen = torch.Generator(device=DEV).manual_seed(3)
    r = lambda *s: torch.randn(*s, generator=gen, device=DEV).bfloat16()
    x, w, dense = r(M, K), (r(N, K) * N ** -0.5).requires_grad_(), r(M, N)
    assert _lib.load().dmf_linear_dgrad_plan(M, N, K) == 1
    own = _lib.linear_dgrad(dense, w.detach())
    _check(own, dense.float() @ w.detach().float())
    for other in (dense[:, ::2], dense.float(), torch._neg_view(dense), r(N, M).t()):
        assert _lib.linear_dgrad(other, w.detach()) is None
    for gy in (dense, r(N, M).t(), torch._neg_view(dense), dense[:1].expand(M, N)):
        ref = gy.float() @ w.detach().float()
        a = x.clone().requires_grad_()
        _check(torch.autograd.grad(block_ops.dual_linear(a, w), a, gy)[0], ref)
        y, *_ = block_ops.DualLinearFunc.apply(a, None, w, None, None, None)
        _check(torch.autograd.grad(y, a, gy)[0], ref)
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t.t().contiguous(), lambda t: t.t()):
            y = block_ops.dual_linear(a, w)
        _check(torch.autograd.grad(y, a, gy)[0], ref)
    a, gy = x.clone().requires_grad_(), dense.clone().requires_grad_()
    gx = torch.autograd.grad(block_ops.dual_linear(a, w), a, gy, create_graph=True)[0]
    _check(torch.autograd.grad(gx, gy, x)[0], x.float() @ w.detach().float().t())


def test_input_gradient_refuses():
    g, w, lib = torch.randn(64, 64, device=DEV).bfloat16(), torch.randn(64, 64, device=DEV).bfloat16(), _lib.load()
    gx = torch.empty(64, 64, device=DEV, dtype=torch.bfloat16)
    call = lambda g, w, o, M, N, K: lib.dmf_linear_dgrad(g, w, o, M, N, K, None)
    p, q, o = g.data_ptr(), w.data_ptr(), gx.data_ptr()
    for size in ((0, 64, 64), (64, 32, 64), (64, 64, 12), (64, 64, 65544), (1 << 25, 64, 8)):
        assert call(p, q, o, *size) == -3 and lib.dmf_linear_dgrad_plan(*size) == 0
    assert call(None, q, o, 64, 64, 64) == -5 and call(p + 2, q, o, 64, 64, 64) == -6


# ---- weight gradient (dmf_linear_wgrad): products exact in fp32, sums in fp32 -- M terms in some order, error below sqrt(M) 2^-24 of the
# sum of magnitudes on random data; 2e-6 covers M = 16389 (7.6e-6 of a worst single element, checked against the largest)
WGRAD = [(1, 8, 8), (63, 64, 64), (64, 128, 192), (65, 136, 200), (129, 120, 184), (333, 1152, 1152), (2048, 384, 1536), (4097, 712, 328),
         (32768, 96, 200), (20001, 384, 384), (16389, 264, 1944)]
# linear_wgrad_wide_kernel: columns that fill no tile on either side, rows that fill no step, one tile, one split (whose sums go straight out)
WGRAD_WIDE = [(6145, 1288, 1032), (4097, 712, 2800), (250001, 184, 200), (8193, 520, 1944), (641, 4088, 3064), (8192, 4608, 1152), (6144, 1152, 4608),
              (8192, 1152, 1152), (8192, 3456, 1152), (4096, 4608, 1152), (4096, 1152, 4608), (16389, 768, 768)]


def trained(which, M, N, K):
    """What dmf_linear_train_plan calls the kernel, for 256 CUs: which 0 the kept form, 1 the input gradient, 2 the weight gradient."""
    name = ctypes.create_string_buffer(128)
    assert _lib.load().dmf_linear_train_plan(which, M, N, K, name, len(name)) == 0
    return name.value.decode()


@pytest.mark.parametrize("M,N,K", WGRAD + WGRAD_WIDE)
def test_weight_gradient(M, N, K):
    assert ("linear_wgrad_wide_kernel, " if (M, N, K) in WGRAD_WIDE else "linear_wgrad_kernel, ") in trained(2, M, N, K)
    assert ((M, N, K) == (641, 4088, 3064)) <= trained(2, M, N, K).endswith(" 1 splits")
    gen = torch.Generator(device=DEV).manual_seed(M + N + K)
    # (rows past the last hold values that would show if they were summed)
    g, x = (torch.randn(M + 64, C, generator=gen, device=DEV).bfloat16() for C in (N, K))
    g[M:], x[M:] = 1e4, 1e4
    lib = _lib.load()
    need = lib.dmf_linear_wgrad_workspace_floats(M, N, K)
    gb = torch.full((N + 4,), 7.0, device=DEV)
    out, ws = torch.full((N + 1, K), 7.0, device=DEV), torch.full((max(need, 4) + 4,), float("nan"), device=DEV)
    assert lib.dmf_linear_wgrad(g.data_ptr(), x.data_ptr(), out.data_ptr(), gb.data_ptr(), ws.data_ptr(), M, N, K, torch.cuda.current_stream().cuda_stream) == 0
    ref = g[:M].double().t() @ x[:M].double()
    sums = g[:M].double().sum(0)
    assert (gb[:N] - sums).norm() <= 2e-6 * sums.norm() and (gb[N:] == 7.0).all()
    assert (out[N] == 7.0).all() and ws[need:].isnan().all()
    assert (out[:N] - ref).norm() <= 2e-6 * ref.norm() and (out[:N] - ref).abs().max() <= 1e-5 * ref.abs().max()


def test_weight_gradient_routes():
    """Layer backward under autocast with dense and strided gradients, native and Python route: the fp32 product of the bf16 operands."""
    x, _, w, b = _operands(130, 256, 128)
    weight, bias, dense = w.float().requires_grad_(), b.float().requires_grad_(), torch.randn(130, 256, device=DEV).bfloat16()
    for gy in (dense, torch.randn(256, 130, device=DEV).bfloat16().t(), dense[:1].expand(130, 256)):
        with torch.autocast("cuda", dtype=torch.bfloat16):
            y = block_ops.dual_linear(x, weight, bias)
        gw, gb = torch.autograd.grad(y, (weight, bias), gy)
        assert (gb - gy.double().sum(0)).norm() <= 2e-6 * gy.double().sum(0).norm()
        ref = gy.double().t() @ x.double()
        assert gw.dtype == torch.float32 and (gw - ref).norm() <= 2e-6 * ref.norm()
    own = _lib.linear_wgrad(dense, x)[0]
    assert (own - dense.double().t() @ x.double()).norm() <= 2e-6 * own.norm()
    assert _lib.linear_wgrad(dense[:, ::2], x) is None and _lib.linear_wgrad(dense.float(), x.float()) is None


@pytest.mark.parametrize("M,N,K", [(130, 256, 128), (3072, 384, 768), (2048, 1152, 1152)])
def test_gradients_that_stand_for_something_else(M, N, K):
    """Gradients, inputs and saved tensors that are views of their buffer's negative, or zeros without storage: every gradient of a layer and of a
    layer with its activation is that of the ordinary tensor, to the bit, on the native and on the Python route."""
    import torch.autograd.forward_ad as fwAD
    x, tx, w, b = _operands(M, N, K)
    dense = torch.randn(M, N, device=DEV).bfloat16()
    zero = torch._efficientzerotensor((M, N), dtype=torch.bfloat16, device=DEV)
    assert zero._is_zerotensor() and torch._neg_view(dense).is_neg()

    def grads(layer, gy, x, hooks=None):
        leaves = [x.detach().requires_grad_() if not x.is_neg() else x, w.float().requires_grad_(), b.float().requires_grad_()]
        wanted = leaves[not leaves[0].requires_grad:]
        with torch.autocast("cuda", dtype=torch.bfloat16):
            if hooks:
                with torch.autograd.graph.saved_tensors_hooks(*hooks):
                    y = layer(*leaves)
            else:
                y = layer(*leaves)
        return torch.autograd.grad(y, wanted, gy)

    def kept(x, w, b):
        with fwAD.dual_level():
            return fwAD.unpack_dual(block_ops.linear_gelu_tanh(fwAD.make_dual(x, tx), w, b))[0]

    def python(x, w, b):
        return block_ops.DualLinearFunc.apply(x, None, w, b, None, None)[0]

    negated = (lambda t: torch.neg(t), lambda t: torch._neg_view(t))
    for layer in (block_ops.dual_linear, python, lambda *a: block_ops.gelu_tanh(block_ops.dual_linear(*a)), kept):
        plain, at_zero = grads(layer, dense, x), grads(layer, zero, x)
        for got, exp in zip(grads(layer, torch._neg_view(-dense), x), plain):
            assert torch.equal(got, exp)
        assert all(bool((g == 0).all()) for g in at_zero)
        for got, exp in zip(grads(layer, dense, torch._neg_view(-x)), plain[1:]):
            assert torch.equal(got, exp)
        for got, exp in zip(grads(layer, dense, x, negated), plain):
            assert torch.equal(got, exp)
    assert _lib.linear_wgrad(torch._neg_view(dense), x) is None and _lib.linear_wgrad(dense, torch._neg_view(x)) is None
    assert _lib.linear_fwd(torch._neg_view(x), None, w, b) is None


def test_weight_gradient_refuses():
    g, x = torch.randn(64, 64, device=DEV).bfloat16(), torch.randn(64, 64, device=DEV).bfloat16()
    out, lib = torch.empty(64, 64, device=DEV), _lib.load()
    call = lambda g, x, o, M, N, K: lib.dmf_linear_wgrad(g, x, o, None, None, M, N, K, None)
    p, q, o = g.data_ptr(), x.data_ptr(), out.data_ptr()
    assert call(p, q, o, 0, 64, 64) == -3 and call(p, q, o, 64, 60, 64) == -3 and call(p, q, o, 64, 64, 12) == -3
    assert call(None, q, o, 64, 64, 64) == -5 and call(p + 2, q, o, 64, 64, 64) == -6
    assert lib.dmf_linear_wgrad_workspace_floats(64, 60, 64) == -1


# sizes that the kernel whose work-groups walk through the tiles takes (256 x 192, 256 x 128; with tangents and gelu 128 rows of each): whole rounds and
# half tiles behind them, only half tiles, a row and a column block that fill neither, one step per tile and fewer steps than stages; outputs whole
WALK = [(2049, 2296, 768), (8193, 1152, 1152), (4100, 1016, 1024), (12345, 1016, 192), (16384, 2304, 64), (2300, 3064, 448)]


@pytest.mark.parametrize("M,N,K", WALK)
def test_products_of_many_tiles(M, N, K):
    x, tx, w, b = _operands(M, N, K)
    ref, tref = torch.nn.functional.linear(x.float(), w.float(), b.float()), tx.float() @ w.float().t()
    gelu = lambda t: torch.nn.functional.gelu(t, approximate="tanh")
    for _ in range(2):   # (a second launch finds its work-groups' LDS as the first left it)
        _check(_call(x, None, w, None, 0)[0], ref - b.float())
        y, ty = _call(x, tx, w, b, 0)
        _check(y, ref)
        _check(ty, tref)
    act, tact = torch.func.jvp(gelu, (ref.double(),), (tref.double(),))
    _check(_call(x, None, w, b, 1)[0], act)
    y, ty = _call(x, tx, w, b, 1)
    _check(y, act)
    _check(ty, tact)


# products of about one tile of 128 x 96 per CU and its neighbours in size, where several kernels are close: a row past a tile, a last column block of
# 8 and of 88 columns, few steps and many; single products, and pairs of half the rows
ONE_ROUND = [(2433, 776, 448), (2561, 1144, 576), (1025, 2296, 448), (2047, 1528, 768), (897, 3064, 768), (4096, 768, 3072)]


@pytest.mark.parametrize("M,N,K", ONE_ROUND)
def test_products_of_one_round(M, N, K):
    x, tx, w, b = _operands(M, N, K)
    ref, tref = torch.nn.functional.linear(x.float(), w.float(), b.float()), tx.float() @ w.float().t()
    half = M // 2 + 1
    for _ in range(2):
        _check(_call(x, None, w, b, 0)[0], ref)
        y, ty = _call(x[:half], tx[:half], w, b, 0)
        _check(y, ref[:half])
        _check(ty, tref[:half])
    act = torch.nn.functional.gelu(ref, approximate="tanh")
    assert (_call(x, None, w, b, 1)[0].float() - act).norm() <= TOL * act.norm()


# Every kernel in every mode, with what dmf_linear_fwd_plan says for 256 CUs asserted: rows and columns that fill no tile, more than one round
# where the kernel is taken there, half tiles and whole ones, one step and many, rows of more than 65536 elements
PLAIN, PAIR, GELU, GELU_PAIR = MODES = [(0, 0), (1, 0), (0, 1), (1, 1)]   # (tangents, gelu)
REACHED = [("linear_kernel<128, 192, 2", (130, 65656, 64), MODES), ("linear_kernel<128, 192, 2", (21778, 264, 128), [PLAIN, GELU]),
           ("linear_kernel<128, 64, 2", (16795, 200, 64), MODES), ("linear_kernel<128, 64, 2", (21851, 392, 128), [PLAIN, GELU]),
           ("linear_kernel<128, 64, 2", (4097, 712, 640), [PLAIN, GELU]), ("linear_kernel<128, 64, 2", (33, 72, 64), [GELU_PAIR]),
           ("linear_kernel<64, 64, 4", (33, 72, 64), [PLAIN, PAIR, GELU]), ("linear_kernel<64, 64, 4", (2049, 776, 3072), [PLAIN, GELU]),
           ("linear_kernel<64, 64, 4", (33, 65680, 128), [PAIR]),
           ("linear_walk_kernel<dmf::WalkTile<1, 3, 4, 5, 5>", (19121, 72, 576), [PLAIN, GELU]),
           ("linear_walk_kernel<dmf::WalkTile<1, 3, 4, 5, 5>", (8200, 72, 640), [PAIR]),
           ("linear_walk_kernel<dmf::WalkTile<1, 3, 4, 5, 5>", (4095, 760, 3072), [PLAIN, GELU]),
           ("linear_walk_kernel<dmf::WalkTile<1, 3, 4, 5, 5>", (2497, 1144, 1152), [PLAIN, GELU]),
           ("linear_walk_kernel<dmf::WalkTile<1, 3, 4, 5, 5>", (1024, 1528, 768), [PAIR]),
           ("linear_walk_kernel<dmf::WalkTile<4, 2, 2, 3, 3>", (23318, 392, 192), MODES),
           ("linear_walk_kernel<dmf::WalkTile<4, 2, 2, 3, 3>", (24656, 200, 64), MODES),
           ("linear_walk_kernel<dmf::WalkTile<4, 2, 2, 3, 3>", (4000, 1016, 1152), MODES),
           ("linear_walk_kernel<dmf::WalkTile<4, 3, 2, 3, 2>", (26350, 520, 128), MODES),
           ("linear_walk_kernel<dmf::WalkTile<4, 3, 2, 3, 2>", (2049, 2296, 768), MODES),
           ("linear_walk_kernel<dmf::WalkTile<4, 3, 2, 3, 2>", (7321, 1144, 1152), MODES)]


def planned(M, N, K, jvp, gelu):
    name = ctypes.create_string_buffer(128)
    assert _lib.load().dmf_linear_fwd_plan(M, N, K, jvp, gelu, name, len(name)) == 0
    return name.value.decode()


@pytest.mark.parametrize("kernel,size,modes", REACHED)
def test_every_kernel(kernel, size, modes):
    M, N, K = size
    x, tx, w, b = _operands(M, N, K)
    ref, tref = torch.nn.functional.linear(x.float(), w.float(), b.float()), tx.float() @ w.float().t()
    act, tact = torch.func.jvp(lambda t: torch.nn.functional.gelu(t, approximate="tanh"), (ref.double(),), (tref.double(),))
    for jvp, gelu in modes:
        assert planned(M, N, K, jvp, gelu) == f"dmf::{kernel}, {gelu + (jvp and gelu)}>"
        y, ty = _call(x, tx if jvp else None, w, b, gelu)
        for got, exp in ((y, act if gelu else ref), (ty, tact if gelu else tref)):
            if got is not None:
                _check(got, exp)


# 256 x 256 tiles, whose results pass through a slot of the stages: rows and columns that fill no tile, one step and two, whole and half tiles behind
# the rounds, no bias and one with its last columns past the tile
WIDE = [((16129, 1016, 64), MODES), ((16129, 2040, 128), MODES), ((8193, 3064, 768), [PLAIN, PAIR, GELU]), ((16300, 2040, 1152), MODES),
        ((21000, 1016, 192), [PAIR, GELU_PAIR]), ((57345, 248, 64), MODES)]


@pytest.mark.parametrize("size,modes", WIDE)
def test_products_of_the_widest_tiles(size, modes):
    M, N, K = size
    x, tx, w, b = _operands(M, N, K)
    ref, tref = torch.nn.functional.linear(x.float(), w.float(), b.float()), tx.float() @ w.float().t()
    act, tact = torch.func.jvp(lambda t: torch.nn.functional.gelu(t, approximate="tanh"), (ref.double(),), (tref.double(),))
    for jvp, gelu in modes:
        assert planned(M, N, K, jvp, gelu) == f"dmf::linear_walk_wide_kernel<{gelu + (jvp and gelu)}>"
        for _ in range(2):
            y, ty = _call(x, tx if jvp else None, w, b, gelu)
            for got, exp in ((y, act if gelu else ref), (ty, tact if gelu else tref)):
                if got is not None:
                    _check(got, exp)
        if not gelu:
            _check(_call(x, tx if jvp else None, w, None, 0)[0], ref - b.float())


# (one of each kernel; a walking kernel's with more columns than one wave's)
UNALIGNED = ["linear_kernel<128, 64", "linear_kernel<64, 64", "WalkTile<1, 3", "WalkTile<4, 2", "WalkTile<4, 3"]


@pytest.mark.parametrize("kernel,size", [(k, next(s for n, s, m in REACHED if k in n and PLAIN in m)) for k in UNALIGNED] + [("wide", WIDE[1][0])])
def test_bias_aligned_to_eight_bytes(kernel, size):
    """The least alignment that the entry takes, with values around the bias that would show."""
    M, N, K = size
    x, tx, w, b = _operands(M, N, K)
    around = torch.full((N + 8,), 1e4, device=DEV, dtype=torch.bfloat16)
    bias = around[4:N + 4]
    bias.copy_(b)
    assert bias.data_ptr() % 16 == 8 and kernel in planned(M, N, K, 0, 0)
    assert torch.equal(_call(x, None, w, bias, 0)[0], _call(x, None, w, b, 0)[0])
    for gelu in (0, 1):
        for got, exp in zip(_call(x, tx, w, bias, gelu), _call(x, tx, w, b, gelu)):
            assert torch.equal(got, exp)
    if _lib.load().dmf_linear_gelu_plan(M, N, K):
        outs = [[torch.empty(M, N, device=DEV, dtype=torch.bfloat16) for _ in range(3)] for _ in range(2)]
        for o, bb in zip(outs, (bias, b)):
            assert _lib.load().dmf_linear_gelu_fwd(x.data_ptr(), tx.data_ptr(), w.data_ptr(), bb.data_ptr(), *(t.data_ptr() for t in o), M, N, K,
                                                   torch.cuda.current_stream().cuda_stream) == 0
        assert all(torch.equal(*t) for t in zip(*outs))


# the MLP's first half with its pre-activation kept, in each of the three tiles: rows and columns that fill none, one step, two and many
KEPT = {"4, 3, 2, 3, 2": [(2049, 2296, 704), (8193, 4088, 128)], "4, 4, 2, 3, 2": [(16129, 1016, 64), (16300, 2040, 1152)],
        "4, 2, 2, 3, 3": [(4000, 1016, 1152), (2300, 3064, 448)]}


@pytest.mark.parametrize("M,N,K,tile", [(*size, tile) for tile, sizes in KEPT.items() for size in sizes])
def test_products_that_keep_their_pre_activation(M, N, K, tile):
    assert trained(0, M, N, K) == f"dmf::linear_walk_pre_kernel<dmf::WalkTile<{tile}> >"
    x, tx, w, b = _operands(M, N, K)
    lib, p = _lib.load(), lambda t: None if t is None else t.data_ptr()
    assert lib.dmf_linear_gelu_plan(M, N, K) == 1
    tref = tx.float() @ w.float().t()
    for bias in (b, None):
        ref = torch.nn.functional.linear(x.float(), w.float(), None if bias is None else bias.float())
        act, tact = torch.func.jvp(lambda t: torch.nn.functional.gelu(t, approximate="tanh"), (ref.double(),), (tref.double(),))
        for _ in range(2):
            out = [torch.full((M + 1, N), 7.0, device=DEV, dtype=torch.bfloat16) for _ in range(3)]
            assert lib.dmf_linear_gelu_fwd(p(x), p(tx), p(w), p(bias), *map(p, out), M, N, K, torch.cuda.current_stream().cuda_stream) == 0
            for got, exp in zip(out, (ref, act, tact)):
                _check(got[:M], exp)
                assert (got[M] == 7.0).all()


def test_the_kept_form_refuses():
    lib, t = _lib.load(), torch.zeros(4096, 64, device=DEV, dtype=torch.bfloat16)
    p = t.data_ptr()
    assert lib.dmf_linear_gelu_plan(64, 64, 64) == 0 and lib.dmf_linear_gelu_fwd(p, p, p, None, p, p, p, 64, 64, 64, None) == -3
    assert lib.dmf_linear_gelu_fwd(p, None, p, None, p, p, p, 2049, 2296, 704, None) == -5
    assert lib.dmf_linear_gelu_fwd(p + 2, p, p, None, p, p, p, 2049, 2296, 704, None) == -6


def test_mlp_first_half_with_a_backward_pass():
    """linear_gelu_tanh at a dual level with gradients: one node, whose gradients are those of the two operators' (the same kernels on the same
    pre-activation, rounded where theirs is), for every choice of what asks for one, under autocast and in bf16, and differentiated again as far as theirs."""
    import torch.autograd.forward_ad as fwAD
    M, N, K = 2049, 2296, 704
    x, tx, w, b = _operands(M, N, K)
    gy = torch.randn(M, N, device=DEV).bfloat16()
    for autocast in (True, False):
        wt, bias = (w.float(), b.float()) if autocast else (w, b)
        for ask in ((1, 1, 1), (1, 0, 0), (0, 1, 0), (0, 0, 1)):
            leaves = [t.detach().clone().requires_grad_(bool(a)) for t, a in zip((x, wt, bias), ask)]
            wanted = [t for t in leaves if t.requires_grad]
            res = []
            for fn in (block_ops.linear_gelu_tanh, lambda *a: block_ops.gelu_tanh(block_ops.dual_linear(*a))):
                with torch.autocast("cuda", dtype=torch.bfloat16, enabled=autocast), fwAD.dual_level():
                    y, ty = fwAD.unpack_dual(fn(fwAD.make_dual(leaves[0], tx), *leaves[1:]))
                res.append((y.detach(), ty.detach(), *torch.autograd.grad(y, wanted, gy)))
                if fn is block_ops.linear_gelu_tanh:
                    assert y.grad_fn.next_functions[0][0].name() == "LinearGeluTanhBackward"   # (behind unpack_dual's view)
            for got, exp in zip(*res):
                assert got.dtype == exp.dtype and got.shape == exp.shape and (got.float() - exp.float()).norm() <= 2 ** -7 * exp.float().norm()
            for got, exp in zip(res[0][2:], res[1][2:]):
                assert torch.equal(got, exp)
    a, wt = x.clone().requires_grad_(), w.clone().requires_grad_()
    with fwAD.dual_level():
        y = fwAD.unpack_dual(block_ops.linear_gelu_tanh(fwAD.make_dual(a, tx), wt, b))[0]
    gx = torch.autograd.grad(y, a, gy, create_graph=True)[0]
    assert torch.autograd.grad(gx, wt, x)[0].shape == wt.shape   # (values: test_mlp_first_half_differentiated_again)


@pytest.mark.parametrize("case", ["second", "over_reverse"])
@pytest.mark.parametrize("autocast", [True, False])
@pytest.mark.parametrize("M,N,K", [(2049, 2296, 704), (2048, 8192, 1024)])
def test_mlp_first_half_differentiated_again(case, autocast, M, N, K):
    """The gradients of the kept form differentiated once more (create_graph=True), and with an incoming gradient that carries a tangent
    (forward over reverse), against the same expressions of torch's operators in fp64 on the same operands.  The weight's copy under autocast is a
    constant where a gradient is differentiated again.  A result is the sum of at most four products of at most five bf16 factors each, every one
    of them rounded once more (2^-9): 2^-9 times 6, and a factor 2 for terms that cancel."""
    import torch.autograd.forward_ad as fwAD
    tol = 12 * 2 ** -9
    gen = torch.Generator(device=DEV).manual_seed(11)
    x, tx, w, b = _operands(M, N, K)
    gy, tgy = ((torch.randn(M, N, generator=gen, device=DEV) * M ** -0.5).bfloat16() for _ in range(2))
    vx, vw = torch.randn(M, K, generator=gen, device=DEV).bfloat16(), (torch.randn(N, K, generator=gen, device=DEV) * K ** -0.5).bfloat16()
    assert _lib.load().dmf_linear_gelu_plan(M, N, K) == 1

    def run(fn, dt, pdt, constant_copy):
        leaves = [x.to(dt).requires_grad_(), w.to(pdt).requires_grad_(), b.to(pdt).requires_grad_()]
        g = gy.to(dt).requires_grad_(case == "second")
        with torch.autocast("cuda", dtype=torch.bfloat16, enabled=autocast and dt != torch.float64), fwAD.dual_level():
            y = fn(fwAD.make_dual(leaves[0], tx.to(dt)), *leaves[1:])
            if case == "over_reverse":
                # (the tangent of x as well as of the gradient)
                grads = torch.autograd.grad(y, leaves, fwAD.make_dual(g, tgy.to(dt)))
                return [fwAD.unpack_dual(t).tangent for t in grads]
            y = fwAD.unpack_dual(y)[0]
        gx, gw = torch.autograd.grad(y, leaves[:2], g, create_graph=True)
        # (a second gradient for x and for what came in; the parameters' too where they are not copied)
        first = (gx * vx.to(gx.dtype)).float().sum() if dt != torch.float64 else (gx * vx.double()).sum()
        second = (gw * vw.to(gw.dtype)).float().sum() if dt != torch.float64 else (gw * vw.double()).sum()
        wanted = [leaves[0], g] + ([] if constant_copy else leaves[1:])
        return [*torch.autograd.grad(first, wanted, retain_graph=True), *torch.autograd.grad(second, wanted)]

    got = run(block_ops.linear_gelu_tanh, torch.bfloat16, torch.float32 if autocast else torch.bfloat16, autocast)
    exp = run(lambda x, w, b: torch.nn.functional.gelu(torch.nn.functional.linear(x, w, b), approximate="tanh"), torch.float64, torch.float64, autocast)
    assert len(got) == len(exp)
    for i, (a, e) in enumerate(zip(got, exp)):
        assert a is not None and a.shape == e.shape, i
        assert (a.double() - e).norm() <= tol * e.norm(), (i, float((a.double() - e).norm() / e.norm()))


def test_the_training_plan_refuses_what_the_entries_refuse():
    plan, name = _lib.load().dmf_linear_train_plan, ctypes.create_string_buffer(4)
    for which, size in ((0, (64, 64, 64)), (0, (2 ** 31, 2296, 704)), (1, (64, 32, 64)), (1, (1 << 25, 64, 8)), (2, (64, 60, 64)), (2, (2 ** 31, 64, 64)), (3, (64, 64, 64))):
        assert plan(which, *size, name, len(name)) == -3
    assert plan(2, 64, 64, 64, None, 0) == -5
    assert plan(2, 64, 64, 64, name, len(name)) == 0 and name.value == b"dmf"   # (cut to the buffer)


def test_the_plan_refuses_what_the_entry_refuses():
    plan, name = _lib.load().dmf_linear_fwd_plan, ctypes.create_string_buffer(4)
    for size in ((64, 64, 32), (64, 60, 64), (0, 64, 64), (2 ** 25, 64, 64)):
        assert plan(*size, 0, 0, name, len(name)) == -3
    assert plan(64, 64, 64, 0, 0, None, 0) == -5
    assert plan(64, 64, 64, 0, 0, name, len(name)) == 0 and name.value == b"dmf"   # (cut to the buffer)
