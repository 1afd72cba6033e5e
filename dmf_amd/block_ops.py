"""Fused DiT-block glue operators with forward-mode (JVP) support.

Host-side counterparts of the small tensor expressions that surround the
attention operator in the reference's block (models/layers.py):

* ``ln_modulate(x, shift, scale)``  = ``modulate(LayerNorm(x), shift, scale)``   (:28-29, :198, :200, :219)
* ``gate_residual(x, gate, h)``     = ``x + gate * h``                           (:198, :200)
* ``residual_ln_modulate(x, gate, h, shift, scale)`` = the two above back to back (:198-200)
* ``gelu_tanh(x)``                  = ``nn.GELU(approximate="tanh")(x)``         (:162, :166)
* ``rms_norm(x, gain)``             = ``RMSNorm.forward``                        (:33-42, :148)
* ``silu(x)``                       = ``nn.SiLU()`` of the adaLN branch          (:185-188, :211-214)
* ``dual_linear(x, weight, bias)``  = ``nn.Linear`` (:131,137,161-165,...) -- library GEMMs, see ``DualLinearFunc``
* ``linear_gelu_tanh(x, weight, bias)`` = ``act(fc1(x))`` of the MLP (:166) -- GELU in the GEMM epilogue when nothing is differentiated

Each follows the protocol of the attention operator (flash_attention_hip_jvp):
a wrapper unpacks forward-AD duals, one ``torch.autograd.Function`` call pushes
primal and tangent through a single fused kernel (C ABI: include/dmf_block.h),
and the result is re-packed with ``fwAD.make_dual``.  ``backward`` propagates
through the primal output only: tangent inputs get no gradient and the
cotangent of the tangent output is dropped -- exact for the MeanFlow loss, whose
JVP target is detached (loss.py:171-172), and the same convention as the
reference's attention ``backward`` (flash_attention_2_jvp.py:260-276).
There is no fallback: without the HIP library every call raises.
"""
from __future__ import annotations

import torch
import torch.autograd.forward_ad as fwAD

from . import _lib


def _unpack(*tensors):
    primals, tangents = [], []
    for t in tensors:
        p, tg = fwAD.unpack_dual(t)
        primals.append(p)
        tangents.append(tg)
    return primals, tangents, any(tg is not None for tg in tangents)


def _primal_only(*tangent_cotangents):
    """These operators differentiate through their primal output only.  A loss that keeps the JVP output attached
    (unlike the MeanFlow loss, loss.py:171-172) would need the second-order terms the reference's tensor expressions
    carry; say so instead of returning gradients that silently lack them."""
    if any(g is not None for g in tangent_cotangents):
        raise NotImplementedError(
            "dmf_amd.block_ops: a gradient arrived at the tangent (JVP) output of a fused block operator; these operators "
            "back-propagate through the primal output only -- detach the JVP output (as DMFLoss does) or build the model "
            "with block_ops='torch'")


def _again(g) -> bool:
    """True where a gradient is to be differentiated again (create_graph=True) or carries a tangent: what can be made of torch's operators is."""
    return torch.is_grad_enabled() or fwAD.unpack_dual(g).tangent is not None


def _like(g, ref):
    """Gradient of a (B, C) modulation operand reshaped to the operand's shape."""
    return g.reshape(ref)


class LNModulateFunc(torch.autograd.Function):
    """(x, shift, scale, tx, tshift, tscale, eps, out_dtype, jvp) -> (y, ty)."""

    @staticmethod
    def forward(x, shift, scale, tx, tshift, tscale, eps, out_dtype, jvp):
        return _lib.ln_modulate_fwd(x, shift, scale, tx, tshift, tscale, eps, out_dtype, jvp)

    @staticmethod
    def setup_context(ctx, inputs, outputs):
        x, shift, scale, _, _, _, eps, _, _ = inputs
        ctx.save_for_backward(x, scale)
        ctx.eps, ctx.mod_shape = eps, (shift.shape, scale.shape)
        ctx.set_materialize_grads(False)

    @staticmethod
    def backward(ctx, gy, gty):
        _primal_only(gty)
        if gy is None:
            return (None,) * 9
        x, scale = ctx.saved_tensors
        gx, gshift, gscale = _lib.ln_modulate_bwd(gy, x, scale, ctx.eps)
        return gx, _like(gshift, ctx.mod_shape[0]), _like(gscale, ctx.mod_shape[1]), None, None, None, None, None, None


class GateResidualFunc(torch.autograd.Function):
    """(x, gate, h, tx, tgate, th, jvp) -> (y, ty)."""

    @staticmethod
    def forward(x, gate, h, tx, tgate, th, jvp):
        return _lib.gate_residual_fwd(x, gate, h, tx, tgate, th, jvp)

    @staticmethod
    def setup_context(ctx, inputs, outputs):
        x, gate, h = inputs[:3]
        ctx.save_for_backward(gate, h)
        ctx.gate_shape, ctx.x_dtype = gate.shape, x.dtype
        ctx.set_materialize_grads(False)

    @staticmethod
    def backward(ctx, gy, gty):
        _primal_only(gty)
        if gy is None:
            return (None,) * 7
        gate, h = ctx.saved_tensors
        gh, ggate = _lib.gate_residual_bwd(gy, gate, h)
        return gy, _like(ggate, ctx.gate_shape), gh, None, None, None, None


class ResidualLNModulateFunc(torch.autograd.Function):
    """(x, gate, h, shift, scale, tx, tgate, th, tshift, tscale, eps, out_dtype, jvp) -> (y, z, ty, tz)."""

    @staticmethod
    def forward(x, gate, h, shift, scale, tx, tgate, th, tshift, tscale, eps, out_dtype, jvp):
        return _lib.residual_ln_modulate_fwd(x, gate, h, shift, scale, tx, tgate, th, tshift, tscale, eps, out_dtype, jvp)

    @staticmethod
    def setup_context(ctx, inputs, outputs):
        x, gate, h, shift, scale = inputs[:5]
        ctx.save_for_backward(outputs[0], h, gate, scale)
        ctx.eps, ctx.shapes = inputs[10], (gate.shape, shift.shape, scale.shape)
        ctx.set_materialize_grads(False)

    @staticmethod
    def backward(ctx, gy, gz, gty, gtz):
        _primal_only(gty, gtz)
        if gy is None and gz is None:
            return (None,) * 13
        y, h, gate, scale = ctx.saved_tensors
        if gz is None:   # only the residual output was used
            gh, ggate = _lib.gate_residual_bwd(gy, gate, h)
            return (gy, _like(ggate, ctx.shapes[0]), gh) + (None,) * 10
        gx, gh, ggate, gshift, gscale = _lib.residual_ln_modulate_bwd(gy, gz, y, h, gate, scale, ctx.eps)
        return (gx, _like(ggate, ctx.shapes[0]), gh, _like(gshift, ctx.shapes[1]), _like(gscale, ctx.shapes[2])) + (None,) * 8


class GeluTanhFunc(torch.autograd.Function):
    """(x, tx) -> (y, ty)."""

    @staticmethod
    def forward(x, tx):
        return _lib.gelu_tanh_fwd(x, tx)

    @staticmethod
    def setup_context(ctx, inputs, outputs):
        ctx.save_for_backward(inputs[0])
        ctx.set_materialize_grads(False)

    @staticmethod
    def backward(ctx, gy, gty):
        _primal_only(gty)
        if gy is None:
            return None, None
        (x,) = ctx.saved_tensors
        if _again(gy):
            return torch.ops.aten.gelu_backward(gy.to(x.dtype), x, approximate="tanh"), None
        return _lib.gelu_tanh_bwd(gy.to(x.dtype), x), None


class SiluFunc(torch.autograd.Function):
    """(x, tx, out_dtype) -> (y, ty)."""

    @staticmethod
    def forward(x, tx, out_dtype):
        return _lib.silu_fwd(x, tx, out_dtype)

    @staticmethod
    def setup_context(ctx, inputs, outputs):
        ctx.save_for_backward(inputs[0])
        ctx.set_materialize_grads(False)

    @staticmethod
    def backward(ctx, gy, gty):
        _primal_only(gty)
        if gy is None:
            return None, None, None
        (x,) = ctx.saved_tensors
        if _again(gy):
            s = torch.sigmoid(x)
            return gy.to(x.dtype) * (s * (1 + x * (1 - s))), None, None
        return _lib.silu_bwd(gy, x), None, None


class RMSNormFunc(torch.autograd.Function):
    """(x, gain, tx, eps, jvp) -> (y, ty); x is (B, L, H, D), normalised over D."""

    @staticmethod
    def forward(x, gain, tx, eps, jvp):
        return _lib.rmsnorm_fwd(x, gain, tx, eps, jvp)

    @staticmethod
    def setup_context(ctx, inputs, outputs):
        x, gain, _, eps, _ = inputs
        ctx.save_for_backward(x, gain)
        ctx.eps = eps
        ctx.set_materialize_grads(False)

    @staticmethod
    def backward(ctx, gy, gty):
        _primal_only(gty)
        if gy is None:
            return (None,) * 5
        x, gain = ctx.saved_tensors
        gx, ggain = _lib.rmsnorm_bwd(gy.to(x.dtype), x, gain, ctx.eps)
        return gx, ggain, None, None, None


def _products(x, tx, w, b):
    """``x w^T + b`` and ``tx w^T`` (None without a tangent): one launch of the package's own product kernel where that is the
    faster one, library products elsewhere."""
    x2 = x.reshape(-1, x.shape[-1])
    own = None if torch.compiler.is_compiling() else _lib.linear_fwd(x2, None if tx is None else tx.reshape(-1, tx.shape[-1]), w, b)
    if own is not None:
        shape = (*x.shape[:-1], w.shape[0])
        return own[0].reshape(shape), (None if tx is None else own[1].reshape(shape))
    linear = torch.nn.functional.linear
    return linear(x, w, b), (None if tx is None else linear(tx, w))


class DualLinearFunc(torch.autograd.Function):
    """(x, tx, weight, bias, w_lp, b_lp) -> (y, ty, w) with y = x W^T + b, ty = tx W^T: exactly
    one product per stream.  torch's own forward-mode rule for ``linear``
    also multiplies the primal input by a materialised all-zero weight tangent
    and adds the two products (three GEMMs, two fills, a copy and an add per
    layer); parameters carry no tangent in the MeanFlow JVP (loss.py:165-170), so
    that work is skipped here.  Under autocast the operands are cast once (``w``,
    the cast weight, is returned so that ``backward`` can reuse it)."""

    @staticmethod
    def forward(x, tx, weight, bias, w_lp, b_lp):
        if x.is_cuda and torch.is_autocast_enabled("cuda"):
            dt = torch.get_autocast_dtype("cuda")
            cached = w_lp is not None and w_lp.dtype == dt
            w = w_lp if cached else weight.to(dt)
            b = None if bias is None else (b_lp if cached and b_lp is not None else bias.to(dt))
            with torch.autocast("cuda", enabled=False):
                y, ty = _products(x.to(dt), None if tx is None else tx.to(dt), w, b)
            # (an input is never handed back as an output: a cached copy reaches backward through the inputs)
            return y, ty, (w if not cached and w is not weight else None)
        return *_products(x, tx, weight, bias), None

    @staticmethod
    def setup_context(ctx, inputs, outputs):
        x, _, weight, bias, w_lp, _ = inputs
        w = outputs[2]
        if w is not None:
            ctx.mark_non_differentiable(w)
        elif w_lp is not None and x.is_cuda and torch.is_autocast_enabled("cuda") and w_lp.dtype == torch.get_autocast_dtype("cuda"):
            w = w_lp
        else:
            w = weight
        ctx.save_for_backward(x, w)
        ctx.weight_dtype = weight.dtype
        ctx.bias_dtype = None if bias is None else bias.dtype
        ctx.set_materialize_grads(False)

    @staticmethod
    def backward(ctx, gy, gty, gw_unused):
        _primal_only(gty)
        if gy is None:
            return (None,) * 6
        x, w = map(_lib.ordinary, ctx.saved_tensors)
        g2 = _lib.ordinary(gy).reshape(-1, gy.shape[-1]).to(w.dtype)
        want_gx, want_gw = ctx.needs_input_grad[0], ctx.needs_input_grad[2]
        want_gb = ctx.bias_dtype is not None and ctx.needs_input_grad[3]
        gx = gw = gb = None
        again = _again(gy)
        # (in one stream: next to each other in two, the products slow one another down and each fork and join idles the GPU)
        if want_gw:
            x2 = x.reshape(-1, x.shape[-1]).to(w.dtype)
            if g2.is_cuda and g2.dtype != ctx.weight_dtype and ctx.weight_dtype == torch.float32:
                own = None if again else _lib.linear_wgrad(g2, x2, want_gb and ctx.bias_dtype == torch.float32)
                if own is not None:
                    gw, gb = own
                elif again:
                    gw = g2.t().float() @ x2.float()
                else:
                    gw = torch.mm(g2.t(), x2, out_dtype=torch.float32)   # the GEMM stores its fp32 accumulators: no cast kernel
            else:
                gw = (g2.t() @ x2).to(ctx.weight_dtype)
        if want_gb and gb is None:
            # torch's multi-block column reduction clears its scratch with a memset node, which does not survive
            # HIP-graph replay; the library's two-stage sum has no such node
            capturing = g2.is_cuda and torch.cuda.is_current_stream_capturing()
            if g2.is_cuda and g2.shape[1] % 8 == 0 and (capturing or not again):
                gb = _lib.colsum(g2.contiguous(), ctx.bias_dtype)
            else:
                if capturing:
                    raise RuntimeError("dual_linear: the bias gradient of a layer whose output width is not a multiple of 8 falls back "
                                       "to torch's column sum, which does not replay correctly from a captured graph")
                gb = g2.sum(0).to(ctx.bias_dtype)
        if want_gx:
            gx = None if again else _lib.linear_dgrad(g2, w)
            gx = (g2 @ w if gx is None else gx).reshape(x.shape).to(x.dtype)
        return gx, None, gw, gb, None, None


def dual_linear(x, weight, bias=None, w_lp=None, b_lp=None):
    """``F.linear(x, weight, bias)``; a forward-AD dual ``x`` gives a dual result
    (weight and bias are constants of the tangent map).  ``w_lp`` / ``b_lp``: optional
    copies of the parameters in the autocast dtype, used instead of casting per call
    (the caller guarantees they are current)."""
    if _lib.native(x, weight, bias):
        out = _lib.host().linear(x, weight, bias, w_lp, b_lp)
        if out is not None:
            return out
    (xp,), (tx,), dual = _unpack(x)
    y, ty, _ = _lib.run_function(DualLinearFunc, xp, tx, weight, bias, w_lp, b_lp)
    return fwAD.make_dual(y, ty) if dual else y


def linear_gelu_tanh(x, weight, bias, w_lp=None, b_lp=None):
    """``gelu_tanh(F.linear(x, weight, bias))`` -- the first half of the MLP
    (reference models/layers.py:161-166).  With nothing to differentiate in reverse the
    activation -- and its derivative on the tangent -- rides in the product's epilogue
    (the pre-activation never reaches HBM); otherwise the pre-activation is needed for
    the backward pass and this is ``dual_linear`` followed by ``gelu_tanh``."""
    if _lib.native(x, weight, bias):
        out = _lib.host().linear_gelu_tanh(x, weight, bias, w_lp, b_lp)
        if out is not None:
            return out
    if torch.is_grad_enabled() or bias is None or not x.is_cuda or fwAD.unpack_dual(x).tangent is not None:
        return gelu_tanh(dual_linear(x, weight, bias, w_lp, b_lp))
    dt = _autocast_dtype(x)
    cached = w_lp is not None and w_lp.dtype == dt
    w = w_lp if cached else weight.to(dt)
    b = b_lp if cached and b_lp is not None else bias.to(dt)
    x2 = _lib._raw(x).reshape(-1, x.shape[-1]).to(dt)
    own = _lib.linear_fwd(x2, None, w, b, gelu=True)
    if own is not None:
        return own[0].reshape(*x.shape[:-1], w.shape[0])
    return torch._addmm_activation(b, x2, _lib._raw(w).t(), use_gelu=True).reshape(*x.shape[:-1], w.shape[0])


def _autocast_dtype(x: torch.Tensor):
    if x.is_cuda and torch.is_autocast_enabled("cuda"):
        return torch.get_autocast_dtype("cuda")
    return x.dtype


def ln_modulate(x, shift, scale, eps: float = 1e-6):
    """``LayerNorm(x) * (1 + scale) + shift`` for x (B, L, C) and shift / scale
    (B, C) or (B, 1, C); LayerNorm over C without affine parameters.  Under
    autocast the result is produced directly in the autocast dtype (it only ever
    feeds a Linear, which would cast it)."""
    if _lib.native(x, shift, scale):
        out = _lib.host().ln_modulate(x, shift, scale, eps)
        if out is not None:
            return out
    (xp, shp, scp), (tx, tsh, tsc), dual = _unpack(x, shift, scale)
    y, ty = _lib.run_function(LNModulateFunc, xp, shp, scp, tx, tsh, tsc, eps, _autocast_dtype(xp), dual)
    return fwAD.make_dual(y, ty) if dual else y


def gate_residual(x, gate, h):
    """``x + gate * h`` for x, h (B, L, C) and gate (B, C) or (B, 1, C); the result
    has the promoted dtype of x and h (the fp32 residual stream under autocast)."""
    if _lib.native(x, gate, h):
        out = _lib.host().gate_residual(x, gate, h)
        if out is not None:
            return out
    (xp, gp, hp), (tx, tg, th), dual = _unpack(x, gate, h)
    dt = torch.promote_types(xp.dtype, hp.dtype)
    if xp.dtype != dt:
        xp, tx = xp.to(dt), (None if tx is None else tx.to(dt))
    y, ty = _lib.run_function(GateResidualFunc, xp, gp, hp, tx, tg, th, dual)
    return fwAD.make_dual(y, ty) if dual else y


def residual_ln_modulate(x, gate, h, shift, scale, eps: float = 1e-6):
    """``y = x + gate * h`` and ``z = LayerNorm(y) * (1 + scale) + shift`` in one pass;
    returns ``(y, z)`` with the dtypes ``gate_residual`` and ``ln_modulate`` would give."""
    if _lib.native(x, gate, h, shift, scale):
        out = _lib.host().residual_ln_modulate(x, gate, h, shift, scale, eps)
        if out is not None:
            return out
    (xp, gp, hp, shp, scp), (tx, tg, th, tsh, tsc), dual = _unpack(x, gate, h, shift, scale)
    dt = torch.promote_types(xp.dtype, hp.dtype)
    if xp.dtype != dt:
        xp, tx = xp.to(dt), (None if tx is None else tx.to(dt))
    y, z, ty, tz = _lib.run_function(ResidualLNModulateFunc, xp, gp, hp, shp, scp, tx, tg, th, tsh, tsc, eps, _autocast_dtype(xp), dual)
    return (fwAD.make_dual(y, ty), fwAD.make_dual(z, tz)) if dual else (y, z)


def gelu_tanh(x):
    """tanh-approximated GELU."""
    if _lib.native(x):
        out = _lib.host().gelu_tanh(x)
        if out is not None:
            return out
    (xp,), (tx,), dual = _unpack(x)
    y, ty = _lib.run_function(GeluTanhFunc, xp, tx)
    return fwAD.make_dual(y, ty) if dual else y


def silu(x):
    """``x * sigmoid(x)``; under autocast the result is produced in the autocast
    dtype (it feeds the adaLN projection, which would cast it)."""
    if _lib.native(x):
        out = _lib.host().silu(x)
        if out is not None:
            return out
    (xp,), (tx,), dual = _unpack(x)
    y, ty = _lib.run_function(SiluFunc, xp, tx, _autocast_dtype(xp))
    return fwAD.make_dual(y, ty) if dual else y


def rms_norm(x, gain, eps: float = 1e-6):
    """Per-head RMS norm of a (B, L, H, D) tensor over D (strided views into a
    packed qkv buffer are read in place); returns a contiguous tensor.  The gain
    is treated as a constant by forward-mode AD (parameters carry no tangent)."""
    (xp,), (tx,), dual = _unpack(x)
    y, ty = _lib.run_function(RMSNormFunc, xp, gain, tx, eps, dual)
    return fwAD.make_dual(y, ty) if dual else y


def chunk_last(x, n: int):
    """``x.chunk(n, dim=-1)`` for a modulation tensor whose width ``n`` divides."""
    if _lib.native(x):
        out = _lib.host().chunk_last(x, n)
        if out is not None:
            return out
    return x.chunk(n, dim=-1)
