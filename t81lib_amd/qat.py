"""Quantization-aware training helpers: the ``t81.qat`` surface ``t8.nn.Linear`` trains with.

``ternary(x, threshold, stochastic)`` (t81/qat.py:49-57) returns balanced-ternary
values in the forward pass and back-propagates through the ``dorso_round``
surrogate (t81/qat.py:28-35): the gradient reaching ``x`` is 2 where |x| < 0.5 and
0 elsewhere (|x| = 0.5 included), not the identity of a plain straight-through
estimator.  Forward values (t81/qat.py:12-25): x is clamped to [-1, 1]; entries
with |x| >= threshold take sign(x), the rest 0; with ``stochastic=True`` each such
entry is kept with probability (|x| - threshold) / (1 - threshold) (clamped to
[0, 1], the denominator floored at 1e-6), drawing one ``torch.rand_like`` sample
per entry from torch's global generator -- the same draw as the reference, so a
seeded run repeats.  Plain torch code, on whatever device the tensors are on.

``TernaryWeight`` and ``TernaryProduct`` are the same expression, ``F.linear(x,
ternary(w / s) * s, b)``, for ``t8.nn.Linear``'s training step on the GPU (csrc/qat.hip): the
weight and its gradient take one pass each instead of about twenty-five, and a float32
product runs over the packed trits with the activations split into three bf16 planes
(exactly, but for digits below 2^-140).  Results keep the tensor expression's roundings (weights and
weight-gradient passes bit for bit); ``weight_on_kernels`` and ``product_on_kernels`` say when
they stand in, everything else (other devices, subclasses, tracing, modes, forward-mode) runs
the expression itself.
"""

from __future__ import annotations

from typing import Optional

import torch
from torch.nn import functional as F
from torch.utils._device import DeviceContext

from . import _lib, ops


def _clamp_threshold(threshold: float) -> float:
    """t81/qat.py:8-9: thresholds are clipped to [0, 1]."""
    return float(max(0.0, min(threshold, 1.0)))


def quantize(x: torch.Tensor, threshold: float, stochastic: bool = False) -> torch.Tensor:
    """The forward value of ``ternary`` (no gradient), t81/qat.py:12-25."""
    c = x.detach().clamp(-1.0, 1.0)
    mag = c.abs()
    keep = mag >= threshold
    if stochastic:
        prob = ((mag - threshold) / max(1.0 - threshold, 1e-6)).clamp(0.0, 1.0)
        keep = keep & (torch.rand_like(prob) < prob)
    return torch.where(keep, torch.sign(c), torch.zeros_like(c))


def dorso_round(x: torch.Tensor) -> torch.Tensor:
    """t81/qat.py:28-35: 1 for x >= 0.5, -1 for x <= -0.5, 2x between (so the gradient is
    2 inside (-0.5, 0.5) and 0 outside)."""
    one = torch.ones_like(x)
    return torch.where(x >= 0.5, one, torch.where(x <= -0.5, -one, 2.0 * x))


class _SurrogateGradient(torch.autograd.Function):
    """Value of ``quantized``, gradient of ``surrogate`` (t81/qat.py:38-46)."""

    @staticmethod
    def forward(ctx, surrogate: torch.Tensor, quantized: torch.Tensor) -> torch.Tensor:
        return quantized.clone()

    @staticmethod
    def backward(ctx, grad_output: torch.Tensor):
        return grad_output, None


def ternary(x: torch.Tensor, threshold: float = 0.45, stochastic: bool = False) -> torch.Tensor:
    """Balanced-ternary quantization of ``x`` for training (t81/qat.py:49-57)."""
    threshold = _clamp_threshold(threshold)
    return _SurrogateGradient.apply(dorso_round(x), quantize(x, threshold, stochastic))


# ------------------------------------------------------------- the kernels' training step --

def observed() -> bool:
    """Whether something sees or rewrites tensor operations, which kernels would hide from it:
    tracing, dispatch and torch-function modes, function transforms, forward-mode.  (A device
    context is a torch-function mode that only fills in the device of new tensors.)"""
    if torch.compiler.is_compiling() or torch.jit.is_tracing():
        return True
    if torch._C._len_torch_function_stack() > 0 and any(
            type(m) is not DeviceContext
            for m in torch.overrides._get_current_function_mode_stack()):
        return True
    return (torch._C._len_torch_dispatch_stack() > 0 or
            torch._C._functorch.peek_interpreter_stack() is not None or
            torch.autograd.forward_ad._current_level >= 0)


def _ordinary(*tensors: Optional[torch.Tensor]) -> bool:
    """Contiguous tensors on the current GPU, of no subclass.  (A batch of gradients taken through
    one graph at once has no storage of its own.)"""
    for t in tensors:
        if t is None:
            continue
        if type(t) not in (torch.Tensor, torch.nn.Parameter) or t.device.type != "cuda" or \
                t.layout != torch.strided or not torch._C._has_storage(t) or \
                not t.is_contiguous():
            return False
        if t.device.index != torch.cuda.current_device():
            return False
    return True


def _plain(*tensors: Optional[torch.Tensor]) -> bool:
    """Ordinary tensors, and nothing that observes."""
    return not observed() and _ordinary(*tensors)


def _as_saved(t: torch.Tensor, dtype: torch.dtype, *shape: int) -> bool:
    """Whether a saved tensor came back as it was (saved-tensor hooks may return another)."""
    return t.dtype == dtype and t.shape == shape and _ordinary(t)


def weight_on_kernels(weight: torch.Tensor, threshold: float) -> bool:
    return (_plain(weight) and weight.ndim == 2 and weight.numel() > 0 and
            weight.dtype in ops._FLOAT_CODES and threshold == threshold)


# tokens x inputs x outputs from which the three-plane products are taken: a step of 512 x 4096
# -> 4096 went 451 -> 343 us, 1623 x 1015 -> 3520 454 -> 344; 256 x 4096 -> 4096 stayed at
# 286, and below that both are bound by the host, whose calls cost 30 us more (128 x 4096 ->
# 4096 251 -> 282).
MIN_PRODUCT = 1 << 32


def product_on_kernels(x: torch.Tensor, weight: torch.Tensor,
                       bias: Optional[torch.Tensor]) -> bool:
    """Large float32 products (MIN_PRODUCT); autocast changes F.linear's own type."""
    return (_plain(x, bias) and x.ndim >= 2 and x.dtype == torch.float32 and
            weight.dtype == torch.float32 and x.shape[-1] == weight.shape[1] and
            x.numel() > 0 and x.numel() * weight.shape[0] >= MIN_PRODUCT and
            (bias is None or (bias.dtype == torch.float32 and bias.shape == weight.shape[:1])) and
            not torch.is_autocast_enabled("cuda") and
            _workspace(x.numel() // weight.shape[1], *weight.shape) > 0 and
            _workspace(x.numel() // weight.shape[1], weight.shape[1], weight.shape[0]) > 0)


def scale_on_kernels(existing: Optional[torch.Tensor]) -> bool:
    """(asked where weight_on_kernels holds)"""
    return existing is None or (_ordinary(existing) and existing.ndim == 0 and
                                existing.dtype == torch.float32 and not existing.requires_grad)


def training_scale(weight: torch.Tensor, previous: Optional[torch.Tensor]) -> torch.Tensor:
    """max |w| (at least 1e-6), or the 0.99 / 0.01 mean of it and the previous scale
    (t81/nn/linear.py:72-85)."""
    w = weight.detach()
    scale = torch.empty((), dtype=torch.float32, device=w.device)
    scratch = torch.empty(1024, dtype=torch.int32, device=w.device)
    _lib.check(_lib.lib().t81_hip_qat_scale(
        w.data_ptr(), ops._FLOAT_CODES[w.dtype], w.numel(),
        previous.data_ptr() if previous is not None else None, scale.data_ptr(),
        scratch.data_ptr(), ops._stream()))
    return scale


def _workspace(m: int, n: int, k: int) -> int:
    return int(_lib.lib().t81_hip_qat_matmul_workspace_size(m, n, k))


def _scratch(nbytes: int, device: torch.device) -> Optional[torch.Tensor]:
    """None where the device has no room for it: the library's product then runs, which needs
    none (the planes take up to 512 MiB, the weight gradient's 1 GiB)."""
    try:
        return torch.empty(nbytes, dtype=torch.uint8, device=device)
    except torch.OutOfMemoryError:
        return None


def _matmul(x: torch.Tensor, packed: torch.Tensor, n: int, scale: torch.Tensor,
            bias: Optional[torch.Tensor]) -> Optional[torch.Tensor]:
    m, k = x.shape
    need = _workspace(m, n, k)
    ws = _scratch(need, x.device)
    if ws is None:
        return None
    out = torch.empty((m, n), dtype=torch.float32, device=x.device)
    _lib.check(_lib.lib().t81_hip_qat_matmul(
        x.data_ptr(), packed.data_ptr(), out.data_ptr(), m, n, k, scale.data_ptr(),
        bias.data_ptr() if bias is not None else None, ws.data_ptr(), need, ops._stream()))
    return out


# outputs from which the six-plane product stands in for the float32 one: its 256 x 256 tiles
# split the tokens below, and the library's smaller tiles are faster there (4096 tokens,
# 1024 x 1024: 63 us against 81; 2048 x 2048 232 -> 188, 1623 tokens, 3520 x 1015 154 -> 106,
# 2048 tokens, 4096 x 4096 479 -> 302).
MIN_WEIGHTS = 3 << 20


def weight_product(grad: torch.Tensor, x: torch.Tensor) -> torch.Tensor:
    """grad^T @ x for contiguous float32 grad (m, n) and x (m, k)."""
    (m, n), k = grad.shape, x.shape[1]
    lib = _lib.lib()
    need = lib.t81_hip_qat_weight_product_workspace_size(m, n, k) if n * k >= MIN_WEIGHTS else 0
    ws = _scratch(need, x.device) if need > 0 else None
    if ws is None:  # (or operands whose planes pass the workspace's bound)
        return grad.t() @ x
    out = torch.empty((n, k), dtype=torch.float32, device=x.device)
    _lib.check(lib.t81_hip_qat_weight_product(grad.data_ptr(), x.data_ptr(), out.data_ptr(), m, n,
                                              k, ws.data_ptr(), need, ops._stream()))
    return out


class TernaryWeight(torch.autograd.Function):
    """(weight, scale, threshold) -> ternary(weight / scale) * scale and its packed trits."""

    @staticmethod
    def forward(ctx, weight: torch.Tensor, scale: torch.Tensor, threshold: float):
        rows, cols = weight.shape
        limbs = ops.limbs_for(cols)
        wq = torch.empty_like(weight)
        packed = torch.empty((rows, limbs, 16), dtype=torch.uint8, device=weight.device)
        inner = torch.empty((rows, limbs, 4), dtype=torch.uint16, device=weight.device)
        code = ops._FLOAT_CODES[weight.dtype]
        _lib.check(_lib.lib().t81_hip_qat_quantize(
            weight.data_ptr(), code, scale.data_ptr(), _clamp_threshold(threshold), wq.data_ptr(),
            packed.data_ptr(), inner.data_ptr(), rows, cols, ops._stream()))
        ctx.save_for_backward(scale, inner)
        ctx.mark_non_differentiable(packed)
        ctx.set_materialize_grads(False)  # no zeros for packed
        return wq, packed

    @staticmethod
    def backward(ctx, grad: torch.Tensor, _packed):
        if grad is None:
            return None, None, None
        scale, inner = ctx.saved_tensors
        rows, cols = grad.shape
        if torch.is_grad_enabled() or not _plain(grad) or \
                not _as_saved(scale, torch.float32) or \
                not _as_saved(inner, torch.uint16, rows, ops.limbs_for(cols), 4):
            # a graph of the gradient is wanted, or tensors that the kernel does not take
            shifts = torch.arange(12, device=grad.device, dtype=torch.int32)
            mask = (inner.to(torch.int32).unsqueeze(-1) >> shifts) & 1
            mask = mask.reshape(rows, -1)[:, :cols] != 0
            kept = torch.where(mask, grad * scale, torch.zeros_like(grad))
            return kept * 2.0 / scale, None, None
        out = torch.empty_like(grad)
        _lib.check(_lib.lib().t81_hip_qat_weight_grad(
            grad.data_ptr(), ops._FLOAT_CODES[grad.dtype], scale.data_ptr(), inner.data_ptr(),
            out.data_ptr(), rows, cols, ops._stream()))
        return out, None, None


class TernaryProduct(torch.autograd.Function):
    """F.linear(x, wq, bias) for 2-D float32 x, with wq = scale * (the packed trits)."""

    @staticmethod
    def forward(ctx, x: torch.Tensor, wq: torch.Tensor, bias: Optional[torch.Tensor],
                packed: torch.Tensor, scale: torch.Tensor) -> torch.Tensor:
        ctx.save_for_backward(x, wq, packed, scale)
        out = _matmul(x, packed, wq.shape[0], scale, bias)
        return F.linear(x, wq, bias) if out is None else out

    @staticmethod
    def backward(ctx, grad: torch.Tensor):
        x, wq, packed, scale = ctx.saved_tensors
        need_x, need_w, need_b = ctx.needs_input_grad[:3]
        n, k = wq.shape
        dx = dw = db = None
        grad_c = grad.contiguous()
        if torch.is_grad_enabled() or not _plain(grad_c) or \
                not _as_saved(x, torch.float32, grad.shape[0], k) or \
                not _as_saved(scale, torch.float32) or \
                not _as_saved(packed, torch.uint8, n, ops.limbs_for(k), ops.BYTES_PER_LIMB):
            # a graph of the gradient is wanted, or tensors that the kernels do not take
            if need_x:
                dx = grad @ wq
            if need_w:
                dw = grad.t() @ x
            if need_b:
                db = grad.sum(0)
            return dx, dw, db, None, None
        if need_x:
            dx = _matmul(grad_c, ops.transpose_packed(packed, n, k), k, scale, None)
            if dx is None:
                dx = grad_c @ wq
        if need_w:
            dw = weight_product(grad_c, x)
        if need_b:
            db = ops.column_sum(grad_c)
        return dx, dw, db, None, None


__all__ = ["ternary", "dorso_round", "quantize"]
