"""Gradient-norm clipping over mixed torch.Tensor / ScalingTensor gradients (msamp/nn/clip_grad.py:11-88)."""

import torch

from msamp import _backend
from msamp.common.dtype import Dtypes
from msamp.common.tensor import ScalingTensor


_KINDS = (1.0, 2.0, float('inf'))
_PLAIN = (torch.float32, torch.float16, torch.bfloat16)


def _table(grads, norm_type):
    """Descriptors of the gradients for the kernels that take the whole list at once, or None if one of them is not a
    contiguous FP8 ScalingTensor or plain tensor on the current GPU, or shares memory with another."""
    if norm_type not in _KINDS or not grads:
        return None
    entries, seen, device = [], set(), None
    for g in grads:
        if type(g) is ScalingTensor:
            value, si = g.value, g.meta.scale_inv
            if not Dtypes.is_fp8_qtype(g.qtype) or si.dtype != torch.float32 or si.numel() != 1 or si.device != value.device:
                return None
            dtype, si, at = int(g.qtype), si.data_ptr(), si.data_ptr()
        else:
            value, si = g, 0
            if type(g) not in (torch.Tensor, torch.nn.Parameter) or g.layout != torch.strided or g.dtype not in _PLAIN or \
                    g.requires_grad:
                return None
            dtype, at = _backend.hp_dt(g), g.data_ptr()
        if device is None:
            device = value.device
        n = value.numel()
        if n == 0 or not value.is_cuda or value.device != device or not value.is_contiguous() or at in seen:
            return None
        seen.add(at)
        entries.append((value.data_ptr(), si, n, dtype))
    return _backend.grad_table(entries) if device.index == torch.cuda.current_device() else None


def _compute_total_norm(grads, norm_type):
    device = grads[0].device
    norms = []
    for g in grads:
        g32 = g.to(torch.float32).detach()
        norms.append((g32.abs().max() if norm_type == float('inf') else torch.norm(g32, norm_type)).to(device))
    if norm_type == float('inf'):
        return norms[0] if len(norms) == 1 else torch.max(torch.stack(norms))
    return torch.norm(torch.stack(norms), norm_type)


def clip_grad_norm_(parameters, max_norm, norm_type=2.0, error_if_nonfinite=False):
    """Clip the global gradient norm in place and return it.  ScalingTensor gradients are dequantized
    for the norm and clipped by scaling their scale_inv (no pass over the payload)."""
    if isinstance(parameters, (torch.Tensor, ScalingTensor)):
        parameters = [parameters]
    else:
        parameters = list(parameters)
    grads = [p.grad for p in parameters if p.grad is not None]
    norm_type, max_norm = float(norm_type), float(max_norm)
    table = _table(grads, norm_type)
    if table is not None:
        # norms, factor and clipping without the host waiting for any of them
        _, total_norm, factor = _backend.grad_norms(table, len(grads), norm_type, max_norm, grads[0].device)
    else:
        total_norm = _compute_total_norm(grads, norm_type) if grads else torch.tensor(0.)
    if error_if_nonfinite and torch.logical_or(total_norm.isnan(), total_norm.isinf()):
        raise RuntimeError(
            f'The total norm of order {norm_type} for gradients from `parameters` is non-finite, so it cannot be '
            'clipped. To disable this error and scale the gradients by the non-finite norm anyway, set '
            '`error_if_nonfinite=False`'
        )
    if max_norm > 0 and table is not None:
        _backend.grad_clip(table, len(grads), factor)
        # (what autograd saved of them, if anything, has changed)
        changed = [g.meta.scale_inv if type(g) is ScalingTensor else g for g in grads]
        torch.autograd.graph.increment_version([t for t in changed if not t.is_inference()])
    elif max_norm > 0:
        coef = torch.clamp(max_norm / (total_norm + 1e-6), max=1.0)
        if coef.item() < 1.0:
            for g in grads:
                g.detach().mul_(coef)
    return total_norm
