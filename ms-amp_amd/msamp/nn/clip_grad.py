"""Gradient-norm clipping over mixed torch.Tensor / ScalingTensor gradients (msamp/nn/clip_grad.py:11-88)."""

import torch

from msamp import _backend
from msamp.common.dtype import Dtypes
from msamp.common.tensor import ScalingTensor


_KINDS = (1.0, 2.0, float('inf'))
_PLAIN = {torch.float32: _backend.DT_F32, torch.float16: _backend.DT_F16, torch.bfloat16: _backend.DT_BF16}


def _entries(grads):
    """Per gradient its descriptor for the kernels that take a whole list at once, or None if it is not a contiguous FP8
    ScalingTensor or plain tensor on the current GPU."""
    current, entries = None, []
    for g in grads:
        kind = type(g)
        if kind is ScalingTensor:
            value, si = g.value, g.meta.scale_inv
            device, word, dtype = value.get_device(), si.data_ptr(), int(g.qtype) if Dtypes.is_fp8_qtype(g.qtype) else 0
            if si.dtype != torch.float32 or si.numel() != 1 or si.get_device() != device:
                dtype = 0
        else:
            value, word, dtype = g, 0, 0
            if (kind is torch.Tensor or kind is torch.nn.Parameter) and g.layout == torch.strided and not g.requires_grad:
                device, dtype = g.get_device(), _PLAIN.get(g.dtype, 0)
        if dtype and device >= 0:
            if current is None:
                current = torch.cuda.current_device()
            numel = value.numel()
            if numel and device == current and value.is_contiguous():
                entries.append((value.data_ptr(), word, numel, dtype))
                continue
        entries.append(None)
    return entries


def _rounds(entries):
    """The entries in as few lists as it takes so that clipping those of one list writes no word twice (an FP8 gradient's
    scale_inv, a plain one's values): what a launch scales at the same time must not overlap."""
    words = {e[1] for e in entries}
    if 0 not in words and len(words) == len(entries):
        return [entries]    # (FP8 throughout: words of four bytes, aligned)
    spans = sorted([(e[1], e[1] + 4, e) if e[1] else (e[0], e[0] + e[2] * _backend.dt_size(e[3]), e) for e in entries])
    end, apart = 0, True
    for lo, hi, _ in spans:
        if lo < end:
            apart = False
            break
        end = hi
    if apart:
        return [entries]
    rounds, ends = [], []
    for lo, hi, e in spans:
        at = next((i for i, end in enumerate(ends) if end <= lo), len(ends))
        if at == len(ends):
            rounds.append([])
            ends.append(hi)
        ends[at] = hi
        rounds[at].append(e)
    return rounds


def _norm(g, norm_type):
    g32 = g.to(torch.float32).detach()
    return g32.abs().max() if norm_type == float('inf') else torch.norm(g32, norm_type)


def _join(norms, norm_type):
    if norm_type == float('inf'):
        return norms[0] if len(norms) == 1 else torch.max(torch.stack(norms))
    return torch.norm(torch.stack(norms), norm_type)


def _held_elsewhere(owners, grads):
    """True if a graph may have saved one of the gradients: something holds it beside its owner and Python, or a view of it."""
    for p, g in zip(owners, grads):
        if type(g) is ScalingTensor:
            if g.meta.scale_inv._use_count() > 1:
                return True
        elif g._use_count() > (2 if isinstance(p, torch.Tensor) else 1) or \
                torch._C._storage_Use_Count(g.untyped_storage()._cdata) > 2:    # (the gradient, and the handle it is asked through)
            return True
    return False


def clip_grad_norm_(parameters, max_norm, norm_type=2.0, error_if_nonfinite=False):
    """Clip the global gradient norm in place and return it.  ScalingTensor gradients are dequantized
    for the norm and clipped by scaling their scale_inv (no pass over the payload)."""
    if isinstance(parameters, (torch.Tensor, ScalingTensor)):
        parameters = [parameters]
    else:
        parameters = list(parameters)
    owners, grads = [], []
    for p in parameters:
        g = p.grad
        if g is not None:
            owners.append(p)
            grads.append(g)
    norm_type, max_norm = float(norm_type), float(max_norm)
    # contiguous FP8 and plain gradients on this GPU go through the kernels that take them all at once, the others one by one
    entries = _entries(grads) if norm_type in _KINDS else [None] * len(grads)
    listed = entries if None not in entries else [e for e in entries if e is not None]
    if listed:
        # norms, factor and clipping without the host waiting for any of them
        table = _backend.grad_table(listed)
        norms, total_norm, coef = _backend.grad_norms(table, len(listed), norm_type, max_norm)
    if len(listed) < len(grads):
        listed_norms = iter(norms.unbind()) if listed else None
        total_norm = _join([(_norm(g, norm_type) if e is None else next(listed_norms)).to(grads[0].device)
                            for g, e in zip(grads, entries)], norm_type)
    elif not grads:
        total_norm = torch.tensor(0.)
    if error_if_nonfinite and torch.logical_or(total_norm.isnan(), total_norm.isinf()):
        raise RuntimeError(
            f'The total norm of order {norm_type} for gradients from `parameters` is non-finite, so it cannot be '
            'clipped. To disable this error and scale the gradients by the non-finite norm anyway, set '
            '`error_if_nonfinite=False`'
        )
    if not max_norm > 0 or not grads:
        return total_norm
    if len(listed) < len(grads):
        coef = torch.clamp(max_norm / (total_norm + 1e-6), max=1.0)
        if not coef.item() < 1.0:
            return total_norm
        for g, e in zip(grads, entries):
            if e is None:
                g.detach().mul_(coef)
        if listed:
            coef = coef.to(norms.device)
    elif max_norm == float('inf') or (_held_elsewhere(owners, grads) and
                                      not torch.cuda.is_current_stream_capturing() and not coef.item() < 1.0):
        # nothing to clip; what a graph has saved must then not count as changed, so the host waits to know, but only for those
        return total_norm
    if listed:
        for part in _rounds(listed):
            _backend.grad_clip(table if part is listed else _backend.grad_table(part), len(part), coef)
        changed = [g.meta.scale_inv if type(g) is ScalingTensor else g for g, e in zip(grads, entries) if e is not None]
        torch.autograd.graph.increment_version([t for t in changed if not t.is_inference()])
    return total_norm
