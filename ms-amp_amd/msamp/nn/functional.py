"""F.linear with ScalingTensor weights: FP8 forward, dgrad and wgrad (msamp/nn/functional.py:16-194)."""

import torch
import torch.nn.functional as F

from msamp import _backend
from msamp.common.dtype import Dtypes
from msamp.common.tensor import ScalingMeta, ScalingTensor, TypeCast
from msamp.operators.gemm import Gemm
from msamp.nn.state import model_state


# What the library's calls for a whole direction take; everything else goes through the same entry points one by one, with
# their own checks.  (A problem whose tile walks are yet to be timed is one of those.)
_FLOATS = (torch.float32, torch.float16, torch.bfloat16)


def _walk_settled(d_in, d_out, *problem):
    # Only the calls for a direction read codes in padded rows, and they time no walks: a gradient product of a ragged width
    # that waited to be timed waited for ever, and its layer went over transposed copies (forward and backward, bfloat16, us:
    # 8192 x 4096 -> 50257 5911, 4596 so; 8192 x 4100 -> 4096 with a bias 629, 536).  Any walk gives the same bits.
    return d_in % 16 != 0 or d_out % 16 != 0 or _backend.gemm_walk_settled(*problem)


def _forward_in_one_call(x, meta, weight, output_dtype, bias):
    w, w_meta = weight.value, weight.meta
    if not (meta.scaling_mode() == 'gated' and meta.qtype == Dtypes.kfloat8_e4m3 and x.dim() == 2 and x.numel() > 0 and x.is_cuda and
            x.dtype in _FLOATS and output_dtype in _FLOATS and meta.scale.is_cuda):
        return False
    (tokens, d_in), device = x.shape, x.device
    return w.dim() == 2 and w.numel() > 0 and w.shape[1] == d_in and w.dtype in _FLOATS and w.device == device and \
        w.is_contiguous() and w_meta.amax.device == device and 1 <= w_meta.window_size <= w_meta.amax.numel() and \
        (bias is None or (bias.device == device and bias.dtype in _FLOATS and bias.numel() == w.shape[0])) and \
        (d_in % 16 == 0 and w.shape[0] % 16 == 0 or _backend.linear_fits(tokens, d_in, w.shape[0])) and \
        _backend.gemm_walk_settled(w.shape[0], tokens, _backend.linear_pitch(d_in), False, False)


def _backward_in_one_call(ctx, dy, d_in, need_dgrad):
    meta = ctx.metas['ograd']
    (tokens, d_out), device = dy.shape, dy.device
    # (under create_graph the casts themselves may have to be recorded)
    return not torch.is_grad_enabled() and meta.scaling_mode() == 'gated' and meta.qtype == Dtypes.kfloat8_e5m2 and \
        meta.scale.is_cuda and dy.numel() > 0 and dy.dtype in _FLOATS and ctx.output_dtype in _FLOATS and \
        ctx.input_codes.device == device and (not need_dgrad or _walk_settled(d_in, d_out, d_in, tokens, d_out, True, False))


def _wgrad_in_one_call(ctx, tokens, d_in, d_out):
    meta, old = ctx.metas['wgrad'], ctx.weight.grad
    if model_state.use_fp8_ddp or _backend._shared_device() or meta.scaling_mode() != 'in_time' or \
            meta.qtype != Dtypes.kfloat8_e4m3 or not _backend.gemm_cast_declines(d_in, d_out, tokens):
        return False
    if old is None:
        return _walk_settled(d_in, d_out, d_in, d_out, tokens, True, True)
    # (a product that is added to something is not timed)
    return type(old) is ScalingTensor and old.meta.qtype == Dtypes.kfloat8_e4m3 and old.value.shape == (d_out, d_in) and \
        old.value.device == ctx.input_codes.device and old.value.is_contiguous()


class _FP8GemmFunction(torch.autograd.Function):
    """y = x W^T (+ bias) with x, W in E4M3; dx = dy W and dW = dy^T x with dy in E5M2; fp32 accumulation.

    The reference adds the bias in a separate elementwise pass after the function (nn/functional.py:184-185); here it
    rides in the epilogue of the forward GEMM (fma(acc, scale, bias), one rounding to the output type instead of
    two) and its gradient, the column sums of dy in the output type, is returned from backward as autograd would
    have formed it."""
    @staticmethod
    def forward(ctx, input, weight, metas, dtype_holder, bias=None, differentiable=True):
        ctx.metas = metas
        model_state.check_metas_in_flat(metas)
        output_dtype = dtype_holder.dtype
        ctx.need_input_grad = input.requires_grad
        ctx.weight, ctx.d_in = weight, input.shape[1]
        ctx.output_dtype = output_dtype
        ctx.bias_dtype = None if bias is None else bias.dtype
        ctx.need_bias_grad = bias is not None and bias.requires_grad
        if bias is not None and not (bias.dtype == output_dtype and bias.is_contiguous()):
            bias = bias.detach().to(output_dtype).contiguous()
        src = input.contiguous()
        meta = metas['input']
        if _forward_in_one_call(src, meta, weight, output_dtype, bias):
            out, ctx.input_codes, ctx.weight_codes, ctx.weight_words = _backend.linear_forward(
                src, meta, weight.value, weight.meta, output_dtype, bias, differentiable
            )
            return out
        input_fp8 = src.cast(Dtypes.kfloat8_e4m3, meta=meta)
        weight_fp8 = weight.cast(Dtypes.kfloat8_e4m3)
        ctx.input_codes, ctx.weight_codes = input_fp8.value, weight_fp8.value
        ctx.weight_words = weight_fp8.meta
        return Gemm.fp8_gemm(weight_fp8, input_fp8, Dtypes.dtype_to_qtype[output_dtype], bias=bias, use_split_accumulator=False)

    @staticmethod
    def backward(ctx, output_grad):
        output_grad = output_grad.contiguous()
        metas = ctx.metas
        tokens, d_out = output_grad.shape
        d_in = ctx.d_in
        input_codes, weight_codes = ctx.input_codes, ctx.weight_codes
        need_dgrad, need_wgrad = ctx.need_input_grad, ctx.weight.requires_grad
        # The reference materializes dy^T, W^T and x^T (fused cast-transpose + two FP8 transposes) because its
        # GEMM reads K-contiguous operands only.  This kernel also reads [K, rows] operands in place, so when
        # the shapes allow, dy is only cast and W, x, dy go to the GEMMs as they are (same results, up to the order of
        # the float32 sum where the weight gradient is taken in parts of K).
        # Codes of widths that are no multiples of 16 come from the forward call in padded rows, which linear_backward reads.
        pitched = input_codes.shape[1] != d_in or weight_codes.shape[0] != d_out
        if pitched and not ((not need_wgrad or _wgrad_in_one_call(ctx, tokens, d_in, d_out)) and
                            _backward_in_one_call(ctx, output_grad, d_in, need_dgrad)):
            pitched = False
            input_codes, weight_codes = input_codes[:, :d_in].contiguous(), weight_codes[:d_out, :d_in].contiguous()
        in_place = pitched or (not need_dgrad or Gemm.kmajor_supported(d_in, tokens, d_out, True, False)) and \
            (not need_wgrad or Gemm.kmajor_supported(d_in, d_out, tokens, True, True))
        if not in_place and (not need_wgrad or _wgrad_in_one_call(ctx, tokens, d_in, d_out)):
            in_place = _backend.linear_takes_short_k(tokens, d_in, d_out) and _backward_in_one_call(ctx, output_grad, d_in, need_dgrad)
        output_qtype = Dtypes.dtype_to_qtype[ctx.output_dtype]
        words = ctx.weight_words
        input_grad = bias_grad = None
        column_sums = in_place and ctx.need_bias_grad and TypeCast.takes_column_sums(output_grad, metas['ograd'], ctx.bias_dtype)
        if in_place and _backward_in_one_call(ctx, output_grad, d_in, need_dgrad):
            # (a weight gradient that is cast inside its product keeps a call of its own)
            with_wgrad = need_wgrad and _wgrad_in_one_call(ctx, tokens, d_in, d_out)
            payload, input_grad, wgrad, bias_grad = _backend.linear_backward(
                output_grad, d_in, metas['ograd'], input_codes, metas['input'].scale_inv, weight_codes,
                words.scale_inv.data_ptr() if isinstance(words, ScalingMeta) else words.data_ptr() + 4, ctx.output_dtype, need_dgrad,
                metas['wgrad'] if with_wgrad else None, ctx.weight.grad, ctx.bias_dtype if column_sums else None
            )
            if with_wgrad:
                ctx.weight.backward_grad_update(ScalingTensor(wgrad, metas['wgrad']))
                need_wgrad = False
            need_dgrad = False
            ograd_fp8, ograd_fp8_t = ScalingTensor(payload, metas['ograd']), None
        elif column_sums:
            payload, bias_grad = TypeCast.cast_to_fp8_with_column_sums(output_grad, metas['ograd'], ctx.bias_dtype)
            ograd_fp8, ograd_fp8_t = ScalingTensor(payload, metas['ograd']), None
        elif in_place:
            ograd_fp8 = output_grad.cast(Dtypes.kfloat8_e5m2, meta=metas['ograd'])
            ograd_fp8_t = None
        else:
            ograd_fp8, ograd_fp8_t = output_grad.fused_cast_transpose(Dtypes.kfloat8_e5m2, meta=metas['ograd'])

        if need_dgrad or need_wgrad:
            input_fp8 = ScalingTensor(input_codes, metas['input'])
            weight_fp8 = ScalingTensor(weight_codes, words if isinstance(words, ScalingMeta) else
                                       ScalingMeta._of_words(Dtypes.kfloat8_e4m3, words))
        if need_dgrad:
            if in_place:
                input_grad = Gemm.fp8_gemm(weight_fp8, ograd_fp8, output_qtype, use_split_accumulator=True, a_kmajor=True)
            else:
                weight_fp8_t = weight_fp8.fp8_transpose()
                input_grad = Gemm.fp8_gemm(weight_fp8_t, ograd_fp8, output_qtype, use_split_accumulator=True)

        if need_wgrad:
            if in_place:
                mat_a, mat_b, layout = input_fp8, ograd_fp8, dict(a_kmajor=True, b_kmajor=True)
            else:
                mat_a, mat_b, layout = input_fp8.fp8_transpose(), ograd_fp8_t, {}
            wgrad = None
            old_wgrad = None
            if ctx.weight.grad is not None:
                # gradient accumulation: add into the dequantized previous gradient
                old_wgrad = ctx.weight.grad.to(ctx.output_dtype)
            if not model_state.use_fp8_ddp:
                # GEMM and cast without reading the product back, where the kernel takes the problem (same bits as the
                # two steps below)
                wgrad = Gemm.fp8_gemm_cast(
                    mat_a, mat_b, output_qtype, metas['wgrad'], sync=True, accumulate=old_wgrad is not None, out=old_wgrad,
                    **layout
                )
            if wgrad is None:
                if old_wgrad is None:
                    wgrad = Gemm.fp8_gemm(mat_a, mat_b, output_qtype, use_split_accumulator=True, **layout)
                else:
                    wgrad = Gemm.fp8_gemm(
                        mat_a, mat_b, output_qtype, accumulate=True, out=old_wgrad, use_split_accumulator=True, **layout
                    )
                if model_state.use_fp8_ddp:
                    wgrad.meta = metas['wgrad']
                else:
                    wgrad = wgrad.cast(Dtypes.kfloat8_e4m3, meta=metas['wgrad'], sync=True)
            del old_wgrad
            ctx.weight.backward_grad_update(wgrad)

        if ctx.need_bias_grad and bias_grad is None:
            bias_grad = output_grad.sum(0).to(ctx.bias_dtype)
        return input_grad, None, None, None, bias_grad, None


class FunctionalOverider:
    """Replaces torch.nn.functional.linear with a version that routes ScalingTensor weights to FP8."""
    EMPTY_GRAD_TENSOR = torch.nn.Parameter(torch.tensor([]))
    _installed = False

    @classmethod
    def override(cls):
        if cls._installed:
            return
        cls._installed = True
        F.linear = cls._get_wrapper_for_linear(F.linear)

    @classmethod
    def _get_wrapper_for_linear(cls, old_fn):
        def new_fn(input, weight, bias=None):
            """linear(input, weight, bias=None): y = x A^T + b; `weight` may be a ScalingTensor carrying
            `_scaling_metas`, in which case the three GEMMs run in FP8 and the bias, rounded to the output dtype
            (the autocast dtype if autocast is on, else the input's), is added in the forward GEMM's epilogue."""
            if not isinstance(input, torch.Tensor):
                raise TypeError(f'input should be a torch.Tensor. current type: {type(input)}')
            if not isinstance(weight, (torch.Tensor, ScalingTensor)):
                raise TypeError(f'weight should be a torch.Tensor or ScalingTensor. current type: {type(weight)}')
            if bias is not None and not isinstance(bias, torch.Tensor):
                raise TypeError(f'bias should be a torch.Tensor. current type: {type(bias)}')
            if isinstance(weight, torch.Tensor):
                return old_fn(input, weight, bias=bias)
            if not hasattr(weight, '_scaling_metas'):
                raise ValueError('weight (ScalingTensor) should have _scaling_metas attribute.')

            model_state.ready_to_scale_tensor = True
            shape = input.shape
            if len(shape) != 2:
                input = input.reshape(-1, shape[-1])
            if torch.is_autocast_enabled():
                output_dtype = torch.get_autocast_dtype('cuda')
            else:
                output_dtype = input.dtype
            out = _FP8GemmFunction.apply(input, weight, weight._scaling_metas, cls.EMPTY_GRAD_TENSOR.type(output_dtype), bias,
                                         torch.is_grad_enabled())
            if len(shape) != 2:
                out = out.view(shape[:-1] + (-1, ))
            return out

        return new_fn


FunctionalOverider.override()
