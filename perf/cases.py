"""Performance cases: what programs built on msamp spend their GPU time on, through the public entry points.

Five kinds of work, each a function of a case's plain values:

train   one training step of a residual MLP set up by msamp.initialize: zero_grad, forward, loss, backward, gradient
        clipping, optimizer step (opt_level O1: float32 moments, O2: E4M3 / scaled-float16 moments).
linear  forward and backward of one FP8Linear in the steady state of delayed scaling, over one or more micro-batches
        (from the second on the weight gradient is added into the FP8 gradient of the ones before).
eval    forward of one FP8Linear without gradients.
cast    Tensor.cast to FP8 with a fresh meta, and back to a float type.
adamw   LBAdamW.step() over a list of FP8 / scaled-float16 parameters with FP8 gradients.
bucket  GradientBucket.quantize over the gradients of a bucket, and msamp.clip_grad_norm_ over the result.
"""

import math
import os
import sys

import torch

sys.path.insert(0, os.path.abspath('ms-amp_amd'))    # the package of the tree that is the working folder

import msamp    # noqa: E402
from msamp.common.dtype import Dtypes    # noqa: E402
from msamp.common.tensor import ScalingTensor    # noqa: E402
from msamp.nn import GradientBucket, LinearReplacer, ScalingParameter, model_state    # noqa: E402
from msamp.optim import LBAdamW    # noqa: E402

_DTYPES = {'fp32': torch.float32, 'fp16': torch.float16, 'bf16': torch.bfloat16}
_QTYPES = {'e4m3': Dtypes.kfloat8_e4m3, 'e5m2': Dtypes.kfloat8_e5m2, 'fp16': Dtypes.kfloat16}
_SIZE = {'fp32': 4, 'fp16': 2, 'bf16': 2, 'e4m3': 1, 'e5m2': 1}
_WINDOW = 16    # amax windows of FP8Linear: after this many updates scaling is delayed, as for the rest of a run


# ---- the cases --------------------------------------------------------------------------------------------------
def listed():
    return [
        # A toy-sized model (the sizes of the unit tests): every call is launch and host latency.
        dict(name='train_tiny_o2', kind='train', level='O2', dtype='fp32', tokens=96, hidden=128, blocks=2, autocast=False),
        # The default opt_level on a small transformer's MLPs, float32 model under autocast as training scripts have it.
        dict(name='train_small_o1', kind='train', level='O1', dtype='fp32', tokens=2048, hidden=1024, blocks=2, autocast=True),
        # A bfloat16 model of medium width under O2: GEMMs, casts and the optimizer all weigh in.
        dict(name='train_medium_o2', kind='train', level='O2', dtype='bf16', tokens=8192, hidden=2048, blocks=2, autocast=False),
        # One square projection at 8192 tokens: the single-layer configuration of the benchmark.
        dict(name='linear_square', kind='linear', dtype='bf16', tokens=8192, d_in=4096, d_out=4096, bias=False, micro=1),
        # The down projection of a Llama-70B layer: the longest K, the largest call.
        dict(name='linear_long_k', kind='linear', dtype='bf16', tokens=16384, d_in=28672, d_out=8192, bias=False, micro=1),
        # The gate projection of a Llama-7B layer with gradient accumulation over two micro-batches.
        dict(name='linear_accumulate', kind='linear', dtype='bf16', tokens=16384, d_in=4096, d_out=11008, bias=False, micro=2),
        # Packed sequences of uneven length, float16 with a bias, widths that are no multiple of a tile.
        dict(name='linear_ragged', kind='linear', dtype='fp16', tokens=12605, d_in=1200, d_out=4304, bias=True, micro=1),
        # Evaluation on a handful of tokens: the layer's weight is most of what is read.
        dict(name='eval_few_tokens', kind='eval', dtype='bf16', tokens=48, d_in=4096, d_out=12288, bias=True),
        # Quantize and dequantize a float32 tensor with rare outliers.
        dict(name='cast_round_trip', kind='cast', dtype='fp32', rows=4096, cols=4096, qtype='e4m3', back='fp32', outliers=100.0),
        # One MLP weight of a Llama-70B layer to FP8.
        dict(name='cast_weight', kind='cast', dtype='bf16', rows=28672, cols=8192, qtype='e4m3', back='', outliers=50.0),
        # The optimizer step of two Llama-7B layers (QKV, O, gate, up, down each), E4M3 weights, E5M2 gradients.
        dict(name='adamw_layers', kind='adamw', level='O2', weight='e4m3', grad='e5m2', tensors=10, rows=9881, cols=4096),
        # A bucket of 32 gradients on its way into a data-parallel reduction, then clipped.
        dict(name='bucket_clip', kind='bucket', dtype='bf16', tensors=32, rows=4096, cols=1024, even=True),
    ]


def _log(rng, low, high):
    return math.exp(rng.uniform(math.log(low), math.log(high)))


def _width(rng, low, high):
    """A layer width: mostly a multiple of 64 or 16, sometimes any number."""
    unit = rng.choice((256, 64, 16, 16, 8, 1))
    return max(1, round(_log(rng, low, high) / unit)) * unit if unit < high else int(high)


def _most_flops():
    return max(work(c)['flops'] for c in listed())


def draw(rng):
    kind = rng.choice(('train', 'linear', 'linear', 'eval', 'cast', 'adamw', 'bucket'))
    if kind == 'train':
        autocast = rng.random() < 0.5
        case = dict(kind=kind, level=rng.choice(('O1', 'O2')), dtype='fp32' if autocast else rng.choice(('fp32', 'bf16')),
                    tokens=int(_log(rng, 32, 8192)), hidden=_width(rng, 64, 2048), blocks=rng.randint(1, 2),
                    autocast=autocast)
    elif kind == 'linear':
        case = dict(kind=kind, dtype=rng.choice(('bf16', 'bf16', 'fp16')), tokens=int(_log(rng, 64, 16384)),
                    d_in=_width(rng, 128, 28672), d_out=_width(rng, 128, 28672), bias=rng.random() < 0.5,
                    micro=rng.choice((1, 1, 2)))
    elif kind == 'eval':
        case = dict(kind=kind, dtype=rng.choice(('bf16', 'fp16')), tokens=int(_log(rng, 1, 4096)),
                    d_in=_width(rng, 256, 16384), d_out=_width(rng, 256, 16384), bias=rng.random() < 0.5)
    elif kind == 'cast':
        case = dict(kind=kind, dtype=rng.choice(('fp32', 'bf16', 'fp16')), rows=int(_log(rng, 16, 28672)),
                    cols=_width(rng, 64, 8192), qtype=rng.choice(('e4m3', 'e5m2')),
                    back=rng.choice(('', 'fp32', 'bf16', 'fp16')), outliers=rng.choice((1.0, 50.0, 100.0)))
    elif kind == 'adamw':
        level = rng.choice(('O1', 'O2', 'O2'))
        case = dict(kind=kind, level=level, weight='fp16' if level == 'O1' else rng.choice(('e4m3', 'fp16')),
                    grad=rng.choice(('e4m3', 'e5m2')), tensors=rng.randint(1, 10), rows=int(_log(rng, 16, 9881)),
                    cols=_width(rng, 64, 4096))
    else:
        case = dict(kind=kind, dtype=rng.choice(('fp32', 'bf16', 'fp16')), tensors=rng.randint(2, 32),
                    rows=int(_log(rng, 16, 4096)), cols=_width(rng, 16, 1024), even=rng.random() < 0.5)
    # a drawn case costs no more than the largest listed one
    while 'tokens' in case and case['tokens'] > 1 and work(case)['flops'] > _most_flops():
        case['tokens'] //= 2
    return case


def _adamw_rows(case):
    """Rows of each parameter: like the five projections of a layer, of three different lengths."""
    r = case['rows']
    lengths = (r * 12288 // 9881, r * 4096 // 9881, r * 11008 // 9881, r * 11008 // 9881, r * 11008 // 9881)
    return [max(1, lengths[i % 5]) for i in range(case['tensors'])]


def _bucket_rows(case):
    return [case['rows'] if case['even'] else max(1, case['rows'] >> i % 3) for i in range(case['tensors'])]


# ---- inputs ------------------------------------------------------------------------------------------------------
class _Block(torch.nn.Module):
    """x + down(gelu(up(norm(x))))"""
    def __init__(self, hidden):
        super().__init__()
        self.norm = torch.nn.LayerNorm(hidden)
        self.up = torch.nn.Linear(hidden, 4 * hidden)
        self.down = torch.nn.Linear(4 * hidden, hidden)

    def forward(self, x):
        return x + self.down(torch.nn.functional.gelu(self.up(self.norm(x))))


def _randn(gen, shape, dtype, std=1.0):
    return (torch.randn(shape, device='cuda', generator=gen) * std).to(dtype)


def _prepare_train(case, gen):
    dtype = _DTYPES[case['dtype']]
    model = torch.nn.Sequential(*[_Block(case['hidden']) for _ in range(case['blocks'])]).cuda()
    with torch.no_grad():
        # weights as in a run: no parameter is zero or one throughout, the projections back into the residual stream are
        # the smaller ones (0.02 / sqrt(2 * 12), as for a stack of twelve blocks)
        for name, p in model.named_parameters():
            std = 0.004 if name.endswith('down.weight') else 0.02
            p.copy_(_randn(gen, p.shape, p.dtype, std) + (1.0 if name.endswith('norm.weight') else 0.0))
    model = model.to(dtype)
    optimizer = torch.optim.AdamW(model.parameters(), lr=3e-5, weight_decay=0.1)
    model, optimizer = msamp.initialize(model, optimizer, opt_level=case['level'])
    x = _randn(gen, (case['tokens'], case['hidden']), dtype)
    target = _randn(gen, (case['tokens'], case['hidden']), dtype)
    return dict(model=model, optimizer=optimizer, params=list(model.parameters()), x=x, target=target)


def _layer(case, gen):
    dtype = _DTYPES[case['dtype']]
    linear = torch.nn.Linear(case['d_in'], case['d_out'], bias=case['bias'], device='cuda', dtype=dtype)
    with torch.no_grad():
        linear.weight.copy_(_randn(gen, linear.weight.shape, dtype, 0.02))
        if case['bias']:
            linear.bias.copy_(_randn(gen, linear.bias.shape, dtype, 0.02))
    return LinearReplacer.replace(linear)


def _prepare_linear(case, gen):
    dtype = _DTYPES[case['dtype']]
    layer = _layer(case, gen)
    optimizer = LBAdamW(layer.parameters(), lr=0.0, weight_decay=0.0)
    xs, dys = [], []
    for _ in range(case['micro']):
        xs.append(_randn(gen, (case['tokens'], case['d_in']), dtype).requires_grad_(True))
        dys.append(_randn(gen, (case['tokens'], case['d_out']), dtype, 1e-3))
    state = dict(layer=layer, xs=xs, dys=dys)
    _fill_windows(layer, optimizer, lambda: layer(xs[0]).backward(dys[0]))
    return state


def _fill_windows(layer, optimizer, one_pass):
    """The first steps of a run, up to where the amax windows are full and scaling is delayed from then on."""
    for _ in range(_WINDOW + 1):
        one_pass()
        layer.weight.grad = None
        if layer.bias is not None:
            layer.bias.grad = None
        optimizer.step()    # no gradients: only the windows move


def _prepare_eval(case, gen):
    layer = _layer(case, gen)
    optimizer = LBAdamW(layer.parameters(), lr=0.0, weight_decay=0.0)
    x = _randn(gen, (case['tokens'], case['d_in']), _DTYPES[case['dtype']])
    state = dict(layer=layer.eval(), x=x)

    def one_pass():
        with torch.no_grad():
            layer(x)

    _fill_windows(layer, optimizer, one_pass)
    return state


def _prepare_cast(case, gen):
    x = _randn(gen, (case['rows'], case['cols']), _DTYPES[case['dtype']])
    n = x.numel()
    at = torch.randint(0, n, (max(1, n // 1000), ), device='cuda', generator=gen)
    x.view(-1)[at] *= case['outliers']
    return dict(x=x, qtype=_QTYPES[case['qtype']], back=case['back'])


def _prepare_adamw(case, gen):
    params = []
    for rows in _adamw_rows(case):
        shape = (rows, case['cols'])
        p = ScalingParameter(_randn(gen, shape, torch.float32, 0.02).cast(_QTYPES[case['weight']]))
        p.grad = _randn(gen, shape, torch.float32, 1e-3).cast(_QTYPES[case['grad']])
        params.append(p)
    moments = dict(exp_avg_dtype=torch.float32, exp_avg_sq_dtype=torch.float32) if case['level'] == 'O1' else {}
    optimizer = LBAdamW(params, lr=3e-4, betas=(0.9, 0.95), weight_decay=0.1, **moments)
    return dict(optimizer=optimizer, params=params)


def _prepare_bucket(case, gen):
    dtype = _DTYPES[case['dtype']]
    shapes = [(rows, case['cols']) for rows in _bucket_rows(case)]
    grads = [_randn(gen, shape, dtype, 1e-3) for shape in shapes]
    params = [ScalingParameter(_randn(gen, shape, torch.float32, 0.02).cast(Dtypes.kfloat16)) for shape in shapes]
    return dict(bucket=GradientBucket([g.numel() for g in grads]), grads=grads, params=params)


_PREPARE = dict(train=_prepare_train, linear=_prepare_linear, eval=_prepare_eval, cast=_prepare_cast, adamw=_prepare_adamw,
                bucket=_prepare_bucket)


def prepare(case, seed):
    gen = torch.Generator(device='cuda').manual_seed(seed)
    model_state.clear()    # a program has one model: every state here is one program's
    state = _PREPARE[case['kind']](case, gen)
    state['kind'] = case['kind']
    state['autocast'] = case.get('autocast', False)
    state['metas'] = model_state.flattened_scaling_metas
    return state


# ---- one pass ----------------------------------------------------------------------------------------------------
def _parts(tensors):
    """Payloads and scales of ScalingTensors, plain tensors as they are."""
    out = []
    for t in tensors:
        if isinstance(t, ScalingTensor):
            out += [t.value, t.meta.scale_inv]
        elif t is not None:
            out.append(t.detach())
    return out


def _run_train(state):
    model, optimizer, params = state['model'], state['optimizer'], state['params']
    optimizer.zero_grad()
    with torch.autocast('cuda', dtype=torch.bfloat16, enabled=state['autocast']):
        y = model(state['x'])
        loss = torch.nn.functional.mse_loss(y.float(), state['target'].float())
    loss.backward()
    msamp.clip_grad_norm_(params, 1.0)
    optimizer.step()
    return [y.detach(), loss.detach()] + _parts(params)


def _run_linear(state):
    layer = state['layer']
    layer.weight.grad = None
    if layer.bias is not None:
        layer.bias.grad = None
    out = []
    for x, dy in zip(state['xs'], state['dys']):
        x.grad = None
        y = layer(x)
        y.backward(dy)
        out += [y.detach(), x.grad]
    return out + _parts([layer.weight.grad, layer.bias.grad if layer.bias is not None else None])


def _run_eval(state):
    with torch.no_grad():
        return state['layer'](state['x'])


def _run_cast(state):
    q = state['x'].cast(state['qtype'])
    out = [q.value, q.meta.scale_inv, q.meta.amax]
    if state['back']:
        out.append(q.to(_DTYPES[state['back']]))
    return out


def _run_adamw(state):
    optimizer, params = state['optimizer'], state['params']
    optimizer.step()
    out = _parts(params)
    for p in params:
        s = optimizer.state[p]
        out += _parts([s['exp_avg'], s['exp_avg_sq']])
    return out


def _run_bucket(state):
    params = state['params']
    for p, g in zip(params, state['bucket'].quantize(state['grads'], world_size=8)):
        p.grad = g
    norm = msamp.clip_grad_norm_(params, 1.0)
    return [state['bucket'].flat, norm] + [p.grad.meta.scale_inv for p in params]


_RUN = dict(train=_run_train, linear=_run_linear, eval=_run_eval, cast=_run_cast, adamw=_run_adamw, bucket=_run_bucket)


def run(state):
    model_state.flattened_scaling_metas = state['metas']    # (the program whose turn it is)
    return _RUN[state['kind']](state)


# ---- what a pass cannot do without -------------------------------------------------------------------------------
def work(case):
    kind = case['kind']
    if kind == 'train':
        t, h, b = case['tokens'], case['hidden'], case['blocks']
        n = 8 * h * h * b    # FP8 weights
        state = 8 if case['level'] == 'O1' else 3
        # weights (scaled float16) and moments read and written, input, target and output once
        return dict(flops=6.0 * t * n, bytes=float(2 * n * (2 + state) + 3 * t * h * _SIZE[case['dtype']]))
    if kind in ('linear', 'eval'):
        t, i, o, size = case['tokens'], case['d_in'], case['d_out'], _SIZE[case['dtype']]
        if kind == 'eval':
            return dict(flops=2.0 * t * i * o, bytes=float(size * t * (i + o) + 2 * i * o))
        m = case['micro']
        # x, dy in, y, dx out; the float16 weight in, its FP8 gradient out
        return dict(flops=6.0 * m * t * i * o, bytes=float(m * 2 * size * t * (i + o) + 3 * i * o))
    n = case['cols'] * (sum(_adamw_rows(case)) if kind == 'adamw' else sum(_bucket_rows(case)) if kind == 'bucket' else case['rows'])
    if kind == 'cast':
        per = _SIZE[case['dtype']] + 1 + (1 + _SIZE[case['back']] if case['back'] else 0)
    elif kind == 'adamw':
        per = 1 + 2 * (_SIZE[case['weight']] + (8 if case['level'] == 'O1' else 3))
    else:
        per = _SIZE[case['dtype']] + 2    # gradients in, codes out, codes in for the norm
    return dict(flops=0.0, bytes=float(n * per))


def tolerance(case):
    """Casts, optimizer steps on given gradients and quantized buckets are element-wise with exact maxima: the same bits.

    Where FP8 products are summed, another order of the sum moves results by a rounding of the output type and, in the
    weight gradient, codes that lie at a tie.  Measured against float32 products over two halves of K: outputs 2.3e-4
    (bfloat16), at most 7.8e-3 in one value, 7.7e-4 of the gradient's codes; four times that is stated.

    In a training step such roundings are quantized to FP8 again and again on their way (forward, backward): measured
    the same way 6.8e-3 over the output and the updated weights of two blocks, at most 4.2e-2 in one value."""
    if case['kind'] in ('cast', 'adamw'):
        return 'exact'
    if case['kind'] == 'bucket':
        return {'rel': 1e-6, 'max': 1e-5, 'differ': 0.0}
    if case['kind'] == 'train':
        return {'rel': 0.027, 'max': 0.17, 'differ': 0.0}
    return {'rel': 1e-3, 'max': 3.2e-2, 'differ': 3e-3}
