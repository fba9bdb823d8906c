"""The work that users of this framework have it do, as cases to measure through its public entry points.

Four kinds of call, each over the range that it is used on:

* ``mlp``: a quantised multi-layer perceptron as hls4ml models bring it, through ``GPUModel.predict`` (numpy in, numpy
  out: the call that the reference's users make) or ``GPUModel.execute`` (tensors that are on the GPU already);
* ``encoder``: an int8 transformer encoder block as an ONNX Q/DQ export lowers to, through ``GPUModel.execute`` or
  ``GPUModel.capture`` (the recorded form that serving loops replay);
* ``dense``: one layer through the operator level, in every operand format it takes;
* ``attention``: the fused attention core through the operator level.
"""

import math

import numpy as np
import torch

from aie4ml_amd import ops
from aie4ml_amd.aie_types import RoundingMode
from aie4ml_amd.frontends.builder import GraphBuilder, qint
from aie4ml_amd.workloads import c5_encoder_block

FLOATS = {'bfloat16': torch.bfloat16, 'float32': torch.float32, 'fp8_e4m3': torch.float8_e4m3fn}
BYTES = {'int8': 1, 'uint8': 1, 'int16': 2, 'bfloat16': 2, 'float32': 4, 'fp8_e4m3': 1}


def listed():
    return [
        # the benchmark's small classifier on one batch of 1024 events, from host arrays to host arrays: the call in the
        # reference's tutorials and tests, where latency and host work are everything
        {'name': 'mlp_predict', 'kind': 'mlp', 'call': 'predict', 'widths': '16-64-32-32-5', 'rows': 1024},
        # the same network on a long stream of samples that lie on the GPU (a million: off every tile and wave grid)
        {'name': 'mlp_stream', 'kind': 'mlp', 'call': 'execute', 'widths': '16-64-32-32-5', 'rows': 1000000},
        # one sequence through an encoder block: interactive serving, every launch and every host step counts
        {'name': 'encoder_single', 'kind': 'encoder', 'call': 'execute', 'batch': 1, 'seq': 128, 'hidden': 768, 'heads': 12,
         'ffn': 3072, 'softmax': 'hccs'},
        # the benchmark's encoder block: throughput on a full batch
        {'name': 'encoder_block', 'kind': 'encoder', 'call': 'execute', 'batch': 64, 'seq': 128, 'hidden': 768, 'heads': 12,
         'ffn': 3072, 'softmax': 'hccs'},
        # a small vision transformer's 197 tokens (off every tile grid), accurate Softmax, recorded once and replayed
        {'name': 'encoder_vit', 'kind': 'encoder', 'call': 'capture', 'batch': 32, 'seq': 197, 'hidden': 384, 'heads': 6,
         'ffn': 1536, 'softmax': 'exp'},
        # long sequences (documents, large images): attention is as much work as the projections
        {'name': 'encoder_long', 'kind': 'encoder', 'call': 'execute', 'batch': 4, 'seq': 1024, 'hidden': 768, 'heads': 12,
         'ffn': 3072, 'softmax': 'exp'},
        # the benchmark's single Dense layer: the largest call, shifts of its own for every output channel
        {'name': 'dense_large', 'kind': 'dense', 'a': 'int8', 'w': 'int8', 'out': 'int8', 'rows': 8192, 'k': 4096, 'n': 4096,
         'per_channel': True, 'relu': True, 'rounding': 'conv_even'},
        # a wide layer on a handful of samples: low-latency inference, the weights are the traffic
        {'name': 'dense_few_rows', 'kind': 'dense', 'a': 'int8', 'w': 'int8', 'out': 'int8', 'rows': 16, 'k': 4096, 'n': 4096,
         'per_channel': False, 'relu': True, 'rounding': 'conv_even'},
        # a classifier head behind a ReLU (unsigned activations): nothing in it is a multiple of a tile
        {'name': 'dense_ragged', 'kind': 'dense', 'a': 'uint8', 'w': 'int8', 'out': 'int8', 'rows': 5000, 'k': 1001, 'n': 777,
         'per_channel': False, 'relu': False, 'rounding': 'symmetric_inf'},
        # 16-bit activations, as layers with a wide dynamic range keep them
        {'name': 'dense_int16', 'kind': 'dense', 'a': 'int16', 'w': 'int8', 'out': 'int16', 'rows': 8192, 'k': 768, 'n': 768,
         'per_channel': False, 'relu': False, 'rounding': 'conv_even'},
        # the floating-point path (ComputeDtype bfloat16) on a feed-forward layer
        {'name': 'dense_bfloat16', 'kind': 'dense', 'a': 'bfloat16', 'w': 'bfloat16', 'out': 'bfloat16', 'rows': 4096, 'k': 1024,
         'n': 4096, 'per_channel': False, 'relu': True, 'rounding': 'conv_even'},
        # the benchmark's attention core: 512 heads of 512 queries and keys
        {'name': 'attention_core', 'kind': 'attention', 'batch': 32, 'heads': 16, 'sq': 512, 'sk': 512, 'dim': 64,
         'softmax': 'exp'},
    ]


# ---- ranges ----------------------------------------------------------------------------------------------------------
def _log(rng, lo, hi):
    """A whole number spread evenly over the logarithm of [lo, hi]; every third one is rounded to a multiple of 64, where
    layer sizes tend to lie, the others fall where they fall."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if rng.random() < 1 / 3 and v >= 64:
        v = v // 64 * 64
    return max(lo, min(hi, v))


def _draw_mlp(rng):
    widths = [_log(rng, 8, 256)] + [_log(rng, 8, 256) for _ in range(rng.randint(1, 4))] + [_log(rng, 1, 64)]
    call = rng.choice(['predict', 'execute'])
    return {'kind': 'mlp', 'call': call, 'widths': '-'.join(map(str, widths)),
            'rows': _log(rng, 1, 16384 if call == 'predict' else 1000000)}


def _draw_encoder(rng):
    dim = rng.choice([32, 64, 64, 64, 128])
    heads = rng.randint(2, max(2, 1024 // dim))
    seq = _log(rng, 16, 1024)
    return {'kind': 'encoder', 'call': rng.choice(['execute', 'capture']), 'batch': _log(rng, 1, max(1, 16384 // seq)),
            'seq': seq, 'hidden': heads * dim, 'heads': heads, 'ffn': heads * dim * rng.choice([2, 4]),
            'softmax': rng.choice(['exp', 'hccs'])}


def _draw_dense(rng):
    a, w = rng.choice([('int8', 'int8'), ('int8', 'int8'), ('uint8', 'int8'), ('int16', 'int8'), ('int16', 'int16'),
                       ('bfloat16', 'bfloat16'), ('fp8_e4m3', 'fp8_e4m3'), ('float32', 'float32')])
    whole = a not in FLOATS
    return {'kind': 'dense', 'a': a, 'w': w,
            'out': a if not whole else 'int16' if a == 'int16' else rng.choice(['int8', 'int8', 'uint8', 'int16']),
            'rows': _log(rng, 1, 16384), 'k': _log(rng, 32, 8192), 'n': _log(rng, 8, 8192),
            'per_channel': whole and rng.random() < 0.3, 'relu': rng.random() < 0.5,
            'rounding': rng.choice(['conv_even', 'conv_even', 'symmetric_inf', 'floor']) if whole else 'conv_even'}


def _draw_attention(rng):
    dim = rng.choice([32, 64, 64, 64, 128])
    keys = _log(rng, 16, 512 if dim <= 64 else 256)
    return {'kind': 'attention', 'batch': _log(rng, 1, 64), 'heads': rng.randint(1, 16),
            'sq': keys if rng.random() < 0.7 else _log(rng, 1, 512), 'sk': keys, 'dim': dim,
            'softmax': rng.choice(['exp', 'hccs'])}


def _cost(case):
    w = work(case)
    return max(w['bytes'], w['flops'] / 50)


def draw(rng):
    make = rng.choice([_draw_mlp, _draw_encoder, _draw_encoder, _draw_dense, _draw_dense, _draw_dense, _draw_attention])
    most = max(_cost(c) for c in listed())
    while True:
        case = make(rng)
        if _cost(case) <= most:
            return case


# ---- inputs and parameters -------------------------------------------------------------------------------------------
def _normal(gen, shape, sigma, dtype):
    """Rounded, clipped N(0, sigma): the shape that quantised activations and weights have."""
    info = torch.iinfo(dtype)
    x = torch.randn(shape, generator=gen, device='cuda') * sigma
    if not info.min:
        x = x.abs_()
    return x.round_().clamp_(info.min, info.max).to(dtype)


def _prepare_mlp(case, seed):
    r = np.random.default_rng(seed)
    widths = [int(v) for v in case['widths'].split('-')]
    act, wq, bq = qint(8, 4, rounding=RoundingMode.RND), qint(8, 7), qint(32, 11)
    gb = GraphBuilder(config={'Iterations': 1})
    t = gb.input('x', (case['rows'], widths[0]), act)
    for i, (k, n) in enumerate(zip(widths[:-1], widths[1:])):
        weight = np.clip(np.rint(r.normal(0.0, 128.0 / math.sqrt(k), (k, n))), -128, 127) / 128.0
        t = gb.dense(t, weight, wq, act, bias=r.integers(-1024, 1025, n) / 2048.0, bias_precision=bq,
                     relu=i < len(widths) - 2, name='fc%d' % i)
    gb.output(t)
    model = gb.build()
    model.compile()
    if case['call'] == 'predict':
        return {'run': model.predict, 'x': r.standard_normal((case['rows'], widths[0]), dtype=np.float32) * 2}
    gen = torch.Generator(device='cuda').manual_seed(seed)
    return {'run': model.execute, 'x': {'x': _normal(gen, (case['rows'], widths[0]), 32.0, torch.int8)}}


def _prepare_encoder(case, seed):
    model, x = c5_encoder_block(case['batch'], case['seq'], case['hidden'], case['heads'], case['ffn'], case['softmax'], seed)
    model.compile()
    dev = {'x': torch.from_numpy(x).cuda()}
    return {'run': model.capture(dev) if case['call'] == 'capture' else model.execute, 'x': dev}


def _prepare_dense(case, seed):
    gen = torch.Generator(device='cuda').manual_seed(seed)
    m, k, n = case['rows'], case['k'], case['n']
    if case['a'] in FLOATS:
        fmt = FLOATS[case['a']]
        x = torch.randn((m, k), generator=gen, device='cuda').to(fmt)
        weight = (torch.randn((k, n), generator=gen, device='cuda') / math.sqrt(k)).to(fmt)
        packed = ops.pack_dense_float(weight, torch.randn((n,), generator=gen, device='cuda'))
        return {'run': lambda x: ops.dense_float(x, packed, relu=case['relu']), 'x': x}
    wide, wide_w = case['a'] == 'int16', case['w'] == 'int16'
    sigma, sigma_w = 8192.0 if wide else 32.0, 4096.0 if wide_w else 16.0
    x = _normal(gen, (m, k), sigma, getattr(torch, case['a']))
    weight = _normal(gen, (k, n), sigma_w, getattr(torch, case['w']))
    spread = sigma * sigma_w * math.sqrt(k)  # of the accumulators; the results are to spread over their type
    shift = max(1, int(round(math.log2(spread / (8192.0 if case['out'] == 'int16' else 32.0)))))
    bias = torch.randint(-int(spread) // 2, int(spread) // 2 + 1, (n,), generator=gen, device='cuda').clamp_(-2**31, 2**31 - 1).int()
    shifts = torch.randint(max(0, shift - 2), shift + 3, (n,), generator=gen, device='cuda').cpu() if case['per_channel'] else shift
    packed = ops.pack_dense(weight, bias, shifts)
    return {'run': lambda x: ops.dense(x, packed, case['rounding'], relu=case['relu'], out_kind=case['out']), 'x': x}


def _prepare_attention(case, seed):
    gen = torch.Generator(device='cuda').manual_seed(seed)
    lead = (case['batch'], case['heads'])
    q = _normal(gen, lead + (case['sq'], case['dim']), 24.0, torch.int8)
    k, v = (_normal(gen, lead + (case['sk'], case['dim']), 24.0, torch.int8) for _ in range(2))
    keys = case['sk']
    b = min(255, 32767 // keys)
    sm = {'kind': 'exp', 'exp_kq': 23} if case['softmax'] == 'exp' else {
        'kind': 'hccs', 'B': b, 'S': 1, 'Dmax': min(127, b - max(1, -(-256 // keys)))}
    return {'run': lambda x: ops.attention(x[0], x[1], x[2], 6, 'conv_even', sm, 8, 'conv_even'), 'x': (q, k, v)}


def prepare(case, seed):
    make = {'mlp': _prepare_mlp, 'encoder': _prepare_encoder, 'dense': _prepare_dense, 'attention': _prepare_attention}
    return make[case['kind']](case, seed)


def run(state):
    return state['run'](state['x'])


# ---- what a pass cannot do without -----------------------------------------------------------------------------------
def work(case):
    if case['kind'] == 'mlp':
        widths = [int(v) for v in case['widths'].split('-')]
        macs = sum(k * n for k, n in zip(widths[:-1], widths[1:]))
        per_row = 4 * widths[0] + 8 * widths[-1] if case['call'] == 'predict' else widths[0] + widths[-1]
        return {'bytes': case['rows'] * per_row + macs + 4 * sum(widths[1:]), 'flops': 2 * macs * case['rows']}
    if case['kind'] == 'encoder':
        h, f, rows = case['hidden'], case['ffn'], case['batch'] * case['seq']
        weights = 4 * h * h + 2 * h * f
        return {'bytes': 2 * rows * h + weights + 4 * (5 * h + f) + 8 * h,
                'flops': 2 * rows * weights + 4 * rows * case['seq'] * h}
    if case['kind'] == 'dense':
        m, k, n = case['rows'], case['k'], case['n']
        return {'bytes': m * k * BYTES[case['a']] + k * n * BYTES[case['w']] + m * n * BYTES[case['out']] + 4 * n,
                'flops': 2 * m * k * n}
    heads = case['batch'] * case['heads']
    return {'bytes': heads * case['dim'] * 2 * (case['sq'] + case['sk']), 'flops': 4 * heads * case['sq'] * case['sk'] * case['dim']}


# Whole-number formats are exact. The float formats: a sum in another order moves a result by float32 rounding errors, which
# the rounding to the result's format either hides or turns into one step of that format. Measured over reductions of 32 to
# 8192 against sums in 64 bits and against float32 sums in another order (2-norm; largest value): bfloat16 4.1e-5 and 7.8e-3,
# float32 1.2e-6 and 8.8e-6, fp8 5.9e-4 and 0.11; four times that is allowed.
FLOAT_TOLERANCE = {'bfloat16': {'rel': 1.7e-4, 'max': 0.032}, 'float32': {'rel': 5e-6, 'max': 3.6e-5},
                   'fp8_e4m3': {'rel': 2.4e-3, 'max': 0.45}}


def tolerance(case):
    return FLOAT_TOLERANCE.get(case.get('a'), 'exact')
