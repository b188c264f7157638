"""The work that a user of this framework has it do, as cases to time: quantized linear layers at decode and prefill
sizes, quantized attention products, mixture-of-experts layers, and the quantization of weights.

Every pass goes through the public surface: a model under `quantize_model`, `quantize` + `dot_general`,
`hadamard_quantized_matmul`, `ragged_dot`, `quantize` + `dequantize`.  Weights are quantized beforehand, as post-training
quantization does; activations arrive in floating point and are quantized inside the pass.
"""
from __future__ import annotations

import math

import torch

import qwix_amd
from qwix_amd import nn
from qwix_amd.contrib import hadamard_rot

_DEV = 'cuda'
_DN = (((1,), (0,)), ((), ()))
_FLOAT = {'bf16': torch.bfloat16, 'f32': torch.float32}


def listed():
  return [
      # The two-layer network of the PTQ example on a batch of 256, through the provider: four small launches.
      dict(name='mlp_w8a8', kind='mlp', rows=256, d_in=1024, hidden=4096, d_out=1024, dtype='f32', scheme='w8a8'),
      # One decode step of one sequence against the up-projection of an FFN, weights in int4 groups of 128.
      dict(name='w4a16_decode', kind='linear', rows=1, k=4096, n=14336, weight='int4', group=128, act='', zero_point=False),
      # A short prompt (a length that divides nothing) against the same weight.
      dict(name='w4a16_prompt', kind='linear', rows=333, k=4096, n=14336, weight='int4', group=128, act='', zero_point=False),
      # A decode step of 64 sequences with int8 weights and activations quantized per token.
      dict(name='w8a8_decode', kind='linear', rows=64, k=4096, n=14336, weight='int8', group=0, act='int8', zero_point=False),
      # Prefill of a square projection, int8 per token and per channel.
      dict(name='w8a8_prefill', kind='linear', rows=4096, k=4096, n=4096, weight='int8', group=0, act='int8', zero_point=False),
      # Prefill of a large FFN in float8: the largest product.
      dict(name='fp8_ffn', kind='linear', rows=8192, k=8192, n=28672, weight='float8_e4m3fn', group=0, act='float8_e4m3fn',
           zero_point=False),
      # Sub-channel scales on both operands, as a rule with tile_size=128 gives.
      dict(name='w8a8_subchannel', kind='linear', rows=4096, k=4096, n=4096, weight='int8', group=128, act='int8',
           zero_point=False),
      # Activations rotated, quantized to int8 and multiplied with an int4 weight that was rotated before.
      dict(name='hadamard_a8w4', kind='hadamard', rows=2048, k=8192, n=8192, group=128),
      # Mixture of experts, prefill: rows sorted by expert, uneven groups, int8.
      dict(name='moe_w8a8_prefill', kind='moe', rows=8192, experts=8, k=4096, n=14336, weight='int8', act='int8'),
      # Mixture of experts, decode: a few tokens for each of many experts, weights in int4 groups of 128.
      dict(name='moe_w4a16_decode', kind='moe', rows=256, experts=64, k=2048, n=4096, weight='int4', act=''),
      # Attention scores of 32 heads, both operands quantized inside the model.
      dict(name='attention_qk', kind='attention', product='qk', batch=32, q=2048, kv=2048, d=128, qtype='int8'),
      # A weight quantized per channel and read back, as when its quantization error is looked at.
      dict(name='weight_fp8', kind='weight', k=8192, n=28672, qtype='float8_e4m3fn', group=0, dtype='bf16'),
  ]


def _log(rng, lo, hi, step=1):
  """A multiple of `step` from lo to hi, spread over the logarithm."""
  v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
  return max(lo, min(hi, int(round(v / step)) * step))


_MOST_OPS = 2.0 * 8192 * 8192 * 28672 / 4  # a quarter of the largest listed product


def _rows_within(rng, lo, hi, ops_per_row):
  return _log(rng, lo, max(lo, min(hi, int(_MOST_OPS / ops_per_row))))


def draw(rng):
  kind = rng.choice(['mlp', 'linear', 'linear', 'linear', 'linear', 'hadamard', 'moe', 'moe', 'attention', 'weight'])
  if kind == 'mlp':
    scheme = rng.choice(['w8a8', 'fp8', 'w4a16'])
    d_in, hidden = _log(rng, 256, 4096, 128), _log(rng, 1024, 14336, 128)
    return dict(kind=kind, rows=_log(rng, 1, 2048), d_in=d_in, hidden=hidden, d_out=d_in,
                dtype='bf16' if scheme == 'w4a16' else rng.choice(['f32', 'bf16']), scheme=scheme)
  if kind == 'linear':
    weight, act, group, zero_point = rng.choice([
        ('int4', '', 128, False), ('int4', '', 128, True), ('int8', '', 128, False), ('int8', '', 0, False),
        ('float8_e4m3fn', '', 128, False), ('int8', 'int8', 0, False), ('int8', 'int8', 0, True),
        ('int8', 'int8', 128, False), ('int4', 'int8', 128, False), ('float8_e4m3fn', 'float8_e4m3fn', 0, False),
        ('float8_e4m3fn', 'float8_e4m3fn', 128, False)])
    k = _log(rng, 1024, 14336, 256)
    n = _log(rng, 1024, 28672, rng.choice([8, 64, 256]))
    most = 16 if rng.random() < 0.4 else 8192  # decode batches are as common as prompts
    return dict(kind=kind, rows=_rows_within(rng, 1, most, 2.0 * k * n), k=k, n=n, weight=weight, group=group, act=act,
                zero_point=zero_point)
  if kind == 'hadamard':
    return dict(kind=kind, rows=_log(rng, 1, 4096), k=1 << rng.randint(10, 13), n=_log(rng, 1024, 14336, 64), group=128)
  if kind == 'moe':
    weight, act = rng.choice([('int8', 'int8'), ('float8_e4m3fn', 'float8_e4m3fn'), ('int4', ''), ('int8', '')])
    experts = rng.choice([8, 16, 32, 64])
    k, n = _log(rng, 1024, 4096, 128), _log(rng, 1024, 65536 // experts if experts > 8 else 14336, 64)
    return dict(kind=kind, rows=_rows_within(rng, 8, 8192, 2.0 * k * n), experts=experts, k=k, n=n, weight=weight, act=act)
  if kind == 'attention':
    batch, d = _log(rng, 1, 64), rng.choice([64, 128])
    kv = _log(rng, 128, 8192, 16)
    most = max(1, min(4096, (32 * 2048 * 2048) // (batch * kv)))  # scores no larger than the listed ones
    return dict(kind=kind, product=rng.choice(['qk', 'pv']), batch=batch, q=1 if rng.random() < 0.25 else _log(rng, 1, most),
                kv=kv, d=d, qtype=rng.choice(['int8', 'float8_e4m3fn']))
  qtype, group = rng.choice([('int8', 0), ('int8', 128), ('int4', 128), ('float8_e4m3fn', 0), ('float8_e4m3fn', 128)])
  return dict(kind='weight', k=_log(rng, 512, 8192, 128), n=_log(rng, 512, 28672, rng.choice([8, 64])), qtype=qtype,
              group=group, dtype=rng.choice(['bf16', 'bf16', 'f32']))


# ------------------------------------------------------------------------------------------
# what a program has in hand before the call
# ------------------------------------------------------------------------------------------


def _normal(g, *shape, std=1.0, dtype=torch.bfloat16):
  return (torch.randn(*shape, generator=g, device=_DEV) * std).to(dtype)


def _weight(g, k, n, qtype, group, method='absmax'):
  return qwix_amd.quantize(_normal(g, k, n, std=0.02), qtype, channelwise_axes=[1], tiled_axes={0: group} if group else {},
                           calibration_method=method)


def _scores(params, q, k):
  del params
  return nn.ops.einsum('bqd,bkd->bqk', q, k)


def _mix(params, p, v):
  del params
  return nn.ops.einsum('bqk,bkd->bqd', p, v)


_SCHEMES = {'w8a8': ('int8', 'int8', None), 'fp8': ('float8_e4m3fn', 'float8_e4m3fn', None), 'w4a16': ('int4', None, 128)}


def prepare(case, seed):
  g = torch.Generator(device=_DEV).manual_seed(seed)
  kind = case['kind']
  if kind == 'mlp':
    weight, act, tile = _SCHEMES[case['scheme']]
    dtype = _FLOAT[case['dtype']]
    rule = qwix_amd.QuantizationRule(module_path='.*', weight_qtype=weight, act_qtype=act, tile_size=tile)
    model = qwix_amd.quantize_model(nn.MLP(case['hidden'], case['d_out']), qwix_amd.PtqProvider([rule]))
    params = {'Dense_0': {'kernel': _normal(g, case['d_in'], case['hidden'], std=0.02, dtype=dtype)},
              'Dense_1': {'kernel': _normal(g, case['hidden'], case['d_out'], std=0.02, dtype=dtype)}}
    x = _normal(g, case['rows'], case['d_in'], dtype=dtype)
    return dict(kind=kind, model=model, params=qwix_amd.quantize_params(params, model.init(params, x)), x=x)
  if kind == 'linear':
    method = 'minmax' if case['zero_point'] else 'absmax'
    x = _normal(g, case['rows'], case['k'])
    # an asymmetric operand is the weight where activations stay in bf16, else the activation (shifted, as after a GELU)
    w = _weight(g, case['k'], case['n'], case['weight'], case['group'], 'absmax' if case['act'] else method)
    if case['act'] and case['zero_point']:
      x = x + 0.5
    # per-token scales, or one for each token and group where the rule tiles both operands
    tiled = {1: case['group']} if case['group'] and case['weight'] != 'int4' else {}
    return dict(kind=kind, x=x, w=w, act=case['act'], tiled=tiled, method=method)
  if kind == 'hadamard':
    x = _normal(g, case['rows'], case['k'])
    signs = (torch.randint(0, 2, (case['k'],), generator=g, device=_DEV) * 2 - 1).to(torch.bfloat16)
    return dict(kind=kind, x=x, w=_weight(g, case['k'], case['n'], 'int4', case['group']), signs=signs)
  if kind == 'moe':
    e, k, n = case['experts'], case['k'], case['n']
    w = torch.empty(e, k, n, dtype=torch.bfloat16, device=_DEV)
    for i in range(e):
      w[i] = _normal(g, k, n, std=0.02)
    w = qwix_amd.quantize(w, case['weight'], channelwise_axes=[0, 2], tiled_axes={1: 128} if not case['act'] else {})
    # every token to an expert at random, some experts more popular than others
    popular = torch.rand(e, generator=g, device=_DEV) + 0.5
    expert = torch.multinomial(popular, case['rows'], replacement=True, generator=g)
    sizes = torch.bincount(expert, minlength=e).to(torch.int32)
    return dict(kind=kind, x=_normal(g, case['rows'], k), w=w, sizes=sizes, act=case['act'])
  if kind == 'attention':
    rule = qwix_amd.QuantizationRule(module_path='.*', weight_qtype=case['qtype'], act_qtype=case['qtype'])
    b, q, kv, d = case['batch'], case['q'], case['kv'], case['d']
    if case['product'] == 'qk':
      fn, lhs, rhs = _scores, _normal(g, b, q, d), _normal(g, b, kv, d)
    else:
      probs = torch.softmax(torch.randn(b, q, kv, generator=g, device=_DEV) * 2, dim=-1).to(torch.bfloat16)
      fn, lhs, rhs = _mix, probs, _normal(g, b, kv, d)
    return dict(kind=kind, model=qwix_amd.quantize_model(fn, qwix_amd.PtqProvider([rule])), lhs=lhs, rhs=rhs)
  w = _normal(g, case['k'], case['n'], std=0.02, dtype=_FLOAT[case['dtype']])
  return dict(kind=kind, w=w, qtype=case['qtype'], tiled={0: case['group']} if case['group'] else {})


# ------------------------------------------------------------------------------------------
# one pass
# ------------------------------------------------------------------------------------------


def run(state):
  kind = state['kind']
  if kind == 'mlp':
    return state['model'].apply(state['params'], state['x'])
  if kind == 'linear':
    x = state['x']
    if state['act']:
      x = qwix_amd.quantize(x, state['act'], channelwise_axes=[0], tiled_axes=state['tiled'],
                            calibration_method=state['method'])
    return qwix_amd.dot_general(x, state['w'], _DN)
  if kind == 'hadamard':
    return hadamard_rot.hadamard_quantized_matmul(state['x'], state['w'], state['signs'])
  if kind == 'moe':
    x = state['x']
    if state['act']:
      x = qwix_amd.quantize(x, state['act'], channelwise_axes=[0])
    return qwix_amd.ragged_dot(x, state['w'], state['sizes'])
  if kind == 'attention':
    return state['model'].apply({}, state['lhs'], state['rhs'])
  q = qwix_amd.quantize(state['w'], state['qtype'], channelwise_axes=[1], tiled_axes=state['tiled'])
  values = q.qvalue.data if isinstance(q.qvalue, qwix_amd.Int4Tensor) else q.qvalue
  return [values, q.scale, qwix_amd.dequantize(q)]


# ------------------------------------------------------------------------------------------
# what a pass cannot do without, and how far two correct results may be apart
# ------------------------------------------------------------------------------------------

_SIZE = {'int8': 1.0, 'int4': 0.5, 'float8_e4m3fn': 1.0}


def _weight_bytes(k, n, qtype, group, copies=1):
  return copies * (k * n * _SIZE[qtype] + (k // group if group else 1) * n * 2)


def work(case):
  kind = case['kind']
  if kind == 'mlp':
    weight, _, tile = _SCHEMES[case['scheme']]
    f = 4 if case['dtype'] == 'f32' else 2
    m, i, h, o = case['rows'], case['d_in'], case['hidden'], case['d_out']
    # the hidden layer is written by the first product and read by the second
    return dict(bytes=_weight_bytes(i, h, weight, tile) + _weight_bytes(h, o, weight, tile) + f * m * (i + 2 * h + o),
                flops=2.0 * m * h * (i + o))
  if kind in ('linear', 'hadamard'):
    m, k, n = case['rows'], case['k'], case['n']
    return dict(bytes=_weight_bytes(k, n, case.get('weight', 'int4'), case['group']) + 2 * m * (k + n), flops=2.0 * m * k * n)
  if kind == 'moe':
    m, k, n = case['rows'], case['k'], case['n']
    used = min(case['experts'], m)
    return dict(bytes=_weight_bytes(k, n, case['weight'], 0 if case['act'] else 128, used) + 2 * m * (k + n),
                flops=2.0 * m * k * n)
  if kind == 'attention':
    b, q, kv, d = case['batch'], case['q'], case['kv'], case['d']
    return dict(bytes=2.0 * b * (q * d + kv * d + q * kv), flops=2.0 * b * q * kv * d)
  f = 4 if case['dtype'] == 'f32' else 2
  k, n = case['k'], case['n']
  # the weight in, its codes out; the codes in, the weight out
  return dict(bytes=2.0 * (k * n * f + _weight_bytes(k, n, case['qtype'], case['group'])), flops=0.0)


# Measured against 64-bit sums of the same quantized operands (and, in the MLP, against hidden activations quantized again
# from 64-bit values: a code that falls on the other side of a rounding step moves the result by a step), then times four.
_MLP = {('w8a8', 'f32'): (1.6e-4, 8e-3), ('fp8', 'f32'): (4e-3, 7e-2), ('w8a8', 'bf16'): (0.03, 0.21),
        ('fp8', 'bf16'): (0.03, 0.5), ('w4a16', 'bf16'): (0.013, 0.062)}


def tolerance(case):
  if case['kind'] == 'weight':
    return 'exact'  # every operation of the quantization is rounded as the reference rounds it
  rel, largest = _MLP[case['scheme'], case['dtype']] if case['kind'] == 'mlp' else (0.0116, 0.043)
  return {'rel': rel, 'max': largest}
