"""GPU parity through the provider surface: QuantizationRule -> PtqProvider -> quantize_model /
quantize_params, on the PTQ MLP benchmark configuration and on an einsum layer."""
import numpy as np
import pytest
import torch

from oracle import qwix_oracle as O
from tests import util

pytestmark = pytest.mark.gpu
DN = (((1,), (0,)), ((), ()))


def _mlp_setup(batch=256, d_in=1024, hidden=4096, d_out=1024):
  import qwix_amd
  from qwix_amd import nn
  model = nn.MLP(hidden, d_out)
  g = torch.Generator().manual_seed(1001)
  params = model.init(g, d_in, torch.float32, util.DEV)
  x = torch.rand(batch, d_in, generator=g, dtype=torch.float32).to(util.DEV)
  rules = [qwix_amd.QuantizationRule(module_path='.*', weight_qtype='int8', act_qtype='int8')]
  return model, params, x, rules


def _oracle_mlp(params, x):
  """The reference's flow restated with the oracle: per-channel int8 weights, per-token int8 activations."""
  w1 = util.farr(params['Dense_0']['kernel'])
  w2 = util.farr(params['Dense_1']['kernel'])
  hw = O.HowToQuantize(qtype='int8', channelwise_axes=[1])
  ha = O.HowToQuantize(qtype='int8', channelwise_axes=[0])
  w1q, w2q = O.quantize(w1, hw), O.quantize(w2, hw)
  xq = O.quantize(util.farr(x), ha)
  h, acc1 = O.fast_dot_general(xq, w1q, DN, return_acc=True)
  h = O.FArr(np.maximum(h.v, 0), O.F32)
  hq = O.quantize(h, ha)
  out, acc2 = O.fast_dot_general(hq, w2q, DN, return_acc=True)
  return dict(w1q=w1q, w2q=w2q, xq=xq, hq=hq, acc1=acc1, acc2=acc2, out=out)


def test_config1_ptq_mlp_quantize_params_then_apply():
  import qwix_amd
  from qwix_amd.providers.ptq import WithAux
  model, params, x, rules = _mlp_setup()
  ptq_model = qwix_amd.quantize_model(model, qwix_amd.PtqProvider(rules))
  abstract = ptq_model.init(params, x)                        # PTQ param tree with `how`
  qparams = qwix_amd.quantize_params(params, abstract)        # offline weight quantization
  want = _oracle_mlp(params, x)
  for name, key, n in (('Dense_0', 'w1q', 4096), ('Dense_1', 'w2q', 1024)):
    leaf = qparams[name]['kernel']
    assert isinstance(leaf, WithAux) and tuple(leaf.array.scale.shape) == (1, n) and leaf.array.scale.dtype == torch.float32
    assert leaf.array.qvalue.dtype == torch.int8 and tuple(leaf.array.shape) == tuple(params[name]['kernel'].shape)
    util.assert_qarray_equal(leaf.array, want[key], name)
  out = ptq_model.apply(qparams, x)
  assert out.dtype == torch.float32 and tuple(out.shape) == (256, 1024)
  got = util.f32np(out)
  assert np.array_equal(got, want['out'].v), np.abs(got - want['out'].v).max()
  # quantize_params == implicit quantization on first use (ptq_test.py:68-80)
  for name in ('Dense_0', 'Dense_1'):
    a, b = abstract[name]['kernel'].array, qparams[name]['kernel'].array
    assert torch.equal(a.qvalue, b.qvalue) and torch.equal(a.scale, b.scale)
  # and close to the float model
  ref = model(params, x)
  assert (out - ref).abs().mean() / ref.abs().mean() < 0.02


def test_config1_intermediate_accumulators_and_activation_quantization():
  from qwix_amd.core import dot_general as dg
  from qwix_amd.core import qarray
  model, params, x, _ = _mlp_setup()
  want = _oracle_mlp(params, x)
  hw = qarray.HowToQuantize(qtype='int8', channelwise_axes=[1])
  ha = qarray.HowToQuantize(qtype='int8', channelwise_axes=[0])
  w1q, w2q = qarray.quantize(params['Dense_0']['kernel'], hw), qarray.quantize(params['Dense_1']['kernel'], hw)
  xq = qarray.quantize(x, ha)
  util.assert_qarray_equal(xq, want['xq'], 'x')
  h, acc1 = dg._fast_dot_general(xq, w1q, DN, return_accumulators=True)
  assert np.array_equal(acc1.cpu().numpy(), want['acc1'])
  hq = qarray.quantize(torch.relu(h), ha)
  util.assert_qarray_equal(hq, want['hq'], 'hidden')
  _, acc2 = dg._fast_dot_general(hq, w2q, DN, return_accumulators=True)
  assert np.array_equal(acc2.cpu().numpy(), want['acc2'])


def test_unquantized_rule_and_unused_rules():
  import qwix_amd
  model, params, x, _ = _mlp_setup(batch=16, d_in=128, hidden=256, d_out=64)
  rules = [qwix_amd.QuantizationRule(module_path='Dense_0', weight_qtype='int8'),
           qwix_amd.QuantizationRule(module_path='nothing', weight_qtype='int4')]
  prov = qwix_amd.PtqProvider(rules)
  pm = qwix_amd.quantize_model(model, prov)
  p = pm.init(params, x)
  from qwix_amd.providers.ptq import WithAux
  assert isinstance(p['Dense_0']['kernel'], WithAux) and isinstance(p['Dense_1']['kernel'], torch.Tensor)
  assert [r.module_path for r in prov.get_unused_rules()] == ['nothing']
  out = pm.apply(p, x)   # weight-only int8 on layer 0 (dequantize path), float layer 1
  ref = model(params, x)
  assert (out - ref).abs().mean() / ref.abs().mean() < 0.01
  with pytest.raises(ValueError, match='not found in the abstract'):
    qwix_amd.quantize_params({'Other': {'kernel': params['Dense_0']['kernel']}}, p)
  assert qwix_amd.quantize_params({'Other': {'kernel': params['Dense_0']['kernel']}}, p, allow_extra_params=True) == {}


def test_einsum_layer_with_subchannel_rule():
  """'btd,dnh->btnh' weight (d, n, h) contracting d, tile 128: scale (d/128, n, h) (ptq_test.py shapes)."""
  import qwix_amd
  from qwix_amd import nn
  layer = nn.Einsum('btd,dnh->btnh', (256, 4, 32))
  g = torch.Generator().manual_seed(5)
  params = layer.init(g, torch.bfloat16, util.DEV)
  x = torch.randn(2, 24, 256, generator=g).to(torch.bfloat16).to(util.DEV)
  rules = [qwix_amd.QuantizationRule(weight_qtype='int4', act_qtype='int8', tile_size=128)]
  pm = qwix_amd.quantize_model(lambda p, x: layer(p, x), qwix_amd.PtqProvider(rules))
  qp = pm.init(params, x)
  wq = qp['kernel'].array
  assert tuple(wq.scale.shape) == (2, 4, 32) and wq.qtype == 'int4'
  out = pm.apply(qp, x)
  assert tuple(out.shape) == (2, 24, 4, 32)
  ow = O.quantize(util.farr(params['kernel']), O.HowToQuantize(qtype='int4', channelwise_axes=[1, 2], tiled_axes={0: 128}))
  util.assert_qarray_equal(wq, ow, 'einsum weight')
  ox = O.quantize(util.farr(x), O.HowToQuantize(qtype='int8', channelwise_axes=[0, 1], tiled_axes={2: 128}))
  want, wacc = O.fast_dot_general(ox, ow, (((2,), (0,)), ((), ())), return_acc=True)
  got = util.f32np(out)
  sx = ox.scale.v.reshape(-1, 2)
  mag = (np.abs(wacc.reshape(2, 48, 128)).astype(np.float64) * sx.T[:, :, None] * ow.scale.v.reshape(2, 1, 128)).sum(0).reshape(want.v.shape)
  assert np.all(np.abs(got - want.v) <= 1e-2 * np.abs(want.v) + 2.0**-7 * mag)


def test_small_tile_rule_takes_the_dequantize_path():
  """(12, 5) kernel with tile 4 -> scale (3, 5) (ptq_test.py:698-730); tile < 128 => slow path."""
  import qwix_amd
  from qwix_amd import nn
  layer = nn.Dense(5, name='Dense_0')
  g = torch.Generator().manual_seed(6)
  params = layer.init(g, 12, torch.float32, util.DEV, std=1.0)
  x = torch.randn(3, 12, generator=g).to(util.DEV)
  pm = qwix_amd.quantize_model(lambda p, x: layer(p, x), qwix_amd.PtqProvider([qwix_amd.QuantizationRule(weight_qtype='int8', tile_size=4)]))
  qp = pm.init(params, x)
  assert tuple(qp['kernel'].array.scale.shape) == (3, 5)
  out = pm.apply(qp, x)
  ow = O.quantize(util.farr(params['kernel']), O.HowToQuantize(qtype='int8', channelwise_axes=[1], tiled_axes={0: 4}))
  util.assert_qarray_equal(qp['kernel'].array, ow, 'tile 4 weight')
  want = O.dot_general(util.farr(x), ow, DN)
  assert np.allclose(util.f32np(out), want.v, rtol=1e-5, atol=1e-6)


def test_two_dim_tile_rule():
  """ptq_test.py:698-730: tile_size given as a mapping {0: 2, 1: 2} is used verbatim: an (8, 16) kernel gets
  (4, 8) scales, through Dense and through an einsum, and the weight-only forward dequantizes per block."""
  import qwix_amd
  from qwix_amd import nn
  layer = nn.Dense(16, name='Dense_0')
  g = torch.Generator().manual_seed(7)
  params = layer.init(g, 8, torch.float32, util.DEV, std=1.0)
  x = torch.ones(2, 8, device=util.DEV)
  rules = [qwix_amd.QuantizationRule(weight_qtype='int8', tile_size={0: 2, 1: 2})]
  pm = qwix_amd.quantize_model(lambda p, x: layer(p, x), qwix_amd.PtqProvider(rules))
  qp = pm.init(params, x)
  assert tuple(qp['kernel'].array.scale.shape) == (4, 8)
  out = pm.apply(qp, x)
  assert tuple(out.shape) == (2, 16)
  how = O.HowToQuantize(qtype='int8', tiled_axes={0: 2, 1: 2})
  ow = O.quantize(util.farr(params['kernel']), how)
  util.assert_qarray_equal(qp['kernel'].array, ow, '2 x 2 block weight')
  want = O.dot_general(util.farr(x), ow, DN)
  bias = util.f32np(params['bias']) if 'bias' in params else 0.0
  assert np.allclose(util.f32np(out), want.v + bias, rtol=1e-5, atol=1e-6)

  ein = nn.Einsum('ij,jk->ik', (8, 16))
  eparams = ein.init(g, torch.float32, util.DEV)
  pm = qwix_amd.quantize_model(lambda p, x: ein(p, x), qwix_amd.PtqProvider(rules))
  qp = pm.init(eparams, x)
  assert tuple(qp['kernel'].array.scale.shape) == (4, 8)
  out = pm.apply(qp, x)
  want = O.dot_general(util.farr(x), O.quantize(util.farr(eparams['kernel']), how), DN)
  assert tuple(out.shape) == (2, 16) and np.allclose(util.f32np(out), want.v, rtol=1e-5, atol=1e-6)


@pytest.mark.parametrize('method', ['absmax', 'minmax'])
def test_static_range_rule_end_to_end(method):
  """ptq_test.py:86-143 without the training-time provider: statistics collected over three batches
  ({'count', 'sum_of_*'}, averaging.py:38-64), the PTQ model's abstract params hold `dot_general0_lhs_scale`
  as a (1, 1) WithAux (plus `_zero_point` for minmax), quantize_params turns the statistics into scale and
  zero point (ptq.py:106-129), and the forward uses them; every stage is checked against the oracle."""
  import qwix_amd
  from qwix_amd import averaging, nn
  from qwix_amd.core import qarray
  from qwix_amd.providers import ptq
  dense = nn.Dense(5, name='Dense_0')
  g = torch.Generator().manual_seed(8)
  params = dense.init(g, 12, torch.float32, util.DEV, std=1.0)
  rules = [qwix_amd.QuantizationRule(module_path='.*', weight_qtype='int8', act_qtype='int8', act_static_scale=True,
                                     act_calibration_method=method)]
  how = qarray.HowToQuantize(qtype='int8', channelwise_axes=[0], calibration_method=method)
  agg = averaging.SimpleMovingAverage()
  stat, batches = None, []
  for _ in range(3):
    xb = (torch.randn(10, 12, generator=g) + 0.3).to(util.DEV)
    batches.append(xb)
    cal = {k: v.mean(dim=0, keepdim=True) for k, v in qarray.calibrate(xb, how).items()}  # act_batch_axes = (0,)
    stat = agg.init(cal) if stat is None else stat
    assert stat['count'].shape == () and all(v.shape == (1, 1) for k, v in stat.items() if k != 'count')
    stat = agg.update(stat, cal)
  assert int(stat['count']) == 3
  with pytest.raises(ValueError, match='Shape mismatch'):
    agg.update(stat, {k: v.reshape(1) for k, v in cal.items()})

  x = batches[0]
  pm = qwix_amd.quantize_model(lambda p, x: dense(p, x), qwix_amd.PtqProvider(rules))
  abstract = pm.init(params, x)
  assert isinstance(abstract['dot_general0_lhs_scale'], ptq.WithAux)
  assert abstract['dot_general0_lhs_scale'].array.shape == (1, 1)
  if method == 'minmax':
    assert abstract['dot_general0_lhs_zero_point'].shape == (1, 1)
  with pytest.raises(ValueError, match='not initialized'):
    qwix_amd.quantize_params(params, abstract, {'dot_general0_lhs': agg.init(cal)})
  qp = qwix_amd.quantize_params(params, abstract, {'dot_general0_lhs': stat})
  assert set(qp) == set(abstract)

  # the oracle's side of the same computation
  keys = ['absmax'] if method == 'absmax' else ['min', 'max']
  avg = {k: O.FArr((util.f32np(stat['sum_of_' + k]) / np.float32(3)).astype(np.float32), O.F32) for k in keys}
  oscale, ozp = O.compute_scale_zero_point(avg, 'int8')
  assert np.array_equal(util.f32np(qp['dot_general0_lhs_scale'].array), oscale.v)
  if method == 'minmax':
    assert np.array_equal(qp['dot_general0_lhs_zero_point'].cpu().numpy(), ozp)
  out = pm.apply(qp, x)
  oxq = O.quantize_with_scale_zero_point(util.farr(x), 'int8', oscale, ozp)
  owq = O.quantize(util.farr(params['kernel']), O.HowToQuantize(qtype='int8', channelwise_axes=[1]))
  util.assert_qarray_equal(qp['kernel'].array, owq, 'weight')
  want = O.dot_general(oxq, owq, DN)
  bias = util.f32np(params['bias']) if 'bias' in params else np.float32(0)
  assert np.allclose(util.f32np(out), want.v + bias, rtol=1e-6, atol=1e-6)
  # without statistics the scale comes from the first input itself
  first = pm.init(params, x)['dot_general0_lhs_scale'].array
  cal0 = {k: O.FArr(util.f32np(v.mean(dim=0, keepdim=True)), O.F32) for k, v in qarray.calibrate(x, how).items()}
  assert np.allclose(util.f32np(first), O.compute_scale_zero_point(cal0, 'int8')[0].v, rtol=1e-6)


def test_ptq_mlp_forward_replays_from_a_hip_graph():
  """The launch-bound configuration (four small kernels per forward) captured once and replayed: no entry
  point allocates or synchronises, so the whole quantized forward is graph-safe.  Every replay, with the
  program's own eager work and synchronisations in between, must reproduce the eager result bit for bit."""
  import qwix_amd
  model, params, x, rules = _mlp_setup()
  ptq_model = qwix_amd.quantize_model(model, qwix_amd.PtqProvider(rules))
  qparams = qwix_amd.quantize_params(params, ptq_model.init(params, x))
  static_x = x.clone()
  s = torch.cuda.Stream()
  s.wait_stream(torch.cuda.current_stream())
  with torch.cuda.stream(s):
    for _ in range(2):
      ptq_model.apply(qparams, static_x)      # warm-up on the side stream (lazy initialisations)
  torch.cuda.current_stream().wait_stream(s)
  graph = torch.cuda.CUDAGraph()
  with torch.cuda.graph(graph):
    static_out = ptq_model.apply(qparams, static_x)
  g = torch.Generator().manual_seed(5)
  for i in range(4):
    xi = torch.rand(x.shape, generator=g, dtype=torch.float32).to(util.DEV) * (i + 1)
    eager = ptq_model.apply(qparams, xi)       # eager work between the replays
    torch.cuda.synchronize()
    static_x.copy_(xi)
    graph.replay()
    torch.cuda.synchronize()
    assert torch.equal(static_out, eager), i


def test_decode_size_calls_fold_the_activation_quantization_into_the_gemm(monkeypatch):
  """Through the provider, a call with at most 32 tokens takes the fused kernel (one launch) and gives the bits
  of the two-step route; more tokens, static scales or sub-channel tiles keep the two-step route."""
  import qwix_amd
  from qwix_amd import nn
  from qwix_amd.core import dot_general as dg
  model = nn.MLP(2048, 512)
  g = torch.Generator().manual_seed(3)
  params = model.init(g, 1024, torch.bfloat16, util.DEV)
  rules = [qwix_amd.QuantizationRule(module_path='.*', weight_qtype='int8', act_qtype='int8')]
  ptq_model = qwix_amd.quantize_model(model, qwix_amd.PtqProvider(rules))
  x = torch.rand(8, 1024, generator=g, dtype=torch.float32).to(torch.bfloat16).to(util.DEV)
  qparams = qwix_amd.quantize_params(params, ptq_model.init(params, x))
  calls = []
  real = dg.fused_act_dot_general
  monkeypatch.setattr(dg, 'fused_act_dot_general', lambda *a, **k: (calls.append(1), real(*a, **k))[1])
  out = ptq_model.apply(qparams, x)
  assert len(calls) == 2
  monkeypatch.setattr(dg, 'fused_act_dot_general', lambda *a, **k: None)   # force the two-step route
  assert torch.equal(out, ptq_model.apply(qparams, x))
  monkeypatch.setattr(dg, 'fused_act_dot_general', lambda *a, **k: (calls.append(1), real(*a, **k))[1])
  big = torch.rand(64, 1024, generator=g, dtype=torch.float32).to(torch.bfloat16).to(util.DEV)
  fused = ptq_model.apply(qparams, big)
  assert len(calls) == 4                                                   # 64 tokens: the same entry point, two launches
  monkeypatch.setattr(dg, 'fused_act_dot_general', lambda *a, **k: None)
  assert torch.equal(fused, ptq_model.apply(qparams, big))


@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16])
@pytest.mark.parametrize('qtype', ['int8', 'float8_e4m3fn'])
@pytest.mark.parametrize('rows,hidden', [(1, 256), (20, 2048), (33, 2048), (32, 2176), (300, 4096), (65, 8320), (9, 16512)])
def test_relu_inside_the_quantization_of_the_next_layer(rows, hidden, qtype, dtype, monkeypatch):
  """The MLP's second layer takes max(h, 0) from h itself: against a ReLU of its own in front of the plain operation, bit for bit,
  with rows that are negative throughout and with the kernel that quantizes in the product (up to 32 rows, K up to 2048); rows of
  more than 32 KB keep the ReLU of their own."""
  import qwix_amd
  from qwix_amd import _lib, nn
  print('case relu', rows, hidden, qtype, dtype, flush=True)
  g = torch.Generator(device=util.DEV).manual_seed(rows + hidden)

  class Plain(nn.MLP):
    def __call__(self, params, x):
      return self.layers[1](params['Dense_1'], torch.relu(self.layers[0](params['Dense_0'], x)))
  rule = qwix_amd.QuantizationRule(module_path='.*', weight_qtype=qtype, act_qtype=qtype)
  params = {'Dense_0': {'kernel': torch.randn(128, hidden, generator=g, device=util.DEV).to(dtype)},
            'Dense_1': {'kernel': torch.randn(hidden, 136, generator=g, device=util.DEV).to(dtype)}}
  x = torch.randn(rows, 128, generator=g, device=util.DEV).to(dtype)
  models = [qwix_amd.quantize_model(m(hidden, 136), qwix_amd.PtqProvider([rule])) for m in (nn.MLP, Plain)]
  negative = {'Dense_0': {'kernel': -params['Dense_0']['kernel'].abs() - 1}, 'Dense_1': params['Dense_1']}
  params = qwix_amd.quantize_params(params, models[0].init(params, x))
  names, call = [], _lib.call
  monkeypatch.setattr(_lib, 'call', lambda *a: names.append(a[0]) or call(*a))
  for _ in range(6):  # the ordinary path, then its plan
    got, want = (m.apply(params, x) for m in models)
    assert got.dtype == dtype and torch.equal(got, want)
  assert ('qwix_hip_qgemm_dynamic_relu' in names) == (hidden * x.element_size() <= 32768)
  negative = qwix_amd.quantize_params(negative, models[0].init(negative, x))
  x = x.abs() + 1
  x[1::2] *= -1  # every second row of h positive throughout, the others negative
  got, want = (m.apply(negative, x) for m in models)
  assert torch.equal(got, want)
  assert torch.count_nonzero(got[::2]).item() == 0 and bool((got[1::2] != 0).any(-1).all())
  assert torch.equal(models[0].apply(params, torch.zeros_like(x)), models[1].apply(params, torch.zeros_like(x)))
  want = models[1].apply(params, x)
  # a provider with a dot_general of its own never sees the option
  class Own(qwix_amd.PtqProvider):
    def dot_general(self, lhs, rhs, dimension_numbers, precision=None, preferred_element_type=None, *, out_sharding=None):
      return super().dot_general(lhs, rhs, dimension_numbers, precision, preferred_element_type, out_sharding=out_sharding)
  assert torch.equal(qwix_amd.quantize_model(nn.MLP(hidden, 136), Own([rule])).apply(params, x), want)


@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16])
@pytest.mark.parametrize('qtype', ['int8', 'float8_e4m3fn'])
@pytest.mark.parametrize('rows,k', [(3, 256), (70, 1032)])
def test_relu_inside_the_quantization_keeps_nan(rows, k, qtype, dtype):
  """NaN of either sign, the smallest and the largest of each, and infinities pass max(x, 0) as torch.relu passes them: in the product
  (3 rows, int8) and in a launch of its own."""
  import qwix_amd
  from qwix_amd import nn
  print('case relu of NaN', rows, k, qtype, dtype, flush=True)
  g = torch.Generator(device=util.DEV).manual_seed(rows + k)

  class Layer:
    def __init__(self, inside):
      self.inside, self.dense = inside, nn.Dense(136)

    def __call__(self, params, x):
      return self.dense(params['Dense_0'], x, relu=True) if self.inside else self.dense(params['Dense_0'], torch.relu(x))
  rule = qwix_amd.QuantizationRule(module_path='.*', weight_qtype=qtype, act_qtype=qtype)
  x = torch.randn(rows, k, generator=g, device=util.DEV).to(dtype)
  bits = x.view(torch.int16 if dtype == torch.bfloat16 else torch.int32)
  inf = 0x7F80 if dtype == torch.bfloat16 else 0x7F800000
  low = -0x8000 if dtype == torch.bfloat16 else -0x80000000
  for i, v in enumerate((inf + 1, low + inf + 1, low + (-low - 1), -low - 1, low + inf, low)):
    bits[i % 2, 5 * i] = v  # NaN, -NaN (the smallest, the largest), NaN, -infinity, -0
  params = {'Dense_0': {'kernel': torch.randn(k, 136, generator=g, device=util.DEV).to(dtype)}}
  models = [qwix_amd.quantize_model(Layer(inside), qwix_amd.PtqProvider([rule])) for inside in (True, False)]
  params = qwix_amd.quantize_params(params, models[0].init(params, x))
  got, want = (m.apply(params, x) for m in models)
  assert torch.equal(got.nan_to_num(nan=12345.0), want.nan_to_num(nan=12345.0))
