"""Launch plans: what the recorder accepts (CPU), and that replayed calls give what the ordinary path gives (GPU)."""
import _thread
import ctypes
import dataclasses
import functools
import sys
import threading
import weakref

import pytest
import torch

from qwix_amd import _lib
from qwix_amd import plans
from tests import util

_DN = (((1,), (0,)), ((), ()))


# ---- the recorder, on host memory: addresses are addresses


def _recorded(fn, *operands):
  with plans.Recorder(operands) as rec:
    out = fn(rec)
  return rec, out


def _note(rec, q, x):
  rec.note('qwix_hip_ksum_i8', (q.data_ptr(), 64, 4, 64, x.data_ptr(), 7))


def test_recorder_tells_operands_buffers_and_constants_apart():
  q = torch.zeros(8, 64, dtype=torch.int8)

  def fn(rec):
    out = torch.empty(4, 2, dtype=torch.int32)
    _note(rec, q[4:], out)
    return out.t()
  rec, out = _recorded(fn, q)
  assert rec.ok and len(rec.buffers) == 1
  name, args = rec.calls[0]
  assert name == 'qwix_hip_ksum_i8'
  assert args == [(plans._OPERAND, 0, 256), (plans._CONST, 0, 64), (plans._CONST, 0, 4), (plans._CONST, 0, 64),
                  (plans._BUFFER, 0, 0), (plans._STREAM, 0, 0)]
  assert rec.results((out,)) == [(0, (2, 4), (1, 2), 0)]
  assert rec.results((torch.zeros(3),)) is None   # not a buffer of the call


@pytest.mark.parametrize('inference', [False, True])
@pytest.mark.parametrize('what', ['copy', 'reshape', 'conversion', 'fill', 'reduction', 'foreign pointer', 'overlapping operands', 'item'])
def test_recorder_refuses(what, inference):
  with torch.inference_mode(inference):
    _check_refused(what)


def _check_refused(what):
  q = torch.zeros(8, 64, dtype=torch.int8)
  kept = torch.zeros(64, 8, dtype=torch.int8)
  second = q[2:] if what == 'overlapping operands' else torch.zeros(1, dtype=torch.int8)

  def fn(rec):
    out = torch.empty(4, dtype=torch.int32)
    if what == 'copy':
      _note(rec, q.t().contiguous(), out)
    elif what == 'reshape':
      _note(rec, q.t().reshape(-1), out)
    elif what == 'conversion':
      _note(rec, q.to(torch.int32), out)
    elif what == 'foreign pointer':
      _note(rec, kept, out)
    else:
      _note(rec, q, out)
      if what == 'fill':
        out.zero_()
      elif what == 'reduction':
        out.sum()
      elif what == 'item':
        out[0].item()
    return out
  rec, _ = _recorded(fn, q, second)
  assert not rec.ok


@pytest.mark.parametrize('inference', [False, True])
def test_recorder_takes_views_by_their_effect(inference):
  """Operations that may copy and do not here; inference mode hands them to the recorder whole."""
  with torch.inference_mode(inference):
    q = torch.zeros(8, 64, dtype=torch.int8)

    def fn(rec):
      out = torch.empty(4, 2, dtype=torch.int32)
      _note(rec, q.contiguous().to(torch.int8).reshape(4, 128).unbind(0)[1].expand(2, 128).narrow(0, 0, 1).flatten(), out)
      return out.reshape(8).view(2, 4)
    rec, out = _recorded(fn, q)
    assert rec.ok and rec.calls[0][1][0] == (plans._OPERAND, 0, 128)
    assert rec.results((out,)) == [(0, (2, 4), (4, 1), 0)]


class _StandIn:
  """In place of the library: every entry point succeeds and writes nothing, no workspace is needed."""

  def __getattr__(self, name):
    return lambda *args: 0


@pytest.fixture
def stand_in(monkeypatch):
  from qwix_amd.core import dot_general as dg
  monkeypatch.setattr(_lib, 'load', _StandIn)
  monkeypatch.setattr(_lib, 'stream_of', lambda t: 0)
  yield
  for cache in (dg._splitk_bytes, dg._dynamic_act_bytes):   # answers of the stand-in
    cache.cache_clear()


def _host_weight(qtype, k, n, layout, zero_point=False):
  """A (k, n) weight in host memory, one scale per 128 rows and column."""
  from qwix_amd.core.qarray import Int4Tensor, QArray
  scale = torch.ones(k // 128, n, dtype=torch.bfloat16)
  if qtype == 'int4':
    data = torch.zeros(*((k, n // 2) if layout == 'natural' else (n, k // 2)), dtype=torch.uint8)
    q = Int4Tensor(data, (k, n), 1) if layout == 'natural' else Int4Tensor(data.t(), (k, n), 0)
  else:
    q = torch.zeros(*((k, n) if layout == 'natural' else (n, k)), dtype=torch.int8)
    q = q if layout == 'natural' else q.t()
  return QArray(q, scale, torch.zeros(k // 128, n, dtype=torch.int8) if zero_point else None, qtype)


def _parts(*operands):
  from qwix_amd.core.qarray import Int4Tensor, QArray
  out = []
  for x in operands:
    for t in ((x.qvalue, x.scale, x.zero_point) if isinstance(x, QArray) else (x,)):
      if t is not None:
        out.append(t.data if isinstance(t, Int4Tensor) else t)
  return out


@pytest.mark.parametrize('qtype', ['int8', 'int4'])
def test_recorder_refuses_what_is_prepared_once_per_weight(stand_in, qtype):
  """A weight in the natural layout is transposed at its first use and the copy is kept: a plan recorded at the first use of
  yet another layer's weight would transpose every layer's weight on every call."""
  from qwix_amd.core import dot_general as dg
  x = torch.zeros(3, 256, dtype=torch.bfloat16)
  for _ in range(4):
    w = _host_weight(qtype, 256, 64, 'natural')
    rec, _ = _recorded(lambda rec: dg._dot_general(x, w, _DN), *_parts(x, w))
    assert not rec.ok
  ready = _host_weight(qtype, 256, 64, 'reduce_minor')   # nothing to prepare
  rec, _ = _recorded(lambda rec: dg._dot_general(x, ready, _DN), *_parts(x, ready))
  assert rec.ok and [name for name, _ in rec.calls] == ['qwix_hip_gemv_wq']


def test_recorder_refuses_sums_kept_per_weight(stand_in):
  """The K-sums of a weight under an asymmetric activation are kept too."""
  from qwix_amd.core import dot_general as dg
  from qwix_amd.core.qarray import QArray
  w = QArray(torch.zeros(64, 256, dtype=torch.int8).t(), torch.ones(1, 64, dtype=torch.bfloat16), None, 'int8')
  recorded = []

  def fn(rec):
    def compute():
      out = torch.empty(64, dtype=torch.int32)
      _note(rec, w.qvalue, out)
      return out
    recorded.append(dg._weight_ksums(w.qvalue, w.qvalue, (), compute))
  rec, _ = _recorded(fn, *_parts(w))
  assert not rec.ok and len(rec.calls) == 1 and recorded[0] is not None


@pytest.mark.parametrize('M,K,N,act,weight,both,dtype,split', [
    (318, 3328, 1280, 'int8', 'int8', True, torch.bfloat16, True), (318, 3328, 1280, 'float8_e4m3fn', 'float8_e4m3fn', True, torch.bfloat16, True),
    (100, 4096, 264, 'int8', 'int8', True, torch.bfloat16, False),  # (few tiles: the wavefronts share K)
    (100, 4096, 264, 'int8', 'int8', True, torch.float32, False), (100, 4096, 264, 'int8', 'int4', True, torch.bfloat16, False),
    (100, 4096, 264, 'int8', 'int4', False, torch.float32, True), (100, 4096, 264, 'float8_e4m3fn', 'float8_e4m3fn', True, torch.bfloat16, False),
    (100, 4096, 264, 'float8_e4m3fn', 'float8_e4m3fn', True, torch.float32, False)])
def test_sub_channel_calls_that_are_not_split_get_no_workspace(stand_in, monkeypatch, M, K, N, act, weight, both, dtype, split):
  from qwix_amd.core import dot_general as dg
  from qwix_amd.core.qarray import Int4Tensor, QArray
  real = ctypes.CDLL(_lib.LIB_PATH)

  class Sizes(_StandIn):
    def __getattr__(self, name):
      if not name.endswith('_bytes'):
        return super().__getattr__(name)
      fn = getattr(real, name)
      fn.restype, fn.argtypes = _lib.SIGNATURES[name]
      return fn
  monkeypatch.setattr(_lib, 'load', Sizes)
  values = lambda t, *shape: torch.zeros(*shape, dtype=torch.int8 if t == 'int8' else torch.float8_e4m3fn)
  wv = Int4Tensor(torch.zeros(N, K // 2, dtype=torch.uint8).t(), (K, N), 0) if weight == 'int4' else values(weight, N, K).t()
  x = QArray(values(act, M, K), torch.ones(M, K // 128 if both else 1, dtype=dtype), None, act)
  w = QArray(wv, torch.ones(K // 128, N, dtype=dtype), None, weight)
  rec, _ = _recorded(lambda rec: dg._dot_general(x, w, _DN), *_parts(x, w))
  assert [name for name, _ in rec.calls] == ['qwix_hip_qgemm_grouped_ws']
  assert len(rec.buffers) == (2 if split else 1)


def test_more_rows_than_one_launch_takes_go_group_by_group(stand_in):
  """Weight-only experts in one launch end at 65535 * 16 rows; with enough groups even a few rows each come to more."""
  from qwix_amd.core import ragged_dot as rd
  from qwix_amd.core.qarray import QArray
  G = 21846
  w = QArray(torch.empty(G, 8, 128, dtype=torch.int8).permute(0, 2, 1), torch.empty(1, 1, 8, dtype=torch.bfloat16), None, 'int8')
  sizes = torch.zeros(G, dtype=torch.int32)
  for rows, taken in ((65535 * 16, True), (65535 * 16 + 1, False)):
    out = rd._weight_only_groups(torch.empty(rows, 128, dtype=torch.bfloat16), w, sizes, torch.bfloat16)
    assert (out is not None) == taken


# ---- the table


def _empty_the_table():
  for k in range(9000):   # more signatures than are remembered
    plans.native().run(('filler', k))


def test_a_plan_in_use_outlives_a_table_that_starts_anew():
  """`rebuild` is Python: what it runs, or another thread meanwhile, may fill the table until it is emptied."""
  n = plans.native()
  seen = []

  def fill(value):
    _empty_the_table()
    seen.append(alive() is not None)
    return value
  rebuild = functools.partial(fill, 'done')
  alive = weakref.ref(rebuild)
  from qwix_amd.core import qarray
  n.setup(qarray.QArray, qarray.Int4Tensor, lambda device: 0, _lib.raise_status, 1)
  try:
    assert n.run(('outlives',)) is None
    assert n.keep(('outlives',), (), [], [], [], rebuild)
    del rebuild   # the table's is the only reference
    assert n.run(('outlives',)) == 'done'
    assert seen == [True] and alive() is None   # let go after the call, not under it
    assert n.run(('outlives',)) is None
  finally:
    plans._native = None
    plans.native()


def test_a_replay_lets_other_threads_run():
  """Allocations can wait for the device and launches for room in its queue: a replay does both without the interpreter lock.
  With a switch interval longer than the test another thread runs only when the lock is let go."""
  from qwix_amd.core import qarray
  n = plans.native()
  n.setup(qarray.QArray, qarray.Int4Tensor, lambda device: 0, _lib.raise_status, 1)
  interval = sys.getswitchinterval()
  ran, alive = [], []   # (results stay: torch lets the lock go where a tensor dies)
  size = 1 << 20   # a mapping of its own, never touched: the allocation takes a while
  try:
    assert n.run(('unlocked',)) is None
    assert n.keep(('unlocked',), (), [((size,), (1,), torch.empty(1, dtype=torch.uint8))], [], [(0, (size,), (1,), 0)], None)
    sys.setswitchinterval(1000.0)
    _thread.start_new_thread(ran.append, (True,))   # (does not wait for the thread to run)
    while not ran and len(alive) < 5000:
      alive.append(n.run(('unlocked',)))
    assert ran
  finally:
    sys.setswitchinterval(interval)
    plans._native = None
    plans.native()


# ---- replay


def _rand(shape, seed, dtype=torch.bfloat16, std=1.0):
  g = torch.Generator(device='cpu').manual_seed(seed)
  return (torch.randn(shape, generator=g) * std).to(dtype).to(util.DEV)


def _same(a, b):
  from qwix_amd.core.qarray import Int4Tensor, QArray
  if isinstance(a, QArray):
    assert a.qtype == b.qtype and tuple(a.shape) == tuple(b.shape) and (a.zero_point is None) == (b.zero_point is None)
    values = lambda q: q.unpack() if isinstance(q, Int4Tensor) else q.view(torch.uint8) if q.dtype == torch.float8_e4m3fn else q
    assert type(a.qvalue) is type(b.qvalue) and torch.equal(values(a.qvalue), values(b.qvalue))
    assert torch.equal(a.scale, b.scale) and (a.zero_point is None or torch.equal(a.zero_point, b.zero_point))
  else:
    assert a.shape == b.shape and a.stride() == b.stride() and a.dtype == b.dtype and torch.equal(a, b)


def _cases():
  """name -> (operands of a seed, the operator, its ordinary path)"""
  import qwix_amd
  from qwix_amd.contrib import hadamard_rot as hr
  from qwix_amd.core import dot_general as dg, einsum as es, qarray as qa, ragged_dot as rd
  def weight(s, qtype, tile=None, method='absmax', k=512, n=200):
    return qwix_amd.quantize(_rand((k, n), s, std=0.05), qtype, channelwise_axes=[1], tiled_axes={0: tile} if tile else {},
                             calibration_method=method)
  act = lambda s, qtype: qwix_amd.quantize(_rand((24, 512), s), qtype, channelwise_axes=[0])
  how = lambda qtype, **kw: qwix_amd.HowToQuantize(qtype=qtype, **kw)
  dot = (lambda a, b: qwix_amd.dot_general(a, b, _DN), lambda a, b: dg._dot_general(a, b, _DN))
  cases = {}
  for q, method in (('int8', 'absmax'), ('int8', 'minmax'), ('int4', 'absmax'), ('float8_e4m3fn', 'absmax')):
    rows, cols = how(q, channelwise_axes=[0], calibration_method=method), how(q, channelwise_axes=[1], calibration_method=method)
    cases[f'rows {q} {method}'] = (lambda s: (_rand((24, 512), s),), lambda x, h=rows: qwix_amd.core.qarray.quantize(x, h),
                                   lambda x, h=rows: qa._quantize_any(x, h, None))
    cases[f'columns {q} {method}'] = (lambda s: (_rand((512, 72), s),), lambda x, h=cols: qwix_amd.core.qarray.quantize(x, h),
                                      lambda x, h=cols: qa._quantize_any(x, h, None))
    cases[f'dequantize {q} {method}'] = (lambda s, q=q, m=method: (weight(s, q, method=m),), qwix_amd.dequantize, qa._dequantize)
  for q in ('int8', 'float8_e4m3fn'):
    cases[f'dot {q}'] = (lambda s, q=q: (act(s, q), weight(s + 1, q)),) + dot
    cases[f'fused act {q}'] = (lambda s, q=q: (_rand((24, 512), s, torch.float32), weight(s + 1, q)),
                               lambda a, b, q=q: dg.fused_act_dot_general(a, b, _DN, act_qtype=q),
                               lambda a, b, q=q: dg._fused_act_dot_general(a, b, _DN, None, q))
  for tile in (128, 256):
    cases[f'dot int8 x int4 {tile}'] = (lambda s, t=tile: (act(s, 'int8'), weight(s + 1, 'int4', t)),) + dot
  for q, method in (('int4', 'absmax'), ('int4', 'minmax'), ('int8', 'minmax')):
    cases[f'weight only {q} {method}'] = (lambda s, q=q, m=method: (_rand((24, 512), s), weight(s + 1, q, 128, m)),) + dot
  cases['einsum'] = (lambda s: tuple(qwix_amd.quantize(_rand((3, 40, 64), s + i), 'int8', channelwise_axes=[0, 1]) for i in (0, 1)),
                     lambda a, b: qwix_amd.einsum('bqd,bkd->bqk', a, b),
                     lambda a, b: es._einsum(('bqd,bkd->bqk', a, b), dg.dot_general, None, {}))
  sizes = lambda s: torch.tensor([s % 5, 9, 0, 7], dtype=torch.int32, device=util.DEV)
  cases['ragged int8'] = (lambda s: (act(s, 'int8'), qwix_amd.quantize(_rand((4, 512, 72), s), 'int8', channelwise_axes=[0, 2]), sizes(s)),
                          qwix_amd.ragged_dot,
                          lambda *a: rd.ragged_dot_general(*a, rd._BASIC_RAGGED_DOT_DIMENSION_NUMBERS))
  for q in ('int4', 'int8'):   # group sizes of their own in every call, empty groups and rows left over among them
    experts = lambda s, q=q: qwix_amd.quantize(_rand((4, 512, 72), s + 1, std=0.05), q, channelwise_axes=[0, 2], tiled_axes={1: 128})
    cases[f'experts {q}'] = (lambda s, e=experts: (_rand((40, 512), s), e(s), torch.roll(sizes(s), s // 10)), qwix_amd.ragged_dot,
                             lambda *a: rd.ragged_dot_general(*a, rd._BASIC_RAGGED_DOT_DIMENSION_NUMBERS))
    # prompt sizes: the weight dequantized inside the product, its contraction cut into ranges, and dequantized in front of it
    for rows, k, n in ((200, 512, 8192), (100, 4096, 256), (1100, 512, 200) if q == 'int4' else (520, 512, 11008)):
      cases[f'weight only {q} {rows} rows'] = (
          lambda s, q=q, m=rows, k=k, n=n: (_rand((m, k), s), weight(s + 1, q, 128, k=k, n=n)),) + dot
  cases['hadamard'] = (lambda s: (_rand((24, 512), s), weight(s + 1, 'int4', 128)), hr.hadamard_quantized_matmul,
                       lambda a, b: hr._hadamard_quantized_matmul(a, b, None, None, None, None))
  return cases


_NAMES = (['%s %s %s' % (w, q, m) for w in ('rows', 'columns', 'dequantize')
           for q, m in (('int8', 'absmax'), ('int8', 'minmax'), ('int4', 'absmax'), ('float8_e4m3fn', 'absmax'))] +
          ['%s %s' % (w, q) for w in ('dot', 'fused act') for q in ('int8', 'float8_e4m3fn')] +
          ['dot int8 x int4 128', 'dot int8 x int4 256', 'weight only int4 absmax', 'weight only int4 minmax',
           'weight only int8 minmax', 'einsum', 'ragged int8', 'hadamard'])
_ENTRIES = {f'experts {q}': ['gemv_wq_groups'] for q in ('int4', 'int8')}   # what the ordinary path of a case runs
_ENTRIES.update({f'weight only {q} {rows} rows': ['gemm_bf16_wq_ws'] for q in ('int4', 'int8') for rows in (200, 100)})
_ENTRIES.update({f'weight only {q} rows': ['dequantize_rm', 'gemm_bf16'] for q in ('int4 1100', 'int8 520')})


@pytest.mark.gpu
@pytest.mark.parametrize('inference', [False, True])
@pytest.mark.parametrize('name', _NAMES + list(_ENTRIES))
def test_replay_equals_the_ordinary_path(name, inference):
  """New operands (other data, other addresses) on every call: the first ones go the ordinary way, the others replay."""
  _empty_the_table()   # (what the other mode recorded)
  make, op, ordinary = _cases()[name]
  alive = []
  for seed in range(plans.RECORD_AT + 2):
    operands = make(10 * seed)
    alive.append(operands)   # no address comes up twice
    with torch.inference_mode(inference):   # (the weights are older than a server's inference mode)
      _same(op(*operands), ordinary(*operands))
  calls = []
  call, _lib.call = _lib.call, lambda *a: calls.append(a[0]) or call(*a)
  try:
    with torch.inference_mode(inference):
      if name in _ENTRIES:
        ordinary(*alive[0])
        assert calls == ['qwix_hip_' + entry for entry in _ENTRIES[name]]
        calls.clear()
      _same(op(*alive[0]), op(*alive[0]))
    assert not calls, 'no plan is kept for this kind of call'
  finally:
    _lib.call = call


def _asymmetric(seed, k, n):
  import qwix_amd
  x = qwix_amd.quantize(_rand((40, k), seed) + 0.5, 'int8', channelwise_axes=[0], calibration_method='minmax')
  return x, qwix_amd.quantize(_rand((k, n), seed + 1), 'int8', channelwise_axes=[1])


@pytest.mark.gpu
def test_asymmetric_rows_replay_with_their_weight_s_sums():
  """Weights of one shape share a plan, each with its own K-sums as an operand; a weight that is written to gets new ones."""
  import qwix_amd
  from qwix_amd.core import dot_general as dg
  _empty_the_table()
  dn = (((1,), (0,)), ((), ()))
  pairs = [_asymmetric(10 * i, 256, 72) for i in range(3)]
  for _ in range(plans.RECORD_AT + 2):
    for x, w in pairs:
      _same(qwix_amd.dot_general(x, w, dn), dg._dot_general(x, w, dn))
  calls = []
  call, _lib.call = _lib.call, lambda *a: calls.append(a[0]) or call(*a)
  try:
    for x, w in pairs:
      qwix_amd.dot_general(x, w, dn)
    assert not calls, 'no plan is kept'
  finally:
    _lib.call = call
  x, w = pairs[0]
  w.qvalue.copy_(pairs[1][1].qvalue)
  _same(qwix_amd.dot_general(x, w, dn), dg._dot_general(x, qwix_amd.QArray(w.qvalue.clone(), w.scale, None, w.qtype), dn))


def _by_hand(x, w):
  """dot_general of one asymmetric and one symmetric array in 64 bits, rounded once (bf16 scales: exact products of integers)."""
  a = (x.qvalue.to(torch.float64) - x.zero_point.to(torch.float64)) * x.scale.to(torch.float64)
  return a @ (w.qvalue.to(torch.float64) * w.scale.to(torch.float64))


def _close(out, want):
  return bool(((out.to(torch.float64) - want).abs() <= 2.0 ** -6 * want.abs() + 2.0 ** -7 * want.abs().mean()).all())


@pytest.mark.gpu
@pytest.mark.parametrize('planned', [False, True])
@pytest.mark.parametrize('change', ['copy_', 'other memory', 'other order', 'forget_weight'])
def test_a_weight_s_sums_follow_its_changes(planned, change):
  """Zero points far from 0 multiply the sums: a result with another weight's sums is off by far more than the rounding of its
  bf16 steps."""
  import qwix_amd
  from qwix_amd.core import dot_general as dg
  _empty_the_table()
  x = qwix_amd.quantize(_rand((40, 256), 1) + 3, 'int8', channelwise_axes=[0], calibration_method='minmax')
  w = qwix_amd.quantize(_rand((256, 256), 2) + 1, 'int8', channelwise_axes=[1])
  for _ in range(plans.RECORD_AT + 2 if planned else 1):
    assert _close(qwix_amd.dot_general(x, w, _DN), _by_hand(x, w))
  other = (-w.qvalue).roll(5, 0) // 2
  if change == 'copy_':
    w.qvalue.copy_(other)
  elif change == 'other memory':
    w.qvalue.data = other.t().contiguous().t()
  elif change == 'other order':
    w.qvalue.data = w.qvalue.data.t()
  else:
    w.qvalue.data.copy_(other)
    dg.forget_weight(w)
  assert _close(qwix_amd.dot_general(x, w, _DN), _by_hand(x, w))


@pytest.mark.gpu
@pytest.mark.parametrize('planned', [False, True])
def test_a_weight_s_sums_are_awaited_on_another_stream(planned):
  """The first call's stream is still busy when a call on another one wants the sums that it will compute."""
  import qwix_amd
  _empty_the_table()
  x, w = _asymmetric(3, 256, 4096)
  if planned:
    for i in range(plans.RECORD_AT + 2):
      a, b = _asymmetric(30 + i, 256, 4096)
      for _ in range(2):
        qwix_amd.dot_general(a, b, _DN)
  want = _by_hand(x, w)
  first, second = torch.cuda.Stream(), torch.cuda.Stream()
  with torch.cuda.stream(first):   # what an allocation for the sums finds there
    torch.full((4096,), 1 << 20, dtype=torch.int32, device=util.DEV)
  torch.cuda.synchronize()
  with torch.cuda.stream(first):
    torch.cuda._sleep(200_000_000)
    qwix_amd.dot_general(x, w, _DN)
  with torch.cuda.stream(second):
    out = qwix_amd.dot_general(x, w, _DN)
  torch.cuda.synchronize()
  assert _close(out, want)


@pytest.mark.gpu
@pytest.mark.parametrize('inference', [False, True])
@pytest.mark.parametrize('qtype,layout', [('int8', 'natural'), ('int4', 'natural'), ('int8', 'reduce_minor'), ('int4', 'reduce_minor')])
def test_a_weight_s_kept_layout_follows_other_memory_and_streams(qtype, layout, inference):
  """What a weight-only call keeps of its weight (a transposed copy, a view) under 'tensor.data = other', and for a call on another
  stream while the one that makes the copy is busy."""
  import qwix_amd
  from qwix_amd.core import dot_general as dg
  make = lambda seed: qwix_amd.quantize(_rand((512, 200), seed, std=0.05), qtype, channelwise_axes=[1], tiled_axes={0: 128}, layout=layout)
  store = lambda w: w.qvalue.data if qtype == 'int4' else w.qvalue
  x, w, other = _rand((5, 512), 1), make(2), make(3)
  fresh = lambda w: dg._slow_dot_general(x, dataclasses.replace(w), _DN)   # an object of its own: nothing is kept for it yet
  with torch.inference_mode(inference):
    assert torch.equal(dg._dot_general(x, w, _DN), fresh(w))
  store(w).data = store(other).clone(memory_format=torch.preserve_format)
  w.scale.data = other.scale.clone()
  with torch.inference_mode(inference):
    assert torch.equal(dg._dot_general(x, w, _DN), fresh(other))
  late = make(4)
  want = fresh(late)
  first, second = torch.cuda.Stream(), torch.cuda.Stream()
  with torch.cuda.stream(first):
    torch.full((512, 200), 127, dtype=torch.int8, device=util.DEV)
  torch.cuda.synchronize()
  with torch.cuda.stream(first):
    torch.cuda._sleep(200_000_000)
    dg._dot_general(x, late, _DN)
  with torch.cuda.stream(second):
    out = dg._dot_general(x, late, _DN)
  torch.cuda.synchronize()
  assert torch.equal(out, want)


@pytest.mark.gpu
def test_a_weight_s_sums_and_a_captured_graph():
  """Sums that only the replay computes are no other call's: the first use of a weight is captured, the next one is not."""
  import qwix_amd
  _empty_the_table()
  x, w = _asymmetric(5, 256, 512)
  warm = _asymmetric(6, 256, 512)
  qwix_amd.dot_general(*warm, _DN)
  torch.cuda.synchronize()
  graph = torch.cuda.CUDAGraph()
  with torch.cuda.graph(graph):
    captured = qwix_amd.dot_general(x, w, _DN)
  assert _close(qwix_amd.dot_general(x, w, _DN), _by_hand(x, w))
  for _ in range(3):
    graph.replay()
    assert _close(captured, _by_hand(x, w))
    assert _close(qwix_amd.dot_general(*warm, _DN), _by_hand(*warm))


@pytest.mark.gpu
@pytest.mark.parametrize('scheme', [('int8', 'int8', None), ('float8_e4m3fn', 'float8_e4m3fn', 128), ('int4', None, 128)])
def test_a_provider_s_operation_is_one_plan(scheme):
  """The operations of a quantized model, activations of other shapes and data in between: replayed without the provider's own
  path, equal to it; static ranges and float kernels keep that path."""
  import qwix_amd
  from qwix_amd import nn
  _empty_the_table()
  weight, act, tile = scheme
  rule = qwix_amd.QuantizationRule(module_path='.*', weight_qtype=weight, act_qtype=act, tile_size=tile)
  provider = qwix_amd.PtqProvider([rule])
  mlp = qwix_amd.quantize_model(nn.MLP(512, 256), provider)
  params = {'Dense_0': {'kernel': _rand((256, 512), 1)}, 'Dense_1': {'kernel': _rand((512, 256), 2)}}

  def attend(params, q, k):
    return nn.ops.einsum('bqd,bkd->bqk', q, k)
  scores = qwix_amd.quantize_model(attend, provider)
  ordinary, calls = qwix_amd.PtqProvider._planned, []
  for i in range(plans.RECORD_AT + 3):
    for rows in (3, 40):
      x, q, k = _rand((rows, 256), 7 * i + rows), _rand((2, rows, 128), 5 * i + rows), _rand((2, 48, 128), 3 * i)
      got = [mlp.apply(params, x)] + ([scores.apply({}, q, k)] if act else [])
      qwix_amd.PtqProvider._planned = lambda self, op, arg, rule, lhs, rhs, fn: fn()
      try:
        want = [mlp.apply(params, x)] + ([scores.apply({}, q, k)] if act else [])
      finally:
        qwix_amd.PtqProvider._planned = ordinary
      for a, b in zip(got, want):
        _same(a, b)
  call, _lib.call = _lib.call, lambda *a: calls.append(a[0]) or call(*a)
  try:
    mlp.apply(params, x)
    if act:
      scores.apply({}, q, k)
  finally:
    _lib.call = call
  assert not calls, 'no plan is kept for an operation of the model'


@pytest.mark.gpu
@pytest.mark.parametrize('first', ['stock', 'subclass', 'instance'])
@pytest.mark.parametrize('op', ['einsum', 'dot_general'])
def test_a_provider_s_own_policy_is_not_replaced_by_a_plan(op, first):
  """Providers that quantize to another type than their rule says beside the stock one, on equal shapes, whichever comes first: each
  gets its own results on every call."""
  import qwix_amd
  from qwix_amd import nn
  _empty_the_table()

  def another(prepare):
    return lambda lhs, rhs, rule, *rest, **kw: prepare(lhs, rhs, dataclasses.replace(rule, act_qtype='float8_e4m3fn'), *rest, **kw)

  class Other(qwix_amd.PtqProvider):
    def _prepare(self, *args, **kw):
      return another(super()._prepare)(*args, **kw)

    def _fusable(self, rule):
      return None

  def run(provider, a, b):
    fn = ((lambda params, q, k: nn.ops.einsum('bqd,bkd->bqk', q, k)) if op == 'einsum' else
          (lambda params, q, k: nn.ops.dot_general(q[0], k[0], (((1,), (1,)), ((), ())))))
    return qwix_amd.quantize_model(fn, provider).apply({}, a, b)
  rule = qwix_amd.QuantizationRule(module_path='.*', weight_qtype='int8', act_qtype='int8')
  providers = {'stock': qwix_amd.PtqProvider([rule]), 'subclass': Other([rule]), 'instance': qwix_amd.PtqProvider([rule])}
  own = providers['instance']
  own._prepare, own._fusable = another(own._prepare), lambda rule: None
  # the same arithmetic under another identity of the module: no plan of a whole operation is kept for it
  plain = {name: qwix_amd.PtqProvider([dataclasses.replace(rule, act_qtype='int8' if name == 'stock' else 'float8_e4m3fn')],
                                      _qarray_module=_OrdinaryModule()) for name in providers}
  order = [first] + [name for name in providers if name != first]
  for i in range(plans.RECORD_AT + 3):   # in turn
    a, b = _rand((2, 24, 128), 3 * i), _rand((2, 40, 128), 3 * i + 1)
    for name in order:
      assert torch.equal(run(providers[name], a, b), run(plain[name], a, b)), (name, i)
  for name in order:   # ... and one after the other
    for i in range(plans.RECORD_AT + 1):
      a, b = _rand((2, 56, 128), 3 * i), _rand((2, 72, 128), 3 * i + 1)
      assert torch.equal(run(providers[name], a, b), run(plain[name], a, b)), (name, i)


class _OrdinaryModule:

  def __getattr__(self, name):
    from qwix_amd.core import qarray
    return getattr(qarray, name)


@pytest.mark.gpu
@pytest.mark.parametrize('qtype', ['int8', 'int4'])
def test_layers_of_one_shape_are_laid_out_once_each(monkeypatch, qtype):
  """More weights of one shape than calls up to the recorded one, in the natural layout: each is transposed at its first use
  and never again."""
  import qwix_amd
  from qwix_amd.core import dot_general as dg
  ws = [qwix_amd.quantize(_rand((512, 200), s, std=0.05), qtype, channelwise_axes=[1], tiled_axes={0: 128}, layout='natural')
        for s in range(plans.RECORD_AT + 2)]
  names, call = [], _lib.call
  monkeypatch.setattr(_lib, 'call', lambda *a: names.append(a[0]) or call(*a))
  for turn in range(4):
    names.clear()
    x = _rand((5, 512), turn)
    outs = [qwix_amd.dot_general(x, w, _DN) for w in ws]
    assert names.count('qwix_hip_transpose_q') == (len(ws) if turn == 0 else 0), names
    assert names.count('qwix_hip_gemv_wq') == len(ws)   # (a replayed plan is not seen here)
    for out, w in zip(outs, ws):
      _same(out, dg._dot_general(x, w, _DN))


@pytest.mark.gpu
def test_replay_with_other_layouts_options_and_errors():
  import qwix_amd
  w = qwix_amd.quantize(_rand((512, 200), 1, std=0.05), 'int8', channelwise_axes=[1])
  big = _rand((40, 1100), 2)
  for _ in range(plans.RECORD_AT + 2):
    for x in (big[:24, :512], big[3:27, 8:520], big[3:27, 3:515], big[:24, :512].contiguous()):   # pitches and alignments
      got = qwix_amd.quantize(x, 'int8', channelwise_axes=[0])
      want = qwix_amd.core.qarray._quantize_any(x.contiguous(), qwix_amd.HowToQuantize(qtype='int8', channelwise_axes=[0]), None)
      _same(got, want)
      out = qwix_amd.dot_general(got, w, _DN)
      assert out.dtype == torch.bfloat16
      assert qwix_amd.dot_general(got, w, _DN, preferred_element_type=torch.float32).dtype == torch.float32
  with pytest.raises(ValueError, match='differ'):
    qwix_amd.dot_general(got, qwix_amd.quantize(_rand((256, 200), 1), 'int8', channelwise_axes=[1]), _DN)
  # one array on both sides: its memory belongs to both operands
  a = qwix_amd.quantize(_rand((64, 64), 5), 'int8', channelwise_axes=[0])
  dn = (((1,), (1,)), ((), ()))
  for _ in range(plans.RECORD_AT + 2):
    _same(qwix_amd.dot_general(a, a, dn), qwix_amd.core.dot_general._dot_general(a, a, dn))


@pytest.mark.gpu
@pytest.mark.parametrize('first,second', [(1, 1.0), (1.0, 1)])
def test_a_tile_of_one_element_is_not_the_whole_axis(first, second):
  """1 == 1.0, but an integer is a size and a float a share of the axis: each has plans of its own."""
  import qwix_amd
  x = _rand((64, 72 if isinstance(first, float) else 80), 3)
  for tile in (first, second):
    how = qwix_amd.HowToQuantize(qtype='int8', channelwise_axes=[1], tiled_axes={0: tile})
    want = qwix_amd.core.qarray._quantize_any(x, how, None)
    for _ in range(plans.RECORD_AT + 2):
      _same(qwix_amd.quantize(x, 'int8', channelwise_axes=[1], tiled_axes={0: tile}), want)
      _same(qwix_amd.core.qarray.quantize(x, how), want)


@pytest.mark.gpu
def test_replay_on_threads_and_streams():
  import qwix_amd
  w = qwix_amd.quantize(_rand((512, 200), 1, std=0.05), 'int8', channelwise_axes=[1])
  xs = [_rand((24, 512), 20 + i) for i in range(4)]
  step = lambda x: qwix_amd.dot_general(qwix_amd.quantize(x, 'int8', channelwise_axes=[0]), w, _DN)
  want = [step(x) for x in xs]
  torch.cuda.synchronize()
  bad = []

  def work(i):
    with torch.cuda.stream(torch.cuda.Stream()):
      for _ in range(50):
        out = step(xs[i])
        torch.cuda.current_stream().synchronize()
        if not torch.equal(out, want[i]):
          bad.append(i)
          return
  threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
  for t in threads:
    t.start()
  for t in threads:
    t.join()
  assert not bad


@pytest.mark.gpu
def test_replay_inside_a_captured_graph():
  """Captured calls are replayed plans; every replay of the graph against the eager result."""
  import qwix_amd
  w = qwix_amd.quantize(_rand((512, 200), 1, std=0.05), 'int8', channelwise_axes=[1])
  x = _rand((24, 512), 30)
  step = lambda: qwix_amd.dot_general(qwix_amd.quantize(x, 'int8', channelwise_axes=[0]), w, _DN)
  side = torch.cuda.Stream()
  side.wait_stream(torch.cuda.current_stream())
  with torch.cuda.stream(side):
    for _ in range(plans.RECORD_AT + 1):
      step()
  torch.cuda.current_stream().wait_stream(side)
  graph = torch.cuda.CUDAGraph()
  with torch.cuda.graph(graph):
    out = step()
  for seed in range(31, 35):
    x.copy_(_rand((24, 512), seed))
    graph.replay()
    torch.cuda.synchronize()
    assert torch.equal(out, step())
