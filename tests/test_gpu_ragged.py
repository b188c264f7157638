"""GPU parity: ragged (mixture-of-experts) quantized GEMM through qwix_amd.ragged_dot vs the CPU oracle.

int8 x int8: the int32 sums are exact and the epilogue is elementwise, so outputs are compared bit for
bit.  e4m3 x e4m3: the matrix instruction's internal accumulation differs from the oracle's single
rounding of an exact sum (up to 1e-4 of the largest output), so outputs are compared at rtol 1e-2 for
bf16 results and 1e-3 for f32 results, the tolerances of the dense fp8 GEMM tests."""
import types

import numpy as np
import pytest
import torch

from oracle import qwix_oracle as O
from tests import util

pytestmark = pytest.mark.gpu


def _how(qtype, channelwise, tiled=None):
  from qwix_amd.core import qarray
  return (qarray.HowToQuantize(qtype=qtype, channelwise_axes=list(channelwise), tiled_axes=dict(tiled or {})),
          O.HowToQuantize(qtype=qtype, channelwise_axes=list(channelwise), tiled_axes=dict(tiled or {})))


def _quantized(shape, dtype, seed, how, scale=1.0):
  from qwix_amd.core import qarray
  x_np, x_t = util.make(shape, dtype, seed=seed, scale=scale)
  q = qarray.quantize(x_t, how[0])
  oq = O.quantize(O.FArr(x_np, dtype), how[1])
  util.assert_qarray_equal(q, oq, 'operand')
  return q, oq


def _sizes(t):
  return torch.tensor(t, dtype=torch.int32, device=util.DEV)


def _check_exact(out, want):
  got = util.f32np(out)
  assert tuple(got.shape) == tuple(want.v.shape)
  bad = np.flatnonzero(got.ravel() != want.v.ravel())
  assert bad.size == 0, f'{bad.size} outputs differ: {got.ravel()[bad[:5]]} vs {want.v.ravel()[bad[:5]]}'


INT8_CASES = [
    # name, (M, K, G, N), group sizes, lhs channelwise, rhs channelwise, rhs tiled
    ('per-tensor', (128, 256, 4, 64), (64, 32, 16, 16), (), (), None),
    ('channelwise', (128, 256, 4, 64), (128, 100, 0, 28), (0,), (2,), None),
    ('group+channel', (128, 256, 4, 64), (50, 50, 28, 0), (0,), (0, 2), None),
    ('group only', (128, 256, 4, 64), (128, 0, 0, 0), (), (0,), None),
    ('short of M', (300, 384, 5, 200), (10, 0, 130, 1, 70), (0,), (0, 2), None),
    ('tile edges', (700, 128, 3, 260), (128, 129, 256), (0,), (0, 2), None),
    ('K not a multiple of 128', (200, 80, 3, 72), (60, 0, 100), (0,), (0, 2), None),
    ('many groups', (1000, 256, 64, 136), tuple((i * 7) % 31 for i in range(64)), (0,), (0, 2), None),
    ('k tiled', (128, 256, 4, 512), (10, 20, 30, 68), (0,), (0, 2), {1: 128}),
    ('k tiled, shared over groups', (128, 256, 4, 512), (10, 20, 30, 68), (0,), (2,), {1: 128}),
    ('k and n tiled', (128, 256, 4, 512), (10, 20, 30, 68), (0,), (0,), {1: 128, 2: 128}),
    ('decode: a few rows per group (weight-streaming kernel), empty groups, rows of no group', (40, 256, 12, 200),
     (0, 3, 16, 1, 0, 7, 2, 0, 5, 2, 1, 1), (0,), (0, 2), None),
    ('decode: one group takes several 16-row passes', (60, 384, 6, 72), (0, 40, 1, 0, 9, 3), (0,), (0, 2), None),
    ('decode: one row per group, shared weight scale', (16, 128, 16, 48), (1,) * 16, (0,), (2,), None),
    ('a few dozen rows per group (64-row tiles, deep weight prefetch), some groups empty or taller than a tile',
     (1700, 1024, 40, 520), tuple((i * 37) % 60 if i % 9 else (0 if i % 2 else 130) for i in range(40)), (0,), (0, 2), None),
    ('big groups', (2100, 512, 2, 2304), (1100, 900), (0,), (0, 2), None),
    ('big groups on a full chip (256-row tiles, ping-pong schedule)', (4096, 384, 4, 3072), (1000, 1100, 900, 1000), (0,), (0, 2), None),
]


@pytest.mark.parametrize('dtype', [O.BF16, O.F32])
@pytest.mark.parametrize('name,shape,sizes,lcw,rcw,rtiled', INT8_CASES)
def test_ragged_dot_int8_bit_exact(name, shape, sizes, lcw, rcw, rtiled, dtype):
  import qwix_amd
  print('case ragged int8', name, shape, sizes, dtype, flush=True)
  M, K, G, N = shape
  xq, oxq = _quantized((M, K), dtype, 100 + M, _how('int8', lcw))
  wq, owq = _quantized((G, K, N), dtype, 200 + N, _how('int8', rcw, rtiled), scale=0.05)
  out = qwix_amd.ragged_dot(xq, wq, _sizes(sizes))
  torch.cuda.synchronize()
  _check_exact(out, O.ragged_dot(oxq, owq, sizes))


def test_ragged_dot_both_sides_k_tiled():
  import qwix_amd
  xq, oxq = _quantized((128, 256), O.BF16, 7, _how('int8', (0,), {1: 128}))
  wq, owq = _quantized((4, 256, 512), O.BF16, 8, _how('int8', (0, 2), {1: 128}), scale=0.05)
  out = qwix_amd.ragged_dot(xq, wq, _sizes((10, 20, 30, 68)))
  _check_exact(out, O.ragged_dot(oxq, owq, (10, 20, 30, 68)))
  bad, _ = _quantized((128, 256), O.BF16, 7, _how('int8', (0,), {1: 64}))
  with pytest.raises(ValueError, match='same tile size'):
    qwix_amd.ragged_dot(bad, wq, _sizes((10, 20, 30, 68)))


def test_ragged_dot_weights_stored_k_contiguous():
  """A weight kept as (G, N, K) storage and handed over as its (G, K, N) view is used in place."""
  import qwix_amd
  from qwix_amd.core.qarray import QArray
  xq, oxq = _quantized((256, 256), O.BF16, 17, _how('int8', (0,)))
  wq, owq = _quantized((3, 256, 192), O.BF16, 18, _how('int8', (0, 2)), scale=0.05)
  stored = wq.qvalue.permute(0, 2, 1).contiguous()
  view = QArray(stored.permute(0, 2, 1), wq.scale, None, wq.qtype)
  out = qwix_amd.ragged_dot(xq, view, _sizes((100, 56, 100)))
  _check_exact(out, O.ragged_dot(oxq, owq, (100, 56, 100)))


def test_ragged_dot_raw_int8_gives_int32():
  import qwix_amd
  rng = util.rng(3)
  a = rng.integers(-128, 128, (260, 128)).astype(np.int8)
  b = rng.integers(-128, 128, (3, 128, 136)).astype(np.int8)
  sizes = (130, 0, 100)
  out = qwix_amd.ragged_dot(torch.from_numpy(a).to(util.DEV), torch.from_numpy(b).to(util.DEV), _sizes(sizes))
  assert out.dtype == torch.int32
  assert np.array_equal(out.cpu().numpy(), O.ragged_dot(a, b, sizes))


def test_ragged_dot_out_of_range_sizes_are_clamped():
  """Negative sizes count as empty groups and a group that would pass the last row is cut off there
  (the kernel takes group_sizes from device memory and must stay inside the operands whatever it holds)."""
  import qwix_amd
  xq, oxq = _quantized((200, 128), O.BF16, 27, _how('int8', (0,)))
  wq, owq = _quantized((4, 128, 64), O.BF16, 28, _how('int8', (0, 2)), scale=0.05)
  out = qwix_amd.ragged_dot(xq, wq, _sizes((50, -3, 400, 10)))
  _check_exact(out, O.ragged_dot(oxq, owq, (50, 0, 150, 0)))


@pytest.mark.parametrize('dtype', [O.BF16, O.F32])
@pytest.mark.parametrize('shape,sizes,rcw', [((128, 256, 4, 64), (128, 100, 0, 28), (2,)),
                                             ((520, 512, 6, 384), (100, 3, 0, 257, 60, 50), (0, 2)),
                                             ((4096, 256, 4, 3072), (1000, 1100, 900, 1000), (0, 2)),
                                             ((48, 256, 8, 200), (5, 0, 9, 1, 20, 3, 2, 4), (0, 2))])   # decode sizes
def test_ragged_dot_fp8(shape, sizes, rcw, dtype):
  import qwix_amd
  M, K, G, N = shape
  xq, oxq = _quantized((M, K), dtype, 300 + M, _how(O.E4M3, (0,)))
  wq, owq = _quantized((G, K, N), dtype, 400 + N, _how(O.E4M3, rcw), scale=0.05)
  out = qwix_amd.ragged_dot(xq, wq, _sizes(sizes))
  want = O.ragged_dot(oxq, owq, sizes).v
  got = util.f32np(out)
  tol = 1e-2 if dtype == O.BF16 else 1e-3
  np.testing.assert_allclose(got, want, rtol=tol, atol=tol * np.abs(want).max())
  assert np.all(got[min(sum(sizes), M):] == 0)


@pytest.mark.parametrize('dtype', [O.BF16, O.F32])
@pytest.mark.parametrize('shape,sizes,rtiled', [((200, 256, 4, 136), (50, 0, 130, 20), None),
                                                ((300, 512, 3, 264), (100, 100, 60), {1: 128}),
                                                ((64, 1024, 6, 128), (1, 0, 30, 3, 0, 9), {1: 256})])
def test_ragged_dot_int4_expert_weights(shape, sizes, rtiled, dtype):
  """int8 activations x int4 expert weights (per channel and sub-channel along K): the sub-channel MFMA GEMM of
  dot_general, group by group.  Its f32 sum of the scaled partials is ordered differently from the oracle's, so
  the comparison is the one of the dense sub-channel tests (rtol 1e-2 for bf16 results, 1e-3 for f32)."""
  import qwix_amd
  M, K, G, N = shape
  xq, oxq = _quantized((M, K), dtype, 61, _how('int8', (0,)))
  wq, owq = _quantized((G, K, N), dtype, 62, _how('int4', (0, 2), rtiled), scale=0.05)
  out = qwix_amd.ragged_dot(xq, wq, _sizes(sizes))
  torch.cuda.synchronize()
  want = O.ragged_dot(oxq, owq, sizes).v
  got = util.f32np(out)
  assert out.dtype == util.TORCH_DT[dtype] and tuple(got.shape) == (M, N)
  # The reference rounds every K tile's scaled partial to the result dtype before summing them; the default
  # kernel keeps them in f32 (as for dot_general): with bf16 results that is up to half a bf16 step of the
  # largest partial per tile, on top of the 1e-2 bar.
  tol = 1e-2 if dtype == O.BF16 else 1e-3
  ntiles = K // (rtiled or {1: K})[1]
  atol = tol * np.abs(want).mean() + (ntiles * 2.0 ** -8 * np.abs(want).max() if dtype == O.BF16 else 0.0)
  np.testing.assert_allclose(got, want, rtol=tol, atol=atol)
  assert np.all(got[min(sum(sizes), M):] == 0)


@pytest.mark.parametrize('wq_type,tiled', [('int4', {1: 128}), ('int8', None), ('float8_e4m3fn', None)])
@pytest.mark.parametrize('sizes', [(3, 0, 20, 1), (300, 40, 0, 172)])
def test_ragged_dot_weight_only_experts(sizes, wq_type, tiled):
  """bf16 activations x quantized expert weights (the dequantize-first path, ragged_dot.py:229-241), group by group
  on this library's weight-only kernels: a few rows per expert (fused dequantize + bf16 MFMA) and hundreds
  (dequantize, then the bf16 MFMA GEMM)."""
  import qwix_amd
  M, K, G, N = 512, 512, 4, 192
  x_np, x_t = util.make((M, K), O.BF16, seed=71)
  wq, owq = _quantized((G, K, N), O.BF16, 72, _how(wq_type, (0, 2), tiled), scale=0.05)
  out = qwix_amd.ragged_dot(x_t, wq, _sizes(sizes))
  torch.cuda.synchronize()
  want = O.ragged_dot(O.FArr(x_np, O.BF16), owq, sizes).v
  got = util.f32np(out)
  assert out.dtype == torch.bfloat16
  np.testing.assert_allclose(got, want, rtol=1e-2, atol=1e-2 * np.abs(want).max())   # as for the fp8 experts above
  assert np.all(got[min(sum(sizes), M):] == 0)


@pytest.mark.parametrize('G,K,N,M,sizes', [
    (4, 128, 200, 40, (0, 17, 16, 1)),           # few workgroups (8 wavefronts), one K block, rows left over
    (4, 384, 72, 100, (33, 0, 70, 50)),          # two row tiles, an odd number of K blocks, sizes past the last row
    (8, 256, 2568, 60, (1, 15, 0, 16, 3, 17, 2, 0)),   # 4 wavefronts x 32 columns, a column tile that ends early
    (64, 256, 1000, 128, tuple(i % 4 for i in range(64))),        # several rounds: int4 4 wavefronts x 64 columns, bytes x 32
    (64, 384, 1000, 1100, tuple((7 * i) % 35 for i in range(64))),  # int4: 2 wavefronts x 64 columns; bytes: 4, two row tiles; several passes
    (4, 256, 1480, 80, (40, 0, 23, 17)),               # two row tiles on eight wavefronts, 32 columns
    (16, 256, 4400, 740, tuple((37 * i) % 93 for i in range(16))),   # bytes: 2 wavefronts, two row tiles
    (8, 640, 1032, 120, (40, 0, 33, 16, 1, 17, 2, 3)),             # two row tiles, 64 columns on eight wavefronts
    (32, 640, 1032, 12, (3, 0, 1) + (0,) * 20 + (5, 2) + (0,) * 7),   # most groups empty
    (64, 384, 1000, 420, tuple((5 * i) % 18 for i in range(64))),  # bytes: 4 wavefronts x 64 columns, second passes of one row
    (64, 384, 2000, 800, tuple((11 * i) % 26 for i in range(64))),  # int4: 2 wavefronts, one row tile, second passes of up to 9 rows
    (64, 384, 1000, 770, tuple((11 * i) % 25 for i in range(64))),
])
@pytest.mark.parametrize('wq_type,tiled,dtype', [('int4', {1: 128}, O.BF16), ('int8', {1: 128}, O.BF16), ('int8', None, O.F32),
                                                 ('float8_e4m3fn', {1: 128}, O.BF16), ('int4', None, O.F32)])
def test_ragged_dot_weight_only_one_launch(G, K, N, M, sizes, wq_type, tiled, dtype):
  """A few rows per group against weight-only experts in one launch, at the edges of its row tiles, column tiles and K
  blocks.  The kernel keeps weight x scale in f32, so a bf16 result is off by its own rounding (half a step, 2^-8 of the
  magnitude between powers of two) plus the f32 sums (below 1e-5 of the largest)."""
  import qwix_amd
  x_np, x_t = util.make((M, K), O.BF16, seed=81)
  wq, owq = _quantized((G, K, N), dtype, 82, _how(wq_type, (0, 2), tiled), scale=0.05)
  assert qwix_amd.core.ragged_dot._weight_only_groups(x_t, wq, _sizes(sizes), torch.float32) is not None
  out = qwix_amd.ragged_dot(x_t, wq, _sizes(sizes), preferred_element_type=torch.float32)
  q = O.qvalue_as_f32(owq).astype(np.float64) * np.repeat(owq.scale.v.astype(np.float64), K // owq.scale.v.shape[1], axis=1)
  want, start = np.zeros((M, N)), 0
  for g, size in enumerate(sizes):
    stop = min(start + size, M)
    want[start:stop] = x_np[start:stop].astype(np.float64) @ q[g]
    start = stop
  np.testing.assert_allclose(util.f32np(out), want, rtol=0, atol=1e-5 * np.abs(want).max())
  low = qwix_amd.ragged_dot(x_t, wq, _sizes(sizes), preferred_element_type=torch.bfloat16)
  np.testing.assert_allclose(util.f32np(low), want, rtol=2.0 ** -8, atol=2e-5 * np.abs(want).max())
  assert np.all(util.f32np(out)[min(sum(sizes), M):] == 0)


def _grouped_reference(x, wq, sizes):
  """Rows of x against the dequantized weight of their own group, in 64 bits."""
  q = (wq.qvalue.unpack() if wq.qtype == 'int4' else wq.qvalue).to(torch.float64)
  w = q * wq.scale.to(torch.float64).repeat_interleave(q.shape[1] // wq.scale.shape[1], 1)
  want, start = torch.zeros(x.shape[0], w.shape[2], dtype=torch.float64, device=x.device), 0
  for g, size in enumerate(sizes):
    stop = min(start + max(size, 0), x.shape[0])
    if stop > start:
      want[start:stop] = x[start:stop].to(torch.float64) @ w[g]
    start = stop
  return want


@pytest.mark.parametrize('G,N,M', [(64, 520, 1400), (16, 4232, 960)])
def test_ragged_dot_weight_only_second_row_tile_over_a_long_contraction(G, N, M):
  """int4 weights take two row tiles only where K is long: four wavefronts, and two where there are thousands of workgroups (tolerance:
  f32 sums of a few thousand products)."""
  import qwix_amd
  gen = torch.Generator().manual_seed(G)
  sizes = torch.bincount(torch.multinomial(torch.rand(G, generator=gen) + 0.2, M, replacement=True, generator=gen), minlength=G).tolist()
  print('case long contraction', G, N, M, flush=True)
  _, x = util.make((M, 2048), O.BF16, seed=95)
  g = torch.Generator(device=util.DEV).manual_seed(N)
  wq = qwix_amd.quantize(torch.randn(G, 2048, N, generator=g, device=util.DEV).to(torch.bfloat16), 'int4', channelwise_axes=[0, 2], tiled_axes={1: 128})
  out = qwix_amd.core.ragged_dot._weight_only_groups(x, wq, _sizes(sizes), torch.float32)
  want = _grouped_reference(x, wq, sizes)
  assert float((out.to(torch.float64) - want).abs().max()) <= 1e-5 * float(want.abs().max())


@pytest.mark.parametrize('G,N,M,sizes', [
    (8, 200, 384, (1, 0, 370, 0, 0, 3, 0, 10)),                   # one group with nearly all rows, two row tiles
    (64, 72, 600, (0,) * 63 + (600,)),                            # all rows in the last group of a wavefront, one row tile
    (130, 72, 700, tuple(417 if g == 100 else 2 * (g % 2) for g in range(130))),     # groups past the first 64, rows left over
    (300, 72, 900, tuple(500 if g == 290 else -1 if g % 5 == 0 else 1 for g in range(300))),   # found in two steps; negative sizes
    (300, 72, 3500, tuple(2 ** 31 - 1 if g in (200, 250) else 16 + g % 2 for g in range(300))),   # sizes that reach past all rows
])
@pytest.mark.parametrize('wq_type', ['int4', 'int8'])
def test_ragged_dot_weight_only_skewed(G, N, M, sizes, wq_type):
  """Row tiles spread over workgroups wherever the rows lie (tolerance: f32 sums, as in the test above)."""
  import qwix_amd
  _, x = util.make((M, 256), O.BF16, seed=91)
  _, w = util.make((G, 256, N), O.BF16, seed=92, scale=0.05)
  wq = qwix_amd.quantize(w, wq_type, channelwise_axes=[0, 2], tiled_axes={1: 128})
  assert qwix_amd.core.ragged_dot._weight_only_groups(x, wq, _sizes(sizes), torch.float32) is not None
  out = qwix_amd.ragged_dot(x, wq, _sizes(sizes), preferred_element_type=torch.float32)
  want = _grouped_reference(x, wq, sizes)
  assert float((out.to(torch.float64) - want).abs().max()) <= 1e-5 * float(want.abs().max())
  assert not out[max(0, min(sum(max(s, 0) for s in sizes), M)):].any()


@pytest.mark.parametrize('G,K,N,M,sizes', [
    (3, 256, 136, 400, (129, 0, 257)),                  # one and two 128-row tiles and a row, rows left over, four slabs
    (4, 384, 72, 700, (128, 1, 500, 300)),              # six slabs; sizes past the last row
    (2, 640, 264, 600, (256, 300)),                     # ten slabs, 64-column tiles of 256 rows
    (2, 1152, 18440, 514, (257, 257)),                  # 128-column tiles of 256 rows
    (70, 384, 72, 5000, tuple(-3 if g == 5 else 2 ** 31 - 1 if g == 69 else 70 + g % 3 for g in range(70))),  # past 64 groups
    (300, 256, 72, 20000, tuple(-1 if g == 7 else 0 if g % 50 == 3 else 2 ** 31 - 1 if g == 297 else 60 + g % 140 if g % 3 else 17
                                for g in range(300))),   # past 256 groups, the last one cut at the last row
])
@pytest.mark.parametrize('wq_type,tiled,dtype', [('int4', {1: 128}, O.BF16), ('int8', {1: 128}, O.BF16), ('int8', None, O.F32),
                                                 ('float8_e4m3fn', {1: 128}, O.F32), ('int4', None, O.F32)])
@pytest.mark.parametrize('most', [None, 0, 70, 130])
def test_ragged_dot_weight_only_tiles(G, K, N, M, sizes, wq_type, tiled, dtype, most, monkeypatch):
  """Too many rows to stream the weights of all groups: those of up to `streamed_rows` rows (and of `most`, also none) are streamed,
  their weights unrounded; tiles of 128 and 256 rows dequantize the others' to bf16, as `dequantize` gives them.  f32 results
  are off by their f32 sums (below 1e-5 of the largest), bf16 results by half a step."""
  import qwix_amd
  from qwix_amd.core import dot_general as dg
  if most is None:
    most = dg.streamed_rows(N, wq_type == 'int4', K, 128 if tiled else K)
  else:
    monkeypatch.setattr(dg, 'streamed_rows', lambda *a: most)
  _, x = util.make((M, K), O.BF16, seed=93)
  _, w = util.make((G, K, N), dtype, seed=94, scale=0.05)
  wq = qwix_amd.quantize(w, wq_type, channelwise_axes=[0, 2], tiled_axes=tiled or {})
  rounded = qwix_amd.dequantize(wq).to(torch.bfloat16).to(torch.float64)
  codes = (wq.qvalue.unpack() if wq_type == 'int4' else wq.qvalue).to(torch.float64)
  exact = codes * wq.scale.to(torch.float64).repeat_interleave(K // wq.scale.shape[1], 1)
  want, start = torch.zeros(M, N, dtype=torch.float64, device=x.device), 0
  for g, size in enumerate(sizes):
    stop = min(start + max(size, 0), M)
    want[start:stop] = x[start:stop].to(torch.float64) @ (exact if stop - start <= most else rounded)[g]
    start = stop
  largest = float(want.abs().max())
  out = qwix_amd.core.ragged_dot._weight_only_groups(x, wq, _sizes(sizes), torch.float32)
  assert float((out.to(torch.float64) - want).abs().max()) <= 1e-5 * largest
  low = qwix_amd.core.ragged_dot._weight_only_groups(x, wq, _sizes(sizes), torch.bfloat16)
  assert bool(((low.to(torch.float64) - want).abs() <= 2.0 ** -8 * want.abs() + 2e-5 * largest).all())
  assert not out[start:].any()


@pytest.mark.parametrize('K,N,sizes,streamed', [(512, 136, (64, 300, 20, 200), (0, 2)), (384, 72, (256, 17, 257, 0), (0, 1))])
@pytest.mark.parametrize('wq_type', ['int4', 'int8', 'float8_e4m3fn'])
def test_small_groups_keep_their_weights_unrounded_beside_large_ones(K, N, sizes, streamed, wq_type):
  """What a group's weights are rounded to does not depend on the other groups' rows: up to 64 rows (256 with K of 128 mod 256)
  f32 sums of unrounded weights, (K / 16 + 16) roundings of 2^-24 of the terms' magnitude."""
  import qwix_amd
  _, x = util.make((sum(sizes), K), O.BF16, seed=95)
  _, w = util.make((len(sizes), K, N), O.F32, seed=96, scale=0.05)
  wq = qwix_amd.quantize(w, wq_type, channelwise_axes=[0, 2], tiled_axes={1: 128})
  out = qwix_amd.ragged_dot(x, wq, _sizes(sizes), preferred_element_type=torch.float32).to(torch.float64)
  want = _grouped_reference(x, wq, sizes)
  codes = wq.qvalue.unpack() if wq_type == 'int4' else wq.qvalue
  terms = _grouped_reference(x.abs(), types.SimpleNamespace(qtype='int8', qvalue=codes.to(torch.float32).abs(), scale=wq.scale), sizes)
  bound = (K / 16 + 16) * 2.0 ** -24 * terms
  for g in streamed:
    rows = slice(sum(sizes[:g]), sum(sizes[:g + 1]))
    assert bool(((out - want).abs() <= bound)[rows].all()), (g, float(((out - want).abs() / terms)[rows].max()))


@pytest.mark.parametrize('G,K,rows', [(65, 256, 60), (130, 128, 130), (64, 144, 3)])
def test_ragged_dot_looks_at_64_groups_at_a_time(G, K, rows):
  """Groups of every chunk of 64 find their rows and tiles: uneven, empty, negative and overlong sizes, raw sums exact."""
  import qwix_amd
  rng = util.rng(G)
  sizes = [int(v) for v in rng.integers(0, 2 * rows, G)]
  sizes[3], sizes[G // 2], sizes[-1] = -7, 0, 2 ** 31 - 1
  M, N = sum(max(v, 0) for v in sizes[:-1]) + rows + 1, 136
  a = torch.from_numpy(rng.integers(-128, 128, (M, K)).astype(np.int8)).to(util.DEV)
  b = torch.from_numpy(rng.integers(-128, 128, (G, K, N)).astype(np.int8)).to(util.DEV)
  out = qwix_amd.ragged_dot(a, b, _sizes(sizes))
  start = 0
  for g, size in enumerate(sizes):
    stop = min(start + max(size, 0), M)
    assert torch.equal(out[start:stop].to(torch.float64), a[start:stop].to(torch.float64) @ b[g].to(torch.float64)), g
    start = stop
  assert start == M


@pytest.mark.parametrize('kind', ['int8', 'float8_e4m3fn'])
@pytest.mark.parametrize('M,K,N,sizes', [
    (400, 1536, 317, (1, 0, 127, 129, 65)),                                    # 128 rows
    (2499, 384, 2076, (1, 192, 193, 0) + (120,) * 15 + (300,)),                # 192
    (3973, 640, 2565, (1, 256, 257, 0, 1460, 1900, 2 ** 31 - 1)),              # 256; last tiles of 1, 180, 108 and 98 rows
    (3329, 256, 4100, (3300, 0, 1)),                                           # 256: a group of many tiles
])
def test_ragged_dot_tiles_of_128_to_256_rows(M, K, N, sizes, kind):
  """Tile heights are chosen from the average size: groups of one row at the front, a tile and a row more, none; the last rows in no group.
  Small integers under scales that are powers of two: every step of the rounding chain is applied to exact values."""
  import qwix_amd
  g = torch.Generator().manual_seed(K + N)
  dt = torch.int8 if kind == 'int8' else torch.float8_e4m3fn
  G = len(sizes)
  a_i = torch.randint(-7, 8, (M, K), generator=g, dtype=torch.int8).to(util.DEV)
  b_i = torch.randint(-7, 8, (G, K, N), generator=g, dtype=torch.int8).to(util.DEV)
  sa = 2.0 ** torch.randint(-3, 3, (M, 1), generator=g).to(util.DEV)
  sb = 2.0 ** torch.randint(-3, 3, (G, 1, N), generator=g).to(util.DEV)
  print('case ragged tile rows', M, K, N, kind, flush=True)
  x = qwix_amd.QArray(a_i.to(torch.float32).to(dt), sa.to(torch.bfloat16), None, kind)
  w = qwix_amd.QArray(b_i.to(torch.float32).to(dt), sb.to(torch.bfloat16), None, kind)
  out = qwix_amd.ragged_dot(x, w, _sizes(sizes))
  start = 0
  for i, size in enumerate(sizes):
    stop = min(start + size, M)
    want = (a_i[start:stop].to(torch.float64) @ b_i[i].to(torch.float64)).to(torch.float32).to(torch.bfloat16)
    assert torch.equal(out[start:stop], want * sa[start:stop].to(torch.bfloat16) * sb[i].to(torch.bfloat16)), i
    start = stop
  assert torch.count_nonzero(out[start:]).item() == 0


@pytest.mark.parametrize('kind', ['int8', 'float8_e4m3fn'])
@pytest.mark.parametrize('M,K,N,sizes', [(400, 1536, 317, (1, 0, 127, 129, 65)), (2499, 384, 2076, (1, 192, 193, 0) + (120,) * 15 + (300,)),
                                         (3973, 640, 2565, (1, 256, 257, 0, 1460, 1900, 2 ** 31 - 1))])  # as above: 64 to 256 rows
def test_ragged_product_with_a_pitch(M, K, N, sizes, kind):
  """Rows of both operands, and the groups' weights, further apart than they are long, through the C ABI: exact as above."""
  from qwix_amd import _lib
  g = torch.Generator().manual_seed(K + N)
  dt, qt, acc = (torch.int8, _lib.INT8, _lib.I32) if kind == 'int8' else (torch.float8_e4m3fn, _lib.E4M3, _lib.F32)
  G = len(sizes)
  a_i = torch.randint(-7, 8, (M, K), generator=g, dtype=torch.int8).to(util.DEV)
  b_i = torch.randint(-7, 8, (G, N, K), generator=g, dtype=torch.int8).to(util.DEV)
  a = torch.full((M, K + 48), 0x7F, dtype=torch.uint8, device=util.DEV)  # (0x7F: a NaN of e4m3)
  b = torch.full((G, N + 3, K + 16), 0x7F, dtype=torch.uint8, device=util.DEV)
  a[:, :K], b[:, :N, :K] = a_i.to(torch.float32).to(dt).view(torch.uint8), b_i.to(torch.float32).to(dt).view(torch.uint8)
  out = torch.full((M, N + 8), 7.0, dtype=torch.float32, device=util.DEV)
  counts = _sizes(sizes)
  print('case ragged pitch', M, K, N, kind, flush=True)
  _lib.call('qwix_hip_qgemm_ragged', a.data_ptr(), a.stride(0), b.data_ptr(), b.stride(1), b.stride(0), qt, M, N, K, counts.data_ptr(), G, None, 0,
            None, 0, 0, acc, out.data_ptr(), _lib.F32, N + 8, _lib.stream_of(a))
  start = 0
  for i, size in enumerate(sizes):
    stop = min(start + size, M)
    assert torch.equal(out[start:stop, :N].to(torch.float64), a_i[start:stop].to(torch.float64) @ b_i[i].to(torch.float64).T), i
    start = stop
  assert torch.count_nonzero(out[start:, :N]).item() == 0 and bool((out[:, N:] == 7.0).all())


def test_ragged_dot_weight_only_more_row_tiles_than_a_grid():
  """65534 groups of 17 and 3 rows: 98301 row tiles, more than a grid's y axis holds."""
  import qwix_amd
  G, M = 65534, 655340
  g = torch.Generator(device=util.DEV).manual_seed(5)
  x = torch.randn(M, 128, generator=g, device=util.DEV).to(torch.bfloat16)
  wq = qwix_amd.quantize((torch.randn(G, 128, 16, generator=g, device=util.DEV) * 0.05).to(torch.bfloat16), 'int8', channelwise_axes=[0, 2])
  sizes = torch.tensor([17, 3] * (G // 2), dtype=torch.int32, device=util.DEV)
  out = qwix_amd.core.ragged_dot._weight_only_groups(x, wq, sizes, torch.float32)
  group = torch.repeat_interleave(torch.arange(G, device=util.DEV), sizes.long())
  top = 0.0
  for rows in torch.arange(M, device=util.DEV).split(65536):
    w = wq.qvalue[group[rows]].double() * wq.scale[group[rows]].double()
    want = (x[rows].double()[:, :, None] * w).sum(1)
    top = max(top, float((out[rows].double() - want).abs().max() / want.abs().max()))
  assert top <= 1e-5   # f32 sums


def test_ragged_dot_weight_only_popular_group_is_shared_out():
  """Half of the rows in one group cost no more than twice what even groups cost (49 us for 41; with one workgroup
  per group and 64 columns it was 184 for 44)."""
  import qwix_amd
  G, M, K, N = 64, 1024, 2048, 1408
  wq = qwix_amd.quantize((torch.randn(G, K, N, device=util.DEV) * 0.05).to(torch.bfloat16), 'int8', channelwise_axes=[0, 2])
  x = torch.randn(M, K, device=util.DEV).to(torch.bfloat16)
  even, skewed = [16] * G, [8] * G
  skewed[20] = M - 8 * (G - 1)

  def best(sizes):
    sizes, times = _sizes(sizes), []
    for _ in range(8):
      ev = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
      ev[0].record()
      for _ in range(5):
        qwix_amd.ragged_dot(x, wq, sizes)
      ev[1].record()
      torch.cuda.synchronize()
      times.append(ev[0].elapsed_time(ev[1]))
    return min(times)
  assert best(skewed) < 2.0 * best(even)


def test_ragged_dot_dequantize_first_path():
  """A raw float lhs or a zero point sends the call to the dequantize-first path (ragged_dot.py:278-292)."""
  import qwix_amd
  from qwix_amd.core import qarray
  x_np, x_t = util.make((128, 256), O.F32, seed=31)
  wq, owq = _quantized((4, 256, 64), O.F32, 32, _how('int8', (0, 2)), scale=0.05)
  sizes = (50, 50, 28, 0)
  out = qwix_amd.ragged_dot(x_t, wq, _sizes(sizes))
  want = O.ragged_dot(O.FArr(x_np, O.F32), owq, sizes).v
  np.testing.assert_allclose(util.f32np(out), want, rtol=1e-4, atol=1e-4 * np.abs(want).max())
  xz = qarray.quantize(x_t, qarray.HowToQuantize(qtype='int8', calibration_method='minmax'))
  oxz = O.quantize(O.FArr(x_np, O.F32), O.HowToQuantize(qtype='int8', calibration_method='minmax'))
  out = qwix_amd.ragged_dot(xz, wq, _sizes(sizes))
  want = O.ragged_dot(oxz, owq, sizes).v
  np.testing.assert_allclose(util.f32np(out), want, rtol=1e-4, atol=1e-4 * np.abs(want).max())


def test_ragged_dot_errors():
  import qwix_amd
  from qwix_amd.core import ragged_dot as rd
  xq, _ = _quantized((128, 256), O.BF16, 41, _how('int8', (0,)))
  wq, _ = _quantized((4, 256, 64), O.BF16, 42, _how('int8', (0, 2)), scale=0.05)
  with pytest.raises(ValueError, match='one entry per group'):
    qwix_amd.ragged_dot(xq, wq, _sizes((64, 64)))
  with pytest.raises(NotImplementedError, match='group_offset'):
    qwix_amd.ragged_dot(xq, wq, _sizes((64, 64, 0, 0)), group_offset=_sizes((0,)))
  dn = rd.RaggedDotDimensionNumbers((((0,), (1,)), ((), ())), (1,), (0,))   # contracts 128 rows with K = 256
  with pytest.raises(ValueError, match='differ'):
    qwix_amd.ragged_dot_general(xq, wq, _sizes((64, 64, 0, 0)), dn)
  dn = rd.RaggedDotDimensionNumbers((((1,), (1,)), ((), ())), (0,), ())     # no group axis: another ragged mode
  with pytest.raises(NotImplementedError, match='one group axis'):
    qwix_amd.ragged_dot_general(xq, wq, _sizes((64, 64, 0, 0)), dn)


def _rdn(dn, ragged, group):
  from qwix_amd.core.ragged_dot import RaggedDotDimensionNumbers
  return RaggedDotDimensionNumbers(dot_dimension_numbers=dn, lhs_ragged_dimensions=(ragged,), rhs_group_dimensions=(group,))


GENERAL_CASES = [
    # name, lhs shape, rhs shape, dot dimension numbers, ragged axis, group axis, sizes, lhs how, rhs how
    ("the reference's non-basic case: a batch axis, K in tiles of 64, no free axis on the rhs", (8, 620, 256), (8, 4, 256),
     (((2,), (2,)), ((0,), (0,))), 1, 1, (60, 120, 190, 250), dict(tiled_axes={2: 64}), dict(tiled_axes={2: 64})),
    ('weights stored (G, N, K)', (200, 128), (3, 72, 128), (((1,), (2,)), ((), ())), 0, 0, (60, 0, 100),
     dict(channelwise_axes=[0]), dict(channelwise_axes=[0, 1])),
    ('rows last on the lhs, group axis in the middle of the rhs', (128, 300), (128, 5, 40), (((0,), (0,)), ((), ())), 1, 1,
     (10, 0, 130, 1, 70), dict(channelwise_axes=[1]), dict(channelwise_axes=[1, 2])),
    ('two contracting axes', (96, 4, 64), (3, 4, 64, 24), (((1, 2), (1, 2)), ((), ())), 0, 0, (30, 50, 16),
     dict(channelwise_axes=[0]), dict(channelwise_axes=[0, 3])),
    ('batch axis and K in tiles of 128', (2, 150, 256), (2, 4, 256, 136), (((2,), (2,)), ((0,), (0,))), 1, 1, (40, 0, 100, 10),
     dict(channelwise_axes=[0, 1], tiled_axes={2: 128}), dict(channelwise_axes=[0, 1, 3], tiled_axes={2: 128})),
]


@pytest.mark.parametrize('dtype', [O.BF16, O.F32])
@pytest.mark.parametrize('name,lshape,rshape,dn,ragged,group,sizes,lhow,rhow', GENERAL_CASES)
def test_ragged_dot_general_dimension_numbers(name, lshape, rshape, dn, ragged, group, sizes, lhow, rhow, dtype):
  """Dimension numbers other than ragged_dot's (ragged_dot.py:123-226 passes any to lax.ragged_dot_general): the ragged
  axis as the only free axis of the lhs, with batch axes, several contracting axes and any axis order.  int8: exact
  sums and an elementwise epilogue, so bit for bit wherever a single K tile is scaled; f32 sums of tile partials at
  1e-5."""
  import qwix_amd
  from qwix_amd.core import qarray
  print('case ragged general', name, dtype, flush=True)
  x_np, x_t = util.make(lshape, dtype, seed=len(name))
  w_np, w_t = util.make(rshape, dtype, seed=len(name) + 1, scale=0.05)
  xq, oxq = qarray.quantize(x_t, qarray.HowToQuantize(qtype='int8', **lhow)), O.quantize(O.FArr(x_np, dtype), O.HowToQuantize(qtype='int8', **lhow))
  wq, owq = qarray.quantize(w_t, qarray.HowToQuantize(qtype='int8', **rhow)), O.quantize(O.FArr(w_np, dtype), O.HowToQuantize(qtype='int8', **rhow))
  util.assert_qarray_equal(xq, oxq, 'lhs')
  util.assert_qarray_equal(wq, owq, 'rhs')
  out = qwix_amd.ragged_dot_general(xq, wq, _sizes(sizes), _rdn(dn, ragged, group))
  want = O.ragged_dot_general(oxq, owq, sizes, dn, ragged, group)
  assert out.dtype == util.TORCH_DT[want.dtype]
  tiled = 'tiled_axes' in lhow or 'tiled_axes' in rhow
  if tiled and dtype == O.F32:
    np.testing.assert_allclose(util.f32np(out), want.v, rtol=0, atol=1e-5 * float(np.abs(want.v).max()))
  elif tiled:
    # bf16 partials: the reference rounds each three times before the f32 sum; the default mode keeps them in f32
    np.testing.assert_allclose(util.f32np(out), want.v, rtol=0, atol=2e-2 * float(np.abs(want.v).max()))
  else:
    _check_exact(out, want)


def test_ragged_dot_general_weight_only_and_errors():
  import qwix_amd
  from qwix_amd.core import qarray
  x_np, x_t = util.make((200, 128), O.BF16, seed=3)
  w_np, w_t = util.make((3, 72, 128), O.BF16, seed=4, scale=0.05)
  how = dict(qtype='int8', channelwise_axes=[0, 1])
  wq, owq = qarray.quantize(w_t, qarray.HowToQuantize(**how)), O.quantize(O.FArr(w_np, O.BF16), O.HowToQuantize(**how))
  dn = (((1,), (2,)), ((), ()))
  out = qwix_amd.ragged_dot_general(x_t, wq, _sizes((60, 0, 100)), _rdn(dn, 0, 0))     # float lhs: dequantize first
  want = O.ragged_dot_general(O.FArr(x_np, O.BF16), owq, (60, 0, 100), dn, 0, 0)
  np.testing.assert_allclose(util.f32np(out), want.v, rtol=1e-2, atol=1e-2 * float(np.abs(want.v).max()))
  assert np.all(util.f32np(out)[160:] == 0)
  with pytest.raises(NotImplementedError, match='ragged contracting or batch axis'):
    qwix_amd.ragged_dot_general(x_t, wq, _sizes((60, 0, 100)), _rdn(dn, 1, 0))
  x3 = torch.zeros(4, 200, 128, dtype=torch.bfloat16, device=util.DEV)
  with pytest.raises(NotImplementedError, match='only free axis'):
    qwix_amd.ragged_dot_general(x3, wq, _sizes((60, 0, 100)), _rdn((((2,), (2,)), ((), ())), 1, 0))
