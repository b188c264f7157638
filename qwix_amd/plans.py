"""Launch plans for the operators: recorded from one ordinary call, replayed by the native module `_plans`.

An operator's Python decides from shapes, strides, dtypes and options which buffers to allocate and which entry points to
call; at decode sizes that takes longer than the kernels (quantize + dot_general of 64 rows: 50 us of Python for 21 us on the
device).  `call` looks the operands' metadata up in a native table and replays the plan kept for it in a few microseconds.

A plan is recorded when a kind of call comes up for the `RECORD_AT`-th time: the ordinary path runs once under a `Recorder`, which
notes every allocation and every entry point call with its constants, and tells operands, buffers and constants apart.  A
plan is kept only if that is all the path did: any other device operation of torch (a copy, a padding, a reduction), a pointer
to memory that is neither an operand nor a buffer of this call (a re-laid-out weight kept from earlier), work whose result
is kept for later calls (`kept_aside`), operands that overlap, or a result that is not one of the buffers leave the call to
the ordinary path for good.
"""
from __future__ import annotations

import ctypes
import threading

import torch
from torch.utils._python_dispatch import TorchDispatchMode

from qwix_amd import _lib

_CONST, _FLOAT, _OPERAND, _BUFFER, _STREAM = range(5)  # argument kinds of plans.cpp

# Recording costs a few hundred microseconds once, replaying saves 20 to 50 each time: shapes that come up a few times and
# never again (a cache that grows with every token) are not worth it.
RECORD_AT = 4

_native = None


def native():
  """The native module, loaded with the library it calls."""
  global _native
  if _native is None:
    _lib.load()
    try:
      from qwix_amd import _plans
    except ImportError as e:
      raise _lib.QwixHipError('qwix_amd/_plans.so is missing or does not load: build it with '
                              '`python qwix_amd/csrc/build.py`') from e
    from qwix_amd.core import qarray
    _plans.setup(qarray.QArray, qarray.Int4Tensor, torch._C._cuda_getCurrentRawStream, _lib.raise_status,
                 RECORD_AT)
    _native = _plans
  return _native


_ALLOCATIONS = frozenset(('aten::empty.memory_format', 'aten::empty_strided', 'aten::empty_like', 'aten::new_empty'))
_ON_THE_HOST = frozenset(('aten::promote_types', 'aten::record_stream'))   # dtypes alone; the allocator's book-keeping


def _storages(values) -> set:
  return {t.untyped_storage().data_ptr() for v in values for t in (v if isinstance(v, (list, tuple)) else (v,))
          if isinstance(t, torch.Tensor)}


def _is_view(func, args, out) -> bool:
  """Whether an operation did nothing on the device: it writes to none of its arguments and all it returns are tensors in an
  argument's memory.  (Told by the effect: `reshape`, `contiguous` and `to` are views or copies, and reach the recorder by
  these names in inference mode, where torch does not take them apart before.)"""
  outs = out if isinstance(out, (list, tuple)) else (out,)
  return (not func._schema.is_mutable and all(isinstance(t, torch.Tensor) for t in outs)
          and _storages(outs) <= _storages(args))


def _extent(t: torch.Tensor) -> tuple[int, int]:
  """First byte and one past the last byte that the tensor's elements occupy."""
  start = t.data_ptr()
  if t.numel() == 0:
    return start, start
  return start, start + (sum((n - 1) * s for n, s in zip(t.shape, t.stride())) + 1) * t.element_size()


class Recorder(TorchDispatchMode):
  """Notes what one call of an operator does on the device; `ok` turns False when it is more than a plan can say."""

  _active = threading.local()

  def __init__(self, operands):
    super().__init__()
    self.ok = True
    self.buffers: list[torch.Tensor] = []   # kept alive, so that no address comes up twice
    self.calls: list = []
    self.operands = operands
    spans = sorted(_extent(t) for t in operands)
    if any(a[1] > b[0] for a, b in zip(spans, spans[1:])):
      self.ok = False

  def __enter__(self):
    self._active.recorder = self
    _lib.recorder_of = self._active
    return super().__enter__()

  def __exit__(self, *exc):
    self._active.recorder = None
    return super().__exit__(*exc)

  def __torch_dispatch__(self, func, types, args=(), kwargs=None):
    out = func(*args, **(kwargs or {}))
    name = func._schema.name + ('.' + func._schema.overload_name if func._schema.overload_name else '')
    if name in _ALLOCATIONS:
      self.buffers.append(out)
    elif name not in _ON_THE_HOST and not _is_view(func, args, out):
      self.ok = False
    return out

  def _place(self, pointer: int):
    """(kind, index, byte offset) of a device pointer, or None."""
    found = []
    for kind, tensors in ((_OPERAND, self.operands), (_BUFFER, self.buffers)):
      for k, t in enumerate(tensors):
        first, last = _extent(t)
        if first <= pointer < last:
          found.append((kind, k, pointer - first))
    return found[0] if len(found) == 1 else None

  def note(self, name: str, args) -> None:
    """One call of a library entry point: its last argument is the stream, the others are told apart by their types."""
    types = _lib.SIGNATURES[name][1]
    noted = []
    for value, kind in zip(args[:-1], types[:-1]):
      if kind is ctypes.c_void_p and value:
        place = self._place(value) if isinstance(value, int) else None
        if place is None:
          self.ok = False
          return
        noted.append(place)
      elif kind is ctypes.c_float:
        noted.append((_FLOAT, 0, float(value)))
      elif value is None or isinstance(value, int):
        noted.append((_CONST, 0, int(value or 0)))
      else:
        self.ok = False
        return
    noted.append((_STREAM, 0, 0))
    self.calls.append((name, noted))

  def results(self, tensors):
    """The buffers that the results are views of: [(buffer, sizes, strides, offset in elements)], or None."""
    out = []
    for t in tensors:
      if not isinstance(t, torch.Tensor) or t.numel() == 0:
        return None
      for k, b in enumerate(self.buffers):
        if b.untyped_storage().data_ptr() == t.untyped_storage().data_ptr() and b.dtype == t.dtype:
          out.append((k, tuple(t.shape), tuple(t.stride()), t.storage_offset() - b.storage_offset()))
          break
      else:
        return None
    return out


def kept_aside() -> None:
  """Called where an operator has just prepared something from a weight that it keeps and later calls read (a re-laid-out
  copy, sums): a plan recorded around it would repeat the preparation on every replay."""
  recorder = getattr(Recorder._active, 'recorder', None)
  if recorder is not None:
    recorder.ok = False


def record(fixed, operands, fn, split):
  """fn() under a recorder; the plan is kept if the recorder understood everything.  `split(result)` gives the result's tensors
  and what puts them together again (None: the result is the tensor itself)."""
  n = native()
  tensors = n.tensors(*operands)
  if tensors is None:
    return fn()
  n.recording(1)
  try:
    with Recorder(tensors) as rec:
      out = fn()
  finally:
    n.recording(-1)
  if rec.ok and rec.calls:
    parts, rebuild = split(out)
    results = rec.results(parts)
    if results is not None:
      n.keep(fixed, tuple(operands), [(tuple(b.shape), tuple(b.stride()), b) for b in rec.buffers], rec.calls, results,
             rebuild)
  return out


def single(out):
  """`split` for operators that return one tensor."""
  return (out,), None
