"""Quantization rules and the provider base class (host-side configuration only).

Mirror of qwix/_src/qconfig.py: `QuantizationRule` (:31-92, same field names and defaults) and
the rule lookup of `QuantizationProvider._get_current_rule_and_op_id` (:209-240): the first rule
whose `module_path` regex fully matches '/'.join(current module path) and whose `op_names` (if
any) contains the op wins; per (module, op) an op id '<op><n>' numbers repeated ops.

There is no Flax here, so the "current module path" comes from `module_scope`, a thread-local
stack that the bundled `qwix_amd.nn` modules (or user code) push while they run.
"""
from __future__ import annotations

import contextlib
import dataclasses
import re
import threading
from typing import Any, Collection, Sequence


@dataclasses.dataclass(frozen=True, kw_only=True)
class QuantizationRule:
  """Which modules / ops to quantize, and how.  Fields as in the reference."""

  module_path: str = '.*'
  op_names: Collection[str] = ()
  weight_qtype: Any = None
  act_qtype: Any = None
  tile_size: int | float | None = None
  act_static_scale: bool | None = None
  weight_calibration_method: str = 'absmax'
  act_calibration_method: str | None = None
  act_batch_axes: Collection[int] = (0,)


_tls = threading.local()


def current_module_path() -> tuple[str, ...]:
  return tuple(getattr(_tls, 'path', ()))


class module_scope(contextlib.ContextDecorator):
  """Pushes `name` on this thread's module path for the duration of the block (or of the decorated function's calls)."""

  def __init__(self, name: str):
    self._name = name
    self._old = None

  def _recreate_cm(self) -> 'module_scope':
    return module_scope(self._name)  # calls may nest

  def __enter__(self) -> None:
    if self._old is not None:  # it holds one path to go back to
      raise RuntimeError('a module_scope is entered once: make another one')
    self._old = current_module_path()
    _tls.path = self._old + (self._name,)

  def __exit__(self, *exc) -> None:
    _tls.path = self._old


class QuantizationProvider:
  """Holds the rules and resolves the rule that applies to the op being executed."""

  def __init__(self, rules: Sequence[QuantizationRule], *, disable_jit: bool = False):
    self._rules = [self._init_rule(rule) for rule in rules]
    self._rule_matches = [False] * len(self._rules)
    self._rule_of: dict[tuple[tuple[str, ...], str], int] = {}  # (module path, op) -> the rule that applies, -1: none
    self._op_counts: dict[tuple[tuple[str, ...], str], int] = {}
    self._initial_run_complete = False  # set by the model wrapper once the model has run under this provider
    self.disable_jit = disable_jit

  @staticmethod
  def _init_rule(rule: QuantizationRule) -> QuantizationRule:
    """Validates a rule and fills its defaults (qconfig.py:122-135)."""
    if rule.act_qtype is None and rule.act_static_scale is not None:
      raise ValueError(f'Invalid rule: act_static_scale is set to {rule.act_static_scale} but act_qtype is None. '
                       'Please either unset act_static_scale, or set act_qtype to enable activation quantization. '
                       f'(Rule: {rule})')
    if rule.act_static_scale is None:
      rule = dataclasses.replace(rule, act_static_scale=False)
    if rule.act_calibration_method is None:
      rule = dataclasses.replace(rule, act_calibration_method='absmax')
    return rule

  def reset_op_ids(self) -> None:
    """Op ids restart at 0 for every model call, so that the same op gets the same id each time."""
    self._op_counts = {}

  def _get_current_rule_and_op_id(self, op_name: str, *, only_rule: bool = False):
    path = current_module_path()
    key = (path, op_name)
    i = self._rule_of.get(key)
    if i is None:
      path_str = '/'.join(path)
      i = next((i for i, r in enumerate(self._rules)
                if re.fullmatch(r.module_path, path_str) and (not r.op_names or op_name in r.op_names)), -1)
      if len(self._rule_of) < 4096:
        self._rule_of[key] = i
    rule = None
    if i >= 0:
      rule = self._rules[i]
      self._rule_matches[i] = True
    if only_rule:
      return rule, None
    n = self._op_counts.get(key, 0)
    self._op_counts[key] = n + 1
    return rule, f'{op_name}{n}'

  def get_unused_rules(self) -> list[QuantizationRule]:
    """Rules that never matched (qconfig.py:242-262); only meaningful once the model has run."""
    if not self._initial_run_complete:
      raise ValueError('Quantization is not completed yet. Please call `quantize_model` and run the model '
                       'before calling `get_unused_rules`.')
    return [r for r, used in zip(self._rules, self._rule_matches) if not used]
