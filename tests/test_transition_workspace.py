"""Workspace of the transitions: none where one kernel does it all, whatever addresses the call comes
with, and what the general path refuses stays refused.  Decided on the host, nothing is launched."""
import ctypes

import pytest

from sparsefold_amd import _lib

BASE = 1 << 32                                          # never dereferenced


def _args(C=128, I=512, rows=384 * 384, **over):
  a = _lib.TransitionArgs()
  a.S, a.N, a.C, a.I = 1, rows, C, I
  for key, value in over.items():
    setattr(a, key, value)
  return a


def _bytes(a):
  return int(_lib.load().sf_hip_transition_workspace_bytes(ctypes.byref(a)))


def test_the_one_kernel_form_needs_none():
  pointers = {"x": BASE, "out": 2 * BASE, "w1": 3 * BASE, "w2": 4 * BASE}
  assert _bytes(_args()) == 0 and _bytes(_args(**pointers)) == 0
  assert _bytes(_args(**{**pointers, "out": 2 * BASE + 2})) == 0


@pytest.mark.parametrize("over", [{"C": 384, "I": 1536}, {"I": 96}, {"cond": BASE, "Cs": 384}, {"pre_scale": BASE}])
def test_the_general_form_holds_both_intermediates(over):
  a = _args(**over)
  assert _bytes(a) >= a.N * (a.C + a.I) * 2


@pytest.mark.parametrize("key", ["x", "w1", "w2"])
def test_misaligned_operands_are_refused(key):
  pointers = {"x": BASE, "out": 2 * BASE, "w1": 3 * BASE, "w2": 4 * BASE}
  pointers[key] += 8
  a = _args(**pointers)
  assert _lib.load().sf_hip_transition_fwd(ctypes.byref(a), None, 0, None) != 0
  assert "aligned" in _lib.last_error()


def test_the_general_form_refuses_a_missing_workspace():
  a = _args(I=96, x=BASE, out=2 * BASE, w1=3 * BASE, w2=4 * BASE)
  assert _lib.load().sf_hip_transition_fwd(ctypes.byref(a), None, 0, None) != 0
  assert "workspace" in _lib.last_error()
