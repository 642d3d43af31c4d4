"""Gathered K/V rows (kv_index) need the direct-to-LDS route's alignments: each refusal is decided on
the host, before anything is launched, so no GPU is needed."""
import ctypes as C

import pytest

from sparsefold_amd import _lib


def _args(**over):
  a = _lib.AttentionArgs()
  a.B0, a.B1, a.Q, a.K, a.H, a.D, a.Dv = 1, 1, 32, 128, 4, 32, 32
  a.scale = 1.0
  base = 1 << 20                                        # never dereferenced: the calls are refused
  for key in ("q", "k", "v", "out", "bias", "kv_index"):
    setattr(a, key, base)
  rows = (C.c_int64 * 4)(0, 0, 128, 32)
  a.q_s = a.k_s = a.v_s = a.o_s = rows
  a.bias_s = (C.c_int64 * 4)(0, 0, 32 * 128, 128)
  a.kv_zero_row = 128
  for key, value in over.items():
    setattr(a, key, value)
  return a


@pytest.mark.parametrize("over", [{"bias": (1 << 20) + 2}, {"bias_s": (C.c_int64 * 4)(0, 0, 32 * 129, 129)},
                                  {"q": (1 << 20) + 8}, {"kv_zero_row": -1}])
def test_gathered_rows_refuse_unaligned_operands(over):
  assert _lib.load().sf_hip_attention_fwd(C.byref(_args(**over)), None) != 0
  assert "gathered K/V rows" in _lib.last_error()
