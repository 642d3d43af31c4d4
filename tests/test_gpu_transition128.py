"""The one-kernel transition of 128 channels (csrc/transition.hip) against the 64-bit result, at the
edges of its 32-row items, its 256-row passes and its blocks of intermediate channels, and the
general path (I not a multiple of 64) beside it.

Bound: h, the gated intermediate c and the result are rounded to bf16, 2^-9 of their value each.  With y =
h W1^T and c = silu(a) b over its channel pairs, the first two reach the result as
  |dy| <= 2^-9 |h| |W1|^T,  |dc| <= 2^-9 |c| + |silu'(a) b| |dy_a| + |silu(a)| |dy_b|,  |du| <= |dc| |W2|^T
element by element (10% on top for the second order and the fp32 sums); over all elements the
roundings have random signs, and three of 2^-9 with a gain of up to 2 at the gate stay below 4 x 2^-9."""
import ctypes

import pytest
import torch

from sparsefold_amd import _lib

pytestmark = pytest.mark.gpu


def _weights(I, seed):
  g = torch.Generator(device="cuda").manual_seed(seed)
  r = lambda *s: torch.randn(*s, generator=g, device="cuda")
  return (1 + 0.2 * r(128), 0.2 * r(128), (r(2 * I, 128) / 128 ** 0.5).bfloat16(), (r(128, I) / I ** 0.5).bfloat16(), r)


def _call(x, out, ln_w, ln_b, w1, w2, residual):
  a = _lib.TransitionArgs()
  a.S, a.N, a.C, a.I, a.add_residual = 1, x.shape[0], 128, w2.shape[1], int(residual)
  p = lambda t: None if t is None else t.data_ptr()
  a.x, a.out, a.ln_w, a.ln_b, a.w1, a.w2 = p(x), p(out), p(ln_w), p(ln_b), p(w1), p(w2)
  lib = _lib.load()
  ws = torch.empty(int(lib.sf_hip_transition_workspace_bytes(ctypes.byref(a))), dtype=torch.uint8, device="cuda")
  _lib.check(lib.sf_hip_transition_fwd(ctypes.byref(a), ctypes.c_void_p(ws.data_ptr()), ws.numel(),
                                       ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)), "sf_hip_transition_fwd")
  return out


def _reference(x, ln_w, ln_b, w1, w2):
  """The update and the bound of its error before its own rounding."""
  x, w1, w2 = x.double(), w1.double(), w2.double()
  h = torch.nn.functional.layer_norm(x, (128,), None if ln_w is None else ln_w.double(), None if ln_b is None else ln_b.double())
  y, dy = h @ w1.t(), 2.0 ** -9 * (h.abs() @ w1.abs().t())
  a, b, da, db = y[:, 0::2], y[:, 1::2], dy[:, 0::2], dy[:, 1::2]
  s = torch.sigmoid(a)
  c = a * s * b
  dc = 2.0 ** -9 * c.abs() + (s * (1 + a * (1 - s)) * b).abs() * da + (a * s).abs() * db
  return c @ w2.t(), dc @ w2.abs().t()


def _check(out, ref, update, bound):
  err = (out.double() - ref).abs()
  bound = 1.1 * bound + ref.abs() * 2.0 ** -8
  assert bool((err <= bound).all()), float((err - bound).max())
  assert err.norm() <= 4 * 2.0 ** -9 * update.norm() + 2.0 ** -9 * ref.norm(), float(err.norm() / update.norm())


@pytest.mark.parametrize("rows,I", [(1, 64), (31, 128), (33, 512), (255, 512), (257, 64), (8191, 128), (256 * 257 + 5, 512), (300, 96)])
@pytest.mark.parametrize("affine", [True, False])
def test_update_and_residual(rows, I, affine):
  ln_w, ln_b, w1, w2, r = _weights(I, rows + I)
  if not affine:
    ln_w = ln_b = None
  x = (2 * r(rows, 128) + 0.5).bfloat16()
  upd, bound = _reference(x, ln_w, ln_b, w1, w2)
  _check(_call(x, torch.full_like(x, 7.0), ln_w, ln_b, w1, w2, False), upd, upd, bound)
  _check(_call(x, torch.full_like(x, 7.0), ln_w, ln_b, w1, w2, True), x.double() + upd, upd, bound)


@pytest.mark.parametrize("rows", [33, 300])
def test_output_at_any_even_address_without_a_workspace(rows):
  ln_w, ln_b, w1, w2, r = _weights(128, rows)
  x = r(rows, 128).bfloat16()
  want = _call(x, torch.empty_like(x), ln_w, ln_b, w1, w2, True)
  buf = torch.full((rows * 128 + 8,), 7.0, device="cuda").bfloat16()
  _call(x, buf[3:3 + rows * 128].view(rows, 128), ln_w, ln_b, w1, w2, True)
  assert torch.equal(buf[3:3 + rows * 128].view(rows, 128), want)
  assert bool((buf[:3] == 7).all()) and bool((buf[3 + rows * 128:] == 7).all())


def test_in_place():
  ln_w, ln_b, w1, w2, r = _weights(512, 3)
  x = r(70001, 128).bfloat16()
  want = _call(x, torch.empty_like(x), ln_w, ln_b, w1, w2, True)
  y = x.clone()
  _call(y, y, ln_w, ln_b, w1, w2, True)
  assert torch.equal(y, want)
