"""Sizes whose rows start at any even address: the attention's bias tiles (rows of any alignment and
length through LDS), the pair-logit planes of an odd number of positions, and the shared-tile
schedule on small grids, each against a 64-bit reference."""
import pytest
import torch

from sparsefold_amd.backends.hip import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _attention(q, k, v, bias, mask, scale):
  s = torch.einsum("bqhd,bkhd->bhqk", q.cpu().double(), k.cpu().double()) * scale + bias.cpu().double()
  s = s.masked_fill(~mask.cpu().bool()[None, None, None, :], -1e30)
  return torch.einsum("bhqk,bkhd->bqhd", torch.softmax(s, -1), v.cpu().double())


# the fewest keys of the LDS form (8), the ends of a 64-key tile, one key past it, odd rows
@pytest.mark.parametrize("D", [24, 48])
@pytest.mark.parametrize("Q,K", [(128, 8), (130, 9), (129, 63), (131, 65), (200, 127), (32, 129), (437, 437), (741, 741)])
@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("schedule", [0, 1, 2])
def test_attention_bias_rows_of_any_alignment(D, Q, K, offset, schedule):
  B, H = 2, 4
  g = torch.Generator(device=DEV).manual_seed(Q + K + D)
  r = lambda *s: torch.randn(*s, generator=g, device=DEV)
  q, k, v = (r(B, n, H, D).bfloat16() for n in (Q, K, K))
  bias = r(H * Q * K + offset).bfloat16()[offset:].view(H, Q, K)      # ends at its buffer's last byte
  mask = (r(K) > -1.0).to(torch.uint8)
  mask[0] = 1
  out = ops.attention(q[:, None], k[:, None], v[:, None], scale=D ** -0.5, bias=bias.expand(B, 1, H, Q, K),
                      mask_k=mask.expand(B, 1, K), schedule=schedule)[:, 0]
  ref = _attention(q, k, v, bias[None], mask, D ** -0.5)
  err = (out.cpu().double() - ref).norm() / ref.norm()
  # bf16 weights and result: 2^-9 each, random signs
  assert err <= 2.0 ** -7.5, float(err)


@pytest.mark.parametrize("H", [1, 16, 33, 64, 130])
@pytest.mark.parametrize("P", [1, 7, 8, 9, 121, 127, 128, 129, 437 * 437, 1023 * 3 + 2])
def test_pair_logit_planes_of_any_length(P, H):
  g = torch.Generator(device=DEV).manual_seed(P + H)
  z = torch.randn(P, 128, generator=g, device=DEV).bfloat16()
  ln_w, ln_b = (torch.randn(128, generator=g, device=DEV) * 0.2 + c for c in (1.0, 0.0))
  w = (torch.randn(H, 128, generator=g, device=DEV) / 128 ** 0.5).bfloat16()
  out = ops.pair_logits(z, ln_w, ln_b, w)
  h = torch.nn.functional.layer_norm(z.double(), (128,), ln_w.double(), ln_b.double())
  ref = w.double() @ h.t()
  assert out.shape == (H, P)
  err = (out.double() - ref).abs()
  # h and the folded weight are rounded to bf16 (2^-9 each, over 128 terms), and the result
  bound = ref.abs() * 2.0 ** -8 + 2 * 2.0 ** -9 * (w.double().abs() @ (h.abs() + ln_b.double().abs()).t())
  assert bool((err <= bound).all()), float((err - bound).max())


def test_noalloc_runs_what_only_the_slices_would_not_fit():
  """Odd N takes key-range slices now; where they alone pass the fixed scratch, the entry point without
  a workspace still runs (without slices), as before."""
  from sparsefold_amd import _lib
  import ctypes
  N, C, H, D = 3801, 768, 16, 48
  a = _lib.SelfAttentionArgs()
  a.S, a.N, a.C, a.H, a.D = 1, N, C, H, D
  w = {"w_qkvg": torch.randn(4 * C, C, device=DEV).bfloat16() / 28, "b_qkvg": torch.zeros(4 * C, device=DEV),
       "w_t2": torch.randn(C, C, device=DEV).bfloat16() / 28, "ln_w": torch.ones(C, device=DEV)}
  x = torch.randn(1, N, C, device=DEV).bfloat16()
  bias = torch.randn(H, N, N, device=DEV).bfloat16()
  with_ws = ops.self_attention_module(x, None, bias, None, w, num_head=H, head_dim=D)
  without = ops.self_attention_module(x, None, bias, None, w, num_head=H, head_dim=D, noalloc=True)
  err = (with_ws.float() - without.float()).norm() / with_ws.float().norm()
  assert err <= 2.0 ** -8, float(err)
