"""The attention's numeric domain: biases of -inf, NaN or +inf at masked keys, and finite biases up to
2^127, in every schedule, with bias rows of any alignment and with the key range in slices."""
import pytest
import torch

from oracle import modules as OM
from sparsefold_amd import workloads as W
from sparsefold_amd.backends.hip import ops
from tests._metrics import assert_close_bf16
from tests.test_gpu_modules import DEV, _params, _prepared, hip_backend   # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu
INF, NAN = float("inf"), float("nan")
B, H = 2, 4
# aligned rows, rows of an even number of elements that is no multiple of 8, odd rows; a ragged last tile
SIZES = [(128, 320), (130, 300), (129, 301)]


def _case(Q, K, D):
  g = torch.Generator().manual_seed(Q + K + D)
  r = lambda *s: torch.randn(*s, generator=g).bfloat16()
  return r(B, Q, H, D), r(B, K, H, D), r(B, K, H, D), r(B, H, Q, K), torch.rand(B, K, generator=g) > 0.3


def _reference(q, k, v, bias, mask, scale):
  """64 bits; a masked key's logit is one finite value whatever its q.k and bias are."""
  s = torch.matmul(q.double().transpose(1, 2), k.double().permute(0, 2, 3, 1).contiguous()) * scale + bias.double()
  s = torch.where(mask[:, None, None, :], s, torch.full_like(s, -1e300))
  return torch.matmul(torch.softmax(s, -1), v.double().transpose(1, 2)).transpose(1, 2)


def _check(q, k, v, bias, mask, schedule):
  scale = q.shape[-1] ** -0.5
  d = lambda t: t.to(DEV)
  out = ops.attention(d(q)[:, None], d(k)[:, None], d(v)[:, None], scale=scale, bias=d(bias)[:, None],
                      mask_k=d(mask)[:, None].to(torch.uint8), schedule=schedule)[:, 0].cpu().double()
  ref = _reference(q, k, v, bias, mask, scale)
  assert bool(torch.isfinite(ref).all()) and bool(torch.isfinite(out).all())
  # bf16 weights and result: 2^-9 each, random signs
  err = float((out - ref).norm() / ref.norm())
  assert err <= 2.0 ** -7.5, err


@pytest.mark.parametrize("D", [24, 48])
@pytest.mark.parametrize("Q,K", SIZES)
@pytest.mark.parametrize("schedule", [0, 1, 2])
def test_minus_infinity_over_whole_tiles(Q, K, D, schedule):
  q, k, v, bias, mask = _case(Q, K, D)
  mask[:] = True
  bias[0, :, :, :128] = -INF                           # the first tiles
  bias[1, :, 5:, 64:192] = -INF                        # tiles in between
  bias[1, 1, :5, :K - 1] = -INF                        # all but the last key
  _check(q, k, v, bias, mask, schedule)
  excluded = bias == -INF
  for value in (torch.finfo(torch.bfloat16).min, -1e9):  # the other usual ways to exclude keys
    bias[excluded] = value
    _check(q, k, v, bias, mask, schedule)


@pytest.mark.parametrize("D", [24, 48])
@pytest.mark.parametrize("Q,K", SIZES)
@pytest.mark.parametrize("schedule", [0, 1, 2])
def test_masked_keys_weigh_nothing_whatever_they_hold(Q, K, D, schedule):
  q, k, v, bias, mask = _case(Q, K, D)
  mask[0, :70] = False                                 # a whole tile among them
  mask[1, K - 3:] = False                              # the last key, which the copies past K repeat
  hidden = ~mask[:, None, None, :].expand_as(bias)
  for value in (INF, -INF, NAN, 3e38):
    _check(q, k, v, torch.where(hidden, torch.full_like(bias, value), bias), mask, schedule)
  k[~mask] = NAN
  out = ops.attention(q.to(DEV)[:, None], k.to(DEV)[:, None], v.to(DEV)[:, None], scale=D ** -0.5, bias=bias.to(DEV)[:, None],
                      mask_k=mask.to(DEV)[:, None].to(torch.uint8), schedule=schedule)[:, 0].cpu().double()
  ref = _reference(q, torch.nan_to_num(k), v, bias, mask, D ** -0.5)
  assert float((out - ref).norm() / ref.norm()) <= 2.0 ** -7.5


@pytest.mark.parametrize("Q,K", SIZES)
@pytest.mark.parametrize("schedule", [0, 1, 2])
def test_all_keys_masked_weigh_alike(Q, K, schedule):
  q, k, v, bias, mask = _case(Q, K, 48)
  mask[1] = False
  bias[1] = NAN
  _check(q, k, v, bias, mask, schedule)


@pytest.mark.parametrize("D", [24, 48])
@pytest.mark.parametrize("Q,K", SIZES)
@pytest.mark.parametrize("schedule", [0, 1, 2])
def test_large_finite_biases(Q, K, D, schedule):
  """|log2(e) bias| up to the largest float; bf16 holds 2e38 and 1.9e38 as different values."""
  q, k, v, bias, mask = _case(Q, K, D)
  mask[:] = True
  bias[0, 0] = -2e38                                   # every key alike
  bias[0, 1] = -2e38
  bias[0, 1, :, 70] = -1.9e38                          # one key above the others, past the first tile
  bias[0, 2] = 1.9e38
  bias[0, 2, :, K - 1] = 2e38
  bias[0, 3, :, :64] = -2e38                           # a first tile far below the rest
  bias[1, 0] = 2e38
  _check(q, k, v, bias, mask, schedule)


@pytest.mark.parametrize("N", [301, 304, 437])
def test_minus_infinity_at_the_start_of_a_key_slice(N):
  """One sample: few enough tasks that the module runs the key range in slices."""
  mod, x, cond, bias, mask = W.make_diffusion(N, S=1, C=384, H=8, seed=N, sharp=True)
  bias[:, :, 128:192] = -INF
  bias[1, :7, :N - 40] = -INF
  hip = _prepared(mod)
  out = hip(x.to(DEV), mask.to(DEV), pair_logits=bias.to(DEV), single_cond=cond.to(DEV), add_residual=False)
  ref = OM.self_attention(x.float(), mask, _params(hip), pair_logits=bias.float(), single_cond=cond.float(), return_update=True)
  assert_close_bf16(out, ref, f"slices N={N}", max_abs=2e-2 * max(1.0, ref.abs().max().item()))
