"""Conditioning widths and channel counts that the one-launch conditioning kernel does not take (channels
not a multiple of 128, conditions wider than 384 or not a multiple of 16): LayerNorm and one product a term."""
import pytest
import torch

from oracle import modules as OM
from sparsefold_amd import workloads as W
from tests._metrics import assert_close_bf16
from tests.test_gpu_modules import DEV, _params, _prepared, hip_backend   # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu
SIZES = [(192, 64, 4), (64, 384, 4), (384, 392, 8), (768, 24, 16), (256, 512, 8)]


@pytest.mark.parametrize("C,C_cond,H", SIZES)
def test_self_attention(C, C_cond, H):
  mod, x, cond, bias, mask = W.make_diffusion(100, S=2, C=C, C_cond=C_cond, H=H, seed=C + C_cond, sharp=True, padded=True)
  hip = _prepared(mod)
  out = hip(x.to(DEV), mask.to(DEV), pair_logits=bias.to(DEV), single_cond=cond.to(DEV), add_residual=False)
  ref = OM.self_attention(x.float(), mask, _params(hip), pair_logits=bias.float(), single_cond=cond.float(), return_update=True)
  assert_close_bf16(out, ref, f"attention C={C} Cs={C_cond}", max_abs=2e-2 * max(1.0, ref.abs().max().item()))


@pytest.mark.parametrize("C,C_cond,H", SIZES)
def test_diffusion_transition(C, C_cond, H):
  mod, x, cond = W.make_diffusion_transition(100, S=2, C=C, C_cond=C_cond, seed=C + C_cond, sharp=True)
  hip = _prepared(mod)
  out = hip(x.to(DEV), single_cond=cond.to(DEV), add_residual=False)
  ref = OM.diffusion_transition_block(x.float(), cond.float(), _params(hip), return_update=True)
  assert_close_bf16(out, ref, f"transition C={C} Cs={C_cond}", max_abs=2e-2 * max(1.0, ref.abs().max().item()))
