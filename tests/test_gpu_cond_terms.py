"""AdaLN conditioning terms of one layer (scale, shift, zero gate in one launch): the condition width
known when the kernel is compiled (384), the other allowed ones, and the ends of a 64-row block."""
import pytest
import torch

from oracle import modules as OM
from sparsefold_amd import workloads as W
from tests._metrics import assert_close_bf16
from tests.test_gpu_modules import DEV, _params, _prepared, hip_backend   # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("C_cond", [16, 128, 368, 384])
@pytest.mark.parametrize("N", [1, 63, 64, 65])
def test_diffusion_attention_condition_widths(C_cond, N):
  mod, x, cond, bias, mask = W.make_diffusion(N, S=2, C_cond=C_cond, seed=N + C_cond, sharp=True)
  hip = _prepared(mod)
  out = hip(x.to(DEV), mask.to(DEV), pair_logits=bias.to(DEV), single_cond=cond.to(DEV), add_residual=False)
  ref = OM.self_attention(x.float(), mask, _params(hip), pair_logits=bias.float(), single_cond=cond.float(), return_update=True)
  assert_close_bf16(out, ref, f"diffusion attention N={N} Cs={C_cond}", max_abs=2e-2 * max(1.0, ref.abs().max().item()))
