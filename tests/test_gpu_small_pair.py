"""Triangle attention and triangle multiplication around the sizes that run the split projection and
output stages (up to 512 items of 32 positions: 128 tokens) and the first past them, against the
oracle.  Tolerances are the modules' own: bf16 rounding of operands and result, 2% of the largest
update."""
import pytest
import torch

from oracle import modules as OM
from sparsefold_amd import workloads as W
from tests._metrics import assert_close_bf16
from tests.test_gpu_modules import DEV, _params, _prepared, hip_backend   # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu
# one item, an exact block of 32 positions and one past it, the last split size and the first unsplit one
SIZES = [1, 31, 32, 33, 127, 128, 129]


@pytest.mark.parametrize("N", SIZES)
@pytest.mark.parametrize("C", [64, 128])
@pytest.mark.parametrize("transpose", [False, True])
def test_triangle_attention(N, C, transpose):
  mod, z, seq = W.make_triangle(N, C=C, H=4, transpose=transpose, padded=N > 32, seed=N + C, sharp=True, act_norm_bias=True)
  hip = _prepared(mod)
  zd, sd = z.to(DEV), seq.to(DEV)
  upd = hip(zd, sd, add_residual=False)
  ref = OM.grid_self_attention(z.float(), seq, _params(hip), transpose=transpose, return_update=True)
  assert_close_bf16(upd, ref, f"triangle N={N} C={C}", max_abs=2e-2 * max(1.0, ref.abs().max().item()))
  assert_close_bf16(hip(zd, sd), OM.grid_self_attention(z.float(), seq, _params(hip), transpose=transpose), f"triangle N={N} C={C}")


@pytest.mark.parametrize("N", SIZES)
@pytest.mark.parametrize("incoming", [False, True])
def test_triangle_multiplication(N, incoming):
  mod, z, mask = W.make_trimul(N, incoming=incoming, padded=N > 32, seed=7 + N)
  hip = _prepared(mod)
  zd, md = z.to(DEV), None if mask is None else mask.to(DEV)
  upd = hip(zd, md, add_residual=False)
  ref = OM.triangle_multiplication(z.float(), mask, _params(hip), equation=mod.EQUATIONS[int(incoming)], return_update=True)
  assert_close_bf16(upd, ref, f"trimul N={N}", max_abs=2e-2 * max(1.0, ref.abs().max().item()))
  assert torch.equal(hip(zd, md), (upd.float() + zd.float()).to(z.dtype))
