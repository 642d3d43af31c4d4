"""What a workspace held before a call decides nothing: the triangle attention (dense, fused output,
block-sparse) leaves q, k and v of the attention rows past N unwritten and still multiplies them, and
its padding bias is written by two kernels.  A workspace of NaNs (0xFF bytes) gives the bits of one of zeros."""
import pytest
import torch

from sparsefold_amd import _lib
from sparsefold_amd import workloads as W
from sparsefold_amd.backends.hip import ops
from tests.test_gpu_modules import DEV, _prepared, hip_backend   # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu
# one row, a key past a 64-key tile, whole tiles with a padding tile after them, a query past a block of 128
SIZES = [1, 63, 64, 65, 127, 129, 192, 200, 300]


def _weights(hip):
  return hip._hip_ln_w, hip._hip_ln_b, hip._hip_w_qkvgb, hip._hip_w_o


def _same_bits(call, nbytes):
  outs = []
  for fill in (0, 255):
    ws = torch.full((nbytes,), fill, dtype=torch.uint8, device=DEV)
    out = call(ws)
    torch.cuda.synchronize()
    outs.append(out if isinstance(out, tuple) else (out,))
  for zeros, nans in zip(*outs):
    assert bool(torch.isfinite(zeros.float()).all())
    assert torch.equal(zeros, nans)


@pytest.mark.parametrize("N", SIZES)
@pytest.mark.parametrize("C", [64, 128])
@pytest.mark.parametrize("transpose", [False, True])
@pytest.mark.parametrize("limit", [0.0, 1.0])            # 1: every (row, head) goes to the exact fix-up
def test_triangle_attention(N, C, transpose, limit):
  mod, z, seq = W.make_triangle(N, C=C, transpose=transpose, padded=N > 32, seed=N + C, sharp=True)
  hip = _prepared(mod)
  zd, sd = z.to(DEV), seq.to(DEV)
  stages = [_lib.TRI_STAGE_ALL] + ([_lib.TRI_STAGE_ALL | _lib.TRI_STAGE_FUSE] if C == 128 else [])
  for s in stages:
    _same_bits(lambda ws: ops.triangle_attention(zd, sd, *_weights(hip), num_head=4, transpose=transpose, stages=s,
                                                 workspace=ws, fixup_sum_limit=limit),
               ops.triangle_workspace_bytes(N, C, 4, C // 4))


@pytest.mark.parametrize("N", SIZES)
@pytest.mark.parametrize("transpose", [False, True])
@pytest.mark.parametrize("samples", [2, 16])             # fewer than the key blocks of the larger sizes, and more
def test_block_sparse_triangle_attention(N, transpose, samples):
  mod, z, seq = W.make_triangle(N, transpose=transpose, padded=N > 32, seed=3 * N, sharp=True)
  hip = _prepared(mod)
  zd, sd = z.to(DEV), seq.to(DEV)
  _same_bits(lambda ws: ops.triangle_attention_ibs(zd, sd, *_weights(hip), num_head=4, transpose=transpose, num_samples=samples,
                                                   num_rand_blocks=1, t_prob=0.5, tr_prob=0.9, u_prob=0.1, seed=5, workspace=ws),
             ops.triangle_ibs_workspace_bytes(N, 128, 4, 32))
