"""The 256 x 256-tile GEMM behind sf_hip_linear_fwd (csrc/linear_pp.hip).

CPU: its tile order, the addresses of its copies and stores at the operands' edges, the LDS layout of a
step (what the copies write against what the operand reads fetch) and the epilogue's private block,
restated from the kernel.  GPU: parity with an fp32
product at the edges of its tiles and of its K steps, every epilogue, and the calls that must stay
on the general kernels (an update in place).  Which kernel a call takes is asked of the library."""
import ctypes

import numpy as np
import pytest
import torch

TILE, BAND = 256, 5


@pytest.mark.parametrize("gx,gy,batch", [(1, 1, 1), (20, 12, 1), (15, 12, 1), (16, 13, 1), (20, 17, 1), (3, 3, 128), (2, 2, 128), (7, 1, 9)])
def test_every_tile_is_taken_once(gx, gy, batch):
  total = gx * gy * batch
  t = np.arange(total)
  bz = t // (gx * gy)
  r = t - bz * gx * gy
  band = r // (BAND * gy)
  q = r - band * BAND * gy
  bh = np.minimum(BAND, gx - band * BAND)
  by = q // bh
  bx = band * BAND + q - by * bh
  assert (bx >= 0).all() and (bx < gx).all() and (by < gy).all() and (bz < batch).all()
  assert np.unique(bx + gx * (by + gy * bz)).size == total
  # the workgroups' walks: XCD ranges of ceil(total / 8), each dealt over the XCD's workgroups
  grid = min(256, (total + 7) // 8 * 8)
  per, seen = (total + 7) // 8, np.zeros(total, int)
  for b in range(grid):
    tile, end = (b & 7) * per + (b >> 3), min(total, ((b & 7) + 1) * per)
    while tile < end:
      seen[tile] += 1
      tile += grid >> 3
  assert (seen == 1).all()


def test_step_layout_and_bank_groups():
  """A chunk's lanes write (row, piece) where the operand reads of that row and piece look, and the 16
  lanes served together read 16 different 16-byte columns of the 256-byte bank span."""
  lane = np.arange(64)
  crow, cpiece = lane >> 2, (lane & 3) ^ ((lane >> 4) & 3)
  where = {}
  for chunk in range(TILE // 16):
    for l in range(64):
      where[(16 * chunk + crow[l], cpiece[l])] = chunk * 1024 + 16 * l
  half, li = lane >> 5, lane & 31
  for block in range(TILE // 32):
    for kk in range(2):
      addr = (block * 2048 + li * 64 + (half ^ ((li >> 2) & 3)) * 16) ^ (32 * kk)
      for l in range(64):
        assert addr[l] == where[(32 * block + li[l], 2 * kk + half[l])]
      for g in range(4):
        assert np.unique(addr[16 * g:16 * g + 16] % 256).size == 16


@pytest.mark.parametrize("M,N,K,pad", [(256, 256, 128, 0), (3850, 3080, 192, 0), (300, 272, 128, 8), (4097, 3576, 256, 64), (257, 8, 320, 0)])
def test_copies_stay_inside_the_operands(M, N, K, pad):
  """Every 16-byte piece a step's copies read, at the tiles on the operands' edges: rows past the end
  read the last row, 32-bit lane offsets, x rows at a stride of K + pad."""
  lane = np.arange(64)
  crow, cpiece = lane >> 2, (lane & 3) ^ ((lane >> 4) & 3)
  for rows, rs, waves in ((M, K + pad, range(4)), (N, K, range(4, 8))):
    size = ((rows - 1) * rs + K) * 2
    pieces = set()
    for b in range((rows + TILE - 1) // TILE):
      r0 = b * TILE
      lastr = rows - 1 - r0
      for wave in waves:
        for u in range(4):
          local = np.minimum(16 * ((wave % 4) * 4 + u) + crow, lastr)
          vo = local * 2 * rs + cpiece * 16
          assert (vo >= 0).all() and (vo < 1 << 32).all()
          for t in range(K // 32):
            at = r0 * rs * 2 + vo + t * 64
            assert (at + 16 <= size).all()
            pieces.update(zip((r0 + local).tolist(), (4 * t + cpiece).tolist()))
    assert pieces == {(r, p) for r in range(rows) for p in range(K // 8)}     # every piece of every row


@pytest.mark.parametrize("glu", [False, True])
@pytest.mark.parametrize("M,N", [(256, 256), (300, 272), (129, 16), (511, 1040), (257, 528)])
def test_stores_cover_the_result(M, N, glu):
  """Rows past the end store the last row again, columns past the end the last valid piece, a wave with no
  column nothing: inside the result, each lane the element its data belongs to, all of it."""
  ncols, rb = (N // 2, 64) if glu else (N, 128)
  rp = rb // 16
  lane = np.arange(64)
  written = np.zeros((M, ncols), np.int64)
  for bx in range((M + TILE - 1) // TILE):
    for by in range((N + TILE - 1) // TILE):
      for wave in range(8):
        m0, n0 = bx * TILE + 128 * (wave // 4), by * TILE + 64 * (wave % 4)
        nc0 = n0 // 2 if glu else n0
        if nc0 >= ncols:
          continue
        pc = np.minimum(lane % rp, (ncols - nc0) // 8 - 1)
        for mb in range(4):
          for i in range(32 // (64 // rp)):
            m = np.minimum(m0 + 32 * mb + i * (64 // rp) + lane // rp, M - 1)
            assert (pc >= 0).all() and (nc0 + 8 * pc + 7 < ncols).all()
            for e in range(8):
              np.add.at(written, (m, nc0 + 8 * pc + e), 1)
  assert (written >= 1).all()


@pytest.mark.parametrize("rb", [128, 64])
def test_epilogue_block_is_a_permutation(rb):
  row, piece = np.meshgrid(np.arange(32), np.arange(rb // 16), indexing="ij")
  slot = row * rb + ((piece ^ ((row * rb >> 8) & (rb // 16 - 1))) << 4)
  assert np.array_equal(np.sort(slot.ravel()), np.arange(32 * rb // 16) * 16)


def _args(M, N, K, *, x=1 << 32, wt=2 << 32, y=3 << 32, batch=0, **over):
  """Arguments for the route query; the addresses are never dereferenced."""
  from sparsefold_amd import _lib
  a = _lib.LinearArgs()
  a.M, a.N, a.K, a.mul_rows, a.batch = M, N, K, 1, batch
  a.x, a.x_rs, a.wt, a.y, a.y_rs = x, K, wt, y, N
  if batch > 1:
    a.x_bs, a.w_bs, a.y_bs = M * K, N * K, M * N
  for key, value in over.items():
    setattr(a, key, value)
  return a


def _large_tiles(a):
  from sparsefold_amd import _lib
  return bool(_lib.load().sf_hip_linear_large_tiles(ctypes.byref(a)))


# (M, N, K) of the parity cases: whole tiles; remainders of rows and columns (8 the smallest); the fewest K
# steps; several tiles to a workgroup, the last round partly filled
SHAPES = [(5120, 3072, 768), (3850, 3080, 192), (5000, 4104, 128), (6400, 6152, 448), (4097, 3576, 256)]


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_route_of_the_parity_shapes(M, N, K):
  assert _large_tiles(_args(M, N, K))
  assert _large_tiles(_args(M, N // 16 * 16, K, glu=1, y_rs=N // 16 * 8))
  rows = 4 << 32
  assert _large_tiles(_args(M, N, K, residual=rows, r_rs=N))
  assert not _large_tiles(_args(M, N, K, y=rows, residual=rows, r_rs=N))       # in place
  assert not _large_tiles(_args(M, N, K, y=rows, mul=rows + 2 * N * (M - 1), mul_rs=N))
  # rows that are no whole number of 16-byte pieces, another output form, too few K steps
  for over in ({"y": (3 << 32) + 2}, {"y_rs": N + 4}, {"yt": 5 << 32}, {"ycols": 8}, {"bias": (6 << 32) + 4}):
    assert not _large_tiles(_args(M, N, K, **over)), over
  assert not _large_tiles(_args(M, N, 64)) and not _large_tiles(_args(M, N, K + 8))


@pytest.mark.parametrize("n,large", [(256, False), (257, False), (300, False), (344, False), (384, False),
                                     (392, True), (436, True), (511, True), (600, True), (768, True), (1024, True)])
def test_route_of_batched_products(n, large):
  """128 planes of n x n: between one and one and a half tiles a side (257 .. 384) the smaller tiles win."""
  assert _large_tiles(_args(n, (n + 7) // 8 * 8, (n + 63) // 64 * 64, batch=128)) == large


@pytest.mark.parametrize("M,N,K,large", [(3700, 3072, 768, True), (6000, 1536, 384, True), (65536, 264, 768, True),
                                         (5120, 768, 768, False), (1000, 3072, 768, False), (33000, 264, 768, False)])
def test_route_of_single_products(M, N, K, large):
  assert _large_tiles(_args(M, N, K)) == large


def _check(y, ref, what):
  """bf16 rounding of the result (2^-8 of its value, half a step and the sum's fp32 error with it)."""
  err = (y.float() - ref).abs()
  bound = ref.abs() * 2.0 ** -8 + 1e-3 * ref.square().mean().sqrt()
  assert bool((err <= bound).all()), f"{what}: {int((err > bound).sum())} values off, worst {float((err - bound).max()):.3e}"


def _inputs(M, N, K, seed=3):
  g = torch.Generator(device="cuda").manual_seed(seed)
  r = lambda *s: torch.randn(*s, generator=g, device="cuda")
  return (r(M, K).bfloat16(), (r(N, K) / K ** 0.5).bfloat16(), r(N), r(M, N).bfloat16(), r(96, N).bfloat16())


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("epilogue", ["plain", "bias", "sigmoid_mul", "mul_residual", "glu"])
def test_parity(M, N, K, epilogue):
  from sparsefold_amd import _lib
  from sparsefold_amd.backends.hip import ops
  x, w, b, res, mul = _inputs(M, N, K)
  assert _large_tiles(_args(M, N, K))
  ref = x.float() @ w.float().t()
  if epilogue == "plain":
    _check(ops.linear(x, w), ref, epilogue)
  elif epilogue == "bias":
    _check(ops.linear(x, w, b), ref + b, epilogue)
  elif epilogue == "sigmoid_mul":
    rows = torch.arange(M, device="cuda") % 96
    _check(ops.linear(x, w, b, post_sigmoid=True, mul=mul), torch.sigmoid(ref + b) * mul.float()[rows], epilogue)
  elif epilogue == "mul_residual":
    rows = torch.arange(M, device="cuda") % 96
    _check(ops.linear(x, w, mul=mul, residual=res), ref * mul.float()[rows] + res.float(), epilogue)
  else:
    n = N // 16 * 16
    y = torch.empty(M, n // 2, dtype=torch.bfloat16, device="cuda")
    a = _lib.LinearArgs()
    a.M, a.N, a.K, a.mul_rows, a.glu = M, n, K, 1, 1
    a.x, a.x_rs, a.wt = x.data_ptr(), K, w.data_ptr()
    a.y, a.y_rs = y.data_ptr(), n // 2
    assert _large_tiles(a)
    _lib.check(_lib.load().sf_hip_linear_fwd(ctypes.byref(a), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)), "linear")
    h = ref[:, :n]
    _check(y, torch.nn.functional.silu(h[:, 0::2]) * h[:, 1::2], epilogue)


@pytest.mark.gpu
def test_update_in_place_adds_its_residual_once():
  from sparsefold_amd import _lib
  M, N, K = 3850, 3080, 192
  x, w, _, res, _ = _inputs(M, N, K)
  ref = x.float() @ w.float().t() + res.float()
  a = _lib.LinearArgs()
  a.M, a.N, a.K, a.mul_rows = M, N, K, 1
  a.x, a.x_rs, a.wt = x.data_ptr(), K, w.data_ptr()
  a.y, a.y_rs, a.residual, a.r_rs = torch.empty_like(res).data_ptr(), N, res.data_ptr(), N
  assert _large_tiles(a)
  a.y = res.data_ptr()
  assert not _large_tiles(a)
  _lib.check(_lib.load().sf_hip_linear_fwd(ctypes.byref(a), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)), "linear")
  _check(res, ref, "in place")


@pytest.mark.gpu
@pytest.mark.parametrize("N", [300, 436, 511, 768])
def test_products_of_the_triangle_multiplication(N):
  """The batched form (a plane per channel, several tiles to a workgroup), sizes whose rows are not a
  whole number of pieces, against the 64-bit update; 300 is the largest listed that takes smaller tiles."""
  assert _large_tiles(_args(N, (N + 7) // 8 * 8, (N + 63) // 64 * 64, batch=128)) == (N > 384)
  from oracle import modules as OM
  from sparsefold_amd import workloads as W
  from sparsefold_amd import modules as M
  from sparsefold_amd.backends.hip import modules as HM
  mod, z, mask = W.make_trimul(N, padded=True, incoming=bool(N % 2), seed=N)
  hip = HM.TriangleMultiplicationHip(mod.config, M.GlobalConfig(), num_channels=128)
  hip.load_state_dict(mod.state_dict())
  hip = hip.cuda()
  hip.prepare_native()
  out = hip(z.cuda(), mask.cuda())
  p = {k: v.cuda().bfloat16().float() if v.ndim == 2 else v.cuda() for k, v in mod.state_dict().items()}
  ref = OM.triangle_multiplication(z.cuda().float(), mask.cuda(), p, equation=mod.equation)
  rel = ((out.float() - ref).norm() / ref.norm()).item()
  assert rel <= 1e-2, rel
