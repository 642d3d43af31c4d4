"""CPU model of every global memory access of the triangle multiplicative update's kernels
(csrc/trimul.hip: the prologue, the batched NT product through the library's GEMM, the epilogue)
and of the host's launch arithmetic, checked against the buffer sizes the host allocates, for both
edges and sizes on both sides of each choice: the split prologue and epilogue (up to 512 items of 32
positions, in 8 or 4 parts) and the persistent ones, linear64_kernel and linear_pp_kernel, rows of the
product padded to 8 columns (N = 1, 37, 97, 129, 300, 437) and not, a last block of 32 positions that
is partly past the end.  The index expressions are the kernels' own, restated; nothing here runs on a
GPU."""
import ctypes

import numpy as np
import pytest

from sparsefold_amd import _lib

KC, KTW = 128, 8                 # channels, waves per workgroup of the persistent position kernels
KWS, KTP, KOP = 136, 34, 36      # LDS pitches: weight rows, the staged product block, split output rows
RESIDENT = 256                   # resident workgroups of the position kernels (one per CU)
SPLIT_ITEMS, SPLIT_WAVES = 512, 4
SIZES = [1, 37, 64, 97, 128, 129, 300, 437, 768]


def _pn(n):
  return (n + 63) & ~63


def _cols(n):
  return (n + 7) & ~7


def _pp(n):
  return (n * _cols(n) + 31) & ~31


def _grid(items):
  """launch_grid + the host's items-per-wave / group arithmetic."""
  waves = max(1, min(RESIDENT * KTW, items))
  ipw = (items + waves - 1) // waves
  groups = (items + ipw * KTW - 1) // (ipw * KTW)
  return ipw, groups


def _covered(items, ipw, groups):
  """Every item is processed by exactly one wave: workgroup g's wave w takes items
  g * KTW * ipw + k * KTW + w, k < ipw, until the first one past the end."""
  g, w, k = np.meshgrid(np.arange(groups), np.arange(KTW), np.arange(ipw), indexing="ij")
  item = (g * KTW * ipw + k * KTW + w).ravel()
  return np.array_equal(np.sort(item[item < items]), np.arange(items))


def _proj_parts(items):
  """(first channel row of the parts, blocks of 32 channels in each): blockIdx.y of the split kernel,
  or all 8 blocks in turn."""
  if items > SPLIT_ITEMS:
    return [0], 8
  bpw = 1 if items <= 128 else 2
  return [32 * bpw * y for y in range(8 // bpw)], bpw


@pytest.mark.parametrize("incoming", [False, True])
@pytest.mark.parametrize("N", SIZES)
def test_prologue(N, incoming):
  Pn = _pn(N)
  items, cbs = Pn * (Pn // 32), Pn // 32
  if items > SPLIT_ITEMS:
    assert _covered(items, *_grid(items))
  else:
    assert items % SPLIT_WAVES == 0              # item = 4 blockIdx.x + wave, no test for the end
  item = np.arange(items)[:, None]
  lane = np.arange(64)[None, :]
  half, li = lane >> 5, lane & 31
  R, col = item // cbs, 32 * (item % cbs) + li
  za, zb = (col, R) if incoming else (R, col)
  ok = (za < N) & (zb < N)
  # z reads, every lane (unconditional): 8 x 16 bytes at element (za * N + zb) * 128 + 8 * half
  # + 16 kk, position 0 where not ok; mask[za], mask[zb] likewise
  assert int((np.where(ok, za * N + zb, 0) * KC + 8 * half).max()) + 16 * 7 + 7 < N * N * KC
  assert int(np.where(ok, np.maximum(za, zb), 0).max()) < N
  # plane stores (2 bytes): the uniform base of channel 32 nb + 8 (r / 4) + r % 4 plus the lane offset
  # (4 half plane + R Pn + col): every element of both sides' 128 planes exactly once
  plane = Pn * Pn
  pos = R * Pn + col
  rows, bpw = _proj_parts(items)
  seen = np.zeros(2 * KC, np.int64)              # (side, channel) rows taken by the parts
  lanes = [pos[:, np.flatnonzero(half[0] == h)].ravel() for h in (0, 1)]
  for h in (0, 1):
    assert np.array_equal(np.sort(lanes[h]), np.arange(plane))    # a half's lanes cover a plane once
  for rg in rows:
    for j in range(bpw):
      first = rg + 32 * j                        # gate row of the block: side kC + channel
      side, ch0 = first // KC, first % KC
      assert (rg % KC) + 32 * j < KC or bpw == 8
      for h in (0, 1):
        for r in range(16):
          ch = ch0 + 8 * (r >> 2) + 4 * h + (r & 3)
          seen[side * KC + ch] += 1
          assert 0 <= ch * plane + int(lanes[h].min()) and ch * plane + int(lanes[h].max()) < KC * plane
  assert (seen == 1).all()


@pytest.mark.parametrize("bpw", [1, 2])
def test_split_prologue_staging(bpw):
  """The part's gate and projection rows: every LDS row from its own weight row, no access past either."""
  G = 32 * bpw
  stage = 2 * G * (KC // 8) // 256
  t = np.arange(256)[:, None] + 256 * np.arange(stage)[None, :]
  n, c8 = t >> 4, (t & 15) * 8
  assert np.array_equal(np.unique(n * KC + c8), np.arange(2 * G * KC // 8) * 8)
  for y in range(8 // bpw):
    rg = G * y
    row = (n // G) * 2 * KC + rg + n % G
    assert row.max() < 4 * KC                                       # folded GLU rows
    # LDS row j of the gate half is channel row rg + j, of the projection half 2 kC + rg + j
    assert all(((row == rg + j) == (n == j)).all() and ((row == 2 * KC + rg + j) == (n == G + j)).all() for j in (0, G - 1))
    tid = np.arange(2 * G)
    assert ((tid // G) * 2 * KC + rg + tid % G).max() < 4 * KC
  assert 2 * G <= 256 and (2 * G - 1) * KWS + KC <= bpw * 64 * KWS


def _large_tiles(N):
  a = _lib.LinearArgs()
  a.M, a.N, a.K, a.mul_rows, a.batch = N, _cols(N), _pn(N), 1, KC
  a.x, a.wt, a.y = 1 << 32, 2 << 32, 3 << 32
  a.x_rs, a.y_rs, a.x_bs, a.w_bs, a.y_bs = _pn(N), _cols(N), _pn(N) ** 2, _pn(N) ** 2, _pp(N)
  return bool(_lib.load().sf_hip_linear_large_tiles(ctypes.byref(a)))


@pytest.mark.parametrize("N", SIZES)
def test_product(N):
  """Loads clamp rows to M - 1 / N - 1 of the planes (rows of K = Pn); the product's rows hold Nt
  columns, all of them stored."""
  Pn, Nt = _pn(N), _cols(N)
  assert Nt <= Pn and Pn % 64 == 0                     # the columns past N come from planes' zero rows
  ab, t_elems = KC * Pn * Pn, KC * _pp(N)
  assert (KC - 1) * Pn * Pn + (N - 1) * Pn + Pn - 1 < ab and (KC - 1) * Pn * Pn + (Nt - 1) * Pn + Pn - 1 < ab
  assert (KC - 1) * _pp(N) + (N - 1) * Nt + Nt - 1 < t_elems
  written = np.zeros((N, Nt), np.int64)
  if _large_tiles(N):
    assert N > 384
    # a wave's part: 128 rows x 64 columns in blocks of 32 rows; lane: row 8 i + lane / 8, piece lane % 8,
    # rows past the end the last row, pieces past the end the last valid one (the same bytes again)
    lane = np.arange(64)
    for bx in range((N + 255) // 256):
      for by in range((Nt + 255) // 256):
        for wave in range(8):
          m0, n0 = 256 * bx + 128 * (wave // 4), 256 * by + 64 * (wave % 4)
          if n0 >= Nt:
            continue
          pc = np.minimum(lane % 8, (Nt - n0) // 8 - 1)
          for mb in range(4):
            for i in range(4):
              m = np.minimum(m0 + 32 * mb + 8 * i + lane // 8, N - 1)
              assert (n0 + 8 * pc + 7 < Nt).all() and ((m * Nt + n0 + 8 * pc) % 8 == 0).all()
              for e in range(8):
                np.add.at(written, (m, n0 + 8 * pc + e), 1)
    assert (written >= 1).all()
  else:
    for bm, bn in ((128, 128), (64, 128), (64, 64)):
      gm, gn = (N + bm - 1) // bm, (Nt + bn - 1) // bn
      assert gm * bm >= N and gn * bn >= Nt and gm < 2 ** 31 and KC <= 65535


def _positions(N, items):
  """out_position of the 32 positions of every item: the element of z and out, or -1."""
  p = np.arange(items * 32).reshape(items, 32)
  row, col = p // _cols(N), p % _cols(N)
  return np.where((p < N * _cols(N)) & (col < N), row * N + col, -1)


@pytest.mark.parametrize("N", SIZES)
def test_epilogue(N):
  Pp = _pp(N)
  items = (N * _cols(N) + 31) // 32
  split = items <= SPLIT_ITEMS
  if not split:
    assert _covered(items, *_grid(items))
  pos = _positions(N, items)
  assert np.array_equal(np.sort(pos[pos >= 0]), np.arange(N * N))   # every position of z and out once
  # the product loads, 16 bytes each, whatever the position: channel w / 4, pieces of 8 positions
  threads, loads = (256, 2) if split else (64, 8)
  w = np.arange(threads)[:, None] + threads * np.arange(loads)[None, :]
  c, seg = w >> 2, w & 3
  start = c * Pp + (items - 1) * 32 + 8 * seg
  assert (start % 8 == 0).all() and int(start.max()) + 7 < KC * Pp
  assert np.array_equal(np.sort((c * 32 + 8 * seg).ravel()), np.arange(KC * 32 // 8) * 8)
  # staged at pitch 34 and read back as channels 16 kk + 8 half + 0..7 of position li
  lds = 4 * 32 * KOP if split else 32 * KWS
  assert int((c * KTP + 8 * seg + 7).max()) < lds and ((c * KTP + 8 * seg) % 2 == 0).all()
  assert (16 * 7 + 8 + 2 * 3 + 1) * KTP + 31 < lds
  # z: every lane, position 0 where there is none
  assert int(np.maximum(pos, 0).max()) * KC + 8 + 16 * 7 + 7 < N * N * KC
  if split:
    # residual and output of wave w: channels 32 w + 8 g + 4 half .. + 3, and whole pieces of 8 through LDS
    lane = np.arange(64)
    got = sorted((16 * u + l // 4, 32 * wv + (l % 4) * 8) for wv in range(4) for u in range(2) for l in lane)
    assert got == [(r, 8 * k) for r in range(32) for k in range(16)]
    assert 3 * 32 * KOP + 31 * KOP + 24 + 7 < lds
    assert 32 * 3 + 8 * 3 + 4 + 3 < KC
  else:
    w = np.arange(64)[:, None] + 64 * np.arange(8)[None, :]
    got = sorted(zip((w >> 4).ravel().tolist(), ((w & 15) * 8).ravel().tolist()))
    assert got == [(r, 8 * k) for r in range(32) for k in range(16)]


@pytest.mark.parametrize("N", SIZES)
def test_trimul_workspace_covers_the_modelled_buffers(N):
  lib = _lib.load()
  Pn, Pp = _pn(N), _pp(N)
  need = 2 * KC * Pn * Pn * 2 + KC * Pp * 2 + (4 * KC * KC + 2 * KC * KC) * 2 + 6 * KC * 4
  assert lib.sf_hip_triangle_mult_workspace_bytes(N, KC) >= need


@pytest.mark.parametrize("grid", [(6, 6, 128), (12, 12, 128), (1, 1, 8), (3, 2, 5), (320, 2, 5), (7, 3, 8)])
def test_batched_gemm_tile_remap_is_a_permutation(grid):
  """linear64_kernel's batched tile order (XCD-contiguous ranges when the tile count is a multiple
  of 8, dispatch order otherwise) visits every (x, y, z) tile exactly once."""
  gx, gy, gz = grid
  total = gx * gy * gz
  L = np.arange(total, dtype=np.int64)
  t = (L & 7) * (total >> 3) + (L >> 3) if total % 8 == 0 else L
  bx, by, bz = t % gx, (t // gx) % gy, t // (gx * gy)
  assert np.unique(bx + gx * (by + gy * bz)).size == total and bz.max() < gz
  if total % 8 == 0 and gz % 8 == 0:
    # each XCD (L % 8) holds whole batch members
    for x in range(8):
      members = np.unique(bz[(L & 7) == x])
      assert members.size == gz // 8
