"""CPU model of the operand layouts and the global / LDS accesses of the dense triangle attention
fast path (csrc/triangle.hip: tri_fold_kernel's padding bias, tri_proj_kernel and its split form,
tri_attn_kernel, tri_fixup_kernel, tri_out_kernel and its split form) for both of its instances --
KC = 2 (C = 128, head dim 32) and KC = 1 (C = 64, head dim 16) -- checked against the buffers the host
carves.
The index expressions are the kernels' own, restated; nothing here runs on a GPU."""
import numpy as np
import pytest

from sparsefold_amd import _lib

H = 4
KT, TR, AW = 64, 4, 8                         # keys per tile, rows per task, waves per workgroup


def _np(n):
  return (n + 127) & ~127


def _ql_off(KC, r, h, NP, p, kk, hf):
  return ((((r * H + h) * (NP >> 5) + (p >> 5)) * (2 * KC) + kk * 2 + hf) * 256 + (p & 31) * 8)


def _vl_off(KC, r, h, NP, c16, hf, d):
  return ((((r * H + h) * (NP >> 4) + c16) * 2 + hf) * (128 * KC) + d * 8)


def _o_off(KC, h, r, i, hf, kk, N, NP):
  return ((((h * N + r) * (NP >> 5) + (i >> 5)) * (512 * KC)) + ((((KC * hf + kk) << 5) + (i & 31)) << 3))


def _bias_pos64(j):
  j32 = j & 31
  return (j & 32) + 16 * ((j32 >> 2) & 1) + 4 * (j32 >> 3) + (j32 & 3)


def _bias_off(h, i, j, NP):
  js = (j & ~63) + _bias_pos64(j & 63)
  jp, pc = js & 63, (js & 63) >> 3
  k, hf = 2 * (pc >> 2) + (pc & 1), (pc >> 1) & 1
  return ((((h * (NP >> 5) + (i >> 5)) * (NP >> 6) + (js >> 6)) << 11) + ((k * 64 + 32 * hf + (i & 31)) << 3) + (jp & 7))


@pytest.mark.parametrize("KC", [1, 2])
def test_operand_layouts_are_bijections(KC):
  """Q/K, V^T and o: every (row, head, position, dim group) has its own 8-element slot, and the
  slots tile the buffers with no gap."""
  D, NP, N = 16 * KC, 128, 100
  q = np.array([_ql_off(KC, r, h, NP, p, kk, hf) for r in range(3) for h in range(H) for p in range(NP)
                for kk in range(KC) for hf in range(2)])
  assert len(set(q.tolist())) == len(q) and q.max() + 8 == 3 * H * NP * D and (q % 8 == 0).all()
  v = np.array([_vl_off(KC, r, h, NP, c, hf, d) for r in range(3) for h in range(H) for c in range(NP // 16)
                for hf in range(2) for d in range(D)])
  assert len(set(v.tolist())) == len(v) and v.max() + 8 == 3 * H * NP * D
  o = np.array([_o_off(KC, h, r, i, hf, kk, N, NP) for h in range(H) for r in range(N) for i in range(0, NP, 1)
                for hf in range(2) for kk in range(KC)])
  assert len(set(o.tolist())) == len(o) and o.max() + 8 == H * N * NP * D
  # a 64-key tile of one row is 2 KC KB of contiguous K (and of V^T): the attention kernel's
  # 1 KB copies at j0 * 32 KC bytes past the row's base
  for j0 in (0, 64, NP - 64):
    ks = {_ql_off(KC, 1, 2, NP, p, kk, hf) for p in range(j0, j0 + 64) for kk in range(KC) for hf in range(2)}
    base = _ql_off(KC, 1, 2, NP, 0, 0, 0) + j0 * 16 * KC
    assert ks == set(range(base, base + 1024 * KC, 8))
    vs = {_vl_off(KC, 1, 2, NP, c, hf, d) for c in range(j0 // 16, j0 // 16 + 4) for hf in range(2) for d in range(D)}
    vb = _vl_off(KC, 1, 2, NP, 0, 0, 0) + j0 * 16 * KC
    assert vs == set(range(vb, vb + 1024 * KC, 8))


@pytest.mark.parametrize("KC", [1, 2])
def test_lds_tile_reads_match_the_copies(KC):
  """The K and V^T operand reads of a tile hit the 16-byte slots the copies filled with the
  wanted key / dim: K slot (rr, kb, kk, half, li) holds key 32 kb + li, k-chunk kk, lane half
  half of row rr; V^T slot (rr, c16, half, li) holds dim li (li mod 16 for KC = 1)."""
  row_bytes = KT * 16 * KC * 2
  k_bytes = TR * row_bytes
  cpw = 2 * k_bytes // 1024 // AW
  assert cpw == 2 * KC
  # copy: wave w chunk u -> LDS bytes (w cpw + u) KB; source = row (w mod 4) of K (w < 4) or V^T
  # (w >= 4), bytes u KB .. of that row's tile; lane L -> 16 L
  filled = {}
  for w in range(AW):
    for u in range(cpw):
      for L in range(64):
        filled[(w * cpw + u) * 1024 + 16 * L] = ("K" if w < 4 else "V", w % 4, u * 1024 + 16 * L)
  assert max(filled) + 16 <= 2 * k_bytes
  for rr in range(TR):
    for kb in range(2):
      for kk in range(KC):
        for half in range(2):
          for li in range(32):
            slot = rr * row_bytes + (kb * 2 * KC + kk * 2 + half) * 512 + li * 16
            src, row, off = filled[slot]
            # offset within the row's tile of K [key block][k-chunk][half][key 32][16 B]
            assert (src, row) == ("K", rr)
            assert off == ((kb * 2 * KC + kk * 2 + half) * 32 + li) * 16
    for c16 in range(4):
      for half in range(2):
        for li in range(32):
          d = li if KC == 2 else li & 15
          slot = k_bytes + rr * row_bytes + (c16 * 2 + half) * 256 * KC + d * 16
          src, row, off = filled[slot]
          assert (src, row) == ("V", rr)
          assert off == ((c16 * 2 + half) * 16 * KC + d) * 16


@pytest.mark.parametrize("KC", [1, 2])
@pytest.mark.parametrize("N", [1, 37, 65, 257, 768])
def test_fast_path_accesses_stay_in_bounds(KC, N):
  D, C = 16 * KC, 64 * KC
  NP = _np(N)
  E = NP * NP * H * D                       # elements of each of Q, K, V^T
  EO = N * NP * H * D                       # elements of o
  EB = NP * NP * H                          # bias elements
  lane = np.arange(64)
  half, li = lane >> 5, lane & 31
  # workspace: the host's size covers Q, K, V^T, bias and o (each rounded to 256 bytes) plus the
  # folded weight, offsets, flags and counters
  ws = int(_lib.load().sf_hip_triangle_workspace_bytes(N, C, H, D))
  assert ws >= 3 * 2 * E + 2 * EB + 2 * EO + (4 * C + 32) * C * 2
  # projection: rows r < N, positions p < NP; Q/K stores of head hd (16 bytes), V^T stores (the
  # attention kernel reads the rows up to NP: below)
  r, p = N - 1, NP - 1
  for hd in range(H):
    for kk in range(KC):
      assert _ql_off(KC, r, hd, NP, p, kk, 1) + 8 <= E
    assert _vl_off(KC, r, hd, NP, NP // 16 - 1, 1, D - 1) + 8 <= E
  assert max(_bias_off(H - 1, NP - 1, j, NP) for j in range(NP - 64, NP)) < EB
  # attention: persistent tasks (head, row group, block of 256 queries); K / V^T copies of the
  # last tile of the last row, the bias loads of the last query tile, Q of the last query
  r0 = NP - TR
  for w in range(AW):
    rr = w % 4
    base = _ql_off(KC, r0 + rr, H - 1, NP, 0, 0, 0) if w < 4 else _vl_off(KC, r0 + rr, H - 1, NP, 0, 0, 0)
    j0 = NP - KT
    hi = base + j0 * 16 * KC + (2 * KC - 1) * 512 + lane.max() * 8 + 8
    assert hi <= E
  qt = NP // 32 - 1
  bias_base = ((H - 1) * (NP >> 5) + qt) * (NP >> 6) << 11
  assert bias_base + (NP - KT) * 32 + 3 * 512 + lane.max() * 8 + 8 <= EB
  for rr in range(TR):
    for kk in range(KC):
      assert _ql_off(KC, r0 + rr, H - 1, NP, NP - 1, kk, 1) + 8 <= E
  # o stores (rows r < N, queries i < N) and the output stage's o reads
  for kk in range(KC):
    assert _o_off(KC, H - 1, N - 1, N - 1, 1, kk, N, NP) + 8 <= EO
  for ch in range(C // 16):
    hd, hf, k2 = (ch >> 1, ch & 1, 1) if KC == 2 else (ch, 1, 0)
    assert _o_off(KC, hd, N - 1, N - 1, hf, k2, N, NP) + 8 <= EO
  # output stage: a block of 32 queries (i0 = 32 ib < N) stores rows i0 + min(row, N - 1 - i0),
  # the rows past N storing the block's last valid row again (no branch around the stores)
  for i0 in range(0, N, 32):
    for row in range(32):
      ro = i0 + min(row, N - 1 - i0)
      assert 0 <= ro < N and (ro == i0 + row or i0 + row >= N)
  # fix-up: mean of V over every 16-key chunk (parts pp of 256 / D threads, 4 chunks per pass)
  npart = 256 // D
  chunks = set()
  for pp in range(npart):
    for c0 in range(pp, NP // 16, npart * 4):
      for u in range(8):
        c16 = c0 + npart * (u >> 1)
        if c16 < NP // 16:
          chunks.add(c16)
          assert _vl_off(KC, N - 1, H - 1, NP, c16, u & 1, D - 1) + 8 <= E
  assert chunks == set(range(NP // 16))


# ---- the bias of the padding: filled by the fold kernel, the rest written by the projection ----

def _fill(N, NP, transpose):
  """fill_padding_bias: (query, key) and value (-1: -inf, 0) of every element of one head's pieces."""
  q0, pc0 = (0, (N >> 6) * 8) if transpose else (N, 0)
  pcs = NP // 8 - pc0
  f = np.arange((NP - q0) * pcs)
  js, i = 8 * (pc0 + f % pcs), q0 + f // pcs
  e = np.arange(8)
  s0 = (js[:, None] & 63) + e
  j = (js[:, None] & ~63) + (s0 & 32) + 8 * ((s0 >> 2) & 3) + 4 * ((s0 >> 4) & 1) + (s0 & 3)
  assert (_bias_pos64(j & 63) == s0).all()               # the stored position inverted
  return np.broadcast_to(i[:, None], j.shape), j, np.where(j >= N, -1, 0)


@pytest.mark.parametrize("transpose", [False, True])
@pytest.mark.parametrize("N", [1, 31, 32, 37, 63, 64, 65, 96, 127, 128, 129, 192, 200, 257])
def test_fill_and_projection_cover_the_bias(N, transpose):
  """-inf for keys past N, 0 for the valid keys of queries past N, the projection's values (and the
  masked logit) elsewhere: every element written, in that order of kernels, and none outside."""
  NP = _np(N)
  unset, pad, zero, value = 0, 1, 2, 3
  state = np.full((NP, NP), unset)                       # [query][key]
  if N != NP:
    i, j, v = _fill(N, NP, transpose)
    assert i.min() >= 0 and i.max() < NP and j.min() >= 0 and j.max() < NP
    state[i, j] = np.where(v == -1, pad, zero)
  # items of 32 positions p of rows r < N: query r, key p (starting node) or query p, key r
  r, p = np.meshgrid(np.arange(N), np.arange(NP), indexing="ij")
  za, zb = (p, r) if transpose else (r, p)
  state[za, zb] = np.where(zb >= N, pad, np.where(za >= N, zero, value))
  i, j = np.meshgrid(np.arange(NP), np.arange(NP), indexing="ij")
  assert np.array_equal(state, np.where(j >= N, pad, np.where(i >= N, zero, value)))
  # and the offsets of a head are a permutation of its plane
  off = np.array([_bias_off(1, a, b, NP) for a, b in ((0, 0), (NP - 1, NP - 1))])
  assert (off >= NP * NP).all() and (off < 2 * NP * NP).all()


@pytest.mark.parametrize("NP", [128, 256])
def test_bias_offsets_are_a_permutation(NP):
  i, j = np.meshgrid(np.arange(NP), np.arange(NP), indexing="ij")
  off = np.concatenate([_bias_off(h, i, j, NP).ravel() for h in range(2)])
  assert np.array_equal(np.sort(off), np.arange(2 * NP * NP))


# ---- the split projection and output stages (up to 512 items) ----

@pytest.mark.parametrize("N", [1, 2, 31, 33, 64, 65, 100, 127, 128])
def test_split_projection_takes_every_item_once(N):
  """Grid (items / 4, 4 parts), a wave per item, no test for the end: the items are a multiple of 4."""
  NP = _np(N)
  items, bpr = N * (NP // 32), NP // 32
  assert items <= 512 and items % 4 == 0
  item = (np.arange(items // 4)[:, None] * 4 + np.arange(4)).ravel()
  r, p0 = item // bpr, (item % bpr) * 32
  assert r.max() < N and p0.max() + 32 <= NP
  assert np.unique(r * NP + p0).size == items
  for transpose in (False, True):
    p = p0[:, None] + np.arange(32)
    za, zb = (p, r[:, None]) if transpose else (r[:, None], p)
    valid = (za < N) & (zb < N)
    assert int(np.where(valid, za * N + zb, 0).max()) < N * N      # z and, by zb, the mask


@pytest.mark.parametrize("KC", [1, 2])
def test_split_projection_staging(KC):
  """Part y's folded rows (q, k, v: C rows; bias: 32, the last repeated) and their place in LDS."""
  C, cols = 64 * KC, (4 * 2 * KC + 1) * 32
  stage = C * (C // 8) // 256
  t = np.arange(256)[:, None] + 256 * np.arange(stage)[None, :]
  for part in range(4):
    rows, src = (32, 4 * C) if part == 3 else (C, C * part)
    n = np.minimum(t // (C // 8), rows - 1)
    assert (src + n).max() < cols and ((src + n) * C + (t % (C // 8)) * 8 + 7).max() < cols * C
    assert rows <= 256 and src + rows <= cols
  assert np.array_equal(np.unique(t // (C // 8)), np.arange(C))    # every LDS row is stored
  assert (C - 1) * (C + 8) + C <= C * (C + 8)


@pytest.mark.parametrize("KC", [1, 2])
@pytest.mark.parametrize("N", [1, 31, 32, 33, 100, 127, 128])
def test_split_output_writes_every_position_once(KC, N):
  NB, C, NP = 2 * KC, 64 * KC, _np(N)
  ib = (N + 31) >> 5
  items = N * ib
  assert items <= 512
  lane = np.arange(64)
  count = np.zeros((N, N, C // 8), np.int64)
  for b in range(items):
    r, i0 = b // ib, (b % ib) * 32
    li = lane & 31
    i = np.where(i0 + li < N, i0 + li, 0)                          # lanes past N read query 0
    for wave in range(NB):
      for j in range(2):                                           # o pieces 2 wave + j of the item
        hd, hf, kk = _piece(KC, 2 * wave + j, lane >> 5)
        assert (_o_off(KC, hd, r, i, hf, kk, N, NP) + 8 <= H * N * NP * 16 * KC).all()
      for u in range(2):
        row, ch = 16 * u + (lane >> 2), (lane & 3) * 8
        keep = i0 + row < N
        np.add.at(count, (np.full(64, r)[keep], (i0 + row)[keep], (32 * wave + ch)[keep] // 8), 1)
  assert (count == 1).all()
  # the waves' output rows (pitch 36) lie where W_g was, the gated o operands hold NC x 64 lanes x 8
  assert NB * 32 * 36 <= C * (C + 8) and (2 * (NB - 1) + 1) * 64 * 8 + 63 * 8 + 8 <= (C // 16) * 64 * 8


def _piece(KC, chunk, half):
  """Head, piece and k-chunk of the output operand's 16-feature chunk for lane half `half`."""
  if KC == 2:
    return chunk >> 1, chunk & 1, half
  return chunk, half, 0
