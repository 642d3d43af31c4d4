// Linear (Y = epilogue(X Wt^T)) on large grids, gfx950: sf_hip_linear_fwd's kernel where the grid
// fills the chip with 256 x 256 tiles.
//
// 8 waves (2 x 4, wave tiles of 128 x 64), two per SIMD, K in steps of 32 through a ring of four LDS
// stages, persistent (a workgroup's tiles run through one continuous ring).  The
// waves form two groups of one wave per SIMD that run half a step apart: while one group reads a
// step's operands from LDS, the other group's MFMAs run, so the matrix cores see work while LDS
// latency passes.  One s_barrier separates the halves:
//   slot 2t      early: reads step t, copies step t + A (A = S - 1) | late: MFMAs of step t - 1
//   slot 2t + 1  early: MFMAs of step t                             | late: reads step t, copies step t + A
// Hand-offs (every barrier is met by all waves): the copies of step t + A overwrite the stage of
// step t - 1, whose last reads (late, slot 2t - 1, lgkmcnt(0) inside the reading asm block) end
// before slot 2t; a wave's own copies of step t + 1 are waited for (vmcnt, issue order) before the
// barrier that ends slot 2t + 1, and step t + 1 is read from slot 2t + 2 on.
// LDS stage: rows of 32 k (64 bytes), 16-byte pieces XOR-swizzled by (row / 4) % 4, so that the 16
// lanes whose operand reads are served together cover all 64 banks (two rows per 128-byte line
// swizzled by the line measured half that rate).
// A step's copies go out between its operand reads and the reads' wait: issued ahead of the reads they
// held them back by 500 cycles a slot, and between the MFMAs they stalled those (8192 x 8192 x 1024:
// 159, 141 and 127 us).  The reads and copies are one asm block with the wait inside: before an LDS
// read it can see, the compiler waits for every outstanding direct-to-LDS copy.
// Epilogue: each wave finishes its own part, 32 rows at a time through a private 32-row LDS
// block outside the ring (no barrier): residual and multiplier rows come in as whole 16-byte
// pieces and are read back in the accumulator's layout, the results go out as whole rows.  (fp32
// tiles through LDS and a barrier, as in linear64_kernel, cost 6 to 8 us per 256 x 256 tile.)
//
// Measured against linear64_kernel (random bf16 data, us a call): 8192 x 8192 x 1024 134 against 174,
// 5120 x 3072 x 768 32 against 38, 3700 x 3072 x 768 27 against 35, 128 batched 768^3 148 against 196
// (the triangle multiplication around them 411 against 458).  At 5120 x 3072 x 768 (a tile for each of 240
// workgroups) a workgroup is resident for 47 thousand cycles, and its SIMDs' matrix cores are busy for 24.6
// of them; the rest is first copies, barriers and the result's stores (5 us at the memory's write rate).
#include <algorithm>

#include "sf_common.h"

namespace {

typedef __attribute__((address_space(3))) uint32_t lds_u32;
constexpr int kTile = 256;

template <int N>
__device__ __forceinline__ void pp_wait() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"i"(N) : "memory");
}
// vmcnt(n * CPW), n = the steps that may stay in flight (uniform)
template <int CPW, int MAX>
__device__ __forceinline__ void pp_wait_steps(int n) {
  if (n >= MAX) pp_wait<MAX * CPW>();
  else if constexpr (MAX > 0) pp_wait_steps<CPW, MAX - 1>(n);
}
__device__ __forceinline__ void pp_ds_write8(uint32_t addr, u32x2 v) { asm volatile("ds_write_b64 %0, %1" ::"v"(addr), "v"(v) : "memory"); }
__device__ __forceinline__ void pp_ds_write4(uint32_t addr, uint32_t v) { asm volatile("ds_write_b32 %0, %1" ::"v"(addr), "v"(v) : "memory"); }
__device__ __forceinline__ void pp_ds_write16(uint32_t addr, u32x4 v) { asm volatile("ds_write_b128 %0, %1" ::"v"(addr), "v"(v) : "memory"); }
// four 8-byte reads: the four 8-column groups of one 32-column block
__device__ __forceinline__ void pp_ds_read8x4(const uint32_t (&ad)[4], u32x2 (&v)[4]) {
  asm volatile("ds_read_b64 %0, %4\n\tds_read_b64 %1, %5\n\tds_read_b64 %2, %6\n\tds_read_b64 %3, %7\n\ts_waitcnt lgkmcnt(0)"
               : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]) : "v"(ad[0]), "v"(ad[1]), "v"(ad[2]), "v"(ad[3]) : "memory");
}
template <int N>
__device__ __forceinline__ void pp_ds_read16(const uint32_t (&ad)[N], u32x4 (&v)[N]) {
  if constexpr (N == 4) {
    asm volatile("ds_read_b128 %0, %4\n\tds_read_b128 %1, %5\n\tds_read_b128 %2, %6\n\tds_read_b128 %3, %7\n\ts_waitcnt lgkmcnt(0)"
                 : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]) : "v"(ad[0]), "v"(ad[1]), "v"(ad[2]), "v"(ad[3]) : "memory");
  } else {
    static_assert(N == 2, "2 or 4 reads");
    asm volatile("ds_read_b128 %0, %2\n\tds_read_b128 %1, %3\n\ts_waitcnt lgkmcnt(0)"
                 : "=&v"(v[0]), "=&v"(v[1]) : "v"(ad[0]), "v"(ad[1]) : "memory");
  }
}
// The operands of one step of a wave (MB row blocks and NB column blocks of 32, k-chunks 0 and 1),
// then -- COPY -- the wave's CPW direct-to-LDS copies of a later step, then the wait for the reads:
// the copies go out while the reads return.  m0: LDS address of the first copy (the others follow
// 1 KB apart); sa: the copies' uniform base, vo: their lane offsets.
#define PP_COPY1 "s_mov_b32 m0, %[m0]\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %[v0], %[sa]\n\t"
#define PP_COPYN(V) "s_add_u32 m0, m0, 0x400\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %[" V "], %[sa]\n\t"
#define PP_WAIT "s_waitcnt lgkmcnt(0)"
#define PP_ARGS [a0] "v"(a0), [a1] "v"(a1), [b0] "v"(b0), [b1] "v"(b1)
template <int MB, int NB, int CPW, bool COPY>
__device__ __forceinline__ void pp_read(uint32_t a0, uint32_t a1, uint32_t b0, uint32_t b1, u32x4 (&xa)[2][MB], u32x4 (&wb)[2][NB],
                                        uint32_t m0, const char* sa, const uint32_t (&vo)[CPW]) {
  static_assert(MB == 4 && NB == 2 && CPW == 4, "wave tiles of 128 x 64, four copies a step");
#define PP_READS "ds_read_b128 %0, %[a0]\n\tds_read_b128 %8, %[b0]\n\tds_read_b128 %1, %[a0] offset:2048\n\t" \
                 "ds_read_b128 %9, %[b0] offset:2048\n\tds_read_b128 %2, %[a0] offset:4096\n\tds_read_b128 %3, %[a0] offset:6144\n\t" \
                 "ds_read_b128 %4, %[a1]\n\tds_read_b128 %10, %[b1]\n\tds_read_b128 %5, %[a1] offset:2048\n\t" \
                 "ds_read_b128 %11, %[b1] offset:2048\n\tds_read_b128 %6, %[a1] offset:4096\n\tds_read_b128 %7, %[a1] offset:6144\n\t"
#define PP_OUTS "=&v"(xa[0][0]), "=&v"(xa[0][1]), "=&v"(xa[0][2]), "=&v"(xa[0][3]), "=&v"(xa[1][0]), "=&v"(xa[1][1]), \
                "=&v"(xa[1][2]), "=&v"(xa[1][3]), "=&v"(wb[0][0]), "=&v"(wb[0][1]), "=&v"(wb[1][0]), "=&v"(wb[1][1])
  if constexpr (COPY)
    asm volatile(PP_READS PP_COPY1 PP_COPYN("v1") PP_COPYN("v2") PP_COPYN("v3") PP_WAIT : PP_OUTS
                 : PP_ARGS, [m0] "s"(m0), [sa] "s"(sa), [v0] "v"(vo[0]), [v1] "v"(vo[1]), [v2] "v"(vo[2]), [v3] "v"(vo[3])
                 : "memory", "m0", "scc");
  else asm volatile(PP_READS PP_WAIT : PP_OUTS : PP_ARGS : "memory");
#undef PP_READS
#undef PP_OUTS
}
#undef PP_COPY1
#undef PP_COPYN
#undef PP_WAIT
#undef PP_ARGS

template <bool GLU>
__global__ __launch_bounds__(512) void linear_pp_kernel(const sf_linear_args a, const int gx, const int gy, const int total) {
  constexpr int BM = kTile, BN = kTile, WM = 2, WN = 4, S = 4;
  constexpr int ABYTES = BM * 64, STAGE = (BM + BN) * 64, A = S - 1;
  constexpr int CPW = STAGE / 1024 / 8;                       // 1 KB copies per wave per step
  constexpr int WR = BM / WM, WC = BN / WN, MB = WR / 32, NB = WC / 32;
  constexpr int XB = 64 * NB;                                 // bytes per row of a wave's bf16 block (operands)
  constexpr int RB = GLU ? XB / 2 : XB;                       // ... of its results
  constexpr int EPI = 32 * XB;                                // a wave's private epilogue block
  static_assert(WM * WN == 8 && MB >= 1 && NB >= 1 && STAGE % 8192 == 0 && (S & A) == 0, "8 waves, whole copies per wave");
  __shared__ __attribute__((aligned(1024))) uint8_t smem[S * STAGE + 8 * EPI];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int half = lane >> 5, li = lane & 31;
  const int wm = wave / WN, wn = wave % WN;
  const bool late = wave >= 4;                                // the second wave of each SIMD
  // Workgroup b is assumed to run on XCD b % 8 (round-robin dispatch); each XCD takes a contiguous
  // range of tiles for its L2: batch members one after another, a member's tiles in bands of kBand
  // tile rows, so that the 32 tiles an XCD runs together form a block of both operands (in plain
  // row order they read nearly every row of one operand: 8192 x 8192 x 1024 ran at the L2 fill rate)
  constexpr int kBand = 5;
  const int per = (total + 7) >> 3, xcd = blockIdx.x & 7, G8 = gridDim.x >> 3;
  const int tend = min(total, (xcd + 1) * per);
  int tile = xcd * per + (int)(blockIdx.x >> 3);
  if (tile >= tend) return;                                   // uniform over the workgroup
  // this wave's copies: 1 KB chunk c = rows 16 c .. 16 c + 15 of the stage (A rows, then B rows);
  // lane L fills row L / 4, slot L % 4, with piece (L % 4) ^ ((row / 4) % 4).  Rows past the end
  // read the last row (their results are never stored).
  const int crow = lane >> 2, cpiece = (lane & 3) ^ ((lane >> 4) & 3);
  auto place = [&](int t, int& bx, int& by, int& bz) __attribute__((always_inline)) {
    bz = t / (gx * gy);
    const int r = t - bz * gx * gy, band = r / (kBand * gy), q = r - band * kBand * gy;
    const int bh = min(kBand, gx - band * kBand);
    by = q / bh;
    bx = band * kBand + q - by * bh;
  };
  static_assert((BM / 16) % CPW == 0, "a wave copies rows of one operand");
  const bool wave_a = wave * CPW < BM / 16;                   // uniform: this wave copies A rows, else B rows
  const int chunk0 = wave_a ? wave * CPW : wave * CPW - BM / 16;
  auto sources = [&](int t, const char*& sa, uint32_t (&vo)[CPW]) __attribute__((always_inline)) {
    int bx, by, bz;
    place(t, bx, by, bz);
    const int64_t r0 = wave_a ? (int64_t)bx * BM : (int64_t)by * BN;   // first row of the operand's tile
    const int64_t rs = wave_a ? a.x_rs : (int64_t)a.K;
    const int lastr = (int)min((wave_a ? a.M : (int64_t)a.N) - 1 - r0, (int64_t)1 << 30);
    sa = (const char*)((wave_a ? (const uint16_t*)a.x + bz * a.x_bs : (const uint16_t*)a.wt + bz * a.w_bs) + r0 * rs);
#pragma unroll
    for (int u = 0; u < CPW; ++u)
      vo[u] = (uint32_t)min(16 * (chunk0 + u) + crow, lastr) * (uint32_t)(2 * rs) + cpiece * 16;
  };
  // operand addresses: row r of a region at 64 r, slot piece ^ ((r / 4) % 4); k-chunk kk, lane
  // half: piece 2 kk + half (kk = 1 flips bit 1 of the slot)
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_u32*)smem;
  const uint32_t rowoff = (uint32_t)(li * 64 + ((half ^ ((li >> 2) & 3)) * 16));
  const uint32_t abase = lds0 + wm * WR * 64 + rowoff, bbase = lds0 + ABYTES + wn * WC * 64 + rowoff;
  auto barrier = [&]() __attribute__((always_inline)) {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  // private epilogue block: row r of 16-byte pieces, slot piece ^ (row of the 256-byte line)
  const uint32_t epi = lds0 + S * STAGE + wave * EPI;
  auto slot = [&](int rb, int row, int piece) __attribute__((always_inline)) -> uint32_t {
    return epi + row * rb + ((piece ^ ((row * rb >> 8) & (rb / 16 - 1))) << 4);
  };

  const int n = a.K / 32;                                     // >= A (host rule)
  const char* sa;                                             // this tile's copies: uniform base
  uint32_t vo[CPW];                                           // ... and lane offsets
  sources(tile, sa, vo);
#pragma unroll
  for (int t = 0; t < A; ++t)
#pragma unroll
    for (int u = 0; u < CPW; ++u) {
      const uint32_t off = vo[u] + t * 64;
      const char* from = sa + off;
      __builtin_amdgcn_global_load_lds(from, (lds_u32*)(smem + t * STAGE + (wave * CPW + u) * 1024), 16, 0, 0);
    }
  pp_wait<(A - 1) * CPW>();
  barrier();
  if (late) barrier();
  // The stores of a tile's epilogue sit in the memory counter between the copies of the next tile's
  // steps A - 1 and A: the first A - 1 waits of a tile leave them in flight (all waves store at
  // once, 32 MB over the chip; waited for at the first step they cost 3 us a tile).
  constexpr int kStores = MB * (32 * RB / 1024);
  bool stored = false;                                        // the previous tile's epilogue issued kStores stores
  int T = 0;                                                  // steps done: the stage of step t is (T + t) % S
  for (;;) {
    const int next = tile + G8;
    const bool has_next = next < tend;                        // uniform
    const char* nsa;
    uint32_t nvo[CPW];
    sources(has_next ? next : tile, nsa, nvo);
    f32x16 acc[MB][NB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[mb][nb][r] = 0.f;
    u32x4 xa[2][MB], wb[2][NB];
    for (int t = 0; t < n; ++t) {
      const uint32_t so = (uint32_t)((T + t) & A) * STAGE;
      const uint32_t a0 = abase + so, b0 = bbase + so;
      // read step t; copy step t + A of this tile, or step t + A - n of the next one
      const uint32_t m0 = lds0 + (uint32_t)((T + t + A) & A) * STAGE + wave * CPW * 1024;   // uniform
      if (t + A < n) pp_read<MB, NB, CPW, true>(a0, a0 ^ 32u, b0, b0 ^ 32u, xa, wb, m0, sa + (int64_t)(t + A) * 64, vo);
      else if (has_next) pp_read<MB, NB, CPW, true>(a0, a0 ^ 32u, b0, b0 ^ 32u, xa, wb, m0, nsa + (int64_t)(t + A - n) * 64, nvo);
      else pp_read<MB, NB, CPW, false>(a0, a0 ^ 32u, b0, b0 ^ 32u, xa, wb, m0, sa, vo);
      // the copies of step t + 1 have landed (in issue order); those of steps t + 2 .. t + A may stay
      // in flight (left: how many of them exist), and the stores issued between A - 1 and A
      const int left = has_next ? A : n - 2 - t;
      const bool relax = stored && t < A - 1 && left >= A - 1;   // uniform
      auto landed = [&]() __attribute__((always_inline)) {
        if (relax) pp_wait<(A - 1) * CPW + kStores>();
        else pp_wait_steps<CPW, A - 1>(left);
      };
      if (late) landed();
      barrier();
#pragma unroll
      for (int kk = 0; kk < 2; ++kk)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
#pragma unroll
          for (int nb = 0; nb < NB; ++nb) acc[mb][nb] = mfma32(as_bf16x8(wb[kk][nb]), as_bf16x8(xa[kk][mb]), acc[mb][nb]);
      if (!late) landed();
      barrier();
    }
    T += n;

    // ---- epilogue of this wave's WR x WC part ----
    {
      int bx, by, bz;
      place(tile, bx, by, bz);
      const int64_t m0 = (int64_t)bx * BM + wm * WR;
      const int n0 = by * BN + wn * WC;
      uint16_t* const yp = (uint16_t*)a.y + bz * a.y_bs;
      const uint16_t* const rp = (const uint16_t*)a.residual;
      const uint16_t* const mp = (const uint16_t*)a.mul;
      const float* const bp = a.bias;
      constexpr int XP = XB / 16, XI = 32 / (64 / XP);        // pieces per operand row, loads per 32 rows
      constexpr int RP = RB / 16, RI = 32 / (64 / RP);        // ... of the results
      // every load of the epilogue comes before its first store: the memory counter is in order, so a
      // load between the stores would wait for them
      if (bp) {                                               // (uniform branches)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            const f32x4 b4 = *reinterpret_cast<const f32x4*>(bp + min(n0 + 32 * nb + 8 * c + 4 * half, a.N - 4));
#pragma unroll
            for (int mb = 0; mb < MB; ++mb)
#pragma unroll
              for (int e = 0; e < 4; ++e) acc[mb][nb][4 * c + e] += b4[e];
          }
      }
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
        f32x16 (&v)[NB] = acc[mb];
        // a [32 rows][32 NB columns] block of mul / residual -> this lane's row li, columns
        // 32 nb + 8 c + 4 half .. + 3 (rows and columns past the end read the last ones)
        auto fetch = [&](const uint16_t* base, int64_t rs, bool wrap, u32x2 (&f)[NB][4]) __attribute__((always_inline)) {
          u32x4 w[XI];
#pragma unroll
          for (int i = 0; i < XI; ++i) {
            const int64_t m = min(m0 + 32 * mb + i * (64 / XP) + lane / XP, a.M - 1);
            const int64_t row = wrap ? (int64_t)((uint32_t)m % (uint32_t)a.mul_rows) : m;
            w[i] = ld16(base + row * rs + min(n0 + 8 * (lane % XP), a.N - 8));
          }
#pragma unroll
          for (int i = 0; i < XI; ++i) pp_ds_write16(slot(XB, i * (64 / XP) + lane / XP, lane % XP), w[i]);
#pragma unroll
          for (int nb = 0; nb < NB; ++nb) {
            uint32_t ad[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) ad[c] = slot(XB, li, 4 * nb + c) + 8 * half;
            pp_ds_read8x4(ad, f[nb]);
          }
        };
        if constexpr (!GLU) {
          if (a.post_sigmoid) {
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
#pragma unroll
              for (int r = 0; r < 16; ++r) v[nb][r] = sigmoidf_(v[nb][r]);
          }
          if (mp) {
            u32x2 f[NB][4];
            fetch(mp, a.mul_rs, true, f);
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
#pragma unroll
              for (int c = 0; c < 4; ++c) {
                v[nb][4 * c] *= bflo(f[nb][c][0]); v[nb][4 * c + 1] *= bfhi(f[nb][c][0]);
                v[nb][4 * c + 2] *= bflo(f[nb][c][1]); v[nb][4 * c + 3] *= bfhi(f[nb][c][1]);
              }
          }
          if (rp) {
            u32x2 f[NB][4];
            fetch(rp, a.r_rs, false, f);
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
#pragma unroll
              for (int c = 0; c < 4; ++c) {
                v[nb][4 * c] += bflo(f[nb][c][0]); v[nb][4 * c + 1] += bfhi(f[nb][c][0]);
                v[nb][4 * c + 2] += bflo(f[nb][c][1]); v[nb][4 * c + 3] += bfhi(f[nb][c][1]);
              }
          }
        }
      }
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
        f32x16 (&v)[NB] = acc[mb];
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            const float x0 = v[nb][4 * c], x1 = v[nb][4 * c + 1], x2 = v[nb][4 * c + 2], x3 = v[nb][4 * c + 3];
            if constexpr (GLU)     // gated pairs: columns 2j (swish) and 2j + 1 of the interleaved weight -> column j
              pp_ds_write4(slot(RB, li, 2 * nb + (c >> 1)) + 8 * (c & 1) + 4 * half,
                           pack_bf2(x0 * sigmoidf_(x0) * x1, x2 * sigmoidf_(x2) * x3));
            else
              pp_ds_write8(slot(RB, li, 4 * nb + c) + 8 * half, u32x2{pack_bf2(x0, x1), pack_bf2(x2, x3)});
          }
        // rows past the end store the last row again and columns past the end the last valid piece:
        // the same bytes their owners store (rows past the end were computed from the last row), so
        // that the number of stores does not depend on the tile.  A wave with no column stores nothing.
        uint32_t ad[RI];
        u32x4 w[RI];
        const int ncols = GLU ? a.N / 2 : a.N, nc0 = GLU ? n0 / 2 : n0;
        const int pc = min(lane % RP, (ncols - nc0) / 8 - 1);
        stored = nc0 < ncols;                                 // uniform
        if (stored) {
#pragma unroll
          for (int i = 0; i < RI; ++i) ad[i] = slot(RB, i * (64 / RP) + lane / RP, pc);
          pp_ds_read16<RI>(ad, w);
#pragma unroll
          for (int i = 0; i < RI; ++i) {
            const int64_t m = min(m0 + 32 * mb + i * (64 / RP) + lane / RP, a.M - 1);
            st16(yp + m * a.y_rs + nc0 + 8 * pc, w[i]);
          }
        }
      }
    }
    if (!has_next) break;
    tile = next;
    sa = nsa;
#pragma unroll
    for (int u = 0; u < CPW; ++u) vo[u] = nvo[u];
  }
  if (!late) barrier();                                       // the late group's extra first barrier
}

bool al16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

int64_t tiles(const sf_linear_args* a, int side) {
  return ((a->M + side - 1) / side) * (((int64_t)a->N + side - 1) / side) * (a->batch > 1 ? a->batch : 1);
}

// Workgroups of a launch: as many as are resident at once, a multiple of 8 (XCDs).  256 where no device
// is there to ask (the host-only query).
int64_t workgroups(const sf_linear_args* a) {
  const void* kernel = a->glu ? reinterpret_cast<const void*>(linear_pp_kernel<true>) : reinterpret_cast<const void*>(linear_pp_kernel<false>);
  const int n = sf_resident_workgroups(kernel, 512) / 8 * 8;
  return n > 0 ? n : 256;
}

// bytes [p, p + ((rows - 1) rs + n) * 2) of a row-strided bf16 operand (rs > 0) meet y's
bool meets_y(const sf_linear_args* a, const void* p, int64_t rows, int64_t rs) {
  const uintptr_t p0 = reinterpret_cast<uintptr_t>(p), p1 = p0 + ((rows - 1) * rs + a->N) * 2;
  const uintptr_t y0 = reinterpret_cast<uintptr_t>(a->y), y1 = y0 + ((a->M - 1) * a->y_rs + a->N) * 2;
  return p0 < y1 && y0 < p1;
}

}  // namespace

bool sf_linear_pp_ok(const sf_linear_args* a) {
  // what the kernel assumes: whole 16-byte pieces in every row, at least four K steps, 32-bit row
  // offsets inside a tile, no transposed or partial output
  const bool fits = a->K % 64 == 0 && a->K >= 128 && a->K <= (1 << 22) && a->x_rs > 0 && a->x_rs <= (1 << 22) && a->y != nullptr &&
                    a->yt == nullptr && a->N % (a->glu ? 16 : 8) == 0 && (a->ycols == 0 || a->ycols == a->N) &&
                    al16(a->y) && a->y_rs % 8 == 0 && (a->batch <= 1 || a->y_bs % 8 == 0) && a->M < (1ll << 31) &&
                    (!a->bias || al16(a->bias)) &&
                    a->y_rs > 0 &&
                    (!a->mul || (al16(a->mul) && a->mul_rs > 0 && a->mul_rs % 8 == 0 && a->mul_rows < (1ll << 31))) &&
                    (!a->residual || (al16(a->residual) && a->r_rs > 0 && a->r_rs % 8 == 0));
  if (!fits) return false;
  // rows past the end are computed and stored twice (see the epilogue): an update in place would
  // add its residual twice there
  if ((a->residual && meets_y(a, a->residual, a->M, a->r_rs)) || (a->mul && meets_y(a, a->mul, a->mul_rows, a->mul_rs))) return false;
  // One round of 256 tiles here takes as long as about 540 of linear64_kernel's 128 x 128 tiles
  // (5120 x 3072 x 768: one round 33 us, 960 tiles 38; 3700 x 3072 x 768: one round 27 us, 696
  // tiles 34; 6000 x 1536 x 384: one round 19 us, 564 tiles 23; 5120 x 768 x 768: one round 24 us,
  // 240 tiles 15), where this kernel's tiles cover at most half as much again as those.  Beyond that the
  // two tie on some cards and it loses on others: 128 batched products of 300 x 304 x 320 (2 x 2 tiles
  // against 3 x 3, 1.78 times the area) 28.0 here and 28.5 there on one card, 32.7 and 29.5 on another,
  // 344 x 344 x 384 31.5 and 31.4, 37.3 and 32.7.  At 1.44 times the area 600 x 600 x 640 109 and 120, 110
  // and 123 (520 x 520 x 576 85.4 and 85.2, 94.7 and 90.0); at 1.33 65536 x 264 x 768 56 and 67.
  const int64_t big = tiles(a, kTile), small = tiles(a, 128), wgs = workgroups(a);
  return big < (1ll << 30) && 540 * wgs * ((big + wgs - 1) / wgs) <= 256 * small && 8 * big <= 3 * small;
}

extern "C" int sf_hip_linear_large_tiles(const sf_linear_args* a) {
  return a != nullptr && a->K % 64 == 0 && sf_linear_pp_ok(a);
}

int sf_linear_pp_launch(const sf_linear_args* a, hipStream_t stream) {
  const int64_t gx = (a->M + kTile - 1) / kTile, gy = ((int64_t)a->N + kTile - 1) / kTile;
  const int64_t total = tiles(a, kTile);
  const dim3 grid((unsigned)std::min<int64_t>(workgroups(a), (total + 7) / 8 * 8));
  if (a->glu) hipLaunchKernelGGL(linear_pp_kernel<true>, grid, dim3(512), 0, stream, *a, (int)gx, (int)gy, (int)total);
  else hipLaunchKernelGGL(linear_pp_kernel<false>, grid, dim3(512), 0, stream, *a, (int)gx, (int)gy, (int)total);
  return sf_check_launch("linear_pp_kernel");
}
