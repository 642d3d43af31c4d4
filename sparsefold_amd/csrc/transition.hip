// The trunk's pair transition (TransitionBlock.forward, blocks.py:84-96) at C = 128 channels in one
// kernel: out = x + (swish(h W1a) * (h W1b)) W2, h = LayerNorm(x), per row of 128 channels.
//
// The LayerNorm, GLU GEMM and output GEMM launches it replaces move every row five times and the
// gated intermediate (I = 512 channels, 1 KB a row) twice through memory: 147456 rows took 44 + 136 +
// 50 us, against 15 us to read x and write out.  Here a wave keeps 32 rows from the first load to the
// last store: h as MFMA operands (32 registers), the 128 x 32 output accumulators (64), and the
// intermediate 32 channels at a time, which never leaves the registers -- the rows of W1 are staged in
// the order in which the first product's accumulator registers are the second one's operand.
//
// A workgroup (8 waves, 256 rows, one per CU) streams the weights through LDS, 24 KB per step of 32
// intermediate channels, double-buffered; one LDS barrier per step.  Step i runs the first product
// (W1) of channels 32 (i + 1) .. and the second (W2) of channels 32 i ..: the gating of one block of
// channels sits in the shadow of the next block's MFMAs.
//
// 147456 rows (N = 384): 206 -> 75 us for the call, 5000 (N = 70) 34 -> 22: the host's part, one launch
// for three.  (On the GPU a pass is 23 us however few rows there are, the three launches 15 to 18 up to
// 4096: replayed from a graph, such calls took less before.)  A pass of 256 rows a workgroup takes 24 us: 11 us
// of MFMAs (384 a wave, two waves per SIMD), 5 of gating beside them, 4 of LayerNorm, 2 of stores, the
// rest operand reads, barriers and staging.  Built and not kept: the two waves of a SIMD changing
// rows two steps apart (the barrier of every step makes one wait through the other's change: 26 us).
#include <algorithm>
#include <type_traits>

#include "sf_common.h"

namespace {

constexpr int kC = 128;
constexpr int kWaves = 8;
constexpr int kP1 = kC + 8;            // LDS pitch (elements) of W1 rows and of x rows: 16 rows cover all banks
constexpr int kP2 = 32 + 8;            // LDS pitch of W2 rows (32 intermediate channels)
constexpr int kStage = 64 * kP1 + kC * kP2;   // elements of one weight stage

typedef u32x4 u32x4_any __attribute__((aligned(2)));   // a 16-byte store at any even address (out alone may be one)

struct TransArgs {
  int64_t rows; int I, items, add_residual;   // items = ceil(rows / 32)
  const uint16_t* x;                   // [rows, 128]
  const float *ln_w, *ln_b;            // [128] or null
  const uint16_t* w1;                  // [2 I, 128]: row 2 i swish channel i, row 2 i + 1 its factor
  const uint16_t* w2;                  // [128, I]
  uint16_t* out;                       // [rows, 128]
};

__global__ __launch_bounds__(64 * kWaves) void transition128_kernel(const TransArgs a) {
  __shared__ __attribute__((aligned(16))) uint16_t sW[2 * kStage];
  __shared__ __attribute__((aligned(16))) uint16_t sX[kWaves][32 * kP1];   // each wave's rows: x, then out
  __shared__ __attribute__((aligned(16))) float sG[kC], sB[kC];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int half = lane >> 5, li = lane & 31;
  uint16_t* const xr = sX[wave];
  const int nblk = a.I / 32;
  if (tid < kC) {
    sG[tid] = a.ln_w ? a.ln_w[tid] : 1.f;
    sB[tid] = a.ln_b ? a.ln_b[tid] : 0.f;
  }
  // ---- weight staging: step i holds W1 of block (i + 1) % nblk and W2 of block i (i = -1 .. nblk - 1)
  //      thread t: W1 rows t / 16 and 32 + t / 16 (rows 0..31 swish, 32..63 factor), piece t % 16;
  //      W2 row t / 4, piece t % 4.  Staged W1 row m holds channel 16 (m / 16) + 8 ((m / 4) % 2) +
  //      4 ((m / 8) % 2) + m % 4, so that accumulator registers 8 kk .. 8 kk + 7 of lane half h are
  //      channels 16 kk + 8 h .. + 7. ----
  const int m = tid >> 4, ch = 16 * (m >> 4) + 8 * ((m >> 2) & 1) + 4 * ((m >> 3) & 1) + (m & 3);
  const uint16_t* const w1p = a.w1 + (int64_t)2 * ch * kC + 8 * (tid & 15);
  const uint16_t* const w2p = a.w2 + (int64_t)(tid >> 2) * a.I + 8 * (tid & 3);
  u32x4 r1a, r1b, r2;
  auto stage_load = [&](int i) __attribute__((always_inline)) {
    const int b1 = i + 1 < nblk ? i + 1 : 0, b2 = i < 0 ? 0 : i;
    r1a = ld16(w1p + (int64_t)b1 * 64 * kC);
    r1b = ld16(w1p + (int64_t)b1 * 64 * kC + kC);
    r2 = ld16(w2p + 32 * b2);
  };
  auto stage_store = [&](int buf) __attribute__((always_inline)) {
    uint16_t* s = sW + buf * kStage;
    st16(s + m * kP1 + 8 * (tid & 15), r1a);
    st16(s + (32 + m) * kP1 + 8 * (tid & 15), r1b);
    st16(s + 64 * kP1 + (tid >> 2) * kP2 + 8 * (tid & 3), r2);
  };
  auto after = [&](int i) __attribute__((always_inline)) { return i + 1 < nblk ? i + 1 : -1; };   // the step after step i

  const int base = blockIdx.x * kWaves;                 // item of wave 0; the grid steps by gridDim * 8
  int buf = 0;
  stage_load(-1);
  stage_store(0);
  stage_load(after(-1));
  __syncthreads();
  // x rows of an item, 16 lanes a row, four rows an instruction; rows past the end read the last one
  u32x4 xv[8];
  auto load_rows = [&](int it) __attribute__((always_inline)) {
    const int64_t r = (int64_t)(it + wave) * 32 + (lane >> 4);
#pragma unroll
    for (int u = 0; u < 8; ++u) xv[u] = ld16(a.x + min(r + 4 * u, a.rows - 1) * kC + 8 * (lane & 15));
  };
  const int stride = gridDim.x * kWaves;
  load_rows(base);
  for (int it0 = base; it0 < a.items; it0 += stride) {
    const int64_t row0 = (int64_t)(it0 + wave) * 32;     // idle waves (row0 >= rows) run on the last row
#pragma unroll
    for (int u = 0; u < 8; ++u) st16(xr + (4 * u + (lane >> 4)) * kP1 + 8 * (lane & 15), xv[u]);
    asm volatile("" ::: "memory");                       // one wave's LDS accesses run in order
    bf16x8 xo[8];                                        // h of row li, channels 16 kk + 8 half ..
    {
      u32x4 v[8];
#pragma unroll
      for (int kk = 0; kk < 8; ++kk) v[kk] = ld16(xr + li * kP1 + 16 * kk + 8 * half);
      float sm[4] = {0.f, 0.f, 0.f, 0.f}, sv[4] = {0.f, 0.f, 0.f, 0.f};   // four chains each
#pragma unroll
      for (int kk = 0; kk < 8; ++kk)
#pragma unroll
        for (int e = 0; e < 4; ++e) sm[e] += bflo(v[kk][e]) + bfhi(v[kk][e]);
      float sum = (sm[0] + sm[1]) + (sm[2] + sm[3]);
      sum += __shfl_xor(sum, 32);
      const float mean = sum * (1.0f / kC);
#pragma unroll
      for (int kk = 0; kk < 8; ++kk)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float d0 = bflo(v[kk][e]) - mean, d1 = bfhi(v[kk][e]) - mean;
          sv[e] += d0 * d0 + d1 * d1;
        }
      float sq = (sv[0] + sv[1]) + (sv[2] + sv[3]);
      sq += __shfl_xor(sq, 32);
      const float rstd = rsqrtf(sq * (1.0f / kC) + 1e-5f);
#pragma unroll
      for (int kk = 0; kk < 8; ++kk) {
        float g[8], b[8];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const f32x4 g4 = *reinterpret_cast<const f32x4*>(sG + 16 * kk + 8 * half + 4 * q);
          const f32x4 b4 = *reinterpret_cast<const f32x4*>(sB + 16 * kk + 8 * half + 4 * q);
#pragma unroll
          for (int e = 0; e < 4; ++e) { g[4 * q + e] = g4[e]; b[4 * q + e] = b4[e]; }
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const bf16x2 y = cvt_bf2((bflo(v[kk][e]) - mean) * rstd * g[2 * e] + b[2 * e],
                                   (bfhi(v[kk][e]) - mean) * rstd * g[2 * e + 1] + b[2 * e + 1]);
          xo[kk][2 * e] = y[0];
          xo[kk][2 * e + 1] = y[1];
        }
      }
    }
    f32x16 o[4], h[2][2];                                // h[parity of the block]: swish and factor channels
#pragma unroll
    for (int nb = 0; nb < 4; ++nb)
#pragma unroll
      for (int e = 0; e < 16; ++e) o[nb][e] = 0.f;
    auto advance = [&](int i) __attribute__((always_inline)) {   // step i is in buf: bring step after(i) in, load the one after
      stage_store(buf ^ 1);
      stage_load(after(after(i)));
    };
    auto w1op = [&](const uint16_t* s, int kk, int f) __attribute__((always_inline)) {
      return as_bf16x8(ld16(s + (32 * f + li) * kP1 + 16 * kk + 8 * half));
    };
    auto w2op = [&](const uint16_t* s, int kk, int nb) __attribute__((always_inline)) {
      return as_bf16x8(ld16(s + 64 * kP1 + (32 * nb + li) * kP2 + 16 * kk + 8 * half));
    };
    advance(-1);
    {
      const uint16_t* s = sW + buf * kStage;             // W1 of block 0
#pragma unroll
      for (int f = 0; f < 2; ++f)
#pragma unroll
        for (int e = 0; e < 16; ++e) h[0][f][e] = 0.f;
#pragma unroll
      for (int kk = 0; kk < 8; ++kk)
#pragma unroll
        for (int f = 0; f < 2; ++f) h[0][f] = mfma32(w1op(s, kk, f), xo[kk], h[0][f]);
    }
    lds_only_barrier();
    buf ^= 1;
    // One step in six groups of four MFMAs: the first product's k-chunks (two MFMAs each: swish and
    // factor rows) in all six, the second product's as soon as its operand chunk is gated; the gating
    // of four channels in each of the first four groups; every group reads the next one's operands.
    // The group barriers interleave them (left alone, the compiler put all gating before the MFMAs and
    // every operand read right before its use).
    // LAST: no block follows; the next item's rows are loaded instead (into the registers the first
    // product does not need) and land under the gating.
    auto step = [&](int i, auto parity, auto lastc) __attribute__((always_inline)) {
      constexpr int P = decltype(parity)::value;
      constexpr bool LAST = decltype(lastc)::value;
      f32x16 &ha = h[P][0], &hb = h[P][1], &na = h[P ^ 1][0], &nb_ = h[P ^ 1][1];
      const uint16_t* s = sW + buf * kStage;
      bf16x8 cb[2], w[2][4];
      auto gate = [&](int g) __attribute__((always_inline)) {   // channels 4 g .. 4 g + 3 of this lane
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const int r = 4 * g + 2 * e;
          const bf16x2 y = cvt_bf2(ha[r] * sigmoidf_(ha[r]) * hb[r], ha[r + 1] * sigmoidf_(ha[r + 1]) * hb[r + 1]);
          cb[g >> 1][4 * (g & 1) + 2 * e] = y[0];
          cb[g >> 1][4 * (g & 1) + 2 * e + 1] = y[1];
        }
      };
      if constexpr (LAST) {
        advance(i);
        load_rows(min(it0 + stride, a.items - 1));       // (the last item's: unused)
#pragma unroll
        for (int q = 0; q < 4; ++q) w[0][q] = w2op(s, 0, q);
#pragma unroll
        for (int q = 0; q < 4; ++q) w[1][q] = w2op(s, 1, q);
        gate(0); gate(1);
#pragma unroll
        for (int q = 0; q < 4; ++q) o[q] = mfma32(w[0][q], cb[0], o[q]);
        gate(2); gate(3);
#pragma unroll
        for (int q = 0; q < 4; ++q) o[q] = mfma32(w[1][q], cb[1], o[q]);
        lds_only_barrier();
        buf ^= 1;
        return;
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) w[0][q] = w1op(s, q >> 1, q & 1);
      advance(i);
#pragma unroll
      for (int e = 0; e < 16; ++e) { na[e] = 0.f; nb_[e] = 0.f; }
      // the younger wave of each SIMD goes first for most of a step: with age priority the older one
      // finished early and waited at the barrier (2%)
      if (wave >= kWaves / 2) __builtin_amdgcn_s_setprio(1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int g = 0; g < 6; ++g) {
        if (g == 5) __builtin_amdgcn_s_setprio(0);
        bf16x8 (&wc)[4] = w[g & 1], (&wn)[4] = w[(g & 1) ^ 1];
        // operands of group g + 1: groups 0, 1 are k-chunks 2g, 2g + 1; group g >= 2 is k-chunk g + 2
        // and column blocks 2 (g % 2), + 1 of the second product's chunk (g - 2) / 2
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int n = g + 1;
          if (n == 1) wn[q] = w1op(s, 2 + (q >> 1), q & 1);
          else if (n < 6) wn[q] = q < 2 ? w1op(s, n + 2, q) : w2op(s, (n - 2) >> 1, 2 * (n & 1) + q - 2);
        }
        if (g < 2) {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            if (q & 1) nb_ = mfma32(wc[q], xo[2 * g + (q >> 1)], nb_);
            else na = mfma32(wc[q], xo[2 * g + (q >> 1)], na);
          }
        } else {
          const int k2 = (g - 2) >> 1, n2 = 2 * (g & 1);
          na = mfma32(wc[0], xo[g + 2], na);
          o[n2] = mfma32(wc[2], cb[k2], o[n2]);
          nb_ = mfma32(wc[1], xo[g + 2], nb_);
          o[n2 + 1] = mfma32(wc[3], cb[k2], o[n2 + 1]);
        }
        if (g < 4) gate(g);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);         // one MFMA
          if (g < 5) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);   // one LDS read
          if (g < 4) __builtin_amdgcn_sched_group_barrier(0x002, 7, 0);   // a quarter of the gating
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      lds_only_barrier();
      buf ^= 1;
    };
    using F = std::false_type; using T = std::true_type;
    for (int i = 0; i < nblk; i += 2) {                  // nblk is even
      step(i, std::integral_constant<int, 0>{}, F{});
      if (i + 2 < nblk) step(i + 1, std::integral_constant<int, 1>{}, F{});
    }
    step(nblk - 1, std::integral_constant<int, 1>{}, T{});
    // ---- out: channels 32 nb + 8 c + 4 half .. + 3 of row li, plus x, through the wave's rows ----
    const uint32_t rmask = a.add_residual ? ~0u : 0u;
    u32x2 z[4][4];
#pragma unroll
    for (int nb = 0; nb < 4; ++nb)
#pragma unroll
      for (int c = 0; c < 4; ++c) z[nb][c] = *reinterpret_cast<const u32x2*>(xr + li * kP1 + 32 * nb + 8 * c + 4 * half);
#pragma unroll
    for (int nb = 0; nb < 4; ++nb)
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const uint32_t z0 = z[nb][c][0] & rmask, z1 = z[nb][c][1] & rmask;
        *reinterpret_cast<u32x2*>(xr + li * kP1 + 32 * nb + 8 * c + 4 * half) =
            u32x2{pack_bf2(o[nb][4 * c] + bflo(z0), o[nb][4 * c + 1] + bfhi(z0)), pack_bf2(o[nb][4 * c + 2] + bflo(z1), o[nb][4 * c + 3] + bfhi(z1))};
      }
    asm volatile("" ::: "memory");
    u32x4 v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = ld16(xr + (4 * u + (lane >> 4)) * kP1 + 8 * (lane & 15));
    uint16_t* const op = a.out + (row0 + (lane >> 4)) * kC + 8 * (lane & 15);
    if (row0 + 32 <= a.rows) {
#pragma unroll
      for (int u = 0; u < 8; ++u) *reinterpret_cast<u32x4_any*>(op + 4 * u * kC) = v[u];
    } else {
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (row0 + 4 * u + (lane >> 4) < a.rows) *reinterpret_cast<u32x4_any*>(op + 4 * u * kC) = v[u];
    }
    asm volatile("" ::: "memory");                       // (the rows are rewritten by the next item)
  }
}

bool al16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

}  // namespace

// By sizes alone: the workspace query must give the same answer whatever addresses the call comes with.
bool sf_transition128_ok(const sf_transition_args* a) {
  return a->C == kC && a->I % 64 == 0 && a->cond == nullptr && a->pre_scale == nullptr && (int64_t)a->S * a->N < (1ll << 35);
}

int sf_transition128_launch(const sf_transition_args* a, hipStream_t stream) {
  if (!al16(a->x) || !al16(a->w1) || !al16(a->w2)) {
    sf_set_error("transition: x, w1 and w2 must be 16-byte aligned"); return 1;
  }
  TransArgs t{};
  t.rows = (int64_t)a->S * a->N; t.I = a->I; t.items = (int)((t.rows + 31) / 32); t.add_residual = a->add_residual;
  t.x = static_cast<const uint16_t*>(a->x); t.ln_w = a->ln_w; t.ln_b = a->ln_b;
  t.w1 = static_cast<const uint16_t*>(a->w1); t.w2 = static_cast<const uint16_t*>(a->w2);
  t.out = static_cast<uint16_t*>(a->out);
  const int groups = (t.items + kWaves - 1) / kWaves;
  const int resident = sf_resident_workgroups(reinterpret_cast<const void*>(transition128_kernel), 64 * kWaves);
  hipLaunchKernelGGL(transition128_kernel, dim3(std::min(groups, resident)), dim3(64 * kWaves), 0, stream, t);
  return sf_check_launch("transition128_kernel");
}
