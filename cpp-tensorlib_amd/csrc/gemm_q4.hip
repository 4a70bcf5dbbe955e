// Prompt-chunk GEMM over an int4 weight: C[M,N] = A[M,K] f32 . dequant(W)^T, formed as the sum over groups of
// scale * (A . q) - the decode GEMV's arithmetic on the matrix pipe, in the terms of gemm_bf16_nt_kernel's int4 form for
// more than 64 rows: row m of A times 2^ea[m] as two f16 terms (one fp32 rounding per product), nibbles exact in f16, a
// group's sums started at zero and added to the accumulators times its scale.
//
// What bounded that form (244 TFLOP/s): vector instructions. Every block cut its rows of A again, slab by slab
// (128 instructions per lane and slab of 32 k beside 16 MFMAs), and a nibble took two instructions. Here:
//   * A is cut once per product (q4_image_kernel; the pass that found the exponents did half of it) into images of
//     64 rows x 32 k, both terms, 8 KB, rows in the bank-conflict-free order the fragment reads expect, so that a unit
//     of four slabs is 32 contiguous KB that go to LDS by global_load_lds, without registers;
//   * the nibbles a lane multiplies come to it directly: its wavefront owns 64 columns (64 x 64 outputs, four
//     wavefronts side by side), a 16-byte load is one group of one column, and two half-wave swaps per two groups give
//     each half its k. Masked in place, a nibble is an f16 with its value (or 16 times that) in the last bits of 1024, so
//     eight of them take nine instructions; the k order that gives (0 4 1 5 2 6 3 7) is the one the images are
//     written in.
// 102 vector instructions beside 16 MFMAs per slab and wavefront are left, 64 of them the scales'. Behind the MFMAs they and
// the MFMAs of a SIMD's two wavefronts add up (512 x 32768 x 3584: 235 us = 510 TFLOP/s; without the scales 192, without all
// of it and the loads 148; wave priorities and a staggered start change nothing), so they go between them, six of which two
// wavefronts hide behind one: 24 shapes 0.99 to 1.10 times as fast, 1.03 on average, 512 x 37888 x 3584 gated 1.06. Two blocks per CU, one barrier per 128 k.
// Rows come in blocks of 64: 301 rows waste 6 % of the products, 128-row tiles waste 28 %. us, before -> now: 301 rows
// gated 37888 x 3584 303 -> 209, 3584 x 18944 150 -> 113, 4608 x 3584 48 -> 42; 512 rows 393 -> 320, 207 -> 176, 61 -> 58.
#include "gemm_shared.hpp"

namespace tlhip {
namespace q4 {

constexpr int kBM = 64, kBN = 256, kSlab = 32, kPlane = kBM * kSlab * 2, kImage = 2 * kPlane, kUnit = 4 * kImage;

__device__ __forceinline__ int image_off(int row, int chunk) {   // 16-byte chunk (8 k) of a row inside a plane
  return row * (kSlab * 2) + ((chunk ^ ((row >> 1) & 3)) << 4);
}

// One block per row of the images (rows past M are zero rows): the row's exponent and its two f16 terms. The row stays
// in registers between the two steps: up to RR runs of eight k per thread, K <= 2048 RR.
template <int RR>
__global__ __launch_bounds__(256) void q4_image_kernel(const float* __restrict__ A, int* __restrict__ ea, char* __restrict__ img,
                                                       int M, int K) {
  __shared__ uint32_t part[4];
  const int gm = blockIdx.x, t = threadIdx.x, k8 = K / 8, row = gm % kBM;
  typedef float f32x4 __attribute__((ext_vector_type(4)));
  f32x4 v[RR][2];
  uint32_t mx = 0;
  const f32x4* src = reinterpret_cast<const f32x4*>(A + (size_t)min(gm, M - 1) * K);
#pragma unroll
  for (int i = 0; i < RR; i++) {
    const int q = t + 256 * i;
    const bool in = q < k8 && gm < M;
#pragma unroll
    for (int h = 0; h < 2; h++) {
      v[i][h] = in ? src[2 * q + h] : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int e = 0; e < 4; e++) mx = max(mx, __float_as_uint(v[i][h][e]) & 0x7fffffffu);
    }
  }
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) mx = max(mx, (uint32_t)__shfl_xor((int)mx, d));
  if ((t & 63) == 0) part[t >> 6] = mx;
  __syncthreads();
  mx = max(max(part[0], part[1]), max(part[2], part[3]));
  const int e = row_exponent((int)(mx >> 23), mx == 0);
  const float s = pow2f(e);
  if (t == 0 && gm < M) ea[gm] = e;
  char* dst = img + (size_t)(gm / kBM) * (K / kSlab) * kImage;
#pragma unroll
  for (int i = 0; i < RR; i++) {
    const int q = t + 256 * i;                     // run q of the row: slab q / 4, chunk q % 4
    if (q >= k8) break;
    const f32x4 a = v[i][0] * s, b = v[i][1] * s;
    frag16 hi, lo;
#pragma unroll
    for (int p = 0; p < 4; p++) {                  // pairs (0 4) (1 5) (2 6) (3 7)
      uint32_t h2, l2;
      split2_f16<false>(a[p], b[p], h2, l2);
      hi[p] = h2;
      lo[p] = l2;
    }
    char* o = dst + (size_t)(q >> 2) * kImage + image_off(row, q & 3);
    *reinterpret_cast<frag16*>(o) = hi;
    *reinterpret_cast<frag16*>(o + kPlane) = lo;
  }
}

// eight nibbles of a word as f16 weights n - 8, k in the images' order. Masked into the last bits of 1024, upper nibbles sixteen
// times as large: the magic-number conversion of int4 weights (Kim et al., "Who Says Elephants Can't Run", 2022), from the f16 format.
__device__ __forceinline__ frag16 nib8(uint32_t w) {
  const f16x2 off = {(_Float16)-1032.0f, (_Float16)-1032.0f}, sixteenth = {(_Float16)0.0625f, (_Float16)0.0625f}, off16 = {(_Float16)-72.0f, (_Float16)-72.0f};
  const uint32_t u = w >> 8;
  auto low = [&](uint32_t x) { return __builtin_bit_cast(uint32_t, __builtin_bit_cast(f16x2, (x & 0x000f000fu) | 0x64006400u) + off); };
  auto high = [&](uint32_t x) {                    // 1024 + 16 n: (that) / 16 - 72, exact
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(__builtin_bit_cast(f16x2, (x & 0x00f000f0u) | 0x64006400u), sixteenth, off16));
  };
  return frag16{low(w), high(w), low(u), high(u)};
}

__device__ __forceinline__ f32x16 mma(const frag16& a, const frag16& b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

// Grid: x = row blocks (fastest) x column tiles, y = K-split parts of `part_units` units of 128 k; part y goes to
// C + y * M * ldc. n0 in tile columns; N = columns of this launch (gated: features), W and scales at its first row.
// GU: a wavefront's 64 columns are 32 gate features and their up rows (ff rows further down); under a split the raw
// parts are stored in that order and splitk_sum_swiglu_kernel gates after the sum.
template <bool GU>
__global__ __launch_bounds__(256, 2) void gemm_q4_kernel(const char* __restrict__ Aimg, const int* __restrict__ ea, const uint8_t* __restrict__ W,
                                                         const float* __restrict__ scales, float* __restrict__ C, int M, int N, int K,
                                                         int part_units, int ldc, int ff, int row_blocks) {
  typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
  extern __shared__ __attribute__((aligned(1024))) char ring[];   // two units of A
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l32 = lane & 31, half = lane >> 5;
  // (with parts in an XCD's run 301 x 3584 x 18944 in seven 106.1 -> 103.5 us, 130 x 4608 x 3584 27.5 -> 26.0)
  const BlockPlace place = block_place(gridDim.x, gridDim.y);
  const int rb = place.tile % row_blocks, n0 = place.tile / row_blocks * kBN;
  const int groups = K / kSlab, ubeg = place.part * part_units, nu = min((groups + 3) / 4, ubeg + part_units) - ubeg;
  C += (size_t)place.part * M * ldc;

  // this lane's columns (clamped: what lies past the edge is not stored)
  const uint8_t* wrow[2];
  const float* srow[2];
#pragma unroll
  for (int j = 0; j < 2; j++) {
    int64_t r;
    if (GU) r = min((n0 >> 1) + wave * 32 + l32, N - 1) + (j ? (int64_t)ff : 0);
    else r = min(n0 + wave * 64 + j * 32 + l32, N - 1);
    wrow[j] = W + r * (K / 2);
    srow[j] = scales + r * groups;
  }
  const char* asrc = Aimg + ((size_t)rb * groups + 4 * ubeg) * kImage;
  // my quarter of a unit's copy. Groups past the last are zeros in LDS: they are multiplied too, by a scale of zero, and an
  // infinity or NaN left there from another group would come through that.
  auto copy = [&](int u, int stage) {
    const int have = min(4, groups - 4 * (ubeg + u)) * (kImage / 1024);
    const auto piece = [&](int p) {
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(asrc + (size_t)u * kUnit + p * 1024 + lane * 16),
                                       (__attribute__((address_space(3))) void*)(ring + stage * kUnit + p * 1024), 16, 0, 0);
    };
    if (have == kUnit / 1024) {
#pragma unroll
      for (int i = 0; i < 8; i++) piece(wave * 8 + i);
    } else {
      for (int p = wave * 8; p < wave * 8 + 8; p++) {
        if (p < have) piece(p);
        else *reinterpret_cast<frag16*>(ring + stage * kUnit + p * 1024 + lane * 16) = frag16{0, 0, 0, 0};
      }
    }
  };
  struct Words { frag16 w[2][2]; f32x4u s[2]; };   // of a unit: [column tile][groups 0 1 | 2 3], the scales
  auto load_w = [&](Words& x, int u) __attribute__((always_inline)) {
    const int g0 = 4 * (ubeg + u);
#pragma unroll
    for (int j = 0; j < 2; j++) {
#pragma unroll
      for (int p = 0; p < 2; p++) x.w[j][p] = *reinterpret_cast<const frag16*>(wrow[j] + 16 * min(g0 + 2 * p + half, groups - 1));
      if (g0 + 4 <= groups) {
        x.s[j] = *reinterpret_cast<const f32x4u*>(srow[j] + g0);
      } else {
#pragma unroll
        for (int e = 0; e < 4; e++) x.s[j][e] = srow[j][min(g0 + e, groups - 1)];
      }
    }
  };
  frag16 w[2][2];                                  // of the unit in hand: [column tile][16-k step][group of the pair]
  f32x4u s[2];
  auto barrier = [] {                              // without the fence that would wait for every copy in flight
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };

  f32x16 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int v = 0; v < 16; v++) acc[i][j][v] = 0.f;
  int aoff[2];
#pragma unroll
  for (int ks = 0; ks < 2; ks++) aoff[ks] = image_off(l32, ks * 2 + half);   // (32 rows further down: 32 row lengths, the same swizzle)

  // A slab in two halves of 32 rows, i = 0 and 1. Between the matrix instructions of one half go the vector instructions of
  // its neighbours: the scales of the half before it, the nibbles of the next slab. Each half's eight products keep the matrix
  // pipe for 256 clocks; in a run of their own, as the scales after them, they kept the wavefront from issuing anything else.
  frag16 a[4], b[2][2];                            // A: [16-k step, term]; weights: [16-k step][column tile]
  f32x16 grp[2][2];                                // [half][column tile]: the sums of a group, its scales still to come
  float ps[2] = {0.f, 0.f};                        // those of the half before
#pragma unroll
  for (int j = 0; j < 2; j++)
#pragma unroll
    for (int v = 0; v < 16; v++) grp[1][j][v] = 0.f;
  auto fetch = [&](const char* at, int i, int q) __attribute__((always_inline)) { a[q] = *reinterpret_cast<const frag16*>(at + aoff[q >> 1] + (q & 1) * kPlane + i * 32 * kSlab * 2); };
  auto nibbles = [&](int g, int ks, int j) __attribute__((always_inline)) { b[ks][j] = nib8(w[j][g >> 1][2 * ks + (g & 1)]); };
  auto scaled = [&](int i, int q) __attribute__((always_inline)) {   // a quarter of half i's sums
#pragma unroll
    for (int v = 8 * (q & 1); v < 8 * (q & 1) + 8; v++) acc[i][q >> 1][v] = fmaf(grp[i][q >> 1][v], ps[q >> 1], acc[i][q >> 1][v]);
    asm volatile("" : "+v"(acc[i][q >> 1]));       // (here: the compiler would gather the slabs' scales, and spill their sums)
  };
  // next: where the slab after this one lies (nullptr: the unit ends)
  auto slab = [&](const char* at, const char* next, int g) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 2; i++) {
#pragma unroll
      for (int q = 0; q < 4; q++) {                // (the second terms first would cost precision at long K: 1.9e-7 for 1.3e-7)
        const int ks = q >> 1;
#pragma unroll
        for (int j = 0; j < 2; j++) grp[i][j] = mma(a[q], b[ks][j], q == 0 ? f32x16{} : grp[i][j]);
        if (i == 0) fetch(at, 1, q);
        else if (next) fetch(next, 0, q);
        scaled(1 - i, q);
        if (i == 0 && q < 2) nibbles(g, 1, q);
        if (i == 1 && q >= 2 && next) nibbles(g + 1, 0, q - 2);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int j = 0; j < 2; j++) ps[j] = s[j][g];
    }
  };
  // What was asked for of unit u has landed - my copies and loads, and my zeros where it lacks groups - and my reads of the unit
  // before it are done; past the barrier that holds for every wavefront. This stands where nothing younger is in flight, and names
  // the words' registers: the compiler takes copies and register loads to return out of order, so at the first use of a word it waits
  // for everything. With two units asked for ahead that was the whole latency of the second, once per unit (so, and with the rows' exponents
  // below asked for at once, a 301-token prompt of eight 7B layers 3912 -> 3746 us).
  auto landed = [&](Words& x, int u) __attribute__((always_inline)) {
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int j = 0; j < 2; j++) asm volatile("" : "+v"(x.w[j][0]), "+v"(x.w[j][1]), "+v"(x.s[j]));
    barrier();
    // words of groups (half) and 2 + (half): a half's k of both groups of a pair
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int p = 0; p < 2; p++) {
        const auto y = __builtin_amdgcn_permlane32_swap(x.w[j][p][0], x.w[j][p][1], false, false);
        const auto z = __builtin_amdgcn_permlane32_swap(x.w[j][p][2], x.w[j][p][3], false, false);
        w[j][p] = frag16{y[0], y[1], z[0], z[1]};  // [16-k step][group of the pair]
      }
    const int have = groups - 4 * (ubeg + u);      // groups past the last are multiplied, and scaled to nothing
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int g = 0; g < 4; g++) s[j][g] = g < have ? x.s[j][g] : 0.f;
  };
  {
    Words x;
    copy(0, 0);
    load_w(x, 0);
    landed(x, 0);
  }
  for (int u = 0;; u++) {
    Words x;
    const bool more = u + 1 < nu;
    if (more) {                                    // (everyone is done with that stage)
      copy(u + 1, (u + 1) & 1);
      load_w(x, u + 1);
    }
    __builtin_amdgcn_sched_barrier(0);
    const char* at = ring + (u & 1) * kUnit;
#pragma unroll
    for (int q = 0; q < 4; q++) fetch(at, 0, q);
#pragma unroll
    for (int j = 0; j < 2; j++) nibbles(0, 0, j);
#pragma unroll
    for (int g = 0; g < 4; g++) slab(at + g * kImage, g < 3 ? at + (g + 1) * kImage : nullptr, g);
    if (!more) break;
    landed(x, u + 1);
  }

#pragma unroll
  for (int q = 0; q < 4; q++) scaled(1, q);        // the last half's
  // acc[v] of lane l: row 8 (v / 4) + 4 (l / 32) + v % 4, column l % 32. The row's exponent comes back out, exactly.
  const int m0 = rb * kBM;
  int4 e4[2][4];                                   // four rows each; (past M: into the images behind the exponents, not used). Asked for one
#pragma unroll                                     // by one between the stores they were 32 round trips, each behind a store
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int g = 0; g < 4; g++) e4[i][g] = *reinterpret_cast<const int4*>(ea + m0 + i * 32 + 8 * g + 4 * half);
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int g = 0; g < 4; g++) asm volatile("" : "+v"(e4[i][g].x), "+v"(e4[i][g].y), "+v"(e4[i][g].z), "+v"(e4[i][g].w));   // (here, once)
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int v = 0; v < 16; v++) {
      const int gm = m0 + i * 32 + 8 * (v >> 2) + 4 * half + (v & 3);
      if (gm >= M) continue;
      const int4 q4 = e4[i][v >> 2];
      const int e = (v & 3) == 0 ? q4.x : (v & 3) == 1 ? q4.y : (v & 3) == 2 ? q4.z : q4.w;
      if (GU && gridDim.y == 1) {
        const int f = (n0 >> 1) + wave * 32 + l32;
        if (f >= N) continue;
        const float g = ldexpf(acc[i][0][v], -e), sg = 1.0f / (1.0f + expf(-g));   // swiglu_kernel's arithmetic
        C[(size_t)gm * ldc + f] = (g * sg) * ldexpf(acc[i][1][v], -e);
      } else {
#pragma unroll
        for (int j = 0; j < 2; j++) {
          const int gn = n0 + wave * 64 + j * 32 + l32;
          if (!GU && gn >= N) continue;            // gated parts are whole tiles wide
          C[(size_t)gm * ldc + gn] = ldexpf(acc[i][j][v], -e);
        }
      }
    }
}

}  // namespace q4

static int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

// can_split: the part sums work on float4s. Work is shaped to whole rounds of the 2 * CUs block slots: fewer tiles than slots
// -> K split; more -> the columns that make whole rounds with full K, the rest split over K in a second launch. The time, fitted to
// 400 runs (65 to 128 rows, N 256 .. 33000, K 256 .. 18944; error 6 %): 11.2 us for two launches, 4 per million numbers
// cut, a unit of 128 k 2.7 or, with two blocks on a CU, 4.1. Above 128 rows, to 11000 runs (129 to 1024 rows, N 128 .. 40000, K 128 ..
// 20480; error 7 %): the same and the outputs, with whole rounds of blocks: 14 x 37 tiles are two.
Q4Plan plan_gemm_q4(int64_t M, int64_t N, int64_t K, size_t parts_bytes, bool want_parts, bool gu, bool can_split) {
  using namespace q4;
  Q4Plan plan;
  const int per = gu ? 2 : 1;
  const int64_t cus = ctx().cus, w = kBN / per, rb = cdiv(M, kBM), tn = cdiv(N, w), slots = 2 * cus, units = cdiv(K / kSlab, 4);
  auto pick_S = [&](int64_t tiles) {
    if (!can_split || tiles >= slots) return 1;
    int64_t S = std::min<int64_t>(slots / tiles, 16);
    while (S > 1 && units / S < 2) S--;            // at least 256 k per part
    if (want_parts)
      while (S > 1 && (size_t)S * M * N * sizeof(float) > parts_bytes) S--;
    return (int)cdiv(units, cdiv(units, S));
  };
  const int64_t per_round = slots / rb;
  if (rb * tn <= slots || per_round == 0 || !can_split || want_parts) {
    plan.pieces[plan.npieces++] = {0, tn, pick_S(rb * tn)};
  } else {
    const int64_t main_tn = tn / per_round * per_round;
    plan.pieces[plan.npieces++] = {0, main_tn, 1};
    if (main_tn < tn) plan.pieces[plan.npieces++] = {main_tn, tn - main_tn, pick_S(rb * (tn - main_tn))};
  }
  const double outputs = 1e-6 * (double)M * (double)(per * N);
  if (M > 128) {
    plan.us = 9.8 + 2.7e-6 * (double)M * K + 0.88 * outputs + 9 * (plan.npieces - 1);
    for (int i = 0; i < plan.npieces; i++) {
      const Q4Plan::Piece& P = plan.pieces[i];
      const int64_t part_groups = std::min(4 * cdiv(units, P.S), K / kSlab);
      plan.us += (double)part_groups / 4 * rounds_us(rb * P.tcols * P.S, cus, 2.69, 3.7);
      if (P.S > 1) plan.us += 1.04e-6 * P.S * M * per * std::min<int64_t>(N, P.tcols * w) + (want_parts ? 0 : 3.3);
    }
    return plan;
  }
  plan.us = 11.2 + 4e-6 * (double)M * K;
  for (int i = 0; i < plan.npieces; i++) {
    const Q4Plan::Piece& P = plan.pieces[i];
    plan.us += (double)cdiv(units, P.S) * slab_us(rb * P.tcols * P.S, cus, 2.67, 4.1);
    if (P.S > 1) plan.us += 0.35e-6 * P.S * M * per * N * 4 + (want_parts ? 0 : kPartSumUs);
  }
  return plan;
}

// The three forms of gemm_bf16_nt_impl (prefill.hip), which has checked the arguments.
int gemm_q4_prompt(const Q4Plan& plan, const float* A, const uint8_t* W, const float* scales, float* C, int64_t M, int64_t N, int64_t K,
                   int* S_out, bool gu) {
  using namespace q4;
  Context& c = ctx();
  const int64_t w = gu ? kBN / 2 : kBN, rb = cdiv(M, kBM), groups = K / kSlab, units = cdiv(groups, 4);
  const bool want_parts = S_out != nullptr;
  const Q4Plan::Piece* pieces = plan.pieces;
  const int npieces = plan.npieces;
  const size_t ea_bytes = ((size_t)M * sizeof(int) + 1023) & ~(size_t)1023, img_bytes = (size_t)rb * groups * kImage;
  size_t parts_need = 0;
  if (!want_parts)
    for (int i = 0; i < npieces; i++)
      if (pieces[i].S > 1) {
        const int64_t part_w = gu ? pieces[i].tcols * kBN : std::min<int64_t>(pieces[i].tcols * w, N - pieces[i].tn0 * w);
        parts_need = std::max(parts_need, (size_t)pieces[i].S * M * part_w * sizeof(float));
      }
  char* sbase = static_cast<char*>(scratch(ea_bytes + img_bytes + parts_need));
  if (!sbase) return kNoScratch;
  int* ea = reinterpret_cast<int*>(sbase);
  char* img = sbase + ea_bytes;
  const auto image = [&](auto kernel) { kernel<<<dim3((unsigned)(rb * kBM)), dim3(256), 0, c.stream>>>(A, ea, img, (int)M, (int)K); };
  if (K <= 2048) image(q4_image_kernel<1>);
  else if (K <= 4096) image(q4_image_kernel<2>);
  else if (K <= 8192) image(q4_image_kernel<4>);
  else if (K <= 20480) image(q4_image_kernel<10>);
  else image(q4_image_kernel<16>);
  for (int i = 0; i < npieces; i++) {
    const Q4Plan::Piece& P = pieces[i];
    const int64_t n0 = P.tn0 * w, pn = std::min<int64_t>(P.tcols * w, N - n0), part_w = gu ? P.tcols * kBN : pn;
    const int S = P.S;
    const int64_t part_units = cdiv(units, S);
    float* dst = C + n0;
    int64_t ldc = N;
    if (want_parts) {
      *S_out = S;
    } else if (S > 1) {
      dst = reinterpret_cast<float*>(sbase + ea_bytes + img_bytes);
      ldc = part_w;
    }
    if (rb * P.tcols > 0x7fffffff || part_w > 0x7fffffff) return fail(TLHIP_EUNSUPPORTED, "tlhip_gemm_q4_nt: too many tiles for one grid");
    const dim3 grid((unsigned)(rb * P.tcols), (unsigned)S);
    const uint8_t* wp = W + (size_t)n0 * K / 2;
    const float* sp = scales + (size_t)n0 * groups;
    const auto run = [&](auto kernel, hipError_t set) {
      if (set != hipSuccess) return hip_fail(set, "hipFuncSetAttribute");
      kernel<<<grid, dim3(256), 2 * kUnit, c.stream>>>(img, ea, wp, sp, dst, (int)M, (int)pn, (int)K, (int)part_units, (int)ldc, (int)N, (int)rb);
      return 0;
    };
    static const hipError_t set_plain = hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_q4_kernel<false>), hipFuncAttributeMaxDynamicSharedMemorySize, 2 * kUnit);
    static const hipError_t set_gated = hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_q4_kernel<true>), hipFuncAttributeMaxDynamicSharedMemorySize, 2 * kUnit);
    if (int rc = gu ? run(gemm_q4_kernel<true>, set_gated) : run(gemm_q4_kernel<false>, set_plain)) return rc;
    if (S > 1 && !want_parts) launch_part_sum(dst, C + n0, M, pn, part_w, N, S, gu ? 32 : 0);
  }
  return TLHIP_OK;
}

}  // namespace tlhip
