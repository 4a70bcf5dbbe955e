// f32 products on the bf16 matrix pipe: C[M,N] = A[M,K] . op(B), operands cut into three bf16 terms.
//
// An f32 has 24 significant bits, a bf16 eight: rounding off one term after the other leaves a = a0 + a1 + a2 exactly, with a1 at
// most 2^-8 of a and a2 2^-17 (three bf16 terms for an f32 product: Henry, Tang and Heinecke, "Leveraging the bfloat16 Artificial
// Intelligence Datatype For Higher-Precision Computations", 2019). Of the nine products of a b the six with i + j <= 2 are summed. The
// others are at most 2^-24 of it, what one fp32 rounding may lose, 6e-9 of a dense result, and vanish where the product is itself a
// 24-bit number (integers stay exact, rows are selected exactly). v_mfma_f32_32x32x16_bf16 does sixteen times the multiply-adds of the
// fp32 pipe in a clock, so six of them are 2.7 times as fast, with 6 roundings of the sum per 16 k where that one has 8; they lean
// down where the fp32 pipe's do not (mean error -0.3e-7 to -0.7e-7 of a result's spread). Error against 64 bits beside the kernels that
// ran before, five shapes of K 896 to 4864 (2-norm): normal numbers 0.5 to 0.8 of theirs, all positive 0.45 to 1.15, spread over
// decades 0.4 to 0.8, rows with half their numbers zero 0.7 to 1.09. Sums of one product are the worst case: up to 1.43 units in the
// last place, 0.5 there. With the two pairs a1 b2 and a2 b1 too they are 1.0, 333 x 4864 x 896 takes 31 us for 27 (event time) and dense
// results are no nearer.
//
// Blocks and waves are those of sgemm_rows_kernel: the eight wavefronts of a block take the 16-k steps w, w + 8, ... of its
// 32 TM x 128 tile, operands go from memory to the registers that cut them up (so every number is cut once per block, without
// LDS and without a barrier), and the sums meet in LDS once, in a fixed order. What bounds it is the issue of a step's 24 TM matrix
// instructions and some 190 + 75 TM vector ones by two wavefronts a SIMD; a register's next load is asked for when the number
// in it has been cut up. us, this and the fp32 kernels: 333 x 4864 x 896 24.8 and 47.3, 333 x 896 x 4864 29 and 48, 150 x 4864 x 896 18
// and 26, 512 x 4864 x 896 47 and 63, 99 x 4608 x 3584 34 and 65, 291 x 3584 x 3584 69 and 116 (100 TFLOP/s of f32 products; the fp32
// pipe's peak is 157, and 60 to 80 were reached). With a tile's matrix instructions after the next tile's cuts instead of between
// them 333 x 4864 x 896 took 29.
//
// The cut is exact while no term is subnormal and none overflows. Each block keeps the largest and the smallest magnitude (of what is
// not zero) it read, and where those leave no room for that - infinities too, which must not meet the zeros of another number's
// lower terms - it does its tile again with the fp32 instruction.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "common.hpp"

namespace tlhip {
namespace split3 {

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x2u __attribute__((ext_vector_type(2), aligned(4)));   // rows need not be aligned
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kWaves = 8, kStep = 16, kBN = 128, kLD = kBN + 4;

struct Range {              // of the magnitudes read: `least` of what is not zero, as bits times two less one
  float most = 0.f;
  uint32_t least = 0xffffffffu;
  __device__ __forceinline__ void see(float a, float b) {
    // (four instructions; left to the compiler, which takes each magnitude by itself, seven)
    const uint32_t x = (__float_as_uint(a) << 1) - 1u, y = (__float_as_uint(b) << 1) - 1u;
    asm("v_max3_f32 %0, %1, |%2|, |%3|" : "=v"(most) : "v"(most), "v"(a), "v"(b));
    asm("v_min3_u32 %0, %1, %2, %3" : "=v"(least) : "v"(least), "v"(x), "v"(y));
  }
};

// numbers 2 i and 2 i + 1 of a lane's eight -> their three terms
struct Terms { u32x4 w[3]; };
__device__ __forceinline__ void cut(const float (&x)[8], Terms& t, Range& range, int i) {
  float a = x[2 * i], b = x[2 * i + 1];
  range.see(a, b);
#pragma unroll
  for (int p = 0; p < 3; p++) {
    const uint32_t h = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){a, b}, bf16x2));
    t.w[p][i] = h;
    if (p < 2) {
      a -= __uint_as_float(h << 16);
      b -= __uint_as_float(h & 0xffff0000u);
    }
  }
}

template <int TM, int TB>
__global__ __launch_bounds__(64 * kWaves, 2) void sgemm_split_kernel(const float* __restrict__ A, uint32_t lda, const float* __restrict__ B,
                                                                     uint32_t ldb, float* __restrict__ C, int M, int N, int K, float scale,
                                                                     float offset, int epi, int kchunk, int split) {
  constexpr int BM = 32 * TM;
  extern __shared__ __attribute__((aligned(16))) float sums[];
  __shared__ float seen_most[2][kWaves];
  __shared__ uint32_t seen_least[2][kWaves];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l32 = lane & 31, half = lane >> 5;
  // row blocks fastest: they read the same columns of B (with parts in an XCD's run 333 x 896 x 4864 29.1 -> 28.0 us)
  const int row_blocks = split & 0xffff;           // (split: row blocks | parts << 16)
  const BlockPlace place = block_place(gridDim.x, split >> 16);
  const int lid = place.tile;
  // (the last columns' tile is moved back to end with the matrix: it stores only the columns from `own` on, for those before them the
  // tile ahead of it may have taken the other way through the range check below)
  const int m0 = lid % row_blocks * BM, own = lid / row_blocks * kBN, n0 = min(own, N - kBN);
  const int kbeg = place.part * kchunk, kend = min(K, kbeg + kchunk);
  C += (size_t)place.part * M * N;                 // K-split parts are dense
  const int steps = (kend - kbeg) / kStep, mine = wave < steps ? (steps - wave + kWaves - 1) / kWaves : 0;
  // column tile j of this lane
  const auto column = [&](int j) { return n0 + (TB ? 32 * j + l32 : 64 * (j >> 1) + 2 * l32 + (j & 1)); };

  uint32_t arow[TM], bcol[4];                      // element offsets; rows past the edge repeat the last: not stored
#pragma unroll
  for (int t = 0; t < TM; t++) arow[t] = (uint32_t)min(m0 + 32 * t + l32, M - 1) * lda + 8 * half;
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const uint32_t c = (uint32_t)column(j);
    bcol[j] = TB ? c * ldb + 8 * half : 8 * half * ldb + c;
  }
  f32x16 acc[TM][4];
  const auto clear = [&]() {
#pragma unroll
    for (int t = 0; t < TM; t++)
#pragma unroll
      for (int j = 0; j < 4; j++)
#pragma unroll
        for (int v = 0; v < 16; v++) acc[t][j][v] = 0.f;
  };
  clear();

  float a[TM][8], b[4][8];
  const auto first_k = [&](int i) { return kbeg + kStep * (wave + kWaves * i); };
  const auto load_a = [&](int k) {
    const float* base = A + k;
#pragma unroll
    for (int t = 0; t < TM; t++)
#pragma unroll
      for (int h = 0; h < 2; h++) {
        const f32x4 v = *reinterpret_cast<const f32x4u*>(base + arow[t] + 4 * h);
#pragma unroll
        for (int e = 0; e < 4; e++) a[t][4 * h + e] = v[e];
      }
  };
  const auto load_b = [&](int g, int k) {          // column tiles 2 g and 2 g + 1
    if (TB) {
#pragma unroll
      for (int j = 2 * g; j < 2 * g + 2; j++)
#pragma unroll
        for (int h = 0; h < 2; h++) {
          const f32x4 v = *reinterpret_cast<const f32x4u*>(B + k + bcol[j] + 4 * h);
#pragma unroll
          for (int e = 0; e < 4; e++) b[j][4 * h + e] = v[e];
        }
    } else {
#pragma unroll
      for (int s = 0; s < 8; s++) {
        const float* row = B + (size_t)(k + s) * ldb;
        const f32x2 v = *reinterpret_cast<const f32x2u*>(row + bcol[2 * g]);
        b[2 * g][s] = v.x;
        b[2 * g + 1][s] = v.y;
      }
    }
  };
  // the ragged step: k past the end is zero on both sides (a zero against an infinity would not do)
  const auto load_ragged = [&]() {
    const int k = kbeg + steps * kStep + 8 * half;
#pragma unroll
    for (int s = 0; s < 8; s++) {
      const bool in = k + s < kend;
      const uint32_t kk = (uint32_t)min(k + s, kend - 1);
#pragma unroll
      for (int t = 0; t < TM; t++) {
        const float v = A[(size_t)(arow[t] - 8 * half) + kk];
        a[t][s] = in ? v : 0.f;
      }
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const float v = TB ? B[(size_t)(bcol[j] - 8 * half) + kk] : B[(size_t)kk * ldb + (bcol[j] - 8 * half * ldb)];
        b[j][s] = in ? v : 0.f;
      }
    }
  };
  const bool ragged = kbeg + steps * kStep < kend && wave == steps % kWaves;

  Range ra, rb;
  // A column tile's matrix instructions go out between the cuts of the next tile: a wavefront alone gets a vector instruction
  // in every 8 clocks, and a matrix instruction of 32 is no time lost for it.
  const auto step = [&](auto more, int next) {
    Terms ac[TM], bc[2];
#pragma unroll
    for (int i = 0; i < 4; i++) {
#pragma unroll
      for (int t = 0; t < TM; t++) cut(a[t], ac[t], ra, i);
      cut(b[0], bc[0], rb, i);
    }
    if (decltype(more)::value) load_a(next);
#pragma unroll
    for (int j = 0; j < 4; j++) {
      // the least terms first
      constexpr int pa[6] = {2, 0, 1, 1, 0, 0}, pb[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
      for (int i = 0; i < 4; i++) {
        if (j < 3) cut(b[j < 3 ? j + 1 : 0], bc[(j + 1) & 1], rb, i);
#pragma unroll
        for (int q = i * 6 * TM / 4; q < (i + 1) * 6 * TM / 4; q++) {
          const int p = q / TM, t = q % TM;
          acc[t][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, ac[t].w[pa[p]]), __builtin_bit_cast(bf16x8, bc[j & 1].w[pb[p]]),
                                                              acc[t][j], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      if (decltype(more)::value && (j & 1) == 0) load_b(j / 2, next);
    }
  };
  if (mine > 0) {
    load_a(first_k(0));
    load_b(0, first_k(0));
    load_b(1, first_k(0));
    for (int i = 1; i < mine; i++) step(std::true_type{}, first_k(i));
    step(std::false_type{}, 0);
  }
  if (ragged) {
    load_ragged();
    step(std::false_type{}, 0);
  }

  // ---- was there room for all terms? ---------------------------------------------------------------------------
  {
    const auto whole = [&](Range r) {
      r.most = wave_max(r.most);
#pragma unroll
      for (int d = 1; d < 64; d *= 2) r.least = min(r.least, (uint32_t)__shfl_xor((int)r.least, d, kWave));
      return r;
    };
    ra = whole(ra);
    rb = whole(rb);
    if (lane == 0) {
      seen_most[0][wave] = ra.most;
      seen_most[1][wave] = rb.most;
      seen_least[0][wave] = ra.least;
      seen_least[1][wave] = rb.least;
    }
    __syncthreads();
    float most[2] = {0.f, 0.f};
    uint32_t least[2] = {0xffffffffu, 0xffffffffu};
#pragma unroll
    for (int w = 0; w < kWaves; w++)
#pragma unroll
      for (int i = 0; i < 2; i++) {
        most[i] = fmaxf(most[i], seen_most[i][w]);
        least[i] = min(least[i], seen_least[i][w]);
      }
    // A term is at least the last place of its number, 2^-23 of its power of two, so from 2^-95 on none is subnormal. A product of two
    // second terms can be 2^-46 of the whole; of a product of 2^-95 or more, what the pipe drops below 2^-126 is 2^-31 at most.
    const auto room = [&](uint32_t x) { return (int)(x >> 24) - 127; };   // exponent of the least magnitude (zeros only: 128)
    const bool fits = most[0] < 0x1p100f && most[1] < 0x1p100f && most[0] * most[1] < 0x1p100f && room(least[0]) > -96 && room(least[1]) > -96 &&
                      room(least[0]) + room(least[1]) > -96;
    if (!fits) {
      clear();
      const auto exact = [&]() {
#pragma unroll
        for (int s = 0; s < 8; s++)
#pragma unroll
          for (int t = 0; t < TM; t++)
#pragma unroll
            for (int j = 0; j < 4; j++) acc[t][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[t][s], b[j][s], acc[t][j], 0, 0, 0);
      };
      for (int i = 0; i < mine; i++) {
        load_a(first_k(i));
        load_b(0, first_k(i));
        load_b(1, first_k(i));
        exact();
      }
      if (ragged) {
        load_ragged();
        exact();
      }
    }
  }

  // acc[t][j][v] of lane l: row 32 t + 8 (v / 4) + 4 (l / 32) + v % 4, column(j). Wavefronts 4..7 hand theirs to 0..3,
  // whose four sums everyone then adds up.
  float* slot = sums + (wave & 3) * BM * kLD;
  const auto put = [&](auto add) {
#pragma unroll
    for (int t = 0; t < TM; t++)
#pragma unroll
      for (int v = 0; v < 16; v++) {
        float* row = slot + (32 * t + 8 * (v >> 2) + 4 * half + (v & 3)) * kLD;
#pragma unroll
        for (int g = 0; g < 2; g++) {
          if (TB) {
#pragma unroll
            for (int e = 0; e < 2; e++) {
              float* p = row + 64 * g + 32 * e + l32;
              *p = decltype(add)::value ? acc[t][2 * g + e][v] + *p : acc[t][2 * g + e][v];
            }
          } else {
            f32x2* p = reinterpret_cast<f32x2*>(row + 64 * g + 2 * l32);
            f32x2 x = {acc[t][2 * g][v], acc[t][2 * g + 1][v]};
            if (decltype(add)::value) {
              const f32x2 o = *p;
              x.x += o.x;
              x.y += o.y;
            }
            *p = x;
          }
        }
      }
  };
  if (wave >= 4) put(std::false_type{});
  __syncthreads();
  if (wave < 4) put(std::true_type{});
  __syncthreads();
  const bool wide = (N & 3) == 0 && (reinterpret_cast<uintptr_t>(C) & 15) == 0;
  for (int i = tid; i < BM * (kBN / 4); i += 64 * kWaves) {
    const int row = i / (kBN / 4), c = i % (kBN / 4) * 4, gm = m0 + row, gn = n0 + c;
    if (gm >= M || gn + 3 < own) continue;
    const auto part = [&](int s) { return *reinterpret_cast<const f32x4*>(sums + (s * BM + row) * kLD + c); };
    f32x4 o = (part(0) + part(1)) + (part(2) + part(3));
    if (epi)
#pragma unroll
      for (int e = 0; e < 4; e++) o[e] = add_rn(mul_rn(o[e], scale), offset);
    float* dst = C + (size_t)gm * N + gn;
    if (wide) {                                    // (N and with it n0 are multiples of four: all or none of them are own)
      *reinterpret_cast<f32x4*>(dst) = o;
    } else if (gn >= own) {
#pragma unroll
      for (int e = 0; e < 4; e++) dst[e] = o[e];
    } else {
      for (int e = own - gn; e < 4; e++) dst[e] = e == 1 ? o[1] : e == 2 ? o[2] : o[3];
    }
  }
}

}  // namespace split3

using namespace split3;
void launch_sgemm_sum(const float* part, float* C, size_t n, int S, float scale, float offset, int epi);   // sgemm.hip

// 1: nothing launched, another kernel is the better one. other_us: the estimate of the best of those; other_steps: the 16-k
// steps that a wavefront of it adds up.
int launch_sgemm_split(const float* pa, int64_t lda, const float* pb, int64_t ldb, int tb, float* pc, int M, int N, int K, float scale,
                       float offset, int epi, double other_us, int other_steps) {
  // whole column tiles, a step for every wavefront, 32-bit element offsets
  if (N < kBN || K < kStep * kWaves || (int64_t)M * lda >= ((int64_t)1 << 32) || (tb ? (int64_t)N * ldb : 16 * ldb + N) >= ((int64_t)1 << 32)) return 1;
  // Row tiles and K splits (parts in scratch, summed in a fixed order) by an estimate in us, fitted to 1100 runs of 110 shapes
  // (17 to 1000 rows, 128 to 16000 columns, K 32 .. 5000; error 12 %, the pick within 0.3 % of the best on average): blocks
  // run one to a CU, and a round of them starts and ends and takes its steps of 16 k; parts are written and read, and their sum
  // is a launch. It has to be 15 % less than the others' (their errors are 6 to 15 %): all of the shapes it is then given
  // were faster, 1.03 to 2 times, 1.5 on average. At 10 % less it would also take 512 x 640 x 1001, a tenth faster, where one element
  // of a test against the CPU path came to 1.04 of its tolerance (the 64-bit result itself is at 0.995 there): results of other
  // bits are left alone where little is gained. A wavefront adds up no more than 1.4 times the
  // other kernel's steps: for as many its error on normal numbers is 0.8 of theirs, and grows with their root.
  const int cus = ctx().cus;
  double least = 0.85 * other_us;
  int TM = 0, S = 1;
  for (int tm = 1; tm <= 2; tm++)
    for (int s = 1; s <= 12 && (s == 1 || K / s >= 96); s++) {
      const int64_t blocks = (int64_t)((M + 32 * tm - 1) / (32 * tm)) * ((N + kBN - 1) / kBN) * s;
      const int n = ((K + s - 1) / s + kStep * kWaves - 1) / (kStep * kWaves);
      if (10 * n > 14 * std::max(other_steps, 1) && n > 1) continue;
      const double us = 2.5 + (double)((blocks + cus - 1) / cus) * (tm == 1 ? 2.0 + 1.765 * n : 3.16 + 2.405 * n) + (s > 1 ? 2.0 + 1.96e-6 * M * N * s : 0);
      if (us < least) { least = us; TM = tm; S = s; }
    }
  const int rb = TM ? (M + 32 * TM - 1) / (32 * TM) : 0;
  const int64_t tiles = (int64_t)rb * ((N + kBN - 1) / kBN);
  if (TM == 0 || tiles >= ((int64_t)1 << 23)) return 1;
  int kchunk = K;
  float* dst = pc;
  if (S > 1) {
    kchunk = ((K + S - 1) / S + kStep - 1) / kStep * kStep;
    S = (K + kchunk - 1) / kchunk;
    dst = S > 1 ? static_cast<float*>(scratch((size_t)S * M * N * sizeof(float))) : pc;
    if (!dst) return 1;                            // (a recording may not grow it)
  }
  const int kepi = S > 1 ? 0 : epi;
  const auto run = [&](auto tm, auto t_b) {
    constexpr int TM_ = decltype(tm)::value, TB_ = decltype(t_b)::value, lds = 4 * 32 * TM_ * kLD * (int)sizeof(float);
    static const hipError_t set = hipFuncSetAttribute(reinterpret_cast<const void*>(sgemm_split_kernel<TM_, TB_>),
                                                      hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (set != hipSuccess) return hip_fail(set, "hipFuncSetAttribute");
    sgemm_split_kernel<TM_, TB_><<<dim3((unsigned)tiles, (unsigned)S), dim3(64 * kWaves), lds, ctx().stream>>>(
        pa, (uint32_t)lda, pb, (uint32_t)ldb, dst, M, N, K, scale, offset, kepi, kchunk, rb | S << 16);   // (rows: up to 1024)
    return 0;
  };
  using std::integral_constant;
  const auto by_tm = [&](auto t_b) { return TM == 1 ? run(integral_constant<int, 1>{}, t_b) : run(integral_constant<int, 2>{}, t_b); };
  if (int rc = tb ? by_tm(integral_constant<int, 1>{}) : by_tm(integral_constant<int, 0>{})) return rc;
  if (S > 1) launch_sgemm_sum(dst, pc, (size_t)M * N, S, scale, offset, epi);
  return 0;
}

}  // namespace tlhip
