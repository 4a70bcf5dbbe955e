// General f32 GEMM of the tl::gpu seam on the fp32 matrix pipe:
//   C[M,N] = (op(A) . op(B)) * scale + offset,  op = identity or transposed view
// (cuda.h:1408-1460 `gemm`: lda / ldb row strides, ta / tb read a transposed view in
// place). This is what `array::dot` issues for rank-2 f32 operands with M > 1 (prompt-side
// matmuls of the array path, training-style graphs); the decode path never reaches it.
//
// v_mfma_f32_32x32x2_f32 multiplies f32 by f32 exactly and accumulates in fp32, so the
// result differs from the reference's FMA loops in summation order only. One instruction
// consumes ONE float per lane per operand - lane l supplies A[l % 32][l / 32] and
// B[l / 32][l % 32] - so both tiles sit in LDS k-major (As[k][m], Bs[k][n]): the 32 lanes of a
// half-wave then read 32 consecutive floats, conflict-free. An operand whose k index is
// contiguous in memory ([m][k] A, [n][k] B) is transposed on its way into LDS.
//
// 4 wavefronts (2 x 2) per block, 128 x 128 block tile, 64 x 64 per wavefront (2 x 2 MFMA
// tiles, 64 accumulator registers), K slabs of 16; the next slab's global loads are in
// flight while the current one is multiplied.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "common.hpp"

namespace tlhip {

typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kSgBM = 128, kSgBN = 128, kSgBK = 16, kSgPad = 4;

// One 128 x 16 operand tile, moved global -> registers -> LDS (k-major).
//   KC = true : k is the contiguous index in memory  (element (r, k) at base[r * ld + k])
//   KC = false: the tile's row index is contiguous   (element (r, k) at base[k * ld + r])
// r = row of A (m) or column of B (n). `fast` (block-uniform): the whole tile is inside the
// matrix and 16-byte loads are aligned; otherwise every element is bounds-checked.
template <bool KC>
struct TileMover {
  float4 reg[2];
  __device__ __forceinline__ void load(const float* __restrict__ base, int64_t ld, int r0, int k0, int R,
                                       int K, bool fast, int tid) {
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const int idx = tid + i * 256;
      if constexpr (KC) {
        const int r = idx >> 2, c4 = (idx & 3) * 4;          // 4 float4 along k per row
        const float* p = base + (int64_t)(r0 + r) * ld + k0 + c4;
        if (fast) {
          reg[i] = *reinterpret_cast<const float4*>(p);
        } else {
          float v[4];
#pragma unroll
          for (int j = 0; j < 4; j++) v[j] = (r0 + r < R && k0 + c4 + j < K) ? p[j] : 0.f;
          reg[i] = make_float4(v[0], v[1], v[2], v[3]);
        }
      } else {
        const int kk = idx >> 5, r4 = (idx & 31) * 4;        // 32 float4 along r per k row
        const float* p = base + (int64_t)(k0 + kk) * ld + r0 + r4;
        if (fast) {
          reg[i] = *reinterpret_cast<const float4*>(p);
        } else {
          float v[4];
#pragma unroll
          for (int j = 0; j < 4; j++) v[j] = (k0 + kk < K && r0 + r4 + j < R) ? p[j] : 0.f;
          reg[i] = make_float4(v[0], v[1], v[2], v[3]);
        }
      }
    }
  }
  __device__ __forceinline__ void store(float (*tile)[kSgBM + kSgPad], int tid) const {
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const int idx = tid + i * 256;
      if constexpr (KC) {
        const int r = idx >> 2, c4 = (idx & 3) * 4;
        tile[c4 + 0][r] = reg[i].x;
        tile[c4 + 1][r] = reg[i].y;
        tile[c4 + 2][r] = reg[i].z;
        tile[c4 + 3][r] = reg[i].w;
      } else {
        const int kk = idx >> 5, r4 = (idx & 31) * 4;
        *reinterpret_cast<float4*>(&tile[kk][r4]) = reg[i];
      }
    }
  }
};

// TA / TB as the seam passes them: TA = 0 means A is [M][K] (k contiguous), TA = 1 means the
// buffer holds [K][M]; TB = 0 means B is [K][N] (n contiguous), TB = 1 means [N][K].
template <int TA, int TB>
__global__ __launch_bounds__(256, 2) void sgemm_mfma_kernel(const float* __restrict__ A, int64_t lda,
                                                           const float* __restrict__ B, int64_t ldb,
                                                           float* __restrict__ C, int M, int N, int K,
                                                           float scale, float offset, int epi,
                                                           int aligned, int kchunk) {
  __shared__ __attribute__((aligned(16))) float As[kSgBK][kSgBM + kSgPad];
  __shared__ __attribute__((aligned(16))) float Bs[kSgBK][kSgBN + kSgPad];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int m0 = blockIdx.y * kSgBM, n0 = blockIdx.x * kSgBN;
  const bool inside = aligned && m0 + kSgBM <= M && n0 + kSgBN <= N;
  // gridDim.z > 1 is split-K: slice z takes K range [z * kchunk, (z + 1) * kchunk) (kchunk a
  // multiple of the slab) and writes its partial product, without the epilogue, to
  // C + z * M * N, a scratch area that sgemm_sum_kernel adds up in slice order.
  const int kbeg = blockIdx.z * kchunk;
  K = min(K, kbeg + kchunk);
  C += (size_t)blockIdx.z * M * N;

  f32x16 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int v = 0; v < 16; v++) acc[i][j][v] = 0.f;

  TileMover<TA == 0> ma;   // A: k contiguous unless transposed
  TileMover<TB != 0> mb;   // B: k contiguous only when transposed
  ma.load(A, lda, m0, kbeg, M, K, inside && kbeg + kSgBK <= K, tid);
  mb.load(B, ldb, n0, kbeg, N, K, inside && kbeg + kSgBK <= K, tid);
  for (int k0 = kbeg; k0 < K; k0 += kSgBK) {
    __syncthreads();   // the previous slab has been consumed
    ma.store(As, tid);
    mb.store(Bs, tid);
    __syncthreads();
    if (k0 + kSgBK < K) {
      const bool fast = inside && k0 + 2 * kSgBK <= K;
      ma.load(A, lda, m0, k0 + kSgBK, M, K, fast, tid);
      mb.load(B, ldb, n0, k0 + kSgBK, N, K, fast, tid);
    }
    const int kh = lane >> 5, l32 = lane & 31;
#pragma unroll
    for (int s = 0; s < kSgBK / 2; s++) {
      float a[2], b[2];
#pragma unroll
      for (int i = 0; i < 2; i++) a[i] = As[2 * s + kh][wm * 64 + i * 32 + l32];
#pragma unroll
      for (int j = 0; j < 2; j++) b[j] = Bs[2 * s + kh][wn * 64 + j * 32 + l32];
#pragma unroll
      for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], b[j], acc[i][j], 0, 0, 0);
    }
  }

  // acc[v] of lane l: row 8 * (v / 4) + 4 * (l / 32) + v % 4, column l % 32 of the 32 x 32 tile
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++) {
      const int gn = n0 + wn * 64 + j * 32 + (lane & 31);
      if (gn >= N) continue;
#pragma unroll
      for (int v = 0; v < 16; v++) {
        const int gm = m0 + wm * 64 + i * 32 + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
        if (gm < M) {
          const float r = acc[i][j][v];
          // separate multiply and add, like the CPU loops (array.h:1879, 2223)
          C[(size_t)gm * N + gn] = epi ? add_rn(mul_rn(r, scale), offset) : r;
        }
      }
    }
}

// C[i] = (sum over slices of part[s][i]) * scale + offset, slices in ascending order.
__global__ __launch_bounds__(256) void sgemm_sum_kernel(const float* __restrict__ part, float* __restrict__ C,
                                                        size_t n, int S, float scale, float offset, int epi) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const float a = sum_parts(S, [&](int s) { return part[(size_t)s * n + i]; });
  C[i] = epi ? add_rn(mul_rn(a, scale), offset) : a;
}

void launch_sgemm_sum(const float* part, float* C, size_t n, int S, float scale, float offset, int epi) {
  sgemm_sum_kernel<<<dim3((unsigned)((n + 255) / 256)), dim3(256), 0, ctx().stream>>>(part, C, n, S, scale, offset, epi);
}

// 16-byte loads need aligned bases and row strides that keep every row aligned
static bool sgemm_aligned(const float* pa, int64_t lda, const float* pb, int64_t ldb) {
  return aligned16(pa) && aligned16(pb) && (lda % 4) == 0 && (ldb % 4) == 0;
}
// Too few tiles to fill the chip: split K over gridDim.z (at least 256 of K per slice) into
// scratch parts that are summed in a fixed order - deterministic, no atomics.
static int sgemm_mfma_splits(int64_t tiles, int K) {
  int S = 1;
  if (tiles < ctx().cus) {
    S = (int)((2 * (int64_t)ctx().cus + tiles - 1) / tiles);
    if (S > 8) S = 8;
    while (S > 1 && K / S < 256) S--;
  }
  if (S > 1) {
    const int kchunk = ((K + S - 1) / S + kSgBK - 1) / kSgBK * kSgBK;
    S = (K + kchunk - 1) / kchunk;
  }
  return S;
}

// Launches the matrix-pipe GEMM; the caller has checked the arguments.
int launch_sgemm_mfma(const float* pa, int64_t lda, int ta, const float* pb, int64_t ldb, int tb, float* pc,
                      int M, int N, int K, float scale, float offset, int epi) {
  const int64_t tiles = (int64_t)((N + kSgBN - 1) / kSgBN) * ((M + kSgBM - 1) / kSgBM);
  const int S = sgemm_mfma_splits(tiles, K);
  int kchunk = K;
  float* dst = pc;
  if (S > 1) {
    kchunk = ((K + S - 1) / S + kSgBK - 1) / kSgBK * kSgBK;
    dst = static_cast<float*>(scratch((size_t)S * M * N * sizeof(float)));
    if (!dst) return fail(TLHIP_ENOMEM, "tlhip_gemm: no scratch for %d K-splits", S);
  }
  const dim3 grid((unsigned)((N + kSgBN - 1) / kSgBN), (unsigned)((M + kSgBM - 1) / kSgBM), (unsigned)S);
  const int aligned = sgemm_aligned(pa, lda, pb, ldb);
  hipStream_t st = ctx().stream;
  const int kepi = S > 1 ? 0 : epi;   // the part sum applies the epilogue when K is split
#define TLHIP_SGEMM(TA_, TB_)                                                                         \
  sgemm_mfma_kernel<TA_, TB_><<<grid, dim3(256), 0, st>>>(pa, lda, pb, ldb, dst, M, N, K, scale, offset, \
                                                          kepi, aligned, kchunk)
  if (!ta && !tb) TLHIP_SGEMM(0, 0);
  else if (!ta && tb) TLHIP_SGEMM(0, 1);
  else if (ta && !tb) TLHIP_SGEMM(1, 0);
  else TLHIP_SGEMM(1, 1);
#undef TLHIP_SGEMM
  if (S > 1) {
    launch_sgemm_sum(dst, pc, (size_t)M * N, S, scale, offset, epi);
  }
  return 0;
}

// ---- up to a few hundred rows -----------------------------------------------------------------------------
// C[M,N] = A[M,K] . op(B) without LDS in the loop: the eight wavefronts of a block split its K range between them
// (wavefront w takes the 16-k steps w, w + 8, ...), each with the whole 16 TM x 64 tile's accumulators, and both operands
// go from memory into the registers of v_mfma_f32_16x16x4_f32 that uses them, ST steps ahead; the sums meet in LDS
// once, in a fixed order. Lane l supplies row l % 16 of A and, of its quarter q = l / 16, the k 4 q .. 4 q + 3 of a step
// as one 16-byte load, one number per product; B is read four columns wide ([K][N]: columns 4 (l % 16) + j, rows
// 4 q + s, whole 256-byte runs) or like A ([N][K]).
// What bounds it: below about 64 rows reading B, above that the matrix pipe (32 clocks per 2048 operations; 60 to 80 of its
// 157 TFLOP/s, which is also what the LDS-tiled kernel above reaches). That one has two barriers per 16 k and reads
// ragged tiles element by element, the vector-ALU kernel of fewer than 128 rows had no K split at all. us, before ->
// now: 5 x 4864 x 896 164 -> 8.6, 5 x 896 x 4864 865 -> 10.7, 64 x 3584 x 3584 767 -> 32, 158 x 1153 x 901 41 -> 13,
// 333 x 4864 x 896 66 -> 47, 450 x 4608 x 3589 260 -> 218.
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));   // rows need not be 16-byte aligned

constexpr int kSrWaves = 8, kSrStep = 16, kSrBN = 64, kSrLD = kSrBN + 4;

template <int TM, int TB>
__global__ __launch_bounds__(64 * kSrWaves, 2) void sgemm_rows_kernel(const float* __restrict__ A, int64_t lda, const float* __restrict__ B,
                                                                      int64_t ldb, float* __restrict__ C, int M, int N, int K, float scale,
                                                                      float offset, int epi, int kchunk, int row_blocks) {
  constexpr int BM = 16 * TM, ST = TM <= 2 ? 4 : 3;
  extern __shared__ __attribute__((aligned(16))) float sums[];
  float (*red)[BM][kSrLD] = reinterpret_cast<float (*)[BM][kSrLD]>(sums);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r16 = lane & 15, quarter = lane >> 4;
  // row blocks fastest: they read the same columns of B (with parts in an XCD's run 90 x 896 x 4864 16.4 -> 15.7 us, 33 rows 11.9 -> 11.2)
  const BlockPlace place = block_place(gridDim.x, gridDim.y);
  const int lid = place.tile;
  const int m0 = lid % row_blocks * BM, n0 = lid / row_blocks * kSrBN;
  const int kbeg = place.part * kchunk, kend = min(K, kbeg + kchunk);
  C += (size_t)place.part * M * N;                 // K-split parts are dense
  // whole steps, the first `whole` of this block's range; what is left of K is one ragged step
  const int steps = (kend - kbeg) / kSrStep, mine = wave < steps ? (steps - wave + kSrWaves - 1) / kSrWaves : 0;
  const bool edge = n0 + kSrBN > N;                // (the block's last columns are read one by one, clamped)

  const float *arow[TM], *bcol[TB ? 4 : 1];
#pragma unroll
  for (int t = 0; t < TM; t++) arow[t] = A + (size_t)min(m0 + 16 * t + r16, M - 1) * lda;   // (rows past the edge: not stored)
  if (TB) {
#pragma unroll
    for (int j = 0; j < 4; j++) bcol[TB ? j : 0] = B + (size_t)min(n0 + 16 * j + r16, N - 1) * ldb;
  } else {
    bcol[0] = B + (edge ? 0 : n0 + 4 * r16);
  }
  f32x4 acc[TM][4];
#pragma unroll
  for (int t = 0; t < TM; t++)
#pragma unroll
    for (int j = 0; j < 4; j++) acc[t][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  f32x4 a[ST][TM], b[ST][4];                       // b: TB column tile j, k 4 q ..; else row 4 q + s, column tiles 0 .. 3
  auto load = [&](int u, int i) {
    const int k = kbeg + kSrStep * (wave + kSrWaves * i) + 4 * quarter;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      if (TB) {
        b[u][j] = *reinterpret_cast<const f32x4u*>(bcol[TB ? j : 0] + k);
      } else if (!edge) {
        b[u][j] = *reinterpret_cast<const f32x4u*>(bcol[0] + (size_t)(k + j) * ldb);
      } else {
#pragma unroll
        for (int e = 0; e < 4; e++) b[u][j][e] = bcol[0][(size_t)(k + j) * ldb + min(n0 + 4 * r16 + e, N - 1)];
      }
    }
#pragma unroll
    for (int t = 0; t < TM; t++) a[u][t] = *reinterpret_cast<const f32x4u*>(arow[t] + k);
    __builtin_amdgcn_sched_barrier(0);
  };
  auto compute = [&](int u) {
#pragma unroll
    for (int s = 0; s < 4; s++)
#pragma unroll
      for (int t = 0; t < TM; t++)
#pragma unroll
        for (int j = 0; j < 4; j++)
          acc[t][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u][t][s], TB ? b[u][j][s] : b[u][s][j], acc[t][j], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
  };
  // every load is of a step that exists: one past the end would cost what a real one costs
  int it = 0;
#pragma unroll
  for (int u = 0; u < ST; u++)
    if (u < mine) load(u, u);
  for (; it + 2 * ST <= mine; it += ST) {
#pragma unroll
    for (int u = 0; u < ST; u++) {
      compute(u);
      load(u, it + u + ST);
    }
  }
#pragma unroll
  for (int u = 0; u < ST; u++) {
    if (it + u < mine) compute(u);
    if (it + u + ST < mine) load(u, it + u + ST);
  }
#pragma unroll
  for (int u = 0; u < ST; u++)
    if (it + u + ST < mine) compute(u);
  // the ragged step: k past the end is zero on both sides (a zero against an infinity would not do)
  if (kbeg + steps * kSrStep < kend && wave == steps % kSrWaves) {
    const int k = kbeg + steps * kSrStep + 4 * quarter;
#pragma unroll
    for (int s = 0; s < 4; s++) {
      const bool in = k + s < kend;
      const int kk = min(k + s, kend - 1);
      float bv[4];
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const float v = TB ? bcol[TB ? j : 0][kk] : B[(size_t)kk * ldb + min(n0 + 4 * r16 + j, N - 1)];
        bv[j] = in ? v : 0.f;
      }
#pragma unroll
      for (int t = 0; t < TM; t++) {
        const float v = arow[t][kk], av = in ? v : 0.f;
#pragma unroll
        for (int j = 0; j < 4; j++) acc[t][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(av, bv[j], acc[t][j], 0, 0, 0);
      }
    }
  }

  // acc[t][j][v] of lane l: row 16 t + 4 (l / 16) + v, column l % 16 of column tile j. Wavefronts 4..7 hand theirs to
  // 0..3, whose four sums everyone then adds up.
  auto entry = [&](float* dst, int t, int v) { return dst + (16 * t + 4 * quarter + v) * kSrLD + (TB ? r16 : 4 * r16); };
  auto put = [&](float* dst) {
#pragma unroll
    for (int t = 0; t < TM; t++)
#pragma unroll
      for (int v = 0; v < 4; v++) {
        float* p = entry(dst, t, v);
        if (TB) {
#pragma unroll
          for (int j = 0; j < 4; j++) p[16 * j] = acc[t][j][v];
        } else {
          *reinterpret_cast<f32x4*>(p) = f32x4{acc[t][0][v], acc[t][1][v], acc[t][2][v], acc[t][3][v]};
        }
      }
  };
  float* slot = &red[wave & 3][0][0];
  if (wave >= 4) put(slot);
  __syncthreads();
  if (wave < 4) {
#pragma unroll
    for (int t = 0; t < TM; t++)
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const float* p = entry(slot, t, v);
        if (TB) {
#pragma unroll
          for (int j = 0; j < 4; j++) acc[t][j][v] += p[16 * j];
        } else {
          const f32x4 x = *reinterpret_cast<const f32x4*>(p);
#pragma unroll
          for (int j = 0; j < 4; j++) acc[t][j][v] += x[j];
        }
      }
    put(slot);
  }
  __syncthreads();
  const bool wide = (N & 3) == 0 && (reinterpret_cast<uintptr_t>(C) & 15) == 0;
  for (int i = tid; i < BM * (kSrBN / 4); i += 64 * kSrWaves) {
    const int row = i / (kSrBN / 4), c = i % (kSrBN / 4) * 4, gm = m0 + row, gn = n0 + c;
    if (gm >= M || gn >= N) continue;
    f32x4 o = (*reinterpret_cast<const f32x4*>(&red[0][row][c]) + *reinterpret_cast<const f32x4*>(&red[1][row][c])) +
              (*reinterpret_cast<const f32x4*>(&red[2][row][c]) + *reinterpret_cast<const f32x4*>(&red[3][row][c]));
    if (epi)
#pragma unroll
      for (int e = 0; e < 4; e++) o[e] = add_rn(mul_rn(o[e], scale), offset);
    float* dst = C + (size_t)gm * N + gn;
    if (wide) {
      *reinterpret_cast<f32x4*>(dst) = o;
    } else {
#pragma unroll
      for (int e = 0; e < 4; e++)
        if (gn + e < N) dst[e] = o[e];
    }
  }
}

int launch_sgemm_split(const float* pa, int64_t lda, const float* pb, int64_t ldb, int tb, float* pc, int M, int N, int K, float scale,
                       float offset, int epi, double other_us, int other_steps);
// The same for A as it is stored ([M][K]); the caller has checked the arguments. tiled: the LDS-tiled kernel takes the
// product too, else the vector-ALU kernel; 1 is returned, and nothing launched, where that is the better one. whole: the
// LDS-tiled kernel is better than this one in any case. Ahead of either goes the product in bf16 terms (sgemm_split.hip) where its
// estimate is the least.
int launch_sgemm_rows(const float* pa, int64_t lda, const float* pb, int64_t ldb, int tb, float* pc, int M, int N, int K, float scale,
                      float offset, int epi, bool tiled, bool whole) {
  // Row blocks and K splits (parts in scratch, summed in a fixed order) that an estimate in clocks likes best: a block
  // takes 1600 clocks per row tile and 128 k, and 6000 to start and end; blocks run one to a CU, so tiles that make a
  // round and a bit are cut smaller until they make whole rounds; parts are written and read at 2.5 KB a clock, and their
  // launch is 11000. (333 x 3584 x 3584: 175 us with 336 tiles of full K, 128 with three splits.)
  const int t16 = (M + 15) / 16, cus = ctx().cus;
  const int64_t columns = (N + kSrBN - 1) / kSrBN;
  int rb = 1, TM = 1, S = 1;
  double least = -1;
  for (int r = (t16 + 3) / 4; r <= (t16 + 3) / 4 + 2 && r <= t16; r++) {
    const int tm = (t16 + r - 1) / r;
    for (int s = 1; s <= 16 && (s == 1 || K / s >= 64); s++) {
      const double rounds = (double)((r * columns * s + cus - 1) / cus), steps = (double)(((K + s - 1) / s + 127) / 128);
      const double t = rounds * (steps * 1600 * tm + 6000) + (s > 1 ? 11000 + 8.0 * s * M * N / 2500 : 0);
      if (least < 0 || t < least) { least = t; rb = r; TM = tm; S = s; }
    }
  }
  // The LDS-tiled kernel is the better one where blocks in several rounds each start and end for a few steps, and for many
  // columns of a middling K (986 x 7459 x 22: 15 us, 42 here; 864 x 18126 x 308 117 and 181; but 300 x 2000 x 60 11 and 7.6). Both
  // times in us, fitted to 2210 runs (128 to 1024 rows, 128 to 150000 columns, K 16 .. 5000; errors 8 and 6 %): a start; for every
  // round of blocks its own start and end and its steps of 16 k (per row tile here); the outputs' megabytes, twice for parts; and
  // the launch that adds those up.
  const int64_t tiles128 = (int64_t)((N + kSgBN - 1) / kSgBN) * ((M + kSgBM - 1) / kSgBM);
  const int St = sgemm_mfma_splits(tiles128, K);
  const auto steps = [&](int parts) { return (double)(((K + parts - 1) / parts + kSgBK - 1) / kSgBK); };
  const auto mb = [&](int parts) { return 4e-6 * M * N * (parts > 1 ? 2 * parts : 1); };
  const double here = 2.2 + std::ceil((double)rb * columns * S / cus) * (1.15 + TM * (0.25 + (tb ? 0.81 : 0.72) * steps(S) / kSrWaves)) +
                      0.28 * mb(S) + (S > 1 ? 2.2 : 0);
  const double fill = (double)tiles128 * St / cus;   // blocks run two to a CU, and the last round's gaps are partly filled
  const double there = 5.5 + std::max(1.0, 0.14 * fill + 0.86 * std::ceil(fill)) *
                                 (steps(St) * (sgemm_aligned(pa, lda, pb, ldb) ? 1.41 : 1.57) - 1) + 0.16 * mb(St) + (St > 1 ? 7.9 : 0);
  const bool to_tiles = whole || (tiled && here > 1.02 * there);
  // (a wavefront of the LDS-tiled kernel adds up all of its block's K, here an eighth)
  if (const int rc = launch_sgemm_split(pa, lda, pb, ldb, tb, pc, M, N, K, scale, offset, epi, to_tiles ? there : here,
                                        (int)steps(to_tiles ? St : S) / (to_tiles ? 1 : kSrWaves)); rc != 1) return rc;
  // (its parts need scratch, which a recording may not grow: the product stays here then)
  if (to_tiles && (whole || St == 1 || scratch((size_t)St * M * N * sizeof(float)))) return 1;
  const int64_t tiles = rb * columns;
  // Fewer than 128 rows or columns, which is what the vector-ALU kernel is left with: more than one, two and four rounds of
  // these blocks for K up to 16, 32 and 47 cost more than its 64 x 64 tiles, which meet no one at their end (us, here and there: 100 x
  // 25000 x 16 15 and 10, 127 x 60000 x 20 32 and 24, 100 x 60000 x 33 31 and 28; 64 x 12000 x 16 4.6 and 5.6). Up to 32 rows leave
  // half of such a tile empty: twice the rounds (26 x 102934 x 24 22 and 15, 16 x 30000 x 16 4.0 and 5.0).
  if (!tiled && K < 48 && M > 16 && tiles >> ((K + 15) / 16 - (M > 32 ? 1 : 0)) > cus) return 1;
  int kchunk = K;
  float* dst = pc;
  if (S > 1) {
    kchunk = ((K + S - 1) / S + kSrStep - 1) / kSrStep * kSrStep;
    S = (K + kchunk - 1) / kchunk;
    dst = S > 1 ? static_cast<float*>(scratch((size_t)S * M * N * sizeof(float))) : pc;
    if (!dst) {                                    // no scratch to be had (a recording may not grow it): no parts
      dst = pc;
      S = 1;
      kchunk = K;
    }
  }
  const dim3 grid((unsigned)tiles, (unsigned)S);
  const int kepi = S > 1 ? 0 : epi;
  const auto run = [&](auto tm, auto t_b) {
    constexpr int TM_ = decltype(tm)::value, TB_ = decltype(t_b)::value, lds = 4 * 16 * TM_ * kSrLD * (int)sizeof(float);
    static const hipError_t set = hipFuncSetAttribute(reinterpret_cast<const void*>(sgemm_rows_kernel<TM_, TB_>),
                                                      hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (set != hipSuccess) return hip_fail(set, "hipFuncSetAttribute");
    sgemm_rows_kernel<TM_, TB_><<<grid, dim3(64 * kSrWaves), lds, ctx().stream>>>(pa, lda, pb, ldb, dst, M, N, K, scale, offset, kepi, kchunk, rb);
    return 0;
  };
  using std::integral_constant;
  const auto by_tm = [&](auto t_b) {
    return TM == 1 ? run(integral_constant<int, 1>{}, t_b) : TM == 2 ? run(integral_constant<int, 2>{}, t_b)
         : TM == 3 ? run(integral_constant<int, 3>{}, t_b) : run(integral_constant<int, 4>{}, t_b);
  };
  if (int rc = tb ? by_tm(integral_constant<int, 1>{}) : by_tm(integral_constant<int, 0>{})) return rc;
  if (S > 1) {
    launch_sgemm_sum(dst, pc, (size_t)M * N, S, scale, offset, epi);
  }
  return 0;
}

}  // namespace tlhip
