// Products of a few rows: C[M,N] = A[M,K] f32 . W[N,K]^T for a short prompt, W bf16 rows or int4 groups.
//
// What bounds it: with M of a few dozen the weight is read once and hardly reused, and what is left is the
// chain of latencies of one block. gemm_bf16_nt_kernel (prefill.hip) walks K in slabs of 32 through LDS, two
// barriers and one load round trip per slab: ten slabs were 20 us for weights that take 2 us to read. Here a
// block has no barrier until its sums are complete: its eight wavefronts split the block's K range between
// them (wavefront w takes the 32-k steps w, w + 8, ...), each with the WHOLE tile's accumulators; both operands come
// through slots of LDS of the wavefront's own (int4 weights straight into registers). The sums meet in
// LDS once at the end, in a fixed order.
//
// Both operands of v_mfma_f32_16x16x32_bf16 are K-contiguous per lane: lane l supplies row l % 16 and k
// 8 (l / 16) .. + 8 - one 16-byte load of a bf16 weight (64 contiguous bytes of every row), two of an f32
// activation (128). Every activation is cut exactly into three bf16 terms in registers (gemm_bf16_nt_kernel's
// arithmetic: exact products, fp32 sums). Tiles of 16 rows waste less of a ragged M than tiles of 32 or 64.
//
// int4: a lane's 16-byte load is the 32 weights of ONE scale group; four groups lie in the four lane quarters
// and are traded (two swaps of lane halves, two of 16-lane rows, for four steps) so that a step multiplies one
// group: its sums start at zero and join the accumulators times the group's scale, as in gemm_bf16_nt_kernel.
//
// int4 above 64 rows (RANGED): the other kernels for these products scale every row of A by its exponent, so a row of
// any finite magnitude comes out right there, while three bf16 terms as they are lose their last bits below 2^-110 and
// a group's sum of 256 times the magnitude overflows above 2^119. Both show in the results, as values that are not
// finite or as four in a row that are tiny. Only then does a block look for its rows' largest magnitudes, and only where
// one is outside 2^-100 .. 2^100 does it multiply once more with scaled rows and store what comes out of that.
#include <type_traits>

#include "gemm_shared.hpp"

namespace tlhip {
namespace rows {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kWaves = 8, kStep = 32;
constexpr int kMaxTM = 5;

// int4: steps of activations in flight per wavefront (a divisor of four), 2 KB of LDS per row tile each
__host__ __device__ constexpr int stages(int TM) { return TM <= 2 ? 4 : 2; }
__host__ __device__ constexpr int lds_bytes_q4(int TM, int TN) {
  const int ring = kWaves * stages(TM) * TM * 2048, sums = 4 * 16 * TM * (16 * TN + 4) * 4;
  return ring > sums ? ring : sums;
}
// bf16: steps of activations in flight - one, or where a step's loads are few, two and four (8 x 446 x 12032 34.0 -> 28.5 us) -
// and the sums of all wavefronts. Rows of four column tiles lie without padding, their 16-byte chunks XORed with the row (160 KB
// at five row tiles).
__host__ __device__ constexpr int steps_ahead(int TM, int TN) { return TM == 1 && TN <= 2 ? 4 / TN : 1; }
__host__ __device__ constexpr int sum_stride(int TN) { return TN == 4 ? 16 * TN : 16 * TN + 4; }
// Steps of weights in LDS: one more than of activations, or one where only so two blocks fit a CU (128 x 4864 gated x 896, four row tiles
// over two column tiles: 19.0 us so, 21.0 with one block and two steps).
__host__ __device__ constexpr int ring_bf16(int TM, int TN, int WS) { return kWaves * (steps_ahead(TM, TN) * TM * 2048 + WS * TN * 1024); }
__host__ __device__ constexpr int sums_bf16(int TM, int TN) { return kWaves * 16 * TM * sum_stride(TN) * 4; }
__host__ __device__ constexpr int weight_steps(int TM, int TN) {
  const int AS = steps_ahead(TM, TN), half = 80 * 1024;
  return AS == 1 && ring_bf16(TM, TN, 2) > half && ring_bf16(TM, TN, 1) <= half && sums_bf16(TM, TN) <= half ? 1 : AS + 1;
}
__host__ __device__ constexpr int lds_bytes_bf16(int TM, int TN) {
  const int ring = ring_bf16(TM, TN, weight_steps(TM, TN)), sums = sums_bf16(TM, TN);
  return ring > sums ? ring : sums;
}
// Blocks of [row tiles - 1][column tiles - 1] that fit a CU: by their registers, as the compiler reports them (two wavefronts a SIMD each), and
// by the LDS above, of which a CU has 160 KB. The plan prices rounds of blocks by it.
struct BlocksOfACu {
  int n[kMaxTM][4] = {{4, 4, 4, 2}, {4, 3, 2, 2}, {3, 2, 2, 1}, {3, 3, 1, 1}, {2, 2, 1, 1}};
  constexpr BlocksOfACu() {
    for (int TM = 1; TM <= kMaxTM; TM++)
      for (int TN = 1; TN <= 4; TN++) {
        const int by_lds = 160 * 1024 / lds_bytes_bf16(TM, TN);
        if (by_lds < n[TM - 1][TN - 1]) n[TM - 1][TN - 1] = by_lds;
      }
  }
};

// 8 floats -> their three bf16 terms (by truncation: x = hi + mid + lo exactly for normal x)
__device__ __forceinline__ void split3(const f32x4& x0, const f32x4& x1, frag16 p[3]) {
  const float x[8] = {x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
#pragma unroll
  for (int b = 0; b < 4; b++) {
    const uint32_t u0 = __float_as_uint(x[2 * b]), u1 = __float_as_uint(x[2 * b + 1]);
    const float r0 = x[2 * b] - __uint_as_float(u0 & 0xffff0000u), r1 = x[2 * b + 1] - __uint_as_float(u1 & 0xffff0000u);
    const uint32_t m0 = __float_as_uint(r0), m1 = __float_as_uint(r1);
    const float s0 = r0 - __uint_as_float(m0 & 0xffff0000u), s1 = r1 - __uint_as_float(m1 & 0xffff0000u);
    p[0][b] = __builtin_amdgcn_perm(u1, u0, 0x07060302u);
    p[1][b] = __builtin_amdgcn_perm(m1, m0, 0x07060302u);
    p[2][b] = __builtin_amdgcn_perm(__float_as_uint(s1), __float_as_uint(s0), 0x07060302u);
  }
}

// 8 nibbles (k ascending, value = nibble - 8) -> 8 bf16, exact
__device__ __forceinline__ frag16 nib8(uint32_t w) {
  const uint32_t lo = w & 0x0f0f0f0fu, hi = (w >> 4) & 0x0f0f0f0fu;   // even k, odd k
  frag16 o;
#pragma unroll
  for (int b = 0; b < 4; b++) {
    const float e = (float)((lo >> (8 * b)) & 0xffu) - 8.0f, d = (float)((hi >> (8 * b)) & 0xffu) - 8.0f;
    o[b] = __builtin_amdgcn_perm(__float_as_uint(d), __float_as_uint(e), 0x07060302u);
  }
  return o;
}

__device__ __forceinline__ f32x4 mma(const frag16& a, const frag16& b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// Grid: x = row blocks (fastest) x column tiles, y = K-split parts of `part_units` units (bf16: steps of 32 k,
// int4: 128 k); part y goes to C + y * M * ldc. N, ff, GU and the order of a gated tile's columns as in
// gemm_bf16_nt_kernel: a tile's first 8 TN columns are gate features, the rest the same features' up rows.
//
// What bounds the bf16 kernel: the CU returns loads in the order of their requests, so activations (from L2, read by every
// block: 2.5 times the weights' bytes at five row tiles over four column tiles) wait behind weights from HBM. 77 x 9728 gated x 896
// took 14.5 us, 10.0 without the weights' loads, 11.3 without the activations', 8.7 without both, and no less without the
// matrix instructions. So little is in flight beyond what is needed next - one step of activations, each tile requested again
// as soon as it is in registers, two steps of weights - and three column tiles (203 blocks instead of 152) are a choice too:
// 12.3 us. With two steps of activations 13.2, all weights first 12.8. 227 shapes of 1 to 80 rows: 0.98 to 1.4 times as fast.
// Weights in LDS like the activations, and what the first copies need from registers and without a division: 145 shapes of 2 to 300
// rows 1.08 times as fast, 0.98 to 1.18 (37 x 4608 x 3584 16.0 -> 14.4 us, 77 x 4864 gated x 896 12.2 -> 11.4).
template <int TM, int TN, bool GU>
__global__ __launch_bounds__(64 * kWaves, 2) void gemm_rows_bf16_kernel(const float* __restrict__ A, const void* __restrict__ W,
                                                                       float* __restrict__ C, int M, int N, int K, int part_units,
                                                                       int ldc, int ff, int split) {
  constexpr int BM = 16 * TM, BN = 16 * TN, LD = sum_stride(TN), AS = steps_ahead(TM, TN), WS = weight_steps(TM, TN);
  extern __shared__ __attribute__((aligned(1024))) float red[];   // operands in flight, then [8][BM][LD] sums
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r16 = lane & 15, quarter = lane >> 4;
  // row blocks fastest: those share a weight tile in one L2 (split: row blocks | parts << 16, parts 1 where the grid's y is the part;
  // the grid's size from the arguments, which are in registers already, and no division where one block holds all rows)
  constexpr int TW = GU ? BN / 2 : BN;
  const int row_blocks = split & 0xffff;
  const BlockPlace place = block_place(row_blocks * ((N + TW - 1) / TW), split >> 16);
  const int lid = place.tile;
  const int tile = row_blocks == 1 ? lid : lid / row_blocks;
  const int m0 = (lid - tile * row_blocks) * BM, n0 = tile * BN;
  C += (size_t)place.part * M * ldc;
  const int units = K / kStep, ubeg = place.part * part_units, uend = min(units, ubeg + part_units);
  const int first = ubeg + wave, mine = first < uend ? (uend - first + kWaves - 1) / kWaves : 0;

  // byte offsets of this lane's rows (clamped into the operands: what lies past an edge is not stored). A 1 KB copy
  // of activations is eight rows of 128 bytes, the 16-byte chunks of row r in the order c ^ (r & 7), which spreads
  // the fragment reads (16 rows, one chunk) over the LDS banks; of weights sixteen rows of 64, in the order c ^ (r / 2 & 3).
  uint32_t aoff[TM][2], woff[TN];
#pragma unroll
  for (int j = 0; j < TN; j++) {
    const int col = 16 * j + (lane >> 2);
    int r;
    if (GU) {
      const int f = min((n0 >> 1) + col % (BN / 2), N - 1);
      r = f + (col >= BN / 2 ? ff : 0);
    } else {
      r = min(n0 + col, N - 1);
    }
    woff[j] = (uint32_t)r * (uint32_t)(K * 2) + ((lane & 3) ^ (lane >> 3 & 3)) * 16;
  }
#pragma unroll
  for (int t = 0; t < TM; t++)
#pragma unroll
    for (int h = 0; h < 2; h++)
      aoff[t][h] = (uint32_t)min(m0 + 16 * t + 8 * h + (lane >> 3), M - 1) * (uint32_t)(K * 4) + ((lane & 7) ^ (lane >> 3)) * 16;
  const int frag[2] = {r16 * 128 + ((2 * quarter) ^ (r16 & 7)) * 16, r16 * 128 + ((2 * quarter + 1) ^ (r16 & 7)) * 16};
  const int wfrag = r16 * 64 + (quarter ^ (r16 >> 1 & 3)) * 16;
  char* slots = reinterpret_cast<char*>(red) + wave * (AS * TM * 2048 + WS * TN * 1024);
  char* wslots = slots + AS * TM * 2048;
  const char* Ab = reinterpret_cast<const char*>(A) + (uint32_t)first * 128u;
  const char* Wb = static_cast<const char*>(W) + (uint32_t)first * 64u;

  f32x4 acc[TM][TN];
#pragma unroll
  for (int t = 0; t < TM; t++)
#pragma unroll
    for (int j = 0; j < TN; j++) acc[t][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  // Both operands are copied into LDS: weights loaded into registers, beside the activations' copies, were taken by the compiler to
  // return out of order with those, and at the first use of every second step's it waited for all that was in flight.
  auto load_a = [&](char* slot, int t, uint32_t i) {   // row tile t of my i-th step
#pragma unroll
    for (int h = 0; h < 2; h++)
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(Ab + (aoff[t][h] + i * (kWaves * 128u))),
                                       (__attribute__((address_space(3))) void*)(slot + t * 2048 + h * 1024), 16, 0, 0);
  };
  auto load_w = [&](int u, uint32_t i) {
#pragma unroll
    for (int j = 0; j < TN; j++)
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(Wb + (woff[j] + i * (kWaves * 64u))),
                                       (__attribute__((address_space(3))) void*)(wslots + (u * TN + j) * 1024), 16, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
  };
  // My i-th step, weights in slot U, activations in `slot`. R: later steps, capped at WS. Requests go out in the order W(0), A(0),
  // W(1), .., W(AS), then in step i A(i + AS, t) as tile t leaves its slot and W(i + WS) at the end (of one slot W(i + 1) as it
  // is read): what is younger than A(i, t) is counted, and W(i) is older (copies into LDS are waited for by count). W(i + WS) takes the
  // slot that W(i) was read from, by fragments that have arrived.
  auto step = [&](auto U, auto R_, uint32_t i, char* slot) {
    constexpr int u = decltype(U)::value, R = decltype(R_)::value, ahead = R < AS - 1 ? R : AS - 1;
    frag16 w[TN];
    const auto tile = [&](auto T) {
      constexpr int t = decltype(T)::value;
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * (TM - 1 - t) + ahead * (TN + 2 * TM) + (R >= AS ? (WS == 1 && t == 0 ? 0 : TN) + 2 * t : 0)) : "memory");
      const char* at = slot + t * 2048;
      const f32x4 x0 = *reinterpret_cast<const f32x4*>(at + frag[0]), x1 = *reinterpret_cast<const f32x4*>(at + frag[1]);
      if constexpr (t == 0) {
#pragma unroll
        for (int j = 0; j < TN; j++) w[j] = *reinterpret_cast<const frag16*>(wslots + (u * TN + j) * 1024 + wfrag);
      }
      if constexpr (R >= AS) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // read before the copy that takes the slot goes out
        if constexpr (WS == 1 && t == 0) load_w(0, i + 1);
        load_a(slot, t, i + AS);
      }
      frag16 p[3];
      split3(x0, x1, p);
      // the weights are the first operand: the tile comes out transposed, four consecutive columns of a row to a lane.
      // (The small terms first would have 0.85 of the spread, but rounding goes one way and three times the mean error adds up over
      // the layers: a 0.5B prompt 2.2e-7 -> 2.8e-7.)
#pragma unroll
      for (int e = 0; e < 3; e++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[t][j] = mma(w[j], p[e], acc[t][j]);
      if (TM * TN >= 12) __builtin_amdgcn_sched_barrier(0);   // (the registers do not hold two row tiles' terms)
    };
    tile(std::integral_constant<int, 0>{});
    if constexpr (TM > 1) tile(std::integral_constant<int, 1>{});
    if constexpr (TM > 2) tile(std::integral_constant<int, 2>{});
    if constexpr (TM > 3) tile(std::integral_constant<int, 3>{});
    if constexpr (TM > 4) tile(std::integral_constant<int, 4>{});
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (WS > 1 && R >= WS) load_w(u, i + WS);
  };
  if (mine > 0) {
    uint32_t i = 0, turn = 0;                      // turn: the slot of activations of step i
    const auto go = [&](auto U, auto R_) {
      step(U, R_, i, slots + turn * (TM * 2048));
      i++;
      turn = turn + 1 == AS ? 0 : turn + 1;
    };
    // N steps, the last ones
    const auto rest = [&](auto N_, auto self, auto K_) {
      constexpr int n = decltype(N_)::value, k = decltype(K_)::value;
      if constexpr (k < n) {
        go(std::integral_constant<int, k % WS>{}, std::integral_constant<int, (n - 1 - k < WS ? n - 1 - k : WS)>{});
        self(N_, self, std::integral_constant<int, k + 1>{});
      }
    };
    const auto last = [&](auto N_) { rest(N_, rest, std::integral_constant<int, 0>{}); };
#pragma unroll
    for (int q = 0; q < AS; q++)
      if (q < mine) {
        load_w(q, q);
#pragma unroll
        for (int t = 0; t < TM; t++) load_a(slots + q * (TM * 2048), t, q);
        __builtin_amdgcn_sched_barrier(0);
      }
    if (WS > 1 && AS < mine) load_w(AS, AS);
    while ((int)i + 2 * WS <= mine) {
      go(std::integral_constant<int, 0>{}, std::integral_constant<int, WS>{});
      if constexpr (WS > 1) go(std::integral_constant<int, 1>{}, std::integral_constant<int, WS>{});
      if constexpr (WS > 2) go(std::integral_constant<int, 2>{}, std::integral_constant<int, WS>{});
      if constexpr (WS > 3) go(std::integral_constant<int, 3>{}, std::integral_constant<int, WS>{});
      if constexpr (WS > 4) go(std::integral_constant<int, 4>{}, std::integral_constant<int, WS>{});
    }
    static_assert(WS <= 5, "steps left below");
    switch (mine - (int)i) {                       // 1 .. 2 WS - 1
      case 1: last(std::integral_constant<int, 1>{}); break;
      case 2: if constexpr (WS > 1) last(std::integral_constant<int, 2>{}); break;
      case 3: if constexpr (WS > 1) last(std::integral_constant<int, 3>{}); break;
      case 4: if constexpr (WS > 2) last(std::integral_constant<int, 4>{}); break;
      case 5: if constexpr (WS > 2) last(std::integral_constant<int, 5>{}); break;
      case 6: if constexpr (WS > 3) last(std::integral_constant<int, 6>{}); break;
      case 7: if constexpr (WS > 3) last(std::integral_constant<int, 7>{}); break;
      case 8: if constexpr (WS > 4) last(std::integral_constant<int, 8>{}); break;
      case 9: if constexpr (WS > 4) last(std::integral_constant<int, 9>{}); break;
    }
  }

  // acc[t][j] of lane l: row 16 t + l % 16, columns 16 j + 4 (l / 16) ..; every wavefront's into LDS, the eight added up
  auto at = [&](int of, int row, int c4) { return red + ((size_t)of * BM + row) * LD + (TN == 4 ? c4 ^ (row & 7) : c4) * 4; };
  __syncthreads();                                 // (the sums take the place of activations that other wavefronts read)
#pragma unroll
  for (int t = 0; t < TM; t++)
#pragma unroll
    for (int j = 0; j < TN; j++) *reinterpret_cast<f32x4*>(at(wave, 16 * t + r16, 4 * j + quarter)) = acc[t][j];
  __syncthreads();
  const bool wide = (ldc & 3) == 0;
  auto total = [&](int row, int c4) {
    f32x4 x[kWaves];
#pragma unroll
    for (int v = 0; v < kWaves; v++) x[v] = *reinterpret_cast<const f32x4*>(at(v, row, c4));
    return ((x[0] + x[4]) + (x[1] + x[5])) + ((x[2] + x[6]) + (x[3] + x[7]));
  };
  auto store = [&](float* dst, const f32x4& o, int left) {
    if (wide && left >= 4) {
      *reinterpret_cast<f32x4*>(dst) = o;
    } else {
#pragma unroll
      for (int e = 0; e < 4; e++)
        if (e < left) dst[e] = o[e];
    }
  };
  if (GU && gridDim.y == 1) {
    for (int i = tid; i < BM * (BN / 8); i += 64 * kWaves) {
      const int row = i / (BN / 8), c4 = i % (BN / 8), gm = m0 + row, f = (n0 >> 1) + 4 * c4;
      if (gm >= M || f >= N) continue;
      const f32x4 g = total(row, c4), up = total(row, c4 + BN / 8);
      f32x4 o;
#pragma unroll
      for (int e = 0; e < 4; e++) o[e] = (g[e] * (1.0f / (1.0f + expf(-g[e])))) * up[e];   // swiglu_kernel's arithmetic
      store(C + (size_t)gm * ldc + f, o, N - f);
    }
  } else {
    for (int i = tid; i < BM * (BN / 4); i += 64 * kWaves) {
      const int row = i / (BN / 4), c4 = i % (BN / 4), gm = m0 + row, gn = n0 + 4 * c4;
      if (gm >= M || (!GU && gn >= N)) continue;   // gated parts are whole tiles wide
      store(C + (size_t)gm * ldc + gn, total(row, c4), GU ? 4 : N - gn);
    }
  }
}

template <int TM, int TN, bool GU, bool RANGED>
__global__ __launch_bounds__(64 * kWaves, 2) void gemm_rows_q4_kernel(const float* __restrict__ A, const void* __restrict__ W,
                                                                     const float* __restrict__ scales, float* __restrict__ C, int M,
                                                                     int N, int K, int part_units, int ldc, int ff, int row_blocks) {
  constexpr int BM = 16 * TM, BN = 16 * TN, LD = BN + 4;
  constexpr int ST = stages(TM), kSlot = TM * 2048;
  extern __shared__ __attribute__((aligned(1024))) float red[];   // activations in flight, then [4][BM][LD] sums
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r16 = lane & 15, quarter = lane >> 4;
  const int nb = gridDim.x, xcd = blockIdx.x & 7, within = blockIdx.x >> 3, q8 = nb >> 3, r8 = nb & 7;
  const int lid = xcd * q8 + min(xcd, r8) + within;
  const int m0 = lid % row_blocks * BM, n0 = lid / row_blocks * BN;
  C += (size_t)blockIdx.y * M * ldc;
  const int units = K / 128, ubeg = blockIdx.y * part_units, uend = min(units, ubeg + part_units);
  const int first = ubeg + wave, mine = first < uend ? (uend - first + kWaves - 1) / kWaves : 0;

  uint32_t aoff[TM][2], woff[TN], soff[TN];        // as above
#pragma unroll
  for (int t = 0; t < TM; t++)
#pragma unroll
    for (int h = 0; h < 2; h++)
      aoff[t][h] = (uint32_t)min(m0 + 16 * t + 8 * h + (lane >> 3), M - 1) * (uint32_t)(K * 4) + ((lane & 7) ^ (lane >> 3)) * 16;
  const int frag[2] = {r16 * 128 + ((2 * quarter) ^ (r16 & 7)) * 16, r16 * 128 + ((2 * quarter + 1) ^ (r16 & 7)) * 16};
  char* ring = reinterpret_cast<char*>(red) + wave * (ST * kSlot);
#pragma unroll
  for (int j = 0; j < TN; j++) {
    const int col = 16 * j + r16;
    int r;
    if (GU) {
      const int f = min((n0 >> 1) + col % (BN / 2), N - 1);
      r = f + (col >= BN / 2 ? ff : 0);
    } else {
      r = min(n0 + col, N - 1);
    }
    woff[j] = (uint32_t)r * (uint32_t)(K / 2) + quarter * 16;
    soff[j] = (uint32_t)r * (uint32_t)(K / 8);
  }
  const char* Ab = reinterpret_cast<const char*>(A);
  const char* Wb = static_cast<const char*>(W);
  const char* Sb = reinterpret_cast<const char*>(scales);

  f32x4 acc[TM][TN];
  float row_scale[TM];                             // RANGED: of this lane's row in each row tile

  // the wavefront's share of the product into acc; scaled: A's rows times row_scale
  auto multiply = [&](auto scaled) {
#pragma unroll
    for (int t = 0; t < TM; t++)
#pragma unroll
      for (int j = 0; j < TN; j++) acc[t][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (mine == 0) return;
    auto load_a = [&](int u, uint32_t step) {      // u: slot, step: of 32 k
#pragma unroll
      for (int t = 0; t < TM; t++)
#pragma unroll
        for (int h = 0; h < 2; h++)
          __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(Ab + (aoff[t][h] + step * 128u)),
                                           (__attribute__((address_space(3))) void*)(ring + u * kSlot + t * 2048 + h * 1024), 16, 0, 0);
    };
    // all but my youngest `n` loads have landed (copies into LDS are waited for by count: the compiler does not see them)
    auto landed = [](auto n) { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(decltype(n)::value) : "memory"); };
    auto cut = [&](int u, int t, frag16 p[3]) {
      const char* at = ring + u * kSlot + t * 2048;
      f32x4 x0 = *reinterpret_cast<const f32x4*>(at + frag[0]), x1 = *reinterpret_cast<const f32x4*>(at + frag[1]);
      if constexpr (decltype(scaled)::value) {
        x0 *= row_scale[t];
        x1 *= row_scale[t];
      }
      split3(x0, x1, p);
    };
    // a unit is four steps; W and the scales of the next unit and the activations of the next steps are on
    // their way while one is multiplied
    frag16 w[2][TN];
    f32x4 s[2][TN];
    auto load_w = [&](int u, int i) {
      const uint32_t unit = (uint32_t)(first + kWaves * i);
#pragma unroll
      for (int j = 0; j < TN; j++) {
        w[u][j] = *reinterpret_cast<const frag16*>(Wb + (woff[j] + unit * 64u));
        s[u][j] = *reinterpret_cast<const f32x4*>(Sb + (soff[j] + unit * 16u));
      }
    };
    auto step_of = [&](int i) { return (uint32_t)(4 * (first + kWaves * (i >> 2)) + (i & 3)); };   // my i-th step: 4 per unit
    // words of four groups -> one word of each of the four quarters' groups: afterwards w[u][j][g] is the eight
    // weights of group g that this lane's quarter multiplies
    auto trade = [&](int u) {
#pragma unroll
      for (int j = 0; j < TN; j++) {
        uint32_t x[4] = {w[u][j][0], w[u][j][1], w[u][j][2], w[u][j][3]};
        auto y = __builtin_amdgcn_permlane32_swap(x[0], x[2], false, false);
        x[0] = y[0]; x[2] = y[1];
        y = __builtin_amdgcn_permlane32_swap(x[1], x[3], false, false);
        x[1] = y[0]; x[3] = y[1];
        y = __builtin_amdgcn_permlane16_swap(x[0], x[1], false, false);
        x[0] = y[0]; x[1] = y[1];
        y = __builtin_amdgcn_permlane16_swap(x[2], x[3], false, false);
        x[2] = y[0]; x[3] = y[1];
        w[u][j] = frag16{x[0], x[1], x[2], x[3]};
      }
    };
    auto compute = [&](int u, int g) {           // group g of the unit in slot u
      frag16 b[TN];
#pragma unroll
      for (int j = 0; j < TN; j++) b[j] = nib8(w[u][j][g]);
#pragma unroll
      for (int t = 0; t < TM; t++) {
        frag16 p[3];
        cut(g % ST, t, p);
        f32x4 grp[TN];
#pragma unroll
        for (int e = 0; e < 3; e++)
#pragma unroll
          for (int j = 0; j < TN; j++) grp[j] = mma(p[e], b[j], e == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : grp[j]);
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
          for (int v = 0; v < 4; v++) acc[t][j][v] = fmaf(grp[j][v], s[u][j][g], acc[t][j][v]);
        if (TM >= 3) __builtin_amdgcn_sched_barrier(0);   // (the registers do not hold two row tiles' terms)
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    // unit `it` in slot u; `more`: the next unit exists (its activations follow in), `far`: the one after it too
    auto unit = [&](int u, int it, auto steady) {
      const bool more = decltype(steady)::value || it + 1 < mine, far = decltype(steady)::value || it + 2 < mine;
      trade(u);
#pragma unroll
      for (int g = 0; g < 4; g++) {
        // younger than this step's activations: those of ST - 1 steps, and the unit of weights issued between
        if (!decltype(steady)::value) landed(std::integral_constant<int, 0>{});
        else if (g == 0) landed(std::integral_constant<int, (ST - 1) * 2 * TM + 2 * TN>{});
        else if (g == 1) landed(std::integral_constant<int, (ST - 1) * 2 * TM + 2 * TN>{});
        else if (ST == 4) landed(std::integral_constant<int, (ST - 1) * 2 * TM + 2 * TN>{});
        else landed(std::integral_constant<int, (ST - 1) * 2 * TM>{});
        compute(u, g);
        if (g + ST < 4 || more) load_a(g % ST, step_of(4 * it + g + ST));
        __builtin_amdgcn_sched_barrier(0);
      }
      if (far) load_w(u, it + 2);
      __builtin_amdgcn_sched_barrier(0);
    };
    load_w(0, 0);
    if (mine > 1) load_w(1, 1);
#pragma unroll
    for (int u = 0; u < ST; u++) load_a(u, step_of(u));
    __builtin_amdgcn_sched_barrier(0);
    int it = 0;
    if (mine > 3) {                              // (the first unit's weights were not issued between its activations: no count)
      unit(0, 0, std::false_type{});
      it = 1;
      for (; it + 3 < mine; it += 2) {
        unit(1, it, std::true_type{});
        unit(0, it + 1, std::true_type{});
      }
      unit(1, it, std::false_type{});
      it++;
    }
    for (; it < mine; it++) {
      if ((it & 1) == 0) unit(0, it, std::false_type{});
      else unit(1, it, std::false_type{});
    }
  };

  // acc[t][j][v] of lane l: row 16 t + 4 (l / 16) + v, column 16 j + l % 16. Wavefronts 4..7 hand theirs to 0..3,
  // whose four sums everyone then adds up.
  auto put = [&](float* dst) {
#pragma unroll
    for (int t = 0; t < TM; t++)
#pragma unroll
      for (int j = 0; j < TN; j++)
#pragma unroll
        for (int v = 0; v < 4; v++) dst[(16 * t + 4 * quarter + v) * LD + 16 * j + r16] = acc[t][j][v];
  };
  float* slot = red + (size_t)(wave & 3) * BM * LD;
  const bool wide = (ldc & 3) == 0;
  auto total = [&](int row, int col) {
    f32x4 x[4];
#pragma unroll
    for (int w4 = 0; w4 < 4; w4++) x[w4] = *reinterpret_cast<const f32x4*>(red + ((size_t)w4 * BM + row) * LD + col);
    return (x[0] + x[1]) + (x[2] + x[3]);
  };
  auto store = [&](float* dst, const f32x4& o, int left) {
    if (wide && left >= 4) {
      *reinterpret_cast<f32x4*>(dst) = o;
    } else {
#pragma unroll
      for (int e = 0; e < 4; e++)
        if (e < left) dst[e] = o[e];
    }
  };
  auto odd = [](const f32x4& o) {                  // RANGED: not finite, or nothing but tiny values
    const float m = fmaxf(fmaxf(fabsf(o[0]), fabsf(o[1])), fmaxf(fabsf(o[2]), fabsf(o[3])));
    const float z = (o[0] + o[1]) * 0.f + (o[2] + o[3]) * 0.f;
    return m < 0x1p-40f || z != 0.f;
  };
  int* found = reinterpret_cast<int*>(red + 4 * BM * LD);   // RANGED: two words behind the sums
  static_assert(!RANGED || (4 * BM * LD + 2) * 4 <= lds_bytes_q4(TM, TN), "room for the words");
  auto any_of_block = [&](bool mine_too, int word) {
    if (mine_too) found[word] = 1;
    __syncthreads();
    return found[word] != 0;
  };
  // the wavefronts' sums joined and stored; true where a sum of this thread's is odd
  auto finish = [&] {
    bool o_dd = false;
    __syncthreads();                               // (the sums take the place of activations that other wavefronts read)
    if (RANGED && tid < 2) found[tid] = 0;
    if (wave >= 4) put(slot);
    __syncthreads();
    if (wave < 4) {
#pragma unroll
      for (int t = 0; t < TM; t++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
          for (int v = 0; v < 4; v++) acc[t][j][v] += slot[(16 * t + 4 * quarter + v) * LD + 16 * j + r16];
      put(slot);                                   // (the lane's own entries: nobody else reads them before the barrier)
    }
    __syncthreads();
    if (GU && gridDim.y == 1) {
      for (int i = tid; i < BM * (BN / 8); i += 64 * kWaves) {
        const int row = i / (BN / 8), c = i % (BN / 8) * 4, gm = m0 + row, f = (n0 >> 1) + c;
        if (gm >= M || f >= N) continue;
        const f32x4 g = total(row, c), u = total(row, c + BN / 2);
        if (RANGED) o_dd |= odd(g) || odd(u);
        f32x4 o;
#pragma unroll
        for (int e = 0; e < 4; e++) o[e] = (g[e] * (1.0f / (1.0f + expf(-g[e])))) * u[e];   // swiglu_kernel's arithmetic
        store(C + (size_t)gm * ldc + f, o, N - f);
      }
    } else {
      for (int i = tid; i < BM * (BN / 4); i += 64 * kWaves) {
        const int row = i / (BN / 4), c = i % (BN / 4) * 4, gm = m0 + row, gn = n0 + c;
        if (gm >= M || (!GU && gn >= N)) continue;   // gated parts are whole tiles wide
        const f32x4 o = total(row, c);
        if (RANGED) o_dd |= odd(o);
        store(C + (size_t)gm * ldc + gn, o, GU ? 4 : N - gn);
      }
    }
    return o_dd;
  };
  multiply(std::false_type{});
  if constexpr (!RANGED) {
    finish();
  } else if (any_of_block(finish(), 0)) {
    int ex[TM];
    bool far = false;
#pragma unroll
    for (int t = 0; t < TM; t++) {                 // the largest magnitude of what this wavefront cuts of a row
      const char* row = Ab + (size_t)min(m0 + 16 * t + r16, M - 1) * K * 4 + quarter * 32;
      uint32_t m = 0;
#pragma unroll 1
      for (int i = 0; i < 4 * mine; i++) {
        const uint4* x = reinterpret_cast<const uint4*>(row + (size_t)(4 * (first + kWaves * (i >> 2)) + (i & 3)) * 128);
        const uint4 x0 = x[0], x1 = x[1];
        m = max(m, max(max(x0.x & 0x7fffffffu, x0.y & 0x7fffffffu), max(x0.z & 0x7fffffffu, x0.w & 0x7fffffffu)));
        m = max(m, max(max(x1.x & 0x7fffffffu, x1.y & 0x7fffffffu), max(x1.z & 0x7fffffffu, x1.w & 0x7fffffffu)));
      }
      m = max(m, (uint32_t)__shfl_xor((int)m, 16));
      m = max(m, (uint32_t)__shfl_xor((int)m, 32));
      far |= m != 0u && (m < __float_as_uint(0x1p-100f) || m > __float_as_uint(0x1p100f));
      ex[t] = row_exponent((int)(m >> 23), m == 0u);
      row_scale[t] = pow2f(ex[t]);
    }
    if (!any_of_block(far, 1)) return;             // zeros, or weights that are
    __syncthreads();                               // (the words lie where copies are about to land)
    multiply(std::true_type{});
#pragma unroll
    for (int t = 0; t < TM; t++)
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const int e = __shfl(ex[t], 4 * quarter + v);   // the exponent of row 16 t + 4 quarter + v comes back out
#pragma unroll
        for (int j = 0; j < TN; j++) acc[t][j][v] = ldexpf(acc[t][j][v], -e);
      }
    finish();
  }
}

template <int TM, int TN, bool GU>
int run_bf16(const RowsPlan& P, const float* A, const void* W, float* C, int M, int N, int K, int ldc, int ff) {
  constexpr int lds = lds_bytes_bf16(TM, TN);
  static const hipError_t set = hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_rows_bf16_kernel<TM, TN, GU>),
                                                    hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (set != hipSuccess) return hip_fail(set, "hipFuncSetAttribute");
  // Parts and tiles in one run per XCD (block_place) where blocks of a part share weights, or where the tiles are no multiple of
  // 8, so that those an XCD gets change from part to part: 77 x 896 x 4864 in ten parts 7.9 -> 7.2 us, 200 rows 12.3 -> 10.5, 500 24.5 -> 22.3;
  // elsewhere the part from the grid, which takes no division (77 x 1152 x 896 in four parts 4.5 us, 4.65 so).
  const bool pairs = P.row_blocks > 1 || P.tiles % 8 != 0;
  gemm_rows_bf16_kernel<TM, TN, GU><<<dim3((unsigned)(P.tiles * P.row_blocks), (unsigned)P.S), dim3(64 * kWaves), lds, ctx().stream>>>(
      A, W, C, M, N, K, P.part_units, ldc, ff, P.row_blocks | (pairs ? P.S : 1) << 16);
  return TLHIP_OK;
}
template <int TM, int TN, bool GU, bool RANGED = false>
int run_q4(const RowsPlan& P, const float* A, const void* W, const float* scales, float* C, int M, int N, int K, int ldc, int ff) {
  constexpr int lds = lds_bytes_q4(TM, TN);
  static const hipError_t set = hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_rows_q4_kernel<TM, TN, GU, RANGED>),
                                                    hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (set != hipSuccess) return hip_fail(set, "hipFuncSetAttribute");
  gemm_rows_q4_kernel<TM, TN, GU, RANGED><<<dim3((unsigned)(P.tiles * P.row_blocks), (unsigned)P.S), dim3(64 * kWaves), lds, ctx().stream>>>(
      A, W, scales, C, M, N, K, P.part_units, ldc, ff, P.row_blocks);
  return TLHIP_OK;
}

template <int TM>
int run_tm(const RowsPlan& P, const float* A, const void* W, const float* scales, float* C, int M, int N, int K, int ldc, int ff, bool gu) {
  const bool q4 = scales != nullptr;
  if constexpr (TM >= 3) {                         // more than 64 rows are blocks of three to five row tiles
    if (q4 && M > 64) {
      switch (P.TN + (gu ? 16 : 0)) {
        case 1: return run_q4<TM, 1, false, true>(P, A, W, scales, C, M, N, K, ldc, ff);
        case 2: return run_q4<TM, 2, false, true>(P, A, W, scales, C, M, N, K, ldc, ff);
        case 18: return run_q4<TM, 2, true, true>(P, A, W, scales, C, M, N, K, ldc, ff);
      }
      return fail(TLHIP_EUNSUPPORTED, "gemm_rows: no kernel for this plan");
    }
  }
  switch (P.TN + (gu ? 16 : 0) + (q4 ? 32 : 0)) {   // (int4 over four column tiles: the registers hold one row tile)
    case 1: return run_bf16<TM, 1, false>(P, A, W, C, M, N, K, ldc, ff);
    case 2: return run_bf16<TM, 2, false>(P, A, W, C, M, N, K, ldc, ff);
    case 3: return run_bf16<TM, 3, false>(P, A, W, C, M, N, K, ldc, ff);
    case 4: return run_bf16<TM, 4, false>(P, A, W, C, M, N, K, ldc, ff);
    case 18: return run_bf16<TM, 2, true>(P, A, W, C, M, N, K, ldc, ff);
    case 19: return run_bf16<TM, 3, true>(P, A, W, C, M, N, K, ldc, ff);
    case 20: return run_bf16<TM, 4, true>(P, A, W, C, M, N, K, ldc, ff);
    case 33:
      if constexpr (TM <= 4) return run_q4<TM, 1, false>(P, A, W, scales, C, M, N, K, ldc, ff);
      break;
    case 34:
      if constexpr (TM <= 4) return run_q4<TM, 2, false>(P, A, W, scales, C, M, N, K, ldc, ff);
      break;
    case 36:
      if constexpr (TM == 1) return run_q4<TM, 4, false>(P, A, W, scales, C, M, N, K, ldc, ff);
      break;
    case 50:
      if constexpr (TM <= 4) return run_q4<TM, 2, true>(P, A, W, scales, C, M, N, K, ldc, ff);
      break;
    case 52:
      if constexpr (TM == 1) return run_q4<TM, 4, true>(P, A, W, scales, C, M, N, K, ldc, ff);
      break;
  }
  return fail(TLHIP_EUNSUPPORTED, "gemm_rows: no kernel for this plan");
}

}  // namespace rows

// The longest chain of matrix instructions, in steps of 32 k, that a wavefront may form a sum of bf16 products by. The error of a sum
// grows with it (0.9e-7 of the result after a step, 1.3e-7 after 4, 1.7e-7 after 7, 2.0e-7 after 10), and the plan that takes
// least time would trade it: few rows' products of K 896 run as fast unsplit on narrow column tiles, in chains of 4 (24 x 1152 x 896
// 1.3e-7 of error for 0.9e-7). So K is split at least as far as fills the CUs by blocks of wide tiles, where that does not cost more
// than it gives. Up to 128 rows that is what an estimate fitted to 280 runs says (K 384 .. 18944, N 384 .. 37888, M 8 .. 120: clocks
// of a step by the CU's vector memory path or its matrix or vector instructions, 3500 and 60 per accumulator tile for a block, parts
// written and read, a launch that adds them up); wide products, which have a block for every CU, stay whole: 18960 x 2048 at 32 rows takes
// 19.3 us, in two parts 22.9. Above, the 128-row tiles, which run what does not come here, split K up to 16 times and have
// 1.73e-7 at K 3584, 1.9e-7 at 4864, 2.5e-7 at 8192, 3.0e-7 at 12288.
static int64_t longest_chain(int64_t M, int64_t N, int64_t K, bool gu, int64_t max_S) {
  auto cdiv = [](int64_t a, int64_t b) { return (a + b - 1) / b; };
  const int64_t rows_w = (gu ? 2 : 1) * N, cus = cu_count(), units = K / rows::kStep, t16 = cdiv(M, 16), row_blocks = cdiv(t16, rows::kMaxTM);
  if (M > 128) return std::max<int64_t>(7, units * 7 / 128);
  const int TM = (int)cdiv(t16, row_blocks);
  double least = 0;
  int64_t chain = 0;
  for (int TN = 4; TN >= (gu ? 2 : 1); TN /= 2) {
    const int64_t blocks1 = cdiv(rows_w, 16 * TN) * row_blocks;
    for (int64_t S = 1; S <= std::min<int64_t>(max_S, units); S++) {
      const int64_t per = cdiv(units, S), blocks = blocks1 * S, n = cdiv(per, rows::kWaves);
      if (cdiv(units, per) != S) continue;
      if (S > 1 && M > 16 && blocks1 > cus) break;
      const double clocks = (double)n * std::max(96.0 * TM * TN, std::max(352.0 * TM, 8 * (70.0 * TM + 60.0 * TN))) + 3500 + 60 * TM * TN;
      const double rounds = blocks <= cus ? 1 : 1.2 * (blocks <= 4 * cus ? (double)cdiv(blocks, cus) : (double)blocks / cus);
      const double us = rounds * clocks / 2100 + (S > 1 ? 1e-6 * (double)(S * M * rows_w) + (gu || N > 8192 ? 5 : 0) : 0);
      if (chain == 0 || us < least) {
        least = us;
        chain = n;
      }
    }
  }
  return chain;
}

// Row tiles per block, columns per tile and K splits that an estimate of the time likes best; S == 0 where the shape is not
// taken. `us` is the chosen plan's time, the launch that adds parts up not included: the caller weighs it against the time of the
// kernel it would take instead.
//
// bf16: a launch costs a start and its weights' way from HBM; a block starts and ends in a time that grows with its sums, and each
// costs a little for its dispatch; a step of its wavefronts takes the CU's loads of activations and weights, a little less where
// CUs are idle; blocks that share a CU cost half again each, more where their steps are many. Fitted up to 128 rows to 25000
// runs in the chains allowed (2 to 128 rows, 256 to 16000 columns, K 256 to 18944: error 8 %, the shape it chooses 1.1 % slower than the
// fastest one on average), above to 13980 others (12800 runs of 129 to 1024 rows take 1.1 times as much, error 9 %, the shape 1.1 %).
// Since weights are copied into LDS a CU takes other numbers of blocks than those runs had. With them the shape is 1.2 % slower than the
// fastest of up to twelve over 3000 products to 128 rows and 1.7 % over 400 above (1.4 and 2.1 % by the earlier numbers; all constants fitted
// anew 1.5 and 1.4 %, or with the sharing alone 0.95 to 128 rows, but longer chains), constants as they were but for the price of sums
// above 128 rows (0.144 before; 129 x 3085 gated x 1056 takes 12.8 us by 194 blocks and 12.7 by 387). Of drawn products of 2 to 1024 rows
// 3 % are run another way for them: 150 of those take 0.79 to 1.14 of their time, 0.941 on average, 27 of the models' sizes 0.74 to 1.05,
// 0.912 (89 x 4608 x 3584 22.8 -> 16.7 us, 89 x 10304 x 2048 24.2 -> 21.0, 131 x 21064 gated x 352 34.8 -> 28.2; 592 x 13304 gated x 352 70 -> 80).
// Measured, us, tiles -> this kernel: 896 x 896 at 37 / 77 / 512 rows 10.3 / 20.9 / 21.7 -> 3.8 / 4.4 / 7.7; 4864 x 896 gated at 37 / 77 / 256
// 15.0 / 25.2 / 28.3 -> 8.3 / 10.7 / 24.4; 896 x 4864 at 37 / 77 / 150 10.9 / 21.4 / 22.5 -> 6.5 / 8.7 / 10.6; 1152 x 896 at 77 / 300 20.9 / 21.4 -> 5.1 / 7.3;
// 18944 x 3584 gated at 37 / 64 104 / 105 -> 73 / 89.
static RowsPlan plan_rows_bf16(int64_t M, int64_t N, int64_t K, bool gu, int64_t max_S) {
  static constexpr rows::BlocksOfACu kFit;
  auto cdiv = [](int64_t a, int64_t b) { return (a + b - 1) / b; };
  RowsPlan best;
  const int64_t rows_w = (gu ? 2 : 1) * N, cus = cu_count(), units = K / rows::kStep, t16 = cdiv(M, 16);
  struct Cost { double start, share, share_n, steps, fill, whole, rows, cols, idle, sums, dispatch, parts, weights, all; };
  static constexpr Cost kFew = {2.33, 0.40, 0.35, 20, 0.77, 0, 0.229, 0.184, 0.827, 0.165, 0.317, 0, 0.051, 1};
  static constexpr Cost kMany = {2.08, 0.424, 0.593, 10, 0.86, 0.086, 0.194, 0.182, 0.877, 0.141, 0, 0.179, 0.103, 1.1};
  const Cost& k = M > 128 ? kMany : kFew;
  // What adds the parts up beside reading them: a launch, or where a narrow product is left as parts their consumer. (Both
  // forms of a narrow product take one plan: two products of this kernel with room for as many parts are the same bits.)
  const double own_sum = gu || N > 8192 ? 5.4 : M > 128 ? 0.4 : 1.3;
  const int64_t chain = longest_chain(M, N, K, gu, max_S);
  const int most_S = (int)std::min<int64_t>(max_S, units), chain_S = (int)cdiv(units, rows::kWaves * chain);
  // (where K cannot be split so far, the tiles cannot split it either, and their chains are eight times as long)
  const int least_S = (int)cdiv(units, cdiv(units, std::min(chain_S, most_S)));
  double least = 0;
  const int64_t few = cdiv(t16, rows::kMaxTM);
  for (int64_t row_blocks = few; row_blocks <= std::min(few + 1, t16); row_blocks++)
    for (int TN = 4; TN >= (gu ? 2 : 1); TN--) {
      const int TM = (int)cdiv(t16, row_blocks);
      const int64_t tiles = cdiv(rows_w, 16 * TN), fit = kFit.n[TM - 1][TN - 1], at_once = fit * cus;
      if (row_blocks > few && t16 <= 4 && tiles * few > cus / 2) continue;   // (weights read twice for CUs that are busy anyway)
      const int64_t unsplit = tiles * row_blocks;
      // (K is split no further than keeps every CU busy)
      for (int S = least_S; S <= most_S && (S == least_S || unsplit * (S - 1) < cus); S++) {
        const int64_t blocks = unsplit * S;
        const int per = ((int)units + S - 1) / S;
        if (((int)units + per - 1) / per != S) continue;
        const int steps = (per + rows::kWaves - 1) / rows::kWaves;   // of a wavefront
        // (up to 128 rows no split that leaves them as many: parts are added one after the other, which costs a rounding each - 22 x 68
        // gated x 1600, 50 steps, 1.75e-7 of error in 13 parts and 1.51e-7 in 7)
        if (M <= 128 && S > least_S && ((int)units + rows::kWaves * steps - 1) / (rows::kWaves * steps) != S) continue;
        const double n = (double)steps;
        // (blocks of nine accumulator tiles leave each other less from the start: 41 x 18944 gated x 3584 by two of them on a CU 85 us, 78 by
        // one of twelve)
        const Cost& sh = TM * TN > 8 ? kMany : k;
        const auto share = [&](int64_t on_a_cu) { return 1 + (sh.share + sh.share_n * n / (n + sh.steps)) * (double)(on_a_cu - 1); };
        double rounds = 1;
        if (blocks > cus) {
          const int64_t rest = blocks % at_once;
          const double fill = blocks > at_once ? k.fill + (1 - k.fill) * (double)rest / (double)at_once : 1;   // of the last round
          rounds = (double)(blocks / at_once) * share(fit) + (rest > 0 ? share(cdiv(rest, cus)) * fill : 0);
        }
        const double work = (k.whole * n + (1 - k.whole) * (double)per / rows::kWaves) * (k.rows * TM + k.cols * TN) *
                            (k.idle + (1 - k.idle) * std::min(1.0, (double)blocks / (double)cus));
        const double parts = S > 1 ? (double)S * M * (gu ? tiles * 16 * TN : N) * 4e-6 : 0;   // MB
        const double us = k.start + rounds * (k.sums * TM * TN + work) + k.dispatch * (double)blocks / (double)cus + k.parts * parts +
                          k.weights * 2e-6 * (double)rows_w * (double)K;
        const double all = us + 0.25 * parts + (S > 1 ? own_sum : 0);
        if (best.S == 0 || all < least) {
          least = all;
          best.TM = TM;
          best.TN = TN;
          best.S = (int)S;
          best.tiles = (int)tiles;
          best.row_blocks = (int)row_blocks;
          best.part_units = (int)per;
          best.us = k.all * us;
        }
      }
    }
  return best;
}

// int4: the estimate that chooses, fitted to 280 runs (K 384 .. 18944, N 384 .. 37888, M 8 .. 120): a step of a block's eight
// wavefronts takes the CU's vector memory path 35 clocks per KB of activations and 60 per KB of weights (whose lanes cover
// 16 rows each), or its SIMDs, with two wavefronts each, the clocks of their matrix or vector instructions (5.5 per element
// cut, 23 per eight nibbles; measured 1.8 times that); a block starts and ends in 3500 clocks and 60 per accumulator
// tile; a launch costs 2 us. `us` is the chosen plan's time fitted again, to 1000 runs (error 10 to 13 %) and 5 to 12 % up.
static RowsPlan plan_row_blocks_q4(int64_t M, int64_t N, int64_t K, bool gu, int64_t max_S, int64_t row_blocks) {
  RowsPlan best;
  auto cdiv = [](int64_t a, int64_t b) { return (a + b - 1) / b; };
  const int64_t rows_w = (gu ? 2 : 1) * N, cus = ctx().cus, units = K / 128;
  constexpr int steps = 4;
  best.row_blocks = (int)row_blocks;
  const int TM = best.TM = (int)cdiv(cdiv(M, 16), row_blocks);
  double least = 0;
  const double own_sum = gu ? 5 : 0;
  for (int TN = TM > 1 ? 2 : 4; TN >= (gu ? 2 : 1); TN /= 2) {   // (what the registers hold)
    const int64_t tiles = cdiv(rows_w, 16 * TN);
    for (int64_t S = 1; S <= std::min<int64_t>(max_S, units); S++) {
      const int64_t per = cdiv(units, S), blocks = tiles * row_blocks * S;
      if (cdiv(units, per) != S) continue;
      const double n = (double)(cdiv(per, rows::kWaves) * steps);    // steps of a wavefront
      const double mem = 8 * (70.0 * TM + 30.0 * TN);
      const double math = 2 * 1.8 * std::max(48.0 * TM * TN, 176.0 * TM + TN * (92.0 + 16 * TM));
      const double rounds = blocks <= 2 * cus ? (double)cdiv(blocks, cus) : (double)blocks / cus;
      const double parts = S > 1 ? (double)S * M * rows_w * 4 / 1e6 : 0;
      // parts written and read, and their launch, which a gated product has
      const double us = 2 + rounds * (n * std::max(math, mem) + 3500 + 60 * TM * TN) / 2100 + (S > 1 ? parts / 4 + own_sum : 0);
      if (best.S == 0 || us < least) {
        least = us;
        best.TN = TN;
        best.S = (int)S;
        best.tiles = (int)tiles;
        best.part_units = (int)per;
        // fewer steps than wavefronts leave some idle; five row tiles spill, and blocks in turn wait for what
        // they would have loaded ahead; over many blocks, wavefronts with a unit more than others even out (38 x 18088 gated x
        // 2560, 20 units over eight wavefronts: 64 us here, 89 in the 64-row tiles)
        const double own = blocks > 2 * cus && per > rows::kWaves ? 1.05 * (double)per / rows::kWaves * steps : n;
        const double work = rounds * own * std::max(mem * (double)std::min<int64_t>(rows::kWaves, per) / rows::kWaves, per > 4 ? math : math / 2) / 2100;
        best.us = 2 + work * (TM == 5 ? 1.3 : 1.0) * (rounds > 2 ? 1.2 : rounds > 1 ? 0.81 : 0.74) + rounds * (0.3 + 0.18 * TM * TN) + parts;
        // many columns of a short K (14000 runs, N 20000 .. 160000): 24 x 21497 gated x 512 24.8 us for an estimate of 20.3
        if (blocks > 2 * cus && per <= 4) best.us *= 1.2;
      }
    }
  }
  return best;
}

RowsPlan plan_gemm_rows(int64_t M, int64_t N, int64_t K, bool gu, bool q4, int64_t max_S) {
  const int64_t rows_w = (gu ? 2 : 1) * N, t16 = (M + 15) / 16;
  if (M > (q4 ? 128 : kRowsMaxBf16) || K % (q4 ? 128 : 32) != 0 || M * K * 4 >= (int64_t(1) << 32) || rows_w * K * (q4 ? 1 : 4) / 2 >= (int64_t(1) << 32))
    return RowsPlan{};                             // (32-bit byte offsets)
  if (!q4) return plan_rows_bf16(M, N, K, gu, max_S);
  // Up to 16 rows nothing else is as fast, save for so few units that most wavefronts of a block have none and so many
  // columns that blocks come in more rounds than that: up to 65000 columns x 128 twice what the 64-row tiles take, x 256 1.4 times;
  // up to 32768 x 256 0.9 times
  if (M <= 16 && K < 512 && (rows_w + 63) / 64 > K / 128 * (int64_t)ctx().cus) return RowsPlan{};
  const auto plan = [&](int64_t row_blocks) { return plan_row_blocks_q4(M, N, K, gu, max_S, row_blocks); };
  if (t16 != 5) return plan((t16 + rows::kMaxTM - 1) / rows::kMaxTM);
  // 65 to 80 rows: one block of five row tiles, or two of three (77 x 640 x 768 7.8 us and 6.1; 74 x 4609 x 11008, whose
  // K cannot be split, 76 and 107)
  const RowsPlan one = plan(1), two = plan(2);
  const auto all = [](const RowsPlan& P) { return P.us + (P.S > 1 ? kPartSumUs : 0); };
  return two.S > 0 && (one.S == 0 || all(two) < all(one)) ? two : one;
}

int launch_gemm_rows(const RowsPlan& P, const float* A, const void* W, const float* scales, float* C, int64_t M, int64_t N, int64_t K,
                     int64_t ldc, bool gu) {
  switch (P.TM) {
    case 1: return rows::run_tm<1>(P, A, W, scales, C, (int)M, (int)N, (int)K, (int)ldc, (int)N, gu);
    case 2: return rows::run_tm<2>(P, A, W, scales, C, (int)M, (int)N, (int)K, (int)ldc, (int)N, gu);
    case 3: return rows::run_tm<3>(P, A, W, scales, C, (int)M, (int)N, (int)K, (int)ldc, (int)N, gu);
    case 4: return rows::run_tm<4>(P, A, W, scales, C, (int)M, (int)N, (int)K, (int)ldc, (int)N, gu);
    case 5: return rows::run_tm<5>(P, A, W, scales, C, (int)M, (int)N, (int)K, (int)ldc, (int)N, gu);
  }
  return fail(TLHIP_EUNSUPPORTED, "gemm_rows: no kernel for this plan");
}

}  // namespace tlhip
