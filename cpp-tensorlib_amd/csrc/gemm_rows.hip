// Products of a few rows: C[M,N] = A[M,K] f32 . W[N,K]^T for a short prompt, W bf16 rows or int4 groups.
//
// What bounds it: with M of a few dozen the weight is read once and hardly reused, and what is left is the
// chain of latencies of one block. gemm_bf16_nt_kernel (prefill.hip) walks K in slabs of 32 through LDS, two
// barriers and one load round trip per slab: ten slabs were 20 us for weights that take 2 us to read. Here a
// block has no barrier until its sums are complete: its eight wavefronts split the block's K range between
// them (wavefront w takes the 32-k steps w, w + 8, ...), each with the WHOLE tile's accumulators, and loads
// both operands straight into the registers of the MFMA that uses them, several steps ahead. The sums meet in
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

// Steps of activations in flight per wavefront (int4: a divisor of four): 2 KB of LDS per row tile each.
__host__ __device__ constexpr int stages(int TM, bool q4) { return TM <= 2 ? 4 : TM == 3 && !q4 ? 3 : 2; }
__host__ __device__ constexpr int lds_bytes(int TM, int TN, bool q4) {
  const int ring = kWaves * stages(TM, q4) * TM * 2048, sums = 4 * 16 * TM * (16 * TN + 4) * 4;
  return ring > sums ? ring : sums;
}

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
template <int TM, int TN, bool GU, bool Q4, bool RANGED>
__global__ __launch_bounds__(64 * kWaves, 2) void gemm_rows_kernel(const float* __restrict__ A, const void* __restrict__ W,
                                                                  const float* __restrict__ scales, float* __restrict__ C,
                                                                  int M, int N, int K, int part_units, int ldc, int ff,
                                                                  int row_blocks) {
  constexpr int BM = 16 * TM, BN = 16 * TN, LD = BN + 4;
  constexpr int ST = stages(TM, Q4), kSlot = TM * 2048;
  extern __shared__ __attribute__((aligned(1024))) float red[];   // activations in flight, then [4][BM][LD] sums
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r16 = lane & 15, quarter = lane >> 4;
  // one contiguous run of tiles per XCD, row blocks fastest: those share a weight tile in one L2
  const int nb = gridDim.x, xcd = blockIdx.x & 7, within = blockIdx.x >> 3, q8 = nb >> 3, r8 = nb & 7;
  const int lid = xcd * q8 + min(xcd, r8) + within;
  const int m0 = lid % row_blocks * BM, n0 = lid / row_blocks * BN;
  C += (size_t)blockIdx.y * M * ldc;
  const int units = Q4 ? K / 128 : K / kStep, ubeg = blockIdx.y * part_units, uend = min(units, ubeg + part_units);
  const int first = ubeg + wave, mine = first < uend ? (uend - first + kWaves - 1) / kWaves : 0;

  // byte offsets of this lane's rows (clamped into the operands: what lies past an edge is not stored). A 1 KB copy
  // of activations is eight rows of 128 bytes, the 16-byte chunks of row r in the order c ^ (r & 7), which spreads
  // the fragment reads (16 rows, one chunk) over the LDS banks.
  uint32_t aoff[TM][2], woff[TN], soff[Q4 ? TN : 1];
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
    woff[j] = (uint32_t)r * (uint32_t)(Q4 ? K / 2 : K * 2) + quarter * 16;
    if (Q4) soff[j] = (uint32_t)r * (uint32_t)(K / 8);
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
    if constexpr (!Q4) {
      frag16 w[ST][TN];
      auto load = [&](int u, int i) {              // slot u takes my i-th step
        const uint32_t step = (uint32_t)(first + kWaves * i);
        load_a(u, step);
#pragma unroll
        for (int j = 0; j < TN; j++) w[u][j] = *reinterpret_cast<const frag16*>(Wb + (woff[j] + step * 64u));
        __builtin_amdgcn_sched_barrier(0);         // (else the compiler gathers the loads of all slots behind the last one's products)
      };
      auto compute = [&](int u) {
#pragma unroll
        for (int t = 0; t < TM; t++) {
          frag16 p[3];
          cut(u, t, p);
#pragma unroll
          for (int e = 0; e < 3; e++)
#pragma unroll
            for (int j = 0; j < TN; j++) acc[t][j] = mma(p[e], w[u][j], acc[t][j]);
        }
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
          landed(std::integral_constant<int, (ST - 1) * (2 * TM + TN)>{});
          compute(u);
          load(u, it + u + ST);
        }
      }
      landed(std::integral_constant<int, 0>{});
#pragma unroll
      for (int u = 0; u < ST; u++) {
        if (it + u < mine) compute(u);
        if (it + u + ST < mine) load(u, it + u + ST);
      }
      landed(std::integral_constant<int, 0>{});
#pragma unroll
      for (int u = 0; u < ST; u++)
        if (it + u + ST < mine) compute(u);
    } else {
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
  static_assert(!RANGED || (4 * BM * LD + 2) * 4 <= lds_bytes(TM, TN, Q4), "room for the words");
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

template <int TM, int TN, bool GU, bool Q4, bool RANGED = false>
int run(const RowsPlan& P, const float* A, const void* W, const float* scales, float* C, int M, int N, int K, int ldc, int ff) {
  constexpr int lds = lds_bytes(TM, TN, Q4);
  static const hipError_t set = hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_rows_kernel<TM, TN, GU, Q4, RANGED>),
                                                    hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (set != hipSuccess) return hip_fail(set, "hipFuncSetAttribute");
  gemm_rows_kernel<TM, TN, GU, Q4, RANGED><<<dim3((unsigned)(P.tiles * P.row_blocks), (unsigned)P.S), dim3(64 * kWaves), lds, ctx().stream>>>(
      A, W, scales, C, M, N, K, P.part_units, ldc, ff, P.row_blocks);
  return TLHIP_OK;
}

template <int TM>
int run_tm(const RowsPlan& P, const float* A, const void* W, const float* scales, float* C, int M, int N, int K, int ldc, int ff, bool gu) {
  const bool q4 = scales != nullptr;
  if constexpr (TM >= 3) {                         // more than 64 rows are blocks of three to five row tiles
    if (q4 && M > 64) {
      switch (P.TN + (gu ? 16 : 0)) {
        case 1: return run<TM, 1, false, true, true>(P, A, W, scales, C, M, N, K, ldc, ff);
        case 2: return run<TM, 2, false, true, true>(P, A, W, scales, C, M, N, K, ldc, ff);
        case 18: return run<TM, 2, true, true, true>(P, A, W, scales, C, M, N, K, ldc, ff);
      }
      return fail(TLHIP_EUNSUPPORTED, "gemm_rows: no kernel for this plan");
    }
  }
  switch (P.TN + (gu ? 16 : 0) + (q4 ? 32 : 0)) {   // (int4 over four column tiles: the registers hold one row tile)
    case 1: return run<TM, 1, false, false>(P, A, W, scales, C, M, N, K, ldc, ff);
    case 2: return run<TM, 2, false, false>(P, A, W, scales, C, M, N, K, ldc, ff);
    case 4: return run<TM, 4, false, false>(P, A, W, scales, C, M, N, K, ldc, ff);
    case 18: return run<TM, 2, true, false>(P, A, W, scales, C, M, N, K, ldc, ff);
    case 20: return run<TM, 4, true, false>(P, A, W, scales, C, M, N, K, ldc, ff);
    case 33:
      if constexpr (TM <= 4) return run<TM, 1, false, true>(P, A, W, scales, C, M, N, K, ldc, ff);
      break;
    case 34:
      if constexpr (TM <= 4) return run<TM, 2, false, true>(P, A, W, scales, C, M, N, K, ldc, ff);
      break;
    case 36:
      if constexpr (TM == 1) return run<TM, 4, false, true>(P, A, W, scales, C, M, N, K, ldc, ff);
      break;
    case 50:
      if constexpr (TM <= 4) return run<TM, 2, true, true>(P, A, W, scales, C, M, N, K, ldc, ff);
      break;
    case 52:
      if constexpr (TM == 1) return run<TM, 4, true, true>(P, A, W, scales, C, M, N, K, ldc, ff);
      break;
  }
  return fail(TLHIP_EUNSUPPORTED, "gemm_rows: no kernel for this plan");
}

}  // namespace rows

// Row tiles per block, columns per tile and K splits that an estimate of the time likes best; S == 0 where the shape is not
// taken.
//
// The estimate that chooses, fitted to 280 runs (K 384 .. 18944, N 384 .. 37888, M 8 .. 120): a step of a block's eight
// wavefronts takes the CU's vector memory path 35 clocks per KB of activations and 60 per KB of weights (whose lanes cover
// 16 rows each), or its SIMDs, with two wavefronts each, the clocks of their matrix or vector instructions (5.5 per element
// cut, 23 per eight nibbles; int4 measured 1.8 times that); a block starts and ends in 3500 clocks and 60 per accumulator
// tile; bf16 blocks past the first round cost a fifth more; a launch costs 2 us. `us` is the chosen plan's time fitted again,
// to 1000 runs (error 10 to 13 %) and 5 to 12 % up: the caller weighs it against the time of the kernel it would take instead.
// Measured, us, other kernel -> this one: 896 x 896 at 5 / 37 / 77 rows 10.5 / 10.0 / 20.5 -> 3.6 / 3.7 / 4.4; 4864 x 896
// gated 14.4 / 16.0 / 25.4 -> 7.8 / 11.1 / 13.4; 896 x 4864 11.0 / 11.4 / 21.7 -> 4.9 / 7.0 / 9.6; 9728 x 896 at 48 and 64
// rows 16.8 / 17.8 -> 10.8 / 11.9; 18944 x 3584 gated 111 / 111 -> 63 / 92; int4 119 / 127 -> 53 / 93.
static RowsPlan plan_row_blocks(int64_t M, int64_t N, int64_t K, bool gu, bool q4, int64_t max_S, int64_t row_blocks) {
  RowsPlan best;
  auto cdiv = [](int64_t a, int64_t b) { return (a + b - 1) / b; };
  const int64_t rows_w = (gu ? 2 : 1) * N, cus = ctx().cus, units = K / (q4 ? 128 : 32), steps = q4 ? 4 : 1;
  best.row_blocks = (int)row_blocks;
  const int TM = best.TM = (int)cdiv(cdiv(M, 16), row_blocks);
  double least = 0;
  const double own_sum = gu || (!q4 && N > 8192) ? 5 : 0;   // (18960 x 2048 at 32 rows: 33.6 us in two parts)
  for (int TN = q4 && TM > 1 ? 2 : 4; TN >= (gu ? 2 : 1); TN /= 2) {   // (what the registers hold)
    const int64_t tiles = cdiv(rows_w, 16 * TN);
    for (int64_t S = 1; S <= std::min<int64_t>(max_S, units); S++) {
      const int64_t per = cdiv(units, S), blocks = tiles * row_blocks * S;
      if (cdiv(units, per) != S) continue;
      const double n = (double)(cdiv(per, rows::kWaves) * steps);    // steps of a wavefront
      const double mem = 8 * (70.0 * TM + (q4 ? 30.0 : 60.0) * TN);
      const double math = 2 * (q4 ? 1.8 * std::max(48.0 * TM * TN, 176.0 * TM + TN * (92.0 + 16 * TM)) : std::max(48.0 * TM * TN, 176.0 * TM));
      // (every CU is busy without a split, and the parts of more than a row tile cost more than the last round's gaps)
      if (!q4 && S > 1 && M > 16 && tiles * row_blocks > cus) break;
      const double rounds = blocks <= (q4 ? 2 : 4) * cus ? (double)cdiv(blocks, cus) : (double)blocks / cus;
      const double parts = S > 1 ? (double)S * M * rows_w * 4 / 1e6 : 0;
      // parts written and read, and their launch, which a gated product has and a wide one (a narrow one is planned as if
      // left as parts, whose sum its consumer forms: the two are the same bits)
      const double us = 2 + rounds * (!q4 && rounds > 1 ? 1.2 : 1.0) * (n * std::max(math, mem) + 3500 + 60 * TM * TN) / 2100 +
                        (S > 1 ? parts / 4 + own_sum : 0);
      if (best.S == 0 || us < least) {
        least = us;
        best.TN = TN;
        best.S = (int)S;
        best.tiles = (int)tiles;
        best.part_units = (int)per;
        // fewer steps than wavefronts leave some idle; five row tiles of int4 spill, and int4 blocks in turn wait for what
        // they would have loaded ahead; over many blocks, wavefronts with a unit more than others even out (38 x 18088 gated x
        // 2560, 20 units over eight wavefronts: 64 us here, 89 in the 64-row tiles)
        const double own = q4 && blocks > 2 * cus && per > rows::kWaves ? 1.05 * (double)per / rows::kWaves * steps : n;
        const double work = rounds * own * std::max(mem * (double)std::min<int64_t>(rows::kWaves, per) / rows::kWaves, per > 4 ? math : math / 2) / 2100;
        best.us = q4 ? 2 + work * (TM == 5 ? 1.3 : 1.0) * (rounds > 2 ? 1.2 : rounds > 1 ? 0.81 : 0.74) + rounds * (0.3 + 0.18 * TM * TN) + parts
                     : 0.85 + 1.15 * work + rounds * (1.2 + 0.18 * TM * TN) + 0.75 * parts;
        // many columns of a short K (14000 runs, N 20000 .. 160000): 24 x 21497 gated x 512 int4 24.8 us for an estimate of 20.3, 111 x
        // 10540 gated x 256 bf16 15.3 for 19.9
        if (blocks > 2 * cus) best.us *= q4 ? (per <= 4 ? 1.2 : 1.0) : M > 64 && K <= 384 ? 0.78 : 1.0;
      }
    }
  }
  return best;
}

RowsPlan plan_gemm_rows(int64_t M, int64_t N, int64_t K, bool gu, bool q4, int64_t max_S) {
  const int64_t rows_w = (gu ? 2 : 1) * N, t16 = (M + 15) / 16;
  if (M > 128 || K % (q4 ? 128 : 32) != 0 || M * K * 4 >= (int64_t(1) << 32) || rows_w * K * (q4 ? 1 : 4) / 2 >= (int64_t(1) << 32))
    return RowsPlan{};                             // (32-bit byte offsets)
  // Up to 16 rows nothing else is as fast, save for int4 with so few units that most wavefronts of a block have none and so many
  // columns that blocks come in more rounds than that: up to 65000 columns x 128 twice what the 64-row tiles take, x 256 1.4 times;
  // up to 32768 x 256 0.9 times
  if (q4 && M <= 16 && K < 512 && (rows_w + 63) / 64 > K / 128 * (int64_t)ctx().cus) return RowsPlan{};
  const auto plan = [&](int64_t row_blocks) { return plan_row_blocks(M, N, K, gu, q4, max_S, row_blocks); };
  if (!q4 || t16 != 5) return plan((t16 + rows::kMaxTM - 1) / rows::kMaxTM);
  // int4 with 65 to 80 rows: one block of five row tiles, or two of three (77 x 640 x 768 7.8 us and 6.1; 74 x 4609 x 11008, whose
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
