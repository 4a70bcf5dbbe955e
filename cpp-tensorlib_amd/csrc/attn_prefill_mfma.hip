// Causal prefill attention on the fp32 matrix pipe (tlhip_attn_prefill, cuda.h:1165-1201).
//
//   out[h, p, :] = softmax_k( scale * q[h, p, :] . K[kv(h), k, :] ) . V[kv(h), k, :],  k <= pos0 + p
//
// v_mfma_f32_32x32x2_f32 multiplies f32 by f32 exactly and accumulates in fp32, so scores and
// outputs differ from the reference's loops in summation order only.
//
// Two kernels: attn_prefill_small_kernel in tiles of 16 queries and 16 keys for head size 64, and for head size 128 where prompt and
// context are short; attn_prefill_mfma_kernel in tiles of 32 for the rest of head size 128. What follows is the second; the first
// has its own remarks.
//
// A block owns one query head and 32 consecutive query positions; its 8 wavefronts deal the
// 32-key tiles of the causal range round-robin and each keeps a running (max, sum, output) state
// for all 32 queries (online softmax), merged through LDS at the end. Per key tile a wavefront
// issues 2 x D/2 MFMAs (Q.K^T, then P.V):
//   * S[32 q x 32 k] : A = the Q tile (in LDS, shared by the block), B = the K tile from LDS;
//   * the score tile leaves the MFMA as one column (key) per lane and 16 rows (queries) per
//     lane, so row maxima and sums are lane reductions over half a wavefront;
//   * P goes through a 32 x 32 LDS tile to become the A operand of P.V; the output
//     accumulators share the score tile's row layout, so the softmax rescale needs no exchange.
// One MFMA consumes one float per lane per operand: lane l supplies A[l % 32][l / 32] and
// B[l / 32][l % 32]. The reduction index is consumed in the order 8m + 4(l/32) + j, which
// makes a lane's four consecutive steps one 16-byte LDS read (Q and K, or P and V, use the
// same order, and a sum does not care).
//
// K, P and V tiles are private to their wavefront and take turns in ONE LDS region (no block
// barriers inside the loop): K is dead once the scores exist, P once it sits in registers.
// Eight wavefronts are two per SIMD: one's softmax (~750 VALU instructions a tile) and load
// latency run under the other's 64-cycle MFMAs. One block per CU (9 regions of 32 x (D+4) floats).
#include "common.hpp"

namespace tlhip {

typedef float f32x16 __attribute__((ext_vector_type(16)));

template <int CTRL>
__device__ __forceinline__ float dpp_mov(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
// max / sum over the 32 lanes of a half wavefront (lanes that share lane / 32); result in every
// lane. Four DPP steps finish a 16-lane row; v_permlane16_swap (gfx950) then hands each row of a
// pair the other row's value: with both operands = v it returns (rows 0,0,2,2 ; rows 1,1,3,3).
__device__ __forceinline__ float half_max(float v) {
  v = fmaxf(v, dpp_mov<0xB1>(v));    // quad_perm [1,0,3,2]
  v = fmaxf(v, dpp_mov<0x4E>(v));    // quad_perm [2,3,0,1]
  v = fmaxf(v, dpp_mov<0x141>(v));   // row_half_mirror
  v = fmaxf(v, dpp_mov<0x140>(v));   // row_mirror
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float half_sum(float v) {
  v += dpp_mov<0xB1>(v);
  v += dpp_mov<0x4E>(v);
  v += dpp_mov<0x141>(v);
  v += dpp_mov<0x140>(v);
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

__device__ __forceinline__ float4 load_kv4(const float* p) { return *reinterpret_cast<const float4*>(p); }
__device__ __forceinline__ float4 load_kv4(const uint16_t* p) {   // 4 bf16, widened exactly
  const uint2 r = *reinterpret_cast<const uint2*>(p);
  return make_float4(bf16_lo(r.x), bf16_hi(r.x), bf16_lo(r.y), bf16_hi(r.y));
}

// LDS: the Q tile (shared by the block) and one 32 x (D+4) region per wavefront that holds the K
// tile, then P, then the V tile.
struct PrefillLds {
  static constexpr int D = 128;
  static constexpr int KS = D + 4;
  static constexpr int PS = 36;
  static constexpr int kRegion = 32 * KS;                 // floats: Q, and one region per wavefront
  static constexpr size_t kBytes = (size_t)9 * kRegion * sizeof(float);
};

template <typename KT>
__global__ __launch_bounds__(512, 1) void attn_prefill_mfma_kernel(const float* __restrict__ q,
                                                                    const KT* __restrict__ K,
                                                                    const KT* __restrict__ V,
                                                                    float* __restrict__ out, int group, int T,
                                                                    int pos0, int64_t kv_stride, float scale,
                                                                    int64_t o_head, int64_t o_row) {
  using L = PrefillLds;
  constexpr int D = L::D, KS = L::KS, PS = L::PS;
  constexpr int kLoads = 32 * D / 4 / 64;
  extern __shared__ __attribute__((aligned(16))) float lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l31 = lane & 31, hi = lane >> 5;
  const int h = blockIdx.x;
  const int nqt = (T + 31) >> 5;
  const int p0 = (nqt - 1 - (int)blockIdx.y) * 32;
  const KT* Kh = K + (size_t)(h / group) * kv_stride;
  const KT* Vh = V + (size_t)(h / group) * kv_stride;
  float* Qs = lds;
  float* R = lds + (1 + wave) * L::kRegion;
  const int kend = min(pos0 + p0 + 32, pos0 + T);
  const int nkt = (kend + 31) >> 5;

  for (int slot = tid; slot < 32 * D / 4; slot += 512) {   // Q tile -> LDS (rows beyond T clamped, never stored)
    const int row = slot / (D / 4), c4 = slot % (D / 4);
    *reinterpret_cast<float4*>(Qs + row * KS + 4 * c4) =
        *reinterpret_cast<const float4*>(q + ((size_t)h * T + min(p0 + row, T - 1)) * D + 4 * c4);
  }
  __syncthreads();

  f32x16 o[D / 32];
#pragma unroll
  for (int dt = 0; dt < D / 32; dt++)
#pragma unroll
    for (int v = 0; v < 16; v++) o[dt][v] = 0.f;
  float mrow[16], lrow[16];
#pragma unroll
  for (int v = 0; v < 16; v++) { mrow[v] = -INFINITY; lrow[v] = 0.f; }

  // K and V rows of a tile travel through registers into the wavefront's LDS region. The
  // registers are free again as soon as the tile has been written to LDS, so the NEXT tile's
  // rows are requested at that point - K right after the K tile is stored, V right after the V
  // tile is stored - and have a whole tile's arithmetic to arrive in. (Rows past the causal
  // range are clamped to its last row: mapped memory, masked when used.)
  float4 kreg[kLoads], vreg[kLoads];
  const auto request = [&](float4* dst, const KT* base, int tile) {
#pragma unroll
    for (int i = 0; i < kLoads; i++) {
      const int slot = lane + 64 * i, key = slot / (D / 4), c4 = slot % (D / 4);
      dst[i] = load_kv4(base + (size_t)min(tile * 32 + key, kend - 1) * D + 4 * c4);
    }
  };
  request(kreg, Kh, wave);
  request(vreg, Vh, wave);
#ifdef TLHIP_TRACE
  unsigned long long ph[5] = {0, 0, 0, 0, 0}, tc = __builtin_readcyclecounter();
  TLHIP_MARK(0);
#define TLHIP_PHASE(i) do { const unsigned long long n_ = __builtin_readcyclecounter(); ph[i] += n_ - tc; tc = n_; } while (0)
#else
#define TLHIP_PHASE(i)
#endif
  for (int kt = wave; kt < nkt; kt += 8) {
    const int k0 = kt * 32;
#pragma unroll
    for (int i = 0; i < kLoads; i++) {
      const int slot = lane + 64 * i, key = slot / (D / 4), c4 = slot % (D / 4);
      *reinterpret_cast<float4*>(R + key * KS + 4 * c4) = kreg[i];
    }
    request(kreg, Kh, kt + 8);
    TLHIP_PHASE(0);
    f32x16 s;
#pragma unroll
    for (int v = 0; v < 16; v++) s[v] = 0.f;
#pragma unroll
    for (int m = 0; m < D / 8; m++) {
      const float4 qa = *reinterpret_cast<const float4*>(Qs + l31 * KS + 8 * m + 4 * hi);
      const float4 kf = *reinterpret_cast<const float4*>(R + l31 * KS + 8 * m + 4 * hi);
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(qa.x, kf.x, s, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(qa.y, kf.y, s, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(qa.z, kf.z, s, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(qa.w, kf.w, s, 0, 0, 0);
    }
    TLHIP_PHASE(1);
    const int key = k0 + l31;
#pragma unroll
    for (int v = 0; v < 16; v++) {
      const int r = 8 * (v >> 2) + 4 * hi + (v & 3);
      const bool seen = key <= pos0 + p0 + r && key < kend;
      const float sv = seen ? s[v] * scale : -INFINITY;
      const float mnew = fmaxf(mrow[v], half_max(sv));
      const float mref = mnew == -INFINITY ? 0.f : mnew;
      const float corr = __expf(mrow[v] - mref);
      const float p = __expf(sv - mref);
      lrow[v] = lrow[v] * corr + half_sum(p);
      mrow[v] = mnew;
#pragma unroll
      for (int dt = 0; dt < D / 32; dt++) o[dt][v] *= corr;
      R[r * PS + l31] = p;                      // the K tile is dead: P takes its place
    }
    float4 pf[4];
#pragma unroll
    for (int m = 0; m < 4; m++) pf[m] = *reinterpret_cast<const float4*>(R + l31 * PS + 8 * m + 4 * hi);
#pragma unroll
    for (int i = 0; i < kLoads; i++) {          // P is in registers: V takes the region
      const int slot = lane + 64 * i, vkey = slot / (D / 4), c4 = slot % (D / 4);
      *reinterpret_cast<float4*>(R + vkey * D + 4 * c4) = vreg[i];
    }
    request(vreg, Vh, kt + 8);
    TLHIP_PHASE(2);
    // (the D/32 output tiles take turns, so consecutive MFMAs never wait for each other's result)
#pragma unroll
    for (int m = 0; m < 4; m++) {
      const float pj[4] = {pf[m].x, pf[m].y, pf[m].z, pf[m].w};
#pragma unroll
      for (int j = 0; j < 4; j++) {
#pragma unroll
        for (int dt = 0; dt < D / 32; dt++) {
          const float* vp = R + (8 * m + 4 * hi + j) * D + dt * 32 + l31;
          o[dt] = __builtin_amdgcn_mfma_f32_32x32x2f32(pj[j], vp[0], o[dt], 0, 0, 0);
        }
      }
    }
    TLHIP_PHASE(3);
  }
#ifdef TLHIP_TRACE
  {
    const unsigned b = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
    if (lane == 0 && b < kTraceBlocks) {
      unsigned long long* g = &g_trace[(b * kTraceWaves + wave) * kTraceSlots];
      g[1] = ph[0]; g[2] = ph[1]; g[3] = ph[2]; g[4] = ph[3]; g[5] = (nkt - wave + 7) / 8;
    }
  }
  TLHIP_MARK(6);
#endif
#undef TLHIP_PHASE

  // merge: each wavefront leaves O [32][D], m [32], l [32] in its region; 16 threads finish a row
  float* Mw = R + 32 * D;
#pragma unroll
  for (int v = 0; v < 16; v++) {
    const int r = 8 * (v >> 2) + 4 * hi + (v & 3);
#pragma unroll
    for (int dt = 0; dt < D / 32; dt++) R[r * D + dt * 32 + l31] = o[dt][v];
    if (l31 == 0) { Mw[r] = mrow[v]; Mw[32 + r] = lrow[v]; }
  }
  __syncthreads();
  {
    const int row = tid >> 4, d0 = (tid & 15) * (D / 16);
    const float* base = lds + L::kRegion;
    float f[8], M = -INFINITY, Lsum = 0.f;
#pragma unroll
    for (int w = 0; w < 8; w++) M = fmaxf(M, base[w * L::kRegion + 32 * D + row]);
#pragma unroll
    for (int w = 0; w < 8; w++) {
      const float mw = base[w * L::kRegion + 32 * D + row];
      f[w] = mw == -INFINITY ? 0.f : __expf(mw - M);
      Lsum += f[w] * base[w * L::kRegion + 32 * D + 32 + row];
    }
    if (p0 + row < T) {
      const float inv = 1.0f / Lsum;
      float* op = out + (size_t)h * o_head + (size_t)(p0 + row) * o_row + d0;   // [Hq,T,D] or [T,Hq*D]
#pragma unroll
      for (int d = 0; d < D / 16; d += 4) {
        float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int w = 0; w < 8; w++) {
          const float4 ow = *reinterpret_cast<const float4*>(base + w * L::kRegion + row * D + d0 + d);
          a.x += f[w] * ow.x; a.y += f[w] * ow.y; a.z += f[w] * ow.z; a.w += f[w] * ow.w;
        }
        *reinterpret_cast<float4*>(op + d) = make_float4(a.x * inv, a.y * inv, a.z * inv, a.w * inv);
      }
    }
  }
}

// The same in tiles of 16 queries and 16 keys, for prompts so short that the tiles above leave the chip idle: three of a block's
// wavefronts had a key tile each at 77 tokens, and a wavefront alone needs 2.8 us for the softmax of 32 x 32 scores. Both products are
// formed transposed (S^T = K Q^T, O^T = V^T P^T): lane (g, c) = (l / 16, l % 16) then holds the scores of query c for the keys 4 g ..
// 4 g + 3 of a tile, which are its operand of the second product as they are - one running maximum and sum to a lane, two register
// swaps per statistic, no LDS until the wavefronts' states meet. All operands come from memory in 16-byte pieces: reduction step (m, j)
// of the scores takes dims 16 m + 4 g + j, and output tile n of the second product holds the dims 64 (n / 4) + 4 c + n % 4, so
// that a lane's piece of a V row is one element of each of four tiles. The next tile's rows are requested before this one's
// arithmetic. 14 heads of 64, 77 tokens: 7.3 -> 4.9 us; error against 64 bits
// 0.7 of the larger tiles' (shorter sums).
template <int D, typename KT>
__global__ __launch_bounds__(512, 1) void attn_prefill_small_kernel(const float* __restrict__ q, const KT* __restrict__ K,
                                                                     const KT* __restrict__ V, float* __restrict__ out, int group, int T,
                                                                     int pos0, int64_t kv_stride, float scale, int64_t o_head,
                                                                     int64_t o_row) {
  typedef float f32x4 __attribute__((ext_vector_type(4)));
  constexpr int NM = D / 16, OS = D + 4;             // 16-byte pieces of a row per lane; row stride of the states in LDS
  __shared__ __attribute__((aligned(16))) float states[8][16][OS];
  __shared__ float ms[8][16], ls[8][16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, c = lane & 15, g = lane >> 4;
  const int h = blockIdx.x, p0 = ((T + 15) / 16 - 1 - (int)blockIdx.y) * 16;
  const KT* Kh = K + (size_t)(h / group) * kv_stride;
  const KT* Vh = V + (size_t)(h / group) * kv_stride;
  const int kend = min(pos0 + p0 + 16, pos0 + T), nkt = (kend + 15) >> 4;
  const int limit = pos0 + min(p0 + c, T - 1);       // the last key this lane's query sees (queries past T are not stored)

  float4 kr[NM], vr[NM];                             // K: dims 16 m + 4 g .. of key c; V: dims 64 (m / 4) + 4 c .. of key 4 g + m % 4
  const auto request = [&](int tile) {
    const KT* kp = Kh + (size_t)min(tile * 16 + c, kend - 1) * D + 4 * g;
#pragma unroll
    for (int m = 0; m < NM; m++) kr[m] = load_kv4(kp + 16 * m);
#pragma unroll
    for (int m = 0; m < NM; m++)
      vr[m] = load_kv4(Vh + (size_t)min(tile * 16 + 4 * g + (m & 3), kend - 1) * D + 64 * (m >> 2) + 4 * c);
  };
  float4 qr[NM];
  const float* qp = q + ((size_t)h * T + min(p0 + c, T - 1)) * D + 4 * g;
#pragma unroll
  for (int m = 0; m < NM; m++) qr[m] = *reinterpret_cast<const float4*>(qp + 16 * m);
  request(wave);

  f32x4 o[NM];
#pragma unroll
  for (int n = 0; n < NM; n++) o[n] = f32x4{0.f, 0.f, 0.f, 0.f};
  float mrow = -INFINITY, lrow = 0.f;
  for (int kt = wave; kt < nkt; kt += 8) {
    float4 kc[NM], vc[NM];
#pragma unroll
    for (int m = 0; m < NM; m++) { kc[m] = kr[m]; vc[m] = vr[m]; }
    if (kt + 8 < nkt) request(kt + 8);
    f32x4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = s0;
#pragma unroll
    for (int m = 0; m < NM; m++) {
      s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(kc[m].x, qr[m].x, s0, 0, 0, 0);
      s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(kc[m].y, qr[m].y, s1, 0, 0, 0);
      s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(kc[m].z, qr[m].z, s0, 0, 0, 0);
      s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(kc[m].w, qr[m].w, s1, 0, 0, 0);
    }
    float sv[4], mx = -INFINITY;
#pragma unroll
    for (int v = 0; v < 4; v++) {
      sv[v] = kt * 16 + 4 * g + v <= limit ? (s0[v] + s1[v]) * scale : -INFINITY;
      mx = fmaxf(mx, sv[v]);
    }
    const auto over_groups = [](float x, auto op) {   // over the four lanes of a query
      LanePair p = swap16(x, x);
      x = op(p.first, p.second);
      p = swap32(x, x);
      return op(p.first, p.second);
    };
    mx = over_groups(mx, [](float x, float y) { return fmaxf(x, y); });
    const float mnew = fmaxf(mrow, mx), mref = mnew == -INFINITY ? 0.f : mnew, corr = __expf(mrow - mref);
    float p[4], sum = 0.f;
#pragma unroll
    for (int v = 0; v < 4; v++) {
      p[v] = __expf(sv[v] - mref);
      sum += p[v];
    }
    lrow = lrow * corr + sum;                        // of this lane's keys
    mrow = mnew;
    if (__any(corr != 1.f)) {
#pragma unroll
      for (int n = 0; n < NM; n++) o[n] *= corr;
    }
#pragma unroll
    for (int v = 0; v < 4; v++)
#pragma unroll
      for (int half = 0; half < NM / 4; half++) {
        const float4 x = vc[4 * half + v];
        o[4 * half] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.x, p[v], o[4 * half], 0, 0, 0);
        o[4 * half + 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.y, p[v], o[4 * half + 1], 0, 0, 0);
        o[4 * half + 2] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.z, p[v], o[4 * half + 2], 0, 0, 0);
        o[4 * half + 3] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.w, p[v], o[4 * half + 3], 0, 0, 0);
      }
  }
  // o[4 half + e][v]: query c, dim 64 half + 4 (4 g + v) + e
#pragma unroll
  for (int half = 0; half < NM / 4; half++)
#pragma unroll
    for (int v = 0; v < 4; v++)
      *reinterpret_cast<f32x4*>(&states[wave][c][64 * half + 16 * g + 4 * v]) = f32x4{o[4 * half][v], o[4 * half + 1][v], o[4 * half + 2][v], o[4 * half + 3][v]};
  {
    LanePair p = swap16(lrow, lrow);
    const float l = p.first + p.second;
    p = swap32(l, l);
    if (g == 0) { ms[wave][c] = mrow; ls[wave][c] = p.first + p.second; }
  }
  __syncthreads();
  const int used = min(8, nkt);                      // wavefronts that had a tile
  for (int i = tid; i < 16 * D / 4; i += 512) {
    const int row = i / (D / 4), d = 4 * (i % (D / 4));
    if (p0 + row >= T) continue;
    float M = -INFINITY, L = 0.f;
    for (int w = 0; w < used; w++) M = fmaxf(M, ms[w][row]);
    f32x4 a = {0.f, 0.f, 0.f, 0.f};
    for (int w = 0; w < used; w++) {
      const float m = ms[w][row], f = m == -INFINITY ? 0.f : __expf(m - M);
      L += f * ls[w][row];
      a += f * *reinterpret_cast<const f32x4*>(&states[w][row][d]);
    }
    *reinterpret_cast<f32x4*>(out + (size_t)h * o_head + (size_t)(p0 + row) * o_row + d) = a * (1.0f / L);
  }
}

// Which of the two: heads of 64 always the small tiles (58 shapes of 14 to 128 heads, 2 to 1000 keys: 1.01 to 1.95 times as fast);
// heads of 128, whose states fill twice the LDS and whose K and V rows every 16 queries then read again, while their blocks
// make one round of the CUs or the keys are few (28 heads, 77 tokens 10.8 -> 7.0 us, 150 15.7 -> 10.3, 77 after 400 27.6 -> 19.0; but 150
// after 400, 280 blocks, 31.8 -> 33.3, 64 heads of 100 tokens after 150 17.3 -> 21.8).
template <int D, typename KT>
int launch_prefill_mfma(const float* q, const KT* K, const KT* V, float* out, int Hq, int Hkv, int T,
                        int64_t kv_max, float scale, int pos0, int token_major) {
  Context& c = ctx();
  const int64_t o_head = token_major ? D : (int64_t)T * D, o_row = token_major ? (int64_t)Hq * D : D;
  const int t16 = (T + 15) / 16;
  if (D == 64 || (int64_t)Hq * t16 <= c.cus || pos0 + T <= 160) {
    hipLaunchKernelGGL((attn_prefill_small_kernel<D, KT>), dim3((unsigned)Hq, (unsigned)t16), dim3(512), 0, c.stream, q, K, V, out, Hq / Hkv, T, pos0,
                       kv_max * (int64_t)D, scale, o_head, o_row);
    return 0;
  }
  if constexpr (D == 128) {
    auto fn = attn_prefill_mfma_kernel<KT>;
    const int lds = (int)PrefillLds::kBytes;
    if ((size_t)lds > (size_t)c.lds_per_cu) return fail(TLHIP_EUNSUPPORTED, "tlhip_attn_prefill: not enough LDS");
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) return hip_fail(e, "hipFuncSetAttribute(LDS)");
    hipLaunchKernelGGL(fn, dim3((unsigned)Hq, (unsigned)((T + 31) / 32)), dim3(512), (size_t)lds, c.stream, q, K, V, out, Hq / Hkv, T, pos0,
                       kv_max * (int64_t)D, scale, o_head, o_row);
  }
  return 0;
}

template int launch_prefill_mfma<128, float>(const float*, const float*, const float*, float*, int, int, int, int64_t, float, int, int);
template int launch_prefill_mfma<64, float>(const float*, const float*, const float*, float*, int, int, int, int64_t, float, int, int);
template int launch_prefill_mfma<128, uint16_t>(const float*, const uint16_t*, const uint16_t*, float*, int, int, int, int64_t, float, int, int);
template int launch_prefill_mfma<64, uint16_t>(const float*, const uint16_t*, const uint16_t*, float*, int, int, int, int64_t, float, int, int);

}  // namespace tlhip
