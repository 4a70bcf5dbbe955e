// Load-time weight conversion on the device.
//
// A model file stores linear layers as f16 (or f32 / bf16) rows [out, in]. The decode
// path wants bf16 rows [N, K], the int4 group format, or [K, N] for the seam's GEMV.
// The reference converts on the host, one element at a time, before uploading
// (bench/cuda/qwen_model.h:40-131, array.h:639-658, 703-742); here the file's bytes are
// uploaded as they are and these kernels write the decode formats straight into the
// weight buffers. All of it is byte/integer work at HBM speed, bit-identical to the
// host arithmetic.
#include <algorithm>

#include "common.hpp"

namespace tlhip {

// ---- element formats -----------------------------------------------------------------
// IEEE half -> float, every bit pattern (subnormals exact, NaN payload kept, no quieting):
// the values of bench/cuda/qwen_model.h:41-60.
__device__ __forceinline__ float f16_bits_to_f32(uint32_t h) {
  const uint32_t sign = (h & 0x8000u) << 16, exp = (h >> 10) & 31u, man = h & 0x3ffu;
  uint32_t bits;
  if (exp == 0) {
    // zero or subnormal: man * 2^-24, exact in f32 (and a normal f32, so no flush applies)
    bits = __float_as_uint(static_cast<float>(man) * 5.9604644775390625e-8f);
  } else if (exp == 31) {
    bits = 0x7f800000u | (man << 13);
  } else {
    bits = ((exp + 112u) << 23) | (man << 13);
  }
  return __uint_as_float(sign | bits);
}

template <int T> struct Elem;   // T: TLHIP_T_F32 / F16 / BF16
template <> struct Elem<TLHIP_T_F32> {
  using type = float;
  static __device__ __forceinline__ float load(const float* p, int64_t i) { return p[i]; }
  static __device__ __forceinline__ void store(float* p, int64_t i, float v) { p[i] = v; }
};
template <> struct Elem<TLHIP_T_F16> {
  using type = uint16_t;
  static __device__ __forceinline__ float load(const uint16_t* p, int64_t i) { return f16_bits_to_f32(p[i]); }
};
template <> struct Elem<TLHIP_T_BF16> {
  using type = uint16_t;
  static __device__ __forceinline__ float load(const uint16_t* p, int64_t i) {
    return __uint_as_float(static_cast<uint32_t>(p[i]) << 16);
  }
  static __device__ __forceinline__ void store(uint16_t* p, int64_t i, float v) { p[i] = f32_to_bf16_rne(v); }
};

// Eight consecutive source elements as floats (16-byte loads where the type allows).
template <int S>
__device__ __forceinline__ void load8(const typename Elem<S>::type* src, int64_t i, float (&v)[8]) {
  if constexpr (S == TLHIP_T_F32) {
    const float4 a = *reinterpret_cast<const float4*>(src + i), b = *reinterpret_cast<const float4*>(src + i + 4);
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
  } else {
    const uint4 r = *reinterpret_cast<const uint4*>(src + i);
    const uint32_t w[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
    for (int k = 0; k < 4; k++) {
      if constexpr (S == TLHIP_T_F16) {
        v[2 * k] = f16_bits_to_f32(w[k] & 0xffffu);
        v[2 * k + 1] = f16_bits_to_f32(w[k] >> 16);
      } else {
        v[2 * k] = bf16_lo(w[k]);
        v[2 * k + 1] = bf16_hi(w[k]);
      }
    }
  }
}

// ---- dst[i] = narrow(widen(src[i])): same layout, other element type ---------------------
template <int S, int T>
__global__ __launch_bounds__(256) void convert_kernel(const typename Elem<S>::type* __restrict__ src,
                                                      typename Elem<T>::type* __restrict__ dst, int64_t n) {
  const int64_t i = (static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x) * 8;
  if (i + 8 <= n) {
    float v[8];
    load8<S>(src, i, v);
    if constexpr (T == TLHIP_T_F32) {
      *reinterpret_cast<float4*>(dst + i) = make_float4(v[0], v[1], v[2], v[3]);
      *reinterpret_cast<float4*>(dst + i + 4) = make_float4(v[4], v[5], v[6], v[7]);
    } else {
      uint32_t w[4];
#pragma unroll
      for (int k = 0; k < 4; k++)
        w[k] = static_cast<uint32_t>(f32_to_bf16_rne(v[2 * k])) |
               (static_cast<uint32_t>(f32_to_bf16_rne(v[2 * k + 1])) << 16);
      *reinterpret_cast<uint4*>(dst + i) = make_uint4(w[0], w[1], w[2], w[3]);
    }
  } else {
    for (int64_t j = i; j < n; j++) Elem<T>::store(dst, j, Elem<S>::load(src, j));
  }
}

// ---- dst[c * ld + col_base + r] = src[r * cols + c]: file rows [out, in] -> [K, N] -------------
// 64 x 64 tiles through LDS so that both sides move whole cache lines.
template <int S, int T>
__global__ __launch_bounds__(256) void convert_transpose_kernel(
    const typename Elem<S>::type* __restrict__ src, typename Elem<T>::type* __restrict__ dst,
    int64_t rows, int64_t cols, int64_t ld, int64_t col_base) {
  __shared__ float tile[64][65];
  const int64_t r0 = static_cast<int64_t>(blockIdx.y) * 64, c0 = static_cast<int64_t>(blockIdx.x) * 64;
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;   // 64 x 4
  for (int j = ty; j < 64; j += 4) {
    const int64_t r = r0 + j, c = c0 + tx;
    if (r < rows && c < cols) tile[j][tx] = Elem<S>::load(src, r * cols + c);
  }
  __syncthreads();
  for (int j = ty; j < 64; j += 4) {
    const int64_t c = c0 + j, r = r0 + tx;   // output row = source column
    if (r < rows && c < cols) Elem<T>::store(dst, c * ld + col_base + r, tile[tx][j]);
  }
}

// ---- int4 group quantiser (array.h:703-742 on the widened rows) ----------------------------
// Per group of 32 consecutive weights of a row: scale = max(1e-8, maxabs) / 7, q = clamp(lround(w / scale), -8, 7),
// stored nibble q + 8, even k in the low nibble. Rows are contiguous on both sides, so group t reads elements
// [32 t, 32 t + 32) and writes packed bytes [16 t, 16 t + 16) and scale t.
//
// What bounds it: vector instructions. A correctly rounded division and a rounding per weight are some 25 of them (two
// thirds of 58 us for 18944 x 3584), and lround(w / scale) needs neither: with n = floor of an approximate quotient
// the answer is n or n + 1, n + 1 exactly when the ROUNDED quotient reaches h = n + 1/2, i.e. when |w| / scale is at
// least h minus half the spacing of floats below h (a tie rounds to h, whose last bit is even). |w| - h scale is one
// FMA, exact where it matters, and the half spacing is 2^-24 times the power of two at or below h's predecessor.
// An approximate quotient on the wrong side of a whole number gives the same answer. Two lanes share a group, 16
// weights each: the loads of a wavefront cover whole lines. Groups that hold an infinity or a NaN go the long way.
__device__ __forceinline__ uint32_t quantize8_long(const float* w, float scale) {
  uint32_t out = 0u;
#pragma unroll 1
  for (int k = 0; k < 8; k++) {
    float q = roundf(__fdiv_rn(w[k], scale));   // half away from zero, like lround
    q = fminf(fmaxf(q, -8.0f), 7.0f);
    out |= static_cast<uint32_t>(static_cast<int>(q) + 8) << (k * 4);
  }
  return out;
}
__device__ __forceinline__ uint32_t quantize8(const float* w, float scale, float inv, float step) {   // step = scale 2^-24
  uint32_t out = 0x88888888u;
#pragma unroll
  for (int k = 0; k < 8; k++) {
    const float a = fabsf(w[k]), n = floorf(a * inv), h = n + 0.5f;
    const float below = __uint_as_float((__float_as_uint(h) - 1u) & 0x7f800000u);
    const int q = static_cast<int>(n) + (fmaf(-h, scale, a) >= -(below * step) ? 1 : 0), s = __float_as_int(w[k]) >> 31;
    out += static_cast<uint32_t>((q ^ s) - s) << (k * 4);   // bytes in memory order, even k low
  }
  return out;
}

// Eight consecutive source elements as floats; f16 by the conversion instruction, exact for every finite half (a NaN
// may change its payload, which no nibble shows).
template <int S>
__device__ __forceinline__ void widen8(const typename Elem<S>::type* src, int64_t i, float* v) {
  if constexpr (S == TLHIP_T_F16) {
    typedef _Float16 half8 __attribute__((ext_vector_type(8)));
    const half8 h = *reinterpret_cast<const half8*>(src + i);
#pragma unroll
    for (int k = 0; k < 8; k++) v[k] = static_cast<float>(h[k]);
  } else {
    float t[8];
    load8<S>(src, i, t);
#pragma unroll
    for (int k = 0; k < 8; k++) v[k] = t[k];
  }
}

template <int S>
__global__ __launch_bounds__(256) void quantize_q4_kernel(const typename Elem<S>::type* __restrict__ src,
                                                          uint2* __restrict__ packed,
                                                          float* __restrict__ scales, int64_t groups) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;   // half a group
  if (t >= 2 * groups) return;                     // (both halves of a group, or neither)
  float w[16];
  widen8<S>(src, t * 16, w);
  widen8<S>(src, t * 16 + 8, w + 8);
  uint32_t top = 0u;                               // of the magnitudes' bits: in their order, NaN above infinity
#pragma unroll
  for (int k = 0; k < 16; k++) top = max(top, __float_as_uint(w[k]) & 0x7fffffffu);
  top = max(top, static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(top), 0xb1, 0xf, 0xf, true)));   // quad_perm 1 0 3 2
  uint2 out;
  float scale;
  if (top < 0x7f800000u) {
    scale = __fdiv_rn(fmaxf(__uint_as_float(top), 1e-8f), 7.0f);
    const float inv = __builtin_amdgcn_rcpf(scale), step = scale * 5.9604644775390625e-8f;
    out = make_uint2(quantize8(w, scale, inv, step), quantize8(w + 8, scale, inv, step));
  } else {
    float maxabs = 1e-8f;                          // what is not a number is not a maximum
#pragma unroll 1
    for (int k = 0; k < 16; k++) {
      const float a = fabsf(w[k]);
      if (a > maxabs) maxabs = a;
    }
    maxabs = fmaxf(maxabs, __shfl_xor(maxabs, 1));
    scale = __fdiv_rn(maxabs, 7.0f);
    out = make_uint2(quantize8_long(w, scale), quantize8_long(w + 8, scale));
  }
  packed[t] = out;
  if ((t & 1) == 0) scales[t >> 1] = scale;
}

// out[j] = widen(table[tok][j]) for an f16 embedding table, tok read from the device
// (the row gather of bench/cuda/qwen_model.h:531-540 without the host in between).
__global__ __launch_bounds__(256) void embed_gather_f16_kernel(const uint16_t* __restrict__ table,
                                                               const int* __restrict__ d_token,
                                                               float* __restrict__ out, int hidden,
                                                               int vocab) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= hidden) return;
  int tok = *d_token;
  tok = tok < 0 ? 0 : (tok >= vocab ? vocab - 1 : tok);
  out[j] = f16_bits_to_f32(table[static_cast<size_t>(tok) * hidden + j]);
}

// out[t][j] = widen(table[ids[t]][j]). The ids ride in the launch's arguments: no copy to wait for (a prompt of 512 x 3584
// widened on the host and copied took 600 us, this 6). Bound by the launch; V numbers a thread.
template <int M> struct TokenIds { int id[M]; };   // a launch of one id carries few
constexpr int kFewIds = 8, kManyIds = 768;
template <bool F16, int V, int M>
__global__ __launch_bounds__(256) void embed_rows_kernel(const uint16_t* __restrict__ table, const TokenIds<M> ids,
                                                         float* __restrict__ out, int hidden) {
  const int t = blockIdx.y, j = (blockIdx.x * 256 + threadIdx.x) * V;
  if (j >= hidden) return;
  const uint16_t* row = table + (size_t)ids.id[t] * hidden + j;
  float* o = out + (size_t)t * hidden + j;
  if constexpr (V == 8) {
    const uint4 w = *reinterpret_cast<const uint4*>(row);
    const uint32_t d[4] = {w.x, w.y, w.z, w.w};
    float f[8];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      f[2 * i] = F16 ? f16_bits_to_f32((uint16_t)(d[i] & 0xffffu)) : bf16_lo(d[i]);
      f[2 * i + 1] = F16 ? f16_bits_to_f32((uint16_t)(d[i] >> 16)) : bf16_hi(d[i]);
    }
    reinterpret_cast<float4*>(o)[0] = make_float4(f[0], f[1], f[2], f[3]);
    reinterpret_cast<float4*>(o)[1] = make_float4(f[4], f[5], f[6], f[7]);
  } else {
    *o = F16 ? f16_bits_to_f32(*row) : __uint_as_float((uint32_t)*row << 16);
  }
}

template <bool F16, int V, int M>
static void launch_embed_rows(const void* table, const int64_t* ids, int64_t T, float* out, int64_t hidden) {
  const unsigned gx = (unsigned)((hidden + 256 * V - 1) / (256 * V));
  for (int64_t t0 = 0; t0 < T; t0 += M) {
    const int n = (int)std::min<int64_t>(T - t0, M);
    TokenIds<M> a{};
    for (int t = 0; t < n; t++) a.id[t] = (int)ids[t0 + t];
    embed_rows_kernel<F16, V, M><<<dim3(gx, (unsigned)n), dim3(256), 0, ctx().stream>>>(
        static_cast<const uint16_t*>(table), a, out + t0 * hidden, (int)hidden);
  }
}

static bool known_type(int t) { return t == TLHIP_T_F32 || t == TLHIP_T_F16 || t == TLHIP_T_BF16; }

}  // namespace tlhip

using namespace tlhip;

// (S, T) dispatch: sources f32 / f16 / bf16, destinations f32 / bf16
#define TLHIP_CONVERT_DISPATCH(S_, T_, CALL)                                             \
  do {                                                                                   \
    if ((T_) == TLHIP_T_F32) {                                                           \
      if ((S_) == TLHIP_T_F32) { CALL(TLHIP_T_F32, TLHIP_T_F32); }                       \
      else if ((S_) == TLHIP_T_F16) { CALL(TLHIP_T_F16, TLHIP_T_F32); }                  \
      else { CALL(TLHIP_T_BF16, TLHIP_T_F32); }                                          \
    } else {                                                                             \
      if ((S_) == TLHIP_T_F32) { CALL(TLHIP_T_F32, TLHIP_T_BF16); }                      \
      else if ((S_) == TLHIP_T_F16) { CALL(TLHIP_T_F16, TLHIP_T_BF16); }                 \
      else { CALL(TLHIP_T_BF16, TLHIP_T_BF16); }                                         \
    }                                                                                    \
  } while (0)

extern "C" {

int tlhip_convert(const void* src, int src_type, void* dst, int dst_type, int64_t n) {
  TLHIP_REQUIRE_READY();
  if (!src || !dst) return fail(TLHIP_EINVAL, "tlhip_convert: null pointer");
  if (!known_type(src_type) || (dst_type != TLHIP_T_F32 && dst_type != TLHIP_T_BF16))
    return fail(TLHIP_EUNSUPPORTED, "tlhip_convert: element types %d -> %d", src_type, dst_type);
  if (n <= 0) return fail(TLHIP_EINVAL, "tlhip_convert: n must be positive");
  if (!aligned16(src) || !aligned16(dst)) return fail(TLHIP_EINVAL, "tlhip_convert: operands must be 16-byte aligned");
  const int64_t blocks = (n + 2047) / 2048;
  if (blocks > 0x7fffffff) return fail(TLHIP_EUNSUPPORTED, "tlhip_convert: too many elements");
#define CALL(S, T)                                                                              \
  convert_kernel<S, T><<<dim3((unsigned)blocks), dim3(256), 0, ctx().stream>>>(                 \
      static_cast<const Elem<S>::type*>(src), static_cast<Elem<T>::type*>(dst), n)
  TLHIP_CONVERT_DISPATCH(src_type, dst_type, CALL);
#undef CALL
  TLHIP_CHECK_LAUNCH(TLHIP_C_CONVERT);
}

int tlhip_convert_transpose(const void* src, int src_type, void* dst, int dst_type, int64_t rows,
                            int64_t cols, int64_t ld_dst, int64_t col_base) {
  TLHIP_REQUIRE_READY();
  if (!src || !dst) return fail(TLHIP_EINVAL, "tlhip_convert_transpose: null pointer");
  if (!known_type(src_type) || (dst_type != TLHIP_T_F32 && dst_type != TLHIP_T_BF16))
    return fail(TLHIP_EUNSUPPORTED, "tlhip_convert_transpose: element types %d -> %d", src_type, dst_type);
  if (rows <= 0 || cols <= 0 || col_base < 0 || col_base + rows > ld_dst)
    return fail(TLHIP_EINVAL, "tlhip_convert_transpose: need rows, cols > 0 and col_base + rows <= ld_dst");
  const int64_t gx = (cols + 63) / 64, gy = (rows + 63) / 64;
  if (gx > 0x7fffffff || gy > 65535) return fail(TLHIP_EUNSUPPORTED, "tlhip_convert_transpose: shape too large");
#define CALL(S, T)                                                                              \
  convert_transpose_kernel<S, T><<<dim3((unsigned)gx, (unsigned)gy), dim3(256), 0, ctx().stream>>>( \
      static_cast<const Elem<S>::type*>(src), static_cast<Elem<T>::type*>(dst), rows, cols, ld_dst, col_base)
  TLHIP_CONVERT_DISPATCH(src_type, dst_type, CALL);
#undef CALL
  TLHIP_CHECK_LAUNCH(TLHIP_C_CONVERT);
}

int tlhip_quantize_q4(const void* src, int src_type, void* packed, void* scales, int64_t rows,
                      int64_t K, int64_t group) {
  TLHIP_REQUIRE_READY();
  if (!src || !packed || !scales) return fail(TLHIP_EINVAL, "tlhip_quantize_q4: null pointer");
  if (!known_type(src_type)) return fail(TLHIP_EUNSUPPORTED, "tlhip_quantize_q4: element type %d", src_type);
  if (group != 32) return fail(TLHIP_EUNSUPPORTED, "tlhip_quantize_q4: group must be 32");   // types.h:20
  if (rows <= 0 || K <= 0 || K % 32 != 0) return fail(TLHIP_EINVAL, "tlhip_quantize_q4: need rows > 0, K a positive multiple of 32");
  if (!aligned16(src) || !aligned16(packed) || (reinterpret_cast<uintptr_t>(scales) & 3u))
    return fail(TLHIP_EINVAL, "tlhip_quantize_q4: src and packed must be 16-byte aligned, scales 4-byte");
  const int64_t groups = rows * (K / 32);
  if ((groups + 255) / 256 > 0x7fffffff) return fail(TLHIP_EUNSUPPORTED, "tlhip_quantize_q4: too many groups");
  // (a grid's x counts threads in 32 bits, and a group takes two: at most 2^30 groups a launch)
  for (int64_t g0 = 0; g0 < groups; g0 += (int64_t)1 << 30) {
    const int64_t n = std::min<int64_t>(groups - g0, (int64_t)1 << 30);
    uint2* pk = static_cast<uint2*>(packed) + 2 * g0;
    float* sc = static_cast<float*>(scales) + g0;
    const dim3 grid((unsigned)((2 * n + 255) / 256)), block(256);
    if (src_type == TLHIP_T_F32)
      quantize_q4_kernel<TLHIP_T_F32><<<grid, block, 0, ctx().stream>>>(static_cast<const float*>(src) + 32 * g0, pk, sc, n);
    else if (src_type == TLHIP_T_F16)
      quantize_q4_kernel<TLHIP_T_F16><<<grid, block, 0, ctx().stream>>>(static_cast<const uint16_t*>(src) + 32 * g0, pk, sc, n);
    else
      quantize_q4_kernel<TLHIP_T_BF16><<<grid, block, 0, ctx().stream>>>(static_cast<const uint16_t*>(src) + 32 * g0, pk, sc, n);
  }
  TLHIP_CHECK_LAUNCH(TLHIP_C_QUANTIZE_Q4);
}

int tlhip_embed_gather_f16(const void* table, const void* d_token, void* out, int64_t hidden,
                           int64_t vocab) {
  TLHIP_REQUIRE_READY();
  if (!table || !d_token || !out) return fail(TLHIP_EINVAL, "tlhip_embed_gather_f16: null pointer");
  if (hidden <= 0 || vocab <= 0 || hidden > 0x7fffffff || vocab > 0x7fffffff)
    return fail(TLHIP_EINVAL, "tlhip_embed_gather_f16: bad shape");
  embed_gather_f16_kernel<<<dim3((unsigned)((hidden + 255) / 256)), dim3(256), 0, ctx().stream>>>(
      static_cast<const uint16_t*>(table), static_cast<const int*>(d_token), static_cast<float*>(out),
      (int)hidden, (int)vocab);
  hipError_t e_ = hipGetLastError();
  if (e_ != hipSuccess) return hip_fail(e_, "kernel launch");
  return TLHIP_OK;
}

int tlhip_embed_rows(const void* table, int table_type, const int64_t* ids, int64_t T, void* out, int64_t hidden, int64_t vocab) {
  TLHIP_REQUIRE_READY();
  const char* who = "tlhip_embed_rows";
  if (!table || !ids || !out) return fail(TLHIP_EINVAL, "%s: null pointer", who);
  if (table_type != TLHIP_T_F16 && table_type != TLHIP_T_BF16) return fail(TLHIP_EINVAL, "%s: an f16 or bf16 table", who);
  if (T <= 0 || hidden <= 0 || vocab <= 0 || hidden > (1 << 30) || vocab > 0x7fffffff) return fail(TLHIP_EINVAL, "%s: bad shape", who);
  for (int64_t t = 0; t < T; t++)
    if (ids[t] < 0 || ids[t] >= vocab) return fail(TLHIP_EINVAL, "%s: id outside the table", who);
  const bool f16 = table_type == TLHIP_T_F16, wide = hidden % 8 == 0 && aligned16(table) && aligned16(out), few = T <= kFewIds;
  const auto go = wide ? (few ? (f16 ? launch_embed_rows<true, 8, kFewIds> : launch_embed_rows<false, 8, kFewIds>)
                              : (f16 ? launch_embed_rows<true, 8, kManyIds> : launch_embed_rows<false, 8, kManyIds>))
                       : (f16 ? launch_embed_rows<true, 1, kManyIds> : launch_embed_rows<false, 1, kManyIds>);
  go(table, ids, T, static_cast<float*>(out), hidden);
  TLHIP_CHECK_LAUNCH(TLHIP_C_EMBED);
}

}  // extern "C"
