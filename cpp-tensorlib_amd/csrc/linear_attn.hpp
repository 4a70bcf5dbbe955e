// Gated linear attention: what the decode step (hybrid_step.hip) and the prompt-chunk kernels
// (linear_attn.hip) share, and the decode step's block.
//
//   state row c <- a_c row_c + k_c v,   o = sum_c q_c row_c,   ln a_c = -softplus(-z_c) / tau
//
// Everything is f32. Decays are kept as base-2 logarithms.
#pragma once

#include "attn_window.hpp"

namespace tlhip {

// log2 of the decay, -log2(1 + e^-z) / tau, from e = e^-|z| <= 1. log2(1 + e) keeps e's
// relative accuracy down to the smallest e: with w = fl(1 + e), log2(w) e / (w - 1) undoes w's rounding.
__device__ __forceinline__ float log2_decay(float z, float inv_tau) {
  const float e = exp2_native(-fabsf(z) * kLog2e), w = 1.f + e;
  const float l = w == 1.f ? e * kLog2e : log2_native(w) * (e * __builtin_amdgcn_rcpf(w - 1.f));
  return -(fmaxf(-z, 0.f) * kLog2e + l) * inv_tau;
}
// z of channel `ch` (head * dim + d): the low-rank product and its bias
__device__ __forceinline__ float decay_logit(const tlhip_linear_attn& a, const float* __restrict__ low, int ch) {
  const uint16_t* w = static_cast<const uint16_t*>(a.a2) + (size_t)ch * a.rank;
  const int rank = (int)a.rank;
  const float bias = static_cast<const float*>(a.bias)[ch];
  float z = 0.f;
  for (int r0 = 0; r0 < rank; r0 += 16) {          // sixteen at once, not in turn
    uint16_t x[16];
    float l[16];
#pragma unroll
    for (int r = 0; r < 16; r++) x[r] = w[min(r0 + r, rank - 1)], l[r] = low[min(r0 + r, rank - 1)];
#pragma unroll
    for (int r = 0; r < 16; r++)
      if (r0 + r < rank) z = fmaf(__uint_as_float((uint32_t)x[r] << 16), l[r], z);
  }
  return z + bias;
}
__host__ __device__ inline int64_t linear_state_ld(int64_t vdim) { return (vdim + 3) & ~(int64_t)3; }

// Decode step of head h, one block of 512 threads. The state is read from the slot of `pos` and
// written to the other one; a thread owns one float4 column of every ng-th row. (Both slots of a thread's first rows, asked for ahead of a
// position that may be on the device, were more traffic than they saved: the mixers of 7, 16 and 28 heads of 64 x 128 in a turn's trace 5.06,
// 5.14 and 5.12 us, so 4.65, 5.05 and 4.98.)
__device__ __forceinline__ void linear_step_block(const tlhip_linear_attn& a, const float* __restrict__ u,
                                                  float* __restrict__ y, int pos, int h, float* smem) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int dim = (int)a.dim, vdim = (int)a.vdim, ld = (int)linear_state_ld(vdim), nv4 = ld >> 2;
  const int ng = small_div(512, nv4), dg = small_div(tid, nv4), v4 = tid - dg * nv4;
  const bool live = dg < ng;
  float* qs = smem;               // [dim]
  float* ks = qs + dim;
  float* al = ks + dim;
  float* vs = al + dim;           // [ld]
  float* red = vs + ld + ((4 - (3 * dim + ld) % 4) & 3);   // [ng][ld], 16-byte aligned
  float* sums = red + 2048;       // [8]
  const size_t slot = (size_t)a.heads * dim * ld;
  const float* src = static_cast<const float*>(a.state) + (size_t)(pos & 1) * slot + (size_t)h * dim * ld;
  float* dst = static_cast<float*>(a.state) + (size_t)((pos + 1) & 1) * slot + (size_t)h * dim * ld;
  constexpr int PRE = 4;          // rows of this thread requested up front
  float4 st[PRE];
#pragma unroll
  for (int i = 0; i < PRE; i++) st[i] = *reinterpret_cast<const float4*>(src + (size_t)min(dg + i * ng, dim - 1) * ld + 4 * v4);
  const int64_t ch0 = (int64_t)h * vdim + min(tid, vdim - 1);
  const float gate0 = u[a.gate_off + ch0], norm0 = static_cast<const float*>(a.norm)[min(tid, vdim - 1)];   // of what this thread writes first
  for (int d = tid; d < dim; d += 512) {
    const int ch = h * dim + d;
    const float q = u[a.q_off + ch], k = u[a.k_off + ch];
    al[d] = exp2_native(log2_decay(decay_logit(a, u + a.low_off, ch), 1.0f / a.tau));
    qs[d] = q * a.q_scale;
    ks[d] = k;
  }
  for (int v = tid; v < ld; v += 512) vs[v] = v < vdim ? u[a.v_off + (int64_t)h * vdim + v] : 0.f;
  __syncthreads();
  float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
  if (live) {
    const float v0 = vs[4 * v4], v1 = vs[4 * v4 + 1], v2 = vs[4 * v4 + 2], v3 = vs[4 * v4 + 3];
    const auto row = [&](int d, float4 s) {
      const float w = al[d], k = ks[d], q = qs[d];
      s.x = fmaf(w, s.x, k * v0); s.y = fmaf(w, s.y, k * v1); s.z = fmaf(w, s.z, k * v2); s.w = fmaf(w, s.w, k * v3);
      *reinterpret_cast<float4*>(dst + (size_t)d * ld + 4 * v4) = s;
      o.x = fmaf(q, s.x, o.x); o.y = fmaf(q, s.y, o.y); o.z = fmaf(q, s.z, o.z); o.w = fmaf(q, s.w, o.w);
    };
#pragma unroll
    for (int i = 0; i < PRE; i++)
      if (dg + i * ng < dim) row(dg + i * ng, pos > 0 ? st[i] : make_float4(0.f, 0.f, 0.f, 0.f));
    for (int d = dg + PRE * ng; d < dim; d += ng)
      row(d, pos > 0 ? *reinterpret_cast<const float4*>(src + (size_t)d * ld + 4 * v4) : make_float4(0.f, 0.f, 0.f, 0.f));
    *reinterpret_cast<float4*>(red + dg * ld + 4 * v4) = o;
  }
  __syncthreads();
  // o[v] summed over the row groups, its mean square over vdim, norm and gate
  float ss = 0.f;
  for (int v = tid; v < vdim; v += 512) {
    float t = 0.f;
    for (int g0 = 0; g0 < ng; g0 += 8) {           // (eight LDS reads at once)
      float x[8];
#pragma unroll
      for (int g = 0; g < 8; g++) x[g] = red[min(g0 + g, ng - 1) * ld + v];
#pragma unroll
      for (int g = 0; g < 8; g++)
        if (g0 + g < ng) t += x[g];
    }
    vs[v] = t;
    ss = fmaf(t, t, ss);
  }
  ss = wave_sum(ss);
  if (lane == 0) sums[wave] = ss;
  __syncthreads();
  float tot = 0.f;
#pragma unroll
  for (int w = 0; w < 8; w++) tot += sums[w];
  const float inv = 1.0f / sqrtf(tot / (float)vdim + a.eps);
  for (int v = tid; v < vdim; v += 512) {
    const int64_t ch = (int64_t)h * vdim + v;
    const float g = v == tid ? gate0 : u[a.gate_off + ch], nv = v == tid ? norm0 : static_cast<const float*>(a.norm)[v];
    y[a.y_off + ch] = vs[v] * inv * nv * (g * sigmoid_f(g)) * a.out_scale;
  }
}

__host__ __device__ inline size_t linear_step_lds(int64_t dim, int64_t vdim) {
  return (size_t)(3 * dim + linear_state_ld(vdim) + 4 + 2048 + 8) * sizeof(float);
}

int check_linear_attn(const tlhip_linear_attn* a, const char* who);
}  // namespace tlhip
