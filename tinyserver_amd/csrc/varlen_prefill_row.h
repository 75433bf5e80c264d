// One query row of one q-head by one wave, in fp32 on the vector units: any
// strides, head_dim up to 512.
#pragma once

#include "tsa_common.h"
#include "varlen_prefill_gqa.h"

namespace tsa {

// Row qi of q/out (query qq of its sequence), q-head h, over the sequence's
// keys [k_start, k_start + k_len). Every lane of the wave takes part.
template <typename T>
__device__ void prefill_row(const PrefillArgs& a, int64_t qi, int64_t qq, int h, int64_t k_start, int64_t k_len) {
  const int lane = threadIdx.x & 63;
  const int kvh = h / a.G, D = a.D;
  const T* qrow = static_cast<const T*>(a.q) + qi * a.q_st + h * a.q_sh;
  const T* kb = static_cast<const T*>(a.k) + k_start * a.k_st + kvh * a.k_sh;
  const T* vb = static_cast<const T*>(a.v) + k_start * a.v_st + kvh * a.v_sh;
  const int64_t kend = a.causal ? (k_len < qq + 1 ? k_len : qq + 1) : k_len;
  constexpr int kMaxPerLane = 8;
  float acc[kMaxPerLane];
#pragma unroll
  for (int i = 0; i < kMaxPerLane; ++i) acc[i] = 0.f;
  float m = kNegInfP, l = 0.f;
  for (int64_t base = 0; base < kend; base += 64) {
    const int64_t key = base + lane;
    float sc = kNegInfP;
    if (key < kend) {
      float dot = 0.f;
      for (int d = 0; d < D; ++d) dot += to_float(qrow[d * a.q_sd]) * to_float(kb[key * a.k_st + d * a.k_sd]);
      sc = dot * a.scale_log2;
    }
    float cmax = sc;
    for (int off = 32; off >= 1; off >>= 1) cmax = fmaxf(cmax, __shfl_xor(cmax, off, 64));
    const float m_new = fmaxf(m, cmax);
    const float alpha = fast_exp2(m - m_new);
    const float p = fast_exp2(sc - m_new);
    const float pr = to_float(from_float<T>(p));  // P.V in the V dtype, as the reference does
    float psum = p;
    for (int off = 32; off >= 1; off >>= 1) psum += __shfl_xor(psum, off, 64);
    l = l * alpha + psum;
#pragma unroll
    for (int i = 0; i < kMaxPerLane; ++i) acc[i] *= alpha;
    const int n = static_cast<int>(kend - base < 64 ? kend - base : 64);
    for (int j = 0; j < n; ++j) {
      const float pj = __shfl(pr, j, 64);
      const T* vr = vb + (base + j) * a.v_st;
#pragma unroll
      for (int i = 0; i < kMaxPerLane; ++i) {
        const int d = lane + 64 * i;
        if (d < D) acc[i] += pj * to_float(vr[d * a.v_sd]);
      }
    }
    m = m_new;
  }
  T* orow = static_cast<T*>(a.out) + qi * a.o_st + h * a.o_sh;
#pragma unroll
  for (int i = 0; i < kMaxPerLane; ++i) {
    const int d = lane + 64 * i;
    if (d < D) orow[d * a.o_sd] = from_float<T>(acc[i] / l);
  }
}

}  // namespace tsa
