// The argument block of the paged decode kernels (paged_decode.hip,
// paged_decode_f32.hip) and what they share.
#pragma once

#include <cmath>

#include "tsa_common.h"

namespace tsa {

struct DecodeArgs {
  void* out;
  const void* q;
  const void* kc;
  const void* vc;
  const int32_t* bt;
  const int32_t* seq_lens;
  int64_t o_ss, o_sh, o_sd;
  int64_t q_ss, q_sh, q_sd;
  int64_t kc_b, kc_h, kc_s, kc_d;
  int64_t vc_b, vc_h, vc_s, vc_d;
  int64_t bt_s0, bt_s1, sl_s;
  int64_t NB;
  int32_t B, Hq, Hkv, G, BS, max_blocks, D;
  int32_t W;        // workgroups of the stream kernel
  int32_t NW;       // wave workers sharing the tile list (kWaves * W)
  float scale_log2;
  float* part;      // [B * Hkv + NW][G * (D + 2)]: per (unit, worker) acc[G][D], m[G], l[G]
  int32_t* pref_out;  // [B + 1] tile prefix over the sequences, for the merge
  // The fused decode step only: query is the raw projection, and the new
  // token's raw k/v rows (B, Hkv, D), the norm weights (D) and the cos/sin
  // rows (B, D) come in here; eps is the RMSNorm epsilon.
  const void* kn; const void* vn; const void* qw; const void* kw; const void* cos; const void* sin;
  void* kc_out; void* vc_out;  // the caches, written (the new token's rows)
  int64_t kn_ss, kn_sh, vn_ss, vn_sh, cs_ss, sn_ss;
  float eps;
  // Splits of a unit's tiles, in the unit form (16-bit, paged_decode_unit.h; 0:
  // the stream) and in float32 (paged_decode_f32.hip; 0: the generic kernel).
  int32_t S;
};

constexpr float kNegInf = -INFINITY;

// Sequence s's length, within [0, the block table's capacity].
__device__ __forceinline__ int64_t clamp_len(const DecodeArgs& a, int s) {
  int64_t L = a.seq_lens[s * a.sl_s];
  const int64_t cap = static_cast<int64_t>(a.max_blocks) * a.BS;
  return L < 0 ? 0 : (L > cap ? cap : L);
}

// A 16-byte load, non-temporal (the streaming hint) with NT.
template <bool NT, typename T>
__device__ __forceinline__ u32x4 load_stream(const T* p) {
  if constexpr (NT) return __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p));
  else return *reinterpret_cast<const u32x4*>(p);
}

// Online log-sum-exp: (m, l, o) of more tokens into (M, L, O). A part whose
// tokens all score -inf has m = -inf and weighs 0 (a NaN in it stays one).
__device__ __forceinline__ void combine_partial(float& M, float& L, float& O, float m, float l, float o) {
  const float mn = fmaxf(M, m), mu = mn == kNegInf ? 0.f : mn;
  const float c_old = fast_exp2(M - mu), c_new = fast_exp2(m - mu);
  O = fmaf(o, c_new, O * c_old);
  L = fmaf(l, c_new, L * c_old);
  M = mn;
}

// paged_decode_f32.hip: the splits of a unit, whether it takes a float32 call
// (rows checked by the caller), and the launch. a.S splits a unit; their partials go to a.part, or
// with a.part NULL one workgroup computes a unit's splits in turn, with the
// same result.
int decode_f32_splits(int64_t units, int64_t unit_tiles, int64_t slots);
bool decode_f32_takes(const DecodeArgs& a);
int decode_f32_launch(const DecodeArgs& a, hipStream_t stream);

}  // namespace tsa
