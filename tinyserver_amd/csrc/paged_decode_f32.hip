// Paged GQA decode attention in float32.
//
// Reference: server/model/kernels/paged_attention.py:8-121.
//
// What bounds it: HBM for long contexts (each K/V byte is read once), the
// chain of memory round trips (lengths, block table, K/V, partials) for short
// ones. A unit is one (sequence, kv head); its 16-token tiles are split over S
// workgroups of four waves, each wave taking a contiguous run of tiles. S is
// the host's choice from the block tables' width. The waves' partials (m, l,
// acc) meet in LDS; with S = 1 the workgroup writes the output, with more it
// writes one partial a workgroup and a second launch merges the S of a unit.
//
// A tile is 64 matrix instructions (v_mfma_f32_16x16x4_f32, 32 cycles each),
// with the up to 16 q-heads of the kv head as columns. With lane
// (g, c) = (lane / 16, lane % 16):
//   S^T(16 tokens x 16 heads) = K Q^T: step 4 J + i takes dims 16 J + 4 g + i,
//     so K's operand is a 16-byte piece of token c's row and Q's of head c's;
//     element r of the result is the score of token 4 g + r for head c.
//   O^T(dims x 16 heads) += V^T P^T: step r takes tokens 4 g + r, whose weights
//     are element r of the lane's own scores; V's operand of dim tile
//     (half, i) is dim 64 half + 4 c + i, 16-byte pieces of token 4 g + r's
//     row. Column c is head c throughout, so the softmax's scales are the
//     lane's own.
// A wave loads the next tile's K and V before it computes one. A lane looks up
// the page of one token in every run of 64 (four tiles), one run ahead; any
// page size and any cache strides with 16-byte rows.
#include "paged_decode.h"

namespace tsa {

constexpr int kF32Waves = 4;

// Floats of one partial in LDS: acc[G][D], m[G], l[G], padded to 16 bytes. (In
// the workspace they are not padded.)
__host__ __device__ inline int f32_slot_floats(int G, int D) { return (G * (D + 2) + 3) & ~3; }

// Split sp of unit u, by the whole workgroup: the waves' partials into
// slots[wave]. (No barrier at the end.)
template <int D>
__device__ __forceinline__ void f32_split(const DecodeArgs& a, int s, int kvh, int L, int sp, float* slots) {
  constexpr int NJ = D / 16, NH = D / 64;
  const int G = a.G;
  const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t n = (L + 15) >> 4;
  const int lo_wg = static_cast<int>(n * sp / a.S), n_wg = static_cast<int>(n * (sp + 1) / a.S) - lo_wg;
  const int lo = lo_wg + n_wg * wave / kF32Waves, nt = lo_wg + n_wg * (wave + 1) / kF32Waves - lo;

  f32x4 acc[NH][4];
#pragma unroll
  for (int x = 0; x < NH; ++x)
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[x][i] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = kNegInf, l = 0.f;

  if (nt > 0) {
    const int32_t* const bt_row = a.bt + s * a.bt_s0;
    // The cache rows of the 64 tokens from tile t: lane i looks up token
    // 16 t + i. Tokens at or past L and page ids outside the pool are not
    // valid; their lanes read row 0 of page 0 and the tile masks them.
    struct Rows {
      int64_t k, v;
      uint64_t valid;
    };
    auto page_of = [&](int t) __attribute__((always_inline)) {
      const int tok = min(16 * t + lane, L - 1);
      return bt_row[(static_cast<uint32_t>(tok) / static_cast<uint32_t>(a.BS)) * a.bt_s1];
    };
    auto rows_of = [&](int t, int page) __attribute__((always_inline)) {
      const int tok = min(16 * t + lane, L - 1);
      const int slot = tok - static_cast<int>(static_cast<uint32_t>(tok) / static_cast<uint32_t>(a.BS)) * a.BS;
      const bool ok = 16 * t + lane < L && page >= 0 && page < a.NB;
      Rows r;
      r.valid = __ballot(ok);
      r.k = ok ? page * a.kc_b + slot * a.kc_s : 0;
      r.v = ok ? page * a.vc_b + slot * a.vc_s : 0;
      return r;
    };
    auto lane_i64 = [&](int64_t x, int src) __attribute__((always_inline)) {
      const int lo32 = __shfl(static_cast<int>(static_cast<uint32_t>(x)), src, 64);
      const int hi32 = __shfl(static_cast<int>(x >> 32), src, 64);
      return static_cast<int64_t>((static_cast<uint64_t>(static_cast<uint32_t>(hi32)) << 32) |
                                  static_cast<uint32_t>(lo32));
    };
    const float* const kbase = static_cast<const float*>(a.kc) + kvh * a.kc_h + 4 * g;
    const float* const vbase = static_cast<const float*>(a.vc) + kvh * a.vc_h + 4 * c;
    int page_next = page_of(lo + 4);
    Rows rows = rows_of(lo, page_of(lo));
    f32x4 q[NJ];
    {
      const float* qp = static_cast<const float*>(a.q) + s * a.q_ss + (kvh * G + min(c, G - 1)) * a.q_sh + 4 * g;
#pragma unroll
      for (int j = 0; j < NJ; ++j) q[j] = *reinterpret_cast<const f32x4*>(qp + 16 * j);
    }

    struct Tile {
      f32x4 k[NJ], v[4][NH];
      uint32_t valid;
    };
    // Tile lo + i into b (past the wave's last tile: the last one again).
    auto load = [&](Tile& b, int i) __attribute__((always_inline)) {
      if (i < nt && i > 0 && (i & 3) == 0) {  // the next four tiles' rows; their successors' pages
        rows = rows_of(lo + i, page_next);
        page_next = page_of(lo + i + 4);
      }
      const int x = 16 * (min(i, nt - 1) & 3);
      b.valid = static_cast<uint32_t>(rows.valid >> x) & 0xFFFFu;
      const float* kp = kbase + lane_i64(rows.k, x + c);
#pragma unroll
      for (int j = 0; j < NJ; ++j) b.k[j] = *reinterpret_cast<const f32x4*>(kp + 16 * j);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float* vp = vbase + lane_i64(rows.v, x + 4 * g + r);
#pragma unroll
        for (int y = 0; y < NH; ++y) b.v[r][y] = *reinterpret_cast<const f32x4*>(vp + 64 * y);
      }
      __builtin_amdgcn_sched_barrier(0);  // issued before the tile in hand is computed
    };
    auto compute = [&](Tile& b) __attribute__((always_inline)) {
      f32x4 sc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) sc = __builtin_amdgcn_mfma_f32_16x16x4f32(b.k[j][i], q[j][i], sc, 0, 0, 0);
      float sv[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) sv[r] = sc[r] * a.scale_log2;
      if (b.valid != 0xFFFFu) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (!((b.valid >> (4 * g + r)) & 1)) {  // unread rows: no weight, and no V that 0 would not cancel
            sv[r] = kNegInf;
#pragma unroll
            for (int y = 0; y < NH; ++y) b.v[r][y] = f32x4{0.f, 0.f, 0.f, 0.f};
          }
      }
      float mx = fmaxf(fmaxf(sv[0], sv[1]), fmaxf(sv[2], sv[3]));
      mx = fmaxf(mx, __builtin_bit_cast(float, xor_lane32<16>(__builtin_bit_cast(uint32_t, mx), lane)));
      mx = fmaxf(mx, __builtin_bit_cast(float, xor_lane32<32>(__builtin_bit_cast(uint32_t, mx), lane)));
      const float m_new = fmaxf(m, mx);
      const float mu = m_new == kNegInf ? 0.f : m_new;  // (-inf: every score so far is -inf, and weighs 0)
      if (__any(m_new > m)) {
        const float alpha = fast_exp2(m - mu);
        l *= alpha;
#pragma unroll
        for (int y = 0; y < NH; ++y)
#pragma unroll
          for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[y][i][e] *= alpha;
        m = m_new;
      }
      float p[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        p[r] = fast_exp2(sv[r] - mu);
        l += p[r];
      }
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int y = 0; y < NH; ++y)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            acc[y][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(b.v[r][y][i], p[r], acc[y][i], 0, 0, 0);
    };
    Tile t0, t1;
    load(t0, 0);
    for (int i = 0; i < nt; i += 2) {
      load(t1, i + 1);
      compute(t0);
      if (i + 1 < nt) {
        load(t0, i + 2);
        compute(t1);
      }
    }
    l += __builtin_bit_cast(float, xor_lane32<16>(__builtin_bit_cast(uint32_t, l), lane));
    l += __builtin_bit_cast(float, xor_lane32<32>(__builtin_bit_cast(uint32_t, l), lane));
  }
  if (c < G) {
    float* const mine = slots + wave * f32_slot_floats(G, D);
#pragma unroll
    for (int y = 0; y < NH; ++y)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        *reinterpret_cast<f32x4*>(mine + c * D + 64 * y + 4 * (4 * g + e)) =
            f32x4{acc[y][0][e], acc[y][1][e], acc[y][2][e], acc[y][3][e]};
    if (g == 0) {
      mine[G * D + c] = m;
      mine[G * D + G + c] = l;
    }
  }
}

// Grid: units (LOOP: a workgroup computes its unit's splits in turn), or units
// x S.
template <int D, bool LOOP>
__global__ __launch_bounds__(64 * kF32Waves) __attribute__((amdgpu_waves_per_eu(LOOP ? 1 : 2))) void paged_decode_f32(
    DecodeArgs a) {
  extern __shared__ __align__(16) float slots[];  // kF32Waves partials
  const int u = blockIdx.x, s = u / a.Hkv, kvh = u - s * a.Hkv, G = a.G, tid = threadIdx.x;
  const int L = static_cast<int>(clamp_len(a, s));
  const int slot = f32_slot_floats(G, D);
  constexpr int kOut = 16 * D / (64 * kF32Waves);  // outputs a thread, at most (G <= 16)
  float M[kOut], den[kOut], o[kOut];
  if constexpr (LOOP) {
#pragma unroll
    for (int k = 0; k < kOut; ++k) {
      M[k] = kNegInf;
      den[k] = o[k] = 0.f;
    }
  }
  const int sp0 = LOOP ? 0 : blockIdx.y, sp1 = LOOP ? a.S : sp0 + 1;
  for (int sp = sp0; sp < sp1; ++sp) {
    if (LOOP && sp > sp0) __syncthreads();  // the slots are read no more
    f32_split<D>(a, s, kvh, L, sp, slots);
    __syncthreads();
    // The waves in order, then (LOOP) the splits in order, as the merge
    // launch takes them.
#pragma unroll
    for (int k = 0; k < kOut; ++k) {
      const int idx = tid + 64 * kF32Waves * k;
      if (idx >= G * D) break;
      const int hd = idx / D;
      float wm = kNegInf, wl = 0.f, wo = 0.f;
#pragma unroll
      for (int w = 0; w < kF32Waves; ++w) {
        const float* sl = slots + w * slot;
        combine_partial(wm, wl, wo, sl[G * D + hd], sl[G * D + G + hd], sl[idx]);
      }
      if constexpr (LOOP) {
        combine_partial(M[k], den[k], o[k], wm, wl, wo);
      } else if (a.S == 1) {
        M[k] = kNegInf;
        den[k] = o[k] = 0.f;
        combine_partial(M[k], den[k], o[k], wm, wl, wo);
      } else {
        float* const out = a.part + (static_cast<int64_t>(u) * a.S + sp) * (G * (D + 2));
        out[idx] = wo;
        if (idx == hd * D) {
          out[G * D + hd] = wm;
          out[G * D + G + hd] = wl;
        }
      }
    }
  }
  if (LOOP || a.S == 1) {
    float* const orow = static_cast<float*>(a.out) + s * a.o_ss + kvh * G * a.o_sh;
#pragma unroll
    for (int k = 0; k < kOut; ++k) {
      const int idx = tid + 64 * kF32Waves * k;
      if (idx >= G * D) break;
      orow[(idx / D) * a.o_sh + (idx % D) * a.o_sd] = o[k] / den[k];  // no tokens: 0/0 = NaN
    }
  }
}

// A unit's S partials, in order, batches of 8 loaded together (a batch past
// the last repeats it and drops it).
template <int D>
__global__ __launch_bounds__(256) void paged_decode_f32_merge(DecodeArgs a) {
  const int u = blockIdx.x, s = u / a.Hkv, kvh = u - s * a.Hkv, G = a.G;
  const int slot = G * (D + 2);
  const float* const base = a.part + static_cast<int64_t>(u) * a.S * slot;
  float* const orow = static_cast<float*>(a.out) + s * a.o_ss + kvh * G * a.o_sh;
  for (int idx = threadIdx.x; idx < G * D; idx += 256) {
    const int hd = idx / D;
    float M = kNegInf, den = 0.f, o = 0.f;
    for (int sp = 0; sp < a.S; sp += 8) {
      float pm[8], pl[8], po[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const float* sl = base + static_cast<int64_t>(min(sp + k, a.S - 1)) * slot;
        pm[k] = sl[G * D + hd];
        pl[k] = sl[G * D + G + hd];
        po[k] = sl[idx];
      }
#pragma unroll
      for (int k = 0; k < 8; ++k)
        if (sp + k < a.S) combine_partial(M, den, o, pm[k], pl[k], po[k]);
    }
    orow[hd * a.o_sh + (idx % D) * a.o_sd] = o / den;
  }
}

// Splits of a unit whose block table holds unit_tiles tiles: two tiles a wave
// (the loads of both are in flight together, so fewer would add workgroups
// and partials without shortening the chain), as far as the workspace's
// slots go (units + 4 * workgroups).
int decode_f32_splits(int64_t units, int64_t unit_tiles, int64_t slots) {
  const int64_t want = (unit_tiles + 2 * kF32Waves - 1) / (2 * kF32Waves), room = slots / units;
  const int64_t n = want < room ? want : room;
  return static_cast<int>(n < 1 ? 1 : n);
}

bool decode_f32_takes(const DecodeArgs& a) {
  return (a.D == 64 || a.D == 128) && a.G <= 16 && a.NB > 0 && int64_t{a.B} * a.Hkv < (int64_t{1} << 31);
}

int decode_f32_launch(const DecodeArgs& a, hipStream_t stream) {
  const int units = a.B * a.Hkv;
  const size_t lds = static_cast<size_t>(kF32Waves) * f32_slot_floats(a.G, a.D) * sizeof(float);
  const bool loop = a.S > 1 && a.part == nullptr;
  const dim3 grid(units, loop ? 1 : a.S), threads(64 * kF32Waves);
  if (a.D == 128) {
    if (loop) paged_decode_f32<128, true><<<grid, threads, lds, stream>>>(a);
    else paged_decode_f32<128, false><<<grid, threads, lds, stream>>>(a);
  } else {
    if (loop) paged_decode_f32<64, true><<<grid, threads, lds, stream>>>(a);
    else paged_decode_f32<64, false><<<grid, threads, lds, stream>>>(a);
  }
  if (int rc = check_launch("tsa_paged_decode")) return rc;
  if (loop || a.S == 1) return TSA_OK;
  if (a.D == 128) paged_decode_f32_merge<128><<<dim3(units), dim3(256), 0, stream>>>(a);
  else paged_decode_f32_merge<64><<<dim3(units), dim3(256), 0, stream>>>(a);
  return check_launch("tsa_paged_decode");
}

}  // namespace tsa
