// The unit form of the 16-bit paged decode, for batches whose block tables
// are small: one workgroup of eight waves takes 32 tiles (512 tokens) of one
// (sequence, kv head) unit, all of them in one shot. Shared by tsa_paged_decode,
// the fused decode step and the mixed kernel's decode role.
//
// What bounds it: the chain of memory round trips and the instructions behind
// the last of them. So nothing is computed from the other sequences (no tile
// prefix, no cursors), the block-table entries load beside the sequence
// length, every K/V row of the workgroup's 512 tokens is in flight at once,
// and a wave scores its four tiles together: one row maximum, one
// exponential pass, no rescaling, and pairs of tiles share the 32-token form of
// the P V product. Wave w takes tiles w, w + 8, w + 16 and w + 24 of the 32.
// The waves' partials meet in LDS. A unit of more than 32 tiles is split over
// S workgroups of four waves and 16 tiles (256 tokens), which leave one partial
// each for a merge launch (decode_split_merge).
//
// Measured against the form before it (four waves a unit, one tile at a time
// through a register ring, three tiles ahead; the fused step staged its rows
// by LDS DMA and normalised them in every wave): fused step of 4 sequences of
// 16-512 tokens, 16/8 heads, 15.4 -> 9.0 us replayed from a graph; decode of 4
// x 256-512 12.1 -> 8.5. Against the stream and its merge: 32 x 64-512, 32/8
// heads, 18.8 -> 12.6; fused step of 8 x 128-4096, 16/8 heads, 26.8 -> 22.5
// (70 MB of K/V, 14 us at a large copy's rate). Splits of eight waves took
// 24.9 there: at the fused step's 173 registers (two waves a SIMD) one such
// workgroup fills a CU, where two of four waves overlap. (The plain form has 153:
// three waves a SIMD.)
//
// The fused step adds the norm and RoPE of the unit's q rows and of the new
// token's k row: 16 lanes a row, four rows a wave, in the first waves, while
// the K/V rows arrive; every wave then reads the q operand from LDS.
#pragma once

#include "norm_rope_row.h"
#include "paged_decode.h"

namespace tsa {

constexpr int kWaveTiles = 4;   // tiles of one wave
// Waves a workgroup's tiles are dealt to: eight where a unit has one
// workgroup (its tables hold at most 32 tiles), four where it is split.
constexpr int kUnitWaves = 8;
constexpr int kSplitWaves = 4;
// Units of this many splits or more (8,192 tokens) read K/V with non-temporal
// loads: batch 1 x 20,000-32,768 tokens, 32/8 heads, 33.3 -> 29.5 us, batch 8 x
// 8,192 57 -> 49. Batches of shorter ones, which the last-level cache may hold
// from one pass to the next, lose by them (batch 8 x 128-4,096: 22.7 -> 24.9).
constexpr int kNtSplits = 32;
constexpr int kUnitRowBytes = 256;  // fused: an LDS row (head_dim 128)
constexpr int kUnitFusedBytes = 9 * kUnitRowBytes;  // G <= 8 q rows and the new k row

// Sequence s's length as the unit form takes it (no pages: no tokens).
__device__ __forceinline__ int unit_len(const DecodeArgs& a, int s) {
  return a.NB > 0 ? static_cast<int>(clamp_len(a, s)) : 0;
}

// Floats of one wave's partial in LDS: acc[G][D], m[G], l[G].
__host__ __device__ inline int unit_slot_floats(int G, int D) { return (G * (D + 2) + 3) & ~3; }
__host__ __device__ inline int unit_lds_bytes(int G, int D, bool fused) {
  return (fused ? kUnitFusedBytes : 0) + kUnitWaves * unit_slot_floats(G, D) * 4;  // (enough for either)
}

// Virtual wave vw of NW, of unit u, split sp (NW * kWaveTiles tiles): its
// partial to slots[vw]. Every lane of the wave takes part; with FUSED every
// wave of the workgroup does (one barrier), and vw is the wave's own number.
// The split has a tile.
template <typename T, int D, bool PAGE16, bool CONTIG, bool FUSED, int NW, bool NT>
__device__ __forceinline__ void unit_wave(const DecodeArgs& a, const int32_t* __restrict__ bt, int s, int kvh, int sp,
                                          int L, int vw, char* fused_rows, float* slots) {
  constexpr int KJ = D / 32, kTiles = NW * kWaveTiles;
  const int G = a.G;
  const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
  const int t0 = kTiles * sp;
  const int n = (L + 15) >> 4;  // tiles of the unit
  const bool v_lane = 8 * c < D;
  const int64_t ks = CONTIG ? D : a.kc_s, vs = CONTIG ? D : a.vc_s;

  // ---- Block-table entries. 16-token multiples of a page: lane j holds the
  // split's tile j, its page and first slot. Other pages: lane j holds token
  // j % 16 of the wave's tile j / 16.
  const int my_tile = PAGE16 ? t0 + (lane & (kTiles - 1)) : t0 + vw + NW * (lane >> 4);
  const int my_tok = 16 * my_tile + (PAGE16 ? 0 : c);
  const uint32_t my_lb = static_cast<uint32_t>(my_tok) / static_cast<uint32_t>(a.BS);
  const int my_slot = my_tok - static_cast<int>(my_lb) * a.BS;
  const int my_page = bt[s * a.bt_s0 + min(static_cast<int>(my_lb), a.max_blocks - 1) * a.bt_s1];
  const bool my_ok = my_tok < L && my_page >= 0 && my_page < a.NB;
  const uint64_t ok64 = __ballot(my_ok);

  // ---- Q (plain), or the fused step's norm inputs.
  u32x4 q[KJ];
  u32x4 nx = {}, nw = {}, nc = {}, ns = {};
  const int n_row = min(4 * vw + g, G);  // fused: this lane's row, 0 .. G-1 a q head, G the new k
  const bool norm_wave = FUSED && 4 * vw <= G;
  if constexpr (FUSED) {
    if (norm_wave) {  // (uniform)
      const T* x = n_row < G ? static_cast<const T*>(a.q) + s * a.q_ss + (kvh * G + n_row) * a.q_sh
                             : static_cast<const T*>(a.kn) + s * a.kn_ss + kvh * a.kn_sh;
      const T* w = static_cast<const T*>(n_row < G ? a.qw : a.kw);
      nx = *reinterpret_cast<const u32x4*>(x + 8 * c);
      nw = *reinterpret_cast<const u32x4*>(w + 8 * c);
      nc = *reinterpret_cast<const u32x4*>(static_cast<const T*>(a.cos) + s * a.cs_ss + 8 * c);
      ns = *reinterpret_cast<const u32x4*>(static_cast<const T*>(a.sin) + s * a.sn_ss + 8 * c);
    }
  } else {
    const T* qrow = static_cast<const T*>(a.q) + s * a.q_ss + (kvh * G + c % G) * a.q_sh + 8 * g;
#pragma unroll
    for (int j = 0; j < KJ; ++j) q[j] = *reinterpret_cast<const u32x4*>(qrow + 32 * j);
  }

  // ---- K operands (lane (g, c): token c, dims 8 (g + 4 j)..+8) and V rows
  // (tokens 4 g .. 4 g + 3, dims 8 c..+8) of the wave's tiles. Rows that are
  // not valid read row 0 of page 0 and are masked; tiles past the unit's end
  // are not read.
  u32x4 ko[kWaveTiles][KJ], vo[kWaveTiles][4];
  uint32_t valid[kWaveTiles];  // bit i: token i of the tile
  const T* const kbase = static_cast<const T*>(a.kc) + kvh * a.kc_h + 8 * g;
  const T* const vbase = static_cast<const T*>(a.vc) + kvh * a.vc_h + (v_lane ? 8 * c : 0);
  auto lane_i64 = [&](int64_t x, int src) {
    const int lo = __shfl(static_cast<int>(static_cast<uint32_t>(x)), src, 64);
    const int hi = __shfl(static_cast<int>(x >> 32), src, 64);
    return static_cast<int64_t>((static_cast<uint64_t>(static_cast<uint32_t>(hi)) << 32) | static_cast<uint32_t>(lo));
  };
  const int64_t my_k = !PAGE16 && my_ok ? my_page * a.kc_b + my_slot * ks : 0;
  const int64_t my_v = !PAGE16 && my_ok ? my_page * a.vc_b + my_slot * vs : 0;
#pragma unroll
  for (int x = 0; x < kWaveTiles; ++x) {
    const int j = vw + NW * x, tile = t0 + j;
    valid[x] = 0;
    if (tile < n) {  // (uniform)
      const T *kp, *vp[4];
      if constexpr (PAGE16) {
        const bool ok = (ok64 >> j) & 1;
        const int64_t page = ok ? __builtin_amdgcn_readlane(my_page, j) : 0;
        const int slot0 = ok ? __builtin_amdgcn_readlane(my_slot, j) : 0;
        const int left = L - 16 * tile;
        valid[x] = !ok ? 0u : left >= 16 ? 0xFFFFu : (1u << left) - 1u;
        kp = kbase + page * a.kc_b + (slot0 + c) * ks;
        vp[0] = vbase + page * a.vc_b + (slot0 + 4 * g) * vs;
#pragma unroll
        for (int r = 1; r < 4; ++r) vp[r] = vp[0] + r * vs;
      } else {
        valid[x] = static_cast<uint32_t>(ok64 >> (16 * x)) & 0xFFFFu;
        kp = kbase + lane_i64(my_k, 16 * x + c);
#pragma unroll
        for (int r = 0; r < 4; ++r) vp[r] = vbase + lane_i64(my_v, 16 * x + 4 * g + r);
      }
#pragma unroll
      for (int i = 0; i < KJ; ++i) ko[x][i] = load_stream<NT>(kp + 32 * i);
#pragma unroll
      for (int r = 0; r < 4; ++r) vo[x][r] = load_stream<NT>(vp[r]);
    } else {
#pragma unroll
      for (int i = 0; i < KJ; ++i) ko[x][i] = u32x4{0, 0, 0, 0};
#pragma unroll
      for (int r = 0; r < 4; ++r) vo[x][r] = u32x4{0, 0, 0, 0};
    }
  }

  if constexpr (FUSED) {
    // The new token, position L - 1: this wave's tile xn, token cn, if the
    // wave has it. Its raw V row replaces the cache's here and is stored.
    const int tn = (L - 1) >> 4, cn = (L - 1) & 15, jn = tn - t0;
    const bool mine = jn >= 0 && jn < kTiles && jn % NW == vw;
    const int xn = jn / NW;
    const bool in_split = jn >= 0 && jn < kTiles;
    const bool stored = in_split && ((ok64 >> (in_split ? jn : 0)) & 1);  // (a page outside the pool is not written)
    const int64_t page = stored ? __builtin_amdgcn_readlane(my_page, in_split ? jn : 0) : 0;
    const int64_t slot = (stored ? __builtin_amdgcn_readlane(my_slot, in_split ? jn : 0) : 0) + cn;
    u32x4 vnew = {};
    if (mine)
      vnew = *reinterpret_cast<const u32x4*>(static_cast<const T*>(a.vn) + s * a.vn_ss + kvh * a.vn_sh + 8 * c);
    __builtin_amdgcn_sched_barrier(0);
    if (norm_wave) {  // (uniform) four rows' norm and RoPE, as the norm/RoPE kernels compute them
      float x[8], w[8], cs[8], sn[8], o[8];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        x[2 * i] = lo_f<T>(nx[i]); x[2 * i + 1] = hi_f<T>(nx[i]);
        w[2 * i] = lo_f<T>(nw[i]); w[2 * i + 1] = hi_f<T>(nw[i]);
        cs[2 * i] = lo_f<T>(nc[i]); cs[2 * i + 1] = hi_f<T>(nc[i]);
        sn[2 * i] = lo_f<T>(ns[i]); sn[2 * i + 1] = hi_f<T>(ns[i]);
      }
      norm_rope_row<T, 128>(x, w, cs, sn, a.eps, c, o);
      const u32x4 row = u32x4{pack2<T>(o[0], o[1]), pack2<T>(o[2], o[3]), pack2<T>(o[4], o[5]), pack2<T>(o[6], o[7])};
      if (4 * vw + g <= G) {
        *reinterpret_cast<u32x4*>(fused_rows + kUnitRowBytes * n_row + 16 * c) = row;
        if (n_row == G && stored)
          *reinterpret_cast<u32x4*>(static_cast<T*>(a.kc_out) + kvh * a.kc_h + page * a.kc_b + slot * ks + 8 * c) = row;
      }
    }
    lds_barrier();
#pragma unroll
    for (int j = 0; j < KJ; ++j)
      q[j] = *reinterpret_cast<const u32x4*>(fused_rows + kUnitRowBytes * (c % G) + 16 * (g + 4 * j));
    if (mine) {  // (uniform)
#pragma unroll
      for (int x = 0; x < kWaveTiles; ++x) {
        if (x != xn) continue;
#pragma unroll
        for (int j = 0; j < KJ; ++j) {
          const u32x4 kn = *reinterpret_cast<const u32x4*>(fused_rows + kUnitRowBytes * G + 16 * (g + 4 * j));
          if (c == cn) ko[x][j] = kn;
        }
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (4 * g + r == cn) vo[x][r] = vnew;
      }
      if (stored && g == 0)
        *reinterpret_cast<u32x4*>(static_cast<T*>(a.vc_out) + kvh * a.vc_h + page * a.vc_b + slot * vs + 8 * c) = vnew;
    }
  }
  if (t0 + vw >= n) return;  // (uniform) no tiles

  // ---- Scores: element r of sc[x] is token 4 g + r of the tile, head c.
  float sv[kWaveTiles][4], m = kNegInf;
#pragma unroll
  for (int x = 0; x < kWaveTiles; ++x) {
    f32x4 sc = f32x4{0.f, 0.f, 0.f, 0.f};
    if (t0 + vw + NW * x < n) {  // (uniform)
#pragma unroll
      for (int j = 0; j < KJ; ++j) sc = mfma_k32<T>(ko[x][j], q[j], sc);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) sv[x][r] = sc[r] * a.scale_log2;
    if (valid[x] != 0xFFFFu) {  // (uniform) unread tokens: no weight, and no V that 0 would not cancel
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (!((valid[x] >> (4 * g + r)) & 1)) {
          sv[x][r] = kNegInf;
          vo[x][r] = u32x4{0, 0, 0, 0};
        }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) m = fmaxf(m, sv[x][r]);
  }
  m = fmaxf(m, __builtin_bit_cast(float, xor_lane32<16>(__builtin_bit_cast(uint32_t, m), lane)));
  m = fmaxf(m, __builtin_bit_cast(float, xor_lane32<32>(__builtin_bit_cast(uint32_t, m), lane)));
  const float mu = m == kNegInf ? 0.f : m;  // (-inf: every score is -inf, and weighs 0)
  float l = 0.f;
  // P as two cache-dtype halves, hi + lo (the reference's P V is fp32): 16
  // (bf16) or 22 (f16) significant bits; l sums the fp32 p.
  u32x2 phi[kWaveTiles], plo[kWaveTiles];
#pragma unroll
  for (int x = 0; x < kWaveTiles; ++x) {
    float p[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      p[r] = fast_exp2(sv[x][r] - mu);
      l += p[r];
    }
    phi[x] = u32x2{pack2<T>(p[0], p[1]), pack2<T>(p[2], p[3])};
    plo[x] = u32x2{pack2<T>(p[0] - lo_f<T>(phi[x][0]), p[1] - hi_f<T>(phi[x][0])),
                   pack2<T>(p[2] - lo_f<T>(phi[x][1]), p[3] - hi_f<T>(phi[x][1]))};
  }
  // ---- O(heads x dims) += P V, a pair of tiles at a time: reduction slots
  // 8 g .. 8 g + 3 are the first tile's tokens 4 g .. 4 g + 3, the next four
  // the second's. acc[u][r] = O[head 4 g + r][dim 8 c + u].
  f32x4 acc[8];
#pragma unroll
  for (int u = 0; u < 8; ++u) acc[u] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int x = 0; x < kWaveTiles; x += 2) {
    if (t0 + vw + NW * x >= n) continue;  // (uniform)
    const u32x4 hi4 = u32x4{phi[x][0], phi[x][1], phi[x + 1][0], phi[x + 1][1]};
    const u32x4 lo4 = u32x4{plo[x][0], plo[x][1], plo[x + 1][0], plo[x + 1][1]};
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int w = u >> 1;
      u32x4 b;
#pragma unroll
      for (int y = 0; y < 2; ++y)
#pragma unroll
        for (int h = 0; h < 2; ++h)
          b[2 * y + h] = (u & 1) ? pack_hi(vo[x + y][2 * h][w], vo[x + y][2 * h + 1][w])
                                 : pack_lo(vo[x + y][2 * h][w], vo[x + y][2 * h + 1][w]);
      acc[u] = mfma_k32<T>(hi4, b, acc[u]);
      acc[u] = mfma_k32<T>(lo4, b, acc[u]);
    }
  }
  l += __builtin_bit_cast(float, xor_lane32<16>(__builtin_bit_cast(uint32_t, l), lane));
  l += __builtin_bit_cast(float, xor_lane32<32>(__builtin_bit_cast(uint32_t, l), lane));
  float* const slot = slots + vw * unit_slot_floats(G, D);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int hd = 4 * g + r;
    if (hd < G && v_lane) {
      float* const dst = slot + hd * D + 8 * c;
      *reinterpret_cast<f32x4*>(dst) = f32x4{acc[0][r], acc[1][r], acc[2][r], acc[3][r]};
      *reinterpret_cast<f32x4*>(dst + 4) = f32x4{acc[4][r], acc[5][r], acc[6][r], acc[7][r]};
    }
  }
  if (g == 0 && c < G) {
    slot[G * D + c] = m;
    slot[G * D + G + c] = l;
  }
}

// Unit u, split sp of NW virtual waves, by a workgroup of WAVES waves (NW, or
// fewer that take the virtual waves in turn: the same partials in the same
// slots, so the same result bit for bit).
template <typename T, int D, bool PAGE16, bool CONTIG, bool FUSED, int NW, int WAVES, bool NT = false>
__device__ __forceinline__ void decode_unit_body(const DecodeArgs& a, const int32_t* __restrict__ bt,
                                                 const int32_t* __restrict__ sl, float* __restrict__ part, int u,
                                                 int sp, char* lds) {
  static_assert(!FUSED || WAVES == NW, "the fused step takes a wave per virtual wave");
  static_assert(!FUSED || 4 * NW > 8, "the fused step's waves cover G <= 8 q rows and the k row, four rows each");
  constexpr int kTiles = NW * kWaveTiles;
  const int G = a.G, tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int s = u / a.Hkv, kvh = u - s * a.Hkv;
  DecodeArgs b = a;  // (seq_lens through the __restrict__ pointer: a scalar load)
  b.seq_lens = sl;
  const int L = __builtin_amdgcn_readfirstlane(unit_len(b, s));
  const int nt = min(max(((L + 15) >> 4) - kTiles * sp, 0), kTiles);  // the split's tiles
  if (nt == 0 && a.S > 1) return;  // (the merge takes the splits that have tiles)
  char* const rows = lds;
  float* const slots = reinterpret_cast<float*>(lds + (FUSED ? kUnitFusedBytes : 0));
  if (nt > 0) {
    for (int vw = wave; vw < NW; vw += WAVES)
      unit_wave<T, D, PAGE16, CONTIG, FUSED, NW, NT>(a, bt, s, kvh, sp, L, vw, rows, slots);
  }
  lds_barrier();
  const int nw = min(nt, NW), slot = unit_slot_floats(G, D);
  for (int idx = tid; idx < G * D; idx += 64 * WAVES) {
    const int hd = idx / D;
    float M = kNegInf, den = 0.f, o = 0.f;
    for (int w = 0; w < nw; ++w) {
      const float* const x = slots + w * slot;
      combine_partial(M, den, o, x[G * D + hd], x[G * D + G + hd], x[idx]);
    }
    if (a.S == 1) {  // no tokens: 0/0 = NaN, as the reference's
      static_cast<T*>(a.out)[s * a.o_ss + (kvh * G + hd) * a.o_sh + (idx - hd * D) * a.o_sd] = from_float<T>(o / den);
    } else {
      float* const out = part + (static_cast<int64_t>(u) * a.S + sp) * (G * (D + 2));
      out[idx] = o;
      if (idx == hd * D) {
        out[G * D + hd] = M;
        out[G * D + G + hd] = den;
      }
    }
  }
}

// Unit u's output from the partials of its splits that have tiles: 64
// outputs a workgroup, each wave a quarter of the splits in batches whose
// loads are issued together (past the last: repeated and dropped), then the
// four quarters in order.
template <typename T>
__global__ __launch_bounds__(256) void decode_split_merge(DecodeArgs a) {
  constexpr int kTokens = 16 * kSplitWaves * kWaveTiles;
  __shared__ float part[4][3][64];
  const int u = blockIdx.x, s = u / a.Hkv, kvh = u - s * a.Hkv, G = a.G, D = a.D;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int L = unit_len(a, s);
  const int n = (L + kTokens - 1) / kTokens, per = (n + 3) / 4;
  const int first = min(n, wave * per), last = min(n, first + per);
  const int64_t slot = static_cast<int64_t>(G) * (D + 2);
  const float* const base = a.part + static_cast<int64_t>(u) * a.S * slot;
  const int idx = min(64 * static_cast<int>(blockIdx.y) + lane, G * D - 1), hd = idx / D;
  float M = kNegInf, den = 0.f, o = 0.f;
  for (int sp = first; sp < last; sp += 8) {
    float pm[8], pl[8], po[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const float* const x = base + min(sp + k, last - 1) * slot;
      pm[k] = x[G * D + hd];
      pl[k] = x[G * D + G + hd];
      po[k] = x[idx];
    }
#pragma unroll
    for (int k = 0; k < 8; ++k)
      if (sp + k < last) combine_partial(M, den, o, pm[k], pl[k], po[k]);
  }
  part[wave][0][lane] = M;
  part[wave][1][lane] = den;
  part[wave][2][lane] = o;
  __syncthreads();
  if (wave > 0 || 64 * static_cast<int>(blockIdx.y) + lane >= G * D) return;
#pragma unroll
  for (int w = 1; w < 4; ++w) combine_partial(M, den, o, part[w][0][lane], part[w][1][lane], part[w][2][lane]);
  static_cast<T*>(a.out)[s * a.o_ss + (kvh * G + hd) * a.o_sh + (idx - hd * D) * a.o_sd] = from_float<T>(o / den);
}

}  // namespace tsa
