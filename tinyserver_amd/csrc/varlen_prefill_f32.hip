// Varlen causal prefill in float32 on the f32 matrix instructions.
//
// Reference: server/model/kernels/varlen_attention.py:8-142.
//
// What bounds it: v_mfma_f32_16x16x4_f32, 32 cycles for 2,048 FLOP a SIMD (a
// large float32 matrix product reaches 133 TFLOP/s on this card; one
// 8192-token sequence of 16/8 heads, 275 GFLOP, runs at 121 here). Small
// batches are bound by the items' serial parts -- the search, the first loads
// and the merge, about 7 us a workgroup, of which two share a CU: 8 prompts of
// 32-512 tokens, 3.5 GFLOP, take 55.5 us where the products alone need 26
// (57.9 with the sequence's ranges read after the search and K after Q; the
// one-wave-per-row kernel took 3,355).
//
// Work item: 32 rows of one (sequence, kv head), a row being one (query,
// q-head of the kv head's group), query-major, so one K/V read serves the
// whole GQA group and a tile spans only 32 / G queries of the causal diagonal.
// One 4-wave workgroup takes an item and deals its 16-key blocks to the waves
// in turn: short items then finish in a quarter of the time one wave would
// take, which is what fills 1,024 SIMDs from a few thousand tokens. The waves'
// partials (m, l, O^T) meet in LDS once per item. Two workgroups share a CU
// (at most 256 registers a wave). K and V come from global memory (the L2
// after the first touch) straight into registers: V is in flight under the
// score products, the next block's K under the softmax and P V. Blocks of 32
// keys on the 32x32x2 form took 68 us for that batch (coarser blocks to deal,
// more masked work); workgroups that stay and walk a precomputed item plan
// took 59 against 58, and 2,430 against 2,264 for the long sequence.
//
// Layouts. With lane (g, c) = (lane / 16, lane % 16) and row tiles t = 0, 1:
//   S^T(16 keys x 16 rows) = K Q^T: step 4 j + i takes dims 16 j + 4 g + i, so
//     a lane's K and Q operands are 16-byte pieces of key c's and row c's
//     vectors; element r of the accumulator is the score of key 4 g + r.
//   O^T(dims x 16 rows) += V^T P^T: step r takes keys 4 g + r, whose weights are
//     element r of the lane's own scores: P never leaves its registers. Dim
//     tile (y, i) has dim 64 y + 4 c + i in its row c, so a lane's V operands
//     are 16-byte pieces of a key's row. A lane holds row c's outputs, so the
//     softmax's scales are the lane's own.
#include <cmath>

#include "tsa_common.h"
#include "varlen_prefill_gqa.h"
#include "varlen_prefill_row.h"

namespace tsa {

constexpr int kF32Rows = 32;     // rows of an item
constexpr int kF32Threads = 256;

// Tiles of 32 (query, head-of-group) rows of sequence b.
__device__ __forceinline__ int f32_tiles(const PrefillArgs& a, int b) {
  int64_t s, n;
  seq_range(a.cu_q, a.cuq_s, b, a.total_q, s, n);
  return static_cast<int>((n * a.G + kF32Rows - 1) / kF32Rows);
}

__device__ __forceinline__ int wave_sum(int x) {
  return __builtin_amdgcn_readlane(static_cast<int>(wave_scan_u32(static_cast<uint32_t>(x))), 63);
}

// Item j (of the launch's tiles, all kv heads together) -> its tile t and its
// sequence's query and key ranges.
// Up to 64 sequences: latest (heaviest) tiles first over all sequences, by a
// binary search on the level (the number of tiles at or above a level, summed
// over the wave's lanes). More sequences: sequence by sequence, latest tile
// first. Returns false past the last item. Wave-uniform.
__device__ __forceinline__ bool f32_item(const PrefillArgs& a, int j, int& t, int64_t& q_start, int64_t& q_len,
                                         int64_t& k_start, int64_t& k_len) {
  const int lane = threadIdx.x & 63;
  int b;
  if (a.nseq <= 64) {
    // (lane b holds sequence b's ranges: one round trip for all that is read)
    int64_t qs, ql, ks, kl;
    const int mine = min(lane, a.nseq - 1);
    seq_range(a.cu_q, a.cuq_s, mine, a.total_q, qs, ql);
    seq_range(a.cu_k, a.cuk_s, mine, a.total_k, ks, kl);
    const int nt = lane < a.nseq ? static_cast<int>((ql * a.G + kF32Rows - 1) / kF32Rows) : 0;
    int mx = nt;
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) mx = max(mx, __shfl_xor(mx, o, 64));
    mx = __builtin_amdgcn_readfirstlane(mx);
    if (j >= wave_sum(nt)) return false;
    int lo = 0, hi = mx - 1;  // the largest level Q with (tiles above or at Q) > j
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (wave_sum(max(0, nt - mid)) > j) lo = mid; else hi = mid - 1;
    }
    int rank = j - wave_sum(max(0, nt - lo - 1));
    uint64_t mask = __ballot(nt > lo);
    while (rank-- > 0) mask &= mask - 1;
    b = __builtin_ctzll(mask);
    t = lo;
    // (starts and lengths fit 31 bits: the host takes calls of fewer rows)
    q_start = __builtin_amdgcn_readlane(static_cast<int>(qs), b);
    q_len = __builtin_amdgcn_readlane(static_cast<int>(ql), b);
    k_start = __builtin_amdgcn_readlane(static_cast<int>(ks), b);
    k_len = __builtin_amdgcn_readlane(static_cast<int>(kl), b);
    return true;
  }
  const int per = (a.nseq + 63) / 64, b0 = min(a.nseq, lane * per), b1 = min(a.nseq, b0 + per);
  int mine = 0;
  for (int i = b0; i < b1; ++i) mine += f32_tiles(a, i);
  const int incl = static_cast<int>(wave_scan_u32(static_cast<uint32_t>(mine)));
  const uint64_t past = __ballot(incl > j);
  if (past == 0) return false;
  const int src = __builtin_ctzll(past);
  int run = __builtin_amdgcn_readlane(incl - mine, src);
  b = src * per;
  int nt = f32_tiles(a, b);
  while (run + nt <= j) {
    run += nt;
    nt = f32_tiles(a, ++b);
  }
  b = __builtin_amdgcn_readfirstlane(b);
  t = __builtin_amdgcn_readfirstlane(nt - 1 - (j - run));
  seq_range(a.cu_q, a.cuq_s, b, a.total_q, q_start, q_len);
  seq_range(a.cu_k, a.cuk_s, b, a.total_k, k_start, k_len);
  return true;
}

template <int D>
constexpr int f32_row_floats() { return D + 4; }  // LDS row pitch: 16-byte aligned, rows 4 banks apart
// LDS: three waves' partials (Q's rows sit in the first until the merge) and
// all four waves' m and l.
template <int D>
constexpr int f32_smem_floats() { return 3 * kF32Rows * f32_row_floats<D>() + 2 * 4 * kF32Rows; }

template <int D>
__global__ __launch_bounds__(kF32Threads) __attribute__((amdgpu_waves_per_eu(2, 2))) void varlen_prefill_f32(
    PrefillArgs a) {
  constexpr int NJ = D / 16;  // 16-byte pieces of a lane's K or Q operand
  constexpr int NH = D / 64;  // 16-byte pieces of a lane's V operand of one key
  constexpr int RP = f32_row_floats<D>();
  __shared__ __align__(16) float smem[f32_smem_floats<D>()];
  float* const ml = smem + 3 * kF32Rows * RP;  // m[4][32], l[4][32]

  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, c = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kvh = static_cast<int>(blockIdx.x) % a.Hkv;
  int tile;
  int64_t q_start, q_len, k_start, k_len;
  if (!f32_item(a, static_cast<int>(blockIdx.x) / a.Hkv, tile, q_start, q_len, k_start, k_len)) return;
  const int G = a.G;
  // (32-bit rows: the host takes calls of fewer than 2^31 rows)
  const uint32_t row0 = static_cast<uint32_t>(tile) * kF32Rows, n_rows = static_cast<uint32_t>(q_len) * G;
  const int rows = static_cast<int>(min(n_rows - row0, static_cast<uint32_t>(kF32Rows)));
  // Row r of the item: query (row0 + r) / G, q-head kvh G + (row0 + r) % G.
  auto q_of = [&](int r) { return static_cast<int>((row0 + r) / static_cast<uint32_t>(G)); };
  auto head_of = [&](int r, int qq) { return kvh * G + static_cast<int>(row0 + r - static_cast<uint32_t>(qq) * G); };
  const int q_first = q_of(0), q_last = q_of(rows - 1);
  const int kl = static_cast<int>(k_len);
  const int kend = a.causal ? min(kl, q_last + 1) : kl;
  const int nblk = (kend + 15) / 16;
  const int full = a.causal ? min(kl, q_first + 1) : kl;  // keys below it are seen by every row

  // The item's Q rows (rows past the last repeat it), then the first K block,
  // all in flight before Q goes to LDS.
  constexpr int kQ = kF32Rows * (D / 4) / kF32Threads;  // 16-byte pieces a thread
  f32x4 qv[kQ];
#pragma unroll
  for (int x = 0; x < kQ; ++x) {
    const int i = tid + x * kF32Threads, r = i / (D / 4), ch = i - r * (D / 4);
    const int rr = min(r, rows - 1), qq = q_of(rr);
    qv[x] = *reinterpret_cast<const f32x4*>(static_cast<const float*>(a.q) + (q_start + qq) * a.q_st +
                                            head_of(rr, qq) * a.q_sh + 4 * ch);
  }

  const float* const kb = static_cast<const float*>(a.k) + k_start * a.k_st + kvh * a.k_sh + 4 * g;
  const float* const vb = static_cast<const float*>(a.v) + k_start * a.v_st + kvh * a.v_sh + 4 * c;
  f32x4 kop[NJ];
  // Keys past the sequence's last re-read it; their scores are masked.
  auto load_k = [&](int blk) __attribute__((always_inline)) {
    const float* p = kb + static_cast<int64_t>(min(blk * 16 + c, kl - 1)) * a.k_st;
#pragma unroll
    for (int j = 0; j < NJ; ++j) kop[j] = *reinterpret_cast<const f32x4*>(p + 16 * j);
  };
  if (wave < nblk) load_k(wave);
#pragma unroll
  for (int x = 0; x < kQ; ++x) {
    const int i = tid + x * kF32Threads, r = i / (D / 4), ch = i - r * (D / 4);
    *reinterpret_cast<f32x4*>(smem + r * RP + 4 * ch) = qv[x];
  }
  int my_end[2];  // keys that rows c and 16 + c see
#pragma unroll
  for (int t = 0; t < 2; ++t) my_end[t] = a.causal ? min(kl, q_of(min(16 * t + c, rows - 1)) + 1) : kl;
  __syncthreads();

  float m[2] = {kNegInfP, kNegInfP}, l[2] = {0.f, 0.f};
  bool bad = false;
  f32x4 acc[2][NH][4];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int y = 0; y < NH; ++y)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[t][y][i] = f32x4{0.f, 0.f, 0.f, 0.f};

  for (int blk = wave; blk < nblk; blk += 4) {
    const int k0 = blk * 16;
    f32x4 vop[4][NH];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float* p = vb + static_cast<int64_t>(min(k0 + 4 * g + r, kl - 1)) * a.v_st;
#pragma unroll
      for (int y = 0; y < NH; ++y) vop[r][y] = *reinterpret_cast<const f32x4*>(p + 64 * y);
    }
    __builtin_amdgcn_sched_barrier(0);  // in flight under the score products
    f32x4 sc[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
    const float* qrow = smem + c * RP + 4 * g;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const f32x4 q0 = *reinterpret_cast<const f32x4*>(qrow + 16 * j);
      const f32x4 q1 = *reinterpret_cast<const f32x4*>(qrow + 16 * RP + 16 * j);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        sc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(kop[j][i], q0[i], sc[0], 0, 0, 0);
        sc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(kop[j][i], q1[i], sc[1], 0, 0, 0);
      }
    }
    load_k(min(blk + 4, nblk - 1));     // the wave's next block (its last: a repeat)
    __builtin_amdgcn_sched_barrier(0);  // in flight under the softmax and P V

    const bool edge = k0 + 16 > full;  // some row does not see some key of the block
    float p[2][4];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      float s[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) s[r] = sc[t][r] * a.scale_log2;
      if (edge) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (k0 + 4 * g + r >= my_end[t]) s[r] = kNegInfP;
      }
      float mx = fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]));
      mx = fmaxf(mx, __builtin_bit_cast(float, xor_lane32<16>(__builtin_bit_cast(uint32_t, mx), lane)));
      mx = fmaxf(mx, __builtin_bit_cast(float, xor_lane32<32>(__builtin_bit_cast(uint32_t, mx), lane)));
      const float m_new = fmaxf(m[t], mx);
      const float mu = m_new == kNegInfP ? 0.f : m_new;  // (-inf: every score of the row so far is -inf, and weighs 0)
      if (__any(m_new > m[t])) {
        const float alpha = fast_exp2(m[t] - mu);
        l[t] *= alpha;
#pragma unroll
        for (int y = 0; y < NH; ++y)
#pragma unroll
          for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[t][y][i][e] *= alpha;
        m[t] = m_new;
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        p[t][r] = fast_exp2(s[r] - mu);
        l[t] += p[t][r];
      }
    }
    // A key that some row does not see must not reach that row: its weight is
    // 0, but 0 times an infinity or NaN in its V row is NaN. An item that
    // meets one is computed again, row by row, below.
    if (edge) {
      float z = 0.f;
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int y = 0; y < NH; ++y)
#pragma unroll
          for (int i = 0; i < 4; ++i) z = fmaf(vop[r][y][i], 0.f, z);
      bad |= z != 0.f;  // NaN
    }
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int y = 0; y < NH; ++y)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          acc[0][y][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(vop[r][y][i], p[0][r], acc[0][y][i], 0, 0, 0);
          acc[1][y][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(vop[r][y][i], p[1][r], acc[1][y][i], 0, 0, 0);
        }
  }
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    l[t] += __builtin_bit_cast(float, xor_lane32<16>(__builtin_bit_cast(uint32_t, l[t]), lane));
    l[t] += __builtin_bit_cast(float, xor_lane32<32>(__builtin_bit_cast(uint32_t, l[t]), lane));
  }

  if (__syncthreads_or(bad)) {
    for (int r = wave; r < rows; r += 4) {
      const int qq = q_of(r);
      prefill_row<float>(a, q_start + qq, qq, head_of(r, qq), k_start, k_len);
    }
    return;
  }

  // The waves' partials: waves 1 to 3 leave theirs in LDS (Q is no longer
  // read), wave 0 adds them to its registers and writes the rows.
  // Element e of acc[t][y][i] is row 16 t + c, dim 64 y + 4 (4 g + e) + i.
#pragma unroll
  for (int t = 0; t < 2; ++t)
    if (g == 0) {
      ml[wave * kF32Rows + 16 * t + c] = m[t];
      ml[(4 + wave) * kF32Rows + 16 * t + c] = l[t];
    }
  if (wave > 0) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      float* const mine = smem + ((wave - 1) * kF32Rows + 16 * t + c) * RP + 16 * g;
#pragma unroll
      for (int y = 0; y < NH; ++y)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          *reinterpret_cast<f32x4*>(mine + 64 * y + 4 * e) =
              f32x4{acc[t][y][0][e], acc[t][y][1][e], acc[t][y][2][e], acc[t][y][3][e]};
    }
  }
  __syncthreads();
  if (wave > 0) return;
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int r = 16 * t + c;
    float f[4], M = kNegInfP, den = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) M = fmaxf(M, ml[w * kF32Rows + r]);
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float mw = ml[w * kF32Rows + r];
      f[w] = mw == kNegInfP ? 0.f : fast_exp2(mw - M);  // (a wave without a seen key: l = 0 and O = 0)
      den = fmaf(f[w], ml[(4 + w) * kF32Rows + r], den);
    }
    if (r >= rows) continue;
    const int qq = q_of(r);
    float* const dst = static_cast<float*>(a.out) + (q_start + qq) * a.o_st + head_of(r, qq) * a.o_sh + 16 * g;
#pragma unroll
    for (int y = 0; y < NH; ++y)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        f32x4 o = f32x4{acc[t][y][0][e], acc[t][y][1][e], acc[t][y][2][e], acc[t][y][3][e]} * f[0];
#pragma unroll
        for (int w = 1; w < 4; ++w)
          o += *reinterpret_cast<const f32x4*>(smem + ((w - 1) * kF32Rows + r) * RP + 64 * y + 16 * g + 4 * e) * f[w];
        *reinterpret_cast<f32x4*>(dst + 64 * y + 4 * e) = o / den;
      }
  }
}

// Float32 rows of 64 or 128 dims in 16-byte pieces. The grid covers every
// item there can be: each sequence adds at most one partial tile to
// total_q * G / 32.
bool prefill_f32_takes(const PrefillArgs& a) {
  const int64_t rows = a.total_q * a.G;
  return (a.D == 64 || a.D == 128) && a.total_k > 0 && rows < (int64_t{1} << 31) - kF32Rows && a.total_k < (1 << 30) &&
         ((rows + kF32Rows - 1) / kF32Rows + a.nseq) * a.Hkv < (int64_t{1} << 31);
}
int prefill_f32_launch(const PrefillArgs& a, hipStream_t stream) {
  const int64_t items = ((a.total_q * a.G + kF32Rows - 1) / kF32Rows + a.nseq) * a.Hkv;
  if (a.D == 128) varlen_prefill_f32<128><<<dim3(items), dim3(kF32Threads), 0, stream>>>(a);
  else varlen_prefill_f32<64><<<dim3(items), dim3(kF32Threads), 0, stream>>>(a);
  return check_launch("tsa_varlen_prefill");
}

}  // namespace tsa
