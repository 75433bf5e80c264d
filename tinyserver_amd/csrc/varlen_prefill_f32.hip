// Varlen causal prefill in float32 on the f32 matrix instructions.
//
// Reference: server/model/kernels/varlen_attention.py:8-142.
//
// What bounds it: v_mfma_f32_32x32x2_f32, 64 cycles for 4,096 FLOP a SIMD (a
// large float32 matrix product reaches 133 TFLOP/s on this card), so the
// kernel keeps that pipe fed and nothing else matters much: the operands come
// straight from global memory (the L2 after the first touch) into registers,
// a K/V block of 32 keys feeding 128 instructions, 8,192 cycles.
//
// Work item: 32 rows of one (sequence, kv head), a row being one (query,
// q-head of the kv head's group), query-major, so one K/V read serves the
// whole GQA group and a tile spans only 32 / G queries of the causal diagonal.
// One 4-wave workgroup takes an item and deals its 32-key blocks to the waves
// in turn: short items then finish in a quarter of the time one wave would
// take, which is what fills 1,024 SIMDs from a few thousand tokens. The waves'
// partials (m, l, O^T) meet in LDS once per item. Two workgroups share a CU
// (68 KB of LDS each, at most 256 registers a wave).
//
// Layouts. With lane (h, c) = (lane / 32, lane % 32):
//   S^T(32 keys x 32 rows) = K Q^T: step 4 J + i takes dims 8 J + 4 h + i, so a
//     lane's K and Q operands are 16-byte pieces of key c's and row c's vectors;
//     element e of the accumulator is the score of key 8 (e/4) + 4 h + e%4 for
//     row c.
//   O^T(dims x rows) += V^T P^T: step e takes keys 8 (e/4) + e%4 (+ 4 for h = 1),
//     whose probabilities are element e of the scores' lanes: P never leaves its
//     registers. Tile u's row r is dim NU r + u, so a lane's V operands of a key
//     are NU consecutive floats. A lane holds row c's outputs, so the softmax's
//     scales are the lane's own.
//
// Measured: 8 prompts of 32-512 tokens, 16/8 heads of 128 dims
// (perf case sizes, 3.5 GFLOP): see kept figures at the launch below.
#include <cmath>

#include "tsa_common.h"
#include "varlen_prefill_gqa.h"
#include "varlen_prefill_row.h"

namespace tsa {

constexpr int kF32Rows = 32;     // rows of an item
constexpr int kF32Threads = 256;

typedef float f32x16v __attribute__((ext_vector_type(16)));

// Tiles of 32 (query, head-of-group) rows of sequence b.
__device__ __forceinline__ int f32_tiles(const PrefillArgs& a, int b) {
  int64_t s, n;
  seq_range(a.cu_q, a.cuq_s, b, a.total_q, s, n);
  return static_cast<int>((n * a.G + kF32Rows - 1) / kF32Rows);
}

__device__ __forceinline__ int wave_sum(int x) {
  return __builtin_amdgcn_readlane(static_cast<int>(wave_scan_u32(static_cast<uint32_t>(x))), 63);
}

// Item j (of the launch's tiles, all kv heads together) -> sequence b, tile t.
// Up to 64 sequences: latest (heaviest) tiles first over all sequences, by a
// binary search on the level (the number of tiles at or above a level, summed
// over the wave's lanes). More sequences: sequence by sequence, latest tile
// first. Returns false past the last item. Wave-uniform.
__device__ __forceinline__ bool f32_item(const PrefillArgs& a, int j, int& b, int& t) {
  const int lane = threadIdx.x & 63;
  if (a.nseq <= 64) {
    const int nt = lane < a.nseq ? f32_tiles(a, lane) : 0;
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
  return true;
}

template <int D>
constexpr int f32_row_floats() { return D + 4; }  // LDS row pitch: 16-byte aligned, rows 4 banks apart
template <int D>
constexpr int f32_smem_floats() { return 4 * kF32Rows * f32_row_floats<D>() + 2 * 4 * kF32Rows; }

template <int D>
__global__ __launch_bounds__(kF32Threads) __attribute__((amdgpu_waves_per_eu(2, 2))) void varlen_prefill_f32(
    PrefillArgs a) {
  constexpr int NJ = D / 8;   // 16-byte pieces of a lane's K or Q operand
  constexpr int NU = D / 32;  // output tiles: consecutive dims a lane reads of a V row
  constexpr int RP = f32_row_floats<D>();
  typedef float vrow_t __attribute__((ext_vector_type(NU)));
  __shared__ __align__(16) float smem[f32_smem_floats<D>()];
  float* const ml = smem + 4 * kF32Rows * RP;  // m[4][32], l[4][32]

  const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, c = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kvh = static_cast<int>(blockIdx.x) % a.Hkv;
  int b, tile;
  if (!f32_item(a, static_cast<int>(blockIdx.x) / a.Hkv, b, tile)) return;
  int64_t q_start, q_len, k_start, k_len;
  seq_range(a.cu_q, a.cuq_s, b, a.total_q, q_start, q_len);
  seq_range(a.cu_k, a.cuk_s, b, a.total_k, k_start, k_len);
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
  const int nblk = (kend + 31) / 32;
  const int full = a.causal ? min(kl, q_first + 1) : kl;  // keys below it are seen by every row
  const int my_q = q_of(min(c, rows - 1));
  const int my_end = a.causal ? min(kl, my_q + 1) : kl;    // keys row c sees

  // The item's Q rows into LDS (rows past the last repeat it).
  for (int i = tid; i < kF32Rows * (D / 4); i += kF32Threads) {
    const int r = i / (D / 4), ch = i - r * (D / 4);
    const int rr = min(r, rows - 1), qq = q_of(rr);
    const float* src = static_cast<const float*>(a.q) + (q_start + qq) * a.q_st + head_of(rr, qq) * a.q_sh + 4 * ch;
    *reinterpret_cast<f32x4*>(smem + r * RP + 4 * ch) = *reinterpret_cast<const f32x4*>(src);
  }

  const float* const kb = static_cast<const float*>(a.k) + k_start * a.k_st + kvh * a.k_sh + 4 * h;
  const float* const vb = static_cast<const float*>(a.v) + k_start * a.v_st + kvh * a.v_sh + NU * c;
  f32x4 kop[NJ];
  // Keys past the sequence's last re-read it; their scores are masked.
  auto load_k = [&](int blk) __attribute__((always_inline)) {
    const float* p = kb + static_cast<int64_t>(min(blk * 32 + c, kl - 1)) * a.k_st;
#pragma unroll
    for (int j = 0; j < NJ; ++j) kop[j] = *reinterpret_cast<const f32x4*>(p + 8 * j);
  };
  if (wave < nblk) load_k(wave);
  __syncthreads();

  float m = kNegInfP, l = 0.f;
  bool bad = false;
  f32x16v acc[NU];
#pragma unroll
  for (int u = 0; u < NU; ++u)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[u][e] = 0.f;

  for (int blk = wave; blk < nblk; blk += 4) {
    const int k0 = blk * 32;
    vrow_t vop[16];
    auto load_v = [&](int e0) __attribute__((always_inline)) {  // eight of the lane's sixteen V operands
#pragma unroll
      for (int e = e0; e < e0 + 8; ++e) {
        const int key = min(k0 + 8 * (e / 4) + 4 * h + e % 4, kl - 1);
        vop[e] = *reinterpret_cast<const vrow_t*>(vb + static_cast<int64_t>(key) * a.v_st);
      }
    };
    load_v(0);
    __builtin_amdgcn_sched_barrier(0);  // in flight under the score products
    f32x16v sc;
#pragma unroll
    for (int e = 0; e < 16; ++e) sc[e] = 0.f;
    const float* qrow = smem + c * RP + 4 * h;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const f32x4 qv = *reinterpret_cast<const f32x4*>(qrow + 8 * j);
#pragma unroll
      for (int i = 0; i < 4; ++i) sc = __builtin_amdgcn_mfma_f32_32x32x2f32(kop[j][i], qv[i], sc, 0, 0, 0);
    }
    load_v(8);
    __builtin_amdgcn_sched_barrier(0);

    float s[16];
    const bool edge = k0 + 32 > full;  // some row does not see some key of the block
#pragma unroll
    for (int e = 0; e < 16; ++e) s[e] = sc[e] * a.scale_log2;
    if (edge) {
#pragma unroll
      for (int e = 0; e < 16; ++e)
        if (k0 + 8 * (e / 4) + 4 * h + e % 4 >= my_end) s[e] = kNegInfP;
    }
    float mx = s[0];
#pragma unroll
    for (int e = 1; e < 16; ++e) mx = fmaxf(mx, s[e]);
    mx = fmaxf(mx, __builtin_bit_cast(float, xor_lane32<32>(__builtin_bit_cast(uint32_t, mx), lane)));
    const float m_new = fmaxf(m, mx);
    const float mu = m_new == kNegInfP ? 0.f : m_new;  // (-inf: every score of row c so far is -inf, and weighs 0)
    if (__any(m_new > m)) {
      const float alpha = fast_exp2(m - mu);
      l *= alpha;
#pragma unroll
      for (int u = 0; u < NU; ++u)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[u][e] *= alpha;
      m = m_new;
    }
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      s[e] = fast_exp2(s[e] - mu);
      l += s[e];
    }
    // A key that some row does not see must not reach that row: its weight is
    // 0, but 0 times an infinity or NaN in its V row is NaN. An item that
    // meets one is computed again, row by row, below.
    if (edge) {
      float z = 0.f;
#pragma unroll
      for (int e = 0; e < 16; ++e)
#pragma unroll
        for (int u = 0; u < NU; ++u) z = fmaf(vop[e][u], 0.f, z);
      bad |= z != 0.f;  // NaN
    }
    auto pv = [&](int e0) __attribute__((always_inline)) {
#pragma unroll
      for (int e = e0; e < e0 + 8; ++e)
#pragma unroll
        for (int u = 0; u < NU; ++u)
          acc[u] = __builtin_amdgcn_mfma_f32_32x32x2f32(vop[e][u], s[e], acc[u], 0, 0, 0);
    };
    pv(0);
    // The next block's K, into the registers that V's first half leaves
    // (the wave's last block loads itself again).
    load_k(min(blk + 4, nblk - 1));
    __builtin_amdgcn_sched_barrier(0);  // under the second half of P V
    pv(8);
  }
  l += __builtin_bit_cast(float, xor_lane32<32>(__builtin_bit_cast(uint32_t, l), lane));

  if (__syncthreads_or(bad)) {
    for (int r = wave; r < rows; r += 4) {
      const int qq = q_of(r);
      prefill_row<float>(a, q_start + qq, qq, head_of(r, qq), k_start, k_len);
    }
    return;
  }

  // The four waves' partials meet in LDS (Q is no longer read).
  float* const mine = smem + (wave * kF32Rows + c) * RP;
#pragma unroll
  for (int e = 0; e < 16; ++e) {
    vrow_t o;
#pragma unroll
    for (int u = 0; u < NU; ++u) o[u] = acc[u][e];
    *reinterpret_cast<vrow_t*>(mine + NU * (8 * (e / 4) + 4 * h + e % 4)) = o;
  }
  if (h == 0) {
    ml[wave * kF32Rows + c] = m;
    ml[(4 + wave) * kF32Rows + c] = l;
  }
  __syncthreads();
  for (int i = tid; i < rows * (D / 4); i += kF32Threads) {
    const int r = i / (D / 4), ch = i - r * (D / 4);
    float mw[4], M = kNegInfP;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      mw[w] = ml[w * kF32Rows + r];
      M = fmaxf(M, mw[w]);
    }
    f32x4 o = f32x4{0.f, 0.f, 0.f, 0.f};
    float den = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float f = mw[w] == kNegInfP ? 0.f : fast_exp2(mw[w] - M);
      // A wave without a seen key has l = 0 and O = 0, and weighs nothing.
      den += f * ml[(4 + w) * kF32Rows + r];
      const f32x4 p = *reinterpret_cast<const f32x4*>(smem + (w * kF32Rows + r) * RP + 4 * ch);
#pragma unroll
      for (int x = 0; x < 4; ++x) o[x] += f * p[x];
    }
    const int qq = q_of(r);
    float* dst = static_cast<float*>(a.out) + (q_start + qq) * a.o_st + head_of(r, qq) * a.o_sh + 4 * ch;
#pragma unroll
    for (int x = 0; x < 4; ++x) o[x] /= den;
    *reinterpret_cast<f32x4*>(dst) = o;
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
