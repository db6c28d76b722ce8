// Packed chunked-prefill attention for fp32 storage (head_dim 128, page 16),
// bottom-right causal, on the fp32 matrix instructions.
//
// A workgroup of 8 waves owns 32 query rows of one (sequence, query head);
// wave w takes the 32-key tiles w, w + 8, ... and the waves merge at the end.
// Bound by the matrix cores: v_mfma_f32_32x32x2 multiplies 256 flop per cycle
// and CU, so a wave spends 8192 cycles on a tile's 128 instructions, beside
// which loading the tile straight into operand registers costs nothing that
// LDS staging would save (K: 16 bytes of 32 rows per load; V: whole rows).
// Three chunks of 84-176 rows over contexts of 116-583 more: 36 us, where the
// per-token path (every row a decode of its whole context) took 182 us.
// With few rows the chip is filled from the key side, which is why a row tile
// is 32 rows and the waves split its keys; with too few it is not taken at all
// (f32_kernel_pays in paged_prefill.hip).
//
// Operand layouts (lane l: i = l % 32, half = l / 32).  The products sum over
// dims, resp. keys, in any order, so the order is the one the loads come in:
//   S^T = K Q^T   k-step (s, e): dims 8s + e (half 0) and 8s + 4 + e (half 1);
//     a lane's 16 bytes at dims 8s + 4half of key i feed four k-steps.
//   O^T = V^T P^T k-step r: keys 8(r/4) + r%4 (half 0) and + 4 (half 1), which
//     is where the S^T accumulator leaves element r: P needs no exchange.
//     Output tile c holds dims 4i + c, so a lane's 16 bytes at dims 4i of one
//     key feed all four tiles.
#include <algorithm>

#include "common.hpp"
#include "mfma.hpp"
#include "prefill_f32.hpp"

namespace rlt {
namespace {

constexpr int kRows = 32;   // query rows per workgroup
constexpr int kKeys = 32;   // keys per tile
constexpr int kWaves = 8;
constexpr int kD = 128;
constexpr int kPage = 16;
constexpr int kSteps = kD / 8;  // 16-byte loads of a K row per lane

// Block b is (row tile b / hq, head b % hq): with hq a multiple of 8 one head's
// row tiles share an XCD and its L2.
__global__ __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(2))) void paged_prefill_f32_kernel(
    PrefillF32Args a) {
  // q as S^T's B operand, then the waves' accumulators and (max, sum).
  __shared__ __align__(16) f32x4 lds[kWaves * 16 * 64];
  __shared__ float2 lds_ml[kWaves][64];
  __shared__ int lds_odd;  // a masked tile's V holds elements that are not finite
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = uniform(tid >> 6);
  const int half = lane >> 5, i = lane & 31;
  const int h = static_cast<int>(blockIdx.x) % a.hq;
  int tile = static_cast<int>(blockIdx.x) / a.hq;

  // The tile's sequence: 64 at a time, one per lane, by a scan of their tiles.
  int row0 = 0, nq = 0, seq = -1;
  for (int s0 = 0; s0 < a.num_seqs; s0 += 64) {
    const int s = min(s0 + lane, a.num_seqs - 1);
    const int r0 = min(max(a.cu[s], 0), a.total_q);
    const int n = min(max(a.cu[s + 1], r0), a.total_q) - r0;
    const int mine = s0 + lane < a.num_seqs ? (n + kRows - 1) / kRows : 0;
    int incl = mine;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int y = __shfl_up(incl, o, 64);
      if (lane >= o) incl += y;
    }
    const uint64_t hit = __builtin_amdgcn_ballot_w64(tile < incl);
    if (hit) {
      const int at = __builtin_ctzll(hit);
      seq = s0 + at;
      row0 = __builtin_amdgcn_readlane(r0, at);
      nq = __builtin_amdgcn_readlane(n, at);
      tile -= __builtin_amdgcn_readlane(incl - mine, at);
      break;
    }
    tile -= __builtin_amdgcn_readlane(incl, 63);
  }
  if (seq < 0) return;
  const int64_t max_len = a.width * kPage;
  const int len = static_cast<int>(min<int64_t>(a.lens[seq], max_len));
  const int prefix = len - nq;
  tile = (nq + kRows - 1) / kRows - 1 - tile;  // longest first
  const int t0 = tile * kRows;
  const int rows = min(nq - t0, kRows);
  const int my_row = t0 + min(i, rows - 1);
  const int limit = prefix + my_row;             // last key of the lane's query
  const int keys = prefix + t0 + rows;           // keys of the tile's last row
  const int ntiles = keys > 0 ? (keys + kKeys - 1) / kKeys : 0;
  const int last = len - 1;
  const int open = prefix + t0;                  // last key that every row of the tile sees
  const int kvh = h / (a.hq / a.hkv);

  if (tid == 0) lds_odd = 0;
  // q rows into LDS, laid out as the lanes read them.
  for (int u = tid; u < kSteps * 64; u += 64 * kWaves) {
    const int s = u >> 6, l = u & 63;
    const int r = t0 + min(l & 31, rows - 1);
    f32x4 v = *reinterpret_cast<const f32x4*>(a.q + (row0 + r) * a.q_row + static_cast<int64_t>(h) * a.q_head + 8 * s +
                                              4 * (l >> 5));
    lds[u] = a.negate ? -v : v;  // a negative scale, exactly
  }
  __syncthreads();

  f32x16 acc[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) acc[c] = f32x16{};
  float m = -INFINITY, lsum = 0.f;

  const int32_t* const trow = a.tables + static_cast<int64_t>(seq) * a.table_stride;
  const float* const kbase = a.k + static_cast<int64_t>(kvh) * a.kv_head;
  const float* const vbase = a.v + static_cast<int64_t>(kvh) * a.kv_head;
  // Page ids of the wave's next 32 tiles, two per tile, one per lane.
  int32_t ids = 0;
  auto load_ids = [&](int n) {  // n: the wave's tile count so far, a multiple of 32
    const int page = 2 * (wave + kWaves * (n + (lane >> 1))) + (lane & 1);
    ids = trow[min(page, last / kPage)];
  };
  auto block = [&](int lane_index) -> int64_t {
    const int32_t b = __builtin_amdgcn_readlane(ids, lane_index);
    return (b < 0 || b >= a.num_blocks) ? 0 : b;
  };
  // The last slot that holds a key in page p (0 or 1) of the tile at key0.
  // Keys past the sequence re-read its last one (masked, and never unwritten):
  // load_ids gives a page past it the last page's id.
  auto last_slot = [&](int key0, int p) {
    const int at = last - (key0 + kPage * p);
    return at < 0 ? last % kPage : min(at, kPage - 1);
  };
  const uint32_t token_bytes = static_cast<uint32_t>(a.kv_token * sizeof(float));
  f32x4 kr[kSteps];
  auto load_k = [&](int n) {
    const int key0 = kKeys * (wave + kWaves * n);
    const int64_t b = i < kPage ? block(2 * (n & 31)) : block(2 * (n & 31) + 1);
    const int slot = min(i & (kPage - 1), i < kPage ? last_slot(key0, 0) : last_slot(key0, 1));
    const float* p = kbase + b * a.kv_block + slot * a.kv_token + 4 * half;
#pragma unroll
    for (int s = 0; s < kSteps; ++s) kr[s] = *reinterpret_cast<const f32x4*>(p + 8 * s);
  };
  // V rows 8(r/4) + r%4 + 4half of page r/8: a scalar page base and 32-bit
  // lane offsets.
  f32x4 vr[8];
  auto load_v = [&](int n, int p, int u0, int u1) __attribute__((always_inline)) {
    int h4 = 4 * half;
    asm volatile("" : "+v"(h4));  // the rows' offsets are cheaper recomputed than kept in registers
    const int lim = last_slot(kKeys * (wave + kWaves * n), p);
    const char* const page = reinterpret_cast<const char*>(vbase + block(2 * (n & 31) + p) * a.kv_block);
#pragma unroll
    for (int u = u0; u < u1; ++u) {
      const uint32_t slot = min(8 * (u >> 2) + (u & 3) + h4, lim);
      vr[u] = *reinterpret_cast<const f32x4*>(page + (slot * token_bytes + 16u * i));
    }
  };

  // Tiles with keys that some row does not see.  P = 0 keeps a masked key's V
  // out of a row only while it is finite, so what is not leaves the products
  // here, and the store adds it to the rows that see it.  One product an element
  // finds out whether there is any (comparing each cost 2% of the kernel).
  auto confine = [&](int n) __attribute__((always_inline)) {
    if (kKeys * (wave + kWaves * n) + kKeys - 1 <= open) return;
    float t = 0.f;  // 0 times what is not finite is a NaN
#pragma unroll
    for (int u = 0; u < 8; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e) t = fmaf(vr[u][e], 0.f, t);
    if (__builtin_amdgcn_ballot_w64(t != t) == 0) return;
    lds_odd = 1;
#pragma unroll
    for (int u = 0; u < 8; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if ((__float_as_uint(vr[u][e]) & 0x7f800000u) == 0x7f800000u) vr[u][e] = 0.f;
  };

  const int mine = ntiles > wave ? (ntiles - wave + kWaves - 1) / kWaves : 0;
  if (mine > 0) {
    load_ids(0);
    load_k(0);
  }
  for (int n = 0; n < mine; ++n) {
    const int key0 = kKeys * (wave + kWaves * n);
    // Short chains of 8 products each, added up as a tree: one chain over the
    // 128 dims loses twice what the per-token path's lane sums do (against 64
    // bits 2.1e-7 on average, 1.5e-7 as here), and two run side by side, so
    // consecutive products do not wait for each other.
    f32x16 tree[4];
#pragma unroll
    for (int b = 0; b < kSteps / 2; ++b) {
      f32x16 c0 = {}, c1 = {};
      const f32x4 q0 = lds[(2 * b) * 64 + lane], q1 = lds[(2 * b + 1) * 64 + lane];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        c0 = __builtin_amdgcn_mfma_f32_32x32x2f32(kr[2 * b][e], q0[e], c0, 0, 0, 0);
        c1 = __builtin_amdgcn_mfma_f32_32x32x2f32(kr[2 * b + 1][e], q1[e], c1, 0, 0, 0);
      }
      if (b == kSteps / 4) {  // V's first rows, once half of K's registers are free
        __builtin_amdgcn_sched_barrier(0);
        load_v(n, 0, 0, 4);
        __builtin_amdgcn_sched_barrier(0);
      }
      c0 += c1;
      int level = 0;
#pragma unroll
      for (int n2 = b; n2 & 1; n2 >>= 1) c0 += tree[level++];
      tree[level] = c0;
      __builtin_amdgcn_sched_barrier(0);  // chains of one pair at a time: 32 registers
    }
    const f32x16 score = tree[3];
    load_v(n, 0, 4, 8);
    float p[16];
    float tmax = -INFINITY;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int key = key0 + 8 * (r >> 2) + 4 * half + (r & 3);
      p[r] = key > limit ? -INFINITY : score[r];
      tmax = fmaxf(tmax, p[r]);
    }
    tmax = max_across_halves(tmax) * a.qscale;
    const float mn = fmaxf(m, tmax);
    const float corr = mn == -INFINITY ? 1.f : fast_exp2(m - mn);
    const float mb = mn == -INFINITY ? 0.f : mn;
    m = mn;
#pragma unroll
    for (int r = 0; r < 16; ++r) p[r] = fast_exp2(fmaf(p[r], a.qscale, -mb));  // one rounding of the exponent
    lsum = fmaf(lsum, corr, (((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]))) +
                                (((p[8] + p[9]) + (p[10] + p[11])) + ((p[12] + p[13]) + (p[14] + p[15]))));
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[c][r] *= corr;
    confine(n);
#pragma unroll
    for (int r = 0; r < 8; ++r)
#pragma unroll
      for (int c = 0; c < 4; ++c) acc[c] = __builtin_amdgcn_mfma_f32_32x32x2f32(vr[r][c], p[r], acc[c], 0, 0, 0);
    load_v(n, 1, 0, 8);
    if (n + 1 < mine) {
      if (((n + 1) & 31) == 0) load_ids(n + 1);
      load_k(n + 1);
    }
    __builtin_amdgcn_sched_barrier(0);
    confine(n);
#pragma unroll
    for (int r = 0; r < 8; ++r)
#pragma unroll
      for (int c = 0; c < 4; ++c) acc[c] = __builtin_amdgcn_mfma_f32_32x32x2f32(vr[r][c], p[8 + r], acc[c], 0, 0, 0);
  }

  // Merge: every wave hands over its accumulators; wave w then sums element
  // pair 2w, 2w + 1 (dims 4i' .. + 3 of two i') over the waves, in wave order.
  __syncthreads();  // q has been read
#pragma unroll
  for (int r = 0; r < 16; ++r) lds[(wave * 16 + r) * 64 + lane] = f32x4{acc[0][r], acc[1][r], acc[2][r], acc[3][r]};
  lsum += __shfl_xor(lsum, 32, 64);  // the other half's keys
  lds_ml[wave][lane] = make_float2(m, lsum);
  __syncthreads();
  float M = -INFINITY;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) M = fmaxf(M, lds_ml[w][lane].x);
  float f[kWaves], total = 0.f;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    const float2 ml = lds_ml[w][lane];
    f[w] = ml.x == -INFINITY ? 0.f : fast_exp2(ml.x - M);
    total = fmaf(ml.y, f[w], total);
  }
  const float inv = total > 0.f ? 1.f / total : 0.f;  // a row that sees no key is written as zeros
  if (i >= rows) return;
  const bool odd = uniform(lds_odd);
  float* const orow = a.out + (row0 + my_row) * a.o_row + static_cast<int64_t>(h) * a.o_head;
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int r = 2 * wave + u;
    f32x4 o = {};
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      const f32x4 x = lds[(w * 16 + r) * 64 + lane];
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = fmaf(x[e], f[w], o[e]);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] *= inv;
    const int dim = 4 * (8 * (r >> 2) + 4 * half + (r & 3));
    if (odd) {
      for (int key = max(open + 1, 0) / kKeys * kKeys; key <= limit; ++key) {
        const int32_t b = trow[key / kPage];
        const int64_t blk = (b < 0 || b >= a.num_blocks) ? 0 : b;
        const f32x4 v = *reinterpret_cast<const f32x4*>(vbase + blk * a.kv_block + key % kPage * a.kv_token + dim);
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if ((__float_as_uint(v[e]) & 0x7f800000u) == 0x7f800000u) o[e] += v[e];
      }
    }
    *reinterpret_cast<f32x4*>(orow + dim) = o;
  }
}

}  // namespace

int launch_prefill_f32(const PrefillF32Args& a, hipStream_t stream) {
  const int64_t blocks = (static_cast<int64_t>(a.total_q) / kRows + a.num_seqs) * a.hq;
  if (blocks > 0x7fffffff) return fail(RLT_EUNSUPPORTED, "rlt_paged_prefill: too many query tiles");
  hipLaunchKernelGGL(paged_prefill_f32_kernel, dim3(static_cast<unsigned>(blocks)), dim3(64 * kWaves), 0, stream, a);
  return check_launch("rlt_paged_prefill(fp32)");
}

}  // namespace rlt
