// Class-A token scores of the decode step (gfx950).
//
// A class-A KV head's query heads rate every audio token of their own
// segment by its softmax weight; the weights, summed over the heads, are
// added to a per-sample accumulator that the chunk planner ranks
// (reference: q1_decode_attn_score, src/common/kv/fused_attn.py:68-156, and
// fused_score_accumulate, src/algorithms/wnw/code/kernels.py:302-370).
//
// Both operators need each head's final softmax normaliser before any
// weight can be formed.  Here it comes from
//   * the attention kernel itself (q1_decode_attn_score): it hands out each
//     segment's final (max, sum) in the log2 domain, so one pass over the
//     audio rows of the flagged segments remains;
//   * or a statistics pass (fused_score_accumulate, which scores a subset of
//     a group's heads with its own scale): the rows of each segment are cut
//     into slices whose partial (max, sum) pairs the scoring pass merges.
// The scoring pass gives one (sample, row range) to one workgroup, which
// sums over heads (and over flagged KV heads) in registers and adds to the
// accumulator once per token: no atomics, deterministic results.
//
// Row dot products are 16 x 16 matrix instructions (rows x heads) in the
// fused_score_accumulate passes.  In attn_score_kernel (where no logits were
// kept: callers without room for them, fp32 head_dim 256, whose attention
// kernel keeps none, more than 64 KV heads) a row of D elements is read by
// D / EPC lanes, 16 bytes each, and reduced across those lanes with a
// butterfly; q lives in LDS as fp32.
#include <math.h>

#include <algorithm>
#include <type_traits>

#include "wnw_dot.h"

namespace wnw {

static constexpr int kScoreThreads = 256;
// Row iterations per scoring workgroup: 16, or 4 when 16 would leave CUs idle
// (few samples or short audio).
static constexpr int kIters = 16;
static constexpr int kItersSmall = 4;
static constexpr int kMaxHeads = 16;
static constexpr float kLog2eS = 1.4426950408889634f;
static constexpr float kNegBigS = -1e30f;

template <typename T>
struct RowGeom {
  static constexpr int EPC = 16 / (int)sizeof(T);  // elements per 16-byte chunk
};
// Rows one scoring workgroup covers: `iters` iterations of kScoreThreads / LPR
// rows, LPR = head_dim / EPC lanes per row.
__host__ __device__ constexpr int score_rows_per_wg(int head_dim, int elem_bytes, int iters = kIters) {
  return iters * kScoreThreads / (head_dim / (16 / elem_bytes));
}

// 16-byte chunk -> EPC floats
template <typename T>
__device__ __forceinline__ void chunk_to_f32(const u32x4& w, float* f) {
  if constexpr (sizeof(T) == 4) {
#pragma unroll
    for (int i = 0; i < 4; ++i) f[i] = __uint_as_float(w[i]);
  } else {
    unpack8(w, f, (T*)nullptr);
  }
}

// Sum over the LPR lanes of a row group (lanes are contiguous, LPR a power of two).
template <int LPR>
__device__ __forceinline__ float group_sum(float x) {
#pragma unroll
  for (int o = LPR / 2; o >= 1; o >>= 1) x += __shfl_xor(x, o);
  return x;
}

// Loads nh query heads ([nh][D] of T) into LDS as fp32.
template <typename T>
__device__ __forceinline__ void stage_q(float* qf, const T* q, int nh, int D) {
  for (int i = threadIdx.x; i < nh * D; i += blockDim.x) qf[i] = Elem<T>::to_f32(q, i);
}

// ---------------------------------------------------------------------------
// scores from the attention kernel's normalisers (q1_decode_attn_score)
// ---------------------------------------------------------------------------
struct AttnScoreParams {
  const void* q;        // [n_seg, G, D]
  const void* k;        // [kv_rows, D]
  const int32_t* cu;    // [n_seg + 1]
  const int64_t* base;  // [n_seg] or null
  const float* lse;     // [n_seg, G, 2] log2 domain
  const int32_t* mask;  // [Hkv], non-zero = score this KV head
  const int32_t* audio_s;  // [B] audio range relative to the segment start
  const int32_t* audio_e;
  const int32_t* acc_off;  // [B + 1]
  float* acc;
  int32_t* err;
  int64_t kv_rows, acc_len;
  int32_t n_seg, G, Hkv;
  float scale_log2;
};

template <typename T, int D, int IT>
__global__ __launch_bounds__(kScoreThreads) void attn_score_kernel(AttnScoreParams p) {
  constexpr int EPC = RowGeom<T>::EPC;
  constexpr int LPR = D / EPC;            // lanes per row
  constexpr int RPI = kScoreThreads / LPR;  // rows per workgroup iteration
  __shared__ float qf[kMaxHeads * D];
  __shared__ float stat[kMaxHeads][2];    // (max, 1 / sum)
  const int b = blockIdx.y;
  const int tid = threadIdx.x;
  const int sub = tid % LPR;              // this lane's chunk of the row
  const int rl = tid / LPR;               // row slot in an iteration
  const int a0 = p.audio_s[b], a1 = p.audio_e[b];
  const int n_audio = a1 - a0;
  const int j0 = blockIdx.x * RPI * IT;
  if (j0 >= n_audio) return;  // workgroup-uniform
  const int64_t off = p.acc_off[b];
  if (off < 0 || off + n_audio > p.acc_len) {  // the accumulator cannot hold this sample's tokens
    if (tid == 0 && blockIdx.x == 0) raise_device_error(p.err, WNW_DEVERR_BOUNDS);
    return;  // workgroup-uniform
  }
  float total[IT];
#pragma unroll
  for (int i = 0; i < IT; ++i) total[i] = 0.f;
  const T* kp = (const T*)p.k;
  for (int kv = 0; kv < p.Hkv; ++kv) {
    if (!p.mask[kv]) continue;
    const int s = b * p.Hkv + kv;
    if (s >= p.n_seg) break;
    const int64_t len = (int64_t)p.cu[s + 1] - p.cu[s];
    const int64_t base = p.base ? p.base[s] : (int64_t)p.cu[s];
    if (a0 < 0 || a1 > len || base < 0 || base + len > p.kv_rows) {
      if (tid == 0) raise_device_error(p.err, WNW_DEVERR_BOUNDS);
      continue;  // uniform
    }
    __syncthreads();  // previous head's q / stat reads are done
    stage_q<T>(qf, (const T*)p.q + (int64_t)s * p.G * D, p.G, D);
    if (tid < p.G) {
      stat[tid][0] = p.lse[((int64_t)s * p.G + tid) * 2];
      stat[tid][1] = 1.f / p.lse[((int64_t)s * p.G + tid) * 2 + 1];
    }
    __syncthreads();
#pragma unroll
    for (int it = 0; it < IT; ++it) {
      const int j = j0 + it * RPI + rl;
      const bool valid = j < n_audio;
      const int64_t row = base + a0 + (valid ? j : 0);
      u32x4 w = *(const u32x4*)(kp + row * D + sub * EPC);
      float kf[EPC];
      chunk_to_f32<T>(w, kf);
      float sc = 0.f;
      for (int g = 0; g < p.G; ++g) {
        float d = 0.f;
#pragma unroll
        for (int i = 0; i < EPC; ++i) d += qf[g * D + sub * EPC + i] * kf[i];
        d = group_sum<LPR>(d);
        sc += exp2f(d * p.scale_log2 - stat[g][0]) * stat[g][1];
      }
      total[it] += valid ? sc : 0.f;
    }
  }
  if (sub == 0) {
#pragma unroll
    for (int it = 0; it < IT; ++it) {
      const int j = j0 + it * RPI + rl;
      if (j < n_audio) p.acc[off + j] += total[it];
    }
  }
}

// ---------------------------------------------------------------------------
// scores from the logits the streaming attention kernel kept
// ---------------------------------------------------------------------------
// The attention kernel already computed every scaled logit x = q.k * scale
// (log2 domain) of the scored audio rows; with its final (max, sum) per head
// a weight is exp2(x - max) / sum.  One thread per audio token of a sample
// sums the weights over the flagged KV heads and their query heads, and
// adds the total to the accumulator once (no atomics).  The validity rules
// are those of attn_score_kernel, so both passes score the same rows.
// The fields of the first loads are the kernel's leading scalar arguments
// (see logit_score_kernel); the rest come in this aggregate.
struct LogitScoreParams {
  const float* xlog;       // [n_seg, G, max_audio]
  const int32_t* acc_off;  // [B + 1]
  float* acc;
  int32_t* err;
  int64_t kv_rows, acc_len, max_audio;
};

static constexpr int kLogitThreads = 256;
static constexpr int kLogitKv = 64;  // KV heads per sample this pass takes (a lane of wave 0 each)
static constexpr int kLogitG = 8;    // query heads per KV head of a score slot

// Latency, not bytes, bounds this pass (a few hundred KB per launch), so
// its loads go out in two batches instead of a chain: wave 0 reads every
// KV head's flag, bounds and normalisers at once (lane = KV head; the
// sample's audio range and offset arrive in the same round trip) and lists
// the flagged, valid segments in LDS; then every thread issues the loads
// of all its logits and of its accumulator entry together.  Loads are
// unconditional (indices clamped into range) and the checks combine with
// bitwise operators, so no load waits behind a branch on another load.
//
// score.hip is built with 16 preloaded argument dwords, of which gfx950
// delivers 14 in SGPRs at dispatch: the six tables of the first round trip
// and the sizes their addresses need (hg = Hkv | G << 16, n_seg), so those
// loads issue before any argument load returns.
// KG: room for the query heads of a group (8, or 16 for wider groups, whose
// first round trip loads twice the normalisers).
template <int KG>
__global__ __launch_bounds__(kLogitThreads) void logit_score_kernel(
    const int32_t* audio_s, const int32_t* audio_e, const int32_t* mask, const int32_t* cu, const int64_t* seg_base,
    const float* lse, int32_t hg, int32_t n_seg, LogitScoreParams p) {
  __shared__ int32_t seg_sh[kLogitKv];
  __shared__ float m_sh[kLogitKv * KG], inv_sh[kLogitKv * KG];
  __shared__ int32_t n_sh;
  const int b = blockIdx.y;
  const int tid = threadIdx.x;
  const int Hkv = hg & 0xffff, G = hg >> 16;
  const int a0 = audio_s[b], a1 = audio_e[b];
  if (tid < 64) {  // wave 0
    const int kv = min(tid, Hkv - 1);
    const int s = min(b * Hkv + kv, n_seg - 1);
    const int32_t flag = mask[kv];
    const int64_t bv = seg_base ? seg_base[s] : 0;
    const int64_t c0 = cu[s], c1 = cu[s + 1];
    float m[KG], l[KG];
#pragma unroll
    for (int g = 0; g < KG; ++g) {
      const int64_t e = ((int64_t)s * G + min(g, G - 1)) * 2;
      m[g] = lse[e];
      l[g] = lse[e + 1];
    }
    const int64_t len = c1 - c0;
    const int64_t base = seg_base ? bv : c0;
    const bool flagged = (tid < Hkv) & (b * Hkv + tid < n_seg) & (flag != 0);
    const bool oob = (a0 < 0) | (a1 > len) | (base < 0) | (base + len > p.kv_rows);
    const bool use = flagged & !oob;
    if (flagged & oob & (blockIdx.x == 0)) raise_device_error(p.err, WNW_DEVERR_BOUNDS);
    const uint64_t bal = __ballot(use);
    if (use) {
      const int pos = __popcll(bal & ((1ull << tid) - 1ull));
      seg_sh[pos] = s;
#pragma unroll
      for (int g = 0; g < KG; ++g) {
        m_sh[pos * KG + g] = m[g];
        inv_sh[pos * KG + g] = 1.f / l[g];
      }
    }
    if (tid == 0) n_sh = __popcll(bal);
  }
  const int64_t off = p.acc_off[b];
  const int n_audio = a1 - a0;
  if ((int64_t)blockIdx.x * kLogitThreads >= min((int64_t)n_audio, p.max_audio)) return;  // uniform
  if (off < 0 || off + n_audio > p.acc_len) {  // the accumulator cannot hold this sample's tokens
    if (tid == 0 && blockIdx.x == 0) raise_device_error(p.err, WNW_DEVERR_BOUNDS);
    return;  // uniform
  }
  __syncthreads();
  const int64_t j = (int64_t)blockIdx.x * kLogitThreads + tid;
  const bool valid = j < n_audio && j < p.max_audio;
  const int64_t jc = valid ? j : 0;  // loads stay unconditional; `valid` gates the store
  const float prior = p.acc[off + jc];
  const int nt = n_sh * G;
  float total = 0.f, sc = 0.f;  // a segment's heads are summed first, then added to the total
  // pair t = (segment i, head g), counted rather than divided by G (uniform);
  // loads past the last pair repeat it
  int i = 0, g = 0;
  for (int t0 = 0; t0 < nt; t0 += 8) {
    float x[8];
    int li = i, lg = g;
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const bool in = t0 + u < nt;
      const int ii = in ? li : n_sh - 1, gg = in ? lg : G - 1;
      x[u] = p.xlog[((int64_t)seg_sh[ii] * G + gg) * p.max_audio + jc];
      if (++lg == G) {
        lg = 0;
        ++li;
      }
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      if (t0 + u < nt) {
        // v_exp_f32 directly: arguments are <= 0 (m is the maximum) and
        // weights below 2^-126 (flushed to zero) are negligible
        sc += __builtin_amdgcn_exp2f(x[u] - m_sh[i * KG + g]) * inv_sh[i * KG + g];
        if (g == G - 1) {
          total += sc;
          sc = 0.f;
        }
      }
      if (++g == G) {
        g = 0;
        ++i;
      }
    }
  }
  if (valid) p.acc[off + j] = prior + total;
}

// ---------------------------------------------------------------------------
// fused_score_accumulate: statistics pass + scoring pass
// ---------------------------------------------------------------------------
struct SegScoreParams {
  const void* q;           // [S, nh, D]
  const void* k;           // [k_rows, D]
  const int32_t* seg_s;    // [S] physical first row
  const int32_t* seg_e;    // [S] physical end row
  const int32_t* audio_s;  // [S] relative to seg_s
  const int32_t* audio_e;
  const int32_t* acc_off;  // [S + 1]
  float* acc;
  float* part;             // [S, slices, nh, 2] (max, sum) in the log2 domain
  int32_t* err;
  int64_t k_rows, acc_len;
  int32_t S, nh;
  float scale_log2;
};

__device__ __forceinline__ void merge_ml(float& m, float& l, float m2, float l2) {
  const float mn = fmaxf(m, m2);
  l = l * exp2f(m - mn) + l2 * exp2f(m2 - mn);
  m = mn;
}

// The 16 bytes at p, read whole where q is 16-byte aligned, else by element.
template <typename T>
__device__ __forceinline__ u32x4 load_chunk(const T* p, bool aligned) {
  if (aligned) return *gptr<u32x4>(p);
  constexpr int N = 16 / (int)sizeof(T);
  u32x4 r = u32x4{0, 0, 0, 0};
#pragma unroll
  for (int i = 0; i < N; ++i) {
    if constexpr (sizeof(T) == 4)
      r[i] = gptr<uint32_t>(p)[i];
    else
      r[i / 2] |= (uint32_t)gptr<uint16_t>(p)[i] << (16 * (i & 1));
  }
  return r;
}

// Slices per item, from the number of items alone (the workspace is sized
// before the lengths are known): two workgroups per CU of a 256-CU device from
// 4 items on (8 items of 7,564 rows: 64 slices of 118 rows), at most 128 slices,
// which the merge takes two per lane, and at least 8.  One to three items thus
// fill half to all of the CUs once, and the slices of short items hold less
// than a tile (300 rows: 2-3 rows each; such a call is bound by its two
// launches, 10.2 us like the 32 slices of the earlier kernels).
static int64_t score_slices(int64_t n_samples) {
  return std::min<int64_t>(128, std::max<int64_t>(8, (512 + n_samples - 1) / std::max<int64_t>(n_samples, 1)));
}

// Both passes, one workgroup per slice of an item's rows (SCORE 0: the
// slice's partial softmax statistics of every head; SCORE 1: every head's
// statistics merged, then each audio row's weights summed over the heads and
// added to its accumulator entry).  The passes cut the rows alike, so as long
// as K fits the eight L2s (4 MB each) the second one's comes from the L2 of the
// XCD that the first one's workgroups filled; larger K (16 items of 24,000 bf16
// rows: 98 MB) is streamed twice.  Bound by the K stream and by two launches' fixed round
// trips; a row dot by 16-lane butterflies (six lane exchanges per row and
// head) had bound it before: 25.1 + 10.4 us for 8 items of 7,564 rows, 4 heads,
// bf16 D = 128 (15.5 MB), now 5.9 + 7.8 us.
template <typename T, int D, bool SCORE>
__global__ __launch_bounds__(kScoreThreads) void seg_score_kernel(SegScoreParams p) {
  constexpr int EPC = RowGeom<T>::EPC;
  constexpr int NC = D / EPC / 4;           // chunks of a row per lane
  constexpr int U = NC >= 8 ? 1 : 8 / NC;   // tiles whose loads are in flight per wave
  constexpr int NW = kScoreThreads / 64;
  __shared__ float stat[kMaxHeads][2];
  __shared__ float red[SCORE ? 1 : NW][kMaxHeads][2];
  const int s = blockIdx.y, c = blockIdx.x, C = gridDim.x;
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lq = lane >> 4, lc = lane & 15;
  const int nh = p.nh;
  const int64_t r0 = gptr<int32_t>(p.seg_s)[s], r1 = gptr<int32_t>(p.seg_e)[s];
  int64_t c0, c1;       // this workgroup's rows of k
  int64_t off = 0, a_row = 0;
  if constexpr (SCORE) {
    const int a0 = gptr<int32_t>(p.audio_s)[s], a1 = gptr<int32_t>(p.audio_e)[s];
    const int n_audio = a1 - a0;
    off = gptr<int32_t>(p.acc_off)[s];
    if (n_audio <= 0) return;
    if (r0 < 0 || r1 < r0 || r1 > p.k_rows || a0 < 0 || r0 + a1 > r1 || off < 0 || off + n_audio > p.acc_len) {
      if (tid == 0) raise_device_error(p.err, WNW_DEVERR_BOUNDS);
      return;
    }
    a_row = r0 + a0;
    c0 = max(r0 + (r1 - r0) * c / C, a_row);
    c1 = min(r0 + (r1 - r0) * (c + 1) / C, r0 + a1);
    if (c0 >= c1) return;  // workgroup-uniform
  } else {
    const bool ok = r0 >= 0 && r1 >= r0 && r1 <= p.k_rows;
    if (!ok && tid == 0 && c == 0) raise_device_error(p.err, WNW_DEVERR_BOUNDS);
    const int64_t len = ok ? r1 - r0 : 0;
    c0 = r0 + len * c / C;
    c1 = r0 + len * (c + 1) / C;
  }
  const int ntiles = (int)((c1 - c0 + 15) / 16);
  const T* kp = (const T*)p.k;
  u32x4 kb[U][NC];
  // tile t0 + NW u of the slice into kb[u]; rows past the slice repeat its last
  auto load = [&](int t0) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t row = min(c0 + 16 * (int64_t)(t0 + NW * u) + lc, c1 - 1);
#pragma unroll
      for (int n = 0; n < NC; ++n) kb[u][n] = *gptr<u32x4>(kp + row * D + (4 * n + lq) * EPC);
    }
  };
  u32x4 qb[NC];
  {
    const T* qs = (const T*)p.q + ((int64_t)s * nh + min(lc, nh - 1)) * D;
    const bool al = ((uintptr_t)p.q & 15) == 0;
#pragma unroll
    for (int n = 0; n < NC; ++n) {
      qb[n] = load_chunk<T>(qs + (4 * n + lq) * EPC, al);
      if (lc >= nh) qb[n] = u32x4{0, 0, 0, 0};
    }
  }
  if (w < ntiles) load(w);
  float m = kNegBigS, l = 0.f;  // SCORE 0: running statistics of head lc; SCORE 1: its (max, 1 / sum)
  if constexpr (SCORE) {
    // merge the slices' statistics: wave w takes heads w, w + NW, ...
    for (int h = w; h < nh; h += NW) {
      const WNW_GLOBAL float* pp = gptr<float>(p.part) + ((int64_t)s * C * nh + h) * 2;
      float mq[2], lsum[2];  // C <= 128
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const int i = lane + 64 * k;
        mq[k] = i < C ? pp[(int64_t)min(i, C - 1) * nh * 2] : kNegBigS;
        lsum[k] = i < C ? pp[(int64_t)min(i, C - 1) * nh * 2 + 1] : 0.f;
      }
      const float M = wave_max(fmaxf(mq[0], mq[1]));
      const float L = wave_sum(lsum[0] * exp2f(mq[0] - M) + lsum[1] * exp2f(mq[1] - M));
      if (lane == 0) {
        stat[h][0] = M;
        stat[h][1] = 1.f / L;
      }
    }
    __syncthreads();
    m = stat[min(lc, nh - 1)][0];
    l = lc < nh ? stat[lc][1] : 0.f;
  }
  for (int t0 = w; t0 < ntiles; t0 += NW * U) {
    f32x4 x[U];
#pragma unroll
    for (int u = 0; u < U; ++u) x[u] = dot_rows<T, NC>(kb[u], qb);
    if (t0 + NW * U < ntiles) load(t0 + NW * U);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t row = c0 + 16 * (int64_t)(t0 + NW * u) + 4 * lq;  // of x[u][0]
      if constexpr (SCORE) {
        float sc[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          sc[i] = lc < nh ? exp2f(fmaf(x[u][i], p.scale_log2, -m)) * l : 0.f;
          // the 16 heads of the lane's row group
#pragma unroll
          for (int o = 8; o >= 1; o >>= 1) sc[i] += __shfl_xor(sc[i], o);
        }
        const float mine = lc == 0 ? sc[0] : lc == 1 ? sc[1] : lc == 2 ? sc[2] : sc[3];
        if (lc < 4 && row + lc < c1) {
          WNW_GLOBAL float* a = gptr_w<float>(p.acc) + off + (row + lc - a_row);
          *a += mine;
        }
      } else {
        // the scaled dot enters the exponent unrounded, as it does in the scores
        float mx = m;
#pragma unroll
        for (int i = 0; i < 4; ++i) mx = fmaxf(mx, row + i < c1 ? x[u][i] * p.scale_log2 : -INFINITY);
        l *= exp2f(m - mx);
#pragma unroll
        for (int i = 0; i < 4; ++i) l += row + i < c1 ? exp2f(fmaf(x[u][i], p.scale_log2, -mx)) : 0.f;
        m = mx;
      }
    }
  }
  if constexpr (!SCORE) {
#pragma unroll
    for (int o = 16; o < 64; o <<= 1) {  // the lane quarters of head lc
      const float m2 = __shfl_xor(m, o), l2 = __shfl_xor(l, o);
      merge_ml(m, l, m2, l2);
    }
    if (lane < 16) {
      red[w][lane][0] = m;
      red[w][lane][1] = l;
    }
    __syncthreads();
    if (tid < nh) {
      float M = kNegBigS, L = 0.f;
#pragma unroll
      for (int ww = 0; ww < NW; ++ww) merge_ml(M, L, red[ww][tid][0], red[ww][tid][1]);
      WNW_GLOBAL float* out = gptr_w<float>(p.part) + (((int64_t)s * C + c) * nh + tid) * 2;
      out[0] = M;
      out[1] = L;
    }
  }
}

// Calls f with a T and the head_dim as compile-time constants; false for a
// type or head_dim without an instance.
template <typename F, typename T>
static bool with_dim(int64_t D, F f, T t) {
  switch (D) {
    case 64: return f(t, std::integral_constant<int, 64>()), true;
    case 128: return f(t, std::integral_constant<int, 128>()), true;
    case 256: return f(t, std::integral_constant<int, 256>()), true;
  }
  return false;
}
template <typename F>
static bool with_type(int dtype, int64_t D, F f) {
  switch (dtype) {
    case WNW_BF16: return with_dim(D, f, bf16_t());
    case WNW_F16: return with_dim(D, f, f16_t());
    case WNW_F32: return with_dim(D, f, float());
  }
  return false;
}

// Rows per iteration count for a scoring grid of `ny` rows of workgroups over
// max_audio rows: 16 iterations when that still gives two workgroups per CU,
// else 4 (more, shorter workgroups).
static int score_iters(int64_t max_audio, int64_t ny, int64_t head_dim, int elem_bytes) {
  const int cus = device_cus();
  const int64_t rows16 = score_rows_per_wg((int)head_dim, elem_bytes, kIters);
  return ((max_audio + rows16 - 1) / rows16) * ny >= 2 * (int64_t)cus ? kIters : kItersSmall;
}

}  // namespace wnw

using namespace wnw;

static int64_t up256(int64_t x) { return (x + 255) / 256 * 256; }

// Workspace of wnw_decode_attn_score: attention workspace, normalisers, then
// (max_audio > 0) the logits of the scored audio rows.
static int64_t score_logits_offset(int64_t attn_ws, int64_t n_seg, int64_t group) {
  return attn_ws + up256(n_seg * group * 2 * 4);
}

extern "C" int64_t wnw_decode_attn_score_workspace_bytes(int64_t n_seg, int64_t group, int64_t head_dim,
                                                         int64_t max_audio) {
  const int64_t a = wnw_decode_attn_workspace_bytes(n_seg, group, head_dim);
  if (a < 0 || max_audio < 0) return -1;
  return score_logits_offset(a, n_seg, group) + up256(n_seg * group * max_audio * 4);
}

// Attention (with the step's append when app is given) + class-A scoring.
static int decode_attn_score_impl(const void* q, const void* k, const void* v, const int32_t* cu_k,
                                  const int64_t* seg_base, int64_t n_seg, int64_t group, int64_t head_dim,
                                  int64_t total_rows, int64_t kv_rows, float scale, int dtype, void* out,
                                  const int32_t* ca_kv_mask, int64_t num_kv_heads, const int32_t* audio_starts,
                                  const int32_t* audio_ends, float* score_acc, const int32_t* score_offsets,
                                  int64_t acc_len, int64_t max_audio, void* workspace, int64_t workspace_bytes,
                                  void* stream, const AttnAppend* app) {
  WNW_CHECK_ARG(num_kv_heads >= 1 && n_seg % num_kv_heads == 0,
                "n_seg (%lld) must be a multiple of num_kv_heads (%lld)", (long long)n_seg,
                (long long)num_kv_heads);
  WNW_CHECK_ARG(ca_kv_mask && audio_starts && audio_ends && score_acc && score_offsets,
                "null pointer argument");
  WNW_CHECK_ARG(max_audio >= 0 && acc_len >= 0, "negative max_audio / acc_len");
  WNW_CHECK_ARG(n_seg / num_kv_heads <= 65535, "at most 65535 samples (the scoring grid's y extent)");
  const int64_t attn_ws = wnw_decode_attn_workspace_bytes(n_seg, group, head_dim);
  WNW_CHECK_ARG(attn_ws >= 0 && workspace_bytes >= attn_ws + up256(n_seg * group * 8),
                "workspace too small for attention + normalisers");
  float* lse = (float*)((char*)workspace + attn_ws);
  // With room for them, the logits of the scored rows are kept by the
  // attention kernel (when the streaming kernel runs) and the scoring pass
  // reads 4 bytes per row and head instead of the K row.
  const int64_t xoff = score_logits_offset(attn_ws, n_seg, group);
  AttnLogits lg;
  lg.xlog = (float*)((char*)workspace + xoff);
  lg.mask = ca_kv_mask;
  lg.audio_s = audio_starts;
  lg.audio_e = audio_ends;
  lg.max_audio = max_audio;
  lg.hkv = (int32_t)num_kv_heads;
  const bool room = max_audio > 0 && num_kv_heads <= kLogitKv && group <= kMaxHeads &&
                    workspace_bytes >= xoff + n_seg * group * max_audio * 4;
  int kept = 0;
  int rc = decode_attn_impl(q, k, v, cu_k, seg_base, n_seg, group, head_dim, total_rows, kv_rows, scale,
                            dtype, out, workspace, attn_ws, WNW_ATTN_AUTO, 0, lse, room ? &lg : nullptr, &kept,
                            stream, false, app);
  if (rc != WNW_OK || n_seg == 0 || max_audio == 0) return rc;
  const int32_t* cu_scored = app ? app->cu_out : cu_k;  // the segments as the attention saw them
  if (kept) {
    LogitScoreParams lp;
    lp.xlog = lg.xlog;
    lp.acc_off = score_offsets;
    lp.acc = score_acc;
    lp.err = device_error_word();
    lp.kv_rows = kv_rows;
    lp.acc_len = acc_len;
    lp.max_audio = max_audio;
    const int32_t hg = (int32_t)num_kv_heads | ((int32_t)group << 16);  // room: Hkv <= 64, G <= 16
    const dim3 grid((unsigned)((max_audio + kLogitThreads - 1) / kLogitThreads), (unsigned)(n_seg / num_kv_heads));
    hipLaunchKernelGGL(group <= kLogitG ? logit_score_kernel<kLogitG> : logit_score_kernel<kMaxHeads>, grid,
                       dim3(kLogitThreads), 0, (hipStream_t)stream, audio_starts, audio_ends, ca_kv_mask, cu_scored,
                       seg_base, (const float*)lse, hg, (int32_t)n_seg, lp);
    WNW_CHECK_HIP(hipGetLastError(), "logit score launch");
    return WNW_OK;
  }
  AttnScoreParams sp;
  sp.q = q;
  sp.k = k;
  sp.cu = cu_scored;
  sp.base = seg_base;
  sp.lse = lse;
  sp.mask = ca_kv_mask;
  sp.audio_s = audio_starts;
  sp.audio_e = audio_ends;
  sp.acc_off = score_offsets;
  sp.acc = score_acc;
  sp.err = device_error_word();
  sp.kv_rows = kv_rows;
  sp.acc_len = acc_len;
  sp.n_seg = (int32_t)n_seg;
  sp.G = (int32_t)group;
  sp.Hkv = (int32_t)num_kv_heads;
  sp.scale_log2 = scale * kLog2eS;
  const int iters = score_iters(max_audio, n_seg / num_kv_heads, head_dim, elem_bytes(dtype));
  const int rows_wg = score_rows_per_wg((int)head_dim, elem_bytes(dtype), iters);
  const dim3 grid((unsigned)((max_audio + rows_wg - 1) / rows_wg), (unsigned)(n_seg / num_kv_heads));
  const bool known = with_type(dtype, head_dim, [&](auto t, auto d) {
    typedef decltype(t) T;
    constexpr int D = decltype(d)::value;
    hipLaunchKernelGGL((iters == kIters ? attn_score_kernel<T, D, kIters> : attn_score_kernel<T, D, kItersSmall>), grid,
                       dim3(kScoreThreads), 0, (hipStream_t)stream, sp);
  });
  WNW_CHECK_HIP(known ? hipGetLastError() : hipErrorInvalidValue, "attention score launch");
  return WNW_OK;
}

extern "C" int wnw_decode_attn_score(const void* q, const void* k, const void* v, const int32_t* cu_k,
                                     const int64_t* seg_base, int64_t n_seg, int64_t group, int64_t head_dim,
                                     int64_t total_rows, int64_t kv_rows, float scale, int dtype, void* out,
                                     const int32_t* ca_kv_mask, int64_t num_kv_heads,
                                     const int32_t* audio_starts, const int32_t* audio_ends,
                                     float* score_acc, const int32_t* score_offsets, int64_t acc_len,
                                     int64_t max_audio, void* workspace, int64_t workspace_bytes,
                                     void* stream) {
  return decode_attn_score_impl(q, k, v, cu_k, seg_base, n_seg, group, head_dim, total_rows, kv_rows, scale, dtype,
                                out, ca_kv_mask, num_kv_heads, audio_starts, audio_ends, score_acc, score_offsets,
                                acc_len, max_audio, workspace, workspace_bytes, stream, nullptr);
}

extern "C" int wnw_decode_attn_score_append(
    const void* q, void* k_pool, void* v_pool, const void* new_k, const void* new_v, const int32_t* cu_old,
    int32_t* cu_new, const int64_t* seg_base, const int32_t* seg_cap, int64_t n_seg, int64_t group,
    int64_t head_dim, int64_t total_rows, int64_t pool_rows, float scale, int dtype, void* out,
    const int32_t* ca_kv_mask, int64_t num_kv_heads, const int32_t* audio_starts, const int32_t* audio_ends,
    float* score_acc, const int32_t* score_offsets, int64_t acc_len, int64_t max_audio, void* workspace,
    int64_t workspace_bytes, void* stream) {
  AttnAppend app;
  app.new_k = new_k;
  app.new_v = new_v;
  app.cu_out = cu_new;
  app.cap = seg_cap;
  return decode_attn_score_impl(q, k_pool, v_pool, cu_old, seg_base, n_seg, group, head_dim, total_rows, pool_rows,
                                scale, dtype, out, ca_kv_mask, num_kv_heads, audio_starts, audio_ends, score_acc,
                                score_offsets, acc_len, max_audio, workspace, workspace_bytes, stream, &app);
}

// ---------------------------------------------------------------------------
// deferred scoring: score slots handed from one streaming launch to the next
// ---------------------------------------------------------------------------
// A slot holds one launch's final normalisers [n_seg, G, 2] and its kept
// logits [n_seg, G, max_audio] (fp32, 256-byte aligned parts).
static int64_t slot_logits_offset(int64_t n_seg, int64_t group) { return up256(n_seg * group * 2 * 4); }

extern "C" int64_t wnw_score_slot_bytes(int64_t n_seg, int64_t group, int64_t max_audio) {
  if (n_seg < 0 || group <= 0 || max_audio < 0) return -1;
  return slot_logits_offset(n_seg, group) + up256(n_seg * group * max_audio * 4);
}

// The logit pass over a slot (the scores of a launch that kept them and had
// no later launch to carry them).
extern "C" int wnw_score_kept_logits(const int32_t* kv_mask, const float* slot, const int32_t* cu,
                                     const int64_t* seg_base, int64_t kv_rows, int64_t n_seg, int64_t group,
                                     int64_t num_kv_heads, const int32_t* audio_starts, const int32_t* audio_ends,
                                     int64_t max_audio, float* score_acc, const int32_t* score_offsets,
                                     int64_t acc_len, void* stream) {
  WNW_CHECK_ARG(kv_mask && slot && cu && audio_starts && audio_ends && score_acc && score_offsets,
                "null pointer argument");
  WNW_CHECK_ARG(n_seg >= 0 && group >= 1 && group <= kLogitG && num_kv_heads >= 1 && num_kv_heads <= kLogitKv &&
                    n_seg % num_kv_heads == 0,
                "bad geometry: n_seg %lld, group %lld, num_kv_heads %lld", (long long)n_seg, (long long)group,
                (long long)num_kv_heads);
  WNW_CHECK_ARG(max_audio >= 0 && acc_len >= 0 && kv_rows >= 0, "negative size");
  WNW_CHECK_ARG(n_seg / num_kv_heads <= 65535, "at most 65535 samples (the scoring grid's y extent)");
  if (n_seg == 0 || max_audio == 0) return WNW_OK;
  LogitScoreParams lp;
  lp.xlog = slot + slot_logits_offset(n_seg, group) / 4;
  lp.acc_off = score_offsets;
  lp.acc = score_acc;
  lp.err = device_error_word();
  lp.kv_rows = kv_rows;
  lp.acc_len = acc_len;
  lp.max_audio = max_audio;
  const int32_t hg = (int32_t)num_kv_heads | ((int32_t)group << 16);
  const dim3 grid((unsigned)((max_audio + kLogitThreads - 1) / kLogitThreads), (unsigned)(n_seg / num_kv_heads));
  hipLaunchKernelGGL(logit_score_kernel<kLogitG>, grid, dim3(kLogitThreads), 0, (hipStream_t)stream, audio_starts,
                     audio_ends, kv_mask, cu, seg_base, slot, hg, (int32_t)n_seg, lp);
  WNW_CHECK_HIP(hipGetLastError(), "logit score launch");
  return WNW_OK;
}

extern "C" int wnw_decode_attn_append_deferred(
    const void* q, void* k_pool, void* v_pool, const void* new_k, const void* new_v, const int32_t* cu_old,
    int32_t* cu_new, const int64_t* seg_base, const int32_t* seg_cap, int64_t n_seg, int64_t group,
    int64_t head_dim, int64_t total_rows, int64_t pool_rows, float scale, int dtype, void* out,
    int64_t num_kv_heads, const int32_t* audio_starts, const int32_t* audio_ends, int64_t max_audio,
    float* score_acc, const int32_t* score_offsets, int64_t acc_len, const int32_t* keep_mask, float* keep_slot,
    uint64_t prev_kv_bits, const float* prev_slot, const int32_t* prev_cu, const int64_t* prev_base,
    int64_t prev_pool_rows, void* workspace, int64_t workspace_bytes, void* stream) {
  WNW_CHECK_ARG(num_kv_heads >= 1 && num_kv_heads <= kLogitKv && n_seg % num_kv_heads == 0,
                "n_seg (%lld) must be a multiple of num_kv_heads (%lld), at most %d KV heads", (long long)n_seg,
                (long long)num_kv_heads, kLogitKv);
  WNW_CHECK_ARG((keep_mask == nullptr) == (keep_slot == nullptr), "the keep mask and its slot come together");
  WNW_CHECK_ARG(!(keep_slot && prev_slot) || (const float*)keep_slot != prev_slot,
                "this launch's slot must not be the slot it scores");
  WNW_CHECK_ARG(max_audio > 0 || (!keep_mask && !prev_slot), "scoring needs max_audio > 0");
  WNW_CHECK_ARG(!prev_slot || (prev_cu && acc_len > 0), "the scored slot needs its offsets and an accumulator");
  // the kept logits need the streaming kernel (the only one that keeps them)
  if ((keep_mask || prev_slot) &&
      !((dtype == WNW_BF16 || dtype == WNW_F16) && (head_dim == 64 || head_dim == 128) && group <= kLogitG)) {
    set_error("deferred scoring needs the streaming kernel (bf16/f16, head_dim 64 or 128, group <= %d)", kLogitG);
    return WNW_ENOTSUP;
  }
  AttnAppend app;
  app.new_k = new_k;
  app.new_v = new_v;
  app.cu_out = cu_new;
  app.cap = seg_cap;
  AttnLogits lg;
  if (keep_mask) {
    WNW_CHECK_ARG(audio_starts && audio_ends, "null audio range");
    lg.xlog = keep_slot + slot_logits_offset(n_seg, group) / 4;
    lg.mask = keep_mask;
    lg.audio_s = audio_starts;
    lg.audio_e = audio_ends;
    lg.max_audio = max_audio;
    lg.hkv = (int32_t)num_kv_heads;
  }
  AttnPrevScore pv;
  if (prev_slot) {
    pv.lse = prev_slot;
    pv.xlog = prev_slot + slot_logits_offset(n_seg, group) / 4;
    pv.kv_bits = prev_kv_bits;
    pv.cu = prev_cu;
    pv.base = prev_base;
    pv.kv_rows = prev_pool_rows;
    pv.acc = score_acc;
    pv.acc_off = score_offsets;
    pv.acc_len = acc_len;
    pv.audio_s = audio_starts;
    pv.audio_e = audio_ends;
    pv.max_audio = max_audio;
    pv.hkv = (int32_t)num_kv_heads;
  }
  int kept = 0;
  const int rc = decode_attn_impl(q, k_pool, v_pool, cu_old, seg_base, n_seg, group, head_dim, total_rows, pool_rows,
                                  scale, dtype, out, workspace, workspace_bytes, WNW_ATTN_STREAM, 0,
                                  keep_mask ? keep_slot : nullptr, keep_mask ? &lg : nullptr, &kept, stream, false,
                                  &app, prev_slot ? &pv : nullptr);
  if (rc == WNW_OK && keep_mask && !kept) {  // cannot happen with the streaming kernel
    set_error("the logits were not kept");
    return WNW_EHIP;
  }
  return rc;
}

extern "C" int64_t wnw_fused_score_workspace_bytes(int64_t n_samples, int64_t n_heads) {
  if (n_samples < 0 || n_heads <= 0) return -1;
  return up256(n_samples * score_slices(n_samples) * n_heads * 2 * 4);
}

extern "C" int wnw_fused_score_accumulate(const void* q, const void* k, const int32_t* seg_starts,
                                          const int32_t* seg_ends, const int32_t* audio_starts,
                                          const int32_t* audio_ends, float* accumulator,
                                          const int32_t* accum_offsets, int64_t n_samples, int64_t n_heads,
                                          int64_t head_dim, int64_t k_rows, int64_t acc_len, int64_t max_audio,
                                          float scale, int dtype, void* workspace, int64_t workspace_bytes,
                                          void* stream) {
  WNW_CHECK_ARG(n_samples >= 0 && n_samples < 65536, "n_samples out of range");
  if (n_samples == 0 || max_audio == 0) return WNW_OK;
  WNW_CHECK_ARG(n_heads >= 1 && n_heads <= kMaxHeads, "n_heads must be in [1, %d]", kMaxHeads);
  WNW_CHECK_ARG(head_dim == 64 || head_dim == 128 || head_dim == 256, "head_dim must be 64, 128 or 256");
  WNW_CHECK_ARG(dtype == WNW_F32 || dtype == WNW_F16 || dtype == WNW_BF16, "bad dtype %d", dtype);
  WNW_CHECK_ARG(q && k && seg_starts && seg_ends && audio_starts && audio_ends && accumulator && accum_offsets &&
                    workspace,
                "null pointer argument");
  WNW_CHECK_ARG(((uintptr_t)k % 16) == 0, "k must be 16-byte aligned");
  WNW_CHECK_ARG(max_audio > 0 && k_rows >= 0 && acc_len >= 0, "bad sizes");
  WNW_CHECK_ARG(workspace_bytes >= wnw_fused_score_workspace_bytes(n_samples, n_heads), "workspace too small");
  SegScoreParams sp;
  sp.q = q;
  sp.k = k;
  sp.seg_s = seg_starts;
  sp.seg_e = seg_ends;
  sp.audio_s = audio_starts;
  sp.audio_e = audio_ends;
  sp.acc_off = accum_offsets;
  sp.acc = accumulator;
  sp.part = (float*)workspace;
  sp.err = device_error_word();
  sp.k_rows = k_rows;
  sp.acc_len = acc_len;
  sp.S = (int32_t)n_samples;
  sp.nh = (int32_t)n_heads;
  sp.scale_log2 = scale * kLog2eS;
  hipStream_t st = (hipStream_t)stream;
  const dim3 grid((unsigned)score_slices(n_samples), (unsigned)n_samples);
  const bool known = with_type(dtype, head_dim, [&](auto t, auto d) {
    typedef decltype(t) T;
    constexpr int D = decltype(d)::value;
    hipLaunchKernelGGL((seg_score_kernel<T, D, false>), grid, dim3(kScoreThreads), 0, st, sp);
    hipLaunchKernelGGL((seg_score_kernel<T, D, true>), grid, dim3(kScoreThreads), 0, st, sp);
  });
  WNW_CHECK_HIP(known ? hipGetLastError() : hipErrorInvalidValue, "score launch");
  return WNW_OK;
}

// First-use set-up of this file's kernels on the current device (the runtime
// resolves a kernel the first time it is used: ~2 ms on MI355X); called by
// wnw_prepare_kernels.
namespace wnw {
void touch_score_kernels() {
  hipFuncAttributes a;
  (void)hipFuncGetAttributes(&a, (const void*)&logit_score_kernel<kLogitG>);
}
}  // namespace wnw
