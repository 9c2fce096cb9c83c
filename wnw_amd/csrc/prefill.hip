// Prompt kernels of the session's prefill branch (gfx950): causal attention
// of a whole prompt, and the token scores that prune it.
//
// Reference: src/algorithms/wnw/code/session.py:50-74 (SDPA with the model's
// mask, causal when there is none) and :119-170 (class-A scores of the last
// prompt token; per KV head the last token's or the mean of the text's
// softmax weights over the audio rows).
#include <math.h>

#include <algorithm>
#include <type_traits>

#include "wnw_dot.h"

namespace wnw {

typedef float f32x16 __attribute__((ext_vector_type(16)));
static constexpr float kLog2eP = 1.4426950408889634f;

template <typename T>
struct PromptOps;
template <>
struct PromptOps<bf16_t> {
  typedef __bf16 v4 __attribute__((ext_vector_type(4)));
  __device__ static f32x16 mma32(const u32x4& a, const u32x4& b, const f32x16& c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                   0, 0);
  }
  __device__ static uint64_t read_tr(const uint8_t* lds) {
    return __builtin_bit_cast(uint64_t,
                              __builtin_amdgcn_ds_read_tr16_b64_v4bf16((__attribute__((address_space(3))) v4*)lds));
  }
  // two values, round to nearest even
  __device__ static uint32_t pack2(float a, float b) {
    typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
    typedef float f2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f2){a, b}, bf2));
  }
};
template <>
struct PromptOps<f16_t> {
  typedef __fp16 h4 __attribute__((__vector_size__(4 * sizeof(__fp16))));
  __device__ static f32x16 mma32(const u32x4& a, const u32x4& b, const f32x16& c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0,
                                                  0);
  }
  __device__ static uint64_t read_tr(const uint8_t* lds) {
    return __builtin_bit_cast(uint64_t,
                              __builtin_amdgcn_ds_read_tr16_b64_v4f16((__attribute__((address_space(3))) h4*)lds));
  }
  __device__ static uint32_t pack2(float a, float b) { return f32_to_f16_bits(a) | (f32_to_f16_bits(b) << 16); }
};
// ---------------------------------------------------------------------------
// causal attention of a prompt (bf16 / f16, head_dim 64 or 128)
// ---------------------------------------------------------------------------
// A workgroup takes 128 queries of one head, a wave 32 of them, and walks the
// 64-key tiles up to its diagonal through two LDS buffers (the next tile's
// copies, direct global->LDS, are in flight while a tile is used; one barrier
// per tile).  Per wave and tile:
//   S^T (64 keys x 32 queries) = K x Q^T: 2 x D/16 v_mfma_f32_32x32x16, Q in
//       registers, K rows from LDS (16-byte chunks XOR-swizzled by the row);
//   O^T (D x 32) += V^T x P^T: D/32 x 4 of the same; lane (hi, n) of S^T holds
//       keys 8 j + 4 hi + 0..3 of query n, which is already the P^T operand
//       when V^T's k-slots follow the same order: two ds_read_b64_tr_b16 per
//       operand (4 keys x 1 column per lane each; V chunks swizzled by 2 (row % 4)).
// Online softmax in-lane (queries are columns) against the running maximum: the
// sums are rescaled in the tiles where some query's maximum grew (with 32
// queries per wave most of the first 50).  A row's largest weight is then 1,
// exact in 16 bits; against a reference that trails the maximum by up to 2^8 it
// would be rounded beside a sum that is not (178 us instead of 187, error
// against 64 bits 3 % larger at a standard deviation of the scores of 1, 16 %
// at 2, 20 % at 4).  Only the diagonal tile masks, and only the last tile clamps
// its rows.  P goes through 16 bits, its sum stays 32-bit.
// Bound by the issue of vector instructions (exponentials above all) beside
// the matrix instructions: two waves per SIMD overlap them only in part.
// bf16, D = 128, 32 heads: 4,564 rows 588 us (SDPA's flash kernel, 290 TFLOP/s) ->
// 187 us (914; 202 with a mask in every tile and the copies' offsets worked out
// per tile), 2 x 28 heads of 2,000 rows 85 -> 73 us; SDPA's error against 64 bits
// to four digits.  Measured and not kept: 64 queries per wave and one wave per
// SIMD (306 us: sums move through accumulator registers), the next tile's
// scores issued ahead of a tile's softmax (189-190 against 194 us, more
// registers), the first values of a tile read ahead of its softmax (the same).
struct PromptAttnParams {
  const void *q, *k, *v;
  void* out;
  int64_t qb, qh, qs, kb, kh, ks, vb, vh, vs, ob, oh, os;  // strides in elements; head_dim is contiguous
  int32_t Hq, G, S, BH, nqb;
  float scale_log2;
};

static constexpr int kPaQ = 128;   // queries per workgroup
static constexpr int kPaKeys = 64;  // keys per tile

// 16 bytes per lane from gbase + voff into LDS at lds_addr + 16 * lane (M0
// carries the LDS address and is restored).  One wait state between M0's write
// and the load, five between a vector instruction's write of the base and the
// load, the two moves among them.
__device__ __forceinline__ void prompt_copy16(const void* gbase, uint32_t voff, uint32_t lds_addr) {
  uint32_t save;
  asm volatile(
      "s_mov_b32 %0, m0\n\t"
      "s_mov_b32 m0, %3\n\t"
      "s_nop 2\n\t"
      "global_load_lds_dwordx4 %1, %2\n\t"
      "s_mov_b32 m0, %0"
      : "=&s"(save)
      : "v"(voff), "s"(gbase), "s"(lds_addr)
      : "memory");
}
__device__ __forceinline__ const void* uniform_ptr(const void* p) {
  const uint64_t x = (uint64_t)(uintptr_t)p;
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)x), hi = __builtin_amdgcn_readfirstlane((uint32_t)(x >> 32));
  return (const void*)(uintptr_t)(((uint64_t)hi << 32) | lo);
}

template <typename T, int D>
__global__ __launch_bounds__(256, 2) void prefill_attn_kernel(PromptAttnParams p) {
  using Ops = PromptOps<T>;
  constexpr int RB = D * 2, CH = RB / 16, TB = kPaKeys * RB;
  constexpr int KK = D / 16, DT = D / 32;
  constexpr int NI = TB / 1024 / 4;  // 1 KB copies per wave and tensor
  constexpr int RPI = 1024 / RB;     // rows per copy
  __shared__ __attribute__((aligned(16))) uint8_t lds[2][2 * TB];
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hi = lane >> 5, n = lane & 31;
  // heavy query blocks first; the blocks of one head share its K and V in the
  // L2 of one XCD when the head count is a multiple of 8
  const int bh = blockIdx.x % p.BH, qblk = p.nqb - 1 - blockIdx.x / p.BH;
  const int b = bh / p.Hq, h = bh - b * p.Hq, hk = h / p.G;
  const int S = p.S;
  const int q0 = qblk * kPaQ + 32 * w, qi = q0 + n;
  const T* kp = (const T*)p.k + b * p.kb + hk * p.kh;
  const T* vp = (const T*)p.v + b * p.vb + hk * p.vh;
  u32x4 qr[KK];
  {
    const T* qp = (const T*)p.q + b * p.qb + h * p.qh + (int64_t)min(qi, S - 1) * p.qs + 8 * hi;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) qr[kk] = *gptr<u32x4>(qp + 16 * kk);
  }
  const uint32_t lds0 =
      __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)lds);
  // lane offsets of a tile's copies: those of a whole tile, until the last one clamps its rows
  uint32_t kdma[NI], vdma[NI];
  auto copy_offsets = [&](int last) {
#pragma unroll
    for (int u = 0; u < NI; ++u) {
      const int r = (w * NI + u) * RPI + lane / CH;
      const int rr = min(r, last), c = lane % CH;
      kdma[u] = (uint32_t)(rr * (int)p.ks * 2 + (c ^ (r % CH)) * 16);
      vdma[u] = (uint32_t)(rr * (int)p.vs * 2 + (c ^ (2 * (r & 3))) * 16);
    }
  };
  copy_offsets(kPaKeys - 1);
  auto issue = [&](int tile, int buf) {  // tiles in ascending order
    const int key0 = tile * kPaKeys;
    const void* kt = uniform_ptr(kp + (int64_t)key0 * p.ks);
    const void* vt = uniform_ptr(vp + (int64_t)key0 * p.vs);
    const uint32_t dst = lds0 + buf * 2 * TB;
    // rows past the prompt repeat its last (masked: later than every query)
    if (key0 + kPaKeys > S) copy_offsets(S - 1 - key0);
#pragma unroll
    for (int u = 0; u < NI; ++u) {
      prompt_copy16(kt, kdma[u], dst + (w * NI + u) * 1024);
      prompt_copy16(vt, vdma[u], dst + TB + (w * NI + u) * 1024);
    }
  };
  // lane offsets of the operands inside a tile
  uint32_t koff[KK], voff[DT];
#pragma unroll
  for (int kk = 0; kk < KK; ++kk) koff[kk] = n * RB + (((2 * kk + hi) ^ (n % CH)) * 16);
  {
    const int lc = lane & 15, dsub = (lane >> 4) & 1;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
      voff[dt] = (4 * hi + (lc >> 2)) * RB + (((4 * dt + 2 * dsub + ((lc & 3) >> 1)) ^ (2 * (lc >> 2))) * 16) +
                 (lc & 1) * 8;
  }
  f32x16 o[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) o[dt] = f32x16{};
  // the running maximum starts below every score (a fully masked value is -inf)
  float m = -3.402823466e38f, l = 0.f;
  const int ntile = min((qblk + 1) * (kPaQ / kPaKeys), (S + kPaKeys - 1) / kPaKeys);
  const int mine = min((q0 + 31) / kPaKeys, ntile - 1);  // the wave's diagonal tile
  auto tile = [&](int i, auto masked) {
    const uint8_t* kt = lds[i & 1];
    const uint8_t* vt = kt + TB;
    f32x16 s[2];
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) s[mt] = f32x16{};
#pragma unroll
    for (int kk = 0; kk < KK; ++kk)
#pragma unroll
      for (int mt = 0; mt < 2; ++mt) s[mt] = Ops::mma32(*(const u32x4*)(kt + koff[kk] + mt * 32 * RB), qr[kk], s[mt]);
    if constexpr (decltype(masked)::value) {
      const int lim = qi - i * kPaKeys - 4 * hi;  // keys 32 mt + 8 j + c (+ 4 hi) up to the query
#pragma unroll
      for (int mt = 0; mt < 2; ++mt)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (32 * mt + 8 * (r >> 2) + (r & 3) > lim) s[mt][r] = -INFINITY;
    }
    float mx = m;
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
      for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[mt][r]);
    mx = max_x32(mx);
    if (__ballot(mx > m)) {
      const float alpha = __builtin_amdgcn_exp2f((m - mx) * p.scale_log2);
      l *= alpha;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) o[dt] *= alpha;
      m = mx;
    }
    const float mc = m * p.scale_log2;
    u32x4 pb[4];
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float x0 = __builtin_amdgcn_exp2f(fmaf(s[kk >> 1][8 * (kk & 1) + 2 * j], p.scale_log2, -mc));
        const float x1 = __builtin_amdgcn_exp2f(fmaf(s[kk >> 1][8 * (kk & 1) + 2 * j + 1], p.scale_log2, -mc));
        l += x0 + x1;
        pb[kk][j] = Ops::pack2(x0, x1);
      }
    }
    // the rows past the prompt repeat its last one: their weights are 0, and V
    // is made 0 too (an infinity there would give NaN with them)
    uint64_t vm[4][2];
    const int end = p.S - i * kPaKeys;  // keys of the prompt in this tile
    bool cut = false;
    if constexpr (decltype(masked)::value) {
      cut = end < kPaKeys;
      if (cut)
#pragma unroll
        for (int kk = 0; kk < 4; ++kk)
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            const int left = end - (16 * kk + 8 * j + 4 * hi);  // of the lane's 4 keys
            vm[kk][j] = left <= 0 ? 0 : left >= 4 ? ~0ull : (1ull << (16 * left)) - 1;
          }
    }
    __builtin_amdgcn_s_setprio(1);  // a wave at its products before another's softmax: 185 -> 183 us
#pragma unroll
    for (int kk = 0; kk < 4; ++kk)
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        uint64_t v0 = Ops::read_tr(vt + voff[dt] + 16 * kk * RB);
        uint64_t v1 = Ops::read_tr(vt + voff[dt] + (16 * kk + 8) * RB);
        if (cut) {
          v0 &= vm[kk][0];
          v1 &= vm[kk][1];
        }
        const u32x4 a = u32x4{(uint32_t)v0, (uint32_t)(v0 >> 32), (uint32_t)v1, (uint32_t)(v1 >> 32)};
        o[dt] = Ops::mma32(a, pb[kk], o[dt]);
      }
    __builtin_amdgcn_s_setprio(0);
  };
  auto turn = [&](int i) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();  // tile i has landed; everyone is done with tile i - 1
    if (i + 1 < ntile) issue(i + 1, (i + 1) & 1);
  };
  issue(0, 0);
  // the tiles up to the wave's diagonal, the diagonal one, the turns of the
  // workgroup's later waves
  for (int i = 0; i < mine; ++i) {
    turn(i);
    tile(i, std::false_type());
  }
  turn(mine);
  tile(mine, std::true_type());
  for (int i = mine + 1; i < ntile; ++i) turn(i);
  if (qi >= S) return;
  const float inv = 1.f / sum_x32(l);
  T* op = (T*)p.out + b * p.ob + h * p.oh + (int64_t)qi * p.os;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
      const float x[4] = {o[dt][4 * j] * inv, o[dt][4 * j + 1] * inv, o[dt][4 * j + 2] * inv, o[dt][4 * j + 3] * inv};
      *(WNW_GLOBAL u32x2_t*)(op + 32 * dt + 8 * j + 4 * hi) = u32x2_t{Ops::pack2(x[0], x[1]), Ops::pack2(x[2], x[3])};
    }
}

// ---------------------------------------------------------------------------
// prompt token scores
// ---------------------------------------------------------------------------
// An item is one score row of one sample: softmax weights over all keys of one
// KV head, summed over a list of queries (class A: the last row of the layer's
// class-A heads; a KV head: its group's heads, the last row or every row
// after the audio) and divided by the rows per head, at the audio keys.
//
// Two launches over (key slice, item, sample): the slice's (max, sum) of every
// query, then with every query's statistics merged the slice's weights summed
// over the queries.  A wave keeps its keys' rows in registers (tiles of 16
// keys as matrix operands) and streams the queries past them, 16 per matrix
// tile, so K is read once per launch.  Latency bound (a few MB): the torch form
// it replaces was ~10 launches per KV head plus an S x S mask, ~500 us a layer
// at 4,564 rows of 8 KV heads (50 text rows); now 13.5 + 15.3 us.  Logits are
// 32-bit sums of exact 16-bit products (that form rounded them to 16 bits twice);
// fp32 dots are added as trees of chains of 8, no less exact than that form's
// library products (as one chain 2-3 times their error for the last row; 4,564
// rows 56 -> 67 us with the torch calls around the launches, 300 text rows of
// 28 heads of 64 380 -> 520 us).
static constexpr int kPsThreads = 256;
static constexpr int kPsMax = 64;       // KV heads, class-A heads and samples a launch describes
static constexpr int kPsQueries = 512;  // queries whose statistics sit in LDS at a time

struct PromptScoreParams {
  const void *q, *k, *mask;
  int64_t qb, qh, qs, kb, kh, ks, mb, ms;  // strides in elements
  float* out_a;       // [B, max_audio]
  float* out_h;       // [B, n_kv, max_audio]
  float* part;        // [B, items, slices, max_queries, 2]
  int32_t S, G, n_a, n_kv, a_kv, last, max_audio, max_queries, mask_dtype;
  float scale;
  uint16_t a_heads[kPsMax];  // class-A query heads
  uint16_t kv[kPsMax];       // KV heads scored
  int32_t ra[kPsMax], re[kPsMax];
};

// Keys of one workgroup: 4 waves x tiles of 16, as many tiles as fit 64
// registers of row chunks.
template <typename T, int D>
struct PromptScoreGeom {
  static constexpr int NC = D * (int)sizeof(T) / 64;  // 16-byte chunks of a row per lane
  static constexpr int KT = NC <= 4 ? 4 : NC == 8 ? 2 : 1;
  static constexpr int kKeys = 4 * 16 * KT;
};

__device__ __forceinline__ float mask_at(const void* m, int64_t i, int dtype) {
  if (dtype == WNW_F32) return gptr<float>(m)[i];
  const uint32_t h = gptr<uint16_t>(m)[i];
  return dtype == WNW_BF16 ? __uint_as_float(h << 16) : f16_bits_to_f32(h);
}

template <typename T, int D, bool SUM>
__global__ __launch_bounds__(kPsThreads) void prompt_score_kernel(PromptScoreParams p) {
  using Ge = PromptScoreGeom<T, D>;
  constexpr int NC = Ge::NC, KT = Ge::KT, EPC = 16 / (int)sizeof(T);
  constexpr float kLowest = -3.402823466e38f;
  __shared__ float st[SUM ? 1 : 4][kPsQueries][2];
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lq = lane >> 4, lc = lane & 15;
  const int slice = blockIdx.x, nsl = gridDim.x, item = blockIdx.y, b = blockIdx.z;
  const bool cls_a = p.n_a > 0 && item == gridDim.y - 1;
  // the lists, indexed at run time, are read where the arguments lie (an
  // index into p itself would copy all of it to scratch memory first)
  const auto* lists = (const __attribute__((address_space(4))) PromptScoreParams*)__builtin_amdgcn_kernarg_segment_ptr();
  const int ra = lists->ra[b], re = lists->re[b], S = p.S;
  const int rows = cls_a || p.last ? 1 : S - re;  // query rows per head
  const int row0 = cls_a || p.last ? S - 1 : re;
  const int nq = (cls_a ? p.n_a : p.G) * rows;
  const int kvh = cls_a ? p.a_kv : lists->kv[item];
  const int key0 = slice * Ge::kKeys + w * 16 * KT;  // this wave's keys
  const T* kp = (const T*)p.k + b * p.kb + kvh * p.kh;
  const T* qp = (const T*)p.q + b * p.qb;
  u32x4 kr[KT][NC];
#pragma unroll
  for (int t = 0; t < KT; ++t) {
    const T* r = kp + (int64_t)min(key0 + 16 * t + lc, S - 1) * p.ks;
#pragma unroll
    for (int n = 0; n < NC; ++n) kr[t][n] = *gptr<u32x4>(r + (4 * n + lq) * EPC);
  }
  f32x4 acc[KT];
#pragma unroll
  for (int t = 0; t < KT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  float* part = p.part + (((int64_t)b * gridDim.y + item) * nsl) * p.max_queries * 2;
  for (int c0 = 0; c0 < nq; c0 += kPsQueries) {
    const int cn = min(kPsQueries, nq - c0);
    if constexpr (SUM) {  // every slice's statistics of this chunk's queries: (max, 1 / sum)
      __syncthreads();
      for (int x = tid; x < cn; x += kPsThreads) {
        float M = kLowest, L = 0.f;
        for (int s0 = 0; s0 < nsl; s0 += 8) {
          float ms[8], ls[8];
#pragma unroll
          for (int u = 0; u < 8; ++u) {
            const WNW_GLOBAL float* e = gptr<float>(part) + ((int64_t)min(s0 + u, nsl - 1) * p.max_queries + c0 + x) * 2;
            ms[u] = e[0];
            ls[u] = s0 + u < nsl ? e[1] : 0.f;
          }
          float Mn = M;
#pragma unroll
          for (int u = 0; u < 8; ++u) Mn = fmaxf(Mn, ms[u]);
          L *= __builtin_amdgcn_exp2f((M - Mn) * kLog2eP);
#pragma unroll
          for (int u = 0; u < 8; ++u) L += ls[u] * __builtin_amdgcn_exp2f((ms[u] - Mn) * kLog2eP);
          M = Mn;
        }
        st[0][x][0] = M;
        st[0][x][1] = 1.f / L;
      }
      __syncthreads();
    }
    u32x4 qn[NC];
    int row_n = 0;
    auto load_q = [&](int x0) {  // this lane's query of tile x0 (the last one again past the end)
      const int qi = c0 + min(x0 + lc, cn - 1);
      const int g = qi / rows;
      row_n = row0 + qi - g * rows;
      const int head = cls_a ? lists->a_heads[g] : kvh * p.G + g;
      const T* qr = qp + head * p.qh + (int64_t)row_n * p.qs;
#pragma unroll
      for (int n = 0; n < NC; ++n) qn[n] = *gptr<u32x4>(qr + (4 * n + lq) * EPC);
    };
    load_q(0);
    for (int x0 = 0; x0 < cn; x0 += 16) {
      const int x = min(x0 + lc, cn - 1), row = row_n;
      u32x4 qc[NC];
#pragma unroll
      for (int n = 0; n < NC; ++n) qc[n] = qn[n];
      if (x0 + 16 < cn) load_q(x0 + 16);  // in flight during this tile's products
      f32x4 v[KT];
#pragma unroll
      for (int t = 0; t < KT; ++t) {
        v[t] = dot_rows<T, NC, sizeof(T) == 4 ? 2 : NC>(kr[t], qc) * p.scale;
      }
      if (p.mask) {  // wave-uniform, as the tests below
#pragma unroll
        for (int t = 0; t < KT; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            v[t][i] += mask_at(p.mask, b * p.mb + row * p.ms + min(key0 + 16 * t + 4 * lq + i, S - 1), p.mask_dtype);
      }
      if (key0 + 16 * KT > (p.mask ? S : row0)) {  // the causal limit (the last row is S - 1 at most), the prompt's end
        const int lim = p.mask ? S - 1 : row;
#pragma unroll
        for (int t = 0; t < KT; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (key0 + 16 * t + 4 * lq + i > lim) v[t][i] = -INFINITY;
      }
      if constexpr (SUM) {
        const float m = st[0][x][0], inv = x0 + lc < cn ? st[0][x][1] : 0.f;
#pragma unroll
        for (int t = 0; t < KT; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[t][i] += __builtin_amdgcn_exp2f((v[t][i] - m) * kLog2eP) * inv;
      } else {
        float mx = kLowest;
#pragma unroll
        for (int t = 0; t < KT; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i) mx = fmaxf(mx, v[t][i]);
        mx = max_x32(max_x16(mx));
        float l = 0.f;
#pragma unroll
        for (int t = 0; t < KT; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i) l += __builtin_amdgcn_exp2f((v[t][i] - mx) * kLog2eP);
        l = sum_x32(sum_x16(l));
        if (lq == 0 && x0 + lc < cn) {
          st[w][x][0] = mx;
          st[w][x][1] = l;
        }
      }
    }
    if constexpr (!SUM) {
      __syncthreads();
      for (int x = tid; x < cn; x += kPsThreads) {
        float M = kLowest, L = 0.f;
#pragma unroll
        for (int u = 0; u < 4; ++u) M = fmaxf(M, st[u][x][0]);
#pragma unroll
        for (int u = 0; u < 4; ++u) L += st[u][x][1] * __builtin_amdgcn_exp2f((st[u][x][0] - M) * kLog2eP);
        WNW_GLOBAL float* e = gptr_w<float>(part) + ((int64_t)slice * p.max_queries + c0 + x) * 2;
        e[0] = M;
        e[1] = L;
      }
      __syncthreads();
    }
  }
  if constexpr (SUM) {
    float* out = cls_a ? p.out_a + (int64_t)b * p.max_audio : p.out_h + ((int64_t)b * p.n_kv + item) * p.max_audio;
    const float per = 1.f / (float)max(rows, 1);
#pragma unroll
    for (int t = 0; t < KT; ++t) {
      f32x4 sum = acc[t];
#pragma unroll
      for (int o = 8; o >= 1; o >>= 1)
#pragma unroll
        for (int i = 0; i < 4; ++i) sum[i] += __shfl_xor(sum[i], o);
      const float lo = lc & 1 ? sum[1] : sum[0], hi = lc & 1 ? sum[3] : sum[2];
      const float mine = lc & 2 ? hi : lo;
      const int key = key0 + 16 * t + 4 * lq + lc;
      if (lc < 4 && key >= ra && key < re) gptr_w<float>(out)[key - ra] = mine * per;
    }
  }
}

}  // namespace wnw

using namespace wnw;

extern "C" int wnw_prefill_attn(const void* q, const void* k, const void* v, int64_t batch, int64_t n_heads,
                                int64_t n_kv_heads, int64_t seq, int64_t head_dim, const int64_t* strides, float scale,
                                int dtype, void* out, void* stream) {
  WNW_CHECK_ARG(batch >= 0 && n_heads >= 0 && seq >= 0 && n_kv_heads >= 1 && n_heads % n_kv_heads == 0,
                "bad prompt geometry: batch %lld, heads %lld / %lld, rows %lld", (long long)batch, (long long)n_heads,
                (long long)n_kv_heads, (long long)seq);
  if (batch == 0 || n_heads == 0 || seq == 0) return WNW_OK;
  WNW_CHECK_ARG(q && k && v && out && strides, "null pointer argument");
  if (!((dtype == WNW_BF16 || dtype == WNW_F16) && (head_dim == 64 || head_dim == 128) && scale > 0.f)) {
    set_error("the prompt attention takes bf16/f16, head_dim 64 or 128 and a positive scale");
    return WNW_ENOTSUP;
  }
  const void* ptrs[4] = {q, k, v, out};
  for (int t = 0; t < 4; ++t) {
    WNW_CHECK_ARG(((uintptr_t)ptrs[t] % 16) == 0, "q, k, v and out must be 16-byte aligned");
    for (int i = 0; i < 3; ++i)
      WNW_CHECK_ARG(strides[3 * t + i] >= 0 && strides[3 * t + i] % 8 == 0, "strides must be multiples of 16 bytes");
    WNW_CHECK_ARG(strides[3 * t + 2] <= (1ll << 22), "row stride too large");  // a tile's offsets fit 32 bits
  }
  WNW_CHECK_ARG(seq < (1ll << 30), "prompt too long");
  PromptAttnParams p;
  p.q = q;
  p.k = k;
  p.v = v;
  p.out = out;
  p.qb = strides[0], p.qh = strides[1], p.qs = strides[2];
  p.kb = strides[3], p.kh = strides[4], p.ks = strides[5];
  p.vb = strides[6], p.vh = strides[7], p.vs = strides[8];
  p.ob = strides[9], p.oh = strides[10], p.os = strides[11];
  p.Hq = (int32_t)n_heads;
  p.G = (int32_t)(n_heads / n_kv_heads);
  p.S = (int32_t)seq;
  const int64_t bh = batch * n_heads, nqb = (seq + kPaQ - 1) / kPaQ;
  WNW_CHECK_ARG(bh * nqb < (1ll << 31), "too many query blocks");
  p.BH = (int32_t)bh;
  p.nqb = (int32_t)nqb;
  p.scale_log2 = scale * kLog2eP;
  const dim3 grid((unsigned)(bh * nqb));
  hipStream_t st = (hipStream_t)stream;
  if (dtype == WNW_BF16) {
    if (head_dim == 128)
      hipLaunchKernelGGL((prefill_attn_kernel<bf16_t, 128>), grid, dim3(256), 0, st, p);
    else
      hipLaunchKernelGGL((prefill_attn_kernel<bf16_t, 64>), grid, dim3(256), 0, st, p);
  } else {
    if (head_dim == 128)
      hipLaunchKernelGGL((prefill_attn_kernel<f16_t, 128>), grid, dim3(256), 0, st, p);
    else
      hipLaunchKernelGGL((prefill_attn_kernel<f16_t, 64>), grid, dim3(256), 0, st, p);
  }
  WNW_CHECK_HIP(hipGetLastError(), "prompt attention launch");
  return WNW_OK;
}

namespace wnw {
// Calls f with a T and the head_dim as compile-time constants; false for a
// type or head_dim without an instance.
template <typename F, typename T>
static bool prompt_dim(int64_t D, F f, T t) {
  switch (D) {
    case 64: return f(t, std::integral_constant<int, 64>()), true;
    case 128: return f(t, std::integral_constant<int, 128>()), true;
    case 256: return f(t, std::integral_constant<int, 256>()), true;
  }
  return false;
}
template <typename F>
static bool prompt_type(int dtype, int64_t D, F f) {
  switch (dtype) {
    case WNW_BF16: return prompt_dim(D, f, bf16_t());
    case WNW_F16: return prompt_dim(D, f, f16_t());
    case WNW_F32: return prompt_dim(D, f, float());
  }
  return false;
}

static int64_t prompt_slices(int64_t seq, int64_t head_dim, int dtype) {
  int64_t keys = 0;
  if (!prompt_type(dtype, head_dim, [&](auto t, auto d) { keys = PromptScoreGeom<decltype(t), decltype(d)::value>::kKeys; }))
    return -1;
  return (seq + keys - 1) / keys;
}
}  // namespace wnw

extern "C" int64_t wnw_prefill_scores_workspace_bytes(int64_t batch, int64_t n_items, int64_t seq, int64_t head_dim,
                                                      int64_t max_queries, int dtype) {
  const int64_t sl = prompt_slices(seq, head_dim, dtype);
  if (batch < 0 || n_items < 0 || seq < 0 || max_queries < 0 || sl < 0) return -1;
  return std::max<int64_t>(256, batch * n_items * sl * max_queries * 8);
}

extern "C" int wnw_prefill_scores(const void* q, const void* k, const void* mask, const int64_t* strides, int64_t batch,
                                  int64_t n_heads, int64_t n_kv_heads, int64_t seq, int64_t head_dim,
                                  const int32_t* audio_starts,
                                  const int32_t* audio_ends, const int32_t* a_heads, int64_t n_a,
                                  const int32_t* kv_heads, int64_t n_kv, int last_row, float scale, int dtype,
                                  int mask_dtype, int64_t max_audio, int64_t max_queries, float* out_a, float* out_h,
                                  void* workspace, int64_t workspace_bytes, void* stream) {
  const int64_t items = n_kv + (n_a > 0 ? 1 : 0), nsl = prompt_slices(seq, head_dim, dtype);
  if (batch > kPsMax || n_a > kPsMax || n_kv > kPsMax || nsl < 0) {
    set_error("the prompt scores take up to %d samples, class-A heads and KV heads, head_dim 64, 128 or 256", kPsMax);
    return WNW_ENOTSUP;
  }
  WNW_CHECK_ARG(batch >= 0 && seq >= 0 && seq < (1ll << 30) && n_a >= 0 && n_kv >= 0 && max_audio >= 0 &&
                    max_queries >= 0 && max_queries < (1ll << 31),
                "bad prompt score geometry");
  WNW_CHECK_ARG(n_kv_heads >= 1 && n_heads >= 1 && n_heads % n_kv_heads == 0 && n_heads <= 65536,
                "bad head counts %lld / %lld", (long long)n_heads, (long long)n_kv_heads);
  const int64_t group = n_heads / n_kv_heads;
  if (batch == 0 || items == 0 || seq == 0 || max_audio == 0) return WNW_OK;
  WNW_CHECK_ARG(q && k && strides && audio_starts && audio_ends && workspace && (n_a == 0 || (a_heads && out_a)) &&
                    (n_kv == 0 || (kv_heads && out_h)),
                "null pointer argument");
  WNW_CHECK_ARG(mask_dtype == WNW_F32 || mask_dtype == WNW_F16 || mask_dtype == WNW_BF16, "bad mask dtype %d",
                mask_dtype);
  const int64_t per = 16 / elem_bytes(dtype);
  for (int i = 0; i < 6; ++i)
    WNW_CHECK_ARG(strides[i] >= 0 && strides[i] % per == 0, "q and k strides must be multiples of 16 bytes");
  WNW_CHECK_ARG(!mask || (strides[6] >= 0 && strides[7] >= 0), "negative mask stride");
  for (int64_t i = 0; i < n_a; ++i)
    WNW_CHECK_ARG(a_heads[i] >= 0 && a_heads[i] < n_heads, "class-A head %d is not one of %lld", a_heads[i],
                  (long long)n_heads);
  for (int64_t i = 0; i < n_kv; ++i)
    WNW_CHECK_ARG(kv_heads[i] >= 0 && kv_heads[i] < n_kv_heads, "KV head %d is not one of %lld", kv_heads[i],
                  (long long)n_kv_heads);
  WNW_CHECK_ARG(((uintptr_t)q % 16) == 0 && ((uintptr_t)k % 16) == 0, "q and k must be 16-byte aligned");
  WNW_CHECK_ARG(workspace_bytes >= wnw_prefill_scores_workspace_bytes(batch, items, seq, head_dim, max_queries, dtype),
                "workspace too small");
  PromptScoreParams p;
  p.q = q;
  p.k = k;
  p.mask = mask;
  p.qb = strides[0], p.qh = strides[1], p.qs = strides[2];
  p.kb = strides[3], p.kh = strides[4], p.ks = strides[5];
  p.mb = strides[6], p.ms = strides[7];
  p.out_a = out_a;
  p.out_h = out_h;
  p.part = (float*)workspace;
  p.S = (int32_t)seq;
  p.G = (int32_t)group;
  p.n_a = (int32_t)n_a;
  p.n_kv = (int32_t)n_kv;
  p.a_kv = n_a > 0 ? a_heads[0] / (int32_t)group : 0;
  p.last = last_row != 0;
  p.max_audio = (int32_t)max_audio;
  p.max_queries = (int32_t)max_queries;
  p.mask_dtype = mask_dtype;
  p.scale = scale;
  int64_t most = n_a;
  for (int64_t b = 0; b < batch; ++b) {
    p.ra[b] = audio_starts[b];
    p.re[b] = audio_ends[b];
    WNW_CHECK_ARG(p.ra[b] >= 0 && p.re[b] >= p.ra[b] && p.re[b] <= seq && p.re[b] - p.ra[b] <= max_audio,
                  "bad audio range [%d, %d) of sample %lld", p.ra[b], p.re[b], (long long)b);
    if (n_kv > 0) most = std::max<int64_t>(most, group * (last_row ? 1 : seq - p.re[b]));
  }
  WNW_CHECK_ARG(most <= max_queries, "max_queries %lld is less than the %lld of an item", (long long)max_queries,
                (long long)most);
  for (int64_t i = 0; i < n_a; ++i) p.a_heads[i] = (uint16_t)a_heads[i];
  for (int64_t i = 0; i < n_kv; ++i) p.kv[i] = (uint16_t)kv_heads[i];
  const dim3 grid((unsigned)nsl, (unsigned)items, (unsigned)batch);
  hipStream_t st = (hipStream_t)stream;
  prompt_type(dtype, head_dim, [&](auto t, auto d) {
    typedef decltype(t) T;
    constexpr int D = decltype(d)::value;
    hipLaunchKernelGGL((prompt_score_kernel<T, D, false>), grid, dim3(kPsThreads), 0, st, p);
    hipLaunchKernelGGL((prompt_score_kernel<T, D, true>), grid, dim3(kPsThreads), 0, st, p);
  });
  WNW_CHECK_HIP(hipGetLastError(), "prompt score launch");
  return WNW_OK;
}
