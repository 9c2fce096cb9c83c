// Decode attention: the arguments and limits its kernels (decode_attn_kernels.h)
// and its host side (decode_attn.hip) share.
#pragma once

#include "wnw_common.h"

namespace wnw {

static constexpr int kMaxGroup = 16;
static constexpr int kMaxGroupS = 8;    // heads per group with q in LDS slots (streaming kernel)
static constexpr int kSplitWaves = 4;   // waves a workgroup's row range is cut into
static constexpr int kPrevLogits = 16;  // pairs per sample the deferred form takes (<= 8 KV heads)
static constexpr float kLog2e = 1.4426950408889634f;

static constexpr int kMaxWgs = 2048;  // workgroups per launch at most

// Two-level merge of long segments (streaming kernel): block partials, two per
// 16 workgroups, and an arrival counter each.  They lie just before the
// partials and counters of the segments, at distances that depend on G and D
// alone, so a kernel finds them without arguments of their own.
static constexpr int kPiecesPerBlock = 16;
static constexpr int kMaxBlocks = 2 * (kMaxWgs / kPiecesPerBlock + 1);
__host__ __device__ constexpr int64_t up256(int64_t x) { return (x + 255) / 256 * 256; }
__host__ __device__ constexpr int64_t blk_counter_bytes() { return up256(kMaxBlocks * 4); }
__host__ __device__ constexpr int64_t blk_ml_bytes(int64_t G) { return up256(kMaxBlocks * G * 2 * 4); }
__host__ __device__ constexpr int64_t blk_acc_bytes(int64_t GD) { return up256(kMaxBlocks * GD * 4); }

struct AttnParams {
  const void* q;        // [n_seg, G, D]
  const void* k;        // [phys_rows, D]
  const void* v;        // [phys_rows, D]
  const int32_t* cu;    // [n_seg + 1] logical offsets (before the append, with APPEND)
  const int64_t* base;  // [n_seg] physical first row, or null (= cu)
  void* out;            // [n_seg, G, D]
  float* part_acc;      // [slots, G, D]
  float* part_ml;       // [slots, G, 2]
  int32_t* counters;    // [n_seg]
  float* lse;           // [n_seg, G, 2] final (max, sum) of each softmax, log2 domain, or null
  int32_t* err;
  uint64_t split_inv;  // ceil(2^64 / (gridDim.x * kSplitWaves)): range bounds without a division
  int64_t phys_rows;   // rows of k / v (bounds)
  int32_t n_seg;
  int32_t G;
  float scale_log2;  // scale * log2(e)
  // Streaming kernel only, null otherwise: the scaled logits (log2 domain)
  // of the audio rows of the segments whose KV head is flagged, for the
  // class-A scoring pass: xlog[(s * G + g) * max_audio + t] for audio row t
  // (relative to audio_s[s / Hkv]) of segment s, t < max_audio.
  float* xlog;
  const int32_t* xmask;    // [Hkv] non-zero: KV head scored
  const int32_t* audio_s;  // [n_seg / Hkv] audio range of each sample, relative to its segments' starts
  const int32_t* audio_e;
  int64_t max_audio;
  int32_t Hkv;
  // APPEND only: the step's rows, the post-append offsets and the capacity
  // of each segment (rows from base[s] it may occupy)
  const void* new_k;   // [n_seg, D]
  const void* new_v;
  int32_t* cu_out;     // [n_seg + 1], must not alias cu
  const int32_t* cap;  // [n_seg]
  // Streaming kernel, direct table only, null otherwise: a previous launch's
  // kept logits (pv_xlog) and normalisers (pv_lse), scored into the class-A
  // accumulator by this launch (AttnPrevScore); audio_s / audio_e /
  // max_audio / Hkv above describe both launches.  Workgroup i takes the
  // 256 tokens of slice i = (sample, block of 256 audio tokens).
  const float* pv_xlog;
  const float* pv_lse;
  uint64_t pv_kvlist;  // the KV heads that launch scored, ascending, 8 bits each (pv_nkv of them)
  int32_t pv_nkv;
  const int32_t* pv_cu;
  const int64_t* pv_base;
  int64_t pv_kv_rows;
  float* pv_acc;
  const int32_t* pv_acc_off;
  int64_t pv_acc_len;
  int32_t pv_nblk;  // 256-token blocks per sample
  int32_t pv_slices;  // samples x pv_nblk (<= the grid)
};

// Launches kernel WNW_ATTN_{MFMA,VALU,STREAM} for element type T.
template <typename T>
hipError_t launch_attn_d(int kernel, int64_t D, const AttnParams& ap, int64_t n_wg, hipStream_t st);

}  // namespace wnw
