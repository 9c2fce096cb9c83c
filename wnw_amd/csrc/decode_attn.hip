// Host side of the split-K decode attention: the choice of kernel and grid,
// the workspace, and the C entry points.  The kernels are in
// decode_attn_kernels.h, compiled per element type.
#include <stdarg.h>
#include <stdio.h>

#include <algorithm>
#include <mutex>
#include <vector>

#include "decode_attn.h"

namespace wnw {

struct DeviceInfo {
  int cus = 0;
  int max_wg = 0;  // upper bound of workgroups per launch (sizes the workspace)
};

static DeviceInfo& device_info() {
  static std::mutex mu;
  static std::vector<DeviceInfo> infos;
  int dev = 0;
  (void)hipGetDevice(&dev);
  std::lock_guard<std::mutex> lock(mu);
  if ((int)infos.size() <= dev) infos.resize(dev + 1);
  DeviceInfo& di = infos[dev];
  if (di.cus == 0) {
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
      cus = 256;
    di.cus = cus;
    di.max_wg = std::min(cus * 8, kMaxWgs);
  }
  return di;
}

struct WsLayout {
  int64_t counters, ml, acc, total;
};
static int64_t blk_bytes(int64_t G, int64_t D) { return blk_counter_bytes() + blk_ml_bytes(G) + blk_acc_bytes(G * D); }

// Arrival counters of the block partials and of cap_seg segments first (their
// place depends on nothing but cap_seg: a launch with another group or
// head_dim finds them cleared), then the (m, l) pairs and the accumulators,
// each time the block partials' before those of `slots` partial slots.
static WsLayout make_layout(int64_t cap_seg, int64_t slots, int64_t G, int64_t D) {
  WsLayout L;
  L.counters = blk_counter_bytes();
  L.ml = L.counters + up256(cap_seg * 4) + blk_ml_bytes(G);
  L.acc = L.ml + up256(slots * G * 2 * 4) + blk_acc_bytes(G * D);
  L.total = L.acc + up256(slots * G * D * 4);
  return L;
}

// Caller-owned workspace: sized before the grid is known, so for the
// largest grid a launch may use.
static WsLayout ws_layout(int64_t n_seg, int64_t G, int64_t D) {
  return make_layout(n_seg, device_info().max_wg + n_seg, G, D);
}

// ---------------------------------------------------------------------------
// The library's own attention scratch (wnw_decode_attn_noalloc)
// ---------------------------------------------------------------------------
// A file-scope device array: each device holds its own copy, at its own
// address, for as long as the process lives.  Host code uses only the
// per-device address from hipGetSymbolAddress (resolved once per device,
// with that device current), never the array's name.  The counters region
// is sized for WNW_NOALLOC_MAX_SEG segments whatever a call's n_seg, so
// calls with different n_seg never turn partial bytes into counters; every
// launch leaves the counters of its segments at zero, the others are never
// touched, and the array is zero at load (cleared again on first use).
// WNW_NOALLOC_SCRATCH_BYTES bound a call's partials and segment counters; the
// block partials have room of their own (grids of up to kNoAllocWgs).
static constexpr int64_t kNoAllocWgs = 1024;
static constexpr int64_t kNoAllocBytes =
    WNW_NOALLOC_SCRATCH_BYTES + blk_counter_bytes() + blk_ml_bytes(kMaxGroup) + blk_acc_bytes(kMaxGroup * 256);
static __device__ __align__(256) uint8_t g_attn_scratch[kNoAllocBytes];

struct ScratchSlot {
  void* ptr = nullptr;
  bool cleared = false;
};

__global__ void fill_zero_kernel(uint32_t* p, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    p[i] = 0u;
}

}  // namespace wnw

using namespace wnw;

extern "C" int64_t wnw_decode_attn_workspace_bytes(int64_t n_seg, int64_t group, int64_t head_dim) {
  if (n_seg < 0 || group <= 0 || head_dim <= 0) return -1;
  return ws_layout(n_seg, group, head_dim).total;
}

extern "C" int wnw_workspace_init(void* workspace, int64_t workspace_bytes, void* stream) {
  WNW_CHECK_ARG(workspace != nullptr || workspace_bytes == 0, "workspace is null");
  WNW_CHECK_ARG(workspace_bytes % 4 == 0, "workspace_bytes must be a multiple of 4");
  if (workspace_bytes == 0) return WNW_OK;
  const int64_t n = workspace_bytes / 4;
  const int64_t blocks = std::min<int64_t>((n + 255) / 256, 4096);
  hipLaunchKernelGGL(fill_zero_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream,
                     (uint32_t*)workspace, n);
  WNW_CHECK_HIP(hipGetLastError(), "workspace init launch");
  return WNW_OK;
}

namespace wnw {
// The current device's scratch address (resolved once per device; the
// counters region is cleared with a fill kernel on the first call, which
// may be under graph capture, so no memset node is recorded).
static int noalloc_scratch(hipStream_t st, void** out) {
  static std::mutex mu;
  static std::vector<ScratchSlot> slots;
  int dev = 0;
  WNW_CHECK_HIP(hipGetDevice(&dev), "hipGetDevice");
  std::lock_guard<std::mutex> lock(mu);
  if ((int)slots.size() <= dev) slots.resize(dev + 1);
  ScratchSlot& sl = slots[dev];
  if (!sl.ptr) {
    void* p = nullptr;
    WNW_CHECK_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(g_attn_scratch)), "resolving the attention scratch");
    WNW_CHECK_ARG(p != nullptr, "the attention scratch has no device address");
    sl.ptr = p;
  }
  if (!sl.cleared) {
    const int64_t n = (int64_t)WNW_NOALLOC_MAX_SEG + blk_counter_bytes() / 4;  // counters, 4 bytes each
    hipLaunchKernelGGL(fill_zero_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, (uint32_t*)sl.ptr, n);
    WNW_CHECK_HIP(hipGetLastError(), "clearing the attention scratch counters");
    sl.cleared = true;
  }
  *out = sl.ptr;
  return WNW_OK;
}

int decode_attn_impl(const void* q, const void* k, const void* v, const int32_t* cu_k,
                     const int64_t* seg_base, int64_t n_seg, int64_t group, int64_t head_dim,
                     int64_t total_rows, int64_t kv_rows, float scale, int dtype, void* out,
                     void* workspace, int64_t workspace_bytes, int kernel, int64_t n_wg, float* lse,
                     const AttnLogits* logits, int* logits_kept, void* stream, bool noalloc,
                     const AttnAppend* app, const AttnPrevScore* prev) {
  if (logits_kept) *logits_kept = 0;
  WNW_CHECK_ARG(n_seg >= 0 && n_seg < (1ll << 30), "n_seg out of range: %lld", (long long)n_seg);
  if (n_seg == 0) return WNW_OK;
  WNW_CHECK_ARG(q && cu_k && out && (workspace || noalloc) && ((k && v) || kv_rows == 0),
                "null pointer argument");
  WNW_CHECK_ARG(group >= 1 && group <= kMaxGroup, "group must be in [1, %d], got %lld", kMaxGroup,
                (long long)group);
  WNW_CHECK_ARG(head_dim == 64 || head_dim == 128 || head_dim == 256,
                "head_dim must be 64, 128 or 256, got %lld", (long long)head_dim);
  WNW_CHECK_ARG(dtype == WNW_F32 || dtype == WNW_F16 || dtype == WNW_BF16, "bad dtype %d", dtype);
  WNW_CHECK_ARG(total_rows >= 0 && kv_rows >= 0, "negative row count");
  if (app) {
    WNW_CHECK_ARG(seg_base && app->new_k && app->new_v && app->cu_out && app->cap,
                  "the fused append needs seg_base, new rows, cu_out and seg_cap");
    WNW_CHECK_ARG((const void*)app->cu_out != (const void*)cu_k, "cu_out must not alias cu");
    WNW_CHECK_ARG(((uintptr_t)app->new_k % 16) == 0 && ((uintptr_t)app->new_v % 16) == 0,
                  "new_k and new_v must be 16-byte aligned");
  }
  WNW_CHECK_ARG(kv_rows < (1ll << 40), "kv_rows too large");
  WNW_CHECK_ARG(((uintptr_t)q % 16) == 0 && ((uintptr_t)k % 16) == 0 && ((uintptr_t)v % 16) == 0 &&
                    ((uintptr_t)out % 16) == 0,
                "q, k, v and out must be 16-byte aligned");
  int kern = kernel;
  // rows of up to 512 bytes stream through a wave's two 16-row LDS buffers;
  // longer ones (fp32, head_dim 256) would need the whole LDS of a CU for them
  if (kern == WNW_ATTN_AUTO) kern = head_dim * elem_bytes(dtype) <= 512 ? WNW_ATTN_STREAM : WNW_ATTN_VALU;
  WNW_CHECK_ARG(kern == WNW_ATTN_MFMA || kern == WNW_ATTN_VALU || kern == WNW_ATTN_STREAM, "bad kernel id %d",
                kernel);
  if (kernel == WNW_ATTN_STREAM)
    WNW_CHECK_ARG(dtype != WNW_F32 && (head_dim == 64 || head_dim == 128) && group <= kMaxGroupS,
                  "the streaming kernel, chosen by name, needs bf16/f16, head_dim 64 or 128 and group <= %d",
                  kMaxGroupS);
  if (kern == WNW_ATTN_MFMA)
    WNW_CHECK_ARG(dtype != WNW_F32 && (head_dim == 64 || head_dim == 128),
                  "the MFMA kernel needs bf16/f16 and head_dim 64 or 128");
  const DeviceInfo& di = device_info();
  int64_t P = n_wg;
  if (P <= 0) {
    // Balanced split of the rows, never fewer than ~64 rows per workgroup:
    // one workgroup per CU for the streaming kernel (its four waves keep
    // enough loads in flight, and fewer workgroups mean fewer partials to
    // merge), two per CU for the others.
    const int64_t by_rows = std::max<int64_t>(1, (total_rows + 63) / 64);
    P = std::min<int64_t>((int64_t)di.cus * (kern == WNW_ATTN_STREAM ? 1 : 2), by_rows);
  }
  P = std::max<int64_t>(1, std::min<int64_t>(P, di.max_wg));
  WsLayout L;
  if (noalloc) {
    WNW_CHECK_ARG(n_seg <= WNW_NOALLOC_MAX_SEG, "the no-alloc entry point takes at most %d segments, got %lld",
                  WNW_NOALLOC_MAX_SEG, (long long)n_seg);
    // the limit's grid: two workgroups per CU outside 16-bit rows of 64 or
    // 128 elements and groups of up to 8, whatever the kernel launches
    const bool narrow = dtype != WNW_F32 && head_dim <= 128 && group <= kMaxGroupS;
    const int64_t P_lim = std::min<int64_t>((int64_t)di.cus * (narrow ? 1 : 2), std::max<int64_t>(1, (total_rows + 63) / 64));
    P = std::min(P, kNoAllocWgs);
    L = make_layout(WNW_NOALLOC_MAX_SEG, std::max(P, P_lim) + n_seg, group, head_dim);
    const int64_t need = L.total - blk_bytes(group, head_dim);
    WNW_CHECK_ARG(need <= WNW_NOALLOC_SCRATCH_BYTES,
                  "this launch needs %lld bytes of split-K scratch; the no-alloc entry point holds %lld "
                  "(fewer segments or a smaller group / head_dim fit)",
                  (long long)need, (long long)WNW_NOALLOC_SCRATCH_BYTES);
    const int rc = noalloc_scratch((hipStream_t)stream, &workspace);
    if (rc != WNW_OK) return rc;
  } else {
    L = ws_layout(n_seg, group, head_dim);
    WNW_CHECK_ARG(workspace_bytes >= L.total, "workspace too small: %lld < %lld bytes",
                  (long long)workspace_bytes, (long long)L.total);
  }

  AttnParams ap;
  ap.q = q;
  ap.k = k;
  ap.v = v;
  ap.cu = cu_k;
  ap.base = seg_base;
  ap.out = out;
  ap.counters = (int32_t*)((char*)workspace + L.counters);
  ap.lse = lse;
  ap.part_ml = (float*)((char*)workspace + L.ml);
  ap.part_acc = (float*)((char*)workspace + L.acc);
  ap.err = device_error_word();
  ap.split_inv = ~0ull / (uint64_t)(P * kSplitWaves) + 1;  // ceil(2^64 / (P * kSplitWaves))
  ap.phys_rows = kv_rows;
  ap.n_seg = (int32_t)n_seg;
  ap.G = (int32_t)group;
  ap.scale_log2 = scale * kLog2e;
  ap.xlog = nullptr;
  ap.xmask = ap.audio_s = ap.audio_e = nullptr;
  ap.max_audio = 0;
  ap.Hkv = 1;
  ap.new_k = ap.new_v = nullptr;
  ap.cu_out = nullptr;
  ap.cap = nullptr;
  ap.pv_xlog = ap.pv_lse = nullptr;
  ap.pv_kvlist = 0;
  ap.pv_nkv = 0;
  ap.pv_slices = 0;
  ap.pv_cu = ap.pv_acc_off = nullptr;
  ap.pv_base = nullptr;
  ap.pv_acc = nullptr;
  ap.pv_kv_rows = ap.pv_acc_len = 0;
  ap.pv_nblk = 0;
  if (prev) {
    // deferred scoring rides in the streaming kernel's direct-table form
    // only, one slice of 256 tokens per workgroup: elsewhere the caller
    // scores the slot in its own launch
    WNW_CHECK_ARG(prev->xlog && prev->lse && prev->cu && prev->acc && prev->acc_off && prev->audio_s &&
                      prev->audio_e,
                  "null deferred-scoring argument");
    WNW_CHECK_ARG(prev->hkv >= 1 && n_seg % prev->hkv == 0 && prev->max_audio > 0 && prev->kv_rows >= 0 &&
                      prev->acc_len >= 0,
                  "bad deferred-scoring geometry");
    const int64_t nblk = (prev->max_audio + 255) / 256;
    int nkv = 0;
    uint64_t kvlist = 0;
    for (int h = 0; h < prev->hkv && h < 64; ++h)
      if ((prev->kv_bits >> h) & 1) {
        if (nkv < 8) kvlist |= (uint64_t)h << (8 * nkv);
        ++nkv;
      }
    WNW_CHECK_ARG(prev->hkv <= 64 && (prev->hkv == 64 || (prev->kv_bits >> prev->hkv) == 0),
                  "deferred-scoring KV heads outside [0, %d)", prev->hkv);
    if (kern != WNW_ATTN_STREAM || n_seg > 64 || nkv > 8 || nkv * group > kPrevLogits ||
        (n_seg / prev->hkv) * nblk > P) {
      set_error("deferred scoring needs the streaming kernel, at most 64 segments, at most 8 scored KV heads "
                "and %d (KV head, query head) pairs, and one 256-token slice per workgroup (%lld slices, %lld "
                "workgroups)",
                kPrevLogits, (long long)((n_seg / prev->hkv) * nblk), (long long)P);
      return WNW_ENOTSUP;
    }
    if (logits && kern == WNW_ATTN_STREAM)
      WNW_CHECK_ARG(logits->hkv == prev->hkv && logits->max_audio == prev->max_audio &&
                        logits->audio_s == prev->audio_s && logits->audio_e == prev->audio_e,
                    "the deferred scoring and this launch's logits must share the audio geometry");
    ap.pv_xlog = nkv > 0 ? prev->xlog : nullptr;  // nothing scored: nothing to do
    ap.pv_lse = prev->lse;
    ap.pv_kvlist = kvlist;
    ap.pv_nkv = nkv;
    ap.pv_slices = (int32_t)((n_seg / prev->hkv) * nblk);
    ap.pv_cu = prev->cu;
    ap.pv_base = prev->base;
    ap.pv_kv_rows = prev->kv_rows;
    ap.pv_acc = prev->acc;
    ap.pv_acc_off = prev->acc_off;
    ap.pv_acc_len = prev->acc_len;
    ap.pv_nblk = (int32_t)nblk;
    ap.audio_s = prev->audio_s;
    ap.audio_e = prev->audio_e;
    ap.max_audio = prev->max_audio;
    ap.Hkv = prev->hkv;
  }
  hipStream_t st = (hipStream_t)stream;
  if (app) {
    if (kern == WNW_ATTN_STREAM) {  // fused into the launch
      ap.new_k = app->new_k;
      ap.new_v = app->new_v;
      ap.cu_out = app->cu_out;
      ap.cap = app->cap;
    } else {  // the in-place append first, then attention over the new offsets
      const int rc = wnw_append_inplace(const_cast<void*>(k), const_cast<void*>(v), app->new_k, app->new_v, cu_k,
                                        app->cu_out, seg_base, app->cap, n_seg, kv_rows, head_dim, dtype, stream);
      if (rc != WNW_OK) return rc;
      ap.cu = app->cu_out;
    }
  }
  if (logits && kern == WNW_ATTN_STREAM) {
    WNW_CHECK_ARG(logits->xlog && logits->mask && logits->audio_s && logits->audio_e, "null logits argument");
    WNW_CHECK_ARG(logits->hkv >= 1 && n_seg % logits->hkv == 0 && logits->max_audio > 0,
                  "bad logits geometry");
    ap.xlog = logits->xlog;
    ap.xmask = logits->mask;
    ap.audio_s = logits->audio_s;
    ap.audio_e = logits->audio_e;
    ap.max_audio = logits->max_audio;
    ap.Hkv = logits->hkv;
    if (logits_kept) *logits_kept = 1;
  }
  hipError_t e = hipErrorInvalidValue;
  switch (dtype) {
    case WNW_BF16: e = launch_attn_d<bf16_t>(kern, head_dim, ap, P, st); break;
    case WNW_F16: e = launch_attn_d<f16_t>(kern, head_dim, ap, P, st); break;
    case WNW_F32: e = launch_attn_d<float>(kern, head_dim, ap, P, st); break;
  }
  WNW_CHECK_HIP(e, "decode attention launch");
  return WNW_OK;
}

}  // namespace wnw

extern "C" int wnw_decode_attn_ex(const void* q, const void* k, const void* v, const int32_t* cu_k,
                                  const int64_t* seg_base, int64_t n_seg, int64_t group,
                                  int64_t head_dim, int64_t total_rows, int64_t kv_rows, float scale,
                                  int dtype, void* out, void* workspace, int64_t workspace_bytes,
                                  int kernel, int64_t n_wg, void* stream) {
  return decode_attn_impl(q, k, v, cu_k, seg_base, n_seg, group, head_dim, total_rows, kv_rows, scale,
                          dtype, out, workspace, workspace_bytes, kernel, n_wg, nullptr, nullptr, nullptr,
                          stream, false, nullptr);
}

extern "C" int wnw_decode_attn(const void* q, const void* k, const void* v, const int32_t* cu_k,
                               const int64_t* seg_base, int64_t n_seg, int64_t group,
                               int64_t head_dim, int64_t total_rows, int64_t kv_rows, float scale,
                               int dtype, void* out, void* workspace, int64_t workspace_bytes,
                               void* stream) {
  return wnw_decode_attn_ex(q, k, v, cu_k, seg_base, n_seg, group, head_dim, total_rows, kv_rows,
                            scale, dtype, out, workspace, workspace_bytes, WNW_ATTN_AUTO, 0, stream);
}

extern "C" int wnw_decode_attn_noalloc(const void* q, const void* k, const void* v, const int32_t* cu_k,
                                       const int64_t* seg_base, int64_t n_seg, int64_t group,
                                       int64_t head_dim, int64_t total_rows, int64_t kv_rows, float scale,
                                       int dtype, void* out, void* stream) {
  return decode_attn_impl(q, k, v, cu_k, seg_base, n_seg, group, head_dim, total_rows, kv_rows, scale,
                          dtype, out, nullptr, 0, WNW_ATTN_AUTO, 0, nullptr, nullptr, nullptr, stream, true,
                          nullptr);
}

extern "C" int wnw_decode_attn_append(const void* q, void* k_pool, void* v_pool, const void* new_k,
                                      const void* new_v, const int32_t* cu_old, int32_t* cu_new,
                                      const int64_t* seg_base, const int32_t* seg_cap, int64_t n_seg,
                                      int64_t group, int64_t head_dim, int64_t total_rows, int64_t pool_rows,
                                      float scale, int dtype, void* out, void* workspace,
                                      int64_t workspace_bytes, void* stream) {
  AttnAppend app;
  app.new_k = new_k;
  app.new_v = new_v;
  app.cu_out = cu_new;
  app.cap = seg_cap;
  return decode_attn_impl(q, k_pool, v_pool, cu_old, seg_base, n_seg, group, head_dim, total_rows, pool_rows,
                          scale, dtype, out, workspace, workspace_bytes, WNW_ATTN_AUTO, 0, nullptr, nullptr,
                          nullptr, stream, false, &app);
}
