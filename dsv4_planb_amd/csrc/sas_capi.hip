// sas_capi.hip -- extern "C" entry points of libsas_hip.so (declared in include/sas.h).
//
// Host side of the drop-in boundary: argument validation mirroring the
// reference's guards (api.py:187-191, 279-282; kernel.py:96-108) as status
// codes, workspace / plan sizing, and the stream-ordered launches of the
// planner, resolver, attention and combine kernels.  Nothing here allocates
// device memory or synchronises the host.
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <mutex>

#include "sas_common.h"
#include "sas_kernels.hip"
#include "sas_attend.hip"
#include "sas_attend_narrow.hip"
#include "sas_backward.hip"
#include "sas_backward_tile.hip"

namespace {

int esize(int dt) { return dt == SAS_DT_FP8E4M3 ? 1 : 2; }

// Compressed slots per token: top-k index slots (scenario 3) or the compressed
// row-list capacity (scenario 2).
int list_k(const sas_params_t* p) { return p->scenario >= 2 ? p->topk : 0; }

int query_num_cus() {
  int dev = 0, n = 0;
  if (hipGetDevice(&dev) != hipSuccess) return 0;
  if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
  return n;
}

int target_units(const sas_params_t* p) {
  int cus = p->num_cus > 0 ? p->num_cus : query_num_cus();
  if (cus <= 0) cus = 256;
  int per = p->units_per_cu > 0 ? p->units_per_cu : 1;
  return cus * per;
}

bool aligned16(const void* ptr) { return ((uintptr_t)ptr & 15u) == 0; }

SasFwdArgs fwd_args(const sas_params_t* p, int target) {
  SasFwdArgs a;
  std::memset(&a, 0, sizeof(a));
  a.T = p->total_tokens;
  a.H = p->num_heads_q;
  a.B = p->batch;
  a.scenario = p->scenario;
  a.K = list_k(p);
  a.cmp_ratio = p->cmp_ratio > 0 ? p->cmp_ratio : 1;
  a.ori_block_size = p->ori_block_size;
  a.ori_table_len = p->ori_table_len;
  a.ori_block_num = p->ori_block_num;
  a.cmp_block_size = p->scenario >= 2 ? p->cmp_block_size : 1;
  a.cmp_table_len = p->scenario >= 2 ? p->cmp_table_len : 1;
  a.cmp_block_num = p->scenario >= 2 ? p->cmp_block_num : 1;
  a.ori_block_stride = p->ori_block_stride;
  a.ori_row_stride = p->ori_row_stride;
  a.cmp_block_stride = p->scenario >= 2 ? p->cmp_block_stride : 0;
  a.cmp_row_stride = p->scenario >= 2 ? p->cmp_row_stride : 0;
  a.scale_log2 = p->softmax_scale * 1.4426950408889634f;
  a.win_left = p->ori_win_left;
  a.list_stride = (int)sas_row_list_stride(p->ori_win_left, a.K, p->scenario);
  a.unit_cap = (int)sas_plan_layout(p->total_tokens, target).unit_cap;
  a.split_cap = target;
  a.slot_cap = 2 * target;
  return a;
}

SasPlanArgs plan_args(const sas_params_t* p, int target, bool cu_ends = false) {
  SasPlanArgs a;
  a.T = p->total_tokens;
  a.B = p->batch;
  a.scenario = p->scenario;
  a.win_left = p->ori_win_left;
  a.cmp_ratio = p->cmp_ratio > 0 ? p->cmp_ratio : 1;
  a.K = list_k(p);
  a.H = p->num_heads_q;
  a.target = target;
  a.cu_ends = cu_ends;
  return a;
}

int check_tensors(const sas_params_t* p, const sas_tensors_t* t) {
  if (!t) return SAS_ERR_NULL;
  if (!t->q || !t->ori_kv || !t->ori_block_table || !t->q_prefix || !t->act_q_lens ||
      !t->seqused_kv || !t->sinks || !t->out)
    return SAS_ERR_NULL;
  if (p->scenario >= 2 && (!t->cmp_kv || !t->cmp_block_table)) return SAS_ERR_SCENARIO;
  if (p->scenario == 3 && !t->cmp_sparse_indices) return SAS_ERR_SCENARIO;
  if (p->kv_dtype == SAS_DT_FP8E4M3 &&
      (!t->ori_kv_scale || (p->scenario >= 2 && !t->cmp_kv_scale)))
    return SAS_ERR_NULL;
  if (!aligned16(t->q) || !aligned16(t->out) || !aligned16(t->ori_kv) ||
      (t->cmp_kv && !aligned16(t->cmp_kv)))
    return SAS_ERR_SHAPE;
  return SAS_OK;
}

struct Ws {
  int* status;
  int* rows;
  uint64_t* addr;
  float* scale;  // fp8 KV only
  int2* tok;     // per token: (window rows, compressed rows) at the call's lengths
  int* plan;
  float* o;
  float* ml;
};

int carve(const sas_params_t* p, void* ws, size_t ws_bytes, int target, Ws* out) {
  const SasWsLayout W = sas_ws_layout(p->total_tokens, list_k(p),
                                      p->num_heads_q, p->head_dim_v, target, p->scenario,
                                      p->ori_win_left, p->kv_dtype == SAS_DT_FP8E4M3);
  if (!ws || ws_bytes < W.total) return SAS_ERR_WORKSPACE;
  if (((uintptr_t)ws & 255u) != 0) return SAS_ERR_WORKSPACE;
  char* base = static_cast<char*>(ws);
  out->status = reinterpret_cast<int*>(base + W.off_status);
  out->rows = reinterpret_cast<int*>(base + W.off_rows);
  out->addr = reinterpret_cast<uint64_t*>(base + W.off_addr);
  out->scale = p->kv_dtype == SAS_DT_FP8E4M3 ? reinterpret_cast<float*>(base + W.off_scale) : nullptr;
  out->tok = reinterpret_cast<int2*>(base + W.off_tok);
  out->plan = reinterpret_cast<int*>(base + W.off_plan);
  out->o = reinterpret_cast<float*>(base + W.off_o);
  out->ml = reinterpret_cast<float*>(base + W.off_ml);
  return SAS_OK;
}

typedef void (*attend_fn_t)(SasFwdArgs, const uint16_t*, const uint64_t*, const float*,
                            const int2*, const float*, const int*, uint16_t*, float*, float*, float*,
                            sas::SasResolveArgs);

// Resolution's inputs and outputs in the workspace.
sas::SasResolveArgs resolve_args(const sas_params_t* p, const sas_tensors_t* t, const Ws& w,
                                 bool cu_ends = false) {
  sas::SasResolveArgs r;
  r.q_prefix = t->q_prefix;
  r.act_q = t->act_q_lens;
  r.cu_ends = cu_ends;
  r.seqused_kv = t->seqused_kv;
  r.ori_bt = t->ori_block_table;
  r.idx = t->cmp_sparse_indices;
  r.cmp_bt = t->cmp_block_table;
  r.rows = w.rows;
  r.tok = w.tok;
  r.addr = w.addr;
  r.ori_kv = static_cast<const uint8_t*>(t->ori_kv);
  r.cmp_kv = static_cast<const uint8_t*>(t->cmp_kv);
  r.esz = p->kv_dtype == SAS_DT_FP8E4M3 ? 1 : 2;
  r.ori_scale = t->ori_kv_scale;
  r.cmp_scale = t->cmp_kv_scale;
  r.scale = w.scale;
  r.t0 = 0;
  r.inv = nullptr;
  r.inv_rows = 0;
  r.local = nullptr;
  r.copies = 0;
  return r;
}

template <int DQK, bool NT, bool KV8>
attend_fn_t attend_ptr(bool f16) {
  return f16 ? &sas::attend_kernel<DQK, 1, NT, KV8> : &sas::attend_kernel<DQK, 0, NT, KV8>;
}

template <int DQK, bool KV8>
attend_fn_t attend_ptr(bool f16, bool nt) {
  return nt ? attend_ptr<DQK, true, KV8>(f16) : attend_ptr<DQK, false, KV8>(f16);
}

template <int DQK>
attend_fn_t narrow_ptr(bool f16, bool nt) {
  return nt ? (f16 ? &sas::attend_narrow_kernel<DQK, 1, true> : &sas::attend_narrow_kernel<DQK, 0, true>)
            : (f16 ? &sas::attend_narrow_kernel<DQK, 1, false> : &sas::attend_narrow_kernel<DQK, 0, false>);
}

// Does the forward let every unit resolve its own rows?  With at most as many
// tokens as target units every unit starts in the first wave of workgroups, and
// each resolves its rows before its first DMA (one launch fewer).  Otherwise units
// queue behind each other on a CU, and the resolver runs first as a stage of its own.
bool fused_resolution(const sas_params_t* p, int target) {
  return (int64_t)p->total_tokens <= (int64_t)target;
}

// At most 64 heads (16-bit KV) and more tokens than target units: the two-wave kernel, two
// of whose workgroups share a CU, so that one's start and epilogue run under the other's
// tiles.  Where every unit starts at once nothing runs beside it, and the four-wave
// kernel's wider gather and resolution win (32 sequences of 4k to 32k tokens, 64 heads,
// top-k 512, a graph replay: 32.6 us against 35.2 us with two waves; 101 tokens of 16
// heads, top-k 1024, an eager step with its plan: 125 against 147 us).  Below 33 heads the
// second wave's heads do not exist either, of two instead of four: forward calls of three
// prompts of 2,000 tokens, top-k 512, d_qk 576, take 391 (16 heads), 408 (32), 409 (33) and
// 463 us (64) against 641, 666, 668 and 709 with four waves; a window-only prompt of 8,192,
// d_qk 512, 244 (8), 253 (16), 282 (32) and 342 (64) against 381, 393, 433 and 490; 300
// tokens of one prompt 35 (16) and 39 (64) against 44 and 49.
bool narrow_heads(const sas_params_t* p, int target) {
  return p->num_heads_q <= 64 && p->kv_dtype != SAS_DT_FP8E4M3 && !fused_resolution(p, target);
}

// Decode-like calls (at most 4 query tokens per sequence on average) read each KV
// row for one token only: their gather uses non-temporal loads.  Prefill-like calls,
// where nearby tokens share most of their rows, keep the default cache policy.
attend_fn_t pick_attend(const sas_params_t* p, int target) {
  const bool f16 = p->q_dtype == SAS_DT_FP16;
  const bool nt = (int64_t)p->total_tokens <= 4 * (int64_t)p->batch;
  const bool kv8 = p->kv_dtype == SAS_DT_FP8E4M3;
  if (narrow_heads(p, target)) return p->head_dim_qk == 576 ? narrow_ptr<576>(f16, nt) : narrow_ptr<512>(f16, nt);
  if (p->head_dim_qk == 576)
    return kv8 ? attend_ptr<576, true>(f16, nt) : attend_ptr<576, false>(f16, nt);
  return kv8 ? attend_ptr<512, true>(f16, nt) : attend_ptr<512, false>(f16, nt);
}

int launch_status() { return hipGetLastError() == hipSuccess ? SAS_OK : SAS_ERR_LAUNCH; }

// The attention kernel over the plan's units.  resolve: each unit first resolves
// its own rows (the resolver stage is then not launched).  With events, the
// dispatch itself records its start and end into them.
int launch_attend(const sas_params_t* p, const sas_tensors_t* t, const int32_t* plan, const Ws& w,
                  int target, sas_stream_t stream, void* start_event, void* stop_event,
                  bool resolve, uint64_t* stamps = nullptr, bool cu_ends = false) {
  SasFwdArgs a = fwd_args(p, target);
  a.stamps = stamps;
  // the two-wave kernel reads the workspace's plan (the resolver has copied a caller's to it)
  if (narrow_heads(p, target)) plan = w.plan;
  sas::SasResolveArgs r = resolve_args(p, t, w, cu_ends);
  if (!resolve) r.addr = nullptr;
  r.rows = nullptr;  // the forward needs addresses only (sas_resolve also writes the codes)
  // With at most `target` tokens (the units resolve their own rows) the planner makes
  // at most `target` units (a plan that does not is refused: PS_UNITS_OVER_TARGET), so
  // no workgroup past the last unit is launched only to exit; otherwise the grid is
  // the plan's unit capacity and those past the plan's count exit at once.
  const int grid = resolve ? target : a.unit_cap;
  hipExtLaunchKernelGGL(pick_attend(p, target), dim3(grid), dim3(narrow_heads(p, target) ? sas::NW_NT : 256), 0, (hipStream_t)stream,
                        (hipEvent_t)start_event, (hipEvent_t)stop_event, 0, a,
                        static_cast<const uint16_t*>(t->q), static_cast<const uint64_t*>(w.addr),
                        static_cast<const float*>(w.scale), static_cast<const int2*>(w.tok),
                        t->sinks, static_cast<const int*>(plan), static_cast<uint16_t*>(t->out),
                        t->lse, w.o, w.ml, r);
  return launch_status();
}

// The resolver stage; codes: also write the row codes (the forward reads addresses
// only; the backward and sas_debug_rows read the codes).  inv: also the inverse lists.
// local: a caller's plan is copied to the workspace's, for kernels that read that one.
// t0, t1: the tokens (t1 < 0: all).
int resolve_stage(const sas_params_t* p, const sas_tensors_t* t, const int32_t* plan, void* ws,
                  size_t ws_bytes, sas_stream_t stream, bool codes, bool local,
                  uint32_t* inv = nullptr, int inv_rows = 0, bool cu_ends = false, int t0 = 0,
                  int t1 = -1) {
  int rc = sas_validate(p);
  if (rc) return rc;
  if ((rc = check_tensors(p, t))) return rc;
  const int target = target_units(p);
  Ws w;
  if ((rc = carve(p, ws, ws_bytes, target, &w))) return rc;
  if (!plan) plan = w.plan;
  if (p->total_tokens == 0) return SAS_OK;
  sas::SasResolveArgs r = resolve_args(p, t, w, cu_ends);
  if (!codes) r.rows = nullptr;
  r.inv = inv;
  r.inv_rows = inv_rows;
  r.t0 = t0;
  if (t1 < 0) t1 = p->total_tokens;
  if (local && plan != w.plan) {
    const SasPlanLayout L = sas_plan_layout(p->total_tokens, target);
    r.local = w.plan;
    r.copies = (int)((L.off_split_tokens + sas::RS_COPY - 1) / sas::RS_COPY);
  }
  hipLaunchKernelGGL(inv ? &sas::resolve_kernel<true> : &sas::resolve_kernel<false>,
                     dim3(t1 - t0 + r.copies), dim3(sas::RS_NT), 0, (hipStream_t)stream,
                     fwd_args(p, target), plan, r);
  return launch_status();
}

// The split combine, which also writes the call's status word (to the workspace
// and, when given, to status_out).
int combine_stage(const sas_params_t* p, const sas_tensors_t* t, const int32_t* plan, void* ws,
                  size_t ws_bytes, sas_stream_t stream, int32_t* status_out) {
  int rc = sas_validate(p);
  if (rc) return rc;
  if ((rc = check_tensors(p, t))) return rc;
  const int target = target_units(p);
  Ws w;
  if ((rc = carve(p, ws, ws_bytes, target, &w))) return rc;
  if (!plan) plan = w.plan;
  if (p->total_tokens == 0) return SAS_OK;
  const SasFwdArgs a = fwd_args(p, target);
  // at most one wave per (split token, head); split tokens number fewer than `target`
  const int waves = target * p->num_heads_q;
  const int per_cu = p->q_dtype == SAS_DT_BF16 ? sas::COMBINE_WGS_PER_CU<0> : sas::COMBINE_WGS_PER_CU<1>;
  const dim3 grid(std::min((waves + sas::COMBINE_WAVES - 1) / sas::COMBINE_WAVES,
                           per_cu * std::max(1, query_num_cus())));
  const dim3 block(64 * sas::COMBINE_WAVES);
  if (p->q_dtype == SAS_DT_BF16)
    hipLaunchKernelGGL(sas::combine_kernel<0>, grid, block, 0, (hipStream_t)stream, a, plan, w.o,
                       w.ml, w.tok, static_cast<uint16_t*>(t->out), t->lse, w.status, status_out);
  else
    hipLaunchKernelGGL(sas::combine_kernel<1>, grid, block, 0, (hipStream_t)stream, a, plan, w.o,
                       w.ml, w.tok, static_cast<uint16_t*>(t->out), t->lse, w.status, status_out);
  return launch_status();
}

int forward_impl(const sas_params_t* p, const sas_tensors_t* t, const int32_t* plan, void* ws,
                 size_t ws_bytes, sas_stream_t stream, int32_t* status_out, bool cu_ends = false) {
  int rc = sas_validate(p);
  if (rc) return rc;
  if ((rc = check_tensors(p, t))) return rc;
  const int target = target_units(p);
  Ws w;
  if ((rc = carve(p, ws, ws_bytes, target, &w))) return rc;
  if (p->total_tokens == 0) return SAS_OK;
  if (!plan) {
    hipLaunchKernelGGL(sas::plan_kernel, dim3(1), dim3(sas::PLAN_NT), 0, (hipStream_t)stream,
                       plan_args(p, target, cu_ends), t->q_prefix, t->act_q_lens, t->seqused_kv, w.plan);
    if ((rc = launch_status())) return rc;
    plan = w.plan;
  }
  if (fused_resolution(p, target)) {
    if ((rc = launch_attend(p, t, plan, w, target, stream, nullptr, nullptr, true, nullptr, cu_ends))) return rc;
  } else {
    if ((rc = resolve_stage(p, t, plan, ws, ws_bytes, stream, false, narrow_heads(p, target), nullptr, 0,
                            cu_ends)))
      return rc;
    if ((rc = launch_attend(p, t, plan, w, target, stream, nullptr, nullptr, false, nullptr, cu_ends))) return rc;
  }
  return combine_stage(p, t, plan, ws, ws_bytes, stream, status_out);
}

int bwd_layout(const sas_params_t* p, SasBwdLayout* L) {
  size_t fwd = 0;
  const int rc = sas_workspace_size(p, &fwd);
  if (rc) return rc;
  const int64_t cmp_cap = p->scenario >= 2 ? (int64_t)p->cmp_table_len * p->cmp_block_size : 0;
  *L = sas_bwd_layout(fwd, p->total_tokens, p->batch, p->num_heads_q, p->scenario, p->ori_win_left,
                      list_k(p), cmp_cap);
  return SAS_OK;
}

}  // namespace

extern "C" {

const char* sas_strerror(int code) {
  switch (code) {
    case SAS_OK: return "ok";
    case SAS_ERR_NULL: return "a required pointer is NULL";
    case SAS_ERR_SHAPE: return "inconsistent or unsupported shape, stride or alignment";
    case SAS_ERR_DTYPE: return "unsupported dtype combination";
    case SAS_ERR_SCENARIO: return "scenario must be 1 (SWA), 2 (CFA) or 3 (SCFA) with its inputs";
    case SAS_ERR_MASK_MODE: return "only ori_mask_mode=4, cmp_mask_mode=3, ori_win_right=0 supported";
    case SAS_ERR_HEADS: return "num_heads_kv must be 1 and num_heads_q in [1, 128]";
    case SAS_ERR_WORKSPACE: return "workspace missing, misaligned or too small";
    case SAS_ERR_PLAN: return "plan buffer too small, or a plan built for other arguments";
    case SAS_ERR_LAUNCH: return "HIP kernel launch failed";
    case SAS_ERR_METADATA: return "invalid metadata arguments";
    case SAS_ERR_GRAPH: return "hipGraph capture or instantiation failed";
    case SAS_ERR_NOT_IMPLEMENTED: return "not implemented";
    case SAS_ERR_SCRATCH:
      return "the call needs more workspace than the fixed scratch buffer of "
             "sas_forward_noalloc (SAS_SCRATCH_BYTES); use sas_forward with a workspace";
    default: return "unknown error";
  }
}

int sas_version(void) { return 1; }

int sas_validate(const sas_params_t* p) {
  if (!p) return SAS_ERR_NULL;
  if (p->num_heads_kv != 1 || p->num_heads_q < 1 || p->num_heads_q > 128) return SAS_ERR_HEADS;
  if (p->scenario < 1 || p->scenario > 3) return SAS_ERR_SCENARIO;
  if (p->ori_mask_mode != 4 || p->ori_win_right != 0 || p->ori_win_left < 0) return SAS_ERR_MASK_MODE;
  if (p->scenario >= 2 && p->cmp_mask_mode != 3) return SAS_ERR_MASK_MODE;
  if (p->q_dtype != SAS_DT_BF16 && p->q_dtype != SAS_DT_FP16) return SAS_ERR_DTYPE;
  if (p->kv_dtype != p->q_dtype && p->kv_dtype != SAS_DT_FP8E4M3) return SAS_ERR_DTYPE;
  if (p->batch < 1 || p->total_tokens < 0) return SAS_ERR_SHAPE;
  if (p->head_dim_qk != 512 && p->head_dim_qk != 576) return SAS_ERR_SHAPE;
  if (p->head_dim_v != 512) return SAS_ERR_SHAPE;
  if (!std::isfinite(p->softmax_scale)) return SAS_ERR_SHAPE;
  if (p->num_cus < 0 || p->units_per_cu < 0) return SAS_ERR_SHAPE;
  const int es = esize(p->kv_dtype);
  if (p->ori_block_num < 1 || p->ori_block_size < 1 || p->ori_table_len < 1) return SAS_ERR_SHAPE;
  if (p->ori_row_stride < p->head_dim_qk ||
      p->ori_block_stride < (int64_t)p->ori_block_size * p->ori_row_stride)
    return SAS_ERR_SHAPE;
  if ((p->ori_row_stride * es) % 16 != 0 || (p->ori_block_stride * es) % 16 != 0) return SAS_ERR_SHAPE;
  // row codes (page * block_size + offset) are int32
  if ((int64_t)p->ori_block_num * p->ori_block_size >= (int64_t)1 << 31) return SAS_ERR_SHAPE;
  if (p->scenario >= 2) {
    if (p->cmp_ratio < 1) return SAS_ERR_SCENARIO;
    if (p->cmp_block_num < 1 || p->cmp_block_size < 1 || p->cmp_table_len < 1) return SAS_ERR_SHAPE;
    if (p->cmp_row_stride < p->head_dim_qk ||
        p->cmp_block_stride < (int64_t)p->cmp_block_size * p->cmp_row_stride)
      return SAS_ERR_SHAPE;
    if ((p->cmp_row_stride * es) % 16 != 0 || (p->cmp_block_stride * es) % 16 != 0)
      return SAS_ERR_SHAPE;
    if ((int64_t)p->cmp_block_num * p->cmp_block_size >= (int64_t)1 << 31) return SAS_ERR_SHAPE;
  }
  if (p->scenario >= 2 && p->topk < 1) return SAS_ERR_SCENARIO;
  if ((int64_t)p->total_tokens * sas_row_list_stride(p->ori_win_left, list_k(p), p->scenario) >=
      (int64_t)1 << 31)
    return SAS_ERR_SHAPE;
  return SAS_OK;
}

int sas_target_units(const sas_params_t* p, int32_t* units) {
  if (!p || !units) return SAS_ERR_NULL;
  *units = target_units(p);
  return SAS_OK;
}

int sas_plan_size(const sas_params_t* p, size_t* n) {
  int rc = sas_validate(p);
  if (rc) return rc;
  if (!n) return SAS_ERR_NULL;
  *n = (size_t)sas_plan_layout(p->total_tokens, target_units(p)).total;
  return SAS_OK;
}

int sas_workspace_size(const sas_params_t* p, size_t* bytes) {
  int rc = sas_validate(p);
  if (rc) return rc;
  if (!bytes) return SAS_ERR_NULL;
  *bytes = sas_ws_layout(p->total_tokens, list_k(p), p->num_heads_q, p->head_dim_v,
                         target_units(p), p->scenario, p->ori_win_left,
                         p->kv_dtype == SAS_DT_FP8E4M3)
               .total;
  return SAS_OK;
}

int sas_plan(const sas_params_t* p, const int32_t* q_prefix, const int32_t* act_q_lens,
             const int32_t* seqused_kv, int32_t* plan, size_t plan_n, sas_stream_t stream) {
  int rc = sas_validate(p);
  if (rc) return rc;
  if (!q_prefix || !act_q_lens || !seqused_kv || !plan) return SAS_ERR_NULL;
  if (!aligned16(plan)) return SAS_ERR_SHAPE;  // the planner writes 16-B records
  const int target = target_units(p);
  if (plan_n < (size_t)sas_plan_layout(p->total_tokens, target).total) return SAS_ERR_PLAN;
  hipLaunchKernelGGL(sas::plan_kernel, dim3(1), dim3(sas::PLAN_NT), 0, (hipStream_t)stream,
                     plan_args(p, target), q_prefix, act_q_lens, seqused_kv, plan);
  return launch_status();
}

int sas_resolve(const sas_params_t* p, const sas_tensors_t* t, const int32_t* plan, void* ws,
                size_t ws_bytes, sas_stream_t stream) {
  if (!p) return SAS_ERR_NULL;
  return resolve_stage(p, t, plan, ws, ws_bytes, stream, true, narrow_heads(p, target_units(p)));
}

int sas_attend_timed(const sas_params_t* p, const sas_tensors_t* t, const int32_t* plan, void* ws,
                     size_t ws_bytes, sas_stream_t stream, void* start_event, void* stop_event,
                     uint64_t* stamps) {
  int rc = sas_validate(p);
  if (rc) return rc;
  if ((rc = check_tensors(p, t))) return rc;
  const int target = target_units(p);
  Ws w;
  if ((rc = carve(p, ws, ws_bytes, target, &w))) return rc;
  if (!plan) plan = w.plan;
  if (p->total_tokens == 0) return SAS_OK;
  // the dispatch exactly as sas_forward launches it (with the units' own row
  // resolution where the forward fuses it)
  return launch_attend(p, t, plan, w, target, stream, start_event, stop_event,
                       fused_resolution(p, target), stamps);
}

int sas_attend(const sas_params_t* p, const sas_tensors_t* t, const int32_t* plan, void* ws,
               size_t ws_bytes, sas_stream_t stream) {
  return sas_attend_timed(p, t, plan, ws, ws_bytes, stream, nullptr, nullptr, nullptr);
}


int sas_combine(const sas_params_t* p, const sas_tensors_t* t, const int32_t* plan, void* ws,
                size_t ws_bytes, sas_stream_t stream) {
  return combine_stage(p, t, plan, ws, ws_bytes, stream, nullptr);
}

int sas_forward(const sas_params_t* p, const sas_tensors_t* t, const int32_t* plan, void* ws,
                size_t ws_bytes, sas_stream_t stream) {
  return forward_impl(p, t, plan, ws, ws_bytes, stream, nullptr);
}

int sas_forward_cu(const sas_params_t* p, const sas_tensors_t* t, const int32_t* plan, void* ws,
                   size_t ws_bytes, sas_stream_t stream) {
  return forward_impl(p, t, plan, ws, ws_bytes, stream, nullptr, true);
}

int sas_call_sizes(const sas_params_t* p, int64_t* sizes) {
  const int rc = sas_validate(p);
  if (rc) return rc;
  if (!sizes) return SAS_ERR_NULL;
  const int target = target_units(p);
  sizes[0] = target;
  sizes[1] = sas_plan_layout(p->total_tokens, target).total;
  sizes[2] = (int64_t)sas_ws_layout(p->total_tokens, list_k(p), p->num_heads_q, p->head_dim_v, target,
                                    p->scenario, p->ori_win_left, p->kv_dtype == SAS_DT_FP8E4M3).total;
  return SAS_OK;
}

int sas_backward_workspace_size(const sas_params_t* p, size_t* bytes) {
  return sas_backward_workspace_size_for(p, 1, bytes);
}

int sas_backward_workspace_size_for(const sas_params_t* p, int kv_grad, size_t* bytes) {
  int rc = sas_validate(p);
  if (rc) return rc;
  if (!bytes) return SAS_ERR_NULL;
  SasBwdLayout L;
  if ((rc = bwd_layout(p, &L))) return rc;
  *bytes = kv_grad ? L.total : L.base_total;
  return SAS_OK;
}

int sas_backward(const sas_params_t* p, const sas_tensors_t* t, const int32_t* plan,
                 const void* dout, const float* dlse, float* dq, float* dsinks, float* d_ori_kv,
                 float* d_cmp_kv, void* ws, size_t ws_bytes, sas_stream_t stream) {
  int rc = sas_validate(p);
  if (rc) return rc;
  if ((rc = check_tensors(p, t))) return rc;
  if (!dout || !dq || !dsinks || !t->lse) return SAS_ERR_NULL;
  if (p->kv_dtype == SAS_DT_FP8E4M3) return SAS_ERR_NOT_IMPLEMENTED;
  if (!aligned16(dout) || !aligned16(dq)) return SAS_ERR_SHAPE;
  const bool kv_grad = d_ori_kv || d_cmp_kv;
  SasBwdLayout L;
  if ((rc = bwd_layout(p, &L))) return rc;
  if (!ws || ws_bytes < (kv_grad ? L.total : L.base_total)) return SAS_ERR_WORKSPACE;
  const int target = target_units(p);
  Ws w;
  if ((rc = carve(p, ws, ws_bytes, target, &w))) return rc;
  hipStream_t s = (hipStream_t)stream;
  const int T = p->total_tokens, H = p->num_heads_q;
  char* base = static_cast<char*>(ws);
  float* dterm = reinterpret_cast<float*>(base + L.off_dterm);
  float* sterm = reinterpret_cast<float*>(base + L.off_sterm);
  if (T == 0) {  // no tokens: dsinks = 0 (a kernel, not a memset, so the call can be captured)
    hipLaunchKernelGGL(sas::bwd_dsink_kernel, dim3(H), dim3(256), 0, s, 0, H,
                       static_cast<const float*>(sterm), dsinks);
    return launch_status();
  }
  if (!plan) {
    hipLaunchKernelGGL(sas::plan_kernel, dim3(1), dim3(sas::PLAN_NT), 0, s, plan_args(p, target),
                       t->q_prefix, t->act_q_lens, t->seqused_kv, w.plan);
    if ((rc = launch_status())) return rc;
    plan = w.plan;
  }
  const bool tiles = kv_grad && L.tile;
  const bool use_inv = tiles && p->scenario == 3 && L.cmp_rows > 0;
  uint32_t* inv = use_inv ? reinterpret_cast<uint32_t*>(base + L.off_inv) : nullptr;
  const SasFwdArgs a = fwd_args(p, target);
  const bool f16 = p->q_dtype == SAS_DT_FP16, d576 = p->head_dim_qk == 576;
  const uint16_t* q = static_cast<const uint16_t*>(t->q);
  const uint16_t* go = static_cast<const uint16_t*>(dout);
  const int2* tok = w.tok;
  const uint64_t* addr = w.addr;
  int* flags = tiles ? reinterpret_cast<int*>(base + L.off_flags) : nullptr;
  const dim3 grid(a.unit_cap * ((H + sas::BW_HEADS - 1) / sas::BW_HEADS));
  typedef void (*bwd_fn_t)(SasFwdArgs, const uint16_t*, const uint16_t*, const uint64_t*,
                           const int2*, const float*, sas::SasBwdTerms, const int*, float*,
                           sas::SasBwdSpill);
  const bwd_fn_t fn = tiles ? (d576 ? (f16 ? &sas::bwd_dq_kernel<576, 1, true> : &sas::bwd_dq_kernel<576, 0, true>)
                                    : (f16 ? &sas::bwd_dq_kernel<512, 1, true> : &sas::bwd_dq_kernel<512, 0, true>))
                            : (d576 ? (f16 ? &sas::bwd_dq_kernel<576, 1, false> : &sas::bwd_dq_kernel<576, 0, false>)
                                    : (f16 ? &sas::bwd_dq_kernel<512, 1, false> : &sas::bwd_dq_kernel<512, 0, false>));
  const sas::SasBwdTerms bt = {static_cast<const uint16_t*>(t->out), dlse, t->sinks, dterm, sterm};
  sas::SasBwdSpill sp = {};
  sas::SasTileArgs ta = {};
  if (tiles) {
    sp.stride = L.stride;
    sp.row_bytes = L.row_bytes;
    sp.data = reinterpret_cast<uint8_t*>(base + L.off_spill);
    sp.flags = flags;
    ta.q_prefix = t->q_prefix;
    ta.act_q = t->act_q_lens;
    ta.seqused_kv = t->seqused_kv;
    ta.ori_bt = t->ori_block_table;
    ta.cmp_bt = t->cmp_block_table;
    ta.inv = inv;
    ta.cmp_rows = L.cmp_rows;
    // one workgroup per CU (its LDS), a multiple of the XCDs
    ta.workers = std::max(8, query_num_cus() / 8 * 8);
    ta.item_cap = (int)L.item_cap;
    ta.want_ori = d_ori_kv != nullptr;
    ta.want_cmp = L.cmp_rows > 0 && d_cmp_kv != nullptr;
    ta.items = reinterpret_cast<int4*>(base + L.off_items);
  }
  // the tokens in runs that the spill and the inverse lists hold (one run where nothing is
  // spilled)
  const int chunk = tiles ? L.chunk_tokens : T;
  for (int t0 = 0; t0 < T; t0 += chunk) {
    sp.t0 = t0;
    sp.t1 = std::min(T, t0 + chunk);
    if ((rc = resolve_stage(p, t, plan, ws, ws_bytes, stream, true, t0 == 0, inv, L.cmp_rows, false, t0, sp.t1)))
      return rc;
    plan = w.plan;  // (the first run's resolver has copied a caller's to it)
    const int run = sp.t1 - t0;
    hipLaunchKernelGGL(sas::bwd_prep_kernel, dim3(run * ((H + sas::BP_HEADS - 1) / sas::BP_HEADS)), dim3(256), 0, s,
                       a, p->head_dim_qk, t0, plan, tok, dterm, sterm, dq, flags);
    if ((rc = launch_status())) return rc;
    hipLaunchKernelGGL(fn, grid, dim3(256), 0, s, a, q, go, addr, tok,
                       static_cast<const float*>(t->lse), bt, plan, dq, sp);
    if ((rc = launch_status())) return rc;
    if (!tiles) break;
    hipLaunchKernelGGL(sas::bwd_items_kernel, dim3(1), dim3(1024), 0, s, a, ta, sp, plan);
    if ((rc = launch_status())) return rc;
    typedef void (*tile_fn_t)(SasFwdArgs, sas::SasTileArgs, sas::SasBwdSpill, const uint16_t*,
                              const uint16_t*, const int2*, const int*, float*, float*);
    const tile_fn_t tf = d576 ? (f16 ? &sas::bwd_dkv_tile_kernel<576, 1> : &sas::bwd_dkv_tile_kernel<576, 0>)
                              : (f16 ? &sas::bwd_dkv_tile_kernel<512, 1> : &sas::bwd_dkv_tile_kernel<512, 0>);
    hipLaunchKernelGGL(tf, dim3(ta.workers), dim3(sas::TK_NT), 0, s, a, ta, sp,
                       q, go, tok, plan, d_ori_kv, d_cmp_kv);
    if ((rc = launch_status())) return rc;
  }
  if (kv_grad) {  // the KV pools' gradient (accumulated into the buffers)
    // what the tiles leave: everything without them; the compressed rows where they are
    // not covered; the tokens marked for an infinity or a NaN
    const int mode = !tiles ? 0 : p->scenario >= 2 && L.cmp_rows == 0 ? 1 : 2;
    const dim3 gkv(mode == 2 ? std::min(a.unit_cap, std::max(1, query_num_cus())) : a.unit_cap);
    typedef void (*dkv_fn_t)(SasFwdArgs, const uint16_t*, const uint16_t*, const uint64_t*,
                             const int*, const int2*, const float*, const float*, const int*,
                             float*, float*, int, const int*);
    const dkv_fn_t kf = d576 ? (f16 ? &sas::bwd_dkv_kernel<576, 1> : &sas::bwd_dkv_kernel<576, 0>)
                             : (f16 ? &sas::bwd_dkv_kernel<512, 1> : &sas::bwd_dkv_kernel<512, 0>);
    hipLaunchKernelGGL(kf, gkv, dim3(256), 0, s, a, q, go, addr, static_cast<const int*>(w.rows), tok,
                       static_cast<const float*>(t->lse), static_cast<const float*>(dterm), plan,
                       d_ori_kv, p->scenario >= 2 ? d_cmp_kv : nullptr, mode,
                       static_cast<const int*>(flags));
    if ((rc = launch_status())) return rc;
  }
  hipLaunchKernelGGL(sas::bwd_dsink_kernel, dim3(H), dim3(256), 0, s, T, H,
                     static_cast<const float*>(sterm), dsinks);
  return launch_status();
}

int sas_debug_rows(const sas_params_t* p, const void* ws, int32_t* rows, int32_t* counts,
                   sas_stream_t stream) {
  int rc = sas_validate(p);
  if (rc) return rc;
  if (!ws || !rows || !counts) return SAS_ERR_NULL;
  const int K = list_k(p);
  const SasWsLayout W = sas_ws_layout(p->total_tokens, K, p->num_heads_q, p->head_dim_v,
                                      target_units(p), p->scenario, p->ori_win_left,
                                      p->kv_dtype == SAS_DT_FP8E4M3);
  // the workspace lists sit at the tile-rounded stride; rows gets the capacity
  const size_t stride = (size_t)sas_row_list_stride(p->ori_win_left, K, p->scenario);
  const size_t cap = (size_t)sas_row_list_cap(p->ori_win_left, K, p->scenario);
  const char* base = static_cast<const char*>(ws);
  if (p->total_tokens > 0 &&
      hipMemcpy2DAsync(rows, cap * 4, base + W.off_rows, stride * 4, cap * 4, (size_t)p->total_tokens,
                       hipMemcpyDeviceToDevice, (hipStream_t)stream) != hipSuccess)
    return SAS_ERR_LAUNCH;
  // the compressed counts: the second int of each token's (window, compressed) record
  if (p->total_tokens > 0 &&
      hipMemcpy2DAsync(counts, 4, base + W.off_tok + 4, 8, 4, (size_t)p->total_tokens,
                       hipMemcpyDeviceToDevice, (hipStream_t)stream) != hipSuccess)
    return SAS_ERR_LAUNCH;
  return SAS_OK;
}

int sas_debug_lists(const sas_params_t* p, const void* ws, uint64_t* addr, float* scale,
                    int32_t* counts, sas_stream_t stream) {
  int rc = sas_validate(p);
  if (rc) return rc;
  if (!ws || !addr || !counts) return SAS_ERR_NULL;
  const bool kv8 = p->kv_dtype == SAS_DT_FP8E4M3;
  const int K = list_k(p);
  const SasWsLayout W = sas_ws_layout(p->total_tokens, K, p->num_heads_q, p->head_dim_v,
                                      target_units(p), p->scenario, p->ori_win_left, kv8);
  const size_t stride = (size_t)sas_row_list_stride(p->ori_win_left, K, p->scenario);
  const size_t cap = (size_t)sas_row_list_cap(p->ori_win_left, K, p->scenario);
  const size_t T = (size_t)p->total_tokens;
  const char* base = static_cast<const char*>(ws);
  hipStream_t s = (hipStream_t)stream;
  if (T == 0) return SAS_OK;
  if (hipMemcpy2DAsync(addr, cap * 8, base + W.off_addr, stride * 8, cap * 8, T,
                       hipMemcpyDeviceToDevice, s) != hipSuccess)
    return SAS_ERR_LAUNCH;
  if (kv8 && scale &&
      hipMemcpy2DAsync(scale, cap * 4, base + W.off_scale, stride * 4, cap * 4, T,
                       hipMemcpyDeviceToDevice, s) != hipSuccess)
    return SAS_ERR_LAUNCH;
  if (hipMemcpyAsync(counts, base + W.off_tok, T * 8, hipMemcpyDeviceToDevice, s) != hipSuccess)
    return SAS_ERR_LAUNCH;
  return SAS_OK;
}

}  // extern "C"

// ---- the allocation-free variant of sas_forward ----
// Its workspace is this fixed device array (one copy per GPU, held until the
// process ends).  In host code `scratch` names a host-side stand-in, not device
// memory: its device address comes from hipGetSymbolAddress, once per device with
// that device current, and only that address is ever handed to a kernel.
static __device__ __attribute__((aligned(256))) uint8_t scratch[SAS_SCRATCH_BYTES];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};

// The current device's copy of `scratch` (looked up on the first call per device).
int scratch_for_current_device(void** out) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return SAS_ERR_LAUNCH;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* ptr = nullptr;
    if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess || !ptr) return SAS_ERR_LAUNCH;
    g_scratch_ptr[dev] = ptr;
  }
  *out = g_scratch_ptr[dev];
  return SAS_OK;
}
}  // namespace

extern "C" {

int sas_forward_noalloc(const sas_params_t* p, const sas_tensors_t* t, const int32_t* plan,
                        int32_t* status, sas_stream_t stream) {
  void* ws = nullptr;
  int rc = scratch_for_current_device(&ws);  // first, so that any call sets the device up
  if (rc) return rc;
  if ((rc = sas_validate(p))) return rc;
  size_t need = 0;
  if ((rc = sas_workspace_size(p, &need))) return rc;
  if (need > (size_t)SAS_SCRATCH_BYTES) return SAS_ERR_SCRATCH;
  return forward_impl(p, t, plan, ws, (size_t)SAS_SCRATCH_BYTES, stream, status);
}

int sas_graph_capture(const sas_params_t* p, const sas_tensors_t* t, const int32_t* plan, void* ws,
                      size_t ws_bytes, sas_stream_t stream, void** graph_exec) {
  if (!graph_exec) return SAS_ERR_NULL;
  int rc = sas_validate(p);
  if (rc) return rc;
  if ((rc = check_tensors(p, t))) return rc;
  hipStream_t s = (hipStream_t)stream;
  hipGraph_t graph = nullptr;
  if (hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal) != hipSuccess) return SAS_ERR_GRAPH;
  rc = sas_forward(p, t, plan, ws, ws_bytes, stream);
  hipError_t e = hipStreamEndCapture(s, &graph);
  if (rc) {
    if (graph) (void)hipGraphDestroy(graph);
    return rc;
  }
  if (e != hipSuccess || !graph) return SAS_ERR_GRAPH;
  hipGraphExec_t exec = nullptr;
  e = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
  (void)hipGraphDestroy(graph);
  if (e != hipSuccess) return SAS_ERR_GRAPH;
  *graph_exec = exec;
  return SAS_OK;
}

int sas_graph_launch(void* graph_exec, sas_stream_t stream) {
  if (!graph_exec) return SAS_ERR_NULL;
  return hipGraphLaunch((hipGraphExec_t)graph_exec, (hipStream_t)stream) == hipSuccess
             ? SAS_OK
             : SAS_ERR_GRAPH;
}

int sas_graph_destroy(void* graph_exec) {
  if (!graph_exec) return SAS_ERR_NULL;
  return hipGraphExecDestroy((hipGraphExec_t)graph_exec) == hipSuccess ? SAS_OK : SAS_ERR_GRAPH;
}

}  // extern "C"

