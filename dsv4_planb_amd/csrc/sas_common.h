// sas_common.h -- shared definitions of the gfx950 sparse shared-KV attention
// kernels and their host launchers (plan layout, workspace layout, params).
#pragma once
#include <stddef.h>
#include <stdint.h>

#include "../../include/sas.h"

#ifdef __HIPCC__
#define SAS_HD __host__ __device__
#else
#define SAS_HD
#endif

// ---- split-KV plan (int32 buffer written by the planner kernel) ----
// header
#define SAS_PLAN_MAGIC 0x53415350  // 'SASP'
#define SAS_PLAN_VERSION 3
#define SAS_PLAN_HDR 24
// PH_T .. PH_CMP_RATIO record the arguments the plan was built for; the kernels
// refuse a plan whose record differs from the call's (plan_matches below).
// PH_STATUS holds the planner's own invariant checks (PS_* bits, 0 = sound).
enum {
  PH_MAGIC = 0, PH_VERSION, PH_T, PH_UNITS, PH_CHUNK, PH_TARGET, PH_NSPLIT_TOKENS,
  PH_NSLOTS, PH_TOTAL_ROWS_LO, PH_TOTAL_ROWS_HI, PH_H, PH_UNIT_CAP, PH_SCENARIO, PH_K,
  PH_WIN_LEFT, PH_B, PH_CMP_RATIO, PH_STATUS
};
// PS_UNITS_OVER_TARGET: at most `target` tokens, yet more than `target` units (the
// attention kernel then launches `target` workgroups, one per unit).
enum {
  PS_UNITS_OVER_CAP = 1, PS_SLOTS_OVER_CAP = 2, PS_SPLIT_TOKENS_OVER_CAP = 4,
  PS_UNITS_OVER_TARGET = 8
};
// per-token record [T][8]: the owning batch and position (TK_B = -1: no batch owns
// the token; TK_SG then holds the last batch whose q_prefix is at most t, or -1), and
// the spans at the lengths the plan was built for.  The kernels take the work
// partition and the ownership from the plan, and the window and the compressed
// threshold from the call's seqused_kv (see live_token in sas_kernels.hip).
#define SAS_TOK_W 8
enum { TK_B = 0, TK_S, TK_SG, TK_NWIN, TK_WINLO, TK_NCMPMAX, TK_SPLITS, TK_WSBASE };
// per-unit record [unit_cap][4]: token, first row, end row, split index (-1 = padded token)
#define SAS_UNIT_W 4

// KV rows processed per inner tile by the attention kernel.
#define SAS_TILE 32
#define SAS_MIN_CHUNK 64

struct SasPlanLayout {
  int64_t T, target, unit_cap, split_cap;
  // int32 offsets: token records, units, split tokens, and per split token its
  // (split count, first workspace slot)
  int64_t off_tok, off_units, off_split_tokens, off_split_meta, total;
};

SAS_HD static inline SasPlanLayout sas_plan_layout(int64_t T, int64_t target) {
  SasPlanLayout L;
  L.T = T;
  L.target = target;
  L.unit_cap = T + target;
  L.split_cap = target;
  L.off_tok = SAS_PLAN_HDR;
  L.off_units = L.off_tok + SAS_TOK_W * T;
  L.off_split_tokens = L.off_units + SAS_UNIT_W * L.unit_cap;
  L.off_split_meta = L.off_split_tokens + L.split_cap;
  L.total = L.off_split_meta + 2 * L.split_cap;
  // A plan is never SAS_META_SIZE (1024) entries long, so a caller-supplied table
  // is told apart from the reference's int32[1024] metadata by its size alone.
  if (L.total == SAS_META_SIZE) L.total += 1;
  return L;
}

// ---- workspace (bytes, each region 256-B aligned) ----
// The first int32 of the workspace is the status word of the last forward call on
// it: 0, or SAS_ERR_PLAN when the plan did not match the call (the outputs are then
// zeros: all of them when the plan's header differs, those of the refused tokens
// when a token's batch differs under the call's q_prefix / act_q).  The combine
// kernel, the last of every forward call, writes it.
struct SasWsLayout {
  size_t off_status, off_rows, off_addr, off_scale, off_tok, off_plan, off_o, off_ml, total;
  int64_t slot_cap;
};

SAS_HD static inline size_t sas_align256(size_t x) { return (x + 255) & ~(size_t)255; }

// Row-code list of one token: its window rows, then directly after them its
// compressed rows (scenario 3: the resolved top-k; scenario 2: every causally
// valid row, up to K of them).  Capacity: win_left + 1 + K slots.
SAS_HD static inline int64_t sas_row_list_cap(int64_t win_left, int64_t K, int scenario) {
  return win_left + 1 + (scenario >= 2 ? K : 0);
}
// Distance between two tokens' lists: the capacity rounded up to whole tiles.  Work
// units of different tokens resolve and read their lists concurrently; so no 64-B
// line of the code, address or scale lists holds rows of two tokens, and a unit's
// last tile, read whole, stays inside its own token's list.
SAS_HD static inline int64_t sas_row_list_stride(int64_t win_left, int64_t K, int scenario) {
  return (sas_row_list_cap(win_left, K, scenario) + SAS_TILE - 1) / SAS_TILE * SAS_TILE;
}

SAS_HD static inline SasWsLayout sas_ws_layout(int64_t T, int64_t K, int64_t H, int64_t Dv,
                                        int64_t target, int scenario, int64_t win_left,
                                        bool kv8) {
  SasWsLayout W;
  size_t off = 0;
  W.off_status = off;
  off = sas_align256(off + 4);
  W.off_rows = off;
  off = sas_align256(off + (size_t)(T > 0 ? T : 1) * sas_row_list_stride(win_left, K, scenario) * 4);
  // 64-bit row addresses, same shape as the code lists, plus one tile of slack
  // (the attention kernel reads row addresses 8 at a time with scalar loads)
  W.off_addr = off;
  off = sas_align256(off + ((size_t)(T > 0 ? T : 1) * sas_row_list_stride(win_left, K, scenario) +
                            SAS_TILE) * 8);
  // fp8 KV: the fp32 dequantisation scale s of every listed row, then a second list
  // of 1 / s (0 where s = 0), same shape
  W.off_scale = off;
  if (kv8)
    off = sas_align256(off + 2 * (size_t)(T > 0 ? T : 1) * sas_row_list_stride(win_left, K, scenario) * 4);
  // per token: int2 (window rows, compressed rows) at the call's lengths; a window
  // count of -1 marks a token refused for a plan that no longer matches it
  W.off_tok = off;
  off = sas_align256(off + (size_t)(T > 0 ? T : 1) * 8);
  W.off_plan = off;
  off = sas_align256(off + (size_t)sas_plan_layout(T, target).total * 4);
  // split tokens have more rows than the chunk (>= total / target), so fewer
  // than `target` of them exist and their units number at most 2 * target.
  W.slot_cap = 2 * target;
  W.off_o = off;
  off = sas_align256(off + (size_t)W.slot_cap * H * Dv * 4);
  W.off_ml = off;  // per (slot, head): float4 (m, l_w, l_e, 0)
  off = sas_align256(off + (size_t)W.slot_cap * H * 4 * 4);
  W.total = off;
  return W;
}

// ---- backward workspace: the forward's, then (bytes, each region 256-B aligned) ----
// The KV pools' gradient by key tiles (bwd_dkv_tile_kernel) reads every row's P and dS
// back from memory: the dq kernel spills them, one record per list position (2 B dS and
// 2 B P per head, heads padded to whole 32-head chunks), and in scenario 3 the resolver's
// inverse lists.  Both are bounded together: the tokens are taken in runs of chunk_tokens.
#define SAS_BWD_KEYS 128                          // keys per tile item
#define SAS_BWD_SPILL_BYTES ((size_t)2 << 30)     // bound of a run's spill and inverse lists
#define SAS_BWD_MIN_GROUP 8                       // fewest tokens per tile item
#define SAS_BWD_MAX_B 2048                        // sequences the item list handles
// Tiles for compressed rows when the table holds at most this times K rows: a tile visit
// (a token against 128 keys) costs about 17 ns of the chip's time, an atomic row 1.75 ns
// (576 adds at 330 G/s), so the two meet where a token lists about 10 of 128 rows; at a
// sixth of them (21) the tiles are ahead, with room for lists that are shorter than K.
#define SAS_BWD_DENSE 6

struct SasBwdLayout {
  size_t off_dterm, off_sterm;  // D and the sink term per (token, head)
  size_t base_total;            // without the KV pools' gradient
  size_t off_flags, off_inv, off_items, off_spill, total;
  int tile;           // key tiles for the window rows
  int cmp_rows;       // compressed rows per sequence covered by tiles (0: none)
  int stride;         // spilled list positions per token
  int row_bytes;      // bytes per spilled position
  int chunk_tokens;   // tokens per run
  int64_t item_cap;
};

SAS_HD static inline SasBwdLayout sas_bwd_layout(size_t fwd_total, int64_t T, int64_t B, int64_t H,
                                                 int scenario, int64_t win_left, int64_t K,
                                                 int64_t cmp_cap) {
  SasBwdLayout L;
  const size_t th = (size_t)(T > 0 ? T : 1) * (size_t)H;
  L.off_dterm = fwd_total;
  L.off_sterm = L.off_dterm + sas_align256(th * 4);
  L.base_total = L.off_sterm + sas_align256(th * 4);
  L.row_bytes = (int)((H + 31) / 32) * 128;
  // tiles pay where several tokens of a sequence share their rows
  L.tile = T >= 8 * B && B <= SAS_BWD_MAX_B;
  const int64_t full = sas_row_list_stride(win_left, K, scenario);
  int64_t stride = sas_row_list_stride(win_left, 0, 1);
  // Compressed rows: a tile visits every token that may list one of its 128 rows, so
  // it pays while a token lists a fair share of them; list positions fit 16 bits.
  L.cmp_rows = 0;
  if (L.tile && scenario >= 2 && full < 65536 && (scenario == 2 || cmp_cap <= SAS_BWD_DENSE * K)) {
    L.cmp_rows = (int)cmp_cap;
    stride = full;
  }
  const size_t inv_bytes = scenario == 3 ? (size_t)L.cmp_rows * 4 : 0;  // per token
  const size_t per_token = (size_t)stride * (size_t)L.row_bytes + inv_bytes;
  if (per_token > SAS_BWD_SPILL_BYTES) L.tile = L.cmp_rows = 0;
  L.stride = (int)stride;
  L.off_flags = L.off_inv = L.off_items = L.off_spill = L.total = L.base_total;
  L.chunk_tokens = (int)(T > 0 ? T : 1);
  L.item_cap = 0;
  if (!L.tile) return L;
  // (at least one: per_token is within the bound); the runs are of about equal length, in
  // whole groups of 64 tokens where the bound leaves room for that
  const int64_t most = (int64_t)(SAS_BWD_SPILL_BYTES / per_token);
  const int64_t runs = (T + most - 1) / most;
  int64_t chunk = ((T + runs - 1) / runs + 63) / 64 * 64;
  if (chunk > most) chunk = most;
  if (chunk > T) chunk = T;
  L.chunk_tokens = (int)chunk;
  // groups of a run: at most chunk / group + one partial group per sequence; tiles of a
  // group: those its window span and its compressed rows touch
  const int64_t groups = chunk / SAS_BWD_MIN_GROUP + B + 1;
  const int64_t tiles = (win_left + 64) / SAS_BWD_KEYS + 2 +
                        (L.cmp_rows + SAS_BWD_KEYS - 1) / SAS_BWD_KEYS;
  L.item_cap = groups * tiles;
  L.off_flags = L.total;
  L.total += sas_align256((size_t)(T + 1) * 4);
  L.off_inv = L.total;
  L.total += sas_align256((size_t)chunk * inv_bytes);
  L.off_items = L.total;
  L.total += sas_align256((size_t)(L.item_cap + 1) * 16);
  L.off_spill = L.total;
  L.total += sas_align256(((size_t)chunk * (size_t)stride + 1) * (size_t)L.row_bytes);
  return L;
}

// ---- kernel parameter blocks (passed by value) ----
// cu_ends (here and in the resolution's arguments): act_q holds the sequences' cumulative
// ends (q_prefix's successors), not their lengths.
struct SasPlanArgs {
  int32_t T, B, scenario, win_left, cmp_ratio, K, H, target, cu_ends;
};

struct SasFwdArgs {
  int32_t T, H, B;
  int32_t scenario, K, cmp_ratio;
  int32_t win_left, list_stride;  // row-code list capacity: win_left + 1 (+ K)
  int32_t ori_block_size, ori_table_len, ori_block_num;
  int32_t cmp_block_size, cmp_table_len, cmp_block_num;
  int64_t ori_block_stride, ori_row_stride, cmp_block_stride, cmp_row_stride;  // elements
  float scale_log2;  // softmax_scale * log2(e)
  int32_t unit_cap, split_cap;  // plan capacities (split_cap = target units)
  int32_t slot_cap;             // split partial slots in the workspace (2 * target)
  // Optional (nullptr: none): the attention dispatch's span on the GPU's 100 MHz
  // real-time counter, {earliest workgroup start, latest workgroup end}; the
  // caller fills {UINT64_MAX, 0} first.
  uint64_t* stamps;
};

// Does the plan describe this call?  Magic and version, the token and batch
// counts, the scenario, the window, the ratio (scenarios 2 and 3), the balance
// target (which sizes the plan and the partial slots) and, in scenario 3, the
// index slots per token; and the planner's own invariants held.  (Scenario 2
// plans may bound the compressed list differently: the resolver caps it at the
// call's K, and each token's row count is min(K, thr) either way.)
// Every field is read before any is compared (& rather than &&): on the device the
// reads then issue together, one memory round trip rather than one per field.
SAS_HD static inline bool plan_matches(const int* plan, const SasFwdArgs& a) {
  int f[PH_STATUS + 1];
#pragma unroll
  for (int i = 0; i <= PH_STATUS; ++i) f[i] = plan[i];
  return (f[PH_MAGIC] == SAS_PLAN_MAGIC) & (f[PH_VERSION] == SAS_PLAN_VERSION) &
         (f[PH_T] == a.T) & (f[PH_B] == a.B) & (f[PH_SCENARIO] == a.scenario) &
         (f[PH_WIN_LEFT] == a.win_left) & (a.scenario == 1 || f[PH_CMP_RATIO] == a.cmp_ratio) &
         (f[PH_TARGET] == a.split_cap) & (a.scenario != 3 || f[PH_K] == a.K) &
         (f[PH_STATUS] == 0);
}
