// sas_kernels.hip -- gfx950 kernels of the sparse shared-KV attention path.
//
//   plan_kernel     split-KV scheduler: per-token row spans (window + compressed)
//                   and work units balanced over the CUs; replaces the reference
//                   scheduler metadata.py:1018-1086 with a GPU pass that needs
//                   only the per-batch lengths.
//   resolve_kernel  compressed top-k index resolution (reference golden.py:28-66):
//                   examine the first min(K, thr) slots, -1 terminates, ids >= thr
//                   are skipped, survivors are compacted in slot order and mapped
//                   through the paged block table to pool rows.
//   combine_kernel  log-sum-exp merge of split partials.
// The attention kernel itself (bf16 / fp16 and fp8 KV) is in sas_attend.hip.
//
// Work decomposition: one work unit = (token, contiguous range of its row list);
// the row list of a token is its window rows (raw KV pool) followed by its
// compressed rows (compressed KV pool).  All heads of the token are processed by
// one workgroup (heads x keys MFMA tiles, 32 heads per wave), so each KV row is
// read from HBM once per token.
#include <hip/hip_runtime.h>

#include "sas_common.h"

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

namespace sas {

__device__ __forceinline__ int floor_div(int a, int b) {
  int q = a / b;
  if ((a % b != 0) && ((a < 0) != (b < 0))) --q;
  return q;
}

// ===========================================================================
// Planner
// ===========================================================================
struct TokInfo {
  int b, s, sg, nwin, winlo, ncmpmax;
};

// Token -> (batch, local position) through q_prefix / act_q: the owning batch is
// the last b with q_prefix[b] <= t (equal prefixes only occur for empty batches,
// which precede the batch that owns the tokens).  A token past its batch's query
// count is owned by none (b = -1); sg then records that batch (the candidate the
// kernels check the call's lengths against), or -1 when no q_prefix is <= t.
__device__ TokInfo token_info(const SasPlanArgs& a, const int* q_prefix, const int* act_q,
                              const int* seqused_kv, int t) {
  TokInfo ti{-1, 0, -1, 0, 0, 0};
  int lo = 0, hi = a.B - 1, b = -1;
  while (lo <= hi) {
    int mid = (lo + hi) >> 1;
    if (q_prefix[mid] <= t) {
      b = mid;
      lo = mid + 1;
    } else {
      hi = mid - 1;
    }
  }
  if (b < 0) return ti;
  int s = t - q_prefix[b];
  int aq = act_q[b] - (a.cu_ends ? q_prefix[b] : 0);
  ti.sg = b;
  if (s >= aq) return ti;
  int sg = seqused_kv[b] - aq + s;                    // golden.py:125
  int winlo = max(sg - a.win_left, 0);                // golden.py:130
  int nwin = max(sg + 1 - winlo, 0);                  // golden.py:129-131
  int ncmp = 0;
  if (a.scenario >= 2) {
    int thr = floor_div(sg + 1, a.cmp_ratio);         // golden.py:44, 147
    ncmp = a.K > 0 ? min(a.K, thr) : thr;             // golden.py:48 / 148 (list capacity)
    ncmp = max(ncmp, 0);
  }
  ti.b = b;
  ti.s = s;
  ti.sg = sg;
  ti.nwin = nwin;
  ti.winlo = winlo;
  ti.ncmpmax = ncmp;
  return ti;
}

constexpr int PLAN_NT = 1024;
constexpr int PLAN_WAVES = PLAN_NT / 64;
// Batches up to this many sequences have q_prefix / act_q / seqused_kv staged in LDS
// for the token lookups (larger ones search global memory).
constexpr int PLAN_LDS_B = 2048;
// Up to this many tokens, each token's row count stays in LDS between the planner's
// passes (beyond it, every pass recomputes it from the inputs).
constexpr int PLAN_LDS_T = 8192;

// Workgroup of the unit emitted k-th: within each full group of 16, emission order
// 2j and 2j + 1 go to workgroups j and j + 8 (one XCD); the last partial group keeps
// its order.  A bijection on [0, U).
__device__ __forceinline__ int xcd_pair_slot(int k, int U) {
  const int base = k & ~15;
  if (base + 16 > U) return k;
  const int r = k & 15;
  return base + (r >> 1) + 8 * (r & 1);
}

// Workgroup of the unit emitted k-th when every unit starts in the first wave of
// workgroups: consecutive runs of P = floor(U / 8) units go to one XCD (workgroups
// x, x + 8, x + 16, ... all run on XCD x mod 8), so the splits of a token, which
// each reload its query rows, and the MTP tokens of a sequence, which share their
// window rows, meet in one L2.  The last U mod 8 keep their order.  A bijection on
// [0, U).
__device__ __forceinline__ int xcd_run_slot(int k, int U) {
  const int P = U >> 3;
  if (P == 0 || k >= 8 * P) return k;
  return 8 * (k % P) + k / P;
}

__global__ __launch_bounds__(PLAN_NT) void plan_kernel(SasPlanArgs a,
                                                       const int* __restrict__ q_prefix,
                                                       const int* __restrict__ act_q,
                                                       const int* __restrict__ seqused_kv,
                                                       int* __restrict__ plan) {
  // Every pass reads its inputs from LDS or registers: nothing the kernel stores is
  // read back from global memory, and the reductions and the scan go through wave
  // shuffles with one LDS step (two barriers each).
  __shared__ int s_qp[PLAN_LDS_B], s_aq[PLAN_LDS_B], s_su[PLAN_LDS_B];
  __shared__ int s_rows[PLAN_LDS_T];  // a token's rows, -1: no sequence owns it
  __shared__ long long s_red[PLAN_WAVES];
  __shared__ int s_fit[2][PLAN_WAVES];
  __shared__ int s_wsum[3][PLAN_WAVES];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const SasPlanLayout L = sas_plan_layout(a.T, a.target);
  int* tok = plan + L.off_tok;
  int* units = plan + L.off_units;
  int* stoks = plan + L.off_split_tokens;
  int* smeta = plan + L.off_split_meta;
  const bool staged_b = a.B <= PLAN_LDS_B, staged_t = a.T <= PLAN_LDS_T;
  if (staged_b) {
    for (int i = tid; i < a.B; i += PLAN_NT) {
      s_qp[i] = q_prefix[i];
      s_aq[i] = act_q[i];
      s_su[i] = seqused_kv[i];
    }
    __syncthreads();
  }
  // (one call per source, so that each reads its own address space: a pointer that
  // may be either becomes FLAT loads)
  auto tinfo = [&](int t) -> TokInfo {
    return staged_b ? token_info(a, s_qp, s_aq, s_su, t) : token_info(a, q_prefix, act_q, seqused_kv, t);
  };

  // Token records (their first six fields) and row counts; tokens interleaved over
  // the threads, so that the record stores are contiguous.
  long long my_rows = 0, my_longest = 0;
  for (int t = tid; t < a.T; t += PLAN_NT) {
    const TokInfo ti = tinfo(t);
    int* r = tok + (size_t)t * SAS_TOK_W;
    *reinterpret_cast<int4*>(r) = make_int4(ti.b, ti.s, ti.sg, ti.nwin);
    *reinterpret_cast<int2*>(r + TK_WINLO) = make_int2(ti.winlo, ti.ncmpmax);
    const int rows = ti.b >= 0 ? ti.nwin + ti.ncmpmax : -1;
    if (staged_t) s_rows[t] = rows;
    if (rows >= 0) {
      my_rows += rows;
      my_longest = max(my_longest, (long long)rows);
    }
  }
  __syncthreads();
  // token t's rows (-1: no sequence owns it)
  auto tok_rows = [&](int t) -> int {
    if (staged_t) return s_rows[t];
    const TokInfo ti = tinfo(t);
    return ti.b >= 0 ? ti.nwin + ti.ncmpmax : -1;
  };
  // Block-wide sum (max_op: maximum); every thread gets the result.
  auto block_reduce = [&](long long v, bool max_op) -> long long {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      const long long o = __shfl_xor(v, off);
      v = max_op ? max(v, o) : v + o;
    }
    __syncthreads();  // earlier readers of s_red are done
    if (lane == 0) s_red[wave] = v;
    __syncthreads();
    long long r = s_red[0];
#pragma unroll
    for (int i = 1; i < PLAN_WAVES; ++i) r = max_op ? max(r, s_red[i]) : r + s_red[i];
    return r;
  };
  const long long R = block_reduce(my_rows, false);
  long long chunk = (R + a.target - 1) / a.target;
  if (chunk < SAS_MIN_CHUNK) chunk = SAS_MIN_CHUNK;
  chunk = (chunk + SAS_TILE - 1) / SAS_TILE * SAS_TILE;

  // From here on each thread owns a contiguous range of tokens (the scan below gives
  // its first unit, slot and split-token index).
  const int per = (a.T + PLAN_NT - 1) / PLAN_NT;
  const int t0 = min(a.T, tid * per), t1 = min(a.T, t0 + per);
  // At most `target` tokens: the smallest chunk (a multiple of the tile) whose units
  // number at most `target`, so that every unit starts in the first wave of
  // workgroups (and the attention kernel, whose units then resolve their own rows,
  // launches exactly `target` workgroups).  R / target alone leaves a second, partial
  // wave of units after the first, which doubles the time of the CUs that run one,
  // and it splits more tokens (each split unit writes a partial the combine pass
  // reads back).
  if (a.T <= a.target) {
    const long long longest = block_reduce(my_longest, true);
    // In tiles: the smallest chunk that fits lies in [ta, tb], and tb (one unit per
    // token) fits.  Each pass tests PLAN_WAVES chunks at once, wave w the one of
    // ta + (w + 1) (tb - ta) / (PLAN_WAVES + 1) tiles (its lanes striding over the
    // tokens), and keeps the interval between the largest that does not fit and the
    // smallest that does: a 17-way search, one barrier per pass (the flags alternate
    // between two buffers, so no pass overwrites flags another wave still reads).
    // (32-bit divides: a token's rows and the chunk fit, and the GPU has no 64-bit
    // integer divide.)
    long long ta = chunk / SAS_TILE;
    long long tb = max(ta, (longest + SAS_TILE - 1) / SAS_TILE);
    int buf = 0;
    while (ta < tb) {
      const long long n = tb - ta;
      const unsigned c = (unsigned)((ta + (long long)(wave + 1) * n / (PLAN_WAVES + 1)) * SAS_TILE);
      long long u = 0;
      for (int t = lane; t < a.T; t += 64) {
        const unsigned rows = (unsigned)max(tok_rows(t), 0);
        u += rows > c ? (long long)((rows + c - 1) / c) : 1;
      }
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) u += __shfl_xor(u, off);
      if (lane == 0) s_fit[buf][wave] = u <= a.target;
      __syncthreads();
      int k = PLAN_WAVES;  // the first chunk tested that fits
      for (int i = PLAN_WAVES - 1; i >= 0; --i)
        if (s_fit[buf][i]) k = i;
      if (k < PLAN_WAVES) tb = ta + (long long)(k + 1) * n / (PLAN_WAVES + 1);
      if (k > 0) ta += (long long)k * n / (PLAN_WAVES + 1) + 1;
      buf ^= 1;
    }
    chunk = ta * SAS_TILE;
  }

  // a token's split count (32-bit division when the chunk fits, as it always does in
  // practice: a token's rows fit an int)
  auto splits_of = [&](long long rows) -> int {
    if (rows <= chunk) return 1;
    if (chunk <= 0x7fffffffll) return (int)(((unsigned)rows + (unsigned)chunk - 1u) / (unsigned)chunk);
    return (int)((rows + chunk - 1) / chunk);
  };
  int my_u = 0, my_s = 0, my_k = 0;
  for (int t = t0; t < t1; ++t) {
    const long long rows = max(tok_rows(t), 0);
    int splits = splits_of(rows);
    my_u += splits;
    if (splits > 1) {
      my_s += splits;
      my_k += 1;
    }
  }
  // Inclusive scans over the threads: within each wave by shuffles, then across the
  // waves' totals.
  int iu = my_u, is = my_s, ik = my_k;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int ou = __shfl_up(iu, off), os = __shfl_up(is, off), ok = __shfl_up(ik, off);
    if (lane >= off) {
      iu += ou;
      is += os;
      ik += ok;
    }
  }
  if (lane == 63) {
    s_wsum[0][wave] = iu;
    s_wsum[1][wave] = is;
    s_wsum[2][wave] = ik;
  }
  __syncthreads();
  int U = 0, NS = 0, NK = 0, pu = 0, ps = 0, pk = 0;
#pragma unroll
  for (int i = 0; i < PLAN_WAVES; ++i) {
    if (i < wave) {
      pu += s_wsum[0][i];
      ps += s_wsum[1][i];
      pk += s_wsum[2][i];
    }
    U += s_wsum[0][i];
    NS += s_wsum[1][i];
    NK += s_wsum[2][i];
  }
  int ub = pu + iu - my_u, sb = ps + is - my_s, kb = pk + ik - my_k;
  const bool decode_like = (long long)a.T <= 4 * (long long)a.B;
  // runs: every unit starts at once and some token is split (its units share Q rows)
  const bool runs = U <= a.target && U > a.T;
  for (int t = t0; t < t1; ++t) {
    int* r = tok + (size_t)t * SAS_TOK_W;
    const int rv = tok_rows(t);
    const long long rows = max(rv, 0);
    const int splits = splits_of(rows);
    *reinterpret_cast<int2*>(r + TK_SPLITS) = make_int2(splits, splits > 1 ? sb : -1);
    long long ct = rows;
    if (splits > 1) ct = ((rows + splits - 1) / splits + SAS_TILE - 1) / SAS_TILE * SAS_TILE;
    for (int i = 0; i < splits; ++i) {
      // units are emitted in reverse order so the longest (latest prefill) tokens start
      // first.  Decode-like plans (at most 4 query tokens per sequence) also keep
      // neighbouring units on one XCD: runs of U / 8 when all units start at once and
      // tokens are split, else pairs 8 workgroups apart (workgroups go to the 8 XCDs
      // in turn).
      const int k = U - 1 - (ub + i);
      const int slot = !decode_like ? k : runs ? xcd_run_slot(k, U) : xcd_pair_slot(k, U);
      if (slot < 0 || slot >= L.unit_cap) continue;  // (U <= unit_cap: flagged below if not)
      long long r0 = (long long)i * ct, r1 = r0 + ct < rows ? r0 + ct : rows;
      *reinterpret_cast<int4*>(units + (size_t)slot * SAS_UNIT_W) =
          make_int4(t, (int)r0, (int)r1, rv >= 0 ? i : -1);
    }
    ub += splits;
    if (splits > 1) {
      if (kb < L.split_cap) {
        stoks[kb] = t;
        smeta[2 * kb] = splits;
        smeta[2 * kb + 1] = sb;
      }
      ++kb;
      sb += splits;
    }
  }
  if (tid == 0) {
    plan[PH_MAGIC] = SAS_PLAN_MAGIC;
    plan[PH_VERSION] = SAS_PLAN_VERSION;
    plan[PH_T] = a.T;
    plan[PH_UNITS] = U;
    plan[PH_CHUNK] = (int)chunk;
    plan[PH_TARGET] = a.target;
    plan[PH_NSPLIT_TOKENS] = NK;
    plan[PH_NSLOTS] = NS;
    plan[PH_TOTAL_ROWS_LO] = (int)(R & 0xffffffff);
    plan[PH_TOTAL_ROWS_HI] = (int)(R >> 32);
    plan[PH_H] = a.H;
    plan[PH_UNIT_CAP] = (int)L.unit_cap;
    plan[PH_SCENARIO] = a.scenario;
    plan[PH_K] = a.K;
    plan[PH_WIN_LEFT] = a.win_left;
    plan[PH_B] = a.B;
    plan[PH_CMP_RATIO] = a.cmp_ratio;
    // The capacities hold by construction (split tokens have more rows than the
    // chunk >= R / target, so fewer than `target` of them exist, with at most
    // 2 * target units; every token has at most rows / chunk + 1 units); a plan
    // that broke one is refused by every kernel.
    int status = 0;
    if ((long long)U > L.unit_cap) status |= PS_UNITS_OVER_CAP;
    if ((long long)NS > 2 * (long long)a.target) status |= PS_SLOTS_OVER_CAP;
    if ((long long)NK > L.split_cap) status |= PS_SPLIT_TOKENS_OVER_CAP;
    if (a.T <= a.target && U > a.target) status |= PS_UNITS_OVER_TARGET;
    plan[PH_STATUS] = status;
    for (int i = PH_STATUS + 1; i < SAS_PLAN_HDR; ++i) plan[i] = 0;
  }
}

// ===========================================================================
// Row resolution.  Writes each token's row-code list: the
// window rows (golden.py:129-131, paged as golden.py:247-268) and, in scenario 3,
// the resolved compressed rows (golden.py:28-66).  A code is a flat pool row
// (page * block_size + offset) or -1 for a row the reference reads as zeros
// (unused page).  Window codes index the raw pool, later codes the compressed pool.
// ===========================================================================
// The row every -1 code reads (zeros).
__device__ __attribute__((aligned(16))) uint8_t g_zero_row[1152] = {};

// Pool address of a row code (-1: the shared zero row).
__device__ __forceinline__ uint64_t code_addr(int code, const uint8_t* pool, int block_size,
                                              int64_t block_stride, int64_t row_stride, int esz) {
  if (code < 0) return (uint64_t)g_zero_row;
  const int page = (int)((unsigned)code / (unsigned)block_size), off = code - page * block_size;
  return (uint64_t)(pool + ((size_t)page * block_stride + (size_t)off * row_stride) * esz);
}

__device__ __forceinline__ int paged_code(const int* __restrict__ bt_row, int table_len,
                                          int block_size, int block_num, int pos) {
  const int blk = (int)((unsigned)pos / (unsigned)block_size);  // pos >= 0
  const int page = blk < table_len ? bt_row[blk] : -1;
  return (page < 0 || page >= block_num) ? -1 : page * block_size + (pos - blk * block_size);
}

// A token is resolved by one workgroup of RS_NT threads: the resolver's own, or the
// four-wave attention kernel's of one of its units.
constexpr int RS_NT = 256;
constexpr int RS_WAVES = RS_NT / 64;

// Workgroup barrier for the resolver: its threads exchange data only through LDS,
// so it waits for LDS operations alone.  (__syncthreads() would also drain every
// outstanding global load and store, putting their latency on each pass.)
__device__ __forceinline__ void rs_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}
constexpr int RS_PER = 8;  // slabs of RS_NT index slots per pass

constexpr int RS_CBT_LDS = 4096;  // compressed block-table entries staged in LDS

// LDS of one token's resolution (the attention kernel lends it the start of its
// tile ring, which is empty until the unit's first DMA).
struct RsShared {
  int wmin[RS_WAVES];
  int cnt[RS_PER][RS_WAVES];
  int cbt[RS_CBT_LDS];
};

// Inputs and outputs of row resolution.
struct SasResolveArgs {
  const int* q_prefix;    // the call's lengths (per batch)
  const int* act_q;
  int cu_ends;            // act_q holds cumulative ends
  const int* seqused_kv;
  const int* ori_bt;
  const int* idx;
  const int* cmp_bt;
  int* rows;              // row codes (nullptr: not written)
  int2* tok;              // per token (window rows, compressed rows) (nullptr: not written)
  uint64_t* addr;         // row addresses (nullptr: the rows were resolved beforehand)
  const uint8_t* ori_kv;
  const uint8_t* cmp_kv;
  int esz;                // bytes per KV element
  const float* ori_scale;
  const float* cmp_scale;
  float* scale;           // fp8: s, then (T * list_stride on) 1 / s; nullptr for 16-bit KV
  int t0;                 // the launch's first token
  // INV: scenario 3's inverse list, [tokens of the launch][inv_rows]: for compressed row j of
  // the token's sequence, the list position of its first occurrence (low 16 bits) and how
  // often it is listed (high 16 bits; 0: not).  Entries below the token's threshold are set.
  uint32_t* inv;
  int inv_rows;
  int* local;             // the workspace's plan, to which a caller's is copied (resolve_kernel)
  int copies;             // by that many workgroups (0: no copy)
};

// List positions [lo, hi) of token t (its window rows, then its compressed rows)
// resolved into codes, pool addresses and (fp8) scales, by the workgroup's RS_NT
// threads.  The first min(K, thr) index slots are taken in passes of RS_PER slabs
// of RS_NT slots; thread i owns slot i of every slab, so each load and store
// instruction of a wave covers 64 consecutive slots.  The first -1 (a block-wide
// minimum) ends the list, ids outside [0, thr) are skipped, and the survivors keep
// their slot order: a wave ranks its survivors of a slab with one ballot, and the
// per-(slab, wave) counts go through LDS.  Returns the token's compressed row count
// when the scan reached the list's end, else a number >= hi - nwin (the scan stops
// after the pass that resolves position hi - 1), and sets nwin_live to the token's
// window row count.  A token no batch owns, or a refused plan, resolves to nothing.
//
// The plan gives the token's batch and position (b, s); its window and threshold
// come from the call's seqused_kv, as the reference's kernel reads the lengths on
// every call: a plan stays valid while the KV lengths change (a decode loop that
// reuses its metadata).  Where the call's q_prefix / act_q no longer give the token
// to batch b at position s (or give a token the plan left unowned to its candidate
// batch), the token is refused: nwin_live = -1, nothing is resolved.
template <bool INV>
__device__ int resolve_rows(const SasFwdArgs& a, const int* tk, bool plan_ok, int t, int lo, int hi,
                            RsShared& sh, const SasResolveArgs& r, int& nwin_live) {
  const int tid = threadIdx.x;
  const int lane = tid & 63, w = tid >> 6;
  const int* ir = r.idx + (size_t)t * a.K;
  // This thread's slot of every slab of the pass at c0, all loaded before any is
  // used (-2: at or past the bound).
  auto load_slots = [&](int (&v)[RS_PER], int c0, int bound) {
#pragma unroll
    for (int k = 0; k < RS_PER; ++k) {
      const int sl = c0 + k * RS_NT + tid;
      v[k] = sl < bound ? ir[sl] : -2;
    }
  };
  // First memory round trip: the token's plan record and, independent of it, the
  // first pass of its index slots.
  int v0[RS_PER];
  if (a.scenario == 3) load_slots(v0, 0, a.K);
  nwin_live = 0;
  if (!plan_ok) return 0;
  const int b = tk[TK_B], s = tk[TK_S], sg_plan = tk[TK_SG];
  if (b < 0 || b >= a.B) {
    // unowned when the plan was built: refused if the call's lengths give the token
    // to the candidate batch (sg_plan)
    if (b < 0 && sg_plan >= 0 && sg_plan < a.B) {
      const int q0 = r.q_prefix[sg_plan], nq = r.act_q[sg_plan] - (r.cu_ends ? q0 : 0);
      if (q0 <= t && t - q0 < nq) nwin_live = -1;
    }
    return 0;
  }
  // The batch's live lengths, issued before (and so landing with) the block-table
  // loads below, which start at the plan's window.
  const int q0 = r.q_prefix[b], nq = r.act_q[b] - (r.cu_ends ? q0 : 0), kv_live = r.seqused_kv[b];
  int* out = r.rows ? r.rows + (size_t)t * a.list_stride : nullptr;
  uint64_t* aout = r.addr + (size_t)t * a.list_stride;
  // fp8 KV: each row's dequantisation scale s and 1 / s beside its address (a -1
  // code reads the zero row: s = 1, so that its P counts in the output normaliser
  // as a zero row of a 16-bit pool does)
  float* sout = r.scale ? r.scale + (size_t)t * a.list_stride : nullptr;
  const size_t inv_off = (size_t)a.T * a.list_stride;  // the 1 / s list follows the s list
  auto put_scale = [&](int p, float s) {
    sout[p] = s;
    sout[inv_off + p] = s != 0.f ? 1.f / s : 0.f;
  };
  // Second: the window's block-table entries and the batch's compressed block-table
  // row, staged in LDS so the per-id page lookups below stay on chip.
  const int* cbt_g = r.cmp_bt + (size_t)b * a.cmp_table_len;
  const bool cbt_lds = a.scenario >= 2 && a.cmp_table_len <= RS_CBT_LDS;
  if (cbt_lds)
    for (int i = tid; i < a.cmp_table_len; i += RS_NT) sh.cbt[i] = cbt_g[i];
  const int* obt = r.ori_bt + (size_t)b * a.ori_table_len;
  auto window = [&](int nwin, int winlo) {
    for (int p = lo + tid; p < min(hi, nwin); p += RS_NT) {
      const int code = paged_code(obt, a.ori_table_len, a.ori_block_size, a.ori_block_num, winlo + p);
      if (out) out[p] = code;
      aout[p] = code_addr(code, r.ori_kv, a.ori_block_size, a.ori_block_stride, a.ori_row_stride, r.esz);
      if (sout) put_scale(p, code < 0 ? 1.f : r.ori_scale[code]);
    }
  };
  // the window at the plan's lengths (the usual case: the call's are the same)
  window(min(tk[TK_NWIN], a.win_left + 1), tk[TK_WINLO]);
  if (q0 + s != t || s < 0 || s >= nq) {  // the call gives this token to another batch
    nwin_live = -1;
    return 0;
  }
  const int sg = kv_live - nq + s;                               // golden.py:125
  const int winlo = max(sg - a.win_left, 0);                     // golden.py:130
  const int nwin = min(max(sg + 1 - winlo, 0), a.win_left + 1);  // golden.py:129-131
  if (sg != sg_plan) {  // the KV length changed since the plan: the window again
    window(nwin, winlo);
    // Positions from nwin on, written above at the plan's window by one thread, may
    // take compressed rows below from another: every store lands before those.
    __syncthreads();
  }
  nwin_live = nwin;
  if (a.scenario == 1) return 0;
  rs_barrier();  // sh.cbt
  const int thr = floor_div(sg + 1, a.cmp_ratio);
  // compressed rows j sit at list position nwin + j; [lo, hi) holds j in [jlo, jhi)
  const int jlo = max(lo - nwin, 0), jhi = hi - nwin;
  if (a.scenario == 2) {  // golden.py:146-150: every compressed row below thr
    const int n = max(min(thr, a.K), 0);
    // One loop per source of the table row: a pointer that may be either (LDS or
    // global) turns its loads into FLAT instructions.
    auto cmp_rows = [&](const int* bt) {
      for (int j = jlo + tid; j < min(n, jhi); j += RS_NT) {
        const int code = paged_code(bt, a.cmp_table_len, a.cmp_block_size, a.cmp_block_num, j);
        if (out) out[nwin + j] = code;
        aout[nwin + j] = code_addr(code, r.cmp_kv, a.cmp_block_size, a.cmp_block_stride, a.cmp_row_stride, r.esz);
        if (sout) put_scale(nwin + j, code < 0 ? 1.f : r.cmp_scale[code]);
      }
    };
    if (cbt_lds)
      cmp_rows(sh.cbt);
    else
      cmp_rows(cbt_g);
    return n;
  }
  const int limit = max(min(a.K, thr), 0);  // golden.py:48
  typedef __attribute__((address_space(1))) uint32_t g_u32;
  g_u32* inv = nullptr;
  if constexpr (INV) {
    if (r.inv) {
      inv = (g_u32*)(uintptr_t)(r.inv + (size_t)(t - r.t0) * r.inv_rows);
      for (int i = tid; i < min(thr, r.inv_rows); i += RS_NT) inv[i] = 0;
      __syncthreads();  // the zeros are in place before the first count below
    }
  }
  // Passes of RS_PER slabs of RS_NT slots; the terminator, the survivors and their
  // slot-order positions come from ballots and two LDS exchanges per pass.
  int emitted = 0;  // compressed rows found so far (block-uniform)
  const uint64_t below = (1ull << lane) - 1;  // lanes ranked before this one
  for (int c0 = 0; c0 < limit && emitted < jhi; c0 += RS_NT * RS_PER) {
    int v[RS_PER];
    if (c0 == 0) {
#pragma unroll
      for (int k = 0; k < RS_PER; ++k) v[k] = k * RS_NT + tid < limit ? v0[k] : -2;
    } else {
      load_slots(v, c0, limit);
    }
    // golden.py:52-53: the first -1 terminates the list.  Slab k precedes slab
    // k + 1, and within a slab wave w's 64 slots precede wave w + 1's, so a wave's
    // first -1 is the lowest lane of its first slab that has one.
    int first = limit;
#pragma unroll
    for (int k = RS_PER - 1; k >= 0; --k) {
      const uint64_t m = __ballot(v[k] == -1);
      if (m) first = c0 + k * RS_NT + w * 64 + (int)__builtin_ctzll(m);
    }
    if (lane == 0) sh.wmin[w] = first;
    rs_barrier();
    int term = sh.wmin[0];
#pragma unroll
    for (int j = 1; j < RS_WAVES; ++j) term = min(term, sh.wmin[j]);
    // golden.py:58-59: ids at or beyond thr are skipped (other negatives too).
    // Survivors of slab k are ranked within the wave by a ballot; the counts of
    // every (slab, wave) give each wave's base position.
    bool keep[RS_PER];
    int rank[RS_PER];
#pragma unroll
    for (int k = 0; k < RS_PER; ++k) {
      keep[k] = c0 + k * RS_NT + tid < term && v[k] >= 0 && v[k] < thr;
      const uint64_t m = __ballot(keep[k]);
      rank[k] = __popcll(m & below);
      if (lane == 0) sh.cnt[k][w] = __popcll(m);
    }
    rs_barrier();
    int pos[RS_PER];
    int total = emitted;
#pragma unroll
    for (int k = 0; k < RS_PER; ++k) {
      int before = 0, slab = 0;
#pragma unroll
      for (int j = 0; j < RS_WAVES; ++j) {
        const int c = sh.cnt[k][j];
        before += j < w ? c : 0;
        slab += c;
      }
      pos[k] = total + before + rank[k];
      total += slab;
      keep[k] = keep[k] && pos[k] >= jlo && pos[k] < jhi;  // inside [lo, hi)
    }
    // The page lookups of the pass, then its codes, then every scale load, then the
    // stores: each load waits only for what it depends on (the block-table row is
    // read through its own address space, so the lookups issue together).
    int code[RS_PER], blk[RS_PER], page[RS_PER];
#pragma unroll
    for (int k = 0; k < RS_PER; ++k) {
      blk[k] = keep[k] ? (int)((unsigned)v[k] / (unsigned)a.cmp_block_size) : -1;
      if (blk[k] >= a.cmp_table_len) blk[k] = -1;
    }
    if (cbt_lds) {
#pragma unroll
      for (int k = 0; k < RS_PER; ++k) page[k] = blk[k] >= 0 ? sh.cbt[blk[k]] : -1;
    } else {
      // typed global: two loads of one pointer type would be merged into one from a
      // pointer that may be either, a FLAT load
      typedef __attribute__((address_space(1))) const int g_int;
      const g_int* cbt = (const g_int*)cbt_g;
#pragma unroll
      for (int k = 0; k < RS_PER; ++k) page[k] = blk[k] >= 0 ? cbt[blk[k]] : -1;
    }
#pragma unroll
    for (int k = 0; k < RS_PER; ++k)
      code[k] = (page[k] < 0 || page[k] >= a.cmp_block_num)
                    ? -1
                    : page[k] * a.cmp_block_size + (v[k] - blk[k] * a.cmp_block_size);
    float sc[RS_PER];
    if (sout) {
#pragma unroll
      for (int k = 0; k < RS_PER; ++k) sc[k] = code[k] >= 0 ? r.cmp_scale[code[k]] : 1.f;
    }
#pragma unroll
    for (int k = 0; k < RS_PER; ++k)
      if (keep[k]) {
        const int p = nwin + pos[k];
        if (out) out[p] = code[k];
        if (sout) put_scale(p, sc[k]);
        aout[p] = code_addr(code[k], r.cmp_kv, a.cmp_block_size, a.cmp_block_stride, a.cmp_row_stride, r.esz);
        if constexpr (INV) {
          if (inv && v[k] < r.inv_rows &&
              __hip_atomic_fetch_add(inv + v[k], 1u << 16, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < (1u << 16))
            __hip_atomic_fetch_or(inv + v[k], (uint32_t)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
      }
    emitted = total;
    if (term < limit) break;  // the list ended in this pass
    rs_barrier();          // wmin / cnt are rewritten by the next pass
  }
  return emitted;
}

// The resolver, one workgroup (RS_NT threads) per token: its whole list.
//
// Ahead of those, with r.local, r.copies workgroups that copy the caller's plan (header,
// token records, units) to the workspace's, which is as long as this call's plan whatever
// the caller's buffer holds: the entry points take no plan size, and a plan built for fewer
// tokens or a smaller target is a shorter buffer, so nothing past its header is read unless
// the header matches (a refused plan leaves a header of zeros).  The kernels behind the
// resolver then read a unit's record together with the header that vouches for it, one
// memory round trip of each unit's start: a window-only prefill of 8,192 tokens (64
// heads, d_qk 512, fp16) took 1 to 2% longer where they read a caller's header first (332
// -> 336 .. 339 us).  (In workgroups of their own: at the end of every token's the copy
// made the resolver 2 us longer.)
constexpr int RS_COPY = 8 * RS_NT;  // plan entries per copying workgroup
template <bool INV>
__global__ __launch_bounds__(RS_NT) void resolve_kernel(SasFwdArgs a, const int* __restrict__ plan,
                                                        SasResolveArgs r) {
  __shared__ RsShared sh;
  // A plan built for other arguments is refused: every token resolves to no rows,
  // the attention kernel writes zeros and the combine kernel sets the status word.
  const bool plan_ok = plan_matches(plan, a);
  const int t = (int)blockIdx.x - r.copies + r.t0;
  if ((int)blockIdx.x < r.copies) {
    // (to the unit capacity, which a matching plan's buffer holds)
    const int64_t n = SAS_PLAN_HDR + (int64_t)a.T * SAS_TOK_W + (int64_t)a.unit_cap * SAS_UNIT_W;
    const int64_t i0 = (int64_t)blockIdx.x * RS_COPY + threadIdx.x;
    if (!plan_ok) {
      if (i0 < SAS_PLAN_HDR) r.local[i0] = 0;
      return;
    }
#pragma unroll
    for (int k = 0; k < RS_COPY / RS_NT; ++k)
      if (i0 + k * RS_NT < n) r.local[i0 + k * RS_NT] = plan[i0 + k * RS_NT];
    return;
  }
  const int* tk = plan + SAS_PLAN_HDR + (size_t)t * SAS_TOK_W;
  int nwin = 0;
  const int n = resolve_rows<INV>(a, tk, plan_ok, t, 0, a.list_stride, sh, r, nwin);
  if (threadIdx.x == 0 && r.tok) r.tok[t] = make_int2(nwin, nwin < 0 ? 0 : n);
}

// ===========================================================================
// 16-bit conversions (attention and combine kernels)
// ===========================================================================
// float -> 16-bit payload of the query dtype, round to nearest even.
template <int QT>
__device__ __forceinline__ uint32_t to_q16(float x) {
  if constexpr (QT == 0)
    return (uint32_t)__builtin_bit_cast(uint16_t, (__bf16)x);
  else
    return (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)x);
}

// Two floats -> two 16-bit values of the query dtype (round to nearest even),
// packed low = a, high = b: one v_cvt_pk_bf16_f32 for bf16.
template <int QT>
__device__ __forceinline__ uint32_t pack2_q16(float a, float b) {
  if constexpr (QT == 0) {
    typedef __bf16 b2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, b2{(__bf16)a, (__bf16)b});
  } else {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, h2{(_Float16)a, (_Float16)b});
  }
}

// 16-bit payload of the query dtype -> float (exact).
template <int QT>
__device__ __forceinline__ float q16_to_f32(uint32_t v) {
  if constexpr (QT == 0)
    return __uint_as_float(v << 16);
  else
    return (float)__builtin_bit_cast(_Float16, (uint16_t)v);
}

// acc + the two 16-bit values packed in v (exact products with 1, fp32 sum).
template <int QT>
__device__ __forceinline__ float sum2_q16(uint32_t v, float acc) {
  if constexpr (QT == 0) {
    typedef __bf16 b2 __attribute__((ext_vector_type(2)));
    const b2 one = {(__bf16)1.f, (__bf16)1.f};
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(b2, v), one, acc, false);
  } else {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    const h2 one = {(_Float16)1.f, (_Float16)1.f};
    return __builtin_amdgcn_fdot2(__builtin_bit_cast(h2, v), one, acc, false);
  }
}

// Split partials: with bf16 queries a split unit stores its O normalised, in fp16
// (11 significant bits against the bf16 output's 8; the merge runs in fp32; a unit
// with some |O| / l_w at fp16's range is redone and stores fp32); with fp16 queries,
// whose output would feel a second rounding of the same width, un-normalised in fp32.
template <int QT>
constexpr bool PART16 = QT == 0;

// ===========================================================================
// Split-KV merge (log-sum-exp) of one (token, head): lane l merges columns
// [8 l, 8 l + 8) of the d_v = 512 partial outputs.  A partial holds O and its two
// normalisers (l_w: sum of the rounded P that entered O, for the output; l_e: sum
// of the exact P, for the LSE) in its own frame m; the merge rescales each by
// 2^(m_s - max_s m_s).  Only split 0 carries the sink, so it enters once.
// ===========================================================================
__device__ __forceinline__ float wave_max(float x) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) x = fmaxf(x, __shfl_xor(x, off));
  return x;
}
__device__ __forceinline__ float wave_sum(float x) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off);
  return x;
}

// Log-sum-exp merge of the S split partials of head h of token t (partial slots
// base ..), by one wave: lane l owns d = 8 l .. 8 l + 7.  Partial row (slot, h) sits
// at float offset (slot H + h) d_v, with its record (m, l_w, l_e, fmt): fmt 0, the
// un-normalised O in fp32 (2 KB); fmt 1, O / l_w in fp16 (the first 1 KB).  The
// records are read 64 at a time (lane j holds record j of a chunk).  With at most
// COMBINE_BATCH splits the rows are read all at once before any is accumulated, as
// fp16 together with the records (one memory round trip for both; a row the record
// says is fp32 is read again); with more, in batches of COMBINE_BATCH_LONG.
constexpr int COMBINE_BATCH = 8;
// Rows per batch of the general merge (more than COMBINE_BATCH splits; the next batch
// is loaded while one is accumulated): few rows in flight, so that the common path's
// register count, not this rare one's, sets the kernel's occupancy.
constexpr int COMBINE_BATCH_LONG = 2;

// rows s0 + j0 .. s0 + j0 + NB - 1 of a chunk of n rows, 16 B per lane: the fp16
// view (fmt 1) when PART16, else fp32 (8 floats as two 16-B halves)
template <int QT, int NB>
using MergeRows = u32x4_t[NB][PART16<QT> ? 1 : 2];

template <int QT>
__device__ __forceinline__ const float* partial_row(const float* ws_o, int H, int h, int slot) {
  return ws_o + ((size_t)slot * H + h) * 512;
}

template <int QT>
__device__ __forceinline__ float4 merge_record(const float* ws_ml, int H, int h, int S, int base, int s0) {
  const int lane = threadIdx.x & 63;
  return s0 + lane < S ? reinterpret_cast<const float4*>(ws_ml)[(size_t)(base + s0 + lane) * H + h]
                       : make_float4(-INFINITY, 0.f, 0.f, 0.f);
}

template <int QT, int NB>
__device__ __forceinline__ void merge_load(MergeRows<QT, NB>& v, const float* ws_o, int H, int h,
                                           int base, int s0, int j0, int n) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    if (j0 + j >= n) break;  // (wave-uniform)
    const u32x4_t* src = reinterpret_cast<const u32x4_t*>(partial_row<QT>(ws_o, H, h, base + s0 + j0 + j));
    if constexpr (PART16<QT>) {
      v[j][0] = src[lane];
    } else {
      v[j][0] = src[2 * lane];
      v[j][1] = src[2 * lane + 1];
    }
  }
}

// The merge of one head given its first record chunk and first row batch (loaded
// beforehand, so that several heads' loads can be in flight together).
template <int QT, int NB>
__device__ __forceinline__ void merge_finish(int t, int h, int H, int S, int base,
                                             const float* __restrict__ ws_o,
                                             const float* __restrict__ ws_ml, const float4 rec0,
                                             const MergeRows<QT, NB>& v0, uint16_t* __restrict__ out,
                                             float* __restrict__ lse) {
  constexpr int DV = 512;
  const int lane = threadIdx.x & 63;
  float mx = rec0.x;
  for (int s0 = 64; s0 < S; s0 += 64) mx = fmaxf(mx, merge_record<QT>(ws_ml, H, h, S, base, s0).x);
  mx = wave_max(mx);  // the merged frame
  float l = 0.f, le = 0.f;
  float o[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  for (int s0 = 0; s0 < S; s0 += 64) {
    const float4 rec = s0 == 0 ? rec0 : merge_record<QT>(ws_ml, H, h, S, base, s0);
    const float wgt = rec.x == -INFINITY ? 0.f : exp2f(rec.x - mx);
    l += wgt * rec.y;
    le += wgt * rec.z;
    // the row's weight: an fp16 row is O / l_w
    const float wrow = rec.w != 0.f ? wgt * rec.y : wgt;
    const int n = min(64, S - s0);
    // batch j0 + NB is loaded before batch j0 is accumulated
    MergeRows<QT, NB> vn;
    for (int j0 = 0; j0 < n; j0 += NB) {
      MergeRows<QT, NB> v;
      if (s0 == 0 && j0 == 0) {
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
          for (int k = 0; k < (PART16<QT> ? 1 : 2); ++k) v[j][k] = v0[j][k];
      } else if (j0 == 0) {
        merge_load<QT, NB>(v, ws_o, H, h, base, s0, j0, n);
      } else {
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
          for (int k = 0; k < (PART16<QT> ? 1 : 2); ++k) v[j][k] = vn[j][k];
      }
      if (j0 + NB < n) merge_load<QT, NB>(vn, ws_o, H, h, base, s0, j0 + NB, n);
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        if (j0 + j >= n) break;
        const float w = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(wrow), j0 + j));
        float x[8];
        if constexpr (PART16<QT>) {
          const bool f16 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(rec.w), j0 + j)) != 0.f;
          if (f16) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              x[2 * e] = q16_to_f32<1>(v[j][0][e] & 0xffffu);
              x[2 * e + 1] = q16_to_f32<1>(v[j][0][e] >> 16);
            }
          } else {  // a redone unit's fp32 row
            const u32x4_t* src =
                reinterpret_cast<const u32x4_t*>(partial_row<QT>(ws_o, H, h, base + s0 + j0 + j));
            const u32x4_t a = src[2 * lane], b = src[2 * lane + 1];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              x[e] = __uint_as_float(a[e]);
              x[4 + e] = __uint_as_float(b[e]);
            }
          }
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            x[e] = __uint_as_float(v[j][0][e]);
            x[4 + e] = __uint_as_float(v[j][1][e]);
          }
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] += w * x[e];
      }
    }
  }
  l = wave_sum(l);
  le = wave_sum(le);
  const float inv = l > 0.f ? 1.f / l : 0.f;
  u32x4_t ov;
#pragma unroll
  for (int e = 0; e < 4; ++e) ov[e] = to_q16<QT>(o[2 * e] * inv) | (to_q16<QT>(o[2 * e + 1] * inv) << 16);
  // (non-temporal, as the attention kernel's output rows)
  __builtin_nontemporal_store(ov, reinterpret_cast<u32x4_t*>(out + ((size_t)t * H + h) * DV) + lane);
  if (lse && lane == 0) lse[(size_t)t * H + h] = (mx + __log2f(le)) * 0.6931471805599453f;
}

template <int QT>
__device__ __forceinline__ void combine_head(int t, int h, int H, int S, int base,
                                             const float* __restrict__ ws_o,
                                             const float* __restrict__ ws_ml,
                                             uint16_t* __restrict__ out, float* __restrict__ lse) {
  // One memory round trip for the records and the first rows: the rows depend on
  // the slot range alone, not on the merged frame.
  const float4 rec0 = merge_record<QT>(ws_ml, H, h, S, base, 0);
  MergeRows<QT, COMBINE_BATCH_LONG> v0;
  merge_load<QT, COMBINE_BATCH_LONG>(v0, ws_o, H, h, base, 0, 0, min(64, S));
  merge_finish<QT, COMBINE_BATCH_LONG>(t, h, H, S, base, ws_o, ws_ml, rec0, v0, out, lse);
}

// log2(e): logits are kept in log2 units (scale_log2 = softmax_scale * log2(e)).
constexpr float LOG2E = 1.4426950408889634f;

// ===========================================================================
// Split combine: one wave per (split token, head), grid-stride over the split
// tokens the plan recorded (a call without split tokens exits at once).
// ===========================================================================
constexpr int COMBINE_WAVES = 4;  // waves per workgroup
// Workgroups per CU the kernel is compiled for (and launched with): every wave runs its
// (token, head) items one memory round trip after another, so more resident waves keep
// more of them in flight.  fp32 partials (fp16 queries) take twice the row registers.
template <int QT>
constexpr int COMBINE_WGS_PER_CU = PART16<QT> ? 4 : 2;

// The combine kernel is the last of every forward call: its workgroup 0 also
// writes the call's status word (SAS_OK, or SAS_ERR_PLAN when the plan's header
// differs from the call or some token was refused), to the workspace and, when
// given, to status_out.
template <int QT>
__global__ __launch_bounds__(64 * COMBINE_WAVES, COMBINE_WGS_PER_CU<QT>) void combine_kernel(
    SasFwdArgs a, const int* __restrict__ plan, const float* __restrict__ ws_o,
    const float* __restrict__ ws_ml, const int2* __restrict__ tok, uint16_t* __restrict__ out,
    float* __restrict__ lse, int* __restrict__ status, int* __restrict__ status_out) {
  const int H = a.H;
  const SasPlanLayout L = sas_plan_layout(a.T, a.split_cap);
  const int wave = blockIdx.x * COMBINE_WAVES + (threadIdx.x >> 6);
  const bool plan_ok = plan_matches(plan, a);
  if (blockIdx.x == 0) {
    // any token refused (window count -1)?  Two tokens per 16-B load.
    int bad = 0;
    if (plan_ok) {
      const int4* t4 = reinterpret_cast<const int4*>(tok);
      for (int i = threadIdx.x; i < a.T / 2; i += blockDim.x) {
        const int4 v = t4[i];
        bad |= (v.x < 0) | (v.z < 0);
      }
      if ((a.T & 1) && threadIdx.x == 0) bad |= tok[a.T - 1].x < 0;
    }
    bad = __syncthreads_or(bad);
    if (threadIdx.x == 0) {
      const int st = plan_ok && !bad ? SAS_OK : SAS_ERR_PLAN;
      *status = st;
      if (status_out) *status_out = st;
    }
  }
  if (!plan_ok) return;  // refused plan: the attention kernel wrote zeros (see plan_unit)
  // The split token's record (token, split count, first slot) is loaded before it is
  // known whether there are that many split tokens: its index is clamped into the
  // list, and a record past the count is never used.
  auto split_record = [&](int i) {
    const int ic = min(i, (int)L.split_cap - 1);
    return make_int3(plan[L.off_split_tokens + ic], plan[L.off_split_meta + 2 * ic],
                     plan[L.off_split_meta + 2 * ic + 1]);
  };
  // Per (split token, head): with at most COMBINE_BATCH splits, its records and rows
  // are loaded with the token's refusal flag, and the next item's split record
  // while this one merges: one memory round trip per item.
  const int stride = gridDim.x * COMBINE_WAVES;
  int3 rec = split_record(wave / H);
  const int items = plan[PH_NSPLIT_TOKENS] * H;  // (split token, head) pairs
  const int lane = threadIdx.x & 63;
  for (int item = wave; item < items; item += stride) {
    const int h = item % H;
    const int t = rec.x, S = rec.y, base = rec.z;
    const bool refused = tok[t].x < 0;
    float4 r0;
    MergeRows<QT, COMBINE_BATCH> v0;
    if (S <= COMBINE_BATCH) {
      r0 = merge_record<QT>(ws_ml, H, h, S, base, 0);
      merge_load<QT, COMBINE_BATCH>(v0, ws_o, H, h, base, 0, 0, S);
    }
    if (item + stride < items) rec = split_record((item + stride) / H);
    if (refused) {  // a refused token: zeros, as its units wrote
      reinterpret_cast<u32x4_t*>(out + ((size_t)t * H + h) * 512)[lane] = u32x4_t{0, 0, 0, 0};
      if (lse && lane == 0) lse[(size_t)t * H + h] = 0.f;
    } else if (S <= COMBINE_BATCH) {
      merge_finish<QT, COMBINE_BATCH>(t, h, H, S, base, ws_o, ws_ml, r0, v0, out, lse);
    } else {
      combine_head<QT>(t, h, H, S, base, ws_o, ws_ml, out, lse);
    }
  }
}

}  // namespace sas
