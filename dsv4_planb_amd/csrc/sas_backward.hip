// sas_backward.hip -- gfx950 kernels of the backward pass: queries, sinks and the
// KV pools.
//
// The reference has no backward; it returns the LSE for one (api.py:32-35,
// 176-184).  With the forward's out and lse, P_j = e^(s_j - lse) is known exactly
// (no running maximum and no frame), and
//   D = <dO, out> - dlse,  dS_j = P_j (<dO, V_j> - D),  dq = scale sum_j dS_j K_j,
//   dsink = -sum_t e^(sink - lse) D
// over the same row lists the forward attends (the resolver's output).
//
//   bwd_prep_kernel   D and the sink term per (token, head); zeroes the dq rows
//                     that are accumulated by several units (split tokens) or
//                     that no batch owns.
//   bwd_dq_kernel     one workgroup per (work unit, 64 heads): each wave owns 16
//                     heads.  Per 32-row tile: S^T = K Q^T and dP^T = V dO^T as
//                     16x16x32 MFMAs (K rows from LDS, Q^T and dO^T fragments in
//                     registers), P and dS in registers, then dq^T += K^T dS^T
//                     (K^T read transposed from the same row-major tile, dS^T
//                     straight from the accumulator layout).  Two tile buffers: the
//                     next tile's rows are loaded into registers during this one's
//                     MFMAs and stored after them.
//   bwd_dkv_kernel    the KV pools' gradient (dK from dS and q, dV from P and
//                     dO): one workgroup per work unit, the tile's gradient summed
//                     over all heads in registers, then fp32 atomics into
//                     pool-shaped buffers (one per element and tile).
//   bwd_dsink_kernel  dsink[h] summed over tokens in a fixed order (one wave per
//                     head), so it is deterministic.
//
// MFMA 16x16x32 operand layouts (lane l, n = l & 15, g = l >> 4): A (16 x 32)
// lane holds row n, columns 8 g .. 8 g + 7; B (32 x 16) lane holds rows 8 g .. 8 g
// + 7 of column n; C (16 x 16) lane holds rows 4 g .. 4 g + 3 of column n.  For
// dq^T the contraction runs over the tile's 32 keys in the order k = 8 g + e ->
// key (e < 4 ? 4 g + e : 16 + 4 g + e - 4): exactly the keys the two S^T blocks
// leave in lane l, so dS^T needs no data movement.
#include <hip/hip_runtime.h>

#include "sas_common.h"

namespace sas {

typedef __bf16 bw_bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 bw_f16x8 __attribute__((ext_vector_type(8)));
typedef float bw_f32x4 __attribute__((ext_vector_type(4)));

constexpr int BW_HEADS = 64;  // heads per workgroup: 4 waves x 16
constexpr int BW_AHEAD = 3;    // LDS fragment reads ahead of the MFMA using them
constexpr int BW_AHEAD_T = 4;  // the same, for the transposed reads of dq's K^T
constexpr int BW_AHEAD_A = 2;  // the same, in the dK/dV kernel's two phases
#define BW_SB() __builtin_amdgcn_sched_barrier(0)

// Loads and atomics through row addresses the kernels compute are issued as global
// (not FLAT) instructions: a FLAT access counts on the LDS counter too, so while one
// is in flight every wait for an LDS read would wait for it as well.
typedef __attribute__((address_space(1))) const u32x4_t g_u32x4;
typedef __attribute__((address_space(1))) float g_float;
__device__ __forceinline__ u32x4_t gload16(uint64_t addr) { return *(g_u32x4*)(uintptr_t)addr; }
__device__ __forceinline__ void gatomic_add(float* p, float v) {
  __hip_atomic_fetch_add((g_float*)p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
constexpr int BW_TILE = 32;   // keys per tile

template <int QT>
__device__ __forceinline__ bw_f32x4 bw_mfma(const u32x4_t& a, const u32x4_t& b, const bw_f32x4& c) {
  if constexpr (QT == 0)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bw_bf16x8, a),
                                                   __builtin_bit_cast(bw_bf16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(bw_f16x8, a),
                                                  __builtin_bit_cast(bw_f16x8, b), c, 0, 0, 0);
}

// D = <dO, out> (less dlse when the LSE has a gradient) and the sink term
// -e^(sink - lse) D, one wave per (token, head): workgroup x takes token x / HB and
// heads 4 (x % HB) .. + 3, HB = ceil(H / 4) (lane l covers dimensions 8 l .. 8 l + 7
// of d_v = 512).  One wave per head keeps every head's loads in flight at once; a
// wave walking a token's heads in turn waits for each head's rows before the next.
template <int QT>
__global__ __launch_bounds__(256) void bwd_prep_kernel(SasFwdArgs a, int dqk,
                                                       const int* __restrict__ plan,
                                                       const int2* __restrict__ tok,
                                                       const uint16_t* __restrict__ dout,
                                                       const uint16_t* __restrict__ out,
                                                       const float* __restrict__ lse,
                                                       const float* __restrict__ dlse,
                                                       const float* __restrict__ sinks,
                                                       float* __restrict__ dterm,
                                                       float* __restrict__ sterm,
                                                       float* __restrict__ dq,
                                                       int* __restrict__ flags) {
  constexpr int DV = 512;
  const int HB = (a.H + 3) / 4;
  const int t = blockIdx.x / HB, h = (blockIdx.x - t * HB) * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (flags && threadIdx.x == 0 && blockIdx.x == t * HB) {
    flags[1 + t] = 0;
    if (t == 0) flags[0] = 0;
  }
  if (h >= a.H) return;
  const bool ok = plan_matches(plan, a);
  const int* tk = plan + SAS_PLAN_HDR + (size_t)t * SAS_TOK_W;
  const int b = ok ? tk[TK_B] : -1;
  // (a token the resolver refused for a stale plan counts as unowned)
  const bool owned = b >= 0 && b < a.B && tok[t].x >= 0;
  const bool zero_dq = !owned || tk[TK_SPLITS] > 1;
  {
    const size_t th = (size_t)t * a.H + h;
    float d = 0.f;
    if (owned) {
      const u32x4_t go = reinterpret_cast<const u32x4_t*>(dout + th * DV)[lane];
      const u32x4_t oo = reinterpret_cast<const u32x4_t*>(out + th * DV)[lane];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        d = fmaf(q16_to_f32<QT>(go[e] & 0xffffu), q16_to_f32<QT>(oo[e] & 0xffffu), d);
        d = fmaf(q16_to_f32<QT>(go[e] >> 16), q16_to_f32<QT>(oo[e] >> 16), d);
      }
      d = wave_sum(d);
      // a gradient of the LSE: d lse / d s_j = P_j and d lse / d sink = P_sink, so it
      // enters as dS = P (dP - (D - dlse)) and dsink = -P_sink (D - dlse)
      if (dlse) d -= dlse[th];
    }
    if (lane == 0) {
      dterm[th] = d;
      const float s = sinks[h];
      // a sink of -inf has P_sink = 0 (lse may be -inf too when nothing is attended)
      sterm[th] = (!owned || s == -INFINITY || d == 0.f) ? 0.f : -__expf(s - lse[th]) * d;
    }
    if (zero_dq) {
      float4* row = reinterpret_cast<float4*>(dq + th * dqk);
      for (int i = lane; i < dqk / 4; i += 64) row[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
  }
}

// The spill (see SasBwdLayout): record 0 is all zeros, then record 1 + (t - t0) stride
// + p for list position p of token t; a record is, per 32-head chunk, 64 B of
// scale dS and 64 B of P in the query dtype.  flags[0] counts and flags[1 + t] marks
// the tokens with an infinity or a NaN in q or dO: the tile kernel, whose masked rows
// multiply a token's q and dO by zeros, leaves those to the per-unit kernel.
struct SasBwdSpill {
  int t0, t1;      // tokens of this run
  int stride;      // list positions per token
  int row_bytes;
  uint8_t* data;
  int* flags;
};

template <int DQK, int QT, bool SPILL>
__global__ __launch_bounds__(256, 1) void bwd_dq_kernel(SasFwdArgs a, const uint16_t* __restrict__ q,
                                                        const uint16_t* __restrict__ dout,
                                                        const uint64_t* __restrict__ addr_list,
                                                        const int2* __restrict__ tok,
                                                        const float* __restrict__ lse,
                                                        const float* __restrict__ dterm,
                                                        const int* __restrict__ plan,
                                                        float* __restrict__ dq, SasBwdSpill sp) {
  constexpr int DV = 512;
  constexpr int KS = DQK / 32;         // k-steps of S^T = K Q^T (18 / 16)
  constexpr int VKS = DV / 32;         // k-steps of dP^T = V dO^T (16)
  constexpr int NDB = DQK / 16;        // 16-dimension blocks of dq^T (36 / 32)
  constexpr int CH = DQK / 8;          // 16-B chunks per row
  constexpr int KSTR = DQK * 2 + 16;   // row-major tile: row stride in bytes
  constexpr int NLD = (BW_TILE * CH + 255) / 256;  // chunks per thread and tile (9 / 8)
  // two tiles: the one computed on and the next one, stored from registers after
  // the MFMAs of this one
  __shared__ __attribute__((aligned(16))) uint8_t kt[2][BW_TILE * KSTR];
  // SPILL: a wave's P and dS of a tile, [16 heads][32 keys] each, for the transpose
  __shared__ __attribute__((aligned(16))) uint8_t tp[SPILL ? 4 * 2048 : 16];

  const int HG = (a.H + BW_HEADS - 1) / BW_HEADS;
  const int u = blockIdx.x / HG, hg = blockIdx.x - u * HG;
  if (!plan_matches(plan, a) || u >= plan[PH_UNITS]) return;  // refused plan: prep zeroed dq
  const int* ur = plan + SAS_PLAN_HDR + (size_t)SAS_TOK_W * a.T + (size_t)u * SAS_UNIT_W;
  const int t = ur[0], split = ur[3];
  if (SPILL && (t < sp.t0 || t >= sp.t1)) return;  // a token of another run
  if (split < 0) return;  // a q row no batch owns: zero (bwd_prep_kernel)
  const int* tk = plan + SAS_PLAN_HDR + (size_t)t * SAS_TOK_W;
  const int splits = tk[TK_SPLITS];
  const int2 tr = tok[t];  // row counts at the call's lengths (the resolver's)
  if (tr.x < 0) return;    // refused token: zero (bwd_prep_kernel)
  const int r0 = ur[1];
  const int r1 = min(split == splits - 1 ? tr.x + tr.y : min(ur[2], tr.x + tr.y), a.list_stride);
  const int ntiles = r1 > r0 ? (r1 - r0 + BW_TILE - 1) / BW_TILE : 0;
  const uint64_t* alist = addr_list + (size_t)t * a.list_stride;

  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int n16 = lane & 15, g = lane >> 4;
  const int h = hg * BW_HEADS + w * 16 + n16;
  const bool hvalid = h < a.H;
  const int hc = min(h, a.H - 1);
  const size_t th = (size_t)t * a.H + hc;

  // A tile's rows: chunk ch = tid + 256 c (row ch / CH, 16-B chunk ch % CH).  The
  // row addresses of tile i + 2 and the chunks of tile i + 1 are loaded while tile i
  // is computed; rows past the unit's end (address 0) are zeros.
  uint64_t ra[NLD];
  u32x4_t pre[NLD];
  auto addrs = [&](int i) {
    const int rb = r0 + i * BW_TILE;
#pragma unroll
    for (int c = 0; c < NLD; ++c) {
      const int ch = tid + 256 * c, row = ch / CH;
      ra[c] = ch < BW_TILE * CH && rb + row < r1 ? alist[rb + row] : 0;
    }
  };
  auto fetch = [&]() {
#pragma unroll
    for (int c = 0; c < NLD; ++c) {
      const int ch = tid + 256 * c, cc = ch - (ch / CH) * CH;
      pre[c] = ra[c] ? gload16(ra[c] + 16 * cc) : u32x4_t{0, 0, 0, 0};
    }
  };
  auto stash = [&](int buf) {
#pragma unroll
    for (int c = 0; c < NLD; ++c) {
      const int ch = tid + 256 * c, row = ch / CH, cc = ch - row * CH;
      if (ch < BW_TILE * CH) *reinterpret_cast<u32x4_t*>(kt[buf] + row * KSTR + cc * 16) = pre[c];
    }
  };
  if (ntiles > 0) {
    addrs(0);
    fetch();
    if (ntiles > 1) addrs(1);
  }

  u32x4_t qf[KS], of[VKS];
  {
    const u32x4_t* qr = reinterpret_cast<const u32x4_t*>(q + th * DQK);
    const u32x4_t* orow = reinterpret_cast<const u32x4_t*>(dout + th * DV);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qf[ks] = qr[4 * ks + g];
#pragma unroll
    for (int ks = 0; ks < VKS; ++ks) of[ks] = orow[4 * ks + g];
  }
  const float lse2 = lse[th] * LOG2E, dh = dterm[th];
  const float c = a.scale_log2;
  const float scale = c * 0.6931471805599453f;
  if constexpr (SPILL) {
    // an infinity or a NaN: all exponent bits set (both halves of each dword)
    constexpr uint32_t EXP = QT == 0 ? 0x7f80u : 0x7c00u;
    bool bad = false;
    auto check = [&](const u32x4_t& v) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        bad = bad || (v[e] & EXP) == EXP || ((v[e] >> 16) & EXP) == EXP;
    };
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) check(qf[ks]);
#pragma unroll
    for (int ks = 0; ks < VKS; ++ks) check(of[ks]);
    if (__any(bad) && lane == 0) {
      sp.flags[1 + t] = 1;
      atomicAdd(sp.flags, 1);
    }
  }
  // SPILL: the wave's P and dS go through LDS: lane (n16, g) writes its 8 keys of head
  // n16 (16 B: positions 8 g .. + 7 of the head's 64-B row, key 16 kb + 4 g + r at
  // position 8 g + 4 kb + r), and ds_read_b64_tr_b16 returns 4 heads (4 g .. + 3) of
  // one position per lane, stored as 8 B of its key's record.  The 32-B halves of a row
  // are swapped for heads 4 .. 7 and 12 .. 15, so that the transposed reads touch every
  // bank once per 256 B.
  uint8_t* const tpw = tp + (SPILL ? w * 2048 : 0);
  const bool sp_wave = SPILL && hg * BW_HEADS + w * 16 < sp.row_bytes / 4;  // a padded head chunk ends
  uint8_t* sp_row = nullptr;
  if constexpr (SPILL)
    sp_row = sp.data + (1 + (size_t)(t - sp.t0) * sp.stride) * sp.row_bytes +
             (2 * hg + (w >> 1)) * 128 + (16 * (w & 1) + 4 * g) * 2;
  bw_f32x4 acc[NDB];
#pragma unroll
  for (int i = 0; i < NDB; ++i) acc[i] = bw_f32x4{0.f, 0.f, 0.f, 0.f};
  if (ntiles > 0) stash(0);
  __syncthreads();

  typedef short tr_s4 __attribute__((ext_vector_type(4)));
  for (int i = 0; i < ntiles; ++i) {
    const int rb = r0 + i * BW_TILE;
    const uint8_t* tl = kt[i & 1];
    if (i + 1 < ntiles) fetch();
    if (i + 2 < ntiles) addrs(i + 2);
    // S^T and dP^T: two blocks of 16 keys each, one chain of 2 KS steps (block
    // kb = st / KS, k-step st % KS).  The K fragments are read BW_AHEAD steps ahead
    // (an LDS read takes several MFMAs' time to return, and this wave is the
    // SIMD's only one); the scheduling barriers keep that order.
    bw_f32x4 s[2], dp[2];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
      s[kb] = bw_f32x4{0.f, 0.f, 0.f, 0.f};
      dp[kb] = bw_f32x4{0.f, 0.f, 0.f, 0.f};
    }
    {
      auto kfrag = [&](int st) -> u32x4_t {
        const int kb = st / KS, ks = st - kb * KS;
        return *reinterpret_cast<const u32x4_t*>(tl + (16 * kb + n16) * KSTR + 16 * g + 64 * ks);
      };
      u32x4_t kf[BW_AHEAD + 1];
#pragma unroll
      for (int st = 0; st < BW_AHEAD; ++st) kf[st] = kfrag(st);
      BW_SB();
#pragma unroll
      for (int st = 0; st < 2 * KS; ++st) {
        if (st + BW_AHEAD < 2 * KS) kf[(st + BW_AHEAD) % (BW_AHEAD + 1)] = kfrag(st + BW_AHEAD);
        const int kb = st / KS, ks = st - kb * KS;
        const u32x4_t av = kf[st % (BW_AHEAD + 1)];
        s[kb] = bw_mfma<QT>(av, qf[ks], s[kb]);
        if (ks < VKS) dp[kb] = bw_mfma<QT>(av, of[ks], dp[kb]);
        BW_SB();
      }
    }
    // P = e^(s - lse) and dS = P (dP - D) for keys 16 kb + 4 g + r of head n16
    float ds[8], pr[8];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const bool valid = rb + 16 * kb + 4 * g + r < r1;
        const float p = valid ? exp2f(fmaf(s[kb][r], c, -lse2)) : 0.f;
        pr[4 * kb + r] = p;
        ds[4 * kb + r] = p * (dp[kb][r] - dh);
      }
    u32x4_t bds;
#pragma unroll
    for (int e = 0; e < 4; ++e) bds[e] = pack2_q16<QT>(ds[2 * e], ds[2 * e + 1]);
    if constexpr (SPILL) {
      if (sp_wave) {
        u32x4_t xs, xp;
#pragma unroll
        for (int e = 0; e < 4; ++e) {  // (heads at or past H: zeros)
          xs[e] = hvalid ? pack2_q16<QT>(ds[2 * e] * scale, ds[2 * e + 1] * scale) : 0u;
          xp[e] = hvalid ? pack2_q16<QT>(pr[2 * e], pr[2 * e + 1]) : 0u;
        }
        const int wo = 64 * n16 + 16 * (g ^ (2 * ((n16 >> 2) & 1)));
        *reinterpret_cast<u32x4_t*>(tpw + wo) = xs;
        *reinterpret_cast<u32x4_t*>(tpw + 1024 + wo) = xp;
        const uint8_t* ro = tpw + 64 * (4 * g + (n16 >> 2)) + 8 * (n16 & 3);
        tr_s4 v[2][2];
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
          for (int z = 0; z < 2; ++z)
            v[x][z] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (__attribute__((address_space(3))) tr_s4*)(ro + 1024 * z + 32 * (x ^ (g & 1))));
#pragma unroll
        for (int x = 0; x < 2; ++x) {
          const int p = rb + 16 * ((n16 >> 2) & 1) + 4 * (2 * x + (n16 >> 3)) + (n16 & 3);
          if (p < r1 && p < sp.stride) {
            typedef __attribute__((address_space(1))) tr_s4 g_s4;
            uint8_t* dst = sp_row + (size_t)p * sp.row_bytes;
            *(g_s4*)(uintptr_t)dst = v[x][0];
            *(g_s4*)(uintptr_t)(dst + 64) = v[x][1];
          }
        }
      }
    }
    // dq^T += K^T dS^T.  A = dimensions 16 db + n16 of keys 4 g .. 4 g + 3 (then 16 +
    // 4 g ..), read transposed from the row-major tile: within each 16-lane block,
    // ds_read_b64_tr_b16 gives lane j element j & 3 of the 8 bytes lane (j >> 2) + 4 e
    // addresses, for e = 0 .. 3; so lane i of block g addresses key 4 g + (i >> 2)
    // (+ 16), dimensions 16 db + 4 (i & 3) .. + 3.
    const uint8_t* ta = tl + (4 * g + (n16 >> 2)) * KSTR + 8 * (n16 & 3);
    {
      // the K^T fragments, read BW_AHEAD_T blocks ahead
      auto kt_frag = [&](int db) -> u32x4_t {
        const tr_s4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) tr_s4*)(ta + 32 * db));
        const tr_s4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) tr_s4*)(ta + 16 * KSTR + 32 * db));
        return u32x4_t{(uint32_t)(uint16_t)lo[0] | ((uint32_t)(uint16_t)lo[1] << 16),
                       (uint32_t)(uint16_t)lo[2] | ((uint32_t)(uint16_t)lo[3] << 16),
                       (uint32_t)(uint16_t)hi[0] | ((uint32_t)(uint16_t)hi[1] << 16),
                       (uint32_t)(uint16_t)hi[2] | ((uint32_t)(uint16_t)hi[3] << 16)};
      };
      u32x4_t tf[BW_AHEAD_T + 1];
#pragma unroll
      for (int db = 0; db < BW_AHEAD_T; ++db) tf[db] = kt_frag(db);
      BW_SB();
#pragma unroll
      for (int db = 0; db < NDB; ++db) {
        if (db + BW_AHEAD_T < NDB) tf[(db + BW_AHEAD_T) % (BW_AHEAD_T + 1)] = kt_frag(db + BW_AHEAD_T);
        acc[db] = bw_mfma<QT>(tf[db % (BW_AHEAD_T + 1)], bds, acc[db]);
        BW_SB();
      }
    }
    if (i + 1 < ntiles) stash((i + 1) & 1);
    __syncthreads();  // tile i + 1 stored; every wave is done with tile i
  }
  if (!hvalid) return;
  // lane holds dimensions 16 db + 4 g .. + 3 of head h
  float* dqr = dq + ((size_t)t * a.H + h) * DQK + 4 * g;
#pragma unroll
  for (int db = 0; db < NDB; ++db) {
    const float4 v = make_float4(acc[db][0] * scale, acc[db][1] * scale, acc[db][2] * scale,
                                 acc[db][3] * scale);
    if (splits > 1) {
      atomicAdd(dqr + 16 * db + 0, v.x);
      atomicAdd(dqr + 16 * db + 1, v.y);
      atomicAdd(dqr + 16 * db + 2, v.z);
      atomicAdd(dqr + 16 * db + 3, v.w);
    } else {
      *reinterpret_cast<float4*>(dqr + 16 * db) = v;
    }
  }
}

// ---------------------------------------------------------------------------
// The KV pools' gradient.  Row j of token t's list (pool row R_j) receives
//   dK_j = scale sum_h dS_hj q_h  (all d_qk dimensions)  +  dV_j = sum_h P_hj dO_h
// (the first d_v dimensions), summed over every token and list position that reads
// R_j (window overlap, repeated top-k ids): fp32 atomics into a gradient buffer
// laid out like the pool (same block and row strides, in elements).  Rows read as
// zeros (-1 codes) and rows past a unit's end receive nothing.
//
// One workgroup per work unit, all heads.  Per 32-row tile the gradient of the
// tile's rows, G = scale dS^T Q + P^T dO (32 keys x d_qk), accumulates in registers
// over the heads, 32 at a time, and goes to the pools with one atomic add per
// element and tile (at H = 128 a quarter of one add per 32-head group).  Per group of 32
// heads, their q and dO rows are staged row-major in LDS (16-B copies), then
//   phase A  wave w computes S^T and dP^T for keys 16 (w & 1) .. + 15 and heads
//            16 (w >> 1) .. + 15 of the group (16x16x32 MFMAs, K rows from the LDS
//            tile, Q^T / dO^T fragments from the staged rows), then P = e^(S - lse)
//            and dS = P (dP - D), written to LDS as scale dS^T and P^T ([key][head],
//            rounded to the query dtype)
//   phase B  G += (scale dS^T) Q + P^T dO (32 heads contracted in one MFMA per 16 x 16
//            block; the Q and dO operands read transposed from the staged rows with
//            ds_read_b64_tr_b16): wave w takes key block w & 1 and half of the
//            dimension blocks.
// After the last group each lane adds 4 keys of one dimension to the pool rows (16
// lanes: 16 consecutive dimensions).
// ---------------------------------------------------------------------------
constexpr int DK_HEADS = 32;  // heads per group

//
// tiles (the rows bwd_dkv_tile_kernel takes): 0 none, 1 the window rows, 2 all; then
// flags marks the tokens whose rows all stay here.
template <int DQK, int QT>
struct DkvLds {
  static constexpr int KSTR = DQK * 2 + 16;      // row-major K tile and staged q: row stride in bytes
  static constexpr int OSTR = 512 * 2 + 16;      // staged dO: row stride in bytes
  static constexpr int TS = 2 * DK_HEADS + 16;   // [key][head] rows of dS^T and P^T: bytes per key
  __attribute__((aligned(16))) uint8_t kt[BW_TILE * KSTR];
  __attribute__((aligned(16))) uint8_t qs[DK_HEADS * KSTR];
  __attribute__((aligned(16))) uint8_t os[DK_HEADS * OSTR];
  __attribute__((aligned(16))) uint8_t dst[BW_TILE * TS];
  __attribute__((aligned(16))) uint8_t ptr[BW_TILE * TS];
};

template <int DQK, int QT>
__device__ __forceinline__ void dkv_unit(
    int u, DkvLds<DQK, QT>& sm, const SasFwdArgs& a, const uint16_t* __restrict__ q,
    const uint16_t* __restrict__ dout, const uint64_t* __restrict__ addr_list,
    const int* __restrict__ row_codes, const int2* __restrict__ tok, const float* __restrict__ lse,
    const float* __restrict__ dterm, const int* __restrict__ plan, float* __restrict__ d_ori,
    float* __restrict__ d_cmp, int tiles, const int* __restrict__ flags) {
  constexpr int DV = 512;
  constexpr int KS = DQK / 32;         // k-steps of S^T = K Q^T (18 / 16)
  constexpr int VKS = DV / 32;         // k-steps of dP^T = V dO^T (16)
  constexpr int NDB = DQK / 16;        // 16-dimension blocks of G (36 / 32)
  constexpr int CH = DQK / 8;          // 16-B chunks per row of K or q
  constexpr int CHO = DV / 8;          // 16-B chunks per row of dO
  constexpr int KSTR = DkvLds<DQK, QT>::KSTR, OSTR = DkvLds<DQK, QT>::OSTR, TS = DkvLds<DQK, QT>::TS;
  uint8_t* const kt = sm.kt;
  uint8_t* const qs = sm.qs;
  uint8_t* const os = sm.os;
  uint8_t* const dst = sm.dst;
  uint8_t* const ptr = sm.ptr;

  const int* ur = plan + SAS_PLAN_HDR + (size_t)SAS_TOK_W * a.T + (size_t)u * SAS_UNIT_W;
  const int t = ur[0], split = ur[3];
  if (split < 0) return;  // a q row no batch owns: it reads no rows
  const int* tk = plan + SAS_PLAN_HDR + (size_t)t * SAS_TOK_W;
  const int2 tr = tok[t];  // row counts at the call's lengths (the resolver's)
  if (tr.x < 0) return;    // refused token: it reads no rows
  const int nwin = tr.x;   // list positions below it are window rows (raw pool)
  int r0 = ur[1];
  if (tiles && !flags[1 + t]) {  // the window rows, or all, are bwd_dkv_tile_kernel's
    if (tiles == 2) return;
    r0 = max(r0, nwin);
  }
  const int r1 = min(ur[3] == tk[TK_SPLITS] - 1 ? tr.x + tr.y : min(ur[2], tr.x + tr.y),
                     a.list_stride);
  const int ntiles = r1 > r0 ? (r1 - r0 + BW_TILE - 1) / BW_TILE : 0;
  if (ntiles == 0) return;
  const uint64_t* alist = addr_list + (size_t)t * a.list_stride;
  const int* codes = row_codes + (size_t)t * a.list_stride;

  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int n16 = lane & 15, g = lane >> 4;
  const int NG = (a.H + DK_HEADS - 1) / DK_HEADS;
  const float c = a.scale_log2;
  const float scale = c * 0.6931471805599453f;
  // phase A role: keys 16 kb .. + 15, heads 16 hb + n16 of the group
  const int kb = w & 1, hb = w >> 1;
  // phase B role: key block kb (as in phase A), dimension blocks [db0, db0 + NDB / 2)
  const int db0 = hb * (NDB / 2);
  typedef short tr_s4 __attribute__((ext_vector_type(4)));
  auto tr_pair = [](const uint8_t* p0, const uint8_t* p1) -> u32x4_t {
    const tr_s4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) tr_s4*)p0);
    const tr_s4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) tr_s4*)p1);
    return u32x4_t{(uint32_t)(uint16_t)lo[0] | ((uint32_t)(uint16_t)lo[1] << 16),
                   (uint32_t)(uint16_t)lo[2] | ((uint32_t)(uint16_t)lo[3] << 16),
                   (uint32_t)(uint16_t)hi[0] | ((uint32_t)(uint16_t)hi[1] << 16),
                   (uint32_t)(uint16_t)hi[2] | ((uint32_t)(uint16_t)hi[3] << 16)};
  };

  // Software pipeline over the steps (tile i, group grp): the next step's q / dO rows
  // (and, before a new tile, its K rows) are loaded into registers during this step's
  // MFMAs, and stored to LDS once every wave is done with the current ones.  Those
  // loads are issued ahead of the tile's atomics, so no wait for them waits for the
  // atomics too (vector memory operations complete in order).
  constexpr int NST = (DK_HEADS * (CH + CHO) + 255) / 256;  // staging chunks per thread (17 / 16)
  constexpr int NLD = (BW_TILE * CH + 255) / 256;          // K-tile chunks per thread (9 / 8)
  u32x4_t stg[NST], pre[NLD];
  uint64_t ra[NLD];
  auto stage_load = [&](int grp) {
    const int h0 = grp * DK_HEADS;
#pragma unroll
    for (int c = 0; c < NST; ++c) {
      const int ch = tid + 256 * c;
      const bool isq = ch < DK_HEADS * CH;
      const int k = isq ? ch : ch - DK_HEADS * CH;
      const int hh = isq ? k / CH : k / CHO, cc = isq ? k - hh * CH : k - hh * CHO;
      stg[c] = u32x4_t{0, 0, 0, 0};
      if (ch < DK_HEADS * (CH + CHO) && h0 + hh < a.H) {
        const size_t th = (size_t)t * a.H + h0 + hh;
        stg[c] = isq ? reinterpret_cast<const u32x4_t*>(q + th * DQK)[cc]
                     : reinterpret_cast<const u32x4_t*>(dout + th * DV)[cc];
      }
    }
  };
  auto stage_store = [&]() {
#pragma unroll
    for (int c = 0; c < NST; ++c) {
      const int ch = tid + 256 * c;
      if (ch >= DK_HEADS * (CH + CHO)) break;
      const bool isq = ch < DK_HEADS * CH;
      const int k = isq ? ch : ch - DK_HEADS * CH;
      const int hh = isq ? k / CH : k / CHO, cc = isq ? k - hh * CH : k - hh * CHO;
      *reinterpret_cast<u32x4_t*>((isq ? qs + hh * KSTR : os + hh * OSTR) + cc * 16) = stg[c];
    }
  };
  auto tile_addrs = [&](int i) {
    const int rb = r0 + i * BW_TILE;
#pragma unroll
    for (int c = 0; c < NLD; ++c) {
      const int ch = tid + 256 * c, row = ch / CH;
      ra[c] = ch < BW_TILE * CH && rb + row < r1 ? alist[rb + row] : 0;
    }
  };
  auto tile_load = [&]() {
#pragma unroll
    for (int c = 0; c < NLD; ++c) {
      const int ch = tid + 256 * c, cc = ch - (ch / CH) * CH;
      pre[c] = ra[c] ? gload16(ra[c] + 16 * cc) : u32x4_t{0, 0, 0, 0};
    }
  };
  auto tile_store = [&]() {
#pragma unroll
    for (int c = 0; c < NLD; ++c) {
      const int ch = tid + 256 * c, row = ch / CH, cc = ch - row * CH;
      if (ch < BW_TILE * CH) *reinterpret_cast<u32x4_t*>(kt + row * KSTR + cc * 16) = pre[c];
    }
  };
  // The LSE and D of this lane's head in each group (H <= 128: at most 4 groups),
  // loaded once.  Vector memory operations complete in order, so a value loaded in
  // the group loop would wait for every load issued before it, the next step's rows
  // included.
  float lse2g[4], dhg[4];
#pragma unroll
  for (int gi = 0; gi < 4; ++gi) {
    const int h = min(gi * DK_HEADS + 16 * hb + n16, a.H - 1);
    lse2g[gi] = lse[(size_t)t * a.H + h] * LOG2E;
    dhg[gi] = dterm[(size_t)t * a.H + h];
  }
  tile_addrs(0);
  tile_load();
  stage_load(0);

  for (int i = 0; i < ntiles; ++i) {
    const int rb = r0 + i * BW_TILE;
    if (i + 1 < ntiles) tile_addrs(i + 1);
    // the codes of the tile's rows this lane adds to (keys 16 kb + 4 g + r), used
    // after the group loop
    int code[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int j = rb + 16 * kb + 4 * g + r;  // list position
      code[r] = j < r1 ? codes[j] : -1;
    }
    bw_f32x4 gacc[NDB / 2];
#pragma unroll
    for (int k = 0; k < NDB / 2; ++k) gacc[k] = bw_f32x4{0.f, 0.f, 0.f, 0.f};

    for (int grp = 0; grp < NG; ++grp) {
      __syncthreads();  // every wave is done with the previous step's tile and rows
      if (grp == 0) tile_store();
      stage_store();
      // the next step's loads: the next group's rows, or the next tile's K rows and
      // its first group's rows
      const bool last = grp + 1 == NG;
      if (!last || i + 1 < ntiles) {
        if (last) tile_load();
        stage_load(last ? 0 : grp + 1);
      }
      const int hl = 16 * hb + n16, h = grp * DK_HEADS + hl;
      const bool hvalid = h < a.H;
      const float lse2 = grp == 0 ? lse2g[0] : grp == 1 ? lse2g[1] : grp == 2 ? lse2g[2] : lse2g[3];
      const float dh = grp == 0 ? dhg[0] : grp == 1 ? dhg[1] : grp == 2 ? dhg[2] : dhg[3];
      __syncthreads();
      // phase A: S^T and dP^T of 16 keys x 16 heads; lane holds keys 16 kb + 4 g + r
      {
        const uint8_t* kr = kt + (16 * kb + n16) * KSTR + 16 * g;
        const uint8_t* qr = qs + hl * KSTR + 16 * g;
        const uint8_t* orow = os + hl * OSTR + 16 * g;
        bw_f32x4 s = bw_f32x4{0.f, 0.f, 0.f, 0.f}, dp = s;
        // the step's three fragments, read BW_AHEAD_A steps ahead
        constexpr int NA = BW_AHEAD_A + 1;
        u32x4_t fk[NA], fq[NA], fo[NA];
        auto frag_a = [&](int ks) {
          fk[ks % NA] = *reinterpret_cast<const u32x4_t*>(kr + 64 * ks);
          fq[ks % NA] = *reinterpret_cast<const u32x4_t*>(qr + 64 * ks);
          if (ks < VKS) fo[ks % NA] = *reinterpret_cast<const u32x4_t*>(orow + 64 * ks);
        };
#pragma unroll
        for (int ks = 0; ks < BW_AHEAD_A; ++ks) frag_a(ks);
        BW_SB();
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          if (ks + BW_AHEAD_A < KS) frag_a(ks + BW_AHEAD_A);
          s = bw_mfma<QT>(fk[ks % NA], fq[ks % NA], s);
          if (ks < VKS) dp = bw_mfma<QT>(fk[ks % NA], fo[ks % NA], dp);
          BW_SB();
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int key = 16 * kb + 4 * g + r;
          const bool valid = hvalid && rb + key < r1;
          const float p = valid ? exp2f(fmaf(s[r], c, -lse2)) : 0.f;
          const float ds = p * (dp[r] - dh);
          const uint32_t pk = pack2_q16<QT>(ds * scale, p);
          *reinterpret_cast<uint16_t*>(dst + key * TS + 2 * hl) = (uint16_t)(pk & 0xffffu);
          *reinterpret_cast<uint16_t*>(ptr + key * TS + 2 * hl) = (uint16_t)(pk >> 16);
        }
      }
      __syncthreads();
      // phase B: G += (scale dS^T) Q + P^T dO for keys 16 kb .. + 15 and this wave's
      // dimension blocks; lane holds keys 16 kb + 4 g + r of dimension 16 db + n16.
      // B operands (heads 8 g .. + 7 of one dimension) read transposed from the
      // staged rows: lane i of block g addresses head 8 g + (i >> 2) (+ 4),
      // dimensions 16 db + 4 (i & 3) .. + 3.
      {
        const u32x4_t ads = *reinterpret_cast<const u32x4_t*>(dst + (16 * kb + n16) * TS + 16 * g);
        const u32x4_t ap = *reinterpret_cast<const u32x4_t*>(ptr + (16 * kb + n16) * TS + 16 * g);
        const int hq = 8 * g + (n16 >> 2);
        const uint8_t* qb = qs + hq * KSTR + 8 * (n16 & 3);
        const uint8_t* ob = os + hq * OSTR + 8 * (n16 & 3);
        // the step's two transposed operands, read BW_AHEAD_A steps ahead (dO's block
        // clamped below d_v, unused past it)
        constexpr int NA = BW_AHEAD_A + 1;
        u32x4_t tq[NA], to[NA];
        auto frag_b = [&](int k) {
          const int db = db0 + k, dbo = min(db, DV / 16 - 1);
          tq[k % NA] = tr_pair(qb + 32 * db, qb + 4 * KSTR + 32 * db);
          to[k % NA] = tr_pair(ob + 32 * dbo, ob + 4 * OSTR + 32 * dbo);
        };
#pragma unroll
        for (int k = 0; k < BW_AHEAD_A; ++k) frag_b(k);
        BW_SB();
#pragma unroll
        for (int k = 0; k < NDB / 2; ++k) {
          if (k + BW_AHEAD_A < NDB / 2) frag_b(k + BW_AHEAD_A);
          const int db = db0 + k;
          gacc[k] = bw_mfma<QT>(ads, tq[k % NA], gacc[k]);
          if (16 * db < DV) gacc[k] = bw_mfma<QT>(ap, to[k % NA], gacc[k]);
          BW_SB();
        }
      }
    }
    // the tile's gradient to the pool rows: one atomic add per element
    float* rowp[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int j = rb + 16 * kb + 4 * g + r;
      float* pool = j < nwin ? d_ori : d_cmp;
      const int bs = j < nwin ? a.ori_block_size : a.cmp_block_size;
      const int64_t bstr = j < nwin ? a.ori_block_stride : a.cmp_block_stride;
      const int64_t rstr = j < nwin ? a.ori_row_stride : a.cmp_row_stride;
      rowp[r] = nullptr;
      if (code[r] >= 0 && pool) {
        const int page = (int)((unsigned)code[r] / (unsigned)bs), off = code[r] - page * bs;
        rowp[r] = pool + (size_t)page * bstr + (size_t)off * rstr;
      }
    }
#pragma unroll
    for (int k = 0; k < NDB / 2; ++k) {
      const int dim = 16 * (db0 + k) + n16;
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (rowp[r]) gatomic_add(rowp[r] + dim, gacc[k][r]);
    }
  }
}

// Workgroup x takes units x, x + gridDim, ...  Where the tiles take every row
// (tiles == 2), one look at the count of marked tokens ends it.
template <int DQK, int QT>
__global__ __launch_bounds__(256, 1) void bwd_dkv_kernel(
    SasFwdArgs a, const uint16_t* __restrict__ q, const uint16_t* __restrict__ dout,
    const uint64_t* __restrict__ addr_list, const int* __restrict__ row_codes,
    const int2* __restrict__ tok, const float* __restrict__ lse, const float* __restrict__ dterm,
    const int* __restrict__ plan, float* __restrict__ d_ori, float* __restrict__ d_cmp, int tiles,
    const int* __restrict__ flags) {
  __shared__ DkvLds<DQK, QT> sm;
  if (tiles == 2 && flags[0] == 0) return;
  if (!plan_matches(plan, a)) return;
  const int units = plan[PH_UNITS];
  for (int u = blockIdx.x; u < units; u += gridDim.x) {
    dkv_unit<DQK, QT>(u, sm, a, q, dout, addr_list, row_codes, tok, lse, dterm, plan, d_ori, d_cmp,
                      tiles, flags);
    __syncthreads();  // every wave is done with the unit's LDS
  }
}

// dsink[h] = sum over tokens of the sink terms: one workgroup per head, thread i
// taking tokens i, i + 256, ... into eight partial sums (eight loads in flight),
// combined in a fixed order within the thread, the wave and the workgroup:
// deterministic.
__global__ __launch_bounds__(256) void bwd_dsink_kernel(int T, int H, const float* __restrict__ sterm,
                                                        float* __restrict__ dsinks) {
  __shared__ float wsum[4];
  const int h = blockIdx.x, tid = threadIdx.x;
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  for (int t0 = 0; t0 < T; t0 += 256 * 8) {
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int t = t0 + 256 * k + tid;
      if (t < T) acc[k] += sterm[(size_t)t * H + h];
    }
  }
  float v = ((acc[0] + acc[1]) + (acc[2] + acc[3])) + ((acc[4] + acc[5]) + (acc[6] + acc[7]));
  v = wave_sum(v);
  if ((tid & 63) == 0) wsum[tid >> 6] = v;
  __syncthreads();
  if (tid == 0) dsinks[h] = (wsum[0] + wsum[1]) + (wsum[2] + wsum[3]);
}

}  // namespace sas
