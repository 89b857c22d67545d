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
//   bwd_prep_kernel   zeroes the dq rows that are accumulated by several units (split
//                     tokens) or that no batch owns.
//   bwd_dq_kernel     one workgroup per (work unit, 64 heads): each wave owns 16
//                     heads.  D and the sink term per (token, head); then, per 32-row
//                     tile: S^T = K Q^T and dP^T = V dO^T as
//                     16x16x32 MFMAs (K rows from LDS, Q^T and dO^T fragments in
//                     registers), P and dS in registers, then dq^T += K^T dS^T
//                     (K^T read transposed from the same row-major tile, dS^T
//                     straight from the accumulator layout).  Three tile buffers,
//                     filled by LDS-direct DMA, one barrier per tile.
//   bwd_dkv_kernel    the KV pools' gradient (dK from dS and q, dV from P and
//                     dO): one workgroup per work unit, the tile's gradient summed
//                     over all heads in registers, then fp32 atomics into
//                     pool-shaped buffers (one per element and tile).
//   bwd_dsink_kernel  dsink[h] summed over tokens in a fixed order (one workgroup per
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

// acc + the two 16-bit values of v, each times zero: acc, or a NaN where one is not finite.
template <int QT>
__device__ __forceinline__ float dot2_zero(uint32_t v, uint32_t zero, float acc) {
  if constexpr (QT == 0) {
    typedef __bf16 b2 __attribute__((ext_vector_type(2)));
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(b2, v), __builtin_bit_cast(b2, zero), acc, false);
  } else {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    return __builtin_amdgcn_fdot2(__builtin_bit_cast(h2, v), __builtin_bit_cast(h2, zero), acc, false);
  }
}

// What the dq kernel leaves out, per (token from t0 on, BP_HEADS heads): the terms of tokens that no
// batch owns (or whose plan is refused), and the zeros of their dq rows and of those that
// several units add to; and the flags of a call whose P and dS are spilled (else null).
constexpr int BP_HEADS = 64;
__global__ __launch_bounds__(256) void bwd_prep_kernel(SasFwdArgs a, int dqk, int t0, const int* __restrict__ plan,
                                                       const int2* __restrict__ tok,
                                                       float* __restrict__ dterm, float* __restrict__ sterm,
                                                       float* __restrict__ dq, int* __restrict__ flags) {
  const int HB = (a.H + BP_HEADS - 1) / BP_HEADS;
  const int tb = blockIdx.x / HB, t = t0 + tb, h0 = (blockIdx.x - tb * HB) * BP_HEADS;
  const int tid = threadIdx.x, nh = min(BP_HEADS, a.H - h0);
  if (flags && tid == 0 && h0 == 0) {
    flags[1 + t] = 0;
    if (t == 0) flags[0] = 0;
  }
  const bool ok = plan_matches(plan, a);
  const int* tk = plan + SAS_PLAN_HDR + (size_t)t * SAS_TOK_W;
  const int b = ok ? tk[TK_B] : -1;
  // (a token the resolver refused for a stale plan counts as unowned)
  const bool owned = b >= 0 && b < a.B && tok[t].x >= 0;
  const size_t th = (size_t)t * a.H + h0;
  if (!owned && tid < nh) {
    dterm[th + tid] = 0.f;
    sterm[th + tid] = 0.f;
  }
  if (!owned || tk[TK_SPLITS] > 1) {
    float4* row = reinterpret_cast<float4*>(dq + th * dqk);
    for (int i = tid; i < nh * dqk / 4; i += 256) row[i] = make_float4(0.f, 0.f, 0.f, 0.f);
  }
}

// D = <dO, out> (less dlse when the LSE has a gradient) and the sink term -e^(sink - lse) D,
// which the dq kernel computes where it holds the dO rows and writes for the kernels after
// it: a kernel of its own reads dO once more and was bound by that (4 documents of 608 ..
// 1,697 tokens, 128 heads: 221 us; now 8 us for bwd_prep_kernel and 100 us more in the dq
// kernel; documents of 1,082 and 971 tokens, 64 heads: 59 us, now 6 and 25).
struct SasBwdTerms {
  const uint16_t* out;
  const float* dlse;  // or null
  const float* sinks;
  float* dterm;  // [T][H]
  float* sterm;
};

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

// A tile's LDS layout: latent rows at a 1088-B stride, 16-B chunk c of row r at c ^ f(r), f
// = 2 (r bit 2) + (r bit 3); rope rows of 128 B, chunk c at c ^ fr(r), fr the three bits of
// (r >> 1) & 7 rotated left by one.  The b128 reads (16 rows, one chunk) and the
// transposed ones (rows 4 g .. 4 g + 3 and 4 g + 4 .. 4 g + 7 x 32 B per 32 lanes) then
// touch every bank once per 256 B.
template <int DQK, bool SPILL>
struct DqLds {
  static constexpr int STRA = 1024 + 64, ROWR = (DQK - 512) * 2;
  static constexpr int TILEA = BW_TILE * STRA, TILEB = TILEA + BW_TILE * ROWR;
  __attribute__((aligned(16))) uint8_t tiles[3 * TILEB];
  // SPILL: a wave's P and dS of a tile, [16 heads][32 keys] each, for the transpose
  __attribute__((aligned(16))) uint8_t tp[SPILL ? 4 * 2048 : 16];
};

// Ring of three tiles, one barrier per tile: tile i + 2's DMAs (wave w: rows 8 w .. + 7, 8
// latent and one rope instruction) are issued between the MFMAs of tile i's S / dP chain.
// They have that one tile's time to arrive, not two: the row addresses of tile i + 3 are
// loaded behind them, vector memory completes in order, and the next iteration begins by
// waiting for those addresses, so two of the three slots are in flight or in use.
//
// What bounds it: a workgroup reads its 64 heads' q, dO and out rows and writes their dq in
// fp32, 352 KB (328 KB at d_qk 512), before and after its tiles and, one workgroup
// per CU (125 KB of LDS, 380 registers), beside nothing else; at the rate of a large copy
// that is 17.7 us (16.5) when every CU does it.  Window-only calls of 8,192 tokens whose
// units have 1, 2, 4, 8, 16 and 32 tiles take 22.0, 22.8, 24.7, 31.0, 46.4 and 71.0 us per
// workgroup at 128 heads with the spill (21.4, 22.9, 25.7, 28.5, 38.8, 58.5 without it) and
// 18.5, 20.9, 24.2, 30.1, 42.7 and 61.4 us at 64 heads, d_qk 512: a long unit's tile is
// 1.2 to 1.9 us (1.1 to 1.3), 0.7 of them MFMA (104 per wave, 1,664 cycles).
//
// Before, the next tile's rows went through registers and a second barrier, the first tile
// was fetched after the query's rows, and the check for infinities and NaNs took four
// instructions per value.  Measured, with the spill: 4 documents of 608 .. 1,697 tokens, 128
// heads, top-k 512, 1,390 -> 1,070 us; documents of 1,082 and 971 tokens, 64 heads, window
// only, d_qk 512, 232 -> 185 us (and since it computes D too 1,175 and 217 us).
template <int DQK, int QT, bool SPILL>
__device__ __forceinline__ void dq_unit(DqLds<DQK, SPILL>& sm, const int4 ur, int hg, const SasFwdArgs& a,
                                        const uint16_t* __restrict__ q, const uint16_t* __restrict__ dout,
                                        const uint64_t* __restrict__ addr_list,
                                        const int2* __restrict__ tok, const float* __restrict__ lse,
                                        const SasBwdTerms& bt, const int* __restrict__ plan,
                                        float* __restrict__ dq, const SasBwdSpill& sp) {
  constexpr int DV = 512;
  constexpr bool ROPE = DQK > DV;
  constexpr int KS = DQK / 32;         // k-steps of S^T = K Q^T (18 / 16)
  constexpr int VKS = DV / 32;         // k-steps of dP^T = V dO^T (16)
  constexpr int NDB = DQK / 16;        // 16-dimension blocks of dq^T (36 / 32)
  constexpr int STRA = DqLds<DQK, SPILL>::STRA, ROWR = DqLds<DQK, SPILL>::ROWR;
  constexpr int TILEA = DqLds<DQK, SPILL>::TILEA, TILEB = DqLds<DQK, SPILL>::TILEB;
  constexpr int CPT = ROPE ? 9 : 8;    // DMA instructions per wave and tile
  typedef __attribute__((address_space(3))) uint8_t l_u8;
  typedef __attribute__((address_space(3))) void l_void;
  typedef short tr_s4 __attribute__((ext_vector_type(4)));
  l_u8* const lds = (l_u8*)sm.tiles;

  const int t = ur.x, split = ur.w;
  if (split < 0) return;  // a q row no batch owns: zero (bwd_prep_kernel)
  if (SPILL && (t < sp.t0 || t >= sp.t1)) return;  // a token of another run
  const int r0 = ur.y;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n16 = lane & 15, g = lane >> 4;
  const int h = hg * BW_HEADS + w * 16 + n16;
  const bool hvalid = h < a.H;
  const int hc = min(h, a.H - 1);
  const size_t th = (size_t)t * a.H + hc;
  // a tile's row addresses of this wave: lane l holds row 8 w + (l & 7)
  const uint64_t* alist = addr_list + (size_t)t * a.list_stride;
  typedef __attribute__((address_space(1))) const uint64_t g_u64;
  auto addrs = [&](int i) -> uint64_t {
    return ((g_u64*)(uintptr_t)alist)[min(r0 + i * BW_TILE + 8 * w + (lane & 7), a.list_stride - 1)];
  };
  uint64_t av = addrs(0), av1 = addrs(1), av2 = addrs(2);
  const int* tk = plan + SAS_PLAN_HDR + (size_t)t * SAS_TOK_W;
  const int splits = tk[TK_SPLITS];
  const int2 tr = tok[t];  // row counts at the call's lengths (the resolver's)
  if (tr.x < 0) return;    // refused token: zero (bwd_prep_kernel)
  const int r1 = min(split == splits - 1 ? tr.x + tr.y : min(ur.z, tr.x + tr.y), a.list_stride);
  const int ntiles = r1 > r0 ? (r1 - r0 + BW_TILE - 1) / BW_TILE : 0;

  // row 8 w + k: lane l fetches latent chunk l ^ f, f = 2 (k >> 2) + (w & 1); rope: lane 8 k +
  // j fetches chunk j ^ fr of row 8 w + k
  const uint32_t vlat = 16u * ((uint32_t)lane ^ (uint32_t)(w & 1));
  const uint32_t rx = (uint32_t)((8 * w + (lane >> 3)) >> 1) & 7u;
  const uint32_t vrope = 1024u + 16u * (((uint32_t)lane & 7u) ^ (((rx & 3u) << 1) | (rx >> 2)));
  auto tail = [&](uint64_t v, int i) -> uint64_t {  // rows past r1 read the zero row
    return r0 + i * BW_TILE + 8 * w + (lane & 7) < r1 ? v : (uint64_t)g_zero_row;
  };
  auto dma_lat = [&](int sl, uint64_t v, int k) {
    const uint64_t ra = ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(v >> 32), k) << 32) |
                        (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, k);
    uint32_t vo = vlat;
    if (k >= 4) {  // (formed here rather than kept across the loop)
      asm volatile("" : "+v"(vo));
      vo ^= 32u;
    }
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        __builtin_amdgcn_make_buffer_rsrc((void*)ra, (short)0, 1024, 0x00020000),
        (l_void*)(lds + sl * TILEB + (8 * w + k) * STRA), 16, vo, 0, 0, 0);
  };
  // (in assembly: the compiler takes a global LDS-direct load for a FLAT access and then
  // drains both counters at the next wait of either)
  auto dma_rope = [&](int sl, uint64_t v) {
    if constexpr (ROPE) {
      const int from = lane >> 3;
      const uint64_t src = (((uint64_t)(uint32_t)__shfl((int)(v >> 32), from) << 32) |
                            (uint32_t)__shfl((int)(uint32_t)v, from)) + vrope;
      const uint32_t m0 = (uint32_t)(uintptr_t)(lds + sl * TILEB + TILEA + 8 * w * ROWR);
      uint32_t keep;  // the compiler's own value of m0
      asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off\n\t"
                   "s_mov_b32 m0, %0" : "=&s"(keep) : "v"(src), "s"(m0) : "memory");
    }
  };
  // tiles 0 and 1 (dead tiles too), ahead of the query's loads
  av = tail(av, 0);
  av1 = tail(av1, 1);
#pragma unroll
  for (int k = 0; k < 8; ++k) dma_lat(0, av, k);
  dma_rope(0, av);
#pragma unroll
  for (int k = 0; k < 8; ++k) dma_lat(1, av1, k);
  dma_rope(1, av1);
  asm volatile("" ::: "memory");

  u32x4_t qf[KS], of[VKS], ot[VKS];
  {
    const u32x4_t* qr = reinterpret_cast<const u32x4_t*>(q + th * DQK);
    const u32x4_t* orow = reinterpret_cast<const u32x4_t*>(dout + th * DV);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qf[ks] = qr[4 * ks + g];
#pragma unroll
    for (int ks = 0; ks < VKS; ++ks) of[ks] = orow[4 * ks + g];
    const u32x4_t* trow = reinterpret_cast<const u32x4_t*>(bt.out + th * DV);
#pragma unroll
    for (int ks = 0; ks < VKS; ++ks) ot[ks] = trow[4 * ks + g];
  }
  const float lse_h = lse[th], lse2 = lse_h * LOG2E, sink = bt.sinks[hc];
  const float dl = bt.dlse ? bt.dlse[th] : 0.f;
  const float c = a.scale_log2;
  const float scale = c * 0.6931471805599453f;
  if constexpr (SPILL) {
    // an infinity or a NaN times zero is a NaN: one dot product with zeros per two values
    uint32_t zero = 0;
    asm volatile("" : "+v"(zero));  // (opaque: the products are not folded)
    float z = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int e = 0; e < 4; ++e) z = dot2_zero<QT>(qf[ks][e], zero, z);
#pragma unroll
    for (int ks = 0; ks < VKS; ++ks)
#pragma unroll
      for (int e = 0; e < 4; ++e) z = dot2_zero<QT>(of[ks][e], zero, z);
    if (__any(z != 0.f) && lane == 0) {
      sp.flags[1 + t] = 1;
      atomicAdd(sp.flags, 1);
    }
  }
  // D: the diagonal of the 16 heads' dO out^T (fragments of a row are the same registers as
  // an A and as a B operand): head h sits in lane (n = h, g = h >> 2), element h & 3
  float dh;
  {
    bw_f32x4 d0 = bw_f32x4{0.f, 0.f, 0.f, 0.f}, d1 = d0;
#pragma unroll
    for (int ks = 0; ks < VKS; ks += 2) {
      d0 = bw_mfma<QT>(of[ks], ot[ks], d0);
      d1 = bw_mfma<QT>(of[ks + 1], ot[ks + 1], d1);
    }
    const int e = n16 & 3;
    const float v0 = e & 1 ? d0[1] + d1[1] : d0[0] + d1[0], v1 = e & 1 ? d0[3] + d1[3] : d0[2] + d1[2];
    // a gradient of the LSE: d lse / d s_j = P_j and d lse / d sink = P_sink, so it
    // enters as dS = P (dP - (D - dlse)) and dsink = -P_sink (D - dlse)
    dh = __shfl(e & 2 ? v1 : v0, n16 + 16 * (n16 >> 2)) - dl;
    if (split == 0 && g == 0 && hvalid) {
      bt.dterm[th] = dh;
      // a sink of -inf has P_sink = 0 (lse may be -inf too when nothing is attended)
      bt.sterm[th] = sink == -INFINITY || dh == 0.f ? 0.f : -__expf(sink - lse_h) * dh;
    }
  }
  // SPILL: the wave's P and dS go through LDS: lane (n16, g) writes its 8 keys of head
  // n16 (16 B: positions 8 g .. + 7 of the head's 64-B row, key 16 kb + 4 g + r at
  // position 8 g + 4 kb + r), and ds_read_b64_tr_b16 returns 4 heads (4 g .. + 3) of
  // one position per lane, stored as 8 B of its key's record.  The 32-B halves of a row
  // are swapped for heads 4 .. 7 and 12 .. 15, so that the transposed reads touch every
  // bank once per 256 B.  Every wave makes the same four stores in every tile (positions
  // past the end, and waves past the padded heads, at an offset past the buffer, which
  // drops them), so that the waits for the ring's DMAs can count them.
  l_u8* const tpw = (l_u8*)sm.tp + (SPILL ? w * 2048 : 0);
  const bool sp_wave = SPILL && hg * BW_HEADS + w * 16 < sp.row_bytes / 4;  // (a padded head chunk ends)
  const auto sp_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(SPILL ? sp.data : nullptr), (short)0,
      (int)((1u + (uint32_t)(sp.t1 - sp.t0) * (uint32_t)sp.stride) * (uint32_t)sp.row_bytes), 0x00020000);
  const uint32_t sp_off = (1u + (uint32_t)(t - sp.t0) * (uint32_t)sp.stride) * (uint32_t)sp.row_bytes +
                          (uint32_t)((2 * hg + (w >> 1)) * 128 + (16 * (w & 1) + 4 * g) * 2);
  bw_f32x4 acc[NDB];
#pragma unroll
  for (int i = 0; i < NDB; ++i) acc[i] = bw_f32x4{0.f, 0.f, 0.f, 0.f};

  // K fragments: row 16 kb + n16, chunk 4 ks + g; K^T fragments: rows 4 g + (n16 >> 2) (+ 16),
  // dimensions 16 db + 4 (n16 & 3) .. + 3
  const uint32_t kf0 = n16 * STRA + 16 * (g ^ (2 * ((n16 >> 2) & 1) + ((n16 >> 3) & 1)));
  const uint32_t kx = (uint32_t)(n16 >> 1) & 7u;
  const uint32_t kfr = TILEA + n16 * ROWR + 16 * (g ^ (int)(((kx & 3u) << 1) | (kx >> 2)));
  const int trow = 4 * g + (n16 >> 2);
  const uint32_t tb0 = trow * STRA + 32 * (g & 1) + 16 * (((n16 >> 1) & 1) ^ ((g >> 1) & 1)) + 8 * (n16 & 1);
  const uint32_t tx = (uint32_t)(trow >> 1) & 7u;
  const uint32_t tbr = TILEA + trow * ROWR + 16 * (((n16 >> 1) & 1) ^ (int)(((tx & 3u) << 1) | (tx >> 2))) + 8 * (n16 & 1);

  int sl = 0;
  for (int i = 0; i < ntiles; ++i) {
    const int rb = r0 + i * BW_TILE;
    // Tile i has landed: younger are tile i + 1's DMAs, an address load and, from the
    // second tile on, the last tile's stores (in the first, the query's loads).  (The wait
    // for the addresses behind the barrier, which the compiler places, is the stricter one
    // from the second tile on: all but those stores.)
    if (i == 0)
      __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, 0));
    else
      __builtin_amdgcn_s_waitcnt(waitcnt_imm(CPT + 1 + (SPILL ? 4 : 0), 0));
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    const l_u8* tl = lds + sl * TILEB;
    const int s2 = sl == 0 ? 2 : sl - 1;  // tile i + 2's slot: tile i - 1's
    const uint64_t vn = tail(av2, i + 2);
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
        return ks < 16 ? lds_read_b128(tl + kf0 + 16 * STRA * kb + 64 * ks)
                       : lds_read_b128(tl + ((kfr + 16 * ROWR * kb) ^ (64u * (uint32_t)(ks - 16))));
      };
      u32x4_t kf[BW_AHEAD + 1];
#pragma unroll
      for (int st = 0; st < BW_AHEAD; ++st) kf[st] = kfrag(st);
      BW_SB();
#pragma unroll
      for (int st = 0; st < 2 * KS; ++st) {
        if (st + BW_AHEAD < 2 * KS) kf[(st + BW_AHEAD) % (BW_AHEAD + 1)] = kfrag(st + BW_AHEAD);
        const int kb = st / KS, ks = st - kb * KS;
        const u32x4_t av_ = kf[st % (BW_AHEAD + 1)];
        s[kb] = bw_mfma<QT>(av_, qf[ks], s[kb]);
        if (ks < VKS) dp[kb] = bw_mfma<QT>(av_, of[ks], dp[kb]);
        if ((st & 3) == 1 && (st >> 2) < 8) dma_lat(s2, vn, st >> 2);
        BW_SB();
      }
      dma_rope(s2, vn);
    }
    av2 = addrs(i + 3);
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
      {
        u32x4_t xs, xp;
#pragma unroll
        for (int e = 0; e < 4; ++e) {  // (heads at or past H: zeros)
          xs[e] = hvalid ? pack2_q16<QT>(ds[2 * e] * scale, ds[2 * e + 1] * scale) : 0u;
          xp[e] = hvalid ? pack2_q16<QT>(pr[2 * e], pr[2 * e + 1]) : 0u;
        }
        const int wo = 64 * n16 + 16 * (g ^ (2 * ((n16 >> 2) & 1)));
        *reinterpret_cast<__attribute__((address_space(3))) u32x4_t*>(tpw + wo) = xs;
        *reinterpret_cast<__attribute__((address_space(3))) u32x4_t*>(tpw + 1024 + wo) = xp;
        const l_u8* ro = tpw + 64 * (4 * g + (n16 >> 2)) + 8 * (n16 & 3);
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
          const uint32_t off = sp_wave && p < r1 && p < sp.stride ? sp_off + (uint32_t)p * (uint32_t)sp.row_bytes : ~0u - 127u;
          typedef uint32_t u2 __attribute__((ext_vector_type(2)));
          __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u2, v[x][0]), sp_rsrc, off, 0, 0);
          __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u2, v[x][1]), sp_rsrc, off + 64u, 0, 0);
        }
      }
    }
    // dq^T += K^T dS^T.  A = dimensions 16 db + n16 of keys 4 g .. 4 g + 3 (then 16 +
    // 4 g ..), read transposed from the row-major tile: within each 16-lane block,
    // ds_read_b64_tr_b16 gives lane j element j & 3 of the 8 bytes lane (j >> 2) + 4 e
    // addresses, for e = 0 .. 3; so lane i of block g addresses key 4 g + (i >> 2)
    // (+ 16), dimensions 16 db + 4 (i & 3) .. + 3.
    {
      // the K^T fragments, read BW_AHEAD_T blocks ahead
      auto kt_frag = [&](int db) -> u32x4_t {
        const l_u8* p = db < 32 ? tl + (tb0 ^ (32u * (uint32_t)(db & 1))) + 64 * (db >> 1)
                                : tl + (tbr ^ (32u * (uint32_t)(db - 32)));
        const int up = db < 32 ? 16 * STRA : 16 * ROWR;
        const tr_s4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) tr_s4*)p);
        const tr_s4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) tr_s4*)(p + up));
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
    sl = sl == 2 ? 0 : sl + 1;
  }
  __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, 15));  // the dead tiles' DMAs have landed
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

template <int DQK, int QT, bool SPILL>
__global__ __launch_bounds__(256, 1) void bwd_dq_kernel(SasFwdArgs a, const uint16_t* __restrict__ q,
                                                        const uint16_t* __restrict__ dout,
                                                        const uint64_t* __restrict__ addr_list,
                                                        const int2* __restrict__ tok,
                                                        const float* __restrict__ lse, SasBwdTerms bt,
                                                        const int* __restrict__ plan,
                                                        float* __restrict__ dq, SasBwdSpill sp) {
  __shared__ DqLds<DQK, SPILL> sm;
  const int HG = (a.H + BW_HEADS - 1) / BW_HEADS;
  const int u = blockIdx.x / HG, hg = blockIdx.x - u * HG;
  // (the unit's record with the plan's header: one memory round trip for both; plan is the
  // workspace's, which holds the grid's unit capacity: see resolve_kernel)
  const int* up = plan + SAS_PLAN_HDR + (size_t)SAS_TOK_W * a.T + (size_t)u * SAS_UNIT_W;
  int4 ur = make_int4(up[0], up[1], up[2], up[3]);
  const int units = plan[PH_UNITS];
  const bool ok = plan_matches(plan, a);
  asm volatile("" : "+s"(ur.x), "+s"(ur.y), "+s"(ur.z), "+s"(ur.w));
  if (!ok || u >= units) return;  // refused plan: prep zeroed dq
  dq_unit<DQK, QT, SPILL>(sm, ur, hg, a, q, dout, addr_list, tok, lse, bt, plan, dq, sp);
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
