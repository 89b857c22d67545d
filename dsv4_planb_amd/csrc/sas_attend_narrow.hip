// sas_attend_narrow.hip -- the attention kernel for at most 64 heads (16-bit KV).
//
// The pipeline of sas_attend.hip (Q in VGPRs, fp32 O^T in AGPRs, KV rows gathered
// straight into an LDS ring, S of the next tile under the softmax of this one, one frame
// per unit, the same epilogue and partials) with half the heads: that kernel's four waves
// hold 128 heads, so at 64 two of them, and at 16 three, would work on clamped heads.  Here
// a workgroup is two waves of 32 heads and a tile is 16 keys, so its ring takes 76 KB and
// two workgroups share a CU: one unit's start and epilogue (about 27,000 cycles, twice
// the loop of a 128-row window) run under the other's tiles.
//
// A tile, per wave (16 keys x 32 heads):
//   S = K Q^T     2 x 18 MFMA 16x16x32 (16 keys x 16 heads, heads 0 .. 15 and 16 .. 31 of
//                 the wave), one K fragment (ds_read_b128) for both.
//                 v_permlane16_swap of the two blocks' results then leaves lane l with
//                 head l & 31, keys 8 (l >> 5) .. + 7: the B operand's layout.
//   O^T += V^T P^T  16 MFMA 32x32x16, V^T read transposed (ds_read_b64_tr_b16).
// The same LDS bytes per FLOP as 32-key tiles (a K or V byte is used for 32 heads).
//
// Measured (attention and resolver, before: the four-wave kernel): packed prompts of 2,068
// to 3,684 tokens, 64 heads, top-k 512, 1,245 -> 818 us (480 -> 740 TFLOP/s); a
// window-only prompt of 8,192 tokens, 64 heads, d_qk 512, fp16, 493 -> 335 us.  A unit's
// cycles (window only: start to its token's record 11,800, query and first DMAs 4,200,
// eight tiles 16,800 of which 8,200 are MFMA, epilogue 8,800): half of a short unit is
// latency, which is why two share a CU and why the unit's record is read with the plan's
// header.
//
// LDS tile: latent rows at a 1088-B stride with the 16-B chunk c of row r at c ^ ((r >> 2)
// & 3), rope rows of 128 B with chunk c at c ^ ((r >> 1) & 7), as in the 32-key tile: the
// b128 K reads (16 rows, one chunk) and the transposed V reads (4 rows x 4 chunks per 16
// lanes) touch every bank once per 256 B.  A wave's 8 rope rows are one DMA (lane 8 k + j:
// chunk j of row k; the row addresses, in SGPRs a tile ahead, are moved into the lanes
// before it) instead of one of 8 lanes per row.
#include <hip/hip_runtime.h>

#include "sas_common.h"

namespace sas {

constexpr int NW_NT = 128;    // threads per workgroup
constexpr int NW_TILE = 16;   // keys per tile
constexpr int NW_STAGES = 4;  // ring slots
constexpr int NW_AHEAD = 4;   // K fragments read ahead of their MFMAs

template <int DQK>
struct NarrowLds {
  static constexpr int TILEB = NW_TILE * (1024 + 64) + NW_TILE * (DQK - 512) * 2;
  __attribute__((aligned(16))) uint8_t tiles[NW_STAGES * TILEB];
  int far;           // a logit of some head outgrew the frame
  uint64_t* stamps;  // as in AttendLds
  uint64_t t0;
};

// d = a b^T + 0 / d += a b^T in VGPRs, 16 x 16 x 32 (see vmfma_first).
template <int QT>
__device__ __forceinline__ void vmfma16_first(f32x4_t& d, const u32x4_t& a, const u32x4_t& b) {
  if constexpr (QT == 0)
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=&v"(d) : "v"(a), "v"(b));
  else
    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, 0" : "=&v"(d) : "v"(a), "v"(b));
}
template <int QT>
__device__ __forceinline__ void vmfma16_acc(f32x4_t& d, const u32x4_t& a, const u32x4_t& b) {
  if constexpr (QT == 0)
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(d) : "v"(a), "v"(b));
  else
    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+v"(d) : "v"(a), "v"(b));
}

// One work unit (its record ur); see attend_unit.
template <int DQK, int QT, bool STREAM, bool REDO>
__device__ __forceinline__ bool narrow_unit(
    int4 ur, NarrowLds<DQK>& sm, const SasFwdArgs& a, const uint16_t* __restrict__ q,
    const uint64_t* __restrict__ addr_list, const int2* __restrict__ tokr,
    const float* __restrict__ sinks, const int* __restrict__ plan, uint16_t* __restrict__ out,
    float* __restrict__ lse, float* __restrict__ ws_o, float* __restrict__ ws_ml, float& m_obs) {
  constexpr int DV = 512;
  constexpr bool ROPE = DQK > DV;
  constexpr int ROWA = DV * 2, STRA = ROWA + 64, ROWR = (DQK - DV) * 2;
  constexpr int TILE = NW_TILE, TILEA = TILE * STRA, TILEB = NarrowLds<DQK>::TILEB;
  constexpr int KS = DQK / 32;             // k-steps of Q K^T (18 / 16)
  constexpr int CPT = ROPE ? 9 : 8;        // DMA instructions per wave and tile
  static_assert(2 * EPI_WAVE <= NW_STAGES * TILEB, "the epilogue staging fits the ring");
  lds_u8* const tiles = (lds_u8*)sm.tiles;

  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));  // (so that the redo's copy does not share, and keep, these)
  const int lane = tid & 63, w = tid >> 6;
  const int g = lane >> 5, li = lane & 31;     // PV and softmax: keys 8 g .., head li
  const int n16 = lane & 15, g4 = lane >> 4;   // QK: row / head n16, dimensions 8 g4 ..

  const int t = ur.x, split = ur.w;
  const int H = a.H;
  auto zero_token = [&]() {
    for (int i = tid; i < H * DV / 8; i += NW_NT)
      reinterpret_cast<u32x4_t*>(out + (size_t)t * H * DV)[i] = u32x4_t{0, 0, 0, 0};
    if (lse)
      for (int i = tid; i < H; i += NW_NT) lse[(size_t)t * H + i] = 0.f;
  };
  if (!REDO && split < 0) {  // a q row no batch owns
    zero_token();
    return false;
  }
  const int r0 = ur.y;
  const int h = w * 32 + li;
  const bool hvalid = h < H;
  const float sink_raw = sinks[min(h, H - 1)];

  // The first four tiles' row addresses of this wave (lane 8 i + k: tile i, row 8 w + k), in
  // one vector load inside the token's list, issued ahead of the query's.
  const int pro_row = r0 + ((lane >> 3) & 3) * TILE + 8 * w + (lane & 7);
  const int pro_ld = min(pro_row, a.list_stride - 1);
  typedef __attribute__((address_space(1))) const uint64_t g_u64;
  uint64_t pro_addr = ((g_u64*)(uintptr_t)addr_list)[(size_t)t * a.list_stride + pro_ld];
  asm volatile("" ::: "memory");
  u32x4_t qf[2][KS];  // heads 16 hb + n16 of the wave, dimensions 32 ks + 8 g4 .. + 7
#pragma unroll
  for (int hb = 0; hb < 2; ++hb) {
    const u32x4_t* qrow =
        reinterpret_cast<const u32x4_t*>(q + ((size_t)t * H + min(w * 32 + 16 * hb + n16, H - 1)) * DQK);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qf[hb][ks] = qrow[4 * ks + g4];
  }
  const int* tk = plan + SAS_PLAN_HDR + (size_t)t * SAS_TOK_W;
  const int splits = tk[TK_SPLITS], wsbase = tk[TK_WSBASE];
  const int2 tr = tokr[t];
  if (!REDO && tr.x < 0) {  // a token refused for a plan that no longer matches it
    zero_token();
    return false;
  }
  const int rows_live = tr.x + tr.y;
  const int r1 = min(split == splits - 1 ? rows_live : min(ur.z, rows_live), a.list_stride);
  const int ntiles = r1 > r0 ? (r1 - r0 + TILE - 1) / TILE : 0;
  const uint64_t* alist = addr_list + (size_t)t * a.list_stride + r0;
  const float sink2 = split == 0 ? sink_raw * LOG2E : -INFINITY;

  if (!REDO && ntiles == 0) {  // O = 0 and the normalisers are the sink's alone
    if (!hvalid) return false;
    const float l_sink = split == 0 ? 1.f : 0.f;
    if (splits == 1) {
      uint16_t* orow = out + ((size_t)t * H + h) * DV + 16 * g;
#pragma unroll
      for (int mb = 0; mb < 16; ++mb)
#pragma unroll
        for (int hf = 0; hf < 2; ++hf)
          *reinterpret_cast<u32x4_t*>(orow + 32 * mb + 8 * hf) = u32x4_t{0, 0, 0, 0};
      if (lse && g == 0) lse[(size_t)t * H + h] = (sink2 + __log2f(l_sink)) * 0.6931471805599453f;
    } else {
      const int slot = wsbase + split;
      if (slot < 0 || slot >= a.slot_cap) return false;  // (a sound plan never gets here)
      uint8_t* orow = reinterpret_cast<uint8_t*>(ws_o + ((size_t)slot * H + h) * DV) + 16 * g;
#pragma unroll
      for (int k = 0; k < (PART16<QT> ? 32 : 64); ++k)
        *reinterpret_cast<u32x4_t*>(orow + 32 * k) = u32x4_t{0, 0, 0, 0};
      if (g == 0)
        reinterpret_cast<float4*>(ws_ml)[(size_t)slot * H + h] =
            make_float4(sink2, l_sink, l_sink, PART16<QT> ? 1.f : 0.f);
    }
    return false;
  }

  // ---- per-lane LDS offsets (bytes within a tile) ----
  // K, latent k-step ks: row n16, chunk 4 ks + g4 -> kofs + 64 ks; rope k-step 16 + j: rope
  // chunk 4 j + g4 -> kofs_r ^ 64 j.
  const uint32_t kofs = n16 * STRA + 16 * (g4 ^ swz_a(n16));
  const uint32_t kofs_r = TILEA + n16 * ROWR + 16 * (g4 ^ swz_b(n16));
  // V^T (A of O^T += V^T P^T): MFMA row m of d-block mb is d = 32 mb + dmap(m) (see
  // attend_unit), k index 8 g + e is key 8 g + e.  Lane l supplies row 8 (l >> 5) + ((l >>
  // 2) & 3) + 4 hf (hf = e >> 2) at column 32 mb + 16 (l & 1) + 8 ((l >> 4) & 1) + 4 ((l >>
  // 1) & 1): vofs[hf] + 64 mb.
  uint32_t vofs[2];
  {
    const int clo = 2 * (lane & 1) + ((lane >> 4) & 1);
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) {
      const int row = 8 * (lane >> 5) + ((lane >> 2) & 3) + 4 * hf;
      vofs[hf] = row * STRA + 16 * (clo ^ swz_a(row)) + 8 * ((lane >> 1) & 1);
    }
  }

  f32x16_t acc[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i] = f32x16_t{};
  float m_run = REDO ? m_obs : sink2;  // redo: the frame is the maximum pass 1 observed

  // ---- gather: tile i goes to ring slot i & 3; wave w copies its rows 8 w .. 8 w + 7 ----
  const int wu = __builtin_amdgcn_readfirstlane(w);
  const uint32_t ulane = (uint32_t)lane;
  // row 8 w + k: lane l fetches source chunk l ^ swz_a(8 w + k) = l ^ ((2 w + (k >> 2)) & 3)
  const uint32_t voffA0 = 16u * (ulane ^ (uint32_t)((2 * wu) & 3));
  // rope: lane 8 k + j fetches chunk j ^ swz_b(8 w + k) of row 8 w + k
  const uint32_t vrope = ROWA + 16u * ((ulane & 7u) ^ (uint32_t)swz_b(8 * wu + (lane >> 3)));
  typedef uint64_t RowAddrs __attribute__((ext_vector_type(8)));
  auto fix_tail = [&](RowAddrs ra, int i) -> RowAddrs {  // rows past r1 read the zero row
    const int rb = r0 + i * TILE + 8 * wu;
    if (rb + 8 > r1) {
#pragma unroll
      for (int k = 0; k < 8; ++k)
        if (rb + k >= r1) ra[k] = (uint64_t)g_zero_row;
    }
    return ra;
  };
  auto load_addrs = [&](int i) -> RowAddrs {
    const int il = min(i, ntiles - 1);  // dead tiles (i >= ntiles) read zeros
    typedef __attribute__((address_space(4))) const RowAddrs c_RowAddrs;
    return fix_tail(*(c_RowAddrs*)(uintptr_t)(alist + il * TILE + 8 * wu), i);
  };
  if (pro_row >= r1) pro_addr = (uint64_t)g_zero_row;
  auto pro_addrs = [&](int i) -> RowAddrs {
    RowAddrs ra;
#pragma unroll
    for (int k = 0; k < 8; ++k)
      ra[k] = ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(pro_addr >> 32), 8 * i + k) << 32) |
              (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)pro_addr, 8 * i + k);
    return ra;
  };
  auto dma_lat = [&](int i, const RowAddrs& ra, int k) {
    lds_u8* dst = tiles + (i & (NW_STAGES - 1)) * TILEB + (8 * wu + k) * STRA;
    // (rows 4 .. 7: 2 w + 1 instead of 2 w, formed here rather than kept across the loop)
    uint32_t vo = voffA0;
    if (k >= 4) {
      asm volatile("" : "+v"(vo));
      vo ^= 16u;
    }
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        __builtin_amdgcn_make_buffer_rsrc((void*)ra[k], (short)0, ROWA, 0x00020000),
        (void __attribute__((address_space(3)))*)dst, 16, vo, 0, 0,
        gather_cpol<STREAM>());
  };
  // The 8 rope rows in one DMA: lane 8 k + j's row address is ra[k], moved from the SGPRs
  // into the lanes eight at a time (a vector load of the addresses would be one more
  // outstanding load, which the compiler waits for where the loop's paths join).  In
  // assembly also the DMA: the compiler takes a global LDS-direct load for a FLAT access
  // and then drains both counters at the next wait of either.  (It does not count this
  // load, so its own vector memory waits are stricter by one.)
  auto dma_rope = [&](int i, const RowAddrs& ra) {
    if constexpr (ROPE) {
      lds_u8* dst = tiles + (i & (NW_STAGES - 1)) * TILEB + TILEA + 8 * wu * ROWR;
      uint32_t lo, hi;
      uint64_t ex;
      asm volatile(
          "s_mov_b64 %[ex], exec\n\t"
          "s_mov_b64 exec, 0xff\n\t" "v_mov_b32 %[lo], %[l0]\n\t" "v_mov_b32 %[hi], %[h0]\n\t"
          "s_lshl_b64 exec, exec, 8\n\t" "v_mov_b32 %[lo], %[l1]\n\t" "v_mov_b32 %[hi], %[h1]\n\t"
          "s_lshl_b64 exec, exec, 8\n\t" "v_mov_b32 %[lo], %[l2]\n\t" "v_mov_b32 %[hi], %[h2]\n\t"
          "s_lshl_b64 exec, exec, 8\n\t" "v_mov_b32 %[lo], %[l3]\n\t" "v_mov_b32 %[hi], %[h3]\n\t"
          "s_lshl_b64 exec, exec, 8\n\t" "v_mov_b32 %[lo], %[l4]\n\t" "v_mov_b32 %[hi], %[h4]\n\t"
          "s_lshl_b64 exec, exec, 8\n\t" "v_mov_b32 %[lo], %[l5]\n\t" "v_mov_b32 %[hi], %[h5]\n\t"
          "s_lshl_b64 exec, exec, 8\n\t" "v_mov_b32 %[lo], %[l6]\n\t" "v_mov_b32 %[hi], %[h6]\n\t"
          "s_lshl_b64 exec, exec, 8\n\t" "v_mov_b32 %[lo], %[l7]\n\t" "v_mov_b32 %[hi], %[h7]\n\t"
          "s_mov_b64 exec, %[ex]"
          : [lo] "=&v"(lo), [hi] "=&v"(hi), [ex] "=&s"(ex)
          : [l0] "s"((uint32_t)ra[0]), [h0] "s"((uint32_t)(ra[0] >> 32)),
            [l1] "s"((uint32_t)ra[1]), [h1] "s"((uint32_t)(ra[1] >> 32)),
            [l2] "s"((uint32_t)ra[2]), [h2] "s"((uint32_t)(ra[2] >> 32)),
            [l3] "s"((uint32_t)ra[3]), [h3] "s"((uint32_t)(ra[3] >> 32)),
            [l4] "s"((uint32_t)ra[4]), [h4] "s"((uint32_t)(ra[4] >> 32)),
            [l5] "s"((uint32_t)ra[5]), [h5] "s"((uint32_t)(ra[5] >> 32)),
            [l6] "s"((uint32_t)ra[6]), [h6] "s"((uint32_t)(ra[6] >> 32)),
            [l7] "s"((uint32_t)ra[7]), [h7] "s"((uint32_t)(ra[7] >> 32))
          : "scc");  // (the shifts of exec)
      const uint64_t src = (((uint64_t)hi << 32) | lo) + vrope;
      const uint32_t m0 = (uint32_t)(uintptr_t)dst;
      uint32_t keep;  // the compiler's own value of m0
      if constexpr (STREAM)
        asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off nt\n\t"
                     "s_mov_b32 m0, %0" : "=&s"(keep) : "v"(src), "s"(m0) : "memory");
      else
        asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off\n\t"
                     "s_mov_b32 m0, %0" : "=&s"(keep) : "v"(src), "s"(m0) : "memory");
    }
  };

  // ---- S = K Q^T: work(ks) runs after step ks's MFMAs issue (ks = -1: before the first;
  // ks = KS: after the last) ----
  auto kread = [&](const lds_u8* tl, int ks, uint32_t kr) -> u32x4_t {
    return ks < 16 ? lds_read_b128(tl + kofs + 64 * ks)
                   : lds_read_b128(tl + (kr ^ (64u * (uint32_t)(ks - 16))));
  };
  auto qk = [&](const lds_u8* tl, f32x4_t (&s)[2], auto&& work) {
    uint32_t kr = kofs_r;
    asm volatile("" : "+v"(kr));
    u32x4_t kb[NW_AHEAD];
#pragma unroll
    for (int j = 0; j < NW_AHEAD; ++j) kb[j] = kread(tl, j, kr);
    SB();
    work(-1);
    SB();
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      if (ks == 0) {
        vmfma16_first<QT>(s[0], kb[0], qf[0][0]);
        vmfma16_first<QT>(s[1], kb[0], qf[1][0]);
      } else {
        vmfma16_acc<QT>(s[0], kb[ks % NW_AHEAD], qf[0][ks]);
        vmfma16_acc<QT>(s[1], kb[ks % NW_AHEAD], qf[1][ks]);
      }
      // (an MFMA reads its operands when it issues: the fragment is free)
      if (ks + NW_AHEAD < KS) kb[ks % NW_AHEAD] = kread(tl, ks + NW_AHEAD, kr);
      work(ks);
      SB();
    }
    work(KS);
    SB();
  };

  // ---- O^T += V^T P^T: one inline-assembly block that also carries the scalar load of a
  // later tile's row addresses (see attend_unit) ----
  auto pv_asm = [&](const lds_u8* tl, const u32x4_t& pk, const uint64_t* aptr) -> RowAddrs {
    const uint32_t a0 = (uint32_t)(uintptr_t)tl + vofs[0];
    const uint32_t a1 = (uint32_t)(uintptr_t)tl + vofs[1];
    typedef uint32_t u32x16_t __attribute__((ext_vector_type(16)));
    u32x16_t sa;
#define NV_RD(j, b) \
    "ds_read_b64_tr_b16 v[" #b ":" #b "+1], %[a0] offset:" #j "\n\t" \
    "ds_read_b64_tr_b16 v[" #b "+2:" #b "+3], %[a1] offset:" #j "\n\t"
#define NV_MM(MN, c, b) MN " %[c" #c "], v[" #b ":" #b "+3], %[p], %[c" #c "]\n\t"
#define NV_ASM(MN) \
    asm volatile( \
        "s_load_dwordx16 %[sa], %[ap], 0x0\n\t" \
        NV_RD(0, 244) NV_RD(64, 248) NV_RD(128, 252) \
        "s_waitcnt lgkmcnt(4)\n\t" NV_MM(MN, 0, 244) NV_RD(192, 244) \
        "s_waitcnt lgkmcnt(4)\n\t" NV_MM(MN, 1, 248) NV_RD(256, 248) \
        "s_waitcnt lgkmcnt(4)\n\t" NV_MM(MN, 2, 252) NV_RD(320, 252) \
        "s_waitcnt lgkmcnt(4)\n\t" NV_MM(MN, 3, 244) NV_RD(384, 244) \
        "s_waitcnt lgkmcnt(4)\n\t" NV_MM(MN, 4, 248) NV_RD(448, 248) \
        "s_waitcnt lgkmcnt(4)\n\t" NV_MM(MN, 5, 252) NV_RD(512, 252) \
        "s_waitcnt lgkmcnt(4)\n\t" NV_MM(MN, 6, 244) NV_RD(576, 244) \
        "s_waitcnt lgkmcnt(4)\n\t" NV_MM(MN, 7, 248) NV_RD(640, 248) \
        "s_waitcnt lgkmcnt(4)\n\t" NV_MM(MN, 8, 252) NV_RD(704, 252) \
        "s_waitcnt lgkmcnt(4)\n\t" NV_MM(MN, 9, 244) NV_RD(768, 244) \
        "s_waitcnt lgkmcnt(4)\n\t" NV_MM(MN, 10, 248) NV_RD(832, 248) \
        "s_waitcnt lgkmcnt(4)\n\t" NV_MM(MN, 11, 252) NV_RD(896, 252) \
        "s_waitcnt lgkmcnt(4)\n\t" NV_MM(MN, 12, 244) NV_RD(960, 244) \
        "s_waitcnt lgkmcnt(4)\n\t" NV_MM(MN, 13, 248) \
        "s_waitcnt lgkmcnt(2)\n\t" NV_MM(MN, 14, 252) \
        "s_waitcnt lgkmcnt(0)\n\t" NV_MM(MN, 15, 244) \
        : [sa] "=s"(sa), [c0] "+a"(acc[0]), [c1] "+a"(acc[1]), [c2] "+a"(acc[2]), [c3] "+a"(acc[3]), \
          [c4] "+a"(acc[4]), [c5] "+a"(acc[5]), [c6] "+a"(acc[6]), [c7] "+a"(acc[7]), \
          [c8] "+a"(acc[8]), [c9] "+a"(acc[9]), [c10] "+a"(acc[10]), [c11] "+a"(acc[11]), \
          [c12] "+a"(acc[12]), [c13] "+a"(acc[13]), [c14] "+a"(acc[14]), [c15] "+a"(acc[15]) \
        : [a0] "v"(a0), [a1] "v"(a1), [p] "v"(pk), [ap] "s"(aptr) \
        : "v244", "v245", "v246", "v247", "v248", "v249", "v250", "v251", "v252", "v253", \
          "v254", "v255", "memory");
    if constexpr (QT == 0) {
      NV_ASM("v_mfma_f32_32x32x16_bf16")
    } else {
      NV_ASM("v_mfma_f32_32x32x16_f16")
    }
#undef NV_ASM
#undef NV_RD
#undef NV_MM
    return __builtin_bit_cast(RowAddrs, sa);
  };

  // ---- softmax of one tile: x[e] is key 8 g + e of head li ----
  float pe = 0.f, pw = 0.f;  // sums of P (LSE) and of the rounded P (output), per lane
  float xo = -INFINITY;      // max of x - m over the unit, for the overflow guard
  const float c = a.scale_log2;
  typedef float f32x8_t __attribute__((ext_vector_type(8)));
  // the two 16 x 16 blocks' results: lane (n16, g4) holds keys 4 g4 + r of head 16 hb + n16
  auto hand_off = [&](f32x4_t (&s)[2]) -> f32x8_t {
    f32x8_t x;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const auto sw = __builtin_amdgcn_permlane16_swap(__float_as_uint(s[0][r]), __float_as_uint(s[1][r]), false, false);
      x[r] = __uint_as_float(sw[0]);
      x[4 + r] = __uint_as_float(sw[1]);
    }
    return x;
  };
  auto tile_max = [&](const f32x8_t& x) {
    float mt = fmaxf(fmaxf(x[0], x[1]), x[2]);
    mt = fmaxf(mt, fmaxf(x[3], x[4]));
    mt = fmaxf(mt, fmaxf(x[5], x[6]));
    mt = fmaxf(mt, x[7]);
    const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(mt), __float_as_uint(mt), false, false);
    return fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
  };
  // one phase of chunk k (keys 2 k, 2 k + 1), pinned where it stands (see attend_unit)
  auto sm_phase = [&](f32x8_t& x, u32x4_t& pk, int k, int ph, bool scaled) {
    float x0 = x[2 * k], x1 = x[2 * k + 1];
    if (ph == 0) {
      x0 = scaled ? x0 - m_run : fmaf(x0, c, -m_run);
      x1 = scaled ? x1 - m_run : fmaf(x1, c, -m_run);
      float m = fmaxf(xo, fmaxf(x0, x1));
      asm volatile("" : "+v"(x0), "+v"(x1), "+v"(m));
      xo = m;
    } else if (ph == 1) {
      x0 = __builtin_amdgcn_exp2f(x0);
      x1 = __builtin_amdgcn_exp2f(x1);
      asm volatile("" : "+v"(x0), "+v"(x1));
    } else if (ph == 2) {
      uint32_t p = pack2_q16<QT>(x0, x1);
      float e = pe + (x0 + x1);
      asm volatile("" : "+v"(p), "+v"(e));
      pk[k] = p;
      pe = e;
    } else {
      float w2 = sum2_q16<QT>(pk[k], pw);
      asm volatile("" : "+v"(w2));
      pw = w2;
    }
    x[2 * k] = x0;
    x[2 * k + 1] = x1;
  };
  // work items of the next tile's QK chain: chunk i >> 2's phase i & 3 at step i - 1
  auto sm_step = [&](f32x8_t& x, u32x4_t& pk, int ks) {
    const int i = ks + 1;
    if (i >= 0 && i < 16) sm_phase(x, pk, i >> 2, i & 3, false);
  };
  auto softmax_last = [&](f32x8_t& x, u32x4_t& pk, bool first, int nvalid) {
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] *= c;
    if (nvalid < TILE) {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (8 * g + e >= nvalid) x[e] = -INFINITY;
    }
    if (first) m_run = fmaxf(m_run, tile_max(x));
#pragma unroll
    for (int i = 0; i < 16; ++i) sm_phase(x, pk, i >> 2, i & 3, true);
  };

  if (!REDO && tid == 0) sm.far = 0;
  {
    // Ring schedule as in attend_unit: iteration i waits for tile i + 1, computes S(i + 1)
    // under the softmax of tile i and the issue of tile i + 3's DMAs, then PV(i).
    RowAddrs ra_next;
#pragma unroll
    for (int i0 = 0; i0 < 3; ++i0) {
      ra_next = pro_addrs(i0);
#pragma unroll
      for (int k = 0; k < 8; ++k) dma_lat(i0, ra_next, k);
      dma_rope(i0, ra_next);
    }
    ra_next = load_addrs(3);

    f32x4_t s2[2];
    __builtin_amdgcn_s_waitcnt(waitcnt_imm(2 * CPT, 15));  // tile 0 landed
    wait_barrier();
    qk(tiles, s2, [](int) {});
    // S(0) is read by VALU next: wait out the XDL-write -> VALU-read hazard
    asm volatile("s_nop 7\n\ts_nop 7" : "+v"(s2[0]), "+v"(s2[1]));
    f32x8_t x = hand_off(s2);

    for (int i = 0; i < ntiles; ++i) {
      u32x4_t pk;
      if (i + 1 < ntiles) {
        __builtin_amdgcn_s_waitcnt(waitcnt_imm(CPT, 15));  // tile i + 1 landed
        wait_barrier();
        const RowAddrs ra_cur = ra_next;
        const lds_u8* tn = tiles + ((i + 1) & (NW_STAGES - 1)) * TILEB;
        auto gather = [&](int ks) {
          if (ks >= 0 && (ks & 1) && (ks >> 1) < 8) dma_lat(i + 3, ra_cur, ks >> 1);
          if (ks == KS - 2) dma_rope(i + 3, ra_cur);  // (no softmax work left)
        };
        if (!REDO && i == 0) {
          // The unit's frame: the maximum of its first 32 keys, as in the 128-head kernel
          // (16 keys would make the largest P exactly 1, free of rounding, half as
          // often), so the first tile's softmax follows the second one's S.
          qk(tn, s2, gather);
          asm volatile("s_nop 7\n\ts_nop 7" : "+v"(s2[0]), "+v"(s2[1]));
          f32x4_t sc[2] = {s2[0], s2[1]};
          f32x8_t x1 = hand_off(sc);
          const int nv = r1 - (r0 + TILE) - 8 * g;  // the second tile may be the last one
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            x[e] *= c;
            x1[e] = e < nv ? x1[e] * c : -INFINITY;
          }
          m_run = fmaxf(m_run, fmaxf(tile_max(x), tile_max(x1)));
#pragma unroll
          for (int k = 0; k < 16; ++k) sm_phase(x, pk, k >> 2, k & 3, true);
        } else {
          qk(tn, s2, [&](int ks) {
            sm_step(x, pk, ks);
            gather(ks);
          });
        }
      } else {
        softmax_last(x, pk, !REDO && i == 0, r1 - (r0 + i * TILE));
      }
      SB();
      {
        const int il = min(i + 4, ntiles - 1);  // dead tiles (>= ntiles) read zeros
        ra_next = fix_tail(pv_asm(tiles + (i & (NW_STAGES - 1)) * TILEB, pk, alist + il * TILE + 8 * wu), i + 4);
      }
      // S(i + 1) is handed over after PV's MFMAs, which covers the XDL-write -> VALU-read
      // hazard of the chain's last two
      asm volatile("" : "+v"(s2[0]), "+v"(s2[1]));
      x = hand_off(s2);
    }
    __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, 15));  // the dead-tile DMAs have landed
    asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7" ::: "memory");
  }
  // (the epilogue's lane numbers are formed again here: kept across the loop, they and the
  // addresses made of them would not fit the registers)
  int etid = threadIdx.x;
  asm volatile("" : "+v"(etid));
  const int el = etid & 63, ew = etid >> 6, eg = (etid >> 5) & 1, eli = etid & 31, eh = ew * 32 + eli;
  const bool ehv = eh < H;
  // both half-waves of a head, summed in the same order in both
  float pes = pe, pws = pw, xobs = xo;
  {
    const auto a1 = __builtin_amdgcn_permlane32_swap(__float_as_uint(pes), __float_as_uint(pes), false, false);
    const auto a2 = __builtin_amdgcn_permlane32_swap(__float_as_uint(pws), __float_as_uint(pws), false, false);
    const auto a3 = __builtin_amdgcn_permlane32_swap(__float_as_uint(xobs), __float_as_uint(xobs), false, false);
    pes = __uint_as_float(a1[0]) + __uint_as_float(a1[1]);
    pws = __uint_as_float(a2[0]) + __uint_as_float(a2[1]);
    xobs = fmaxf(__uint_as_float(a3[0]), __uint_as_float(a3[1]));
  }
  const float l_sink = split != 0 ? 0.f : (sink2 == m_run ? 1.f : exp2f(sink2 - m_run));
  const float l_e = l_sink + pes, l_w = l_sink + pws;

  // ---- overflow guard: a logit far above the frame redoes the whole unit ----
  if (!REDO) {
    if (__any(xobs > redo_slack<QT>()) && el == 0) atomicOr(&sm.far, 1);
    lds_barrier();
    if (sm.far) {
      m_obs = m_run + xobs;
      return true;
    }
  }

  // ---- epilogue: the output leaves through LDS (see attend_unit) ----
  if constexpr (REDO) lds_barrier();
  lds_u8* const ob = tiles + ew * EPI_WAVE;
  const int nrows = min(32, H - 32 * ew);  // this wave's heads below H (wave-uniform)
  auto rows_out = [&](auto* dst, size_t row_elems) {
#pragma unroll
    for (int r0 = 0; r0 < 32; r0 += 8) {
      u32x4_t v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = lds_read_b128(ob + (r0 + j) * EPI_STRIDE + 16 * el);
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (r0 + j < nrows)
          __builtin_nontemporal_store(
              v[j], reinterpret_cast<u32x4_t*>(reinterpret_cast<uint8_t*>(dst + (r0 + j) * row_elems) + 16 * el));
    }
  };
  auto lds_w128 = [&](int off, u32x4_t v) {
    *reinterpret_cast<__attribute__((address_space(3))) u32x4_t*>(ob + off) = v;
  };
  float mx = 0.f;
  auto stage16 = [&](auto pk, float sc, auto track) {
#pragma unroll
    for (int mb = 0; mb < 16; ++mb) {
      f32x16_t v = acc[mb];
      asm volatile("" : "+v"(v));
      if constexpr (decltype(track)::value) {
#pragma unroll
        for (int r = 0; r < 16; ++r) mx = fmaxf(mx, fabsf(v[r]));
      }
#pragma unroll
      for (int hf = 0; hf < 2; ++hf) {
        u32x4_t o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = pk(v[8 * hf + 2 * e] * sc, v[8 * hf + 2 * e + 1] * sc);
        lds_w128(eli * EPI_STRIDE + 64 * mb + 32 * eg + 16 * hf, o);
      }
      SB();  // (one block's values in VGPRs at a time)
    }
  };
  const float inv = l_w > 0.f ? 1.f / l_w : 0.f;
  if (splits == 1) {
    stage16([](float x, float y) { return pack2_q16<QT>(x, y); }, inv, std::false_type{});
    rows_out(out + ((size_t)t * H + 32 * ew) * DV, DV);
    if (lse && eg == 0 && ehv) lse[(size_t)t * H + eh] = (m_run + __log2f(l_e)) * 0.6931471805599453f;
    return false;
  }
  const int slot = wsbase + split;
  if (slot < 0 || slot >= a.slot_cap) return false;  // (a sound plan never gets here)
  if constexpr (PART16<QT> && !REDO) {
    stage16([](float x, float z) { return pack2_q16<1>(x, z); }, inv, std::true_type{});
    const bool over = ehv && mx * inv >= 65504.f;
    if (__any(over) && el == 0) atomicOr(&sm.far, 1);
    lds_barrier();
    if (sm.far) {
      m_obs = m_run + xobs;
      return true;
    }
    rows_out(reinterpret_cast<uint16_t*>(ws_o + ((size_t)slot * H + 32 * ew) * DV), 2 * DV);
    if (eg == 0 && ehv)
      reinterpret_cast<float4*>(ws_ml)[(size_t)slot * H + eh] = make_float4(m_run, l_w, l_e, 1.f);
  } else {
#pragma unroll
    for (int half = 0; half < 2; ++half) {
#pragma unroll
      for (int mb = 8 * half; mb < 8 * half + 8; ++mb) {
        const int mo = 128 * (mb - 8 * half);
        f32x16_t v = acc[mb];
        asm volatile("" : "+v"(v));
#pragma unroll
        for (int qd = 0; qd < 4; ++qd) {
          u32x4_t o;
#pragma unroll
          for (int e = 0; e < 4; ++e) o[e] = __float_as_uint(v[4 * qd + e]);
          lds_w128(eli * EPI_STRIDE + mo + 64 * eg + 16 * qd, o);
        }
        SB();
      }
      rows_out(ws_o + ((size_t)slot * H + 32 * ew) * DV + 256 * half, DV);
    }
    if (eg == 0 && ehv)
      reinterpret_cast<float4*>(ws_ml)[(size_t)slot * H + eh] = make_float4(m_run, l_w, l_e, 0.f);
  }
  return false;
}

// One workgroup per work unit, behind the resolver stage; see attend_kernel (the same
// arguments; no scales and no resolution).
template <int DQK, int QT, bool STREAM>
__global__ __launch_bounds__(NW_NT, 1) void attend_narrow_kernel(
    SasFwdArgs a, const uint16_t* __restrict__ q, const uint64_t* __restrict__ addr_list,
    const float*, const int2* __restrict__ tokr, const float* __restrict__ sinks,
    const int* __restrict__ plan, uint16_t* __restrict__ out, float* __restrict__ lse,
    float* __restrict__ ws_o, float* __restrict__ ws_ml, SasResolveArgs) {
  __shared__ __attribute__((aligned(16))) NarrowLds<DQK> sm;
  const int u = blockIdx.x;
  sm.stamps = a.stamps;
  sm.t0 = __builtin_amdgcn_s_memrealtime();
  // The unit's record with the plan's header, before the header says whether the plan and
  // the unit are sound: one memory round trip for both, of the unit's three.  (plan is the
  // workspace's, which holds the grid's unit capacity; see resolve_kernel.)
  const int units = plan[PH_UNITS];
  const int* up = plan + SAS_PLAN_HDR + (size_t)SAS_TOK_W * a.T + (size_t)u * SAS_UNIT_W;
  int4 ur = make_int4(up[0], up[1], up[2], up[3]);
  const bool plan_ok = plan_matches(plan, a);
  asm volatile("" : "+s"(ur.x), "+s"(ur.y), "+s"(ur.z), "+s"(ur.w));
  if (!plan_ok) {  // a plan built for other arguments: zeros
    if (u < a.T) {
      for (int i = threadIdx.x; i < a.H * 512 / 8; i += NW_NT)
        reinterpret_cast<u32x4_t*>(out + (size_t)u * a.H * 512)[i] = u32x4_t{0, 0, 0, 0};
      if (lse)
        for (int i = threadIdx.x; i < a.H; i += NW_NT) lse[(size_t)u * a.H + i] = 0.f;
    }
    return;
  }
  if (u >= units) return;
  float m_obs = 0.f;
  if (narrow_unit<DQK, QT, STREAM, false>(ur, sm, a, q, addr_list, tokr, sinks, plan, out, lse, ws_o,
                                          ws_ml, m_obs)) {
    lds_barrier();  // every wave is done with the ring before the redo refills it
    narrow_unit<DQK, QT, STREAM, true>(ur, sm, a, q, addr_list, tokr, sinks, plan, out, lse, ws_o, ws_ml,
                                       m_obs);
  }
  uint64_t* stamps = sm.stamps;
  if (stamps) {
    __syncthreads();
    typedef __attribute__((address_space(1))) unsigned long long g_u64;
    if (threadIdx.x == 0) {
      __hip_atomic_fetch_min((g_u64*)(uintptr_t)stamps, (unsigned long long)sm.t0,
                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_fetch_max((g_u64*)(uintptr_t)(stamps + 1),
                             (unsigned long long)__builtin_amdgcn_s_memrealtime(), __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
    }
  }
}

}  // namespace sas
