// sas_attend.hip -- pipelined gfx950 attention kernel for bf16 / fp16 and fp8 e4m3 KV.
//
// One workgroup (4 waves, one per SIMD) processes one work unit of the split-KV
// plan: a contiguous range of one query token's row list (its window rows, then
// its compressed rows).  Wave w owns query heads [32 w, 32 w + 32); Q stays in
// VGPRs (36 x 16-B fragments at d_qk = 576) and the fp32 O^T accumulator of
// 512 x 32 fills the AGPRs.  KV rows are gathered 32 at a time (one tile) by
// buffer loads that write LDS directly, into a 4-slot ring.
//
// Iteration i, per wave (32 keys x 32 heads per tile):
//   wait for tile i+1, workgroup barrier
//   S^T(i+1) = K Q^T   36 MFMA 32x32x16 into a VGPR accumulator, A = K rows from
//                      LDS (ds_read_b128, QK_RING in flight), B = Q; the softmax of tile i
//                      and the DMA of tile i+3 (into tile i-1's slot) are issued
//                      between these MFMAs, so the VALU and DMA work overlaps the
//                      matrix core
//   softmax(i)         P = 2^(x - m) in a per-unit frame m, bf16(P)
//   O^T += V^T P^T     32 MFMA into the AGPRs, A = V^T read transposed from LDS
//                      (ds_read_b64_tr_b16, three ahead), B = P^T; one inline-assembly
//                      block that also carries the scalar load of tile i+4's row
//                      addresses
// Tiles i (V), i+1 (K) and i+3 (landing) sit in distinct slots; tiles i+2 and i+3
// are in flight while tile i+1 is computed.
//
// Row addresses: the resolve kernel turns each row code into a 64-bit pool
// address (the shared zero row for -1).  Each wave gathers 8 rows per tile
// through raw buffer resources based at those addresses, so the addresses are
// wave-uniform (SGPRs) and nothing in the loop divides or indexes page tables.
// Every DMA is a buffer load, never the FLAT form: an outstanding FLAT load that
// writes LDS makes the compiler drain every later LDS wait to zero.
//
// Softmax (reference golden.py:156-200): the state of a head is (m, l, O) seeded
// with (sink, 1, 0) on the unit that holds the token's first rows.  O / l and
// m + ln l do not depend on the frame m, so the kernel fixes m after the first
// tile and never rescales the AGPR-resident O inside the loop (a VALU pass over
// 256 accumulators would cost as much as a tile of MFMA work and, worse, makes
// the compiler keep O in VGPRs).  Two normalisers are kept: l_w sums the
// bf16-rounded P that enter PV, so O / l_w is exactly a convex combination of
// the V rows (a one-hot softmax returns its row unchanged, as the reference's
// P = 1 does); l_e sums the unrounded P and gives the LSE.  A logit more than
// redo_slack() above the frame (64 for bf16 queries, 15 for fp16, whose largest
// finite value is below 2^16; with fp8 KV and fp16 queries also a rounded P s
// above 2^15) makes the workgroup discard the pass and recompute the unit framed
// on the maximum each head observed (a second, separately inlined copy of the
// unit body, so the common path carries no extra live state).
//
// LDS tile = latent region (32 rows x 512 dims at a 1088-B row stride, i.e. 64 B
// of padding per row) + rope region (32 rows x 64 dims, 128-B rows; absent at
// d_qk = 512).  Latent 16-B chunk c of row r lives at chunk c ^ ((r >> 2) & 3);
// the padding puts rows r .. r+3 in different quarters of the 256-B bank line,
// the XOR separates rows 4 apart.  Rope chunk c of row r lives at c ^ ((r >> 1) & 7).
// With these, the b128 K reads (16 consecutive rows, one chunk) and the b64
// transposed V reads (4 rows x 4 chunks per 16 lanes) touch every bank once per
// 256 B, and the per-lane read offsets reduce to two registers plus immediates.
// A latent DMA instruction copies one whole row (64 lanes x 16 B), so its source
// is a wave-uniform row base plus a per-lane offset.
//
// fp8 e4m3 KV (KV8; each row 576 B of codes plus an fp32 scale): the tile holds the
// codes and every MFMA operand is converted in registers (v_cvt_scalef32_pk_bf16_fp8,
// exact: every e4m3 value is a bf16 / fp16 value).  Row r sits at 1056 r; its 16-B
// chunk c at c ^ (9 ((r >> 3) & 1)).  One DMA instruction per row (64 lanes x 16 B:
// lanes past the 36 chunks read out of range and write zeros into the row's
// padding).  K fragments come from ds_read_b128 (two k-steps each; the Q fragments
// follow the same dimension order); V^T fragments from ds_read_b64_tr_b8, whose
// lane i of each 16-lane block receives byte i & 7 of lanes 2 p + (i >> 3), p = 0..7:
// 8 keys of one dimension, one MFMA operand after four conversions.  With this
// layout the b128 K reads (16 rows, one chunk) and the transposed V reads (8 rows x
// 32 B per 32 lanes) touch every bank once per 256 B.  The scale multiplies S
// (x = S c s) and is folded into P before its rounding (O = sum bf16(P s) V8, the
// reference's dequantised V = V8 s).  The output normaliser sums the weights that
// entered PV, bf16(P s) / s, so that O / l_w stays a convex combination of the rows
// s V8 (a one-hot softmax returns s V8 exactly); l_e sums the unrounded P (LSE).
#include <hip/hip_runtime.h>

#include "sas_common.h"

namespace sas {

// How far (log2 units) a logit may rise above the unit's frame before the unit is
// redone in a frame set on the observed maximum: P = 2^(x - m) enters PV rounded
// to the query dtype, so 2^SLACK must stay finite there (bf16: 2^64, far inside its
// range, with 2^64 times the row count far inside fp32's; fp16: 2^15 <= 65504).
template <int QT>
constexpr float redo_slack() { return QT == 0 ? 64.f : 15.f; }

// K fragments in flight ahead of the QK chain's MFMAs (16-bit KV): each b128 read is
// issued QK_RING - 1 MFMAs (32 cycles each) before its use.  Four measured 0.4% faster
// than three on prefill (interleaved, three rounds), five no better than three.
constexpr int QK_RING = 4;

typedef __attribute__((address_space(3))) uint8_t lds_u8;
typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

// Workgroup barrier without the memory fences of __syncthreads(): those wait for
// every outstanding global load (vmcnt(0)), which would drain the DMA prefetch.
// LDS writes of this wave are completed first (lgkmcnt(0)); DMA landings are
// waited for explicitly with vmcnt before the barrier where needed.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

__device__ __forceinline__ u32x4_t lds_read_b128(const lds_u8* p) {
  return *reinterpret_cast<const __attribute__((address_space(3))) u32x4_t*>(p);
}

// Swizzle of the latent region: chunk c of row r sits at c ^ swz_a(r).
__device__ __forceinline__ int swz_a(int r) { return (r >> 2) & 3; }
// Swizzle of the rope region.
__device__ __forceinline__ int swz_b(int r) { return (r >> 1) & 7; }

// fp8 tiles: 32 rows at a 1056-B stride, then one 512-B scale block per wave: its 8
// rows' scales s (then zeros) and, 256 B on, their 1 / s.
constexpr int KV8_STRIDE = 1056;
constexpr int KV8_SCALES = SAS_TILE * KV8_STRIDE;

// Epilogue staging: each wave's 32 output rows (1 KB each: 512 16-bit values, or half a
// row of fp32 partials) at a 1040-B stride, which spreads the rows' 16-B writes over
// the banks.
constexpr int EPI_STRIDE = 1040;
constexpr int EPI_WAVE = 32 * EPI_STRIDE;

template <int DQK, bool KV8>
struct AttendLds {
  static constexpr int TILEB =
      KV8 ? KV8_SCALES + 4 * 512 : SAS_TILE * (1024 + 64) + SAS_TILE * (DQK - 512) * 2;
  uint8_t tiles[4 * TILEB];
  int far;  // a logit of some head outgrew the frame
  // the dispatch's stamp buffer (nullptr: none) and the workgroup's start on the
  // real-time counter, parked here for the workgroup's end: values kept in
  // registers across the tile loop would crowd it
  uint64_t* stamps;
  uint64_t t0;
};

// Two e4m3 codes (the low or the high half of a dword) -> two 16-bit values of the
// query dtype, exactly.
template <int QT, bool HI>
__device__ __forceinline__ uint32_t fp8x2_to_q16(uint32_t v) {
  if constexpr (QT == 0)
    return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(v, 1.0f, HI));
  else
    return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(v, 1.0f, HI));
}

// d = a b^T + 0 / d += a b^T in VGPRs (the O accumulator owns the AGPRs).  Written as
// inline assembly so the S accumulator is a VGPR tuple; the chain's only hazard, a
// VALU read of d, is covered by vgpr_mfma_drain.
// CVT: the A operand was just written by VALU conversions, which an MFMA may read
// only two wait states later (s_nop 1).
template <int QT, bool CVT = false>
__device__ __forceinline__ void vmfma_first(f32x16_t& d, const u32x4_t& a, const u32x4_t& b) {
  if constexpr (CVT && QT == 0)
    asm volatile("s_nop 1\n\tv_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(d) : "v"(a), "v"(b));
  else if constexpr (CVT)
    asm volatile("s_nop 1\n\tv_mfma_f32_32x32x16_f16 %0, %1, %2, 0" : "=&v"(d) : "v"(a), "v"(b));
  else if constexpr (QT == 0)
    asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(d) : "v"(a), "v"(b));
  else
    asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, %2, 0" : "=&v"(d) : "v"(a), "v"(b));
}
template <int QT, bool CVT = false>
__device__ __forceinline__ void vmfma_acc(f32x16_t& d, const u32x4_t& a, const u32x4_t& b) {
  if constexpr (CVT && QT == 0)
    asm volatile("s_nop 1\n\tv_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(d) : "v"(a), "v"(b));
  else if constexpr (CVT)
    asm volatile("s_nop 1\n\tv_mfma_f32_32x32x16_f16 %0, %1, %2, %0" : "+v"(d) : "v"(a), "v"(b));
  else if constexpr (QT == 0)
    asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(d) : "v"(a), "v"(b));
  else
    asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, %2, %0" : "+v"(d) : "v"(a), "v"(b));
}
// An 8-pass XDL result read by a VALU needs NumPasses + 4 wait states on gfx950;
// 24 covers it with margin.
__device__ __forceinline__ void vgpr_mfma_drain(f32x16_t& d) {
  asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7" : "+v"(d));
}

// d = a b^T + 0 / d += a b^T on 32 x 32 x 64 e4m3 operands (8 VGPRs each): lane l
// holds row / column l % 32 and k = 32 (l >> 5) .. + 31, one code per byte.  A
// 16-pass XDL op: its result needs 20 wait states before a VALU read.
typedef int i32x8_t __attribute__((ext_vector_type(8)));
__device__ __forceinline__ void vmfma8_first(f32x16_t& d, const i32x8_t& a, const i32x8_t& b) {
  asm volatile("v_mfma_f32_32x32x64_f8f6f4 %0, %1, %2, 0" : "=&v"(d) : "v"(a), "v"(b));
}
__device__ __forceinline__ void vmfma8_acc(f32x16_t& d, const i32x8_t& a, const i32x8_t& b) {
  asm volatile("v_mfma_f32_32x32x64_f8f6f4 %0, %1, %2, %0" : "+v"(d) : "v"(a), "v"(b));
}

#define SB() __builtin_amdgcn_sched_barrier(0)

// s_waitcnt immediates (gfx9 encoding: vmcnt[3:0] | expcnt[6:4] | lgkmcnt[11:8] |
// vmcnt[5:4] << 14).  Issued through the builtin so the compiler's own wait
// insertion knows these counters are drained.
constexpr int waitcnt_imm(int vm, int lgkm) {
  return (vm & 15) | (7 << 4) | ((lgkm & 15) << 8) | (((vm >> 4) & 3) << 14);
}
__device__ __forceinline__ void wait_barrier() {
  __builtin_amdgcn_s_waitcnt(waitcnt_imm(63, 0));
  __builtin_amdgcn_s_barrier();
}

// One work unit u.  Returns true (workgroup-uniform) when the first pass must be
// redone; m_obs then holds each lane's observed maximum (log2 units), which the
// REDO instance takes as its frame.
// Cache policy of the gather DMA: STREAM (non-temporal loads) when every row is
// read by one token (decode: the rows would only displace reused lines from L2 and
// MALL), the default when nearby tokens re-read the same rows (prefill).
template <bool STREAM>
constexpr int gather_cpol() { return STREAM ? 2 : 0; }  // 2: the NT bit of the buffer load

// The token's row counts come from `live` when the unit resolved its own rows
// (fused), else from the resolver's per-token record tokr[t]; own_hi bounds the list
// positions the unit may read before its token record is known (its own resolved
// range when fused: other units of the token write theirs concurrently).
template <int DQK, int QT, bool STREAM, bool KV8, bool REDO>
__device__ __forceinline__ bool attend_unit(
    int u, AttendLds<DQK, KV8>& sm, const SasFwdArgs& a, const uint16_t* __restrict__ q,
    const uint64_t* addr_list, const float* scale_list, const int2* tokr, bool fused, int2 live,
    int own_hi, const float* __restrict__ sinks, const int* __restrict__ plan,
    uint16_t* __restrict__ out, float* __restrict__ lse, float* __restrict__ ws_o,
    float* __restrict__ ws_ml, float& m_obs) {
  constexpr int DV = 512;
  constexpr int NT = 256;
  constexpr int TILE = SAS_TILE;          // 32 keys
  constexpr int NSTAGE = 4;
  constexpr bool ROPE = DQK > DV;         // d_qk = 576: 64 rope dims after the latent 512
  static_assert(DQK == DV || DQK == DV + 64, "d_qk must be 512 or 576");
  constexpr int ROWA = DV * 2;            // latent bytes per row (1024)
  constexpr int STRA = ROWA + 64;         // latent LDS row stride
  constexpr int ROWR = (DQK - DV) * 2;    // rope bytes per row (128 or 0)
  constexpr int TILEA = TILE * STRA;
  constexpr int TILEB = KV8 ? KV8_SCALES + 4 * 512 : TILEA + TILE * ROWR;
  constexpr int KSTEPS = DQK / 16;        // MFMA k-steps of Q K^T: 36 / 32
  // DMA instructions per wave per tile: 8 latent rows (+ 8 rope rows), or 8 fp8
  // rows and their scales and inverse scales
  constexpr int CPT = KV8 ? 10 : 8 + (ROPE ? 8 : 0);
  static_assert(TILE == 32, "the MFMA tiling assumes 32-key tiles");
  // fp8 KV with bf16 queries: QK on the fp8 MFMA, 64 dimensions per op
  constexpr bool F8Q = KV8 && QT == 0;
  constexpr int QM = DQK / 64;  // fp8 ops per QK chain: 9 / 8
  static_assert(AttendLds<DQK, KV8>::TILEB == TILEB, "LDS layout");
  static_assert(4 * EPI_WAVE <= 4 * TILEB, "the epilogue staging fits the ring");
  lds_u8* const tiles = (lds_u8*)sm.tiles;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = tid >> 6;
  const int g = lane >> 5;   // half-wave
  const int li = lane & 31;  // MFMA column (head) / row index

  const int* ur = plan + SAS_PLAN_HDR + (size_t)SAS_TOK_W * a.T + (size_t)u * SAS_UNIT_W;
  const int t = ur[0], split = ur[3];
  const int H = a.H;

  // zeros for every head of the token, as the reference's padded slots
  auto zero_token = [&]() {
    for (int i = tid; i < H * DV / 8; i += NT)
      reinterpret_cast<u32x4_t*>(out + (size_t)t * H * DV)[i] = u32x4_t{0, 0, 0, 0};
    if (lse)
      for (int i = tid; i < H; i += NT) lse[(size_t)t * H + i] = 0.f;
  };
  if (split < 0) {  // a q row no batch owns
    zero_token();
    return false;
  }

  const int r0 = ur[1];
  // Head indices past H are clamped onto a valid head and never stored.
  const int h = w * 32 + li;
  const bool hvalid = h < H;
  const int hc = min(h, H - 1);
  // the head's sink, read by every unit (first, so that the wait for it is not a wait
  // for the loads below: vector loads complete in order)
  const float sink_raw = sinks[hc];

  // The first three tiles' row addresses of this wave (lane 8 i + k: tile i, row
  // 8 w + k) in one vector load, issued with the query's loads before the token record
  // is read: one memory round trip for the unit's start, where a scalar load per tile
  // chains three.  Rows past the unit's end become the zero row once the end is known.
  // The load itself stays inside the unit's own rows [r0, own_hi) (clamped), so it
  // never touches lines another unit writes when the units resolve their own rows.
  // (Lanes 24 .. 63 load tile 3's rows and repeats, unused: no divergent branch, which
  // would move the list pointer to VGPRs.)
  const int pro_row = r0 + ((lane >> 3) & 3) * TILE + 8 * w + (lane & 7);
  const int pro_ld = min(max(min(pro_row, own_hi - 1), r0), a.list_stride - 1);
  // (a global load: through a generic pointer it would be a FLAT load, which every
  // later wait on vector or LDS counters has to drain)
  typedef __attribute__((address_space(1))) const uint64_t g_u64;
  uint64_t pro_addr = ((g_u64*)(uintptr_t)addr_list)[(size_t)t * a.list_stride + pro_ld];
  // The fence keeps this load ahead of the query's (vector loads complete in order:
  // the DMAs then wait for the addresses only, not for the query too).
  asm volatile("" ::: "memory");
  u32x4_t qf[F8Q ? 1 : KSTEPS];
  u32x4_t qraw[F8Q ? 4 * QM : 1];  // F8Q: op m, lane half g: dimensions 64 m + 32 g + 8 j .. + 7
  {
    const u32x4_t* qrow = reinterpret_cast<const u32x4_t*>(q + ((size_t)t * H + hc) * DQK);
    if constexpr (F8Q) {
#pragma unroll
      for (int m = 0; m < QM; ++m)
#pragma unroll
        for (int j = 0; j < 4; ++j) qraw[4 * m + j] = qrow[8 * m + 4 * g + j];
    } else {
      // fp8 (fp16 queries): k-step 2 j + h covers dimensions 32 j + 16 g + 8 h .. + 7
      // (the K order)
#pragma unroll
      for (int ks = 0; ks < KSTEPS; ++ks)
        qf[ks] = KV8 ? qrow[4 * (ks >> 1) + 2 * g + (ks & 1)] : qrow[2 * ks + g];
    }
  }

  const int* tk = plan + SAS_PLAN_HDR + (size_t)t * SAS_TOK_W;
  const int splits = tk[TK_SPLITS], wsbase = tk[TK_WSBASE];
  // the token's row counts at the call's lengths: read here, with the token record
  // (one round trip for both), unless the unit resolved its rows itself
  const int2 tr = fused ? live : tokr[t];
  if (tr.x < 0) {  // a token refused for a plan that no longer matches it
    zero_token();
    return false;
  }
  // The token's last unit takes its rows to the list's end: the plan's ranges are at
  // the lengths it was built for, and the call's KV lengths may have grown since.
  const int rows_live = tr.x + tr.y;
  const int r1 = min(split == splits - 1 ? rows_live : min(ur[2], rows_live), a.list_stride);
  const int ntiles = r1 > r0 ? (r1 - r0 + TILE - 1) / TILE : 0;
  // row addresses of this unit's list (pool addresses; -1 codes read the zero row)
  const uint64_t* alist = addr_list + (size_t)t * a.list_stride + r0;
  // fp8: this unit's row scales; their inverses follow the whole scale list
  const float* slist = KV8 ? scale_list + (size_t)t * a.list_stride + r0 : nullptr;
  const size_t inv_off = (size_t)a.T * a.list_stride;

  // ---- per-lane LDS offsets (bytes within a tile) ----
  // K, latent k-step ks < 32: row li, chunk 2 ks + g -> kofs[ks & 1] + 64 (ks >> 1).
  // K, rope k-step 32 + j: row li, rope chunk 2 j + g -> kofs_r ^ 32 j (the row
  // offset TILEA + 128 li has clear bits 4..6, which carry the swizzled chunk).
  // fp8: K k-steps 2 j, 2 j + 1 come from one b128 read of row li, chunk 2 j + g at
  // position (2 j + g) ^ 9 b3 (b3 = (li >> 3) & 1): byte 32 (j ^ 4 b3) + 16 (g ^ b3),
  // i.e. kofs[(j >> 2) & 1] + 32 (j & ~4).
  // fp8 KV, bf16 queries (F8Q): QK runs on the fp8 MFMA, 64 dimensions per op.  Op m
  // takes row li, dimensions 64 m + 32 g .. + 31: chunks c = 4 m + 2 g + {0, 1} at
  // positions c ^ 9 b3, i.e. bytes k8o[j][h] + 64 (m & ~2) with h = (m >> 1) & 1.
  uint32_t kofs[2], kofs_r = 0, k8o[2][2];
  if constexpr (KV8) {
    const uint32_t b3 = (li >> 3) & 1;
    const uint32_t base = li * KV8_STRIDE + 16 * (g ^ b3);
    kofs[0] = base + 128 * b3;
    kofs[1] = base + 128 * (1 - b3);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      k8o[0][h] = li * KV8_STRIDE + 32 * g + 16 * b3 + 128 * (h ^ b3);
      k8o[1][h] = k8o[0][h] + 16 - 32 * b3;
    }
  } else {
    const int f = swz_a(li);
#pragma unroll
    for (int j = 0; j < 2; ++j) kofs[j] = li * STRA + 16 * ((2 * j + g) ^ f);
    kofs_r = TILEA + li * ROWR + 16 * (g ^ swz_b(li));
  }
  // V^T (A of O^T += V^T P^T).  MFMA row m of d-block mb is d = 32 mb + dmap(m) with
  // dmap(m) = 16 ((m >> 2) & 1) + 4 (m >> 3) + (m & 3), so accumulator register r of
  // lane (li, g) holds d = 32 mb + 16 g + r.  MFMA k index 8 g + e of k-step kk is key
  // 16 kk + 8 (e >> 2) + 4 g + (e & 3), matching where P^T sits in the S^T registers.
  // Lane l therefore supplies row 16 kk + 4 (l >> 5) + ((l >> 2) & 3) + 8 hf (hf = e >> 2)
  // at column 32 mb + 16 (l & 1) + 8 ((l >> 4) & 1) + 4 ((l >> 1) & 1): latent chunk
  // 4 mb + clo, clo = 2 (l & 1) + ((l >> 4) & 1), byte 8 ((l >> 1) & 1) within it.  The
  // row's swizzle only touches clo and depends on hf alone, so the offset is
  // vofs[hf] + 64 mb + 16 kk STRA.
  // fp8 (ds_read_b64_tr_b8): MFMA row m of d-block mb is d = 32 mb + m.  Lane s of
  // 16-lane block blk (p = (s & 15) >> 1, g = blk >> 1) supplies the row of the key
  // that P^T's k index 8 g + p holds, 16 kk + 8 (p >> 2) + 4 g + (p & 3), at
  // dimensions 32 mb + 16 (blk & 1) + 8 (s & 1) .. + 7: chunk 2 mb + (blk & 1) at
  // position 2 (mb ^ 4 b3) + ((blk & 1) ^ b3), b3 = p >> 2, i.e.
  // vofs[(mb >> 2) & 1] + 32 (mb & ~4) + 16 kk KV8_STRIDE.
  uint32_t vofs[2];
  if constexpr (KV8) {
    const int blk = lane >> 4, p = (lane & 15) >> 1;
    const uint32_t b3 = p >> 2;
    const int row = 8 * (p >> 2) + 4 * (blk >> 1) + (p & 3);
    const uint32_t base = row * KV8_STRIDE + 16 * ((blk & 1) ^ b3) + 8 * (lane & 1);
    vofs[0] = base + 128 * b3;
    vofs[1] = base + 128 * (1 - b3);
  } else {
    const int clo = 2 * (lane & 1) + ((lane >> 4) & 1);
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) {
      const int row = 4 * (lane >> 5) + ((lane >> 2) & 3) + 8 * hf;
      vofs[hf] = row * STRA + 16 * (clo ^ swz_a(row)) + 8 * ((lane >> 1) & 1);
    }
  }

  // ---- per-wave state: 32 heads per wave ----
  // golden.py:162-163: the unit holding the token's first rows carries the sink
  const float sink2 = split == 0 ? sink_raw * LOG2E : -INFINITY;

  // A unit without rows (a redo always has some): O = 0 and the normalisers are
  // the sink's alone.  Returning here also keeps the accumulators below on a
  // single path, so the epilogue does not have to merge them with zeros.
  if (ntiles == 0) {
    if (REDO || !hvalid) return false;  // (a redo always has rows)
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
      // lane (li, g) zeroes half of row li: 16 B per step, fp16 (fmt 1) or fp32 (fmt 0)
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

  // F8Q: the query, scaled by 2^e so that its largest |q| lies in [128, 256), as two
  // e4m3 parts hi = rne(q 2^e) and lo = rne(q 2^e - hi), op m's B operands.  A bf16
  // value has 8 significant bits and each part 4: hi + lo = q 2^e exactly for every
  // element of magnitude >= 2^-10 of the head's largest (smaller ones are off by at
  // most 2^-10 in the scaled units), so S 2^-e is the bf16 product.  ck = c 2^-e.
  i32x8_t qh[F8Q ? QM : 1], ql[F8Q ? QM : 1];
  float ck = a.scale_log2;
  // F8Q: the split, run once the first tiles' DMAs are issued (its VALU work then
  // overlaps their flight instead of delaying it)
  auto split_query = [&]() {
    if constexpr (F8Q) {
      // the head's largest |q| over both half-waves (bf16 magnitudes order as integers)
      uint32_t mx = 0;
#pragma unroll
      for (int i = 0; i < 4 * QM; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const uint32_t w = qraw[i][e] & 0x7fff7fffu;
          mx = max(mx, max(w & 0xffffu, w >> 16));
        }
      {
        const auto sw = __builtin_amdgcn_permlane32_swap(mx, mx, false, false);
        mx = max(sw[0], sw[1]);
      }
      const float qmax = __uint_as_float(mx << 16);
      // |e| <= 126 keeps 2^e and 2^-e normal floats: every finite bf16 qmax up to
      // 2^128 is placed in [128, 256); only a head whose largest |q| is below 2^-118
      // is placed lower (off by at most 2^-136 per element, far below its own size
      // times 2^-8 that bf16 rounding already allows)
      const int e = qmax > 0.f ? min(max(8 - __builtin_amdgcn_frexp_expf(qmax), -126), 126) : 0;
      const float qs = __builtin_amdgcn_ldexpf(1.f, e);
      ck = a.scale_log2 * __builtin_amdgcn_ldexpf(1.f, -e);
#pragma unroll
      for (int m = 0; m < QM; ++m)
#pragma unroll
        for (int d = 0; d < 8; ++d) {  // codes 4 d .. 4 d + 3 of op m
          const uint32_t w0 = qraw[4 * m + (d >> 1)][2 * (d & 1)];
          const uint32_t w1 = qraw[4 * m + (d >> 1)][2 * (d & 1) + 1];
          const float a0 = __uint_as_float(w0 << 16) * qs, a1 = __uint_as_float(w0 & 0xffff0000u) * qs;
          const float a2 = __uint_as_float(w1 << 16) * qs, a3 = __uint_as_float(w1 & 0xffff0000u) * qs;
          int hw = __builtin_amdgcn_cvt_pk_fp8_f32(a0, a1, 0, false);
          hw = __builtin_amdgcn_cvt_pk_fp8_f32(a2, a3, hw, true);
          const auto h01 = __builtin_amdgcn_cvt_pk_f32_fp8(hw, false);
          const auto h23 = __builtin_amdgcn_cvt_pk_f32_fp8(hw, true);
          int lw = __builtin_amdgcn_cvt_pk_fp8_f32(a0 - h01[0], a1 - h01[1], 0, false);
          lw = __builtin_amdgcn_cvt_pk_fp8_f32(a2 - h23[0], a3 - h23[1], lw, true);
          qh[m][d] = hw;
          ql[m][d] = lw;
        }
    }
  };
  f32x16_t acc[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i] = f32x16_t{};
  float m_run = REDO ? m_obs : sink2;  // redo: the frame is the maximum pass 1 observed

  // ---- gather: tile i goes to ring slot i & 3 ----
  // Wave w copies rows 8 w .. 8 w + 7 of every tile.  Latent: instruction k copies
  // row 8 w + k, lane l fetching source chunk l ^ swz_a(8 w + k) =
  // l ^ ((2 w + (k >> 2)) & 3) into slot l.  Row addresses reach SGPRs by scalar
  // loads an iteration before their DMA (tiles 0 .. 2: by lane reads of the
  // prologue's vector load).
  const int wu = __builtin_amdgcn_readfirstlane(w);  // the wave index as a scalar
  const uint32_t ulane = (uint32_t)lane;
  // fp8: every row of wave w has bit 3 of its tile row equal to w & 1, so lane l
  // fetches chunk l ^ 9 (w & 1) of each of its rows (chunks past the row: zeros).
  const uint32_t voffA0 = KV8 ? 16u * (ulane ^ (9u * (uint32_t)(wu & 1)))
                              : 16u * (ulane ^ (uint32_t)((2 * wu) & 3));
  const uint32_t voffA1 = 16u * (ulane ^ (uint32_t)((2 * wu + 1) & 3));
  // rope DMA of row 8 w + k: lane l fetches chunk l ^ ((4 w + (k >> 1)) & 7)
  const uint32_t voffR0 = 16u * (ulane & 7u);
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
    // through the constant address space: a scalar load, whatever stores the kernel
    // made before (its DMA waits count vector-memory instructions)
    typedef __attribute__((address_space(4))) const RowAddrs c_RowAddrs;
    return fix_tail(*(c_RowAddrs*)(uintptr_t)(alist + il * TILE + 8 * wu), i);
  };
  // Tile i < 3's row addresses, read out of the lanes of the prologue's vector load
  // (rows past r1, dead tiles' included, already hold the zero row).  Tile 3's come
  // by a scalar load: they stay live into the loop, where SGPRs filled from lanes
  // push the fp8 variants' registers over the limit.
  if (pro_row >= r1) pro_addr = (uint64_t)g_zero_row;
  auto pro_addrs = [&](int i) -> RowAddrs {
    RowAddrs ra;
#pragma unroll
    for (int k = 0; k < 8; ++k)
      ra[k] = ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(pro_addr >> 32), 8 * i + k) << 32) |
              (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)pro_addr, 8 * i + k);
    return ra;
  };
  // One row through a raw buffer resource based at the row (loads directly into
  // LDS, never the FLAT form: an outstanding FLAT load that writes LDS makes every
  // later LDS wait a full drain).
  auto row_rsrc = [&](uint64_t addr) {
    return __builtin_amdgcn_make_buffer_rsrc((void*)addr, (short)0, KV8 ? DQK : ROWA + ROWR,
                                             0x00020000);
  };
  // 16-bit KV: the latent 1024 B of row 8 w + k; fp8: the whole row
  auto dma_lat = [&](int i, const RowAddrs& ra, int k) {
    lds_u8* dst = tiles + (i & (NSTAGE - 1)) * TILEB + (8 * wu + k) * (KV8 ? KV8_STRIDE : STRA);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(row_rsrc(ra[k]), (void __attribute__((address_space(3)))*)dst, 16,
                                             KV8 || k < 4 ? voffA0 : voffA1, 0, 0, gather_cpol<STREAM>());
  };
  // fp8: the scales of this wave's 8 rows of tile i into its block, then their
  // inverses 256 B on (lane l writes float l; rows past the unit's end, and lanes
  // 8 .. 63, read as zeros)
  auto dma_scale = [&](int i) {
    // (readfirstlane: a clamp selects v_med3, and a buffer resource in VGPRs would
    // be issued lane by lane)
    const int n = __builtin_amdgcn_readfirstlane(max(0, min(8, r1 - (r0 + i * TILE + 8 * wu))));
    lds_u8* dst = tiles + (i & (NSTAGE - 1)) * TILEB + KV8_SCALES + 512 * wu;
    const float* src = slist + i * TILE + 8 * wu;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        __builtin_amdgcn_make_buffer_rsrc((void*)src, (short)0, 4 * n, 0x00020000),
        (void __attribute__((address_space(3)))*)dst, 4, 4u * ulane, 0, 0, gather_cpol<STREAM>());
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        __builtin_amdgcn_make_buffer_rsrc((void*)(src + inv_off), (short)0, 4 * n, 0x00020000),
        (void __attribute__((address_space(3)))*)(dst + 256), 4, 4u * ulane, 0, 0,
        gather_cpol<STREAM>());
  };
  // Rope: lanes 0..7 copy the 128-B rope of one row per instruction, chunk
  // l ^ swz_b(8 w + k) = l ^ ((4 w + (k >> 1)) & 7) into slot l.  It runs after every
  // other use of the row addresses in its block: a uniform value used on both
  // sides of the divergent lane < 8 branch can end up in VGPRs.
  auto dma_rope = [&](int i, const RowAddrs& ra) {
    if constexpr (ROPE) {
      lds_u8* dst = tiles + (i & (NSTAGE - 1)) * TILEB + TILEA + 8 * wu * ROWR;
      if (lane < 8) {
        // formed here rather than kept across the loop: registers are the limit
        uint32_t vb = voffR0;
        asm volatile("" : "+v"(vb));
#pragma unroll
        for (int k = 0; k < 8; ++k)
          __builtin_amdgcn_raw_ptr_buffer_load_lds(
              row_rsrc(ra[k]), (void __attribute__((address_space(3)))*)(dst + k * ROWR), 16,
              ROWA + (vb ^ (16u * (uint32_t)((4 * wu + (k >> 1)) & 7))), 0, 0, gather_cpol<STREAM>());
      }
    }
  };

  // ---- S^T = K Q^T: the chain of KSTEPS accumulating MFMAs, K fragments QK_RING - 1 ahead ----
  // work(ks) runs right after step ks's MFMA issues (ks = -1: before the first one,
  // while the first K fragments are in flight; ks = KSTEPS: after the last one).
  // The loop hangs the previous tile's softmax and a later tile's DMA on it, so that
  // VALU, SALU and DMA issue overlap the matrix core instead of following it.
  auto kread = [&](const lds_u8* tl, int ks, uint32_t kr) -> u32x4_t {
    return ks < 32 ? lds_read_b128(tl + kofs[ks & 1] + 64 * (ks >> 1))
                   : lds_read_b128(tl + (kr ^ (32u * (uint32_t)(ks - 32))));
  };
  // fp8: b128 read j holds k-steps 2 j (dwords 0, 1) and 2 j + 1 (dwords 2, 3)
  auto kpair8 = [&](const lds_u8* tl, int j) -> u32x4_t {
    return lds_read_b128(tl + kofs[(j >> 2) & 1] + 32 * (j & ~4));
  };
  // F8Q: K operand of op m (two b128 reads of row li)
  auto kread8 = [&](const lds_u8* tl, int m) -> i32x8_t {
    const int h = (m >> 1) & 1, off = 64 * (m & ~2);
    const u32x4_t c0 = lds_read_b128(tl + k8o[0][h] + off);
    const u32x4_t c1 = lds_read_b128(tl + k8o[1][h] + off);
    return i32x8_t{(int)c0[0], (int)c0[1], (int)c0[2], (int)c0[3],
                   (int)c1[0], (int)c1[1], (int)c1[2], (int)c1[3]};
  };
  auto qk = [&](const lds_u8* tl, f32x16_t& s, auto&& work) {
    if constexpr (F8Q) {
      // op m with hi, then with lo (the K operand read once); two work items per op,
      // whose 64 cycles match two 16-bit k-steps, so the schedule's steps are kept
      i32x8_t kr[2];
      kr[0] = kread8(tl, 0);
      SB();
      work(-1);
      SB();
#pragma unroll
      for (int m = 0; m < QM; ++m) {
        if (m == 0)
          vmfma8_first(s, kr[0], qh[0]);
        else
          vmfma8_acc(s, kr[m & 1], qh[m]);
        if (m + 1 < QM) kr[(m + 1) & 1] = kread8(tl, m + 1);
        work(4 * m);
        SB();
        work(4 * m + 1);
        SB();
        vmfma8_acc(s, kr[m & 1], ql[m]);
        work(4 * m + 2);
        SB();
        work(4 * m + 3);
        SB();
      }
      work(KSTEPS);
      SB();
      return;
    } else if constexpr (KV8) {
      u32x4_t rw[2];
      rw[0] = kpair8(tl, 0);
      rw[1] = kpair8(tl, 1);
      SB();
      work(-1);
      SB();
#pragma unroll
      for (int ks = 0; ks < KSTEPS; ++ks) {
        const int j = ks >> 1, h2 = 2 * (ks & 1);
        u32x4_t kf;
        kf[0] = fp8x2_to_q16<QT, false>(rw[j & 1][h2]);
        kf[1] = fp8x2_to_q16<QT, true>(rw[j & 1][h2]);
        kf[2] = fp8x2_to_q16<QT, false>(rw[j & 1][h2 + 1]);
        kf[3] = fp8x2_to_q16<QT, true>(rw[j & 1][h2 + 1]);
        if (ks == 0)
          vmfma_first<QT, true>(s, kf, qf[0]);
        else
          vmfma_acc<QT, true>(s, kf, qf[ks]);
        if ((ks & 1) && j + 2 < KSTEPS / 2) rw[j & 1] = kpair8(tl, j + 2);
        work(ks);
        SB();
      }
      // the steady-state fp8 softmax ends at step 32: past the last MFMA at d_qk 512
      work(KSTEPS);
      SB();
      return;
    }
    // the rope offset, formed per chain rather than kept across the loop
    uint32_t kr = kofs_r;
    asm volatile("" : "+v"(kr));
    constexpr int KR = QK_RING;
    u32x4_t kb[KR];
#pragma unroll
    for (int j = 0; j < KR; ++j) kb[j] = kread(tl, j, kr);
    SB();
    work(-1);
    SB();
    vmfma_first<QT>(s, kb[0], qf[0]);
    work(0);
    SB();
#pragma unroll
    for (int ks = 1; ks < KSTEPS; ++ks) {
      if (ks + KR - 1 < KSTEPS) kb[(ks + KR - 1) % KR] = kread(tl, ks + KR - 1, kr);
      vmfma_acc<QT>(s, kb[ks % KR], qf[ks]);
      work(ks);
      SB();
    }
  };
  // Tile i's DMA over a QK chain: one latent row every fourth step, the rope rows
  // (behind a lane < 8 branch) after the last MFMA.
  auto dma_step = [&](int ks, int i, const RowAddrs& ra) {
    if (ks >= 0 && (ks & 3) == 1 && (ks >> 2) < 8) dma_lat(i, ra, ks >> 2);
    if (ks == KSTEPS - 1) {
      if constexpr (KV8)
        dma_scale(i);
      else
        dma_rope(i, ra);
    }
  };

  // ---- O^T += V^T P^T ----
  // PV in one inline-assembly block that also carries the scalar load of a later
  // tile's row addresses: its latency hides under the 32 MFMAs, and the block's
  // own LDS waits count only the V^T reads (a scalar load in flight can only make
  // them stricter), so the loaded SGPRs are valid when the block ends.
  // V^T operand ring: three 4-VGPR buffers v[244:255] (clobbered), reads 3 MFMAs ahead.
  // The MFMAs run accumulator-outer: all 16 d-blocks of key half 0, then of half 1.
  auto pv_asm = [&](const lds_u8* tl, const u32x4_t(&pk)[2], const uint64_t* aptr) -> RowAddrs {
    const uint32_t a0 = (uint32_t)(uintptr_t)tl + vofs[0];
    const uint32_t a1 = (uint32_t)(uintptr_t)tl + vofs[1];
    typedef uint32_t u32x16_t __attribute__((ext_vector_type(16)));
    u32x16_t sa;
    if constexpr (KV8) {
      // fp8: V^T fragments by ds_read_b64_tr_b8 into a three-deep ring v[250:255],
      // three MFMAs ahead; four conversions into v[242:245] / v[246:249] each, two
      // wait states (s_nop 1, after the next read) before the MFMA reads them.
#define PV8_ASM(MN, CVT) \
    asm volatile( \
        "s_load_dwordx16 %[sa], %[ap], 0x0\n\t" \
        "ds_read_b64_tr_b8 v[250:251], %[a0] offset:0\n\t" "ds_read_b64_tr_b8 v[252:253], %[a0] offset:32\n\t" "ds_read_b64_tr_b8 v[254:255], %[a0] offset:64\n\t" \
        "s_waitcnt lgkmcnt(2)\n\t" CVT " v242, v250, 1.0\n\t" CVT " v243, v250, 1.0 op_sel:[1,0,0]\n\t" CVT " v244, v251, 1.0\n\t" CVT " v245, v251, 1.0 op_sel:[1,0,0]\n\t" "ds_read_b64_tr_b8 v[250:251], %[a0] offset:96\n\t" "s_nop 1\n\t" MN " %[c0], v[242:245], %[p0], %[c0]\n\t" \
        "s_waitcnt lgkmcnt(2)\n\t" CVT " v246, v252, 1.0\n\t" CVT " v247, v252, 1.0 op_sel:[1,0,0]\n\t" CVT " v248, v253, 1.0\n\t" CVT " v249, v253, 1.0 op_sel:[1,0,0]\n\t" "ds_read_b64_tr_b8 v[252:253], %[a1] offset:0\n\t" "s_nop 1\n\t" MN " %[c1], v[246:249], %[p0], %[c1]\n\t" \
        "s_waitcnt lgkmcnt(2)\n\t" CVT " v242, v254, 1.0\n\t" CVT " v243, v254, 1.0 op_sel:[1,0,0]\n\t" CVT " v244, v255, 1.0\n\t" CVT " v245, v255, 1.0 op_sel:[1,0,0]\n\t" "ds_read_b64_tr_b8 v[254:255], %[a1] offset:32\n\t" "s_nop 1\n\t" MN " %[c2], v[242:245], %[p0], %[c2]\n\t" \
        "s_waitcnt lgkmcnt(2)\n\t" CVT " v246, v250, 1.0\n\t" CVT " v247, v250, 1.0 op_sel:[1,0,0]\n\t" CVT " v248, v251, 1.0\n\t" CVT " v249, v251, 1.0 op_sel:[1,0,0]\n\t" "ds_read_b64_tr_b8 v[250:251], %[a1] offset:64\n\t" "s_nop 1\n\t" MN " %[c3], v[246:249], %[p0], %[c3]\n\t" \
        "s_waitcnt lgkmcnt(2)\n\t" CVT " v242, v252, 1.0\n\t" CVT " v243, v252, 1.0 op_sel:[1,0,0]\n\t" CVT " v244, v253, 1.0\n\t" CVT " v245, v253, 1.0 op_sel:[1,0,0]\n\t" "ds_read_b64_tr_b8 v[252:253], %[a1] offset:96\n\t" "s_nop 1\n\t" MN " %[c4], v[242:245], %[p0], %[c4]\n\t" \
        "s_waitcnt lgkmcnt(2)\n\t" CVT " v246, v254, 1.0\n\t" CVT " v247, v254, 1.0 op_sel:[1,0,0]\n\t" CVT " v248, v255, 1.0\n\t" CVT " v249, v255, 1.0 op_sel:[1,0,0]\n\t" "ds_read_b64_tr_b8 v[254:255], %[a0] offset:256\n\t" "s_nop 1\n\t" MN " %[c5], v[246:249], %[p0], %[c5]\n\t" \
        "s_waitcnt lgkmcnt(2)\n\t" CVT " v242, v250, 1.0\n\t" CVT " v243, v250, 1.0 op_sel:[1,0,0]\n\t" CVT " v244, v251, 1.0\n\t" CVT " v245, v251, 1.0 op_sel:[1,0,0]\n\t" "ds_read_b64_tr_b8 v[250:251], %[a0] offset:288\n\t" "s_nop 1\n\t" MN " %[c6], v[242:245], %[p0], %[c6]\n\t" \
        "s_waitcnt lgkmcnt(2)\n\t" CVT " v246, v252, 1.0\n\t" CVT " v247, v252, 1.0 op_sel:[1,0,0]\n\t" CVT " v248, v253, 1.0\n\t" CVT " v249, v253, 1.0 op_sel:[1,0,0]\n\t" "ds_read_b64_tr_b8 v[252:253], %[a0] offset:320\n\t" "s_nop 1\n\t" MN " %[c7], v[246:249], %[p0], %[c7]\n\t" \
        "s_waitcnt lgkmcnt(2)\n\t" CVT " v242, v254, 1.0\n\t" CVT " v243, v254, 1.0 op_sel:[1,0,0]\n\t" CVT " v244, v255, 1.0\n\t" CVT " v245, v255, 1.0 op_sel:[1,0,0]\n\t" "ds_read_b64_tr_b8 v[254:255], %[a0] offset:352\n\t" "s_nop 1\n\t" MN " %[c8], v[242:245], %[p0], %[c8]\n\t" \
        "s_waitcnt lgkmcnt(2)\n\t" CVT " v246, v250, 1.0\n\t" CVT " v247, v250, 1.0 op_sel:[1,0,0]\n\t" CVT " v248, v251, 1.0\n\t" CVT " v249, v251, 1.0 op_sel:[1,0,0]\n\t" "ds_read_b64_tr_b8 v[250:251], %[a1] offset:256\n\t" "s_nop 1\n\t" MN " %[c9], v[246:249], %[p0], %[c9]\n\t" \
        "s_waitcnt lgkmcnt(2)\n\t" CVT " v242, v252, 1.0\n\t" CVT " v243, v252, 1.0 op_sel:[1,0,0]\n\t" CVT " v244, v253, 1.0\n\t" CVT " v245, v253, 1.0 op_sel:[1,0,0]\n\t" "ds_read_b64_tr_b8 v[252:253], %[a1] offset:288\n\t" "s_nop 1\n\t" MN " %[c10], v[242:245], %[p0], %[c10]\n\t" \
        "s_waitcnt lgkmcnt(2)\n\t" CVT " v246, v254, 1.0\n\t" CVT " v247, v254, 1.0 op_sel:[1,0,0]\n\t" CVT " v248, v255, 1.0\n\t" CVT " v249, v255, 1.0 op_sel:[1,0,0]\n\t" "ds_read_b64_tr_b8 v[254:255], %[a1] offset:320\n\t" "s_nop 1\n\t" MN " %[c11], v[246:249], %[p0], %[c11]\n\t" \
        "s_waitcnt lgkmcnt(2)\n\t" CVT " v242, v250, 1.0\n\t" CVT " v243, v250, 1.0 op_sel:[1,0,0]\n\t" CVT " v244, v251, 1.0\n\t" CVT " v245, v251, 1.0 op_sel:[1,0,0]\n\t" "ds_read_b64_tr_b8 v[250:251], %[a1] offset:352\n\t" "s_nop 1\n\t" MN " %[c12], v[242:245], %[p0], %[c12]\n\t" \
        "s_waitcnt lgkmcnt(2)\n\t" CVT " v246, v252, 1.0\n\t" CVT " v247, v252, 1.0 op_sel:[1,0,0]\n\t" CVT " v248, v253, 1.0\n\t" CVT " v249, v253, 1.0 op_sel:[1,0,0]\n\t" "ds_read_b64_tr_b8 v[252:253], %[a0] offset:16896\n\t" "s_nop 1\n\t" MN " %[c13], v[246:249], %[p0], %[c13]\n\t" \
        "s_waitcnt lgkmcnt(2)\n\t" CVT " v242, v254, 1.0\n\t" CVT " v243, v254, 1.0 op_sel:[1,0,0]\n\t" CVT " v244, v255, 1.0\n\t" CVT " v245, v255, 1.0 op_sel:[1,0,0]\n\t" "ds_read_b64_tr_b8 v[254:255], %[a0] offset:16928\n\t" "s_nop 1\n\t" MN " %[c14], v[242:245], %[p0], %[c14]\n\t" \
        "s_waitcnt lgkmcnt(2)\n\t" CVT " v246, v250, 1.0\n\t" CVT " v247, v250, 1.0 op_sel:[1,0,0]\n\t" CVT " v248, v251, 1.0\n\t" CVT " v249, v251, 1.0 op_sel:[1,0,0]\n\t" "ds_read_b64_tr_b8 v[250:251], %[a0] offset:16960\n\t" "s_nop 1\n\t" MN " %[c15], v[246:249], %[p0], %[c15]\n\t" \
        "s_waitcnt lgkmcnt(2)\n\t" CVT " v242, v252, 1.0\n\t" CVT " v243, v252, 1.0 op_sel:[1,0,0]\n\t" CVT " v244, v253, 1.0\n\t" CVT " v245, v253, 1.0 op_sel:[1,0,0]\n\t" "ds_read_b64_tr_b8 v[252:253], %[a0] offset:16992\n\t" "s_nop 1\n\t" MN " %[c0], v[242:245], %[p1], %[c0]\n\t" \
        "s_waitcnt lgkmcnt(2)\n\t" CVT " v246, v254, 1.0\n\t" CVT " v247, v254, 1.0 op_sel:[1,0,0]\n\t" CVT " v248, v255, 1.0\n\t" CVT " v249, v255, 1.0 op_sel:[1,0,0]\n\t" "ds_read_b64_tr_b8 v[254:255], %[a1] offset:16896\n\t" "s_nop 1\n\t" MN " %[c1], v[246:249], %[p1], %[c1]\n\t" \
        "s_waitcnt lgkmcnt(2)\n\t" CVT " v242, v250, 1.0\n\t" CVT " v243, v250, 1.0 op_sel:[1,0,0]\n\t" CVT " v244, v251, 1.0\n\t" CVT " v245, v251, 1.0 op_sel:[1,0,0]\n\t" "ds_read_b64_tr_b8 v[250:251], %[a1] offset:16928\n\t" "s_nop 1\n\t" MN " %[c2], v[242:245], %[p1], %[c2]\n\t" \
        "s_waitcnt lgkmcnt(2)\n\t" CVT " v246, v252, 1.0\n\t" CVT " v247, v252, 1.0 op_sel:[1,0,0]\n\t" CVT " v248, v253, 1.0\n\t" CVT " v249, v253, 1.0 op_sel:[1,0,0]\n\t" "ds_read_b64_tr_b8 v[252:253], %[a1] offset:16960\n\t" "s_nop 1\n\t" MN " %[c3], v[246:249], %[p1], %[c3]\n\t" \
        "s_waitcnt lgkmcnt(2)\n\t" CVT " v242, v254, 1.0\n\t" CVT " v243, v254, 1.0 op_sel:[1,0,0]\n\t" CVT " v244, v255, 1.0\n\t" CVT " v245, v255, 1.0 op_sel:[1,0,0]\n\t" "ds_read_b64_tr_b8 v[254:255], %[a1] offset:16992\n\t" "s_nop 1\n\t" MN " %[c4], v[242:245], %[p1], %[c4]\n\t" \
        "s_waitcnt lgkmcnt(2)\n\t" CVT " v246, v250, 1.0\n\t" CVT " v247, v250, 1.0 op_sel:[1,0,0]\n\t" CVT " v248, v251, 1.0\n\t" CVT " v249, v251, 1.0 op_sel:[1,0,0]\n\t" "ds_read_b64_tr_b8 v[250:251], %[a0] offset:17152\n\t" "s_nop 1\n\t" MN " %[c5], v[246:249], %[p1], %[c5]\n\t" \
        "s_waitcnt lgkmcnt(2)\n\t" CVT " v242, v252, 1.0\n\t" CVT " v243, v252, 1.0 op_sel:[1,0,0]\n\t" CVT " v244, v253, 1.0\n\t" CVT " v245, v253, 1.0 op_sel:[1,0,0]\n\t" "ds_read_b64_tr_b8 v[252:253], %[a0] offset:17184\n\t" "s_nop 1\n\t" MN " %[c6], v[242:245], %[p1], %[c6]\n\t" \
        "s_waitcnt lgkmcnt(2)\n\t" CVT " v246, v254, 1.0\n\t" CVT " v247, v254, 1.0 op_sel:[1,0,0]\n\t" CVT " v248, v255, 1.0\n\t" CVT " v249, v255, 1.0 op_sel:[1,0,0]\n\t" "ds_read_b64_tr_b8 v[254:255], %[a0] offset:17216\n\t" "s_nop 1\n\t" MN " %[c7], v[246:249], %[p1], %[c7]\n\t" \
        "s_waitcnt lgkmcnt(2)\n\t" CVT " v242, v250, 1.0\n\t" CVT " v243, v250, 1.0 op_sel:[1,0,0]\n\t" CVT " v244, v251, 1.0\n\t" CVT " v245, v251, 1.0 op_sel:[1,0,0]\n\t" "ds_read_b64_tr_b8 v[250:251], %[a0] offset:17248\n\t" "s_nop 1\n\t" MN " %[c8], v[242:245], %[p1], %[c8]\n\t" \
        "s_waitcnt lgkmcnt(2)\n\t" CVT " v246, v252, 1.0\n\t" CVT " v247, v252, 1.0 op_sel:[1,0,0]\n\t" CVT " v248, v253, 1.0\n\t" CVT " v249, v253, 1.0 op_sel:[1,0,0]\n\t" "ds_read_b64_tr_b8 v[252:253], %[a1] offset:17152\n\t" "s_nop 1\n\t" MN " %[c9], v[246:249], %[p1], %[c9]\n\t" \
        "s_waitcnt lgkmcnt(2)\n\t" CVT " v242, v254, 1.0\n\t" CVT " v243, v254, 1.0 op_sel:[1,0,0]\n\t" CVT " v244, v255, 1.0\n\t" CVT " v245, v255, 1.0 op_sel:[1,0,0]\n\t" "ds_read_b64_tr_b8 v[254:255], %[a1] offset:17184\n\t" "s_nop 1\n\t" MN " %[c10], v[242:245], %[p1], %[c10]\n\t" \
        "s_waitcnt lgkmcnt(2)\n\t" CVT " v246, v250, 1.0\n\t" CVT " v247, v250, 1.0 op_sel:[1,0,0]\n\t" CVT " v248, v251, 1.0\n\t" CVT " v249, v251, 1.0 op_sel:[1,0,0]\n\t" "ds_read_b64_tr_b8 v[250:251], %[a1] offset:17216\n\t" "s_nop 1\n\t" MN " %[c11], v[246:249], %[p1], %[c11]\n\t" \
        "s_waitcnt lgkmcnt(2)\n\t" CVT " v242, v252, 1.0\n\t" CVT " v243, v252, 1.0 op_sel:[1,0,0]\n\t" CVT " v244, v253, 1.0\n\t" CVT " v245, v253, 1.0 op_sel:[1,0,0]\n\t" "ds_read_b64_tr_b8 v[252:253], %[a1] offset:17248\n\t" "s_nop 1\n\t" MN " %[c12], v[242:245], %[p1], %[c12]\n\t" \
        "s_waitcnt lgkmcnt(2)\n\t" CVT " v246, v254, 1.0\n\t" CVT " v247, v254, 1.0 op_sel:[1,0,0]\n\t" CVT " v248, v255, 1.0\n\t" CVT " v249, v255, 1.0 op_sel:[1,0,0]\n\t" "s_nop 1\n\t" MN " %[c13], v[246:249], %[p1], %[c13]\n\t" \
        "s_waitcnt lgkmcnt(1)\n\t" CVT " v242, v250, 1.0\n\t" CVT " v243, v250, 1.0 op_sel:[1,0,0]\n\t" CVT " v244, v251, 1.0\n\t" CVT " v245, v251, 1.0 op_sel:[1,0,0]\n\t" "s_nop 1\n\t" MN " %[c14], v[242:245], %[p1], %[c14]\n\t" \
        "s_waitcnt lgkmcnt(0)\n\t" CVT " v246, v252, 1.0\n\t" CVT " v247, v252, 1.0 op_sel:[1,0,0]\n\t" CVT " v248, v253, 1.0\n\t" CVT " v249, v253, 1.0 op_sel:[1,0,0]\n\t" "s_nop 1\n\t" MN " %[c15], v[246:249], %[p1], %[c15]\n\t" \
        : [sa] "=s"(sa), [c0] "+a"(acc[0]), [c1] "+a"(acc[1]), [c2] "+a"(acc[2]), [c3] "+a"(acc[3]), \
          [c4] "+a"(acc[4]), [c5] "+a"(acc[5]), [c6] "+a"(acc[6]), [c7] "+a"(acc[7]), \
          [c8] "+a"(acc[8]), [c9] "+a"(acc[9]), [c10] "+a"(acc[10]), [c11] "+a"(acc[11]), \
          [c12] "+a"(acc[12]), [c13] "+a"(acc[13]), [c14] "+a"(acc[14]), [c15] "+a"(acc[15]) \
        : [a0] "v"(a0), [a1] "v"(a1), [p0] "v"(pk[0]), [p1] "v"(pk[1]), [ap] "s"(aptr) \
        : "v242", "v243", "v244", "v245", "v246", "v247", "v248", "v249", "v250", "v251", \
          "v252", "v253", "v254", "v255", "memory");
      if constexpr (QT == 0) {
        PV8_ASM("v_mfma_f32_32x32x16_bf16", "v_cvt_scalef32_pk_bf16_fp8")
      } else {
        PV8_ASM("v_mfma_f32_32x32x16_f16", "v_cvt_scalef32_pk_f16_fp8")
      }
#undef PV8_ASM
      return __builtin_bit_cast(RowAddrs, sa);
    }
#define PV_RD(j, b) \
    "ds_read_b64_tr_b16 v[" #b ":" #b "+1], %[a0] offset:" #j "\n\t" \
    "ds_read_b64_tr_b16 v[" #b "+2:" #b "+3], %[a1] offset:" #j "\n\t"
#define PV_MM(MN, c, b, p) MN " %[c" #c "], v[" #b ":" #b "+3], %[p" #p "], %[c" #c "]\n\t"
#define PV_ASM(MN) \
    asm volatile( \
        "s_load_dwordx16 %[sa], %[ap], 0x0\n\t" \
        PV_RD(0, 244) PV_RD(64, 248) PV_RD(128, 252) \
        "s_waitcnt lgkmcnt(4)\n\t" PV_MM(MN, 0, 244, 0) PV_RD(192, 244) \
        "s_waitcnt lgkmcnt(4)\n\t" PV_MM(MN, 1, 248, 0) PV_RD(256, 248) \
        "s_waitcnt lgkmcnt(4)\n\t" PV_MM(MN, 2, 252, 0) PV_RD(320, 252) \
        "s_waitcnt lgkmcnt(4)\n\t" PV_MM(MN, 3, 244, 0) PV_RD(384, 244) \
        "s_waitcnt lgkmcnt(4)\n\t" PV_MM(MN, 4, 248, 0) PV_RD(448, 248) \
        "s_waitcnt lgkmcnt(4)\n\t" PV_MM(MN, 5, 252, 0) PV_RD(512, 252) \
        "s_waitcnt lgkmcnt(4)\n\t" PV_MM(MN, 6, 244, 0) PV_RD(576, 244) \
        "s_waitcnt lgkmcnt(4)\n\t" PV_MM(MN, 7, 248, 0) PV_RD(640, 248) \
        "s_waitcnt lgkmcnt(4)\n\t" PV_MM(MN, 8, 252, 0) PV_RD(704, 252) \
        "s_waitcnt lgkmcnt(4)\n\t" PV_MM(MN, 9, 244, 0) PV_RD(768, 244) \
        "s_waitcnt lgkmcnt(4)\n\t" PV_MM(MN, 10, 248, 0) PV_RD(832, 248) \
        "s_waitcnt lgkmcnt(4)\n\t" PV_MM(MN, 11, 252, 0) PV_RD(896, 252) \
        "s_waitcnt lgkmcnt(4)\n\t" PV_MM(MN, 12, 244, 0) PV_RD(960, 244) \
        "s_waitcnt lgkmcnt(4)\n\t" PV_MM(MN, 13, 248, 0) PV_RD(17408, 248) \
        "s_waitcnt lgkmcnt(4)\n\t" PV_MM(MN, 14, 252, 0) PV_RD(17472, 252) \
        "s_waitcnt lgkmcnt(4)\n\t" PV_MM(MN, 15, 244, 0) PV_RD(17536, 244) \
        "s_waitcnt lgkmcnt(4)\n\t" PV_MM(MN, 0, 248, 1) PV_RD(17600, 248) \
        "s_waitcnt lgkmcnt(4)\n\t" PV_MM(MN, 1, 252, 1) PV_RD(17664, 252) \
        "s_waitcnt lgkmcnt(4)\n\t" PV_MM(MN, 2, 244, 1) PV_RD(17728, 244) \
        "s_waitcnt lgkmcnt(4)\n\t" PV_MM(MN, 3, 248, 1) PV_RD(17792, 248) \
        "s_waitcnt lgkmcnt(4)\n\t" PV_MM(MN, 4, 252, 1) PV_RD(17856, 252) \
        "s_waitcnt lgkmcnt(4)\n\t" PV_MM(MN, 5, 244, 1) PV_RD(17920, 244) \
        "s_waitcnt lgkmcnt(4)\n\t" PV_MM(MN, 6, 248, 1) PV_RD(17984, 248) \
        "s_waitcnt lgkmcnt(4)\n\t" PV_MM(MN, 7, 252, 1) PV_RD(18048, 252) \
        "s_waitcnt lgkmcnt(4)\n\t" PV_MM(MN, 8, 244, 1) PV_RD(18112, 244) \
        "s_waitcnt lgkmcnt(4)\n\t" PV_MM(MN, 9, 248, 1) PV_RD(18176, 248) \
        "s_waitcnt lgkmcnt(4)\n\t" PV_MM(MN, 10, 252, 1) PV_RD(18240, 252) \
        "s_waitcnt lgkmcnt(4)\n\t" PV_MM(MN, 11, 244, 1) PV_RD(18304, 244) \
        "s_waitcnt lgkmcnt(4)\n\t" PV_MM(MN, 12, 248, 1) PV_RD(18368, 248) \
        "s_waitcnt lgkmcnt(4)\n\t" PV_MM(MN, 13, 252, 1) \
        "s_waitcnt lgkmcnt(2)\n\t" PV_MM(MN, 14, 244, 1) \
        "s_waitcnt lgkmcnt(0)\n\t" PV_MM(MN, 15, 248, 1) \
        : [sa] "=s"(sa), [c0] "+a"(acc[0]), [c1] "+a"(acc[1]), [c2] "+a"(acc[2]), [c3] "+a"(acc[3]), \
          [c4] "+a"(acc[4]), [c5] "+a"(acc[5]), [c6] "+a"(acc[6]), [c7] "+a"(acc[7]), \
          [c8] "+a"(acc[8]), [c9] "+a"(acc[9]), [c10] "+a"(acc[10]), [c11] "+a"(acc[11]), \
          [c12] "+a"(acc[12]), [c13] "+a"(acc[13]), [c14] "+a"(acc[14]), [c15] "+a"(acc[15]) \
        : [a0] "v"(a0), [a1] "v"(a1), [p0] "v"(pk[0]), [p1] "v"(pk[1]), [ap] "s"(aptr) \
        : "v244", "v245", "v246", "v247", "v248", "v249", "v250", "v251", "v252", "v253", \
          "v254", "v255", "memory");
    if constexpr (QT == 0) {
      PV_ASM("v_mfma_f32_32x32x16_bf16")
    } else {
      PV_ASM("v_mfma_f32_32x32x16_f16")
    }
#undef PV_ASM
#undef PV_RD
#undef PV_MM
    return __builtin_bit_cast(RowAddrs, sa);
  };

  // ---- softmax of one tile: P = 2^(S c - m) rounded to bf16, sums ----
  float pe = 0.f;          // sum of P (LSE), per lane
  float pw = 0.f;          // sum of bf16(P): what entered PV (output normaliser)
  float pmax = 0.f;        // fp16 q with fp8 KV: the largest P s rounded for PV
  float xo = -INFINITY;    // max of x - m over the unit, for the overflow guard
  const float c = a.scale_log2;
  // The max over the tile of both half-waves (lane l and lane l ^ 32 hold the two
  // halves of a head's 32 keys).
  auto tile_max = [&](const f32x16_t& x) {
    float mt = fmaxf(fmaxf(x[0], x[1]), x[2]);
#pragma unroll
    for (int r = 3; r < 15; r += 2) mt = fmaxf(mt, fmaxf(x[r], x[r + 1]));
    mt = fmaxf(mt, x[15]);
    const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(mt), __float_as_uint(mt),
                                                     false, false);
    return fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
  };
  // One phase of chunk k (rows 2k, 2k+1) of a tile held in x (in place):
  //   0: x = S c - m (or x - m on the first tile, already scaled), overflow max
  //   1: 2^x (underflow -> 0)
  //   2: bf16 pack into P^T, sum of P
  //   3: sum of bf16(P)
  // Every phase ends by pinning what it wrote (an empty volatile asm that takes and
  // gives the values): volatile asm keeps its place among the MFMA statements, so
  // the optimiser can neither sink the work out of the chain nor merge phases.
  // fp8: sc holds the scales of rows 2 k, 2 k + 1 and iv their inverses (x = S c s;
  // bf16(P s) enters PV and bf16(P s) / s the output normaliser).
  auto sm_phase = [&](f32x16_t& x, u32x4_t(&pk)[2], int k, int ph, bool scaled, f32x2_t sc,
                      f32x2_t iv) {
    const int r = 2 * k;
    float x0 = x[r], x1 = x[r + 1];
    if (ph == 0) {
      if (scaled) {
        x0 -= m_run;
        x1 -= m_run;
      } else if constexpr (KV8) {
        x0 = fmaf(x0, ck * sc[0], -m_run);
        x1 = fmaf(x1, ck * sc[1], -m_run);
      } else {
        x0 = fmaf(x0, c, -m_run);
        x1 = fmaf(x1, c, -m_run);
      }
      float m = fmaxf(xo, fmaxf(x0, x1));
      asm volatile("" : "+v"(x0), "+v"(x1), "+v"(m));
      xo = m;
    } else if (ph == 1) {
      x0 = __builtin_amdgcn_exp2f(x0);
      x1 = __builtin_amdgcn_exp2f(x1);
      asm volatile("" : "+v"(x0), "+v"(x1));
    } else if (ph == 2) {
      const float y0 = KV8 ? x0 * sc[0] : x0, y1 = KV8 ? x1 * sc[1] : x1;
      uint32_t p = pack2_q16<QT>(y0, y1);
      float e = pe + (x0 + x1);
      asm volatile("" : "+v"(p), "+v"(e));
      pk[k >> 2][k & 3] = p;
      pe = e;
      if constexpr (KV8 && QT == 1) {  // the scale can push P s past fp16's range
        float pm = fmaxf(pmax, fmaxf(y0, y1));
        asm volatile("" : "+v"(pm));
        pmax = pm;
      }
    } else if constexpr (KV8) {
      const uint32_t p = pk[k >> 2][k & 3];
      float w2 = fmaf(q16_to_f32<QT>(p >> 16), iv[1], fmaf(q16_to_f32<QT>(p & 0xffffu), iv[0], pw));
      asm volatile("" : "+v"(w2));
      pw = w2;
    } else {
      float w2 = sum2_q16<QT>(pk[k >> 2][k & 3], pw);
      asm volatile("" : "+v"(w2));
      pw = w2;
    }
    x[r] = x0;
    x[r + 1] = x1;
  };
  // The softmax of a tile as work items of the next tile's QK chain (steps -1 ..
  // KSTEPS - 1).  Steady state: chunk k's phase p at step 4k + p - 1 (steps -1 ..
  // 30).  First tile of the unit (the frame is not fixed yet): scale at steps -1
  // and 0, the tile max at step 1, then chunk k's phase p at step 3k + p + 2
  // (steps 2 .. 26).
  // fp8 (tc: the tile being softmaxed, whose scale blocks hold its row scales):
  //   steady: chunk k's phase p at step 4k + p + 1; its scales are read a chunk ahead
  //   into sc8[k & 1] (chunk 0's at step -1), its inverse scales at its phase 1;
  //   first tile: all 16 scales at step -1 (s16), x = S c s at steps 0 and 1, the tile
  //   max at step 2, chunk k's phase p at step 3k + p + 3, its scales read again at
  //   its phase 0 and its inverse scales at its phase 1.
  // Register r of S^T is key 8 (r >> 2) + 4 g + (r & 3), whose scale is at byte
  // 512 (r >> 2) + 16 g + 4 (r & 3) of the scale blocks and its inverse 256 B on.
  auto scl2 = [&](const lds_u8* tl, int k, int inv) -> f32x2_t {
    return *reinterpret_cast<const __attribute__((address_space(3))) f32x2_t*>(
        tl + KV8_SCALES + 256 * inv + 512 * (k >> 1) + 16 * g + 8 * (k & 1));
  };
  auto scl4 = [&](const lds_u8* tl, int qd) -> f32x4_t {
    return *reinterpret_cast<const __attribute__((address_space(3))) f32x4_t*>(
        tl + KV8_SCALES + 512 * qd + 16 * g);
  };
  auto s16_pair = [](const f32x4_t (&s16)[4], int k) -> f32x2_t {
    const f32x4_t v = s16[k >> 1];
    return (k & 1) ? f32x2_t{v[2], v[3]} : f32x2_t{v[0], v[1]};
  };
  auto s16_at = [](const f32x4_t (&s16)[4], int r) -> float { return s16[r >> 2][r & 3]; };
  auto sm_step8 = [&](f32x16_t& x, u32x4_t(&pk)[2], int ks, bool first, const lds_u8* tc,
                      f32x2_t (&sc8)[2], f32x2_t& iv8, f32x4_t (&s16)[4]) {
    if (!first) {
      if (ks == -1) sc8[0] = scl2(tc, 0, 0);
      const int k = (ks - 1) >> 2, ph = (ks - 1) & 3;
      if (ks >= 1 && k < 8) {
        if (ph == 0 && k + 1 < 8) sc8[(k + 1) & 1] = scl2(tc, k + 1, 0);
        if (ph == 1) iv8 = scl2(tc, k, 1);
        sm_phase(x, pk, k, ph, false, sc8[k & 1], iv8);
      }
    } else if (ks == -1) {
#pragma unroll
      for (int qd = 0; qd < 4; ++qd) s16[qd] = scl4(tc, qd);
    } else if (ks == 0 || ks == 1) {
#pragma unroll
      for (int r = 0; r < 8; r += 2) {
        const int rr = 8 * ks + r;
        float x0 = x[rr] * (ck * s16_at(s16, rr)), x1 = x[rr + 1] * (ck * s16_at(s16, rr + 1));
        asm volatile("" : "+v"(x0), "+v"(x1));
        x[rr] = x0;
        x[rr + 1] = x1;
      }
    } else if (ks == 2) {
      float m = fmaxf(m_run, tile_max(x));
      asm volatile("" : "+v"(m));
      m_run = m;
    } else {
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const int ph = ks - 3 - 3 * k;
        if (ph == 0) sc8[k & 1] = scl2(tc, k, 0);
        if (ph == 1) iv8 = scl2(tc, k, 1);
        if (ph >= 0 && ph < 4) sm_phase(x, pk, k, ph, true, sc8[k & 1], iv8);
      }
    }
  };
  auto sm_step = [&](f32x16_t& x, u32x4_t(&pk)[2], int ks, bool first) {
    const f32x2_t none = {1.f, 1.f};
    if (!first) {
      const int k = (ks + 1) >> 2, ph = (ks + 1) & 3;
      if (ks >= -1 && k < 8) sm_phase(x, pk, k, ph, false, none, none);
    } else if (ks == -1 || ks == 0) {
#pragma unroll
      for (int r = 0; r < 8; r += 2) {
        float x0 = x[8 * (ks + 1) + r] * c, x1 = x[8 * (ks + 1) + r + 1] * c;
        asm volatile("" : "+v"(x0), "+v"(x1));
        x[8 * (ks + 1) + r] = x0;
        x[8 * (ks + 1) + r + 1] = x1;
      }
    } else if (ks == 1) {
      float m = fmaxf(m_run, tile_max(x));
      asm volatile("" : "+v"(m));
      m_run = m;
    } else {
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const int ph = ks - 2 - 3 * k;
        if (ph >= 0 && ph < 4) sm_phase(x, pk, k, ph, true, none, none);
      }
    }
  };
  // The unit's last tile, on its own (rows past r1 masked).
  auto softmax_last = [&](f32x16_t& x, u32x4_t(&pk)[2], bool first, int nvalid, const lds_u8* tc) {
    f32x4_t s16[4];
    if constexpr (KV8) {
#pragma unroll
      for (int qd = 0; qd < 4; ++qd) s16[qd] = scl4(tc, qd);
#pragma unroll
      for (int r = 0; r < 16; ++r) x[r] *= ck * s16_at(s16, r);
    } else {
#pragma unroll
      for (int r = 0; r < 16; ++r) x[r] *= c;
    }
    if (nvalid < TILE) {
      const int lim = nvalid - 4 * g;
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (8 * (r >> 2) + (r & 3) >= lim) x[r] = -INFINITY;
    }
    if (first) m_run = fmaxf(m_run, tile_max(x));
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const f32x2_t iv = KV8 ? scl2(tc, k, 1) : f32x2_t{1.f, 1.f};
#pragma unroll
      for (int ph = 0; ph < 4; ++ph)
        sm_phase(x, pk, k, ph, true, KV8 ? s16_pair(s16, k) : f32x2_t{1.f, 1.f}, iv);
    }
  };

  if (!REDO && tid == 0) sm.far = 0;
  {  // ntiles >= 1
    // Ring schedule.  Iteration i: wait for tile i+1 and barrier (tile i+1 visible;
    // every wave is done with tile i-1), then S(i+1) = K(i+1) Q^T with the softmax
    // of tile i and tile i+3's DMA (into tile i-1's slot) interleaved, then
    // O += V(i)^T P(i)^T.  Tiles i, i+1 and i+3 sit in distinct slots; tiles
    // i+2 and i+3 are in flight while i+1 is computed.  Tiles past the last one
    // are DMA'd from the zero row, so every wait counts the same instructions.
    RowAddrs ra_next;
#pragma unroll
    for (int i0 = 0; i0 < 3; ++i0) {
      ra_next = pro_addrs(i0);
#pragma unroll
      for (int k = 0; k < 8; ++k) dma_lat(i0, ra_next, k);
      if constexpr (KV8)
        dma_scale(i0);
      else
        dma_rope(i0, ra_next);
    }
    ra_next = load_addrs(3);

    f32x16_t s_cur, s_next;
    split_query();
    __builtin_amdgcn_s_waitcnt(waitcnt_imm(2 * CPT, 15));  // tile 0 landed
    wait_barrier();
    qk(tiles, s_cur, [](int) {});
    // S(0) is read by VALU next: wait out the XDL-write -> VALU-read hazard
    vgpr_mfma_drain(s_cur);
    if constexpr (F8Q) asm volatile("s_nop 7" : "+v"(s_cur));

    // One PV call site for every tile: the O accumulators are inline-assembly
    // operands, and two call sites in the loop would be given different AGPRs,
    // shuffled through VGPRs on every trip.
    for (int i = 0; i < ntiles; ++i) {
      u32x4_t pk[2];
      if (i + 1 < ntiles) {
        __builtin_amdgcn_s_waitcnt(waitcnt_imm(CPT, 15));  // tile i+1 landed
        wait_barrier();
        const RowAddrs ra_cur = ra_next;
        const lds_u8* tn = tiles + ((i + 1) & (NSTAGE - 1)) * TILEB;
        const lds_u8* tc = tiles + (i & (NSTAGE - 1)) * TILEB;  // tile i (its scales)
        f32x2_t sc8[2], iv8;
        f32x4_t s16[4];
        if (!REDO && i == 0) {
          qk(tn, s_next, [&](int ks) {
            if constexpr (KV8)
              sm_step8(s_cur, pk, ks, true, tc, sc8, iv8, s16);
            else
              sm_step(s_cur, pk, ks, true);
            dma_step(ks, i + 3, ra_cur);
          });
        } else {
          qk(tn, s_next, [&](int ks) {
            if constexpr (KV8)
              sm_step8(s_cur, pk, ks, false, tc, sc8, iv8, s16);
            else
              sm_step(s_cur, pk, ks, false);
            dma_step(ks, i + 3, ra_cur);
          });
        }
      } else {
        softmax_last(s_cur, pk, !REDO && i == 0, r1 - (r0 + i * TILE),
                     tiles + (i & (NSTAGE - 1)) * TILEB);
      }
      SB();
      // PV of tile i, carrying the scalar load of tile i+4's row addresses (after
      // this tile's LDS reads, so the LDS waits in it count exactly; the next
      // barrier's lgkmcnt(0) covers the scalar load).
      {
        const int il = min(i + 4, ntiles - 1);  // dead tiles (>= ntiles) read zeros
        ra_next = fix_tail(pv_asm(tiles + (i & (NSTAGE - 1)) * TILEB, pk, alist + il * TILE + 8 * wu),
                           i + 4);
      }
      // S(i+1) becomes the tile the next trip softmaxes.  The pin orders the copy
      // after PV's 32 MFMAs, which covers the XDL-write -> VALU-read hazard of the
      // chain's last MFMA.
      asm volatile("" : "+v"(s_next));
      s_cur = s_next;
    }
    __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, 15));  // the dead-tile DMAs have landed
    // the last PV MFMAs (inline assembly) write the accumulators: wait out the
    // XDL-write -> VALU-read hazard before the epilogue reads them
    asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7" ::: "memory");
  }
  // both half-waves of a head (lanes l and l ^ 32), summed in the same order in both
  float pes = pe, pws = pw, xobs = xo;
  {
    const auto a1 = __builtin_amdgcn_permlane32_swap(__float_as_uint(pes), __float_as_uint(pes), false, false);
    const auto a2 = __builtin_amdgcn_permlane32_swap(__float_as_uint(pws), __float_as_uint(pws), false, false);
    const auto a3 = __builtin_amdgcn_permlane32_swap(__float_as_uint(xobs), __float_as_uint(xobs), false, false);
    pes = __uint_as_float(a1[0]) + __uint_as_float(a1[1]);
    pws = __uint_as_float(a2[0]) + __uint_as_float(a2[1]);
    xobs = fmaxf(__uint_as_float(a3[0]), __uint_as_float(a3[1]));
  }
  // golden.py:162-163: the sink seeds (m, l) = (sink, 1) on the token's first unit
  const float l_sink = split != 0 ? 0.f : (sink2 == m_run ? 1.f : exp2f(sink2 - m_run));
  const float l_e = l_sink + pes, l_w = l_sink + pws;

  // ---- overflow guard: a logit far above the frame redoes the whole unit ----
  if (!REDO) {
    bool over = xobs > redo_slack<QT>();
    if constexpr (KV8 && QT == 1) over = over || pmax > 32768.f;  // 2^15, as the slack
    if (__any(over) && lane == 0) atomicOr(&sm.far, 1);
    lds_barrier();
    if (sm.far) {
      m_obs = m_run + xobs;
      return true;
    }
  }

  // ---- epilogue: the output leaves through LDS ----
  // Each wave writes its 32 heads' rows into its own region of the ring (idle now:
  // every wave has passed its last PV and its DMAs have landed, which the guard's
  // barrier, or the redo's own below, establishes), then stores them one row per
  // instruction: 64 lanes x 16 B, one contiguous 1 KB.  Stored straight from the
  // accumulator layout, each instruction would write 32 B into each of 32 rows, which
  // the memory pipeline moves at about a quarter of its rate.
  // Accumulator layout: 16-bit KV: register r of block mb of lane (li, g) is d =
  // 32 mb + 16 g + r of head li; fp8: register 4 q + e is d = 32 mb + 8 q + 4 g + e.
  if constexpr (REDO) lds_barrier();
  lds_u8* const ob = tiles + w * EPI_WAVE;
  const int nrows = min(32, H - 32 * w);  // this wave's heads below H (wave-uniform)
  // rows [0, nrows) of the wave's region to dst + r * row_elems (1 KB per row).  The
  // stores are non-temporal: no workgroup of this kernel reads the rows, and lines
  // left dirty in the L2 are written back by the end-of-kernel release, after the
  // last workgroup has finished.
  auto rows_out = [&](auto* dst, size_t row_elems) {
#pragma unroll
    for (int r0 = 0; r0 < 32; r0 += 8) {
      u32x4_t v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = lds_read_b128(ob + (r0 + j) * EPI_STRIDE + 16 * lane);
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (r0 + j < nrows)
          __builtin_nontemporal_store(
              v[j], reinterpret_cast<u32x4_t*>(reinterpret_cast<uint8_t*>(dst + (r0 + j) * row_elems) + 16 * lane));
    }
  };
  auto lds_w128 = [&](int off, u32x4_t v) {
    *reinterpret_cast<__attribute__((address_space(3))) u32x4_t*>(ob + off) = v;
  };
  // Row li of the wave's region: 512 16-bit values (d at 2 d), each O * sc packed by
  // pk (the output dtype, or fp16 for a partial); with track, the largest |O| of the
  // lane's values into mx (from the same reads: a second pass over the accumulators
  // would keep all 256 of them in VGPRs at once).
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
      if constexpr (KV8) {
#pragma unroll
        for (int q2 = 0; q2 < 4; ++q2) {
          const uint32_t p0 = pk(v[4 * q2] * sc, v[4 * q2 + 1] * sc);
          const uint32_t p1 = pk(v[4 * q2 + 2] * sc, v[4 * q2 + 3] * sc);
          typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
          *reinterpret_cast<__attribute__((address_space(3))) u32x2_t*>(
              ob + li * EPI_STRIDE + 64 * mb + 16 * q2 + 8 * g) = u32x2_t{p0, p1};
        }
      } else {
#pragma unroll
        for (int hf = 0; hf < 2; ++hf) {
          u32x4_t o;
#pragma unroll
          for (int e = 0; e < 4; ++e) o[e] = pk(v[8 * hf + 2 * e] * sc, v[8 * hf + 2 * e + 1] * sc);
          lds_w128(li * EPI_STRIDE + 64 * mb + 32 * g + 16 * hf, o);
        }
      }
    }
  };
  const float inv = l_w > 0.f ? 1.f / l_w : 0.f;
  if (splits == 1) {
    stage16([](float x, float y) { return pack2_q16<QT>(x, y); }, inv, std::false_type{});
    rows_out(out + ((size_t)t * H + 32 * w) * DV, DV);
    if (lse && g == 0 && hvalid) lse[(size_t)t * H + h] = (m_run + __log2f(l_e)) * 0.6931471805599453f;
    return false;
  }
  const int slot = wsbase + split;
  if (slot < 0 || slot >= a.slot_cap) return false;  // (a sound plan never gets here)
  // A split unit's partial row of head h sits at float offset (slot H + h) d_v of the
  // partial buffer, with its record (m, l_w, l_e, fmt) for the combine pass.
  if constexpr (PART16<QT> && !REDO) {
    // fmt 1: O / l_w in fp16, in the row's first 1 KB.  Should some head's |O| / l_w
    // reach fp16's range (some |V| does), the unit is redone, and the redo stores
    // fp32 rows.
    stage16([](float x, float z) { return pack2_q16<1>(x, z); }, inv, std::true_type{});
    const bool over = hvalid && mx * inv >= 65504.f;
    if (__any(over) && lane == 0) atomicOr(&sm.far, 1);
    lds_barrier();
    if (sm.far) {
      m_obs = m_run + xobs;
      return true;
    }
    rows_out(reinterpret_cast<uint16_t*>(ws_o + ((size_t)slot * H + 32 * w) * DV), 2 * DV);
    if (g == 0 && hvalid)
      reinterpret_cast<float4*>(ws_ml)[(size_t)slot * H + h] = make_float4(m_run, l_w, l_e, 1.f);
  } else {
    // fmt 0: the un-normalised O in fp32, in two halves of 256 dimensions (1 KB per
    // row each)
#pragma unroll
    for (int half = 0; half < 2; ++half) {
#pragma unroll
      for (int mb = 8 * half; mb < 8 * half + 8; ++mb) {
        const int mo = 128 * (mb - 8 * half);
#pragma unroll
        for (int qd = 0; qd < 4; ++qd) {
          u32x4_t o;
#pragma unroll
          for (int e = 0; e < 4; ++e) o[e] = __float_as_uint(acc[mb][4 * qd + e]);
          lds_w128(li * EPI_STRIDE + mo + (KV8 ? 32 * qd + 16 * g : 64 * g + 16 * qd), o);
        }
      }
      rows_out(ws_o + ((size_t)slot * H + 32 * w) * DV + 256 * half, DV);
    }
    if (g == 0 && hvalid)
      reinterpret_cast<float4*>(ws_ml)[(size_t)slot * H + h] = make_float4(m_run, l_w, l_e, 0.f);
  }
  return false;
}

}  // namespace sas

namespace sas {

// One workgroup per work unit.  rs.addr set: the resolver stage did not run, and
// each unit first resolves its own rows (pool addresses, fp8 scales and the token's
// row counts; rs.rows is null, so no row codes) into the workspace.
template <int DQK, int QT, bool STREAM, bool KV8>
__global__ __launch_bounds__(256, 1) void attend_kernel(
    SasFwdArgs a, const uint16_t* __restrict__ q, const uint64_t* addr_list,
    const float* scale_list, const int2* __restrict__ tokr,
    const float* __restrict__ sinks, const int* __restrict__ plan, uint16_t* __restrict__ out,
    float* __restrict__ lse, float* __restrict__ ws_o, float* __restrict__ ws_ml,
    SasResolveArgs rs) {
  __shared__ __attribute__((aligned(16))) AttendLds<DQK, KV8> sm;
  static_assert(sizeof(RsShared) <= sizeof(sm.tiles), "the resolution borrows the tile ring");
  const int u = blockIdx.x;
  // (every thread writes the same value, so each one's read at the end sees it,
  // whatever barriers the unit's path has)
  sm.stamps = a.stamps;
  // the workgroup's start, kept in LDS until its end (every thread writes its own
  // reading, all within a few cycles of each other; the atomics all wait for the
  // end, where they cost the loop no registers)
  sm.t0 = __builtin_amdgcn_s_memrealtime();
  const int units = plan[PH_UNITS];  // (read with the header: one round trip)
  const bool plan_ok = plan_matches(plan, a);
  if (!plan_ok) {  // a plan built for other arguments: zeros (the combine kernel sets
    if (u < a.T) { // the call's status word)
      for (int i = threadIdx.x; i < a.H * 512 / 8; i += 256)
        reinterpret_cast<u32x4_t*>(out + (size_t)u * a.H * 512)[i] = u32x4_t{0, 0, 0, 0};
      if (lse)
        for (int i = threadIdx.x; i < a.H; i += 256) lse[(size_t)u * a.H + i] = 0.f;
    }
    return;
  }
  if (u >= units) return;
  const int* ur = plan + SAS_PLAN_HDR + (size_t)SAS_TOK_W * a.T + (size_t)u * SAS_UNIT_W;
  const int t = ur[0];
  // resolved here: the token's window and compressed row counts (the compressed
  // count at least what this unit needs)
  int2 live = make_int2(0, 0);
  int own_hi = a.list_stride;
  if (rs.addr) {
    const int* tk = plan + SAS_PLAN_HDR + (size_t)t * SAS_TOK_W;
    const int split = ur[3];
    // The token's last unit resolves to the list's end (its count is then exact; the
    // call's KV lengths may exceed the plan's), the others their planned ranges.
    const bool last = split < 0 || split == tk[TK_SPLITS] - 1;
    own_hi = last ? a.list_stride : min(ur[2], a.list_stride);
    int nwin = 0;
    const int nc = resolve_rows<false>(a, tk, true, t, ur[1], own_hi,
                                       *reinterpret_cast<RsShared*>(sm.tiles), rs, nwin);
    live = make_int2(nwin, nwin < 0 ? 0 : nc);
    if (rs.tok && threadIdx.x == 0 && last) rs.tok[t] = live;
    // Every wave's stores have reached L2 before any wave reads the lists back
    // (vector and scalar loads, the scale DMA), and every wave is done with the
    // borrowed LDS.
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
  }
  // The lists are read through pointers the compiler cannot trace to the stores
  // above, so none of those loads moves before the barrier.
  asm volatile("" : "+s"(addr_list), "+s"(scale_list));
  float m_obs = 0.f;
  const bool fused = rs.addr != nullptr;
  if (attend_unit<DQK, QT, STREAM, KV8, false>(u, sm, a, q, addr_list, scale_list, tokr, fused,
                                               live, own_hi, sinks, plan, out, lse, ws_o, ws_ml,
                                               m_obs)) {
    lds_barrier();  // every wave is done with the ring before the redo refills it
    attend_unit<DQK, QT, STREAM, KV8, true>(u, sm, a, q, addr_list, scale_list, tokr, fused, live,
                                            own_hi, sinks, plan, out, lse, ws_o, ws_ml, m_obs);
  }
  // the workgroup's end on the real-time counter, after every wave's stores have
  // completed (the pointer read back from LDS)
  uint64_t* stamps = sm.stamps;
  if (stamps) {
    __syncthreads();
    // (global atomics: through a generic pointer they would be FLAT ones)
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
