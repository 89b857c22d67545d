// sas_backward_tile.hip -- the KV pools' gradient by key tiles, for calls whose tokens
// share their rows (prefill-like).
//
// The per-unit kernel (bwd_dkv_kernel) walks a token's rows and adds every row's
// gradient to its pool row with fp32 atomics: d_qk of them per (token, row) pair, and
// the chip sustains about 330 G fp32 atomic adds/s (1.3 TB/s of floats, whatever the
// rows or the lane layout).  Here a workgroup keeps the gradient of 128 consecutive
// positions of a sequence in registers over a group of tokens and adds it to the pool
// once: 128 d_qk atomics per (tile, group) instead of d_qk per pair.  P and dS come
// from the dq kernel's spill, so nothing is recomputed.
//
//   bwd_items_kernel     the (token group, key tile) items of a run of tokens.
//   bwd_dkv_tile_kernel  G += (scale dS)^T Q + P^T dO over the item's tokens.
//
// One item, 8 waves: wave w takes dimension quarter w & 3 (128 latent dimensions and,
// at d_qk 576, 16 of rope) of the 64 keys of half w >> 2: 4 x 9 accumulator blocks of
// 16 keys x 16 dimensions (144 registers, two waves per SIMD).  A step is 32 heads of
// one token: their q and dO rows (68 KB) and the keys' spilled dS and P (16 KB) are DMA'd
// to LDS through a ring of half steps; q and dO are read transposed (ds_read_b64_tr_b16)
// as the B operands, dS and P 16 B per lane (8 heads of one key).  At 128 keys a
// step's matrix work is 2,176 cycles per SIMD, its LDS traffic about 1,900 and its loads
// 1,300 at 64 B per clock: half as many keys per item would leave the loads and the LDS
// as the bound.
//
// Measured (the pools' gradient of packed training batches, before: the per-unit kernel):
// 4 documents of 608 .. 1,697 tokens, 128 heads, top-k 512: 2,424 -> 565 us (and 300 us
// for the spill in the dq kernel as it was then); documents of 1,082 and 971 tokens, 64
// heads, window only, d_qk 512: 424 -> 107 us (and 50 us).
// What bounds it now is memory: 3.2 GB read in 565 us (5.7 TB/s), of which 1.7
// GB are first reads.  A operands loaded by every wave that uses them (64 loads of 16
// rows per step, instead of 16 DMAs into the ring) doubled its time: a load of 16
// 64-B rows occupies the vector memory pipe about 40 cycles.
#include <hip/hip_runtime.h>

#include "sas_common.h"

namespace sas {

constexpr int TK_KEYS = SAS_BWD_KEYS;  // keys per item
constexpr int TK_NT = 512;             // threads per workgroup

// The call's lengths and tables, and the run's items.
struct SasTileArgs {
  const int* q_prefix;
  const int* act_q;
  const int* seqused_kv;
  const int* ori_bt;
  const int* cmp_bt;
  const uint32_t* inv;  // scenario 3: the resolver's inverse lists, [the run's tokens][cmp_rows]
  int cmp_rows;         // compressed rows covered by tiles (0: none)
  int item_cap;
  int workers;          // workgroups of bwd_dkv_tile_kernel
  int want_ori, want_cmp;
  int4* items;  // [0].x: their number; item i at 1 + i: (sequence, first token, tokens |
                // compressed << 16, key tile)
};

// Block-wide inclusive scan of one int per thread (1024 threads); total: the sum.
__device__ __forceinline__ int items_scan(int v, int* wsum, int& total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int o = __shfl_up(v, off);
    if (lane >= off) v += o;
  }
  __syncthreads();  // earlier readers of wsum are done
  if (lane == 63) wsum[wave] = v;
  __syncthreads();
  total = 0;
  int before = 0;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    if (i < wave) before += wsum[i];
    total += wsum[i];
  }
  return v + before;
}

// One workgroup of 1024 threads: the token groups of every sequence (its tokens of this
// run, `group` at a time), then per group its window tiles and its compressed tiles.  A
// group's items are consecutive, so that its tokens' q and dO rows are read by
// workgroups of one XCD at about the same time (bwd_dkv_tile_kernel's item order).
//
// The group size: every item costs about its tokens' visits plus a fixed part (its
// prologue and the tile's atomics, about TILE_FIXED visits), and the workgroups take the
// items round by round, so the sizes tried are ranked by rounds x (group + TILE_FIXED).
constexpr int TILE_FIXED = 8;
__device__ constexpr int TILE_GROUPS[] = {64, 48, 40, 32, 28, 24, 20, 18, 16, 14, 12, 10, 8};

__global__ __launch_bounds__(1024) void bwd_items_kernel(SasFwdArgs a, SasTileArgs ta, SasBwdSpill sp,
                                                         const int* __restrict__ plan) {
  __shared__ int gpre[SAS_BWD_MAX_B + 1];  // a sequence's first group
  __shared__ int qlo[SAS_BWD_MAX_B], qn[SAS_BWD_MAX_B], sg_lo[SAS_BWD_MAX_B];
  __shared__ int wsum[16];
  __shared__ long long cost[16];
  const int tid = threadIdx.x;
  // the spill's zero record
  for (int i = tid; i < sp.row_bytes / 4; i += 1024) reinterpret_cast<int*>(sp.data)[i] = 0;
  if (!plan_matches(plan, a)) {
    if (tid == 0) ta.items[0] = make_int4(0, 0, 0, 0);
    return;
  }
  // sequence b's tokens in this run (a token past the next sequence's first belongs to
  // that one): the first, their number and the first one's position
  for (int b = tid; b < a.B; b += 1024) {
    const int q0 = ta.q_prefix[b], nq = ta.act_q[b], next = b + 1 < a.B ? ta.q_prefix[b + 1] : a.T;
    const int lo = max(q0, sp.t0);
    qlo[b] = lo;
    qn[b] = max(0, min(min(q0 + nq, next), min(sp.t1, a.T)) - lo);
    sg_lo[b] = ta.seqused_kv[b] - nq + lo - q0;
  }
  __syncthreads();
  // group i of G tokens of sequence b: its token count, first window tile, window tiles
  // and compressed tiles
  struct Group {
    int n, wlo, nw, nc;
  };
  auto group_of = [&](int b, int i, int G) -> Group {
    Group r = {min(G, qn[b] - i * G), 0, 0, 0};
    const int sg0 = sg_lo[b] + i * G, sg1 = sg0 + r.n - 1;
    if (sg1 >= 0) {
      r.wlo = max(sg0 - a.win_left, 0) / TK_KEYS;
      if (ta.want_ori) r.nw = sg1 / TK_KEYS - r.wlo + 1;
      if (ta.want_cmp) r.nc = (min((sg1 + 1) / a.cmp_ratio, ta.cmp_rows) + TK_KEYS - 1) / TK_KEYS;
    }
    return r;
  };
  // wave k counts the items of groups of TILE_GROUPS[k] tokens: its lanes over the groups
  // of one sequence after another, or (many sequences) over the sequences
  constexpr int NG = sizeof(TILE_GROUPS) / sizeof(int);
  static_assert(NG <= 16, "one wave per group size");
  const int lane = tid & 63, wave = tid >> 6;
  if (wave < NG) {
    const int G = TILE_GROUPS[wave];
    const bool by_seq = a.B >= 64;
    int n = 0;
    for (int b = by_seq ? lane : 0; b < a.B; b += by_seq ? 64 : 1)
      for (int i = by_seq ? 0 : lane; i * G < qn[b]; i += by_seq ? 1 : 64) {
        const Group r = group_of(b, i, G);
        n += r.nw + r.nc;
      }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) n += __shfl_xor(n, off);
    if (lane == 0) cost[wave] = (long long)((n + ta.workers - 1) / ta.workers) * (G + TILE_FIXED);
  }
  __syncthreads();
  int G = TILE_GROUPS[0];
  for (int k = 1, best = 0; k < NG; ++k)
    if (cost[k] < cost[best]) {
      best = k;
      G = TILE_GROUPS[k];
    }
  // each sequence's first group
  int carry = 0, total;
  for (int base = 0; base < a.B; base += 1024) {
    const int b = base + tid;
    const int n = b < a.B ? (qn[b] + G - 1) / G : 0;
    const int inc = items_scan(n, wsum, total);
    if (b < a.B) gpre[b] = carry + inc - n;
    carry += total;
  }
  const int groups = carry;
  __syncthreads();
  carry = 0;
  for (int base = 0; base < groups; base += 1024) {
    const int g = base + tid;
    Group r = {0, 0, 0, 0};
    int b = 0, at = 0;
    if (g < groups) {
      int hi = a.B - 1;  // the last sequence with gpre <= g
      while (b < hi) {
        const int mid = (b + hi + 1) >> 1;
        if (gpre[mid] <= g) b = mid; else hi = mid - 1;
      }
      at = g - gpre[b];
      r = group_of(b, at, G);
    }
    const int n = r.nw + r.nc, first = qlo[b] + at * G;
    int o = carry + items_scan(n, wsum, total) - n;
    for (int i = 0; i < n; ++i, ++o)
      if (o < ta.item_cap)
        ta.items[1 + o] = make_int4(b, first, r.n | (i < r.nw ? 0 : 1 << 16), i < r.nw ? r.wlo + i : i - r.nw);
    carry += total;
  }
  if (tid == 0) ta.items[0] = make_int4(min(carry, ta.item_cap), G, 0, 0);
}

// A slot holds half a step: 32 heads' q rows and the 128 keys' dS, or their dO rows and P.
template <int DQK>
struct TileLds {
  static constexpr int ROPE = (DQK - 512) * 2;             // rope bytes per row
  static constexpr int QL = 32 * 1024, QR = 32 * ROPE;     // latent rows (or dO's), rope rows
  static constexpr int SLOT = QL + QR + TK_KEYS * 64;      // and the keys' A rows
  __attribute__((aligned(16))) uint8_t slot[3 * SLOT];
};

template <int DQK, int QT>
__device__ __forceinline__ void dkv_tile(TileLds<DQK>& sm, const int4 it, const SasFwdArgs& a, const SasTileArgs& ta,
                                         const SasBwdSpill& sp, const uint16_t* __restrict__ q,
                                         const uint16_t* __restrict__ dout,
                                         const int2* __restrict__ tok, const int* __restrict__ plan,
                                         float* __restrict__ d_ori, float* __restrict__ d_cmp) {
  constexpr bool ROPE = DQK > 512;
  constexpr int NDB = ROPE ? 9 : 8;  // 16-dimension blocks per wave
  constexpr int SLOT = TileLds<DQK>::SLOT, QL = TileLds<DQK>::QL, QR = TileLds<DQK>::QR;
  typedef __attribute__((address_space(3))) uint8_t l_u8;
  typedef short tr_s4 __attribute__((ext_vector_type(4)));
  l_u8* const lds = (l_u8*)sm.slot;

  const int b = it.x, first = it.y, n = it.z & 0xffff, space = it.z >> 16, tile = it.w;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n16 = lane & 15, g = lane >> 4;
  const int dq4 = w & 3, half = w >> 2;
  const int p0 = tile * TK_KEYS;            // the tile's first position
  const int pa = p0 + 16 * w + (lane >> 2);  // the key whose A row this lane copies
  const int NG = (a.H + 31) / 32;
  const bool use_inv = space == 1 && a.scenario == 3;

  // ---- the visits: lane i holds token first + i ----
  // Positions lo .. hi are the token's; position p sits at list position p + delta
  // (with use_inv, where the inverse list says).  cnt: how often the visit's rows are
  // taken (a row listed several times; 0: no visit).
  int v_lo = 0, v_hi = -1, v_delta = 0, v_cnt = 0;
  const int kv = ta.seqused_kv[b], nq = ta.act_q[b], q0 = ta.q_prefix[b];
  if (lane < n) {
    const int t = first + lane;
    const int2 tr = tok[t];
    const bool ok = plan[SAS_PLAN_HDR + (size_t)t * SAS_TOK_W + TK_B] == b && tr.x >= 0 &&
                    sp.flags[1 + t] == 0;
    const int sg = kv - nq + t - q0;
    if (space == 0) {
      v_lo = max(sg - a.win_left, 0);
      v_hi = min(sg, v_lo + tr.x - 1);
      v_delta = -v_lo;
    } else {
      v_hi = a.scenario == 2 ? tr.y - 1 : min((sg + 1) / a.cmp_ratio, ta.cmp_rows) - 1;
      v_delta = tr.x;
    }
    v_cnt = ok && v_lo < p0 + TK_KEYS && v_hi >= p0 ? 1 : 0;
  }
  if (use_inv) {  // the rows of the tile that each token lists: the largest count
    int* const mx = reinterpret_cast<int*>(sm.slot);
    for (int i = w; i < n; i += TK_NT / 64) {
      const int hi = __builtin_amdgcn_readlane(v_hi, i), c = __builtin_amdgcn_readlane(v_cnt, i);
      int m = 0;
      if (c) {
        const uint32_t* iv = ta.inv + (size_t)(first + i - sp.t0) * ta.cmp_rows;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          const int p = p0 + 64 * k + lane;
          if (p <= hi) m = max(m, (int)(iv[p] >> 16));
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) m = max(m, __shfl_xor(m, off));
      }
      if (lane == 0) mx[i] = m;
    }
    __syncthreads();
    if (lane < n) v_cnt = mx[lane];
    __syncthreads();
  }
  uint64_t left = __ballot(v_cnt > 0);  // visits not yet begun
  if (left == 0) return;  // (the same in every wave)

  // ---- half a step to LDS: part 0 q and dS, part 1 dO and P, of 32 heads (chunk c) ----
  // Latent (and dO) rows of 1 KB: the 32-B pair P of row r at P ^ f(r), f = (r & 3) |
  // (r bit 3) << 2; rope rows of 128 B: pair P at P ^ ((r bit 1) | (r bit 3) << 1).  A
  // transposed read addresses 8 rows (r, r + 8 of 0 .. 3) x 32 B per 32 lanes, which then
  // touch every bank once per 256 B.  Wave w copies rows 4 w .. 4 w + 3 of each part and
  // the A rows (64 B: 32 heads of one key) of keys 16 w .. + 15; heads at or past H are
  // empty ranges (zeros).
  const uint32_t fb = (uint32_t)((w >> 1) & 1);
  const uint32_t vlat = 16u * ((uint32_t)lane ^ (8u * fb));
  const uint32_t rr = (uint32_t)(4 * w + ((lane >> 3) & 3));  // rope: row of lanes 0 .. 31
  const uint32_t vrope = ((uint32_t)(lane >> 3) & 3u) * DQK * 2 + 1024u +
                         16u * (((uint32_t)lane & 7u) ^ (2u * (((rr >> 1) & 1u) | ((rr >> 3) & 1u) << 1)));
  auto rsrc = [&](const void* p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc((void*)p, (short)0, (int)bytes, 0x00020000);
  };
  typedef __attribute__((address_space(3))) void l_void;
  const uint32_t spill_bytes = (1u + (uint32_t)(sp.t1 - sp.t0) * (uint32_t)sp.stride) * (uint32_t)sp.row_bytes;
  uint32_t off = 0;  // byte offset of the record of the lane's key (0: the zero record)
  auto dma = [&](int t, int c, auto part, int sl) {
    constexpr bool Q = decltype(part)::value == 0;
    constexpr int LD = Q ? DQK : 512;
    const uint16_t* src = Q ? q : dout;
    l_u8* const dst = lds + sl * SLOT;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int r = 4 * w + k, h = 32 * c + r;
      const size_t th = (size_t)t * a.H + min(h, a.H - 1);
      uint32_t vo = vlat;  // formed here rather than kept across the loop
      asm volatile("" : "+v"(vo));
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc(src + th * LD, h < a.H ? 1024u : 0u),
                                               (l_void*)(dst + 1024 * r), 16, vo ^ (32u * k), 0, 0, 0);
    }
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc(sp.data, spill_bytes), (l_void*)(dst + QL + QR + 1024 * w), 16,
                                             off + 16u * ((uint32_t)lane & 3u), 128 * c + (Q ? 0 : 64), 0, 0);
    if constexpr (Q && ROPE) {
      const int h0 = 32 * c + 4 * w;
      // (readfirstlane: the clamp selects v_med3, and a buffer resource in VGPRs would be
      // issued lane by lane)
      const int rows = __builtin_amdgcn_readfirstlane(max(0, min(4, a.H - h0)));
      const size_t th = (size_t)t * a.H + __builtin_amdgcn_readfirstlane(min(h0, a.H - 1));
      const auto rs = rsrc(q + th * DQK, (uint32_t)rows * DQK * 2);
      if (lane < 32)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (l_void*)(dst + QL + 512 * w), 16, vrope, 0, 0, 0);
    }
  };
  typedef std::integral_constant<int, 0> PartQ;
  typedef std::integral_constant<int, 1> PartO;
  constexpr int NQ = ROPE ? 6 : 5, NO = 5;  // DMA instructions of a wave per part
  // The inverse-list entry of the lane's key for visit i (without inverse lists: an
  // unused word), a plain load in every step: a load behind a branch is waited for where
  // the paths join.
  auto load_inv = [&](int i) -> uint32_t {
    typedef __attribute__((address_space(1))) const uint8_t g_u8;
    const g_u8* iv = use_inv ? (const g_u8*)(uintptr_t)(ta.inv + (size_t)(first + i - sp.t0) * ta.cmp_rows)
                             : (const g_u8*)(uintptr_t)sp.data;
    // (positions past the token's last read that one: set_rows drops them)
    const int hi = use_inv ? __builtin_amdgcn_readlane(v_hi, i) : 0;
    return *(__attribute__((address_space(1))) const uint32_t*)(iv + 4u * (uint32_t)min(pa, hi));
  };
  uint32_t ivn;        // the entry that the next set_rows uses
  bool touched = false;  // some token took the lane's key
  // the lane's record for visit i, round r (rows listed more than r times); returns
  // whether the wave's 64 keys hold any of the token's positions
  auto set_rows = [&](int i, int r) -> bool {
    const int lo = __builtin_amdgcn_readlane(v_lo, i), hi = __builtin_amdgcn_readlane(v_hi, i);
    const int delta = __builtin_amdgcn_readlane(v_delta, i);
    bool ok = pa >= lo && pa <= hi;
    uint32_t pos = (uint32_t)(pa + delta);
    if (use_inv) {
      ok = ok && (int)(ivn >> 16) > r;
      pos = ivn & 0xffffu;
    }
    off = ok ? (1u + (uint32_t)(first + i - sp.t0) * (uint32_t)sp.stride + pos) * (uint32_t)sp.row_bytes : 0u;
    touched = touched || ok;
    return lo < p0 + 64 * half + 64 && hi >= p0 + 64 * half;
  };

  bw_f32x4 acc[4][NDB];
#pragma unroll
  for (int kb = 0; kb < 4; ++kb)
#pragma unroll
    for (int k = 0; k < NDB; ++k) acc[kb][k] = bw_f32x4{0.f, 0.f, 0.f, 0.f};

  // B operands: lane i of block g addresses head 8 g + (i >> 2) (+ 4), dimensions 16 db
  // + 4 (i & 3) .. + 3 of the staged rows
  const uint32_t br = (uint32_t)(8 * g + (n16 >> 2));
  const uint32_t bf = (br & 3u) | (((br >> 3) & 1u) << 2);
  const uint32_t blat = br * 1024u + 256u * (uint32_t)dq4 + 32u * bf + 8u * (uint32_t)(n16 & 3);
  const uint32_t brope = (uint32_t)QL + br * 128u +
                         32u * ((uint32_t)dq4 ^ (((br >> 1) & 1u) | (((br >> 3) & 1u) << 1))) +
                         8u * (uint32_t)(n16 & 3);
  auto tr2 = [&](const l_u8* p, int hi_off) -> u32x4_t {
    const tr_s4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) tr_s4*)p);
    const tr_s4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) tr_s4*)(p + hi_off));
    return u32x4_t{(uint32_t)(uint16_t)lo[0] | ((uint32_t)(uint16_t)lo[1] << 16),
                   (uint32_t)(uint16_t)lo[2] | ((uint32_t)(uint16_t)lo[3] << 16),
                   (uint32_t)(uint16_t)hi[0] | ((uint32_t)(uint16_t)hi[1] << 16),
                   (uint32_t)(uint16_t)hi[2] | ((uint32_t)(uint16_t)hi[3] << 16)};
  };
  const uint32_t ba = (uint32_t)(QL + QR) + 4096u * (uint32_t)half + 64u * (uint32_t)n16 + 16u * (uint32_t)g;
  constexpr int AHEAD = 3;  // B fragments read ahead of their MFMAs
  auto phase = [&](const l_u8* tl, auto part) {
    constexpr int NB = decltype(part)::value == 0 && ROPE ? 9 : 8;
    // (the block offsets are formed per read rather than kept across the loop)
    uint32_t bl = blat;
    asm volatile("" : "+v"(bl));
    auto frag = [&](int k) -> u32x4_t {
      return k < 8 ? tr2(tl + (bl ^ (32u * (uint32_t)k)), 4096) : tr2(tl + brope, 512);
    };
    u32x4_t f[4], bq[AHEAD + 1];
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) f[kb] = lds_read_b128(tl + ba + 1024 * kb);
#pragma unroll
    for (int k = 0; k < AHEAD; ++k) bq[k] = frag(k);
    BW_SB();
#pragma unroll
    for (int k = 0; k < NB; ++k) {
      if (k + AHEAD < NB) bq[(k + AHEAD) % (AHEAD + 1)] = frag(k + AHEAD);
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) acc[kb][k] = bw_mfma<QT>(f[kb], bq[k % (AHEAD + 1)], acc[kb][k]);
      BW_SB();
    }
  };

  // ---- the steps: (visit, round, 32 heads), half a step at a time ----
  // Ring of three slots: half a step is computed while the next one, issued a half step
  // earlier, arrives and the one after is issued (the last step issues itself again,
  // unused).  The wait at the top of a half leaves the next half's loads in flight.
  int vi = (int)__builtin_ctzll(left), rnd = 0, c = 0, sl = 0;
  left &= left - 1;
  // the visit that the set_rows after (visit i, round r) takes
  auto inv_of = [&](int i, int r) -> int {
    return left && r + 1 >= __builtin_amdgcn_readlane(v_cnt, i) ? (int)__builtin_ctzll(left) : i;
  };
  ivn = load_inv(vi);
  bool busy = set_rows(vi, 0);
  ivn = load_inv(inv_of(vi, 0));
  asm volatile("" ::: "memory");
  dma(first + vi, 0, PartQ{}, 0);
  dma(first + vi, 0, PartO{}, 1);
  asm volatile("" ::: "memory");
  bool more = true;
  while (more) {
    // the next step
    int vi2 = vi, rnd2 = rnd, c2 = c + 1;
    bool fresh = false;  // another visit or round
    if (c2 == NG) {
      fresh = true;
      c2 = 0;
      if (rnd + 1 < __builtin_amdgcn_readlane(v_cnt, vi)) {
        ++rnd2;
      } else if (left) {
        vi2 = (int)__builtin_ctzll(left);
        rnd2 = 0;
        left &= left - 1;
      } else {
        more = false;
        fresh = false;
        c2 = c;
      }
    }
    const bool busy_now = busy;
    const int s1 = sl == 2 ? 0 : sl + 1, s2 = s1 == 2 ? 0 : s1 + 1;
    __builtin_amdgcn_s_waitcnt(waitcnt_imm(NO, 0));  // q and dS have landed
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (fresh) busy = set_rows(vi2, rnd2);
    dma(first + vi2, c2, PartQ{}, s2);
    ivn = load_inv(inv_of(vi2, rnd2));
    asm volatile("" ::: "memory");
    BW_SB();
    if (busy_now) phase(lds + sl * SLOT, PartQ{});
    BW_SB();
    __builtin_amdgcn_s_waitcnt(waitcnt_imm(NQ + 1, 0));  // dO and P have landed
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    dma(first + vi2, c2, PartO{}, sl);
    asm volatile("" ::: "memory");
    BW_SB();
    if (busy_now) phase(lds + s1 * SLOT, PartO{});
    BW_SB();
    vi = vi2;
    rnd = rnd2;
    c = c2;
    sl = s2;
  }
  // the last step's unused DMA has landed in every wave, and every wave is done reading
  __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, 0));
  __syncthreads();
  uint8_t* const took = sm.slot;  // which of the tile's keys some token took
  if ((lane & 3) == 0) took[16 * w + (lane >> 2)] = touched;
  __syncthreads();

  // ---- the tile's gradient to the pool rows: keys 16 kb + 4 g + r of the half ----
  const int* bt = space ? ta.cmp_bt + (size_t)b * a.cmp_table_len : ta.ori_bt + (size_t)b * a.ori_table_len;
  const int bs = space ? a.cmp_block_size : a.ori_block_size;
  const int tl_len = space ? a.cmp_table_len : a.ori_table_len;
  const int bnum = space ? a.cmp_block_num : a.ori_block_num;
  const int64_t bstr = space ? a.cmp_block_stride : a.ori_block_stride;
  const int64_t rstr = space ? a.cmp_row_stride : a.ori_row_stride;
  float* const pool = space ? d_cmp : d_ori;
#pragma unroll
  for (int kb = 0; kb < 4; ++kb)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int k = 4 * g + r;
      const int key = 64 * half + 16 * kb + k;
      const int code = took[key] ? paged_code(bt, tl_len, bs, bnum, p0 + key) : -1;
      if (code >= 0) {
        const int page = (int)((unsigned)code / (unsigned)bs);
        float* row = pool + (size_t)page * bstr + (size_t)(code - page * bs) * rstr + n16;
#pragma unroll
        for (int d = 0; d < NDB; ++d)
          gatomic_add(row + (d < 8 ? 128 * dq4 + 16 * d : 512 + 16 * dq4), acc[kb][d][r]);
      }
    }
}

template <int DQK, int QT>
__global__ __launch_bounds__(TK_NT) void bwd_dkv_tile_kernel(
    SasFwdArgs a, SasTileArgs ta, SasBwdSpill sp, const uint16_t* __restrict__ q,
    const uint16_t* __restrict__ dout, const int2* __restrict__ tok, const int* __restrict__ plan,
    float* __restrict__ d_ori, float* __restrict__ d_cmp) {
  __shared__ TileLds<DQK> sm;
  // The items in rounds of one per workgroup; workgroups x, x + 8, ... run on XCD x mod 8,
  // which takes a run of consecutive items of every round.
  const int items = ta.items[0].x, W = gridDim.x, run = W >> 3;
  const int at = (int)(blockIdx.x & 7) * run + (int)(blockIdx.x >> 3);
  for (int r = 0; r < items; r += W) {
    // (a partial round is spread over the XCDs as a full one)
    const int left = min(items - r, W), per = (left + 7) >> 3;
    const int x = at / run, k = at - x * run;
    const int i = k < per ? x * per + k : left;
    if (i < left) dkv_tile<DQK, QT>(sm, ta.items[1 + r + i], a, ta, sp, q, dout, tok, plan, d_ori, d_cmp);
    __syncthreads();  // every wave is done with the item's LDS
  }
}

}  // namespace sas
