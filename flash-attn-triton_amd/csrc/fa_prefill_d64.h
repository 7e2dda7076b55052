// FlashAttention-2 prefill forward for gfx950 at head dim 64, plain epilogue
// (scale, causal and window masks), fp16 / bf16: dense, cross, varlen, and
// chunks of queries against a KV cache.
//
// Semantics are those of prefill_pp_kernel (fa_prefill_pp.h), the same launch
// forms at head dim 128; row packing, key splits, block-table reads and the
// precision of the KV-cache and paged forms are described there.
//
// At head dim 64 a 64-key tile of a wave's 32 rows holds 16 MFMAs (512 matrix
// cycles) and as many scores as at 128: per score a scale, an exp2 and parts
// of the max, packing and row sum, about 680 vector-ALU cycles.  The vector
// ALU is the longer side, so the ping-pong schedule's lockstep phases would
// leave the matrix core idle; here three waves per SIMD run freely and cover
// for each other.  What is done about the vector and scalar work of a tile:
//  * the S^T products start from -m (the running max in raw score units, kept
//    in 16 registers), so the exp2 argument is one multiply per score and no
//    accumulator is cleared;
//  * tiles go global -> LDS by LDS-DMA into three stages of 8 KiB each for K
//    and V (48 KiB per workgroup, three workgroups per CU), two tiles ahead,
//    without staging registers;
//  * tiles are walked downwards in three runs: those that may cut the upper
//    bound, those every row sees whole (unrolled by the three stages, so that
//    every LDS address is a per-lane offset plus an immediate, and without any
//    mask or range test), those that may cut the lower bound;
//  * the S^T products run at raised wave priority, so that they are not queued
//    behind the other waves' vector work.
// LDS rows are 128 bytes without padding; 16-byte chunk c of row r sits at
// c ^ (r / 2 % 8) (K) or c ^ 4 (r / 2 % 2) (V), so the 16 rows of a K read and
// the 4 x 4 chunks of a transposed V read touch distinct banks (256 bytes).
//
// Bound: issue on the vector ALU (busy 70 % of the cycles, the matrix core
// 48 %, at the 1.6 GHz the chip holds under this load; B4 H32 S4096).
// Measured on one MI355X against prefill_kernel (4 waves, tiles staged through
// VGPRs), per call, fp16, B / S / Hq / Hk:
//   non-causal  4 / 1024 / 32 / 32   58.7 ->  45.2 us (760 TFLOP/s)
//   non-causal  4 / 4096 / 32 / 32    762 ->   598 us (920 TFLOP/s)
//   causal      8 / 1024 / 16 / 16   52.4 ->  33.9 us
//   causal      2 / 3001 / 32 / 8     145 ->  92.6 us
//   causal      4 / 4096 / 32 / 32    432 ->   316 us (870 TFLOP/s)
// Tried and dropped: four waves per SIMD (128 registers, 12 spilled; equal at
// S = 4096, 6 % slower at 1024), 32-key tiles (10 % slower), two stages (1 %
// slower at S = 4096), row sums on the matrix core (5 % slower), all K reads
// ahead of the products or the V reads ahead of the exps (within 1 %).
#pragma once

#include <type_traits>

#include "fa_prefill_pp.h"

namespace fa {

struct D64Tile {
  static constexpr int NW = 4;
  static constexpr int BM = 32 * NW, NT = 64 * NW;
  static constexpr int BN = 64;             // keys per tile
  static constexpr int NS = 3;              // LDS stages per operand
  static constexpr int ROWB = 128;          // bytes per K / V row
  static constexpr int TILEB = BN * ROWB;   // bytes per K or V tile
  static constexpr int LDS_BYTES = 2 * NS * TILEB;
  static constexpr int IPW = TILEB / 1024 / NW;   // DMA instructions per wave and tile
  static_assert(IPW * NW * 1024 == TILEB, "tile must split evenly over the waves");
};

// Waits until at most N vector-memory instructions of this wave are
// outstanding (and keeps LDS reads from moving ahead of the wait).
template <int N>
__device__ inline void wait_loads() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// Ring step barrier: at most N tile loads of this wave are outstanding, and
// every LDS read it has issued has returned, so that after it any wave may
// refill what was read.  (The products that use the reads are not memory
// operations: without the scheduling barriers nothing keeps them, and with
// them the compiler's own wait, on this side of the barrier.)
template <int N>
__device__ inline void ring_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// MODE: kPpDense / kPpVarlen / kPpCache (fa_prefill_pp.h).
template <class T, int MODE, bool PAGED>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3, 3)))
void prefill_d64_kernel(const FwdParams p) {
  using Tile = D64Tile;
  constexpr int D = 64, NW = Tile::NW, BM = Tile::BM, BN = Tile::BN, NS = Tile::NS;
  constexpr int ROWB = Tile::ROWB, TILEB = Tile::TILEB, IPW = Tile::IPW;
  constexpr int NKC = D / 16, NDB = D / 32, NKB = BN / 32, NCC = BN / 16;
  constexpr bool VARLEN = MODE == kPpVarlen, CACHE = MODE == kPpCache;
  static_assert(!PAGED || MODE != kPpDense, "dense K/V are not paged");
  // The KV-cache and paged forms raise the max with every larger score and
  // sum the fp32 P.
  constexpr float kSlack = CACHE || PAGED ? 0.f : kRescaleSlack;
  constexpr bool kSumRounded = T::kSumRounded && !CACHE && !PAGED;

  extern __shared__ __attribute__((aligned(1024))) uint8_t smem_d64[];
  uint8_t* const k_ring = smem_d64;
  uint8_t* const v_ring = smem_d64 + NS * TILEB;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c32 = lane & 31;
  const int g = lane >> 5;

  // ------------------------------------------------------------ work item
  int mb, hh, b, kvh, split = 0;
  if constexpr (CACHE) {
    int c;
    work_item_cache(blockIdx.x, p.total_blocks, p.n_mblocks, p.batch * p.heads_k, mb, split, c);
    if (p.heavy_first) mb = p.n_mblocks - 1 - mb;
    b = c / p.heads_k;
    kvh = c % p.heads_k;
    hh = kvh * p.group;   // first query head of the group
  } else {
    int id;
    if (!VARLEN ||
        !work_item_kv_rr(blockIdx.x, p.total_blocks, p.n_mblocks, p.group, p.heavy_first != 0, p.span, mb,
                         id))
      work_item(blockIdx.x, p.total_blocks, p.n_mblocks, p.heavy_first != 0, p.span, mb, id);
    hh = id % p.heads_q;
    b = id / p.heads_q;
    kvh = hh / p.group;
  }

  int Sq, Sk, qoff = (int)p.q_offset;
  int64_t q_base, o_base, lse_base, k_base = 0, v_base = 0;
  typedef const __attribute__((address_space(4))) int* table_ptr;
  table_ptr bt_row = nullptr;
  if constexpr (VARLEN) {
    if (guard_failed(p)) return;
    const VarlenSeq sq = nth_longest(p.cu_q, p.cu_k, p.batch, b);
    const int qs = sq.qs, ks = sq.ks;
    b = sq.b;
    Sq = sq.Sq;
    Sk = sq.Sk;
    if (p.seqused_q != nullptr) Sq = max(0, min(Sq, p.seqused_q[b]));
    if (p.seqused_k != nullptr) Sk = max(0, min(Sk, p.seqused_k[b]));
    const int os = p.cu_o != nullptr ? p.cu_o[b] : qs;
    q_base = (int64_t)qs * p.q_ss;
    o_base = (int64_t)os * p.o_ss;
    lse_base = (int64_t)os * p.lse_ss;
    if constexpr (PAGED) {
      if (p.bt_cols > 0) Sk = (int)min((int64_t)Sk, (int64_t)p.bt_cols * p.page_size);
    } else {
      k_base = (int64_t)ks * p.k_ss;
      v_base = (int64_t)ks * p.v_ss;
    }
  } else {
    Sq = p.seqlen_q;
    Sk = p.seqlen_k;
    q_base = (int64_t)b * p.q_sb;
    o_base = (int64_t)b * p.o_sb;
    lse_base = (int64_t)b * p.lse_sb;
    if constexpr (CACHE) {
      int row, lp;
      Sk = cache_keys(p, b, &row, &lp);
      if (p.kv_causal_offset) qoff = Sk - Sq;
      if constexpr (!PAGED) {
        k_base = (int64_t)row * p.k_sb + (int64_t)lp * p.k_ss;
        v_base = (int64_t)row * p.v_sb + (int64_t)lp * p.v_ss;
      }
    } else {
      k_base = (int64_t)b * p.k_sb;
      v_base = (int64_t)b * p.v_sb;
    }
  }
  if constexpr (PAGED) bt_row = (table_ptr)(p.block_table + (int64_t)b * p.bt_stride);
  q_base += (int64_t)hh * p.q_sh;
  o_base += (int64_t)hh * p.o_sh;
  lse_base += (int64_t)hh * p.lse_sh;
  k_base += (int64_t)kvh * p.k_sh;
  v_base += (int64_t)kvh * p.v_sh;

  const int rows = CACHE ? Sq * p.group : Sq;
  auto row_query = [&](int gr) __attribute__((always_inline)) {
    return CACHE ? (int)fdiv((uint32_t)gr, p.fd_group) : gr;
  };
  auto row_head = [&](int gr) __attribute__((always_inline)) {
    return CACHE ? (int)fmod((uint32_t)gr, p.fd_group) : 0;
  };
  // Splits that hold no keys write nothing; split 0 always runs.
  if (CACHE && split > 0 && (int64_t)split * p.split_tiles * BN >= Sk) return;
  const int row0 = mb * BM;
  if (row0 >= rows) return;   // whole workgroup: varlen blocks past this sequence
  const int row_last = min(row0 + BM, rows) - 1;
  const int wrow0 = row0 + 32 * w;
  const int qi = wrow0 + c32;   // this lane's row
  const bool row_valid = qi < rows;
  const bool wave_active = wrow0 <= row_last;
  // Positions fit in 32 bits (the host keeps lengths and offsets below 2^29).
  const int qpos = row_query(qi) + qoff;

  const int wl = p.window_left, wr = p.window_right;
  const bool causal = p.causal != 0;
  int key_hi = Sk - 1;
  if (causal) key_hi = min(key_hi, qpos);
  if (wr >= 0) key_hi = min(key_hi, qpos + wr);
  constexpr int kNoKey = 1 << 30;
  const int key_lo = wl >= 0 ? qpos - wl : -kNoKey;

  // Keys [k_lo, k_hi) any row of the workgroup sees and [f_lo, f_hi) all of
  // its rows see: tiles inside the latter need no mask.
  const int pos_min = row_query(row0) + qoff, pos_max = row_query(row_last) + qoff;
  int k_hi = Sk, f_hi = Sk, k_lo = 0, f_lo = 0;
  if (causal) {
    k_hi = min(k_hi, pos_max + 1);
    f_hi = min(f_hi, pos_min + 1);
  }
  if (wr >= 0) {
    k_hi = min(k_hi, pos_max + wr + 1);
    f_hi = min(f_hi, pos_min + wr + 1);
  }
  if (wl >= 0) {
    k_lo = max(0, pos_min - wl);
    f_lo = max(0, pos_max - wl);
  }
  int t_begin = k_lo / BN;
  int t_end = k_hi > k_lo ? (k_hi + BN - 1) / BN : t_begin;
  if constexpr (CACHE) {   // this split's tiles
    t_begin = max(t_begin, split * p.split_tiles);
    t_end = max(t_begin, min(t_end, (split + 1) * p.split_tiles));
  }
  const int J = t_end - t_begin;
  // Step it works on tile t_end - 1 - it.  Steps [0, n_top) may cut the upper
  // bound, [n_mid, J) the lower one.
  const int n_top = max(0, min(J, t_end - max(f_hi, 0) / BN));
  const int n_mid = max(n_top, min(J, t_end - (f_lo + BN - 1) / BN));

  // ------------------------------------------------------------ tile loads
  // This wave copies rows [16 w, +16) of every tile, 8 per instruction; lane l
  // writes physical chunk l % 8 of row l / 8 of the eight, so it loads the
  // logical chunk that the swizzle puts there.  Paged: the 16 rows lie in one
  // page (page_size % 16 == 0) and offsets count from the first of them.
  auto k_swz = [](int r) __attribute__((always_inline)) { return (r >> 1) & 7; };
  auto v_swz = [](int r) __attribute__((always_inline)) { return 4 * ((r >> 1) & 1); };
  const uint32_t k_row_b = (uint32_t)(p.k_ss * 2);
  const uint32_t v_row_b = (uint32_t)(p.v_ss * 2);
  uint32_t k_off[IPW], v_off[IPW];
#pragma unroll
  for (int i = 0; i < IPW; ++i) {
    const int r = 8 * (IPW * w + i) + (lane >> 3);
    const int rr = PAGED ? r - 8 * IPW * w : r;
    const int pc = lane & 7;
    k_off[i] = (uint32_t)rr * k_row_b + (uint32_t)((pc ^ k_swz(r)) * 16);
    v_off[i] = (uint32_t)rr * v_row_b + (uint32_t)((pc ^ v_swz(r)) * 16);
  }
  const uint32_t k_lds_a = lds_address(k_ring) + IPW * w * 1024;
  const uint32_t v_lds_a = lds_address(v_ring) + IPW * w * 1024;
  const uint16_t* const kg = static_cast<const uint16_t*>(p.k) + k_base;
  const uint16_t* const vg = static_cast<const uint16_t*>(p.v) + v_base;
  const int n0_top = (t_end - 1) * BN;
  const uint16_t* k_next = kg + (int64_t)n0_top * p.k_ss;
  const uint16_t* v_next = vg + (int64_t)n0_top * p.v_ss;
  const int64_t k_step = (int64_t)BN * p.k_ss, v_step = (int64_t)BN * p.v_ss;
  const uint32_t k_full = rows_extent(0, BN, p.k_ss, D);
  const uint32_t v_full = rows_extent(0, BN, p.v_ss, D);
  // Page of this wave's rows of step it's tile, -1 past the keys.
  auto page_of = [&](int it) __attribute__((always_inline)) {
    const int n = (t_end - 1 - it) * BN + 8 * IPW * w;
    return it < J && n < Sk ? bt_row[fdiv((uint32_t)n, p.fd_page)] : -1;
  };
  int page = -1;   // of the next tile to load
  // Loads of step it's tile into ring slot `slot` (called for 0, 1, 2, ... in
  // order).  Only step 0's tile can run past the last key; steps past J get
  // an empty resource: the instructions still retire, which keeps the wait
  // counts uniform.
  auto issue = [&](int it, int slot) __attribute__((always_inline)) {
    u32x4 rk, rv;
    if constexpr (PAGED) {
      const int n = (t_end - 1 - it) * BN + 8 * IPW * w;
      const bool live = page >= 0 && page < p.cache_blocks;
      const int at = live ? (int)fmod((uint32_t)n, p.fd_page) : 0;
      const int left = min(8 * IPW, Sk - n);
      rk = make_rsrc_words(kg + (live ? (int64_t)page * p.k_sb + (int64_t)at * p.k_ss : 0),
                           live ? rows_extent(0, left, p.k_ss, D) : 0u);
      rv = make_rsrc_words(vg + (live ? (int64_t)page * p.v_sb + (int64_t)at * p.v_ss : 0),
                           live ? rows_extent(0, left, p.v_ss, D) : 0u);
    } else {
      rk = make_rsrc_words(k_next, it >= J ? 0u : it > 0 ? k_full : rows_extent(n0_top, Sk, p.k_ss, D));
      rv = make_rsrc_words(v_next, it >= J ? 0u : it > 0 ? v_full : rows_extent(n0_top, Sk, p.v_ss, D));
      k_next -= k_step;
      v_next -= v_step;
    }
#pragma unroll
    for (int i = 0; i < IPW; ++i) buf_load16_lds(rk, k_lds_a + slot * TILEB + i * 1024, k_off[i]);
#pragma unroll
    for (int i = 0; i < IPW; ++i) buf_load16_lds(rv, v_lds_a + slot * TILEB + i * 1024, v_off[i]);
  };
  // Step it's tile sits in slot (it - n_top) mod 3: the unmasked run starts at 0.
  const int slot0 = (NS - n_top % NS) % NS;
  auto slot_at = [&](int it) __attribute__((always_inline)) { return (slot0 + it) % NS; };

  // ------------------------------------------------------------ prologue
  // Q rows by DMA into the slot of step 2 (waves 0 and 1 in its K half, 2 and
  // 3 in its V half), ahead of the tiles of steps 0 and 1.
  u32x4 qreg[NKC];
  {
    uint8_t* const q_st = (w < NW / 2 ? k_ring + w * 4096 : v_ring + (w - NW / 2) * 4096) +
                          slot_at(2) * TILEB;
    static_assert(NW / 2 * 4096 <= TILEB, "Q staging must fit one tile slot");
    const uint16_t* const qg = static_cast<const uint16_t*>(p.q) + q_base;
    const int i0 = row_query(wrow0);
    const u32x4 rq = make_rsrc_words(qg + (int64_t)i0 * p.q_ss,
                                     CACHE ? 0x80000000u : rows_extent(wrow0, Sq, p.q_ss, D));
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = 8 * i + (lane >> 3), gr = wrow0 + r;
      const uint32_t ro =
          CACHE ? (uint32_t)((row_query(gr) - i0) * (int)p.q_ss + row_head(gr) * (int)p.q_sh) * 2
                : (uint32_t)r * (uint32_t)(p.q_ss * 2);
      buf_load16_lds(rq, lds_address(q_st) + i * 1024,
                     CACHE && gr >= rows ? 0xfffffff0u : ro + (uint32_t)(((lane & 7) ^ k_swz(r)) * 16));
    }
    if constexpr (PAGED) page = page_of(0);
    issue(0, slot_at(0));
    if constexpr (PAGED) page = page_of(1);
    issue(1, slot_at(1));
    if constexpr (PAGED) page = page_of(2);
    wait_loads<4 * IPW>();
#pragma unroll
    for (int kc = 0; kc < NKC; ++kc)
      qreg[kc] = *reinterpret_cast<const u32x4*>(q_st + c32 * ROWB + ((2 * kc + g) ^ k_swz(c32)) * 16);
    // The rows are read before the barrier after which the slot is refilled.
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }

  // Per-lane LDS offsets: K rows (A operand of S^T, row kb * 32 + c32, chunk
  // 2 kc + g) and V^T (ds_read_b64_tr_b16: lane j of its 16 lanes reads key
  // row 16 cc + 4 g + j / 4 (+ 8), dims db * 32 + 16 (c32 / 16) + 4 (j % 4)).
  uint32_t k_rd[NKC], v_rd[NDB];
  {
    const int j16 = lane & 15;
    const uint32_t vr = (uint32_t)(4 * g + (j16 >> 2)) * ROWB + (uint32_t)((j16 & 1) * 8);
    const int v_cx = 2 * (c32 >> 4) + ((j16 & 3) >> 1);
#pragma unroll
    for (int kc = 0; kc < NKC; ++kc)
      k_rd[kc] = (uint32_t)c32 * ROWB + ((uint32_t)(2 * kc + g) ^ (uint32_t)k_swz(c32)) * 16;
#pragma unroll
    for (int db = 0; db < NDB; ++db)
      v_rd[db] = vr + ((uint32_t)(4 * db + v_cx) ^ (uint32_t)v_swz(j16 >> 2)) * 16;
  }

  const float sl = p.scale_log2;
  const float slack = kSlack / sl;
  f32x16 acc[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db) acc[db] = f32x16{};
  float l_run = 0.f;   // this lane's partial row sum
  // m_c: the finite max, in raw score units, that P is taken against (every
  // register of cneg holds -m_c); thr: the score above m_c at which it moves,
  // -inf until the row has seen a key.  Boundary tiles may show a row only a
  // few keys, so the slack applies once an unmasked tile has set m_c (the
  // largest P being exactly 1 is worth 1 % of the error to float64).
  float m_c = 0.f, thr = -INFINITY;
  f32x16 cneg = f32x16{};

  // One tile: S^T - m = K Q^T - m, boundary mask, lazy max / O^T rescale,
  // P = exp2(sl (s - m)), O^T += V^T P^T, row sums.
  auto compute = [&](int slot, int n0, auto mask_c) __attribute__((always_inline)) {
    constexpr bool MASK = decltype(mask_c)::value;
    const uint8_t* const Ks = k_ring + slot * TILEB;
    const uint8_t* const Vs = v_ring + slot * TILEB;
    f32x16 s[NKB];
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
      for (int kc = 0; kc < NKC; ++kc) {
        const u32x4 a = *reinterpret_cast<const u32x4*>(Ks + k_rd[kc] + kb * 32 * ROWB);
        s[kb] = T::mfma32(a, qreg[kc], kc == 0 ? cneg : s[kb]);
      }
    __builtin_amdgcn_s_setprio(0);
    if constexpr (MASK) {
      const int hi0 = key_hi - n0 - 4 * g;
      const int lo0 = key_lo - n0 - 4 * g;
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int ko = kb * 32 + 8 * (v >> 2) + (v & 3);
          if (ko > hi0 || ko < lo0) s[kb][v] = -INFINITY;
        }
    }
    float mq[4] = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
#pragma unroll
    for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
      for (int v = 0; v < 16; v += 8)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          mq[q] = fmaxf(fmaxf(mq[q], s[kb][v + 2 * q]), s[kb][v + 2 * q + 1]);
    const float mx = halves_max(fmaxf(fmaxf(mq[0], mq[1]), fmaxf(mq[2], mq[3])));
    const bool raise = mx > thr;
    if (__builtin_amdgcn_ballot_w64(raise)) {
      const float up = raise ? mx : 0.f;
      // (A row's first keys: nothing is accumulated yet, and -mx may be large.)
      const float alpha = raise ? (thr == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(-mx * sl)) : 1.f;
      m_c += up;
      if (MASK ? raise : raise || thr == 0.f) thr = MASK ? 0.f : slack;
      l_run *= alpha;
#pragma unroll
      for (int db = 0; db < NDB; ++db) acc[db] *= alpha;
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb) s[kb] -= up;
#pragma unroll
      for (int v = 0; v < 16; ++v) cneg[v] = -m_c;
    }
    float lq[4] = {0.f, 0.f, 0.f, 0.f};
    u32x4 pb[NCC];
#pragma unroll
    for (int cc = 0; cc < NCC; ++cc) {
      const f32x16& sv = s[cc >> 1];
      const int o8 = (cc & 1) * 8;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float e0 = __builtin_amdgcn_exp2f(sv[o8 + 2 * j] * sl);
        const float e1 = __builtin_amdgcn_exp2f(sv[o8 + 2 * j + 1] * sl);
        pb[cc][j] = T::pack2(e0, e1);
        if (kSumRounded)
          lq[j] = T::sum2(pb[cc][j], lq[j]);
        else
          lq[j] += e0 + e1;
      }
    }
    l_run += (lq[0] + lq[1]) + (lq[2] + lq[3]);
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int cc = 0; cc < NCC; ++cc)
#pragma unroll
      for (int db = 0; db < NDB; ++db) {
        const uint16_t* vp = reinterpret_cast<const uint16_t*>(Vs + v_rd[db] + cc * 16 * ROWB);
        const u32x2 lo = lds_read_tr16(vp);
        const u32x2 hi = lds_read_tr16(vp + 8 * D);
        acc[db] = T::mfma32(u32x4{lo[0], lo[1], hi[0], hi[1]}, pb[cc], acc[db]);
      }
    __builtin_amdgcn_s_setprio(0);
  };

  // ------------------------------------------------------------ main loop
  // Top of step it: this wave's loads of its tile have landed once at most
  // those of step it + 1 are outstanding; the barrier makes everyone's
  // visible, and every wave has its reads of step it - 1, whose slot the loads
  // of step it + 2 refill.
  auto top = [&](int it, int refill) __attribute__((always_inline)) {
    ring_barrier<2 * IPW>();
    issue(it + 2, refill);
  };
  // After a step: the block-table entry the next step's loads need, in flight
  // while this wave waits for the others.
  auto bottom = [&](int it) __attribute__((always_inline)) {
    if constexpr (PAGED) page = page_of(it + 3);
  };
  const int qw_min = row_query(wrow0) + qoff;
  const int qw_max = row_query(min(wrow0 + 31, row_last)) + qoff;
  int it = 0;
#pragma nounroll
  for (int part = 0; part < 2; ++part) {
    const int end = part == 0 ? n_top : J;
    for (; it < end; ++it) {
      top(it, slot_at(it + 2));
      // Tiles no row of this wave sees are skipped.
      const int n0 = (t_end - 1 - it) * BN;
      bool skip = !wave_active;
      if (causal) skip = skip || n0 > qw_max;
      if (wr >= 0) skip = skip || n0 > qw_max + wr;
      if (wl >= 0) skip = skip || n0 + BN - 1 < qw_min - wl;
      if (!skip) compute(slot_at(it), n0, std::true_type{});
      bottom(it);
    }
    if (part == 0) {
      while (it < n_mid) {
        top(it, 2);
        compute(0, 0, std::false_type{});
        bottom(it);
        if (++it >= n_mid) break;
        top(it, 0);
        compute(1, 0, std::false_type{});
        bottom(it);
        if (++it >= n_mid) break;
        top(it, 1);
        compute(2, 0, std::false_type{});
        bottom(it);
        ++it;
      }
    }
  }
  // Every load (including the empty ones past the last tile) has landed and
  // every wave is done reading before the rings become the output staging.
  wait_loads<0>();
  __syncthreads();

  // ------------------------------------------------------------ epilogue
  if (!wave_active) return;
  const float l_tot = halves_sum(l_run);
  const float inv_l = l_tot > 0.f ? 1.f / l_tot : 0.f;
  const float lse_val = l_tot > 0.f ? (m_c * sl + __log2f(l_tot)) * kLn2 : -INFINITY;
  static_assert(NW * stage_part_bytes(NDB) <= Tile::LDS_BYTES &&
                    NW * stage_out_bytes(NDB) <= Tile::LDS_BYTES,
                "output staging must fit the rings");
  if constexpr (CACHE) {
    if (Sk > p.split_tiles * BN) {
      const int64_t prow0 = ((int64_t)split * p.batch + b) * Sq;
      uint8_t* const st = smem_d64 + w * stage_part_bytes(NDB);
      stage_part_write<NDB>(acc, inv_l, st, c32, g);
      const uint8_t* const rd = st + (lane >> 4) * stage_part_pitch(NDB) + (lane & 15) * 16;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const f32x4 val = *reinterpret_cast<const f32x4*>(rd + i * 4 * stage_part_pitch(NDB));
        const int gr = wrow0 + 4 * i + (lane >> 4);
        if (gr < rows) {
          const int64_t prow = (prow0 + row_query(gr)) * p.heads_q + hh + row_head(gr);
          *reinterpret_cast<f32x4*>(p.o_part + prow * D + (lane & 15) * 4) = val;
        }
      }
      if (g == 0 && row_valid)
        p.lse_part[(prow0 + row_query(qi)) * p.heads_q + hh + row_head(qi)] = lse_val;
      return;
    }
    uint16_t* const og = static_cast<uint16_t*>(p.o) + o_base;
    u32x4 out[2 * NDB];
    stage_rows_gather<T, NDB>(acc, inv_l, smem_d64 + w * stage_out_bytes(NDB), c32, g, lane, out);
#pragma unroll
    for (int i = 0; i < 2 * NDB; ++i) {
      const int gr = wrow0 + 8 * i + (lane >> 3);
      if (gr < rows)
        store16(og + (int64_t)row_query(gr) * p.o_ss + (int64_t)row_head(gr) * p.o_sh + (lane & 7) * 8,
                out[i]);
    }
    if (p.lse != nullptr && g == 0 && row_valid)
      p.lse[lse_base + (int64_t)row_query(qi) * p.lse_ss + (int64_t)row_head(qi) * p.lse_sh] = lse_val;
  } else {
    stage_rows_store<T, NDB>(acc, inv_l, smem_d64 + w * stage_out_bytes(NDB), c32, g, lane,
                             static_cast<uint16_t*>(p.o) + o_base + (int64_t)wrow0 * p.o_ss, p.o_ss,
                             Sq - wrow0);
    if (p.lse != nullptr && g == 0 && row_valid) p.lse[lse_base + (int64_t)qi * p.lse_ss] = lse_val;
  }
}

}  // namespace fa
