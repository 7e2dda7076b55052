// Ping-pong FlashAttention-2 prefill forward for gfx950 at head dim 128,
// fp16 / bf16 (dense, cross, varlen, and chunks of queries against a KV cache).
//
// Semantics are those of prefill_kernel (fa_prefill_kernel.h), i.e. the
// reference's dense and varlen forward kernels
// (/root/reference/flash_attn_triton/triton_kernel/attention_kernel.py:424-533,
// :275-372, :27-104).  The schedule is built around two measured properties
// of the CDNA4 SIMD:
//
// * An MFMA issued by one wave and VALU work (exp2, max, pack) issued by
//   another wave on the same SIMD run concurrently; inside one wave only a
//   few VALU instructions hide under each MFMA.
// * The two waves w and w + 4 of a 512-thread workgroup share a SIMD.
//
// So the workgroup's 8 waves form two groups, G0 = waves 0-3 and G1 = waves
// 4-7, which alternate between a GEMM phase and a softmax phase, separated by
// workgroup barriers.  While G0 runs the GEMM phase of key tile j
// (S_j = K_j Q^T and O^T += V_{j-1}^T P_{j-1}: 32 MFMAs per wave), G1 runs the
// softmax of tile j - 1 (VALU only), and the other way round in the next
// phase: each SIMD's matrix core is fed by one of its two waves in every
// phase.
//
// Tiles: a wave owns 32 query rows (row block 2 (w % 4) + w / 4, so both
// groups reach the causal diagonal at the same tile); keys come in tiles of
// 64.  K and V tiles are copied global -> LDS by the buffer loads' LDS mode
// (no VGPR staging): one instruction moves 64 x 16 bytes to 1 KiB of
// consecutive LDS.  Four stages per operand; the loads of K_{j+3} and V_{j+2}
// are issued in the softmax phase of tile j and waited for one softmax phase
// later, two phases before their first use.  Rows past the end of the
// sequence come back as zeros (raw buffer range check), so no load branches.
//
// LDS layout: rows of D = 128 halfs (256 B) without padding; the 16-byte
// chunk c of row r is stored at chunk position c ^ (r & 15) for K and
// c ^ 4 (r & 3) for V, so the K reads of the S^T product (16 rows, one chunk
// column per 16 lanes) and the V^T transpose reads (ds_read_b64_tr_b16, 4 rows
// x 4 chunks per 32 lanes) touch distinct bank groups.
//
// Paged K/V (varlen with a block table, and the paged cache): the 8 rows a
// wave copies of every tile lie in one page (page_size % 8 == 0), so a tile
// load costs the wave one block-table entry, read through the scalar cache
// one tile ahead and shared by K and V, and the loads stay whole-row DMA.
//
// KV-cache mode (kPpCache): the rows of a workgroup are (query, head) pairs of
// one KV head, head fastest, so the query heads of a group share every K/V
// tile, and the keys of a sequence are split into ranges of split_tiles tiles
// (cache_combine_kernel merges them; a sequence that fits one range is written
// directly).  These forms keep fwd_kernel's precision, which they replaced:
// unpre-scaled Q, row sums over the fp32 P, and the running max raised with
// every larger score (slack 0): the largest P of a row is then exactly 1,
// where a stale max rounds it (measured 2.25e-3 against 2.34e-3 relative error
// to float64 in bf16, for 5 % of the time).  What bounds them is the
// GEMM / softmax phase pair, as in the dense form.  Measured on one MI355X,
// causal, bf16, Hq32 Hk8, page 256: 512 queries against 4 caches of 512 to
// 8192 keys 584 + 16 us (fwd_kernel + combine) -> 147 + 12 us; 4 full
// caches of 8192 keys 796 -> 342 us per call.
#pragma once

#include <type_traits>

#include "fa_prefill_kernel.h"

namespace fa {

template <int D>
struct PingPongTile {
  static constexpr int NW = 8;
  static constexpr int NT = 512;
  static constexpr int BM = 256;          // query rows per workgroup (32 per wave)
  static constexpr int BN = 64;           // keys per tile
  static constexpr int NS = 4;            // LDS stages per operand
  static constexpr int ROWB = D * 2;      // bytes per K / V row
  static constexpr int TILEB = BN * ROWB; // bytes per K or V tile
  // Past the K and V rings: 8 KiB per wave of one group for staging Q and
  // output rows (stage_rows_* below).
  static constexpr int STAGE_OFF = 2 * NS * TILEB;
  static constexpr int LDS_BYTES = STAGE_OFF + 4 * 8192;
  static constexpr int RPI = 1024 / ROWB;              // rows per 1-KiB load instruction
  static constexpr int IPW = TILEB / 1024 / NW;        // load instructions per wave per tile
  static_assert(D == 128, "ping-pong tiles are laid out for head dim 128");
  static_assert(IPW * NW * 1024 == TILEB, "tile must split evenly over the waves");
};

// Workgroup barrier that the scheduler may not move instructions across (the
// phase structure depends on every MFMA of a GEMM phase being issued before
// it).  LDS visibility is handled by the kernel's explicit waits.
__device__ inline void pp_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_barrier" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// The launch forms, instantiations of their own so that the dense kernel
// carries none of the others' work-item code: dense / cross, cu_seqlens
// addressing, and a few queries per sequence against a KV cache.
enum { kPpDense = 0, kPpVarlen = 1, kPpCache = 2 };

// Work item of a KV-cache launch: row block mb, key split and KV group
// c = b * heads_k + kvh.  Row blocks vary fastest (the blocks of a KV head
// share its tiles in one L2), the split slowest, so that every sequence's
// full leading splits go out before the short or empty trailing ones.  KV
// groups are dealt round-robin over the 8 XCDs; with 1, 2 or 4 groups each
// takes 8 / n_kv XCDs.
__device__ inline void work_item_cache(int L, int total, int n_mblocks, int n_kv, int& mb,
                                       int& split, int& c) {
  constexpr int kXcds = 8;
  int k = L;
  if (n_kv % kXcds == 0) {
    const int per = n_kv / kXcds;
    k = L / kXcds;
    mb = k % n_mblocks;
    k /= n_mblocks;
    c = (k % per) * kXcds + L % kXcds;
    split = k / per;
  } else if (kXcds % n_kv == 0 && total % kXcds == 0) {
    c = (L % kXcds) % n_kv;
    k = (L / kXcds) * (kXcds / n_kv) + (L % kXcds) / n_kv;
    mb = k % n_mblocks;
    split = k / n_mblocks;
  } else {
    mb = k % n_mblocks;
    k /= n_mblocks;
    c = k % n_kv;
    split = k / n_kv;
  }
}

// Visible keys of sequence b of a KV-cache call, clamped to what the cache and
// the block table hold whatever the device arrays contain; *row is the batched
// cache's row and *pad its left padding.
__device__ inline int cache_keys(const FwdParams& p, int b, int* row, int* pad) {
  int L = p.seqlens_k != nullptr ? p.seqlens_k[b] : p.seqlen_k;
  int lp = 0;
  *row = b;
  if (p.block_table == nullptr) {
    if (p.cache_rows != nullptr) *row = p.cache_rows[b];
    if (p.leftpad != nullptr) lp = max(0, min(p.leftpad[b], p.seqlen_k));
    if (*row < 0 || *row >= p.cache_blocks) L = 0;
  }
  *pad = lp;
  return max(0, min(L, p.seqlen_k - lp));
}

template <class T, int D, int MODE, bool PAGED>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
void prefill_pp_kernel(const FwdParams p) {
  using Tile = PingPongTile<D>;
  constexpr int BM = Tile::BM;
  constexpr int BN = Tile::BN;
  constexpr int NS = Tile::NS;
  constexpr int ROWB = Tile::ROWB;
  constexpr int TILEB = Tile::TILEB;
  constexpr int IPW = Tile::IPW;
  constexpr int RPI = Tile::RPI;
  constexpr int NKC = D / 16;      // 16-dim k-steps of S^T
  constexpr int NDB = D / 32;      // 32-dim blocks of O^T
  constexpr int NKB = BN / 32;     // 32-key blocks per tile
  constexpr int NCC = BN / 16;     // 16-key k-steps of O^T
  constexpr bool VARLEN = MODE == kPpVarlen;
  constexpr bool CACHE = MODE == kPpCache;
  static_assert(!PAGED || MODE != kPpDense, "dense K/V are not paged");
  static_assert(!PAGED || RPI * IPW == 8, "a wave's rows of a tile must be 8 consecutive keys");

  extern __shared__ __attribute__((aligned(1024))) uint8_t smem_pp[];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = w >> 2;             // 0: GEMM first, 1: softmax first
  const int sid = w & 3;
  const int rb = 2 * sid + grp;       // this wave's 32-row block
  const int c32 = lane & 31;
  const int g = lane >> 5;

  // ------------------------------------------------------------ work item
  // Varlen: K/V heads round-robin over the XCDs (ragged sequences load
  // contiguous group ranges unevenly).
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
      work_item(blockIdx.x, p.total_blocks, p.n_mblocks, p.heavy_first != 0, kCausalSpan, mb, id);
    hh = id % p.heads_q;
    b = id / p.heads_q;
    kvh = hh / p.group;
  }

  int Sq, Sk, qoff32 = (int)p.q_offset;
  int64_t q_base, o_base, lse_base, k_base = 0, v_base = 0;
  // Block table of this sequence, in the constant address space: its entries
  // are wave-uniform and go through the scalar cache, off the vector-memory
  // counter the tile loads are waited on with.
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
      if (p.kv_causal_offset) qoff32 = Sk - Sq;
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

  // Rows: query rows of one head, or (cache) the group's heads of query
  // gr / group as rows gr = query * group + head.
  const int rows = CACHE ? Sq * p.group : Sq;
  auto row_query = [&](int gr) __attribute__((always_inline)) {
    return CACHE ? (int)fdiv((uint32_t)gr, p.fd_group) : gr;
  };
  auto row_head = [&](int gr) __attribute__((always_inline)) {
    return CACHE ? (int)fmod((uint32_t)gr, p.fd_group) : 0;
  };
  // Splits that hold no keys write nothing (the combine skips them); split 0
  // always runs, so that an empty sequence still gets its rows.
  if (CACHE && split > 0 && (int64_t)split * p.split_tiles * BN >= Sk) return;

  const int row0 = mb * BM;
  if (row0 >= rows) return;   // whole workgroup: varlen blocks past this sequence
  const int row_last = min(row0 + BM, rows) - 1;

  const int wrow0 = row0 + 32 * rb;
  const int qi = wrow0 + c32;   // this lane's row
  const bool row_valid = qi < rows;
  // Positions fit in 32 bits (the host keeps lengths and offsets below 2^29).
  const int qpos = row_query(qi) + qoff32;
  const int qpos_w_min = row_query(wrow0) + qoff32;
  const int qpos_w_max = row_query(min(wrow0 + 31, row_last)) + qoff32;

  const int wl = p.window_left, wr = p.window_right;
  const bool causal = p.causal != 0;
  int key_hi = Sk - 1;
  if (causal) key_hi = min(key_hi, qpos);
  if (wr >= 0) key_hi = min(key_hi, qpos + wr);
  // key_lo stays above -2^30 so that key - key_lo cannot overflow.
  const int key_lo = wl >= 0 ? max(qpos - wl, -(1 << 30)) : -(1 << 30);

  // Key tiles [t_begin, t_end) any row of the workgroup can see.
  int k_hi = Sk;
  if (causal) k_hi = min(k_hi, row_query(row_last) + qoff32 + 1);
  if (wr >= 0) k_hi = min(k_hi, row_query(row_last) + qoff32 + wr + 1);
  int k_lo = 0;
  if (wl >= 0) k_lo = max(0, row_query(row0) + qoff32 - wl);
  int t_begin = k_lo / BN;
  int t_end = k_hi > k_lo ? (k_hi + BN - 1) / BN : t_begin;
  if constexpr (CACHE) {   // this split's tiles
    t_begin = max(t_begin, split * p.split_tiles);
    t_end = max(t_begin, min(t_end, (split + 1) * p.split_tiles));
  }
  const int J = t_end - t_begin;

  // ------------------------------------------------------------ Q^T in VGPRs
  // fp16: Q is pre-scaled by scale * log2(e) and rounded back to fp16, as the
  // reference's forward kernel does (attention_kernel.py:492-495), so the
  // scores come out of the MFMAs in log2 units.  bf16 keeps Q as given (its
  // 8-bit mantissa would move the log-sum-exp by ~1.5e-3) and scales every
  // score in the softmax; so do the KV-cache and paged forms, whose callers
  // have always had the unrounded Q.
  constexpr bool kPre = std::is_same<T, F16>::value && !CACHE && !PAGED;
  constexpr float kSlack = CACHE || PAGED ? 0.f : kRescaleSlack;
  constexpr bool kSumRounded = T::kSumRounded && !CACHE && !PAGED;
  const uint16_t* qg = static_cast<const uint16_t*>(p.q);
  u32x4 qreg[NKC];
  // This wave's 32 Q rows are staged through LDS with whole-row DMA (rows past
  // the sequence read as zeros): G0 in V stages 2-3, which the V loads first
  // fill in the softmax phases after G0 has read its rows, G1 in the staging
  // area past the rings.
  static_assert(D == 128, "Q staging holds 256-byte rows");
  uint8_t* const q_st = smem_pp + (grp == 0 ? NS * TILEB + 2 * TILEB : Tile::STAGE_OFF) + sid * 8192;
  if constexpr (CACHE) {
    // Row r of the wave is query row_query(wrow0 + r), head row_head: offsets
    // from the wave's first query (the host routes only strides whose offsets
    // stay far below 2^31); rows past the last one lie beyond the resource.
    const int i0 = row_query(wrow0);
    const u32x4 rs = make_rsrc_words(qg + q_base + (int64_t)i0 * p.q_ss, 0x80000000u);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int r = 4 * i + (lane >> 4);
      const int gr = wrow0 + r;
      const uint32_t ro = (uint32_t)((row_query(gr) - i0) * (int)p.q_ss + row_head(gr) * (int)p.q_sh) * 2;
      buf_load16_lds(rs, lds_address(q_st) + i * 1024,
                     gr < rows ? ro + (uint32_t)(((lane & 15) ^ (r & 15)) * 16) : 0xfffffff0u);
    }
  } else {
    stage_rows_load(make_rsrc_words(qg + q_base + (int64_t)wrow0 * p.q_ss,
                                    rows_extent(wrow0, Sq, p.q_ss, D)),
                    lds_address(q_st), (uint32_t)(p.q_ss * 2), lane);
  }
  auto prescale_q = [&]() {
    if constexpr (kPre) {
      const float qs = p.scale_log2;
#pragma unroll
      for (int kc = 0; kc < NKC; ++kc)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const uint32_t w2 = qreg[kc][i];
          qreg[kc][i] = T::pack2(T::to_float((uint16_t)(w2 & 0xffffu)) * qs,
                                 T::to_float((uint16_t)(w2 >> 16)) * qs);
        }
    }
  };

  // ------------------------------------------------------------ tile loads
  // This wave copies rows [RPI * (IPW * w + i), +RPI) of every K and V tile,
  // i < IPW.  Lane l writes physical chunk l % 16 of row RPI*(...) + l / 16,
  // so it loads the logical chunk that the swizzle puts there.
  const uint16_t* kg = static_cast<const uint16_t*>(p.k) + k_base;
  const uint16_t* vg = static_cast<const uint16_t*>(p.v) + v_base;
  const uint32_t k_row_b = (uint32_t)(p.k_ss * 2);
  const uint32_t v_row_b = (uint32_t)(p.v_ss * 2);
  uint32_t k_off[IPW], v_off[IPW];
#pragma unroll
  for (int i = 0; i < IPW; ++i) {
    const int r = RPI * (IPW * w + i) + (lane >> 4);
    const int pc = lane & 15;
    const int rr = PAGED ? r - RPI * IPW * w : r;   // paged: from the wave's first row
    k_off[i] = (uint32_t)rr * k_row_b + (uint32_t)((pc ^ (r & 15)) * 16);
    v_off[i] = (uint32_t)rr * v_row_b + (uint32_t)((pc ^ (4 * (r & 3))) * 16);
  }
  uint8_t* const k_lds = smem_pp;
  uint8_t* const v_lds = smem_pp + NS * TILEB;
  // Tile rel (relative to t_begin) of K / V into its stage.  Tiles past the
  // workgroup's range get an empty resource: the instruction still retires
  // (keeping the wait counts uniform) and writes zeros.
  const uint32_t k_lds_a = lds_address(k_lds) + IPW * w * 1024;
  const uint32_t v_lds_a = lds_address(v_lds) + IPW * w * 1024;
  // Paged: first key of this wave's rows of tile rel, its page (-1 past the
  // last key) and the resource that ends at the last valid one of its 8 rows.
  auto wave_key = [&](int rel) __attribute__((always_inline)) {
    return (t_begin + rel) * BN + RPI * IPW * w;
  };
  auto page_of = [&](int rel) __attribute__((always_inline)) {
    const int n = wave_key(rel);
    return rel < J && n < Sk ? bt_row[fdiv((uint32_t)n, p.fd_page)] : -1;
  };
  auto page_rsrc = [&](const uint16_t* base, int64_t sb, int64_t ss, int rel, int page)
      __attribute__((always_inline)) {
    const int n = wave_key(rel);
    const bool live = page >= 0 && page < p.cache_blocks;   // page -1: no key of this tile is left
    const int slot = live ? (int)fmod((uint32_t)n, p.fd_page) : 0;
    return make_rsrc_words(base + (live ? (int64_t)page * sb + (int64_t)slot * ss : 0),
                           live ? rows_extent(0, min(RPI * IPW, Sk - n), ss, D) : 0u);
  };
  int page_k = -1, page_v = -1;   // pages of the next K and V tile to load
  auto load_k = [&](int rel) {
    const int n0 = (t_begin + rel) * BN;
    const uint32_t ext = rel < J ? rows_extent(n0, Sk, p.k_ss, D) : 0u;
    const u32x4 rs = PAGED ? page_rsrc(kg, p.k_sb, p.k_ss, rel, page_k)
                           : make_rsrc_words(kg + (int64_t)(rel < J ? n0 : 0) * p.k_ss, ext);
    const uint32_t dst = k_lds_a + (rel % NS) * TILEB;
#pragma unroll
    for (int i = 0; i < IPW; ++i) buf_load16_lds(rs, dst + i * 1024, k_off[i]);
  };
  auto load_v = [&](int rel) {
    const int n0 = (t_begin + rel) * BN;
    const uint32_t ext = rel < J ? rows_extent(n0, Sk, p.v_ss, D) : 0u;
    const u32x4 rs = PAGED ? page_rsrc(vg, p.v_sb, p.v_ss, rel, page_v)
                           : make_rsrc_words(vg + (int64_t)(rel < J ? n0 : 0) * p.v_ss, ext);
    const uint32_t dst = v_lds_a + (rel % NS) * TILEB;
#pragma unroll
    for (int i = 0; i < IPW; ++i) buf_load16_lds(rs, dst + i * 1024, v_off[i]);
  };

  // Per-lane LDS read offsets.  K (A operand of S^T, 16 B per lane): key row
  // kb*32 + c32, logical chunk 2 kc + g.  V^T (ds_read_b64_tr_b16, 8 B per
  // lane): lane j of its 16-lane group reads key row 16 cc + 4 g + j / 4 (+8),
  // dims db*32 + 16 (c32 / 16) + 4 (j % 4).
  const int kx = c32 & 15;
  const uint32_t k_rd = (uint32_t)c32 * ROWB;
  const int j16 = lane & 15;
  const uint32_t v_rd = (uint32_t)(4 * g + (j16 >> 2)) * ROWB + (uint32_t)((j16 & 1) * 8);
  const int v_cx = 2 * (c32 >> 4) + ((j16 & 3) >> 1);   // chunk within a 32-dim block
  const int v_sw = j16 >> 2;                             // row & 3 of every V^T read

  auto wave_masks = [&](int rel) {
    const int n0 = (t_begin + rel) * BN, n1 = n0 + BN;
    bool need = n1 > Sk;
    if (causal) need = need || n1 - 1 > qpos_w_min;
    if (wr >= 0) need = need || n1 - 1 > qpos_w_min + wr;
    if (wl >= 0) need = need || n0 < qpos_w_max - wl;
    return need;
  };

  f32x16 acc[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db) acc[db] = f32x16{};
  float m_run = -INFINITY;   // running (possibly stale) max, log2 units
  float l_run = 0.f;         // this lane's partial row sum
  // m_c: the finite max that P is taken against (m_run, or 0 while the row
  // has seen no key).  fp16: the S^T products start from -m_c instead of
  // zero (every lane of cneg holds -m_c of its query row), so they produce
  // the exponent s - m_c of P directly.
  float m_c = 0.f;
  f32x16 cneg = f32x16{};
  const float sl = kPre ? 1.f : p.scale_log2;
  f32x16 s[NKB];
  u32x4 pbuf[NCC];

  // LDS operand reads.  The per-lane swizzled offsets are computed once
  // (8 for K, one per 16-dim step; 4 for V^T, one per 32-dim block), so that
  // a GEMM phase issues no VALU work of its own: it would queue behind the
  // other group's softmax on the shared VALU port and starve the MFMAs.
  uint32_t k_ofs[NKC], v_ofs[NDB];
#pragma unroll
  for (int kc = 0; kc < NKC; ++kc) k_ofs[kc] = k_rd + (((uint32_t)(2 * kc + g)) ^ (uint32_t)kx) * 16;
#pragma unroll
  for (int db = 0; db < NDB; ++db)
    v_ofs[db] = v_rd + ((((uint32_t)db ^ (uint32_t)v_sw) << 2) + (uint32_t)v_cx) * 16;
  auto k_read = [&](const uint8_t* Ks, int kc, int kb) {
    return *reinterpret_cast<const u32x4*>(Ks + k_ofs[kc] + kb * 32 * ROWB);
  };
  auto v_read = [&](const uint8_t* Vs, int db, int cc) {
    const uint16_t* vp = reinterpret_cast<const uint16_t*>(Vs + v_ofs[db] + cc * 16 * ROWB);
    const u32x2 lo = lds_read_tr16(vp);
    const u32x2 hi = lds_read_tr16(vp + 8 * D);
    return u32x4{lo[0], lo[1], hi[0], hi[1]};
  };
  constexpr int NQK = NKC * NKB;   // MFMAs of S^T per tile
  constexpr int NPV = NDB * NCC;   // MFMAs of O^T per tile
  // One GEMM phase: S^T = K Q^T from K stage kst (DO_QK) and O^T += V^T P^T
  // from V stage vst (DO_PV).  The operand reads run ahead of the MFMAs that
  // consume them (8 K reads before the first product, then one read per
  // product; the V^T reads under the second half of S^T), pinned with
  // scheduling groups: left to itself the scheduler keeps two reads in flight
  // and every pair of MFMAs waits out the LDS latency.
  auto gemm = [&](int kst, int vst, auto do_qk_c, auto do_pv_c) {
    constexpr bool DO_QK = decltype(do_qk_c)::value;
    constexpr bool DO_PV = decltype(do_pv_c)::value;
    // The matrix-core phase of the SIMD: its instructions go first.
    __builtin_amdgcn_s_setprio(1);
    const uint8_t* Ks = k_lds + kst * TILEB;
    const uint8_t* Vs = v_lds + vst * TILEB;
    u32x4 ka[DO_QK ? NQK : 1];
    u32x4 va[DO_PV ? NPV : 1];
    if constexpr (DO_QK) {
#pragma unroll
      for (int i = 0; i < NQK; ++i) ka[i] = k_read(Ks, i / NKB, i % NKB);
    }
    if constexpr (DO_PV) {
#pragma unroll
      for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int cc = 0; cc < NCC; ++cc) va[db * NCC + cc] = v_read(Vs, db, cc);
    }
    if constexpr (DO_QK) {
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb) s[kb] = kPre ? cneg : f32x16{};
#pragma unroll
      for (int kc = 0; kc < NKC; ++kc)
#pragma unroll
        for (int kb = 0; kb < NKB; ++kb) s[kb] = T::mfma32(ka[kc * NKB + kb], qreg[kc], s[kb]);
    }
    if constexpr (DO_PV) {
#pragma unroll
      for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int cc = 0; cc < NCC; ++cc)
          acc[db] = T::mfma32(va[db * NCC + cc], pbuf[cc], acc[db]);
    }
    // Scheduling groups (mask 0x100 = LDS read, 0x008 = MFMA): 8 reads up
    // front, then two reads behind every product until all are issued, so
    // the reads run as far ahead as the 15-entry LDS counter allows (a
    // measured 1.46x over one read per product for this phase in isolation).
    constexpr int NRD = (DO_QK ? NQK : 0) + (DO_PV ? 2 * NPV : 0);   // LDS reads
    constexpr int NMF = (DO_QK ? NQK : 0) + (DO_PV ? NPV : 0);       // MFMAs
    constexpr int NPAIR = (NRD - 8 + 1) / 2;
    __builtin_amdgcn_sched_group_barrier(0x100, 8, 0);
#pragma unroll
    for (int i = 0; i < NPAIR; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, NMF - NPAIR, 0);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(0);
  };
  using yes = std::true_type;
  using no = std::false_type;
  // Softmax of the tile starting at key n0 (s: the exponents s - m_c for
  // fp16, the raw scores for bf16): boundary mask, lazy max / O rescale,
  // P = exp2(s - m_c) packed as the B operand of pv, row sums.
  auto softmax_tile = [&](int n0, bool masked) {
    if (masked) {
      // Keys outside [key_lo, key_hi] -> -inf, branch-free: the sign of
      // (key_hi - key) | (key - key_lo) selects the -inf bit pattern.
      const int hi0 = key_hi - n0 - 4 * g;
      const int lo0 = n0 + 4 * g - key_lo;
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb) {
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int ko = kb * 32 + 8 * (v >> 2) + (v & 3);
          const uint32_t m = (uint32_t)(((hi0 - ko) | (lo0 + ko)) >> 31);
          // (A scalar copy first: bit_cast of a vector element reference
          // reads element 0 with this compiler.)
          const float sv = s[kb][v];
          s[kb][v] = __uint_as_float((__float_as_uint(sv) & ~m) | (m & 0xff800000u));
        }
      }
    }
    float mq[4] = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
#pragma unroll
    for (int kb = 0; kb < NKB; ++kb) {
#pragma unroll
      for (int v = 0; v < 16; v += 8) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
          mq[q] = fmaxf(fmaxf(mq[q], s[kb][v + 2 * q]), s[kb][v + 2 * q + 1]);
      }
    }
    const float mq4 = halves_max(fmaxf(fmaxf(mq[0], mq[1]), fmaxf(mq[2], mq[3])));
    const float mx = kPre ? mq4 + m_c : mq4 * sl;
    const bool raise = mx > m_run + kSlack;
    if (__builtin_amdgcn_ballot_w64(raise)) {
      const float m_new = raise ? mx : m_run;
      const float alpha = m_new == m_run ? 1.f : __builtin_amdgcn_exp2f(m_run - m_new);
      l_run *= alpha;
#pragma unroll
      for (int db = 0; db < NDB; ++db) acc[db] *= alpha;
      m_run = m_new;
      const float m_use = m_run == -INFINITY ? 0.f : m_run;
      if constexpr (kPre) {
        const float shift = m_use - m_c;   // 0 on the lanes that did not raise
#pragma unroll
        for (int kb = 0; kb < NKB; ++kb) s[kb] -= shift;
#pragma unroll
        for (int v = 0; v < 16; ++v) cneg[v] = -m_use;
      }
      m_c = m_use;
    }
    // exp2 argument of score x.
    auto expo = [&](float x) { return kPre ? x : fmaf(x, sl, -m_c); };
    float lq[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int cc = 0; cc < NCC; ++cc) {
      const f32x16& sv = s[cc >> 1];
      const int o8 = (cc & 1) * 8;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float e0 = __builtin_amdgcn_exp2f(expo(sv[o8 + 2 * j]));
        const float e1 = __builtin_amdgcn_exp2f(expo(sv[o8 + 2 * j + 1]));
        pbuf[cc][j] = T::pack2(e0, e1);
        if (kSumRounded)
          lq[j] = T::sum2(pbuf[cc][j], lq[j]);
        else
          lq[j] += e0 + e1;
      }
    }
    l_run += (lq[0] + lq[1]) + (lq[2] + lq[3]);
  };

  // ------------------------------------------------------------ prologue
  // Stages 0..NS-2 of K and 0..NS-3 of V; the Q rows retire with them.
  if constexpr (PAGED) {
#pragma unroll
    for (int r = 0; r < NS - 1; ++r) {
      page_k = page_v = page_of(r);
      load_k(r);
      if (r < NS - 2) load_v(r);
    }
    page_k = page_of(NS - 1);   // (page_v: that of tile NS - 2)
  } else {
#pragma unroll
    for (int r = 0; r < NS - 1; ++r) load_k(r);
#pragma unroll
    for (int r = 0; r < NS - 2; ++r) load_v(r);
  }
  __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0)
  pp_barrier();
  stage_rows_read_operand<NKC>(q_st, c32, g, qreg);
  prescale_q();

  // ------------------------------------------------------------ phases
  // Every wave runs the same straight-line sequence GEMM(0), softmax(0),
  // GEMM(1), ..., softmax(J-1), GEMM(J) with a barrier after each step; G1
  // enters one barrier later than G0 (and G0 leaves one later), so in every
  // phase one group multiplies while the other exponentiates.
  // GEMM(j) = S_j (j < J) and O^T += V_{j-1}^T P_{j-1} (j >= 1).  Tiles that
  // hold no visible key for some of this wave's rows are computed anyway with
  // the mask applied: in lockstep, skipping them would not shorten a phase.
  auto softmax_step = [&](int j) {
    load_k(j + NS - 1);
    load_v(j + NS - 2);
    if constexpr (PAGED) {
      page_v = page_k;
      page_k = page_of(j + NS);
    }
    softmax_tile((t_begin + j) * BN, wave_masks(j));
    // The table entry has arrived before the GEMM phase: a scalar load in
    // flight there would turn every counted wait for LDS reads into a full one.
    if constexpr (PAGED) asm volatile("" : "+s"(page_k));
    // This wave's loads from the previous softmax step have landed.
    __builtin_amdgcn_s_waitcnt(0x0f70 | (2 * IPW));
  };
  if (grp == 1) pp_barrier();
  if (J > 0) {
    gemm(0, 0, yes{}, no{});
    pp_barrier();
    softmax_step(0);
    pp_barrier();
    for (int j = 1; j < J; ++j) {
      gemm(j % NS, (j - 1) % NS, yes{}, yes{});
      pp_barrier();
      softmax_step(j);
      pp_barrier();
    }
    gemm(0, (J - 1) % NS, no{}, yes{});
  }
  pp_barrier();
  if (grp == 0) pp_barrier();
  // Every wave's tile loads (including the empty ones past the last tile)
  // have landed before the rings are reused as the output staging area.
  __builtin_amdgcn_s_waitcnt(0x0f70);
  pp_barrier();

  // ------------------------------------------------------------ epilogue
  const float l_tot = halves_sum(l_run);
  const float inv_l = l_tot > 0.f ? 1.f / l_tot : 0.f;
  const float lse_val = l_tot > 0.f ? (m_run + __log2f(l_tot)) * kLn2 : -INFINITY;
  if constexpr (CACHE) {
    uint16_t* const og = static_cast<uint16_t*>(p.o) + o_base;
    if (Sk > p.split_tiles * BN) {
      // One of several splits: the normalized fp32 rows, staged through LDS so
      // that every store covers two whole 512-byte rows of the workspace.
      static_assert(Tile::NW * stage_part_bytes(NDB) <= Tile::LDS_BYTES, "partial rows must fit the LDS");
      const int64_t prow0 = ((int64_t)split * p.batch + b) * Sq;
      uint8_t* const st = smem_pp + w * stage_part_bytes(NDB);
      stage_part_write<NDB>(acc, inv_l, st, c32, g);
      const uint8_t* const rd = st + (lane >> 5) * stage_part_pitch(NDB) + (lane & 31) * 16;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const f32x4 val = *reinterpret_cast<const f32x4*>(rd + i * 2 * stage_part_pitch(NDB));
        const int gr = wrow0 + 2 * i + (lane >> 5);
        if (gr < rows) {
          const int64_t prow = (prow0 + row_query(gr)) * p.heads_q + hh + row_head(gr);
          *reinterpret_cast<f32x4*>(p.o_part + prow * D + (lane & 31) * 4) = val;
        }
      }
      if (g == 0 && row_valid)
        p.lse_part[(prow0 + row_query(qi)) * p.heads_q + hh + row_head(qi)] = lse_val;
      return;
    }
    u32x4 out[8];
    stage_rows_gather<T, NDB>(acc, inv_l, smem_pp + w * kStageOutBytes, c32, g, lane, out);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int gr = wrow0 + 4 * i + (lane >> 4);
      if (gr < rows)
        store16(og + (int64_t)row_query(gr) * p.o_ss + (int64_t)row_head(gr) * p.o_sh + (lane & 15) * 8,
                out[i]);
    }
    if (p.lse != nullptr && g == 0 && row_valid)
      p.lse[lse_base + (int64_t)row_query(qi) * p.lse_ss + (int64_t)row_head(qi) * p.lse_sh] = lse_val;
  } else {
    stage_rows_store<T, NDB>(acc, inv_l, smem_pp + w * kStageOutBytes, c32, g, lane,
                             static_cast<uint16_t*>(p.o) + o_base + (int64_t)wrow0 * p.o_ss,
                             p.o_ss, Sq - wrow0);
    if (p.lse != nullptr && g == 0 && row_valid) p.lse[lse_base + (int64_t)qi * p.lse_ss] = lse_val;
  }
}

// Merge of the key splits of a KV-cache launch: out = sum_s exp(lse_s - lse)
// o_s, lse = log sum_s exp(lse_s) over the splits that hold keys of the row's
// sequence.  Sequences of one split were written by the split kernel.  One
// thread per row and 4 dims, kCacheMergeBatch splits' loads in flight: bound
// by reading the partials.
constexpr int kCacheMergeBatch = 4;
template <class T>
__global__ __launch_bounds__(256) void cache_combine_kernel(const FwdParams p, int D) {
  const int quads = D / 4;
  const int64_t nrows = (int64_t)p.batch * p.seqlen_q * p.heads_q;
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= nrows * quads) return;
  const int64_t row = idx / quads;
  const int qd = (int)(idx % quads);
  const int h = (int)(row % p.heads_q);
  const int i = (int)((row / p.heads_q) % p.seqlen_q);
  const int b = (int)(row / ((int64_t)p.heads_q * p.seqlen_q));
  int crow, pad;
  const int L = cache_keys(p, b, &crow, &pad);
  const int split_keys = p.split_tiles * 64;
  if (L <= split_keys) return;
  const int n = min(p.num_splits, (L + split_keys - 1) / split_keys);
  float m = -INFINITY, tot = 0.f;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int s0 = 0; s0 < n; s0 += kCacheMergeBatch) {
    float ls[kCacheMergeBatch];
    f32x4 o[kCacheMergeBatch];
#pragma unroll
    for (int u = 0; u < kCacheMergeBatch; ++u) {
      const int s = s0 + u;
      ls[u] = s < n ? p.lse_part[(int64_t)s * nrows + row] : -INFINITY;
      o[u] = s < n ? *reinterpret_cast<const f32x4*>(p.o_part + ((int64_t)s * nrows + row) * D + qd * 4)
                   : f32x4{0.f, 0.f, 0.f, 0.f};
    }
    float mb = m;
#pragma unroll
    for (int u = 0; u < kCacheMergeBatch; ++u) mb = fmaxf(mb, ls[u]);
    if (mb == -INFINITY) continue;
    const float rescale = __expf(m - mb);   // m == -inf -> 0
    tot *= rescale;
    acc *= rescale;
#pragma unroll
    for (int u = 0; u < kCacheMergeBatch; ++u) {
      const float wgt = ls[u] == -INFINITY ? 0.f : __expf(ls[u] - mb);
      tot += wgt;
      acc += wgt * o[u];
    }
    m = mb;
  }
  const float inv = tot > 0.f ? 1.f / tot : 0.f;
  uint16_t* orow = static_cast<uint16_t*>(p.o) + (int64_t)b * p.o_sb + (int64_t)i * p.o_ss +
                   (int64_t)h * p.o_sh;
  u32x2 val;
  val[0] = T::pack2(acc[0] * inv, acc[1] * inv);
  val[1] = T::pack2(acc[2] * inv, acc[3] * inv);
  *reinterpret_cast<u32x2*>(orow + qd * 4) = val;
  if (p.lse != nullptr && qd == 0)
    p.lse[(int64_t)b * p.lse_sb + (int64_t)i * p.lse_ss + (int64_t)h * p.lse_sh] =
        tot > 0.f ? m + __logf(tot) : -INFINITY;
}

}  // namespace fa
