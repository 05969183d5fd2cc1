// Flash-attention backward for gfx950: dQ kernel (query-stationary; also produces delta) and dK/dV
// kernel (kv-stationary, all query heads of a GQA group reduced in registers), run in that order.
//
// Semantics: reference kvax/ops/flash_attention_triton.py:373-410 (delta = rowsum(O * dO)),
// :526-617 / :620-871 (dQ: P = exp2(S * scale * log2e - lse), dS = P * (dP - delta),
// dQ = scale * dS K) and :413-523 / :874-1191 (dV = P^T dO, dK = scale * dS^T Q, summed over the
// query heads of each kv head as :1855-1868 does).  P and dS are rounded to the input dtype
// before the second contractions, as in the reference.  Padding tokens take part in nothing and
// get exact-zero gradients.
//
// Layout trick shared with the forward: each contraction is arranged so that the tile produced
// by the first MFMA stage (P or dS in C layout: one column per lane) is directly the B operand
// of the second stage, whose A operand is gathered with transposing LDS reads.
//   dQ kernel:    S^T, dP^T [kv x q]  ->  dQ^T [d x q]  += K^T [d x kv]  dS^T [kv x q]
//   dK/dV kernel: S,   dP   [q x kv]  ->  dV^T [d x kv] += dO^T [d x q]  P  [q x kv]
//                                         dK^T [d x kv] += Q^T  [d x q]  dS [q x kv]
// The dK/dV kernel passes P between the two wavefronts of a pair through LDS (see there); no
// atomics are used and the result is deterministic.
#include "common.h"
#include "fa_common.h"

namespace kvax {
int validate_fa_common(const kvax_fa_args* a);

namespace {

constexpr int kTile = kTileRows;  // rows of the streamed operand per LDS stage

struct BwdParams {
  const char* q;
  const char* k;
  const char* v;
  const char* out;
  const char* dout;
  char* dq;
  char* dk;
  char* dv;
  const float* lse;
  float* delta;
  const int32_t* q_pos;
  const int32_t* q_seg;
  const int32_t* kv_pos;
  const int32_t* kv_seg;
  const int32_t* dq_mask[4];
  const int32_t* dkdv_mask[4];
  int64_t q_sb, q_ss, q_sh;
  int64_t k_sb, k_ss, k_sh;
  int64_t v_sb, v_ss, v_sh;
  int64_t o_sb, o_ss, o_sh;
  int64_t do_sb, do_ss, do_sh;
  int64_t dq_sb, dq_ss, dq_sh;
  int64_t dk_sb, dk_ss, dk_sh;
  int64_t dv_sb, dv_ss, dv_sh;
  int batch, q_len, kv_len, num_heads, num_kv_heads, group;
  int bq, bk;  // backward block sizes: the dQ mask has query blocks of bk and kv blocks of bq
  int n_dq_blocks, n_kv_blocks;
  int num_shards, shard_rows;  // context shards of the query axis the dK/dV mask has rows for, queries per shard
  int num_tiles, total_items;
  int dkdv_f32;  // dK / dV are fp32 tensors (strides still in elements)
  const int4* kv_tiles;  // tile summaries [batch, n_kv_tiles, 2]
  const int4* q_tiles;   // tile summaries [batch, n_q_tiles, 2]
  int n_kv_tiles, n_q_tiles;
  int list_tiles;  // dK/dV kernel: query tiles per chunk of the live-tile bookkeeping
  int32_t* order_ws;           // room for the dK/dV dispatch order and its scratch
  const int32_t* dkdv_order;   // dispatch order of the kv tiles [batch, tiles], or null
  int32_t* dkdv_queue;         // dK/dV kernel: one item counter per XCD, zero at launch
  int dkdv_parts;              // work-groups that share the steps of a dK/dV work item (see plan_dkdv_parts)
  int64_t dk_part, dv_part;    // bytes between the partial results of two parts
  float* parts_ws;             // room for them
  int flags;
  float scale, scale_log2;
  float scale_log2_abs;  // |scale| * log2(e) > 0, used with K negated when the scale is negative
  uint32_t k_sign;       // 0x80008000 when the scale is negative
  // Where the device decides whether work items are shared (see shares_items): the ordering pass's sum and maximum of the
  // items' work, and what dk, dv, their strides and dkdv_f32 are without parts; else null.
  const int32_t* work_stats;
  char *whole_dk, *whole_dv;
  int64_t whole_dk_sb, whole_dk_ss, whole_dk_sh, whole_dv_sb, whole_dv_ss, whole_dv_sh;
  int whole_f32;
  int dq_head_shift;     // log2 of the heads per dQ work-group (see heads_shift)
};

// ---------------------------------------------------------------------------------------------
// Merged range of the streamed axis for a work-group that covers several mask blocks of the
// stationary axis: union of [lower, upper) over the blocks that are its `own`, intersection of [lower_full, upper_full)
// over all of [blk0, blk1], in elements.
// ---------------------------------------------------------------------------------------------
struct Range {
  int lo, hi, flo, fhi;
};

template <class Own>
__device__ __forceinline__ Range merged_range(const int32_t* const mask[4], int64_t base, int blk0,
                                              int blk1, int unit, int limit, Own own) {
  Range r{0x7fffffff, 0, 0, 0x7fffffff};
  for (int blk = blk0; blk <= blk1; blk++) {
    const int l_ = mask[0][base + blk] * unit, u_ = mask[1][base + blk] * unit;
    r.flo = max(r.flo, mask[2][base + blk] * unit);
    r.fhi = min(r.fhi, mask[3][base + blk] * unit);
    if (u_ > l_ && own(blk)) {
      r.lo = min(r.lo, l_);
      r.hi = max(r.hi, u_);
    }
  }
  r.hi = min(r.hi, limit);
  return r;
}

// A stationary MFMA operand.  PINNED, at one wavefront per SIMD: put into the accumulation registers for
// good (left to itself the register allocator parks such fragments there, too, and copies them back for
// their use: 36 copies per 32 MFMAs in the dQ kernel at head_dim 256, 16 per 16 in dK/dV, none at 192).  8k
// tokens, heads 16/4 of 256, without / with it in turn on one machine: dQ 409 / 398 us, dK/dV 828 / 798; dQ
// at 192 equal.  Nothing looks into inline asm for the two wait states between such a write and an MFMA
// that reads it: the loops that do lie behind a barrier.
template <class Vec8, bool PINNED>
__device__ __forceinline__ Vec8 operand(uint4 u) {
  if constexpr (PINNED) {
    uint32_t a0, a1, a2, a3;
    asm volatile("v_accvgpr_write_b32 %0, %1" : "=a"(a0) : "v"(u.x));
    asm volatile("v_accvgpr_write_b32 %0, %1" : "=a"(a1) : "v"(u.y));
    asm volatile("v_accvgpr_write_b32 %0, %1" : "=a"(a2) : "v"(u.z));
    asm volatile("v_accvgpr_write_b32 %0, %1" : "=a"(a3) : "v"(u.w));
    u = make_uint4(a0, a1, a2, a3);
  }
  return __builtin_bit_cast(Vec8, u);
}

// ---------------------------------------------------------------------------------------------
// dQ: one work-group = NW wavefronts x 32 query rows of one (batch, kv head), of one head or the same rows of several
// heads of the group (see heads_shift); streams the live K/V tiles through a ring of LDS stages filled by asynchronous copies.
// ---------------------------------------------------------------------------------------------
template <int D, int DV, int STAGES>
struct DqSmem {
  static constexpr int kTileBytes = kTile * D * 2;  // K tile; swizzled, unpadded
  static constexpr int kIds = kTileBytes + kTile * DV * 2;  // behind the V tile
  static constexpr int kStage = kIds + 2 * kTile * 4;
  static constexpr int kTotal = STAGES * kStage;
};

template <class Tr, int D, int DV, int NW, int WPS, int STAGES>
__global__ __launch_bounds__(NW * 64, WPS) void fa_bwd_dq_kernel(const BwdParams p) {
  using vec8 = typename Tr::vec8;
  using Smem = DqSmem<D, DV, STAGES>;
  constexpr int TQ = NW * 32;
  constexpr int KSTEPS = D / 16, VSTEPS = DV / 16;  // contraction steps of S^T = K Q^T and dP^T = V dO^T
  constexpr int DT = D / 32;
  constexpr int RB = D * 2, RBV = DV * 2;
  // operand address registers (see kNatRegs): at one wavefront per SIMD there is room for one per step
  constexpr int kNat = WPS == 1 ? KSTEPS : kNatRegs<D>, kNatV = WPS == 1 ? VSTEPS : kNatRegs<DV>;
  constexpr int kTr = WPS == 1 ? DT : kTrRegs<D>;
  constexpr int kCopies = async_tile_copies_per_wave<kTile, D, NW>() + async_tile_copies_per_wave<kTile, DV, NW>() + 1;
  static_assert(STAGES == 2 || STAGES == 3, "the loop below keeps STAGES - 1 tiles in flight");
  extern __shared__ __attribute__((aligned(16))) char smem[];

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64), lane = tid % 64;  // wave-uniform on purpose
  const int c = lane % 32, h = lane / 32;

  int group, rank, g;
  const int head_shift = kHeadsPerWorkGroup<D> ? p.dq_head_shift : 0;
  const ItemMap items{p.batch * p.num_kv_heads, p.num_tiles, p.group >> head_shift};
  if (!items.decode(blockIdx.x, group, rank, g)) return;
  const int kv_head = group % p.num_kv_heads;
  const int b = group / p.num_kv_heads;
  const int q_tile = p.num_tiles - 1 - rank;
  // rows of a work-group per head, the wavefront's head among those of the work-group and its block of rows
  const int TR = TQ >> head_shift;
  static_assert(NW == 4 || NW == 8, "wavefronts are dealt to heads by shifts");
  const int wave_shift = (NW == 8 ? 3 : 2) - head_shift;
  const int row_block = kHeadsPerWorkGroup<D> ? wave & ((1 << wave_shift) - 1) : wave;
  const int head0 = kv_head * p.group + (g << head_shift);
  const int head = kHeadsPerWorkGroup<D> ? head0 + (wave >> wave_shift) : head0;
  const int q0 = q_tile * TR;

  const int32_t* kv_seg = p.kv_seg + (int64_t)b * p.kv_len;
  const int32_t* kv_pos = p.kv_pos + (int64_t)b * p.kv_len;
  const char* kbase = p.k + ((int64_t)b * p.k_sb + (int64_t)kv_head * p.k_sh) * 2;
  const char* vbase = p.v + ((int64_t)b * p.v_sb + (int64_t)kv_head * p.v_sh) * 2;

  const int qbs = p.bk, kbs = p.bq;  // the dQ mask swaps the backward block sizes
  const int64_t mbase = (int64_t)b * p.n_dq_blocks;
  // (the full ranges over TQ rows whatever the rows per head: see the forward)
  const int blk0 = q0 / TQ * TQ / qbs, blk1 = min((q0 / TQ * TQ + TQ - 1) / qbs, p.n_dq_blocks - 1);
  int own0 = blk0, own1 = blk1;
  if (head_shift > 0) own0 = q0 / qbs, own1 = (q0 + TR - 1) / qbs;
  const Range r = merged_range(p.dq_mask, mbase, blk0, blk1, kbs, p.kv_len, [&](int blk) { return blk >= own0 && blk <= own1; });
  const int t_lo = r.lo / kTile;
  const int t_hi = r.hi > r.lo ? (r.hi + kTile - 1) / kTile : t_lo;
  const int tf_lo = (r.flo + kTile - 1) / kTile, tf_hi = r.fhi / kTile;

  if (t_hi <= t_lo) {
    // No row of the tile can attend to anything (padding queries): zeros for dQ and delta, and
    // nothing is read.  Whole rows, 16 bytes per lane.
    constexpr int kChunks = D * 2 / 16;
    const int rows = min(TR, p.q_len - q0);
    for (int hd = head0; hd < head0 + (1 << head_shift); hd++) {
      char* dq0 = p.dq + ((int64_t)b * p.dq_sb + (int64_t)hd * p.dq_sh) * 2;
      for (int i = tid; i < rows * kChunks; i += NW * 64)
        *reinterpret_cast<uint4*>(dq0 + (int64_t)(q0 + i / kChunks) * p.dq_ss * 2 + (i % kChunks) * 16) =
            make_uint4(0, 0, 0, 0);
      for (int i = tid; i < rows; i += NW * 64)
        p.delta[((int64_t)b * p.num_heads + hd) * p.q_len + q0 + i] = 0.f;
    }
    return;
  }

  // per-lane query column.  Its ids, its row of the block mask and lse are read without waiting
  // for one another (index 0 stands in for rows beyond the sequence), as are dO, O, Q and the first
  // 64 tile summaries below: one trip to memory for the whole prologue instead of several in a row.
  const int qrow = q0 + row_block * 32 + c;
  const bool in = qrow < p.q_len;
  const int qi = in ? qrow : 0;
  const int qseg_raw = p.q_seg[(int64_t)b * p.q_len + qi];
  const int qpos_raw = p.q_pos[(int64_t)b * p.q_len + qi];
  const int lower_raw = p.dq_mask[0][mbase + qi / qbs], upper_raw = p.dq_mask[1][mbase + qi / qbs];
  const float lse_raw = p.lse[((int64_t)b * p.num_heads + head) * p.q_len + qi];
  const int4* kv_summaries = p.kv_tiles + 2 * (int64_t)b * p.n_kv_tiles;
  const WordSummaries first_word = load_word_summaries(kv_summaries, t_lo >> 6, t_lo, t_hi, lane);
  // dO fragments (B operand of dP^T = V dO^T): lane holds 8 consecutive head-dim elements per
  // step, i.e. half of its row; with the same half of O they give delta = rowsum(O * dO)
  // (reference attn_bwd_preprocess, flash_attention_triton.py:373-410), which is also written out
  // for the dK/dV kernel.
  uint4 draw[VSTEPS];
  // Q fragments (B operand of S^T = K Q^T), requested with dO and O so that their latency does not
  // follow that of the live-tile bookkeeping below
  uint4 qraw[KSTEPS], oraw[VSTEPS];
  {
    // rows beyond the sequence read row 0 and are zeroed afterwards: no load sits behind a branch
    const char* qr = p.q + ((int64_t)b * p.q_sb + (int64_t)head * p.q_sh + (int64_t)qi * p.q_ss) * 2;
    const char* dr = p.dout + ((int64_t)b * p.do_sb + (int64_t)head * p.do_sh + (int64_t)qi * p.do_ss) * 2;
    const char* orow = p.out + ((int64_t)b * p.o_sb + (int64_t)head * p.o_sh + (int64_t)qi * p.o_ss) * 2;
#pragma unroll
    for (int ks = 0; ks < VSTEPS; ks++) {
      draw[ks] = *reinterpret_cast<const uint4*>(dr + (16 * ks + 8 * h) * 2);
      oraw[ks] = *reinterpret_cast<const uint4*>(orow + (16 * ks + 8 * h) * 2);
    }
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ks++) qraw[ks] = make_uint4(0, 0, 0, 0);
    if (t_hi > t_lo) {  // wave-uniform: nothing to attend to, no Q
#pragma unroll
      for (int ks = 0; ks < KSTEPS; ks++) qraw[ks] = *reinterpret_cast<const uint4*>(qr + (16 * ks + 8 * h) * 2);
    }
  }
  float delta_q = 0.f;
  {
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ks++)
      if (!in) qraw[ks] = make_uint4(0, 0, 0, 0);
#pragma unroll
    for (int ks = 0; ks < VSTEPS; ks++) {
      if (!in) draw[ks] = oraw[ks] = make_uint4(0, 0, 0, 0);
      const uint4 o4 = oraw[ks];
      const uint32_t ow[4] = {o4.x, o4.y, o4.z, o4.w}, gw[4] = {draw[ks].x, draw[ks].y, draw[ks].z, draw[ks].w};
#pragma unroll
      for (int w = 0; w < 4; w++) {
        delta_q += Tr::to_float((uint16_t)(ow[w] & 0xffff)) * Tr::to_float((uint16_t)(gw[w] & 0xffff));
        delta_q += Tr::to_float((uint16_t)(ow[w] >> 16)) * Tr::to_float((uint16_t)(gw[w] >> 16));
      }
    }
    delta_q += xor32(delta_q);
    if (in && h == 0) p.delta[((int64_t)b * p.num_heads + head) * p.q_len + qrow] = delta_q;
  }
  const int qseg = in ? qseg_raw : -1;
  const int qpos = in ? qpos_raw : 0;
  int col_lo = 0;
  unsigned col_width = 0;
  float lse_q = 0.f;
  if (in && qseg != -1) {
    col_lo = lower_raw * kbs;
    col_width = (unsigned)max(min(upper_raw * kbs, p.kv_len) - col_lo, 0);
    lse_q = lse_raw;
  }
  TileParts mine[1];
  mine[0] = wave_parts(col_width > 0, qseg, qpos);

  // live kv tiles of [t_lo, t_hi): per-wave bitmaps, compacted into one list
  int* live_count = reinterpret_cast<int*>(smem + Smem::kTotal);
  unsigned long long* live_bits = reinterpret_cast<unsigned long long*>(smem + Smem::kTotal + 16);
  const int word0 = t_lo >> 6;
  const int words = t_hi > t_lo ? ((t_hi - 1) >> 6) - word0 + 1 : 0;
  const uint32_t* live_list = reinterpret_cast<const uint32_t*>(live_bits + NW * (cdiv_dev(p.n_kv_tiles, 64) + 1));
  mark_live_tiles<true, 1>(kv_summaries, mine, t_lo, t_hi, live_bits + wave * words, word0, lane, first_word);
  __syncthreads();
  if (wave == 0)
    compact_live_tiles<NW>(live_bits, words, word0, const_cast<uint32_t*>(live_list), live_count, lane);
  __syncthreads();
  const int n_live = *live_count;

  f32x16 dq[DT];
#pragma unroll
  for (int dt = 0; dt < DT; dt++)
#pragma unroll
    for (int i = 0; i < 16; i++) dq[dt][i] = 0.f;

  if (n_live > 0) {
    vec8 qf[KSTEPS], dof[VSTEPS];
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ks++) qf[ks] = operand<vec8, WPS == 1>(qraw[ks]);
#pragma unroll
    for (int ks = 0; ks < VSTEPS; ks++) dof[ks] = operand<vec8, WPS == 1>(draw[ks]);
    int nat_off[kNat], nat_off_v[kNatV], tr_off[kTr][2];
#pragma unroll
    for (int ks = 0; ks < kNat; ks++) nat_off[ks] = nat_offset<D>(c, ks, h);
#pragma unroll
    for (int ks = 0; ks < kNatV; ks++) nat_off_v[ks] = nat_offset<DV>(c, ks, h);
#pragma unroll
    for (int dt = 0; dt < kTr; dt++) {
      tr_off[dt][0] = tr_offset<D>(lane, dt, 0);
      tr_off[dt][1] = tr_offset<D>(lane, dt, 1);
    }

    const uint32_t smem_addr = (uint32_t)(uintptr_t)smem;
    const int32_t* id_src = (wave & 1) ? kv_pos : kv_seg;
    const AsyncTileCopy<kTile, D, NW> copy_k(p.k_ss * 2, wave, lane);
    const AsyncTileCopy<kTile, DV, NW> copy_v(p.v_ss * 2, wave, lane);
    auto issue = [&](int tile, int stage) {
      const uint32_t base = smem_addr + stage * Smem::kStage;
      copy_k(kbase, tile * kTile, p.kv_len, base);
      copy_v(vbase, tile * kTile, p.kv_len, base + Smem::kTileBytes);
      async_copy_b32(id_src + min(tile * kTile + lane, p.kv_len - 1),
                     __builtin_amdgcn_readfirstlane(base + Smem::kIds + (wave & 1) * (kTile * 4)));
    };

    uint32_t e0 = live_list[0];
    uint32_t e1 = n_live > 1 ? live_list[1] : 0;
    uint32_t e2 = n_live > 2 ? live_list[2] : 0;
    issue(e0 & 0xffffff, 0);
    if (STAGES == 3 && n_live > 1) issue(e1 & 0xffffff, 1);

    int stage = 0;
    for (int i = 0; i < n_live; i++) {
      if (STAGES == 3 && i + 1 < n_live) wait_vmcnt<kCopies>(); else wait_vmcnt<0>();
      __syncthreads();
      const uint32_t e3 = i + 3 < n_live ? live_list[i + 3] : 0;
      if (STAGES == 3) {
        if (i + 2 < n_live) issue(e2 & 0xffffff, stage >= 1 ? stage - 1 : STAGES - 1);  // (stage + 2) % 3
      } else {
        if (i + 1 < n_live) issue(e1 & 0xffffff, stage ^ 1);
      }
      const int t = e0 & 0xffffff;

      if ((e0 >> (24 + wave)) & 1) {
        const int kv0 = t * kTile;
        const char* ktile = smem + stage * Smem::kStage;
        const char* vtile = ktile + Smem::kTileBytes;
        const int32_t* ids = reinterpret_cast<const int32_t*>(ktile + Smem::kIds);
        const bool full = t >= tf_lo && t < tf_hi;

#pragma unroll 1
        for (int kt = 0; kt < 2; kt++) {
          // S^T = K Q^T and dP^T = V dO^T for 32 kv rows: 16 MFMAs, operand reads four ahead
          f32x16 s, dp;
#pragma unroll
          for (int i2 = 0; i2 < 16; i2++) s[i2] = 0.f, dp[i2] = 0.f;
          // Fenced above head_dim 128, see the dK/dV kernel: at 192 with 128 178 -> 171 us on 2 x 4k tokens, 16
          // heads.  At 128 the scheduling groups are heeded well enough and the freedom they leave is better:
          // 1484 us on 32k tokens, heads 32/8, against 1508 fenced.
          if constexpr (D > 128) {
            constexpr int N = KSTEPS + VSTEPS, kAheadOps = WPS == 2 && D > 128 ? 3 : 4;
            vec8 op[N];
            // operand i: K and V rows in turn while there are both, then K rows
            auto is_v = [](int i) { return i < 2 * VSTEPS && i % 2 == 1; };
            auto step = [](int i) { return i < 2 * VSTEPS ? i / 2 : i - VSTEPS; };
            auto read = [&](int i) {
              const int ks = step(i);
              return is_v(i) ? *reinterpret_cast<const vec8*>(vtile + 32 * kt * RBV + nat_off_v[ks % kNatV] + ks / kNatV * kGroupBytes<DV>)
                             : *reinterpret_cast<const vec8*>(ktile + 32 * kt * RB + nat_off[ks % kNat] + ks / kNat * kGroupBytes<D>);
            };
#pragma unroll
            for (int i = 0; i < kAheadOps; i++) op[i] = read(i);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < N; i++) {
              if (is_v(i)) dp = Tr::mfma(op[i], dof[step(i)], dp);
              else s = Tr::mfma(op[i], qf[step(i)], s);
              if (i + kAheadOps < N) op[i + kAheadOps] = read(i + kAheadOps);
              __builtin_amdgcn_sched_barrier(0);
            }
          } else {
#pragma unroll
            for (int ks = 0; ks < KSTEPS; ks++) {
              s = Tr::mfma(*reinterpret_cast<const vec8*>(ktile + 32 * kt * RB + nat_off[ks]), qf[ks], s);
              dp = Tr::mfma(*reinterpret_cast<const vec8*>(vtile + 32 * kt * RBV + nat_off_v[ks]), dof[ks], dp);
            }
            __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
            for (int i2 = 0; i2 < KSTEPS + VSTEPS - 4; i2++) {
              __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
              __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            }
            __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);
          }
          // K^T operands of this block's dQ update, requested before the element-wise work
          // (with two wavefronts per SIMD above head_dim 128 there are no registers to do that in)
          constexpr bool kLean = WPS == 2 && D > 128;
          vec8 ta[DT];
          auto read_kt = [&](int dt, int row0) {
            return tr_read_a_swz<Tr>(ktile + row0 * RB + dt / kTr * kGroupBytes<D>, tr_off[dt % kTr][0], tr_off[dt % kTr][1]);
          };
          if (!kLean) {
#pragma unroll
            for (int dt = 0; dt < DT; dt++) ta[dt] = read_kt(dt, 32 * kt);
          }
#pragma unroll
          for (int i2 = 0; i2 < 16; i2++) s[i2] = fast_exp2(__builtin_fmaf(s[i2], p.scale_log2, -lse_q));
          if (!full)
            mask_c_tile<true>(s, ids, ids + kTile, 32 * kt, kv0, h, qseg, qpos, col_lo, col_width, 0.f);
#pragma unroll
          for (int i2 = 0; i2 < 16; i2++) s[i2] *= dp[i2] - delta_q;
          // dQ^T += K^T dS^T
#pragma unroll
          for (int st = 0; st < 2; st++) {
            const vec8 dsb = pack8<Tr>(s[8 * st + 0], s[8 * st + 1], s[8 * st + 2], s[8 * st + 3],
                                       s[8 * st + 4], s[8 * st + 5], s[8 * st + 6], s[8 * st + 7]);
            if (kLean) {
#pragma unroll
              for (int dt = 0; dt < DT; dt++) dq[dt] = Tr::mfma(read_kt(dt, 32 * kt + 16 * st), dsb, dq[dt]);
              continue;
            }
            vec8 tb[DT];  // second half's operands, requested before the first half's MFMAs
            if (st == 0) {
#pragma unroll
              for (int dt = 0; dt < DT; dt++)
                tb[dt] = read_kt(dt, 32 * kt + 16);
            }
#pragma unroll
            for (int dt = 0; dt < DT; dt++) dq[dt] = Tr::mfma(ta[dt], dsb, dq[dt]);
            if (st == 0) {
#pragma unroll
              for (int dt = 0; dt < DT; dt++) ta[dt] = tb[dt];
            }
          }
        }
      }
      e0 = e1, e1 = e2, e2 = e3;
      stage = stage == STAGES - 1 ? 0 : stage + 1;
    }
  }

  {
    // Rows that attend to nothing (padding) get exact zeros.  Their accumulator is not zero when the
    // block mask declares padding-against-padding blocks mask-free (masks built without skipping
    // padding): the element mask, which is what excludes them, is not applied there.
    // The rows leave through LDS (each wavefront its own part of the tile space, which is done with)
    // as whole rows, 16 bytes per lane, instead of 8-byte pieces of 32 rows per store; rows are
    // swizzled by the row index against bank conflicts.
    const bool dead = col_width == 0;
    __syncthreads();  // every wavefront has read its last tile
    constexpr int PC = NW * 32 * D * 2 <= Smem::kTotal ? D : 64;  // columns per pass
    static_assert(NW * 32 * PC * 2 <= Smem::kTotal, "a wavefront's part of the tile space");
    constexpr int kRowBytes = PC * 2, kChunks = kRowBytes / 16;
    constexpr int kSwz = kChunks % 16 == 0 ? kChunks - 1 : 7;  // chunks are permuted within a power of two of them
    char* stage = smem + wave * (32 * kRowBytes);
    char* mine = stage + c * kRowBytes;
    char* dq0 = p.dq + ((int64_t)b * p.dq_sb + (int64_t)head * p.dq_sh) * 2;
#pragma unroll
    for (int pass = 0; pass < D / PC; pass++) {
#pragma unroll
      for (int dt = 0; dt < PC / 32; dt++)
#pragma unroll
        for (int g4 = 0; g4 < 4; g4++) {
          const f32x16& a = dq[pass * (PC / 32) + dt];
          uint2 u;
          u.x = Tr::pack2(a[4 * g4 + 0] * p.scale, a[4 * g4 + 1] * p.scale);
          u.y = Tr::pack2(a[4 * g4 + 2] * p.scale, a[4 * g4 + 3] * p.scale);
          if (dead) u = make_uint2(0, 0);
          *reinterpret_cast<uint2*>(mine + (((4 * dt + g4) ^ (c & kSwz)) * 16) + 8 * h) = u;
        }
#pragma unroll
      for (int i = 0; i < 32 * kChunks; i += 64) {
        const int row = (i + lane) / kChunks, chunk = (i + lane) % kChunks;
        const uint4 v = *reinterpret_cast<const uint4*>(stage + row * kRowBytes + ((chunk ^ (row & kSwz)) * 16));
        const int qr = q0 + row_block * 32 + row;
        if (qr < p.q_len) *reinterpret_cast<uint4*>(dq0 + (int64_t)qr * p.dq_ss * 2 + pass * kRowBytes + chunk * 16) = v;
      }
    }
  }
}

// ---------------------------------------------------------------------------------------------
// dK/dV: one work-group = 128 kv rows of one (batch, kv head), 8 wavefronts in 4 pairs.  Both
// wavefronts of a pair own the same 32 kv rows and share a SIMD; they split the work by role:
//   P wave, tile t:  S = Q K^T,  P = exp2(S * c - lse) -> LDS,  dV^T += dO^T P
//   S wave, tile t:  dS = P * (dP - delta) and dK^T += Q^T dS of tile t - 1 (P from LDS, dP kept
//                    in registers), then dP = dO V^T of tile t
// so that each holds one accumulator tile set and one fragment set (K or V) - half the registers
// of doing both, which is what lets two wavefronts run per SIMD.  The S wave running one tile
// behind means one barrier per tile, and at any time one wavefront of the pair has element-wise
// work while the other has MFMAs.  The work-group streams the live Q / dO tiles of every query
// head of the group; Q tiles stay one step longer than dO tiles, hence separate rings.
// ---------------------------------------------------------------------------------------------
// Shape of a dK/dV work-group per head_dim.  Up to 192 it is 8 wavefronts (4 role pairs, 128 kv rows) at
// two per SIMD, stepping through 64-row query tiles up to 128.  Above, the Q / dO rings and the scores of
// a step only fit beside the accumulators with 32-row steps: a 64-row tile of the live list is then taken
// as two steps.  At 256 a wavefront's fragments and accumulators need more than half a SIMD's registers,
// so it is 4 wavefronts (2 pairs, 64 kv rows) at one per SIMD.  (Eight at 256 spill 8 registers in the
// step: 16k tokens, heads 16/4 3.56 against 2.04 ms; four at 192 with 128 for the values, 2 x 4k tokens,
// 16 heads: 380 against 244 us.)
template <int D>
struct DkdvCfg {
  static constexpr int kPairs = D > 192 ? 2 : 4;
  static constexpr int kStepRows = D > 128 ? 32 : 64;  // query rows per step (and LDS stage)
  static constexpr int kWps = kPairs == 2 ? 1 : 2;     // wavefronts per SIMD
  static constexpr int kWaves = 2 * kPairs;
  static constexpr int kKvRows = 32 * kPairs;          // kv rows per work-group
  static constexpr int kUnits = kStepRows / 32;        // 32-row MFMA units per step
  static constexpr int kSub = kTile / kStepRows;       // steps per 64-row tile of the live list
};
inline int dkdv_kv_rows(int head_dim) { return head_dim > 192 ? 64 : 128; }

// Whether two work-groups should share each of 257 to 512 items depends on the documents, so the device decides, from the
// work the ordering pass has counted: where the longest item is 15 % and 40 steps longer than a compute unit's share of the
// work.  A step is a live 64-row query tile of one head here and in plan_dkdv_parts (the kernel takes it as two above
// head_dim 128).  us of the dK/dV kernel and the sum in a training pass, items whole -> as decided: 8k tokens in documents of about 2k,
// heads 32/8 of 64 531 -> 373, of 128 664 -> 570, of 192 with 128 806 -> 720, 16/4 of 256 (longest item 232 steps, share 178) 803 ->
// 638; 4 x 4k in documents of 1k, 16/4 of 128, 452 -> 388; 16k in documents of 3k, 8/2 of 256, 1243 -> 878.  Left whole (whole / in
// two parts, the kernel alone on a faster machine): one document of 8k, 16/4 of 256, 1278 / 1327; of 16k, 8/2, 2564 / 2633; without
// the limit of 40 steps 4k in documents of 1k, 16/16 of 192 with 128, 112 / 181, and 2 x 2k in documents of 300, 16/16 of 128,
// 75 / 134.  Deciding against it costs 5 to 6 us of backwards of 100 us (16k in documents of 64, 8/4 of 64) and more, mostly a sum kernel
// that finds nothing to add: only where an item can have 160 steps.
// stats: sum and maximum of the items' work (in tiles, the same for every kv head and query head)
__device__ __forceinline__ bool shares_items(const int32_t* stats, int num_kv_heads, int group) {
  const int64_t longest = (int64_t)stats[1] * group * kNumCus, share = (int64_t)stats[0] * num_kv_heads * group;
  return longest * 20 > share * 23 && longest - share > 40 * kNumCus;
}

template <int D, int DV>
struct DkdvSmem {
  using Cfg = DkdvCfg<D>;
  static constexpr int kQTileBytes = Cfg::kStepRows * D * 2;  // swizzled, unpadded
  static constexpr int kDoTileBytes = Cfg::kStepRows * DV * 2;
  // lse, delta, seg, pos: 64 entries each whatever the step size (a wave-wide copy brings 64)
  static constexpr int kRowData = 4 * kTile * 4;
  static constexpr int kQStages = 4, kDoStages = 3;
  static constexpr int kQ = 0;
  static constexpr int kDo = kQ + kQStages * kQTileBytes;
  static constexpr int kRows = kDo + kDoStages * kDoTileBytes;
  static constexpr int kExchange = kRows + kQStages * kRowData;
  // per pair two slots of P (one kStepRows x 32 tile, 16 bits per element): written for step s while
  // the slot of step s - 1 is read
  static constexpr int kSlotBytes = Cfg::kUnits * 2 * 1024;
  static constexpr int kTotal = kExchange + Cfg::kPairs * 2 * kSlotBytes;
};

// DECIDES: the device decides whether the items are shared (p.work_stats; a kernel of its own, because what it adds costs
// the one at head_dim 128 two more spilled registers and 1.5 to 2 %).
template <class Tr, int D, int DV, bool DECIDES>
__global__ __launch_bounds__(DkdvCfg<D>::kWaves * 64, DkdvCfg<D>::kWps) void fa_bwd_dkdv_kernel(const BwdParams p) {
  using vec8 = typename Tr::vec8;
  using Smem = DkdvSmem<D, DV>;
  using Cfg = DkdvCfg<D>;
  constexpr int NW = Cfg::kWaves;
  constexpr int NP = Cfg::kPairs;
  constexpr int TKV = Cfg::kKvRows;
  constexpr int SR = Cfg::kStepRows;
  constexpr int UNITS = Cfg::kUnits;
  constexpr int SUB = Cfg::kSub;
  static_assert(DV <= D, "the arrays below are sized by the larger head_dim");
  constexpr int KSTEPS = D / 16, VSTEPS = DV / 16;  // contraction steps of S = Q K^T and dP = dO V^T
  constexpr int DT = D / 32, DTV = DV / 32;         // 32-row tiles of dK^T and dV^T
  constexpr int RB = D * 2, RBV = DV * 2;
  // only the P waves issue tile copies: they are the ones with slack before the barrier.  Each
  // also copies its share of the four row-data arrays.
  constexpr int kRowCopies = 4 / NP;
  constexpr int kCopies = async_tile_copies_per_wave<SR, D, NP>() + async_tile_copies_per_wave<SR, DV, NP>() + kRowCopies;
  extern __shared__ __attribute__((aligned(16))) char smem[];

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64), lane = tid % 64;  // wave-uniform on purpose
  const int c = lane % 32, h = lane / 32;
  const int pair = wave % NP;
  const bool p_wave = wave < NP;  // role, wave-uniform

  // The launch is one work-group per compute unit, and each takes work items (128 kv rows of one
  // batch row and kv head) from the queues (see ItemQueue) until none is left.  The ticket for the
  // next item is drawn when the current one's step loop has ended, so that its latency hides behind
  // the final stores and an item is never held back by a long one.
  const bool whole = DECIDES && !shares_items(p.work_stats, p.num_kv_heads, p.group);
  auto parts = [&] { return whole ? 1 : p.dkdv_parts; };
  const ItemMap items{p.batch * p.num_kv_heads, p.num_tiles, parts()};
  ItemQueue work{p.dkdv_queue, DECIDES ? items.grid() : p.total_items, (int)(blockIdx.x % 8)};  // thread 0's
  auto dkdv_f32 = [&] { return whole ? p.whole_f32 : p.dkdv_f32; };
  int* next_item = reinterpret_cast<int*>(smem + Smem::kTotal) + 1;
  if (tid == 0) *next_item = work.resolve(work.draw());
  __syncthreads();
  for (int item = *next_item; item >= 0; item = *next_item) {
  __syncthreads();  // every wavefront has read next_item
  int ticket = 0;
  // kv tiles in the computed dispatch order (without one: early tiles first, which see the most
  // queries under a causal mask)
  int group, rank, member;  // member: which part of the item's steps
  if (items.decode(item, group, rank, member)) {
  char* const dk_out = whole ? p.whole_dk : p.dk + member * p.dk_part;
  char* const dv_out = whole ? p.whole_dv : p.dv + member * p.dv_part;
  const int kv_head = group % p.num_kv_heads;
  const int b = group / p.num_kv_heads;
  const int entry = p.dkdv_order ? p.dkdv_order[(int64_t)b * p.num_tiles + rank] : rank;
  const int kv_tile = entry & (kDeadItem - 1);
  const int k0 = kv_tile * TKV;
  if (entry & kDeadItem) {
    // no query tile can interact with these kv rows (known from the ordering pass): zeros, no bookkeeping
    if (tid == 0) ticket = work.draw();
    const int esize = dkdv_f32() ? 4 : 2;
    const int rows = min(TKV, p.kv_len - k0);
    auto zero_rows = [&](char* out, int64_t sb, int64_t sh, int64_t ss, int columns) {
      const int chunks = columns * esize / 16;
      for (int i = tid; i < rows * chunks; i += NW * 64)
        *reinterpret_cast<uint4*>(out + ((int64_t)b * sb + (int64_t)kv_head * sh + (int64_t)(k0 + i / chunks) * ss) * esize +
                                  (i % chunks) * 16) = make_uint4(0, 0, 0, 0);
    };
    if (whole) {
      zero_rows(dk_out, p.whole_dk_sb, p.whole_dk_sh, p.whole_dk_ss, D);
      zero_rows(dv_out, p.whole_dv_sb, p.whole_dv_sh, p.whole_dv_ss, DV);
    } else {
      zero_rows(dk_out, p.dk_sb, p.dk_sh, p.dk_ss, D);
      zero_rows(dv_out, p.dv_sb, p.dv_sh, p.dv_ss, DV);
    }
  } else {

  const int kbs = p.bk, qbs = p.bq;
  // per-lane kv column (the same for both wavefronts of a pair)
  const int kvcol = k0 + pair * 32 + c;
  const bool in = kvcol < p.kv_len;
  const int kvseg = in ? p.kv_seg[(int64_t)b * p.kv_len + kvcol] : -1;
  const int kvpos = in ? p.kv_pos[(int64_t)b * p.kv_len + kvcol] : 0;
  TileParts mine[1];
  mine[0] = wave_parts(kvseg != -1, kvseg, kvpos);
  bool dead = true;  // the lane's key is attended by no query of any shard

  f32x16 acc[DT];  // dV^T (P wave) or dK^T (S wave): rows = head dim, columns = the lane's kv row
#pragma unroll
  for (int dt = 0; dt < DT; dt++)
#pragma unroll
    for (int i = 0; i < 16; i++) acc[dt][i] = 0.f;

  // The query range is walked in chunks of at most p.list_tiles tiles, the number whose live-tile
  // bookkeeping fits in the LDS left over (one chunk unless the query sequence is very long).
  int* live_count = reinterpret_cast<int*>(smem + Smem::kTotal);
  unsigned long long* live_bits = reinterpret_cast<unsigned long long*>(smem + Smem::kTotal + 16);
  const uint32_t* live_list = reinterpret_cast<const uint32_t*>(live_bits + NW * (cdiv_dev(p.list_tiles, 64) + 1));
  // Under context parallelism the mask has one row per contiguous shard of the query axis, with
  // shard-local bounds; the shards are walked one after another with the accumulators kept: eight
  // shards of 8k queries x 64k keys (32/8 heads) as one launch instead of eight that leave fp32
  // results to be added (2.1 ms of adds, and 17 GB written and read by them), step 24.8 -> 19.1 ms.
  for (int shard = 0; shard < p.num_shards; shard++) {
  const int q_first = shard * p.shard_rows;
  const int64_t mbase = ((int64_t)b * p.num_shards + shard) * p.n_kv_blocks;
  const Range r = merged_range(p.dkdv_mask, mbase, k0 / kbs,
                               min((k0 + TKV - 1) / kbs, p.n_kv_blocks - 1), qbs, p.shard_rows, [](int) { return true; });
  if (r.hi <= r.lo) continue;
  const int t_lo = (q_first + r.lo) / kTile;
  const int t_hi = (q_first + r.hi + kTile - 1) / kTile;
  const int tf_lo = (q_first + r.flo + kTile - 1) / kTile, tf_hi = (q_first + r.fhi) / kTile;
  int col_lo = 0;
  unsigned col_width = 0;
  if (in && kvseg != -1) {
    const int first = p.dkdv_mask[0][mbase + kvcol / kbs] * qbs;
    // queries at or beyond the end never count (their LDS rows hold a copy of the last row)
    col_width = (unsigned)max(min(p.dkdv_mask[1][mbase + kvcol / kbs] * qbs, p.shard_rows) - first, 0);
    col_lo = q_first + first;
  }
  dead &= col_width == 0;
  for (int c_lo = t_lo; c_lo < t_hi; c_lo += p.list_tiles) {
  const int c_hi = min(c_lo + p.list_tiles, t_hi);
  // live query tiles of [c_lo, c_hi) (the same for every head of the group; both wavefronts of a
  // pair mark the same tiles)
  const int word0 = c_lo >> 6;
  const int words = ((c_hi - 1) >> 6) - word0 + 1;
  const int4* q_summaries = p.q_tiles + 2 * (int64_t)b * p.n_q_tiles;
  mark_live_tiles<false, 1>(q_summaries, mine, c_lo, c_hi, live_bits + wave * words, word0, lane,
                            load_word_summaries(q_summaries, word0, c_lo, c_hi, lane));
  __syncthreads();
  if (wave == 0)
    // highest query tile first: every kv work-group of a document ends on the document's last query
    // tiles, so walking backwards the work-groups that run together stream the same Q/dO tiles at
    // the same time (they start at different tiles when walking forwards) and share them in L2
    compact_live_tiles<NW, true>(live_bits, words, word0, const_cast<uint32_t*>(live_list), live_count, lane);
  __syncthreads();
  const int n_live = *live_count;
  // every head of the group walks the same list; this part's share of the (head, list entry) pairs
  // (the divisions are a microsecond of an item: 16 rows of 1k tokens, 16 heads of 64, 184 -> 181 us without)
  int pair_lo = 0, pair_hi = n_live * p.group, first_head = 0;
  if (parts() > 1) {
    pair_lo = (int)((int64_t)(n_live * p.group) * member / parts());
    pair_hi = (int)((int64_t)(n_live * p.group) * (member + 1) / parts());
    first_head = n_live ? pair_lo / n_live : 0;
  }
  const int steps = (pair_hi - pair_lo) * SUB;

  if (steps > 0) {
    const int first_li = pair_lo - first_head * n_live;
    // stationary fragments: K (negated when the scale is negative) for the P wave, V for the S wave
    // (VSTEPS of them)
    vec8 frag[KSTEPS];
    {
      const char* base = p_wave ? p.k + ((int64_t)b * p.k_sb + (int64_t)kv_head * p.k_sh + (int64_t)(in ? kvcol : 0) * p.k_ss) * 2
                                : p.v + ((int64_t)b * p.v_sb + (int64_t)kv_head * p.v_sh + (int64_t)(in ? kvcol : 0) * p.v_ss) * 2;
      const uint32_t sign = p_wave ? p.k_sign : 0u;
#pragma unroll
      for (int ks = 0; ks < KSTEPS; ks++) {
        uint4 u = make_uint4(0, 0, 0, 0);
        if (in && (ks < VSTEPS || p_wave)) u = *reinterpret_cast<const uint4*>(base + (16 * ks + 8 * h) * 2);
        u.x ^= sign, u.y ^= sign, u.z ^= sign, u.w ^= sign;
        frag[ks] = operand<vec8, Cfg::kWps == 1>(u);
      }
    }
    // Operand addresses.  The P wave reads rows of Q and columns of dO, the S wave rows of dO and
    // columns of Q; with value head_dim of its own each role has its own pattern in the same registers.
    // (At one wavefront per SIMD there is room for one register per step: 16k tokens at head_dim 256 2.04
    // against 2.32 ms with shared ones.)
    constexpr bool kShared = Cfg::kWps == 2;
    constexpr int kNatQ = kShared ? kNatRegs<D> : KSTEPS, kNatDo = kShared ? kNatRegs<DV> : VSTEPS;
    constexpr int kTrQ = kShared ? kTrRegs<D> : DT, kTrDo = kShared ? kTrRegs<DV> : DTV;
    constexpr int kNat = kNatQ > kNatDo ? kNatQ : kNatDo, kTr = kTrQ > kTrDo ? kTrQ : kTrDo;
    int nat_off[kNat], tr_off[kTr][2];
#pragma unroll
    for (int ks = 0; ks < kNat; ks++)
      nat_off[ks] = D == DV || p_wave ? nat_offset<D>(c, ks, h) : nat_offset<DV>(c, ks, h);
#pragma unroll
    for (int dt = 0; dt < kTr; dt++)
#pragma unroll
      for (int half = 0; half < 2; half++)
        tr_off[dt][half] = D == DV || !p_wave ? tr_offset<D>(lane, dt, half) : tr_offset<DV>(lane, dt, half);
    // columns [32 dt, +32) of 16 rows of a Q tile (S wave) or a dO tile (P wave), transposed
    auto read_q_t = [&](const char* rows16, int dt) {
      constexpr int n = kTrQ;
      return tr_read_a_swz<Tr>(rows16 + dt / n * kGroupBytes<D>, tr_off[dt % n][0], tr_off[dt % n][1]);
    };
    auto read_do_t = [&](const char* rows16, int dt) {
      constexpr int n = kTrDo;
      return tr_read_a_swz<Tr>(rows16 + dt / n * kGroupBytes<DV>, tr_off[dt % n][0], tr_off[dt % n][1]);
    };

    const uint32_t smem_addr = (uint32_t)(uintptr_t)smem;
    const AsyncTileCopy<SR, D, NP> copy_q(p.q_ss * 2, pair, lane);
    const AsyncTileCopy<SR, DV, NP> copy_do(p.do_ss * 2, pair, lane);
    // Steps go through the list entries of one head of the group after the other; step s: its Q tile and row data go to
    // slot s % 4 of their rings, its dO tile to slot s % 3.  The issuing side keeps its own cursor
    // (list index, per-head base pointers) and advances it by additions only: divisions and 64-bit
    // multiplies per copy are serial scalar work of the issuing wave.
    const int head0 = kv_head * p.group + first_head;
    const char* is_q = p.q + ((int64_t)b * p.q_sb + (int64_t)head0 * p.q_sh) * 2;
    const char* is_do = p.dout + ((int64_t)b * p.do_sb + (int64_t)head0 * p.do_sh) * 2;
    // row-data arrays this wave copies (array w of lse, delta, seg, pos for w = pair, pair + NP, ...):
    // lse and delta are per head, seg and pos per batch row
    const char* is_rows[kRowCopies];
    int64_t rows_per_head[kRowCopies];
#pragma unroll
    for (int r = 0; r < kRowCopies; r++) {
      const int which = pair + r * NP;
      is_rows[r] = which == 0   ? (const char*)(p.lse + ((int64_t)b * p.num_heads + head0) * p.q_len)
                   : which == 1 ? (const char*)(p.delta + ((int64_t)b * p.num_heads + head0) * p.q_len)
                   : which == 2 ? (const char*)(p.q_seg + (int64_t)b * p.q_len)
                                : (const char*)(p.q_pos + (int64_t)b * p.q_len);
      rows_per_head[r] = which < 2 ? (int64_t)p.q_len * 4 : 0;
    }
    int is_li = first_li, is_sub = 0;
    uint32_t is_entry = live_list[first_li];
    auto issue_next = [&](int q_slot, int do_slot) {
      const int qr0 = (int)(is_entry & 0xffffff) * kTile + is_sub * SR;
      copy_q(is_q, qr0, p.q_len, smem_addr + Smem::kQ + q_slot * Smem::kQTileBytes);
      copy_do(is_do, qr0, p.q_len, smem_addr + Smem::kDo + do_slot * Smem::kDoTileBytes);
#pragma unroll
      for (int r = 0; r < kRowCopies; r++)
        async_copy_b32(is_rows[r] + (int64_t)min(qr0 + lane, p.q_len - 1) * 4,
                       __builtin_amdgcn_readfirstlane(smem_addr + Smem::kRows + q_slot * Smem::kRowData +
                                                      (pair + r * NP) * (kTile * 4)));
      if (++is_sub == SUB) {
        is_sub = 0;
        if (++is_li == n_live) {
          is_li = 0;
          is_q += p.q_sh * 2;
          is_do += p.do_sh * 2;
#pragma unroll
          for (int r = 0; r < kRowCopies; r++) is_rows[r] += rows_per_head[r];
        }
        is_entry = live_list[is_li];
      }
    };

    // P of the pair's tiles, 16-bit floats with a 10-bit mantissa whatever the tensor dtype:
    // [slot][unit mt][half st] x 64 lanes x 16 bytes, in the lane order of the C tile
    char* exchange = smem + Smem::kExchange + pair * 2 * Smem::kSlotBytes + lane * 16;

    // Above head_dim 128 the accumulators and fragments leave no registers for operands requested ahead
    // of the element-wise work.
    constexpr bool kLean = D > 128 && Cfg::kWps == 2;
    // S wave, second part of a tile: dS = P * (dP - delta) rounded to the input dtype (masked
    // entries have P = 0), dK^T += Q^T dS.  x = dP of that tile.
    auto finish_dk = [&](const f32x16 (&x)[UNITS], const char* qtile, const float* delta_rows, const char* pslot) {
      vec8 ta[2][DT];
      if (!kLean) {
#pragma unroll
        for (int st = 0; st < 2; st++)
#pragma unroll
          for (int dt = 0; dt < DT; dt++) ta[st][dt] = read_q_t(qtile + 16 * st * RB, dt);
      }
#pragma unroll
      for (int mt = 0; mt < UNITS; mt++) {
        vec8 dsb[2];
#pragma unroll
        for (int st = 0; st < 2; st++) {
          const uint4 e = *reinterpret_cast<const uint4*>(pslot + (2 * mt + st) * 1024);
          const uint32_t w[4] = {e.x, e.y, e.z, e.w};
          const float4 d0 = *reinterpret_cast<const float4*>(delta_rows + 32 * mt + 8 * (2 * st) + 4 * h);
          const float4 d1 = *reinterpret_cast<const float4*>(delta_rows + 32 * mt + 8 * (2 * st + 1) + 4 * h);
          const float dl[8] = {d0.x, d0.y, d0.z, d0.w, d1.x, d1.y, d1.z, d1.w};
          float ds[8];
#pragma unroll
          for (int j = 0; j < 4; j++) {
            ds[2 * j] = F16::to_float((uint16_t)(w[j] & 0xffff)) * (x[mt][8 * st + 2 * j] - dl[2 * j]);
            ds[2 * j + 1] = F16::to_float((uint16_t)(w[j] >> 16)) * (x[mt][8 * st + 2 * j + 1] - dl[2 * j + 1]);
          }
          dsb[st] = pack8<Tr>(ds[0], ds[1], ds[2], ds[3], ds[4], ds[5], ds[6], ds[7]);
        }
        if (kLean) {
#pragma unroll
          for (int st = 0; st < 2; st++)
#pragma unroll
            for (int dt = 0; dt < DT; dt++)
              acc[dt] = Tr::mfma(read_q_t(qtile + (32 * mt + 16 * st) * RB, dt), dsb[st], acc[dt]);
          continue;
        }
        vec8 tb[2][DT];  // operands of the next unit, requested before this unit's MFMAs
        if (mt + 1 < UNITS) {
#pragma unroll
          for (int st = 0; st < 2; st++)
#pragma unroll
            for (int dt = 0; dt < DT; dt++)
              tb[st][dt] = read_q_t(qtile + (32 * (mt + 1) + 16 * st) * RB, dt);
        }
#pragma unroll
        for (int st = 0; st < 2; st++)
#pragma unroll
          for (int dt = 0; dt < DT; dt++) acc[dt] = Tr::mfma(ta[st][dt], dsb[st], acc[dt]);
        if (mt + 1 < UNITS) {
#pragma unroll
          for (int st = 0; st < 2; st++)
#pragma unroll
            for (int dt = 0; dt < DT; dt++) ta[st][dt] = tb[st][dt];
        }
      }
    };

    int li = first_li, sub = 0;    // list index and sub-step of the current step
    uint32_t e0 = live_list[li];   // its entry
    uint32_t ep = 0;               // entry of the previous step
    if (p_wave) {
      issue_next(0, 0);
      if (steps > 1) issue_next(1, 1);
    }

    f32x16 x[UNITS];  // S of this step (P wave) / dP carried from the previous step (S wave)
    int q_slot = 0, do_slot = 0, q_prev = 0;
    for (int step = 0; step < steps; step++) {
      // the rows of this step have landed; every wavefront is done with the previous step
      if (p_wave) {
        if (step + 1 < steps) wait_vmcnt<kCopies>(); else wait_vmcnt<0>();
      }
      __syncthreads();
      if (p_wave && step + 2 < steps) issue_next((q_slot + 2) & 3, do_slot >= 1 ? do_slot - 1 : 2);
      const int t = e0 & 0xffffff;
      const bool active = (e0 >> (24 + wave)) & 1, active_prev = (ep >> (24 + wave)) & 1;
      const int qr0 = t * kTile + sub * SR;
      const char* qtile = smem + Smem::kQ + q_slot * Smem::kQTileBytes;
      const char* dotile = smem + Smem::kDo + do_slot * Smem::kDoTileBytes;
      const float* rowdata = reinterpret_cast<const float*>(smem + Smem::kRows + q_slot * Smem::kRowData);
      const int32_t* rowids = reinterpret_cast<const int32_t*>(rowdata + 2 * kTile);
      const bool full = t >= tf_lo && t < tf_hi;

      if (!p_wave && active_prev)
        finish_dk(x, smem + Smem::kQ + q_prev * Smem::kQTileBytes,
                  reinterpret_cast<const float*>(smem + Smem::kRows + q_prev * Smem::kRowData) + kTile,
                  exchange + ((step - 1) & 1) * Smem::kSlotBytes);

      // 8 * UNITS * KSTEPS / 8 MFMAs per wavefront, S = Q K^T (P wave) or dP = dO V^T (S wave), the
      // 32-row units interleaved; operand reads run four ahead of the MFMAs
      const char* rows_a = p_wave ? qtile : dotile;
      if (active) {
#pragma unroll
        for (int mt = 0; mt < UNITS; mt++)
#pragma unroll
          for (int i = 0; i < 16; i++) x[mt][i] = 0.f;
        // The order is fenced: with scheduling groups instead, the compiler gave up the reads ahead at
        // head_dim 128 and waited for every operand (dK/dV 2426 -> 2392 us on 32k tokens, 4574 -> 4448 on
        // 4 x 16k short documents, 186 -> 174 on 4k tokens, heads 32/8).  At 64 it does so, too, but mixes
        // the short contraction with what is around it, which is better (one document of 16k, heads 16/4:
        // 1533 against 1620).
#define KVAX_CONTRACT(n, regs)                                                                                       \
  if constexpr (D > 64) {                                                                                            \
    constexpr int N = UNITS * ((n) / 16), kAheadOps = 4;                                                             \
    vec8 op[N];                                                                                                      \
    auto read = [&](int i) {                                                                                         \
      return *reinterpret_cast<const vec8*>(rows_a + 32 * (i % UNITS) * ((n) * 2) + nat_off[i / UNITS % (regs)] +    \
                                            i / UNITS / (regs) * kGroupBytes<n>);                                    \
    };                                                                                                               \
    _Pragma("unroll") for (int i = 0; i < kAheadOps; i++) op[i] = read(i);                                           \
    __builtin_amdgcn_sched_barrier(0);                                                                               \
    _Pragma("unroll") for (int i = 0; i < N; i++) {                                                                  \
      x[i % UNITS] = Tr::mfma(op[i], frag[i / UNITS], x[i % UNITS]);                                                 \
      if (i + kAheadOps < N) op[i + kAheadOps] = read(i + kAheadOps);                                                \
      __builtin_amdgcn_sched_barrier(0);                                                                             \
    }                                                                                                                \
  } else {                                                                                                           \
  _Pragma("unroll") for (int ks = 0; ks < (n) / 16; ks++)                                                            \
      _Pragma("unroll") for (int mt = 0; mt < UNITS; mt++)                                                           \
          x[mt] = Tr::mfma(*reinterpret_cast<const vec8*>(rows_a + 32 * mt * ((n) * 2) + nat_off[ks % (regs)] +      \
                                                          ks / (regs) * kGroupBytes<n>), frag[ks], x[mt]);           \
  __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);                                                                 \
  _Pragma("unroll") for (int i = 0; i < UNITS * ((n) / 16) - 4; i++) {                                               \
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                                                               \
    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);                                                               \
  }                                                                                                                  \
  __builtin_amdgcn_sched_group_barrier(0x008, 4, 0); }
        if constexpr (D == DV) {
          KVAX_CONTRACT(D, kNatQ)
        } else if (p_wave) {
          KVAX_CONTRACT(D, kNatQ)
        } else {
          KVAX_CONTRACT(DV, kNatDo)
        }
#undef KVAX_CONTRACT
      }

      if (p_wave && active) {
        // operands of dV's first unit, requested before the element-wise work
        vec8 ta[2][DTV];
        if (!kLean) {
#pragma unroll
          for (int st = 0; st < 2; st++)
#pragma unroll
            for (int dt = 0; dt < DTV; dt++) ta[st][dt] = read_do_t(dotile + 16 * st * RBV, dt);
        }
        vec8 pb[UNITS][2];
        char* pslot = exchange + (step & 1) * Smem::kSlotBytes;
#pragma unroll
        for (int mt = 0; mt < UNITS; mt++) {
          f32x16& sc = x[mt];
          if (!full)  // raw scores: masked -> -inf, so that P = exp2(-inf) = 0 (scale_log2_abs > 0)
            mask_c_tile<false>(sc, rowids, rowids + kTile, 32 * mt, qr0, h, kvseg, kvpos, col_lo,
                               col_width, -INFINITY);
#pragma unroll
          for (int g4 = 0; g4 < 4; g4++) {
            const float4 l4 = *reinterpret_cast<const float4*>(rowdata + 32 * mt + 8 * g4 + 4 * h);
            sc[4 * g4 + 0] = fast_exp2(__builtin_fmaf(sc[4 * g4 + 0], p.scale_log2_abs, -l4.x));
            sc[4 * g4 + 1] = fast_exp2(__builtin_fmaf(sc[4 * g4 + 1], p.scale_log2_abs, -l4.y));
            sc[4 * g4 + 2] = fast_exp2(__builtin_fmaf(sc[4 * g4 + 2], p.scale_log2_abs, -l4.z));
            sc[4 * g4 + 3] = fast_exp2(__builtin_fmaf(sc[4 * g4 + 3], p.scale_log2_abs, -l4.w));
          }
#pragma unroll
          for (int st = 0; st < 2; st++) {
            pb[mt][st] = pack8<Tr>(sc[8 * st + 0], sc[8 * st + 1], sc[8 * st + 2], sc[8 * st + 3],
                                   sc[8 * st + 4], sc[8 * st + 5], sc[8 * st + 6], sc[8 * st + 7]);
            const uint4 e = make_uint4(F16::pack2(sc[8 * st + 0], sc[8 * st + 1]), F16::pack2(sc[8 * st + 2], sc[8 * st + 3]),
                                       F16::pack2(sc[8 * st + 4], sc[8 * st + 5]), F16::pack2(sc[8 * st + 6], sc[8 * st + 7]));
            *reinterpret_cast<uint4*>(pslot + (2 * mt + st) * 1024) = e;
          }
        }
        // dV^T += dO^T P
#pragma unroll
        for (int mt = 0; mt < UNITS; mt++) {
          if (kLean) {
#pragma unroll
            for (int st = 0; st < 2; st++)
#pragma unroll
              for (int dt = 0; dt < DTV; dt++)
                acc[dt] = Tr::mfma(read_do_t(dotile + (32 * mt + 16 * st) * RBV, dt), pb[mt][st], acc[dt]);
            continue;
          }
          vec8 tb[2][DTV];
          if (mt + 1 < UNITS) {
#pragma unroll
            for (int st = 0; st < 2; st++)
#pragma unroll
              for (int dt = 0; dt < DTV; dt++)
                tb[st][dt] = read_do_t(dotile + (32 * (mt + 1) + 16 * st) * RBV, dt);
          }
#pragma unroll
          for (int st = 0; st < 2; st++)
#pragma unroll
            for (int dt = 0; dt < DTV; dt++) acc[dt] = Tr::mfma(ta[st][dt], pb[mt][st], acc[dt]);
          if (mt + 1 < UNITS) {
#pragma unroll
            for (int st = 0; st < 2; st++)
#pragma unroll
              for (int dt = 0; dt < DTV; dt++) ta[st][dt] = tb[st][dt];
          }
        }
      }
      ep = e0;
      if (++sub == SUB) {
        sub = 0;
        li = li + 1 == n_live ? 0 : li + 1;
        e0 = live_list[li];
      }
      q_prev = q_slot;
      q_slot = (q_slot + 1) & 3;
      do_slot = do_slot == 2 ? 0 : do_slot + 1;
    }
    // the S wave still owes the last tile
    __syncthreads();
    if (!p_wave && ((ep >> (24 + wave)) & 1))
      finish_dk(x, smem + Smem::kQ + q_prev * Smem::kQTileBytes,
                reinterpret_cast<const float*>(smem + Smem::kRows + q_prev * Smem::kRowData) + kTile,
                exchange + ((steps - 1) & 1) * Smem::kSlotBytes);
  }
  __syncthreads();  // the next chunk reuses the bookkeeping, the rings and the exchange slots
  }
  }

  if (tid == 0) ticket = work.draw();
  // ---- epilogue: the P wave holds dV^T, the S wave dK^T (times the scale) ----------------------
  // A lane holds 4 consecutive head-dim elements of its kv row per register group, so storing from
  // the registers would touch 32 rows with 8 or 16 bytes each per instruction.  Each wavefront
  // instead passes its 32 x D tile through its own part of the LDS (the rings are free by now),
  // 128 head-dim columns at a time, and writes whole rows: 16 bytes per lane, consecutive lanes
  // consecutive chunks of a row.  Rows are swizzled by the row index so that neither side has bank
  // conflicts.
  {
    // (padding keys, dead: exact zeros, see the dQ kernel's epilogue)
    const float mul = p_wave ? 1.f : p.scale;
    char* base = p_wave ? dv_out : dk_out;
    int64_t sb = p_wave ? p.dv_sb : p.dk_sb, sh = p_wave ? p.dv_sh : p.dk_sh, ss = p_wave ? p.dv_ss : p.dk_ss;
    if (whole) {
      sb = p_wave ? p.whole_dv_sb : p.whole_dk_sb;
      sh = p_wave ? p.whole_dv_sh : p.whole_dk_sh;
      ss = p_wave ? p.whole_dv_ss : p.whole_dk_ss;
    }
    constexpr int PC = D % 128 == 0 && DV % 128 == 0 ? 128 : 64;  // columns per pass
    constexpr int kDtPerPass = PC / 32;
    const int esize = dkdv_f32() ? 4 : 2;
    const int row_bytes = PC * esize;             // 128, 256 or 512
    const int chunks = row_bytes / 16;            // 8, 16 or 32 per row
    char* stage = smem + wave * (32 * PC * 4);    // room for the fp32 case
    static_assert(NW * 32 * PC * 4 <= Smem::kTotal, "a wavefront's part of the LDS");
    const int64_t tile_off = (int64_t)b * sb + (int64_t)kv_head * sh + (int64_t)(k0 + pair * 32) * ss;
#pragma unroll
    for (int pass = 0; pass < D / PC; pass++) {
      if (D != DV && p_wave && pass >= DV / PC) break;
      char* mine = stage + c * row_bytes;
      if (dkdv_f32()) {
#pragma unroll
        for (int d = 0; d < kDtPerPass; d++)
#pragma unroll
          for (int g4 = 0; g4 < 4; g4++) {
            const f32x16& a = acc[pass * kDtPerPass + d];
            const int chunk = 8 * d + 2 * g4 + h;
            *reinterpret_cast<float4*>(mine + ((chunk ^ (c & (chunks - 1))) * 16)) =
                dead ? make_float4(0.f, 0.f, 0.f, 0.f)
                     : make_float4(a[4 * g4 + 0] * mul, a[4 * g4 + 1] * mul, a[4 * g4 + 2] * mul, a[4 * g4 + 3] * mul);
          }
      } else {
#pragma unroll
        for (int d = 0; d < kDtPerPass; d++)
#pragma unroll
          for (int g4 = 0; g4 < 4; g4++) {
            const f32x16& a = acc[pass * kDtPerPass + d];
            uint2 u;
            u.x = Tr::pack2(a[4 * g4 + 0] * mul, a[4 * g4 + 1] * mul);
            u.y = Tr::pack2(a[4 * g4 + 2] * mul, a[4 * g4 + 3] * mul);
            if (dead) u = make_uint2(0, 0);
            const int chunk = 4 * d + g4;
            *reinterpret_cast<uint2*>(mine + ((chunk ^ (c & (chunks - 1))) * 16) + 8 * h) = u;
          }
      }
      // 32 rows x `chunks` 16-byte pieces, 64 per instruction
      const int per_iter = 64 / chunks;  // rows per instruction: 8, 4 or 2
      for (int r0 = 0; r0 < 32; r0 += per_iter) {
        const int row = r0 + lane / chunks, chunk = lane % chunks;
        const uint4 v = *reinterpret_cast<const uint4*>(stage + row * row_bytes + ((chunk ^ (row & (chunks - 1))) * 16));
        if (k0 + pair * 32 + row < p.kv_len)
          *reinterpret_cast<uint4*>(base + (tile_off + (int64_t)row * ss) * esize + pass * row_bytes + chunk * 16) = v;
      }
    }
  }
  }  // the item has work
  } else if (tid == 0) {
    ticket = work.draw();
  }
  if (tid == 0) *next_item = work.resolve(ticket);
  __syncthreads();
  }  // items of this XCD
}

// Adds the parts' fp32 dK and dV in the order of the parts and writes them in the gradients' type and
// strides.  A copy, bound by memory: 16 bytes per thread and part, four parts in flight.
struct DkdvSumParams {
  const float* parts[2];  // dK, dV: [part][batch, kv_len, kv heads, head_dim]
  char* dst[2];
  int64_t sb[2], ss[2], sh[2];
  int64_t total[2];       // 4-element pieces of a tensor
  int pieces[2];          // and of one of its rows
  int num_parts, kv_len, num_kv_heads, group;
  int f32;
  const int32_t* work_stats;  // null, or as in BwdParams: nothing to add where no items are shared
};

template <class Tr>
__global__ __launch_bounds__(256) void dkdv_sum_kernel(const DkdvSumParams p) {
  const int which = blockIdx.y;
  if (p.work_stats && !shares_items(p.work_stats, p.num_kv_heads, p.group)) return;
  // (one round, but for launches that may have nothing to do)
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < p.total[which]; i += (int64_t)gridDim.x * 256) {
  const float4* src = reinterpret_cast<const float4*>(p.parts[which]) + i;
  float4 sum = src[0];
#pragma unroll 4
  for (int part = 1; part < p.num_parts; part++) {
    const float4 v = src[p.total[which] * part];
    sum.x += v.x, sum.y += v.y, sum.z += v.z, sum.w += v.w;
  }
  int64_t row = i / p.pieces[which];
  const int d = (int)(i % p.pieces[which]) * 4;
  const int head = (int)(row % p.num_kv_heads);
  row /= p.num_kv_heads;
  const int64_t at = row / p.kv_len * p.sb[which] + row % p.kv_len * p.ss[which] + head * p.sh[which] + d;
  if (p.f32)
    *reinterpret_cast<float4*>(p.dst[which] + at * 4) = sum;
  else
    *reinterpret_cast<uint2*>(p.dst[which] + at * 2) = make_uint2(Tr::pack2(sum.x, sum.y), Tr::pack2(sum.z, sum.w));
  }
}

// How many work-groups share the steps of a dK/dV work item.  A launch with fewer items than compute
// units leaves the others idle, and one with few more ends on its longest items (under a causal mask
// the first keys see twice the mean number of queries).  An item costs about 20 us whatever its steps
// (ids, list, first tiles, results), a step 1.2 to 1.8 us, and every part is written and read once
// more: one round of parts on the compute units where each has at least 8 steps, two, which even out
// the items' lengths, where it has 24, three where it has 128.  Steps are counted as if every query
// tile were live.  dK/dV kernel and sum, us, items x steps without parts -> with (number of parts):
//   32 x 128 (2k, heads 8/2 of 64)       126 -> 44 (8), 53 (16)
//   64 x 64 (1k, heads 32/8 of 128)      127 -> 60 (4), 83 (8)
//   128 x 128 (2k, heads 32/8)           178 -> 112 (2), 102 (4), 108 (6), 140 (8)
//   192 x 192 (3k, documents of 1k)      180 -> 121 (2), 149 (4)
//   128 x 512 (8k, heads 8/2, the same)  323 -> 184 (2), 117 (4), 139 (6), 160 (8)
//   256 x 256 (4k, heads 32/8)           450 -> 317 (2), 348 (3)
//   384 x 384 (6k)                       741 -> 683 (2)
//   128 x 1024 (16k, heads 4/1)          622 -> 333 (2), 192 (4), 172 (6), 193 (8)
//   256 x 2048 (32k, heads 4/1)          1179 -> 631 (2), 452 (3)
// A function of the shapes, so that the workspace can be sized up front (at most 768 parts of 128 rows;
// up to 1024 where the device decides, see device_decides_parts).
int plan_dkdv_parts(int batch, int q_len, int kv_len, int num_heads, int num_kv_heads, int head_dim) {
  if (batch <= 0 || q_len <= 0 || kv_len <= 0 || num_kv_heads <= 0 || num_heads % num_kv_heads) return 1;
  const int64_t items = (int64_t)batch * num_kv_heads * cdiv(kv_len, dkdv_kv_rows(head_dim));
  const int64_t steps = (int64_t)cdiv(q_len, kTile) * (num_heads / num_kv_heads);
  const int64_t one_round = min(kNumCus / items, steps / 8), two_rounds = min(2 * kNumCus / items, steps / 24),
                three_rounds = min(3 * kNumCus / items, steps / 128);
  return (int)max(min(max(max(one_round, two_rounds), three_rounds), (int64_t)16), (int64_t)1);
}

// Whether the device decides between one part and two (see shares_items): the order is computed for such launches.
bool device_decides_parts(int batch, int q_len, int kv_len, int num_heads, int num_kv_heads, int head_dim) {
  if (plan_dkdv_parts(batch, q_len, kv_len, num_heads, num_kv_heads, head_dim) > 1) return false;
  if (num_kv_heads <= 0 || (int64_t)cdiv(q_len, kTile) * (num_heads / num_kv_heads) < 160) return false;
  if (cdiv(q_len, kTile) > 1 << 20) return false;  // the sum of 512 items' work stays below 2^31
  const int tiles = cdiv(kv_len, dkdv_kv_rows(head_dim));
  const int64_t items = (int64_t)batch * num_kv_heads * tiles;
  return items > kNumCus && items <= 2 * kNumCus && tiles >= kMinOrderedItems && tiles <= kMaxOrderedItems;
}

template <class K>
int reserve_lds(K kernel, int need, int bytes, LdsReservation* reservation, const char* what) {
  if (need > bytes)
    return fail(KVAX_EUNSUPPORTED, "%s needs %d bytes of LDS for tile bitmaps (limit %d): sequence too long",
                what, need, bytes);
  return reservation->ensure(kernel, bytes, what);
}

// dQ launch: NW wavefronts (32 query rows each) per work-group, WPS per SIMD.
template <class Tr, int D, int DV, int NW, int STAGES, int WPS = 2>
int launch_dq(BwdParams p, hipStream_t stream) {
  auto kernel = fa_bwd_dq_kernel<Tr, D, DV, NW, WPS, STAGES>;
  static LdsReservation done;
  constexpr int kLimit = kLdsPerCu / (4 * WPS / NW);  // work-groups per compute unit share the LDS
  const int smem = DqSmem<D, DV, STAGES>::kTotal + live_tiles_bytes(NW, p.n_kv_tiles);
  if (int rc = reserve_lds(kernel, smem, kLimit, &done, "the dQ kernel")) return rc;
  p.dq_head_shift = kHeadsPerWorkGroup<D> ? heads_shift(p.group, NW) : 0;
  p.num_tiles = cdiv(p.q_len, NW * 32 >> p.dq_head_shift);
  p.total_items = ItemMap{p.batch * p.num_kv_heads, p.num_tiles, p.group >> p.dq_head_shift}.grid();
  hipLaunchKernelGGL(kernel, dim3(p.total_items), dim3(NW * 64), smem, stream, p);
  return check_launch("fa_bwd_dq_kernel");
}

template <class Tr, int D, int DV>
int launch_bwd(BwdParams p, hipStream_t stream) {
  // a key sequence too long for the dQ kernel's largest configuration is refused before anything
  // is enqueued (the dK/dV kernel has no such limit)
  if (p.q_len > 0 && !(p.flags & KVAX_FA_SKIP_DQ)) {
    const int need = D > 128 ? DqSmem<D, DV, 2>::kTotal + live_tiles_bytes(4, p.n_kv_tiles)
                             : DqSmem<D, DV, 3>::kTotal + live_tiles_bytes(8, p.n_kv_tiles);
    if (need > kLdsPerCu)
      return fail(KVAX_EUNSUPPORTED, "the dQ kernel needs %d bytes of LDS for tile bitmaps (limit %d): "
                  "sequence too long", need, kLdsPerCu);
  }
  // tile summaries of both sequences (a few microseconds; needed by dQ and dK/dV)
  {
    TileSummaryJob jobs[2] = {{p.kv_pos, p.kv_seg, (void*)p.kv_tiles, p.kv_len},
                              {p.q_pos, p.q_seg, (void*)p.q_tiles, p.q_len}};
    int32_t* counters = tile_order_counters(p.order_ws, p.batch, cdiv(p.kv_len, DkdvCfg<D>::kKvRows));
    if (int rc = launch_tile_summaries(jobs, 2, p.batch, stream, counters)) return rc;
  }
  // dQ: two work-groups of four wavefronts per compute unit (each hides the other's prologue,
  // barriers and final stores) when the tile bitmaps fit beside the smaller ring, else one of eight;
  // at head_dim 256 (128 accumulator registers for dQ alone) one work-group of four, one per SIMD
  constexpr int kStagesSmall = D == 64 ? 3 : 2;
  using Cfg = DkdvCfg<D>;
  const bool run_dq = p.q_len > 0 && !(p.flags & KVAX_FA_SKIP_DQ);
  const bool run_dkdv = p.kv_len > 0 && !(p.flags & KVAX_FA_SKIP_DKDV);
  const bool dq_small =
      DqSmem<D, DV, kStagesSmall>::kTotal + live_tiles_bytes(4, p.n_kv_tiles) <= kLdsHalfCu;
  // dK/dV runs one long work-group per compute unit: its light work items are dispatched last, by
  // decreasing number of live tiles, so that the launch does not end on a few long ones.  With no more
  // items (parts included) than compute units all start at once and the order decides nothing: a launch of
  // 6 us less (2k tokens, heads 8/2 of 64).
  {
    const int items = cdiv(p.kv_len, Cfg::kKvRows);
    if (run_dkdv && items >= kMinOrderedItems && items <= kMaxOrderedItems &&
        (int64_t)items * p.batch * p.num_kv_heads * p.dkdv_parts > kNumCus &&
        (int64_t)items * (p.n_q_tiles + 2) < 0x7fffffff) {
      const TileOrderJob job{p.kv_tiles, p.q_tiles, p.order_ws, p.n_kv_tiles, p.n_q_tiles,
                             Cfg::kKvRows / kTileRows, items, 0, p.work_stats != nullptr};
      if (int rc = launch_tile_order(job, p.batch, stream)) return rc;
      p.dkdv_order = p.order_ws;
    }
    if (!p.dkdv_order) p.work_stats = nullptr;
  }
  if (run_dq) {
    if constexpr (D == 256) {
      if (int rc = launch_dq<Tr, D, DV, 4, 2, 1>(p, stream)) return rc;
    } else if constexpr (D > 128) {
      // At 192 with 128 for the values eight wavefronts, two per SIMD, just fit their registers (with 192
      // they spill 48 in the step: 175 against 120 us on 4k tokens, 16 heads) and pay where more
      // work-groups than compute units remain (us, eight / four wavefronts, 16 heads): 2 x 4k tokens
      // 201 / 225, 16k 785 / 1055, 6k 318 / 402; 4k 201 / 177, 2k 106 / 86.
      [[maybe_unused]] const bool fills = (int64_t)p.batch * p.num_heads * cdiv(p.q_len, 256) > kNumCus;
      if constexpr (DV == 128) {
        if (fills && DqSmem<D, DV, 2>::kTotal + live_tiles_bytes(8, p.n_kv_tiles) <= kLdsPerCu) {
          if (int rc = launch_dq<Tr, D, DV, 8, 2>(p, stream)) return rc;
        } else {
          if (int rc = launch_dq<Tr, D, DV, 4, 2, 1>(p, stream)) return rc;
        }
      } else {
        if (int rc = launch_dq<Tr, D, DV, 4, 2, 1>(p, stream)) return rc;
      }
    } else {
      if (dq_small) {
        if (int rc = launch_dq<Tr, D, DV, 4, kStagesSmall>(p, stream)) return rc;
      } else {
        if (int rc = launch_dq<Tr, D, DV, 8, 3>(p, stream)) return rc;
      }
    }
  }
  // dK/dV: wavefronts in role pairs (see DkdvCfg)
  if (run_dkdv) {
    constexpr int NW = Cfg::kWaves;
    static LdsReservation done, done_deciding;
    const bool deciding = p.work_stats != nullptr;
    auto kernel = deciding ? fa_bwd_dkdv_kernel<Tr, D, DV, true> : fa_bwd_dkdv_kernel<Tr, D, DV, false>;
    // live-tile bookkeeping for as many query tiles as the remaining LDS holds (a multiple of 64)
    constexpr int kLdsLimit = kLdsPerCu;
    int chunk = 64;
    while (chunk < p.n_q_tiles && DkdvSmem<D, DV>::kTotal + live_tiles_bytes(NW, chunk * 2) <= kLdsLimit) chunk *= 2;
    p.list_tiles = min(chunk, max(p.n_q_tiles, 1));
    const int smem = DkdvSmem<D, DV>::kTotal + live_tiles_bytes(NW, p.list_tiles);
    if (int rc = reserve_lds(kernel, smem, kLdsLimit, deciding ? &done_deciding : &done, "the dK/dV kernel")) return rc;
    p.num_tiles = cdiv(p.kv_len, Cfg::kKvRows);
    p.total_items = ItemMap{p.batch * p.num_kv_heads, p.num_tiles, p.dkdv_parts}.grid();
    DkdvSumParams sum{};
    if (p.work_stats) {
      p.dkdv_parts = 2;
      p.whole_dk = p.dk, p.whole_dk_sb = p.dk_sb, p.whole_dk_ss = p.dk_ss, p.whole_dk_sh = p.dk_sh;
      p.whole_dv = p.dv, p.whole_dv_sb = p.dv_sb, p.whole_dv_ss = p.dv_ss, p.whole_dv_sh = p.dv_sh;
      p.whole_f32 = p.dkdv_f32;
      p.total_items = ItemMap{p.batch * p.num_kv_heads, p.num_tiles, 2}.grid();
      sum.work_stats = p.work_stats;
    }
    if (p.dkdv_parts > 1) {  // the kernel leaves fp32 parts, dkdv_sum_kernel adds them
      const int64_t rows = (int64_t)p.batch * p.kv_len * p.num_kv_heads;
      sum.dst[0] = p.dk, sum.sb[0] = p.dk_sb, sum.ss[0] = p.dk_ss, sum.sh[0] = p.dk_sh;
      sum.dst[1] = p.dv, sum.sb[1] = p.dv_sb, sum.ss[1] = p.dv_ss, sum.sh[1] = p.dv_sh;
      sum.pieces[0] = D / 4, sum.pieces[1] = DV / 4;
      sum.total[0] = rows * (D / 4), sum.total[1] = rows * (DV / 4);
      sum.parts[0] = p.parts_ws, sum.parts[1] = p.parts_ws + rows * D * p.dkdv_parts;
      sum.num_parts = p.dkdv_parts, sum.kv_len = p.kv_len, sum.num_kv_heads = p.num_kv_heads, sum.group = p.group;
      sum.f32 = p.dkdv_f32;
      p.dk = (char*)sum.parts[0], p.dk_sh = D, p.dk_ss = (int64_t)p.num_kv_heads * D, p.dk_sb = p.dk_ss * p.kv_len;
      p.dv = (char*)sum.parts[1], p.dv_sh = DV, p.dv_ss = (int64_t)p.num_kv_heads * DV, p.dv_sb = p.dv_ss * p.kv_len;
      p.dk_part = sum.total[0] * 16, p.dv_part = sum.total[1] * 16;
      p.dkdv_f32 = 1;
    }
    p.dkdv_queue = tile_order_counters(p.order_ws, p.batch, p.num_tiles) + p.batch;
    hipLaunchKernelGGL(kernel, dim3(min(p.total_items, kNumCus)), dim3(NW * 64), smem, stream, p);
    if (int rc = check_launch("fa_bwd_dkdv_kernel")) return rc;
    if (p.dkdv_parts > 1) {
      unsigned grid = (unsigned)((sum.total[0] + 255) / 256);
      if (p.work_stats) grid = grid < 4 * kNumCus ? grid : 4 * kNumCus;
      hipLaunchKernelGGL(dkdv_sum_kernel<Tr>, dim3(grid, 2), dim3(256), 0, stream, sum);
      if (int rc = check_launch("dkdv_sum_kernel")) return rc;
    }
  }
  return KVAX_OK;
}

}  // namespace
}  // namespace kvax

using namespace kvax;

static size_t delta_bytes(const kvax_fa_args* a) {
  return ((size_t)a->batch * a->num_heads * a->q_len * sizeof(float) + 15) / 16 * 16;
}

// Start of the dK/dV parts in the workspace: behind delta [batch, heads, q_len] fp32, the tile summaries
// of the kv and query sequences, and the dispatch order of the dK/dV work items.
static size_t parts_offset(const kvax_fa_args* a) {
  return delta_bytes(a) + tile_summary_bytes(a->batch, a->kv_len) + tile_summary_bytes(a->batch, a->q_len) +
         tile_order_bytes(a->batch, cdiv(a->kv_len, dkdv_kv_rows(a->head_dim)));
}
static int dkdv_parts(const kvax_fa_args* a) {
  return plan_dkdv_parts(a->batch, a->q_len, a->kv_len, a->num_heads, a->num_kv_heads, a->head_dim);
}
static bool dkdv_device_decides(const kvax_fa_args* a) {
  return device_decides_parts(a->batch, a->q_len, a->kv_len, a->num_heads, a->num_kv_heads, a->head_dim);
}
static size_t dkdv_parts_bytes(const kvax_fa_args* a) {
  const int parts = dkdv_device_decides(a) ? 2 : dkdv_parts(a);
  return parts == 1 ? 0 : (size_t)parts * a->batch * a->kv_len * a->num_kv_heads * (a->head_dim + value_head_dim(a)) * sizeof(float);
}

extern "C" size_t kvax_fa_bwd_workspace_bytes(const kvax_fa_args* a) {
  if (!a || a->batch < 0 || a->q_len < 0 || a->kv_len < 0 || a->num_heads < 0) return 0;
  return parts_offset(a) + dkdv_parts_bytes(a);
}

extern "C" int kvax_fa_bwd(const kvax_fa_args* a, void* workspace, size_t workspace_bytes,
                           kvax_stream_t stream_) {
  if (int rc = validate_fa_common(a)) return rc;
  // empty tensors (and the masks over an empty outer axis) may come with null pointers
  const bool has_q = a->batch > 0 && a->q_len > 0, has_kv = a->batch > 0 && a->kv_len > 0;
  if ((has_q && (!a->dout || !a->dq)) || (has_kv && (!a->dk || !a->dv)))
    return fail(KVAX_EINVAL, "null gradient pointer");
  if (a->bwd_query_block <= 0 || a->bwd_kv_block <= 0)
    return fail(KVAX_EINVAL, "backward block sizes must be positive");
  for (int i = 0; i < 4; i++)
    if ((has_q && !a->dq_mask[i]) || (has_kv && !a->dkdv_mask[i]))
      return fail(KVAX_EINVAL, "backward masks are missing");
  const int shards = a->dkdv_shards > 1 ? a->dkdv_shards : 1;
  if (a->dkdv_shards < 0 || a->q_len % shards || (shards > 1 && a->q_len / shards % a->bwd_query_block))
    return fail(KVAX_EINVAL, "q_len %d does not split into %d shards of whole %d-token blocks", a->q_len,
                a->dkdv_shards, a->bwd_query_block);
  const int64_t* strides[] = {a->do_strides, a->dq_strides, a->dk_strides, a->dv_strides};
  for (auto s : strides)
    for (int i = 0; i < 3; i++)
      if (s[i] % 8) return fail(KVAX_EINVAL, "strides must be multiples of 8 elements (16 bytes)");
  for (auto s : strides)
    if (s[1] < 0 || s[1] >= (1 << 24))
      return fail(KVAX_EUNSUPPORTED, "sequence stride of %lld elements is outside [0, 2^24)", (long long)s[1]);
  const void* ptrs[] = {a->dout, a->dq, a->dk, a->dv};
  for (auto ptr : ptrs)
    if ((uintptr_t)ptr % 16) return fail(KVAX_EINVAL, "tensor pointers must be 16-byte aligned");
  const size_t need = kvax_fa_bwd_workspace_bytes(a);
  if (need > workspace_bytes || (need && !workspace))
    return fail(KVAX_EWORKSPACE, "workspace of %zu bytes needed, %zu given", need, workspace_bytes);
  if ((uintptr_t)workspace % 16) return fail(KVAX_EINVAL, "workspace must be 16-byte aligned");
  if (a->batch == 0) return KVAX_OK;

  BwdParams p{};
  p.q = (const char*)a->q, p.k = (const char*)a->k, p.v = (const char*)a->v;
  p.out = (const char*)a->out, p.dout = (const char*)a->dout;
  p.dq = (char*)a->dq, p.dk = (char*)a->dk, p.dv = (char*)a->dv;
  p.lse = a->lse;
  p.delta = (float*)workspace;
  p.kv_tiles = (const int4*)((char*)workspace + delta_bytes(a));
  p.q_tiles = (const int4*)((char*)workspace + delta_bytes(a) + tile_summary_bytes(a->batch, a->kv_len));
  p.n_kv_tiles = cdiv(a->kv_len, kTileRows);
  p.n_q_tiles = cdiv(a->q_len, kTileRows);
  p.order_ws = (int32_t*)((char*)p.q_tiles + tile_summary_bytes(a->batch, a->q_len));
  p.q_pos = a->q_pos, p.q_seg = a->q_seg, p.kv_pos = a->kv_pos, p.kv_seg = a->kv_seg;
  for (int i = 0; i < 4; i++) p.dq_mask[i] = a->dq_mask[i], p.dkdv_mask[i] = a->dkdv_mask[i];
  p.q_sb = a->q_strides[0], p.q_ss = a->q_strides[1], p.q_sh = a->q_strides[2];
  p.k_sb = a->k_strides[0], p.k_ss = a->k_strides[1], p.k_sh = a->k_strides[2];
  p.v_sb = a->v_strides[0], p.v_ss = a->v_strides[1], p.v_sh = a->v_strides[2];
  p.o_sb = a->o_strides[0], p.o_ss = a->o_strides[1], p.o_sh = a->o_strides[2];
  p.do_sb = a->do_strides[0], p.do_ss = a->do_strides[1], p.do_sh = a->do_strides[2];
  p.dq_sb = a->dq_strides[0], p.dq_ss = a->dq_strides[1], p.dq_sh = a->dq_strides[2];
  p.dk_sb = a->dk_strides[0], p.dk_ss = a->dk_strides[1], p.dk_sh = a->dk_strides[2];
  p.dv_sb = a->dv_strides[0], p.dv_ss = a->dv_strides[1], p.dv_sh = a->dv_strides[2];
  p.batch = a->batch, p.q_len = a->q_len, p.kv_len = a->kv_len;
  p.num_heads = a->num_heads, p.num_kv_heads = a->num_kv_heads;
  p.group = a->num_heads / a->num_kv_heads;
  p.bq = a->bwd_query_block, p.bk = a->bwd_kv_block;
  p.n_dq_blocks = cdiv(a->q_len, a->bwd_kv_block);
  p.n_kv_blocks = cdiv(a->kv_len, a->bwd_kv_block);
  p.dkdv_parts = dkdv_parts(a);
  if (dkdv_device_decides(a))
    p.work_stats = tile_order_counters(p.order_ws, a->batch, cdiv(a->kv_len, dkdv_kv_rows(a->head_dim))) + a->batch + kQueueCounters;
  p.parts_ws = (float*)((char*)workspace + parts_offset(a));
  p.num_shards = shards;
  p.shard_rows = a->q_len / shards;
  p.dkdv_f32 = (a->flags & KVAX_FA_DKDV_F32) != 0;
  p.flags = a->flags;
  p.scale = a->scale;
  p.scale_log2 = a->scale * 1.4426950408889634f;
  p.scale_log2_abs = fmaxf(fabsf(a->scale), 1e-30f) * 1.4426950408889634f;
  p.k_sign = a->scale < 0.f ? 0x80008000u : 0u;
  hipStream_t stream = (hipStream_t)stream_;
  return dispatch_heads(a, [&](auto tr, auto d, auto dv) {
    return launch_bwd<decltype(tr), decltype(d)::value, decltype(dv)::value>(p, stream);
  });
}
