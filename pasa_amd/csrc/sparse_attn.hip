// K4: block-sparse flash attention with per-group first-order correction.
//
// Reference: pisa_pg_fwd_kernel, svg/kernels/triton/group_pisa_attention.py:135-262
//   Phase 1 (:170-186): exact online softmax (base 2) over the selected key
//     blocks; columns >= T masked.
//   Phase 2 (:212-253): per group g of 32 key blocks, the blocks not selected
//     contribute p_j (V^_j + s * Hbar_g^T q) with p_j = 2^(c q.kbar_j - m);
//     A and L are rescaled when the running max rises, Gamma = sum p_j n_j is
//     not (the reference's literal form, :201/:243; gamma_literal = 0 gives the
//     rescaled "consistent" form).
//   Finalize (:258-262): o = A / (L + Gamma).
//
// MI355X mapping.  One workgroup = one (slice, query block) of BT rows, or two blocks of 64
// (PAIR); one wavefront per 32 query rows.  Everything is computed transposed so that the
// softmax statistics of a query row stay in the lanes that hold it:
//   S^T[key][q]  = K  * Q^T    (16x16x32 MFMA, K from LDS, Q in VGPRs)
//   O^T[e][q]   += V^T * P^T   (V^T read from the row-major V tile with
//                               ds_read_b64_tr_b16, P from the S^T accumulators)
// The lane layout is described at k4_body.
//
// Phase 1 walks the selected blocks in ascending block order (the selection
// bitmask) instead of top-k order: exact online softmax is order-independent up
// to rounding, and the ascending sweep keeps the workgroups of one XCD on
// nearby key blocks at the same time, so the K/V tiles they share hit in L2.
// Workgroups are mapped XCD-aware: each XCD walks a contiguous run of query
// blocks of the same head.
//
// One body, k4_body, for head dims 64 and 128 (kernels k4_sparse_attn, k4_sparse_attn_dma and
// k4_cross_attn): K/V tiles go straight into LDS (buffer_load ... lds, XOR-swizzled rows),
// double-buffered between the K and V tiles, with an exact online softmax (rescale whenever a
// row's max rises).  At BT = 64 a four-wave workgroup runs two query blocks (PAIR), each wave
// pair on its own selected tiles in lock step: co-resident workgroups on a CU drift into
// start-time cohorts, each sweeping a different region of key space, and pairing halves the
// number of cohorts (and so the L2 working set), while each group's phase-2 operands are loaded
// once for both blocks.
//
// The row sum of P is kept in fp32 (adds, not v_dot2c_f32_bf16: on gfx950 a dot
// instruction issues only between the MFMAs of the SIMD's other wave, so it stalls
// its wave behind the partner's MFMA stream).
//
// Phase-2 operands (kbar, V^ transposed, Hbar transposed; in the input's 16-bit type) are
// packed per (slice, group) by k4_pack_xor into the exact LDS image K4 copies in.  That type
// is a template argument (Bf16, or F16 at D = 128).
#include "common.h"
#include "k4_layout.h"
#include "kernels.h"

namespace pasa {

// ---- phase-2 operand pack ---------------------------------------------------

// One workgroup per (group, slice).  Every output element is written once, as part of
// a 16-byte chunk: Hbar^T goes through LDS (coalesced fp32 reads of Hbar rows, column
// reads from a padded tile), kbar rows are read as 32-byte runs, V^T columns with the
// token index fastest across lanes.  Rounding is round-to-nearest-even, as everywhere.
template <int D, typename E = Bf16>
__global__ __launch_bounds__(256) void k4_pack_xor(const float* __restrict__ kc,
                                                   const float* __restrict__ vc,
                                                   const float* __restrict__ hgroup,
                                                   unsigned char* __restrict__ pack, int NT, int NG) {
  using P = K4Pack<D>;
  using TL = K4Tile<D>;
  constexpr int CH = D / 8;   // 16-byte chunks per row
  constexpr int HS = D + 1;  // padded row of the fp32 Hbar tile
  __shared__ float hs[D * HS];
  const int g = blockIdx.x;
  const int bh = blockIdx.y;
  const int tid = threadIdx.x;
  unsigned char* out = pack + ((int64_t)bh * NG + g) * P::BYTES;
  const float* kb = kc + (int64_t)bh * NT * D;
  const float* vb = vc + (int64_t)bh * NT * D;
  const float* hb = hgroup + ((int64_t)bh * NG + g) * D * D;
#pragma unroll 4
  for (int it = 0; it < D * D / 4 / 256; ++it) {
    const int idx = it * 256 + tid;
    const int d = idx / (D / 4);
    const int e4 = (idx % (D / 4)) * 4;
    const float4 x = *(const float4*)(hb + d * D + e4);
    hs[d * HS + e4 + 0] = x.x;
    hs[d * HS + e4 + 1] = x.y;
    hs[d * HS + e4 + 2] = x.z;
    hs[d * HS + e4 + 3] = x.w;
  }
  // kbar: rows m (block of the group) x D / 8 chunks of 8 features, K layout.
  unsigned char* part2 = out + P::HT_BYTES;
#pragma unroll
  for (int it = 0; it < kGroup * D / 8 / 256; ++it) {
    const int qi = it * 256 + tid;
    const int m = qi / CH;
    const int cc = qi % CH;
    const int jj = g * kGroup + m;
    float f[8];
    if (jj < NT) {
      const float4 x0 = *(const float4*)(kb + (int64_t)jj * D + cc * 8);
      const float4 x1 = *(const float4*)(kb + (int64_t)jj * D + cc * 8 + 4);
      f[0] = x0.x; f[1] = x0.y; f[2] = x0.z; f[3] = x0.w;
      f[4] = x1.x; f[5] = x1.y; f[6] = x1.z; f[7] = x1.w;
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) f[i] = 0.f;
    }
    const uint4 w = make_uint4(E::pack2(f[0], f[1]), E::pack2(f[2], f[3]), E::pack2(f[4], f[5]), E::pack2(f[6], f[7]));
    *(uint4*)(part2 + P::KB_OFF + TL::k_byte(m, cc * 8)) = w;
  }
  // V^T: feature rows e x 4 chunks of 8 blocks (vt_block_of order), kVtRow bytes per row.
#pragma unroll
  for (int it = 0; it < D * kGroup / 8 / 256; ++it) {
    const int qi = it * 256 + tid;
    const int e = qi & (D - 1);
    const int cc = qi / D;
    float f[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int jj = g * kGroup + vt_block_of(cc, i);
      f[i] = jj < NT ? vb[(int64_t)jj * D + e] : 0.f;
    }
    const uint4 w = make_uint4(E::pack2(f[0], f[1]), E::pack2(f[2], f[3]), E::pack2(f[4], f[5]), E::pack2(f[6], f[7]));
    *(uint4*)(part2 + P::VT_OFF + e * kVtRow + cc * 16) = w;
  }
  __syncthreads();
  // Hbar^T: row e, chunk cc holds Hbar[8 cc .. 8 cc + 7][e].
#pragma unroll 2
  for (int it = 0; it < D * D / 8 / 256; ++it) {
    const int qi = it * 256 + tid;
    const int e = qi / CH;
    const int cc = qi % CH;
    float f[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) f[i] = hs[(cc * 8 + i) * HS + e];
    const uint4 w = make_uint4(E::pack2(f[0], f[1]), E::pack2(f[2], f[3]), E::pack2(f[4], f[5]), E::pack2(f[6], f[7]));
    *(uint4*)(out + TL::k_byte(e, cc * 8)) = w;
  }
}

// ---- tiles loaded straight into LDS -----------------------------------------
//
// The K/V tiles never pass through VGPRs: buffer_load_dwordx4 ... lds writes each lane's
// 16 bytes to LDS directly (zeros past the end of the slice), which frees the
// staging registers for deeper LDS-operand prefetching while two workgroups
// still share each CU.  Per block i, with one K and one V buffer, two barriers:
//   wait K_i -> barrier -> load V_i -> S = K_i Q^T -> softmax
//   -> wait V_i -> barrier -> load K_{i+1} -> O += V_i P
// Each barrier both publishes a landed tile and frees the other buffer, so V_i
// streams in during S + softmax and K_{i+1} during P.V.
//
// The products run on the 16x16x32 MFMA (v_mfma_f32_16x16x32_bf16 / _f16).  Under the
// chip's power limit it sustains about 11% more FLOP/s than the 32x32x16 form on
// real-valued operands (1.94 against 1.75 PFLOP/s in a bare MFMA stream, at 1.93
// against 1.72 GHz): the same work per cycle for less energy.  Lane l of a wave owns
// query rows l % 16 and 16 + l % 16 of the wave's 32 (query tiles qt = 0, 1), and holds,
// per 16-key tile kt of S^T = K Q^T, keys 16 kt + 4 (l / 16) + {0..3} of both rows; a
// row's statistics are reduced over its four lanes l % 16 + 16 g.  For P.V the 8 keys of
// a 32-key step s a lane holds (tiles 2s and 2s + 1) are its B-operand k-slots as they
// stand, and two transposing LDS reads fetch the V^T A-operand slots for the same keys.
//
// Tiles at D = 128 use 256-byte rows with XOR-swizzled 16-byte chunks: K chunk c of row r sits at
// c ^ (r & 15) (the A-operand reads of 16 rows by one 16-lane group touch 16 distinct
// chunks), V chunk c at c ^ 2 (r & 7) (the transposing reads of 32 lanes, rows 8 apart,
// touch 16 distinct chunks).  The phase-2 pack image is loaded the same way.

// PAIR: two query blocks per workgroup, one wave group (QWAVES waves) each, with
// their K/V tiles side by side in the K and V buffers.
template <int D_, int BT, bool PAIR = false>
struct K4D {
  static constexpr int D = D_;
  static constexpr int ROWB = 2 * D;                       // bytes of a tile row
  static constexpr int QWAVES = BT / 32;                   // waves of one query block
  static constexpr int QBLOCKS = PAIR ? 2 : 1;             // query blocks per workgroup
  static constexpr int WAVES = QWAVES * QBLOCKS;
  static constexpr int THREADS = WAVES * 64;
  static constexpr int TILE = BT * ROWB;                   // bytes of one K or V tile
  // A 1 KB direct load covers RPL rows; a query block's waves cover SPAN rows (a multiple of 16,
  // the period of the swizzles) in VW loads each.
  static constexpr int RPL = 1024 / ROWB;
  static constexpr int SPAN = RPL * QWAVES > 16 ? RPL * QWAVES : 16;
  static constexpr int VW = SPAN / (RPL * QWAVES);
  static constexpr int KT = BT / 16;                       // 16-key tiles of S per block
  static constexpr int KS = D / 32;                        // 32-feature k-steps
  static constexpr int DT = D / 16;                        // 16-feature tiles of O
  using PK = K4Pack<D>;
  static constexpr int KBUF = QBLOCKS * TILE > PK::HT_BYTES ? QBLOCKS * TILE : PK::HT_BYTES;
  static constexpr int VBUF = QBLOCKS * TILE > PK::PART2 ? QBLOCKS * TILE : PK::PART2;
  static_assert(BT % SPAN == 0, "load schedule");
  static_assert(WAVES == 4, "four-wave workgroups (BT = 128, or BT = 64 in pairs)");
  static_assert(PK::PART2 % (1024 * WAVES) == 0 && PK::HT_BYTES % (1024 * WAVES) == 0, "pack split");
};

// Byte offset in a V tile of the 8 bytes lane `lane` reads with ds_read_b64_tr_b16 for
// 16-feature tile dt and key rows row0 + 4 (lane / 16) + {0..3}: row row0 + 4 (lane / 16)
// + (lane % 16) / 4, features 16 dt + 4 (lane % 4) .. + 3 (chunk 2 dt + (lane % 4) / 2,
// half lane % 2).  row0 is a multiple of 16.
template <int D>
__device__ __forceinline__ int vtile_tr_byte(int row0, int dt, int lane) {
  const int r = row0 + 4 * (lane >> 4) + ((lane & 15) >> 2);
  const int c = 2 * dt + ((lane & 3) >> 1);
  return r * K4Tile<D>::ROWB + ((c ^ K4Tile<D>::vx(r)) << 4) + 8 * (lane & 1);
}

// Instruction-group masks of __builtin_amdgcn_sched_group_barrier.
constexpr int kSchedMfma = 0x008;
constexpr int kSchedDsRead = 0x100;

// ALL: dense attention (every key block exact, no selection read, no correction); a
// separate instantiation so that profiles tell the two launches apart.
// PERM: k and v are the token-major view (as pasa_block_stats_placed writes it), q is
// frame-major, and o is stored frame-major: the load and the store of a query row go
// through map_row.
// PAIR: two consecutive query blocks (or text query tiles) per workgroup (not ALL,
// not PERM).  Video blocks visit NS selected tiles each, so their barriers match
// (a shorter selection row, or a text pair spanning the prompt and the padding
// segment, idles through its partner's extra tiles); a pair past the last block
// repeats it and stores nothing.  Phase 2 visits the groups
// either block approximates; a wave whose block selects the whole group adds nothing
// there, so each block's result is the one the unpaired kernel computes.
// CROSS (with ALL): the slices of q and o have q_len rows, those of k and v T; the query tiles
// cover q's rows and each visits all of k's.
// o_heads (ALL): 0, o is [slice, row, D] as q; else o is [batch, row, head, D] with o_heads heads, the
// layout the projection after the attention reads.
// AL: k, v and pack are 16-byte aligned.
template <int D, int BT, bool ALL, bool PERM, bool PAIR, typename E, bool CROSS = false, bool AL = true>
__device__ __forceinline__ void k4_body(const uint16_t* __restrict__ q, const uint16_t* __restrict__ k,
                                        const uint16_t* __restrict__ v, const unsigned char* __restrict__ pack,
                                        const uint32_t* __restrict__ selmask, uint16_t* __restrict__ o, float scale,
                                        float c, int T, int NT, int NG, int NW, int xcd_chunk, int gamma_literal,
                                        int text, int text_valid, int n_text_wg, int nbh, int o_heads, int q_len,
                                        const RowMap& rm) {
  static_assert(!CROSS || (ALL && !PERM), "separate key rows: dense attention only");
  static_assert(!PAIR || (!ALL && !PERM), "pairs run selected video blocks only");
  constexpr bool all_tiles = ALL;
  using C = K4D<D, BT, PAIR>;
  using TL = K4Tile<D>;
  using PK = typename C::PK;
  using vec8 = typename E::vec8;
  constexpr int ROWB = C::ROWB;
  constexpr int KT = C::KT, KS = C::KS, DT = C::DT;
  // Two distinct LDS objects, so the compiler can tell loads into one from reads of the other.
  __shared__ __attribute__((aligned(1024))) unsigned char Ks[C::KBUF];
  __shared__ __attribute__((aligned(1024))) unsigned char Vs[C::VBUF];

  // Each slice holds T blocked (video) rows followed by `text` text rows, of which the
  // first text_valid are the prompt and the rest padding.  Two segments attend only
  // within themselves: [0, seg) with seg = T + text_valid, and the padding [seg, T + text).
  // The first n_text_wg workgroups (a multiple of 8) each own one tile of text query
  // rows of one segment and attend densely to that segment's keys; they are the
  // longest-running ones, so they go first.  The rest own one query block (a pair of
  // blocks with PAIR) of the video rows; wg & 7 names their XCD, and each XCD takes a
  // contiguous run of a slice's query blocks (shared K/V tiles in its L2).
  const int wg = blockIdx.x;
  const bool dense = wg < n_text_wg;
  const int seg = T + text_valid;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int half = PAIR ? wave / C::QWAVES : 0;  // query block (tile) of this wave within the workgroup
  const int qw = PAIR ? wave - half * C::QWAVES : wave;  // wave within its query block
  // A pair's second block (tile) past the last one repeats it and stores nothing.
  bool store_rows = true;
  int bh, qb, qbw = 0, qrow0, row_limit, kbeg = 0, kend = seg;
  int pair_tiles = 0;  // PAIR: tiles of the longer half (the shorter one idles through the rest)
  if (dense) {
    const int vtiles = (text_valid + BT - 1) / BT;
    const int qtiles = vtiles + (text - text_valid + BT - 1) / BT;
    const int units = (qtiles + C::QBLOCKS - 1) / C::QBLOCKS;
    bh = wg / units;
    if (bh >= nbh) return;  // padding of the text range to a multiple of 8
    qb = 0;
    const int t0 = (wg - bh * units) * C::QBLOCKS;
    store_rows = t0 + half < qtiles;
    const int qt = store_rows ? t0 + half : t0;
    auto seg_tiles = [&](int t) { return t < vtiles ? (seg + BT - 1) / BT : (T + text - seg + BT - 1) / BT; };
    if (PAIR) pair_tiles = max(seg_tiles(t0), seg_tiles(min(t0 + 1, qtiles - 1)));
    if (qt < vtiles) {
      qrow0 = T + qt * BT;
      row_limit = seg;
    } else {
      qrow0 = seg + (qt - vtiles) * BT;
      row_limit = T + text;
      kbeg = seg;
      kend = T + text;
    }
  } else {
    const int w = wg - n_text_wg;
    const int xcd = w & 7;
    const int slot = w >> 3;
    bh = slot / xcd_chunk;
    qb = (xcd * xcd_chunk + (slot - bh * xcd_chunk)) * C::QBLOCKS;
    const int nq = CROSS ? (q_len + BT - 1) / BT : NT;
    if (qb >= nq) return;
    store_rows = qb + half < nq;
    qbw = qb + (store_rows ? half : 0);
    qrow0 = qbw * BT;
    row_limit = CROSS ? q_len : T;
  }

  const int l16 = lane & 15;  // query row within a 16-row query tile; A-operand row
  const int g4 = lane >> 4;   // which 8 k-slots of an operand, which 4 rows of a result
  const int Ttot = T + text;
  const int64_t slice = (int64_t)bh * Ttot * D;
  const bool perm = PERM && slice_permuted(rm, bh);
  // This lane's two query rows (query tiles qt = 0, 1), and the frame-major rows their
  // output goes to (PERM: q is gathered through the same map).
  int qrow[2], qrow_st[2];
#pragma unroll
  for (int qt = 0; qt < 2; ++qt) {
    qrow[qt] = qrow0 + qw * 32 + 16 * qt + l16;
    qrow_st[qt] = perm ? map_row(qrow[qt], rm) : qrow[qt];
  }

  const uint32_t slice_bytes = (uint32_t)Ttot * D * 2u;
  const int q_rows = CROSS ? q_len : Ttot;
  const rsrc_t qr = make_rsrc(q + (int64_t)bh * q_rows * D, (uint32_t)q_rows * D * 2u);
  // Q as B operands: qf[qt][ks] holds features 32 ks + 8 g4 .. + 7 of row qrow[qt].
  vec8 qf[2][KS];
#pragma unroll
  for (int qt = 0; qt < 2; ++qt)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      qf[qt][ks] = as_vec8<E>(buf_load16(qr, ((uint32_t)(perm ? qrow_st[qt] : qrow[qt]) * D + ks * 32 + g4 * 8) * 2u));
  // Complete the Q loads now: vector-memory waits the compiler would place at their
  // first use inside the loop would also wait for the tile loads in flight there.
  wait_vmcnt<0>();

  // O^T accumulators: oacc[dt][qt] element i is feature 16 dt + 4 g4 + i of row qrow[qt].
  f32x4_t oacc[DT][2];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int qt = 0; qt < 2; ++qt)
#pragma unroll
      for (int i = 0; i < 4; ++i) oacc[dt][qt][i] = 0.f;
  // Running max, row sum and Gamma of the two rows: m is the same on the four lanes of a
  // row; l and Gamma are this lane's partial sums (its keys), added over the four at the end.
  float l_run[2] = {0.f, 0.f};
  float g_run[2] = {0.f, 0.f};
  float m_run[2] = {-INFINITY, -INFINITY};

  // The selection row is read-only here: constant address space -> scalar loads,
  // which wait on lgkmcnt and leave the in-flight tile loads alone.
  typedef const __attribute__((address_space(4))) uint32_t* const_u32_ptr;
  const const_u32_ptr mrow = (const_u32_ptr)(selmask + ((int64_t)bh * NT + qbw) * NW);
  // PAIR: the rows of both blocks (phase 2 visits the groups either approximates).
  const const_u32_ptr mrow0 = (const_u32_ptr)(selmask + ((int64_t)bh * NT + qb) * NW);
  const const_u32_ptr mrow1 = (const_u32_ptr)(selmask + ((int64_t)bh * NT + min(qb + 1, NT - 1)) * NW);

  // Direct-load lane constants.  Load (vw, n) of this wave covers RPL tile rows from
  // SPAN n + RPL (qw + QWAVES vw) of its query block's tile; lane l's 16 bytes land at chunk
  // l % CPR of row l / CPR (CPR chunks per row), so it fetches the logical chunk stored there.
  constexpr int RPL = C::RPL, SPAN = C::SPAN, CPR = ROWB / 16;
  const int lrow = lane / CPR;
  const int lch = lane % CPR;
  uint32_t k_lane[C::VW], v_lane[C::VW];
#pragma unroll
  for (int vw = 0; vw < C::VW; ++vw) {
    const int r = RPL * (qw + C::QWAVES * vw) + lrow;  // row mod SPAN
    k_lane[vw] = (uint32_t)(r * ROWB + ((lch ^ TL::kx(r)) << 4));
    v_lane[vw] = (uint32_t)(r * ROWB + ((lch ^ TL::vx(r)) << 4));
  }

  auto tile_load = [](u32x4_t rsrc, uint32_t lds, uint32_t off, uint32_t so) {
    if constexpr (AL)
      dma_load16_lds(rsrc, lds, off, so);
    else
      staged_load16_lds(rsrc, lds, off, so);
  };
  const u32x4_t kd = make_rsrc_words(k + slice, slice_bytes);
  const u32x4_t vd = make_rsrc_words(v + slice, slice_bytes);
  const uint32_t ks_lds = lds_addr(Ks);
  const uint32_t vs_lds = lds_addr(Vs);
  // This query block's K and V tiles (phase 1); phase 2 uses the whole buffers.
  const int tile_off = half * C::TILE;
  const uint32_t kt_lds = ks_lds + tile_off;
  const uint32_t vt_lds = vs_lds + tile_off;
  // A tile is BT key rows starting at row `row0` of the slice (rows past the slice read as zero).
  auto load_k = [&](int row0) {
    const uint32_t soff = (uint32_t)row0 * (uint32_t)ROWB;
#pragma unroll
    for (int vw = 0; vw < C::VW; ++vw)
#pragma unroll
      for (int n = 0; n < BT / SPAN; ++n)
        tile_load(kd, kt_lds + (SPAN * n + RPL * (qw + C::QWAVES * vw)) * ROWB, k_lane[vw] + SPAN * n * ROWB, soff);
  };
  auto load_v = [&](int row0) {
    const uint32_t soff = (uint32_t)row0 * (uint32_t)ROWB;
#pragma unroll
    for (int vw = 0; vw < C::VW; ++vw)
#pragma unroll
      for (int n = 0; n < BT / SPAN; ++n)
        tile_load(vd, vt_lds + (SPAN * n + RPL * (qw + C::QWAVES * vw)) * ROWB, v_lane[vw] + SPAN * n * ROWB, soff);
  };

  // MFMA A-operand offsets of K-layout tiles (K, Hbar^T, kbar): row l16 of a 16-row tile,
  // chunk 4 ks + g4 (features 32 ks + 8 g4 .. + 7).
  int kofs[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) kofs[ks] = l16 * ROWB + (((4 * ks + g4) ^ TL::kx(l16)) << 4);
  // The transposing V reads of 32-key step s: keys 32 s + 16 h2 + 4 g4 + {0..3} (h2 = 0, 1).
  int vofs[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) vofs[dt] = vtile_tr_byte<D>(0, dt, lane);

  int wsel = 0;
  int jall = 0;
  uint32_t bits = (!dense && !all_tiles && NW > 0) ? mrow[0] : 0u;
  auto next_selected = [&]() -> int {
    while (bits == 0u) {
      if (++wsel >= NW) return -1;
      bits = mrow[wsel];
    }
    const int j = 32 * wsel + __builtin_ctz(bits);
    bits &= bits - 1u;
    return j;
  };
  // Exact tiles in visiting order: a video query block takes its selected blocks in
  // ascending order, then the prompt rows [T, seg); a text query tile takes every row
  // of its segment [kbeg, kend).  Returns the tile's first row (-1 when done) and its
  // number of valid rows in nv.
  int tt = 0;
  auto next_tile = [&](int& nv) -> int {
    if (!dense) {
      const int j = all_tiles ? (jall < NT ? jall++ : -1) : next_selected();
      if (j >= 0) {
        nv = min(BT, T - j * BT);
        return j * BT;
      }
      kbeg = T;  // then the prompt rows
    }
    const int r = kbeg + tt * BT;
    if (r >= kend) return -1;
    ++tt;
    nv = min(BT, kend - r);
    return r;
  };

  // ---------------- Phase 1 ------------------------------------------------------
  // PAIR: the tile count of the longer half: for video blocks the longer of the two
  // selection rows (rows written by pasa_select all hold NS bits) plus the prompt
  // tiles; for text tiles, set above from the two segments.  The shorter half idles
  // through its partner's extra tiles below, so that the workgroup barriers match.
  int tiles_done = 0;
  if (PAIR && !dense) {
    int n0 = 0, n1 = 0;
    for (int w = 0; w < NW; ++w) {
      n0 += __builtin_popcount(mrow0[w]);
      n1 += __builtin_popcount(mrow1[w]);
    }
    pair_tiles = max(n0, n1) + (text_valid + BT - 1) / BT;
  }
  int nv_cur = 0;
  int blk = next_tile(nv_cur);
  if (blk >= 0) load_k(blk);
  while (blk >= 0) {
    int nv_nxt = 0;
    const int nxt = next_tile(nv_nxt);
    wait_vmcnt<0>();           // this wave's K_blk loads landed
    barrier_lds_reads_done();  // ... and every wave's; every wave is done reading the V buffer
    load_v(blk);

    // S^T = K Q^T: sacc[kt][qt] element i = key 16 kt + 4 g4 + i against row qrow[qt].
    f32x4_t sacc[KT][2];
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int qt = 0; qt < 2; ++qt)
#pragma unroll
        for (int i = 0; i < 4; ++i) sacc[kt][qt][i] = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int kt = 0; kt < KT; ++kt) {
        const vec8 a = as_vec8<E>(lds_ld<uint4>(Ks + tile_off, kofs[ks] + kt * 16 * ROWB));
#pragma unroll
        for (int qt = 0; qt < 2; ++qt) sacc[kt][qt] = E::mfma16(a, qf[qt][ks], sacc[kt][qt]);
      }
    // Keep 8 fragment reads in flight: each read feeds two MFMAs, consumed ~16 MFMAs
    // (~256 cycles) after it was issued, which covers the LDS latency.
    {
      constexpr int NR = KS * KT;
#pragma unroll
      for (int i = 0; i < 8; ++i) __builtin_amdgcn_sched_group_barrier(kSchedDsRead, 1, 0);
#pragma unroll
      for (int i = 0; i < NR - 8; ++i) {
        __builtin_amdgcn_sched_group_barrier(kSchedMfma, 2, 0);
        __builtin_amdgcn_sched_group_barrier(kSchedDsRead, 1, 0);
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) __builtin_amdgcn_sched_group_barrier(kSchedMfma, 2, 0);
    }

    const int nvalid = nv_cur;
    if (nvalid < BT) {
      // key 16 kt + 4 g4 + i is past the tile's rows iff 16 kt + i reaches lim;
      // comparing against immediates keeps no per-key constants live.
      const int lim = nvalid - 4 * g4;
#pragma unroll
      for (int kt = 0; kt < KT; ++kt)
#pragma unroll
        for (int qt = 0; qt < 2; ++qt)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (kt * 16 + i >= lim) sacc[kt][qt][i] = -INFINITY;
    }
    float mxc[2];
#pragma unroll
    for (int qt = 0; qt < 2; ++qt) {
      float mx = -INFINITY;
#pragma unroll
      for (int kt = 0; kt < KT; ++kt)
#pragma unroll
        for (int i = 0; i < 4; ++i) mx = fmaxf(mx, sacc[kt][qt][i]);
      mxc[qt] = quad16_max(mx) * c;
    }
    // One wave-uniform test per query tile: a tile whose 16 rows all kept their max skips
    // the 32 products of its O (they would multiply by exactly 1).
#pragma unroll
    for (int qt = 0; qt < 2; ++qt) {
      if (__any(mxc[qt] > m_run[qt])) {
        const float m_new = fmaxf(m_run[qt], mxc[qt]);
        const float alpha = fast_exp2(m_run[qt] - m_new);  // 0 on the first block, 1 if the max held
        m_run[qt] = m_new;
        l_run[qt] *= alpha;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
          for (int i = 0; i < 4; ++i) oacc[dt][qt][i] *= alpha;
      }
    }
    // P in the B-operand layout of 32-key step s: slots 0-3 = tile 2s, 4-7 = tile 2s + 1.
    // The row sum adds the fp32 p (as gpa.py:182-184 sums `score` before its bf16
    // cast), then adds the tile's sum to the rescaled l.
    vec8 pf[KT / 2][2];
#pragma unroll
    for (int qt = 0; qt < 2; ++qt) {
      float lsum[2] = {0.f, 0.f};
#pragma unroll
      for (int s = 0; s < KT / 2; ++s) {
        uint32_t w[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const f32x4_t& src = sacc[2 * s + (j >> 1)][qt];
          const float p0 = fast_exp2(fmaf(src[2 * (j & 1)], c, -m_run[qt]));
          const float p1 = fast_exp2(fmaf(src[2 * (j & 1) + 1], c, -m_run[qt]));
          w[j] = E::pack2(p0, p1);
          lsum[j & 1] += p0 + p1;
        }
        pf[s][qt] = as_vec8<E>((u32x4_t){w[0], w[1], w[2], w[3]});
      }
      l_run[qt] += lsum[0] + lsum[1];
    }
    // V_blk is waited for only now, so its load overlaps S and the softmax.
    wait_vmcnt<0>();
    barrier_lds_reads_done();  // every wave's part of V_blk landed; every wave is done reading K_blk
    if (nxt >= 0) load_k(nxt);
#pragma unroll
    for (int s = 0; s < KT / 2; ++s)
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        const uint2 lo = lds_read_tr16(Vs + tile_off, vofs[dt] + s * 32 * ROWB);
        const uint2 hi = lds_read_tr16(Vs + tile_off, vofs[dt] + s * 32 * ROWB + 16 * ROWB);
        const vec8 a = as_vec8<E>((u32x4_t){lo.x, lo.y, hi.x, hi.y});
#pragma unroll
        for (int qt = 0; qt < 2; ++qt) oacc[dt][qt] = E::mfma16(a, pf[s][qt], oacc[dt][qt]);
      }
    // Read-ahead for the transposing V reads: two per A operand, which feeds two MFMAs.
    {
      constexpr int NM = (KT / 2) * DT * 2;
#pragma unroll
      for (int i = 0; i < 8; ++i) __builtin_amdgcn_sched_group_barrier(kSchedDsRead, 1, 1);
#pragma unroll
      for (int i = 0; i < NM - 8; ++i) {
        __builtin_amdgcn_sched_group_barrier(kSchedMfma, 1, 1);
        __builtin_amdgcn_sched_group_barrier(kSchedDsRead, 1, 1);
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) __builtin_amdgcn_sched_group_barrier(kSchedMfma, 1, 1);
    }
    blk = nxt;
    nv_cur = nv_nxt;
    if (PAIR) ++tiles_done;
  }
  if (PAIR) {
    for (; tiles_done < pair_tiles; ++tiles_done)
#pragma unroll
      for (int b = 0; b < 2; ++b) barrier_lds_reads_done();  // the loop's barriers per tile
  }
  barrier_lds_reads_done();  // every wave is done reading the V buffer

  // ---------------- Phase 2 ------------------------------------------------------
  const int last_len = T - (NT - 1) * BT;
  const u32x4_t pd = make_rsrc_words(pack + (int64_t)bh * NG * PK::BYTES, (uint32_t)(NG * PK::BYTES));
  // V^T of the group: row 16 dt + l16, chunk g4 (blocks 4 g4 + {0..3}, 16 + 4 g4 + {0..3}).
  const int pv_base = PK::VT_OFF + l16 * kVtRow + g4 * 16;
  const int ng_run = (dense || all_tiles) ? 0 : NG;  // text rows and dense attention: no correction term
  // Groups with at least one unselected in-range block (of either block of a pair),
  // in ascending order.
  auto inrange_of = [&](int g) -> uint32_t {
    const int nin = min(kGroup, NT - g * kGroup);
    return nin >= 32 ? 0xffffffffu : ((1u << nin) - 1u);
  };
  auto approx_of = [&](int g) -> uint32_t { return inrange_of(g) & ~mrow[g]; };
  auto visit_of = [&](int g) -> uint32_t {
    return PAIR ? inrange_of(g) & ~(mrow0[g] & mrow1[g]) : approx_of(g);
  };
  auto next_group = [&](int g) -> int {
    for (++g; g < ng_run; ++g)
      if (visit_of(g) != 0u) return g;
    return -1;
  };
  // A group's pack is two parts: kbar + V^T (part 2, into Vs) and Hbar^T (into Ks).
  // Part 2 of the next group loads while this group's Hbar^T product runs, and the
  // next Hbar^T loads while the next group's scores and P.V^ run.  Two barriers per
  // group: after P.V^ (part 2 of g read everywhere, Hbar^T of g landed) and after the
  // Hbar^T product (Hbar^T of g read everywhere, part 2 of the next group landed).
  constexpr int HT_LOADS = PK::HT_BYTES / 1024 / C::WAVES;
  constexpr int P2_LOADS = PK::PART2 / 1024 / C::WAVES;
  auto load_part2 = [&](int g) {
    const uint32_t gsoff = (uint32_t)(g * PK::BYTES);
#pragma unroll
    for (int n = 0; n < P2_LOADS; ++n) {
      const int kb = n * C::WAVES + wave;
      tile_load(pd, vs_lds + kb * 1024, (uint32_t)(PK::HT_BYTES + kb * 1024 + lane * 16), gsoff);
    }
  };
  auto load_ht = [&](int g) {
    const uint32_t gsoff = (uint32_t)(g * PK::BYTES);
#pragma unroll
    for (int n = 0; n < HT_LOADS; ++n) {
      const int kb = n * C::WAVES + wave;  // 1 KB piece of Hbar^T
      tile_load(pd, ks_lds + kb * 1024, (uint32_t)(kb * 1024 + lane * 16), gsoff);
    }
  };
  int g = next_group(-1);
  if (g >= 0) {  // phase 1 ended with a barrier after the last reads of Ks and Vs
    load_part2(g);
    load_ht(g);
    wait_vmcnt<HT_LOADS>();    // this wave's part 2 of group g landed (Hbar^T may be in flight)
    barrier_lds_reads_done();  // ... and every wave's
  }
  while (g >= 0) {
    const int gn = next_group(g);
    const uint32_t approx = approx_of(g);

    // PAIR: a wave whose block selects the whole group adds nothing to o (its weights are 0, and 0 times a
    // sum that is not finite would be NaN).  The branches enclose just the two sums: around the scores and
    // q Hbar as well they cost 1 to 2%, so 0 to 0.5% (24 heads x 119 k rows, three comparisons with neither:
    // 28.3 ms against 28.2, 27.7 against 27.6, 27.9 against 28.3).
    const bool mine = !PAIR || approx != 0u;
    // s-bar^T = kbar Q^T: sb[bt][qt] element i = block 16 bt + 4 g4 + i of the group.
    f32x4_t sb[2][2];
#pragma unroll
    for (int bt = 0; bt < 2; ++bt)
#pragma unroll
      for (int qt = 0; qt < 2; ++qt)
#pragma unroll
        for (int i = 0; i < 4; ++i) sb[bt][qt][i] = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int bt = 0; bt < 2; ++bt) {
        const vec8 a = as_vec8<E>(lds_ld<uint4>(Vs, PK::KB_OFF + kofs[ks] + bt * 16 * ROWB));
#pragma unroll
        for (int qt = 0; qt < 2; ++qt) sb[bt][qt] = E::mfma16(a, qf[qt][ks], sb[bt][qt]);
      }
    // Blocks of the group that are selected (or past NT) drop out: element i of sb[bt]
    // is block 16 bt + 4 g4 + i, so its keep mask is one sign-extended bit of approx >> 4 g4.
    const uint32_t ah = approx >> (4 * g4);
    float m_new[2], alpha[2];
#pragma unroll
    for (int qt = 0; qt < 2; ++qt) {
      float gmx = -INFINITY;
#pragma unroll
      for (int bt = 0; bt < 2; ++bt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const uint32_t keep = (uint32_t)__builtin_amdgcn_sbfe((int)ah, 16 * bt + i, 1);
          sb[bt][qt][i] = __uint_as_float((__float_as_uint(sb[bt][qt][i]) & keep) | (~keep & 0xff800000u));  // -inf if dropped
          gmx = fmaxf(gmx, sb[bt][qt][i]);
        }
      m_new[qt] = fmaxf(m_run[qt], quad16_max(gmx) * c);
      alpha[qt] = fast_exp2(m_run[qt] - m_new[qt]);
      m_run[qt] = m_new[qt];
      l_run[qt] *= alpha[qt];
      if (!gamma_literal) g_run[qt] *= alpha[qt];
    }
#pragma unroll
    for (int qt = 0; qt < 2; ++qt)
      if (__any(alpha[qt] != 1.f)) {
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
          for (int i = 0; i < 4; ++i) oacc[dt][qt][i] *= alpha[qt];
      }
    float psum[2];
    vec8 pbf[2];
#pragma unroll
    for (int qt = 0; qt < 2; ++qt) {
      uint32_t w[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const f32x4_t& src = sb[j >> 1][qt];
        const float p0 = fast_exp2(fmaf(src[2 * (j & 1)], c, -m_new[qt]));
        const float p1 = fast_exp2(fmaf(src[2 * (j & 1) + 1], c, -m_new[qt]));
        psum[qt] = j == 0 ? p0 + p1 : psum[qt] + (p0 + p1);  // no 0 + x: x may be -0
        w[j] = E::pack2(p0, p1);
      }
      pbf[qt] = as_vec8<E>((u32x4_t){w[0], w[1], w[2], w[3]});
    }
    // Gamma += sum_j p_j * n_j.  Every block holds BT rows except the last one, NT - 1,
    // which holds last_len: BT * sum(p) (exact, BT being a power of two), corrected for
    // that block in the one group holding it.
    float gsum[2] = {psum[0] * (float)BT, psum[1] * (float)BT};
    if (g == NG - 1 && last_len != BT) {
      const int mm_last = (NT - 1) - g * kGroup;  // block 16 bt + 4 g4 + i of the group
      if (g4 == ((mm_last >> 2) & 3)) {
#pragma unroll
        for (int qt = 0; qt < 2; ++qt) {
          float sl = sb[0][qt][0];
#pragma unroll
          for (int bt = 0; bt < 2; ++bt)
#pragma unroll
            for (int i = 0; i < 4; ++i)
              if (16 * bt + i == (mm_last & 16) + (mm_last & 3)) sl = sb[bt][qt][i];
          gsum[qt] += fast_exp2(fmaf(sl, c, -m_new[qt])) * (float)(last_len - BT);
        }
      }
    }
#pragma unroll
    for (int qt = 0; qt < 2; ++qt) {
      g_run[qt] += gsum[qt];
      psum[qt] = quad16_sum(psum[qt]);
    }
    if (mine) {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        const vec8 a = as_vec8<E>(lds_ld<uint4>(Vs, pv_base + dt * 16 * kVtRow));
#pragma unroll
        for (int qt = 0; qt < 2; ++qt) oacc[dt][qt] = E::mfma16(a, pbf[qt], oacc[dt][qt]);
      }
    }
    wait_vmcnt<0>();           // this wave's Hbar^T of group g landed (nothing else is in flight)
    barrier_lds_reads_done();  // every wave is done reading part 2 of group g; Hbar^T of g is in place
    if (gn >= 0) load_part2(gn);

    // r^T = Hbar^T Q^T: racc[dt][qt] element i = feature 16 dt + 4 g4 + i of q.Hbar.
    f32x4_t racc[DT][2];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int qt = 0; qt < 2; ++qt)
#pragma unroll
        for (int i = 0; i < 4; ++i) racc[dt][qt][i] = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        const vec8 a = as_vec8<E>(lds_ld<uint4>(Ks, kofs[ks] + dt * 16 * ROWB));
#pragma unroll
        for (int qt = 0; qt < 2; ++qt) racc[dt][qt] = E::mfma16(a, qf[qt][ks], racc[dt][qt]);
      }
    if (mine) {
#pragma unroll
      for (int qt = 0; qt < 2; ++qt) {
        const float f = psum[qt] * scale;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
          for (int i = 0; i < 4; ++i) oacc[dt][qt][i] = fmaf(racc[dt][qt][i], f, oacc[dt][qt][i]);
      }
    }
    if (gn >= 0) wait_vmcnt<0>();  // this wave's part 2 of group gn landed
    barrier_lds_reads_done();      // every wave is done reading Hbar^T of g; part 2 of gn is in place
    if (gn >= 0) load_ht(gn);
    g = gn;
  }

  const int ob = ALL && o_heads > 0 ? bh / o_heads : bh;  // o's rows are o_heads (or one) rows of D apart
  const int on = ALL && o_heads > 0 ? o_heads : 1;
  uint16_t* const oslice = o + ((int64_t)ob * q_rows * on + (bh - ob * on)) * D;
  const int ostride = on * D;
  // O = A / (L + Gamma): one correctly rounded reciprocal per row, then products.
#pragma unroll
  for (int qt = 0; qt < 2; ++qt) {
    const float inv = 1.f / (quad16_sum(l_run[qt]) + quad16_sum(g_run[qt]));
    if (store_rows && qrow[qt] < row_limit) {
      uint16_t* orow = oslice + (int64_t)qrow_st[qt] * ostride;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        uint2 w;
        w.x = E::pack2(oacc[dt][qt][0] * inv, oacc[dt][qt][1] * inv);
        w.y = E::pack2(oacc[dt][qt][2] * inv, oacc[dt][qt][3] * inv);
        *(uint2*)(orow + dt * 16 + 4 * g4) = w;
      }
    }
  }
}

#define PASA_K4_PARAMS                                                                                         \
  const uint16_t *__restrict__ q, const uint16_t *__restrict__ k, const uint16_t *__restrict__ v,              \
      const unsigned char *__restrict__ pack, const uint32_t *__restrict__ selmask, uint16_t *__restrict__ o,  \
      float scale, float c, int T, int NT, int NG, int NW, int xcd_chunk, int gamma_literal, int text,         \
      int text_valid, int n_text_wg, int nbh, int o_heads, int q_len, RowMap rm
#define PASA_K4_ARGS                                                                                        \
  q, k, v, pack, selmask, o, scale, c, T, NT, NG, NW, xcd_chunk, gamma_literal, text, text_valid, n_text_wg, \
      nbh, o_heads, q_len, rm

// D = 128: two waves per SIMD (256 VGPRs each), two workgroups of 64 KB of LDS per CU.
template <int BT, bool ALL, bool PERM, bool PAIR = false, typename E = Bf16>
__global__ __attribute__((amdgpu_flat_work_group_size(1, 256), amdgpu_waves_per_eu(2, 2)))
void k4_sparse_attn_dma(PASA_K4_PARAMS) {
  k4_body<128, BT, ALL, PERM, PAIR, E>(PASA_K4_ARGS);
}

// Dense attention of q_len query rows to T key rows per slice (the text cross-attention of a DiT
// block).  32,760 x 512 at 12 heads: 128 us, where PyTorch's SDPA takes 244.
template <typename E>
__global__ __attribute__((amdgpu_flat_work_group_size(1, 256), amdgpu_waves_per_eu(2, 2)))
void k4_cross_attn(PASA_K4_PARAMS) {
  k4_body<128, 128, true, false, false, E, true>(PASA_K4_ARGS);
}

// D = 64: half the accumulators, operands and tile bytes.
template <int D, int BT, bool AL>
__global__ __attribute__((amdgpu_flat_work_group_size(1, 256), amdgpu_waves_per_eu(2)))
void k4_sparse_attn(PASA_K4_PARAMS) {
  k4_body<D, BT, false, false, BT == 64, Bf16, false, AL>(PASA_K4_ARGS);
}

// The D = 128 kernels where k, v or pack is not 16-byte aligned: tiles staged through registers (a few of
// which spill at block 128).
template <int BT, bool ALL, bool PERM, bool PAIR, typename E, bool CROSS = false>
__global__ __attribute__((amdgpu_flat_work_group_size(1, 256), amdgpu_waves_per_eu(2, 2)))
void k4_staged(PASA_K4_PARAMS) {
  k4_body<128, BT, ALL, PERM, PAIR, E, CROSS, false>(PASA_K4_ARGS);
}
#undef PASA_K4_PARAMS
#undef PASA_K4_ARGS

// Whether K and V tiles (and the pack) can load straight into LDS.
static bool aligned16(const void* k, const void* v, const void* pack = nullptr) {
  return (((uintptr_t)k | (uintptr_t)v | (uintptr_t)pack) & 15u) == 0;
}

size_t k4_pack_bytes(int D, int BT) {
  if (BT != 64 && BT != 128) return 0;
  return D == 128 ? K4Pack<128>::BYTES : (D == 64 ? K4Pack<64>::BYTES : 0);
}

hipError_t launch_pack_phase2(const float* kc, const float* vc, const float* hgroup, void* pack,
                              int bh, int T, int D, int BT, bool f16, hipStream_t stream) {
  const int NT = (T + BT - 1) / BT;
  const int NG = (NT + kGroup - 1) / kGroup;
  dim3 grid(NG, bh);
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, grid, dim3(256), 0, stream, kc, vc, hgroup, (unsigned char*)pack, NT, NG);
    return hipGetLastError();
  };
  if ((BT != 64 && BT != 128) || (D != 64 && D != 128) || (f16 && D != 128)) return hipErrorInvalidValue;
  if (f16) return go(k4_pack_xor<128, F16>);
  return D == 128 ? go(k4_pack_xor<128, Bf16>) : go(k4_pack_xor<64, Bf16>);
}

hipError_t launch_sparse_attn(const void* q, const void* k, const void* v, const void* pack,
                              const int32_t* idx, const uint32_t* selmask, void* o, float scale,
                              int bh, int T, int text, int text_valid, int D, int BT, int NS,
                              int gamma_literal, const RowMap* rm, bool f16, hipStream_t stream) {
  if (text > 0 && D != 128) return hipErrorInvalidValue;  // the text segment is a D = 128 feature
  if (f16 && D != 128) return hipErrorInvalidValue;       // so are fp16 inputs
  if (text_valid < 0 || text_valid > text) return hipErrorInvalidValue;
  const int NT = (T + BT - 1) / BT;
  const int NG = (NT + kGroup - 1) / kGroup;
  const int NW = (NT + 31) / 32;
  const int xcd_chunk = (NT + 7) / 8;
  const int text_qtiles = (text_valid + BT - 1) / BT + (text - text_valid + BT - 1) / BT;
  const int n_text_wg = (bh * text_qtiles + 7) / 8 * 8;
  dim3 grid(n_text_wg + 8 * bh * xcd_chunk);
  const float c = scale * kLog2e;
  auto a = (const uint16_t*)q;
  auto b = (const uint16_t*)k;
  auto cc = (const uint16_t*)v;
  auto pk = (const unsigned char*)pack;
  auto oo = (uint16_t*)o;
  const bool aligned = aligned16(k, v, pack);
  auto dma = [&](auto direct, auto staged, dim3 g, int chunk, int n_text, const RowMap& map) {
    hipLaunchKernelGGL((aligned ? direct : staged), g, dim3(256), 0, stream, a, b, cc, pk, selmask, oo, scale, c, T, NT,
                       NG, NW, chunk, gamma_literal, text, text_valid, n_text, bh, 0, 0, map);
  };
  static_assert(K4D<128, 128>::THREADS == 256 && K4D<128, 64, true>::THREADS == 256 &&
                    K4D<64, 128>::THREADS == 256 && K4D<64, 64, true>::THREADS == 256,
                "four-wave workgroups");
  // Query blocks (and text tiles) in pairs at block size 64: each XCD takes a contiguous run of a
  // slice's pairs.
  const int pair_chunk = ((NT + 1) / 2 + 7) / 8;
  const int n_text_pairs = (bh * ((text_qtiles + 1) / 2) + 7) / 8 * 8;
  const dim3 grid_pairs(n_text_pairs + 8 * bh * pair_chunk);
  if (rm != nullptr) {  // token-major view of frame-major slices: D = 128, BT = 128 only
    if (D != 128 || BT != 128) return hipErrorInvalidValue;
    if (f16)
      dma(k4_sparse_attn_dma<128, false, true, false, F16>, k4_staged<128, false, true, false, F16>, grid, xcd_chunk,
          n_text_wg, *rm);
    else
      dma(k4_sparse_attn_dma<128, false, true, false, Bf16>, k4_staged<128, false, true, false, Bf16>, grid, xcd_chunk,
          n_text_wg, *rm);
  } else if (D == 128 && BT == 128) {
    if (f16)
      dma(k4_sparse_attn_dma<128, false, false, false, F16>, k4_staged<128, false, false, false, F16>, grid, xcd_chunk,
          n_text_wg, RowMap{});
    else
      dma(k4_sparse_attn_dma<128, false, false, false, Bf16>, k4_staged<128, false, false, false, Bf16>, grid, xcd_chunk,
          n_text_wg, RowMap{});
  } else if (D == 128 && BT == 64) {
    if (f16)
      dma(k4_sparse_attn_dma<64, false, false, true, F16>, k4_staged<64, false, false, true, F16>, grid_pairs, pair_chunk,
          n_text_pairs, RowMap{});
    else
      dma(k4_sparse_attn_dma<64, false, false, true, Bf16>, k4_staged<64, false, false, true, Bf16>, grid_pairs,
          pair_chunk, n_text_pairs, RowMap{});
  } else if (D == 64 && BT == 128) {
    dma(k4_sparse_attn<64, 128, true>, k4_sparse_attn<64, 128, false>, grid, xcd_chunk, 0, RowMap{});
  } else if (D == 64 && BT == 64) {
    dma(k4_sparse_attn<64, 64, true>, k4_sparse_attn<64, 64, false>, grid_pairs, pair_chunk, 0, RowMap{});
  } else {
    return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_dense_attn(const void* q, const void* k, const void* v, void* o, float scale, int bh,
                             int T, int text, int text_valid, int o_heads, bool f16, hipStream_t stream) {
  constexpr int BT = 128;
  if (T < 1 || text < 0 || text_valid < 0 || text_valid > text) return hipErrorInvalidValue;
  const int NT = (T + BT - 1) / BT;
  const int xcd_chunk = (NT + 7) / 8;
  const int text_qtiles = (text_valid + BT - 1) / BT + (text - text_valid + BT - 1) / BT;
  const int n_text_wg = (bh * text_qtiles + 7) / 8 * 8;
  dim3 grid(n_text_wg + 8 * bh * xcd_chunk);
  auto launch = [&](auto direct, auto staged) {
    hipLaunchKernelGGL((aligned16(k, v) ? direct : staged), grid, dim3(K4D<128, BT>::THREADS), 0, stream, (const uint16_t*)q, (const uint16_t*)k,
                       (const uint16_t*)v, nullptr, nullptr, (uint16_t*)o, scale, scale * kLog2e, T, NT, 0, 0,
                       xcd_chunk, 1, text, text_valid, n_text_wg, bh, o_heads, 0, RowMap{});
  };
  if (f16)
    launch(k4_sparse_attn_dma<BT, true, false, false, F16>, k4_staged<BT, true, false, false, F16>);
  else
    launch(k4_sparse_attn_dma<BT, true, false, false, Bf16>, k4_staged<BT, true, false, false, Bf16>);
  return hipGetLastError();
}

hipError_t launch_cross_attn(const void* q, const void* k, const void* v, void* o, float scale, int bh, int q_len,
                             int kv_len, int o_heads, bool f16, hipStream_t stream) {
  constexpr int BT = 128;
  if (q_len < 1 || kv_len < 1) return hipErrorInvalidValue;
  const int xcd_chunk = ((q_len + BT - 1) / BT + 7) / 8;
  auto launch = [&](auto direct, auto staged) {
    hipLaunchKernelGGL((aligned16(k, v) ? direct : staged), dim3(8 * bh * xcd_chunk), dim3(K4D<128, BT>::THREADS), 0, stream, (const uint16_t*)q,
                       (const uint16_t*)k, (const uint16_t*)v, nullptr, nullptr, (uint16_t*)o, scale, scale * kLog2e,
                       kv_len, (kv_len + BT - 1) / BT, 0, 0, xcd_chunk, 1, 0, 0, 0, bh, o_heads, q_len, RowMap{});
  };
  if (f16)
    launch(k4_cross_attn<F16>, k4_staged<BT, true, false, false, F16, true>);
  else
    launch(k4_cross_attn<Bf16>, k4_staged<BT, true, false, false, Bf16, true>);
  return hipGetLastError();
}

}  // namespace pasa
