// K4 for shapes the tuned kernels do not take: fp32 q, k, v; any head dim up to 128; any
// group size; block sizes 16 .. 256; dense attention of those types and head dims.
//
// Reference: pisa_pg_fwd_kernel, svg/kernels/triton/group_pisa_attention.py:135-262; any float
// dtype (:380), any group size (:312) and any power-of-two block size (:311).  Rounding: for
// 16-bit inputs kc, vc and Hbar are rounded to the input type at their use, P and P-bar before
// their products, and the output at its store, as the reference does; fp32 inputs are not
// rounded anywhere.
//
// Every product runs on the 16x16 MFMAs: 16x16x32 for bf16 and fp16, 16x16x4 (fp32 operands,
// fp32 accumulation) for fp32.  Both leave element i of lane l = row 4 (l / 16) + i, column
// l % 16 of the result, so one kernel serves the three types: S^T[key][q] = K Q^T,
// O^T[e][q] += V^T P^T and O^T += Hbar^T Q^T f, a lane holding query l % 16 of each 16-row
// query tile throughout (the softmax of a row stays in its four lanes, and P never moves
// between lanes).
//   16 bits: a k-step of 32 takes slots {4g .. 4g + 3, 16 + 4g .. 16 + 4g + 3} (g = l / 16),
//     the slots the transposing LDS reads deliver for V^T and Hbar^T and the ones a lane's
//     scores already are; K rows are staged with their features in that order, so a K operand
//     is one 16-byte read.
//   fp32: a step of 4 takes slots {4g + i}, so one 16-byte read of a K row feeds four steps and
//     the scores are P's operands as they stand; V and Hbar operands are 4-byte reads.
//
// Work split.  A workgroup is four waves of RW query rows.  BT >= 64 (TEAM = 4): the waves share
// a 64-row (RW 16) or 128-row (RW 32) tile of one query block, its selected blocks and the K/V
// chunks staged in LDS.  BT < 64 (TEAM = 1): each wave owns a 16- or 32-row query block (fp32: 16
// rows of one) and walks its own selected blocks through chunks of its own in LDS, with no
// workgroup barrier; so all 64 lanes work at any block size, and the four waves share the
// operands of phase 2, which every query block reads in full.  The next chunk's rows load into
// registers while one is multiplied.
//
// fp32 with TEAM = 4 (Split32) runs on the bf16 MFMA: every operand is split into three bf16 planes,
// x = x1 + x2 + x3 to its last bit (q in registers, K/V/V^/Hbar as they are staged, P after its
// exponential), and a product is six MFMAs: x1 y1 into one sum, the smaller five into another, so
// that they round at their own size.  Six bf16 MFMAs take 3/8 of the fp32 MFMA's time for the same
// product, and round less: one addition per 32 terms where the fp32 MFMA rounds after every product.
// Error against 64 bits at 12 heads x 7,800 rows, D 128, block 64: 7.2e-7 with one FMA per lane,
// 5.0e-7 on the fp32 MFMA, 3.8e-7 so (with q and k of mean 1 and 3, where the scores cancel, 1.8e-6
// and 1.7e-6 at 2 heads x 3,000 rows; one sum over all 128 features rounds 8% more than one FMA per
// lane); K4 there 2.07 ms, 0.66 and 0.46.
// TEAM = 1 stays on the fp32 MFMA (Any32): a wave would split its own K/V rows for 16 queries.
// Its fp32 sums are taken in short chains (16 features, a chunk of keys, 32 rows of Hbar) that are
// then added: where q and k have a common mean the scores' rounding is the error, and it grows with
// the chain (2 heads x 1,000 rows, D 128, block 32, means 1 and 3: 1.6e-6 with one FMA per lane, 3.0e-6
// with chains of 64 features, which are 1 to 3% faster, 1.4e-6 so).
//
// What bounds it: Split32, the MFMA pipe (75 GFLOP of fp32, so 450 of bf16, in 0.46 ms, where a
// large bf16 product takes 0.34), with a third as many VALU instructions for the splits;
// Any32, the fp32 MFMA (153 TFLOP/s in a large product); 16 bits, the latency of the staged loads
// and, in phase 2, of Hbar (16 heads x 8,610 rows, D 96, block 32, groups of 16: 149 GFLOP in
// 0.35 ms, half of it phase 2, where one FMA per lane took 9.7 ms with half its lanes idle).
#include <initializer_list>
#include <type_traits>

#include "common.h"
#include "kernels.h"

namespace pasa {

namespace {

struct Split32 {  // fp32 rows, three bf16 planes of each in LDS
  using M = Bf16;
  static constexpr int ES = 4;
  static constexpr bool SPLIT = true;
  using frag = bf16x8_t;
};
struct Any32 {  // fp32 rows in LDS, fp32 MFMA
  static constexpr int ES = 4;
  static constexpr bool SPLIT = false;
  using frag = f32x4_t;
  using Team4 = Split32;
};
template <typename M_>
struct Any16 {
  using M = M_;
  static constexpr int ES = 2;
  static constexpr bool SPLIT = false;
  using frag = typename M::vec8;
  using Team4 = Any16;
};

constexpr int pow2_at_least(int x) {
  int p = 1;
  while (p < x) p *= 2;
  return p;
}

// DP: the head dim padded to 64, 96 or 128 (zeros in LDS and registers).
template <typename E, int DP, int TEAM, int RW>
struct AnyCfg {
  static constexpr int ES = E::ES;
  static constexpr bool SPLIT = E::SPLIT;
  static constexpr bool F32 = ES == 4 && !SPLIT;
  static constexpr int LE = F32 ? 4 : 2;         // bytes of an element in LDS
  static constexpr int NPL = SPLIT ? 3 : 1;      // planes of every row in LDS
  static constexpr int QT = RW / 16;             // 16-row query tiles per wave
  static constexpr int ROWS = 4 * RW;            // query rows per workgroup (TEAM = 4)
  static constexpr int NF = DP * LE / 64;  // 64-byte feature steps per row: one fragment each
  static constexpr int DT = DP / 16;       // 16-feature tiles of O
  // Keys per chunk: what two workgroups per CU leave room for (fp32 planes: 27 KB each of K and V; the
  // fp32 pass over a split tile keeps its count, whose registers the split pass needs too).
  static constexpr int KC = TEAM == 1 ? (F32 ? 16 : 32) : (ES == 4 ? 32 : 64);
  // Row strides.  K: an odd number of 16-byte chunks, so that 16 rows read at one chunk touch 16
  // distinct bank groups.  V in 16 bits: twice an odd number of chunks, so that the 8 rows x 32
  // bytes half a wave transposes do; in fp32 4 rows x 64 bytes, four rows apart, already do.
  static constexpr int KROW = DP * LE + 16;
  static constexpr int VROW = DP * LE + (F32 ? 16 : 32);
  static constexpr int SLAB = NPL * KC * (KROW + VROW);
  static constexpr int KZ = 32;                  // blocks per zero-order chunk
  static constexpr int HR = F32 || (SPLIT && DP == 96) ? 32 : (SPLIT ? 64 : DP);  // Hbar rows staged at a time
  static constexpr int Z_BYTES = NPL * KZ * (KROW + VROW);
  static constexpr int H_BYTES = NPL * HR * VROW;
  static constexpr int P1 = (4 / TEAM) * SLAB;
  // SPLIT: Hbar takes the place of the zero-order rows, whose chunk is done by then.
  static constexpr int P2 = SPLIT ? (Z_BYTES > H_BYTES ? Z_BYTES : H_BYTES) : Z_BYTES + H_BYTES;
  static constexpr int LDS = P1 > P2 ? P1 : P2;
  static constexpr int CH = DP * ES / 16;        // 16-byte chunks per row
  static constexpr int CHP = pow2_at_least(CH);  // lanes per staged row
  static constexpr int TT = 64 * TEAM;
  static constexpr int RPP = TT / CHP;           // rows per staging pass
  static constexpr int PASSES = KC / RPP;
  static constexpr int C4 = DP / 4;              // 4-feature pieces of a statistics row
  static constexpr int C4P = pow2_at_least(C4);
  static constexpr int RPP4 = 256 / C4P;
  static_assert(PASSES * RPP == KC && KZ % RPP4 == 0 && HR % RPP4 == 0, "staging split");
};

// Element-wise forms, for rows that are not whole 16-byte chunks or not aligned to them: 16 bytes of
// a row from chunk c on, and four floats of a statistics row; elements past D are zero.
template <int ES>
__device__ __forceinline__ uint4 load_elems(const unsigned char* row, int c, int D) {
  uint32_t w[4] = {0u, 0u, 0u, 0u};
  if constexpr (ES == 2) {
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (8 * c + i < D) w[i >> 1] |= (uint32_t)reinterpret_cast<const uint16_t*>(row)[8 * c + i] << (16 * (i & 1));
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (4 * c + i < D) w[i] = reinterpret_cast<const uint32_t*>(row)[4 * c + i];
  }
  return make_uint4(w[0], w[1], w[2], w[3]);
}

// Four fp32 as three bf16 each, x = x1 + x2 + x3, each part the rounded rest of the ones before it;
// together they hold all 24 bits of x down to 2^-110, below which x3 is a bf16 subnormal: operands are
// split times a power of two (kUp below), which makes the parts of every fp32 exact.  The rest of an
// infinity, of a NaN or of an x that rounds to infinity is NaN.
__device__ __forceinline__ void split4(const float (&x)[4], uint2 (&pl)[3]) {
  float r[4] = {x[0], x[1], x[2], x[3]};
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    pl[i] = make_uint2(Bf16::pack2(r[0], r[1]), Bf16::pack2(r[2], r[3]));
    r[0] -= __uint_as_float(pl[i].x << 16);
    r[1] -= __uint_as_float(pl[i].x & 0xffff0000u);
    r[2] -= __uint_as_float(pl[i].y << 16);
    r[3] -= __uint_as_float(pl[i].y & 0xffff0000u);
  }
}

// For j = 0, 1: hi[j] += a1 b1 and lo[j] += the five products of the next orders of a = a[j], smallest
// first.  With |x2| <= 2^-8 |x| and |x3| <= 2^-17 |x| what is left out (x2 y3 + x3 y2 + x3 y3) is at most
// 2^-24 (1 + 2^-10) of a b, 0.054 of 2^-24 on average (up to 3.9 with x1 cut instead of rounded).  The two
// sums alternate, held in this order: an MFMA that adds to the one before waits for it (the call above,
// when its loads were slower: 625 us with one after the other, 615 in the compiler's order, 609 so).
__device__ __forceinline__ void mfma_split(const bf16x8_t (&a)[2][3], const bf16x8_t (&b)[3], f32x4_t* const (&hi)[2],
                                           f32x4_t* const (&lo)[2]) {
  constexpr int PA[6] = {2, 0, 0, 1, 1, 0}, PB[6] = {0, 0, 2, 1, 0, 1};
#pragma unroll
  for (int i = 0; i < 6; ++i) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      f32x4_t& t = PA[i] + PB[i] == 0 ? *hi[j] : *lo[j];
      t = Bf16::mfma16(a[j][PA[i]], b[PB[i]], t);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
}

// Powers of two that Split32 multiplies operands by before their split (16 or more cover the subnormals,
// whose last bit is 2^-149 where a bf16 part's is 2^-133).  The scores are then 2^40, O 2^56 times
// their values, in P V^ as in q Hbar.  K stays as it is: with q below 2^88 (above, its parts are not
// finite) a part below 2^-133 of it moves no exponent c s by more than 2^-27.
// Without them v of 2^-118 comes out to 6.7e-6, of 2^-130 to 2.8e-2; with them as with fp32 products.
// They cost 1 to 2% (12 heads x 7,800 rows, block 64: D 128 564 -> 571 us, D 64 276 -> 281).
constexpr float kUpQ = 0x1p40f, kUpP = 0x1p16f, kUpV = 0x1p40f, kUpH = 0x1p16f;
constexpr float kDownS = 0x1p-40f, kDownO = 0x1p-56f;
constexpr float kMinSplitC = 0x1p-40f, kMaxSplitC = 0x1p12f;  // the c that this holds for

constexpr uint32_t kOutside = 0x80000000u;  // a buffer offset past every chunk: the load gives zeros

// One workgroup's tile of k4_any_mfma, in the workgroup's `lds`; false: the tile is not finite and
// nothing has been stored (split fp32 only).
// VEC: the rows of q, k, v, o, kc, vc and hgroup are whole aligned 16-byte chunks.  They are then
// loaded through buffer resources over just the rows wanted, so rows past them read as zero with
// no branch around any load (a branch per load makes the compiler wait for each by itself: the
// bf16 call above took 0.67 ms, now 0.42, with a run-time test of the alignment in its load loop).
// all: dense (every key of the segment, no selection, no correction; BT is then ROWS).
// nvt: the first nvt tiles are query blocks (0: the text rows alone, where the blocks run with
// TEAM = 1), the rest up to ntiles text rows.
template <typename E, int DP, int TEAM, int RW, bool VEC>
__device__ __forceinline__ bool any_tile(
    unsigned char* lds, const unsigned char* __restrict__ q, const unsigned char* __restrict__ k,
    const unsigned char* __restrict__ v, const float* __restrict__ kc, const float* __restrict__ vc,
    const float* __restrict__ hgroup, const uint32_t* __restrict__ selmask, unsigned char* __restrict__ o, float scale,
    float c, int T, int text, int text_valid, int D, int BT, int NT, int G, int NG, int NW, int gamma_literal, int all,
    int nvt, int ntiles) {
  using C = AnyCfg<E, DP, TEAM, RW>;
  using frag = typename E::frag;
  constexpr int ES = C::ES, QT = C::QT, NF = C::NF, DT = C::DT, KC = C::KC;
  constexpr int KROW = C::KROW, VROW = C::VROW;
  constexpr bool F32 = C::F32, SPLIT = C::SPLIT;
  constexpr int NPL = C::NPL;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15;
  const int g4 = lane >> 4;
  const int bh = blockIdx.y;
  // Consecutive workgroups go to consecutive XCDs; each takes a contiguous run of a slice's tiles.
  const int tile = (int)(blockIdx.x & 7) * (int)(gridDim.x >> 3) + (int)(blockIdx.x >> 3);
  if (tile >= ntiles) return true;

  const int Ttot = T + text;
  const int seg = T + text_valid;
  // This wave's rows [row0, row_end), its query block I (video tiles of a sparse call) and the
  // run of keys [cur, cend) that follows its selected blocks.
  int I = -1, row0, row_end, cur, cend;
  const int upb = TEAM == 1 ? BT / RW : 1;  // TEAM = 1: waves per query block
  if (TEAM == 1) {
    const int u = tile * 4 + wave;  // RW rows of a block; a wave past the last block repeats it and stores nothing
    I = min(u / upb, NT - 1);
    row0 = I * BT + (u - u / upb * upb) * RW;
    row_end = u < NT * upb ? min(T, row0 + RW) : row0;
    cur = T;
    cend = seg;
  } else if (tile < nvt) {
    const int tpb = (BT + C::ROWS - 1) / C::ROWS;
    I = tile / tpb;
    const int r0 = I * BT + (tile - I * tpb) * C::ROWS;
    row_end = min(T, min(r0 + C::ROWS, (I + 1) * BT));
    if (r0 >= row_end) return true;  // a tile past the last block's rows
    row0 = r0 + wave * RW;
    cur = all ? 0 : T;
    cend = seg;
    if (all) I = -1;
  } else {
    const int t = tile - nvt;
    const int ptiles = (text_valid + C::ROWS - 1) / C::ROWS;
    row0 = (t < ptiles ? T + t * C::ROWS : seg + (t - ptiles) * C::ROWS) + wave * RW;
    row_end = t < ptiles ? seg : Ttot;
    cur = t < ptiles ? 0 : seg;
    cend = row_end;
  }
  const int64_t row_bytes = (int64_t)D * ES;
  const int64_t slice = (int64_t)bh * Ttot * row_bytes;
  const unsigned char* ksl = k + slice;
  const unsigned char* vsl = v + slice;

  // Q as B operands: fragment f of query tile qt holds the slots of feature step f.
  frag qf[QT][NF][NPL];
  const rsrc_t qrs = make_rsrc(q + slice + (int64_t)row0 * row_bytes,
                               (uint32_t)(min(RW, max(0, row_end - row0)) * (int)row_bytes));
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    const int r = 16 * qt + l16;
    const unsigned char* qrow = q + slice + (int64_t)(row0 + r) * row_bytes;
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      u32x4_t w = {0u, 0u, 0u, 0u};
      if constexpr (SPLIT) {
        u32x4_t pw[3];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int d = 32 * f + 16 * h + 4 * g4;
          u32x4_t x4 = {0u, 0u, 0u, 0u};
          if constexpr (VEC) {
            x4 = __builtin_amdgcn_raw_buffer_load_b128(
                qrs, d < D ? (uint32_t)(r * (int)row_bytes + d * 4) : kOutside, 0, 0);
          } else if (row0 + r < row_end) {
            const uint4 y = load_elems<4>(qrow, d / 4, D);
            x4 = (u32x4_t){y.x, y.y, y.z, y.w};
          }
          const float x[4] = {__uint_as_float(x4[0]) * kUpQ, __uint_as_float(x4[1]) * kUpQ,
                              __uint_as_float(x4[2]) * kUpQ, __uint_as_float(x4[3]) * kUpQ};
          uint2 pl[3];
          split4(x, pl);
#pragma unroll
          for (int i = 0; i < 3; ++i) {
            pw[i][2 * h] = pl[i].x;
            pw[i][2 * h + 1] = pl[i].y;
          }
        }
#pragma unroll
        for (int i = 0; i < NPL; ++i) qf[qt][f][i] = __builtin_bit_cast(frag, pw[i]);
        continue;
      }
      if constexpr (F32) {
        const int d = 16 * f + 4 * g4;
        if constexpr (VEC) {
          w = __builtin_amdgcn_raw_buffer_load_b128(qrs, d < D ? (uint32_t)(r * (int)row_bytes + d * 4) : kOutside, 0, 0);
        } else if (row0 + r < row_end) {
          const uint4 x = load_elems<4>(qrow, d / 4, D);
          w = (u32x4_t){x.x, x.y, x.z, x.w};
        }
      } else {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int d = 32 * f + 16 * h + 4 * g4;
          if constexpr (VEC) {
            const auto x = __builtin_amdgcn_raw_buffer_load_b64(
                qrs, d < D ? (uint32_t)(r * (int)row_bytes + d * 2) : kOutside, 0, 0);
            w[2 * h] = x[0];
            w[2 * h + 1] = x[1];
          } else if (row0 + r < row_end) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
              if (d + i < D)
                w[2 * h + (i >> 1)] |= (uint32_t)reinterpret_cast<const uint16_t*>(qrow)[d + i] << (16 * (i & 1));
          }
        }
      }
      qf[qt][f][0] = __builtin_bit_cast(frag, w);
    }
  }

  f32x4_t oacc[DT][QT];
  float l_run[QT], g_run[QT], m_run[QT];  // m: on all four lanes of a row; l, Gamma: this lane's keys
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    m_run[qt] = -INFINITY;
    l_run[qt] = g_run[qt] = 0.f;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) oacc[dt][qt] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
  }

  // A operands of O^T from `rows` (V, V^ or Hbar rows in LDS): feature tile dt, row step s.
  auto vt16 = [&](const unsigned char* rows, int s, int dt) {
    const unsigned char* p = rows + (32 * s + 4 * g4 + (l16 >> 2)) * VROW + dt * 32 + (l16 & 3) * 8;
    const uint2 lo = lds_read_tr16(p, 0);
    const uint2 hi = lds_read_tr16(p, 16 * VROW);
    return __builtin_bit_cast(frag, (u32x4_t){lo.x, lo.y, hi.x, hi.y});
  };
  // The three planes of a fragment: K rows of tile kt at step f (planes kp bytes apart), and the V
  // form (planes vp bytes apart).
  auto kfrag3 = [&](const unsigned char* rows, int kp, int f, int kt, frag (&a)[3]) {
#pragma unroll
    for (int i = 0; i < 3; ++i) a[i] = lds_ld<frag>(rows, i * kp + (kt * 16 + l16) * KROW + f * 64 + g4 * 16);
  };
  auto vfrag3 = [&](const unsigned char* rows, int vp, int s, int dt, frag (&a)[3]) {
#pragma unroll
    for (int i = 0; i < 3; ++i) a[i] = vt16(rows + i * vp, s, dt);
  };
  auto vt32 = [&](const unsigned char* rows, int r, int dt) {
    return lds_ld<float>(rows, (r + 4 * g4) * VROW + dt * 64 + l16 * 4);
  };

  // Four fp32, times `up`, as their three parts, one plane each.
  auto st_split = [&](unsigned char* base, int plane, int off, const uint4& x, float up) {
    const float f[4] = {__uint_as_float(x.x) * up, __uint_as_float(x.y) * up, __uint_as_float(x.z) * up,
                        __uint_as_float(x.w) * up};
    uint2 pl[3];
    split4(f, pl);
#pragma unroll
    for (int i = 0; i < 3; ++i) lds_st(base, i * plane + off, pl[i]);
  };

  const float cs = SPLIT ? c * kDownS : c;
  // One online-softmax step over the 16 KTN rows at Kb / Vb.  mask(s) drops scores (to -inf),
  // on_rescale(qt, alpha) sees a rise of the running max, add(qt, key, p) every weight; rows_v(a, key)
  // sees every operand of V: key 16 kt + i of this lane in fp32, the eight of a 32-key step in 16 bits.
  auto step = [&](const unsigned char* Kb, const unsigned char* Vb, auto ktn, auto mask, auto on_rescale, auto add,
                  auto rows_v) __attribute__((always_inline)) {
    constexpr int KTN = decltype(ktn)::value;
    f32x4_t s[KTN][QT];
    if constexpr (SPLIT) {
      constexpr int KP = 16 * KTN * KROW;
      // Feature steps per sum of first-order products: half of them (one of 96's three).
      constexpr int HC = NF % 2 ? 1 : NF / 2;
      f32x4_t hi[KTN][QT], sb[KTN][QT];
#pragma unroll
      for (int kt = 0; kt < KTN; ++kt)
#pragma unroll
        for (int qt = 0; qt < QT; ++qt) s[kt][qt] = sb[kt][qt] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int f = 0; f < NF; ++f)
        for (int kt = 0; kt < KTN; kt += 2) {
          frag a[2][3];
          kfrag3(Kb, KP, f, kt, a[0]);
          kfrag3(Kb, KP, f, kt + 1, a[1]);
#pragma unroll
          for (int qt = 0; qt < QT; ++qt) {
            if (f % HC == 0) hi[kt][qt] = hi[kt + 1][qt] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
            mfma_split(a, qf[qt][f], {&hi[kt][qt], &hi[kt + 1][qt]}, {&sb[kt][qt], &sb[kt + 1][qt]});
            if (f % HC == HC - 1) {
              s[kt][qt] += hi[kt][qt];
              s[kt + 1][qt] += hi[kt + 1][qt];
            }
          }
        }
#pragma unroll
      for (int kt = 0; kt < KTN; ++kt)
#pragma unroll
        for (int qt = 0; qt < QT; ++qt) s[kt][qt] += sb[kt][qt];
    } else if constexpr (F32) {
      // Chains of 16 features (one f), added as a tree: longer chains round more (see above).  Two at
      // a time, so that an MFMA does not wait for the one before it.
#pragma unroll
      for (int kt = 0; kt < KTN; ++kt) {
        f32x4_t half[QT][3];  // [h]: the finished sum of 2^(h + 1) chains that waits for its pair
#pragma unroll
        for (int f = 0; f < NF; f += 2) {
          const frag a0 = lds_ld<frag>(Kb, (kt * 16 + l16) * KROW + f * 64 + g4 * 16);
          const frag a1 = lds_ld<frag>(Kb, (kt * 16 + l16) * KROW + (f + 1) * 64 + g4 * 16);
#pragma unroll
          for (int qt = 0; qt < QT; ++qt) {
            f32x4_t t0 = {0.f, 0.f, 0.f, 0.f}, t1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              t0 = __builtin_amdgcn_mfma_f32_16x16x4f32(a0[i], qf[qt][f][0][i], t0, 0, 0, 0);
              t1 = __builtin_amdgcn_mfma_f32_16x16x4f32(a1[i], qf[qt][f + 1][0][i], t1, 0, 0, 0);
            }
            t0 += t1;
            int h = 0;
#pragma unroll
            for (int p = f / 2; p & 1; p >>= 1) t0 = half[qt][h++] + t0;
            half[qt][h] = t0;
            if (f == NF - 2) s[kt][qt] = NF == 6 ? half[qt][1] + t0 : t0;
          }
        }
      }
    } else {
#pragma unroll
      for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int kt = 0; kt < KTN; ++kt) {
          const frag a = lds_ld<frag>(Kb, (kt * 16 + l16) * KROW + f * 64 + g4 * 16);
#pragma unroll
          for (int qt = 0; qt < QT; ++qt) {
            if (f == 0) s[kt][qt] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
            s[kt][qt] = E::M::mfma16(a, qf[qt][f][0], s[kt][qt]);
          }
        }
    }
    mask(s);
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
      float mx = -INFINITY;
#pragma unroll
      for (int kt = 0; kt < KTN; ++kt)
#pragma unroll
        for (int i = 0; i < 4; ++i) mx = fmaxf(mx, s[kt][qt][i]);
      const float mxc = quad16_max(mx) * cs;
      if (__any(mxc > m_run[qt])) {
        const float m_new = fmaxf(m_run[qt], mxc);
        const float alpha = fast_exp2(m_run[qt] - m_new);  // 0 on the first step
        m_run[qt] = m_new;
        l_run[qt] *= alpha;
        on_rescale(qt, alpha);
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
          for (int i = 0; i < 4; ++i) oacc[dt][qt][i] *= alpha;
      }
#pragma unroll
      for (int kt = 0; kt < KTN; ++kt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float p = fast_exp2(fmaf(s[kt][qt][i], cs, -m_run[qt]));
          add(qt, 16 * kt + i, p);
          s[kt][qt][i] = p;
        }
    }
    if constexpr (F32) {
      // Each chunk's products are summed by themselves and added to o once (shorter fp32 chains).
#pragma unroll
      for (int d2 = 0; d2 < DT; d2 += 2) {
        f32x4_t t[2][QT];
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int qt = 0; qt < QT; ++qt) t[j][qt] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kt = 0; kt < KTN; ++kt)
#pragma unroll
          for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
              const float a = rows_v(vt32(Vb, 16 * kt + i, d2 + j), 16 * kt + i);
#pragma unroll
              for (int qt = 0; qt < QT; ++qt)
                t[j][qt] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, s[kt][qt][i], t[j][qt], 0, 0, 0);
            }
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int qt = 0; qt < QT; ++qt) oacc[d2 + j][qt] += t[j][qt];
      }
    } else if constexpr (SPLIT) {
      constexpr int VP = 16 * KTN * VROW;
      static_assert(KTN == 2, "one 32-key step");
      frag pf[QT][3];
#pragma unroll
      for (int qt = 0; qt < QT; ++qt) {
        u32x4_t pw[3];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const float x[4] = {s[h][qt][0] * kUpP, s[h][qt][1] * kUpP, s[h][qt][2] * kUpP, s[h][qt][3] * kUpP};
          uint2 pl[3];
          split4(x, pl);
#pragma unroll
          for (int i = 0; i < 3; ++i) {
            pw[i][2 * h] = pl[i].x;
            pw[i][2 * h + 1] = pl[i].y;
          }
        }
#pragma unroll
        for (int i = 0; i < 3; ++i) pf[qt][i] = __builtin_bit_cast(frag, pw[i]);
      }
#pragma unroll
      for (int dt = 0; dt < DT; dt += 2) {
        frag a[2][3];
        vfrag3(Vb, VP, 0, dt, a[0]);
        vfrag3(Vb, VP, 0, dt + 1, a[1]);
#pragma unroll
        for (int qt = 0; qt < QT; ++qt) {
          f32x4_t lo[2];  // the first-order products add to o itself: one addition per 32 keys
          lo[0] = lo[1] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
          mfma_split(a, pf[qt], {&oacc[dt][qt], &oacc[dt + 1][qt]}, {&lo[0], &lo[1]});
          oacc[dt][qt] += lo[0];
          oacc[dt + 1][qt] += lo[1];
        }
      }
    } else {
#pragma unroll
      for (int s2 = 0; s2 < KTN / 2; ++s2) {
        frag pf[QT];
#pragma unroll
        for (int qt = 0; qt < QT; ++qt) {
          const f32x4_t &a = s[2 * s2][qt], &b = s[2 * s2 + 1][qt];
          pf[qt] = __builtin_bit_cast(frag, (u32x4_t){E::M::pack2(a[0], a[1]), E::M::pack2(a[2], a[3]),
                                                      E::M::pack2(b[0], b[1]), E::M::pack2(b[2], b[3])});
        }
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
          const frag a = rows_v(vt16(Vb, s2, dt), 32 * s2);
#pragma unroll
          for (int qt = 0; qt < QT; ++qt) oacc[dt][qt] = E::M::mfma16(a, pf[qt], oacc[dt][qt]);
        }
      }
    }
  };

  // ---------------- Phase 1: the selected blocks, then the run [cur, cend) --------
  typedef const __attribute__((address_space(4))) uint32_t* const const_u32_ptr;
  const const_u32_ptr mrow = (const_u32_ptr)(selmask + ((int64_t)bh * NT + (I < 0 ? 0 : I)) * NW);
  {
    unsigned char* Kb = lds + (TEAM == 1 ? wave : 0) * C::SLAB;
    unsigned char* Vb = Kb + NPL * KC * KROW;
    const int tt = tid & (C::TT - 1);
    const int sc = tt % C::CHP;   // this thread's 16-byte chunk of a staged row
    const int sr = tt / C::CHP;   // its row in each pass
    const bool in_row = sc * (16 / ES) < D;
    auto sync = [&]() {
      if (TEAM == 1) {  // LDS operations of a wave complete in order: only its own writes need waiting for
        __builtin_amdgcn_s_waitcnt(0xC07F);
        asm volatile("" ::: "memory");
      } else {
        __syncthreads();
      }
    };
    int w = 0, j0 = 0, j1 = 0;  // the selected block being walked: rows [j0, j1)
    uint32_t bits = I >= 0 && NW > 0 ? mrow[0] : 0u;
    auto next_block = [&]() -> bool {
      if (I < 0) return false;
      while (bits == 0u) {
        if (++w >= NW) return false;
        bits = mrow[w];
      }
      const int j = 32 * w + __builtin_ctz(bits);
      bits &= bits - 1u;
      j0 = j * BT;
      j1 = min(T, j0 + BT);
      return true;
    };
    // The next chunk: rows ra .. (16 rows from ra, then from rb, where a chunk holds two 16-row
    // blocks); returns its number of rows, 0 at the end.
    bool tail = false;
    auto next_chunk = [&](int& ra, int& rb) -> int {
      if (j0 >= j1 && !tail && !next_block()) {
        tail = true;
        j0 = cur;
        j1 = cend;
      }
      if (j0 >= j1) return 0;
      ra = j0;
      int n = min(KC, j1 - j0);
      j0 += n;
      rb = ra + 16;
      if (TEAM == 1 && KC == 32 && RW == 16 && BT == 16 && !tail && n == 16 && next_block()) {
        rb = j0;
        n += j1 - j0;
        j0 = j1;
      }
      return n;
    };
    uint4 kreg[C::PASSES], vreg[C::PASSES];
    // Rows r of a chunk: ra + r, and rb + r - 16 from row 16 on where each wave stages its own.
    const uint32_t lane_off = in_row ? (uint32_t)(sr * (int)row_bytes + sc * 16) : kOutside;
    auto fetch = [&](int ra, int rb, int n) {
      constexpr int RUN = TEAM == 1 && KC == 32 && RW == 16 ? 16 : KC;  // 32-row blocks (RW 32) fill a chunk
      const int na = min(n, RUN), nb = n - na;
      const unsigned char* base_k[2] = {ksl + (int64_t)ra * row_bytes, ksl + (int64_t)rb * row_bytes};
      const unsigned char* base_v[2] = {vsl + (int64_t)ra * row_bytes, vsl + (int64_t)rb * row_bytes};
      const rsrc_t rk[2] = {make_rsrc(base_k[0], (uint32_t)(na * (int)row_bytes)),
                            make_rsrc(base_k[1], (uint32_t)(nb * (int)row_bytes))};
      const rsrc_t rv[2] = {make_rsrc(base_v[0], (uint32_t)(na * (int)row_bytes)),
                            make_rsrc(base_v[1], (uint32_t)(nb * (int)row_bytes))};
#pragma unroll
      for (int p = 0; p < C::PASSES; ++p) {
        const int h = p * C::RPP >= RUN ? 1 : 0;
        const int r0 = p * C::RPP - h * RUN;  // of the pass, within its run
        if constexpr (VEC) {
          const uint32_t off = lane_off + (uint32_t)(r0 * (int)row_bytes);
          kreg[p] = buf_load16(rk[h], off);
          vreg[p] = buf_load16(rv[h], off);
        } else {
          kreg[p] = vreg[p] = make_uint4(0u, 0u, 0u, 0u);
          if (r0 + sr < (h ? nb : na) && in_row) {
            kreg[p] = load_elems<ES>(base_k[h] + (int64_t)(r0 + sr) * row_bytes, sc, D);
            vreg[p] = load_elems<ES>(base_v[h] + (int64_t)(r0 + sr) * row_bytes, sc, D);
          }
        }
      }
    };
    auto stash = [&]() {
      if (sc >= C::CH) return;
#pragma unroll
      for (int p = 0; p < C::PASSES; ++p) {
        const int r = p * C::RPP + sr;
        if constexpr (SPLIT) {
          st_split(Kb, KC * KROW, r * KROW + (sc >> 3) * 64 + (sc & 3) * 16 + ((sc >> 2) & 1) * 8, kreg[p], 1.f);
          st_split(Vb, KC * VROW, r * VROW + sc * 8, vreg[p], kUpV);
          continue;
        }
        if constexpr (F32) {
          lds_st(Kb, r * KROW + sc * 16, kreg[p]);
        } else {  // features in slot order: 8 sc .. + 3 and + 4 .. + 7 are halves of two slots
          const int b = r * KROW + (sc >> 2) * 64 + (sc & 1) * 32 + ((sc >> 1) & 1) * 8;
          lds_st(Kb, b, make_uint2(kreg[p].x, kreg[p].y));
          lds_st(Kb, b + 16, make_uint2(kreg[p].z, kreg[p].w));
        }
        lds_st(Vb, r * VROW + sc * 16, vreg[p]);
      }
    };
    int ra = 0, rb = 0;
    int n = next_chunk(ra, rb);
    if (n > 0) fetch(ra, rb, n);
    while (n > 0) {
      const int n2 = next_chunk(ra, rb);
      sync();  // the previous chunk has been read
      stash();
      sync();
      if (n2 > 0) fetch(ra, rb, n2);
      step(Kb, Vb, std::integral_constant<int, KC / 16>{},
           [&](auto& s) {
             if (n < KC) {
               const int lim = n - 4 * g4;  // key 16 kt + 4 g4 + i is past the chunk iff 16 kt + i >= lim
#pragma unroll
               for (int kt = 0; kt < KC / 16; ++kt)
#pragma unroll
                 for (int qt = 0; qt < QT; ++qt)
#pragma unroll
                   for (int i = 0; i < 4; ++i)
                     if (16 * kt + i >= lim) s[kt][qt][i] = -INFINITY;
             }
           },
           [](int, float) {}, [&](int qt, int, float p) { l_run[qt] += p; }, [](auto a, int) { return a; });
      n = n2;
    }
  }

  // ---------------- Phase 2: zero- and first-order correction per group -----------
  if (I >= 0) {
    const int last_len = T - (NT - 1) * BT;
    const float* kcb = kc + (int64_t)bh * NT * D;
    const float* vcb = vc + (int64_t)bh * NT * D;
    unsigned char* Kz = lds;
    unsigned char* Vz = lds + NPL * C::KZ * KROW;
    unsigned char* Hs = SPLIT ? lds : lds + C::Z_BYTES;
    constexpr int H0 = SPLIT ? 1 : 0;  // the item that Hbar's first rows come with
    const int c4 = tid % C::C4P, r4 = tid / C::C4P;
    // TEAM = 1: blocks of one mask word that some wave of the workgroup does not select.
    auto word_unselected = [&](int wd) -> uint32_t {
      uint32_t m = 0xffffffffu;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        m &= ((const_u32_ptr)(selmask + ((int64_t)bh * NT + min((tile * 4 + i) / upb, NT - 1)) * NW))[wd];
      return ~m;
    };
    auto any_unselected = [&](int a, int b) -> bool {
      for (int wd = a >> 5; wd <= (b - 1) >> 5; ++wd) {
        uint32_t m = word_unselected(wd);
        if (wd == a >> 5) m &= 0xffffffffu << (a & 31);
        if (wd == (b - 1) >> 5) m &= 0xffffffffu >> (31 - ((b - 1) & 31));
        if (m) return true;
      }
      return false;
    };
    // Bit t: block jc + t (t < cn <= 32) is approximated for this wave's query block.
    auto approx_bits = [&](int jc, int cn) -> uint32_t {
      const int wd = jc >> 5, sh = jc & 31;
      uint32_t sel = mrow[wd] >> sh;
      if (sh != 0 && wd + 1 < NW) sel |= mrow[wd + 1] << (32 - sh);
      return ~sel & (cn >= 32 ? 0xffffffffu : (1u << cn) - 1u);
    };
    // Four floats to LDS as four elements of the input type (or their parts, `plane` bytes apart).
    auto st4 = [&](unsigned char* base, int plane, int off16, int off32, const float4& x, float up) {
      if constexpr (SPLIT)
        st_split(base, plane, off16, __builtin_bit_cast(uint4, x), up);
      else if constexpr (F32)
        lds_st(base, off32, x);
      else
        lds_st(base, off16, make_uint2(E::M::pack2(x.x, x.y), E::M::pack2(x.z, x.w)));
    };
    const bool in4 = 4 * c4 < D;
    const uint32_t off4 = in4 ? (uint32_t)(r4 * D + 4 * c4) * 4u : kOutside;
    // Piece c4 of row r0 + r4 of the statistics rows at base, of which n are wanted; zero without `want`.
    auto load4 = [&](const float* base, const rsrc_t& rs, int r0, int n, bool want = true) -> float4 {
      if constexpr (VEC) {
        const uint4 x = buf_load16(rs, want ? off4 + (uint32_t)(r0 * D) * 4u : kOutside);
        return make_float4(__uint_as_float(x.x), __uint_as_float(x.y), __uint_as_float(x.z), __uint_as_float(x.w));
      } else {
        uint4 x = make_uint4(0u, 0u, 0u, 0u);
        if (want && r0 + r4 < n) x = load_elems<4>((const unsigned char*)(base + (int64_t)(r0 + r4) * D), c4, D);
        return make_float4(__uint_as_float(x.x), __uint_as_float(x.y), __uint_as_float(x.z), __uint_as_float(x.w));
      }
    };
    // Work items in order: a group's zero-order chunks of 32 blocks (the first one brings Hbar's
    // first HR rows along, but for the split ones), then the rest of its Hbar HR rows at a time.  The
    // next item's rows load into registers while one is computed (430 -> 391 us at the bf16 shape
    // above, split fp32 0.5%); with the fp32 MFMA that is 2% slower.
    int ig = -1, ijc = 0, ihs = 0;
    auto group_end = [&](int g) -> int { return (int)min((int64_t)NT, (int64_t)(g + 1) * G); };
    uint32_t iap = 0u;  // TEAM = 4: the item's approximated blocks
    auto chunk_from = [&](int g, int jc) -> bool {  // the group's first chunk at or after jc with work
      for (const int jb = group_end(g); jc < jb; jc += C::KZ) {
        const int cn = min(C::KZ, jb - jc);
        if (TEAM != 1) iap = approx_bits(jc, cn);
        if (TEAM == 1 ? any_unselected(jc, jc + cn) : iap != 0u) {
          ijc = jc;
          return true;
        }
      }
      return false;
    };
    auto next_item = [&]() -> bool {
      if (ig >= 0) {
        if (ihs == 0 && chunk_from(ig, ijc + C::KZ)) return true;
        if ((ihs + 1 - H0) * C::HR < D) {
          ++ihs;
          return true;
        }
      }
      ihs = 0;
      while (++ig < NG)
        if (chunk_from(ig, ig * G)) return true;
      return false;
    };
    constexpr int ZP = C::KZ / C::RPP4, HP = C::HR / C::RPP4;
    float4 zk[ZP], zv[ZP], hx[HP];
    auto fetch_h = [&](int g, int hs) {
      const int n = min(C::HR, D - hs * C::HR);
      const float* hb = hgroup + ((int64_t)bh * NG + g) * D * D + (int64_t)hs * C::HR * D;
      const rsrc_t rh = make_rsrc(hb, (uint32_t)(n * D * 4));
#pragma unroll
      for (int p = 0; p < HP; ++p) hx[p] = load4(hb, rh, p * C::RPP4, n);
    };
    // V^ of a selected block is taken as zero: its weight is, but 0 times a sum that left the type's
    // range is NaN.  TEAM = 1: each wave selects its own, and clears them from its operands (below).
    auto fetch_z = [&](int jc, int cn) {
      const uint32_t approx = TEAM == 1 ? 0xffffffffu : iap;
      const float* kb = kcb + (int64_t)jc * D;
      const float* vb = vcb + (int64_t)jc * D;
      const rsrc_t rk = make_rsrc(kb, (uint32_t)(cn * D * 4)), rv = make_rsrc(vb, (uint32_t)(cn * D * 4));
#pragma unroll
      for (int p = 0; p < ZP; ++p) {
        zk[p] = load4(kb, rk, p * C::RPP4, cn);
        zv[p] = load4(vb, rv, p * C::RPP4, cn, (approx >> (p * C::RPP4 + r4)) & 1u);
      }
    };
    auto stash_h = [&]() {
      if (c4 >= C::C4) return;
#pragma unroll
      for (int p = 0; p < HP; ++p) {
        const int r = p * C::RPP4 + r4;
        st4(Hs, C::HR * VROW, r * VROW + c4 * 8, r * VROW + c4 * 16, hx[p], kUpH);
      }
    };
    auto stash_z = [&]() {
      if (c4 >= C::C4) return;
#pragma unroll
      for (int p = 0; p < ZP; ++p) {
        const int r = p * C::RPP4 + r4;
        st4(Kz, C::KZ * KROW, r * KROW + (c4 >> 3) * 64 + (c4 & 3) * 16 + ((c4 >> 2) & 1) * 8, r * KROW + c4 * 16,
            zk[p], 1.f);
        st4(Vz, C::KZ * VROW, r * VROW + c4 * 8, r * VROW + c4 * 16, zv[p], kUpV);
      }
    };
    // Per row, of the current group: the sums of p and of p times the block's length, relative to
    // the running max until the group ends (Gamma itself is rescaled only in the consistent form,
    // :231-235), then f = scale * (sum of p).
    float psum[QT], gsum[QT], f[QT];
    int pg = -1;  // the group of the previous item
    bool mine = true;  // this wave approximates some block of the group (TEAM = 1: another wave may instead)
    bool more = next_item();
    if (more && !F32) {
      fetch_z(ijc, min(C::KZ, group_end(ig) - ijc));
      if (!SPLIT) fetch_h(ig, 0);
    }
    while (more) {
      const int g = ig, jc = ijc, hs = ihs;
      const uint32_t ap = iap;
      const bool first = g != pg;
      pg = g;
      __syncthreads();  // the previous item's rows have been read
      const bool h_rows = hs > 0 || (first && !SPLIT);
      if (F32) {
        if (hs == 0) fetch_z(jc, min(C::KZ, group_end(g) - jc));
        if (h_rows) fetch_h(g, hs);
      }
      if (hs == 0) stash_z();
      if (h_rows) stash_h();
      __syncthreads();
      more = next_item();
      if (more && !F32) {
        if (ihs == 0) fetch_z(ijc, min(C::KZ, group_end(ig) - ijc));
        if (ihs > 0 || (ig != g && !SPLIT)) fetch_h(ig, ihs - H0);
      }
      if (hs == 0) {
        if (first) {
#pragma unroll
          for (int qt = 0; qt < QT; ++qt) psum[qt] = gsum[qt] = 0.f;
          mine = false;
        }
        // Zero order: o += p V^.
        const uint32_t approx = TEAM == 1 ? approx_bits(jc, min(C::KZ, group_end(g) - jc)) : ap;
        const bool visit = TEAM != 1 || approx != 0u;
        if (visit) mine = true;
        const uint32_t ub = approx >> (4 * g4);
        u32x4_t keep;  // 16 bits: keys 4 g4 .. + 3 and 16 + 4 g4 .. + 3 of the step, two to a word
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const uint32_t two = ub >> (2 * (i & 1) + 16 * (i >> 1));
          keep[i] = ((two & 1u) ? 0xffffu : 0u) | ((two & 2u) ? 0xffff0000u : 0u);
        }
        const int last = NT - 1 - jc - 4 * g4;  // this lane's key index of the last block
        if (visit)
          step(Kz, Vz, std::integral_constant<int, C::KZ / 16>{},
               [&](auto& s) {
#pragma unroll
                 for (int kt = 0; kt < C::KZ / 16; ++kt)
#pragma unroll
                   for (int qt = 0; qt < QT; ++qt)
#pragma unroll
                     for (int i = 0; i < 4; ++i)
                       if (!((ub >> (16 * kt + i)) & 1u)) s[kt][qt][i] = -INFINITY;
               },
               [&](int qt, float alpha) {
                 psum[qt] *= alpha;
                 gsum[qt] *= alpha;
                 if (!gamma_literal) g_run[qt] *= alpha;
               },
               [&](int qt, int key, float p) {
                 psum[qt] += p;
                 gsum[qt] += p * (float)(key == last ? last_len : BT);
               },
               [&](auto a, int key) {
                 if constexpr (TEAM != 1)
                   return a;
                 else if constexpr (F32)
                   return (ub >> key) & 1u ? a : 0.f;
                 else
                   return __builtin_bit_cast(frag, __builtin_bit_cast(u32x4_t, a) & keep);
               });
        if (more && ig == g && ihs == 0) continue;  // another chunk of this group
#pragma unroll
        for (int qt = 0; qt < QT; ++qt) {
          g_run[qt] += gsum[qt];
          f[qt] = quad16_sum(psum[qt]) * scale;
        }
        if (SPLIT) continue;  // Hbar comes with the next items
      }
      // First order: o += f (q . Hbar), over this item's rows of Hbar.  A wave that selects the whole
      // group has f = 0 and leaves Hbar, which may not be finite, alone.
      if (TEAM == 1 && !mine) continue;
      if constexpr (F32) {
#pragma unroll
        for (int h = 0; h < DP / C::HR; ++h) {
          if (h != hs) continue;
#pragma unroll
          for (int d2 = 0; d2 < DT; d2 += 2) {
            f32x4_t r[2][QT];
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
              for (int qt = 0; qt < QT; ++qt) r[j][qt] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int cc = 0; cc < C::HR / 16; ++cc)
#pragma unroll
              for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                  const float a = vt32(Hs, 16 * cc + i, d2 + j);
#pragma unroll
                  for (int qt = 0; qt < QT; ++qt)
                    r[j][qt] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, qf[qt][h * (C::HR / 16) + cc][0][i], r[j][qt], 0,
                                                                    0, 0);
                }
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
              for (int qt = 0; qt < QT; ++qt)
#pragma unroll
                for (int i = 0; i < 4; ++i) oacc[d2 + j][qt][i] = fmaf(r[j][qt][i], f[qt], oacc[d2 + j][qt][i]);
          }
        }
      } else if constexpr (SPLIT) {
#pragma unroll
        for (int h = 0; h < DP / C::HR; ++h) {
          if (h != hs - H0) continue;
#pragma unroll
          for (int dt = 0; dt < DT; dt += 2) {
            f32x4_t hi[QT][2], lo[QT][2];
#pragma unroll
            for (int qt = 0; qt < QT; ++qt)
#pragma unroll
              for (int j = 0; j < 2; ++j) hi[qt][j] = lo[qt][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s2 = 0; s2 < C::HR / 32; ++s2) {
              frag a[2][3];
              vfrag3(Hs, C::HR * VROW, s2, dt, a[0]);
              vfrag3(Hs, C::HR * VROW, s2, dt + 1, a[1]);
#pragma unroll
              for (int qt = 0; qt < QT; ++qt)
                mfma_split(a, qf[qt][h * (C::HR / 32) + s2], {&hi[qt][0], &hi[qt][1]}, {&lo[qt][0], &lo[qt][1]});
            }
#pragma unroll
            for (int qt = 0; qt < QT; ++qt)
#pragma unroll
              for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                  oacc[dt + j][qt][i] = fmaf(hi[qt][j][i] + lo[qt][j][i], f[qt], oacc[dt + j][qt][i]);
          }
        }
      } else {
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
          f32x4_t r[QT];
#pragma unroll
          for (int qt = 0; qt < QT; ++qt) r[qt] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int s2 = 0; s2 < NF; ++s2) {
            const frag a = vt16(Hs, s2, dt);
#pragma unroll
            for (int qt = 0; qt < QT; ++qt) r[qt] = E::M::mfma16(a, qf[qt][s2][0], r[qt]);
          }
#pragma unroll
          for (int qt = 0; qt < QT; ++qt)
#pragma unroll
            for (int i = 0; i < 4; ++i) oacc[dt][qt][i] = fmaf(r[qt][i], f[qt], oacc[dt][qt][i]);
        }
      }
    }
  }

  if constexpr (SPLIT) {
    float t = 0.f;
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
      t += l_run[qt] + g_run[qt];
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) t += (oacc[dt][qt][0] + oacc[dt][qt][1]) + (oacc[dt][qt][2] + oacc[dt][qt][3]);
    }
    if (__syncthreads_or(!(fabsf(t) < INFINITY))) return false;
  }

  // o = A / (L + Gamma) (:258-259), stored in the input type (:262).
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    const int r = row0 + 16 * qt + l16;
    const float den = quad16_sum(l_run[qt]) + quad16_sum(g_run[qt]);
    if (r < row_end) {
      unsigned char* orow = o + slice + (int64_t)r * row_bytes;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        const int e = 16 * dt + 4 * g4;
        float x[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) x[i] = SPLIT ? oacc[dt][qt][i] / den * kDownO : oacc[dt][qt][i] / den;
        if (VEC && e < D) {
          if constexpr (ES == 4)
            *reinterpret_cast<float4*>(orow + e * 4) = make_float4(x[0], x[1], x[2], x[3]);
          else
            *reinterpret_cast<uint2*>(orow + e * 2) = make_uint2(E::M::pack2(x[0], x[1]), E::M::pack2(x[2], x[3]));
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (e + i < D) {
              if constexpr (ES == 4)
                reinterpret_cast<float*>(orow)[e + i] = x[i];
              else
                reinterpret_cast<uint16_t*>(orow)[e + i] = (uint16_t)E::M::bits(x[i]);
            }
        }
      }
    }
  }
  return true;
}

}  // namespace

// Three waves per SIMD for Any32 at DP 96: its scores' partial sums take it past 168 registers, and two
// waves are slower than the 20 that then spill (12 heads x 7,800 rows, D 96, block 32: 850 and 779 us).
template <typename E, int DP, int TEAM, int RW, bool VEC>
__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(AnyCfg<E, DP, TEAM, RW>::F32 && DP == 96 ? 3 : 2))) void k4_any_mfma(
    const unsigned char* __restrict__ q, const unsigned char* __restrict__ k, const unsigned char* __restrict__ v,
    const float* __restrict__ kc, const float* __restrict__ vc, const float* __restrict__ hgroup,
    const uint32_t* __restrict__ selmask, unsigned char* __restrict__ o, float scale, float c, int T, int text,
    int text_valid, int D, int BT, int NT, int G, int NG, int NW, int gamma_literal, int all, int nvt,
    int ntiles) {
  using C = AnyCfg<E, DP, TEAM, RW>;
  if constexpr (E::SPLIT) {
    // An infinite operand meets the zero parts of another and gives NaN where an fp32 product would
    // not, and the scaled sums leave the range before the sums themselves: a tile that is not finite is
    // done again in fp32.
    using C32 = AnyCfg<Any32, DP, TEAM, RW>;
    __shared__ __attribute__((aligned(16))) unsigned char lds[C::LDS > C32::LDS ? C::LDS : C32::LDS];
    if (c >= kMinSplitC && c <= kMaxSplitC &&
        any_tile<E, DP, TEAM, RW, VEC>(lds, q, k, v, kc, vc, hgroup, selmask, o, scale, c, T, text, text_valid, D, BT,
                                       NT, G, NG, NW, gamma_literal, all, nvt, ntiles))
      return;
    any_tile<Any32, DP, TEAM, RW, VEC>(lds, q, k, v, kc, vc, hgroup, selmask, o, scale, c, T, text, text_valid, D, BT,
                                       NT, G, NG, NW, gamma_literal, all, nvt, ntiles);
  } else {
    __shared__ __attribute__((aligned(16))) unsigned char lds[C::LDS];
    any_tile<E, DP, TEAM, RW, VEC>(lds, q, k, v, kc, vc, hgroup, selmask, o, scale, c, T, text, text_valid, D, BT, NT,
                                   G, NG, NW, gamma_literal, all, nvt, ntiles);
  }
}

namespace {

struct AnyCall {
  const void *q, *k, *v;
  const float *kc, *vc, *hgroup;
  const uint32_t* selmask;
  void* o;
  float scale;
  int bh, T, text, text_valid, D, BT, G, gamma_literal, all;
  hipStream_t stream;
};

bool aligned16(std::initializer_list<const void*> ps) {
  uintptr_t x = 0;
  for (const void* p : ps) x |= (uintptr_t)p;
  return (x & 15u) == 0;
}

int text_tiles(const AnyCall& a, int rows) {
  return (a.text_valid + rows - 1) / rows + (a.text - a.text_valid + rows - 1) / rows;
}

template <typename E, int DP, int TEAM, int RW, bool VEC>
hipError_t launch_any(const AnyCall& a, int BT, int nvt, int ntiles) {
  const int NT = (a.T + BT - 1) / BT;
  const dim3 grid((unsigned)((ntiles + 7) / 8 * 8), (unsigned)a.bh);
  hipLaunchKernelGGL((k4_any_mfma<E, DP, TEAM, RW, VEC>), grid, dim3(256), 0, a.stream, (const unsigned char*)a.q,
                     (const unsigned char*)a.k, (const unsigned char*)a.v, a.kc, a.vc, a.hgroup, a.selmask,
                     (unsigned char*)a.o, a.scale, a.scale * kLog2e, a.T, a.text, a.text_valid, a.D, BT, NT, a.G,
                     (NT + a.G - 1) / a.G, (NT + 31) / 32, a.gamma_literal, a.all, nvt, ntiles);
  return hipGetLastError();
}

// The workgroup tile of TEAM = 4: 128 rows when the blocks are that long and such tiles fill the
// 256 CUs, else 64.
bool wide_tiles(const AnyCall& a, int BT) {
  return BT >= 128 && (int64_t)a.bh * ((a.T + 127) / 128) >= 256;
}

// WIDE: 32 rows per wave where the blocks are long enough, measured at D 96.  Not in fp32, whose planes
// or wider fragments then spill (283 registers).  At DP 128 the 16-bit ones spill too, 60 VGPRs below
// block 64 and 33 from block 128 on, which every group of phase 2 reloads (16 rows would not; not
// measured there: 12 heads x 16,380 rows, D 128, bf16, block 32 637 us, block 128, groups of 16 400).
template <typename E, int DP, bool VEC, bool WIDE>
hipError_t launch_dp(const AnyCall& a) {
  if (!a.all && a.BT < 64) {
    const int NT = (a.T + a.BT - 1) / a.BT;
    hipError_t e;
    if (!WIDE || a.BT == 16) {
      const int ntiles = (int)(((int64_t)NT * (a.BT / 16) + 3) / 4);
      e = launch_any<E, DP, 1, 16, VEC>(a, a.BT, ntiles, ntiles);
    } else {
      const int ntiles = (NT + 3) / 4;
      e = launch_any<E, DP, 1, WIDE ? 32 : 16, VEC>(a, a.BT, ntiles, ntiles);
    }
    if (e != hipSuccess || a.text == 0) return e;
    return launch_any<typename E::Team4, DP, 4, 16, VEC>(a, a.BT, 0, text_tiles(a, 64));  // the text rows
  }
  const bool wide = WIDE && wide_tiles(a, a.all ? 128 : a.BT);
  const int rows = wide ? 128 : 64;
  const int BT = a.all ? rows : a.BT;
  const int nvt = (a.T + BT - 1) / BT * ((BT + rows - 1) / rows);
  const int ntiles = nvt + text_tiles(a, rows);
  return wide ? launch_any<typename E::Team4, DP, 4, WIDE ? 32 : 16, VEC>(a, BT, nvt, ntiles)
              : launch_any<typename E::Team4, DP, 4, 16, VEC>(a, BT, nvt, ntiles);
}

template <typename E>
hipError_t launch_type(const AnyCall& a) {
  constexpr bool WIDE = E::ES == 2;
  const bool vec = (a.D * E::ES) % 16 == 0 && a.D % 4 == 0 && aligned16({a.q, a.k, a.v, a.o, a.kc, a.vc, a.hgroup});
  if (!vec) return launch_dp<E, 128, false, false>(a);
  return a.D <= 64 ? launch_dp<E, 64, true, WIDE>(a)
                   : (a.D <= 96 ? launch_dp<E, 96, true, WIDE>(a) : launch_dp<E, 128, true, WIDE>(a));
}

}  // namespace

int64_t sparse_attn_any_tiles(int T, int text, int text_valid, int BT) {
  const int64_t NT = (T + BT - 1) / BT;
  const int64_t tpb = (BT + 63) / 64;
  return NT * tpb + (text_valid + 63) / 64 + (text - text_valid + 63) / 64;
}

hipError_t launch_sparse_attn_any(const void* q, const void* k, const void* v, const float* kc, const float* vc,
                                  const float* hgroup, const uint32_t* selmask, void* o, float scale, int bh, int T,
                                  int text, int text_valid, int D, int BT, int G, int gamma_literal, int all,
                                  int dtype, hipStream_t stream) {
  if (D < 1 || D > 128 || BT < 16 || BT > 256 || (BT & (BT - 1)) || G < 1 || text_valid < 0 || text_valid > text)
    return hipErrorInvalidValue;
  if (!all && (kc == nullptr || vc == nullptr || hgroup == nullptr || selmask == nullptr)) return hipErrorInvalidValue;
  const AnyCall a{q, k, v, kc, vc, hgroup, selmask, o, scale, bh, T, text, text_valid, D, BT, G, gamma_literal, all,
                  stream};
  switch (dtype) {
    case kAnyF32: return launch_type<Any32>(a);
    case kAnyBf16: return launch_type<Any16<Bf16>>(a);
    case kAnyF16: return launch_type<Any16<F16>>(a);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace pasa
