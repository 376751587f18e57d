// Statistics and selection scores for shapes the tuned kernels do not take: fp32 q, k, v; any
// head dim up to 128; any group size; block sizes 16 .. 256 (the attention stage of the same
// shapes is any_attn.hip).
//
// Reference: svg/kernels/triton/group_pisa_attention.py
//   k2_block_stats_any   fused_chunk_reduce_kernel :66-129 (+ sqrt :287) and
//                        compute_h_group :291-301
//   k3_scores_any        the selection scores :365-371
// The reference accepts any float dtype (o = torch.empty_like(v), :380; statistics
// stored like q, :275-278), any group size (:312) and any power-of-two block size
// (:311; Triton's tl.arange needs a power of two).  The statistics are fp32 here.
#include "common.h"
#include "kernels.h"

namespace pasa {

namespace {

// The three input types: a 16-byte chunk as fp32, and element i of a chunk's four words taken from
// a row that is not whole aligned chunks.
struct F32E {
  static constexpr int ES = 4;
  __device__ static void put(uint32_t (&w)[4], int i, const unsigned char* row, int d) {
    w[i] = reinterpret_cast<const uint32_t*>(row)[d];
  }
  __device__ static void widen(const uint4& c, float (&f)[4]) {
    f[0] = __uint_as_float(c.x);
    f[1] = __uint_as_float(c.y);
    f[2] = __uint_as_float(c.z);
    f[3] = __uint_as_float(c.w);
  }
};
template <typename M>
struct E16 {
  static constexpr int ES = 2;
  __device__ static void put(uint32_t (&w)[4], int i, const unsigned char* row, int d) {
    w[i >> 1] |= (uint32_t)reinterpret_cast<const uint16_t*>(row)[d] << (16 * (i & 1));
  }
  __device__ static void widen(const uint4& c, float (&f)[8]) { M::widen8(c, f); }
};
using Bf16E = E16<Bf16>;
using F16E = E16<F16>;

constexpr int kAnyChunk = 32;  // rows of a staged K/V chunk

}  // namespace

// ---- block statistics ---------------------------------------------------------
// One workgroup (four waves) per part of a group of G key blocks; the part's blocks in ascending
// order, each in chunks of up to 32 rows of q, k and v staged in LDS as fp32 (feature columns D ..
// DP - 1 zero), the next chunk's rows in registers meanwhile.
//
// H_j = K^T V - kbar_j V^_j^T (:106-107) runs on the 16x16x4 fp32 MFMA for every input type, each
// wave on a quarter of the D x D moment, rows in ascending order: that MFMA is a chain of fused
// multiply-adds in k order, bit for bit, so kc, qc, ||H_j|| and the selection made from them do not
// depend on how the work is split.  ||H_j||^2 is summed in 8 x 8 tiles (H_j through LDS), then over
// the wave, then over the waves; column sums run down a block's rows in order, one column per
// thread.  The group sum stays in registers; with split > 1 each part writes its own to `partials`
// and k2_any_reduce adds the parts in order.
//
// Bound: the fp32 MFMA (2 D^2 FLOP per row) against three rows read; a block of 64 rows at D 128 is
// 3.4 us of MFMA issue.  One workgroup per group left most of the 256 CUs idle and its FMAs waited
// on four LDS reads per row: 12 heads x 7,800 fp32 rows of D 128 took 847 us (now 66 + 12 for the
// reduction), 2 heads x 1,024 of D 64 291 us (now 8 + 6), 16 x 8,610 bf16 of D 96 248 us (66 + 7).
template <typename EL, int DP>
struct StatsCfg {
  static constexpr int CH = kAnyChunk;
  static constexpr int LD = DP + 16;   // four consecutive rows start 16 banks apart
  static constexpr int HLD = DP + 4;   // rows four apart do, and 16-byte rows
  static constexpr int KV_FLOATS = 3 * CH * LD;
  static constexpr int H_FLOATS = DP * HLD;
  static constexpr int LDS_FLOATS = KV_FLOATS > H_FLOATS ? KV_FLOATS : H_FLOATS;  // one after the other
  static constexpr int EPC = 16 / EL::ES;             // elements per 16-byte chunk
  static constexpr int NCH = DP / EPC;                // chunks per row
  static constexpr int NCHP = NCH <= 8 ? 8 : (NCH <= 16 ? 16 : 32);
  static constexpr int RPP = 256 / NCHP;              // rows per staging pass
  static constexpr int PASSES = CH / RPP;
  static constexpr int TL = DP / 32;                  // 16 x 16 tiles per side of a wave's quarter
};

// VEC: rows are whole aligned 16-byte chunks, loaded through a buffer resource over the rows wanted
// (rows past them read as zero, with no branch around a load); else element by element.
template <typename EL, int DP, bool VEC>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k2_block_stats_any(
    const unsigned char* __restrict__ q, const unsigned char* __restrict__ k, const unsigned char* __restrict__ v,
    float* __restrict__ qc, float* __restrict__ kc, float* __restrict__ vc, float* __restrict__ hnorm,
    float* __restrict__ hgroup, float* __restrict__ partials, int T, int Tslice, int D, int BT, int NT, int G,
    int split) {
  using C = StatsCfg<EL, DP>;
  constexpr int CH = C::CH, LD = C::LD, HLD = C::HLD, TL = C::TL, EPC = C::EPC;
  __shared__ __attribute__((aligned(16))) float buf[C::LDS_FLOATS];  // K, V and Q chunk; then H_j
  __shared__ __attribute__((aligned(16))) float kbar[DP];
  __shared__ float vhat[DP];
  __shared__ float red[4];
  float* ks = buf;
  float* vs = buf + CH * LD;
  float* qsm = buf + 2 * CH * LD;
  const int g = blockIdx.x / split;
  const int part = blockIdx.x - g * split;
  const int bh = blockIdx.y;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15;
  const int g4 = lane >> 4;
  const int dq = (wave >> 1) * (DP / 2);
  const int eq = (wave & 1) * (DP / 2);
  const int NG = (NT + G - 1) / G;
  const int nblk = min(G, NT - g * G);
  const int per = (nblk + split - 1) / split;
  const int j0 = g * G + min(part * per, nblk);
  const int j1 = g * G + min((part + 1) * per, nblk);
  const int64_t row_bytes = (int64_t)D * EL::ES;
  const int64_t slice = (int64_t)bh * Tslice * row_bytes;

  if (tid < DP) kbar[tid] = vhat[tid] = 0.f;  // columns past D stay zero

  // Staging: thread (sr, sc) moves chunk sc of rows sr, sr + RPP, ...
  const int sc = tid % C::NCHP;
  const int sr = tid / C::NCHP;
  // Column sums: threads 0 .. 127 column tid of k and q, threads 128 .. 255 column tid - 128 of v.
  const int col = tid & 127;
  const bool kq_side = tid < 128;
  uint4 kreg[C::PASSES], vreg[C::PASSES], qreg[C::PASSES];
  const uint32_t lane_off = sc * EPC < D ? (uint32_t)(sr * (int)row_bytes + sc * 16) : 0x80000000u;
  // Chunk sc of the rows r0 + p RPP + sr, zero past the n rows from r0.
  auto load = [&](const unsigned char* base, int r0, int n, uint4 (&dst)[C::PASSES]) {
    const unsigned char* p0 = base + slice + (int64_t)r0 * row_bytes;
    const rsrc_t rs = make_rsrc(p0, (uint32_t)(n * (int)row_bytes));
#pragma unroll
    for (int p = 0; p < C::PASSES; ++p) {
      if constexpr (VEC) {
        dst[p] = buf_load16(rs, lane_off + (uint32_t)(p * C::RPP * (int)row_bytes));
      } else {
        uint32_t w[4] = {0u, 0u, 0u, 0u};
        if (p * C::RPP + sr < n) {
#pragma unroll
          for (int i = 0; i < EPC; ++i)
            if (sc * EPC + i < D) EL::put(w, i, p0 + (int64_t)(p * C::RPP + sr) * row_bytes, sc * EPC + i);
        }
        dst[p] = make_uint4(w[0], w[1], w[2], w[3]);
      }
    }
  };
  auto fetch = [&](int r0, int n) {
    load(k, r0, n, kreg);
    load(v, r0, n, vreg);
    load(q, r0, n, qreg);
  };
  auto stash1 = [&](float* dst, const uint4& x) {
    float f[EPC];
    EL::widen(x, f);
#pragma unroll
    for (int i = 0; i < EPC; i += 4) *reinterpret_cast<float4*>(dst + i) = make_float4(f[i], f[i + 1], f[i + 2], f[i + 3]);
  };
  auto stash = [&]() {
    if (sc >= C::NCH) return;
#pragma unroll
    for (int p = 0; p < C::PASSES; ++p) {
      const int o = (p * C::RPP + sr) * LD + sc * EPC;
      stash1(ks + o, kreg[p]);
      stash1(vs + o, vreg[p]);
      stash1(qsm + o, qreg[p]);
    }
  };

  f32x4_t gacc[TL][TL];
#pragma unroll
  for (int a = 0; a < TL; ++a)
#pragma unroll
    for (int b = 0; b < TL; ++b) gacc[a][b] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
  if (j0 < j1) fetch(j0 * BT, min(CH, min(BT, T - j0 * BT)));
  for (int j = j0; j < j1; ++j) {
    const int r0 = j * BT;
    const int n = min(BT, T - r0);
    f32x4_t acc[TL][TL];
#pragma unroll
    for (int a = 0; a < TL; ++a)
#pragma unroll
      for (int b = 0; b < TL; ++b) acc[a][b] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    float ksum = 0.f, qs = 0.f;  // ksum: of v on the upper threads
    for (int c0 = 0; c0 < n; c0 += CH) {
      const int cn = min(CH, n - c0);
      __syncthreads();  // the buffers have been read
      stash();
      __syncthreads();
      if (c0 + CH < n)
        fetch(r0 + c0 + CH, min(CH, n - c0 - CH));
      else if (j + 1 < j1)
        fetch(r0 + BT, min(CH, min(BT, T - r0 - BT)));
      if (col < D) {  // rows past cn are zero, and adding them changes no bit
        const float* p = (kq_side ? ks : vs) + col;
#pragma unroll 8
        for (int t = 0; t < CH; ++t) ksum += p[t * LD];
        if (kq_side) {
#pragma unroll 8
          for (int t = 0; t < CH; ++t) qs += qsm[t * LD + col];
        }
      }
      const float* ka = ks + g4 * LD + dq + l16;
      const float* va = vs + g4 * LD + eq + l16;
      for (int t0 = 0; t0 < cn; t0 += 16) {  // 16 rows (rows past cn are zero), four per MFMA
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          float a[TL], b[TL];
#pragma unroll
          for (int t = 0; t < TL; ++t) {
            a[t] = ka[(t0 + 4 * s) * LD + 16 * t];
            b[t] = va[(t0 + 4 * s) * LD + 16 * t];
          }
#pragma unroll
          for (int x = 0; x < TL; ++x)
#pragma unroll
            for (int y = 0; y < TL; ++y)
              acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[x], b[y], acc[x][y], 0, 0, 0);
        }
      }
    }
    if (col < D) {
      const int64_t so = ((int64_t)bh * NT + j) * D + col;
      if (kq_side) {
        const float kb = ksum / (float)n;
        kbar[col] = kb;
        qc[so] = qs / (float)n;  // :101
        kc[so] = kb;             // :102
      } else {
        vhat[col] = ksum;
        vc[so] = ksum;           // :103 (a sum, not a mean)
      }
    }
    __syncthreads();  // the sums are in place, and the K/V chunk has been read
#pragma unroll
    for (int x = 0; x < TL; ++x) {
      const float4 kb = *reinterpret_cast<const float4*>(kbar + dq + 16 * x + 4 * g4);
      const float kbv[4] = {kb.x, kb.y, kb.z, kb.w};
#pragma unroll
      for (int y = 0; y < TL; ++y) {
        const float vh = vhat[eq + 16 * y + l16];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float h = fmaf(-kbv[i], vh, acc[x][y][i]);  // :107 (zero past D)
          gacc[x][y][i] += h;
          buf[(dq + 16 * x + 4 * g4 + i) * HLD + eq + 16 * y + l16] = h;
        }
      }
    }
    __syncthreads();
    float nsq = 0.f;
    const int d0 = 8 * (tid >> 4);
    const int e0 = 8 * (tid & 15);
    if (d0 < D && e0 < D) {
#pragma unroll
      for (int a = 0; a < 8; ++a) {
        const float4 h0 = *reinterpret_cast<const float4*>(buf + (d0 + a) * HLD + e0);
        const float4 h1 = *reinterpret_cast<const float4*>(buf + (d0 + a) * HLD + e0 + 4);
        const float h[8] = {h0.x, h0.y, h0.z, h0.w, h1.x, h1.y, h1.z, h1.w};
#pragma unroll
        for (int b = 0; b < 8; ++b) nsq = fmaf(h[b], h[b], nsq);
      }
    }
    nsq = wave_sum_xor(nsq);
    if (lane == 0) red[wave] = nsq;
    __syncthreads();
    if (tid == 0) hnorm[(int64_t)bh * NT + j] = sqrt_rn((red[0] + red[1]) + (red[2] + red[3]));  // :110, :287
  }
  // hbar_g = (1/G) sum over the group, the missing blocks of the last group counting as zeros (:294-299).
  float* hg = split == 1 ? hgroup + ((int64_t)bh * NG + g) * D * D
                         : partials + (((int64_t)bh * NG + g) * split + part) * D * D;
  const float Gf = split == 1 ? (float)G : 1.f;
#pragma unroll
  for (int x = 0; x < TL; ++x)
#pragma unroll
    for (int y = 0; y < TL; ++y)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int d = dq + 16 * x + 4 * g4 + i;
        const int e = eq + 16 * y + l16;
        if (d < D && e < D) hg[d * D + e] = gacc[x][y][i] / Gf;
      }
}

// hgroup[g] = (sum over the parts of partials[g], in part order) / G; one entry per thread.
__global__ __launch_bounds__(256) void k2_any_reduce(const float* __restrict__ partials, float* __restrict__ hgroup,
                                                     int split, int G, int dd) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= dd) return;
  const int64_t grp = (int64_t)blockIdx.z * gridDim.y + blockIdx.y;
  const float* src = partials + grp * split * dd + i;
  float a = src[0];
  for (int p = 1; p < split; ++p) a += src[(int64_t)p * dd];
  hgroup[grp * dd + i] = a / (float)G;
}

// ---- selection scores -----------------------------------------------------------
// score[I][j] = sum_d qc[I][d] * fl(scale * kc[j][d]) + log(hnorm[j] + 1e-6) [+ noise[j]], the head
// dims k3_scores (64 and 128) does not take.  One workgroup per 64 x 64 tile: 64 rows of qc and of
// scale * kc in LDS, each wave 32 x 32 scores on the 16x16x4 fp32 MFMA with features in ascending
// order, which is the chain of fused multiply-adds over d bit for bit.  Rows of LD floats, LD four
// times an odd number: 16 rows x 4 features fall into 64 distinct banks.
//
// One thread per score instead, each reading both of its rows from L2, took 420 us at 16 heads x
// 270 blocks of D 96 (now 11).
constexpr int kScoreTile = 64;

__global__ __launch_bounds__(256) void k3_scores_any(const float* __restrict__ qc, const float* __restrict__ kc,
                                                     const float* __restrict__ hnorm, const float* __restrict__ noise,
                                                     float scale, int use_cov_bias, float* __restrict__ scores, int NT,
                                                     int D, int LD, int ntj, int vec) {
  __shared__ __attribute__((aligned(16))) float rows[2 * kScoreTile * 132];  // 64 rows of qc, then 64 of scale * kc
  float* qs = rows;
  float* ks = rows + kScoreTile * LD;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int l16 = lane & 15;
  const int g4 = lane >> 4;
  const int bh = blockIdx.z;
  const int ti = blockIdx.x / ntj;
  const int i0 = ti * kScoreTile;
  const int j0 = (blockIdx.x - ti * ntj) * kScoreTile;
  const float* qb = qc + (int64_t)bh * NT * D;
  const float* kb = kc + (int64_t)bh * NT * D;
  const int r = tid >> 2;  // the row this thread stages, four threads to a row
  const bool iq = i0 + r < NT, jk = j0 + r < NT;
  for (int d = 4 * (tid & 3); d < LD; d += 16) {
    float q4[4] = {0.f, 0.f, 0.f, 0.f}, k4[4] = {0.f, 0.f, 0.f, 0.f};
    const float* qp = qb + (int64_t)(i0 + r) * D + d;
    const float* kp = kb + (int64_t)(j0 + r) * D + d;
    if (vec) {
      if (iq && d < D) {
        const float4 x = *reinterpret_cast<const float4*>(qp);
        q4[0] = x.x; q4[1] = x.y; q4[2] = x.z; q4[3] = x.w;
      }
      if (jk && d < D) {
        const float4 x = *reinterpret_cast<const float4*>(kp);
        k4[0] = x.x; k4[1] = x.y; k4[2] = x.z; k4[3] = x.w;
      }
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (iq && d + i < D) q4[i] = qp[i];
        if (jk && d + i < D) k4[i] = kp[i];
      }
    }
    *reinterpret_cast<float4*>(qs + r * LD + d) = make_float4(q4[0], q4[1], q4[2], q4[3]);
    *reinterpret_cast<float4*>(ks + r * LD + d) =
        make_float4(mul_rn(scale, k4[0]), mul_rn(scale, k4[1]), mul_rn(scale, k4[2]), mul_rn(scale, k4[3]));
  }
  __syncthreads();
  f32x4_t acc[2][2];
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y) acc[x][y] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
  const float* qa = qs + ((wave >> 1) * 32 + l16) * LD + g4;
  const float* ka = ks + ((wave & 1) * 32 + l16) * LD + g4;
  for (int d = 0; d < D; d += 4) {
    const float a[2] = {qa[d], qa[16 * LD + d]};
    const float b[2] = {ka[d], ka[16 * LD + d]};
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int y = 0; y < 2; ++y) acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[x], b[y], acc[x][y], 0, 0, 0);
  }
#pragma unroll
  for (int y = 0; y < 2; ++y) {
    const int j = j0 + (wave & 1) * 32 + 16 * y + l16;
    if (j >= NT) continue;
    float bias = 0.f;
    if (use_cov_bias) {
      bias = logf(hnorm[(int64_t)bh * NT + j] + 1e-6f);
      if (noise) bias = bias + noise[(int64_t)bh * NT + j];
    }
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int I = i0 + (wave >> 1) * 32 + 16 * x + 4 * g4 + i;
        if (I < NT) scores[((int64_t)bh * NT + I) * NT + j] = acc[x][y][i] + bias;
      }
  }
}

namespace {

template <typename F>
hipError_t by_dtype(int dtype, F&& f) {
  switch (dtype) {
    case kAnyF32: f(F32E{}); break;
    case kAnyBf16: f(Bf16E{}); break;
    case kAnyF16: f(F16E{}); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace

// Parts per group: about two workgroups per CU (256 CUs), at least one block each.
int block_stats_any_split(int bh, int T, int BT, int G) {
  const int NT = (T + BT - 1) / BT;
  const int64_t groups = (int64_t)((NT + G - 1) / G) * bh;
  const int nblk = min(G, NT);
  int split = 1;
  while (groups * split < 512 && 2 * split <= nblk) split *= 2;
  return split;
}

hipError_t launch_block_stats_any(const void* q, const void* k, const void* v, float* qc, float* kc, float* vc,
                                  float* hnorm, float* hgroup, float* partials, int split, int bh, int T, int Tslice,
                                  int D, int BT, int G, int dtype, hipStream_t stream) {
  if (D < 1 || D > 128 || BT < 1 || G < 1 || split < 1 || (split > 1 && partials == nullptr)) return hipErrorInvalidValue;
  const int NT = (T + BT - 1) / BT;
  const int NG = (NT + G - 1) / G;
  const dim3 grid(NG * split, bh);
  const hipError_t e = by_dtype(dtype, [&](auto el) {
    using EL = decltype(el);
    const bool vec = (D * EL::ES) % 16 == 0 && (((uintptr_t)q | (uintptr_t)k | (uintptr_t)v) & 15u) == 0;
    auto go = [&](auto kern) {
      hipLaunchKernelGGL(kern, grid, dim3(256), 0, stream, (const unsigned char*)q, (const unsigned char*)k,
                         (const unsigned char*)v, qc, kc, vc, hnorm, hgroup, partials, T, Tslice, D, BT, NT, G, split);
    };
    if (!vec)
      go(k2_block_stats_any<EL, 128, false>);
    else if (D <= 64)
      go(k2_block_stats_any<EL, 64, true>);
    else if (D <= 96)
      go(k2_block_stats_any<EL, 96, true>);
    else
      go(k2_block_stats_any<EL, 128, true>);
  });
  if (e != hipSuccess || split == 1) return e;
  hipLaunchKernelGGL(k2_any_reduce, dim3((D * D + 255) / 256, NG, bh), dim3(256), 0, stream, (const float*)partials,
                     hgroup, split, G, D * D);
  return hipGetLastError();
}

hipError_t launch_scores_any(const float* qc, const float* kc, const float* hnorm, const float* noise, float scale,
                             int use_cov_bias, float* scores, int bh, int NT, int D, hipStream_t stream) {
  if (D < 1 || D > 128) return hipErrorInvalidValue;
  const int nt = (NT + kScoreTile - 1) / kScoreTile;
  const int LD = 4 * (((D + 3) / 4) | 1);
  const int vec = D % 4 == 0 && (((uintptr_t)qc | (uintptr_t)kc) & 15u) == 0;
  hipLaunchKernelGGL(k3_scores_any, dim3(nt * nt, 1, bh), dim3(256), 0, stream, qc, kc, hnorm, noise, scale,
                     use_cov_bias, scores, NT, D, LD, nt, vec);
  return hipGetLastError();
}

}  // namespace pasa
