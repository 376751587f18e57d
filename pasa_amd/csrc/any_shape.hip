// Statistics and selection scores for shapes the tuned kernels do not take: fp32 q, k, v; any
// head dim up to 128; any group size; block sizes 16 .. 256 (the attention stage of the same
// shapes is any_attn.hip).  Plain VALU arithmetic, one workgroup per (slice, group).
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

// Element access for the three input types.
struct F32E {
  __device__ static float load(const void* p, int64_t i) { return ((const float*)p)[i]; }
};
struct Bf16E {
  __device__ static float load(const void* p, int64_t i) {
    return bf16_bits_to_f32(((const uint16_t*)p)[i]);
  }
};
struct F16E {
  __device__ static float load(const void* p, int64_t i) { return (float)((const _Float16*)p)[i]; }
};

constexpr int kAnyChunk = 32;   // rows of a staged K/V chunk
constexpr int kAnyLd = 132;     // LDS row stride (floats) of staged rows: 16-byte aligned, so
                                // row pieces are ds_read_b128

}  // namespace

// ---- block statistics ---------------------------------------------------------
// One workgroup (256 threads) per (group of G key blocks, slice); the group's blocks in
// ascending order, each in 32-row chunks of k and v staged in LDS as fp32 (132-float rows,
// feature columns D .. 127 zero).  Thread t owns an 8 x 8 tile of the D x D moment, rows
// d = 8 (t >> 4) .. + 7 and columns e = 8 (t & 15) .. + 7: per staged row, four 16-byte
// reads feed 64 FMAs.  H_j[d][e] = sum_t k_t[d] v_t[e] - kbar_j[d] V^_j[e] (:106-107), the
// sum over the block's rows in order; entries past D stay zero and are not stored.  Threads
// t < D own column t of the block sums of q, k and v.  The group sum adds H_j in block order,
// then / G.
template <typename EL>
__global__ __launch_bounds__(256) void k2_block_stats_any(const void* __restrict__ q, const void* __restrict__ k,
                                                          const void* __restrict__ v, float* __restrict__ qc,
                                                          float* __restrict__ kc, float* __restrict__ vc,
                                                          float* __restrict__ hnorm, float* __restrict__ hgroup,
                                                          int T, int Tslice, int D, int BT, int NT, int G) {
  constexpr int CH = kAnyChunk, LD = kAnyLd;
  __shared__ __attribute__((aligned(16))) float ks[CH * LD];
  __shared__ __attribute__((aligned(16))) float vs[CH * LD];
  __shared__ float qsm[CH * 128];  // the chunk's q rows (only their column sums are needed)
  __shared__ float kbar[128];
  __shared__ float vhat[128];
  __shared__ float red[4];
  const int g = blockIdx.x;
  const int bh = blockIdx.y;
  const int tid = threadIdx.x;
  const int NG = (NT + G - 1) / G;
  const int64_t base = (int64_t)bh * Tslice * D;
  const int d0 = 8 * (tid >> 4);
  const int e0 = 8 * (tid & 15);
  const bool owns = d0 < D && e0 < D;  // the tile holds at least one entry of the moment
  for (int i = tid; i < CH * LD; i += 256) {
    ks[i] = 0.f;
    vs[i] = 0.f;
  }
  if (tid < 128) {
    kbar[tid] = 0.f;
    vhat[tid] = 0.f;
  }
  float gacc[64];
#pragma unroll
  for (int m = 0; m < 64; ++m) gacc[m] = 0.f;
  const int j1 = min(NT, (g + 1) * G);
  for (int j = g * G; j < j1; ++j) {
    const int r0 = j * BT;
    const int n = min(BT, T - r0);
    float hacc[64];
#pragma unroll
    for (int m = 0; m < 64; ++m) hacc[m] = 0.f;
    float qs = 0.f, ksum = 0.f, vsum = 0.f;
    for (int c0 = 0; c0 < n; c0 += CH) {
      const int cn = min(CH, n - c0);
      __syncthreads();  // the previous chunk's reads are done (and the zero fill landed)
      for (int i = tid; i < cn * D; i += 256) {
        const int t = i / D;
        const int d = i - t * D;
        const int64_t off = base + (int64_t)(r0 + c0 + t) * D + d;
        ks[t * LD + d] = EL::load(k, off);
        vs[t * LD + d] = EL::load(v, off);
        qsm[t * 128 + d] = EL::load(q, off);
      }
      __syncthreads();
      if (tid < D) {
        for (int t = 0; t < cn; ++t) {
          ksum += ks[t * LD + tid];
          vsum += vs[t * LD + tid];
          qs += qsm[t * 128 + tid];
        }
      }
      if (owns) {
        for (int t = 0; t < cn; ++t) {
          const float4 k0 = *reinterpret_cast<const float4*>(ks + t * LD + d0);
          const float4 k1 = *reinterpret_cast<const float4*>(ks + t * LD + d0 + 4);
          const float4 v0 = *reinterpret_cast<const float4*>(vs + t * LD + e0);
          const float4 v1 = *reinterpret_cast<const float4*>(vs + t * LD + e0 + 4);
          const float kk[8] = {k0.x, k0.y, k0.z, k0.w, k1.x, k1.y, k1.z, k1.w};
          const float vv[8] = {v0.x, v0.y, v0.z, v0.w, v1.x, v1.y, v1.z, v1.w};
#pragma unroll
          for (int a = 0; a < 8; ++a)
#pragma unroll
            for (int b = 0; b < 8; ++b) hacc[8 * a + b] = fmaf(kk[a], vv[b], hacc[8 * a + b]);
        }
      }
    }
    __syncthreads();
    if (tid < D) {
      const float kb = ksum / (float)n;
      kbar[tid] = kb;
      vhat[tid] = vsum;
      const int64_t so = ((int64_t)bh * NT + j) * D + tid;
      qc[so] = qs / (float)n;  // :101
      kc[so] = kb;             // :102
      vc[so] = vsum;           // :103 (a sum, not a mean)
    }
    __syncthreads();
    float nsq = 0.f;
    if (owns) {
#pragma unroll
      for (int a = 0; a < 8; ++a)
#pragma unroll
        for (int b = 0; b < 8; ++b) {
          const float h = hacc[8 * a + b] - kbar[d0 + a] * vhat[e0 + b];  // :107 (zero past D)
          nsq = fmaf(h, h, nsq);
          gacc[8 * a + b] += h;
        }
    }
    nsq = wave_sum(nsq);
    if ((tid & 63) == 0) red[tid >> 6] = nsq;
    __syncthreads();
    if (tid == 0) hnorm[(int64_t)bh * NT + j] = sqrt_rn((red[0] + red[1]) + (red[2] + red[3]));  // :110, :287
  }
  // hbar_g = (1/G) sum over the group, the missing blocks of the last group counting as zeros (:294-299).
  if (owns) {
    float* hg = hgroup + ((int64_t)bh * NG + g) * D * D;
#pragma unroll
    for (int a = 0; a < 8; ++a)
#pragma unroll
      for (int b = 0; b < 8; ++b)
        if (d0 + a < D && e0 + b < D) hg[(d0 + a) * D + e0 + b] = gacc[8 * a + b] / (float)G;
  }
}

// ---- selection scores -----------------------------------------------------------
// score[I][j] = sum_d qc[I][d] * fl(scale * kc[j][d]) + log(hnorm[j] + 1e-6) [+ noise[j]],
// one thread per score, features in ascending order; one row per grid x index.
__global__ __launch_bounds__(256) void k3_scores_any(const float* __restrict__ qc, const float* __restrict__ kc,
                                                     const float* __restrict__ hnorm, const float* __restrict__ noise,
                                                     float scale, int use_cov_bias, float* __restrict__ scores, int NT,
                                                     int D) {
  const int j = blockIdx.y * 256 + threadIdx.x;
  const int I = blockIdx.x;  // the row on grid x: NT may exceed grid y's 65,535
  const int bh = blockIdx.z;
  if (j >= NT) return;
  const float* qi = qc + ((int64_t)bh * NT + I) * D;
  const float* kj = kc + ((int64_t)bh * NT + j) * D;
  float acc = 0.f;
  for (int d = 0; d < D; ++d) acc = fmaf(qi[d], mul_rn(scale, kj[d]), acc);
  float bias = 0.f;
  if (use_cov_bias) {
    bias = logf(hnorm[(int64_t)bh * NT + j] + 1e-6f);
    if (noise) bias = bias + noise[(int64_t)bh * NT + j];
  }
  scores[((int64_t)bh * NT + I) * NT + j] = acc + bias;
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

hipError_t launch_block_stats_any(const void* q, const void* k, const void* v, float* qc, float* kc, float* vc,
                                  float* hnorm, float* hgroup, int bh, int T, int Tslice, int D, int BT, int G,
                                  int dtype, hipStream_t stream) {
  if (D < 1 || D > 128 || BT < 1 || G < 1) return hipErrorInvalidValue;
  const int NT = (T + BT - 1) / BT;
  const int NG = (NT + G - 1) / G;
  const dim3 grid(NG, bh);
  return by_dtype(dtype, [&](auto el) {
    hipLaunchKernelGGL(k2_block_stats_any<decltype(el)>, grid, dim3(256), 0, stream, q, k, v, qc, kc, vc, hnorm,
                       hgroup, T, Tslice, D, BT, NT, G);
  });
}

hipError_t launch_scores_any(const float* qc, const float* kc, const float* hnorm, const float* noise, float scale,
                             int use_cov_bias, float* scores, int bh, int NT, int D, hipStream_t stream) {
  if (D < 1 || D > 128) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k3_scores_any, dim3(NT, (NT + 255) / 256, bh), dim3(256), 0, stream, qc, kc, hnorm, noise,
                     scale, use_cov_bias, scores, NT, D);
  return hipGetLastError();
}

}  // namespace pasa
