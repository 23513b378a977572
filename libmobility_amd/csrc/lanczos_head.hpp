// The second half of a Lanczos step (LanczosAlgorithm.cu:128-152) for short
// vectors, at the start of the product that follows it: every workgroup of the
// product finishes the step for itself from w = M v_i, so the step needs no
// launch of its own and v_{i+1} is in LDS when the pairs begin.  The sums add
// what k_lanczos_step_1wg adds, in its order (the same bits): its thread t is
// lane t mod 64 of its wave t / 64, whose sums the four waves here take in turn.
#pragma once
#include "kernels.hpp"
#include "lane_sums.hpp"

namespace lm {

// sum over kLanczosFusedThreads virtual threads in k_lanczos_step_1wg's order,
// p[j] the values of virtual wave (wave + 4 j); sh is not reused
__device__ inline double head_sum(double* p, double* sh) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    p[j] = wave_sum(p[j]);
    if (lane == 0) sh[wave + 4 * j] = p[j];
  }
  __syncthreads();
  double t = 0.0;
#pragma unroll
  for (int k = 0; k < kLanczosFusedThreads / 64; ++k) t += sh[k];
  return t;
}

// 256 threads; v_{i+1} to s_v[0 .. n), and with `write` (one workgroup of the
// launch) to memory, with alpha[i] and beta[i].
__device__ inline void lanczos_head(const LanczosHead& h, double* s_v, double (*sh)[16],
                                    bool write) {
  static_assert(kLanczosFusedThreads == 1024 && kLanczosHeadMax == 4096, "4 x 4 entries per thread");
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int n = h.n;
  const double bprev = h.i > 0 ? h.sc->beta[h.i - 1] : 0.0;
  const double normz = h.sc->normz;
  double w[4][4], v[4][4], vp[4][4];
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int k = 64 * (wave + 4 * j) + lane + 1024 * r;
      w[j][r] = v[j][r] = vp[j][r] = 0.0;
      if (k < n) {
        w[j][r] = h.w[k];
        v[j][r] = h.v[k];
        if (h.i > 0) vp[j][r] = h.vp[k];
      }
    }
  double p[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    p[j] = 0.0;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int k = 64 * (wave + 4 * j) + lane + 1024 * r;
      if (k < n) {
        if (h.i > 0) w[j][r] -= bprev * vp[j][r];
        p[j] += w[j][r] * v[j][r];
      }
    }
  }
  const double alpha = head_sum(p, sh[0]);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    p[j] = 0.0;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int k = 64 * (wave + 4 * j) + lane + 1024 * r;
      if (k < n) {
        w[j][r] -= alpha * v[j][r];
        p[j] += w[j][r] * w[j][r];
      }
    }
  }
  double beta = sqrt(head_sum(p, sh[1]));
  if (beta < 1e-3 * alpha / normz) beta = 0.0;  // LanczosAlgorithm.cu:140-142
  const double inv = beta > 0.0 ? 1.0 / beta : 0.0;
  if (write && threadIdx.x == 0) {
    h.sc->alpha[h.i] = alpha;
    h.sc->beta[h.i] = beta;
  }
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int k = 64 * (wave + 4 * j) + lane + 1024 * r;
      if (k < n) {
        const double x = beta > 0.0 ? w[j][r] * inv : (k == 0 ? 1.0 : 0.0);
        s_v[k] = x;
        if (write) h.v_next[k] = x;
      }
    }
  __syncthreads();
}

}  // namespace lm
