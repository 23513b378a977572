// The product of small systems: sources across the lanes.
//
// k_pair (nbody_kernels.hip) puts 256 targets into a workgroup's lanes, so a
// system of 1000 particles fills 4 workgroups, has to be cut into source
// chunks whose partial sums a second kernel adds, and each chunk is a serial
// chain of 64 to 256 pairs behind one LDS tile.  Here a wave holds 64 sources
// in its lanes and meets T targets, whose records it reads through the scalar
// cache; each lane sums its own sources' contributions to the T targets, and
// the wave adds its lanes at the end (lane swaps, then rotations inside the
// rows of 16, a fixed order).  With SPLIT waves per group of T targets (SPLIT
// 4: the whole workgroup) the waves take every SPLIT-th group of 64 sources
// and meet in LDS, added in wave order.  There are N / T units of work instead
// of N / 256, no partial sums in memory and no second launch.
//
// Bound by latency below about 500 particles (2.8-3.5 us: launch, one load of
// the sources, the lane sums) and by VALU issue above.  T = 4: the fold costs
// about 100 instructions per wave against 100 (open) to 770 (wall 6x6) per
// group of 64 sources; T = 8 was 1.2-1.8x slower for 6x6 blocks (196-227
// VGPRs, 2 waves per SIMD) and within 7 % for the translational block.
// Microseconds per product, k_pair + k_chunk_reduce against this kernel:
//   particles          96           512          1024         2000        4096        8192
//   open UF FP64   11.0 / 3.0   13.0 / 3.5   15.0 / 4.6   19.7 / 8.5   33 / 22.5    81 / 74
//   open UF FP32    9.3 / 2.8   11.3 / 3.3   13.2 / 4.2   17.7 / 6.5   25 / 15.3    55 / 44
//   wall 6x6 FP64  40.8 / 4.8   44.4 / 7.1   48.5 / 11.4  61.3 / 31.3  126 / 105   411 / 406
//   wall 6x6 FP32  36.4 / 4.5   39.9 / 6.4   43.8 / 9.9   54.2 / 22.2   95 / 66    242 / 229
#include <type_traits>

#include "kernels.hpp"
#include "lane_sums.hpp"
#include "lm_common.hpp"
#include "pair_device.hpp"
#include "pair_math.hpp"

namespace lm {

namespace {

constexpr int kWideWaves = kPairThreads / 64;

// Sums NV values over the 64 lanes: v[q], q < NV / 4, of row r (lanes 16r ..
// 16r + 15) becomes the sum of value (r / 2) NV/2 + (r mod 2) NV/4 + q.
template <int NV>
__device__ inline void wave_fold(double* v) {
#pragma unroll
  for (int q = 0; q < NV / 2; ++q) v[q] = fold32(v[q], v[q + NV / 2]);
#pragma unroll
  for (int q = 0; q < NV / 4; ++q) v[q] = row_sum(fold16(v[q], v[q + NV / 4]));
}

// The sums of T targets over the sources base, base + 64 * stride, ... < src1
// (64 at a time, one per lane), left in v (T times U, then T times W) per lane.
template <class R, bool WALL, int BLK, int T>
__device__ __attribute__((always_inline)) inline void wide_sources(const typename Rec<R>::T* __restrict__ pos,
                                    const double* __restrict__ F, const double* __restrict__ Tq,
                                    int64_t tgt0, int ntgt, int64_t base, int64_t src1, int stride,
                                    double t0, double rt0, double r0, double* v) {
  using R4 = typename Rec<R>::T;
  constexpr bool kNeedF = (BLK & (kUF | kWF)) != 0;
  constexpr bool kNeedT = (BLK & (kUT | kWT)) != 0;
  constexpr bool kAngular = (BLK & (kWT | kWF)) != 0;
  constexpr int G = T < 4 ? T : 4;  // pairs per overlap test
  const int lane = threadIdx.x & 63;
  const Vec3<R> zero = {R(0), R(0), R(0)};
  R4 pi[T];  // uniform: scalar loads
#pragma unroll
  for (int t = 0; t < T; ++t) pi[t] = pos[tgt0 + (t < ntgt ? t : ntgt - 1)];
  Vec3<R> u[T], w[T], none = zero;
#pragma unroll
  for (int t = 0; t < T; ++t) u[t] = w[t] = zero;
  const R ta = R(r0 / rt0);  // 1/a: symmetric units (pair_math.hpp)
  for (; base < src1; base += 64 * (int64_t)stride) {
    const int64_t j = base + lane;
    R4 pj = far_record<R4>();
    Vec3<R> fj = zero, tj = zero;
    if (j < src1) {
      pj = pos[j];
      const R b = WALL ? pj.w : R(1);  // the wall's damping goes with the force
      if (kNeedF) fj = {b * R(F[3 * j]), b * R(F[3 * j + 1]), b * R(F[3 * j + 2])};
      const R bt = b * ta;
      if (kNeedT) tj = {bt * R(Tq[3 * j]), bt * R(Tq[3 * j + 1]), bt * R(Tq[3 * j + 2])};
    }
    if constexpr (WALL) {
#pragma unroll
      for (int t = 0; t < T; ++t) {
        PairGeo<R> g;
        pair_distances<R, true>(pi[t].x, pi[t].y, pi[t].z, pj.x, pj.y, pj.z, g);
        pair_inverses<R, true>(g);
        pair_unit<R, true, BLK, false>(g, pj.z, fj, tj, zero, zero, u[t], w[t], none, none);
      }
    } else {
#pragma unroll
      for (int g = 0; g < T; g += G) {
        PairGeo<R> q[G];
        RpyCoef<R> cf[G];
        NearTestCmp<R> near;
#pragma unroll
        for (int t = 0; t < G; ++t) {
          pair_distances<R, false>(pi[g + t].x, pi[g + t].y, pi[g + t].z, pj.x, pj.y, pj.z, q[t]);
          pair_inverses<R, false>(q[t]);
          cf[t] = RpyCoef<R>{};
          rpy_unit_far<R, BLK>(q[t].ir, cf[t]);
          near.add(q[t].r2);
        }
        if (__builtin_expect(near.hit(), 0)) {
          lm_rare_path();
#pragma unroll
          for (int t = 0; t < G; ++t) rpy_unit_near_select<R, BLK>(q[t].r2, q[t].ir, cf[t]);
        }
#pragma unroll
        for (int t = 0; t < G; ++t)
          open_unit<R, BLK, false>(q[t].dx, q[t].dy, q[t].dz, cf[t], fj, tj, zero, zero, u[g + t],
                                   w[g + t], none, none);
      }
    }
  }
#pragma unroll
  for (int t = 0; t < T; ++t) {
    const double b = WALL ? (double)pi[t].w : 1.0;
    const double us = 0.75 * t0 * b, ws = rt0 * b;
    v[3 * t + 0] = us * (double)u[t].x;
    v[3 * t + 1] = us * (double)u[t].y;
    v[3 * t + 2] = us * (double)u[t].z;
    if constexpr (kAngular) {
      v[3 * T + 3 * t + 0] = ws * (double)w[t].x;
      v[3 * T + 3 * t + 1] = ws * (double)w[t].y;
      v[3 * T + 3 * t + 2] = ws * (double)w[t].z;
    }
  }
}

// A unit's targets [tgt0, tgt0 + ntgt) and its system's particles [src0, src1).
struct WideUnit {
  int64_t tgt0, src0, src1;
  int ntgt, kind, sys;
};
template <int T>
__device__ inline WideUnit wide_unit(const WideArgs& a, int unit, int kind) {
  WideUnit w;
  w.kind = kind;
  if (a.items != nullptr) {
    const WideItem it = a.items[unit];
    const SymSys S = a.sys[it.sys];
    w.sys = it.sys;
    w.src0 = S.off;
    w.src1 = S.off + S.n;
    w.tgt0 = S.off + it.tgt;
    w.kind = S.wall;
  } else {
    w.sys = unit / a.per_sys;
    w.src0 = (int64_t)w.sys * a.ns;
    w.src1 = w.src0 + a.ns;
    w.tgt0 = w.src0 + (int64_t)(unit - w.sys * a.per_sys) * T;
  }
  w.ntgt = (int)min((int64_t)T, w.src1 - w.tgt0);
  return w;
}

// The wave's sums of v, in value order, to red, or (add) added to it.
template <int NV>
__device__ inline void wide_fold_to(double* v, double* red, bool add = false) {
  wave_fold<NV>(v);
  const int lane = threadIdx.x & 63;
  if ((lane & 15) == 0) {
    const int row = lane >> 4;
    red += (row >> 1) * (NV / 2) + (row & 1) * (NV / 4);
#pragma unroll
    for (int q = 0; q < NV / 4; ++q) red[q] = add ? red[q] + v[q] : v[q];
  }
}

// Value q of the unit: its wave's sum, or the waves' in order.
template <int SPLIT, int NV>
__device__ inline double wide_value(const double (*s_red)[NV], int wave, int q) {
  if (SPLIT == 1) return s_red[wave][q];
  double s = s_red[0][q];
#pragma unroll
  for (int w = 1; w < kWideWaves; ++w) s += s_red[w][q];
  return s;
}

}  // namespace

// Unit of work u: T targets of one system, from the list `items` or, for
// equal systems, by its number.  SPLIT 4: one unit per workgroup; SPLIT 1: one
// per wave.  LONG: the lanes' sums go to FP64 every kWideFp32Sources sources.  It
// takes 6 to 27 more registers, so only where a system has more: 60000 particles
// among 40000 systems of 64, FP32, 2.23 -> 2.31 ms (open UF), 11.1 -> 11.7 (wall 6x6).
template <class R, int KIND, int BLK, int T, int SPLIT, bool LONG>
__global__ __launch_bounds__(kPairThreads) void k_pair_wide(WideArgs a) {
  using R4 = typename Rec<R>::T;
  constexpr bool kAngular = (BLK & (kWT | kWF)) != 0;
  constexpr int NV = (kAngular ? 6 : 3) * T;
  static_assert(NV % 4 == 0, "the lane fold needs a multiple of 4 values");
  __shared__ double s_red[kWideWaves][NV];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (a.stop != nullptr) {
    // one read per workgroup, so that all its threads take the same branch
    __shared__ int s_stop;
    if (threadIdx.x == 0) s_stop = *(volatile const int*)a.stop;
    __syncthreads();
    if (s_stop != 0) return;
  }
  const int unit = SPLIT == 1 ? (int)blockIdx.x * kWideWaves + wave : (int)blockIdx.x;
  bool live = unit < a.nunits;
  WideUnit w{0, 0, 0, 1, KIND, 0};
  if (live) {
    w = wide_unit<T>(a, unit, KIND);
    if (a.active != nullptr && a.active[w.sys] == 0) live = false;  // system already converged
  }
  if (SPLIT != 1 && !live) return;  // the whole workgroup
  double v[NV];
  if (live) {
    const R4* pos = static_cast<const R4*>(a.pos);
    auto sums = [&](int64_t src0, int64_t src1) __attribute__((always_inline)) {
      const int64_t base = src0 + (SPLIT == 1 ? 0 : 64 * wave);
      if (KIND == 2 ? w.kind != 0 : KIND == 1)
        wide_sources<R, KIND != 0, BLK, T>(pos, a.F, a.T, w.tgt0, w.ntgt, base, src1, SPLIT, a.t0,
                                           a.rt0, a.r0, v);
      else
        wide_sources<R, KIND == 1, BLK, T>(pos, a.F, a.T, w.tgt0, w.ntgt, base, src1, SPLIT, a.t0,
                                           a.rt0, a.r0, v);
    };
    if constexpr (LONG) {
#pragma unroll 1
      for (int64_t s0 = w.src0; s0 < w.src1; s0 += kWideFp32Sources) {
        sums(s0, min(s0 + kWideFp32Sources, w.src1));
        wide_fold_to<NV>(v, s_red[wave], s0 > w.src0);
      }
    } else {
      sums(w.src0, w.src1);
      wide_fold_to<NV>(v, s_red[wave]);
    }
  }
  __syncthreads();
  if (!live) return;
  // value q of the unit: component q of its targets' U, then of their W
  const int q = SPLIT == 1 ? lane : (int)threadIdx.x;
  if (q < NV) {
    const double s = wide_value<SPLIT, NV>(s_red, wave, q);
    const int e = q < 3 * T ? q : q - 3 * T;
    if (e < 3 * w.ntgt) (q < 3 * T ? a.U : a.W)[3 * w.tgt0 + e] = s;
  }
}

// WideStep: the product between the two halves of Lanczos steps.  Without it a
// step of 2000 particles with torques took 31 us for the product, 4.8 for w . v
// and 7.0 for one workgroup that normalised; with it 31.8 + 4.7 us in two launches.
template <class R, int BLK, int T, int SPLIT>
__global__ __launch_bounds__(kPairThreads) void k_wide_step(WideArgs a, WideStep h) {
  using R4 = typename Rec<R>::T;
  constexpr bool kAngular = (BLK & (kWT | kWF)) != 0;
  constexpr int NV = (kAngular ? 6 : 3) * T;
  __shared__ double s_red[kWideWaves][NV];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // one read per workgroup, so that all its threads take the same branch
  __shared__ int s_stop;
  if (threadIdx.x == 0) s_stop = a.stop != nullptr ? *(volatile const int*)a.stop : 0;
  __syncthreads();
  if (s_stop != 0) return;
  const int unit = SPLIT == 1 ? (int)blockIdx.x * kWideWaves + wave : (int)blockIdx.x;
  const bool live = unit < a.nunits;
  if (SPLIT != 1 && !live) return;  // the whole workgroup
  // v_i = scale * F
  const double* F = h.v;
  double scale = 1.0, beta = 0.0;
  if (h.i > 0) {
    const int nb = (h.n + kPairThreads - 1) / kPairThreads;
    beta = sqrt(wave_sum(lane < nb ? h.partial_b[lane] : 0.0));
    if (beta < 1e-3 * h.sc->alpha[h.i - 1] / h.sc->normz) beta = 0.0;  // LanczosAlgorithm.cu:140-142
    F = beta > 0.0 ? h.w : h.e1;
    scale = beta > 0.0 ? 1.0 / beta : 1.0;
    if (unit == 0 && threadIdx.x == 0) h.sc->beta[h.i - 1] = beta;
  }
  const int64_t n3 = kAngular ? h.n / 2 : h.n;
  WideUnit w{0, 0, 0, 1, 1, 0};
  if (live) {
    w = wide_unit<T>(a, unit, 1);
    double v[NV];
    wide_sources<R, true, BLK, T>(static_cast<const R4*>(a.pos), F, F + n3, w.tgt0, w.ntgt,
                                  w.src0 + (SPLIT == 1 ? 0 : 64 * wave), w.src1, SPLIT,
                                  scale * a.t0, scale * a.rt0, scale * a.r0, v);
    wide_fold_to<NV>(v, s_red[wave]);
  }
  __syncthreads();
  const int q = SPLIT == 1 ? lane : (int)threadIdx.x;
  if (!live || q >= 64) return;  // whole waves
  double part = 0.0;
  const int e = q < 3 * T ? q : q - 3 * T;
  if (q < NV && e < 3 * w.ntgt) {
    const int64_t k = 3 * w.tgt0 + e + (q < 3 * T ? 0 : n3);
    const double vk = scale * F[k];
    double wk = wide_value<SPLIT, NV>(s_red, wave, q);
    if (h.i > 0) {
      h.v[k] = vk;
      wk -= beta * h.vp[k];
    }
    h.w_out[k] = wk;
    part = wk * vk;
  }
  part = wave_sum(part);
  if (lane == 0) h.partial_a[unit] = part;
}

template <class R, int BLK>
static void launch_wide_step_split(const WideArgs& a, const WideStep& h, hipStream_t s) {
  if (a.split == 4)
    hipLaunchKernelGGL((k_wide_step<R, BLK, kWideTargets, 4>), dim3((unsigned)a.nunits),
                       dim3(kPairThreads), 0, s, a, h);
  else
    hipLaunchKernelGGL((k_wide_step<R, BLK, kWideTargets, 1>),
                       dim3((unsigned)((a.nunits + kWideWaves - 1) / kWideWaves)),
                       dim3(kPairThreads), 0, s, a, h);
  LM_HIP(hipGetLastError());
}

void launch_wide_step(const WideArgs& a, const WideStep& h, hipStream_t s) {
  constexpr int kAll = kUF | kUT | kWT | kWF;
  if (a.nunits <= 0) return;
  if (a.kind != 1 || a.active || h.n <= 0 || h.n > kWideStepMax || h.w == h.w_out ||
      (a.blocks != kUF && a.blocks != kAll) || (a.split != 1 && a.split != 4))
    throw Error("[libmobility_amd] this product cannot take a Lanczos step");
  if (a.fp32)
    a.blocks == kUF ? launch_wide_step_split<float, kUF>(a, h, s)
                    : launch_wide_step_split<float, kAll>(a, h, s);
  else
    a.blocks == kUF ? launch_wide_step_split<double, kUF>(a, h, s)
                    : launch_wide_step_split<double, kAll>(a, h, s);
}

template <class R, int KIND, int BLK>
static void launch_wide_split(const WideArgs& a, hipStream_t s) {
  const dim3 grid((unsigned)(a.split == 4 ? a.nunits : (a.nunits + kWideWaves - 1) / kWideWaves));
  const dim3 block(kPairThreads);
  if (a.long_sums != 0 && a.split == 1 && std::is_same<R, float>::value)
    hipLaunchKernelGGL((k_pair_wide<R, KIND, BLK, kWideTargets, 1, std::is_same<R, float>::value>),
                       grid, block, 0, s, a);
  else if (a.long_sums != 0)
    throw Error("[libmobility_amd] long sums of the wide kernel: FP32, one wave per unit");
  else if (a.split == 4)
    hipLaunchKernelGGL((k_pair_wide<R, KIND, BLK, kWideTargets, 4, false>), grid, block, 0, s, a);
  else if (a.split == 1)
    hipLaunchKernelGGL((k_pair_wide<R, KIND, BLK, kWideTargets, 1, false>), grid, block, 0, s, a);
  else
    throw Error("[libmobility_amd] wide launch takes 1 or 4 waves per unit");
  LM_HIP(hipGetLastError());
}

template <class R, int KIND>
static void launch_wide_blk(const WideArgs& a, hipStream_t s) {
  switch (a.blocks) {
    case kUF: launch_wide_split<R, KIND, kUF>(a, s); break;
    case kUF | kWF: launch_wide_split<R, KIND, kUF | kWF>(a, s); break;
    case kUT | kWT: launch_wide_split<R, KIND, kUT | kWT>(a, s); break;
    case kUF | kUT | kWT | kWF: launch_wide_split<R, KIND, kUF | kUT | kWT | kWF>(a, s); break;
    default: throw Error("[libmobility_amd] unsupported block combination");
  }
}

template <class R>
static void launch_wide_r(const WideArgs& a, hipStream_t s) {
  switch (a.kind) {
    case 0: launch_wide_blk<R, 0>(a, s); break;
    case 1: launch_wide_blk<R, 1>(a, s); break;
    case 2: launch_wide_blk<R, 2>(a, s); break;
    default: throw Error("[libmobility_amd] invalid kernel kind");
  }
}

void launch_pair_wide(const WideArgs& a, hipStream_t s) {
  if (a.nunits <= 0) return;
  if (a.fp32)
    launch_wide_r<float>(a, s);
  else
    launch_wide_r<double>(a, s);
}

}  // namespace lm
