// One item of the symmetric evaluation in symmetric units (pair_math.hpp),
// shared by the kernels of sym_kernels.hip and nbody_kernels.hip.
//
// A workgroup of NW waves holds a tile of 64 NW TPL targets in its lanes (TPL
// per lane) and streams the partner tiles through LDS in sub-tiles of 64 NW
// sources: NW blocks of 64, each stored twice, so that step k reads lane + k
// without index arithmetic.  At step k, lane l meets source (l + k) mod 64 of
// its wave's block and holds that source's running sums, which move one lane
// down before each step (DPP wave_rol:1).  With NW > 1 wave w takes block
// (w + p) mod NW in phase p, so in every phase the waves hold sums of different
// blocks and add them to one FP64 row per source, a barrier between phases (a
// row per wave and block would take NW times the LDS).  With NW = 1 there are
// no barriers and the sums go straight to the offset's slab.
#pragma once
#include <type_traits>

#include "kernels.hpp"
#include "pair_device.hpp"
#include "pair_math.hpp"

namespace lm {

// Lane l receives lane (l + 1) mod 64.
template <class R>
__device__ inline R lane_rol1(R v);
template <>
__device__ inline float lane_rol1<float>(float v) {
  return __builtin_bit_cast(
      float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x134, 0xf, 0xf, true));
}
template <>
__device__ inline double lane_rol1<double>(double v) {
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo =
      (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, 0x134, 0xf, 0xf, true);
  const uint32_t hi =
      (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), 0x134, 0xf, 0xf, true);
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}
template <class R>
__device__ inline void rol1(Vec3<R>& v) {
  v.x = lane_rol1(v.x);
  v.y = lane_rol1(v.y);
  v.z = lane_rol1(v.z);
}

template <int BLK>
struct SymForm {
  static constexpr bool needF = (BLK & (kUF | kWF)) != 0;
  static constexpr bool needT = (BLK & (kUT | kWT)) != 0;
  static constexpr bool angular = (BLK & (kWT | kWF)) != 0;
  static constexpr int comp = angular ? 6 : 3;
  static constexpr int nrec = 1 + (needF ? 1 : 0) + (needT ? 1 : 0);
  static constexpr int recF = 1;
  static constexpr int recT = needF ? 2 : 1;
};

// Staged sources, three components per record (position, force, torque).
// FP32: 16-byte slots.  FP64: one array per component, because a lane stride
// of 32 bytes has bank conflicts.
template <class R, int NREC, int NW>
struct SymStage;
template <int NREC, int NW>
struct SymStage<float, NREC, NW> {
  float4 rec[NREC][128 * NW];
  __device__ void put(int slot, int r, const Vec3<float>& v) {
    const float4 q = {v.x, v.y, v.z, 0.f};
    rec[r][slot] = q;
    rec[r][slot + 64] = q;
  }
  __device__ Vec3<float> get(int r, int i) const {
    const float4 q = rec[r][i];
    return {q.x, q.y, q.z};
  }
};
template <int NREC, int NW>
struct SymStage<double, NREC, NW> {
  double c[3 * NREC][128 * NW];
  __device__ void put(int slot, int r, const Vec3<double>& v) {
    c[3 * r][slot] = c[3 * r][slot + 64] = v.x;
    c[3 * r + 1][slot] = c[3 * r + 1][slot + 64] = v.y;
    c[3 * r + 2][slot] = c[3 * r + 2][slot + 64] = v.z;
  }
  __device__ Vec3<double> get(int r, int i) const {
    return {c[3 * r][i], c[3 * r + 1][i], c[3 * r + 2][i]};
  }
};

// LDS of one item: the staged sources and, with NW > 1, the sources' sums.
template <class R, int BLK, int NW>
struct SymLds {
  SymStage<R, SymForm<BLK>::nrec, NW> st;
  double red[NW > 1 ? SymForm<BLK>::comp * 64 * NW : 1];
};

// A particle's position, force and torque in symmetric units (a.ta = 1/a; the
// wall's damping folded into the last two).
template <class R, bool WALL, int BLK>
struct SymParticle {
  Vec3<R> p, f, t;
  R b;
  __device__ void load(const SymArgs& a, int64_t i, bool ok) {
    using R4 = typename Rec<R>::T;
    const R4 q = ok ? static_cast<const R4*>(a.pos)[i] : far_record<R4>();
    p = {q.x, q.y, q.z};
    b = WALL ? q.w : R(1);
    f = t = {R(0), R(0), R(0)};
    if (SymForm<BLK>::needF && ok)
      f = {b * R(a.F[3 * i]), b * R(a.F[3 * i + 1]), b * R(a.F[3 * i + 2])};
    if (SymForm<BLK>::needT && ok) {
      const R s = b * R(a.r0 / a.rt0);
      t = {s * R(a.T[3 * i]), s * R(a.T[3 * i + 1]), s * R(a.T[3 * i + 2])};
    }
  }
};

template <class R>
__device__ inline void add3(Vec3<R>& d, const Vec3<R>& s) {
  d.x += s.x;
  d.y += s.y;
  d.z += s.z;
}
template <class R>
__device__ inline void add_to(Vec3<double>& d, Vec3<R>& s) {
  d.x += s.x;
  d.y += s.y;
  d.z += s.z;
  s = {R(0), R(0), R(0)};
}
__device__ inline void put3(double* o, double s, double x, double y, double z) {
  o[0] = s * x;
  o[1] = s * y;
  o[2] = s * z;
}

// The step loop of one wave: its lanes' targets against block `b0` (+ lane) of
// the staged sources; DIAG: all ordered pairs, the targets' sums only, which with
// the same b0 in all lanes may end after the block's `cnt` sources.
template <class R, bool WALL, int BLK, int TPL, int NW, bool DIAG>
__device__ inline void sym_steps(const SymStage<R, SymForm<BLK>::nrec, NW>& st, int b0,
                                 const SymParticle<R, WALL, BLK>* me, Vec3<R>* u, Vec3<R>* w,
                                 Vec3<R>& su, Vec3<R>& sw, int cnt = 64) {
  using Fm = SymForm<BLK>;
  const Vec3<R> zero = {R(0), R(0), R(0)};
  // FP32, several targets per lane: a step's terms of a source are added up before
  // they go to its running sum, which so has 64 terms as with one target.
  constexpr bool kOwn = std::is_same<R, float>::value && TPL > 1 && !DIAG;
  if constexpr (!WALL && BLK == kUF) {
    // the open translational block: overlap test over the step's pairs, and in
    // FP32 the fences of sym_item (nbody_kernels.hip)
    constexpr bool kFence = std::is_same<R, float>::value;
#pragma unroll 2
    for (int k = 0; k < cnt; ++k) {
      R dx[TPL], dy[TPL], dz[TPL], r2[TPL], ir[TPL];
      RpyCoef<R> cf[TPL];
      NearTest<R> near;
      const Vec3<R> pg = st.get(0, b0 + k), fg = st.get(1, b0 + k);
#pragma unroll
      for (int t = 0; t < TPL; ++t) {
        dx[t] = me[t].p.x - pg.x;
        dy[t] = me[t].p.y - pg.y;
        dz[t] = me[t].p.z - pg.z;
        r2[t] = dx[t] * dx[t] + dy[t] * dy[t] + dz[t] * dz[t];
        near.add(r2[t]);
      }
      if constexpr (kFence) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int t = 0; t < TPL; ++t) ir[t] = lm_rsqrt(r2[t]);
      if (!DIAG) rol1(su);
      if constexpr (kFence) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int t = 0; t < TPL; ++t) {
        cf[t] = RpyCoef<R>{};
        rpy_far_uf34<R>(ir[t], cf[t]);
      }
      if (__builtin_expect(near.hit(), 0)) {
        lm_rare_path();
#pragma unroll
        for (int t = 0; t < TPL; ++t) rpy_near_select_uf34<R>(r2[t], ir[t], cf[t]);
      }
      Vec3<R> cu = zero, cw = zero;
#pragma unroll
      for (int t = 0; t < TPL; ++t)
        open_unit<R, BLK, !DIAG>(dx[t], dy[t], dz[t], cf[t], fg, zero, me[t].f, zero, u[t], w[t],
                                 kOwn ? cu : su, kOwn ? cw : sw);
      if constexpr (kOwn) add3(su, cu);
    }
  } else {
#pragma unroll 1
    for (int k = 0; k < cnt; ++k) {
      const Vec3<R> pj = st.get(0, b0 + k);
      Vec3<R> fj = zero, tj = zero;
      if (Fm::needF) fj = st.get(Fm::recF, b0 + k);
      if (Fm::needT) tj = st.get(Fm::recT, b0 + k);
      if (!DIAG) {
        rol1(su);
        if (Fm::angular) rol1(sw);
      }
      Vec3<R> cu = zero, cw = zero;
#pragma unroll
      for (int t = 0; t < TPL; ++t) {
        PairGeo<R> g;
        pair_distances<R, WALL>(me[t].p.x, me[t].p.y, me[t].p.z, pj.x, pj.y, pj.z, g);
        pair_inverses<R, WALL>(g);
        pair_unit<R, WALL, BLK, !DIAG>(g, pj.z, fj, tj, me[t].f, me[t].t, u[t], w[t],
                                       kOwn ? cu : su, kOwn ? cw : sw);
      }
      if constexpr (kOwn) {
        add3(su, cu);
        if (Fm::angular) add3(sw, cw);
      }
    }
  }
}

// Targets of tile it.tile against the partner offsets [it.o0, it.o1), or (DIAG)
// against themselves (SHORT: source by source, all lanes at the same one, up to the
// last; a step of the others reads lane + k and takes whole blocks).
template <class R, bool WALL, int BLK, int TPL, int NW, bool DIAG, bool SHORT = false>
__device__ inline void sym_unit_item(const SymItem& it, const SymSys& S, const SymArgs& a,
                                     SymLds<R, BLK, NW>& lds) {
  using Fm = SymForm<BLK>;
  constexpr int kThr = 64 * NW;
  constexpr int kTile = kThr * TPL;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = NW == 1 ? 0 : __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t N = S.off + S.n;  // end of the system's particles
  const int64_t tgt0 = S.off + (int64_t)it.tile * kTile;
  const double us = 0.75 * a.t0, ws = a.rt0;  // units of U and W
  const Vec3<R> zero = {R(0), R(0), R(0)};

  SymParticle<R, WALL, BLK> me[TPL];
  Vec3<R> u[TPL], w[TPL];
  Vec3<double> u64[TPL], w64[TPL];
#pragma unroll
  for (int t = 0; t < TPL; ++t) {
    const int64_t i = tgt0 + tid + t * kThr;
    me[t].load(a, i, i < N);
    u[t] = w[t] = zero;
    u64[t] = w64[t] = {0.0, 0.0, 0.0};
  }
  const int o0 = DIAG ? 0 : it.o0, o1 = DIAG ? 1 : it.o1;
  for (int o = o0; o < o1; ++o) {
    if (!DIAG && 2 * o == S.ntiles && 2 * it.tile >= S.ntiles) continue;  // met from the other side
    int J = it.tile + o;
    if (J >= S.ntiles) J -= S.ntiles;
#pragma unroll 1
    for (int sub = 0; sub < TPL; ++sub) {
      const int64_t base = S.off + (int64_t)J * kTile + sub * kThr;
      if (base >= N) break;
      const int64_t j = base + tid;
      const bool ok = j < N;
      if (NW > 1) __syncthreads();  // the previous sub-tile is done with the LDS
      R bj;
      {
        SymParticle<R, WALL, BLK> src;
        src.load(a, j, ok);
        bj = src.b;
        const int slot = (tid >> 6) * 128 + lane;
        lds.st.put(slot, 0, src.p);
        if (Fm::needF) lds.st.put(slot, Fm::recF, src.f);
        if (Fm::needT) lds.st.put(slot, Fm::recT, src.t);
      }
      if (NW > 1)
        __syncthreads();
      else
        __builtin_amdgcn_wave_barrier();
      Vec3<R> su = zero, sw = zero;
#pragma unroll 1
      for (int p = 0; p < NW; ++p) {
        const int blk = NW == 1 ? 0 : (wave + p) & (NW - 1);
        su = sw = zero;
        // of a tile that the system does not fill: blocks without sources and waves
        // without targets give zeros (uniform per wave)
        if (NW == 1 || (base + 64 * blk < N && tgt0 + 64 * wave < N))
          sym_steps<R, WALL, BLK, TPL, NW, DIAG>(
              lds.st, blk * 128 + (SHORT ? 0 : lane), me, u, w, su, sw,
              SHORT ? (int)min((int64_t)64, N - base - 64 * blk) : 64);
        if constexpr (std::is_same<R, float>::value) {
          // FP32 sums over 64 sources at most
#pragma unroll
          for (int t = 0; t < TPL; ++t) {
            add_to(u64[t], u[t]);
            if (Fm::angular) add_to(w64[t], w[t]);
          }
        }
        if (!DIAG) {
          // lane l holds source l - 1 after 64 steps: one more move
          rol1(su);
          if (Fm::angular) rol1(sw);
          if (NW > 1) {
            const double v[6] = {(double)su.x, (double)su.y, (double)su.z,
                                 (double)sw.x, (double)sw.y, (double)sw.z};
            double* red = lds.red + blk * 64 + lane;
#pragma unroll
            for (int c = 0; c < Fm::comp; ++c)
              red[c * kThr] = p == 0 ? v[c] : red[c * kThr] + v[c];
            __syncthreads();
          }
        }
      }
      if (!DIAG && ok) {
        double v[6] = {(double)su.x, (double)su.y, (double)su.z,
                       (double)sw.x, (double)sw.y, (double)sw.z};
        if (NW > 1) {
#pragma unroll
          for (int c = 0; c < Fm::comp; ++c) v[c] = lds.red[c * kThr + tid];
        }
        const int64_t row = (int64_t)(o - a.obase) * a.n3 + 3 * j;
        put3(a.slab_s + row, us * (double)bj, v[0], v[1], v[2]);
        if (Fm::angular) put3(a.slab_sw + row, ws * (double)bj, v[3], v[4], v[5]);
      }
    }
  }
  if constexpr (std::is_same<R, double>::value) {
#pragma unroll
    for (int t = 0; t < TPL; ++t) {
      u64[t] = u[t];
      w64[t] = w[t];
    }
  }
#pragma unroll
  for (int t = 0; t < TPL; ++t) {
    const int64_t i = tgt0 + tid + t * kThr;
    if (i < N) {
      const int64_t row = (int64_t)it.chunk * a.n3 + 3 * i;
      const double b = (double)me[t].b;
      put3(a.slab_t + row, us * b, u64[t].x, u64[t].y, u64[t].z);
      if (Fm::angular) put3(a.slab_tw + row, ws * b, w64[t].x, w64[t].y, w64[t].z);
    }
  }
}

template <class R, bool WALL, int BLK, int TPL, int NW, bool SHORT = false>
__device__ inline void sym_unit(const SymItem& it, const SymSys& S, const SymArgs& a,
                                SymLds<R, BLK, NW>& lds) {
  if (it.o0 == 0)
    sym_unit_item<R, WALL, BLK, TPL, NW, true, SHORT>(it, S, a, lds);
  else
    sym_unit_item<R, WALL, BLK, TPL, NW, false>(it, S, a, lds);
}

}  // namespace lm
