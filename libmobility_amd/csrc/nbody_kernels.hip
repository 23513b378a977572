// gfx950 kernels of the O(N^2) mobility product and of setPositions.
//
// Pair kernel layout
//   * One workgroup = one PairItem: a tile of targets (256 x TPL, each lane
//     owns TPL targets held in registers) against one chunk of sources of the
//     same system.
//   * Sources stream through LDS in tiles of 256 records; every lane reads the
//     same source at the same time, so LDS reads are broadcasts.
//   * FP32 mode: pair terms and the per-tile sums are FP32, each tile's sum is
//     added into FP64 accumulators (error grows with the tile, not with N).
//   * Partial results of the chunks of one target go to separate slabs and
//     are summed by k_chunk_reduce in a fixed order (bitwise reproducible).
//   * Items are ordered target-tile-major, chunk-minor.  Workgroups are
//     dispatched round-robin over the 8 XCDs, so with 8 chunks every XCD
//     reads one chunk of the sources and its L2 holds only that chunk.
#include <type_traits>

#include "kernels.hpp"
#include "lanczos_head.hpp"
#include "lm_common.hpp"
#include "pair_device.hpp"
#include "pair_math.hpp"
#include "sym_item.hpp"

namespace lm {

// One item: targets [tgt0, tgt0 + ntgt) x sources [src0, src1) of one system.
template <class R, bool WALL, int BLK, int TPL>
__device__ inline void pair_item(const PairItem& it, const typename Rec<R>::T* __restrict__ pos,
                                 const double* __restrict__ F, const double* __restrict__ T,
                                 double* __restrict__ U, double* __restrict__ W, int64_t slab,
                                 double t0, double rt0, double r0, typename Rec<R>::T* s_pos,
                                 typename Rec<R>::T* s_f, typename Rec<R>::T* s_t) {
  using R4 = typename Rec<R>::T;
  constexpr bool kNeedF = (BLK & (kUF | kWF)) != 0;
  constexpr bool kNeedT = (BLK & (kUT | kWT)) != 0;
  constexpr bool kAngular = (BLK & (kWT | kWF)) != 0;
  // open translational block: coefficients times 4/3 (one operation less per
  // pair), undone once on the output
  constexpr bool kUF34 = !WALL && BLK == kUF;
  const int tid = threadIdx.x;

  R4 pi[TPL];
#pragma unroll
  for (int k = 0; k < TPL; ++k) {
    const int loc = tid + k * kPairThreads;
    pi[k] = (loc < it.ntgt) ? pos[it.tgt0 + loc] : far_record<R4>();
  }
  PairAcc<R> acc[TPL];
  PairAcc<double> acc64[TPL];
#pragma unroll
  for (int k = 0; k < TPL; ++k) {
    acc_zero(acc[k]);
    acc_zero(acc64[k]);
  }

  for (int64_t base = it.src0; base < it.src1; base += kPairThreads) {
    const int64_t j = base + tid;
    // sources of this tile (a chunk's last tile may be partial; its padding
    // slots hold far records and zero forces and are skipped)
    const int cnt = (int)min((int64_t)kPairThreads, it.src1 - base);
    __syncthreads();
    if (j < it.src1) {
      s_pos[tid] = pos[j];
      if constexpr (WALL) {
        // symmetric units (pair_math.hpp), the damping with the force
        const R bf = s_pos[tid].w, bt = bf * R(r0 / rt0);
        if (kNeedF) s_f[tid] = R4{bf * R(F[3 * j]), bf * R(F[3 * j + 1]), bf * R(F[3 * j + 2]), R(0)};
        if (kNeedT) s_t[tid] = R4{bt * R(T[3 * j]), bt * R(T[3 * j + 1]), bt * R(T[3 * j + 2]), R(0)};
      } else {
        if (kNeedF) s_f[tid] = R4{R(F[3 * j]), R(F[3 * j + 1]), R(F[3 * j + 2]), R(0)};
        if (kNeedT) s_t[tid] = R4{R(T[3 * j]), R(T[3 * j + 1]), R(T[3 * j + 2]), R(0)};
      }
    } else {
      s_pos[tid] = far_record<R4>();
      if (kNeedF) s_f[tid] = R4{R(0), R(0), R(0), R(0)};
      if (kNeedT) s_t[tid] = R4{R(0), R(0), R(0), R(0)};
    }
    __syncthreads();
    if constexpr (WALL) {
      auto source = [&](int s) __attribute__((always_inline)) {
        const R4 pj = s_pos[s];
        const Vec3<R> zero = {R(0), R(0), R(0)};
        Vec3<R> fj = zero, tj = zero, none = zero;
        if (kNeedF) fj = {s_f[s].x, s_f[s].y, s_f[s].z};
        if (kNeedT) tj = {s_t[s].x, s_t[s].y, s_t[s].z};
#pragma unroll
        for (int k = 0; k < TPL; ++k) {
          // U in acc.uf, W in acc.wf
          PairGeo<R> g;
          pair_distances<R, true>(pi[k].x, pi[k].y, pi[k].z, pj.x, pj.y, pj.z, g);
          pair_inverses<R, true>(g);
          pair_unit<R, true, BLK, false>(g, pj.z, fj, tj, zero, zero, acc[k].uf, acc[k].wf, none,
                                         none);
        }
      };
      if constexpr (std::is_same<R, float>::value && kNeedF && kNeedT) {
        // Sums of forces' and torques' blocks in one accumulator have twice the terms:
        // they go to FP64 every 64 sources.  With 256 their error was 1.2 times that of
        // an accumulator per block, with 64 it is 0.8 times (17000 to 40000 particles);
        // 40000 particles 4.98 -> 4.94 ms.
        for (int s0 = 0; s0 < cnt; s0 += 64) {
          const int s1 = min(s0 + 64, cnt);
          for (int s = s0; s < s1; ++s) source(s);
#pragma unroll
          for (int k = 0; k < TPL; ++k) {
            add_to(acc64[k].uf, acc[k].uf);
            add_to(acc64[k].wf, acc[k].wf);
          }
        }
      } else {
        for (int s = 0; s < cnt; ++s) source(s);
      }
    } else {
      // Open boundaries: a group of SG sources x TPL targets (4 pairs) gets
      // its far-field coefficients first and one overlap test for the whole
      // group; the overlap values (rare: overlapping spheres and the self
      // pair) are patched in by selects inside that single branch.
      constexpr int SG = TPL >= 4 ? 1 : 4 / TPL;
      const int lim = (cnt + SG - 1) / SG * SG;  // padding slots up to a whole group
      for (int s = 0; s < lim; s += SG) {
        R dx[SG][TPL], dy[SG][TPL], dz[SG][TPL], r2[SG][TPL], ir[SG][TPL];
        RpyCoef<R> cf[SG][TPL];
        R4 fj[SG], tj[SG];
        NearTestCmp<R> near;
#pragma unroll
        for (int g = 0; g < SG; ++g) {
          const R4 pj = s_pos[s + g];
          if (kNeedF) fj[g] = s_f[s + g]; else fj[g] = R4{R(0), R(0), R(0), R(0)};
          if (kNeedT) tj[g] = s_t[s + g]; else tj[g] = R4{R(0), R(0), R(0), R(0)};
#pragma unroll
          for (int k = 0; k < TPL; ++k) {
            dx[g][k] = pi[k].x - pj.x;
            dy[g][k] = pi[k].y - pj.y;
            dz[g][k] = pi[k].z - pj.z;
            r2[g][k] = dx[g][k] * dx[g][k] + dy[g][k] * dy[g][k] + dz[g][k] * dz[g][k];
            ir[g][k] = lm_rsqrt(r2[g][k]);
            cf[g][k] = RpyCoef<R>{};
            if constexpr (kUF34)
              rpy_far_uf34<R>(ir[g][k], cf[g][k]);
            else
              rpy_far<R, BLK>(ir[g][k], cf[g][k]);
            near.add(r2[g][k]);
          }
        }
        if (__builtin_expect(near.hit(), 0)) {
          // opaque statement: keep this a branch (not speculated onto every group)
          __asm__ __volatile__("");
#pragma unroll
          for (int g = 0; g < SG; ++g)
#pragma unroll
            for (int k = 0; k < TPL; ++k) {
              if constexpr (kUF34)
                rpy_near_select_uf34<R>(r2[g][k], ir[g][k], cf[g][k]);
              else
                rpy_near_select<R, BLK>(r2[g][k], ir[g][k], cf[g][k]);
            }
        }
#pragma unroll
        for (int g = 0; g < SG; ++g)
#pragma unroll
          for (int k = 0; k < TPL; ++k)
            open_accumulate<R, BLK>(dx[g][k], dy[g][k], dz[g][k], fj[g].x, fj[g].y, fj[g].z,
                                    tj[g].x, tj[g].y, tj[g].z, cf[g][k], acc[k]);
      }
    }
    if constexpr (std::is_same<R, float>::value && !(WALL && kNeedF && kNeedT)) {
#pragma unroll
      for (int k = 0; k < TPL; ++k) {
        acc64[k].uf.x += acc[k].uf.x; acc64[k].uf.y += acc[k].uf.y; acc64[k].uf.z += acc[k].uf.z;
        acc64[k].ut.x += acc[k].ut.x; acc64[k].ut.y += acc[k].ut.y; acc64[k].ut.z += acc[k].ut.z;
        acc64[k].wt.x += acc[k].wt.x; acc64[k].wt.y += acc[k].wt.y; acc64[k].wt.z += acc[k].wt.z;
        acc64[k].wf.x += acc[k].wf.x; acc64[k].wf.y += acc[k].wf.y; acc64[k].wf.z += acc[k].wf.z;
        acc_zero(acc[k]);
      }
    }
  }
  if constexpr (std::is_same<R, double>::value) {
#pragma unroll
    for (int k = 0; k < TPL; ++k) acc64[k] = acc[k];
  }
  double* Uo = U + (int64_t)it.chunk * slab;
  double* Wo = kAngular ? W + (int64_t)it.chunk * slab : nullptr;
  const double tuf = kUF34 ? 0.75 * t0 : t0;
#pragma unroll
  for (int k = 0; k < TPL; ++k) {
    const int loc = tid + k * kPairThreads;
    if (loc < it.ntgt) {
      const int64_t i = it.tgt0 + loc;
      const PairAcc<double>& a = acc64[k];
      if constexpr (WALL) {
        const double b = (double)pi[k].w;
        put3(Uo + 3 * i, 0.75 * t0 * b, a.uf.x, a.uf.y, a.uf.z);
        if (kAngular) put3(Wo + 3 * i, rt0 * b, a.wf.x, a.wf.y, a.wf.z);
        continue;
      }
      Uo[3 * i + 0] = tuf * a.uf.x + rt0 * a.ut.x;
      Uo[3 * i + 1] = tuf * a.uf.y + rt0 * a.ut.y;
      Uo[3 * i + 2] = tuf * a.uf.z + rt0 * a.ut.z;
      if (kAngular) {
        Wo[3 * i + 0] = r0 * a.wt.x + rt0 * a.wf.x;
        Wo[3 * i + 1] = r0 * a.wt.y + rt0 * a.wf.y;
        Wo[3 * i + 2] = r0 * a.wt.z + rt0 * a.wf.z;
      }
    }
  }
}

// KIND: 0 open, 1 wall, 2 per item.  PERSIST: the grid loops over items,
// fetching the next one from `counter` (work queue; every workgroup exits
// once the counter passes nitems).
template <class R, int KIND, int BLK, int TPL, bool PERSIST>
__global__ __launch_bounds__(kPairThreads) void k_pair(
    const PairItem* __restrict__ items, int nitems, unsigned int* __restrict__ counter,
    const typename Rec<R>::T* __restrict__ pos, const double* __restrict__ F,
    const double* __restrict__ T, double* __restrict__ U, double* __restrict__ W, int64_t slab,
    const int* __restrict__ active, const int* stop, double t0, double rt0, double r0) {
  using R4 = typename Rec<R>::T;
  constexpr bool kNeedF = (BLK & (kUF | kWF)) != 0;
  constexpr bool kNeedT = (BLK & (kUT | kWT)) != 0;
  __shared__ R4 s_pos[kPairThreads];
  __shared__ R4 s_f[kNeedF ? kPairThreads : 1];
  __shared__ R4 s_t[kNeedT ? kPairThreads : 1];
  __shared__ int s_item;
  int item = blockIdx.x;
  if (!PERSIST && stop != nullptr) {
    // one read per workgroup, so that all its threads take the same branch
    // (the flag may change while the workgroup starts)
    __shared__ int s_stop;
    if (threadIdx.x == 0) s_stop = *(volatile const int*)stop;
    __syncthreads();
    if (s_stop != 0) return;
  }
  while (true) {
    if (PERSIST) {
      __syncthreads();  // previous item finished with s_item and the tiles
      if (threadIdx.x == 0) s_item = (int)atomicAdd(counter, 1u);
      __syncthreads();
      item = s_item;
    }
    if (item >= nitems) break;
    const PairItem it = items[item];
    if (active != nullptr && active[it.sys] == 0) {  // system already converged
      if (!PERSIST) break;
      continue;
    }
    if (KIND == 2) {
      if (it.wall)
        pair_item<R, true, BLK, TPL>(it, pos, F, T, U, W, slab, t0, rt0, r0, s_pos, s_f, s_t);
      else
        pair_item<R, false, BLK, TPL>(it, pos, F, T, U, W, slab, t0, rt0, r0, s_pos, s_f, s_t);
    } else {
      pair_item<R, KIND == 1, BLK, TPL>(it, pos, F, T, U, W, slab, t0, rt0, r0, s_pos, s_f, s_t);
    }
    if (!PERSIST) break;
  }
}

// ---- symmetric evaluation (open boundaries, translational block) --------------
// Open RPY depends on r only and is even in d, so M_ji F_i uses the pair's
// coefficients unchanged: fuf F_i + guf (d.F_i) d.  An item holds the 256*TPL
// targets of tile I in the lanes and streams each partner tile J through LDS
// in sub-tiles of 256 sources (four blocks of 64, each stored twice).  Lane l
// meets source (l + k) mod 64 of a block at step k (address l + k) and carries
// that source's running sum, which moves one lane down after every step
// (DPP wave_rol:1), so after 64 steps every source has met all targets of the
// wave and its sum sits back in lane (source index).  The four waves' sums are
// added in a fixed order and written once per source to the offset's slab.

template <class R, int TPL, bool FENCE>
__device__ inline void sym_item(const SymItem& it, const SymArgs& a, typename Rec<R>::T* s_pos,
                                typename Rec<R>::T* s_f, R* s_red) {
  using R4 = typename Rec<R>::T;
  constexpr int kTile = kPairThreads * TPL;
  // FP32: one step per overlap test, and the step's reciprocal square roots and
  // lane moves between two scheduling fences, next to each other.  Two waves of
  // a SIMD issue simple FP32 together (1.5-1.7 instructions per CU cycle, other
  // VALU instructions 0.9, v_rsq_f32 0.47), but every v_rsq or DPP move that
  // stands alone in such a stream costs 3-5 issue slots, and a run of them
  // hardly more than one.  FP64 has no such pairing and keeps groups of 4 pairs.
  //   131072 particles, 4 targets per lane 5.94 -> 5.55 ms, 2 per lane 6.25 ->
  //   5.75 ms; 32768, 2 per lane 449 -> 414 us; 20011, 1 per lane 195 -> 186 us.
  // Not where a CU has one or two workgroups (FENCE false, kFenceItems): little issues
  // beside a wave then, and it waits for the latencies of one step instead of four.
  constexpr bool kFence = FENCE && std::is_same<R, float>::value;
  constexpr int SG = kFence || TPL >= 4 ? 1 : 4 / TPL;  // steps per overlap test
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const R4* __restrict__ pos = static_cast<const R4*>(a.pos);
  const double* __restrict__ F = a.F;
  const SymSys S = a.sys[it.sys];
  const int64_t N = S.off + S.n;  // end of the system's particles
  const int64_t tgt0 = S.off + (int64_t)it.tile * kTile;
  const double t0s = 0.75 * a.t0;  // the coefficients carry 4/3 (rpy_far_uf34)

  R4 pi[TPL];
  R fix[TPL], fiy[TPL], fiz[TPL];
#pragma unroll
  for (int t = 0; t < TPL; ++t) {
    const int64_t i = tgt0 + tid + t * kPairThreads;
    if (i < N) {
      pi[t] = pos[i];
      fix[t] = R(F[3 * i]);
      fiy[t] = R(F[3 * i + 1]);
      fiz[t] = R(F[3 * i + 2]);
    } else {
      pi[t] = far_record<R4>();
      fix[t] = fiy[t] = fiz[t] = R(0);
    }
  }
  Vec3<R> acc[TPL];
  Vec3<double> acc64[TPL];
#pragma unroll
  for (int t = 0; t < TPL; ++t) {
    acc[t] = {R(0), R(0), R(0)};
    acc64[t] = {0.0, 0.0, 0.0};
  }
  auto flush = [&]() {
#pragma unroll
    for (int t = 0; t < TPL; ++t) {
      acc64[t].x += acc[t].x;
      acc64[t].y += acc[t].y;
      acc64[t].z += acc[t].z;
      acc[t] = {R(0), R(0), R(0)};
    }
  };

  for (int o = it.o0; o < it.o1; ++o) {
    if (2 * o == S.ntiles && 2 * it.tile >= S.ntiles) continue;  // met from the other side
    int J = it.tile + o;
    if (J >= S.ntiles) J -= S.ntiles;
    double* __restrict__ So = a.slab_s + (int64_t)(o - a.obase) * a.n3;
#pragma unroll 1
    for (int sub = 0; sub < TPL; ++sub) {
      const int64_t base = S.off + (int64_t)J * kTile + sub * kPairThreads;
      if (base >= N) break;
      const int64_t j = base + tid;
      __syncthreads();  // the previous sub-tile is done with s_pos, s_f and s_red
      R4 pj = far_record<R4>();
      R4 fj = R4{R(0), R(0), R(0), R(0)};
      if (j < N) {
        pj = pos[j];
        fj = R4{R(F[3 * j]), R(F[3 * j + 1]), R(F[3 * j + 2]), R(0)};
      }
      s_pos[wave * 128 + lane] = pj;
      s_pos[wave * 128 + 64 + lane] = pj;
      s_f[wave * 128 + lane] = fj;
      s_f[wave * 128 + 64 + lane] = fj;
      __syncthreads();
#pragma unroll 1  // one copy of the step loop (the blocks differ only in address)
      for (int blk = 0; blk < 4; ++blk) {
        const R4* sp = s_pos + blk * 128 + lane;
        const R4* sf = s_f + blk * 128 + lane;
        Vec3<R> sa = {R(0), R(0), R(0)};
#pragma unroll 2
        for (int k = 0; k < 64; k += SG) {
          R dx[SG][TPL], dy[SG][TPL], dz[SG][TPL], r2[SG][TPL], ir[SG][TPL];
          RpyCoef<R> cf[SG][TPL];
          R4 pg[SG], fg[SG];
          NearTest<R> near;
#pragma unroll
          for (int g = 0; g < SG; ++g) {
            pg[g] = sp[k + g];
            fg[g] = sf[k + g];
#pragma unroll
            for (int t = 0; t < TPL; ++t) {
              dx[g][t] = pi[t].x - pg[g].x;
              dy[g][t] = pi[t].y - pg[g].y;
              dz[g][t] = pi[t].z - pg[g].z;
              r2[g][t] = dx[g][t] * dx[g][t] + dy[g][t] * dy[g][t] + dz[g][t] * dz[g][t];
              near.add(r2[g][t]);
            }
          }
          if constexpr (kFence) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int g = 0; g < SG; ++g)
#pragma unroll
            for (int t = 0; t < TPL; ++t) ir[g][t] = lm_rsqrt(r2[g][t]);
          if constexpr (kFence) {
            // the running sum moves here, beside the reciprocal square roots
            sa.x = lane_rol1(sa.x);
            sa.y = lane_rol1(sa.y);
            sa.z = lane_rol1(sa.z);
            __builtin_amdgcn_sched_barrier(0);
          }
#pragma unroll
          for (int g = 0; g < SG; ++g)
#pragma unroll
            for (int t = 0; t < TPL; ++t) {
              cf[g][t] = RpyCoef<R>{};
              rpy_far_uf34<R>(ir[g][t], cf[g][t]);
            }
          if (__builtin_expect(near.hit(), 0)) {
            __asm__ __volatile__("");  // keep this a branch
#pragma unroll
            for (int g = 0; g < SG; ++g)
#pragma unroll
              for (int t = 0; t < TPL; ++t) rpy_near_select_uf34<R>(r2[g][t], ir[g][t], cf[g][t]);
          }
#pragma unroll
          for (int g = 0; g < SG; ++g) {
            // the running sum moves first and the step's terms accumulate
            // into it: one move per component and step, no separate add
            if constexpr (!kFence) {
              sa.x = lane_rol1(sa.x);
              sa.y = lane_rol1(sa.y);
              sa.z = lane_rol1(sa.z);
            }
#pragma unroll
            for (int t = 0; t < TPL; ++t) {
              const R fuf = cf[g][t].fuf, guf = cf[g][t].guf;
              const R st = guf * (dx[g][t] * fg[g].x + dy[g][t] * fg[g].y + dz[g][t] * fg[g].z);
              acc[t].x = lm_fma(st, dx[g][t], lm_fma(fuf, fg[g].x, acc[t].x));
              acc[t].y = lm_fma(st, dy[g][t], lm_fma(fuf, fg[g].y, acc[t].y));
              acc[t].z = lm_fma(st, dz[g][t], lm_fma(fuf, fg[g].z, acc[t].z));
              const R ss = guf * (dx[g][t] * fix[t] + dy[g][t] * fiy[t] + dz[g][t] * fiz[t]);
              sa.x = lm_fma(ss, dx[g][t], lm_fma(fuf, fix[t], sa.x));
              sa.y = lm_fma(ss, dy[g][t], lm_fma(fuf, fiy[t], sa.y));
              sa.z = lm_fma(ss, dz[g][t], lm_fma(fuf, fiz[t], sa.z));
            }
          }
        }
        // after 64 steps lane l holds source l - 1: one more move puts source l in lane l
        s_red[(wave * 3 + 0) * kPairThreads + blk * 64 + lane] = lane_rol1(sa.x);
        s_red[(wave * 3 + 1) * kPairThreads + blk * 64 + lane] = lane_rol1(sa.y);
        s_red[(wave * 3 + 2) * kPairThreads + blk * 64 + lane] = lane_rol1(sa.z);
        // With 2 or 4 targets per lane a source's FP32 sum has 128 or 256 terms;
        // the targets' sums then go to FP64 every 64 sources instead of every
        // 256, so that the error is no larger than with 1 per lane.
        if (std::is_same<R, float>::value && TPL > 1 && a.fine != 0) flush();
      }
      __syncthreads();
      if (j < N) {
        double vx = 0.0, vy = 0.0, vz = 0.0;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          vx += (double)s_red[(w * 3 + 0) * kPairThreads + tid];
          vy += (double)s_red[(w * 3 + 1) * kPairThreads + tid];
          vz += (double)s_red[(w * 3 + 2) * kPairThreads + tid];
        }
        So[3 * j + 0] = t0s * vx;
        So[3 * j + 1] = t0s * vy;
        So[3 * j + 2] = t0s * vz;
      }
      if (std::is_same<R, float>::value && (TPL == 1 || a.fine == 0)) flush();
    }
  }
  if constexpr (std::is_same<R, double>::value) {
#pragma unroll
    for (int t = 0; t < TPL; ++t) acc64[t] = acc[t];
  }
  double* __restrict__ Uo = a.slab_t + (int64_t)it.chunk * a.n3;
#pragma unroll
  for (int t = 0; t < TPL; ++t) {
    const int64_t i = tgt0 + tid + t * kPairThreads;
    if (i < N) {
      Uo[3 * i + 0] = t0s * acc64[t].x;
      Uo[3 * i + 1] = t0s * acc64[t].y;
      Uo[3 * i + 2] = t0s * acc64[t].z;
    }
  }
}

// Open boundaries with angular blocks, in the order of operations that plain
// Lanczos products keep: the same ring, lanes and rotation as sym_item, with
// open_both giving both directions of every block from one set of
// coefficients.  The source sums carry U (units of t0) and, with angular
// blocks, W (units of r0).
template <class R, int BLK, int TPL>
__device__ inline void sym_item_gen(const SymItem& it, const SymArgs& a,
                                    typename Rec<R>::T* s_pos, typename Rec<R>::T* s_f,
                                    typename Rec<R>::T* s_t, R* s_red) {
  using R4 = typename Rec<R>::T;
  constexpr int kTile = kPairThreads * TPL;
  constexpr bool kNeedF = (BLK & (kUF | kWF)) != 0;
  constexpr bool kNeedT = (BLK & (kUT | kWT)) != 0;
  constexpr bool kAngular = (BLK & (kWT | kWF)) != 0;
  constexpr int kComp = kAngular ? 6 : 3;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const R4* __restrict__ pos = static_cast<const R4*>(a.pos);
  const SymSys S = a.sys[it.sys];
  const int64_t N = S.off + S.n;  // end of the system's particles
  const int64_t tgt0 = S.off + (int64_t)it.tile * kTile;
  const R kut = R(a.rt0 / a.t0), kwf = R(a.rt0 / a.r0);
  const Vec3<R> zero = {R(0), R(0), R(0)};

  R4 pi[TPL];
  Vec3<R> fi[TPL], ti[TPL];
#pragma unroll
  for (int t = 0; t < TPL; ++t) {
    const int64_t i = tgt0 + tid + t * kPairThreads;
    const bool ok = i < N;
    pi[t] = ok ? pos[i] : far_record<R4>();
    fi[t] = (kNeedF && ok) ? Vec3<R>{R(a.F[3 * i]), R(a.F[3 * i + 1]), R(a.F[3 * i + 2])} : zero;
    ti[t] = (kNeedT && ok) ? Vec3<R>{R(a.T[3 * i]), R(a.T[3 * i + 1]), R(a.T[3 * i + 2])} : zero;
  }
  PairAcc<R> acc[TPL];
  PairAcc<double> acc64[TPL];
#pragma unroll
  for (int t = 0; t < TPL; ++t) {
    acc_zero(acc[t]);
    acc_zero(acc64[t]);
  }

  for (int o = it.o0; o < it.o1; ++o) {
    if (2 * o == S.ntiles && 2 * it.tile >= S.ntiles) continue;  // met from the other side
    int J = it.tile + o;
    if (J >= S.ntiles) J -= S.ntiles;
    for (int sub = 0; sub < TPL; ++sub) {
      const int64_t base = S.off + (int64_t)J * kTile + sub * kPairThreads;
      if (base >= N) break;
      const int64_t j = base + tid;
      __syncthreads();  // the previous sub-tile is done with the staged sources and s_red
      const bool ok = j < N;
      const R4 pj = ok ? pos[j] : far_record<R4>();
      s_pos[wave * 128 + lane] = pj;
      s_pos[wave * 128 + 64 + lane] = pj;
      if (kNeedF) {
        const R4 fj = ok ? R4{R(a.F[3 * j]), R(a.F[3 * j + 1]), R(a.F[3 * j + 2]), R(0)}
                         : R4{R(0), R(0), R(0), R(0)};
        s_f[wave * 128 + lane] = fj;
        s_f[wave * 128 + 64 + lane] = fj;
      }
      if (kNeedT) {
        const R4 tj = ok ? R4{R(a.T[3 * j]), R(a.T[3 * j + 1]), R(a.T[3 * j + 2]), R(0)}
                         : R4{R(0), R(0), R(0), R(0)};
        s_t[wave * 128 + lane] = tj;
        s_t[wave * 128 + 64 + lane] = tj;
      }
      __syncthreads();
      for (int blk = 0; blk < 4; ++blk) {
        const int b0 = blk * 128 + lane;
        Vec3<R> su = zero, sw = zero;
        for (int k = 0; k < 64; ++k) {
          const R4 pj4 = s_pos[b0 + k];
          Vec3<R> fj = zero, tj = zero;
          if (kNeedF) {
            const R4 v = s_f[b0 + k];
            fj = {v.x, v.y, v.z};
          }
          if (kNeedT) {
            const R4 v = s_t[b0 + k];
            tj = {v.x, v.y, v.z};
          }
          Vec3<R> cu = zero, cw = zero;
#pragma unroll
          for (int t = 0; t < TPL; ++t)
            open_pair_both<R, BLK>(pi[t].x - pj4.x, pi[t].y - pj4.y, pi[t].z - pj4.z, fj, tj,
                                   fi[t], ti[t], kut, kwf, acc[t], cu, cw);
          su.x = lane_rol1(su.x) + cu.x;
          su.y = lane_rol1(su.y) + cu.y;
          su.z = lane_rol1(su.z) + cu.z;
          if (kAngular) {
            sw.x = lane_rol1(sw.x) + cw.x;
            sw.y = lane_rol1(sw.y) + cw.y;
            sw.z = lane_rol1(sw.z) + cw.z;
          }
        }
        // lane l holds source l - 1 after 64 steps: one more move
        R* red = s_red + wave * kComp * kPairThreads + blk * 64 + lane;
        red[0 * kPairThreads] = lane_rol1(su.x);
        red[1 * kPairThreads] = lane_rol1(su.y);
        red[2 * kPairThreads] = lane_rol1(su.z);
        if (kAngular) {
          red[3 * kPairThreads] = lane_rol1(sw.x);
          red[4 * kPairThreads] = lane_rol1(sw.y);
          red[5 * kPairThreads] = lane_rol1(sw.z);
        }
      }
      __syncthreads();
      if (ok) {
        double v[kComp];
#pragma unroll
        for (int q = 0; q < kComp; ++q) v[q] = 0.0;
#pragma unroll
        for (int w = 0; w < 4; ++w)
#pragma unroll
          for (int q = 0; q < kComp; ++q) v[q] += (double)s_red[(w * kComp + q) * kPairThreads + tid];
        double* So = a.slab_s + (int64_t)(o - a.obase) * a.n3;
        So[3 * j + 0] = a.t0 * v[0];
        So[3 * j + 1] = a.t0 * v[1];
        So[3 * j + 2] = a.t0 * v[2];
        if (kAngular) {
          double* Sw = a.slab_sw + (int64_t)(o - a.obase) * a.n3;
          Sw[3 * j + 0] = a.r0 * v[kComp - 3];
          Sw[3 * j + 1] = a.r0 * v[kComp - 2];
          Sw[3 * j + 2] = a.r0 * v[kComp - 1];
        }
      }
      if constexpr (std::is_same<R, float>::value) {
#pragma unroll
        for (int t = 0; t < TPL; ++t) {
          acc64[t].uf.x += acc[t].uf.x; acc64[t].uf.y += acc[t].uf.y; acc64[t].uf.z += acc[t].uf.z;
          acc64[t].ut.x += acc[t].ut.x; acc64[t].ut.y += acc[t].ut.y; acc64[t].ut.z += acc[t].ut.z;
          acc64[t].wt.x += acc[t].wt.x; acc64[t].wt.y += acc[t].wt.y; acc64[t].wt.z += acc[t].wt.z;
          acc64[t].wf.x += acc[t].wf.x; acc64[t].wf.y += acc[t].wf.y; acc64[t].wf.z += acc[t].wf.z;
          acc_zero(acc[t]);
        }
      }
    }
  }
  if constexpr (std::is_same<R, double>::value) {
#pragma unroll
    for (int t = 0; t < TPL; ++t) acc64[t] = acc[t];
  }
  double* Uo = a.slab_t + (int64_t)it.chunk * a.n3;
  double* Wo = kAngular ? a.slab_tw + (int64_t)it.chunk * a.n3 : nullptr;
#pragma unroll
  for (int t = 0; t < TPL; ++t) {
    const int64_t i = tgt0 + tid + t * kPairThreads;
    if (i < N) {
      const PairAcc<double>& c = acc64[t];
      Uo[3 * i + 0] = a.t0 * c.uf.x + a.rt0 * c.ut.x;
      Uo[3 * i + 1] = a.t0 * c.uf.y + a.rt0 * c.ut.y;
      Uo[3 * i + 2] = a.t0 * c.uf.z + a.rt0 * c.ut.z;
      if (kAngular) {
        Wo[3 * i + 0] = a.r0 * c.wt.x + a.rt0 * c.wf.x;
        Wo[3 * i + 1] = a.r0 * c.wt.y + a.rt0 * c.wf.y;
        Wo[3 * i + 2] = a.r0 * c.wt.z + a.rt0 * c.wf.z;
      }
    }
  }
}

// LDS of one item of the order-keeping evaluation.
template <class R, int BLK>
struct SymKeepLds {
  using R4 = typename Rec<R>::T;
  R4 pos[4 * 128];
  R4 f[(BLK & (kUF | kWF)) ? 4 * 128 : 1];
  R4 t[(BLK & (kUT | kWT)) ? 4 * 128 : 1];
  R red[4 * ((BLK & (kWT | kWF)) ? 6 : 3) * kPairThreads];
};

// One item per workgroup: a diagonal tile (all ordered pairs of tile I, the
// self pairs included) or a range of partner offsets.  KIND: 0 open, 2 per
// system (mixed ensembles; their wall systems run in symmetric units).
template <class R, int KIND, int BLK, int TPL, bool FENCE>
__global__ __launch_bounds__(kPairThreads) void k_pair_sym(SymArgs a) {
  using R4 = typename Rec<R>::T;
  using Keep = SymKeepLds<R, BLK>;
  using Unit = SymLds<R, BLK, 4>;
  constexpr size_t kLds =
      KIND == 2 && sizeof(Unit) > sizeof(Keep) ? sizeof(Unit) : sizeof(Keep);
  __shared__ __align__(16) unsigned char s_mem[kLds];
  Keep& lds = *reinterpret_cast<Keep*>(s_mem);
  if (a.stop != nullptr) {
    // one read per workgroup, so that all its threads take the same branch
    __shared__ int s_stop;
    if (threadIdx.x == 0) s_stop = *(volatile const int*)a.stop;
    __syncthreads();
    if (s_stop != 0) return;
  }
  const SymItem it = a.items[blockIdx.x];
  if (a.active != nullptr && a.active[it.sys] == 0) return;  // system already converged
  const SymSys S = a.sys[it.sys];
  if constexpr (KIND == 2) {
    if (S.wall != 0) {
      sym_unit<R, true, BLK, TPL, 4, true>(it, S, a, *reinterpret_cast<Unit*>(s_mem));
      return;
    }
  }
  if (it.o0 == 0) {
    constexpr int kTile = kPairThreads * TPL;
    PairItem p;
    p.tgt0 = S.off + (int64_t)it.tile * kTile;
    const int64_t left = S.off + S.n - p.tgt0;
    p.ntgt = (int32_t)(left < kTile ? left : kTile);
    p.src0 = p.tgt0;
    p.src1 = p.tgt0 + p.ntgt;
    p.chunk = it.chunk;
    p.wall = 0;
    p.sys = it.sys;
    pair_item<R, false, BLK, TPL>(p, static_cast<const R4*>(a.pos), a.F, a.T, a.slab_t, a.slab_tw,
                                  a.n3, a.t0, a.rt0, a.r0, lds.pos, lds.f, lds.t);
    return;
  }
  if constexpr (BLK == kUF)
    sym_item<R, TPL, FENCE>(it, a, lds.pos, lds.f, lds.red);
  else
    sym_item_gen<R, BLK, TPL>(it, a, lds.pos, lds.f, lds.t, lds.red);
}

// Products of plain Lanczos over small open systems: the launch first finishes
// the step before (lanczos_head.hpp), in every workgroup, and reads the forces
// from LDS.  1024 particles, translational, FP64, a step and a product: 17.8 us
// in two launches (this and the chunk sums), 20.4 as product and one-workgroup
// step.  All four blocks:
template <class R>
__global__ __launch_bounds__(kPairThreads) void k_pair_head(
    const PairItem* __restrict__ items, const typename Rec<R>::T* __restrict__ pos,
    double* __restrict__ U, double* __restrict__ W, int64_t slab, const int* stop, double t0,
    double rt0, double r0, LanczosHead h) {
  using R4 = typename Rec<R>::T;
  constexpr int BLK = kUF | kUT | kWT | kWF;
  __shared__ R4 s_pos[kPairThreads];
  __shared__ R4 s_f[kPairThreads];
  __shared__ R4 s_t[kPairThreads];
  __shared__ double s_v[kLanczosHeadMax];
  __shared__ double sh[2][16];
  __shared__ int s_stop;
  // one read per workgroup, so that all its threads take the same branch
  if (threadIdx.x == 0) s_stop = stop != nullptr ? *(volatile const int*)stop : 0;
  const PairItem it = items[blockIdx.x];
  lanczos_head(h, s_v, sh, blockIdx.x == 0);
  if (s_stop != 0) return;  // read after the barriers of the head
  pair_item<R, false, BLK, 1>(it, pos, s_v, s_v + slab, U, W, slab, t0, rt0, r0, s_pos, s_f, s_t);
}

// The same for the translational block alone, where one item's 256 targets x 64
// sources leave a wave 64 pairs in series on a quarter of the chip's CUs: a
// workgroup takes 64 targets, its waves the coefficients of 16 sources each, and
// three of them then add one component each, source by source in k_pair's order
// (the same bits).  1024 particles, FP64: 13.8 -> 10.8 us.
template <class R>
__global__ __launch_bounds__(kPairThreads) void k_pair_head_uf(
    const PairItem* __restrict__ items, const typename Rec<R>::T* __restrict__ pos,
    double* __restrict__ U, int64_t slab, const int* stop, double t0, LanczosHead h) {
  using R4 = typename Rec<R>::T;
  __shared__ R s_p[3][64], s_f[3][64];
  __shared__ R s_fuf[64][64], s_s[64][64];  // per source and target
  __shared__ double s_v[kLanczosHeadMax];
  __shared__ double sh[2][16];
  __shared__ int s_stop;
  if (threadIdx.x == 0) s_stop = stop != nullptr ? *(volatile const int*)stop : 0;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const PairItem it = items[blockIdx.x >> 2];
  const int loc = 64 * (int)(blockIdx.x & 3) + lane;
  const R4 pi = loc < it.ntgt ? pos[it.tgt0 + loc] : far_record<R4>();
  // sources of the first 64, in flight while the step ends
  R4 pj = it.src0 + lane < it.src1 ? pos[it.src0 + lane] : far_record<R4>();
  lanczos_head(h, s_v, sh, blockIdx.x == 0);
  if (s_stop != 0 || 64 * (int)(blockIdx.x & 3) >= it.ntgt) return;  // the whole workgroup
  const R xi = wave == 0 ? pi.x : (wave == 1 ? pi.y : pi.z);
  R acc = R(0);
  double acc64 = 0.0;
  for (int64_t base = it.src0; base < it.src1; base += 64) {
    const int64_t j = base + lane;
    const int cnt = (int)min((int64_t)64, it.src1 - base);
    if (base > it.src0) {
      __syncthreads();  // the block before is done with the LDS
      if (j < it.src1) pj = pos[j];
    }
    if (wave == 0) {
      s_p[0][lane] = pj.x;
      s_p[1][lane] = pj.y;
      s_p[2][lane] = pj.z;
#pragma unroll
      for (int c = 0; c < 3; ++c) s_f[c][lane] = j < it.src1 ? R(s_v[3 * j + c]) : R(0);
    }
    __syncthreads();
#pragma unroll
    for (int s = 16 * wave; s < 16 * wave + 16; s += 4) {
      R dx[4], dy[4], dz[4], r2[4], ir[4];
      RpyCoef<R> cf[4];
      NearTestCmp<R> near;
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int q = s + g < cnt ? s + g : cnt - 1;
        dx[g] = pi.x - s_p[0][q];
        dy[g] = pi.y - s_p[1][q];
        dz[g] = pi.z - s_p[2][q];
        r2[g] = dx[g] * dx[g] + dy[g] * dy[g] + dz[g] * dz[g];
        ir[g] = lm_rsqrt(r2[g]);
        cf[g] = RpyCoef<R>{};
        rpy_far_uf34<R>(ir[g], cf[g]);
        near.add(r2[g]);
      }
      if (__builtin_expect(near.hit(), 0)) {
        lm_rare_path();
#pragma unroll
        for (int g = 0; g < 4; ++g) rpy_near_select_uf34<R>(r2[g], ir[g], cf[g]);
      }
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int q = s + g < cnt ? s + g : cnt - 1;
        s_fuf[s + g][lane] = cf[g].fuf;
        s_s[s + g][lane] =
            cf[g].guf * (dx[g] * s_f[0][q] + dy[g] * s_f[1][q] + dz[g] * s_f[2][q]);
      }
    }
    __syncthreads();
    if (wave < 3) {
#pragma unroll 8
      for (int s = 0; s < cnt; ++s)
        acc = lm_fma(s_s[s][lane], xi - s_p[wave][s], lm_fma(s_fuf[s][lane], s_f[wave][s], acc));
      if constexpr (std::is_same<R, float>::value) {
        // FP64 sums over tiles of kPairThreads sources, as in pair_item
        if ((base - it.src0) % kPairThreads == kPairThreads - 64 || base + 64 >= it.src1) {
          acc64 += acc;
          acc = R(0);
        }
      }
    }
  }
  if constexpr (std::is_same<R, double>::value) acc64 = acc;
  if (wave < 3 && loc < it.ntgt)
    U[(int64_t)it.chunk * slab + 3 * (it.tgt0 + loc) + wave] = 0.75 * t0 * acc64;
}

// ---- several force vectors per pass (translational block) ----------------------
// Same tiling as pair_item; each pair's geometry and coefficients are computed
// once and applied to the NR force vectors staged side by side in LDS.
template <class R, bool WALL, int NR, int TPL>
__device__ inline void pair_item_multi(const PairItem& it, const typename Rec<R>::T* __restrict__ pos,
                                       const double* __restrict__ F, double* __restrict__ U,
                                       int64_t n3, int nch, double t0, typename Rec<R>::T* s_pos,
                                       typename Rec<R>::T* s_f) {
  using R4 = typename Rec<R>::T;
  const int tid = threadIdx.x;
  R4 pi[TPL];
#pragma unroll
  for (int k = 0; k < TPL; ++k) {
    const int loc = tid + k * kPairThreads;
    pi[k] = (loc < it.ntgt) ? pos[it.tgt0 + loc] : far_record<R4>();
  }
  Vec3<R> acc[TPL][NR];
  Vec3<double> acc64[TPL][NR];
#pragma unroll
  for (int k = 0; k < TPL; ++k)
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      acc[k][r] = {R(0), R(0), R(0)};
      acc64[k][r] = {0.0, 0.0, 0.0};
    }
  for (int64_t base = it.src0; base < it.src1; base += kPairThreads) {
    const int64_t j = base + tid;
    __syncthreads();
    if (j < it.src1) {
      const R4 pj = pos[j];
      s_pos[tid] = pj;
      const R b = WALL ? pj.w : R(1);  // the wall's damping goes with the force
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        const double* f = F + (int64_t)r * n3 + 3 * j;
        s_f[r * kPairThreads + tid] = R4{b * R(f[0]), b * R(f[1]), b * R(f[2]), R(0)};
      }
    } else {
      s_pos[tid] = far_record<R4>();
#pragma unroll
      for (int r = 0; r < NR; ++r) s_f[r * kPairThreads + tid] = R4{R(0), R(0), R(0), R(0)};
    }
    __syncthreads();
    for (int s = 0; s < kPairThreads; ++s) {
      const R4 pj = s_pos[s];
      R4 fj[NR];
#pragma unroll
      for (int r = 0; r < NR; ++r) fj[r] = s_f[r * kPairThreads + s];
#pragma unroll
      for (int k = 0; k < TPL; ++k) {
        UFCoef<R> c;
        if constexpr (WALL) {
          uf_coef_wall<R>(pi[k].x, pi[k].y, pi[k].z, pj.x, pj.y, pj.z, c);
#pragma unroll
          for (int r = 0; r < NR; ++r) uf_apply_wall<R>(c, fj[r].x, fj[r].y, fj[r].z, acc[k][r]);
        } else {
          c.dx = pi[k].x - pj.x;
          c.dy = pi[k].y - pj.y;
          c.dz = pi[k].z - pj.z;
          const R r2 = c.dx * c.dx + c.dy * c.dy + c.dz * c.dz;
          const R ir = lm_rsqrt(r2);
          RpyCoef<R> cf{};
          rpy_far_uf34<R>(ir, cf);  // times 4/3, undone on the output
          if (__builtin_expect(r2 < R(4), 0)) {
            lm_rare_path();
            rpy_near_select_uf34<R>(r2, ir, cf);
          }
          c.a0 = cf.fuf;
          c.cd = cf.guf;
#pragma unroll
          for (int r = 0; r < NR; ++r) uf_apply_open<R>(c, fj[r].x, fj[r].y, fj[r].z, acc[k][r]);
        }
      }
    }
    if constexpr (std::is_same<R, float>::value) {
#pragma unroll
      for (int k = 0; k < TPL; ++k)
#pragma unroll
        for (int r = 0; r < NR; ++r) {
          acc64[k][r].x += acc[k][r].x;
          acc64[k][r].y += acc[k][r].y;
          acc64[k][r].z += acc[k][r].z;
          acc[k][r] = {R(0), R(0), R(0)};
        }
    }
  }
  if constexpr (std::is_same<R, double>::value) {
#pragma unroll
    for (int k = 0; k < TPL; ++k)
#pragma unroll
      for (int r = 0; r < NR; ++r) acc64[k][r] = acc[k][r];
  }
#pragma unroll
  for (int k = 0; k < TPL; ++k) {
    const int loc = tid + k * kPairThreads;
    if (loc < it.ntgt) {
      const int64_t i = it.tgt0 + loc;
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        double* o = U + ((int64_t)r * nch + it.chunk) * n3;
        const double tuf = 0.75 * t0 * (WALL ? (double)pi[k].w : 1.0);
        o[3 * i + 0] = tuf * acc64[k][r].x;
        o[3 * i + 1] = tuf * acc64[k][r].y;
        o[3 * i + 2] = tuf * acc64[k][r].z;
      }
    }
  }
}

template <class R, int KIND, int NR>
__global__ __launch_bounds__(kPairThreads) void k_pair_multi(
    const PairItem* __restrict__ items, const typename Rec<R>::T* __restrict__ pos,
    const double* __restrict__ F, double* __restrict__ U, int64_t n3, int nch, double t0) {
  using R4 = typename Rec<R>::T;
  constexpr int TPL = multi_tpl(NR);
  __shared__ R4 s_pos[kPairThreads];
  __shared__ R4 s_f[NR * kPairThreads];
  const PairItem it = items[blockIdx.x];
  if constexpr (KIND == 0) {
    pair_item_multi<R, false, NR, TPL>(it, pos, F, U, n3, nch, t0, s_pos, s_f);
  } else if constexpr (KIND == 1) {
    pair_item_multi<R, true, NR, TPL>(it, pos, F, U, n3, nch, t0, s_pos, s_f);
  } else {
    if (it.wall)
      pair_item_multi<R, true, NR, TPL>(it, pos, F, U, n3, nch, t0, s_pos, s_f);
    else
      pair_item_multi<R, false, NR, TPL>(it, pos, F, U, n3, nch, t0, s_pos, s_f);
  }
}

template <class R, int KIND>
static void launch_pair_multi_k(const PairMultiArgs& a, hipStream_t s) {
  using R4 = typename Rec<R>::T;
  const R4* pos = static_cast<const R4*>(a.pos);
  if (a.nrhs == 4)
    hipLaunchKernelGGL((k_pair_multi<R, KIND, 4>), dim3(a.nitems), dim3(kPairThreads), 0, s,
                       a.items, pos, a.F, a.U, a.n3, a.nch, a.t0);
  else if (a.nrhs == 2)
    hipLaunchKernelGGL((k_pair_multi<R, KIND, 2>), dim3(a.nitems), dim3(kPairThreads), 0, s,
                       a.items, pos, a.F, a.U, a.n3, a.nch, a.t0);
  else
    throw Error("[libmobility_amd] multi-vector launch handles 2 or 4 vectors");
  LM_HIP(hipGetLastError());
}

void launch_pair_multi(const PairMultiArgs& a, hipStream_t s) {
  if (a.nitems <= 0) return;
  if (a.fp32) {
    if (a.kind == 0) launch_pair_multi_k<float, 0>(a, s);
    else if (a.kind == 1) launch_pair_multi_k<float, 1>(a, s);
    else launch_pair_multi_k<float, 2>(a, s);
  } else {
    if (a.kind == 0) launch_pair_multi_k<double, 0>(a, s);
    else if (a.kind == 1) launch_pair_multi_k<double, 1>(a, s);
    else launch_pair_multi_k<double, 2>(a, s);
  }
}

template <class R, int KIND, int BLK, int TPL>
static void launch_pair_t(const PairArgs& a, hipStream_t s) {
  using R4 = typename Rec<R>::T;
  if (a.persistent) {
    if (!a.counter) throw Error("[libmobility_amd] persistent launch without a work counter");
    launch_zero_u32(a.counter, 1, s);
    hipLaunchKernelGGL((k_pair<R, KIND, BLK, TPL, true>), dim3(a.grid), dim3(kPairThreads), 0, s,
                       a.items, a.nitems, a.counter, static_cast<const R4*>(a.pos), a.F, a.T, a.U,
                       a.W, a.slab, a.active, a.stop, a.t0, a.rt0, a.r0);
  } else {
    hipLaunchKernelGGL((k_pair<R, KIND, BLK, TPL, false>), dim3(a.nitems), dim3(kPairThreads), 0,
                       s, a.items, a.nitems, a.counter, static_cast<const R4*>(a.pos), a.F, a.T,
                       a.U, a.W, a.slab, a.active, a.stop, a.t0, a.rt0, a.r0);
  }
  LM_HIP(hipGetLastError());
}

template <class R, int KIND, int BLK>
static void launch_pair_tpl(const PairArgs& a, hipStream_t s) {
  switch (a.tpl) {
    case 1: launch_pair_t<R, KIND, BLK, 1>(a, s); break;
    case 2: launch_pair_t<R, KIND, BLK, 2>(a, s); break;
    case 4:
      if constexpr (KIND == 0 && BLK == kUF) {
        launch_pair_t<R, KIND, BLK, 4>(a, s);
        break;
      }
      [[fallthrough]];
    default: throw Error("[libmobility_amd] unsupported targets-per-lane for this kernel");
  }
}

template <class R, int KIND>
static void launch_pair_blk(const PairArgs& a, hipStream_t s) {
  switch (a.blocks) {
    case kUF: launch_pair_tpl<R, KIND, kUF>(a, s); break;
    case kUF | kWF: launch_pair_tpl<R, KIND, kUF | kWF>(a, s); break;
    case kUT | kWT: launch_pair_tpl<R, KIND, kUT | kWT>(a, s); break;
    case kUF | kUT | kWT | kWF: launch_pair_tpl<R, KIND, kUF | kUT | kWT | kWF>(a, s); break;
    default: throw Error("[libmobility_amd] unsupported block combination");
  }
}

template <class R>
static void launch_pair_kind(const PairArgs& a, hipStream_t s) {
  switch (a.wall) {
    case 0: launch_pair_blk<R, 0>(a, s); break;
    case 1: launch_pair_blk<R, 1>(a, s); break;
    case 2: launch_pair_blk<R, 2>(a, s); break;
    default: throw Error("[libmobility_amd] invalid kernel kind");
  }
}

template <class R>
static void launch_pair_head(const PairArgs& a, hipStream_t s) {
  const auto* pos = static_cast<const typename Rec<R>::T*>(a.pos);
  if (a.blocks == kUF)
    hipLaunchKernelGGL(k_pair_head_uf<R>, dim3(4 * a.nitems), dim3(kPairThreads), 0, s, a.items,
                       pos, a.U, a.slab, a.stop, a.t0, a.head);
  else
    hipLaunchKernelGGL((k_pair_head<R>), dim3(a.nitems), dim3(kPairThreads), 0, s, a.items, pos, a.U,
                       a.W, a.slab, a.stop, a.t0, a.rt0, a.r0, a.head);
  LM_HIP(hipGetLastError());
}

void launch_pair(const PairArgs& a, hipStream_t s) {
  if (a.nitems <= 0) return;
  if (a.head.n > 0) {
    constexpr int kAll = kUF | kUT | kWT | kWF;
    if (a.wall != 0 || a.persistent || a.tpl != 1 || a.active || a.slab <= 0 ||
        a.head.n > kLanczosHeadMax || (a.blocks != kUF && a.blocks != kAll) ||
        a.head.n != a.slab * (a.blocks == kAll ? 2 : 1))
      throw Error("[libmobility_amd] this product cannot finish a Lanczos step");
    if (a.fp32)
      launch_pair_head<float>(a, s);
    else
      launch_pair_head<double>(a, s);
    return;
  }
  if (a.fp32)
    launch_pair_kind<float>(a, s);
  else
    launch_pair_kind<double>(a, s);
}

// Items up to which the open translational kernel runs without fences, one target
// per lane: at most two workgroups per CU.  Ensembles of open systems, FP32, product
// in us with / without: 204 items 54.6 / 45.5, 280 items 57.9 / 47.2, 400 items 61.5 /
// 60.1, 640 and 768 items equal, 1280 items 90.4 / 94.1, 3200 items 151 / 160.
constexpr int kFenceItems = 512;

template <class R, int KIND, int BLK>
static void launch_pair_sym_tpl(const SymArgs& a, hipStream_t s) {
  const dim3 grid((unsigned)a.nitems), block(kPairThreads);
  constexpr bool fence = std::is_same<R, float>::value && BLK == kUF;
  switch (a.tpl) {
    case 1:
      if (fence && a.nitems > kFenceItems)
        hipLaunchKernelGGL((k_pair_sym<R, KIND, BLK, 1, fence>), grid, block, 0, s, a);
      else
        hipLaunchKernelGGL((k_pair_sym<R, KIND, BLK, 1, false>), grid, block, 0, s, a);
      break;
    case 2: hipLaunchKernelGGL((k_pair_sym<R, KIND, BLK, 2, fence>), grid, block, 0, s, a); break;
    case 4:
      if constexpr (KIND == 0 && BLK == kUF) {
        hipLaunchKernelGGL((k_pair_sym<R, KIND, BLK, 4, fence>), grid, block, 0, s, a);
        break;
      }
      [[fallthrough]];
    default: throw Error("[libmobility_amd] unsupported targets-per-lane for the symmetric kernel");
  }
  LM_HIP(hipGetLastError());
}

// Lanczos products have forces, or forces and torques.
template <class R, int KIND>
static void launch_pair_sym_blk(const SymArgs& a, hipStream_t s) {
  switch (a.blocks) {
    case kUF: launch_pair_sym_tpl<R, KIND, kUF>(a, s); break;
    case kUF | kUT | kWT | kWF: launch_pair_sym_tpl<R, KIND, kUF | kUT | kWT | kWF>(a, s); break;
    default: throw Error("[libmobility_amd] unsupported block combination");
  }
}

template <class R>
static void launch_pair_sym_r(const SymArgs& a, hipStream_t s) {
  switch (a.wall) {
    case 0: launch_pair_sym_blk<R, 0>(a, s); break;
    case 2: launch_pair_sym_blk<R, 2>(a, s); break;
    default: throw Error("[libmobility_amd] invalid kernel kind");
  }
}

void launch_pair_sym(const SymArgs& a, hipStream_t s) {
  if (a.nitems <= 0) return;
  if (a.waves != 4) throw Error("[libmobility_amd] unsupported shape of the symmetric kernel");
  if (a.fp32)
    launch_pair_sym_r<float>(a, s);
  else
    launch_pair_sym_r<double>(a, s);
}

// s + p[0] + p[n] + ... + p[(count - 1) n], added in this order; kSlabBatch
// loads are in flight at once (one at a time, a short sum is a chain of memory
// latencies).
constexpr int kSlabBatch = 16;
__device__ inline double add_slabs(double s, const double* __restrict__ p, int count, int64_t n) {
  int c = 0;
  for (; c + kSlabBatch <= count; c += kSlabBatch) {
    double q[kSlabBatch];
#pragma unroll
    for (int k = 0; k < kSlabBatch; ++k) q[k] = p[(int64_t)(c + k) * n];
#pragma unroll
    for (int k = 0; k < kSlabBatch; ++k) s += q[k];
  }
  double q[kSlabBatch];
#pragma unroll
  for (int k = 0; k < kSlabBatch; ++k) q[k] = c + k < count ? p[(int64_t)(c + k) * n] : 0.0;
#pragma unroll
  for (int k = 0; k < kSlabBatch; ++k)
    if (c + k < count) s += q[k];
  return s;
}

// Three workgroups per row block (at most 256 particles of one system), one
// thread per entry.  Bound by HBM for large systems (607 MB at
// 131072 particles and 193 slabs: 116 -> 100 us, 6.0 TB/s) and by latency for
// small ones (20011 particles, 79 slabs: 23.7 -> 8.4 us; 10007, 41 slabs: 6.7
// -> 3.9 us, against one workgroup per row block and one load at a time).
__global__ __launch_bounds__(kPairThreads) void k_sym_reduce(SymReduceArgs r) {
  const SymRows rb = r.rows[blockIdx.x / 3];
  if (r.active != nullptr && r.active[rb.sys] == 0) return;
  const int64_t e = 3 * rb.p0 + (int64_t)(blockIdx.x % 3) * kPairThreads + threadIdx.x;
  if (e >= 3 * (rb.p0 + rb.np)) return;
  const SymSys S = r.sys[rb.sys];
  const int tile = (int)((e / 3 - S.off) / r.tile);
  const int hi = min(r.o1, S.hmax + 1);  // this system's offsets in the pass: [o0, hi)
  const int width = hi - r.o0;
  // target slabs of this system in the pass
  const int nchp =
      width <= 0 ? 0 : (S.per > 0 ? (width + S.per - 1) / S.per : min(r.nch, width));
  // an even tile count meets offset ntiles/2 only from tiles I < ntiles/2, so
  // that slab (the ring's last) holds no rows of tiles J < ntiles/2
  const bool drop = S.ntiles % 2 == 0 && 2 * tile < S.ntiles && hi - 1 == S.ntiles / 2;
  const int64_t n = r.n3;
  double s = r.accumulate ? r.out[e] : 0.0;
  s = add_slabs(s, r.slab_t + e, nchp, n);
  if (r.diag) s += r.slab_t[(int64_t)r.nch * n + e];
  if (width > 0) s = add_slabs(s, r.slab_s + e, drop ? width - 1 : width, n);
  r.out[e] = s;
}

void launch_sym_reduce(const SymReduceArgs& r, hipStream_t s) {
  if (r.nrows <= 0) return;
  hipLaunchKernelGGL(k_sym_reduce, dim3((unsigned)(3 * r.nrows)), dim3(kPairThreads), 0, s, r);
  LM_HIP(hipGetLastError());
}

// out[r] = sum over the chunks c of part[r][c], for the vectors r = blockIdx.y
// of n entries each.  Bound by latency up to some 10^5 entries: 16 loads in
// flight instead of one (4 vectors of 24576 entries, 32 chunks: four launches of
// 9.2 us -> one of 6 us).
__global__ __launch_bounds__(kPairThreads) void k_chunk_reduce(const double* __restrict__ part,
                                                              int nch, int64_t n,
                                                              double* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * kPairThreads + threadIdx.x;
  if (i >= n) return;
  const int64_t r = blockIdx.y;
  out[r * n + i] = add_slabs(0.0, part + r * nch * n + i, nch, n);
}

void launch_chunk_reduce(const double* part, int nch, int64_t n, double* out, hipStream_t s,
                         int nvec) {
  if (n <= 0 || nvec <= 0) return;
  const dim3 grid((unsigned)((n + kPairThreads - 1) / kPairThreads), (unsigned)nvec);
  hipLaunchKernelGGL(k_chunk_reduce, grid, dim3(kPairThreads), 0, s, part, nch, n, out);
  LM_HIP(hipGetLastError());
}

// One workgroup per particle block; blocks of converged systems return at once.
__global__ __launch_bounds__(256) void k_seg_chunk_reduce(const double* __restrict__ part,
                                                          int nch, int64_t n,
                                                          double* __restrict__ out,
                                                          const SegBlock* __restrict__ blocks,
                                                          const int* __restrict__ active) {
  const SegBlock b = blocks[blockIdx.x];
  if (active[b.sys] == 0) return;
  for (int64_t i = 3 * b.p0 + threadIdx.x; i < 3 * b.p1; i += blockDim.x) {
    double s = 0.0;
    for (int c = 0; c < nch; ++c) s += part[(int64_t)c * n + i];
    out[i] = s;
  }
}

void launch_seg_chunk_reduce(const double* part, int nch, int64_t n, double* out,
                             const SegBlock* blocks, int nblocks, const int* active,
                             hipStream_t s) {
  if (n <= 0 || nblocks <= 0) return;
  hipLaunchKernelGGL(k_seg_chunk_reduce, dim3((unsigned)nblocks), dim3(256), 0, s, part, nch, n,
                     out, blocks, active);
  LM_HIP(hipGetLastError());
}

// ---- setPositions -----------------------------------------------------------

// Corners of a box grown by this thread's particles, reduced over the NT
// threads: lo and hi of component c end in sh[c][0] and sh[3 + c][0].
template <int NT>
struct BoxSum {
  double mn[3] = {1e300, 1e300, 1e300}, mx[3] = {-1e300, -1e300, -1e300};
  __device__ void add(double x, double y, double z) {
    mn[0] = fmin(mn[0], x);
    mx[0] = fmax(mx[0], x);
    mn[1] = fmin(mn[1], y);
    mx[1] = fmax(mx[1], y);
    mn[2] = fmin(mn[2], z);
    mx[2] = fmax(mx[2], z);
  }
  __device__ void reduce(double (*sh)[NT / 64]) {
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    for (int c = 0; c < 3; ++c) {
      for (int o = 32; o > 0; o >>= 1) {
        mn[c] = fmin(mn[c], __shfl_xor(mn[c], o));
        mx[c] = fmax(mx[c], __shfl_xor(mx[c], o));
      }
      if (lane == 0) {
        sh[c][wid] = mn[c];
        sh[3 + c][wid] = mx[c];
      }
    }
    __syncthreads();
    if (threadIdx.x < 6) {
      const int c = threadIdx.x;
      double v = sh[c][0];
      for (int w = 1; w < NT / 64; ++w) v = (c < 3) ? fmin(v, sh[c][w]) : fmax(v, sh[c][w]);
      sh[c][0] = v;
    }
    __syncthreads();
  }
};

// One workgroup per system; bound by the latency of its loads: 4 particles per
// thread in flight, and 1024 threads where a system has more than 4096
// particles.  With 256 threads and one particle in flight 2999 particles took
// 4.9 us, 65536 74, 131072 142; now 3.9, 22, 39.  host (may be null): a copy of
// bbox in mapped host memory, where reading it takes no transfer of its own.
// own (may be null): a copy of the positions, so that a wait for the boxes is
// also one for the last read of the caller's array.
template <int NT>
__global__ __launch_bounds__(NT) void k_system_bbox(const double* __restrict__ pos,
                                                   const int64_t* __restrict__ off,
                                                   double wall_shift_in,
                                                   const int* __restrict__ kinds, int wall,
                                                   double* __restrict__ bbox, double* host,
                                                   double* __restrict__ own) {
  __shared__ double sh[6][NT / 64];
  const int s = blockIdx.x;
  const int64_t b = off[s], e = off[s + 1];
  const double wall_shift = (kinds ? kinds[s] : wall) ? wall_shift_in : 0.0;
  BoxSum<NT> box;
  constexpr int kQ = 4;
  for (int64_t i0 = b + threadIdx.x; i0 < e; i0 += kQ * NT) {
    double p[kQ][3];
#pragma unroll
    for (int q = 0; q < kQ; ++q) {
      const int64_t i = i0 + q * NT < e ? i0 + q * NT : i0;  // again: no other box
#pragma unroll
      for (int c = 0; c < 3; ++c) p[q][c] = pos[3 * i + c];
    }
#pragma unroll
    for (int q = 0; q < kQ; ++q) box.add(p[q][0], p[q][1], p[q][2] - wall_shift);
    if (own != nullptr)
#pragma unroll
      for (int q = 0; q < kQ; ++q)
#pragma unroll
        for (int c = 0; c < 3; ++c)
          if (i0 + q * NT < e) own[3 * (i0 + q * NT) + c] = p[q][c];
  }
  box.reduce(sh);
  if (threadIdx.x < 6) {
    bbox[6 * s + threadIdx.x] = sh[threadIdx.x][0];
    if (host != nullptr) host[6 * s + threadIdx.x] = sh[threadIdx.x][0];
  }
}

void launch_system_bbox(const double* pos, const int64_t* sys_off, int nsys, int64_t largest,
                        double wall_shift, const int* kinds, int wall, double* bbox, hipStream_t s,
                        double* host, double* own) {
  if (nsys <= 0) return;
  if (largest > 4096)
    hipLaunchKernelGGL(k_system_bbox<1024>, dim3(nsys), dim3(1024), 0, s, pos, sys_off, wall_shift,
                       kinds, wall, bbox, host, own);
  else
    hipLaunchKernelGGL(k_system_bbox<256>, dim3(nsys), dim3(256), 0, s, pos, sys_off, wall_shift,
                       kinds, wall, bbox, host, own);
  LM_HIP(hipGetLastError());
}

// The records of a particle of an open (wall: bottom-wall) system at (x, y, z),
// in units of a: FP64, and FP32 relative to the centre c of its system's box.
__device__ inline void put_records(int64_t i, int wall, double x, double y, double z, double a,
                                   double cx, double cy, double cz, double4* __restrict__ rec64,
                                   float4* __restrict__ rec32) {
  const double ia = 1.0 / a;
  if (wall) {
    const double h = fmax(z, a) * ia;
    const double b = fmin(fmax(z * ia, 0.0), 1.0);
    rec64[i] = double4{x * ia, y * ia, h, b};
    rec32[i] = float4{(float)((x - cx) * ia), (float)((y - cy) * ia), (float)h, (float)b};
  } else {
    rec64[i] = double4{x * ia, y * ia, z * ia, 1.0};
    rec32[i] = float4{(float)((x - cx) * ia), (float)((y - cy) * ia), (float)((z - cz) * ia), 1.0f};
  }
}

// Boxes, shifted positions and records of small open systems (at most
// kPlaceMax particles) in one launch, a workgroup per system that keeps its
// particles in registers: positions are read once, which matters where they
// lie in host memory, and one launch less of the few that a small step has.
__global__ __launch_bounds__(256) void k_place_small(const double* __restrict__ pos,
                                                     const int64_t* __restrict__ off,
                                                     double* __restrict__ bbox, double a,
                                                     double* __restrict__ shifted,
                                                     double4* __restrict__ rec64,
                                                     float4* __restrict__ rec32) {
  __shared__ double sh[6][4];
  constexpr int kQ = kPlaceMax / 256;
  const int s = blockIdx.x;
  const int64_t b = off[s], e = off[s + 1];
  double p[kQ][3];
  BoxSum<256> box;
#pragma unroll
  for (int q = 0; q < kQ; ++q) {
    const int64_t i = b + threadIdx.x + 256 * q;
    if (i < e) {
#pragma unroll
      for (int c = 0; c < 3; ++c) p[q][c] = pos[3 * i + c];
    }
  }
#pragma unroll
  for (int q = 0; q < kQ; ++q)
    if (b + threadIdx.x + 256 * q < e) box.add(p[q][0], p[q][1], p[q][2]);
  box.reduce(sh);
  if (threadIdx.x < 6) bbox[6 * s + threadIdx.x] = sh[threadIdx.x][0];
  const double cx = 0.5 * (sh[0][0] + sh[3][0]), cy = 0.5 * (sh[1][0] + sh[4][0]),
               cz = 0.5 * (sh[2][0] + sh[5][0]);
#pragma unroll
  for (int q = 0; q < kQ; ++q) {
    const int64_t i = b + threadIdx.x + 256 * q;
    if (i < e) {
#pragma unroll
      for (int c = 0; c < 3; ++c) shifted[3 * i + c] = p[q][c];
      put_records(i, 0, p[q][0], p[q][1], p[q][2], a, cx, cy, cz, rec64, rec32);
    }
  }
}

void launch_place_small(const double* pos, const int64_t* sys_off, int nsys, double* bbox, double a,
                        double* shifted, void* rec64, void* rec32, hipStream_t s) {
  if (nsys <= 0) return;
  hipLaunchKernelGGL(k_place_small, dim3(nsys), dim3(256), 0, s, pos, sys_off, bbox, a, shifted,
                     static_cast<double4*>(rec64), static_cast<float4*>(rec32));
  LM_HIP(hipGetLastError());
}

__global__ void k_make_records(const double* __restrict__ pos, int64_t N,
                               const int64_t* __restrict__ off, int nsys,
                               const double* __restrict__ bbox, const int* __restrict__ kinds,
                               int wall_all, double wall_shift, double a,
                               double* __restrict__ shifted, double4* __restrict__ rec64,
                               float4* __restrict__ rec32) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= N) return;
  int lo = 0, hi = nsys;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (off[mid] <= i) lo = mid; else hi = mid;
  }
  const double* bb = bbox + 6 * lo;
  const int wall = kinds ? kinds[lo] : wall_all;
  const double x = pos[3 * i], y = pos[3 * i + 1], z = pos[3 * i + 2] - (wall ? wall_shift : 0.0);
  if (shifted) {
    shifted[3 * i] = x;
    shifted[3 * i + 1] = y;
    shifted[3 * i + 2] = z;
  }
  put_records(i, wall, x, y, z, a, 0.5 * (bb[0] + bb[3]), 0.5 * (bb[1] + bb[4]),
              0.5 * (bb[2] + bb[5]), rec64, rec32);
}

void launch_make_records(const double* pos, int64_t N, const int64_t* sys_off, int nsys,
                         const double* bbox, const int* kinds, int wall, double wall_shift,
                         double a, double* shifted, void* rec64, void* rec32, hipStream_t s) {
  if (N <= 0) return;
  const int nt = 256;
  hipLaunchKernelGGL(k_make_records, dim3((unsigned)((N + nt - 1) / nt)), dim3(nt), 0, s, pos, N,
                     sys_off, nsys, bbox, kinds, wall, wall_shift, a, shifted,
                     static_cast<double4*>(rec64), static_cast<float4*>(rec32));
  LM_HIP(hipGetLastError());
}

__global__ void k_copy2(const double* __restrict__ x0, double* __restrict__ y0,
                        const double* __restrict__ x1, double* __restrict__ y1, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  if (y0 != nullptr) y0[i] = x0[i];
  if (y1 != nullptr) y1[i] = x1[i];
}

void launch_copy2(const double* x0, double* y0, const double* x1, double* y1, int64_t n,
                  hipStream_t s) {
  if (n <= 0 || (y0 == nullptr && y1 == nullptr)) return;
  hipLaunchKernelGGL(k_copy2, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, x0, y0, x1, y1, n);
  LM_HIP(hipGetLastError());
}

__global__ void k_zero_open(double* __restrict__ v, int64_t N, const int64_t* __restrict__ off,
                            int nsys, const int* __restrict__ kinds) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= N) return;
  int lo = 0, hi = nsys;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (off[mid] <= i) lo = mid; else hi = mid;
  }
  if (!kinds[lo]) {
    v[3 * i] = 0.0;
    v[3 * i + 1] = 0.0;
    v[3 * i + 2] = 0.0;
  }
}

void launch_zero_open_systems(double* v, int64_t N, const int64_t* sys_off, int nsys,
                              const int* kinds, hipStream_t s) {
  if (N <= 0 || !kinds) return;
  hipLaunchKernelGGL(k_zero_open, dim3((unsigned)((N + 255) / 256)), dim3(256), 0, s, v, N, sys_off,
                     nsys, kinds);
  LM_HIP(hipGetLastError());
}

}  // namespace lm
