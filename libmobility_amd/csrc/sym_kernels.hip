// Symmetric evaluation in symmetric units (sym_item.hpp): every form but the
// open translational block in FP32, and products that keep their order of
// operations (nbody_kernels.hip).
#include "kernels.hpp"
#include "lm_common.hpp"
#include "sym_item.hpp"

namespace lm {

namespace {

// Waves per SIMD the registers are cut for: 4 in FP32 (128 registers), 3 in
// FP64 (168).
template <class R>
constexpr int kSymWaves = std::is_same<R, float>::value ? 4 : 3;

}  // namespace

// KIND: 0 open, 1 wall, 2 per system (mixed ensembles).
template <class R, int KIND, int BLK, int TPL, int NW>
__global__ __launch_bounds__(64 * NW, kSymWaves<R>) void k_pair_sym_unit(SymArgs a) {
  __shared__ SymLds<R, BLK, NW> lds;
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
  if constexpr (KIND != 0) {
    if (KIND == 1 || S.wall != 0) {
      sym_unit<R, true, BLK, TPL, NW>(it, S, a, lds);
      return;
    }
  }
  if constexpr (KIND != 1) sym_unit<R, false, BLK, TPL, NW>(it, S, a, lds);
}

__global__ __launch_bounds__(256) void k_sym_items(SymItem* __restrict__ items, int nitems, SymSys S,
                                                  int oa, int ws, int cs, int nch, SymSys* sys,
                                                  SymRows* __restrict__ rows, int64_t nrows) {
  const int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (k == 0) *sys = S;
  const int ring = S.ntiles * cs;
  if (k < ring)
    items[k] = sym_ring_item(S, 0, (int)(k / cs), (int)(k % cs), cs, oa, ws);
  else if (k < nitems)
    items[k] = SymItem{0, (int)k - ring, 0, 0, nch};
  if (k < nrows) {
    const int64_t left = S.n - 256 * k;
    rows[k] = SymRows{S.off + 256 * k, (int32_t)(left < 256 ? left : 256), 0};
  }
}

void launch_sym_items(SymItem* items, int nitems, const SymSys& S, int oa, int ob, int nch, int diag,
                      SymSys* sys, SymRows* rows, int64_t nrows, hipStream_t s) {
  const int ws = (ob < S.hmax + 1 ? ob : S.hmax + 1) - oa;
  const int cs = sym_ring_chunks(S, ws, nch);
  if (nitems != S.ntiles * (cs + diag))
    throw Error("[libmobility_amd] symmetric work list of another size");
  const int64_t n = nitems > nrows ? nitems : nrows;
  if (n <= 0) return;
  hipLaunchKernelGGL(k_sym_items, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, items, nitems,
                     S, oa, ws, cs, nch, sys, rows, nrows);
  LM_HIP(hipGetLastError());
}

template <class R, int KIND, int BLK>
static void launch_unit_shape(const SymArgs& a, hipStream_t s) {
  const dim3 grid((unsigned)a.nitems);
  if (a.waves == 1 && a.tpl == 1)
    hipLaunchKernelGGL((k_pair_sym_unit<R, KIND, BLK, 1, 1>), grid, dim3(64), 0, s, a);
  else if (a.waves == 4 && a.tpl == 1)
    hipLaunchKernelGGL((k_pair_sym_unit<R, KIND, BLK, 1, 4>), grid, dim3(256), 0, s, a);
  else if (a.waves == 4 && a.tpl == 2)
    hipLaunchKernelGGL((k_pair_sym_unit<R, KIND, BLK, 2, 4>), grid, dim3(256), 0, s, a);
  else
    throw Error("[libmobility_amd] unsupported shape of the symmetric kernel");
  LM_HIP(hipGetLastError());
}

template <class R, int KIND>
static void launch_unit_blk(const SymArgs& a, hipStream_t s) {
  switch (a.blocks) {
    case kUF: launch_unit_shape<R, KIND, kUF>(a, s); break;
    case kUF | kWF: launch_unit_shape<R, KIND, kUF | kWF>(a, s); break;
    case kUT | kWT: launch_unit_shape<R, KIND, kUT | kWT>(a, s); break;
    case kUF | kUT | kWT | kWF: launch_unit_shape<R, KIND, kUF | kUT | kWT | kWF>(a, s); break;
    default: throw Error("[libmobility_amd] unsupported block combination");
  }
}

template <class R>
static void launch_unit_kind(const SymArgs& a, hipStream_t s) {
  switch (a.wall) {
    case 0: launch_unit_blk<R, 0>(a, s); break;
    case 1: launch_unit_blk<R, 1>(a, s); break;
    case 2: launch_unit_blk<R, 2>(a, s); break;
    default: throw Error("[libmobility_amd] invalid kernel kind");
  }
}

void launch_pair_sym_unit(const SymArgs& a, hipStream_t s) {
  if (a.nitems <= 0) return;
  if (a.fp32)
    launch_unit_kind<float>(a, s);
  else
    launch_unit_kind<double>(a, s);
}

}  // namespace lm
