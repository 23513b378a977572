// Counting sort of one system's particles into grid cells (cell_sort.hpp).  On
// the host the two grids of the preconditioner took 0.3 ms each for 32768
// particles, with 0.1 ms of transfers, while the GPU had nothing to do; here
// about 25 us each.
#include "cell_sort.hpp"
#include "lm_common.hpp"

namespace lm {

namespace {
constexpr int kCT = 256;
inline unsigned cell_blocks(int64_t n) { return (unsigned)((n + kCT - 1) / kCT); }
}  // namespace

__global__ __launch_bounds__(kCT) void k_record_box(const double4* __restrict__ rec, int64_t N,
                                                   double* host) {
  __shared__ double sh[6][kCT / 64];
  double mn[3] = {1e300, 1e300, 1e300}, mx[3] = {-1e300, -1e300, -1e300};
  for (int64_t i = (int64_t)blockIdx.x * kCT + threadIdx.x; i < N; i += (int64_t)gridDim.x * kCT) {
    const double4 p = rec[i];
    const double x[3] = {p.x, p.y, p.z};
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      mn[c] = fmin(mn[c], x[c]);
      mx[c] = fmax(mx[c], x[c]);
    }
  }
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    for (int o = 32; o > 0; o >>= 1) {
      mn[c] = fmin(mn[c], __shfl_xor(mn[c], o));
      mx[c] = fmax(mx[c], __shfl_xor(mx[c], o));
    }
    if ((threadIdx.x & 63) == 0) {
      sh[c][threadIdx.x >> 6] = mn[c];
      sh[3 + c][threadIdx.x >> 6] = mx[c];
    }
  }
  __syncthreads();
  if (threadIdx.x < 6) {
    const int c = threadIdx.x;
    double v = sh[c][0];
    for (int w = 1; w < kCT / 64; ++w) v = c < 3 ? fmin(v, sh[c][w]) : fmax(v, sh[c][w]);
    host[6 * blockIdx.x + c] = v;
  }
}

void launch_record_box(const double4* rec, int64_t N, double* host, hipStream_t s) {
  hipLaunchKernelGGL(k_record_box, dim3(kBoxBlocks), dim3(kCT), 0, s, rec, N, host);
  LM_HIP(hipGetLastError());
}

__global__ __launch_bounds__(kCT) void k_cell_count(const double4* __restrict__ rec, int64_t N,
                                                   CellGrid grid, int* __restrict__ raw,
                                                   int* __restrict__ count) {
  const int64_t i = (int64_t)blockIdx.x * kCT + threadIdx.x;
  if (i >= N) return;
  const double4 p = rec[i];
  const double x[3] = {p.x, p.y, p.z};
  int q[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    q[k] = 0;
    if (grid.ext[k] > 0.0) {
      const double d = x[k] - grid.lo[k];
      const double f = floor(grid.by_edge ? d / grid.edge[k] : d / grid.ext[k] * grid.g[k]);
      const double top = grid.g[k] - 1, c = 0.0 < f ? f : 0.0;
      q[k] = (int)(c < top ? c : top);
    }
  }
  const int cell = (q[0] * grid.g[1] + q[1]) * grid.g[2] + q[2];
  raw[i] = cell;
  atomicAdd(&count[cell], 1);
}

__global__ __launch_bounds__(kCT) void k_cell_zero(int* __restrict__ count, int n) {
  const int c = blockIdx.x * kCT + threadIdx.x;
  if (c < n) count[c] = 0;
}

void launch_cell_count(const double4* rec, int64_t N, const CellGrid& grid, int* raw, int* count,
                       int ncell, hipStream_t s) {
  hipLaunchKernelGGL(k_cell_zero, dim3(cell_blocks(ncell)), dim3(kCT), 0, s, count, ncell);
  hipLaunchKernelGGL(k_cell_count, dim3(cell_blocks(N)), dim3(kCT), 0, s, rec, N, grid, raw, count);
  LM_HIP(hipGetLastError());
}

// One workgroup; thread t has the cells [t m, (t + 1) m).
constexpr int kScanT = 1024;
__global__ __launch_bounds__(kScanT) void k_cell_scan(CellScan a) {
  __shared__ int64_t s_n[kScanT / 64];
  __shared__ int s_c[kScanT / 64], s_m[kScanT / 64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int m = (a.ncell + kScanT - 1) / kScanT;
  const int c0 = min((int)threadIdx.x * m, a.ncell), c1 = min(c0 + m, a.ncell);
  int64_t n = 0;
  int cells = 0, top = 0;
  for (int c = c0; c < c1; ++c) {
    const int k = a.count[c];
    n += k;
    cells += k > 0;
    top = max(top, k);
  }
  // inclusive sums over the lanes, then over the waves before
  int64_t in = n;
  int ic = cells;
  for (int o = 1; o < 64; o <<= 1) {
    const int64_t vn = __shfl_up((long long)in, o);
    const int vc = __shfl_up(ic, o);
    if (lane >= o) {
      in += vn;
      ic += vc;
    }
  }
  for (int o = 32; o > 0; o >>= 1) top = max(top, __shfl_xor(top, o));
  if (lane == 63) {
    s_n[wave] = in;
    s_c[wave] = ic;
    s_m[wave] = top;
  }
  __syncthreads();
  int64_t bn = in - n;
  int bc = ic - cells;
  for (int w = 0; w < wave; ++w) {
    bn += s_n[w];
    bc += s_c[w];
  }
  for (int c = c0; c < c1; ++c) {
    const int k = a.count[c];
    if (a.start64 != nullptr) a.start64[c] = bn;
    if (a.compact != nullptr) {
      a.compact[c] = k > 0 ? bc : -1;
      if (k > 0) a.start32[bc++] = (int)bn;
    }
    bn += k;
  }
  if (threadIdx.x == kScanT - 1) {
    if (a.start64 != nullptr) a.start64[a.ncell] = bn;
    if (a.compact != nullptr) a.start32[bc] = (int)bn;
    if (a.host != nullptr) {
      int all = 0;
      for (int w = 0; w < kScanT / 64; ++w) all = max(all, s_m[w]);
      a.host[0] = bc;
      a.host[1] = all;
    }
  }
}

void launch_cell_scan(const CellScan& a, hipStream_t s) {
  hipLaunchKernelGGL(k_cell_scan, dim3(1), dim3(kScanT), 0, s, a);
  LM_HIP(hipGetLastError());
}

template <class I>
__global__ __launch_bounds__(kCT) void k_cell_fill(const int* __restrict__ raw, int64_t N,
                                                  const int* __restrict__ compact,
                                                  const I* __restrict__ start,
                                                  int* __restrict__ count, int* __restrict__ list) {
  const int64_t i = (int64_t)blockIdx.x * kCT + threadIdx.x;
  if (i >= N) return;
  const int c = raw[i];
  list[start[compact != nullptr ? compact[c] : c] + atomicSub(&count[c], 1) - 1] = (int)i;
}

void launch_cell_fill64(const int* raw, int64_t N, const int64_t* start, int* count, int* list,
                        hipStream_t s) {
  hipLaunchKernelGGL(k_cell_fill<int64_t>, dim3(cell_blocks(N)), dim3(kCT), 0, s, raw, N,
                     static_cast<const int*>(nullptr), start, count, list);
  LM_HIP(hipGetLastError());
}

void launch_cell_fill32(const int* raw, int64_t N, const int* compact, const int* start, int* count,
                        int* list, hipStream_t s) {
  hipLaunchKernelGGL(k_cell_fill<int>, dim3(cell_blocks(N)), dim3(kCT), 0, s, raw, N, compact,
                     start, count, list);
  LM_HIP(hipGetLastError());
}

__global__ __launch_bounds__(kCT) void k_cell_order(const int* __restrict__ raw, int64_t N,
                                                   const int* __restrict__ compact,
                                                   const int* __restrict__ start, int C,
                                                   const int* __restrict__ list,
                                                   int* __restrict__ perm,
                                                   int* __restrict__ cell_of,
                                                   double* __restrict__ scale) {
  const int64_t t = (int64_t)blockIdx.x * kCT + threadIdx.x;
  if (t < C) scale[t] = 1.0 / sqrt((double)(start[t + 1] - start[t]));
  if (t >= N) return;
  const int i = list[t];  // a wave's particles share their cells
  const int c = compact[raw[i]];
  const int s0 = start[c], s1 = start[c + 1];
  int rank = 0;
  for (int k = s0; k < s1; ++k) rank += list[k] < i;
  perm[s0 + rank] = i;
  cell_of[i] = c;
}

void launch_cell_order(const int* raw, int64_t N, const int* compact, const int* start, int C,
                       const int* list, int* perm, int* cell_of, double* scale, hipStream_t s) {
  hipLaunchKernelGGL(k_cell_order, dim3(cell_blocks(N > C ? N : C)), dim3(kCT), 0, s, raw, N,
                     compact, start, C, list, perm, cell_of, scale);
  LM_HIP(hipGetLastError());
}

}  // namespace lm
