// Coarse level of the two-level sqrtMdotW preconditioner (no counterpart in the
// reference): particles are grouped into spatial cells, separately for every
// system of an ensemble; Q (3N x 3C) holds one orthonormal column per cell
// and direction, Q[3i+a, 3c+a] = 1/sqrt(n_c) for particle i in cell c.  The
// kernels build Mc = Q^T M Q from the pair terms (block-diagonal over the
// systems, one dense block each), factor each block Mc_s = L_s L_s^T, form
// X_s = L_s^{-1}, and apply
//     out = in + Q (T - I) Q^T in,   T = X, X^T or L,
// on the translational entries.  Everything is FP64 except the pair terms of
// Mc (FP32 geometry and coefficients, FP32 sums per lane over one source cell,
// FP64 beyond), which only shape the preconditioner: exactness of the square
// root rests on X and L being inverses of each other, which holds to FP64
// rounding whatever Mc is.
#include <hip/hip_runtime.h>

#include "coarse.hpp"
#include "kernels.hpp"
#include "lm_common.hpp"
#include "pair_math.hpp"

namespace lm {

namespace {

constexpr int kT = kCoarseTile;  // 64: dense tile edge
constexpr int kP = kT + 1;       // LDS row pitch (doubles)
constexpr int kKB = 4;           // tile columns per block of the factorisation updates
constexpr int kWaveRowMax = 2048;  // longest coarse row of the one-wave-per-row matvec
// trailing updates of at least this many tiles use the two-by-two-tile kernels
constexpr int64_t kQuadTiles = 1024;

// ---- cell-sorted records ---------------------------------------------------

template <class R4>
__global__ void k_gather_records(const R4* __restrict__ rec, const int* __restrict__ perm,
                                 int64_t N, R4* __restrict__ out) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k < N) out[k] = rec[perm[k]];
}

// ---- Mc = Q^T M Q ------------------------------------------------------------

// p -> (c, d) with c >= d, p = c (c + 1) / 2 + d
__device__ inline void tri_index(int64_t p, int& c, int& d) {
  int64_t cc = (int64_t)((sqrt(8.0 * (double)p + 1.0) - 1.0) * 0.5);
  while (cc * (cc + 1) / 2 > p) --cc;
  while ((cc + 1) * (cc + 2) / 2 <= p) ++cc;
  c = (int)cc;
  d = (int)(p - cc * (cc + 1) / 2);
}

// s += the 3x3 translational block M_ij / t0 of the pair (ri, rj),
// row-major (open: the six entries of the upper triangle, times 4/3: the
// caller scales the open sums by 3/4)
template <bool WALL, class R, class R4>
__device__ inline void pair_block_sum(const R4 ri, const R4 rj, R s[9]) {
  if (WALL) {
    UFCoef<R> k;
    uf_coef_wall<R>(ri.x, ri.y, ri.z, rj.x, rj.y, rj.z, k);
    // the damping, and back from 4/3 of the block
    const R q = R(0.75) * ri.w * rj.w;
    k.a0 *= q;
    k.cd *= q;
    k.ex *= q;
    k.ey *= q;
    k.ez *= q;
    k.hx *= q;
    k.hy *= q;
    k.hz *= q;
    const R dv[3] = {k.dx, k.dy, k.dz};
    const R ev[3] = {k.ex, k.ey, k.ez};
    const R gv[3] = {k.gx, k.gy, k.gz};
    const R hv[3] = {k.hx, k.hy, k.hz};
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
      for (int b = 0; b < 3; ++b)
        s[3 * a + b] += (a == b ? k.a0 : R(0)) + k.cd * dv[a] * dv[b] + gv[a] * ev[b] +
                        (b == 2 ? hv[a] : R(0));
  } else {
    const R dx = ri.x - rj.x, dy = ri.y - rj.y, dz = ri.z - rj.z;
    const R r2 = dx * dx + dy * dy + dz * dz;
    const R ir = lm_rsqrt(r2);
    RpyCoef<R> cf{};
    rpy_far_uf34<R>(ir, cf);
    if (__builtin_expect(r2 < R(4), 0)) {
      lm_rare_path();
      rpy_near_select_uf34<R>(r2, ir, cf);
    }
    const R fuf = cf.fuf, guf = cf.guf;
    s[0] += fuf + guf * dx * dx;
    s[1] += guf * dx * dy;
    s[2] += guf * dx * dz;
    s[4] += fuf + guf * dy * dy;
    s[5] += guf * dy * dz;
    s[8] += fuf + guf * dz * dz;
  }
}

// s += sum over targets i in [i0, i1) and sources j in [j0, j1) of the
// pair blocks, this lane's share.  The two cells go through the wave's LDS
// (sh: 128 records) in chunks of up to 64 x 64 particles, and the 64 lanes
// walk a chunk's ni x nj pairs in row-major order, lane l taking pairs
// l, l + 64, ...: every lane works whatever the cell sizes.
template <bool WALL, class R, class R4>
__device__ inline void cell_pair_sum(const R4* __restrict__ rec, int i0, int i1, int j0, int j1,
                                     int lane, R4* sh, R s[9]) {
  for (int ib = i0; ib < i1; ib += 64) {
    const int ni = min(64, i1 - ib);
    for (int jb = j0; jb < j1; jb += 64) {
      const int nj = min(64, j1 - jb);
      // The wave's reads of the previous chunk precede these writes in its
      // LDS order.
      if (lane < ni) sh[lane] = rec[ib + lane];
      if (lane < nj) sh[64 + lane] = rec[jb + lane];
      __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
      __builtin_amdgcn_wave_barrier();
      const int di = 64 / nj, dj = 64 - di * nj;  // a step of 64 pairs
      int ii = lane / nj, jj = lane - ii * nj;
      for (int p = lane; p < ni * nj; p += 64) {
        pair_block_sum<WALL, R, R4>(sh[ii], sh[64 + jj], s);
        ii += di;
        jj += dj;
        if (jj >= nj) {
          jj -= nj;
          ++ii;
        }
      }
    }
  }
  if (!WALL) {
    s[3] = s[1];
    s[6] = s[2];
    s[7] = s[5];
  }
}

// One wave per cell pair (c >= d) of one system: the lanes share the pairs
// of the two cells, then a butterfly sums the lanes.  The block and its
// transpose go to the system's matrix (Mc is symmetric because
// M_ji = M_ij^T).  pair_off[s] counts the cell pairs of the systems before s.
template <class R, class R4>
__global__ __launch_bounds__(256) void k_coarse_matrix(const R4* __restrict__ rec,
                                                       const int* __restrict__ start,
                                                       const double* __restrict__ scale,
                                                       const CoarseSys* __restrict__ sys,
                                                       const int64_t* __restrict__ pair_off,
                                                       int nsys, int64_t npairs,
                                                       double* __restrict__ Mc) {
  __shared__ R4 sh[4][128];
  const int lane = threadIdx.x & 63;
  // grid-stride over the cell pairs: one launch may not exceed 2^32 work-items
  for (int64_t p = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); p < npairs;
       p += (int64_t)gridDim.x * 4) {  // uniform per wave
    int lo = 0, hi = nsys;  // the last system with pair_off <= p
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (pair_off[mid] <= p) lo = mid; else hi = mid;
    }
    const CoarseSys S = sys[lo];
    int c, d;
    tri_index(p - pair_off[lo], c, d);
    const int gc = S.c0 + c, gd = S.c0 + d;
    R s[9];
  #pragma unroll
    for (int k = 0; k < 9; ++k) s[k] = R(0);
    R4* w = sh[threadIdx.x >> 6];
    if (S.wall)
      cell_pair_sum<true, R, R4>(rec, start[gc], start[gc + 1], start[gd], start[gd + 1], lane, w, s);
    else
      cell_pair_sum<false, R, R4>(rec, start[gc], start[gc + 1], start[gd], start[gd + 1], lane, w,
                                  s);
    double v[9];
  #pragma unroll
    for (int k = 0; k < 9; ++k) {
      v[k] = (double)s[k];
  #pragma unroll
      for (int o = 32; o > 0; o >>= 1) v[k] += __shfl_xor(v[k], o);
    }
    if (lane == 0) {
      const double f = scale[gc] * scale[gd] * (S.wall ? 1.0 : 0.75);  // open sums carry 4/3
      double* M = Mc + S.moff;
  #pragma unroll
      for (int a = 0; a < 3; ++a)
  #pragma unroll
        for (int b = 0; b < 3; ++b) {
          M[(int64_t)(3 * c + a) * S.n + 3 * d + b] = f * v[3 * a + b];
          if (c != d) M[(int64_t)(3 * d + b) * S.n + 3 * c + a] = f * v[3 * a + b];
        }
    }
  }
}

// unit diagonal on each system's padding rows [3C, n)
__global__ void k_pad_identity(double* __restrict__ A, const CoarseSys* __restrict__ sys) {
  const CoarseSys S = sys[blockIdx.x];
  for (int r = 3 * S.C + (int)threadIdx.x; r < S.n; r += blockDim.x)
    A[S.moff + (int64_t)r * S.n + r] = 1.0;
}

// ---- dense 64 x 64 tiles in LDS ------------------------------------------------

constexpr int kTT = 256;                 // threads of the tile operations
constexpr int kTQ = kT * kT / kTT;       // tile entries per thread

// A tile on its way from memory to LDS: every load of a thread is in flight at
// once (one at a time, a tile took 5 us, most of an operation).
struct TileRegs {
  double v[kTQ];
  __device__ void fetch(const double* __restrict__ g, int64_t ld) {
#pragma unroll
    for (int q = 0; q < kTQ; ++q) {
      const int e = (int)threadIdx.x + kTT * q;
      v[q] = g[(e >> 6) * ld + (e & 63)];
    }
  }
  __device__ void stage(double (*S)[kP]) const {
#pragma unroll
    for (int q = 0; q < kTQ; ++q) {
      const int e = (int)threadIdx.x + kTT * q;
      S[e >> 6][e & 63] = v[q];
    }
  }
};

__device__ inline void tile_load(double (*S)[kP], const double* __restrict__ g, int64_t ld) {
  TileRegs t;
  t.fetch(g, ld);
  t.stage(S);
}

__device__ inline void tile_load2(double (*S0)[kP], const double* __restrict__ g0, int64_t ld0,
                                  double (*S1)[kP], const double* __restrict__ g1, int64_t ld1) {
  TileRegs t0, t1;
  t0.fetch(g0, ld0);
  t1.fetch(g1, ld1);
  t0.stage(S0);
  t1.stage(S1);
}

typedef double d4 __attribute__((ext_vector_type(4)));

__device__ inline void tile_zero(d4 acc[2][2]) {
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) acc[a][b] = d4{0.0, 0.0, 0.0, 0.0};
}

// acc += A * (TB ? B^T : B) for 64 x 64 tiles in LDS on the FP64 matrix cores
// (256 threads): wave w computes the 32 x 32 quadrant (w >> 1, w & 1) as
// 2 x 2 tiles of v_mfma_f64_16x16x4f64.  Operand lanes: A[i][k] from lane
// 16 k + i, B[k][j] from lane 16 k + j; result register r of lane l holds
// row 4 r + (l >> 4) of column l & 15 (layout measured on gfx950).  Every
// index stays in the 64 x 64 tile.
template <bool TB>
__device__ inline void tile_mm_mfma(const double (*A)[kP], const double (*B)[kP], d4 acc[2][2]) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int R0 = (w >> 1) * 32, C0 = (w & 1) * 32;
  const int li = lane & 15, lk = lane >> 4;
#pragma unroll 4
  for (int kk = 0; kk < kT; kk += 4) {
    const double a0 = A[R0 + li][kk + lk], a1 = A[R0 + 16 + li][kk + lk];
    const double b0 = TB ? B[C0 + li][kk + lk] : B[kk + lk][C0 + li];
    const double b1 = TB ? B[C0 + 16 + li][kk + lk] : B[kk + lk][C0 + 16 + li];
    acc[0][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b0, acc[0][0], 0, 0, 0);
    acc[0][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b1, acc[0][1], 0, 0, 0);
    acc[1][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b0, acc[1][0], 0, 0, 0);
    acc[1][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b1, acc[1][1], 0, 0, 0);
  }
}

// Entry (a, b, r) of a lane in the layout of tile_mm_mfma's result: row and column.
__device__ inline int mfma_row(int a, int r) {
  return ((int)threadIdx.x >> 7) * 32 + 16 * a + 4 * r + (((int)threadIdx.x & 63) >> 4);
}
__device__ inline int mfma_col(int b) {
  return (((int)threadIdx.x >> 6) & 1) * 32 + 16 * b + ((int)threadIdx.x & 15);
}

// d = the tile at g in the layout of tile_mm_mfma's result (all loads in flight)
__device__ inline void tile_fetch_mfma(const double* __restrict__ g, int64_t ld, d4 d[2][2]) {
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) d[a][b][r] = g[mfma_row(a, r) * ld + mfma_col(b)];
}

// out[row][col] = the result of tile_mm_mfma
__device__ inline void tile_store_mfma(double* __restrict__ out, int64_t ld, const d4 acc[2][2]) {
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) out[mfma_row(a, r) * ld + mfma_col(b)] = acc[a][b][r];
}

// d -= acc
__device__ inline void tile_sub(d4 d[2][2], const d4 acc[2][2]) {
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) d[a][b] -= acc[a][b];
}

// acc += A * (TB ? B^T : B) for 64 x 64 tiles in LDS, the whole tile by one
// wave: 4 x 4 tiles of v_mfma_f64_16x16x4f64, 16 products per 8 operand
// reads (same lane layout as tile_mm_mfma).
template <bool TB>
__device__ inline void tile_mm_wave(const double (*A)[kP], const double (*B)[kP], d4 acc[4][4]) {
  const int lane = threadIdx.x & 63;
  const int li = lane & 15, lk = lane >> 4;
#pragma unroll 2
  for (int kk = 0; kk < kT; kk += 4) {
    double a[4], b[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      a[q] = A[16 * q + li][kk + lk];
      b[q] = TB ? B[16 * q + li][kk + lk] : B[kk + lk][16 * q + li];
    }
#pragma unroll
    for (int p = 0; p < 4; ++p)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        acc[p][q] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[p], b[q], acc[p][q], 0, 0, 0);
  }
}

// out[row][col] -= the tile result of tile_mm_wave, 16 entries in flight
__device__ inline void tile_sub_wave(double* __restrict__ out, int64_t ld, const d4 acc[4][4]) {
  const int lane = threadIdx.x & 63;
  const int li = lane & 15, lk = lane >> 4;
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    double* o = out + (int64_t)(16 * p + lk) * ld + li;
    double v[4][4];
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int r = 0; r < 4; ++r) v[q][r] = o[4 * r * ld + 16 * q];
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int r = 0; r < 4; ++r) o[4 * r * ld + 16 * q] = v[q][r] - acc[p][q][r];
  }
}

// ---- tile operations of the factorisation (256 threads each) -------------------
// Every operation starts with a workgroup barrier, so that one workgroup can
// run a sequence of them on the same LDS tiles and matrices.  The Cholesky
// is blocked by kKB tile columns: a block [kb, kend) is finished first, and
// the tiles right of it receive its kKB products in one read-modify-write.
// X = L^{-1} is the block forward substitution on L X = I, blocked the same
// way.

// value of v in lane `lane` (uniform) of the wave
__device__ inline double lane_value(double v, int lane) {
  const long long b = __builtin_bit_cast(long long, v);
  const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffLL), lane);
  const int hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
  return __builtin_bit_cast(double, ((long long)hi << 32) | (unsigned int)lo);
}

// Cholesky factor of one 64 x 64 tile in LDS (256 threads).  S: the lower part
// of an SPD tile on entry, L on exit (the part above the diagonal holds
// anything); W: L^{-T} on exit.  The column operations that turn A into L turn
// the identity below it into L^{-T}, so the tile is factored as the 128 x 64
// matrix [A; I], in four panels of 16 columns.  In a panel every wave holds the
// panel's 16 diagonal rows in lanes 0-15 and eliminates them redundantly,
// lanes 16-63 hold further rows (wave 0 those of A, waves 1 and 2 those of W;
// rows of W above the panel's end only, the others are still zero there); a
// column's multipliers reach the lanes by readlane.  The columns to the right
// get the panel's product from the matrix cores.  Bound by the chain of 64
// pivots: one wave with the whole tile in registers, and a forward
// substitution for the inverse, took 43 us; a whole column of L around this
// (k_chol_column) takes 19.
// Returns false if a pivot is not positive.
__device__ inline bool chol_tile(double (*S)[kP], double (*W)[kP]) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int li = lane & 15, lk = lane >> 4;
  bool ok = true;
#pragma unroll
  for (int q = 0; q < kTQ; ++q) {
    const int e = (int)threadIdx.x + kTT * q;
    W[e >> 6][e & 63] = (e >> 6) == (e & 63);
  }
  __syncthreads();
#pragma unroll 1
  for (int p = 0; p < kT / 16; ++p) {
    const int c0 = 16 * p;
    // the row of this lane: of S where it is below 64, of W from 64 on, -1 none
    int row = -1;
    if (wave == 0) {
      if (c0 + lane < kT) row = c0 + lane;
    } else if (wave < 3) {
      const int q = 32 * (wave - 1) + lane - 16;
      if (lane < 16) row = c0 + lane;
      else if (lane < 48 && q < c0 + 16) row = kT + q;
    }
    double* r = row < 0 ? S[0] : (row < kT ? S[row] : W[row - kT]);
    double a[16];
#pragma unroll
    for (int c = 0; c < 16; ++c) a[c] = row < 0 ? 0.0 : r[c0 + c];
    __syncthreads();  // every wave has read the diagonal rows
    if (wave < 3) {
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        double d = lane_value(a[j], j);
        if (!(d > 0.0)) {
          ok = false;
          d = 1.0;
        }
        // sqrt(d) and its reciprocal, each corrected once by its residual
        double ipiv = lm_rsqrt(d);
        double piv = d * ipiv;
        piv = __builtin_fma(0.5 * ipiv, __builtin_fma(-piv, piv, d), piv);
        ipiv = __builtin_fma(ipiv, __builtin_fma(-piv, ipiv, 1.0), ipiv);
        a[j] = lane == j ? piv : a[j] * ipiv;
#pragma unroll
        for (int c = j + 1; c < 16; ++c) a[c] = __builtin_fma(-a[j], lane_value(a[j], c), a[c]);
      }
      if (row >= 0 && (wave == 0 || lane >= 16)) {
#pragma unroll
        for (int c = 0; c < 16; ++c) r[c0 + c] = a[c];
      }
    }
    __syncthreads();
    // 16 x 16 tiles (tr, tc), tc > p: rows tr >= tc of S, rows tr <= p of W
    const int rem = kT / 16 - 1 - p;
    const int ns = rem * (rem + 1) / 2, nw = (p + 1) * rem;
    for (int t = wave; t < ns + nw; t += 4) {  // uniform per wave
      int tr, tc;
      double(*X)[kP] = S;
      if (t < ns) {
        tri_index(t, tr, tc);
        tr += p + 1;
        tc += p + 1;
      } else {
        X = W;
        tr = (t - ns) / rem;
        tc = p + 1 + (t - ns) % rem;
      }
      d4 acc = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int kk = 0; kk < 16; kk += 4)
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(X[16 * tr + li][c0 + kk + lk],
                                                   S[16 * tc + li][c0 + kk + lk], acc, 0, 0, 0);
#pragma unroll
      for (int q = 0; q < 4; ++q) X[16 * tr + 4 * q + lk][16 * tc + li] -= acc[q];
    }
    __syncthreads();
  }
  return ok;
}

// L_kk and Dinv_k = L_kk^{-1} from chol_tile's tiles to memory
__device__ inline void store_diag(double* __restrict__ Lkk, int64_t ld, double* __restrict__ D,
                                  const double (*S)[kP], const double (*W)[kP]) {
#pragma unroll
  for (int q = 0; q < kTQ; ++q) {
    const int e = (int)threadIdx.x + kTT * q;
    const int r = e >> 6, c = e & 63;
    Lkk[(int64_t)r * ld + c] = c <= r ? S[r][c] : 0.0;
    D[e] = W[c][r];
  }
}

// Factor the diagonal tile k in place and write its inverse Dinv_k; info[0] = 1
// when a pivot is not positive.
__device__ inline void op_chol_diag(double* __restrict__ A, int64_t ld, int k,
                                    double* __restrict__ Dinv, int* __restrict__ info,
                                    double (*P0)[kP], double (*P1)[kP]) {
  __syncthreads();
  double* Akk = A + (int64_t)k * kT * ld + (int64_t)k * kT;
  tile_load(P0, Akk, ld);
  __syncthreads();
  if (!chol_tile(P0, P1) && threadIdx.x == 0) info[0] = 1;
  store_diag(Akk, ld, Dinv + (int64_t)k * kT * kT, P0, P1);
}

// L_ik = A_ik L_kk^{-T}
__device__ inline void op_panel(double* __restrict__ A, int64_t ld, int k, int i,
                                const double* __restrict__ Dinv, double (*P0)[kP],
                                double (*P1)[kP]) {
  __syncthreads();
  double* Aik = A + (int64_t)i * kT * ld + (int64_t)k * kT;
  tile_load2(P0, Aik, ld, P1, Dinv + (int64_t)k * kT * kT, kT);
  __syncthreads();
  d4 acc[2][2];
  tile_zero(acc);
  tile_mm_mfma<true>(P0, P1, acc);
  tile_store_mfma(Aik, ld, acc);
}

// out -= sum over s < count of a_s (TB ? b_s^T : b_s), the tiles a_s at a + s sa,
// b_s at b + s sb; the tiles of a step are loaded while the matrix cores work on
// the step before.
template <bool TB>
__device__ inline void op_update(double* out, const double* a, int64_t sa, const double* b,
                                 int64_t sb, int count, int64_t ld, double (*P0)[kP],
                                 double (*P1)[kP]) {
  d4 acc[2][2], d[2][2];
  TileRegs ta, tb;
  __syncthreads();  // what the tiles hold is in memory and LDS is free
  ta.fetch(a, ld);
  tb.fetch(b, ld);
  tile_fetch_mfma(out, ld, d);
  tile_zero(acc);
  for (int s = 0; s < count; ++s) {
    if (s > 0) __syncthreads();
    ta.stage(P0);
    tb.stage(P1);
    __syncthreads();
    if (s + 1 < count) {
      ta.fetch(a + (s + 1) * sa, ld);
      tb.fetch(b + (s + 1) * sb, ld);
    }
    tile_mm_mfma<TB>(P0, P1, acc);
  }
  tile_sub(d, acc);
  tile_store_mfma(out, ld, d);
}

// A_ij -= sum_{k in [k0, k1)} L_ik L_jk^T
__device__ inline void op_chol_update(double* A, int64_t ld, int i, int j, int k0, int k1,
                                      double (*P0)[kP], double (*P1)[kP]) {
  double* Ai = A + (int64_t)i * kT * ld;
  op_update<true>(Ai + (int64_t)j * kT, Ai + (int64_t)k0 * kT, kT,
                  A + (int64_t)j * kT * ld + (int64_t)k0 * kT, kT, k1 - k0, ld, P0, P1);
}

// X_km = Dinv_k X_km
__device__ inline void op_trinv_scale(double* __restrict__ X, int64_t ld, int k, int m,
                                      const double* __restrict__ Dinv, double (*P0)[kP],
                                      double (*P1)[kP]) {
  __syncthreads();
  double* Xkm = X + (int64_t)k * kT * ld + (int64_t)m * kT;
  tile_load2(P0, Xkm, ld, P1, Dinv + (int64_t)k * kT * kT, kT);
  __syncthreads();
  d4 acc[2][2];
  tile_zero(acc);
  tile_mm_mfma<false>(P1, P0, acc);
  tile_store_mfma(Xkm, ld, acc);
}

// X_im -= sum_{k in [k0, k1)} L_ik X_km
__device__ inline void op_trinv_update(double* X, const double* L, int64_t ld, int i, int m, int k0,
                                       int k1, double (*P0)[kP], double (*P1)[kP]) {
  op_update<false>(X + (int64_t)i * kT * ld + (int64_t)m * kT,
                   L + (int64_t)i * kT * ld + (int64_t)k0 * kT, kT,
                   X + (int64_t)k0 * kT * ld + (int64_t)m * kT, kT * ld, k1 - k0, ld, P0, P1);
}

// Xt tile (bj, bi) = (X tile (bi, bj))^T
__device__ inline void op_transpose(const double* __restrict__ X, double* __restrict__ Xt,
                                    int64_t ld, int bi, int bj, double (*P0)[kP]) {
  __syncthreads();
  tile_load(P0, X + (int64_t)bi * kT * ld + (int64_t)bj * kT, ld);
  __syncthreads();
  double* o = Xt + (int64_t)bj * kT * ld + (int64_t)bi * kT;
#pragma unroll
  for (int q = 0; q < kTQ; ++q) {
    const int e = (int)threadIdx.x + kTT * q;
    o[(e >> 6) * ld + (e & 63)] = P0[e & 63][e >> 6];
  }
}

// ---- one matrix, one launch per step ---------------------------------------------

// S = d, in LDS
__device__ inline void tile_put_mfma(double (*S)[kP], const d4 d[2][2]) {
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) S[mfma_row(a, r)][mfma_col(b)] = d[a][b][r];
}

// Tile column k of L, one workgroup per tile row i = k + blockIdx.x, from the
// block's columns before it (left-looking inside the block of kKB columns):
//   A_ik -= sum_{k' in [kb, k)} L_ik' L_kk'^T,   L_ik = A_ik L_kk^{-T}.
// Every workgroup updates and factors the diagonal tile itself, so a column is
// one launch: with launches of their own for the diagonal tile, the column and
// the update of the block's later columns a column took 71 us on average, of
// which most was one wave's chain and the launches' latency; now 19 to 37 us,
// 28 on average (36 tiles).  A_kk is read by all and written by none: workgroup 0 leaves L_kk in
// `Lkk` (row pitch ld) until the whole of L is done.
__global__ __launch_bounds__(256) void k_chol_column(double* __restrict__ A, int64_t ld, int kb,
                                                     int k, double* __restrict__ Lkk,
                                                     double* __restrict__ Dinv,
                                                     int* __restrict__ info) {
  __shared__ double P[4][kT][kP];
  const int i = k + (int)blockIdx.x;
  const bool below = i > k;  // uniform per workgroup
  const double* rowk = A + (int64_t)k * kT * ld;
  double* rowi = A + (int64_t)i * kT * ld;
  d4 dk[2][2], di[2][2], ak[2][2], ai[2][2];
  TileRegs tk, ti;
  if (kb < k) {
    tk.fetch(rowk + (int64_t)kb * kT, ld);
    if (below) ti.fetch(rowi + (int64_t)kb * kT, ld);
  }
  tile_fetch_mfma(rowk + (int64_t)k * kT, ld, dk);
  tile_fetch_mfma(rowi + (int64_t)k * kT, ld, di);
  tile_zero(ak);
  tile_zero(ai);
  for (int q = kb; q < k; ++q) {
    if (q > kb) __syncthreads();
    tk.stage(P[0]);
    if (below) ti.stage(P[1]);
    __syncthreads();
    if (q + 1 < k) {
      tk.fetch(rowk + (int64_t)(q + 1) * kT, ld);
      if (below) ti.fetch(rowi + (int64_t)(q + 1) * kT, ld);
    }
    tile_mm_mfma<true>(P[0], P[0], ak);
    if (below) tile_mm_mfma<true>(P[1], P[0], ai);
  }
  tile_sub(dk, ak);
  tile_put_mfma(P[2], dk);
  __syncthreads();  // the tiles of the last step are read, P[2] is written
  const bool ok = chol_tile(P[2], P[3]);
  if (!below) {
    if (!ok && threadIdx.x == 0) info[0] = 1;
    store_diag(Lkk, ld, Dinv + (int64_t)k * kT * kT, P[2], P[3]);
    return;
  }
  tile_sub(di, ai);
  tile_put_mfma(P[1], di);
  __syncthreads();
  tile_zero(ai);
  tile_mm_mfma<false>(P[1], P[3], ai);
  tile_store_mfma(rowi + (int64_t)k * kT, ld, ai);
}

// A_ij -= sum_{k in [kb, kend)} L_ik L_jk^T for kend <= j <= i < nb
__global__ __launch_bounds__(256) void k_chol_trailing(double* __restrict__ A, int64_t ld, int kb,
                                                       int kend) {
  __shared__ double P0[kT][kP];
  __shared__ double P1[kT][kP];
  int ii, jj;
  tri_index(blockIdx.x, ii, jj);
  op_chol_update(A, ld, kend + ii, kend + jj, kb, kend, P0, P1);
}

// Two tile rows [r0, r0 + 2) by two tile columns [c0, c0 + 2) per workgroup
// (wave w owns tile (r0 + (w >> 1), c0 + (w & 1))), so that every tile
// staged in LDS feeds two output tiles: half the panel bytes per flop of the
// one-tile kernels.  Tiles past the matrix (tile row nb; for X, tile column
// kend) are neither read nor written.
// The four tiles of one k (a0, a1 the row operands, b0, b1 the column
// operands; null for a tile past the matrix) pass through registers: pf is
// loaded for step k + 1 while the matrix cores work on step k.
struct QuadTiles {
  double v[4][kT * kT / 256];
};

__device__ inline void quad_fetch(QuadTiles& pf, const double* __restrict__ a0,
                                  const double* __restrict__ a1, const double* __restrict__ b0,
                                  const double* __restrict__ b1, int64_t ld) {
  const double* src[4] = {a0, a1, b0, b1};
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    if (src[t] == nullptr) continue;  // uniform
#pragma unroll
    for (int q = 0; q < kT * kT / 256; ++q) {
      const int e = (int)threadIdx.x + 256 * q;
      pf.v[t][q] = src[t][(e >> 6) * ld + (e & 63)];
    }
  }
}

__device__ inline void quad_stage(double (*S)[kT][kP], const QuadTiles& pf, bool a1, bool b1) {
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    if ((t == 1 && !a1) || (t == 3 && !b1)) continue;  // uniform
#pragma unroll
    for (int q = 0; q < kT * kT / 256; ++q) {
      const int e = (int)threadIdx.x + 256 * q;
      S[t][e >> 6][e & 63] = pf.v[t][q];
    }
  }
}

// A_ij -= sum_{k in [kb, kend)} L_ik L_jk^T for kend <= j <= i < nb, a 2 x 2
// block of tiles per workgroup (block pair (I, J), I >= J, from blockIdx.x)
__global__ __launch_bounds__(256) void k_chol_trailing2(double* __restrict__ A, int64_t ld, int kb,
                                                        int kend, int nb) {
  __shared__ double S[4][kT][kP];
  int I, J;
  tri_index(blockIdx.x, I, J);
  const int i0 = kend + 2 * I, j0 = kend + 2 * J;
  const int w = threadIdx.x >> 6;
  const int i = i0 + (w >> 1), j = j0 + (w & 1);
  const bool live = i < nb && j <= i;  // uniform per wave
  d4 acc[4][4];
#pragma unroll
  for (int p = 0; p < 4; ++p)
#pragma unroll
    for (int q = 0; q < 4; ++q) acc[p][q] = d4{0.0, 0.0, 0.0, 0.0};
  const bool a1 = i0 + 1 < nb, b1 = j0 + 1 < nb;
  QuadTiles pf;
  const double* ai = A + (int64_t)i0 * kT * ld;
  const double* aj = A + (int64_t)j0 * kT * ld;
  const int64_t row = (int64_t)kT * ld;
  quad_fetch(pf, ai + (int64_t)kb * kT, a1 ? ai + row + (int64_t)kb * kT : nullptr,
             aj + (int64_t)kb * kT, b1 ? aj + row + (int64_t)kb * kT : nullptr, ld);
  for (int k = kb; k < kend; ++k) {
    __syncthreads();  // the previous step is done with S
    quad_stage(S, pf, a1, b1);
    __syncthreads();
    if (k + 1 < kend) {
      const int64_t c = (int64_t)(k + 1) * kT;
      quad_fetch(pf, ai + c, a1 ? ai + row + c : nullptr, aj + c, b1 ? aj + row + c : nullptr, ld);
    }
    if (live) tile_mm_wave<true>(S[w >> 1], S[2 + (w & 1)], acc);
  }
  if (live) tile_sub_wave(A + (int64_t)i * kT * ld + (int64_t)j * kT, ld, acc);
}

// X_im -= sum_{k in [max(kb, m0), kend)} L_ik X_km for kend <= i < nb,
// m < kend, a 2 x 2 block of tiles per workgroup (rows i0, i0 + 1, columns
// m0, m0 + 1).  X_km = 0 for m > k, so the shared k range adds exact zeros
// to column m0 + 1.
__global__ __launch_bounds__(256) void k_trinv_trailing2(double* __restrict__ X,
                                                         const double* __restrict__ L, int64_t ld,
                                                         int kb, int kend, int nb) {
  __shared__ double S[4][kT][kP];
  const int mcols = (kend + 1) / 2;
  const int i0 = kend + 2 * (int)(blockIdx.x / mcols), m0 = 2 * (int)(blockIdx.x % mcols);
  const int w = threadIdx.x >> 6;
  const int i = i0 + (w >> 1), m = m0 + (w & 1);
  const bool live = i < nb && m < kend;  // uniform per wave
  d4 acc[4][4];
#pragma unroll
  for (int p = 0; p < 4; ++p)
#pragma unroll
    for (int q = 0; q < 4; ++q) acc[p][q] = d4{0.0, 0.0, 0.0, 0.0};
  const bool a1 = i0 + 1 < nb, b1 = m0 + 1 < kend;
  const int k0 = m0 > kb ? m0 : kb;
  QuadTiles pf;
  const double* li = L + (int64_t)i0 * kT * ld;  // row operands L_ik, L_(i+1)k
  const double* xm = X + (int64_t)m0 * kT;       // column operands X_km, X_k(m+1)
  const int64_t row = (int64_t)kT * ld;
  quad_fetch(pf, li + (int64_t)k0 * kT, a1 ? li + row + (int64_t)k0 * kT : nullptr,
             xm + (int64_t)k0 * row, b1 ? xm + (int64_t)k0 * row + kT : nullptr, ld);
  for (int k = k0; k < kend; ++k) {
    __syncthreads();  // the previous step is done with S
    quad_stage(S, pf, a1, b1);
    __syncthreads();
    if (k + 1 < kend) {
      const int64_t c = (int64_t)(k + 1) * kT, r = (int64_t)(k + 1) * row;
      quad_fetch(pf, li + c, a1 ? li + row + c : nullptr, xm + r, b1 ? xm + r + kT : nullptr, ld);
    }
    if (live) tile_mm_wave<false>(S[w >> 1], S[2 + (w & 1)], acc);
  }
  if (live) tile_sub_wave(X + (int64_t)i * kT * ld + (int64_t)m * kT, ld, acc);
}

// Tile rows [kb, kend) of X, one workgroup per tile column m < kend:
//   X_km = Dinv_k (X_km - sum_{k' in [max(kb, m), k)} L_kk' X_k'm)
// One launch for the block's 4 rows, which depend on each other, instead of two
// per row (15 us each): 43 to 52 us.
__global__ __launch_bounds__(256) void k_trinv_block(double* __restrict__ X,
                                                     const double* __restrict__ L, int64_t ld,
                                                     int kb, int kend,
                                                     const double* __restrict__ Dinv) {
  __shared__ double P0[kT][kP];
  __shared__ double P1[kT][kP];
  const int m = blockIdx.x;
  const int k0 = m > kb ? m : kb;
  for (int k = k0; k < kend; ++k) {
    if (k > k0) op_trinv_update(X, L, ld, k, m, k0, k, P0, P1);
    op_trinv_scale(X, ld, k, m, Dinv, P0, P1);
  }
}

// X_im -= sum_{k in [max(kb, m), kend)} L_ik X_km for kend <= i < nb, m < kend
// (X_km = 0 for m > k)
__global__ __launch_bounds__(256) void k_trinv_trailing(double* __restrict__ X,
                                                        const double* __restrict__ L, int64_t ld,
                                                        int kb, int kend) {
  __shared__ double P0[kT][kP];
  __shared__ double P1[kT][kP];
  const int m = blockIdx.x % kend;
  const int i = kend + blockIdx.x / kend;
  op_trinv_update(X, L, ld, i, m, m > kb ? m : kb, kend, P0, P1);
}

__global__ void k_identity(double* __restrict__ X, int64_t ld, int n) {
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < (int64_t)n * n;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t r = e / n, c = e % n;
    X[r * ld + c] = r == c ? 1.0 : 0.0;
  }
}

// Xt = X^T; the diagonal tiles of L, until now in Xt, go to A
__global__ __launch_bounds__(256) void k_transpose(const double* __restrict__ X, double* Xt,
                                                   double* __restrict__ A, int64_t ld) {
  __shared__ double P0[kT][kP];
  if (blockIdx.x == blockIdx.y) {
    const int64_t t = (int64_t)blockIdx.x * kT * (ld + 1);
    for (int e = threadIdx.x; e < kT * kT; e += blockDim.x)
      A[t + (e >> 6) * ld + (e & 63)] = Xt[t + (e >> 6) * ld + (e & 63)];
  }
  op_transpose(X, Xt, ld, blockIdx.y, blockIdx.x, P0);
}

// ---- many small matrices: one workgroup per system, the same schedule -----------

__global__ __launch_bounds__(256) void k_factor_small(double* __restrict__ A,
                                                      double* __restrict__ X,
                                                      double* __restrict__ Xt,
                                                      double* __restrict__ Dinv,
                                                      int* __restrict__ info,
                                                      const CoarseSys* __restrict__ sys,
                                                      const int* __restrict__ list) {
  __shared__ double P0[kT][kP];
  __shared__ double P1[kT][kP];
  const CoarseSys S = sys[list[blockIdx.x]];
  const int n = S.n, nb = n / kT;
  double* a = A + S.moff;
  double* x = X + S.moff;
  double* xt = Xt + S.moff;
  double* dinv = Dinv + S.doff;
  for (int kb = 0; kb < nb; kb += kKB) {
    const int kend = kb + kKB < nb ? kb + kKB : nb;
    for (int k = kb; k < kend; ++k) {
      op_chol_diag(a, n, k, dinv, info, P0, P1);
      for (int i = k + 1; i < nb; ++i) op_panel(a, n, k, i, dinv, P0, P1);
      for (int j = k + 1; j < kend; ++j)
        for (int i = j; i < nb; ++i) op_chol_update(a, n, i, j, k, k + 1, P0, P1);
    }
    for (int j = kend; j < nb; ++j)
      for (int i = j; i < nb; ++i) op_chol_update(a, n, i, j, kb, kend, P0, P1);
  }
  __syncthreads();
  for (int64_t e = threadIdx.x; e < (int64_t)n * n; e += blockDim.x)
    x[e] = (e / n) == (e % n) ? 1.0 : 0.0;
  for (int kb = 0; kb < nb; kb += kKB) {
    const int kend = kb + kKB < nb ? kb + kKB : nb;
    for (int k = kb; k < kend; ++k) {
      for (int m = 0; m <= k; ++m) op_trinv_scale(x, n, k, m, dinv, P0, P1);
      for (int i = k + 1; i < kend; ++i)
        for (int m = 0; m <= k; ++m) op_trinv_update(x, a, n, i, m, k, k + 1, P0, P1);
    }
    for (int i = kend; i < nb; ++i)
      for (int m = 0; m < kend; ++m) op_trinv_update(x, a, n, i, m, m > kb ? m : kb, kend, P0, P1);
  }
  for (int bi = 0; bi < nb; ++bi)
    for (int bj = 0; bj < nb; ++bj) op_transpose(x, xt, n, bi, bj, P0);
}

// ---- per-application kernels ------------------------------------------------------

// One particle's entries of a vector: the three translational ones, and with D =
// 6 the angular ones (from 3N on).
template <int D>
__device__ inline int64_t entry(int64_t i, int k, int64_t N) {
  return k < 3 ? 3 * i + k : 3 * N + 3 * i + (k - 3);
}

// y = B_i x or B_i^T x for the D x D block of particle i
template <int D>
__device__ inline void block_times(const double* __restrict__ B, int64_t i, int transpose,
                                   const double x[D], double y[D]) {
  const double* b = B + (int64_t)D * D * i;
#pragma unroll
  for (int r = 0; r < D; ++r) {
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < D; ++k) s += (transpose ? b[D * k + r] : b[D * r + k]) * x[k];
    y[r] = s;
  }
}

// cvec[3c+a] = scale[c] * sum over the particles of cell c of v[3i+a]; one
// wave per cell, lanes stride the cell's sorted list, fixed-order butterfly.
// D = 0: v = in.  D = 3, 6: v = B_i in or B_i^T in, which also goes to `out`
// (every particle is in one cell); the blocks in a launch of their own cost 5 us
// more (32768 particles).
template <int D>
__global__ __launch_bounds__(256) void k_coarse_restrict(const double* in, const double* B,
                                                         int transpose, int64_t N, double* out,
                                                         const int* __restrict__ perm,
                                                         const int* __restrict__ start,
                                                         const double* __restrict__ scale, int C,
                                                         double* __restrict__ cvec) {
  const int lane = threadIdx.x & 63;
  const int c = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (c >= C) return;  // uniform per wave
  double s0 = 0.0, s1 = 0.0, s2 = 0.0;
  for (int k = start[c] + lane; k < start[c + 1]; k += 64) {
    const int64_t i = perm[k];
    constexpr int M = D > 0 ? D : 3;
    double v[M];
#pragma unroll
    for (int q = 0; q < M; ++q) v[q] = in[entry<M>(i, q, N)];
    if constexpr (D > 0) {
      double t[M];
      block_times<D>(B, i, transpose, v, t);
#pragma unroll
      for (int q = 0; q < M; ++q) {
        v[q] = t[q];
        out[entry<M>(i, q, N)] = t[q];
      }
    }
    s0 += v[0];
    s1 += v[1];
    s2 += v[2];
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    s0 += __shfl_xor(s0, o);
    s1 += __shfl_xor(s1, o);
    s2 += __shfl_xor(s2, o);
  }
  if (lane == 0) {
    cvec[3 * c] = scale[c] * s0;
    cvec[3 * c + 1] = scale[c] * s1;
    cvec[3 * c + 2] = scale[c] * s2;
  }
}

// y[r] = sum_m T_s[lr][m] x[r0 + m] - x[r] over the system's rows, m <= lr
// (lower) or m >= lr (upper), m < 3 C_s; r = r0 + lr with r0 = 3 c0 of the
// row's system s; one workgroup per row, fixed-order reduction.
__global__ __launch_bounds__(256) void k_coarse_gemv(const double* __restrict__ T,
                                                     const CoarseSys* __restrict__ sys,
                                                     const int* __restrict__ row_sys, int lower,
                                                     const double* __restrict__ x,
                                                     double* __restrict__ y) {
  __shared__ double red[256];
  const int r = blockIdx.x;
  const CoarseSys S = sys[row_sys[r]];
  const int r0 = 3 * S.c0, lr = r - r0;
  const int m0 = lower ? 0 : lr, m1 = lower ? lr + 1 : 3 * S.C;
  const double* row = T + S.moff + (int64_t)lr * S.n;
  const double* xs = x + r0;
  double s = 0.0;
  for (int m = m0 + (int)threadIdx.x; m < m1; m += 256) s = __builtin_fma(row[m], xs[m], s);
  red[threadIdx.x] = s;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) y[r] = red[0] - x[r];
}

// The same with one wave per row (short rows: many small systems);
// fixed-order butterfly.
__global__ __launch_bounds__(256) void k_coarse_gemv_wave(const double* __restrict__ T,
                                                          const CoarseSys* __restrict__ sys,
                                                          const int* __restrict__ row_sys,
                                                          int rows, int lower,
                                                          const double* __restrict__ x,
                                                          double* __restrict__ y) {
  const int lane = threadIdx.x & 63;
  const int r = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (r >= rows) return;  // uniform per wave
  const CoarseSys S = sys[row_sys[r]];
  const int r0 = 3 * S.c0, lr = r - r0;
  const int m0 = lower ? 0 : lr, m1 = lower ? lr + 1 : 3 * S.C;
  const double* row = T + S.moff + (int64_t)lr * S.n;
  const double* xs = x + r0;
  double s = 0.0;
  for (int m = m0 + lane; m < m1; m += 64) s = __builtin_fma(row[m], xs[m], s);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
  if (lane == 0) y[r] = s - x[r];
}

// out[k] = in[k] + scale[c] * y[3c + a] for k = 3i + a < 3N (c = cell of i),
// out[k] = rest[k] beyond (in and rest may equal out)
__global__ void k_coarse_prolong(const double* in, const double* rest,
                                 const int* __restrict__ cell_of,
                                 const double* __restrict__ scale, const double* __restrict__ y,
                                 int64_t n3, int64_t n, double* out) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  if (k < n3) {
    const int64_t i = k / 3;
    const int c = cell_of[i];
    out[k] = in[k] + scale[c] * y[3 * c + (int)(k - 3 * i)];
  } else {
    out[k] = rest[k];
  }
}

// The same followed by out = B_i (.) or B_i^T (.) per particle, D x D blocks (one
// launch instead of two); with D = 3 entries from 3N on pass through.
template <int D>
__global__ void k_coarse_prolong_blocks(const double* in, const int* __restrict__ cell_of,
                                        const double* __restrict__ scale,
                                        const double* __restrict__ y,
                                        const double* __restrict__ B, int transpose, int64_t N,
                                        int64_t n, double* out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < N) {
    const int c = cell_of[i];
    double v[D], t[D];
#pragma unroll
    for (int q = 0; q < D; ++q) {
      v[q] = in[entry<D>(i, q, N)];
      if (q < 3) v[q] += scale[c] * y[3 * c + q];
    }
    block_times<D>(B, i, transpose, v, t);
#pragma unroll
    for (int q = 0; q < D; ++q) out[entry<D>(i, q, N)] = t[q];
  }
  if (D == 3) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t k = 3 * N + i; k < n; k += stride) out[k] = in[k];
  }
}

inline unsigned blocks_for(int64_t n, int nt) { return (unsigned)((n + nt - 1) / nt); }
// Workgroups of a grid-stride launch: a dispatch holds at most 2^32 work-items.
inline unsigned stride_blocks(int64_t n, int per_block) {
  const int64_t b = (n + per_block - 1) / per_block;
  return (unsigned)(b < (int64_t)1 << 20 ? b : (int64_t)1 << 20);
}

}  // namespace

void launch_coarse_gather(const void* rec, const int* perm, int64_t N, void* out, bool fp64,
                          hipStream_t s) {
  if (N <= 0) return;
  if (fp64)
    hipLaunchKernelGGL(k_gather_records<double4>, dim3(blocks_for(N, 256)), dim3(256), 0, s,
                       static_cast<const double4*>(rec), perm, N, static_cast<double4*>(out));
  else
    hipLaunchKernelGGL(k_gather_records<float4>, dim3(blocks_for(N, 256)), dim3(256), 0, s,
                       static_cast<const float4*>(rec), perm, N, static_cast<float4*>(out));
  LM_HIP(hipGetLastError());
}

void launch_coarse_matrix(const void* rec, bool fp64, const int* start, const double* scale,
                          const CoarseSys* sys, const int64_t* pair_off, int nsys, int64_t npairs,
                          double* Mc, int64_t total, hipStream_t s) {
  launch_zero(Mc, total, s);
  if (npairs > 0) {
    if (fp64)
      hipLaunchKernelGGL((k_coarse_matrix<double, double4>), dim3(stride_blocks(npairs, 4)),
                         dim3(256), 0, s, static_cast<const double4*>(rec), start, scale, sys,
                         pair_off, nsys, npairs, Mc);
    else
      hipLaunchKernelGGL((k_coarse_matrix<float, float4>), dim3(stride_blocks(npairs, 4)), dim3(256),
                         0, s, static_cast<const float4*>(rec), start, scale, sys, pair_off, nsys,
                         npairs, Mc);
    LM_HIP(hipGetLastError());
  }
  hipLaunchKernelGGL(k_pad_identity, dim3(nsys), dim3(64), 0, s, Mc, sys);
  LM_HIP(hipGetLastError());
}

void launch_coarse_factor(double* A, double* X, double* Xt, double* Dinv, int* info, int64_t ld,
                          int n, hipStream_t s, const SideStream& side) {
  const int nb = n / kT;
  hipStream_t x = side.stream;
  // X may still be read by work queued on s before this call.
  LM_HIP(hipEventRecord(side.block, s));
  LM_HIP(hipStreamWaitEvent(x, side.block, 0));
  hipLaunchKernelGGL(k_identity, dim3(stride_blocks((int64_t)n * n, 256)), dim3(256), 0, x, X, ld,
                     n);
  for (int kb = 0; kb < nb; kb += kKB) {
    const int kend = kb + kKB < nb ? kb + kKB : nb;
    for (int k = kb; k < kend; ++k)
      hipLaunchKernelGGL(k_chol_column, dim3(nb - k), dim3(256), 0, s, A, ld, kb, k,
                         Xt + (int64_t)k * kT * (ld + 1), Dinv, info);
    // Columns [kb, kend) of L and their diagonal inverses are final here (the
    // diagonal tiles of L are in Xt).  Block kb of X reads nothing else of L,
    // and the trailing update of L below writes only columns >= kend.
    LM_HIP(hipEventRecord(side.block, s));
    LM_HIP(hipStreamWaitEvent(x, side.block, 0));
    hipLaunchKernelGGL(k_trinv_block, dim3(kend), dim3(256), 0, x, X, A, ld, kb, kend, Dinv);
    const int T = nb - kend;
    const int64_t xtiles = (int64_t)T * kend;
    if (xtiles >= kQuadTiles)
      hipLaunchKernelGGL(k_trinv_trailing2, dim3((unsigned)((int64_t)((T + 1) / 2) * ((kend + 1) / 2))),
                         dim3(256), 0, x, X, A, ld, kb, kend, nb);
    else if (T > 0)
      hipLaunchKernelGGL(k_trinv_trailing, dim3((unsigned)xtiles), dim3(256), 0, x, X, A, ld, kb, kend);
    const int64_t tiles = (int64_t)T * (T + 1) / 2, T2 = (T + 1) / 2;
    if (tiles >= kQuadTiles)
      hipLaunchKernelGGL(k_chol_trailing2, dim3((unsigned)(T2 * (T2 + 1) / 2)), dim3(256), 0, s, A,
                         ld, kb, kend, nb);
    else if (T > 0)
      hipLaunchKernelGGL(k_chol_trailing, dim3((unsigned)tiles), dim3(256), 0, s, A, ld, kb, kend);
  }
  LM_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_transpose, dim3(nb, nb), dim3(256), 0, x, X, Xt, A, ld);
  LM_HIP(hipGetLastError());
  LM_HIP(hipEventRecord(side.done, x));
  LM_HIP(hipStreamWaitEvent(s, side.done, 0));
}

void launch_coarse_factor_small(double* A, double* X, double* Xt, double* Dinv, int* info,
                                const CoarseSys* sys, const int* list, int count, hipStream_t s) {
  if (count <= 0) return;
  hipLaunchKernelGGL(k_factor_small, dim3(count), dim3(256), 0, s, A, X, Xt, Dinv, info, sys, list);
  LM_HIP(hipGetLastError());
}

void launch_coarse_apply(const double* T, const CoarseSys* sys, const int* row_sys, int rows,
                         int max_row, bool lower, const double* in, double* out, int64_t N,
                         int64_t n, const int* perm, const int* start, const int* cell_of,
                         const double* scale, int C, double* cvec, double* yvec,
                         const ParticleBlocks& before, const ParticleBlocks& after,
                         hipStream_t s) {
  for (const ParticleBlocks* b : {&before, &after})
    if (b->B != nullptr && b->dim != 3 && !(b->dim == 6 && n == 6 * N))
      throw Error("[libmobility_amd] 6x6 preconditioner blocks need linear and angular entries");
  const dim3 cells(blocks_for(C, 4)), block(256);
  const int bd = before.B ? before.dim : 0, ad = after.B ? after.dim : 0;
  auto restrict_with = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, cells, block, 0, s, in, before.B, before.transpose, N, out, perm,
                       start, scale, C, cvec);
  };
  if (bd == 0) restrict_with(k_coarse_restrict<0>);
  else if (bd == 3) restrict_with(k_coarse_restrict<3>);
  else restrict_with(k_coarse_restrict<6>);
  LM_HIP(hipGetLastError());
  if (max_row <= kWaveRowMax)
    hipLaunchKernelGGL(k_coarse_gemv_wave, dim3(blocks_for(rows, 4)), block, 0, s, T, sys, row_sys,
                       rows, lower ? 1 : 0, cvec, yvec);
  else
    hipLaunchKernelGGL(k_coarse_gemv, dim3(rows), block, 0, s, T, sys, row_sys, lower ? 1 : 0,
                       cvec, yvec);
  LM_HIP(hipGetLastError());
  const double* trans = bd > 0 ? out : in;  // translational entries so far, and the rest
  const double* rest = bd == 6 ? out : in;
  if (ad == 0) {
    hipLaunchKernelGGL(k_coarse_prolong, dim3(blocks_for(n, 256)), block, 0, s, trans, rest,
                       cell_of, scale, yvec, 3 * N, n, out);
  } else {
    if (bd > 0) throw Error("[libmobility_amd] coarse level: blocks on both sides");
    auto prolong_with = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3(blocks_for(N, 256)), block, 0, s, in, cell_of, scale, yvec,
                         after.B, after.transpose, N, n, out);
    };
    if (ad == 3) prolong_with(k_coarse_prolong_blocks<3>);
    else prolong_with(k_coarse_prolong_blocks<6>);
  }
  LM_HIP(hipGetLastError());
}

}  // namespace lm
