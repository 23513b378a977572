// Particles of one system into the cells of a grid, on the device (the
// preconditioner's neighbour search and its coarse level).  Systems of an
// ensemble are small and many: their grids are built on the host.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace lm {

// Cell of a coordinate along axis k, 0 where ext is 0: floor((x - lo) / edge), or
// with by_edge = 0 floor((x - lo) / ext * g), in both cases cut to [0, g).
struct CellGrid {
  double lo[3], ext[3], edge[3];
  int g[3];
  int by_edge;
};

// Per block the corners of its records' box: host[6 b] lo, host[6 b + 3] hi.
constexpr int kBoxBlocks = 64;
void launch_record_box(const double4* rec, int64_t N, double* host, hipStream_t s);

// Raw cell ids (x-major) and the cells' populations (zeroed here).
void launch_cell_count(const double4* rec, int64_t N, const CellGrid& grid, int* raw, int* count,
                       int ncell, hipStream_t s);
// Exclusive sums of count[0 .. ncell): start64 (ncell + 1), or with `compact` the
// non-empty cells numbered in raw order and their start32 (cells + 1); host: the
// number of non-empty cells and the largest population.
struct CellScan {
  const int* count;
  int ncell;
  int64_t* start64;
  int* compact;
  int* start32;
  int* host;
};
void launch_cell_scan(const CellScan& a, hipStream_t s);
// The particles cell by cell, in no particular order within a cell (count is
// used up).
void launch_cell_fill64(const int* raw, int64_t N, const int64_t* start, int* count, int* list,
                        hipStream_t s);
void launch_cell_fill32(const int* raw, int64_t N, const int* compact, const int* start, int* count,
                        int* list, hipStream_t s);
// perm: the list with ascending particles in each cell; cell_of: compact ids;
// scale[c] = 1 / sqrt(population).  Every particle is ranked against its whole
// cell: for cells of up to kCellRankMax.
constexpr int kCellRankMax = 4096;
void launch_cell_order(const int* raw, int64_t N, const int* compact, const int* start, int C,
                       const int* list, int* perm, int* cell_of, double* scale, hipStream_t s);

}  // namespace lm
