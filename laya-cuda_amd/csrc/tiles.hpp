// Tile walk shared by the GEMM kernels: which output tile a workgroup takes.
#pragma once

#include "common.hpp"

namespace laya {

// Workgroup tile coordinates.  Workgroups are dealt to the 8 XCDs round-robin by linear dispatch
// id, so consecutive ids run on different L2s.  When the workgroup count allows, the logical index
// is laid out instead so that each XCD gets one contiguous share, decoded split-major: with split-K
// an XCD works on whole K-slices (or an equal part of one) and fetches only those slices of both
// operands.  Inside a slice, tiles are walked so the operand that is larger in HBM is fetched into
// one L2 once: with many rows (A larger), groups of 4 tile rows with the column index outer; with
// fewer rows than columns (B, the weights, larger), whole tile columns one after another.
// Coordinates of logical tile `id` (0 .. nx ny nz - 1): the workgroup with linear dispatch id `id`
// in the order above.
__device__ __forceinline__ void tile_of(int id, int nx, int ny, int nz, bool rows_major, int* x, int* y, int* z) {
  const int per_z = nx * ny, total = per_z * nz;
  if (total % 8) {
    *x = id % nx;
    *y = (id / nx) % ny;
    *z = id / per_z;
    return;
  }
  const int l = (id % 8) * (total / 8) + id / 8;
  *z = l / per_z;
  const int t = l - *z * per_z;
  if (rows_major) {
    constexpr int G = 4;
    const int group = t / (G * nx), first = group * G, size = min(G, ny - first), in = t - group * G * nx;
    *y = first + in % size;
    *x = in / size;
  } else {
    *x = t / ny;
    *y = t - *x * ny;
  }
}
__device__ __forceinline__ void tile_coords(int nx, int ny, int nz, bool rows_major, int* x, int* y, int* z) {
  tile_of(blockIdx.x + nx * (blockIdx.y + ny * blockIdx.z), nx, ny, nz, rows_major, x, y, z);
}

// Tile of workgroup `id` of few-row problems: each XCD gets an equal share of whatever count there
// is (one more tile on the first few), walked split by split and whole tile columns at a time, so a
// weight panel is fetched into one L2 and the row tiles that share it run there together.
__device__ __forceinline__ void tile_of_even(int id, int nx, int ny, int nz, int* x, int* y, int* z) {
  const int total = nx * ny * nz, share = total >> 3, rest = total & 7, xcd = id & 7;
  const int l = xcd * share + min(xcd, rest) + (id >> 3);
  *z = l / (nx * ny);
  const int t = l - *z * nx * ny;
  *x = t / ny;
  *y = t - *x * ny;
}

}  // namespace laya
