// Cell sort internals shared with the gravity step.
#pragma once

#include "pm_common.h"

namespace pm {
namespace sort {

int check_sort_args(int64_t n, const int32_t* mesh_shape, const int32_t* brick);
size_t workspace_bytes(int64_t n, const int32_t* mesh_shape, const int32_t* brick);
int sort_cells(const int16_t* pmid, const float* disp, const uint8_t* valid, int64_t n,
               const int32_t* mesh_shape, float cell_size, const int32_t* brick, int32_t* perm,
               int32_t* bin_offsets, int16_t* pmid_s, float* disp_s, Arena& ws, hipStream_t s);

// The tile kernels' particle record (16 bytes, one vector load): the CIC fractions f[3] of the
// base cell (bit for bit what pm_gravity.hip's base_frac gives) and rec_bits of the base cell's place
// (lx, ly, lz) in its brick: the offset of that cell in a tile of (b0+1) x (b1+1) rows of b2 + 2
// words (at most 2^15 words), and in the top bit whether it is in the brick's last z plane.
__host__ __device__ inline uint32_t rec_bits(int lx, int ly, int lz, int b1, int b2) {
  return (uint32_t)((lx * (b1 + 1) + ly) * (b2 + 2) + lz) | (lz == b2 - 1 ? 0x80000000u : 0u);
}
__device__ __forceinline__ int rec_cell(uint32_t bits) { return (int)(bits & 0x7fffffffu); }
__device__ __forceinline__ bool rec_top(uint32_t bits) { return (bits >> 31) != 0; }

// Output of the bucketing: bins (num_bricks + 2 offsets, the last bucket holding invalid
// particles), perm, and either rec (above) or the payload pmid / disp / valid gathered into bucket
// order.
struct Sorted {
  int32_t* bins = nullptr;
  int32_t* perm = nullptr;
  float4* rec = nullptr;
  int16_t* pmid = nullptr;
  float* disp = nullptr;
  uint8_t* valid = nullptr;
};

// Unstable bucketing by the same key (gravity step).  ptcl_grid (may be null) is the Lagrangian
// grid the particles were generated on, a hint that selects grid-block chunks (speed only).
// count (bucket_count_len words, 16-byte aligned) and partial (bucket_partials of that) are
// scratch; cleared: count is zero already.
int64_t bucket_count_len(const int32_t* mesh_shape, const int32_t* brick);
int64_t bucket_partials(int64_t len);
size_t bucket_workspace_bytes(const int32_t* mesh_shape, const int32_t* brick);
int bucket_cells(const int16_t* pmid, const float* disp, const uint8_t* valid, int64_t n, const int32_t* mesh_shape,
                 float cell_size, const int32_t* brick, const int32_t* ptcl_grid, const Sorted& out, int32_t* count,
                 int32_t* partial, bool cleared, hipStream_t s);

// pm_init: resolve the current device's address of the allocation-free binning scratch.
int init_noalloc_scratch();

}  // namespace sort
}  // namespace pm
