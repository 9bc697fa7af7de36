// The single-device PM force step and its reverse (force VJP).
//
// Forward (nbody/gravity.py:786-814 on the streamed single-device branch :597-606, 506-543):
//   1. cell sort (pm_sort.hip) and a gather of the particle payload into key order;
//   2. CIC scatter of v_p = valid * N_m/N_p from sorted particles (spatially coherent atomics);
//   3. z pass r2c with S = (rho - 1) * (1.5 Omega_m) fused into the load;
//   4. y pass forward;
//   5. x pass forward, mask x (-1/k^2), then two inverse x transforms in registers:
//        A <- IFFT_x(phi),  B <- IFFT_x(-i k_x phi)
//   6. y pass inverse on A with two outputs: A <- IFFT_y(A), C <- IFFT_y(-i k_y A);
//      y pass inverse on B;
//   7. z pass c2r of B -> F_x, C -> F_y, (-i k_z) A -> F_z  (1/N normalisation fused);
//   8. CIC gather of (F_x, F_y, F_z) from sorted particles, written back through the
//      permutation in caller order.
// The derivative operators commute with the transforms along the other axes, so the three
// inverse transforms of the reference (one per component, :535-543) share their x and y
// passes: 4R + 14C bytes of mesh traffic instead of 4R + 20C.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "pm_common.h"
#include "pm_fft_launch.h"
#include "pm_sort.h"

namespace pm {
namespace grav {
namespace {

constexpr int kBlock = 256;

__global__ void k_fill(float* __restrict__ p, int64_t n, float v) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    p[i] = v;
}

// dst = src for a mesh handed back to the caller: 16-byte accesses, four in flight per
// thread (a device-to-device hipMemcpyAsync of the 4 GiB density at 1024^3 ran at 2.1 TB/s)
__global__ void __launch_bounds__(kBlock) k_copy_mesh(const float* __restrict__ src, float* __restrict__ dst,
                                                      int64_t n) {
  const int64_t n4 = n / 4;
  const int64_t stride = (int64_t)gridDim.x * kBlock;
  const float4* s4 = reinterpret_cast<const float4*>(src);
  float4* d4 = reinterpret_cast<float4*>(dst);
  int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  for (; i + 3 * stride < n4; i += 4 * stride) {
    const float4 a = s4[i], b = s4[i + stride], c = s4[i + 2 * stride], d = s4[i + 3 * stride];
    d4[i] = a;
    d4[i + stride] = b;
    d4[i + 2 * stride] = c;
    d4[i + 3 * stride] = d;
  }
  for (; i < n4; i += stride) d4[i] = s4[i];
  for (int64_t j = 4 * n4 + (int64_t)blockIdx.x * kBlock + threadIdx.x; j < n; j += stride) dst[j] = src[j];
}

__global__ void __launch_bounds__(kBlock) k_scatter_sorted(const int16_t* __restrict__ pmid,
                                                           const float* __restrict__ disp,
                                                           const uint8_t* __restrict__ valid, int64_t n,
                                                           float val, Geom g, float* __restrict__ mesh) {
  int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= n || !valid[j]) return;
  AxisCic ax[3];
  particle_cic(g, pmid, disp, j, ax);
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    int64_t flat;
    corner_index(g, ax, c, flat);
    atomic_add_f32(mesh + flat, val * corner_weight(ax, c));
  }
}

__global__ void __launch_bounds__(kBlock) k_gather3_sorted(const int16_t* __restrict__ pmid,
                                                           const float* __restrict__ disp,
                                                           const uint8_t* __restrict__ valid,
                                                           const int32_t* __restrict__ perm, int64_t n,
                                                           Geom g, const float* __restrict__ fx,
                                                           const float* __restrict__ fy,
                                                           const float* __restrict__ fz,
                                                           float* __restrict__ acc) {
  int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= n) return;
  float r[3] = {0.f, 0.f, 0.f};
  if (valid[j]) {
    AxisCic ax[3];
    particle_cic(g, pmid, disp, j, ax);
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      int64_t flat;
      corner_index(g, ax, c, flat);
      float w = corner_weight(ax, c);
      r[0] = r[0] + fx[flat] * w;
      r[1] = r[1] + fy[flat] * w;
      r[2] = r[2] + fz[flat] * w;
    }
  }
  int64_t i = perm[j];
  acc[i * 3 + 0] = r[0];
  acc[i * 3 + 1] = r[1];
  acc[i * 3 + 2] = r[2];
}

// ----------------------------------------------------------------------------------------
// Brick-tiled CIC on sorted particles.  The mesh is tiled by bricks of (BX,BY,BZ) cells; the
// cell sort groups particles by the brick of their base (corner-0) cell, so every corner a
// particle touches lies in its brick's tile extended by one cell on the upper side.  One
// workgroup walks a column of bricks (fixed x and y brick coordinates) along z.
//
// Particles come as 16-byte records (pm_sort.h): the fractions and the tile offset of the base cell,
// one vector load instead of six scalar ones and no division per particle (512^3 particles on a 1024^3
// mesh: scatter 2.26 -> 1.54 ms, gather 4.95 -> 4.71 ms).
//
// Scatter (owner computes): a run of a column's bricks is accumulated one after the other into an
// LDS tile of (BX+1)(BY+1)(BZ+1) 64-bit cells (int64 fixed point; the CIC entry points' are float64) with
// LDS atomics.  The tile's upper z
// plane belongs to the next brick of the column and is carried to it inside LDS; the lower plane
// of the run's first brick gets the carry of the brick below (the one above the periodic
// wrap for the first) from that brick's own particles in its last z plane, read a second time.
// So every owned cell is complete when it is stored, once, with plain stores (no zero fill, no
// global atomics), and a column can be cut into runs for different workgroups: with whole
// columns a 128^3 mesh has 64 of them.  The upper x and y planes go to z-contiguous plane buffers
// (XS, YS), which are added to the lower x/y planes of the neighbouring columns later (pull,
// fixed order: deterministic).
// Gather: a run is walked downward in z.  Each force component's tile rows z in [0, BZ)
// are read as aligned rows; the z = BZ plane is the lower plane of the brick above, kept in
// LDS from the previous step (read directly for the first), so no row costs a second cache line.
constexpr int kTileMaxFloats = 19100;  // gather f32 tile: (32+1)*(16+1)*(32+2) = 19074 fits
constexpr int kTileMaxWords = 9900;    // scatter 64-bit tile: (16+1)*(16+1)*(32+2) = 9826 (78.6 KB: 2 WG/CU)
constexpr int kPlaneMax = 1100;        // (b0+1)*(b1+1) cells of one z plane of a tile
// The force step's scatter accumulation is exact 64-bit fixed point (2^-32 units): gfx950's LDS integer atomics run
// an order of magnitude faster than its LDS float32 atomics, and integer sums are order independent,
// so the density is deterministic; each cell is rounded to float32 once when stored.
constexpr float kFix = 4294967296.0f;         // 2^32
constexpr float kUnfix = 2.3283064365386963e-10f;  // 2^-32

struct Bricks {
  int n[3];   // mesh shape
  int b[3];   // brick shape
  int nb[3];  // bricks per axis
};

inline Bricks make_bricks(const int32_t* mesh, const int32_t* brick) {
  Bricks k;
  for (int a = 0; a < 3; ++a) {
    k.n[a] = mesh[a];
    k.b[a] = brick[a];
    k.nb[a] = mesh[a] / brick[a];
  }
  return k;
}

inline bool tiled_ok(const int32_t* mesh, const int32_t* brick) {
  for (int a = 0; a < 3; ++a)
    if (brick[a] < 1 || mesh[a] % brick[a] != 0) return false;
  // LDS tile rows have a z pitch of b2 + 2 words
  const int64_t plane = (int64_t)(brick[0] + 1) * (brick[1] + 1);
  const int64_t words = plane * (brick[2] + 2);
  return words <= kTileMaxFloats && words <= kTileMaxWords && plane <= kPlaneMax;
}

inline bool is_brick(const Bricks& k, int x, int y, int z) { return k.b[0] == x && k.b[1] == y && k.b[2] == z; }

// Upper-plane buffers of the tiled scatter, z-contiguous:
//   XS[(col * (b1+1) + ly) * nz + z]  the x == b0 plane of column col (ly in [0, b1])
//   YS[(col * b0 + lx) * nz + z]      the y == b1 plane of column col (lx in [0, b0))
inline int64_t xs_floats(const Bricks& k) { return (int64_t)k.nb[0] * k.nb[1] * (k.b[1] + 1) * k.n[2]; }
inline int64_t ys_floats(const Bricks& k) { return (int64_t)k.nb[0] * k.nb[1] * k.b[0] * k.n[2]; }

// Workgroups are dispatched round-robin over the 8 XCDs; logical column q runs on workgroup
// (q % g8) * 8 + q / g8 so neighbouring columns (which share halo rows) share an L2.
__device__ __forceinline__ int column_of(int L, int G) {
  if (G % 8 != 0) return L;
  return (L % 8) * (G / 8) + L / 8;
}

// The column walks that read a tile plus its one-cell x/y halo (gather, displacement cotangent):
// XCD x (workgroups L with L % 8 == x) takes the columns cx in [x R, (x + 1) R), R = nb0 / 8, and
// visits them in patches of PX x 8 columns, patch after patch, so the workgroups an XCD runs at
// the same time (about 64) form a compact patch of the (cx, cy) plane and read the halo rows
// they share into one L2 at nearly the same time, instead of a 64-column strip whose x-halo
// rows are read again, long after, by the strip beside it.  Other shapes keep column_of.
__device__ __forceinline__ int patch_column_of(int L, int G, int nb0, int nb1) {
  const int R = nb0 / 8;
  const int PX = R < 8 ? R : 8;
  if (G % 8 != 0 || G != nb0 * nb1 || nb0 % 8 != 0 || nb1 % 8 != 0 || PX == 0 || R % PX != 0) return column_of(L, G);
  const int x = L % 8, j = L / 8;
  const int per = PX * 8;
  const int p = j / per, w = j - p * per;
  const int npy = nb1 / 8;
  const int pxi = p / npy, pyi = p - pxi * npy;
  const int cx = x * R + pxi * PX + w / 8;
  const int cy = pyi * 8 + (w & 7);
  return cx * nb1 + cy;
}

constexpr int kBatch = 8;  // independent loads kept in flight per thread in the runtime-shape tile loops

// Compile-time brick shape when BX > 0 (integer divisions by the tile extents become
// shifts/multiplies); BX = 0 reads the shape from the runtime descriptor.
//
// LDS tile layout: tile[(x * t1 + y) * pitch + z], z in [0, b2], pitch = b2 + 2, so every
// corner of a particle is its corner-0 address plus a compile-time offset, and rows are
// 8-byte aligned for float2 LDS stores when b2 is even.  The spare word z = b2 + 1 of each
// scatter row holds the z carry.
template <int BX, int BY, int BZ>
struct BrickShape {
  int b0, b1, b2;
  static constexpr bool kVec = BX > 0 && BZ % 4 == 0;
  // 8 x 8 x 16 bricks (small meshes) on 256 threads, the others on 512
  static constexpr int NT = BX == 8 ? 256 : 512;
  // particles of one brick processed per tile staging by the gathers: their results wait in LDS,
  // so each tile is read once per brick unless the brick holds more (~2x the mean occupancy at
  // 1/8 particle per cell).  1024 for the small bricks, one staging per brick at one particle per cell
  // (against 512: 128^3 particles on 128^3 53 -> 44 us, 64^3 on 64^3 20 -> 17 us; no different at 1/8 per
  // cell)
  static constexpr int CAP = BX == 8 ? 1024 : 2048;
  static constexpr int PPT = CAP / NT;
  // LDS tile sizes: gather (float), scatter (int64) and one z plane
  static constexpr int TF = BX ? (BX + 1) * (BY + 1) * (BZ + 2) : kTileMaxFloats;
  static constexpr int TW = BX ? (BX + 1) * (BY + 1) * (BZ + 2) : kTileMaxWords;
  static constexpr int PL = BX ? (BX + 1) * (BY + 1) : kPlaneMax;
  __device__ __forceinline__ explicit BrickShape(const Bricks& k)
      : b0(BX ? BX : k.b[0]), b1(BY ? BY : k.b[1]), b2(BZ ? BZ : k.b[2]) {}
  __device__ __forceinline__ int t0() const { return b0 + 1; }
  __device__ __forceinline__ int t1() const { return b1 + 1; }
  __device__ __forceinline__ int t2() const { return b2 + 1; }
  __device__ __forceinline__ int pitch() const { return b2 + 2; }
  __device__ __forceinline__ int rows() const { return (b0 + 1) * (b1 + 1); }
  __device__ __forceinline__ int tfloats() const { return (b0 + 1) * (b1 + 1) * (b2 + 2); }
  __device__ __forceinline__ int cell(int x, int y, int z) const { return (x * (b1 + 1) + y) * (b2 + 2) + z; }
  // offset of corner c relative to corner 0
  __device__ __forceinline__ int corner_off(int c) const {
    return ((c & 1) * (b1 + 1) + ((c >> 1) & 1)) * (b2 + 2) + ((c >> 2) & 1);
  }
};

// CIC weight of corner c from the fractional offsets, in the reference's product order
__device__ __forceinline__ float frac_weight(const float f[3], int c) {
  float wx = (c & 1) ? 1.f - fabsf(f[0] - 1.f) : 1.f - fabsf(f[0]);
  float wy = ((c >> 1) & 1) ? 1.f - fabsf(f[1] - 1.f) : 1.f - fabsf(f[1]);
  float wz = ((c >> 2) & 1) ? 1.f - fabsf(f[2] - 1.f) : 1.f - fabsf(f[2]);
  return wx * wy * wz;
}

// A tile's sum: the force step's fixed point, or (CIC) float64.  The CIC entry points take values of any
// range, so no common unit serves them: their deposits are the float32 products that float atomics
// would add, summed in float64, so that every cell is as good as its own deposits (ds_add_f64: 128^3
// particles on a 256^3 mesh in 36 us, as with the fixed point).
template <bool CIC>
using TileSum = std::conditional_t<CIC, double, unsigned long long>;

template <int BX, int BY, int BZ, bool CIC>
__global__ void __launch_bounds__((BrickShape<BX, BY, BZ>::NT)) k_scatter_columns(
    const float4* __restrict__ rec, const int32_t* __restrict__ bin_off, float val, Bricks k, int run,
    float* __restrict__ mesh, float* __restrict__ xs, float* __restrict__ ys, const float* __restrict__ vals,
    const float* __restrict__ vscale, const float* __restrict__ base) {
  using B_ = BrickShape<BX, BY, BZ>;
  using Sum = TileSum<CIC>;
  constexpr int NT = B_::NT;
  __shared__ __align__(16) Sum tile[B_::TW];
  // fixed point: per-particle values (sorted order) are brought to |v| <= 1 by vscale[0] and scaled
  // back on output; a constant value is used as it is
  const float vs = !CIC && vals ? vscale[0] : 1.f;
  const float us = !CIC && vals ? kUnfix / vs : kUnfix;
  auto unfix = [&](Sum x) {
    if constexpr (CIC)
      return (float)x;
    else
      return (float)(long long)x * us;
  };
  const B_ B(k);
  const int col = column_of(blockIdx.x, gridDim.x);
  const int cx = col / k.nb[1], cy = col - cx * k.nb[1];
  const int P = B.pitch(), rows = B.rows(), carry = B.b2 + 1, tf = B.tfloats();
  const int64_t n1 = k.n[1], n2 = k.n[2];
  const int bz0 = blockIdx.y * run, bz1 = min(k.nb[2], bz0 + run);
  const int32_t* off = bin_off + (int64_t)col * k.nb[2];
  for (int i = threadIdx.x; i < tf; i += NT) tile[i] = Sum(0);
  // Particles stream in chunks of NT * PPT in index order (the bricks' bins are contiguous).  The
  // loads of the next chunk are issued before the current one is accumulated, so they are in
  // flight across the flush between bricks.
  constexpr int PPT = 4;
  constexpr int64_t CH = (int64_t)NT * PPT;
  auto load = [&](float4* r, int64_t start, int64_t end) {  // clamped: unconditional (end > start somewhere)
#pragma unroll
    for (int q = 0; q < PPT; ++q) {
      const int64_t j = start + threadIdx.x + (int64_t)q * NT;
      r[q] = rec[j < end ? j : end - 1];
    }
  };
  auto add = [&](const float4& r, int64_t j, int c0, int c_begin) {  // corners c_begin .. 7 (4: the upper z plane)
    const float fr[3] = {r.x, r.y, r.z};
    const float v = vals ? vals[j] * vs : val;
#pragma unroll
    for (int c = 0; c < 8; ++c)
      if (c >= c_begin) {
        const float dep = v * frac_weight(fr, c);
        if constexpr (CIC)
          atomicAdd(&tile[c0 + B.corner_off(c)], (double)dep);
        else
          atomicAdd(&tile[c0 + B.corner_off(c)], (unsigned long long)__float2ll_rn(dep * kFix));
      }
  };
  const int64_t run0 = off[bz0], run1 = off[bz1];
  float4 raw[PPT];
  if (run1 > run0) load(raw, run0, run1);
  __syncthreads();
  {
    // the brick below the run: its last z plane's upper corners are the first brick's z = 0 plane
    const int bb = bz0 == 0 ? k.nb[2] - 1 : bz0 - 1;
    const int64_t h0 = off[bb], h1 = off[bb + 1];
    for (int64_t c0 = h0; c0 < h1; c0 += CH) {
      float4 h[PPT];
      load(h, c0, h1);
#pragma unroll
      for (int q = 0; q < PPT; ++q) {
        const int64_t j = c0 + threadIdx.x + (int64_t)q * NT;
        const uint32_t bits = __float_as_uint(h[q].w);
        if (j < h1 && sort::rec_top(bits)) add(h[q], j, sort::rec_cell(bits) - B.b2, 4);
      }
    }
  }
  for (int bz = bz0; bz < bz1; ++bz) {
    const int o[3] = {cx * B.b0, cy * B.b1, bz * B.b2};
    const int64_t j0 = off[bz], j1 = off[bz + 1];
    for (int64_t c0 = j0; c0 < j1; c0 += CH) {
      float4 cur[PPT];
#pragma unroll
      for (int q = 0; q < PPT; ++q) cur[q] = raw[q];
      load(raw, c0 + CH < j1 ? c0 + CH : j1, run1);  // next chunk
#pragma unroll
      for (int q = 0; q < PPT; ++q) {
        const int64_t j = c0 + threadIdx.x + (int64_t)q * NT;
        if (j < j1) add(cur[q], j, sort::rec_cell(__float_as_uint(cur[q].w)), 0);
      }
    }
    __syncthreads();
    // z carry: the plane z = b2 is the next brick's z = 0 plane
    for (int r = threadIdx.x; r < rows; r += NT) {
      Sum* row = tile + r * P;
      const Sum cin = row[carry];
      row[carry] = row[B.b2];
      row[B.b2] = Sum(0);
      row[0] += cin;
    }
    __syncthreads();
    // owned cells x < b0, y < b1, z < b2, then the x == b0 and y == b1 planes (z < b2); each cell is
    // cleared for the next brick as it is read
    if constexpr (B_::kVec) {
      constexpr int C4 = BZ / 4;
      constexpr int OWN = BX * BY * C4, XP = (BY + 1) * C4, YP = BX * C4;
      for (int it = threadIdx.x; it < OWN + XP + YP; it += NT) {
        int x, y, c4;
        float* dst;
        if (it < OWN) {
          int r = it / C4;
          c4 = it - r * C4;
          x = r / BY;
          y = r - x * BY;
          dst = &mesh[((int64_t)(o[0] + x) * n1 + (o[1] + y)) * n2 + o[2] + 4 * c4];
        } else if (it < OWN + XP) {
          int r = (it - OWN) / C4;
          c4 = (it - OWN) - r * C4;
          x = BX;
          y = r;
          dst = &xs[((int64_t)col * (BY + 1) + y) * n2 + o[2] + 4 * c4];
        } else {
          int r = (it - OWN - XP) / C4;
          c4 = (it - OWN - XP) - r * C4;
          x = r;
          y = BY;
          dst = &ys[((int64_t)col * BX + x) * n2 + o[2] + 4 * c4];
        }
        Sum* src = &tile[B.cell(x, y, 4 * c4)];  // 16-byte aligned
        const Sum x0 = src[0], x1 = src[1], x2 = src[2], x3 = src[3];
        src[0] = src[1] = src[2] = src[3] = Sum(0);
        float4 o = make_float4(unfix(x0), unfix(x1), unfix(x2), unfix(x3));
        if (CIC && base && it < OWN) {
          const float4 m = *reinterpret_cast<const float4*>(base + (dst - mesh));
          o = make_float4(m.x + o.x, m.y + o.y, m.z + o.z, m.w + o.w);
        }
        *reinterpret_cast<float4*>(dst) = o;
      }
    } else {
      const int own = B.b0 * B.b1 * B.b2, xp = B.t1() * B.b2, yp = B.b0 * B.b2;
      for (int i = threadIdx.x; i < own + xp + yp; i += NT) {
        Sum* src;
        float* dst;
        if (i < own) {
          int r = i / B.b2, z = i - r * B.b2;
          int x = r / B.b1, y = r - x * B.b1;
          dst = &mesh[((int64_t)(o[0] + x) * n1 + (o[1] + y)) * n2 + (o[2] + z)];
          src = &tile[B.cell(x, y, z)];
        } else if (i < own + xp) {
          int r = (i - own) / B.b2, z = (i - own) - r * B.b2;
          dst = &xs[((int64_t)col * B.t1() + r) * n2 + o[2] + z];
          src = &tile[B.cell(B.b0, r, z)];
        } else {
          int r = (i - own - xp) / B.b2, z = (i - own - xp) - r * B.b2;
          dst = &ys[((int64_t)col * B.b0 + r) * n2 + o[2] + z];
          src = &tile[B.cell(r, B.b1, z)];
        }
        float o = unfix(*src);
        if (CIC && base && i < own) o = base[dst - mesh] + o;
        *dst = o;
        *src = Sum(0);
      }
    }
    __syncthreads();
  }
}

// Add the upper x/y planes of the neighbouring columns into the lower x/y planes of each
// column.  A cell with lx = X % b0 and ly = Y % b1 receives
//   lx == 0: XS of column (cx-1, cy) row ly; and when ly == 0 also XS of (cx-1, cy-1) row b1
//   ly == 0: YS of column (cx, cy-1) row lx
// (columns periodic).  One thread per z element, z fastest: every access is coalesced.
__global__ void __launch_bounds__(kBlock) k_fold_xy(Bricks k, const float* __restrict__ xs,
                                                    const float* __restrict__ ys, float* __restrict__ mesh) {
  const int b0 = k.b[0], b1 = k.b[1];
  const int nb0 = k.nb[0], nb1 = k.nb[1];
  const int64_t nx = k.n[0], ny = k.n[1], nz = k.n[2];
  const int64_t nxp = (int64_t)nb0 * ny * nz;        // x-plane cells
  const int64_t nyp = (nx - nb0) * nb1 * nz;         // y-plane cells with lx != 0
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nxp + nyp;
       i += (int64_t)gridDim.x * blockDim.x) {
    int64_t X, Y, Z;
    float add;
    if (i < nxp) {
      Z = i % nz;
      int64_t t = i / nz;
      Y = t % ny;
      const int cxp = (int)(t / ny);
      X = (int64_t)cxp * b0;
      const int cy = (int)(Y / b1), ly = (int)(Y - (int64_t)cy * b1);
      const int sx = cxp == 0 ? nb0 - 1 : cxp - 1;
      add = xs[(((int64_t)sx * nb1 + cy) * (b1 + 1) + ly) * nz + Z];
      if (ly == 0) {
        const int sy = cy == 0 ? nb1 - 1 : cy - 1;
        add += xs[(((int64_t)sx * nb1 + sy) * (b1 + 1) + b1) * nz + Z];
        add += ys[(((int64_t)cxp * nb1 + sy) * b0) * nz + Z];
      }
    } else {
      const int64_t j = i - nxp;
      Z = j % nz;
      int64_t t = j / nz;
      const int64_t xr = t % (nx - nb0);
      const int cyp = (int)(t / (nx - nb0));
      const int cx = (int)(xr / (b0 - 1)), lx = 1 + (int)(xr - (int64_t)cx * (b0 - 1));
      X = (int64_t)cx * b0 + lx;
      Y = (int64_t)cyp * b1;
      const int sy = cyp == 0 ? nb1 - 1 : cyp - 1;
      add = ys[(((int64_t)cx * nb1 + sy) * b0 + lx) * nz + Z];
    }
    const int64_t flat = (X * ny + Y) * nz + Z;
    mesh[flat] = mesh[flat] + add;
  }
}

// Stage rows z in [0, b2) of one component's tile for brick (cx, cy, bz) (rows wrap in x, y).
template <int BX, int BY, int BZ>
__device__ __forceinline__ void stage_rows(float* tile, const float* __restrict__ F, const BrickShape<BX, BY, BZ>& B,
                                           const Bricks& k, int cx, int cy, int bz) {
  constexpr int NT = BrickShape<BX, BY, BZ>::NT;
  const int ox = cx * B.b0, oy = cy * B.b1, oz = bz * B.b2;
  if constexpr (BrickShape<BX, BY, BZ>::kVec) {
    constexpr int C4 = BZ / 4;
    constexpr int ITEMS = (BX + 1) * (BY + 1) * C4;
    constexpr int ONE = (ITEMS + NT - 1) / NT;
    constexpr int ROUND = ONE <= 6 ? ONE : 4;
#pragma unroll 1
    for (int base = 0; base < ITEMS; base += ROUND * NT) {
      float4 v[ROUND];
#pragma unroll
      for (int u = 0; u < ROUND; ++u) {  // unconditional (clamped) loads: the round stays in flight
        int it = min(base + (int)threadIdx.x + u * NT, ITEMS - 1);
        int r = it / C4, c4 = it - r * C4;
        int x = r / (BY + 1), y = r - x * (BY + 1);
        int gx = ox + x, gy = oy + y;
        gx -= gx >= k.n[0] ? k.n[0] : 0;
        gy -= gy >= k.n[1] ? k.n[1] : 0;
        v[u] = *reinterpret_cast<const float4*>(&F[((int64_t)gx * k.n[1] + gy) * k.n[2] + oz + 4 * c4]);
      }
#pragma unroll
      for (int u = 0; u < ROUND; ++u) {
        int it = base + threadIdx.x + u * NT;
        if (it < ITEMS) {
          int r = it / C4, c4 = it - r * C4;
          float* dst = &tile[r * (BZ + 2) + 4 * c4];
          *reinterpret_cast<float2*>(dst) = make_float2(v[u].x, v[u].y);
          *reinterpret_cast<float2*>(dst + 2) = make_float2(v[u].z, v[u].w);
        }
      }
    }
  } else {
    const int t1 = B.t1(), b2 = B.b2, P = B.pitch();
    const int items = B.rows() * b2;
    for (int i0 = 0; i0 < items; i0 += NT * kBatch) {
      float v[kBatch];
      int dst[kBatch];
#pragma unroll
      for (int u = 0; u < kBatch; ++u) {
        int iu = i0 + u * NT + (int)threadIdx.x;
        int i = min(iu, items - 1);
        int r = i / b2, z = i - r * b2;
        int x = r / t1, y = r - x * t1;
        int gx = ox + x, gy = oy + y;
        gx -= gx >= k.n[0] ? k.n[0] : 0;
        gy -= gy >= k.n[1] ? k.n[1] : 0;
        v[u] = F[((int64_t)gx * k.n[1] + gy) * k.n[2] + oz + z];
        dst[u] = iu < items ? r * P + z : -1;
      }
#pragma unroll
      for (int u = 0; u < kBatch; ++u)
        if (dst[u] >= 0) tile[dst[u]] = v[u];
    }
  }
}

// The z = 0 plane of brick (cx, cy, bz) of one component, read directly (rows wrap in x, y).
template <int BX, int BY, int BZ>
__device__ __forceinline__ void load_plane(float* plane, const float* __restrict__ F, const BrickShape<BX, BY, BZ>& B,
                                           const Bricks& k, int cx, int cy, int bz) {
  constexpr int NT = BrickShape<BX, BY, BZ>::NT;
  const int t1 = B.t1();
  for (int r = threadIdx.x; r < B.rows(); r += NT) {
    int x = r / t1, y = r - x * t1;
    int gx = cx * B.b0 + x, gy = cy * B.b1 + y;
    gx -= gx >= k.n[0] ? k.n[0] : 0;
    gy -= gy >= k.n[1] ? k.n[1] : 0;
    plane[r] = F[((int64_t)gx * k.n[1] + gy) * k.n[2] + (int64_t)bz * B.b2];
  }
}

// Invalid particles (binned last, past the last brick: sorted positions [first, n)) get zero rows,
// a share per workgroup of the column walk that writes the others' (n = 0: nothing to do).
__device__ __forceinline__ void zero_invalid(const int32_t* __restrict__ perm, int64_t first, int64_t n,
                                             float* __restrict__ out) {
  const int64_t wg = (int64_t)blockIdx.y * gridDim.x + blockIdx.x;
  for (int64_t j = first + wg * blockDim.x + threadIdx.x; j < n;
       j += (int64_t)gridDim.x * gridDim.y * blockDim.x) {
    const int64_t i = perm[j];
    out[i * 3 + 0] = 0.f;
    out[i * 3 + 1] = 0.f;
    out[i * 3 + 2] = 0.f;
  }
}

template <int BX, int BY, int BZ>
__global__ void __launch_bounds__((BrickShape<BX, BY, BZ>::NT)) k_gather_columns(
    const float4* __restrict__ rec, const int32_t* __restrict__ bin_off, const int32_t* __restrict__ perm, Bricks k,
    int run, const float* __restrict__ f0, const float* __restrict__ f1, const float* __restrict__ f2, int64_t nzero,
    float* __restrict__ acc) {
  using B_ = BrickShape<BX, BY, BZ>;
  constexpr int NT = B_::NT, CAP = B_::CAP, PPT = B_::PPT;
  __shared__ __align__(16) float tile[B_::TF];
  __shared__ float res[3][CAP];
  __shared__ float plane[2][3][B_::PL];  // [parity of bz][component]: lower z plane of brick bz
  const B_ B(k);
  const int col = patch_column_of(blockIdx.x, gridDim.x, k.nb[0], k.nb[1]);
  const int cx = col / k.nb[1], cy = col - cx * k.nb[1];
  const int rows = B.rows(), P = B.pitch(), nb2 = k.nb[2];
  const int bz0 = blockIdx.y * run, bz1 = min(nb2, bz0 + run);
  // the brick above the run (above the top one: brick 0, periodic)
  const int above = bz1 == nb2 ? 0 : bz1;
  load_plane(plane[bz1 & 1][0], f0, B, k, cx, cy, above);
  load_plane(plane[bz1 & 1][1], f1, B, k, cx, cy, above);
  load_plane(plane[bz1 & 1][2], f2, B, k, cx, cy, above);
  for (int bz = bz1 - 1; bz >= bz0; --bz) {
    const int64_t bid = (int64_t)col * nb2 + bz;
    const int64_t j0 = bin_off[bid], j1 = bin_off[bid + 1];
    const int up = (bz + 1) & 1, me = bz & 1;
    if (j0 == j1) {  // no particles: only this brick's lower planes are needed (by the brick below)
      __syncthreads();
      load_plane(plane[me][0], f0, B, k, cx, cy, bz);
      load_plane(plane[me][1], f1, B, k, cx, cy, bz);
      load_plane(plane[me][2], f2, B, k, cx, cy, bz);
      continue;
    }
    for (int64_t s0 = j0; s0 < j1; s0 += CAP) {
      const int64_t s1 = s0 + CAP < j1 ? s0 + CAP : j1;
      // each particle's record, once for the three components (clamped loads; their latency
      // overlaps the first tile's staging)
      float4 r[PPT];
#pragma unroll
      for (int q = 0; q < PPT; ++q) {
        const int64_t j = s0 + threadIdx.x + (int64_t)q * NT;
        r[q] = rec[j < s1 ? j : s1 - 1];
      }
#pragma unroll 1
      for (int comp = 0; comp < 3; ++comp) {
        const float* __restrict__ F = comp == 0 ? f0 : (comp == 1 ? f1 : f2);
        __syncthreads();  // the previous component's interpolation is done with the tile
        stage_rows<BX, BY, BZ>(tile, F, B, k, cx, cy, bz);
        for (int i = threadIdx.x; i < rows; i += NT) tile[i * P + B.b2] = plane[up][comp][i];
        __syncthreads();
        for (int i = threadIdx.x; i < rows; i += NT) plane[me][comp][i] = tile[i * P];
#pragma unroll
        for (int q = 0; q < PPT; ++q) {
          const int jl = threadIdx.x + q * NT;
          if (s0 + jl >= s1) continue;
          const float fr[3] = {r[q].x, r[q].y, r[q].z};
          const int c0 = sort::rec_cell(__float_as_uint(r[q].w));
          float sum = 0.f;
#pragma unroll
          for (int c = 0; c < 8; ++c) sum = sum + tile[c0 + B.corner_off(c)] * frac_weight(fr, c);
          res[comp][jl] = sum;
        }
      }
      __syncthreads();
#pragma unroll
      for (int q = 0; q < PPT; ++q) {
        const int jl = threadIdx.x + q * NT;
        if (s0 + jl < s1) {
          int64_t i = perm[s0 + jl];
          acc[i * 3 + 0] = res[0][jl];
          acc[i * 3 + 1] = res[1][jl];
          acc[i * 3 + 2] = res[2][jl];
        }
      }
    }
  }
  zero_invalid(perm, bin_off[(int64_t)k.nb[0] * k.nb[1] * nb2], nzero, acc);
}

// The displacement cotangent of the force step, tiled like k_gather_columns: for sorted
// particle j, dc = sum_m coef_m(j) sum_c M_m(c) grad W_c(j) with the meshes M = (F_x, F_y, F_z,
// dens_cot) and coef = (acc_cot of j, x, y, z, from the sorted component-major copies; the
// particle value), written as dc / a1 through perm: the reverse of the three gathers
// (pallas.py:321-355) and the scatter adjoint's displacement term (pallas.py:358-409) in one
// pass.  grad W_c = (s_x w_y w_z, w_x s_y w_z, w_x w_y s_z) with s = sign(-(f - b)), sign(0) =
// 0 (the corner_grad convention).  Each mesh's tile is staged in turn, a particle's partial sums
// waiting in its thread's own LDS slots; small bricks' tiles are staged together.  With a zero particle value the density term is skipped.
template <int BX, int BY, int BZ>
__global__ void __launch_bounds__((BrickShape<BX, BY, BZ>::NT)) k_disp_cot_columns(
    const float4* __restrict__ rec, const int32_t* __restrict__ bin_off, const int32_t* __restrict__ perm, float cell,
    Bricks k, int run, const float* __restrict__ f0, const float* __restrict__ f1, const float* __restrict__ f2,
    const float* __restrict__ dcot, const float* __restrict__ cot_s, int64_t n, float val, int64_t nzero,
    float* __restrict__ disp_cot, int accum) {
  using B_ = BrickShape<BX, BY, BZ>;
  constexpr int NT = B_::NT, CAP = B_::CAP, PPT = B_::PPT;
  constexpr bool ALL = BX == 8;  // every mesh's tile at once
  __shared__ __align__(16) float tile[ALL ? 4 * B_::TF : B_::TF];
  __shared__ float res[3][ALL ? 1 : CAP];
  __shared__ float plane[2][4][B_::PL];  // [parity of bz][mesh]: lower z plane of brick bz
  const B_ B(k);
  const int col = patch_column_of(blockIdx.x, gridDim.x, k.nb[0], k.nb[1]);
  const int cx = col / k.nb[1], cy = col - cx * k.nb[1];
  const int rows = B.rows(), P = B.pitch(), nb2 = k.nb[2];
  // the meshes: the force components and (val != 0) the density cotangent; the latter alone (no f0);
  // or one mesh alone (f0 without f1)
  const int nm = f0 && !f1 ? 1 : (val != 0.f ? 4 : 3);
  const int m0 = f0 ? 0 : 3;
  const int bz0 = blockIdx.y * run, bz1 = min(nb2, bz0 + run);
  // the brick above the run (above the top one: brick 0, periodic)
  const int above = bz1 == nb2 ? 0 : bz1;
  for (int m = m0; m < nm; ++m)
    load_plane(plane[bz1 & 1][m], m == 0 ? f0 : (m == 1 ? f1 : (m == 2 ? f2 : dcot)), B, k, cx, cy, above);
  for (int bz = bz1 - 1; bz >= bz0; --bz) {
    const int64_t bid = (int64_t)col * nb2 + bz;
    const int64_t j0 = bin_off[bid], j1 = bin_off[bid + 1];
    const int up = (bz + 1) & 1, me = bz & 1;
    if (j0 == j1) {  // no particles: only this brick's lower planes are needed (by the brick below)
      __syncthreads();
      for (int m = m0; m < nm; ++m)
        load_plane(plane[me][m], m == 0 ? f0 : (m == 1 ? f1 : (m == 2 ? f2 : dcot)), B, k, cx, cy, bz);
      continue;
    }
    auto mesh = [&](int m) { return m == 0 ? f0 : (m == 1 ? f1 : (m == 2 ? f2 : dcot)); };
    // mesh m's tile (and this brick's lower plane, for the brick below)
    auto stage = [&](int m) {
      __syncthreads();  // the previous mesh's pass is done with the tile
      stage_rows<BX, BY, BZ>(tile, mesh(m), B, k, cx, cy, bz);
      for (int i = threadIdx.x; i < rows; i += NT) tile[i * P + B.b2] = plane[up][m][i];
      __syncthreads();
      for (int i = threadIdx.x; i < rows; i += NT) plane[me][m][i] = tile[i * P];
    };
    // a particle's weights and the signs of their derivatives
    struct Weights {
      float w[3][2], sg[3][2];
    };
    auto weights = [&](const float4& r) {
      Weights W;
      const float fr[3] = {r.x, r.y, r.z};
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        float f = fr[a];
        asm volatile("" : "+v"(f));  // weights per mesh pass: kept out of registers between passes
#pragma unroll
        for (int bb = 0; bb < 2; ++bb) {
          const float delta = f - (float)bb;
          W.w[a][bb] = 1.f - fabsf(delta);
          W.sg[a][bb] = cic_sign(delta);
        }
      }
      return W;
    };
    // sum_c M(c) grad W_c over a staged mesh's corners from c0
    auto grads = [&](const Weights& W, int c0, float gs[3]) {
      gs[0] = gs[1] = gs[2] = 0.f;
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        const int bx = c & 1, by = (c >> 1) & 1, bzz = (c >> 2) & 1;
        const float v = tile[c0 + B.corner_off(c)];
        gs[0] = gs[0] + v * (W.sg[0][bx] * W.w[1][by] * W.w[2][bzz]);
        gs[1] = gs[1] + v * (W.w[0][bx] * W.sg[1][by] * W.w[2][bzz]);
        gs[2] = gs[2] + v * (W.w[0][bx] * W.w[1][by] * W.sg[2][bzz]);
      }
    };
    if constexpr (ALL) {
      // Small bricks: the meshes are staged together, once per brick, and a particle's sums stay in
      // registers.  Mesh by mesh and 512 particles at a time, a brick that holds most particles of a
      // state was staged 2048 times: 64^3 particles in one brick of 128^3 3.29 ms (1.89 in the
      // 512-thread walk of large bricks before), the whole VJP 6.07 -> 3.42 ms, CIC gather adjoint 2.21 -> 1.19
      // (float atomics 1.21); VJP of 64^3 on 64^3 204 -> 196 us
      constexpr int U = 4;
      __syncthreads();
      for (int m = m0; m < nm; ++m) {
        float* T = tile + m * B_::TF;
        stage_rows<BX, BY, BZ>(T, mesh(m), B, k, cx, cy, bz);
        for (int i = threadIdx.x; i < rows; i += NT) T[i * P + B.b2] = plane[up][m][i];
      }
      __syncthreads();
      for (int m = m0; m < nm; ++m)
        for (int i = threadIdx.x; i < rows; i += NT) plane[me][m][i] = tile[m * B_::TF + i * P];
      for (int64_t s0 = j0; s0 < j1; s0 += U * NT) {
        float4 r[U];
        float cf[U][4];
        int32_t row[U];
#pragma unroll
        for (int q = 0; q < U; ++q) {  // clamped loads
          int64_t jq = s0 + threadIdx.x + (int64_t)q * NT;
          jq = jq < j1 ? jq : j1 - 1;
          r[q] = rec[jq];
          row[q] = perm[jq];
#pragma unroll
          for (int m = 0; m < 4; ++m) cf[q][m] = m < 3 && m >= m0 && m < nm ? cot_s[(int64_t)m * n + jq] : val;
        }
#pragma unroll
        for (int q = 0; q < U; ++q) {
          if (s0 + threadIdx.x + (int64_t)q * NT >= j1) continue;
          const Weights W = weights(r[q]);
          const int c0 = sort::rec_cell(__float_as_uint(r[q].w));
          float sum[3] = {0.f, 0.f, 0.f};
#pragma unroll
          for (int m = 0; m < 4; ++m) {
            if (m < m0 || m >= nm) continue;  // uniform
            float gs[3];
            grads(W, c0 + m * B_::TF, gs);
#pragma unroll
            for (int a = 0; a < 3; ++a) sum[a] = sum[a] + cf[q][m] * gs[a];
          }
          float* out = disp_cot + (int64_t)row[q] * 3;
#pragma unroll
          for (int a = 0; a < 3; ++a) out[a] = (accum ? out[a] : 0.f) + sum[a] / cell;
        }
      }
    } else if (nm - m0 == 1) {
      // One mesh alone: staged once for the brick and the results written as they come.  With a staging and
      // two barriers per CAP particles, bricks of many particles took long: CIC gather adjoint of 64^3
      // particles in one brick of 256^3 1.00 -> 0.74 ms (float atomics 0.43), 128^3 on 256^3 168 -> 143 us (736)
      constexpr int U = 4;
      stage(m0);
      for (int64_t s0 = j0; s0 < j1; s0 += U * NT) {
        float4 r[U];
        float cf[U];
        int32_t row[U];
#pragma unroll
        for (int q = 0; q < U; ++q) {  // clamped loads
          int64_t jq = s0 + threadIdx.x + (int64_t)q * NT;
          jq = jq < j1 ? jq : j1 - 1;
          r[q] = rec[jq];
          cf[q] = m0 < 3 ? cot_s[(int64_t)m0 * n + jq] : val;
          row[q] = perm[jq];
        }
#pragma unroll
        for (int q = 0; q < U; ++q) {
          if (s0 + threadIdx.x + (int64_t)q * NT >= j1) continue;
          float gs[3];
          grads(weights(r[q]), sort::rec_cell(__float_as_uint(r[q].w)), gs);
          float* out = disp_cot + (int64_t)row[q] * 3;
#pragma unroll
          for (int a = 0; a < 3; ++a) out[a] = (accum ? out[a] : 0.f) + cf[q] * gs[a] / cell;
        }
      }
    } else {
      for (int64_t s0 = j0; s0 < j1; s0 += CAP) {
        const int64_t s1 = s0 + CAP < j1 ? s0 + CAP : j1;
        // each particle's record, once for every mesh
        float4 r[PPT];
#pragma unroll
        for (int q = 0; q < PPT; ++q) {
          const int64_t j = s0 + threadIdx.x + (int64_t)q * NT;
          r[q] = rec[j < s1 ? j : s1 - 1];
        }
#pragma unroll 1
        for (int m = m0; m < nm; ++m) {
          stage(m);
          float cf[PPT];
#pragma unroll
          for (int q = 0; q < PPT; ++q) {  // this mesh's coefficients (clamped loads)
            const int64_t j = s0 + threadIdx.x + (int64_t)q * NT;
            cf[q] = m < 3 ? cot_s[(int64_t)m * n + (j < s1 ? j : s1 - 1)] : val;
          }
#pragma unroll
          for (int q = 0; q < PPT; ++q) {
            const int jl = threadIdx.x + q * NT;
            if (s0 + jl >= s1) continue;
            float gs[3];
            grads(weights(r[q]), sort::rec_cell(__float_as_uint(r[q].w)), gs);
#pragma unroll
            for (int a = 0; a < 3; ++a) res[a][jl] = (m == m0 ? 0.f : res[a][jl]) + cf[q] * gs[a];
          }
        }
#pragma unroll
        for (int q = 0; q < PPT; ++q) {  // a thread's own results: no barrier
          const int jl = threadIdx.x + q * NT;
          if (s0 + jl < s1) {
            const int64_t i = perm[s0 + jl];
#pragma unroll
            for (int a = 0; a < 3; ++a) disp_cot[i * 3 + a] = res[a][jl] / cell;
          }
        }
      }
    }
  }
  zero_invalid(perm, bin_off[(int64_t)k.nb[0] * k.nb[1] * nb2], nzero, disp_cot);
}

// Reverse of the three gathers without brick tiling (gather^T = float-atomic scatter of
// acc_cot, plus the displacement cotangent from the mesh values), pallas.py:321-355 per
// component.
__global__ void __launch_bounds__(kBlock) k_gather3_bwd_sorted(
    const int16_t* __restrict__ pmid, const float* __restrict__ disp, const uint8_t* __restrict__ valid,
    const int32_t* __restrict__ perm, int64_t n, Geom g, const float* __restrict__ fx,
    const float* __restrict__ fy, const float* __restrict__ fz, const float* __restrict__ acc_cot,
    float* __restrict__ gx, float* __restrict__ gy, float* __restrict__ gz, float* __restrict__ disp_cot_s) {
  int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= n) return;
  float dc[3] = {0.f, 0.f, 0.f};
  if (valid[j]) {
    int64_t i = perm[j];
    float ac[3] = {acc_cot[i * 3 + 0], acc_cot[i * 3 + 1], acc_cot[i * 3 + 2]};
    AxisCic ax[3];
    particle_cic(g, pmid, disp, j, ax);
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      int64_t flat;
      corner_index(g, ax, c, flat);
      float w = corner_weight(ax, c);
      float gr[3];
      corner_grad(ax, c, gr);
      atomic_add_f32(gx + flat, ac[0] * w);
      atomic_add_f32(gy + flat, ac[1] * w);
      atomic_add_f32(gz + flat, ac[2] * w);
      float inner = ac[0] * fx[flat] + ac[1] * fy[flat] + ac[2] * fz[flat];
#pragma unroll
      for (int a = 0; a < 3; ++a) dc[a] = dc[a] + inner * gr[a];
    }
  }
#pragma unroll
  for (int a = 0; a < 3; ++a) disp_cot_s[j * 3 + a] = dc[a] / g.a1;
}

// Sorted, component-major copies of the acceleration cotangent (cot_s[c n + j] = acc_cot of
// sorted particle j) for the tiled gather-adjoint scatter, and per-block maxima of |acc_cot|.
__global__ void __launch_bounds__(kBlock) k_cot_sorted(const int32_t* __restrict__ perm,
                                                       const float* __restrict__ acc_cot, int64_t n,
                                                       float* __restrict__ cot_s, float* __restrict__ pmax) {
  float mx = 0.f;  // +inf once a non-finite value is seen (fmaxf alone would skip a NaN)
  for (int64_t j = (int64_t)blockIdx.x * kBlock + threadIdx.x; j < n; j += (int64_t)gridDim.x * kBlock) {
    const int64_t i = perm[j];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const float v = acc_cot[i * 3 + c];
      cot_s[c * n + j] = v;
      mx = isfinite(v) ? fmaxf(mx, fabsf(v)) : INFINITY;
    }
  }
  for (int off = 32; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off));
  __shared__ float part[kBlock / 64];
  if ((threadIdx.x & 63) == 0) part[threadIdx.x / 64] = mx;
  __syncthreads();
  if (threadIdx.x == 0) {
    float m = 0.f;
    for (int w = 0; w < kBlock / 64; ++w) m = fmaxf(m, part[w]);
    pmax[blockIdx.x] = m;
  }
}

// scale[0] = 1 / max |acc_cot| (1 when all are zero; capped at 2^127 when the maximum is so
// small that its reciprocal overflows): the values enter the fixed point at magnitude <= 1.
// A non-finite cotangent makes the scale NaN, and the tiled scatter's output scale (the
// reciprocal) with it, so every mesh cotangent and with them every particle's displacement
// cotangent and the Omega_m cotangent come out NaN, as the unfused float chain would give.
__global__ void k_cot_scale(const float* __restrict__ pmax, int nb, float* __restrict__ scale) {
  float m = 0.f;
  for (int i = threadIdx.x; i < nb; i += 64) m = fmaxf(m, pmax[i]);  // one wave
  for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
  if (threadIdx.x != 0) return;
  scale[0] = !(m <= 3.402823466e38f) ? __int_as_float(0x7fc00000) : (m > 0.f ? fminf(1.f / m, 1.7014118e38f) : 1.f);
}

// Scatter adjoint for the density: disp_cot += v * sum_c dens_cot[c] grad_c / cell, then the
// total is written back in caller order (scatter.py:341-375, pallas.py:358-409).
__global__ void __launch_bounds__(kBlock) k_scatter_bwd_sorted(
    const int16_t* __restrict__ pmid, const float* __restrict__ disp, const uint8_t* __restrict__ valid,
    const int32_t* __restrict__ perm, int64_t n, Geom g, float val, const float* __restrict__ dens_cot,
    const float* __restrict__ disp_cot_s, float* __restrict__ disp_cot) {
  int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= n) return;
  float dc[3] = {0.f, 0.f, 0.f};
  if (valid[j] && val != 0.f) {
    AxisCic ax[3];
    particle_cic(g, pmid, disp, j, ax);
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      int64_t flat;
      corner_index(g, ax, c, flat);
      float gr[3];
      corner_grad(ax, c, gr);
      float mv = dens_cot[flat] * val;
#pragma unroll
      for (int a = 0; a < 3; ++a) dc[a] = dc[a] + mv * gr[a];
    }
  }
  int64_t i = perm[j];
#pragma unroll
  for (int a = 0; a < 3; ++a)  // added to the gather's terms (disp_cot_s), or to disp_cot itself when null
    disp_cot[i * 3 + a] = (disp_cot_s ? disp_cot_s[j * 3 + a] : disp_cot[i * 3 + a]) + dc[a] / g.a1;
}

// omega_cot += 1.5 * sum_x src_cot(x) * (rho(x) [+ rho_add(x)] - 1); dens_cot = src_cot * scale,
// in place, and copied to rho_cot when given (the cotangent of an added density)
__global__ void __launch_bounds__(kBlock) k_source_bwd(float* __restrict__ src_cot,
                                                       const float* __restrict__ rho,
                                                       const float* __restrict__ rho_add,
                                                       float* __restrict__ rho_cot, int64_t n,
                                                       float scale, double* __restrict__ part) {
  // sum_x src_cot (rho - 1): float products, float64 sums (per thread, then per block in a
  // fixed order), one partial per block; float4 accesses when every array is 16-byte aligned
  const bool vec = ((reinterpret_cast<uintptr_t>(src_cot) | reinterpret_cast<uintptr_t>(rho) |
                     reinterpret_cast<uintptr_t>(rho_add) | reinterpret_cast<uintptr_t>(rho_cot)) & 15) == 0;
  const int64_t n4 = vec ? n / 4 : 0;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  const int64_t g0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  double acc = 0.0;
  for (int64_t q = g0; q < n4; q += stride) {
    const float4 sc = reinterpret_cast<const float4*>(src_cot)[q];
    float4 r = reinterpret_cast<const float4*>(rho)[q];
    if (rho_add) {
      const float4 ra = reinterpret_cast<const float4*>(rho_add)[q];
      r = make_float4(r.x + ra.x, r.y + ra.y, r.z + ra.z, r.w + ra.w);
    }
    acc += (double)(sc.x * (r.x - 1.f)) + (double)(sc.y * (r.y - 1.f)) + (double)(sc.z * (r.z - 1.f)) +
           (double)(sc.w * (r.w - 1.f));
    const float4 o = make_float4(sc.x * scale, sc.y * scale, sc.z * scale, sc.w * scale);
    reinterpret_cast<float4*>(src_cot)[q] = o;
    if (rho_cot) reinterpret_cast<float4*>(rho_cot)[q] = o;
  }
  for (int64_t i = 4 * n4 + g0; i < n; i += stride) {
    const float sc = src_cot[i];
    float r = rho[i];
    if (rho_add) r += rho_add[i];
    acc += (double)(sc * (r - 1.f));
    src_cot[i] = sc * scale;
    if (rho_cot) rho_cot[i] = sc * scale;
  }
  for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off);
  __shared__ double wsum[kBlock / 64];
  if ((threadIdx.x & 63) == 0) wsum[threadIdx.x / 64] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int w = 0; w < kBlock / 64; ++w) t += wsum[w];
    part[blockIdx.x] = t;
  }
}

// omega_cot[0] += 1.5 * (the block partials of k_source_bwd, summed in a fixed order)
__global__ void k_source_bwd_sum(const double* __restrict__ part, int nb, float* __restrict__ omega_cot) {
  const double t = wave_sum(part, nb);
  if (threadIdx.x == 0) omega_cot[0] += 1.5f * (float)t;
}

constexpr int kSrcBlocks = 2048;  // blocks of k_source_bwd (and its partials)

struct Layout {
  int nx, ny, nz, m;
  int64_t pitch;  // complex row pitch (float2) of a full half spectrum, >= m+1, multiple of 16
  int64_t nreal;  // nx*ny*nz
  int64_t ncplx;  // nx*ny*pitch
  // Band of the force pipeline.  With the particle-Nyquist filter active every mode with
  // |k_i| > pi/l_p (1 + 8 eps) is zero after the Green multiply, so the passes after the z
  // r2c keep only kz < nkz and, after the y forward pass, only the 2*ky_keep+1 rows with
  // |ky| <= ky_keep (packed).  Unfiltered axes keep everything (nkz = m+1, ky_keep = -1).
  int nkz;         // stored spectrum columns (kz = 0..nkz-1); nkz = m+1 includes Nyquist
  int ky_keep;     // packed y band half-width, -1 = full rows
  int nky;         // rows after the y forward pass (2*ky_keep+1 or ny)
  int64_t pitch1;  // row pitch of the banded spectra, multiple of 16
  int64_t s1;      // nx*ny*pitch1:  full-y banded spectrum
  int64_t s2;      // nx*nky*pitch1: packed-y banded spectrum
};

// Largest |m| on an axis of n points whose wavenumber 2 pi m / (n cell) can pass the
// particle-Nyquist mask |k| <= pi/l_p (1 + 8 eps_f32) (core/utils.py:33-37).  The slack of
// 1e-4 makes the band a superset of the device-side float32 mask, which still decides
// every mode inside the band.
int band_half_width(int n, double cell, double spacing) {
  double kmax = 3.14159265358979323846 / spacing * (1.0 + 8.0 * 1.1920928955078125e-07) * (1.0 + 1e-4);
  double dk = 2.0 * 3.14159265358979323846 / ((double)n * cell);
  return (int)std::floor(kmax / dk);
}

Layout make_layout(const pm_gravity_desc* d) {
  const int32_t* s = d->mesh_shape;
  Layout L;
  L.nx = s[0];
  L.ny = s[1];
  L.nz = s[2];
  L.m = s[2] / 2;
  L.pitch = (int64_t)align_up((size_t)L.m + 1, 16);
  L.nreal = (int64_t)L.nx * L.ny * L.nz;
  L.ncplx = (int64_t)L.nx * L.ny * L.pitch;
  L.nkz = L.m + 1;
  L.ky_keep = -1;
  L.nky = L.ny;
  if (d->mask_active) {
    int kz = band_half_width(L.nz, d->cell_size, d->ptcl_spacing);
    if (kz < L.m) L.nkz = kz + 1;
    int ky = band_half_width(L.ny, d->cell_size, d->ptcl_spacing);
    if (2 * ky + 1 < L.ny) {
      L.ky_keep = ky;
      L.nky = 2 * ky + 1;
    }
  }
  L.pitch1 = (int64_t)align_up((size_t)L.nkz, 16);
  L.s1 = (int64_t)L.nx * L.ny * L.pitch1;
  L.s2 = (int64_t)L.nx * L.nky * L.pitch1;
  return L;
}

int check_desc(const pm_gravity_desc* d, int64_t n) {
  PM_RETURN_IF(d == nullptr, PM_ERROR_INVALID_ARGUMENT, "desc is NULL");
  PM_RETURN_IF(n < 0 || n > INT32_MAX, PM_ERROR_UNSUPPORTED, "particle count must be in [0, 2^31)");
  PM_RETURN_IF(!fft::supported_shape(d->mesh_shape), PM_ERROR_UNSUPPORTED,
               "mesh axes must be powers of two in [2, 2048]");
  PM_RETURN_IF(!(d->cell_size > 0.f), PM_ERROR_INVALID_ARGUMENT, "cell_size must be positive");
  PM_RETURN_IF(d->mask_active && !(d->ptcl_spacing > 0.f), PM_ERROR_INVALID_ARGUMENT,
               "ptcl_spacing must be positive when the particle-Nyquist mask is active");
  return sort::check_sort_args(n, d->mesh_shape, d->brick);
}

constexpr int kCotBlocks = 1024;  // blocks of k_cot_sorted (and slots of their maxima)

struct Buffers {
  sort::Sorted srt;  // the bucketed particles: records when tiled, else the sorted payload
  float* tables;
  bool tiled;      // brick-tiled scatter/gather (the brick divides the mesh and fits LDS)
  float* xs;       // upper x / y planes of every brick column (tiled scatter)
  float* ys;
  float* r0;  // density, then F_x
  float* r1;  // F_y
  float* r2;  // F_z
  float2* ca;  // s1-sized banded spectra: ca, cc, ce
  float2* cb;  // s2-sized (packed y rows): cb, cd, cg
  float2* cc;
  float2* cd;
  float2* ce;
  float2* cg;
  int32_t* count;    // the bucketing's counters and scan partials
  int32_t* partial;
  // reverse only: F_x (the forward keeps rho in r0), three mesh cotangents
  float* g0;
  float* g1;
  float* g2;
  float* g3;
  float* disp_cot_s;
  float* cot_s;      // sorted acc_cot, component-major (tiled reverse)
  float* cot_pmax;   // per-block maxima, then the fixed-point scale
  double* src_part;  // per-block partials of the Omega_m cotangent
};

bool carve(Arena& ws, const Layout& L, int64_t n, const int32_t* shape, const int32_t* brick, bool reverse,
           Buffers& b) {
  b.xs = b.ys = nullptr;
  int64_t nbins = 1;
  for (int a = 0; a < 3; ++a) nbins *= ceil_div(shape[a], brick[a]);
  b.srt = sort::Sorted();
  b.srt.bins = ws.take<int32_t>(nbins + 2);
  b.tiled = tiled_ok(shape, brick);
  if (b.tiled) {
    Bricks k = make_bricks(shape, brick);
    b.xs = ws.take<float>(xs_floats(k));
    b.ys = ws.take<float>(ys_floats(k));
  }
  b.srt.perm = ws.take<int32_t>(n);
  if (b.tiled) {
    b.srt.rec = ws.take<float4>(n);
  } else {
    b.srt.pmid = ws.take<int16_t>(3 * n);
    b.srt.disp = ws.take<float>(3 * n);
    b.srt.valid = ws.take<uint8_t>(n);
  }
  b.tables = ws.take<float>(fft::spec_table_floats(shape));
  b.r0 = ws.take<float>(L.nreal);
  b.r1 = ws.take<float>(L.nreal);
  b.r2 = ws.take<float>(L.nreal);
  // banded force pipeline (see force_mesh_stage and adjoint_spectral_stage)
  // (the x Green pass's two outputs, cb and cg, side by side: 1.34 ms at 1024^3 against 1.47 with cg
  // last, where the three streams of the pass start further apart)
  b.ca = ws.take<float2>(L.s1);
  b.cb = ws.take<float2>(L.s2);
  b.cg = ws.take<float2>(L.s2);
  b.cc = ws.take<float2>(L.s1);
  b.cd = ws.take<float2>(L.s2);
  b.ce = ws.take<float2>(L.s1);
  const int64_t counters = sort::bucket_count_len(shape, brick);
  b.count = ws.take<int32_t>(counters);
  b.partial = ws.take<int32_t>(sort::bucket_partials(counters));
  if (reverse) {
    b.g0 = ws.take<float>(L.nreal);
    b.g1 = ws.take<float>(L.nreal);
    b.g2 = ws.take<float>(L.nreal);
    b.g3 = ws.take<float>(L.nreal);
    b.disp_cot_s = b.tiled ? nullptr : ws.take<float>(3 * n);
    b.cot_s = b.tiled ? ws.take<float>(3 * n) : nullptr;
    b.cot_pmax = b.tiled ? ws.take<float>(kCotBlocks + 1) : nullptr;
    b.src_part = ws.take<double>(kSrcBlocks);
  }
  return ws.ok();
}

size_t workspace_bytes(const pm_gravity_desc* d, int64_t n, bool reverse) {
  Layout L = make_layout(d);
  Arena probe(reinterpret_cast<void*>(uintptr_t(256)), SIZE_MAX / 2);
  Buffers b;
  carve(probe, L, n, d->mesh_shape, d->brick, reverse, b);
  return probe.used + 256;
}

Geom step_geom(const pm_gravity_desc* d) {
  Geom g;
  for (int a = 0; a < 3; ++a) {
    g.ls[a] = d->mesh_shape[a];
    g.gs[a] = d->mesh_shape[a];
    g.off[a] = 0.f;
  }
  g.a1 = d->cell_size;
  g.a2 = 0.f;
  return g;
}

unsigned grid_for(int64_t n) { return (unsigned)std::max<int64_t>(1, ceil_div(n, kBlock)); }

int fill(float* p, int64_t n, hipStream_t s) {
  if (n == 0) return PM_SUCCESS;
  unsigned blocks = (unsigned)std::min<int64_t>(ceil_div(n, kBlock * 4), 1 << 16);
  hipLaunchKernelGGL(k_fill, dim3(blocks), dim3(kBlock), 0, s, p, n, 0.f);
  PM_LAUNCHED("k_fill", s);
  return PM_SUCCESS;
}

// How the column walks cut their columns: `run` bricks per workgroup.  A cut costs the scatter a
// second read of a brick's particles and the gathers a strided plane per component, so columns stay
// whole when there are enough of them for the workgroups the chip holds at once (two per CU of
// 16 x 16 x 32 bricks; 8 x 8 x 16 ones fit more) and are halved until there are otherwise.  256^3
// mesh, 128^3 particles, scatter / gather with 256, 512, 1024 and 2048 workgroups wanted: 37 / 91,
// 33 / 69, 36 / 77, 39 / 83 us; 128^3 mesh in 8 x 8 x 16 bricks with 512, 1024, 2048: 14 / 19, 12 / 17,
// 13 / 15 us.
struct Walk {
  dim3 grid;
  int run;
};
Walk column_walk(const Bricks& k) {
  const int64_t ncols = (int64_t)k.nb[0] * k.nb[1];
  const int64_t want = k.b[0] == 8 ? 1024 : 512;
  int run = k.nb[2];
  while (run > 1 && ncols * ceil_div(k.nb[2], run) < want) run = (run + 1) / 2;
  return {dim3((unsigned)ncols, (unsigned)ceil_div(k.nb[2], run)), run};
}

// The bricks the step uses: the caller's, but 8 x 8 x 16 ones in place of larger ones they divide on
// meshes of up to kSmallMesh cells, where 16 x 16 x 32 columns are too few workgroups (a 64^3
// mesh, 32^3 particles: scatter 16 -> 5, gather 17 -> 6 us; 128^3: 28 -> 11, 36 -> 13 us; at 256^3 their
// additional plane cells cost more, 33 -> 45 and 69 -> 91 us).  The results do not depend on it beyond
// the rounding of the cells that neighbouring columns share.
constexpr int64_t kSmallMesh = int64_t(1) << 21;
int effective_desc(const pm_gravity_desc* d, int64_t n, pm_gravity_desc* out) {
  PM_TRY(check_desc(d, n));
  *out = *d;
  constexpr int small[3] = {8, 8, 16};
  const int64_t cells = (int64_t)d->mesh_shape[0] * d->mesh_shape[1] * d->mesh_shape[2];
  bool use = cells <= kSmallMesh && tiled_ok(d->mesh_shape, d->brick);
  for (int a = 0; a < 3; ++a) use = use && d->brick[a] % small[a] == 0;
  if (use)
    for (int a = 0; a < 3; ++a) out->brick[a] = small[a];
  return PM_SUCCESS;
}

// Tiled CIC scatter of the bucketed particles into mesh (whose every cell it writes): the
// constant particle value, or per-particle values vals (sorted order) with vscale[0] * |vals|
// <= 1; then, with fold, the neighbouring columns' upper x/y planes (otherwise the R2C pass that
// reads the mesh adds them: fold_planes).
int scatter_planes(const Bricks& k, const sort::Sorted& srt, float value, float* mesh, float* xs, float* ys,
                   const float* vals, const float* vscale, bool cic, const float* base, bool fold, hipStream_t s) {
  const Walk w = column_walk(k);
  auto launch = [&](auto kern, int threads) {
    hipLaunchKernelGGL(kern, w.grid, dim3(threads), 0, s, srt.rec, srt.bins, value, k, w.run, mesh, xs, ys, vals,
                       vscale, base);
  };
  if (cic && is_brick(k, 16, 16, 32))
    launch(k_scatter_columns<16, 16, 32, true>, BrickShape<16, 16, 32>::NT);
  else if (cic)  // cic_plan takes no other bricks
    launch(k_scatter_columns<8, 8, 16, true>, BrickShape<8, 8, 16>::NT);
  else if (is_brick(k, 16, 16, 32))
    launch(k_scatter_columns<16, 16, 32, false>, BrickShape<16, 16, 32>::NT);
  else if (is_brick(k, 8, 8, 16))
    launch(k_scatter_columns<8, 8, 16, false>, BrickShape<8, 8, 16>::NT);
  else
    launch(k_scatter_columns<0, 0, 0, false>, BrickShape<0, 0, 0>::NT);
  PM_LAUNCHED("k_scatter_columns", s);
  if (!fold) return PM_SUCCESS;
  const int64_t plane_cells = ((int64_t)k.nb[0] * k.n[1] + (int64_t)(k.n[0] - k.nb[0]) * k.nb[1]) * k.n[2];
  const unsigned blocks = (unsigned)std::max<int64_t>(1, std::min<int64_t>(ceil_div(plane_cells, kBlock), 8192));
  hipLaunchKernelGGL(k_fold_xy, dim3(blocks), dim3(kBlock), 0, s, k, xs, ys, mesh);
  PM_LAUNCHED("k_fold_xy", s);
  return PM_SUCCESS;
}

int scatter_tiled(const pm_gravity_desc* d, const Buffers& b, float* mesh, const float* vals, const float* vscale,
                  bool fold, hipStream_t s) {
  return scatter_planes(make_bricks(d->mesh_shape, d->brick), b.srt, d->particle_value, mesh, b.xs, b.ys, vals, vscale,
                        false, nullptr, fold, s);
}

// The plane buffers of an unfolded tiled scatter, for the R2C pass (mesh and brick extents are
// powers of two: the brick divides the mesh).
fft::FoldPlanes fold_planes(const pm_gravity_desc* d, const Buffers& b) {
  fft::FoldPlanes f;
  f.xs = b.xs;
  f.ys = b.ys;
  f.ny_log = fft::ilog2(d->mesh_shape[1]);
  f.b0_log = fft::ilog2(d->brick[0]);
  f.b1_log = fft::ilog2(d->brick[1]);
  f.nb0 = d->mesh_shape[0] / d->brick[0];
  f.nb1 = d->mesh_shape[1] / d->brick[1];
  return f;
}

// The particles binned by brick into the workspace's sorted copies (b.srt).
int bucket_stage(const int16_t* pmid, const float* disp, const uint8_t* valid, int64_t n,
                 const pm_gravity_desc* d, Buffers& b, hipStream_t s) {
  // the Lagrangian grid the particle count implies (mesh * cell / spacing per axis)
  int32_t grid[3] = {0, 0, 0};
  if (d->ptcl_spacing > 0.f)
    for (int a = 0; a < 3; ++a) {
      const double v = (double)d->mesh_shape[a] * d->cell_size / d->ptcl_spacing;
      grid[a] = (v >= 1.0 && v < 1e9) ? (int32_t)lrint(v) : 0;
    }
  return sort::bucket_cells(pmid, disp, valid, n, d->mesh_shape, d->cell_size, d->brick, grid, b.srt,
                            b.count, b.partial, true, s);
}

// Bucketing by brick (with the payload gathered into bucket order), then the density in b.r0; fold
// as for scatter_tiled.
int density_stage(const int16_t* pmid, const float* disp, const uint8_t* valid, int64_t n,
                  const pm_gravity_desc* d, const Layout& L, Buffers& b, bool fold, hipStream_t s) {
  const Geom g = step_geom(d);
  PM_TRY(bucket_stage(pmid, disp, valid, n, d, b, s));
  if (b.tiled) return scatter_tiled(d, b, b.r0, nullptr, nullptr, fold, s);
  PM_TRY(fill(b.r0, L.nreal, s));
  if (n > 0) {
    hipLaunchKernelGGL(k_scatter_sorted, dim3(grid_for(n)), dim3(kBlock), 0, s, b.srt.pmid, b.srt.disp, b.srt.valid,
                       n, d->particle_value, g, b.r0);
    PM_LAUNCHED("k_scatter_sorted", s);
  }
  return PM_SUCCESS;
}

int gather_stage(const uint8_t* valid, int64_t n, const pm_gravity_desc* d, const Buffers& b, const float* fx,
                 const float* fy, const float* fz, float* acc, hipStream_t s) {
  if (n == 0) return PM_SUCCESS;
  if (b.tiled) {
    Bricks k = make_bricks(d->mesh_shape, d->brick);
    const Walk w = column_walk(k);
    const int64_t nzero = valid ? n : 0;
    auto launch = [&](auto kern, int threads) {
      hipLaunchKernelGGL(kern, w.grid, dim3(threads), 0, s, b.srt.rec, b.srt.bins, b.srt.perm, k, w.run, fx, fy, fz,
                         nzero, acc);
    };
    if (is_brick(k, 16, 16, 32))
      launch(k_gather_columns<16, 16, 32>, BrickShape<16, 16, 32>::NT);
    else if (is_brick(k, 8, 8, 16))
      launch(k_gather_columns<8, 8, 16>, BrickShape<8, 8, 16>::NT);
    else
      launch(k_gather_columns<0, 0, 0>, BrickShape<0, 0, 0>::NT);
    PM_LAUNCHED("k_gather_columns", s);
    return PM_SUCCESS;
  }
  hipLaunchKernelGGL(k_gather3_sorted, dim3(grid_for(n)), dim3(kBlock), 0, s, b.srt.pmid, b.srt.disp, b.srt.valid,
                     b.srt.perm, n, step_geom(d), fx, fy, fz, acc);
  PM_LAUNCHED("k_gather3_sorted", s);
  return PM_SUCCESS;
}

int disp_cot_walk(const Bricks& k, const sort::Sorted& srt, float cell, const float* f0, const float* f1,
                  const float* f2, const float* dcot, const float* cot_s, int64_t n, float val, int64_t nzero,
                  int accum, float* disp_cot, hipStream_t s) {
  const Walk w = column_walk(k);
  auto launch = [&](auto kern, int threads) {
    hipLaunchKernelGGL(kern, w.grid, dim3(threads), 0, s, srt.rec, srt.bins, srt.perm, cell, k, w.run, f0, f1, f2, dcot,
                       cot_s, n, val, nzero, disp_cot, accum);
  };
  if (is_brick(k, 16, 16, 32))
    launch(k_disp_cot_columns<16, 16, 32>, BrickShape<16, 16, 32>::NT);
  else if (is_brick(k, 8, 8, 16))
    launch(k_disp_cot_columns<8, 8, 16>, BrickShape<8, 8, 16>::NT);
  else
    launch(k_disp_cot_columns<0, 0, 0>, BrickShape<0, 0, 0>::NT);
  PM_LAUNCHED("k_disp_cot_columns", s);
  return PM_SUCCESS;
}

// Tiled displacement cotangent of the reverse pass from the meshes f0, f1, f2 (null: none) and the
// density cotangent dcot, with the sorted acc_cot copies in b.cot_s; nzero = n: particles outside
// every brick (the invalid ones) get zero.  accum: added to disp_cot.
int disp_cot_tiled(const pm_gravity_desc* d, const Buffers& b, int64_t n, const float* f0, const float* f1,
                   const float* f2, const float* dcot, int64_t nzero, int accum, float* disp_cot, hipStream_t s) {
  return disp_cot_walk(make_bricks(d->mesh_shape, d->brick), b.srt, d->cell_size, f0, f1, f2, dcot,
                       f0 ? b.cot_s : nullptr, n, d->particle_value, nzero, accum, disp_cot, s);
}
// Density (b.r0) -> force meshes F_x (b.r0, or b.g0 when the density is kept), F_y (b.r1), F_z
// (b.r2); unfolded: b.r0's plane buffers are still to be added (scatter_tiled).
int force_mesh_stage(const pm_gravity_desc* d, const Layout& L, Buffers& b, const fft::SpecTables& tb,
                     hipStream_t s, bool keep_density, bool unfolded, const float* rho_add) {
  using namespace fft;
  const float coef = 1.5f * d->omega_m;  // 1.5 * Omega_m in float32 (gravity.py:630)
  const bool zband = L.nkz <= L.m;      // Nyquist column not stored
  const bool ypack = L.ky_keep >= 0;
  // every pass writes buffers other than those it reads (the passes with several outputs need it):
  //   A (s1) z r2c output, later chi = y inverse of psi (D_z applied by the z c2r)
  //   B (s2) y forward output (packed |ky| band)
  //   G (s2) psi = x inverse of the Green-multiplied spectrum
  //   C (s2) D_x psi
  //   E (s1) D_y chi
  //   H (s1) y inverse of D_x psi
  float2* A = b.ca;
  float2* B = b.cd;
  float2* G = b.cg;
  float2* C = b.cb;
  float2* E = b.ce;
  float2* H = b.cc;
  const int64_t p1 = L.pitch1;
  ZPass z1{};
  z1.rin = b.r0;
  z1.cmain[0] = A;
  z1.pitch_r = L.nz;
  z1.pitch_c = p1;
  z1.nlines = (int64_t)L.nx * L.ny;
  z1.src_shift = -1.f;
  z1.src_scale = coef;
  z1.rin_add = rho_add;  // learned density correction (null: none)
  if (unfolded && b.tiled) z1.fold = fold_planes(d, b);
  z1.kz_lim = L.nkz;
  z1.nyq = zband ? 0 : 1;
  PM_TRY(launch_z(L.nz, false, z1, tb, s));
  const int ncols = L.nkz;
  // y forward, packing the |ky| band when the filter allows it
  ColPass yf{A, B, nullptr, p1, 1, (int64_t)L.ny * p1, ncols, 0, 0, 0, 0, 0};
  yf.o_row = p1;
  yf.o_batch = (int64_t)L.nky * p1;
  yf.keep = L.ky_keep;
  PM_TRY(launch_cols(L.ny, kColFwd, yf, L.nx, tb, 1, s));
  // x: forward, Green, two inverses; columns are kz, batches are the (packed) ky rows
  ColPass xg{B, G, C, (int64_t)L.nky * p1, 1, p1, ncols, 1, 0, 0, 1, 0};
  if (ypack) {
    xg.ky_split = L.ky_keep;
    xg.ky_shift = L.ny - L.nky;
  }
  PM_TRY(launch_cols(L.nx, kColGreen, xg, L.nky, tb, 0, s));
  // the three y inverses expand the band back to full rows, in one launch
  ColPass yi{G, A, E, p1, 1, (int64_t)L.nky * p1, ncols, 0, 0, 0, 0, 0};
  yi.in1 = C;
  yi.out2 = H;
  yi.o_row = p1;
  yi.o_batch = (int64_t)L.ny * p1;
  yi.keep = L.ky_keep;
  yi.compact_in = 1;
  PM_TRY(launch_cols(L.ny, kColInv3, yi, L.nx, tb, 1, s));
  // the three c2r passes, in one launch
  ZPass zc{};
  zc.pitch_r = L.nz;
  zc.pitch_c = p1;
  zc.nlines = (int64_t)L.nx * L.ny;
  zc.out_scale = (float)(2.0 / ((double)L.nx * L.ny * L.nz));
  zc.kz_lim = L.nkz;
  zc.nyq = zband ? 0 : 1;
  zc.ncomp = 3;
  zc.cmain[0] = H;
  zc.cmain[1] = E;
  zc.cmain[2] = A;
  zc.rout[0] = keep_density ? b.g0 : b.r0;  // reverse keeps rho for the Omega_m cotangent
  zc.rout[1] = b.r1;
  zc.rout[2] = b.r2;
  zc.deriv = 1 << 2;  // D_z on the last component
  return launch_z(L.nz, true, zc, tb, s);
}

// Spectral adjoint of the force meshes: src_cot (b.g1, real) = irfftn(G * sum_i conj(D_i) *
// rfftn(g_i)) for the three cotangent meshes g_i (b.g1, b.g2, b.g3; the symbol is Hermitian, so
// the transpose of irfftn(H rfftn(.)) is irfftn(conj(H) rfftn(.))).  G * D_i vanishes outside
// the particle-Nyquist band, so the passes are force_mesh_stage's in reverse on the same band:
// three z r2c passes storing the kz band, three y passes packing the |ky| band, one x pass
// that transforms the three spectra, combines them mode by mode and inverts (kColAdj), the y
// inverse expanding the band and the z c2r.  Buffers: ca, cc, ce (s1) and cb, cd, cg (s2).
// adjoint_z_pass is component c's z r2c, taken right after its scatter (whose plane buffers it
// folds when unfolded).
int adjoint_z_pass(const pm_gravity_desc* d, const Layout& L, Buffers& b, const fft::SpecTables& tb, int c,
                   const float* mesh, bool unfolded, hipStream_t s) {
  using namespace fft;
  const bool zband = L.nkz <= L.m;
  float2* out[3] = {b.ca, b.cc, b.ce};
  ZPass zr{};
  zr.rin = mesh;
  zr.cmain[0] = out[c];
  zr.pitch_r = L.nz;
  zr.pitch_c = L.pitch1;
  zr.nlines = (int64_t)L.nx * L.ny;
  zr.src_shift = 0.f;
  zr.src_scale = 1.f;
  zr.kz_lim = L.nkz;
  zr.nyq = zband ? 0 : 1;
  if (unfolded) zr.fold = fold_planes(d, b);
  return launch_z(L.nz, false, zr, tb, s);
}

int adjoint_spectral_stage(const Layout& L, Buffers& b, const fft::SpecTables& tb, hipStream_t s) {
  using namespace fft;
  const bool zband = L.nkz <= L.m;
  const bool ypack = L.ky_keep >= 0;
  const int64_t p1 = L.pitch1;
  const int ncols = L.nkz;
  float2* s1buf[3] = {b.ca, b.cc, b.ce};
  float2* s2buf[3] = {b.cb, b.cd, b.cg};
  for (int c = 0; c < 3; ++c) {  // y forward, packed
    ColPass yf{s1buf[c], s2buf[c], nullptr, p1, 1, (int64_t)L.ny * p1, ncols, 0, 0, 0, 0, 0};
    yf.o_row = p1;
    yf.o_batch = (int64_t)L.nky * p1;
    yf.keep = L.ky_keep;
    PM_TRY(launch_cols(L.ny, kColFwd, yf, L.nx, tb, 1, s));
  }
  // x: three forward transforms, the combined symbol, one inverse -> cc (packed band)
  ColPass xa{s2buf[0], b.cc, nullptr, (int64_t)L.nky * p1, 1, p1, ncols, 1, 0, 0, 1, 0};
  xa.in1 = s2buf[1];
  xa.in2 = s2buf[2];
  if (ypack) {
    xa.ky_split = L.ky_keep;
    xa.ky_shift = L.ny - L.nky;
  }
  PM_TRY(launch_cols(L.nx, kColAdj, xa, L.nky, tb, 0, s));
  // y inverse expanding the band: cc -> ce
  ColPass yi{b.cc, b.ce, nullptr, p1, 1, (int64_t)L.nky * p1, ncols, 0, 0, 0, 0, 0};
  yi.o_row = p1;
  yi.o_batch = (int64_t)L.ny * p1;
  yi.keep = L.ky_keep;
  yi.compact_in = 1;
  PM_TRY(launch_cols(L.ny, kColInv, yi, L.nx, tb, 1, s));
  ZPass zc{};
  zc.pitch_r = L.nz;
  zc.pitch_c = p1;
  zc.nlines = (int64_t)L.nx * L.ny;
  zc.out_scale = (float)(2.0 / ((double)L.nx * L.ny * L.nz));
  zc.kz_lim = L.nkz;
  zc.nyq = zband ? 0 : 1;
  zc.cmain[0] = b.ce;
  zc.rout[0] = b.g1;
  zc.deriv = 0;
  return launch_z(L.nz, true, zc, tb, s);
}

// The particle-Nyquist-filtered potential of a real mesh on the force step's band:
// out = add + irfftn(mask * (-1/k^2) * rfftn(scale * (in + shift))).  With shift = -1 and
// scale = 1.5 Omega_m on a density mesh it is the potential of the force's source
// (gravity.py:626-633 with the Poisson and filter symbols of :174-196, 263-321); the operator
// is real and symmetric, so with shift = 0 it is also its own adjoint (a cotangent's path back
// to the source).  The passes are force_mesh_stage's for one output: z r2c storing the kz band
// (A), y forward packing the |ky| band (A -> B), the x pass with the Green multiply and one
// inverse (kColPot, B -> G), the y inverse expanding the band (G -> A), z c2r (+ add).
int potential_stage(const Layout& L, float2* A, float2* B, float2* G, const fft::SpecTables& tb, const float* in,
                    float shift, float scale, const float* add, float* out, hipStream_t s) {
  using namespace fft;
  const bool zband = L.nkz <= L.m;
  const int64_t p1 = L.pitch1;
  const int ncols = L.nkz;
  ZPass zr{};
  zr.rin = in;
  zr.cmain[0] = A;
  zr.pitch_r = L.nz;
  zr.pitch_c = p1;
  zr.nlines = (int64_t)L.nx * L.ny;
  zr.src_shift = shift;
  zr.src_scale = scale;
  zr.kz_lim = L.nkz;
  zr.nyq = zband ? 0 : 1;
  PM_TRY(launch_z(L.nz, false, zr, tb, s));
  ColPass yf{A, B, nullptr, p1, 1, (int64_t)L.ny * p1, ncols, 0, 0, 0, 0, 0};
  yf.o_row = p1;
  yf.o_batch = (int64_t)L.nky * p1;
  yf.keep = L.ky_keep;
  PM_TRY(launch_cols(L.ny, kColFwd, yf, L.nx, tb, 1, s));
  ColPass xp{B, G, nullptr, (int64_t)L.nky * p1, 1, p1, ncols, 1, 0, 0, 1, 0};
  if (L.ky_keep >= 0) {
    xp.ky_split = L.ky_keep;
    xp.ky_shift = L.ny - L.nky;
  }
  PM_TRY(launch_cols(L.nx, kColPot, xp, L.nky, tb, 0, s));
  ColPass yi{G, A, nullptr, p1, 1, (int64_t)L.nky * p1, ncols, 0, 0, 0, 0, 0};
  yi.o_row = p1;
  yi.o_batch = (int64_t)L.ny * p1;
  yi.keep = L.ky_keep;
  yi.compact_in = 1;
  PM_TRY(launch_cols(L.ny, kColInv, yi, L.nx, tb, 1, s));
  ZPass zc{};
  zc.pitch_r = L.nz;
  zc.pitch_c = p1;
  zc.nlines = (int64_t)L.nx * L.ny;
  zc.out_scale = (float)(2.0 / ((double)L.nx * L.ny * L.nz));
  zc.kz_lim = L.nkz;
  zc.nyq = zband ? 0 : 1;
  zc.cmain[0] = A;
  zc.rout[0] = out;
  zc.rout_add = add;
  zc.deriv = 0;
  return launch_z(L.nz, true, zc, tb, s);
}

size_t potential_workspace_bytes(const pm_gravity_desc* d) {
  const Layout L = make_layout(d);
  return align_up(sizeof(float) * fft::spec_table_floats(d->mesh_shape), 256) +
         align_up(sizeof(float2) * L.s1, 256) * 2 + align_up(sizeof(float2) * L.s2, 256) + 256;
}

int prepare(const pm_gravity_desc* d, int64_t n, void* workspace, size_t workspace_bytes_, bool reverse,
            Layout& L, Buffers& b, Arena& ws, fft::SpecTables& tb, hipStream_t s) {
  PM_TRY(check_desc(d, n));
  PM_TRY(require_device_tables());
  size_t need = workspace_bytes(d, n, reverse);
  PM_RETURN_IF(workspace == nullptr || workspace_bytes_ < need, PM_ERROR_WORKSPACE,
               "gravity workspace too small: need " + std::to_string(need) + " bytes");
  L = make_layout(d);
  PM_RETURN_IF(!carve(ws, L, n, d->mesh_shape, d->brick, reverse, b), PM_ERROR_WORKSPACE,
               "workspace carve failed");
  const fft::SpecTables sc = fft::spec_scalars(d->cell_size, d->ptcl_spacing, d->mask_active);
  // the bucketing's counters are cleared along (unused by the calls that resume)
  PM_TRY(fft::launch_spec_tables(b.tables, d->mesh_shape, sc, b.count,
                                 sort::bucket_count_len(d->mesh_shape, d->brick), s));
  tb = fft::spec_tables_view(b.tables, d->mesh_shape, sc);
  return PM_SUCCESS;
}

// ---------------------------------------------------------------- tiled CIC seam ----
// The scatter and the gather adjoint of the kernel seam (pm_cic.hip) through the force step's
// binning and column kernels, for one-channel meshes without offset, drops or a cell size of their
// own.  Float atomics run at 23-27 G/s here (128^3 displaced particles onto a 256^3 mesh: 744 us with
// the copy of the mesh); binning the particles (56 us), ordering their values (10), adding each brick up
// in LDS (36) and the column planes (11) take 122 us.
//
// Precision: a deposit is the float32 product v W of the atomics' kernel, and a cell's deposits are added in
// float64 and rounded once per column that touches it, where float atomics round at every addition; so the
// range of the values, zeros, infinities and NaN need no rule.  (Fixed point in units of the largest
// value, tried first, cost the cells far below it their bits: one value 2^16 times the others left 1.2e-4
// rms in the cells without it.)
//
// The values in sorted order.
__global__ void __launch_bounds__(kBlock) k_cic_values(const int32_t* __restrict__ perm,
                                                       const int32_t* __restrict__ bins, int nbins,
                                                       const float* __restrict__ val, float* __restrict__ val_s) {
  const int64_t n = bins[nbins];  // the valid ones
  for (int64_t j = (int64_t)blockIdx.x * kBlock + threadIdx.x; j < n; j += (int64_t)gridDim.x * kBlock)
    val_s[j] = val[perm[j]];
}

struct CicPlan {
  Bricks k;
  int32_t brick[3];
  int64_t cells;
};

// Whether a call takes the tiled path: one channel, no offset, the particles' own cell size, the whole
// periodic mesh, axes in whole bricks, enough particles for the launches and enough per cell for the
// passes over the mesh.  Atomics / tiled, us, of 64^3 particles with normal displacements of 1.5 cells, onto
// meshes of 64^3: 87 / 48, 128^3: 97 / 39, 256^3: 122 / 61, 384^3: 195 / 207, 512^3: 339 / 340; 96^3 on
// 512^3: 551 / 358; 128^3 on 128^3: 704 / 97.
constexpr int64_t kCicTiled = int64_t(1) << 18;
constexpr int64_t kCicSparse = 128;
bool cic_plan(const pm_cic_geom* g, int64_t n, int32_t channels, CicPlan* p) {
  if (channels != 1 || n < kCicTiled || n > INT32_MAX || g->mesh_cell > 0.f) return false;
  p->cells = 1;
  for (int a = 0; a < 3; ++a) {
    if (g->offset[a] != 0.f || g->local_shape[a] != g->global_shape[a] || g->local_shape[a] < 1) return false;
    p->cells *= g->local_shape[a];
  }
  if (p->cells > kCicSparse * n) return false;
  constexpr int32_t large[3] = {16, 16, 32}, small[3] = {8, 8, 16};
  const int32_t* br = nullptr;
  if (p->cells > kSmallMesh && tiled_ok(g->local_shape, large)) br = large;
  if (p->cells <= kSmallMesh && tiled_ok(g->local_shape, small)) br = small;
  if (!br || sort::check_sort_args(n, g->local_shape, br) != PM_SUCCESS) return false;
  for (int a = 0; a < 3; ++a) p->brick[a] = br[a];
  p->k = make_bricks(g->local_shape, br);
  return true;
}

struct CicBuffers {
  sort::Sorted srt;
  int32_t *count, *partial;
  float *xs, *ys, *val_s;
};

bool cic_carve(Arena& ws, const pm_cic_geom* g, const CicPlan& p, int64_t n, CicBuffers& b) {
  const int64_t counters = sort::bucket_count_len(g->local_shape, p.brick);
  b.count = ws.take<int32_t>(counters);
  b.partial = ws.take<int32_t>(sort::bucket_partials(counters));
  b.srt.bins = ws.take<int32_t>((int64_t)p.k.nb[0] * p.k.nb[1] * p.k.nb[2] + 2);
  b.srt.perm = ws.take<int32_t>(n);
  b.srt.rec = ws.take<float4>(n);
  b.xs = ws.take<float>(xs_floats(p.k));
  b.ys = ws.take<float>(ys_floats(p.k));
  b.val_s = ws.take<float>(n);
  return ws.ok();
}

size_t cic_bytes(const pm_cic_geom* g, const CicPlan& p, int64_t n) {
  Arena probe(reinterpret_cast<void*>(uintptr_t(256)), SIZE_MAX / 2);
  CicBuffers b{};
  cic_carve(probe, g, p, n, b);
  return probe.used + 256;
}

// out = base + sum val W (val null: val_scalar) through the tiles.
int cic_scatter_tiled(const int16_t* pmid, const float* disp, const uint8_t* valid, const float* val, float val_scalar,
                      int64_t n, const pm_cic_geom* g, const CicPlan& p, const float* base, float* out, CicBuffers& b,
                      hipStream_t s) {
  // a cube's particles in C order are the usual state: a hint for the binning's chunks only
  const int32_t c = (int32_t)lrint(std::cbrt((double)n));
  const int32_t grid[3] = {c, c, c};
  PM_TRY(sort::bucket_cells(pmid, disp, valid, n, g->local_shape, g->particle_cell, p.brick, grid, b.srt, b.count,
                            b.partial, false, s));
  if (val) {
    const int nbins = p.k.nb[0] * p.k.nb[1] * p.k.nb[2];
    const unsigned nb = (unsigned)std::min<int64_t>(ceil_div(n, kBlock), 1024);
    hipLaunchKernelGGL(k_cic_values, dim3(nb), dim3(kBlock), 0, s, b.srt.perm, b.srt.bins, nbins, val, b.val_s);
    PM_LAUNCHED("k_cic_values", s);
  }
  return scatter_planes(p.k, b.srt, val_scalar, out, b.xs, b.ys, val ? b.val_s : nullptr, nullptr, true, base, true, s);
}

}  // namespace
}  // namespace grav
}  // namespace pm

using namespace pm;

extern "C" {

int pm_gravity_workspace(const pm_gravity_desc* desc, int64_t n, size_t* bytes) {
  pm_gravity_desc eff;
  PM_TRY(grav::effective_desc(desc, n, &eff));
  PM_RETURN_IF(bytes == nullptr, PM_ERROR_INVALID_ARGUMENT, "bytes is NULL");
  *bytes = grav::workspace_bytes(&eff, n, false);
  return PM_SUCCESS;
}

int pm_gravity_vjp_workspace(const pm_gravity_desc* desc, int64_t n, size_t* bytes) {
  pm_gravity_desc eff;
  PM_TRY(grav::effective_desc(desc, n, &eff));
  PM_RETURN_IF(bytes == nullptr, PM_ERROR_INVALID_ARGUMENT, "bytes is NULL");
  *bytes = grav::workspace_bytes(&eff, n, true);
  return PM_SUCCESS;
}

int pm_gravity(const int16_t* pmid, const float* disp, const uint8_t* valid, int64_t n,
               const pm_gravity_desc* desc, float* acc, void* workspace, size_t workspace_bytes,
               void* stream) {
  return pm_gravity_corrected(pmid, disp, valid, n, desc, nullptr, acc, workspace, workspace_bytes, stream);
}

int pm_gravity_corrected(const int16_t* pmid, const float* disp, const uint8_t* valid, int64_t n,
                         const pm_gravity_desc* desc, const float* rho_add, float* acc, void* workspace,
                         size_t workspace_bytes, void* stream) {
  hipStream_t s = as_stream(stream);
  pm_gravity_desc eff;
  PM_TRY(grav::effective_desc(desc, n, &eff));
  desc = &eff;
  grav::Layout L;
  grav::Buffers b{};
  Arena ws(workspace, workspace_bytes);
  fft::SpecTables tb;
  int st = grav::prepare(desc, n, workspace, workspace_bytes, false, L, b, ws, tb, s);
  if (st) return st;
  PM_RETURN_IF(n > 0 && (pmid == nullptr || disp == nullptr || acc == nullptr), PM_ERROR_INVALID_ARGUMENT,
               "pmid/disp/acc NULL");
  st = grav::density_stage(pmid, disp, valid, n, desc, L, b, false, s);
  if (st) return st;
  st = grav::force_mesh_stage(desc, L, b, tb, s, false, true, rho_add);
  if (st) return st;
  return grav::gather_stage(valid, n, desc, b, b.r0, b.r1, b.r2, acc, s);
}

int pm_gravity_corrected_resume(const int16_t* pmid, const float* disp, const uint8_t* valid, int64_t n,
                                const pm_gravity_desc* desc, const float* rho_add, float* acc, void* workspace,
                                size_t workspace_bytes, void* stream) {
  hipStream_t s = as_stream(stream);
  pm_gravity_desc eff;
  PM_TRY(grav::effective_desc(desc, n, &eff));
  desc = &eff;
  grav::Layout L;
  grav::Buffers b{};
  Arena ws(workspace, workspace_bytes);
  fft::SpecTables tb;
  // the same carve as the pm_gravity_density call: the bucketed particles and the density
  // mesh it left are at the same places
  int st = grav::prepare(desc, n, workspace, workspace_bytes, false, L, b, ws, tb, s);
  if (st) return st;
  PM_RETURN_IF(n > 0 && (pmid == nullptr || disp == nullptr || acc == nullptr), PM_ERROR_INVALID_ARGUMENT,
               "pmid/disp/acc NULL");
  st = grav::force_mesh_stage(desc, L, b, tb, s, false, false, rho_add);
  if (st) return st;
  return grav::gather_stage(valid, n, desc, b, b.r0, b.r1, b.r2, acc, s);
}

int pm_gravity_density_offset(const pm_gravity_desc* desc, int64_t n, size_t* offset) {
  pm_gravity_desc eff;
  PM_TRY(grav::effective_desc(desc, n, &eff));
  desc = &eff;
  PM_RETURN_IF(offset == nullptr, PM_ERROR_INVALID_ARGUMENT, "offset is NULL");
  // the forward carve on a stand-in base (never dereferenced): prepare() carves from the
  // workspace start in the same order, so the density's offset is the same there
  char* const base = reinterpret_cast<char*>(uintptr_t(1) << 12);
  Arena ws(base, SIZE_MAX / 2);
  grav::Buffers b{};
  const grav::Layout L = grav::make_layout(desc);
  PM_RETURN_IF(!grav::carve(ws, L, n, desc->mesh_shape, desc->brick, false, b), PM_ERROR_WORKSPACE,
               "workspace carve failed");
  *offset = (size_t)(reinterpret_cast<char*>(b.r0) - base);
  return PM_SUCCESS;
}

int pm_gravity_density(const int16_t* pmid, const float* disp, const uint8_t* valid, int64_t n,
                       const pm_gravity_desc* desc, float* rho, void* workspace, size_t workspace_bytes,
                       void* stream) {
  hipStream_t s = as_stream(stream);
  pm_gravity_desc eff;
  PM_TRY(grav::effective_desc(desc, n, &eff));
  desc = &eff;
  grav::Layout L;
  grav::Buffers b{};
  Arena ws(workspace, workspace_bytes);
  fft::SpecTables tb;
  int st = grav::prepare(desc, n, workspace, workspace_bytes, false, L, b, ws, tb, s);
  if (st) return st;
  PM_RETURN_IF(rho == nullptr || (n > 0 && (pmid == nullptr || disp == nullptr)), PM_ERROR_INVALID_ARGUMENT,
               "pmid/disp/rho NULL");
  st = grav::density_stage(pmid, disp, valid, n, desc, L, b, true, s);
  if (st) return st;
  if (rho == b.r0) return PM_SUCCESS;  // the caller reads the density in place (pm_gravity_density_offset)
  if (((reinterpret_cast<uintptr_t>(rho) | reinterpret_cast<uintptr_t>(b.r0)) & 15) == 0) {
    hipLaunchKernelGGL(grav::k_copy_mesh, dim3(2048), dim3(grav::kBlock), 0, s, b.r0, rho, (int64_t)L.nreal);
    PM_LAUNCHED("k_copy_mesh", s);
  } else {
    PM_HIP_TRY(hipMemcpyAsync(rho, b.r0, sizeof(float) * L.nreal, hipMemcpyDeviceToDevice, s));
  }
  return PM_SUCCESS;
}

int pm_gravity_vjp(const int16_t* pmid, const float* disp, const uint8_t* valid, int64_t n,
                   const pm_gravity_desc* desc, const float* acc_cot, float* disp_cot,
                   float* omega_cot, void* workspace, size_t workspace_bytes, void* stream) {
  return pm_gravity_corrected_vjp(pmid, disp, valid, n, desc, nullptr, acc_cot, disp_cot, omega_cot, nullptr,
                                  workspace, workspace_bytes, stream);
}

// The force VJP; with resume, the forward meshes (and the bucketed particles) are those a
// pm_gravity_keep call left in the same workspace for the same particles.
static int vjp_impl(const int16_t* pmid, const float* disp, const uint8_t* valid, int64_t n,
                    const pm_gravity_desc* desc, const float* rho_add, const float* acc_cot, float* disp_cot,
                    float* omega_cot, float* rho_cot, void* workspace, size_t workspace_bytes, void* stream,
                    bool resume) {
  hipStream_t s = as_stream(stream);
  pm_gravity_desc eff;
  PM_TRY(grav::effective_desc(desc, n, &eff));
  desc = &eff;
  grav::Layout L;
  grav::Buffers b{};
  Arena ws(workspace, workspace_bytes);
  fft::SpecTables tb;
  int st = grav::prepare(desc, n, workspace, workspace_bytes, true, L, b, ws, tb, s);
  if (st) return st;
  PM_RETURN_IF(n > 0 && (pmid == nullptr || disp == nullptr || acc_cot == nullptr || disp_cot == nullptr),
               PM_ERROR_INVALID_ARGUMENT, "pmid/disp/acc_cot/disp_cot NULL");
  PM_RETURN_IF(omega_cot == nullptr, PM_ERROR_INVALID_ARGUMENT, "omega_cot NULL");
  const Geom g = grav::step_geom(desc);
  // recompute the forward meshes: rho stays in r0, F_x goes to g0, F_y r1, F_z r2
  if (!resume) {
    st = grav::density_stage(pmid, disp, valid, n, desc, L, b, true, s);
    if (st) return st;
    st = grav::force_mesh_stage(desc, L, b, tb, s, true, false, rho_add);
    if (st) return st;
  }
  // gather^T: acc_cot scattered into three cotangent meshes, displacement cotangent from F.
  // With brick tiling each component goes through the tiled scatter (sorted, scaled copies of
  // acc_cot); otherwise through float atomics beside the displacement cotangent.
  // The tiled path takes the displacement cotangent after the spectral adjoint, in one pass
  // over F and the density cotangent.
  if (b.tiled) {
    const unsigned nb = (unsigned)std::max<int64_t>(1, std::min<int64_t>(ceil_div(n, grav::kBlock), grav::kCotBlocks));
    hipLaunchKernelGGL(grav::k_cot_sorted, dim3(nb), dim3(grav::kBlock), 0, s, b.srt.perm, acc_cot, n, b.cot_s,
                       b.cot_pmax);
    PM_LAUNCHED("k_cot_sorted", s);
    hipLaunchKernelGGL(grav::k_cot_scale, dim3(1), dim3(64), 0, s, b.cot_pmax, (int)nb, b.cot_pmax + grav::kCotBlocks);
    PM_LAUNCHED("k_cot_scale", s);
    float* gm[3] = {b.g1, b.g2, b.g3};
    for (int c = 0; c < 3; ++c) {
      st = grav::scatter_tiled(desc, b, gm[c], b.cot_s + (int64_t)c * n, b.cot_pmax + grav::kCotBlocks, false, s);
      if (st) return st;
      st = grav::adjoint_z_pass(desc, L, b, tb, c, gm[c], true, s);
      if (st) return st;
    }
  } else {
    st = grav::fill(b.g1, L.nreal, s);
    if (st) return st;
    st = grav::fill(b.g2, L.nreal, s);
    if (st) return st;
    st = grav::fill(b.g3, L.nreal, s);
    if (st) return st;
    if (n > 0) {
      hipLaunchKernelGGL(grav::k_gather3_bwd_sorted, dim3(grav::grid_for(n)), dim3(grav::kBlock), 0, s,
                         b.srt.pmid, b.srt.disp, b.srt.valid, b.srt.perm, n, g, b.g0, b.r1, b.r2, acc_cot, b.g1, b.g2, b.g3,
                         b.disp_cot_s);
      PM_LAUNCHED("k_gather3_bwd_sorted", s);
    }
    float* gm[3] = {b.g1, b.g2, b.g3};
    for (int c = 0; c < 3; ++c) PM_TRY(grav::adjoint_z_pass(desc, L, b, tb, c, gm[c], false, s));
  }
  // spectral adjoint: src_cot (g1) = irfftn(G * sum_i conj(D_i) rfftn(g_i)) on the band
  st = grav::adjoint_spectral_stage(L, b, tb, s);
  if (st) return st;
  {
    const float coef = 1.5f * desc->omega_m;
    const unsigned blocks =
        (unsigned)std::max<int64_t>(1, std::min<int64_t>(ceil_div(L.nreal, grav::kBlock * 16), grav::kSrcBlocks));
    hipLaunchKernelGGL(grav::k_source_bwd, dim3(blocks), dim3(grav::kBlock), 0, s, b.g1, b.r0, rho_add, rho_cot,
                       L.nreal, coef, b.src_part);
    PM_LAUNCHED("k_source_bwd", s);
    hipLaunchKernelGGL(grav::k_source_bwd_sum, dim3(1), dim3(64), 0, s, b.src_part, (int)blocks, omega_cot);
    PM_LAUNCHED("k_source_bwd_sum", s);
  }
  if (n > 0 && b.tiled)
    return grav::disp_cot_tiled(desc, b, n, b.g0, b.r1, b.r2, b.g1, valid ? n : 0, 0, disp_cot, s);
  if (n > 0) {
    hipLaunchKernelGGL(grav::k_scatter_bwd_sorted, dim3(grav::grid_for(n)), dim3(grav::kBlock), 0, s, b.srt.pmid,
                       b.srt.disp, b.srt.valid, b.srt.perm, n, g, desc->particle_value, b.g1, b.disp_cot_s, disp_cot);
    PM_LAUNCHED("k_scatter_bwd_sorted", s);
  }
  return PM_SUCCESS;
}

int pm_gravity_corrected_vjp(const int16_t* pmid, const float* disp, const uint8_t* valid, int64_t n,
                             const pm_gravity_desc* desc, const float* rho_add, const float* acc_cot,
                             float* disp_cot, float* omega_cot, float* rho_cot, void* workspace,
                             size_t workspace_bytes, void* stream) {
  return vjp_impl(pmid, disp, valid, n, desc, rho_add, acc_cot, disp_cot, omega_cot, rho_cot, workspace,
                  workspace_bytes, stream, false);
}

int pm_gravity_keep(const int16_t* pmid, const float* disp, const uint8_t* valid, int64_t n,
                    const pm_gravity_desc* desc, float* acc, void* workspace, size_t workspace_bytes, void* stream) {
  hipStream_t s = as_stream(stream);
  pm_gravity_desc eff;
  PM_TRY(grav::effective_desc(desc, n, &eff));
  desc = &eff;
  grav::Layout L;
  grav::Buffers b{};
  Arena ws(workspace, workspace_bytes);
  fft::SpecTables tb;
  // the VJP's carve: the meshes stay where pm_gravity_vjp_resume finds them
  int st = grav::prepare(desc, n, workspace, workspace_bytes, true, L, b, ws, tb, s);
  if (st) return st;
  PM_RETURN_IF(n > 0 && (pmid == nullptr || disp == nullptr || acc == nullptr), PM_ERROR_INVALID_ARGUMENT,
               "pmid/disp/acc NULL");
  st = grav::density_stage(pmid, disp, valid, n, desc, L, b, true, s);
  if (st) return st;
  st = grav::force_mesh_stage(desc, L, b, tb, s, true, false, nullptr);
  if (st) return st;
  return grav::gather_stage(valid, n, desc, b, b.g0, b.r1, b.r2, acc, s);
}

int pm_gravity_vjp_resume(const int16_t* pmid, const float* disp, const uint8_t* valid, int64_t n,
                          const pm_gravity_desc* desc, const float* acc_cot, float* disp_cot, float* omega_cot,
                          void* workspace, size_t workspace_bytes, void* stream) {
  return vjp_impl(pmid, disp, valid, n, desc, nullptr, acc_cot, disp_cot, omega_cot, nullptr, workspace,
                  workspace_bytes, stream, true);
}

int pm_gravity_density_cot(const int16_t* pmid, const float* disp, const uint8_t* valid, int64_t n,
                           const pm_gravity_desc* desc, const float* dens_cot, float* disp_cot, void* workspace,
                           size_t workspace_bytes, void* stream) {
  hipStream_t s = as_stream(stream);
  pm_gravity_desc eff;
  PM_TRY(grav::effective_desc(desc, n, &eff));
  desc = &eff;
  grav::Layout L;
  grav::Buffers b{};
  Arena ws(workspace, workspace_bytes);
  fft::SpecTables tb;
  int st = grav::prepare(desc, n, workspace, workspace_bytes, false, L, b, ws, tb, s);
  if (st) return st;
  PM_RETURN_IF(n > 0 && (pmid == nullptr || disp == nullptr || dens_cot == nullptr || disp_cot == nullptr),
               PM_ERROR_INVALID_ARGUMENT, "pmid/disp/dens_cot/disp_cot NULL");
  if (n == 0) return PM_SUCCESS;
  PM_TRY(grav::bucket_stage(pmid, disp, valid, n, desc, b, s));
  const Geom g = grav::step_geom(desc);
  if (b.tiled)  // invalid particles are in no bin: their disp_cot stays as it is
    return grav::disp_cot_tiled(desc, b, n, nullptr, nullptr, nullptr, dens_cot, 0, 1, disp_cot, s);
  hipLaunchKernelGGL(grav::k_scatter_bwd_sorted, dim3(grav::grid_for(n)), dim3(grav::kBlock), 0, s, b.srt.pmid,
                     b.srt.disp, b.srt.valid, b.srt.perm, n, g, desc->particle_value, dens_cot, nullptr, disp_cot);
  PM_LAUNCHED("k_scatter_bwd_sorted", s);
  return PM_SUCCESS;
}

int pm_potential_workspace(const pm_gravity_desc* desc, size_t* bytes) {
  PM_TRY(grav::check_desc(desc, 0));
  PM_RETURN_IF(bytes == nullptr, PM_ERROR_INVALID_ARGUMENT, "bytes is NULL");
  *bytes = grav::potential_workspace_bytes(desc);
  return PM_SUCCESS;
}

int pm_gravity_potential(const float* in, float shift, float scale, const float* add, const pm_gravity_desc* desc,
                         float* out, void* workspace, size_t workspace_bytes, void* stream) {
  PM_TRY(grav::check_desc(desc, 0));
  PM_TRY(require_device_tables());
  PM_RETURN_IF(in == nullptr || out == nullptr, PM_ERROR_INVALID_ARGUMENT, "NULL mesh");
  const size_t need = grav::potential_workspace_bytes(desc);
  PM_RETURN_IF(workspace == nullptr || workspace_bytes < need, PM_ERROR_WORKSPACE,
               "potential workspace too small: need " + std::to_string(need) + " bytes");
  hipStream_t s = as_stream(stream);
  const grav::Layout L = grav::make_layout(desc);
  Arena ws(workspace, workspace_bytes);
  float* tables = ws.take<float>(fft::spec_table_floats(desc->mesh_shape));
  float2* A = ws.take<float2>(L.s1);
  float2* G = ws.take<float2>(L.s1);
  float2* B = ws.take<float2>(L.s2);
  PM_RETURN_IF(!ws.ok(), PM_ERROR_WORKSPACE, "potential workspace carve failed");
  const fft::SpecTables sc = fft::spec_scalars(desc->cell_size, desc->ptcl_spacing, desc->mask_active);
  PM_TRY(fft::launch_spec_tables(tables, desc->mesh_shape, sc, nullptr, 0, s));
  const fft::SpecTables tb = fft::spec_tables_view(tables, desc->mesh_shape, sc);
  return grav::potential_stage(L, A, B, G, tb, in, shift, scale, add, out, s);
}

int pm_spectral_workspace(const pm_gravity_desc* desc, size_t* bytes) {
  PM_RETURN_IF(desc == nullptr || bytes == nullptr, PM_ERROR_INVALID_ARGUMENT, "NULL argument");
  PM_RETURN_IF(!fft::supported_shape(desc->mesh_shape), PM_ERROR_UNSUPPORTED,
               "mesh axes must be powers of two in [2, 2048]");
  *bytes = align_up(sizeof(float) * fft::spec_table_floats(desc->mesh_shape), 256);
  return PM_SUCCESS;
}

int pm_spectral_force_multiply(const float* in_complex, float* out_complex, const pm_gravity_desc* desc,
                               int32_t axis, int32_t adjoint, void* workspace, size_t workspace_bytes,
                               void* stream) {
  PM_RETURN_IF(desc == nullptr || in_complex == nullptr || out_complex == nullptr,
               PM_ERROR_INVALID_ARGUMENT, "NULL argument");
  PM_RETURN_IF(axis < -1 || axis > 2, PM_ERROR_INVALID_ARGUMENT, "axis must be -1, 0, 1 or 2");
  size_t need = 0;
  int st = pm_spectral_workspace(desc, &need);
  if (st) return st;
  PM_RETURN_IF(desc->mask_active && !(desc->ptcl_spacing > 0.f), PM_ERROR_INVALID_ARGUMENT,
               "ptcl_spacing must be positive when the particle-Nyquist mask is active");
  PM_RETURN_IF(!(desc->cell_size > 0.f), PM_ERROR_INVALID_ARGUMENT, "cell_size must be positive");
  PM_RETURN_IF(workspace == nullptr || workspace_bytes < need, PM_ERROR_WORKSPACE,
               "spectral workspace too small: need " + std::to_string(need) + " bytes");
  hipStream_t s = as_stream(stream);
  float* tables = static_cast<float*>(workspace);
  const fft::SpecTables sc = fft::spec_scalars(desc->cell_size, desc->ptcl_spacing, desc->mask_active);
  st = fft::launch_spec_tables(tables, desc->mesh_shape, sc, nullptr, 0, s);
  if (st) return st;
  fft::SpecTables tb = fft::spec_tables_view(tables, desc->mesh_shape, sc);
  return fft::launch_spectral_multiply(reinterpret_cast<const float2*>(in_complex),
                                       reinterpret_cast<float2*>(out_complex), desc->mesh_shape, tb, axis,
                                       adjoint, s);
}

int pm_cic_tiled_workspace(int64_t n, int32_t channels, const pm_cic_geom* geom, size_t* bytes) {
  PM_RETURN_IF(geom == nullptr || bytes == nullptr, PM_ERROR_INVALID_ARGUMENT, "NULL argument");
  grav::CicPlan p;
  *bytes = grav::cic_plan(geom, n, channels, &p) ? grav::cic_bytes(geom, p, n) : 0;
  return PM_SUCCESS;
}

static int cic_prepare(const int16_t* pmid, const float* disp, int64_t n, const pm_cic_geom* geom, void* workspace,
                       size_t workspace_bytes, grav::CicPlan& p, grav::CicBuffers& b) {
  PM_RETURN_IF(geom == nullptr || pmid == nullptr || disp == nullptr, PM_ERROR_INVALID_ARGUMENT, "NULL argument");
  PM_RETURN_IF(!(geom->particle_cell > 0.f), PM_ERROR_INVALID_ARGUMENT, "particle_cell must be positive");
  PM_RETURN_IF(!grav::cic_plan(geom, n, 1, &p), PM_ERROR_UNSUPPORTED, "pm_cic_tiled_workspace is 0 for this call");
  const size_t need = grav::cic_bytes(geom, p, n);
  PM_RETURN_IF(workspace == nullptr || workspace_bytes < need, PM_ERROR_WORKSPACE,
               "CIC workspace too small: need " + std::to_string(need) + " bytes");
  Arena ws(workspace, workspace_bytes);
  PM_RETURN_IF(!grav::cic_carve(ws, geom, p, n, b), PM_ERROR_WORKSPACE, "CIC workspace carve failed");
  return PM_SUCCESS;
}

int pm_cic_scatter_tiled(const int16_t* pmid, const float* disp, const uint8_t* valid, const float* val,
                         float val_scalar, int64_t n, const pm_cic_geom* geom, const float* base, float* mesh,
                         void* workspace, size_t workspace_bytes, void* stream) {
  grav::CicPlan p;
  grav::CicBuffers b{};
  PM_TRY(cic_prepare(pmid, disp, n, geom, workspace, workspace_bytes, p, b));
  PM_RETURN_IF(mesh == nullptr || mesh == base, PM_ERROR_INVALID_ARGUMENT, "mesh must be given and differ from base");
  PM_RETURN_IF(((reinterpret_cast<uintptr_t>(mesh) | reinterpret_cast<uintptr_t>(base)) & 15) != 0,
               PM_ERROR_INVALID_ARGUMENT, "meshes must be 16-byte aligned");
  return grav::cic_scatter_tiled(pmid, disp, valid, val, val_scalar, n, geom, p, base, mesh, b, as_stream(stream));
}

int pm_cic_gather_bwd_tiled(const int16_t* pmid, const float* disp, const uint8_t* valid, int64_t n,
                            const pm_cic_geom* geom, const float* mesh, const float* val_cot, float* disp_cot,
                            float* mesh_cot, void* workspace, size_t workspace_bytes, void* stream) {
  grav::CicPlan p;
  grav::CicBuffers b{};
  PM_TRY(cic_prepare(pmid, disp, n, geom, workspace, workspace_bytes, p, b));
  PM_RETURN_IF(mesh == nullptr || val_cot == nullptr || disp_cot == nullptr || mesh_cot == nullptr,
               PM_ERROR_INVALID_ARGUMENT, "NULL argument");
  PM_RETURN_IF(((reinterpret_cast<uintptr_t>(mesh) | reinterpret_cast<uintptr_t>(mesh_cot)) & 15) != 0,
               PM_ERROR_INVALID_ARGUMENT, "meshes must be 16-byte aligned");
  hipStream_t s = as_stream(stream);
  PM_TRY(grav::cic_scatter_tiled(pmid, disp, valid, val_cot, 0.f, n, geom, p, nullptr, mesh_cot, b, s));
  return grav::disp_cot_walk(p.k, b.srt, geom->particle_cell, mesh, nullptr, nullptr, nullptr, b.val_s, n, 0.f,
                             valid ? n : 0, 0, disp_cot, s);
}

}  // extern "C"
