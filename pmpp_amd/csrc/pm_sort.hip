// Stable, deterministic cell sort (least-significant-digit radix, digits of up to 10 bits).
//
// Each pass is a stable counting sort of one digit:
//   1. k_digit_hist   one wave per contiguous segment of kSeg items counts its digits;
//   2. exclusive scan of the digit-major (digit, segment) count matrix;
//   3. k_digit_scatter the same waves walk their segment in order, rank each item among
//      equal digits of its 64-item group with ballot masks, and place it at
//      offset[digit][segment] + running count -- input order is preserved inside every
//      key, so the result equals numpy.argsort(keys, kind="stable") bit for bit.
// The key of the first pass is computed on the fly from (pmid, disp): the raveled brick
// index of the containing cell, with invalid particles mapped to the sentinel.
#include <algorithm>
#include <atomic>
#include <type_traits>

#include "pm_common.h"
#include "pm_sort.h"

namespace pm {
namespace sort {
namespace {

constexpr int kWave = 64;
constexpr int kWavesPerBlock = 4;
constexpr int kIters = 128;               // 64-item groups per segment
constexpr int kSeg = kWave * kIters;      // items per wave segment
constexpr int kMaxDigitBits = 10;
constexpr int kMaxRadix = 1 << kMaxDigitBits;

struct KeyGeom {
  int n[3];
  int b[3];
  int nb[3];
  int nshift[3];  // log2(n) when n is a power of two, else -1
  int bshift[3];  // log2(b) when b is a power of two, else -1
  float cell;
  int sentinel;
};

__device__ __forceinline__ int cell_key(const KeyGeom& g, const int16_t* __restrict__ pmid,
                                        const float* __restrict__ disp,
                                        const uint8_t* __restrict__ valid, int64_t i) {
  if (valid && !valid[i]) return g.sentinel;
  int c[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    // containing cell: the CIC base index with offset 0 (cic/pallas.py:227-236)
    float t = disp[i * 3 + a] / g.cell;
    int base = (int)pmid[i * 3 + a] + (int)floorf(t);
    int cell = g.nshift[a] >= 0 ? (base & (g.n[a] - 1)) : pos_mod(base, g.n[a]);
    c[a] = g.bshift[a] >= 0 ? (cell >> g.bshift[a]) : cell / g.b[a];
  }
  return (c[0] * g.nb[1] + c[1]) * g.nb[2] + c[2];
}

template <bool FIRST>
__global__ void __launch_bounds__(kWave * kWavesPerBlock)
    k_digit_hist(const int32_t* __restrict__ keys, const int16_t* __restrict__ pmid,
                 const float* __restrict__ disp, const uint8_t* __restrict__ valid, KeyGeom g,
                 int64_t n, int shift, int dbits, int64_t nseg, int32_t* __restrict__ hist) {
  __shared__ int32_t h[kWavesPerBlock][kMaxRadix];
  const int lane = threadIdx.x % kWave;
  const int w = threadIdx.x / kWave;
  const int radix = 1 << dbits;
  for (int d = lane; d < radix; d += kWave) h[w][d] = 0;
  __syncthreads();
  const int64_t seg = (int64_t)blockIdx.x * kWavesPerBlock + w;
  if (seg < nseg) {
    // equal digits of a 64-item group are counted by their lowest lane (ballot match), so the
    // wave-private row h[w] needs no atomics and nearly sorted keys do not serialise on one bank
    const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    const int64_t start = seg * kSeg;
    for (int it = 0; it < kIters; ++it) {
      int64_t i = start + it * kWave + lane;
      bool active = i < n;
      int key = 0;
      if (active) key = FIRST ? cell_key(g, pmid, disp, valid, i) : keys[i];
      int d = (key >> shift) & (radix - 1);
      uint64_t peers = __ballot(active);
      for (int bit = 0; bit < dbits; ++bit) {
        bool set = (d >> bit) & 1;
        uint64_t m = __ballot(set);
        peers &= set ? m : ~m;
      }
      if (active && (peers & lt_mask) == 0) h[w][d] += __popcll(peers);
      __builtin_amdgcn_wave_barrier();
    }
  }
  __syncthreads();
  if (seg < nseg)
    for (int d = lane; d < radix; d += kWave) hist[(int64_t)d * nseg + seg] = h[w][d];
}

template <bool FIRST>
__global__ void __launch_bounds__(kWave * kWavesPerBlock)
    k_digit_scatter(const int32_t* __restrict__ keys_in, const int32_t* __restrict__ vals_in,
                    const int16_t* __restrict__ pmid, const float* __restrict__ disp,
                    const uint8_t* __restrict__ valid, KeyGeom g, int64_t n, int shift, int dbits,
                    int64_t nseg, const int32_t* __restrict__ offsets, int32_t* __restrict__ keys_out,
                    int32_t* __restrict__ vals_out) {
  __shared__ int32_t cnt[kWavesPerBlock][kMaxRadix];
  const int lane = threadIdx.x % kWave;
  const int w = threadIdx.x / kWave;
  const int radix = 1 << dbits;
  const int64_t seg = (int64_t)blockIdx.x * kWavesPerBlock + w;
  if (seg >= nseg) return;  // whole wave exits together; no block barriers below
  for (int d = lane; d < radix; d += kWave) cnt[w][d] = offsets[(int64_t)d * nseg + seg];
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  const int64_t start = seg * kSeg;
  for (int it = 0; it < kIters; ++it) {
    int64_t i = start + it * kWave + lane;
    bool active = i < n;
    int key = 0, val = 0;
    if (active) {
      if (FIRST) {
        key = cell_key(g, pmid, disp, valid, i);
        val = (int)i;
      } else {
        key = keys_in[i];
        val = vals_in[i];
      }
    }
    int d = (key >> shift) & (radix - 1);
    uint64_t peers = __ballot(active);
    for (int bit = 0; bit < dbits; ++bit) {
      bool set = (d >> bit) & 1;
      uint64_t m = __ballot(set);
      peers &= set ? m : ~m;
    }
    int rank = __popcll(peers & lt_mask);
    int base = 0;
    if (active) base = cnt[w][d];
    __builtin_amdgcn_wave_barrier();
    if (active) {
      int pos = base + rank;
      if (keys_out) keys_out[pos] = key;
      vals_out[pos] = val;
      if (rank == 0) cnt[w][d] = base + __popcll(peers);
    }
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  }
}

// ---- exclusive scan of int32 counts (3 phases) ----
// Where the scan's results go.  Plain (tail = nullptr): out[i].  Bucketing: the counters are `first`
// bricks, kTails counters of invalid particles and an end marker; out takes the bricks' offsets, the
// invalid bucket's start and the end (out[first + 1]), tail the start of each invalid counter's share.
constexpr int kTails = 64;
struct ScanOut {
  int32_t* out;
  int32_t* tail = nullptr;
  int64_t first = 0;
  __device__ __forceinline__ void put(int64_t i, int32_t v) const {
    if (!tail || i < first) {
      out[i] = v;
      return;
    }
    const int64_t k = i - first;
    if (k == 0) out[first] = v;
    if (k < kTails)
      tail[k] = v;
    else
      out[first + 1] = v;
  }
};

constexpr int kScanBlock = 256;
constexpr int kScanPer = 16;
constexpr int kScanChunk = kScanBlock * kScanPer;

__device__ __forceinline__ int32_t block_exclusive_scan(int32_t v, int32_t* sh, int32_t& total) {
  const int t = threadIdx.x;
  sh[t] = v;
  __syncthreads();
  for (int off = 1; off < kScanBlock; off <<= 1) {
    int32_t a = t >= off ? sh[t - off] : 0;
    __syncthreads();
    sh[t] += a;
    __syncthreads();
  }
  total = sh[kScanBlock - 1];
  int32_t ex = sh[t] - v;
  __syncthreads();
  return ex;
}

__global__ void __launch_bounds__(kScanBlock) k_scan_reduce(const int32_t* __restrict__ in, int64_t len,
                                                            int32_t* __restrict__ partial) {
  __shared__ int32_t sh[kScanBlock];
  int64_t base = (int64_t)blockIdx.x * kScanChunk + threadIdx.x * kScanPer;
  int32_t s = 0;
  for (int j = 0; j < kScanPer; ++j)
    if (base + j < len) s += in[base + j];
  int32_t total;
  block_exclusive_scan(s, sh, total);
  if (threadIdx.x == 0) partial[blockIdx.x] = total;
}

__global__ void __launch_bounds__(kScanBlock) k_scan_partials(int32_t* __restrict__ partial, int64_t len) {
  __shared__ int32_t sh[kScanBlock];
  int32_t carry = 0;
  for (int64_t base = 0; base < len; base += kScanBlock) {
    int64_t i = base + threadIdx.x;
    int32_t v = i < len ? partial[i] : 0;
    int32_t total;
    int32_t ex = block_exclusive_scan(v, sh, total);
    if (i < len) partial[i] = carry + ex;
    carry += total;
  }
}

__global__ void __launch_bounds__(kScanBlock) k_scan_apply(const int32_t* __restrict__ in, int64_t len,
                                                           const int32_t* __restrict__ partial, ScanOut out) {
  __shared__ int32_t sh[kScanBlock];
  int64_t base = (int64_t)blockIdx.x * kScanChunk + threadIdx.x * kScanPer;
  int32_t vals[kScanPer];
  int32_t s = 0;
  for (int j = 0; j < kScanPer; ++j) {
    vals[j] = (base + j < len) ? in[base + j] : 0;
    s += vals[j];
  }
  int32_t total;
  int32_t ex = block_exclusive_scan(s, sh, total) + partial[blockIdx.x];
  for (int j = 0; j < kScanPer; ++j) {
    if (base + j < len) out.put(base + j, ex);
    ex += vals[j];
  }
}

// bin_offsets[b] = first sorted position with key >= b, for b in [0, num_keys]
__global__ void k_bin_bounds(const int32_t* __restrict__ keys, int64_t n, int num_keys,
                             int32_t* __restrict__ bounds) {
  int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j > n) return;
  int lo = (j == 0) ? 0 : keys[j - 1] + 1;
  int hi = (j == n) ? num_keys : keys[j];
  for (int b = lo; b <= hi; ++b) bounds[b] = (int32_t)j;
}

// sorted payload: pmid_s[j] = pmid[perm[j]], disp_s[j] = disp[perm[j]] (either may be null)
__global__ void k_gather_payload(const int32_t* __restrict__ perm, const int16_t* __restrict__ pmid,
                                 const float* __restrict__ disp, int64_t n, int16_t* __restrict__ pmid_s,
                                 float* __restrict__ disp_s) {
  for (int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; j < n; j += (int64_t)gridDim.x * blockDim.x) {
    const int64_t i = perm[j];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      if (pmid_s) pmid_s[j * 3 + a] = pmid[i * 3 + a];
      if (disp_s) disp_s[j * 3 + a] = disp[i * 3 + a];
    }
  }
}

// The same scan in one launch: each workgroup sums everything before its chunk of 4096 itself
// instead of waiting for partials.  The last of 33 workgroups reads 512 KB from L2 for the
// 131,074 bricks of a 1024^3 mesh; the three launches it replaces took 15 us there and 9 us on a
// 64^3 mesh (32 bricks).
constexpr int kScan1Threads = 1024;
constexpr int64_t kScan1Max = 1 << 18;  // beyond it the sums of what came before cost more than two launches
__global__ void __launch_bounds__(kScan1Threads) k_scan_one(const int32_t* __restrict__ in, int64_t len,
                                                            ScanOut out) {
  __shared__ int32_t loc[kScan1Threads / 64], pre[kScan1Threads / 64];
  const int t = threadIdx.x, lane = t % 64, wave = t / 64;
  const int64_t base = (int64_t)blockIdx.x * kScanChunk;
  const int4* in4 = reinterpret_cast<const int4*>(in);  // chunk starts are 16-byte aligned
  int32_t before = 0;
#pragma unroll 8
  for (int64_t i = t; i < base / 4; i += kScan1Threads) {
    const int4 v = in4[i];
    before += (v.x + v.y) + (v.z + v.w);
  }
  int32_t v[4], s = 0;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int64_t i = base + 4 * t + j;
    v[j] = i < len ? in[i] : 0;
    s += v[j];
  }
  int32_t inc = s;
  for (int off = 1; off < 64; off <<= 1) {
    const int32_t u = __shfl_up(inc, off);
    if (lane >= off) inc += u;
  }
  for (int off = 32; off > 0; off >>= 1) before += __shfl_xor(before, off);
  if (lane == 63) loc[wave] = inc;
  if (lane == 0) pre[wave] = before;
  __syncthreads();
  int32_t ex = inc - s;
  for (int w = 0; w < kScan1Threads / 64; ++w) ex += pre[w] + (w < wave ? loc[w] : 0);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int64_t i = base + 4 * t + j;
    if (i < len) out.put(i, ex);
    ex += v[j];
  }
}
static_assert(kScan1Threads * 4 == kScanChunk, "four counts per thread");

int scan_exclusive(const int32_t* in, const ScanOut& out, int64_t len, int32_t* partial, hipStream_t s) {
  if (len == 0) return PM_SUCCESS;
  if (len <= kScan1Max && reinterpret_cast<uintptr_t>(in) % 16 == 0) {
    hipLaunchKernelGGL(k_scan_one, dim3((unsigned)ceil_div(len, kScanChunk)), dim3(kScan1Threads), 0, s, in, len, out);
    PM_LAUNCHED("scan", s);
    return PM_SUCCESS;
  }
  int64_t blocks = ceil_div(len, kScanChunk);
  hipLaunchKernelGGL(k_scan_reduce, dim3((unsigned)blocks), dim3(kScanBlock), 0, s, in, len, partial);
  hipLaunchKernelGGL(k_scan_partials, dim3(1), dim3(kScanBlock), 0, s, partial, blocks);
  hipLaunchKernelGGL(k_scan_apply, dim3((unsigned)blocks), dim3(kScanBlock), 0, s, in, len, partial, out);
  PM_LAUNCHED("scan", s);
  return PM_SUCCESS;
}

KeyGeom make_key_geom(const int32_t* mesh_shape, float cell, const int32_t* brick) {
  KeyGeom g;
  int64_t nbins = 1;
  auto log2_or_neg = [](int v) {
    if (v <= 0 || (v & (v - 1))) return -1;
    int l = 0;
    while ((1 << l) < v) ++l;
    return l;
  };
  for (int a = 0; a < 3; ++a) {
    g.n[a] = mesh_shape[a];
    g.b[a] = brick[a];
    g.nb[a] = (int)ceil_div(mesh_shape[a], brick[a]);
    g.nshift[a] = log2_or_neg(mesh_shape[a]);
    g.bshift[a] = log2_or_neg(brick[a]);
    nbins *= g.nb[a];
  }
  g.cell = cell;
  g.sentinel = (int)nbins;
  return g;
}

// ---- unstable bucketing by key (the gravity step's binning) ----
// The order inside a bucket depends on atomic arrival order, which the tile kernels do not
// see: the scatter sums in exact integer arithmetic and the gather is per particle.
//
// A particle's brick key and, for REC, its record (pm_sort.h): the containing cell's local place in
// the brick as a tile offset, and the fractions t - floor(t) of the CIC weights.
template <bool REC>
__device__ __forceinline__ int raw_cell_key(const KeyGeom& g, const int p[3], const float d[3], bool ok, float4& rec) {
  int c[3], l[3];
  float f[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const float t = d[a] / g.cell;  // the same float32 arithmetic as cell_key and the CIC base cell
    const float lf = floorf(t);
    const int base = p[a] + (int)lf;
    const int cell = g.nshift[a] >= 0 ? (base & (g.n[a] - 1)) : pos_mod(base, g.n[a]);
    c[a] = g.bshift[a] >= 0 ? (cell >> g.bshift[a]) : cell / g.b[a];
    l[a] = cell - c[a] * g.b[a];
    f[a] = t - lf;
  }
  if constexpr (REC)
    rec = make_float4(f[0], f[1], f[2], __uint_as_float(rec_bits(l[0], l[1], l[2], g.b[1], g.b[2])));
  return ok ? (c[0] * g.nb[1] + c[1]) * g.nb[2] + c[2] : g.sentinel;
}

// Bucketing in chunks of NT x 4 x GROUPS particles per workgroup: keys are aggregated in an LDS hash
// table (as many slots as particles, so the linear probe always ends), then one global atomic
// per distinct key and chunk reserves that key's range, and the chunk's particles of one key are
// written contiguously by one workgroup.  A thread takes four consecutive particles at a time: six
// 16- and 8-byte loads instead of 24 scalar ones (when the arrays are so aligned), and a run of
// equal keys among them claims its slot and its ranks once.  When the particles are a whole
// Lagrangian grid in C order (the usual PM state), a chunk is a block of 64 along z of that grid,
// which falls into a few bricks, so a chunk needs only a handful of global atomics and its writes
// fill cache lines (blocks at the grid's upper edges may be partly empty; grids that would leave
// more than 30 % of the slots empty count as index ranges); otherwise chunks are contiguous index
// ranges.  The mapping only affects speed:
// every partition of the particles gives a valid (unstable) bucketing.
//
// Invalid particles would all reserve from one counter, at ~13 ns per chunk and atomic: with every
// 16th of 180^3 slots unused that was most of both passes (83 + 90 us; the whole force 644 us).  They
// are counted in kTails counters instead, chunk c in counter c mod kTails, whose shares the scan lays
// one after the other (the force 608 us).
//
// Bound by HBM and by the latency of a chunk's phases.  512^3 particles: count 0.69 -> 0.52 ms, place
// 2.20 -> 1.55 ms (20 bytes written per particle as two stores, 23 as eight before; 5.1 GB at 3.3
// TB/s).
struct ChunkMap {
  int64_t n;
  int64_t nchunks;
  int tiled;       // 1: BX x BY x 64 blocks of a (g0, g1, g2) particle grid
  int g0, g1, g2;  // grid extents (tiled)
  int nby, nbz;  // blocks along y and z (tiled)
  int vec;       // pmid 8-, disp 16- and valid 4-byte aligned
};

// Chunk shapes by size: level 2 is 4 x 8 x 64 particles on 256 threads; level 1 half of it, which
// holds half the registers and so does not leave a second round of workgroups nearly empty on
// medium problems; level 0 is 2 x 4 x 64 on 128 threads, so that small problems fill the chip
// (32^3 particles: 64 workgroups instead of 16).
template <int LEVEL>
struct ChunkCfg {
  static constexpr int NT = LEVEL == 0 ? 128 : 256;
  static constexpr int GROUPS = LEVEL == 2 ? 2 : 1;  // groups of 4 consecutive particles per thread
  static constexpr int CHUNK = NT * 4 * GROUPS;
  static constexpr int BX = LEVEL == 0 ? 2 : 4, BY = LEVEL == 2 ? 8 : 4;
  static_assert(BX * BY * 64 == CHUNK, "tiled chunk");
  static constexpr int SLOT_BITS = LEVEL == 0 ? 10 : 11;
  static constexpr int SLOTS = 1 << SLOT_BITS;
  static_assert(SLOTS >= CHUNK, "the probe must end");
};
constexpr int kRankBits = 12;  // ranks go up to the largest chunk
// The level for n particles.  Measured (count + place, us): 32^3 particles levels 0 and 2: 20, 25;
// 64^3: 24, 30; 128^3 levels 1 and 2: 58, 62; 512^3: 2143, 2074 (the larger chunk's fewer global
// atomics).  Index ranges cross more bricks per chunk, which favours the largest sooner (180^3:
// 189 against 151; 100^3: 36 against 39).
inline int chunk_level(int64_t n, bool grid) {
  if (n <= (int64_t(1) << 19)) return 0;
  return n <= (int64_t(1) << (grid ? 24 : 21)) ? 1 : 2;
}

// first particle of group q (of 4 consecutive ones) of chunk c, and how many of the 4 there are
template <int LEVEL>
__device__ __forceinline__ int64_t chunk_index(const ChunkMap& m, int64_t c, int q, int& live) {
  using C = ChunkCfg<LEVEL>;
  if (!m.tiled) {
    const int64_t i = c * C::CHUNK + 4 * (int64_t)q;
    live = (int)max(int64_t(0), min(int64_t(4), m.n - i));
    return i;
  }
  const int bz = (int)(c % m.nbz);
  const int64_t r = c / m.nbz;
  const int by = (int)(r % m.nby);
  const int bx = (int)(r / m.nby);
  const int row = q >> 4;  // rows of 64 particles, 16 groups each
  const int ix = bx * C::BX + row / C::BY, iy = by * C::BY + row % C::BY, iz = bz * 64 + 4 * (q & 15);
  live = ix < m.g0 && iy < m.g1 ? max(0, min(4, m.g2 - iz)) : 0;
  return ((int64_t)ix * m.g1 + iy) * m.g2 + iz;
}

template <bool PLACE, bool REC, int LEVEL>
__global__ void __launch_bounds__(ChunkCfg<LEVEL>::NT)
    k_bucket(const int16_t* __restrict__ pmid, const float* __restrict__ disp, const uint8_t* __restrict__ valid,
             KeyGeom g, ChunkMap m, int32_t* __restrict__ count, const int32_t* __restrict__ bins,
             int32_t* __restrict__ perm, int16_t* __restrict__ pmid_s, float* __restrict__ disp_s,
             uint8_t* __restrict__ valid_s, float4* __restrict__ rec_s, const int32_t* __restrict__ tail) {
  using C = ChunkCfg<LEVEL>;
  constexpr int NT = C::NT, G = C::GROUPS, SLOTS = C::SLOTS;
  __shared__ int s_key[SLOTS];
  __shared__ int s_cnt[SLOTS];  // count per slot, then (PLACE) the slot's first destination
  const int t = threadIdx.x;
  for (int h = t; h < SLOTS; h += NT) {
    s_key[h] = -1;
    s_cnt[h] = 0;
  }
  __syncthreads();
  for (int64_t c = blockIdx.x; c < m.nchunks; c += gridDim.x) {
    int code[G * 4];
    // the placing pass keeps each particle in registers between its two phases: its record, or
    // the raw pmid (packed with the valid flag) and disp
    float4 rec[PLACE ? G * 4 : 1];
    uint32_t pk[PLACE && !REC ? G * 4 : 1];
    short4 pr[G][3];
    float4 dr[G][3];
    uchar4 vr[G];
    int live[G];
    // all groups' loads first (in flight together); a group that is not whole, or unaligned
    // arrays, take clamped scalar loads
#pragma unroll
    for (int u = 0; u < G; ++u) {
      const int64_t i0 = chunk_index<LEVEL>(m, c, t + u * NT, live[u]);
      vr[u] = make_uchar4(1, 1, 1, 1);
      if (m.vec && live[u] == 4 && (i0 & 3) == 0) {
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          pr[u][a] = reinterpret_cast<const short4*>(pmid + i0 * 3)[a];
          dr[u][a] = reinterpret_cast<const float4*>(disp + i0 * 3)[a];
        }
        if (valid) vr[u] = *reinterpret_cast<const uchar4*>(valid + i0);
      } else {
        auto at = [&](int64_t i) { return i < m.n ? i : m.n - 1; };
        auto pm = [&](int e) { return pmid[at(i0 + e / 3) * 3 + e % 3]; };
        auto dp = [&](int e) { return disp[at(i0 + e / 3) * 3 + e % 3]; };
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          pr[u][a] = make_short4(pm(4 * a), pm(4 * a + 1), pm(4 * a + 2), pm(4 * a + 3));
          dr[u][a] = make_float4(dp(4 * a), dp(4 * a + 1), dp(4 * a + 2), dp(4 * a + 3));
        }
        if (valid) vr[u] = make_uchar4(valid[at(i0)], valid[at(i0 + 1)], valid[at(i0 + 2)], valid[at(i0 + 3)]);
      }
    }
#pragma unroll
    for (int u = 0; u < G; ++u) {
      const int pf[12] = {pr[u][0].x, pr[u][0].y, pr[u][0].z, pr[u][0].w, pr[u][1].x, pr[u][1].y,
                          pr[u][1].z, pr[u][1].w, pr[u][2].x, pr[u][2].y, pr[u][2].z, pr[u][2].w};
      const float df[12] = {dr[u][0].x, dr[u][0].y, dr[u][0].z, dr[u][0].w, dr[u][1].x, dr[u][1].y,
                            dr[u][1].z, dr[u][1].w, dr[u][2].x, dr[u][2].y, dr[u][2].z, dr[u][2].w};
      const uint8_t vf[4] = {vr[u].x, vr[u].y, vr[u].z, vr[u].w};
      int key[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int p[3] = {pf[3 * e], pf[3 * e + 1], pf[3 * e + 2]};
        const float d[3] = {df[3 * e], df[3 * e + 1], df[3 * e + 2]};
        float4 r;
        key[e] = raw_cell_key<REC>(g, p, d, vf[e] != 0, r);
        if (key[e] == g.sentinel) key[e] += (int)(c % kTails);
        if (e >= live[u]) key[e] = -1;  // no such particle: no bin
        if constexpr (PLACE) {
          if constexpr (REC) {
            rec[u * 4 + e] = r;
          } else {
            rec[u * 4 + e] = make_float4(d[0], d[1], d[2],
                                         __uint_as_float(((uint32_t)p[0] & 0xffffu) | ((uint32_t)p[1] << 16)));
            pk[u * 4 + e] = ((uint32_t)p[2] & 0xffffu) | ((uint32_t)vf[e] << 16);
          }
        }
      }
      // runs of equal keys: length of the run that starts at e
      int len[4];
      len[3] = 1;
#pragma unroll
      for (int e = 2; e >= 0; --e) len[e] = key[e + 1] == key[e] ? len[e + 1] + 1 : 1;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (e > 0 && key[e] == key[e - 1]) {  // continues the run: next rank of the same slot
          code[u * 4 + e] = code[u * 4 + e - 1] + (key[e] >= 0 ? 1 : 0);
          continue;
        }
        code[u * 4 + e] = -1;
        if (key[e] >= 0) {
          unsigned h = ((unsigned)key[e] * 2654435761u) >> (32 - C::SLOT_BITS);
          for (;;) {
            const int prev = atomicCAS(&s_key[h], -1, key[e]);
            if (prev == -1 || prev == key[e]) break;
            h = (h + 1) & (SLOTS - 1);
          }
          code[u * 4 + e] = ((int)h << kRankBits) | atomicAdd(&s_cnt[h], len[e]);
        }
      }
    }
    __syncthreads();
    for (int h = t; h < SLOTS; h += NT) {
      const int k = s_key[h];
      if (k >= 0) {
        const int cnt = s_cnt[h];
        if (PLACE)  // count[k] counts down from the bin's total: no second clearing of the counters
          s_cnt[h] = (k < g.sentinel ? bins[k] : tail[k - g.sentinel]) + atomicSub(&count[k], cnt) - cnt;
        else
          atomicAdd(&count[k], cnt);
      }
    }
    __syncthreads();
    if constexpr (PLACE) {
#pragma unroll
      for (int e = 0; e < G * 4; ++e) {
        if (code[e] < 0) continue;
        int unused;
        const int64_t i = chunk_index<LEVEL>(m, c, t + (e / 4) * NT, unused) + e % 4;
        const int dest = s_cnt[code[e] >> kRankBits] + (code[e] & ((1 << kRankBits) - 1));
        perm[dest] = (int32_t)i;
        if constexpr (REC) {
          rec_s[dest] = rec[e];
        } else {
          const uint32_t pk0 = __float_as_uint(rec[e].w);
          pmid_s[(int64_t)dest * 3 + 0] = (int16_t)(pk0 & 0xffffu);
          pmid_s[(int64_t)dest * 3 + 1] = (int16_t)(pk0 >> 16);
          pmid_s[(int64_t)dest * 3 + 2] = (int16_t)(pk[e] & 0xffffu);
          disp_s[(int64_t)dest * 3 + 0] = rec[e].x;
          disp_s[(int64_t)dest * 3 + 1] = rec[e].y;
          disp_s[(int64_t)dest * 3 + 2] = rec[e].z;
          valid_s[dest] = (uint8_t)(pk[e] >> 16);
        }
      }
    }
    __syncthreads();
    if (c + gridDim.x < m.nchunks) {
      for (int h = t; h < SLOTS; h += NT) {
        s_key[h] = -1;
        s_cnt[h] = 0;
      }
      __syncthreads();
    }
  }
}

inline bool is_grid(int64_t n, const int32_t* grid) {
  return grid && n > 0 && (int64_t)grid[0] * grid[1] * grid[2] == n;
}

template <int LEVEL>
ChunkMap make_chunk_map(const int16_t* pmid, const float* disp, const uint8_t* valid, int64_t n, const int32_t* grid) {
  using C = ChunkCfg<LEVEL>;
  ChunkMap m{};
  m.n = n;
  m.vec = reinterpret_cast<uintptr_t>(pmid) % 8 == 0 && reinterpret_cast<uintptr_t>(disp) % 16 == 0 &&
          reinterpret_cast<uintptr_t>(valid) % 4 == 0;
  const int64_t blocks =
      grid ? ceil_div(grid[0], C::BX) * ceil_div(grid[1], C::BY) * ceil_div(grid[2], 64) : 0;
  if (is_grid(n, grid) && n * 10 >= blocks * C::CHUNK * 7) {
    m.tiled = 1;
    m.g0 = grid[0];
    m.g1 = grid[1];
    m.g2 = grid[2];
    m.nby = (int)ceil_div(grid[1], C::BY);
    m.nbz = (int)ceil_div(grid[2], 64);
    m.nchunks = blocks;
  } else {
    m.nchunks = ceil_div(n, C::CHUNK);
  }
  return m;
}

__global__ void k_zero_i32(int32_t* __restrict__ p, int64_t len) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < len; i += (int64_t)gridDim.x * blockDim.x)
    p[i] = 0;
}

int key_bits(int64_t max_key) {
  int b = 1;
  while ((int64_t(1) << b) <= max_key) ++b;
  return b;
}

}  // namespace

int64_t bucket_count_len(const int32_t* mesh_shape, const int32_t* brick) {
  int64_t nbins = 1;
  for (int a = 0; a < 3; ++a) nbins *= ceil_div(mesh_shape[a], brick[a]);
  return nbins + kTails + 1;  // bricks, invalid particles, the end
}

int64_t bucket_partials(int64_t len) { return ceil_div(len, kScanChunk) + 1 + kTails; }

size_t bucket_workspace_bytes(const int32_t* mesh_shape, const int32_t* brick) {
  const int64_t len = bucket_count_len(mesh_shape, brick);
  return align_up(sizeof(int32_t) * len, 256) + align_up(sizeof(int32_t) * bucket_partials(len), 256);
}

template <bool REC, int LEVEL>
static int launch_bucket(const int16_t* pmid, const float* disp, const uint8_t* valid, int64_t n, const KeyGeom& g,
                         const int32_t* ptcl_grid, const Sorted& out, int32_t* count, int32_t* partial, int64_t len,
                         hipStream_t s) {
  int32_t* tail = partial + bucket_partials(len) - kTails;
  const ChunkMap m = make_chunk_map<LEVEL>(pmid, disp, valid, n, ptcl_grid);
  const dim3 grid((unsigned)std::max<int64_t>(1, std::min<int64_t>(m.nchunks, 4096)));
  const dim3 block(ChunkCfg<LEVEL>::NT);
  if (n > 0) {
    hipLaunchKernelGGL((k_bucket<false, false, LEVEL>), grid, block, 0, s, pmid, disp, valid, g, m, count,
                       (const int32_t*)nullptr, (int32_t*)nullptr, (int16_t*)nullptr, (float*)nullptr,
                       (uint8_t*)nullptr, (float4*)nullptr, (const int32_t*)nullptr);
    PM_LAUNCHED("k_bucket_count", s);
  }
  PM_TRY(scan_exclusive(count, ScanOut{out.bins, tail, g.sentinel}, len, partial, s));
  if (n > 0) {
    hipLaunchKernelGGL((k_bucket<true, REC, LEVEL>), grid, block, 0, s, pmid, disp, valid, g, m, count,
                       (const int32_t*)out.bins, out.perm, out.pmid, out.disp, out.valid, out.rec,
                       (const int32_t*)tail);
    PM_LAUNCHED("k_bucket_place", s);
  }
  return PM_SUCCESS;
}

int bucket_cells(const int16_t* pmid, const float* disp, const uint8_t* valid, int64_t n, const int32_t* mesh_shape,
                 float cell_size, const int32_t* brick, const int32_t* ptcl_grid, const Sorted& out, int32_t* count,
                 int32_t* partial, bool cleared, hipStream_t s) {
  KeyGeom g = make_key_geom(mesh_shape, cell_size, brick);
  const int64_t len = bucket_count_len(mesh_shape, brick);
  if (!cleared) {
    const unsigned zb = (unsigned)std::min<int64_t>(ceil_div(len, 256), 1024);
    hipLaunchKernelGGL(k_zero_i32, dim3(zb), dim3(256), 0, s, count, len);
    PM_LAUNCHED("k_zero_i32", s);
  }
  auto launch = [&](auto rec) {
    constexpr bool REC = decltype(rec)::value;
    const int level = chunk_level(n, is_grid(n, ptcl_grid));
    if (level == 0) return launch_bucket<REC, 0>(pmid, disp, valid, n, g, ptcl_grid, out, count, partial, len, s);
    if (level == 1) return launch_bucket<REC, 1>(pmid, disp, valid, n, g, ptcl_grid, out, count, partial, len, s);
    return launch_bucket<REC, 2>(pmid, disp, valid, n, g, ptcl_grid, out, count, partial, len, s);
  };
  return out.rec ? launch(std::true_type{}) : launch(std::false_type{});
}

// The same with the counters and scan partials carved from an arena.
static int bucket_cells_arena(const int16_t* pmid, const float* disp, const uint8_t* valid, int64_t n,
                              const int32_t* mesh_shape, float cell_size, const int32_t* brick,
                              const int32_t* ptcl_grid, int32_t* perm, int32_t* bin_offsets, int16_t* pmid_s,
                              float* disp_s, uint8_t* valid_s, Arena& ws, hipStream_t s) {
  const int64_t len = bucket_count_len(mesh_shape, brick);
  int32_t* count = ws.take<int32_t>(len);
  int32_t* partial = ws.take<int32_t>(bucket_partials(len));
  PM_RETURN_IF(!ws.ok(), PM_ERROR_WORKSPACE, "bucket workspace too small");
  Sorted out;
  out.perm = perm;
  out.bins = bin_offsets;
  out.pmid = pmid_s;
  out.disp = disp_s;
  out.valid = valid_s;
  return bucket_cells(pmid, disp, valid, n, mesh_shape, cell_size, brick, ptcl_grid, out, count, partial, false, s);
}

int check_sort_args(int64_t n, const int32_t* mesh_shape, const int32_t* brick) {
  PM_RETURN_IF(n < 0 || n > INT32_MAX, PM_ERROR_UNSUPPORTED, "particle count must be in [0, 2^31)");
  PM_RETURN_IF(mesh_shape == nullptr || brick == nullptr, PM_ERROR_INVALID_ARGUMENT, "NULL shape");
  int64_t nbins = 1;
  for (int a = 0; a < 3; ++a) {
    PM_RETURN_IF(mesh_shape[a] < 1 || brick[a] < 1, PM_ERROR_INVALID_ARGUMENT,
                 "mesh_shape and brick must be positive");
    nbins *= ceil_div(mesh_shape[a], brick[a]);
  }
  PM_RETURN_IF(nbins >= INT32_MAX, PM_ERROR_UNSUPPORTED,
               "more than 2^31-1 bricks: use a coarser brick for this mesh");
  return PM_SUCCESS;
}

size_t workspace_bytes(int64_t n, const int32_t* mesh_shape, const int32_t* brick) {
  int64_t nseg = ceil_div(n, kSeg);
  int64_t hist = (int64_t)kMaxRadix * nseg;
  size_t b = 0;
  b += align_up(sizeof(int32_t) * n, 256) * 3;  // keys a/b, vals
  b += align_up(sizeof(int32_t) * hist, 256) * 2;
  b += align_up(sizeof(int32_t) * (ceil_div(hist, kScanChunk) + 1), 256);
  (void)mesh_shape;
  (void)brick;
  return b + 256;
}

int digit_bits_for(int bits, int& passes) {
  passes = (bits + kMaxDigitBits - 1) / kMaxDigitBits;
  return (bits + passes - 1) / passes;
}

int sort_cells(const int16_t* pmid, const float* disp, const uint8_t* valid, int64_t n,
               const int32_t* mesh_shape, float cell_size, const int32_t* brick, int32_t* perm,
               int32_t* bin_offsets, int16_t* pmid_s, float* disp_s, Arena& ws, hipStream_t s) {
  KeyGeom g = make_key_geom(mesh_shape, cell_size, brick);
  if (n == 0) {
    if (bin_offsets) {
      hipLaunchKernelGGL(k_bin_bounds, dim3(1), dim3(1), 0, s, (const int32_t*)nullptr, (int64_t)0,
                         g.sentinel + 1, bin_offsets);
      PM_LAUNCHED("k_bin_bounds", s);
    }
    return PM_SUCCESS;
  }
  const int64_t nseg = ceil_div(n, kSeg);
  // without a validity mask no particle takes the sentinel, so the key range ends at nbins-1
  const int bits = key_bits(valid ? g.sentinel : std::max(g.sentinel - 1, 1));
  int passes = 1;
  const int dbits = digit_bits_for(bits, passes);
  const int64_t hist_len = ((int64_t)1 << dbits) * nseg;
  int32_t* keys_a = ws.take<int32_t>(n);
  int32_t* keys_b = ws.take<int32_t>(n);
  int32_t* vals_t = ws.take<int32_t>(n);
  int32_t* hist = ws.take<int32_t>(hist_len);
  int32_t* offs = ws.take<int32_t>(hist_len);
  int32_t* partial = ws.take<int32_t>(ceil_div(hist_len, kScanChunk) + 1);
  PM_RETURN_IF(!ws.ok(), PM_ERROR_WORKSPACE, "sort workspace too small");

  const dim3 grid((unsigned)ceil_div(nseg, kWavesPerBlock)), block(kWave * kWavesPerBlock);
  // value ping-pong arranged so the last pass writes `perm`
  int32_t* vbuf[2] = {(passes % 2 == 1) ? perm : vals_t, (passes % 2 == 1) ? vals_t : perm};
  int32_t* kbuf[2] = {keys_a, keys_b};
  for (int pass = 0; pass < passes; ++pass) {
    const int shift = dbits * pass;
    const bool last = pass == passes - 1;
    int32_t* kin = kbuf[(pass + 1) % 2];
    int32_t* kout = (last && !bin_offsets) ? nullptr : kbuf[pass % 2];
    int32_t* vin = vbuf[(pass + 1) % 2];
    int32_t* vout = vbuf[pass % 2];
    if (pass == 0)
      hipLaunchKernelGGL(k_digit_hist<true>, grid, block, 0, s, nullptr, pmid, disp, valid, g, n, shift,
                         dbits, nseg, hist);
    else
      hipLaunchKernelGGL(k_digit_hist<false>, grid, block, 0, s, kin, pmid, disp, valid, g, n, shift,
                         dbits, nseg, hist);
    PM_LAUNCHED("k_digit_hist", s);
    int st = scan_exclusive(hist, ScanOut{offs}, hist_len, partial, s);
    if (st) return st;
    if (pass == 0)
      hipLaunchKernelGGL(k_digit_scatter<true>, grid, block, 0, s, nullptr, nullptr, pmid, disp, valid, g,
                         n, shift, dbits, nseg, offs, kout, vout);
    else
      hipLaunchKernelGGL(k_digit_scatter<false>, grid, block, 0, s, kin, vin, pmid, disp, valid, g, n,
                         shift, dbits, nseg, offs, kout, vout);
    PM_LAUNCHED("k_digit_scatter", s);
    if (last && bin_offsets) {
      hipLaunchKernelGGL(k_bin_bounds, dim3((unsigned)ceil_div(n + 1, 256)), dim3(256), 0, s, kout, n,
                         g.sentinel + 1, bin_offsets);
      PM_LAUNCHED("k_bin_bounds", s);
    }
  }
  if (pmid_s || disp_s) {
    const unsigned blocks = (unsigned)std::min<int64_t>(ceil_div(n, 256), 8192);
    hipLaunchKernelGGL(k_gather_payload, dim3(blocks), dim3(256), 0, s, perm, pmid, disp, n, pmid_s, disp_s);
    PM_LAUNCHED("k_gather_payload", s);
  }
  return PM_SUCCESS;
}

// ------------------------------------------------ allocation-free binning ----
// pm_bucket_cells_noalloc takes its bin counters and scan partials from this file-scope
// device array instead of a caller workspace.  On the host the array's name is only a
// stand-in, so host code never passes it to a kernel or a copy: pm_init resolves the
// array's address on each device once (hipGetSymbolAddress, with that device current) and
// the entry point uses the address of the current device.  Every call on a device shares
// that device's copy, so calls that overlap on one device (two streams) race.
constexpr size_t kNoAllocScratchBytes = size_t(8) << 20;  // 8 MiB: up to 2,096,446 bricks
constexpr int64_t kNoAllocBricks = 2096446;
constexpr int kMaxDevices = 64;
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];
static std::atomic<void*> g_scratch_ptr[kMaxDevices];

int init_noalloc_scratch() {
  int dev = 0;
  PM_HIP_TRY(hipGetDevice(&dev));
  PM_RETURN_IF(dev < 0 || dev >= kMaxDevices, PM_ERROR_UNSUPPORTED, "device ordinal >= 64");
  if (g_scratch_ptr[dev].load(std::memory_order_acquire)) return PM_SUCCESS;
  void* p = nullptr;
  PM_HIP_TRY(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
  PM_RETURN_IF(p == nullptr, PM_ERROR_HIP, "hipGetSymbolAddress returned NULL for the binning scratch");
  g_scratch_ptr[dev].store(p, std::memory_order_release);
  return PM_SUCCESS;
}

int check_bucket_args(const int16_t* pmid, const float* disp, int64_t n, const int32_t* mesh_shape, float cell_size,
                      const int32_t* brick, const int32_t* ptcl_grid, const int32_t* perm, const int32_t* bin_offsets,
                      const int16_t* pmid_s, const float* disp_s, const uint8_t* valid_s) {
  int st = check_sort_args(n, mesh_shape, brick);
  if (st) return st;
  PM_RETURN_IF(!(cell_size > 0.f), PM_ERROR_INVALID_ARGUMENT, "cell_size must be positive");
  PM_RETURN_IF(bin_offsets == nullptr, PM_ERROR_INVALID_ARGUMENT, "bin_offsets NULL");
  PM_RETURN_IF(n > 0 && (pmid == nullptr || disp == nullptr || perm == nullptr || pmid_s == nullptr ||
                         disp_s == nullptr || valid_s == nullptr),
               PM_ERROR_INVALID_ARGUMENT, "pmid/disp/perm/sorted payload NULL");
  if (ptcl_grid)
    for (int a = 0; a < 3; ++a)
      PM_RETURN_IF(ptcl_grid[a] < 0, PM_ERROR_INVALID_ARGUMENT, "ptcl_grid must be non-negative");
  return PM_SUCCESS;
}

}  // namespace sort
}  // namespace pm

using namespace pm;

extern "C" {

int pm_sort_cells_workspace(int64_t n, const int32_t mesh_shape[3], const int32_t brick[3],
                            size_t* bytes) {
  int st = sort::check_sort_args(n, mesh_shape, brick);
  if (st) return st;
  PM_RETURN_IF(bytes == nullptr, PM_ERROR_INVALID_ARGUMENT, "bytes is NULL");
  *bytes = sort::workspace_bytes(n, mesh_shape, brick);
  return PM_SUCCESS;
}

int pm_sort_cells(const int16_t* pmid, const float* disp, const uint8_t* valid, int64_t n,
                  const int32_t mesh_shape[3], float cell_size, const int32_t brick[3],
                  int32_t* perm, int32_t* bin_offsets, int16_t* pmid_sorted, float* disp_sorted,
                  void* workspace, size_t workspace_bytes, void* stream) {
  int st = sort::check_sort_args(n, mesh_shape, brick);
  if (st) return st;
  PM_RETURN_IF(!(cell_size > 0.f), PM_ERROR_INVALID_ARGUMENT, "cell_size must be positive");
  PM_RETURN_IF(n > 0 && (pmid == nullptr || disp == nullptr || perm == nullptr),
               PM_ERROR_INVALID_ARGUMENT, "pmid/disp/perm NULL");
  size_t need = sort::workspace_bytes(n, mesh_shape, brick);
  PM_RETURN_IF(workspace == nullptr || workspace_bytes < need, PM_ERROR_WORKSPACE,
               "sort workspace too small: need " + std::to_string(need) + " bytes");
  Arena ws(workspace, workspace_bytes);
  return sort::sort_cells(pmid, disp, valid, n, mesh_shape, cell_size, brick, perm, bin_offsets, pmid_sorted,
                          disp_sorted, ws, as_stream(stream));
}

int pm_bucket_cells_workspace(int64_t n, const int32_t mesh_shape[3], const int32_t brick[3], size_t* bytes) {
  int st = sort::check_sort_args(n, mesh_shape, brick);
  if (st) return st;
  PM_RETURN_IF(bytes == nullptr, PM_ERROR_INVALID_ARGUMENT, "bytes is NULL");
  *bytes = sort::bucket_workspace_bytes(mesh_shape, brick);
  return PM_SUCCESS;
}

int pm_bucket_cells(const int16_t* pmid, const float* disp, const uint8_t* valid, int64_t n,
                    const int32_t mesh_shape[3], float cell_size, const int32_t brick[3], const int32_t ptcl_grid[3],
                    int32_t* perm, int32_t* bin_offsets, int16_t* pmid_sorted, float* disp_sorted,
                    uint8_t* valid_sorted, void* workspace, size_t workspace_bytes, void* stream) {
  int st = sort::check_bucket_args(pmid, disp, n, mesh_shape, cell_size, brick, ptcl_grid, perm, bin_offsets,
                                   pmid_sorted, disp_sorted, valid_sorted);
  if (st) return st;
  const size_t need = sort::bucket_workspace_bytes(mesh_shape, brick);
  PM_RETURN_IF(workspace == nullptr || workspace_bytes < need, PM_ERROR_WORKSPACE,
               "bucket workspace too small: need " + std::to_string(need) + " bytes");
  Arena ws(workspace, workspace_bytes);
  return sort::bucket_cells_arena(pmid, disp, valid, n, mesh_shape, cell_size, brick, ptcl_grid, perm, bin_offsets,
                            pmid_sorted, disp_sorted, valid_sorted, ws, as_stream(stream));
}

int pm_bucket_cells_noalloc(const int16_t* pmid, const float* disp, const uint8_t* valid, int64_t n,
                            const int32_t mesh_shape[3], float cell_size, const int32_t brick[3],
                            const int32_t ptcl_grid[3], int32_t* perm, int32_t* bin_offsets, int16_t* pmid_sorted,
                            float* disp_sorted, uint8_t* valid_sorted, void* stream) {
  int st = sort::check_bucket_args(pmid, disp, n, mesh_shape, cell_size, brick, ptcl_grid, perm, bin_offsets,
                                   pmid_sorted, disp_sorted, valid_sorted);
  if (st) return st;
  const size_t need = sort::bucket_workspace_bytes(mesh_shape, brick);
  const int64_t nbins = sort::bucket_count_len(mesh_shape, brick) - sort::kTails - 1;
  PM_RETURN_IF(need > sort::kNoAllocScratchBytes || nbins > sort::kNoAllocBricks, PM_ERROR_UNSUPPORTED,
               "pm_bucket_cells_noalloc: " + std::to_string(need) + " bytes of bin counters exceed its " +
                   std::to_string(sort::kNoAllocScratchBytes) +
                   "-byte static scratch (at most 2,096,446 bricks): use pm_bucket_cells with a workspace");
  int dev = 0;
  PM_HIP_TRY(hipGetDevice(&dev));
  void* p = (dev >= 0 && dev < sort::kMaxDevices) ? sort::g_scratch_ptr[dev].load(std::memory_order_acquire)
                                                  : nullptr;
  PM_RETURN_IF(p == nullptr, PM_ERROR_INVALID_ARGUMENT,
               "pm_init has not run on the current device (it resolves the binning scratch)");
  Arena ws(p, sort::kNoAllocScratchBytes);
  return sort::bucket_cells_arena(pmid, disp, valid, n, mesh_shape, cell_size, brick, ptcl_grid, perm, bin_offsets,
                            pmid_sorted, disp_sorted, valid_sorted, ws, as_stream(stream));
}

}  // extern "C"
