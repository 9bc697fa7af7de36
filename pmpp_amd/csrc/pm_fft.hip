// FFT passes (real<->half-spectrum along z, complex along y/x) and the fused spectral
// force passes of the PM step.  See pm_fft.h for the decomposition.
#include <algorithm>
#include <atomic>
#include <cmath>
#include <mutex>
#include <vector>

#include "pm_fft.h"
#include "pm_fft_launch.h"

namespace pm {
namespace fft {

// ------------------------------------------------------------ twiddle table ----
static __device__ float2 g_twiddle[kTwN];

namespace {
std::mutex g_tw_mutex;
std::atomic<const float2*> g_tw_ptr[64];
}  // namespace

const float2* twiddle_table() {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return nullptr;
  return g_tw_ptr[dev].load(std::memory_order_acquire);
}

}  // namespace fft

// The one place that uploads the table and synchronises (pm_init): every other entry point
// only enqueues work on its stream, so it can run inside HIP graph capture.
int init_device_tables() {
  int dev = 0;
  PM_HIP_TRY(hipGetDevice(&dev));
  PM_RETURN_IF(dev < 0 || dev >= 64, PM_ERROR_UNSUPPORTED, "device ordinal >= 64");
  std::lock_guard<std::mutex> lock(fft::g_tw_mutex);
  if (fft::g_tw_ptr[dev].load(std::memory_order_acquire)) return PM_SUCCESS;
  std::vector<float2> host(fft::kTwN);
  for (int i = 0; i < fft::kTwN; ++i) {
    // exp(-2 pi i j / 4096) in double, rounded once to float
    long double a = 2.0L * 3.14159265358979323846264338327950288L * (long double)i / fft::kTwN;
    host[i] = make_float2((float)cosl(a), (float)(-sinl(a)));
  }
  host[0] = make_float2(1.f, 0.f);
  host[fft::kTwN / 4] = make_float2(0.f, -1.f);
  host[fft::kTwN / 2] = make_float2(-1.f, 0.f);
  host[3 * fft::kTwN / 4] = make_float2(0.f, 1.f);
  PM_HIP_TRY(hipMemcpyToSymbol(HIP_SYMBOL(fft::g_twiddle), host.data(), sizeof(float2) * fft::kTwN));
  void* ptr = nullptr;
  PM_HIP_TRY(hipGetSymbolAddress(&ptr, HIP_SYMBOL(fft::g_twiddle)));
  PM_HIP_TRY(hipDeviceSynchronize());
  fft::g_tw_ptr[dev].store(static_cast<const float2*>(ptr), std::memory_order_release);
  return PM_SUCCESS;
}

int require_device_tables() {
  PM_RETURN_IF(fft::twiddle_table() == nullptr, PM_ERROR_INVALID_ARGUMENT,
               "pm_init has not run on the current device (it prepares the FFT twiddle table)");
  return PM_SUCCESS;
}

namespace fft {
namespace {

// ----------------------------------------------------------- column passes ----
// T adjacent columns per workgroup.  The y inverse of the three force components (kColInv3) runs
// three workgroups per tile (HALVES), one per output; the first two load the same input tile (the
// second read is served by L2: they run on one XCD at nearly the same time), so no thread
// keeps two spectra live.  The x Green pass (kColGreen) runs one
// workgroup per tile that parks its multiplied spectrum in its first output between the two
// inverses.  Outputs of two-output passes must not alias the input or each other.
template <int N, int T, int HALVES>
struct ColCfg {
  static constexpr int P = Plan<N>::P;
  static constexpr int THREADS = T * P;
  static constexpr int PADK = T;  // per-k1-block LDS pad: spreads the strided rows over banks
  static constexpr int LDS_FLOATS = N * T + Plan<N>::N1 * PADK;
};

// Column tiles are visited in an XCD-aware order: workgroups are dispatched round-robin
// over the 8 XCDs, so logical item q is given to workgroup (q % g8) * 8 + q / g8 ... i.e.
// consecutive logical items (the workgroups of a tile, and neighbouring tiles, which share
// cache lines when T*8 < 128 bytes) run on the same XCD at nearly the same time.
template <int N, int T, int MODE, int HALVES>
__global__ void __launch_bounds__((ColCfg<N, T, HALVES>::THREADS))
    k_cols(ColPass io, SpecTables tb, int dax, const float2* __restrict__ tw, int gx, int gy, int g8) {
  using PL = Plan<N>;
  using CF = ColCfg<N, T, HALVES>;
  constexpr int E = PL::E, N2 = PL::N2;
  __shared__ float lds[CF::LDS_FLOATS];
  const int L = blockIdx.x;
  const int q = (L % 8) * g8 + L / 8;
  const int half = HALVES > 1 ? q % HALVES : 0;
  const int tile = HALVES > 1 ? q / HALVES : q;
  const int tilex = tile % gx;
  const int64_t b = tile / gx;
  if (b >= gy) return;  // padding workgroup of the XCD remap: uniform exit before any barrier
  const int lt = threadIdx.x;
  const int col = lt % T;
  const int p = lt / T;
  const int cg = tilex * T + col;
  const bool cok = cg < io.ncols;
  // loads use a clamped column so they are unconditional (branch-free batches stay in flight)
  const int cgl = cok ? cg : io.ncols - 1;
  const int64_t lbase = b * io.s_batch + (int64_t)cgl * io.s_col;
  const int64_t o_row = io.o_row >= 0 ? io.o_row : io.s_row;
  const int64_t obase = b * (io.o_batch >= 0 ? io.o_batch : io.s_batch) + (int64_t)cg * io.s_col;
  // row r = p + d of this thread's column: base + d * stride, with d a compile-time multiple of
  // the row step for every unrolled slot, so the per-slot offsets are uniform (scalar) and no
  // per-slot row index stays live in a VGPR across the transforms
  const int64_t ibase = lbase + (int64_t)p * io.s_row;
  const int64_t obp = obase + (int64_t)p * o_row;
  const int keep = io.keep;
  // band compaction of the transformed axis (see ColPass::keep)
  auto in_band = [&](int k) { return keep < 0 || k <= keep || k >= N - keep; };
  auto packed = [&](int k) { return (keep < 0 || k <= keep) ? k : k - (N - 2 * keep - 1); };
  float* my = lds;
  auto idx = [&](int row) { return row * T + col + (row / N2) * CF::PADK; };

  static_assert((HALVES == 3) == (MODE == kColInv3 || MODE == kColSym), "three workgroups per tile: one per output");
  float2 v[E];
  if constexpr (MODE == kColAdj) {
    // Spectral adjoint of the force step, x pass (the columns are kz, the batches the packed ky
    // rows, as for kColGreen): sum_i conj(D_i) hat g_i with conj(i negk) = -i negk, then
    // mask * (-1/k^2), then the inverse x transform.  The y and z symbols are constant along
    // an x column, so by linearity those two components are combined before their transform:
    // U = X(negk_y g_y + negk_z g_z), then s = -i (negk_x X(g_x) + U); two lines live per
    // thread instead of three.
    int ky = (int)(b * io.ky_b) + cgl * io.ky_c;
    ky += ky > io.ky_split ? io.ky_shift : 0;
    int kz = (int)(b * io.kz_b) + cgl * io.kz_c + io.kz0;
    const float kyv = tb.k[1][ky], kzv = tb.k[2][kz];
    const float nky = tb.negk[1][ky], nkz = tb.negk[2][kz];
    const bool keep_yz = cok && tb.mask[1][ky] != 0.f && tb.mask[2][kz] != 0.f;
#pragma unroll
    for (int s = 0; s < E; ++s) {
      const int64_t o = ibase + (int64_t)(nrow<N>(p, s) - p) * io.s_row;
      const float2 gy = io.in1[o], gz = io.in2[o];
      v[s] = make_float2(nky * gy.x + nkz * gz.x, nky * gy.y + nkz * gz.y);
    }
    forward_core<N>(v, my, p, idx, tw);
    asm volatile("" ::: "memory");  // the x component's loads after U's transform
    float2 w[E];
#pragma unroll
    for (int s = 0; s < E; ++s) w[s] = io.in[ibase + (int64_t)(nrow<N>(p, s) - p) * io.s_row];
    forward_core<N>(w, my, p, idx, tw);
#pragma unroll
    for (int s = 0; s < E; ++s) {
      const float kxv = spec_k(xrow<N>(p, s), N, false, tb.period);
      const float nkx = spec_negk(kxv, tb);
      const float tx = nkx * w[s].x + v[s].x, ty = nkx * w[s].y + v[s].y;  // s = -i t
      const float k2 = kxv * kxv + kyv * kyv + kzv * kzv;
      const bool keep = keep_yz && spec_keep(kxv, tb) && k2 != 0.f;
      const float r = recip_nr(k2);
      v[s] = keep ? make_float2(-ty * r, tx * r) : make_float2(0.f, 0.f);  // -s / k^2
    }
    inverse_core<N>(v, my, p, idx, tw);
    if (cok) {
#pragma unroll
      for (int s = 0; s < E; ++s) io.out0[obp + (int64_t)(nrow<N>(p, s) - p) * o_row] = v[s];
    }
    return;
  } else if constexpr (MODE == kColFwd || MODE == kColGreen || MODE == kColPot) {
#pragma unroll
    for (int s = 0; s < E; ++s) v[s] = io.in[ibase + (int64_t)(nrow<N>(p, s) - p) * io.s_row];
    forward_core<N>(v, my, p, idx, tw);
  } else {
    const float2* src = MODE == kColInv3 && half == 2 ? io.in1 : io.in;  // uniform
    if (keep >= 0 && io.compact_in) {  // packed band in, zero outside it
#pragma unroll
      for (int s = 0; s < E; ++s) {
        int k = xrow<N>(p, s);
        v[s] = src[lbase + (int64_t)(in_band(k) ? packed(k) : 0) * io.s_row];
      }
#pragma unroll
      for (int s = 0; s < E; ++s)
        if (!in_band(xrow<N>(p, s))) v[s] = make_float2(0.f, 0.f);
    } else {
#pragma unroll
      for (int s = 0; s < E; ++s) v[s] = src[ibase + (int64_t)(xrow<N>(p, s) - p) * io.s_row];
    }
  }

  if constexpr (MODE == kColFwd) {
    if (cok) {
#pragma unroll
      for (int s = 0; s < E; ++s) {
        int k = xrow<N>(p, s);
        if (in_band(k)) io.out0[obase + (int64_t)packed(k) * o_row] = v[s];  // forward: packed output
      }
    }
    return;
  } else {
    if constexpr (MODE == kColGreen || MODE == kColPot) {
      // mask x Poisson symbol (gravity.py:174-196, 263-287); for kColGreen's second output also
      // D_x = i*negk_x (configuration.py:365-376), below
      int ky = (int)(b * io.ky_b) + cgl * io.ky_c;
      ky += ky > io.ky_split ? io.ky_shift : 0;
      int kz = (int)(b * io.kz_b) + cgl * io.kz_c + io.kz0;
      float kyv = tb.k[1][ky], kzv = tb.k[2][kz];
      bool keep_yz = cok && tb.mask[1][ky] != 0.f && tb.mask[2][kz] != 0.f;
      // k_x, its mask and -k_x are evaluated in registers (the same expressions as the
      // tables): 3*E table loads per thread would be hoisted above the transform and stay live
#pragma unroll
      for (int s = 0; s < E; ++s) {
        int kx = xrow<N>(p, s);
        float kxv = spec_k(kx, N, false, tb.period);
        float k2 = kxv * kxv + kyv * kyv + kzv * kzv;
        bool keep = keep_yz && spec_keep(kxv, tb) && k2 != 0.f;
        const float r = recip_nr(k2);
        float g = keep ? -r : 0.f;  // one reciprocal per mode, shared by both parts
        v[s] = make_float2(v[s].x * g, v[s].y * g);
      }
      if constexpr (MODE == kColGreen) {
        // one workgroup per tile: the multiplied spectrum phi is parked in out0 at this
        // thread's own output rows (where it writes its out0 values at the end, so no other
        // thread touches them), D_x phi is inverted into out1, then phi is read back and
        // inverted into out0 -- three transforms per tile instead of four (two workgroups that
        // each redo the forward); the parked tiles overflow L2, so the pass moves 1.8x its
        // algorithmic bytes, and is faster anyway: the transforms bound it, not HBM
        if (cok) {
#pragma unroll
          for (int s = 0; s < E; ++s) io.out0[obp + (int64_t)(nrow<N>(p, s) - p) * o_row] = v[s];
        }
#pragma unroll
        for (int s = 0; s < E; ++s) v[s] = c_imul(spec_negk(spec_k(xrow<N>(p, s), N, false, tb.period), tb), v[s]);
        inverse_core<N>(v, my, p, idx, fresh_table(tw));
        if (cok) {
#pragma unroll
          for (int s = 0; s < E; ++s) io.out1[obp + (int64_t)(nrow<N>(p, s) - p) * o_row] = v[s];
        }
        asm volatile("" ::: "memory");  // no twiddle of the first inverse kept live for the second
#pragma unroll
        for (int s = 0; s < E; ++s)
          v[s] = cok ? io.out0[obp + (int64_t)(nrow<N>(p, s) - p) * o_row] : make_float2(0.f, 0.f);
      }
    } else if constexpr (MODE == kColSym) {
      const ColSymbol sy = half == 0 ? io.sym[0] : (half == 1 ? io.sym[1] : io.sym[2]);  // uniform
      const float ky = tb.k[1][b], kz = tb.k[2][cgl];
      // a wavenumber of axis a with the Nyquist zeroed
      auto live = [&](int a, float k) { return fabsf(fabsf(k) - io.sym_nyq[a]) <= io.sym_tol[a] ? 0.f : k; };
      const bool cross = sy.j != sy.i;  // strains of two axes and gradients zero the Nyquist
#pragma unroll
      for (int s = 0; s < E; ++s) {
        const float kx = tb.k[0][xrow<N>(p, s)];
        float ki = sy.i == 0 ? kx : (sy.i == 1 ? ky : kz);
        if (cross) ki = live(sy.i, ki);
        if (sy.j < 0) {
          v[s] = make_float2(ki * v[s].y, -ki * v[s].x);  // -i k v
        } else {
          float kj = sy.j == 0 ? kx : (sy.j == 1 ? ky : kz);
          if (cross) kj = live(sy.j, kj);
          v[s] = c_scale(v[s], -ki * kj);
        }
      }
    } else if constexpr (MODE == kColInv3) {
      if (half == 1) {
#pragma unroll
        for (int s = 0; s < E; ++s) v[s] = c_imul(tb.negk[dax][xrow<N>(p, s)], v[s]);
      }
    }
    // after a forward transform in the same kernel (kColGreen, kColPot) the inverse's twiddles
    // are loaded afresh instead of kept live from the forward
    inverse_core<N>(v, my, p, idx, (MODE == kColGreen || MODE == kColPot) ? fresh_table(tw) : tw);
    float2* out = (half == 1) ? io.out1 : (half == 2 ? io.out2 : io.out0);
    if (cok) {
#pragma unroll
      for (int s = 0; s < E; ++s) out[obp + (int64_t)(nrow<N>(p, s) - p) * o_row] = v[s];
    }
  }
}

// --------------------------------------------------------------- z passes ----
// Two real lines (2 i and 2 i + 1) of N points per complex transform, z = a + i b: the pair's spectra
// are A = (Z[k] + conj Z[N-k]) / 2 and B = -i (Z[k] - conj Z[N-k]) / 2.  Against one line as N / 2
// complex points this has a tenth more butterflies, but no twiddle, no table load and one LDS round
// less where bins k and N - k meet, which cost as much as the transform: with the loads and stores
// alone the c2r of three 1024^3 components takes 3.8 ms, with the transform 4.4, with the N / 2-point
// pairing it took 5.2; now 4.6.  A pair's threads are in one wave, so nothing waits at a barrier.
// Before -> now, us: c2r 256^3 116 -> 88, 512^3 783 -> 594, 1024^3 5220 -> 4600; r2c with planes
// 43 -> 33, 256 -> 231, 2050 -> 1450.  Now bound by the memory path (c2r 19.3 GB: 4.2 TB/s; a copy
// reaches 4.8).  A line's rounding goes with the larger of its pair: rms error of a forward or
// inverse transform of white noise against 64 bits, before -> now, 64^3 1.50e-7 -> 1.49e-7, 256^3 1.86e-7 ->
// 1.89e-7, 512^3 2.07e-7 -> 2.11e-7; on the smaller half of a log-normal field's cells, of their rms, 256^3
// 8.9e-6 and 512^3 1.2e-5 either way.
template <int N>
struct ZCfg {
  static constexpr int P = Plan<N>::P;
  // long lines: more of them per workgroup, so more adjacent rows are written at about the same time
  // (1024^3, 64 / 128 / 256 / 512 threads: c2r 4.99 / 4.98 / 4.49 / 4.60, r2c 1.70 / 1.65 / 1.62 / 1.45 ms;
  // 512^3, 256 / 512: 594 / 606, 232 / 238 us).  At 2048 points, whose threads hold 64 slots, 512 only helps
  // the r2c of many lines (256 / 512: 64^2 lines c2r 25 / 29, r2c 22 / 26 us; 256^2 311 / 316, 258 / 274; 512^2
  // 1077 / 1138, 945 / 878)
  static constexpr int THREADS = N == 1024 ? 512 : 256;
  static constexpr int PAIRS = THREADS / P;
  // floats per pair's slot (the transform's real / imaginary exchange), with LSTR = P (mod 64) so the
  // 64/P pairs of a wave start on disjoint groups of the 64 LDS banks
  static constexpr int LSTR = ((N + N / Plan<N>::N2 + 63) / 64) * 64 + (P % 64);
  static constexpr int LDS_FLOATS = PAIRS * LSTR;
  static_assert(P <= 64, "a pair's threads are in one wave");
};

// ADD: C2R: the output is rout_add + the scaled line; R2C: rin's planes are folded on load
// (ZPass::fold).  Separate instantiations, so the plain passes keep their register budget.
template <int N, bool C2R, bool ADD = false>
__global__ void __launch_bounds__((ZCfg<N>::THREADS), (C2R && N == 2048 ? 2 : 1))  // c2r: 57 -> 52 us at 64^2 x 2048
    k_zpass(ZPass zp, SpecTables tb, const float2* __restrict__ tw) {
  using PL = Plan<N>;
  using ZC = ZCfg<N>;
  constexpr int P = PL::P, E = PL::E, N2 = PL::N2, M = N / 2;
  __shared__ float lds[ZC::LDS_FLOATS];
  const int p = threadIdx.x % P;
  const int pair = threadIdx.x / P;
  const int64_t pg = (int64_t)blockIdx.x * ZC::PAIRS + pair;
  const bool ok = 2 * pg < zp.nlines;
  const int64_t la = 2 * (ok ? pg : 0);  // clamped: unconditional, batched loads
  float* slot = lds + pair * ZC::LSTR;
  auto idx = [&](int row) { return pair * ZC::LSTR + row + row / N2; };
  float2 v[E];

  if constexpr (!C2R) {
    const float* src = zp.rin + la * zp.pitch_r;
    if constexpr (P == 2) {
      // rows of 4 and 8 points, two threads a pair: whole vectors, of which a thread takes every other
      // element (a scalar load's 64 lanes lie in 32 places: forward transform of 1024^2 lines of 8 points
      // 77 -> 68 us; 64 with one line per half-length transform)
      typedef float Quad __attribute__((ext_vector_type(4), aligned(4)));
#pragma unroll
      for (int q = 0; q < N / 4; ++q) {
        const Quad a = reinterpret_cast<const Quad*>(src)[q], b = reinterpret_cast<const Quad*>(src + zp.pitch_r)[q];
        v[2 * q] = p ? make_float2(a.y, b.y) : make_float2(a.x, b.x);
        v[2 * q + 1] = p ? make_float2(a.w, b.w) : make_float2(a.z, b.z);
      }
    } else {
#pragma unroll
      for (int s = 0; s < E; ++s) v[s] = make_float2(src[nrow<N>(p, s)], src[zp.pitch_r + nrow<N>(p, s)]);
    }
    if constexpr (ADD) {
      // a cell with lx = x mod b0 and ly = y mod b1 takes, from its neighbouring columns (periodic),
      //   lx == 0: XS of column (cx-1, cy) row ly; and when ly == 0 also XS of (cx-1, cy-1) row b1
      //            and YS of (cx, cy-1) row 0
      //   ly == 0: YS of column (cx, cy-1) row lx
      // summed in this order before they are added.  Reading them here saves the pass that
      // would add them in place.
      const FoldPlanes& fp = zp.fold;
      const int x = (int)(la >> fp.ny_log);
      const int lx = x & ((1 << fp.b0_log) - 1);
      const int cx = x >> fp.b0_log, sx = cx == 0 ? fp.nb0 - 1 : cx - 1;
      const int64_t b0 = int64_t(1) << fp.b0_log, b1 = int64_t(1) << fp.b1_log;
      auto xs_line = [&](int ccy, int64_t row) {
        return fp.xs + (((int64_t)sx * fp.nb1 + ccy) * (b1 + 1) + row) * zp.pitch_r;
      };
      auto fold = [&](int y, auto add) {
        const int ly = y & ((1 << fp.b1_log) - 1);
        if (lx != 0 && ly != 0) return;
        const int cy = y >> fp.b1_log, sy = cy == 0 ? fp.nb1 - 1 : cy - 1;
        const float* ysl = fp.ys + (((int64_t)cx * fp.nb1 + sy) * b0 + lx) * zp.pitch_r;
        const float* p0 = lx == 0 ? xs_line(cy, ly) : ysl;
        float w[E];
#pragma unroll
        for (int s = 0; s < E; ++s) w[s] = p0[nrow<N>(p, s)];
        if (lx == 0 && ly == 0) {
          // eight slots at a time: all at once, the loads would be issued one by one for want of
          // registers, and the few corner lines would hold up the whole pass
          const float* p1 = xs_line(sy, b1);
          constexpr int Q = E < 8 ? E : 8;
#pragma unroll
          for (int c = 0; c < E; c += Q) {
            float f[Q], g[Q];
#pragma unroll
            for (int s = 0; s < Q; ++s) {
              f[s] = p1[nrow<N>(p, c + s)];
              g[s] = ysl[nrow<N>(p, c + s)];
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int s = 0; s < Q; ++s) w[c + s] = (w[c + s] + f[s]) + g[s];
            __builtin_amdgcn_sched_barrier(0);
          }
        }
#pragma unroll
        for (int s = 0; s < E; ++s) add(s, w[s]);
      };
      const int y = (int)(la & ((1 << fp.ny_log) - 1));  // even: both lines have the same x
      fold(y, [&](int s, float w) { v[s].x += w; });
      fold(y + 1, [&](int s, float w) { v[s].y += w; });
    }
    if (zp.rin_add) {  // uniform
      const float* src2 = zp.rin_add + la * zp.pitch_r;
#pragma unroll
      for (int s = 0; s < E; ++s) {
        v[s].x += src2[nrow<N>(p, s)];
        v[s].y += src2[zp.pitch_r + nrow<N>(p, s)];
      }
    }
#pragma unroll
    for (int s = 0; s < E; ++s)
      v[s] = make_float2((v[s].x + zp.src_shift) * zp.src_scale, (v[s].y + zp.src_shift) * zp.src_scale);
    forward_core<N, true>(v, lds, p, idx, tw);
    // bins k and N - k meet in a natural-order copy of the transform, real parts first
    constexpr int H = E / 2;  // bins k = p + P j < N / 2 per thread
    float sr[H], dr[H], mr, mi;
#pragma unroll
    for (int s = 0; s < E; ++s) slot[xrow<N>(p, s)] = v[s].x;
    line_sync<true>();
    mr = slot[M];
#pragma unroll
    for (int j = 0; j < H; ++j) {
      const int k = p + P * j;
      const float a = slot[k], b = slot[(N - k) & (N - 1)];
      sr[j] = 0.5f * (a + b);
      dr[j] = 0.5f * (b - a);
    }
    line_sync<true>();
#pragma unroll
    for (int s = 0; s < E; ++s) slot[xrow<N>(p, s)] = v[s].y;
    line_sync<true>();
    mi = slot[M];
    if (!ok) return;
    float2* da = zp.cmain[0] + la * zp.pitch_c;
    float2* db = da + zp.pitch_c;
#pragma unroll
    for (int j = 0; j < H; ++j) {
      const int k = p + P * j;
      if (k < zp.kz_lim) {
        const float a = slot[k], b = slot[(N - k) & (N - 1)];
        da[k] = make_float2(sr[j], 0.5f * (a - b));
        db[k] = make_float2(0.5f * (a + b), dr[j]);
      }
    }
    if (p == 0 && zp.nyq) {
      da[M] = make_float2(mr, 0.f);
      db[M] = make_float2(mi, 0.f);
    }
  } else {
    // Z[k] = A[k] + i B[k], and conj A + i conj B of N - k above N / 2, which a thread gets from the one that
    // read those through a natural-order copy in LDS, real parts first (reading the half spectra a
    // second time, in reverse and from the cache, took 15 % longer at N = 1024)
    const int comp = blockIdx.y;
    const float2* sa = zp.cmain[comp] + la * zp.pitch_c;
    const float2* sb = sa + zp.pitch_c;
    const int klim = zp.kz_lim < M ? zp.kz_lim : M;
    const bool deriv = (zp.deriv >> comp) & 1;
    // slot s < E / 2 in this order has a bin base + p below N / 2, and E - 1 - s the bins N - base - p
    auto bin = [](int s) constexpr { return P * (s / N2) + PL::N1 * (s % N2); };
    float2 ma = make_float2(0.f, 0.f), mb = ma;  // the Nyquist bin
    if (zp.nyq && p == 0) {
      ma = sa[M];
      mb = sb[M];
    }
    // the slots below N / 2, at most 16 at a time (64-slot threads would not have the registers)
    constexpr int H2 = N2 > 1 ? N2 / 2 : 1;
    auto low = [](int i) constexpr { return (i / H2) * N2 + i % H2; };
    constexpr int Q = E / 2 < 16 ? E / 2 : 16;
    static_for<0, E / 2 / Q>([&](auto C) {
      float2 a[Q], b[Q];
      static_for<0, Q>([&](auto I) {
        constexpr int i = decltype(I)::value, k = bin(low(decltype(C)::value * Q + i));
        a[i] = b[i] = make_float2(0.f, 0.f);
        if (k + P <= klim) {  // uniform: the whole slot is in the band
          a[i] = sa[k + p];
          b[i] = sb[k + p];
        } else if (k + p < klim) {
          a[i] = sa[k + p];
          b[i] = sb[k + p];
        }
      });
      if (deriv) {
        static_for<0, Q>([&](auto I) {
          constexpr int i = decltype(I)::value, k = bin(low(decltype(C)::value * Q + i));
          const float m = tb.negk[2][k + p];
          a[i] = c_imul(m, a[i]);
          b[i] = c_imul(m, b[i]);
        });
      }
      static_for<0, Q>([&](auto I) {
        constexpr int i = decltype(I)::value, s = low(decltype(C)::value * Q + i);
        if constexpr (s == 0) {  // irfft uses only the real parts of the DC and Nyquist bins
          if (p == 0) a[i].y = b[i].y = 0.f;
        }
        v[s] = make_float2(a[i].x - b[i].y, a[i].y + b[i].x);
        v[E - 1 - s].y = b[i].x - a[i].y;
        if (bin(s) < klim) slot[bin(s) + p] = a[i].x + b[i].y;
      });
      if constexpr (E / 2 > Q) __builtin_amdgcn_sched_barrier(0);
    });
    if (deriv) {
      ma = c_imul(tb.negk[2][M], ma);
      mb = c_imul(tb.negk[2][M], mb);
    }
    line_sync<true>();
    auto mirrored = [&](auto set) {
      static_for<0, E>([&](auto S) {
        constexpr int s = decltype(S)::value;
        if constexpr (bin(s) >= M) {
          const int k = N - bin(s) - p;  // in (0, N / 2]
          float f = 0.f;
          if (N - bin(s) - P + 1 < klim) f = slot[k];  // uniform
          set(s, k < klim ? f : 0.f);
        }
      });
    };
    float re[E];
    mirrored([&](int s, float f) { re[s] = f; });
    line_sync<true>();
    static_for<0, E>([&](auto S) {
      constexpr int s = decltype(S)::value;
      if constexpr (bin(s) < M) {
        if (bin(s) < klim) slot[bin(s) + p] = v[E - 1 - s].y;
      }
    });
    line_sync<true>();
    mirrored([&](int s, float f) { v[s] = make_float2(re[s], f); });
    line_sync<true>();
    static_for<0, E>([&](auto S) {
      constexpr int s = decltype(S)::value;
      if constexpr (bin(s) == M) {
        if (p == 0) v[s] = make_float2(ma.x, mb.x);
      }
    });
    asm volatile("" ::: "memory");  // no twiddle loaded before the spectra are in
    inverse_core<N, true>(v, lds, p, idx, fresh_table(tw));
    if (!ok) return;
    float* da = zp.rout[comp] + la * zp.pitch_r;
    float* db = da + zp.pitch_r;
    const float sc = 0.5f * zp.out_scale;
    if constexpr (ADD) {
      const float* ea = zp.rout_add + la * zp.pitch_r;
#pragma unroll
      for (int s = 0; s < E; ++s)
        v[s] = make_float2(ea[nrow<N>(p, s)] + v[s].x * sc, ea[zp.pitch_r + nrow<N>(p, s)] + v[s].y * sc);
    } else {
#pragma unroll
      for (int s = 0; s < E; ++s) v[s] = make_float2(v[s].x * sc, v[s].y * sc);
    }
#pragma unroll
    for (int s = 0; s < E; ++s) {
      da[nrow<N>(p, s)] = v[s].x;
      db[nrow<N>(p, s)] = v[s].y;
    }
  }
}

// ------------------------------------------------------------ spectral tables ----
// Angular wavenumbers k = m * (1/n) * (2 pi / cell) evaluated in double and rounded to
// float (numerics/fft.py:30-41), the particle-Nyquist masks (core/utils.py:33-37) and
// negk with the derivative zeroed at the mesh Nyquist (configuration.py:369-376), all
// decided in float32 like the reference.
// Also clears `zero` (counters of the step that follows on the stream: one launch less).
__global__ void k_spec_tables(float* out, int n0, int n1, int n2, SpecTables sc, int32_t* __restrict__ zero,
                              int64_t nzero) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nzero; i += (int64_t)gridDim.x * blockDim.x)
    zero[i] = 0;
  int n[3] = {n0, n1, n2};
  int len[3] = {n0, n1, n2 / 2 + 1};
  int off = 0;
  for (int a = 0; a < 3; ++a) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < len[a]; i += gridDim.x * blockDim.x) {
      const float k = spec_k(i, n[a], a == 2, sc.period);
      out[off + i] = k;
      out[off + len[a] + i] = spec_keep(k, sc) ? 1.f : 0.f;
      out[off + 2 * len[a] + i] = spec_negk(k, sc);
    }
    off += 3 * len[a];
  }
}

// out = (adjoint ? conj(D) : D) * G * in on a standard-layout spectrum; axis < 0: D = 1.
__global__ void k_spectral_multiply(const float2* __restrict__ in, float2* __restrict__ out, int nx,
                                    int ny, int nzh, SpecTables tb, int axis, int adjoint) {
  int64_t total = (int64_t)nx * ny * nzh;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * blockDim.x) {
    int kz = (int)(i % nzh);
    int ky = (int)((i / nzh) % ny);
    int kx = (int)(i / ((int64_t)nzh * ny));
    float kxv = tb.k[0][kx], kyv = tb.k[1][ky], kzv = tb.k[2][kz];
    float k2 = kxv * kxv + kyv * kyv + kzv * kzv;
    bool keep = tb.mask[0][kx] != 0.f && tb.mask[1][ky] != 0.f && tb.mask[2][kz] != 0.f && k2 != 0.f;
    float2 v = in[i];
    float2 phi = keep ? make_float2(-v.x / k2, -v.y / k2) : make_float2(0.f, 0.f);
    if (axis >= 0) {
      int ki = axis == 0 ? kx : (axis == 1 ? ky : kz);
      float nk = tb.negk[axis][ki];
      phi = c_imul(adjoint ? -nk : nk, phi);
    }
    out[i] = phi;
  }
}

template <int N, int T, int MODE, int HALVES>
int launch_cols_cfg(const ColPass& cp, int batches, const SpecTables& tb, int dax, hipStream_t s,
                    const char* name) {
  using CF = ColCfg<N, T, HALVES>;
  const float2* tw = twiddle_table();
  PM_RETURN_IF(tw == nullptr, PM_ERROR_HIP, "twiddle table not initialised");
  const int gx = (int)ceil_div(cp.ncols, T);
  const int64_t tiles = (int64_t)gx * batches;
  const int64_t g = ceil_div(tiles * HALVES, 8) * 8;
  PM_RETURN_IF((HALVES > 1 || MODE == kColGreen) && (cp.in == cp.out0 || cp.in == cp.out1 || cp.out0 == cp.out1),
               PM_ERROR_INVALID_ARGUMENT, "FFT passes with several outputs need them distinct from their input");
  PM_RETURN_IF(MODE == kColInv3 && (cp.in1 == cp.out0 || cp.in1 == cp.out1 || cp.in1 == cp.out2 || cp.in == cp.out2 ||
                                    cp.out0 == cp.out2 || cp.out1 == cp.out2),
               PM_ERROR_INVALID_ARGUMENT, "FFT passes with several outputs need them distinct from their inputs");
  PM_RETURN_IF(g > INT32_MAX, PM_ERROR_UNSUPPORTED, "too many FFT column tiles");
  hipLaunchKernelGGL((k_cols<N, T, MODE, HALVES>), dim3((unsigned)g), dim3(CF::THREADS), 0, s, cp, tb, dax, tw,
                     gx, batches, (int)(g / 8));
  PM_LAUNCH_CHECK(name);
  PM_MARK(name, s);
  return PM_SUCCESS;
}

template <int N>
int launch_cols_n(int mode, const ColPass& cp, int batches, const SpecTables& tb, int dax,
                  hipStream_t s) {
  constexpr int T1 = (N >= 512) ? 8 : 16;  // one-output passes: 64 or 128-byte row segments
  constexpr int T2 = (N >= 2048) ? 4 : 8;   // passes with several outputs
  switch (mode) {
    case kColFwd: return launch_cols_cfg<N, T1, kColFwd, 1>(cp, batches, tb, dax, s, "fft_cols_fwd");
    case kColInv: return launch_cols_cfg<N, T1, kColInv, 1>(cp, batches, tb, dax, s, "fft_cols_inv");
    case kColInv3: return launch_cols_cfg<N, T2, kColInv3, 3>(cp, batches, tb, dax, s, "fft_cols_inv3");
    case kColGreen: return launch_cols_cfg<N, T2, kColGreen, 1>(cp, batches, tb, dax, s, "fft_cols_green");
    case kColSym: return launch_cols_cfg<N, T2, kColSym, 3>(cp, batches, tb, dax, s, "fft_cols_symbol");
    case kColAdj: return launch_cols_cfg<N, T1, kColAdj, 1>(cp, batches, tb, dax, s, "fft_cols_adjoint");
    case kColPot: return launch_cols_cfg<N, T2, kColPot, 1>(cp, batches, tb, dax, s, "fft_cols_potential");
    default: return fail(PM_ERROR_INVALID_ARGUMENT, "bad column mode");
  }
}

template <int N>
int launch_z_n(bool c2r, const ZPass& zp, const SpecTables& tb, hipStream_t s) {
  const float2* tw = twiddle_table();
  PM_RETURN_IF(tw == nullptr, PM_ERROR_HIP, "twiddle table not initialised");
  PM_RETURN_IF(zp.nlines % 2 != 0, PM_ERROR_UNSUPPORTED, "the FFT line passes take pairs of lines");
  if (zp.nlines == 0) return PM_SUCCESS;
  const unsigned blocks = (unsigned)ceil_div(zp.nlines / 2, ZCfg<N>::PAIRS);
  const dim3 threads(ZCfg<N>::THREADS);
  if (c2r) {
    const dim3 grid(blocks, (unsigned)zp.ncomp);
    if (zp.rout_add) {
      hipLaunchKernelGGL((k_zpass<N, true, true>), grid, threads, 0, s, zp, tb, tw);
      PM_LAUNCHED("fft_z_c2r_add", s);
    } else {
      hipLaunchKernelGGL((k_zpass<N, true>), grid, threads, 0, s, zp, tb, tw);
      PM_LAUNCHED("fft_z_c2r", s);
    }
  } else {
    if (zp.fold.xs)
      hipLaunchKernelGGL((k_zpass<N, false, true>), dim3(blocks), threads, 0, s, zp, tb, tw);
    else
      hipLaunchKernelGGL((k_zpass<N, false>), dim3(blocks), threads, 0, s, zp, tb, tw);
    PM_LAUNCHED("fft_z_r2c", s);
  }
  return PM_SUCCESS;
}

}  // namespace

#define PM_POW2_CASES(X) X(2) X(4) X(8) X(16) X(32) X(64) X(128) X(256) X(512) X(1024) X(2048)

int launch_cols(int n, int mode, const ColPass& cp, int batches, const SpecTables& tb, int dax,
                hipStream_t s) {
  if (batches == 0 || cp.ncols == 0) return PM_SUCCESS;
  switch (n) {
#define PM_CASE(V) \
  case V: return launch_cols_n<V>(mode, cp, batches, tb, dax, s);
    PM_POW2_CASES(PM_CASE)
#undef PM_CASE
    default: return fail(PM_ERROR_UNSUPPORTED, "FFT axis length must be a power of two in [2, 2048]");
  }
}

int launch_z(int nz, bool c2r, const ZPass& zp, const SpecTables& tb, hipStream_t s) {
  if (nz < 2 || nz > 2048 || !is_pow2(nz))
    return fail(PM_ERROR_UNSUPPORTED, "last FFT axis must be a power of two in [2, 2048]");
  switch (nz) {
#define PM_CASE(V) \
  case V: return launch_z_n<V>(c2r, zp, tb, s);
    PM_POW2_CASES(PM_CASE)
#undef PM_CASE
    default: return fail(PM_ERROR_UNSUPPORTED, "last FFT axis must be a power of two in [2, 2048]");
  }
}

bool supported_shape(const int32_t* shape) {
  for (int a = 0; a < 3; ++a)
    if (shape[a] < 2 || shape[a] > 2048 || !is_pow2(shape[a])) return false;
  return true;
}

size_t spec_table_floats(const int32_t* shape) {
  return 3 * ((size_t)shape[0] + shape[1] + (shape[2] / 2 + 1));
}

SpecTables spec_scalars(double cell_size, double ptcl_spacing, int mask_active) {
  SpecTables tb{};
  const float eps32 = 1.1920928955078125e-07f;
  tb.period = 2.0 * 3.14159265358979323846 / cell_size;
  const float k_nyq_ptcl = (float)(3.14159265358979323846 / ptcl_spacing);
  // two float32 roundings as the reference (volatile: no contraction into an fma)
  volatile float tol = k_nyq_ptcl * (8.0f * eps32);
  tb.klim = k_nyq_ptcl + tol;
  tb.nyq = (float)(3.14159265358979323846 / cell_size);
  tb.nyq_eps = tb.nyq * eps32;
  tb.mask_active = mask_active;
  return tb;
}

SpecTables spec_tables_view(const float* base, const int32_t* shape, const SpecTables& scalars) {
  SpecTables tb = scalars;
  int len[3] = {shape[0], shape[1], shape[2] / 2 + 1};
  size_t off = 0;
  for (int a = 0; a < 3; ++a) {
    tb.k[a] = base + off;
    tb.mask[a] = base + off + len[a];
    tb.negk[a] = base + off + 2 * len[a];
    off += 3 * (size_t)len[a];
  }
  return tb;
}

int launch_spec_tables(float* out, const int32_t* shape, const SpecTables& scalars, int32_t* zero, int64_t nzero,
                       hipStream_t s) {
  const unsigned blocks = (unsigned)std::max<int64_t>(8, std::min<int64_t>(ceil_div(nzero, 1024), 512));
  hipLaunchKernelGGL(k_spec_tables, dim3(blocks), dim3(256), 0, s, out, shape[0], shape[1], shape[2], scalars, zero,
                     nzero);
  PM_LAUNCHED("k_spec_tables", s);
  return PM_SUCCESS;
}

int launch_spectral_multiply(const float2* in, float2* out, const int32_t* shape, const SpecTables& tb,
                             int axis, int adjoint, hipStream_t s) {
  int64_t total = (int64_t)shape[0] * shape[1] * (shape[2] / 2 + 1);
  unsigned blocks = (unsigned)std::min<int64_t>(ceil_div(total, 256), 65536);
  hipLaunchKernelGGL(k_spectral_multiply, dim3(blocks), dim3(256), 0, s, in, out, shape[0], shape[1],
                     shape[2] / 2 + 1, tb, axis, adjoint);
  PM_LAUNCHED("k_spectral_multiply", s);
  return PM_SUCCESS;
}

// Forward 3D r2c on a half spectrum with row pitch `pitch` (>= nz/2+1), in place over
// `spec` (z pass writes it, y and x passes update it).
int rfft3d_pitched(const float* in, float2* spec, const int32_t* shape, int64_t pitch, float shift,
                   float scale, const SpecTables& tb, hipStream_t s) {
  const int nx = shape[0], ny = shape[1], nz = shape[2], m = nz / 2;
  ZPass zp{};
  zp.rin = in;
  zp.cmain[0] = spec;
  zp.pitch_r = nz;
  zp.pitch_c = pitch;
  zp.nlines = (int64_t)nx * ny;
  zp.src_shift = shift;
  zp.src_scale = scale;
  int st = launch_z(nz, false, zp, tb, s);
  if (st) return st;
  ColPass cy{spec, spec, nullptr, pitch, 1, (int64_t)ny * pitch, m + 1, 0, 0, 0, 0, 0};
  st = launch_cols(ny, kColFwd, cy, nx, tb, 0, s);
  if (st) return st;
  ColPass cx{spec, spec, nullptr, (int64_t)ny * pitch, 1, pitch, m + 1, 0, 0, 0, 0, 0};
  return launch_cols(nx, kColFwd, cx, ny, tb, 0, s);
}

// Row pitch of a scratch half spectrum: rows start on cache lines where they are several lines long.  Shorter
// ones would only get longer: inverse transform with / without, us, 2048^2 x 2 522 / 210, 1024^2 x 8 94 / 72,
// 512 x 256 x 64 57 / 50, 256^2 x 128 51 / 47, but 256^3 79 / 93, 512^3 898 / 1000, 256^2 x 2048 725 / 811.
int64_t scratch_pitch(const int32_t* shape) {
  const int64_t n = shape[2] / 2 + 1;
  return shape[2] >= 256 ? (int64_t)align_up((size_t)n, 16) : n;
}

// The y and z passes of ncomp inverse transforms whose x inverses lie one after the other in
// `spec` (pitched rows), into ncomp meshes one after the other (1/N normalised).
static int inverse_yz(float2* spec, float* out, const int32_t* shape, int64_t pitch, int ncomp, const SpecTables& tb,
                      hipStream_t s) {
  const int nx = shape[0], ny = shape[1], nz = shape[2], m = nz / 2;
  ColPass cy{spec, spec, nullptr, pitch, 1, (int64_t)ny * pitch, m + 1, 0, 0, 0, 0, 0};
  PM_TRY(launch_cols(ny, kColInv, cy, ncomp * nx, tb, 0, s));
  ZPass zp{};
  zp.rout[0] = out;
  zp.cmain[0] = spec;
  zp.pitch_r = nz;
  zp.pitch_c = pitch;
  zp.nlines = (int64_t)ncomp * nx * ny;
  zp.out_scale = (float)(2.0 / ((double)nx * ny * nz));
  return launch_z(nz, true, zp, tb, s);
}

size_t symbol_inverse_bytes(const int32_t* shape) {
  return sizeof(float2) * 3 * (size_t)shape[0] * shape[1] * scratch_pitch(shape);
}

// out[c] = irfftn(symbol_c(k) spec), c = 0..2, for a standard-layout spectrum that is only read: the
// symbols are applied by the x pass, which writes the three components to scratch; the y and z
// passes run over the three in one launch each (nine launches and three passes over a
// spectrum each before: the multiply, its scratch copy, and the transform's three).
int symbol_inverse3(const float2* spec, float* out, const int32_t* shape, const float* const ktab[3],
                    const ColSymbol sym[3], const float nyquist[3], const float tol[3], float2* scratch,
                    hipStream_t s) {
  const int nx = shape[0], ny = shape[1], m = shape[2] / 2;
  const int64_t pitch = scratch_pitch(shape), comp = (int64_t)nx * ny * pitch;
  SpecTables tb{};
  for (int a = 0; a < 3; ++a) tb.k[a] = ktab[a];
  ColPass cx{const_cast<float2*>(spec), scratch, scratch + comp, (int64_t)ny * (m + 1), 1, m + 1, m + 1, 0, 0, 0, 0, 0};
  cx.out2 = scratch + 2 * comp;
  cx.o_row = (int64_t)ny * pitch;
  cx.o_batch = pitch;
  for (int c = 0; c < 3; ++c) {
    cx.sym[c] = sym[c];
    cx.sym_nyq[c] = nyquist[c];
    cx.sym_tol[c] = tol[c];
  }
  PM_TRY(launch_cols(nx, kColSym, cx, ny, tb, 0, s));
  return inverse_yz(scratch, out, shape, pitch, 3, tb, s);
}

// Inverse 3D c2r of a standard-layout spectrum that is only read: the x pass writes the scratch.
int irfft3d_keep(const float2* spec, float* out, const int32_t* shape, float2* scratch, hipStream_t s) {
  const int nx = shape[0], ny = shape[1], m = shape[2] / 2;
  const int64_t pitch = scratch_pitch(shape);
  SpecTables tb{};
  ColPass cx{const_cast<float2*>(spec), scratch, nullptr, (int64_t)ny * (m + 1), 1, m + 1, m + 1, 0, 0, 0, 0, 0};
  cx.o_row = (int64_t)ny * pitch;
  cx.o_batch = pitch;
  PM_TRY(launch_cols(nx, kColInv, cx, ny, tb, 0, s));
  return inverse_yz(scratch, out, shape, pitch, 1, tb, s);
}

// Inverse 3D c2r (1/N normalised); the spectrum is used as scratch.
int irfft3d_pitched(float2* spec, float* out, const int32_t* shape, int64_t pitch, const SpecTables& tb,
                    hipStream_t s) {
  const int nx = shape[0], ny = shape[1], m = shape[2] / 2;
  ColPass cx{spec, spec, nullptr, (int64_t)ny * pitch, 1, pitch, m + 1, 0, 0, 0, 0, 0};
  PM_TRY(launch_cols(nx, kColInv, cx, ny, tb, 0, s));
  return inverse_yz(spec, out, shape, pitch, 1, tb, s);
}

}  // namespace fft
}  // namespace pm

using namespace pm;

extern "C" {

int pm_fft_workspace(const int32_t shape[3], size_t* bytes) {
  PM_RETURN_IF(shape == nullptr || bytes == nullptr, PM_ERROR_INVALID_ARGUMENT, "NULL argument");
  PM_RETURN_IF(!fft::supported_shape(shape), PM_ERROR_UNSUPPORTED,
               "FFT axes must be powers of two in [2, 2048]");
  *bytes = 0;
  return PM_SUCCESS;
}

int pm_rfft3d(const float* in, float* out_complex, const int32_t shape[3], void* workspace,
              size_t workspace_bytes, void* stream) {
  (void)workspace;
  (void)workspace_bytes;
  PM_RETURN_IF(shape == nullptr || in == nullptr || out_complex == nullptr, PM_ERROR_INVALID_ARGUMENT,
               "NULL argument");
  PM_RETURN_IF(!fft::supported_shape(shape), PM_ERROR_UNSUPPORTED,
               "FFT axes must be powers of two in [2, 2048]");
  int st = require_device_tables();
  if (st) return st;
  PM_RETURN_IF((const void*)in == (const void*)out_complex, PM_ERROR_INVALID_ARGUMENT,
               "pm_rfft3d needs distinct input and output buffers");
  fft::SpecTables tb{};
  return fft::rfft3d_pitched(in, reinterpret_cast<float2*>(out_complex), shape, shape[2] / 2 + 1, 0.f,
                             1.f, tb, as_stream(stream));
}

int pm_irfft3d(float* in_complex, float* out, const int32_t shape[3], void* workspace,
               size_t workspace_bytes, void* stream) {
  (void)workspace;
  (void)workspace_bytes;
  PM_RETURN_IF(shape == nullptr || in_complex == nullptr || out == nullptr, PM_ERROR_INVALID_ARGUMENT,
               "NULL argument");
  PM_RETURN_IF(!fft::supported_shape(shape), PM_ERROR_UNSUPPORTED,
               "FFT axes must be powers of two in [2, 2048]");
  int st = require_device_tables();
  if (st) return st;
  PM_RETURN_IF((const void*)in_complex == (const void*)out, PM_ERROR_INVALID_ARGUMENT,
               "pm_irfft3d needs distinct input and output buffers");
  fft::SpecTables tb{};
  return fft::irfft3d_pitched(reinterpret_cast<float2*>(in_complex), out, shape, shape[2] / 2 + 1, tb,
                              as_stream(stream));
}

int pm_irfft3d_keep_workspace(const int32_t shape[3], size_t* bytes) {
  PM_RETURN_IF(shape == nullptr || bytes == nullptr, PM_ERROR_INVALID_ARGUMENT, "NULL argument");
  PM_RETURN_IF(!fft::supported_shape(shape), PM_ERROR_UNSUPPORTED,
               "FFT axes must be powers of two in [2, 2048]");
  *bytes = sizeof(float2) * (size_t)shape[0] * shape[1] * fft::scratch_pitch(shape);
  return PM_SUCCESS;
}

int pm_irfft3d_keep(const float* in_complex, float* out, const int32_t shape[3], void* workspace,
                    size_t workspace_bytes, void* stream) {
  size_t need = 0;
  PM_TRY(pm_irfft3d_keep_workspace(shape, &need));
  PM_RETURN_IF(in_complex == nullptr || out == nullptr, PM_ERROR_INVALID_ARGUMENT, "NULL argument");
  PM_TRY(require_device_tables());
  PM_RETURN_IF(workspace == nullptr || workspace_bytes < need, PM_ERROR_WORKSPACE,
               "inverse FFT workspace too small: need " + std::to_string(need) + " bytes");
  return fft::irfft3d_keep(reinterpret_cast<const float2*>(in_complex), out, shape, static_cast<float2*>(workspace),
                           as_stream(stream));
}

}  // extern "C"
