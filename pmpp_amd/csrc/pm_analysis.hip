// Integer-shell power spectra of half-spectrum meshes (the P(k) metric).
//
// For every stored mode (kx, ky, kz <= Nz/2) of an rfft spectrum: shell = floor(|n| + 1e-9)
// of the integer mode vector, Hermitian multiplicity 2 (1 on the kz = 0 and even-Nz Nyquist
// planes), power |a|^2 (and |b|^2, Re a b*) times the mass-assignment deconvolution
// (sinc(nx/Nx) sinc(ny/Ny) sinc(nz/Nz))^(-2p), accumulated per shell.  Sums are float64:
// registers, per-block LDS accumulators, then one global atomic per shell and block, so the
// summation order (not the value beyond float64 rounding) varies between runs.
#include <algorithm>

#include "pm_common.h"

namespace pm {
namespace analysis {
namespace {

constexpr int kBlock = 256;
constexpr int kMaxShells = 2048;

__device__ __forceinline__ float sinc_f(float x) {
  if (x == 0.f) return 1.f;
  const float px = 3.14159265358979323846f * x;
  return sinpif(x) / px;
}

__global__ void k_zero_f64(double* __restrict__ p, int n) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) p[i] = 0.0;
}

// Bound by reading the spectra once.  A thread keeps one (|kx|, kz) and walks |ky| upwards, taking the
// up to four modes (+-kx, +-ky) of a step together: they share shell and window, the shell only
// grows along the walk, by at most one a step (no square root), and the modes of a shell are added
// up in a register, so an LDS atomic is paid per shell and walk instead of per mode.  Adjacent lanes
// are adjacent in kz.  A walk is cut into `chunk` steps where there are too few of them to fill
// the chip.  The window's factors come per thread (x, z) and from a table of the chunk (y).
// 256^3 (68 MB): 77 us with an atomic, an f64 square root and three sines per mode, 19 us now.
constexpr int kShellBlock = 512;
constexpr int kShellChunk = 1024;  // longest chunk (its window table is in LDS)

template <bool CROSS>
__global__ void __launch_bounds__(kShellBlock) k_shell_sums(const float2* __restrict__ a, const float2* __restrict__ b,
                                                            int nx, int ny, int nz, int mas_power, int num_shells,
                                                            int density, int chunk, double* __restrict__ sums) {
  extern __shared__ double acc[];  // nw * num_shells, then the chunk's window factors
  constexpr int nw = CROSS ? 3 : 1;
  float* sy = reinterpret_cast<float*>(acc + nw * num_shells);
  const int nzh = nz / 2 + 1, hx = nx / 2 + 1, hy = ny / 2 + 1;
  const int y0 = blockIdx.y * chunk, y1 = min(hy, y0 + chunk);
  for (int i = threadIdx.x; i < nw * num_shells; i += kShellBlock) acc[i] = 0.0;
  for (int i = threadIdx.x; i < y1 - y0; i += kShellBlock) sy[i] = sinc_f((float)(y0 + i) / (float)ny);
  __syncthreads();
  const int64_t nm = (int64_t)nx * ny * nz;
  // density inputs: delta_k = rho_k / mean(rho) away from k = 0, mean = Re rho_0 / N_m
  float sa = 1.f, sb = 1.f;
  if (density) {
    sa = (float)((double)nm / (double)a[0].x);
    if (CROSS) sb = (float)((double)nm / (double)b[0].x);
  }
  const int64_t q = (int64_t)blockIdx.x * kShellBlock + threadIdx.x;
  if (q < (int64_t)hx * nzh) {
    const int mx = (int)(q / nzh), mz = (int)(q - (int64_t)mx * nzh);
    const bool dupx = mx > 0 && 2 * mx < nx;
    const float wx = sinc_f((float)mx / (float)nx), wz = sinc_f((float)mz / (float)nz);
    const float mult = (mz == 0 || ((nz % 2) == 0 && mz == nz / 2)) ? 1.f : 2.f;
    const int64_t xoff = dupx ? (int64_t)(nx - 2 * mx) * ny * nzh : 0;  // to the row of -kx
    int64_t msq = (int64_t)mx * mx + (int64_t)mz * mz + (int64_t)y0 * y0;
    int64_t shell = (int64_t)floor(sqrt((double)msq) + 1e-9);
    int64_t next = (shell + 1) * (shell + 1);
    double run[nw] = {};
    auto flush = [&]() {
      const int64_t sh = shell < num_shells ? shell : num_shells - 1;
#pragma unroll
      for (int c = 0; c < nw; ++c) {
        atomicAdd(&acc[c * num_shells + sh], run[c]);
        run[c] = 0.0;
      }
    };
    for (int my = y0; my < y1; ++my) {
      const bool dupy = my > 0 && 2 * my < ny;
      const int64_t i0 = ((int64_t)mx * ny + my) * nzh + mz;
      const int64_t yoff = dupy ? (int64_t)(ny - 2 * my) * nzh : 0;  // to the row of -ky
      float2 va[4], vb[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) {  // absent partners read the mode itself again
        const int64_t i = i0 + ((c & 1) ? yoff : 0) + ((c & 2) ? xoff : 0);
        va[c] = a[i];
        if (CROSS) vb[c] = b[i];
      }
      if (msq >= next) {
        flush();
        ++shell;
        next += 2 * shell + 1;
      }
      msq += 2 * my + 1;
      float w = 1.f;
      if (mas_power > 0) {
        const float win = wx * sy[my - y0] * wz;
        const float inv = 1.f / win;
        const float inv2 = inv * inv;
        for (int p = 0; p < mas_power; ++p) w *= inv2;
      }
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        if (((c & 1) && !dupy) || ((c & 2) && !dupx)) continue;
        const float2 u = make_float2(va[c].x * sa, va[c].y * sa);
        run[0] += (double)((u.x * u.x + u.y * u.y) * w * mult);
        if constexpr (CROSS) {
          const float2 v = make_float2(vb[c].x * sb, vb[c].y * sb);
          run[1] += (double)((v.x * v.x + v.y * v.y) * w * mult);
          run[2] += (double)((u.x * v.x + u.y * v.y) * w * mult);
        }
      }
    }
    flush();
  }
  __syncthreads();
  for (int i = threadIdx.x; i < nw * num_shells; i += kShellBlock) {
    const double v = acc[i];
    if (v != 0.0) atomicAdd(&sums[i], v);
  }
}

// Reverse of the shell sums: grad_k = coef[shell(k)] * window(k) * s^2 * a_k, s the density
// normalisation (1 for an overdensity), shell and window exactly as the forward.  With
// coef[s] = 2 cell^3 dL/dP_s / nmodes_s, irfftn(grad) is dL/d(mesh) of L(P) (the constant
// term from the mean of a density input is left out: it carries no particle gradient).
__global__ void __launch_bounds__(kBlock) k_shell_grad(const float2* __restrict__ a, float2* __restrict__ g, int nx,
                                                       int ny, int nz, int mas_power, int num_shells,
                                                       const float* __restrict__ coef, int density) {
  const int nzh = nz / 2 + 1;
  const int64_t total = (int64_t)nx * ny * nzh;
  const int64_t nm = (int64_t)nx * ny * nz;
  const float s = density ? (float)((double)nm / (double)a[0].x) : 1.f;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
    const int kz = (int)(i % nzh);
    const int ky = (int)((i / nzh) % ny);
    const int kx = (int)(i / ((int64_t)nzh * ny));
    const int mx = kx < (nx + 1) / 2 ? kx : kx - nx;
    const int my = ky < (ny + 1) / 2 ? ky : ky - ny;
    const int mz = kz;
    const int64_t msq = (int64_t)mx * mx + (int64_t)my * my + (int64_t)mz * mz;
    int shell = (int)floor(sqrt((double)msq) + 1e-9);
    shell = shell < num_shells ? shell : num_shells - 1;
    float w = 1.f;
    if (mas_power > 0) {
      const float win = sinc_f((float)mx / (float)nx) * sinc_f((float)my / (float)ny) * sinc_f((float)mz / (float)nz);
      const float inv = 1.f / win;
      const float inv2 = inv * inv;
      for (int p = 0; p < mas_power; ++p) w *= inv2;
    }
    const float f = coef[shell] * w * s * s;
    const float2 v = a[i];
    g[i] = make_float2(f * v.x, f * v.y);
  }
}

}  // namespace
}  // namespace analysis
}  // namespace pm

using namespace pm;

extern "C" {

int pm_power_spectrum(const float* spec_a, const float* spec_b, const int32_t shape[3], int32_t mas_power,
                      int32_t num_shells, int32_t density, double* sums, void* stream) {
  PM_RETURN_IF(spec_a == nullptr || shape == nullptr || sums == nullptr, PM_ERROR_INVALID_ARGUMENT,
               "NULL argument");
  for (int a = 0; a < 3; ++a) PM_RETURN_IF(shape[a] < 1, PM_ERROR_INVALID_ARGUMENT, "mesh axes must be >= 1");
  PM_RETURN_IF(num_shells < 1 || num_shells > analysis::kMaxShells, PM_ERROR_UNSUPPORTED,
               "num_shells must be in [1, 2048]");
  PM_RETURN_IF(mas_power < 0 || mas_power > 4, PM_ERROR_INVALID_ARGUMENT, "mas_power must be in [0, 4]");
  hipStream_t s = as_stream(stream);
  const bool cross = spec_b != nullptr;
  const int nw = cross ? 3 : 1;
  hipLaunchKernelGGL(analysis::k_zero_f64, dim3(1), dim3(256), 0, s, sums, nw * num_shells);
  PM_LAUNCHED("k_zero_f64", s);
  // walks cut until there are about 2^18 of them
  const int64_t walks = (int64_t)(shape[0] / 2 + 1) * (shape[2] / 2 + 1), hy = shape[1] / 2 + 1;
  const int64_t cuts = std::min<int64_t>(hy, std::max<int64_t>(ceil_div(int64_t(1) << 18, walks),
                                                                ceil_div(hy, analysis::kShellChunk)));
  const int chunk = (int)ceil_div(hy, cuts);
  const dim3 grid((unsigned)ceil_div(walks, analysis::kShellBlock), (unsigned)ceil_div(hy, chunk));
  const size_t lds = sizeof(double) * nw * num_shells + sizeof(float) * chunk;
  const float2* a = reinterpret_cast<const float2*>(spec_a);
  const float2* b = reinterpret_cast<const float2*>(spec_b);
  if (cross)
    hipLaunchKernelGGL(analysis::k_shell_sums<true>, grid, dim3(analysis::kShellBlock), lds, s, a, b, shape[0],
                       shape[1], shape[2], mas_power, num_shells, density, chunk, sums);
  else
    hipLaunchKernelGGL(analysis::k_shell_sums<false>, grid, dim3(analysis::kShellBlock), lds, s, a, b, shape[0],
                       shape[1], shape[2], mas_power, num_shells, density, chunk, sums);
  PM_LAUNCHED("k_shell_sums", s);
  return PM_SUCCESS;
}

int pm_power_spectrum_bwd(const float* spec, const int32_t shape[3], int32_t mas_power, int32_t num_shells,
                          int32_t density, const float* shell_coef, float* grad_spec, void* stream) {
  PM_RETURN_IF(spec == nullptr || shape == nullptr || shell_coef == nullptr || grad_spec == nullptr,
               PM_ERROR_INVALID_ARGUMENT, "NULL argument");
  for (int a = 0; a < 3; ++a) PM_RETURN_IF(shape[a] < 1, PM_ERROR_INVALID_ARGUMENT, "mesh axes must be >= 1");
  PM_RETURN_IF(num_shells < 1 || num_shells > analysis::kMaxShells, PM_ERROR_UNSUPPORTED,
               "num_shells must be in [1, 2048]");
  PM_RETURN_IF(mas_power < 0 || mas_power > 4, PM_ERROR_INVALID_ARGUMENT, "mas_power must be in [0, 4]");
  hipStream_t s = as_stream(stream);
  const int64_t total = (int64_t)shape[0] * shape[1] * (shape[2] / 2 + 1);
  const unsigned blocks =
      (unsigned)std::max<int64_t>(1, std::min<int64_t>(ceil_div(total, analysis::kBlock * 4), 65536));
  hipLaunchKernelGGL(analysis::k_shell_grad, dim3(blocks), dim3(analysis::kBlock), 0, s,
                     reinterpret_cast<const float2*>(spec), reinterpret_cast<float2*>(grad_spec), shape[0], shape[1],
                     shape[2], mas_power, num_shells, shell_coef, density);
  PM_LAUNCHED("k_shell_grad", s);
  return PM_SUCCESS;
}

}  // extern "C"
