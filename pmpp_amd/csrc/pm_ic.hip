// Initial conditions on the particle grid: the linear-mode filter and the spectral and
// real-space steps of 2LPT.  Spectra are the standard rfftn layout (n0, n1, n2/2 + 1) complex
// of pm_rfft3d; wavenumbers come from per-axis float32 tables (the angular fftfreq of the
// particle grid), so every mode sees exactly the same k as the reference's float32 kvec.
#include <algorithm>
#include <cmath>

#include "pm_common.h"
#include "pm_fft_launch.h"

namespace pm {
namespace ic {
namespace {

constexpr int kBlock = 256;

unsigned grid_for(int64_t n) {
  return (unsigned)std::max<int64_t>(1, std::min<int64_t>(ceil_div(n, (int64_t)kBlock * 4), 65536));
}

struct KTabs {
  const float* k0;
  const float* k1;
  const float* k2;
  int n0, n1, nzh;
};

__device__ __forceinline__ void mode_k(const KTabs& t, int64_t i, float& a, float& b, float& c) {
  const int kz = (int)(i % t.nzh);
  const int64_t r = i / t.nzh;
  const int ky = (int)(r % t.n1);
  const int kx = (int)(r / t.n1);
  a = t.k0[kx];
  b = t.k1[ky];
  c = t.k2[kz];
}

// linear interpolation on an ascending table, clamped at both ends (numpy/jax interp)
__device__ __forceinline__ float interp(float x, const float* __restrict__ xs, const float* __restrict__ ys, int n) {
  if (x <= xs[0]) return ys[0];
  if (x >= xs[n - 1]) return ys[n - 1];
  int lo = 0, hi = n - 1;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (xs[mid] <= x)
      lo = mid;
    else
      hi = mid;
  }
  const float t = (x - xs[lo]) / (xs[hi] - xs[lo]);
  return ys[lo] + t * (ys[hi] - ys[lo]);
}

// spec *= scale * sqrt(P(k)),  P(k) = coef (k / k_pivot)^n_s T(k)^2, P(0) = 0
__global__ void __launch_bounds__(kBlock) k_linear_modes(float2* __restrict__ spec, KTabs t,
                                                         const float* __restrict__ tk,
                                                         const float* __restrict__ tT, int nt, float coef,
                                                         float k_pivot, float n_s, float scale) {
  const int64_t total = (int64_t)t.n0 * t.n1 * t.nzh;
  for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < total; i += (int64_t)gridDim.x * kBlock) {
    float a, b, c;
    mode_k(t, i, a, b, c);
    const float k = sqrtf(a * a + b * b + c * c);
    float f = 0.f;
    if (k > 0.f) {
      const float T = interp(k, tk, tT, nt);
      const float p = coef * powf(k / k_pivot, n_s) * T * T;
      f = scale * sqrtf(fmaxf(p, 0.f));
    }
    const float2 v = spec[i];
    spec[i] = make_float2(v.x * f, v.y * f);
  }
}

enum Op : int { kScale = 0, kLaplace = 1, kStrain = 2, kNegGrad = 3, kPotential = 4 };

__device__ __forceinline__ float pick(int axis, float a, float b, float c) {
  return axis == 0 ? a : (axis == 1 ? b : c);
}

// out = symbol(k) * in for one of: s (kScale), -1/k^2 with k = 0 -> 0 (kLaplace), the two in
// this order (kPotential),
// -k_i k_j with the Nyquist k zeroed when i != j (kStrain), -i k_i with the Nyquist k
// zeroed (kNegGrad).  nyq[a] = pi / spacing_a, |(|k| - nyq)| <= tol[a] marks the Nyquist.
__global__ void __launch_bounds__(kBlock) k_spectral_op(const float2* __restrict__ in, float2* __restrict__ out,
                                                        KTabs t, int op, int ai, int aj, float s, float3 nyq,
                                                        float3 tol) {
  const int64_t total = (int64_t)t.n0 * t.n1 * t.nzh;
  for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < total; i += (int64_t)gridDim.x * kBlock) {
    float a, b, c;
    mode_k(t, i, a, b, c);
    const float2 v = in[i];
    float2 r;
    if (op == kScale) {
      r = make_float2(v.x * s, v.y * s);
    } else if (op == kLaplace || op == kPotential) {
      const float k2 = a * a + b * b + c * c;
      const float2 w = op == kPotential ? make_float2(v.x * s, v.y * s) : v;
      r = k2 != 0.f ? make_float2(-w.x / k2, -w.y / k2) : make_float2(0.f, 0.f);
    } else {
      float ki = pick(ai, a, b, c);
      const float nqi = pick(ai, nyq.x, nyq.y, nyq.z), tli = pick(ai, tol.x, tol.y, tol.z);
      if (op == kNegGrad) {
        if (fabsf(fabsf(ki) - nqi) <= tli) ki = 0.f;
        r = make_float2(ki * v.y, -ki * v.x);  // -i k v
      } else {
        float kj = pick(aj, a, b, c);
        if (ai != aj) {
          const float nqj = pick(aj, nyq.x, nyq.y, nyq.z), tlj = pick(aj, tol.x, tol.y, tol.z);
          if (fabsf(fabsf(ki) - nqi) <= tli) ki = 0.f;
          if (fabsf(fabsf(kj) - nqj) <= tlj) kj = 0.f;
        }
        const float m = -ki * kj;
        r = make_float2(m * v.x, m * v.y);
      }
    }
    out[i] = r;
  }
}

// acc = (init ? 0 : acc) + coef * a * b  (b == null: + coef * a)
__global__ void __launch_bounds__(kBlock) k_product_acc(float* __restrict__ acc, const float* __restrict__ a,
                                                        const float* __restrict__ b, int64_t n, float coef,
                                                        int init) {
  for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock) {
    const float p = b ? a[i] * b[i] : a[i];
    acc[i] = init ? coef * p : acc[i] + coef * p;
  }
}

// L = d0 d2 + d0 d1 + d1 d2 - d01^2 - d02^2 - d12^2 of the six strain meshes d0, d1, d2, d01, d02, d12
// (n cells each, one after the other): the 2LPT source in one pass over them (six passes before)
__global__ void __launch_bounds__(kBlock) k_lpt2_source(const float* __restrict__ d, int64_t n,
                                                        float* __restrict__ L) {
  for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock) {
    const float d0 = d[i], d1 = d[n + i], d2 = d[2 * n + i];
    const float d01 = d[3 * n + i], d02 = d[4 * n + i], d12 = d[5 * n + i];
    float v = d0 * d2;
    v = v + d0 * d1;
    v = v + d1 * d2;
    v = v - d01 * d01;
    v = v - d02 * d02;
    L[i] = v - d12 * d12;
  }
}

// Particles on the Lagrangian grid (g0, g1, g2) of a mesh (m0, m1, m2): per axis the anchor rint(i
// (m / g)) and what is left of the position as a displacement (i m - anchor g) (cell / g), both in
// float64 as the host would form them (an anchor past int16 wraps as there); to it the LPT terms D1
// grad1 + D2 grad2 (component-major meshes on the grid; null: none), and the velocities V1 grad1 + V2
// grad2.  Bound by HBM (18 bytes written per particle, with LPT 30, and 24 read); four particles per
// thread, whole vectors.
struct LatticeAxes {
  int g[3], m[3];
  double step[3], left[3];  // m / g, cell / g
};

__global__ void __launch_bounds__(kBlock) k_lpt_particles(LatticeAxes ax, const float* __restrict__ grad1,
                                                          const float* __restrict__ grad2, float D1, float V1, float D2,
                                                          float V2, int vec, int16_t* __restrict__ pmid,
                                                          float* __restrict__ disp, float* __restrict__ vel) {
  const int64_t n = (int64_t)ax.g[0] * ax.g[1] * ax.g[2];
  for (int64_t i0 = 4 * ((int64_t)blockIdx.x * kBlock + threadIdx.x); i0 < n; i0 += 4 * (int64_t)gridDim.x * kBlock) {
    const int live = (int)min(int64_t(4), n - i0);
    const bool whole = vec && live == 4;
    int16_t p[12];
    float d[12], v[12];
    float ga[3][4], gb[3][4];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
#pragma unroll
      for (int e = 0; e < 4; ++e) ga[a][e] = gb[a][e] = 0.f;
      if (whole) {
        if (grad1) {
          const float4 t = *reinterpret_cast<const float4*>(grad1 + a * n + i0);
          ga[a][0] = t.x, ga[a][1] = t.y, ga[a][2] = t.z, ga[a][3] = t.w;
        }
        if (grad2) {
          const float4 t = *reinterpret_cast<const float4*>(grad2 + a * n + i0);
          gb[a][0] = t.x, gb[a][1] = t.y, gb[a][2] = t.z, gb[a][3] = t.w;
        }
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (grad1 && e < live) ga[a][e] = grad1[a * n + i0 + e];
          if (grad2 && e < live) gb[a][e] = grad2[a * n + i0 + e];
        }
      }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int64_t i = min(i0 + e, n - 1);
      const int iz = (int)(i % ax.g[2]);
      const int64_t r = i / ax.g[2];
      const int idx[3] = {(int)(r / ax.g[1]), (int)(r % ax.g[1]), iz};
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        const int anchor = (int)rint((double)idx[a] * ax.step[a]);
        const int64_t left = (int64_t)idx[a] * ax.m[a] - (int64_t)anchor * ax.g[a];
        float x = (float)((double)left * ax.left[a]), u = 0.f;
        if (grad1) {
          x += D1 * ga[a][e];
          u += V1 * ga[a][e];
        }
        if (grad2) {
          x += D2 * gb[a][e];
          u += V2 * gb[a][e];
        }
        p[3 * e + a] = (int16_t)anchor;
        d[3 * e + a] = x;
        v[3 * e + a] = u;
      }
    }
    if (whole) {
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        reinterpret_cast<short4*>(pmid + 3 * i0)[q] = make_short4(p[4 * q], p[4 * q + 1], p[4 * q + 2], p[4 * q + 3]);
        reinterpret_cast<float4*>(disp + 3 * i0)[q] = make_float4(d[4 * q], d[4 * q + 1], d[4 * q + 2], d[4 * q + 3]);
        if (vel)
          reinterpret_cast<float4*>(vel + 3 * i0)[q] = make_float4(v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]);
      }
    } else {
#pragma unroll
      for (int e = 0; e < 12; ++e)
        if (e < 3 * live) {
          pmid[3 * i0 + e] = p[e];
          disp[3 * i0 + e] = d[e];
          if (vel) vel[3 * i0 + e] = v[e];
        }
    }
  }
}

// disp[:, axis] += D g, vel[:, axis] += V g for particles in grid order
__global__ void __launch_bounds__(kBlock) k_lpt_acc(float* __restrict__ disp, float* __restrict__ vel,
                                                    const float* __restrict__ g, int64_t n, int axis, float D,
                                                    float V) {
  for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock) {
    const float v = g[i];
    disp[3 * i + axis] += D * v;
    if (vel) vel[3 * i + axis] += V * v;
  }
}

}  // namespace
}  // namespace ic
}  // namespace pm

using namespace pm;

namespace {

int check_ktabs(const int32_t* shape, const float* const* ktab, ic::KTabs& t) {
  PM_RETURN_IF(shape == nullptr || ktab == nullptr, PM_ERROR_INVALID_ARGUMENT, "NULL argument");
  for (int a = 0; a < 3; ++a) {
    PM_RETURN_IF(shape[a] < 1, PM_ERROR_INVALID_ARGUMENT, "grid axes must be >= 1");
    PM_RETURN_IF(ktab[a] == nullptr, PM_ERROR_INVALID_ARGUMENT, "wavenumber table NULL");
  }
  t.k0 = ktab[0];
  t.k1 = ktab[1];
  t.k2 = ktab[2];
  t.n0 = shape[0];
  t.n1 = shape[1];
  t.nzh = shape[2] / 2 + 1;
  return PM_SUCCESS;
}

}  // namespace

extern "C" {

int pm_ic_linear_modes(float* spec, const int32_t shape[3], const float* const ktab[3], const float* table_k,
                       const float* table_T, int32_t table_n, float coef, float k_pivot, float n_s, float scale,
                       void* stream) {
  ic::KTabs t{};
  PM_TRY(check_ktabs(shape, ktab, t));
  PM_RETURN_IF(spec == nullptr || table_k == nullptr || table_T == nullptr, PM_ERROR_INVALID_ARGUMENT,
               "NULL argument");
  PM_RETURN_IF(table_n < 2, PM_ERROR_INVALID_ARGUMENT, "transfer table needs >= 2 entries");
  const int64_t total = (int64_t)t.n0 * t.n1 * t.nzh;
  hipStream_t s = as_stream(stream);
  hipLaunchKernelGGL(ic::k_linear_modes, dim3(ic::grid_for(total)), dim3(ic::kBlock), 0, s,
                     reinterpret_cast<float2*>(spec), t, table_k, table_T, table_n, coef, k_pivot, n_s, scale);
  PM_LAUNCHED("k_linear_modes", s);
  return PM_SUCCESS;
}

int pm_ic_spectral_op(const float* in, float* out, const int32_t shape[3], const float* const ktab[3], int32_t op,
                      int32_t axis_i, int32_t axis_j, float scale, const float nyquist[3], const float tol[3],
                      void* stream) {
  ic::KTabs t{};
  PM_TRY(check_ktabs(shape, ktab, t));
  PM_RETURN_IF(in == nullptr || out == nullptr, PM_ERROR_INVALID_ARGUMENT, "NULL argument");
  PM_RETURN_IF(op < 0 || op > 4, PM_ERROR_INVALID_ARGUMENT, "unknown spectral op");
  const bool axes = op == ic::kStrain || op == ic::kNegGrad;
  PM_RETURN_IF(axes && (axis_i < 0 || axis_i > 2 || axis_j < 0 || axis_j > 2), PM_ERROR_INVALID_ARGUMENT,
               "axis out of range");
  PM_RETURN_IF(axes && (nyquist == nullptr || tol == nullptr), PM_ERROR_INVALID_ARGUMENT,
               "Nyquist tables NULL");
  float3 nq = make_float3(0.f, 0.f, 0.f), tl = make_float3(-1.f, -1.f, -1.f);
  if (axes) {
    nq = make_float3(nyquist[0], nyquist[1], nyquist[2]);
    tl = make_float3(tol[0], tol[1], tol[2]);
  }
  const int64_t total = (int64_t)t.n0 * t.n1 * t.nzh;
  hipStream_t s = as_stream(stream);
  hipLaunchKernelGGL(ic::k_spectral_op, dim3(ic::grid_for(total)), dim3(ic::kBlock), 0, s,
                     reinterpret_cast<const float2*>(in), reinterpret_cast<float2*>(out), t, (int)op, (int)axis_i,
                     (int)axis_j, scale, nq, tl);
  PM_LAUNCHED("k_spectral_op", s);
  return PM_SUCCESS;
}

int pm_ic_product_acc(float* acc, const float* a, const float* b, int64_t n, float coef, int32_t init,
                      void* stream) {
  PM_RETURN_IF(n < 0 || (n > 0 && (acc == nullptr || a == nullptr)), PM_ERROR_INVALID_ARGUMENT, "NULL argument");
  if (n == 0) return PM_SUCCESS;
  hipStream_t s = as_stream(stream);
  hipLaunchKernelGGL(ic::k_product_acc, dim3(ic::grid_for(n)), dim3(ic::kBlock), 0, s, acc, a, b, n, coef, (int)init);
  PM_LAUNCHED("k_product_acc", s);
  return PM_SUCCESS;
}

int pm_ic_lpt_accumulate(float* disp, float* vel, const float* grad, int64_t n, int32_t axis, float D, float V,
                         void* stream) {
  PM_RETURN_IF(n < 0 || (n > 0 && (disp == nullptr || grad == nullptr)), PM_ERROR_INVALID_ARGUMENT, "NULL argument");
  PM_RETURN_IF(axis < 0 || axis > 2, PM_ERROR_INVALID_ARGUMENT, "axis out of range");
  if (n == 0) return PM_SUCCESS;
  hipStream_t s = as_stream(stream);
  hipLaunchKernelGGL(ic::k_lpt_acc, dim3(ic::grid_for(n)), dim3(ic::kBlock), 0, s, disp, vel, grad, n, (int)axis, D,
                     V);
  PM_LAUNCHED("k_lpt_acc", s);
  return PM_SUCCESS;
}

int pm_ic_symbol_inverse_workspace(const int32_t shape[3], size_t* bytes) {
  PM_RETURN_IF(shape == nullptr || bytes == nullptr, PM_ERROR_INVALID_ARGUMENT, "NULL argument");
  PM_RETURN_IF(!fft::supported_shape(shape), PM_ERROR_UNSUPPORTED, "FFT axes must be powers of two in [2, 2048]");
  *bytes = fft::symbol_inverse_bytes(shape);
  return PM_SUCCESS;
}

int pm_ic_symbol_inverse(const float* in, float* out, const int32_t shape[3], const float* const ktab[3], int32_t kind,
                         const float nyquist[3], const float tol[3], void* workspace, size_t workspace_bytes,
                         void* stream) {
  size_t need = 0;
  PM_TRY(pm_ic_symbol_inverse_workspace(shape, &need));
  ic::KTabs t{};
  PM_TRY(check_ktabs(shape, ktab, t));
  PM_RETURN_IF(in == nullptr || out == nullptr || nyquist == nullptr || tol == nullptr, PM_ERROR_INVALID_ARGUMENT,
               "NULL argument");
  PM_RETURN_IF(kind < 0 || kind > 2, PM_ERROR_INVALID_ARGUMENT, "kind must be 0, 1 or 2");
  PM_RETURN_IF(workspace == nullptr || workspace_bytes < need, PM_ERROR_WORKSPACE,
               "symbol inverse workspace too small: need " + std::to_string(need) + " bytes");
  PM_TRY(require_device_tables());
  const fft::ColSymbol sym[3][3] = {{{0, 0}, {1, 1}, {2, 2}}, {{0, 1}, {0, 2}, {1, 2}}, {{0, -1}, {1, -1}, {2, -1}}};
  return fft::symbol_inverse3(reinterpret_cast<const float2*>(in), out, shape, ktab, sym[kind], nyquist, tol,
                              static_cast<float2*>(workspace), as_stream(stream));
}

int pm_ic_lpt2_source(const float* strains, int64_t n, float* out, void* stream) {
  PM_RETURN_IF(n < 0 || (n > 0 && (strains == nullptr || out == nullptr)), PM_ERROR_INVALID_ARGUMENT, "NULL argument");
  if (n == 0) return PM_SUCCESS;
  hipStream_t s = as_stream(stream);
  hipLaunchKernelGGL(ic::k_lpt2_source, dim3(ic::grid_for(n)), dim3(ic::kBlock), 0, s, strains, n, out);
  PM_LAUNCHED("k_lpt2_source", s);
  return PM_SUCCESS;
}

int pm_ic_lpt_particles(const int32_t grid[3], const int32_t mesh[3], double cell_size, const float* grad1,
                        const float* grad2, float D1, float V1, float D2, float V2, int16_t* pmid, float* disp,
                        float* vel, void* stream) {
  PM_RETURN_IF(grid == nullptr || mesh == nullptr, PM_ERROR_INVALID_ARGUMENT, "NULL argument");
  ic::LatticeAxes ax;
  int64_t n = 1;
  for (int a = 0; a < 3; ++a) {
    PM_RETURN_IF(grid[a] < 1 || mesh[a] < grid[a], PM_ERROR_INVALID_ARGUMENT,
                 "the mesh must be at least the particle grid");
    ax.g[a] = grid[a];
    ax.m[a] = mesh[a];
    ax.step[a] = (double)mesh[a] / (double)grid[a];
    ax.left[a] = cell_size / (double)grid[a];
    n *= grid[a];
  }
  PM_RETURN_IF(pmid == nullptr || disp == nullptr, PM_ERROR_INVALID_ARGUMENT, "pmid/disp NULL");
  const int vec = n % 4 == 0 && reinterpret_cast<uintptr_t>(pmid) % 8 == 0 &&
                  ((reinterpret_cast<uintptr_t>(disp) | reinterpret_cast<uintptr_t>(vel) |
                    reinterpret_cast<uintptr_t>(grad1) | reinterpret_cast<uintptr_t>(grad2)) & 15) == 0;
  hipStream_t s = as_stream(stream);
  const unsigned blocks = (unsigned)std::max<int64_t>(1, std::min<int64_t>(ceil_div(n, 4 * ic::kBlock), 8192));
  hipLaunchKernelGGL(ic::k_lpt_particles, dim3(blocks), dim3(ic::kBlock), 0, s, ax, grad1, grad2, D1, V1, D2, V2, vec,
                     pmid, disp, vel);
  PM_LAUNCHED("k_lpt_particles", s);
  return PM_SUCCESS;
}

}  // extern "C"
