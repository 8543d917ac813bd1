// Pointwise kernels of the differentiable band energy sum_b sum_r V |psi_b|^2:
// the energy (one pass over the fields) and the field 2 V psi g that the adjoint
// transform takes (one more). Called by the autograd layer, on its stream.
//
// Both are bound by the bytes of the fields. As tensor expressions the energy
// took five passes over them and the field three: six bands of 60^3 FP64 (20.7
// MB of fields) 43 us and 16 us on the GPU and some ten launches from Python,
// which bound the whole gradient.
#include <hip/hip_runtime.h>

#include "fft_common.hpp"
#include "hip_check.hpp"

namespace spfft {

namespace {

constexpr int kThreads = 256;
constexpr int kEnergyBlocks = 64;  // per band

// Sum over the workgroup, in a fixed order (result in thread 0).
__device__ __forceinline__ double block_sum(double x) {
  __shared__ double part[kThreads / 64];
  for (int d = 32; d > 0; d /= 2) x += __shfl_xor(x, d);
  if (threadIdx.x % 64 == 0) part[threadIdx.x / 64] = x;
  __syncthreads();
  x = part[0];
  for (int w = 1; w < kThreads / 64; ++w) x += part[w];
  return x;
}

// |x|^2. An FP32 field is squared in FP32, operation by operation: the energy is
// the FP64 sum of the FP32 density sum V rho, whatever computes the density.
__device__ __forceinline__ double density(Cx<double> x) { return x.re * x.re + x.im * x.im; }
__device__ __forceinline__ double density(Cx<float> x) {
#pragma clang fp contract(off)
  const float re = x.re * x.re, im = x.im * x.im;
  return static_cast<double>(re + im);
}

// partial[band][block] = the block's share of sum_r V |psi|^2, in FP64.
template <typename T>
__global__ void __launch_bounds__(kThreads)
    k_field_energy(const Cx<T>* psi, const T* v, long long points, double* partial) {
  const Cx<T>* f = psi + blockIdx.y * points;
  double acc = 0.0;
  constexpr int U = 4;
  const long long step = static_cast<long long>(gridDim.x) * kThreads;
  for (long long r = static_cast<long long>(blockIdx.x) * kThreads + threadIdx.x; r < points;
       r += U * step) {
    Cx<T> x[U];
    T w[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const long long i = r + u * step;
      const bool in = i < points;
      x[u] = f[in ? i : r];
      w[u] = v[in ? i : r];
      if (!in) x[u] = Cx<T>{T(0), T(0)}, w[u] = T(0);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      acc += static_cast<double>(w[u]) * density(x[u]);
    }
  }
  acc = block_sum(acc);
  if (threadIdx.x == 0) partial[blockIdx.y * gridDim.x + blockIdx.x] = acc;
}

__global__ void __launch_bounds__(kThreads)
    k_energy_sum(const double* partial, int count, double* energy) {
  double acc = 0.0;
  for (int i = threadIdx.x; i < count; i += kThreads) acc += partial[i];
  acc = block_sum(acc);
  if (threadIdx.x == 0) *energy = acc;
}

// out = (2 V g) psi, g a device scalar (null: 1); out may be psi.
template <typename T>
__global__ void __launch_bounds__(kThreads)
    k_energy_field(const Cx<T>* psi, const T* v, const double* g, long long points, Cx<T>* out) {
  const long long base = blockIdx.y * points;
  const T scale = g ? static_cast<T>(*g) : T(1);
  constexpr int U = 2;
  const long long r0 = static_cast<long long>(blockIdx.x) * U * kThreads + threadIdx.x;
  Cx<T> x[U];
  T w[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const long long i = min(r0 + u * kThreads, points - 1);
    x[u] = psi[base + i];
    w[u] = T(2) * v[i] * scale;
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const long long i = r0 + u * kThreads;
    if (i < points) out[base + i] = Cx<T>{w[u] * x[u].re, w[u] * x[u].im};
  }
}

template <typename T>
void field_energy(const void* psi, const void* v, long long points, int bands, double* partial,
                  double* energy, hipStream_t stream) {
  hipLaunchKernelGGL(k_field_energy<T>, dim3(kEnergyBlocks, bands), dim3(kThreads), 0, stream,
                     static_cast<const Cx<T>*>(psi), static_cast<const T*>(v), points, partial);
  check_launch();
  hipLaunchKernelGGL(k_energy_sum, dim3(1), dim3(kThreads), 0, stream, partial,
                     kEnergyBlocks * bands, energy);
  check_launch();
}

template <typename T>
void energy_field(const void* psi, const void* v, const double* g, long long points, int bands,
                  void* out, hipStream_t stream) {
  const long long blocks = (points + 2 * kThreads - 1) / (2 * kThreads);
  hipLaunchKernelGGL(k_energy_field<T>, dim3(static_cast<unsigned>(blocks), bands),
                     dim3(kThreads), 0, stream, static_cast<const Cx<T>*>(psi),
                     static_cast<const T*>(v), g, points, static_cast<Cx<T>*>(out));
  check_launch();
}

template <typename F>
int guarded(F&& f) {
  try {
    f();
    return 0;
  } catch (const GenericError& e) {
    return static_cast<int>(e.error_code());
  } catch (...) {
    return static_cast<int>(SPFFT_UNKNOWN_ERROR);
  }
}

}  // namespace
}  // namespace spfft

// Hooks of spfft_amd/autograd.py (no counterpart in the reference ABI): device
// pointers of checked tensors on `device`, `stream` the caller's there. valueBytes: 8 or 4 per real
// value. `partial` holds spfft_amd_energy_partials(bands) doubles.
extern "C" __attribute__((visibility("default"))) int spfft_amd_energy_partials(int bands) {
  return spfft::kEnergyBlocks * bands;
}
extern "C" __attribute__((visibility("default"))) int spfft_amd_field_energy(
    int device, int valueBytes, const void* psi, const void* potential, long long points,
    int bands, double* partial, double* energy, void* stream) {
  using namespace spfft;
  const auto s = static_cast<hipStream_t>(stream);
  return guarded([&] {
    if (points < 1 || bands < 1 || bands > 65535) throw InvalidParameterError();
    DeviceGuard guard(device);
    if (valueBytes == 8) {
      field_energy<double>(psi, potential, points, bands, partial, energy, s);
    } else {
      field_energy<float>(psi, potential, points, bands, partial, energy, s);
    }
  });
}
extern "C" __attribute__((visibility("default"))) int spfft_amd_energy_field(
    int device, int valueBytes, const void* psi, const void* potential, const double* grad,
    long long points, int bands, void* out, void* stream) {
  using namespace spfft;
  const auto s = static_cast<hipStream_t>(stream);
  return guarded([&] {
    if (points < 1 || bands < 1 || bands > 65535) throw InvalidParameterError();
    DeviceGuard guard(device);
    if (valueBytes == 8) {
      energy_field<double>(psi, potential, grad, points, bands, out, s);
    } else {
      energy_field<float>(psi, potential, grad, points, bands, out, s);
    }
  });
}
