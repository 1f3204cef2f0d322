// state_init.hip -- populations of a state set from fields or planes, formed
// on the device (lattice_grid_3d.cpp:95-131 per node).
//
// Compiled without fused multiply-adds and with IEEE square roots: the
// equilibria must be the host expressions' values bit for bit (the reference
// forms them on the host, in FP32, product by product).  Bound by the bytes
// of the planes written; on the host the same loop took 45 ms for 96 x 80 x
// 64 D3Q19 nodes, here it is 4 field uploads and one 20 us launch.
#include <hip/hip_runtime.h>

#include "engine.hpp"
#include "lattice.hpp"
#include "node_ops.hpp"

namespace wake_hip {

namespace {

// FP32 population -> storage format (16-bit: the deviation from the weight,
// rounded to nearest even).
template <int STORAGE>
__device__ __forceinline__ void put(void* buf, long long i, float f, float w) {
  if constexpr (STORAGE == kStoreF32) {
    static_cast<float*>(buf)[i] = f;
  } else if constexpr (STORAGE == kStoreF16) {
    static_cast<_Float16*>(buf)[i] = static_cast<_Float16>(f - w);
  } else {
    const uint32_t b = __float_as_uint(f - w);
    static_cast<uint16_t*>(buf)[i] = static_cast<uint16_t>((b + 0x7FFFu + ((b >> 16) & 1u)) >> 16);
  }
}

// Convective outlet record of node n where it lies on x = nx - 1: the FP32
// value of population q (padding entries zero).
template <class L>
__device__ __forceinline__ void put_prev(float* prev, int nx, int n, int q, float f) {
  if ((n + 1) % nx != 0) return;
  float* rec = prev + static_cast<long long>(n / nx) * prev_stride(L::Q);
  rec[q] = f;
  if (q == L::Q - 1)
    for (int k = L::Q; k < prev_stride(L::Q); ++k) rec[k] = 0.0f;
}

template <class L, int STORAGE>
__global__ __launch_bounds__(256) void k_init_fields(const float* __restrict__ rho, const float* __restrict__ ux,
                                                     const float* __restrict__ uy, const float* __restrict__ uz,
                                                     float* __restrict__ speed, void* __restrict__ buf,
                                                     long long stride, float* __restrict__ prev, int nx, int N) {
  const int n = blockIdx.x * 256 + threadIdx.x;
  if (n >= N) return;
  const float r = rho[n], a = ux[n], b = uy[n], c = L::D == 2 ? 0.0f : uz[n];
  const float u_sq = L::D == 2 ? a * a + b * b : a * a + b * b + c * c;
  speed[n] = sqrtf(u_sq);
  static_for<L::Q>([&](auto qc) {
    constexpr int q = decltype(qc)::value;
    float cu = static_cast<float>(L::cx[q]) * a + static_cast<float>(L::cy[q]) * b;
    if constexpr (L::D == 3) cu = cu + static_cast<float>(L::cz[q]) * c;
    const float f = L::w[q] * r * (1.0f + 3.0f * cu + 4.5f * cu * cu - 1.5f * u_sq);
    put<STORAGE>(buf, q * stride + n, f, L::w[q]);
    put_prev<L>(prev, nx, n, q, f);
  });
}

// splitmix64 finaliser (the host's add_noise counter hash).
__device__ __forceinline__ unsigned long long mix64(unsigned long long x) {
  x += 0x9E3779B97F4A7C15ull;
  x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
  x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
  return x ^ (x >> 31);
}

struct Planes {
  const float* p[D3Q27::Q];
};

// FP32 planes of the populations q0 .. q1 - 1 plus seeded noise (amplitude 0:
// none, the planes as they are) -> the state.
template <class L, int STORAGE>
__global__ __launch_bounds__(256) void k_init_planes(const Planes planes, int q0, int q1, float amplitude,
                                                     unsigned long long seed, void* __restrict__ buf,
                                                     long long stride, float* __restrict__ prev, int nx, int N) {
  const int n = blockIdx.x * 256 + threadIdx.x;
  if (n >= N) return;
  static_for<L::Q>([&](auto qc) {
    constexpr int q = decltype(qc)::value;
    if (q < q0 || q >= q1) return;
    float f = planes.p[q][n];
    if (amplitude != 0.0f) {
      const unsigned long long h = mix64(seed ^ (static_cast<unsigned long long>(n) * L::Q + q));
      const double u = static_cast<double>(h >> 40) * (1.0 / 16777216.0);
      f += amplitude * static_cast<float>(2.0 * u - 1.0);
    }
    put<STORAGE>(buf, q * stride + n, f, L::w[q]);
    put_prev<L>(prev, nx, n, q, f);
  });
}

// (a domain may hold up to 2^31 - 1 nodes)
constexpr unsigned blocks_of(int nodes) { return (static_cast<unsigned>(nodes) + 255u) / 256u; }
static_assert(blocks_of(0x7fffffff) == 1u << 23 && blocks_of(0x7fffff01) == 1u << 23 &&
              blocks_of(0x7fffff00) == (1u << 23) - 1 && blocks_of(257) == 2 && blocks_of(1) == 1);

template <class F>
hipError_t with_kind(int lattice, int storage, F&& f) {
  auto with = [&](auto lat) {
    if (storage == kStoreF32) return f(lat, std::integral_constant<int, kStoreF32>{});
    if (storage == kStoreF16) return f(lat, std::integral_constant<int, kStoreF16>{});
    if (storage == kStoreBF16) return f(lat, std::integral_constant<int, kStoreBF16>{});
    return hipErrorInvalidValue;
  };
  if (lattice == 9) return with(D2Q9{});
  if (lattice == 19) return with(D3Q19{});
  if (lattice == 27) return with(D3Q27{});
  return hipErrorInvalidValue;
}

}  // namespace

hipError_t launch_init_fields(int lattice, int storage, const float* rho, const float* ux, const float* uy,
                              const float* uz, float* speed, void* buf, long long stride, float* prev, int nx, int N,
                              hipStream_t s) {
  return with_kind(lattice, storage, [&](auto lat, auto st) {
    k_init_fields<decltype(lat), decltype(st)::value>
        <<<blocks_of(N), 256, 0, s>>>(rho, ux, uy, uz, speed, buf, stride, prev, nx, N);
    return hipGetLastError();
  });
}

hipError_t launch_init_planes(int lattice, int storage, const float* const* planes, int q0, int count,
                              float amplitude, unsigned long long seed, void* buf, long long stride, float* prev,
                              int nx, int N, hipStream_t s) {
  if (q0 < 0 || count < 0 || q0 + count > lattice) return hipErrorInvalidValue;
  return with_kind(lattice, storage, [&](auto lat, auto st) {
    Planes p{};
    for (int k = 0; k < count; ++k) p.p[q0 + k] = planes[k];
    k_init_planes<decltype(lat), decltype(st)::value>
        <<<blocks_of(N), 256, 0, s>>>(p, q0, q0 + count, amplitude, seed, buf, stride, prev, nx, N);
    return hipGetLastError();
  });
}

}  // namespace wake_hip
