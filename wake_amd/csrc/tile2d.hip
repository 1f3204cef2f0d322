// tile2d.hip -- launches of several D2Q9 steps from LDS tiles (gfx950).
#include "tile2d.hpp"

namespace wake_hip {

// Bound by VALU issue: a D2Q9 node costs 100 (BGK) to 190 (TRT) VALU
// instructions a step.  Eight waves a SIMD (two 32 x 32 tiles a compute unit)
// cap the scalar registers at 80: left alone the kernel takes 106, which
// fits seven waves, so one tile -- the MRT + LES channel of 1500 x 403 nodes
// then takes 10.7 us a step instead of 8.3.  (Figures without forces.)
// At 1536 x 1024 nodes FP32: 146 G node-steps/s plain BGK, 90 G for the
// channel (single-step launches: 78 G and 76 G); TRT channel of 240 x 80:
// 1.8 us a step, where a single-step launch takes 4.6.
template <class St, int COLL, bool LES, bool THERMAL, bool FORCE, bool EDGES, int T, int W, int H>
__global__ __launch_bounds__(W * H) __attribute__((amdgpu_waves_per_eu(!THERMAL && H == 32 ? 8 : 4))) void k_tile2d(const StepArgs a, const typename St::T* __restrict__ ain,
                                                  typename St::T* __restrict__ aout, const float* __restrict__ gin,
                                                  float* __restrict__ gout, int nsteps, bool from_s,
                                                  const TileForces mf) {
  static_assert(T <= kTbSteps, "ring and launch bookkeeping");
  __shared__ Tile2dShared<St, THERMAL, W, H> sh;
  // the arguments are the first bytes of the kernel's argument segment
  TileArgs* ap = (TileArgs*)(__builtin_amdgcn_kernarg_segment_ptr());
  tile2d_steps<St, COLL, LES, THERMAL, FORCE, EDGES, T, W, H>(
      sh, ap, ain, aout, gin, gout, static_cast<int>(blockIdx.x) * (W - 2 * T),
      static_cast<int>(blockIdx.y) * (H - 2 * T), nsteps, from_s, ap->s_step, mf);
}

// The per-wave partials of the force samples of steps first .. first +
// gridDim.y - 1 from the nodes' sums: one wave per slot adds its row
// segment's nodes in the butterfly order of a single-step launch, so the
// partials have that launch's bits.
__global__ __launch_bounds__(256) void k_mem_slots(const TileForces mf, const int* __restrict__ row_list,
                                                   int waves_per_row, int nslots, int nx, long long first,
                                                   double* __restrict__ ring) {
  const int slot = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (slot >= nslots) return;
  const long long at = (first + blockIdx.y) % mf.ring;
  const int row = row_list[slot / waves_per_row];
  const int x = 64 * (slot % waves_per_row) + __lane_id();
  const int k = x < nx ? mf.index[row * nx + x] : -1;
  double s0 = 0.0, s1 = 0.0, s2 = 0.0;
  if (__any(k >= 0)) {
    if (k >= 0) {
      const double* p = mf.out + 3 * (at * mf.count + k);
      s0 = p[0];
      s1 = p[1];
      s2 = p[2];
    }
    s0 = wave_sum(s0);
    s1 = wave_sum(s1);
    s2 = wave_sum(s2);
  }
  if (__lane_id() == 0) {
    double* o = ring + 3 * (at * nslots + slot);
    o[0] = s0;
    o[1] = s1;
    o[2] = s2;
  }
}

// The open-boundary closures of step a.s_step at the solid nodes of the inlet
// and outlet rows, in place in the populations that step left (form_s_at
// applies them there each step).  Each forms three populations from six that
// it leaves alone, so the last step's are all that is to be seen of them, and
// closing again changes nothing.
template <class St>
__global__ __launch_bounds__(64) void k_close_solid(const StepArgs a, typename St::T* __restrict__ buf) {
  using L = D2Q9;
  const int y = blockIdx.x * 64 + threadIdx.x, x = blockIdx.y == 0 ? 0 : a.nx - 1;
  if (y >= a.ny) return;
  const int n = y * a.nx + x;
  const uint8_t c = a.cls[n];
  if (!(c & kClsFrozen)) return;
  float f[L::Q];
  static_for<L::Q>([&](auto qc) {
    constexpr int q = decltype(qc)::value;
    f[q] = tb_get<St, L, q>(buf[q * a.stride + n]);
  });
  if (c & kClsInlet) apply_inlet<L>(a, f, y, n, a.s_step);
  if ((c & kClsOutlet) && a.outflow == 1) apply_zh_outflow_d2q9(a, f);
  static_for<L::Q>([&](auto qc) {
    constexpr int q = decltype(qc)::value;
    buf[q * a.stride + n] = tb_put<St, L, q>(f[q]);
  });
}

__global__ __launch_bounds__(256) void k_index_nodes(const int* __restrict__ nodes, int count,
                                                     int* __restrict__ index) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < count) index[nodes[i]] = i;
}

namespace {

// Tiles of W x H nodes with a halo of T own (W - 2 T) x (H - 2 T).
constexpr int kTileW = 32, kTileH = 32, kTileLowH = 24;

template <int T, int W, int H>
dim3 tiles_of(int nx, int ny) {
  constexpr int wx = W - 2 * T, wy = H - 2 * T;
  return dim3((nx + wx - 1) / wx, (ny + wy - 1) / wy);
}

int compute_units() {
  static const int cus = [] {
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
      n = 0;
    return n;
  }();
  return cus;
}

// The low tile owns half the nodes for 3/4 of the waves: worth it while there
// is a compute unit for each tile (240 x 80 nodes, TRT channel without
// forces: 1.69 us a step against 2.07), not beyond (256 x 256: 2.47 against 2.23).
bool low_tiles(const StepArgs& a) {
  const dim3 g = tiles_of<kTbSteps, kTileW, kTileLowH>(a.nx, a.ny);
  return static_cast<long long>(g.x) * g.y <= compute_units();
}

template <class St, int COLL, bool LES, bool THERMAL>
hipError_t go(const StepArgs& a, const void* in, void* out, const float* gin, float* gout, int nsteps, bool from_s,
              bool edges, const TileForces& mf, hipStream_t s) {
  using T_ = typename St::T;
  auto run = [&](auto force, auto edge, auto tc, auto hc) {
    constexpr int T = decltype(tc)::value, H = decltype(hc)::value;
    k_tile2d<St, COLL, LES, THERMAL, decltype(force)::value, decltype(edge)::value, T, kTileW, H>
        <<<tiles_of<T, kTileW, H>(a.nx, a.ny), kTileW * H, 0, s>>>(a, static_cast<const T_*>(in),
                                                                   static_cast<T_*>(out), gin, gout, nsteps, from_s,
                                                                   mf);
    return hipGetLastError();
  };
  using Many = std::integral_constant<int, kTbSteps>;
  using Few = std::integral_constant<int, kTbFewSteps>;
  using High = std::integral_constant<int, kTileH>;
  using Low = std::integral_constant<int, kTileLowH>;
  auto sized = [&](auto force, auto edge) {
    constexpr bool one_per_unit = THERMAL && sizeof(T_) == 4;
    if (nsteps <= kTbFewSteps && tile2d_steps_of(a.nx, a.ny, one_per_unit) == kTbFewSteps)
      return run(force, edge, Few{}, High{});
    if (low_tiles(a)) return run(force, edge, Many{}, Low{});
    return run(force, edge, Many{}, High{});
  };
  auto edged = [&](auto force) {
    if constexpr (!THERMAL) {
      if (!edges) return sized(force, std::false_type{});
    }
    return sized(force, std::true_type{});
  };
  if constexpr (!THERMAL) {
    if (a.gx == 0.0f && a.gy == 0.0f) return edged(std::false_type{});
  }
  return edged(std::true_type{});
}

template <class St, bool THERMAL>
hipError_t go_collision(int collision, bool les, const StepArgs& a, const void* in, void* out, const float* gin,
                        float* gout, int nsteps, bool from_s, bool edges, const TileForces& mf, hipStream_t s) {
  auto with = [&](auto coll) {
    constexpr int C = decltype(coll)::value;
    if constexpr (!THERMAL) {
      if (les) return go<St, C, true, false>(a, in, out, gin, gout, nsteps, from_s, edges, mf, s);
    }
    return go<St, C, false, THERMAL>(a, in, out, gin, gout, nsteps, from_s, edges, mf, s);
  };
  if (collision == kBGK) return with(std::integral_constant<int, kBGK>{});
  if (collision == kTRT) return with(std::integral_constant<int, kTRT>{});
  return with(std::integral_constant<int, kMRT>{});
}

}  // namespace

// The halo is computed again by each neighbour: in issue slots (rows of a
// wave) 8 steps from a 32 x 32 tile cost 2.9 times their own nodes, 4 steps
// 1.5 times, which counts once there are more tiles than the chip holds at a
// time: two a compute unit, one with FP32 temperature (115 KB of LDS).
// Measured, us a step for 8 / 4 steps a launch: MRT + LES channel FP32
// 512 x 256 nodes (512 tiles of 8 steps) 3.60 / 3.85, 768 x 384 (1152)
// 6.70 / 5.27; temperature FP32 256 x 256 (256 tiles) 2.87 / 4.19, 512 x 256
// 5.31 / 4.43.
int tile2d_steps_for(long long tiles_of_most, bool one_per_unit) {
  return tiles_of_most <= (one_per_unit ? 1ll : 2ll) * compute_units() ? kTbSteps : kTbFewSteps;
}
int tile2d_steps_of(int nx, int ny, bool one_per_unit) {
  const dim3 g = tiles_of<kTbSteps, kTileW, kTileH>(nx, ny);
  return tile2d_steps_for(static_cast<long long>(g.x) * g.y, one_per_unit);
}

hipError_t launch_tile2d(int storage, int collision, bool les, bool thermal, bool from_s, bool edges, int nsteps,
                         const StepArgs& a, const void* in, void* out, const float* gin, float* gout,
                         const TileForces& mf, hipStream_t s) {
  if (nsteps < 1 || nsteps > kTbSteps || a.nz != 1) return hipErrorInvalidValue;
  auto with = [&](auto st) {
    using St = decltype(st);
    if (thermal) {
      if constexpr (std::is_same_v<St, StBF16>) return hipErrorInvalidValue;
      else return go_collision<St, true>(collision, false, a, in, out, gin, gout, nsteps, from_s, true, mf, s);
    }
    return go_collision<St, false>(collision, les, a, in, out, gin, gout, nsteps, from_s, edges, mf, s);
  };
  switch (storage) {
    case kStoreF32: return with(StF32{});
    case kStoreF16: return with(StF16{});
    case kStoreBF16: return with(StBF16{});
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_mem_slots(const TileForces& mf, const int* row_list, int nrows, int nx, long long first, int count,
                            double* ring, hipStream_t s) {
  const int waves = mem_waves_per_row(nx), nslots = nrows * waves;
  if (nslots <= 0 || count <= 0) return hipSuccess;
  k_mem_slots<<<dim3((nslots + 3) / 4, count), 256, 0, s>>>(mf, row_list, waves, nslots, nx, first, ring);
  return hipGetLastError();
}

hipError_t launch_close_solid(int storage, const StepArgs& a, void* buf, hipStream_t s) {
  auto with = [&](auto st) {
    using St = decltype(st);
    k_close_solid<St><<<dim3((a.ny + 63) / 64, 2), 64, 0, s>>>(a, static_cast<typename St::T*>(buf));
    return hipGetLastError();
  };
  switch (storage) {
    case kStoreF32: return with(StF32{});
    case kStoreF16: return with(StF16{});
    case kStoreBF16: return with(StBF16{});
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_index_nodes(const int* nodes, int count, int* index, hipStream_t s) {
  if (count <= 0) return hipSuccess;
  k_index_nodes<<<(count + 255) / 256, 256, 0, s>>>(nodes, count, index);
  return hipGetLastError();
}

}  // namespace wake_hip
