// tile2d_batch.hip -- the tile launches of tile2d.hip over the members of a
// batch: one work-group per tile of one member.
//
// A batched single step moves 72 bytes a node (FP32) and one force launch
// follows each; 448-node-wide wakes stepped at 61 G node-steps/s with both.
// Four steps per launch move 25 bytes a node-step and need one force launch,
// most of whose samples the tiles have already formed.
#include "batch.hpp"
#include "tile2d.hpp"

namespace wake_hip {

namespace {
constexpr int kW = 32, kH = 32;
}

// The steps i .. i + nsteps - 1 of the chunk, launch `flip` of it (each
// launch a member takes part in swaps its buffers once).
template <class St, int COLL, bool LES, bool THERMAL, bool FORCE, int T>
__global__ __launch_bounds__(kW * kH) __attribute__((amdgpu_waves_per_eu(THERMAL ? 4 : 8))) void k_tile2d_batch(
    const BatchSlot* __restrict__ slots, const int* __restrict__ tile_slot, int i, int flip, int nsteps) {
  using P = typename St::T;
  __shared__ Tile2dShared<St, THERMAL, kW, kH> sh;
  const int t = blockIdx.x;
  const BatchSlot& sl = slots[__builtin_amdgcn_readfirstlane(tile_slot[t])];
  const unsigned long long cur = sl.step + static_cast<unsigned long long>(i);
  if (cur >= sl.stop_at) return;  // uniform over the work-group
  const unsigned long long left = sl.stop_at - cur;
  const int ns = left < static_cast<unsigned long long>(nsteps) ? static_cast<int>(left) : nsteps;
  const int local = t - sl.ttile0;
  const int ty = local / sl.ttiles_x, tx = local - ty * sl.ttiles_x;
  const int par = (sl.parity + flip) & 1;
  tile2d_steps<St, COLL, LES, THERMAL, FORCE, true, T, kW, kH>(
      sh, (TileArgs*)(&sl.a), static_cast<const P*>(sl.buf[par]), static_cast<P*>(sl.buf[par ^ 1]), sl.gbuf[par],
      sl.gbuf[par ^ 1], tx * (kW - 2 * T), ty * (kH - 2 * T), ns, cur == sl.s_at, cur, sl.tile_forces);
}

// Forces on S after the steps i .. i + nsteps - 1 of the chunk, one
// work-group per member and step: all but the last from the sums the tiles
// left, the last formed from the buffer they wrote, in k_mem_batch's order.
template <class St>
__global__ __launch_bounds__(256) void k_mem_tiles(const BatchSlot* __restrict__ slots, int i, int flip, int nsteps,
                                                   int chunk, double* __restrict__ hist) {
  using L = D2Q9;
  const BatchSlot& sl = slots[blockIdx.x];
  const int j = blockIdx.y;
  const unsigned long long cur = sl.step + static_cast<unsigned long long>(i);
  if (!sl.mem_on || cur + j >= sl.stop_at) return;
  const unsigned long long k = cur + j + 1;  // the sample of S_k
  const bool formed = j + 1 < nsteps && k < sl.stop_at;
  const StepArgs& a = sl.a;
  const auto* buf = static_cast<const typename St::T*>(sl.buf[((sl.parity + flip) & 1) ^ 1]);
  const TileForces& tf = sl.tile_forces;
  double s0 = 0.0, s1 = 0.0, s2 = 0.0;
  for (int m = threadIdx.x; m < sl.mem_count; m += blockDim.x) {
    if (formed) {
      const double* p = tf.out + 3 * (static_cast<long long>(k % tf.ring) * tf.count + m);
      s0 += p[0];
      s1 += p[1];
      s2 += p[2];
    } else {
      const int n = sl.mem_nodes[m];
      const int x = n % a.nx, y = n / a.nx;
      float f[L::Q];
      form_s_at<L, St, false>(a, buf, x, y, 0, n, a.cls[n], false, k, f);
      mem_node<L>(a, x, y, 0, n, f, a.mem_c[0], a.mem_c[1], a.mem_c[2], a.mem_rmax, s0, s1, s2);
    }
  }
  block_sum3(s0, s1, s2);
  if (threadIdx.x == 0) {
    double* o = hist + (static_cast<long long>(blockIdx.x) * chunk + i + j) * 3;
    o[0] = s0;
    o[1] = s1;
    o[2] = s2;
  }
}

namespace {

template <class St, bool THERMAL>
hipError_t go(int collision, bool les, bool force, int span, const BatchSlot* slots, const int* tile_slot, int ntiles,
              int i, int flip, int nsteps, hipStream_t s) {
  auto run = [&](auto coll, auto les_c, auto force_c, auto span_c) {
    k_tile2d_batch<St, decltype(coll)::value, decltype(les_c)::value, THERMAL, decltype(force_c)::value,
                   decltype(span_c)::value><<<ntiles, kW * kH, 0, s>>>(slots, tile_slot, i, flip, nsteps);
    return hipGetLastError();
  };
  auto spanned = [&](auto coll, auto les_c, auto force_c) {
    if (span == kTbSteps) return run(coll, les_c, force_c, std::integral_constant<int, kTbSteps>{});
    return run(coll, les_c, force_c, std::integral_constant<int, kTbFewSteps>{});
  };
  auto forced = [&](auto coll, auto les_c) {
    if constexpr (!THERMAL) {
      if (!force) return spanned(coll, les_c, std::false_type{});
    }
    return spanned(coll, les_c, std::true_type{});
  };
  auto with = [&](auto coll) {
    if constexpr (!THERMAL) {
      if (les) return forced(coll, std::true_type{});
    }
    return forced(coll, std::false_type{});
  };
  if (collision == kBGK) return with(std::integral_constant<int, kBGK>{});
  if (collision == kTRT) return with(std::integral_constant<int, kTRT>{});
  return with(std::integral_constant<int, kMRT>{});
}

}  // namespace

void tile2d_grid(int nx, int ny, int span, int* tiles_x, int* tiles) {
  const int w = kW - 2 * span, h = kH - 2 * span;
  *tiles_x = (nx + w - 1) / w;
  *tiles = *tiles_x * ((ny + h - 1) / h);
}

hipError_t launch_tile2d_batch(int storage, int collision, bool les, bool thermal, bool force, int span,
                               const BatchSlot* slots, const int* tile_slot, int ntiles, int i, int flip, int nsteps,
                               hipStream_t s) {
  if (ntiles <= 0) return hipSuccess;
  if ((span != kTbSteps && span != kTbFewSteps) || nsteps < 1 || nsteps > span) return hipErrorInvalidValue;
  auto with = [&](auto st) {
    using St = decltype(st);
    if (thermal) {
      if constexpr (std::is_same_v<St, StBF16>) return hipErrorInvalidValue;
      else return go<St, true>(collision, false, true, span, slots, tile_slot, ntiles, i, flip, nsteps, s);
    }
    return go<St, false>(collision, les, force, span, slots, tile_slot, ntiles, i, flip, nsteps, s);
  };
  switch (storage) {
    case kStoreF32: return with(StF32{});
    case kStoreF16: return with(StF16{});
    case kStoreBF16: return with(StBF16{});
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_mem_tiles(int storage, const BatchSlot* slots, int nslots, int i, int flip, int nsteps, int chunk,
                            double* hist, hipStream_t s) {
  if (nslots <= 0 || nsteps <= 0) return hipSuccess;
  const dim3 g(nslots, nsteps);
  switch (storage) {
    case kStoreF32: k_mem_tiles<StF32><<<g, 256, 0, s>>>(slots, i, flip, nsteps, chunk, hist); break;
    case kStoreF16: k_mem_tiles<StF16><<<g, 256, 0, s>>>(slots, i, flip, nsteps, chunk, hist); break;
    case kStoreBF16: k_mem_tiles<StBF16><<<g, 256, 0, s>>>(slots, i, flip, nsteps, chunk, hist); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace wake_hip
