// tile2d.hpp -- several D2Q9 steps per launch from an LDS tile (device code).
//
// A 2D single-step launch is bound by latency up to some hundred thousand
// nodes (a 240 x 80 TRT channel takes 4.6 us a step, 6.7 with its forces:
// class byte, bounce mask, own-node populations, one memory round trip after
// another, for 0.3 us of bytes) and by its 72 bytes a node beyond.  Tiles take
// 1.8 us, 2.5 with the forces.  Here each work-group loads a W x H tile of
// A_{k-1} around its (W - 2 T) x (H - 2 T) nodes into LDS, pull-collides up to
// T times there -- the valid region shrinks by one node per step -- and stores
// A of its own nodes; the launch, the class data and the populations' way
// through memory are paid once per T steps, and walls, obstacles and open
// boundaries read their neighbours from LDS.
//
// One thread per tile node; the two population tiles alternate, so a step
// needs one barrier.  Every node update is the pull, boundary closure,
// collision and storage rounding of the single-step kernel, so the result
// has the same bits as that many single steps.  x always wraps; a tile row
// outside a non-periodic y range holds wrapped values that no node inside
// the range keeps (its bounce mask replaces them), as in the single-step
// pull.  Solid nodes in the inlet and outlet rows are not closed here: no node
// reads them, and k_close_solid does it before they are read out (tested for
// in the step loop, they cost a batch of 512 wakes 1.2 %).  Not for curved
// links or the convective outlet (its upstream neighbour reaches two nodes
// per step, past the halo): those domains take single steps.
#pragma once

#include "thermal_impl.hpp"

namespace wake_hip {

template <class St, class L, int q>
__device__ __forceinline__ float tb_get(typename St::T v) {
  if constexpr (sizeof(typename St::T) == 4) {
    return v;
  } else {
    return St::template from_dev_bits<L, q>(__builtin_bit_cast(unsigned short, v));
  }
}
template <class St, class L, int q>
__device__ __forceinline__ typename St::T tb_put(float v) {
  if constexpr (sizeof(typename St::T) == 4) {
    return v;
  } else {
    return __builtin_bit_cast(typename St::T, St::template dev_bits<L, q>(v));
  }
}

// LDS of one tile: two population tiles and, with a temperature, two of its own.
template <class St, bool THERMAL, int W, int H>
struct Tile2dShared {
  typename St::T f[2][D2Q9::Q][W * H];
  float g[2][THERMAL ? D2Q5::Q : 1][THERMAL ? W * H : 1];
};

// The arguments in the constant address space (a kernel's own, or a batch's
// slot table, which no kernel of a step writes): what only boundary nodes
// need is loaded where they need it, through a pointer the compiler cannot
// follow, instead of being held in scalar registers over all steps (held,
// some forty of them spill to VGPR lanes that every node reads back).
using TileArgs = const __attribute__((address_space(4))) StepArgs;
__device__ __forceinline__ TileArgs* opaque_args(TileArgs* p) {
  asm volatile("" : "+s"(p));
  return p;
}

// The same value, as one the compiler knows nothing of.
__device__ __forceinline__ void opaque(float& v) { asm volatile("" : "+v"(v)); }

// Steps s_step + 1 .. s_step + nsteps (nsteps <= T, the tile's halo) of the
// tile whose own nodes start at (ox, oy).  from_s: `ain` holds a materialised S, the
// first step only collides.  mf: where the own nodes' force sums go
// (mf.index null: none); the sample of S_k formed by a step's pull is written
// at ring position k.  FORCE: the body force is not zero.  EDGES: some node
// has a class bit or force sums are taken (false: a plain periodic domain).
template <class St, int COLL, bool LES, bool THERMAL, bool FORCE, bool EDGES, int T, int W, int H>
__device__ __forceinline__ void tile2d_steps(Tile2dShared<St, THERMAL, W, H>& sh, TileArgs* ap,
                                             const typename St::T* __restrict__ ain,
                                             typename St::T* __restrict__ aout, const float* __restrict__ gin,
                                             float* __restrict__ gout, int ox, int oy, int nsteps, bool from_s,
                                             unsigned long long s_step, const TileForces& mf) {
  using L = D2Q9;
  const int nx = ap->nx, ny = ap->ny;
  const long long S = ap->stride;
  const int cell = threadIdx.x;  // this thread's tile node
  const int i = cell % W, j = cell / W;
  // node of the domain (the tile may wrap more than once around a small one)
  int x = (ox - T + i) % nx, y = (oy - T + j) % ny;
  if (x < 0) x += nx;
  if (y < 0) y += ny;
  const int n = y * nx + x;
  // Everything the steps need of this node, in one round trip.
  static_for<L::Q>([&](auto qc) {
    constexpr int q = decltype(qc)::value;
    sh.f[0][q][cell] = ain[q * S + n];
  });
  if constexpr (THERMAL) {
    static_for<D2Q5::Q>([&](auto qc) {
      constexpr int q = decltype(qc)::value;
      sh.g[0][q][cell] = gin[q * S + n];
    });
  }
  const uint8_t c = EDGES ? ap->cls[n] : static_cast<uint8_t>(0);
  uint32_t bm = EDGES ? ap->bmask[n] : 0u;
  const int li = i - T, lj = j - T;
  const bool own = li >= 0 && li < W - 2 * T && lj >= 0 && lj < H - 2 * T && ox + li < nx && oy + lj < ny;
  int force_at = -1;
  if constexpr (EDGES && !THERMAL) {
    if (mf.index && own) force_at = mf.index[n];
  }
  if (!(c & kClsSlow)) bm = 0;
  uint32_t moving = 0;  // directions whose pull source is a moving wall
  float t_wall[D2Q5::Q] = {};
  uint32_t g_wall = 0;  // temperature directions whose pull source reflects
  auto source = [&](int cx, int cy, bool& in) {
    const int sx = wrap(x - cx, nx);
    int sy = y - cy;
    in = true;
    if (ap->per_y) sy = wrap(sy, ny);
    else in = sy >= 0 && sy < ny;
    return in ? sy * nx + sx : n;
  };
  if (bm & kBounceMovingWall) moving = ap->mmask[n];
  if constexpr (THERMAL) {
    if (c & kClsSlow) {
      static_for<D2Q5::Q>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        if constexpr (q > 0) {
          bool in;
          const int sn = source(D2Q5::cx[q], D2Q5::cy[q], in);
          const uint8_t t = (in && !ap->periodic_mode) ? ap->flags[sn] : static_cast<uint8_t>(kFluid);
          t_wall[q] = in ? ap->t_wall[sn] : __builtin_nanf("");
          if (!in || t == kSolid || t == kMovingWall) g_wall |= 1u << q;
        }
      });
    }
  }
  // What the collisions read, kept over the steps.
  StepArgs b;
  b.tau = ap->tau;
  b.cs = ap->cs;
  b.gx = ap->gx;
  b.gy = ap->gy;
  b.nonfinite = ap->nonfinite;
  if constexpr (THERMAL) {
    b.gbeta = ap->gbeta;
    b.t_ref = ap->t_ref;
    b.tau_g = ap->tau_g;
  }
  // The rates 1 / tau: once per launch with FP32 storage, where each is an
  // IEEE division; per step with 16-bit storage (formed outside the node
  // update they make the compiler fuse the TRT force terms differently from
  // the single step's).
  constexpr bool kHoist = !LES && sizeof(typename St::T) == 4;
  constexpr bool kFast = St::kFast && !THERMAL;
  float rate_s = 0.0f, rate_a = 0.0f, rate_g = 0.0f;
  auto rates = [&]() {
    if constexpr (!LES) {
      rate_s = recip<kFast>(b.tau);
      if constexpr (COLL == kTRT) rate_a = recip<kFast>(trt_tau_a(b.tau));
    }
    if constexpr (THERMAL) rate_g = 1.0f / b.tau_g;
  };
  if constexpr (kHoist) rates();
  // What inlet and outlet nodes read; the inlet velocity of a node changes
  // from step to step only with inlet noise.
  StepArgs e;
  e.nx = nx;
  e.ny = ny;
  e.nz = 1;
  e.inflow_parabolic = ap->inflow_parabolic;
  e.uin_x = ap->uin_x;
  e.uin_y = ap->uin_y;
  e.umax = ap->umax;
  e.turb_amp = ap->turb_amp;
  e.turb_seed = ap->turb_seed;
  e.rho_out = ap->rho_out;
  e.outflow = ap->outflow;
  const bool noisy = e.turb_amp != 0.0f;
  float u_edge = 0.0f;
  if ((c & kClsInlet) && !noisy) u_edge = inlet_velocity(e, y, n, 0);
  // One step of the tile; EDGE = false where no node of the tile carries a
  // class bit (most tiles of a large domain), which skips every test for it.
  auto step = [&](auto edge, int s) {
    constexpr bool EDGE = decltype(edge)::value;
    const int src = (s - 1) & 1, dst = s & 1;
    // The parameters as values the compiler takes no product of out of the
    // loop: hoisted, it would no longer fuse into the sum it feeds, and the
    // node would round differently from a single step.
    if constexpr (kHoist) {
      asm volatile("" : "+v"(rate_s));
      if constexpr (COLL == kTRT) asm volatile("" : "+v"(rate_a));
    } else {
      asm volatile("" : "+s"(b.tau));
      if constexpr (LES) asm volatile("" : "+s"(b.cs));
      if constexpr (THERMAL) asm volatile("" : "+s"(b.tau_g));
    }
    if constexpr (FORCE || THERMAL) asm volatile("" : "+s"(b.gx), "+s"(b.gy));
    if constexpr (THERMAL) asm volatile("" : "+s"(b.gbeta), "+s"(b.t_ref));
    if constexpr (THERMAL && EDGE) {
      static_for<D2Q5::Q>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        if constexpr (q > 0) opaque(t_wall[q]);  // 2 w T_wall is such a product
      });
    }
    if (i >= s && i < W - s && j >= s && j < H - s) {
      float f[L::Q];
      const bool pull = !(from_s && s == 1) && !(EDGE && (c & kClsFrozen));
      const unsigned long long k = s_step + static_cast<unsigned long long>(s - 1);  // S_k is formed here
      static_for<L::Q>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        f[q] = tb_get<St, L, q>(sh.f[src][q][cell - L::cy[q] * W - L::cx[q]]);
      });
      if (!pull) {
        static_for<L::Q>([&](auto qc) {
          constexpr int q = decltype(qc)::value;
          f[q] = tb_get<St, L, q>(sh.f[src][q][cell]);
        });
      } else if (EDGE && c) {
        if (c & kClsSlow) {
          // every own-node value is read at once and the bouncing ones kept:
          // one LDS round trip instead of one per bouncing direction
          float own_f[L::Q];
          static_for<L::Q>([&](auto qc) {
            constexpr int q = decltype(qc)::value;
            if constexpr (q > 0) own_f[q] = tb_get<St, L, L::opp[q]>(sh.f[src][L::opp[q]][cell]);
          });
          if (moving) {
            TileArgs* p = opaque_args(ap);
            const float uw[3] = {p->uw[0], p->uw[1], p->uw[2]};
            static_for<L::Q>([&](auto qc) {
              constexpr int q = decltype(qc)::value;
              if constexpr (q > 0) {
                const float ci_uw = static_cast<float>(L::cx[q]) * uw[0] + static_cast<float>(L::cy[q]) * uw[1] +
                                    static_cast<float>(L::cz[q]) * uw[2];
                const float v = own_f[q] + 2.0f * L::w[q] * 1.0f * 3.0f * ci_uw;
                if (moving & (1u << q)) own_f[q] = v;
              }
            });
          }
          static_for<L::Q>([&](auto qc) {
            constexpr int q = decltype(qc)::value;
            if constexpr (q > 0) {
              if (bm & (1u << q)) f[q] = own_f[q];
            }
          });
        }
        if (c & kClsInlet) {
          if (noisy) u_edge = inlet_velocity(e, y, n, k);
          close_inlet<L>(f, u_edge, e.uin_y);
        }
        if ((c & kClsOutlet) && e.outflow == 1) apply_zh_outflow_d2q9(e, f);
      }
      if constexpr (THERMAL) {
        float g[D2Q5::Q];
        static_for<D2Q5::Q>([&](auto qc) {
          constexpr int q = decltype(qc)::value;
          g[q] = sh.g[src][q][cell - D2Q5::cy[q] * W - D2Q5::cx[q]];
          if (!pull) g[q] = sh.g[src][q][cell];
          if constexpr (q > 0) {
            if (EDGE && pull && (g_wall & (1u << q))) {
              const float r = sh.g[src][D2Q5::opp[q]][cell];
              const float tw = t_wall[q];
              g[q] = (tw != tw) ? r : -r + 2.0f * D2Q5::w[q] * tw;
            }
          }
        });
        if (!EDGE || !(c & kClsSolid)) {
          if constexpr (!kHoist) rates();
          thermal_collide_rates<COLL>(b, rate_s, rate_a, rate_g, f, g);
        }
        static_for<D2Q5::Q>([&](auto qc) {
          constexpr int q = decltype(qc)::value;
          sh.g[dst][q][cell] = g[q];
        });
      } else {
        if (EDGE && force_at >= 0 && pull) {
          TileArgs* p = opaque_args(ap);
          StepArgs m;
          m.nx = nx;
          m.ny = ny;
          m.nz = 1;
          m.per_y = p->per_y;
          m.per_z = p->per_z;
          double s0 = 0.0, s1 = 0.0, s2 = 0.0;
          mem_node<L>(m, x, y, 0, n, f, p->mem_c[0], p->mem_c[1], p->mem_c[2], p->mem_rmax, s0, s1, s2, &bm);
          double* o = mf.out + 3 * (static_cast<long long>(k % mf.ring) * mf.count + force_at);
          o[0] = s0;
          o[1] = s1;
          o[2] = s2;
        }
        if (!EDGE || !(c & kClsSolid)) {
          if constexpr (!kHoist) rates();
          const Macro m =
              collide_d2q9_rates<COLL, LES, St::kFast, FORCE>(f, b.tau, rate_s, rate_a, b.cs, b.gx, b.gy);
          flag_nonfinite(b, m.rho);
        }
      }
      static_for<L::Q>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        sh.f[dst][q][cell] = tb_put<St, L, q>(f[q]);
      });
    }
    __syncthreads();
  };
  const bool edges = EDGES && __syncthreads_or(c != 0);
  if constexpr (!EDGES) __syncthreads();
  if (edges) {
#pragma unroll 1
    for (int s = 1; s <= nsteps; ++s) step(std::bool_constant<EDGES>{}, s);
  } else {
#pragma unroll 1
    for (int s = 1; s <= nsteps; ++s) step(std::false_type{}, s);
  }
  if (own) {
    const int last = nsteps & 1;
    static_for<L::Q>([&](auto qc) {
      constexpr int q = decltype(qc)::value;
      aout[q * S + n] = sh.f[last][q][cell];
    });
    if constexpr (THERMAL) {
      static_for<D2Q5::Q>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        gout[q * S + n] = sh.g[last][q][cell];
      });
    }
  }
}

}  // namespace wake_hip
