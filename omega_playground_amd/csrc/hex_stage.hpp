// Per-cell device operators of the one-launch forward stage on the regular
// hexagonal mesh with uniform coefficients (HexStage records and HexCoef,
// checked on the host in hex_layout.cpp), any layer count.
//
// A cell's tendencies are functions of the prognostic rows of its
// neighbourhood alone: its three owned edges' tendencies read 26 velocity and
// 14 thickness rows.  The operators here form every intermediate (vertex
// vorticity and thickness, kinetic energy, divergence) in registers from
// those rows instead of reading what a diagnostics launch stored.
//
// Bits: every sum keeps the reference's order and every product its
// association.  On this mesh all cdiv, cke, crv, cth share one magnitude,
// 1/dc, 1/dv, the scalings and f are one value, and the TRiSK weights are
// exactly (+-2, +-1, 0) times one value, so a product that two stencils form
// with coefficients of either sign is formed once.  Factors 1/2 and 1/4 are
// folded into factors far from the subnormal range, never into one that
// holds a velocity: the tails of a vortex run through that range, where a
// power of two no longer scales exactly.
#pragma once

#include <type_traits>
#include <utility>

#include "device_common.hpp"
#include "hex_lattice.hpp"

namespace omega_hip {
namespace stage {

using namespace dev;
namespace hl = hexl;

// f(0), ..., f(n-1) with compile-time indices
template <class F, int... I>
__device__ __forceinline__ void each_of(F &&f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int n, class F> __device__ __forceinline__ void each(F &&f) {
  each_of(f, std::make_integer_sequence<int, n>{});
}

// What a stage kernel reads and writes; passed by value.
struct Ctx {
  int L;
  unsigned L8;    // bytes of a row
  unsigned k8;    // byte offset of this lane's first level
  int k;          // this lane's first level
};

template <int N> __device__ __forceinline__ Vd<N> ldo(const double *p, unsigned off) {
  return ld<N>(reinterpret_cast<const double *>(reinterpret_cast<const char *>(p) + off));
}
template <int N> __device__ __forceinline__ void sto(double *p, unsigned off, const Vd<N> &x) {
  st<N>(reinterpret_cast<double *>(reinterpret_cast<char *>(p) + off), x);
}

// Coefficients of one leg of a walk, each a copy the compiler does not
// recognise as the other legs' (one scalar move)
struct LegCoef {
  double crv, cth, cke, cdiv, hdiv, idc;
};
template <int tag> __device__ __forceinline__ double own(double x) {
  asm("; leg %1" : "+s"(x) : "i"(tag));
  return x;
}
template <int tag> __device__ __forceinline__ LegCoef leg_coef(const HexCoef &q) {
  return LegCoef{own<tag>(q.crv),  own<tag>(q.cth),  own<tag>(q.cke),
                 own<tag>(q.cdiv), own<tag>(q.hdiv), own<tag>(q.idc)};
}

// x, unknown to the compiler: rows read again through it are loaded again
__device__ __forceinline__ unsigned again(unsigned x) {
  asm volatile("" : "+v"(x));
  return x;
}

// x, read anew each time round a loop: products with it stay in the loop
__device__ __forceinline__ double each_time(double x) {
  asm volatile("" : "+s"(x));
  return x;
}

// Values formed by here: the compiler may not sink their arithmetic below
template <int N> __device__ __forceinline__ void pin(Vd<N> &x) {
#pragma unroll
  for (int i = 0; i < N; ++i) asm volatile("" : "+v"(x[i]));
}
template <int N, class... A> __device__ __forceinline__ void pin(Vd<N> &x, A &...rest) {
  pin(x);
  pin(rest...);
}

// the 19 cells of the neighbourhood (hexl numbering), from the cell's record
__device__ __forceinline__ void load_cells(const int *__restrict__ rec, int c,
                                           int (&id)[hl::kCells]) {
  const int4 *p = reinterpret_cast<const int4 *>(rec + (size_t)c * hl::kRec);
  int t[hl::kRec];
#pragma unroll
  for (int i = 0; i < hl::kRec / 4; ++i) {
    const int4 v = p[i];
    t[4 * i] = v.x;
    t[4 * i + 1] = v.y;
    t[4 * i + 2] = v.z;
    t[4 * i + 3] = v.w;
  }
#pragma unroll
  for (int i = 0; i < hl::kCells; ++i) id[i] = t[i];
}

// ---------------------------------------------------------------------------
// Momentum and thickness of one cell: compute_vn_tendency on the three owned
// edges (PV flux, KE and SSH gradients, del2) and compute_h_tendency.
// ---------------------------------------------------------------------------
template <int N> struct MomOut {
  // terms of the owned edges' tendencies, in the order they are added to the
  // starting value: + u, - ke_grad, - ssh_grad, + visc (V2)
  Vd<N> u[3], ke_grad[3], ssh_grad[3], visc[3];
  Vd<N> h; // thickness tendency
  Vd<N> rv[2], it[2], ke, div; // the cell's own diagnostics
  // PRE: the rows of the owned edges a tendency VJP reads here (PreOut)
  Vd<N> se[3], fu[3], own[3];
};

// The walk keeps few rows live at a time: the four vertices of the owned
// edges, then round the three neighbours across those edges (W, SW, SE, whose
// sides come in the PV stencils' slot order), then the second half of every
// stencil, round the cell itself, whose outer sides' rows are read again.
// Each leg has its own copies of the coefficients (leg_coef), so that
// products two legs form are formed twice instead of staying live between
// them, and FENCE keeps the scheduler from hoisting a later leg's rows above
// an earlier one's arithmetic; without these the walk needs 180 registers
// and half the wavefronts.
// early(o): called once o's rv, it, se and fu are set, to store them before
// the walk goes on.
template <int N, bool V2, bool PRE, class Early>
__device__ __forceinline__ void momentum(const HexCoef &q, const Ctx &x,
                                         const int (&id)[hl::kCells], const double *__restrict__ h,
                                         const double *__restrict__ vn, MomOut<N> &o, Early early) {
  const unsigned L8 = x.L8;
  unsigned k8 = x.k8;
  Vd<N> hv[hl::kCells], v[hl::kEdges];
  Vd<N> P[hl::kVerts], Q[hl::kVerts], rvort[hl::kVerts];
  Vd<N> S[hl::kEdges], T[hl::kEdges], G[hl::kEdges], G2[hl::kEdges], F[hl::kEdges];
  Vd<N> ke[4], dv[4], qs[3], qt[3], curl[3];
  auto H = [&](auto... I) {
    ((hv[I] = ldo<N>(h, __umul24((unsigned)id[I], L8) + k8)), ...);
  };
  auto V = [&](auto... E) {
    ((v[E] = ldo<N>(vn + (E % 3) * x.L, __umul24((unsigned)id[E / 3], 3u * L8) + k8)), ...);
  };
  // a vertex: relative vorticity, 1/thickness, the two PV products
  auto vertex = [&](const LegCoef &c, auto W) {
    constexpr int w = W;
    constexpr hl::Vert t = hl::vert(w);
#pragma unroll
    for (int i = 0; i < N; ++i) {
      double rv = __builtin_fma(t.s[0] * c.crv, v[t.e[0]][i], 0.0);
      rv = rv + t.s[1] * (c.crv * v[t.e[1]][i]);
      rv = rv + t.s[2] * (c.crv * v[t.e[2]][i]);
      double th = __builtin_fma(c.cth, hv[t.c[0]][i], 0.0);
      th = th + c.cth * hv[t.c[1]][i];
      th = th + c.cth * hv[t.c[2]][i];
      const double it = 0.25 / th; // a quarter of 1/thickness
      rvort[w][i] = rv;
      P[w][i] = it * rv;
      Q[w][i] = it * q.f;
      if constexpr (w < 2) {
        o.rv[w][i] = rv;
        o.it[w][i] = 4.0 * it;
      }
    }
  };
  // an edge of the stencils: half the edge means of the PV products, and the
  // weighted thickness flux (w * thickness) * v with the weights it is read
  // with (the smallest one, and twice that)
  auto side = [&](auto E) {
    constexpr int e = E;
    constexpr hl::Edge t = hl::edge(e);
#pragma unroll
    for (int i = 0; i < N; ++i) {
      S[e][i] = P[t.v[0]][i] + P[t.v[1]][i];
      T[e][i] = Q[t.v[0]][i] + Q[t.v[1]][i];
      const double s = hv[t.c[0]][i] + hv[t.c[1]][i];
      G[e][i] = (q.w2 * s) * v[e][i];
      G2[e][i] = (q.w * s) * v[e][i];
      if constexpr (PRE) F[e][i] = (0.5 * s) * v[e][i];
    }
  };
  // slot j of the PV stencil of owned edge K (the slots of weight zero too: an
  // infinity there makes the sum a NaN)
  auto pv = [&](auto KK, auto J) {
    constexpr int K = KK, m = hl::pv_mult(K, J), e = hl::pv_edge(K, J);
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const double nv = (qs[K][i] + S[e][i]) + T[e][i];
      const double t = (m == 2 || m == -2 ? G2[e][i] : G[e][i]) * nv;
      if constexpr (m > 0) qt[K][i] = qt[K][i] + t;
      else if constexpr (m < 0) qt[K][i] = qt[K][i] - t;
      else qt[K][i] = __builtin_fma(t, 0.0, qt[K][i]);
      if constexpr (PRE) {
        // flux-weighted sum: weight times flux, in slot order
        const double x = ((m == 2 || m == -2 ? 2 * q.w : q.w) * F[e][i]);
        if constexpr (m > 0) o.own[K][i] = o.own[K][i] + x;
        else if constexpr (m < 0) o.own[K][i] = o.own[K][i] - x;
        else o.own[K][i] = __builtin_fma(F[e][i], 0.0, o.own[K][i]);
      }
    }
  };
  // kinetic energy and divergence of cell b
  auto cell = [&](const LegCoef &c, auto B) {
    constexpr int b = B;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      double a = 0.0, d = 0.0;
      each<6>([&](auto J) {
        constexpr int j = J, e = hl::cell_edge(b, j);
        const double u = v[e][i];
        a = __builtin_fma((c.cke * u) * u, 0.25, a);
        d = j < 3 ? d - c.cdiv * u : d + c.cdiv * u;
      });
      ke[b][i] = a;
      dv[b][i] = d;
    }
  };
#define HEXC(n) (std::integral_constant<int, n>{})
#define FENCE() __builtin_amdgcn_sched_barrier(0)
  H(HEXC(0), HEXC(1), HEXC(2), HEXC(3), HEXC(4), HEXC(6));
  V(HEXC(0), HEXC(1), HEXC(2), HEXC(12), HEXC(20), HEXC(19), HEXC(5), HEXC(9), HEXC(13));
  FENCE();
  V(HEXC(56), HEXC(3), HEXC(4), HEXC(6), HEXC(18), HEXC(55), HEXC(23));
  H(HEXC(18), HEXC(7), HEXC(8));
  const LegCoef c0 = leg_coef<0>(q);
  vertex(c0, HEXC(0));
  vertex(c0, HEXC(1));
  vertex(c0, HEXC(6));
  vertex(c0, HEXC(9));
  each<3>([&](auto KK) {
    constexpr int K = KK;
    constexpr hl::Edge t = hl::edge(K);
#pragma unroll
    for (int i = 0; i < N; ++i) {
      qs[K][i] = (P[t.v[0]][i] + P[t.v[1]][i]) + (Q[t.v[0]][i] + Q[t.v[1]][i]);
      qt[K][i] = 0.0;
      curl[K][i] = (rvort[t.v[1]][i] - rvort[t.v[0]][i]) * q.idv;
      if constexpr (PRE) {
        o.se[K][i] = 2.0 * qs[K][i];
        o.own[K][i] = 0.0;
        o.fu[K][i] = 0.5 * (hv[t.c[0]][i] + hv[t.c[1]][i]) * v[K][i];
      }
    }
  });
  pin(P[0], Q[0], P[1], Q[1], P[6], Q[6], P[9], Q[9], qs[0], qs[1], qs[2], qt[0], qt[1], qt[2]);
  if constexpr (V2) pin(curl[0], curl[1], curl[2]);
  early(o);
  FENCE();
  // round W: its sides NE, NW, (W), SW, SE
  V(HEXC(7), HEXC(8), HEXC(26), HEXC(10), HEXC(30));
  H(HEXC(9), HEXC(10));
  const LegCoef c1 = leg_coef<1>(q);
  vertex(c1, HEXC(13));
  side(HEXC(19));
  pv(HEXC(0), HEXC(0));
  vertex(c1, HEXC(2));
  side(HEXC(56));
  pv(HEXC(0), HEXC(1));
  vertex(c1, HEXC(3));
  side(HEXC(3));
  pv(HEXC(0), HEXC(2));
  vertex(c1, HEXC(4));
  side(HEXC(4));
  pv(HEXC(0), HEXC(3));
  side(HEXC(5));
  pv(HEXC(0), HEXC(4));
  pv(HEXC(1), HEXC(0));
  cell(c1, HEXC(1));
  pin(qt[0], qt[1], ke[1], P[4], Q[4]);
  if constexpr (PRE) pin(o.own[0], o.own[1]);
  if constexpr (V2) pin(dv[1]);
  FENCE();
  // round SW: its sides W, (SW), SE, E
  V(HEXC(11), HEXC(36), HEXC(33), HEXC(37), HEXC(14));
  H(HEXC(11), HEXC(12));
  const LegCoef c2 = leg_coef<2>(q);
  vertex(c2, HEXC(5));
  side(HEXC(6));
  pv(HEXC(1), HEXC(1));
  vertex(c2, HEXC(20));
  side(HEXC(7));
  pv(HEXC(1), HEXC(2));
  vertex(c2, HEXC(7));
  side(HEXC(8));
  pv(HEXC(1), HEXC(3));
  side(HEXC(9));
  pv(HEXC(1), HEXC(4));
  pv(HEXC(2), HEXC(0));
  cell(c2, HEXC(2));
  pin(qt[1], qt[2], ke[2], P[7], Q[7]);
  if constexpr (PRE) pin(o.own[1], o.own[2]);
  if constexpr (V2) pin(dv[2]);
  FENCE();
  // round SE: its sides W, (SW), SE, E, NE
  const LegCoef c3 = leg_coef<3>(q);
  vertex(c3, HEXC(22));
  side(HEXC(10));
  pv(HEXC(2), HEXC(1));
  vertex(c3, HEXC(25));
  side(HEXC(11));
  pv(HEXC(2), HEXC(2));
  vertex(c3, HEXC(24));
  side(HEXC(36));
  pv(HEXC(2), HEXC(3));
  side(HEXC(13));
  pv(HEXC(2), HEXC(4));
  cell(c3, HEXC(3));
  // round the cell
  k8 = again(k8);
  H(HEXC(4), HEXC(5), HEXC(6));
  V(HEXC(17), HEXC(15), HEXC(12), HEXC(16), HEXC(20));
  pin(qt[2], ke[3]);
  if constexpr (PRE) pin(o.own[2]);
  if constexpr (V2) pin(dv[3]);
  FENCE();
  const LegCoef c4 = leg_coef<4>(q);
  vertex(c4, HEXC(8));
  vertex(c4, HEXC(11));
  side(HEXC(1));
  pv(HEXC(0), HEXC(5));
  side(HEXC(2));
  pv(HEXC(0), HEXC(6));
  pv(HEXC(1), HEXC(5));
  side(HEXC(12));
  pv(HEXC(0), HEXC(7));
  pv(HEXC(1), HEXC(6));
  pv(HEXC(2), HEXC(5));
  side(HEXC(16));
  pv(HEXC(0), HEXC(8));
  pv(HEXC(1), HEXC(7));
  pv(HEXC(2), HEXC(6));
  side(HEXC(20));
  pv(HEXC(0), HEXC(9));
  pv(HEXC(1), HEXC(8));
  pv(HEXC(2), HEXC(7));
  side(HEXC(0));
  pv(HEXC(1), HEXC(9));
  pv(HEXC(2), HEXC(8));
  pv(HEXC(2), HEXC(9));
  cell(c4, HEXC(0));
#undef HEXC
#undef FENCE
#pragma unroll
  for (int i = 0; i < N; ++i) {
    double a = 0.0;
    each<6>([&](auto J) {
      constexpr int j = J, e = hl::cell_edge(0, j);
      const double f = (q.hdiv * (hv[0][i] + hv[1 + j][i])) * v[e][i];
      a = j < 3 ? a + f : a - f;
    });
    o.h[i] = a;
  }
  o.ke = ke[0];
  o.div = dv[0];
  each<3>([&](auto KK) {
    constexpr int K = KK, nb = K + 1; // the neighbour across is the edge's first cell
#pragma unroll
    for (int i = 0; i < N; ++i) {
      o.u[K][i] = qt[K][i];
      o.ke_grad[K][i] = (ke[0][i] - ke[nb][i]) * q.idc;
      o.ssh_grad[K][i] = q.grav * (hv[0][i] - hv[nb][i]) * q.idc;
      if constexpr (V2) {
        const double del2u = (dv[0][i] - dv[nb][i]) * q.idc - curl[K][i];
        o.visc[K][i] = ((x.k + i < q.ml) ? q.cv2 : 0.0) * del2u;
      }
    }
    pin(o.u[K], o.ke_grad[K], o.ssh_grad[K]);
    if constexpr (V2) pin(o.visc[K]);
  });
  pin(o.h);
}

// ---------------------------------------------------------------------------
// Momentum del4 (vel_hyperdiff_edge.hpp:140-237): the Laplacian of an edge
// field x on the three owned edges, (div1 - div0)/dc - (curl1 - curl0)*idv,
// with the divergences of the cells and the curls of the vertices formed from
// the 19 rows of x around.  Applied to the velocity and then to its own
// result.
// ---------------------------------------------------------------------------
template <int N> struct LapOut {
  Vd<N> e[3];         // the Laplacian on the owned edges
  Vd<N> curl[2], div; // of x on the cell's own vertices and at the cell
};

template <int N>
__device__ __forceinline__ void laplacian(const HexCoef &q, double idv, const Ctx &x,
                                          const int (&id)[hl::kCells],
                                          const double *__restrict__ in, LapOut<N> &o) {
  Vd<N> v[hl::kEdges], div[4], curl[hl::kVerts];
  each<hl::kEdges>([&](auto E) {
    constexpr int e = E;
    if constexpr (hl::kNeed.lap[e])
      v[e] = ldo<N>(in + (e % 3) * x.L, __umul24((unsigned)id[e / 3], 3u * x.L8) + x.k8);
  });
  each<4>([&](auto B) {
    constexpr int b = B;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      double d = 0.0;
      each<6>([&](auto J) {
        constexpr int j = J, e = hl::cell_edge(b, j);
        d = j < 3 ? d - q.cdiv * v[e][i] : d + q.cdiv * v[e][i];
      });
      div[b][i] = d;
    }
  });
  each<hl::kVerts>([&](auto W) {
    constexpr int w = W;
    if constexpr (w == 0 || w == 1 || w == 6 || w == 9) {
      constexpr hl::Vert t = hl::vert(w);
#pragma unroll
      for (int i = 0; i < N; ++i) {
        double r = __builtin_fma(t.s[0] * q.crv, v[t.e[0]][i], 0.0);
        r = r + t.s[1] * (q.crv * v[t.e[1]][i]);
        r = r + t.s[2] * (q.crv * v[t.e[2]][i]);
        curl[w][i] = r;
      }
    }
  });
  each<3>([&](auto KK) {
    constexpr int K = KK;
    constexpr hl::Edge t = hl::edge(K);
#pragma unroll
    for (int i = 0; i < N; ++i)
      o.e[K][i] = (div[0][i] - div[K + 1][i]) * q.idc - (curl[t.v[1]][i] - curl[t.v[0]][i]) * idv;
  });
  o.curl[0] = curl[0];
  o.curl[1] = curl[1];
  o.div = div[0];
}

} // namespace stage
} // namespace omega_hip
