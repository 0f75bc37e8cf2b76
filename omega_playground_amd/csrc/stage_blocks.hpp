// Block bodies of the stage kernels, shared by the kernels with a launch of
// their own (kernels_stage.hip) and those that run both in one launch
// (kernels_stage_both.hip).
#pragma once

#include "hex_stage.hpp"
#include "stage_launch.hpp"

namespace omega_hip {
namespace stage {

// Entry of block b of n: workgroups are dealt to the 8 XCDs round-robin, and
// with swz each XCD takes a contiguous range of entries, so that neighbouring
// cells' rows are re-read from one L2.  (Chosen without a branch, which cost
// 0.1 us of a 5 us launch.)
__device__ __forceinline__ int block_entry(int b, int n, int swz) {
  const int e = logical_block(b, n, 1);
  return swz ? e : b;
}
__device__ __forceinline__ int xcd_entry(int n, int swz) { return block_entry((int)blockIdx.x, n, swz); }

// The cell and levels of this thread at an entry (level chunk, cell block);
// false: no work here.
__device__ __forceinline__ bool stage_place(const StageLaunch &p, int entry, int N, int &c, Ctx &x) {
  const int ch = p.tiles == p.ncb ? 0 : uniform(entry / p.ncb);
  const int row = (int)threadIdx.x / p.lx, ln = (int)threadIdx.x - row * p.lx;
  c = (entry - ch * p.ncb) * p.rows + row;
  const int k = (ch * p.lx + ln) * N;
  x = Ctx{p.L, (unsigned)p.L * 8u, (unsigned)k * 8u, k};
  return row < p.rows && c < p.nc && k < p.L;
}

// Momentum and thickness.  Two levels per lane at two waves per SIMD (228
// registers) take 0.68 ms per stage at nx=512, 64 layers (2.25 GB, 3.3 TB/s;
// the vector units half busy, the rest latency), one level per lane at four
// waves 0.83 ms (the same rows in twice the load instructions).
// V4: subtract the del4 rows (p.x) the Laplacian launches left.
template <int N, bool V2, bool V4, bool EMIT, bool PRE = false>
__device__ __forceinline__ void stage_mom(const StageLaunch &p, int entry) {
  int c;
  Ctx x;
  if (!stage_place(p, entry, N, c, x)) return;
  const StageArgs &a = p.a;
  const int L = x.L, k = x.k;
  int id[hl::kCells];
  load_cells(p.rec, c, id);
  const size_t idx = (size_t)c * L + k, e0 = (size_t)(3 * c) * L + k;
  MomOut<N> o;
  momentum<N, V2, PRE>(p.q, x, id, a.h.in, a.vn.in, o, [&](const MomOut<N> &o) {
    if constexpr (EMIT) {
#pragma unroll
      for (int w = 0; w < 2; ++w) {
        const size_t vi = (size_t)(2 * c + w) * L + k;
        st<N>(p.d.rvort_v + vi, o.rv[w]);
        st<N>(p.d.inv_thick_v + vi, o.it[w]);
      }
    }
    if constexpr (PRE) {
#pragma unroll
      for (int K = 0; K < 3; ++K) {
        st<N>(p.pre.se + e0 + K * L, o.se[K]);
        st<N>(p.pre.fu + e0 + K * L, o.fu[K]);
      }
    }
  });
  if constexpr (EMIT) {
    st<N>(p.d.ke_c + idx, o.ke);
    st<N>(p.d.div_c + idx, o.div);
  }
  if constexpr (PRE) {
#pragma unroll
    for (int K = 0; K < 3; ++K) st<N>(p.pre.own + e0 + K * L, o.own[K]);
  }
#pragma unroll
  for (int K = 0; K < 3; ++K) {
    Vd<N> T = tend_base<N>(a, a.vn, e0 + K * L);
#pragma unroll
    for (int i = 0; i < N; ++i) {
      T[i] = T[i] + o.u[K][i];
      T[i] = T[i] - o.ke_grad[K][i];
      T[i] = T[i] - o.ssh_grad[K][i];
      if constexpr (V2) T[i] = T[i] + o.visc[K][i];
    }
    if constexpr (V4) {
      const Vd<N> y = ld<N>(p.x + e0 + K * L);
#pragma unroll
      for (int i = 0; i < N; ++i) T[i] = T[i] - y[i];
    }
    epilogue<N>(a, a.vn, e0 + K * L, T);
  }
  Vd<N> T = tend_base<N>(a, a.h, idx);
#pragma unroll
  for (int i = 0; i < N; ++i) T[i] = T[i] + o.h[i];
  epilogue<N>(a, a.h, idx, T);
}

// A tile's LDS: rows of thickness, tracer ratio and (D4) Laplacian at its places,
// and the cells there
template <int N, int LX, int TW, int TH, bool D4> struct TileRows {
  static constexpr int HALO = D4 ? 2 : 1;
  static constexpr int PLACES = (TW + 2 * HALO) * (TH + 2 * HALO), ROWS = PLACES * LX * N,
                       LAPS = D4 ? ROWS : 1;
  alignas(16) double h[ROWS];
  double ratio[ROWS], lap[LAPS];
  int ids[PLACES];
};

// ---------------------------------------------------------------------------
// Tracers: a block stages a tile of the lattice, TW x TH cells with one ring
// of halo (two with del4) and LX lanes of N levels, in LDS, so that a
// neighbour's tracer ratio and Laplacian are formed once per tile instead of
// once per cell that reads them: 0.86 ms per stage at nx=512, 64 layers, 4
// tracers with del4 (0.64 without, 90 % of a copy's rate), against 1.49 ms
// for one cell per thread with both rings in registers (19 divisions and 19
// rows per cell and tracer).  A thread computes its own cell's Laplacian and
// at most one of the ring's, with the sums of its cell's thicknesses kept in
// registers for all tracers.  Tiles of 64-byte rows (LX = 4, N = 2) ran
// faster than 128-byte ones (6.3 against 7.2 ms per step), three waves per
// SIMD faster than four with 13 registers spilled (6.3 against 7.0).
// ---------------------------------------------------------------------------
template <int N, int LX, int TW, int TH, bool D2, bool D4, bool EMIT>
__device__ __forceinline__ void stage_tile(const TileLaunch &p, int w, int l0, double *Hs, double *Ns,
                                           double *Ds, int *ids) {
  constexpr int HALO = D4 ? 2 : 1, PW = TW + 2 * HALO, PH = TH + 2 * HALO, NP = PW * PH;
  constexpr int CELLS = TW * TH, R = (NP + CELLS - 1) / CELLS;
  constexpr int RING = 2 * (TW + 2) + 2 * TH; // the first ring round the tile
  static_assert(RING <= CELLS, "one place of the ring per row of lanes");
  constexpr int S = LX * N; // doubles per place and array
  const int tile = uniform(w / p.nch), ch = w - tile * p.nch;
  const int ln = (int)threadIdx.x % LX, row = (int)threadIdx.x / LX;
  const int L = p.L, k = (ch * LX + ln) * N;
  const bool lev = k < L;
  const unsigned L8 = (unsigned)L * 8u, k8 = (unsigned)k * 8u;
  const size_t sp = (size_t)p.nc * L;
  const StageArgs &a = p.a;
  const HexCoef &q = p.q;
  const int *tid = p.ids + (size_t)tile * ((TW + 4) * (TH + 4));
  for (int i = (int)threadIdx.x; i < NP; i += LX * CELLS)
    ids[i] = tid[(i / PW + 2 - HALO) * (TW + 4) + i % PW + 2 - HALO];
  __syncthreads();
  const int l1 = min(l0 + p.per_block, a.ntr);
  // the places this thread stages: thickness, its inverse, the first tracer
  Vd<N> inv[R], t[R];
  unsigned off[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int pos = row + r * CELLS;
    if (pos < NP && lev) {
      off[r] = __umul24((unsigned)ids[pos], L8) + k8;
      inv[r] = ldo<N>(a.h.in, off[r]);
      t[r] = ldo<N>(a.tr.in + l0 * sp, off[r]);
    }
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int pos = row + r * CELLS;
    if (pos < NP && lev) {
      st<N>(Hs + pos * S + ln * N, inv[r]);
#pragma unroll
      for (int i = 0; i < N; ++i) inv[r][i] = 1.0 / inv[r][i];
    }
  }
  // A place's neighbours W, SW, SE, E, NE, NW are at fixed distances from it,
  // those of other rows one place further right in odd rows: two bases,
  // lowered by a row so that every distance is positive
  struct Place {
    int same, other; // index of the element a row below and one left
  };
  auto place = [&](int x, int y) {
    const int i = ((y - 1) * PW + x - 1) * S + ln * N;
    return Place{i, i + ((y + HALO) & 1) * S};
  };
  auto get = [&](const double *A, const Place &o, auto J) {
    constexpr int j = J; // 0 the place itself, 1 + d its neighbour in direction d
    constexpr int by[7] = {PW + 1, PW, 0, 1, PW + 2, 2 * PW + 1, 2 * PW};
    constexpr bool same = j < 2 || j == 4;
    return ld<N>(A + (same ? o.same : o.other) + by[j] * S);
  };
  // the thread's own cell (tile rows start at even rows of the lattice, and
  // so do staged rows)
  const int cy = row / TW, cx = row % TW;
  const Place own = place(cx + HALO, cy + HALO);
  const int self = (cy + HALO) * PW + cx + HALO;
  const bool mine = lev && (tile % p.tiles_x) * TW + cx < p.nx && (tile / p.tiles_x) * TH + cy < p.ny;
  Vd<N> v[6];
  if (mine) {
    const int odd = cy & 1;
    const int c4[6] = {ids[self], ids[self], ids[self], ids[self + 1], ids[self + PW + odd],
                       ids[self + PW - 1 + odd]};
#pragma unroll
    for (int j = 0; j < 6; ++j)
      v[j] = ldo<N>(a.vn.in + (j % 3) * L, __umul24((unsigned)c4[j], 3u * L8) + k8);
  }
  __syncthreads();
  Vd<N> f[6];
  {
    const Vd<N> h0 = get(Hs, own, std::integral_constant<int, 0>{});
    each<6>([&](auto J) {
      const Vd<N> hj = get(Hs, own, std::integral_constant<int, 1 + J>{});
#pragma unroll
      for (int i = 0; i < N; ++i) f[J][i] = hj[i] + h0[i];
    });
  }
  const int c = ids[self];
  // this thread's place on the ring: the rows below and above, then the sides
  const int rr = row < RING ? row : 0, side = rr - 2 * (TW + 2);
  const Place ring = side < 0 ? place(rr % (TW + 2) + 1, rr < TW + 2 ? 1 : TH + 2)
                             : place(side & 1 ? TW + 2 : 1, side / 2 + 2);
  for (int l = l0; l < l1; ++l) {
    if (l > l0) __syncthreads();
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int pos = row + r * CELLS;
      if (pos < NP && lev) {
        Vd<N> n;
#pragma unroll
        for (int i = 0; i < N; ++i) n[i] = t[r][i] * inv[r][i];
        st<N>(Ns + pos * S + ln * N, n);
        if (l + 1 < l1) t[r] = ldo<N>(a.tr.in + (l + 1) * sp, off[r]);
      }
    }
    const size_t idx = ((size_t)l * p.nc + c) * L + k;
    EpiIn<N> e;
    if (mine) e = epi_prefetch<N>(a, a.tr, idx);
    __syncthreads();
    // the cell's tracer Laplacian (D4) and advection, from its neighbours' ratios
    const double qdiv = each_time(q.qdiv), hdiv = each_time(q.hdiv);
    const Vd<N> n0 = get(Ns, own, std::integral_constant<int, 0>{});
    Vd<N> d0 = zero<N>(), adv = zero<N>(), dif = zero<N>(), hyp = zero<N>();
    each<6>([&](auto J) {
      constexpr int j = J;
      const Vd<N> nj = get(Ns, own, std::integral_constant<int, 1 + j>{});
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const double g = (j < 3 ? n0[i] - nj[i] : nj[i] - n0[i]) * q.idc;
        const double x = (qdiv * f[j][i]) * (nj[i] + n0[i]) * v[j][i];
        adv[i] = j < 3 ? adv[i] + x : adv[i] - x;
        if constexpr (D2) {
          const double y = q.ct2 * f[j][i] * q.s2 * g;
          dif[i] = j < 3 ? dif[i] - y : dif[i] + y;
        }
        if constexpr (D4) {
          const double z = (hdiv * f[j][i]) * g;
          d0[i] = j < 3 ? d0[i] - z : d0[i] + z;
        }
      }
    });
    pin(adv);
    if constexpr (D2) pin(dif);
    if constexpr (D4) {
      st<N>(Ds + own.same + (PW + 1) * S, d0);
      if (row < RING) {
        Place rim = ring;
        rim.same = (int)again((unsigned)rim.same);
        rim.other = (int)again((unsigned)rim.other);
        const Vd<N> h0 = get(Hs, rim, std::integral_constant<int, 0>{});
        const Vd<N> r0 = get(Ns, rim, std::integral_constant<int, 0>{});
        Vd<N> d = zero<N>();
        each<6>([&](auto J) {
          constexpr int j = J;
          const Vd<N> hj = get(Hs, rim, std::integral_constant<int, 1 + j>{});
          const Vd<N> nj = get(Ns, rim, std::integral_constant<int, 1 + j>{});
#pragma unroll
          for (int i = 0; i < N; ++i) {
            const double m = hdiv * (hj[i] + h0[i]);
            const double y = m * ((j < 3 ? r0[i] - nj[i] : nj[i] - r0[i]) * q.idc);
            d[i] = j < 3 ? d[i] - y : d[i] + y;
          }
        });
        st<N>(Ds + rim.same + (PW + 1) * S, d);
      }
      __syncthreads();
      each<6>([&](auto J) {
        constexpr int j = J;
        const Vd<N> dj = get(Ds, own, std::integral_constant<int, 1 + j>{});
#pragma unroll
        for (int i = 0; i < N; ++i) {
          const double z = q.ct4 * ((j < 3 ? d0[i] - dj[i] : dj[i] - d0[i]) * q.idc);
          hyp[i] = j < 3 ? hyp[i] + z : hyp[i] - z;
        }
      });
      pin(hyp);
    }
    if (mine) {
      Vd<N> T;
#pragma unroll
      for (int i = 0; i < N; ++i) {
        T[i] = e.base[i] + adv[i];
        if constexpr (D2) T[i] = T[i] + dif[i];
        if constexpr (D4) T[i] = T[i] + hyp[i];
      }
      if constexpr (EMIT && D4) st<N>(p.d.trdel2_c + idx, d0);
      epi_finish<N>(a, a.tr, idx, T, e);
    }
  }
}

} // namespace stage
} // namespace omega_hip
