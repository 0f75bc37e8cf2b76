// Forward stage on the regular hexagonal mesh with uniform coefficients, any
// layer count: one launch for momentum and thickness (hex_stage.hpp), one for
// the tracers, two more before them with momentum del4.  No diagnostics
// launch: each kernel forms what it needs from the prognostic rows.
//
// Against a diagnostics launch and a tendency launch that gather about 260
// rows per cell (nx=512, 64 layers, 4 tracers, del2 viscosity, tracer del4):
// 2.37 -> 1.57 ms per RK4 stage, 68 -> 44 rows per cell through HBM.  At 60
// layers, where that pair ran the general kernels, 0.250 -> 0.077 ms (150 x
// 94 cells, 3 tracers); one layer, 512 x 384 cells: 0.135 -> 0.016 ms.
#include <algorithm>

#include "stage_blocks.hpp"

namespace omega_hip {

namespace {

using namespace stage;

template <int N, bool V2, bool V4, bool EMIT>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(N == 1 ? 4 : 2)))
    k_stage_mom(StageLaunch p) {
  stage_mom<N, V2, V4, EMIT>(p, xcd_entry(p.tiles, p.swz));
}

// The same leaving the stage input's diagnostics and the rows its tendency
// VJP reads (the adjoint's stage recomputation): 137 us at nx=256, 32 layers
// with del2 viscosity, against 309 for a diagnostics and a tendency launch
// that gather the stored rows (with the tracers, 47 us here).  Two levels per
// lane spill up to 12 registers and are still the faster form (2.27 against
// 2.34 ms per step adjoint).
template <int N, bool V2, bool V4>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(N == 1 ? 3 : 2)))
    k_stage_mom_pre(StageLaunch p) {
  stage_mom<N, V2, V4, true, true>(p, xcd_entry(p.tiles, p.swz));
}

// A parameter block through the constant address space (no kernel writes one):
// its scalar loads then move over the row stores like those of a kernel's
// arguments (1012 -> 967 us per step of 16 mixed members).
template <class T> __device__ __forceinline__ const T &constant_at(const T *t, int i) {
  return *(const T *)((const __attribute__((address_space(4))) T *)t + i);
}

// Ensemble form: block b belongs to member who[b] (-1: none), whose parameter
// block is read in place through scalar loads and whose blocks start at a
// multiple of 8, so that each XCD takes a contiguous eighth of every member.
// Members of any terms share the launch (StageKind): with a launch for each
// set of terms small members waited for one another, 24 members of 576 cells
// with 8 sets of terms and 3 layer counts 1660 us per LSRK5 step, 107 so.
template <int N, int V2, bool EMIT>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(N == 1 ? 4 : 2)))
    k_batch_mom(const StageLaunch *__restrict__ desc, const int *__restrict__ who) {
  const int w = uniform(who[blockIdx.x]);
  if (w < 0) return;
  const StageLaunch &p = constant_at(desc, w);
  const int entry = block_entry((int)blockIdx.x - p.block0, p.tiles, p.swz);
  if constexpr (V2 != kAny) {
    stage_mom<N, V2 != 0, false, EMIT>(p, entry);
  } else {
    if (p.a.terms & T_VDEL2) stage_mom<N, true, false, EMIT>(p, entry);
    else stage_mom<N, false, false, EMIT>(p, entry);
  }
}

// The edge Laplacian: of the velocity (FINAL false), then of that result,
// with the masked coefficient applied (FINAL).
template <int N, bool FINAL, bool EMIT>
__global__ void __launch_bounds__(256) k_stage_lap(StageLaunch p) {
  int c;
  Ctx x;
  if (!stage_place(p, xcd_entry(p.tiles, p.swz), N, c, x)) return;
  int id[hl::kCells];
  load_cells(p.rec, c, id);
  LapOut<N> o;
  laplacian<N>(p.q, FINAL ? p.q.idv : p.q.idv4, x, id, p.x, o);
  const size_t e0 = (size_t)(3 * c) * x.L + x.k;
#pragma unroll
  for (int K = 0; K < 3; ++K) {
    if constexpr (FINAL) {
#pragma unroll
      for (int i = 0; i < N; ++i)
        o.e[K][i] = ((x.k + i < p.q.ml) ? p.q.cv4 : 0.0) * o.e[K][i];
    }
    st<N>(p.y + e0 + K * x.L, o.e[K]);
  }
  if constexpr (EMIT) {
#pragma unroll
    for (int w = 0; w < 2; ++w) st<N>(p.d.vdel2_rv_v + (size_t)(2 * c + w) * x.L + x.k, o.curl[w]);
    st<N>(p.d.vdel2_div_c + (size_t)c * x.L + x.k, o.div);
  }
}

template <int N, int LX, int TW, int TH, bool D2, bool D4, bool EMIT>
__global__ void __launch_bounds__(LX *TW *TH) __attribute__((amdgpu_waves_per_eu(N == 2 ? 3 : 4)))
    k_stage_tile(TileLaunch p) {
  using R = TileRows<N, LX, TW, TH, D4>;
  __shared__ double h[R::ROWS], ratio[R::ROWS], lap[R::LAPS];
  __shared__ int ids[R::PLACES];
  stage_tile<N, LX, TW, TH, D2, D4, EMIT>(p, xcd_entry(p.work, p.swz), (int)blockIdx.y * p.per_block, h,
                                          ratio, lap, ids);
}

// Ensemble form (k_batch_mom); tiles of all shapes share the LDS.  D4: some
// member has del4 (without it the bodies leave room for four waves per SIMD).
template <int N, int LX, int TW, int TH, int D2, bool D4, bool EMIT>
__device__ __forceinline__ void batch_tile(const TileLaunch &p, int entry, char *mem) {
  auto body = [&](auto D2_, auto D4_) {
    constexpr bool d2 = decltype(D2_)::value, d4 = decltype(D4_)::value;
    // without del4 there is no Laplacian to emit
    auto &r = *reinterpret_cast<TileRows<N, LX, TW, TH, d4> *>(mem);
    stage_tile<N, LX, TW, TH, d2, d4, EMIT && d4>(p, entry, 0, r.h, r.ratio, r.lap, r.ids);
  };
  constexpr std::true_type yes{};
  constexpr std::false_type no{};
  if constexpr (D2 != kAny) {
    body(std::bool_constant<D2 != 0>{}, std::bool_constant<D4>{});
  } else {
    const bool d2 = p.a.terms & T_TDEL2;
    if (D4 && (p.a.terms & T_TDEL4)) {
      if (d2) body(yes, std::bool_constant<D4>{});
      else body(no, std::bool_constant<D4>{});
    } else if (d2) {
      body(yes, no);
    } else {
      body(no, no);
    }
  }
}

template <int N, int LX, int D2, bool D4, bool EMIT>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(N == 2 && (D4 || D2 != kAny) ? 3 : 4)))
    k_batch_tile(const TileLaunch *__restrict__ desc, const int *__restrict__ who) {
  constexpr size_t of[3] = {sizeof(TileRows<N, 4, 8, 8, D4>), sizeof(TileRows<N, 2, 16, 8, D4>),
                            sizeof(TileRows<N, 1, 16, 16, D4>)};
  __shared__ alignas(16) char mem[LX == 4 ? of[0] : LX == 2 ? of[1] : LX == 1 ? of[2]
                                                                  : std::max({of[0], of[1], of[2]})];
  const int w = uniform(who[blockIdx.x]);
  if (w < 0) return;
  const TileLaunch &p = constant_at(desc, w);
  const int entry = block_entry((int)blockIdx.x - p.block0, p.work, p.swz);
  if (LX == 4 || (LX == kAny && p.lx == 4)) batch_tile<N, 4, 8, 8, D2, D4, EMIT>(p, entry, mem);
  else if (LX == 2 || (LX == kAny && p.lx == 2)) batch_tile<N, 2, 16, 8, D2, D4, EMIT>(p, entry, mem);
  else batch_tile<N, 1, 16, 16, D2, D4, EMIT>(p, entry, mem);
}

using StageFn = void (*)(StageLaunch);

template <int N, bool EMIT> StageFn pick_mom(bool v2, bool v4) {
  if (v4) return v2 ? k_stage_mom<N, true, true, EMIT> : k_stage_mom<N, false, true, EMIT>;
  return v2 ? k_stage_mom<N, true, false, EMIT> : k_stage_mom<N, false, false, EMIT>;
}

template <int N> StageFn pick_pre(bool v2, bool v4) {
  if (v4) return v2 ? k_stage_mom_pre<N, true, true> : k_stage_mom_pre<N, false, true>;
  return v2 ? k_stage_mom_pre<N, true, false> : k_stage_mom_pre<N, false, false>;
}

// without del4 there is no Laplacian to emit
template <int N, int LX, int TW, int TH, bool EMIT> auto pick_shape(bool d2, bool d4) {
  if (d4)
    return d2 ? k_stage_tile<N, LX, TW, TH, true, true, EMIT>
              : k_stage_tile<N, LX, TW, TH, false, true, EMIT>;
  return d2 ? k_stage_tile<N, LX, TW, TH, true, false, false>
            : k_stage_tile<N, LX, TW, TH, false, false, false>;
}
template <int N, bool EMIT> auto pick_tile_of(int lx, bool d2, bool d4) {
  if (lx == 4) return pick_shape<N, 4, 8, 8, EMIT>(d2, d4);
  if (lx == 2) return pick_shape<N, 2, 16, 8, EMIT>(d2, d4);
  return pick_shape<N, 1, 16, 16, EMIT>(d2, d4);
}
auto pick_tile(int N, int lx, bool d2, bool d4, bool emit) {
  if (N == 2) return emit ? pick_tile_of<2, true>(lx, d2, d4) : pick_tile_of<2, false>(lx, d2, d4);
  return emit ? pick_tile_of<1, true>(lx, d2, d4) : pick_tile_of<1, false>(lx, d2, d4);
}

constexpr int kTileThreads = 256; // every tile shape's

} // namespace

int stage_levels(const MeshView &m, const Launch &lc) {
  return lc.lpt == 2 && m.L % 2 == 0 ? 2 : 1;
}

void stage_launch(const MeshView &m, const Launch &lc, int N, const HexCoef &q, const StageArgs &a,
                  const DiagOut &d, StageLaunch &p, TileLaunch &t) {
  const int lanes = (m.L + N - 1) / N;
  // lanes per cell and block: up to 16 (32 levels), so that a block's cells
  // share more of their neighbours' rows in L1 (2.81 against 2.85 ms per step
  // for momentum alone at nx=512, 64 layers with 32, 2.94 with 8)
  const int want = lc.chunk > 0 ? std::min(std::max(1, lc.chunk / N), 64) : 16;
  const int nch = (lanes + want - 1) / want;
  p = StageLaunch{};
  p.q = q;
  p.rec = m.hexc;
  p.nc = m.nc;
  p.L = m.L;
  p.lx = (lanes + nch - 1) / nch;
  p.rows = lc.rows > 0 ? std::min(lc.rows, 256 / p.lx) : 256 / p.lx;
  p.ncb = (m.nc + p.rows - 1) / p.rows;
  p.tiles = p.ncb * nch;
  p.swz = lc.swizzle;
  p.a = a;
  p.d = d;
  t = TileLaunch{};
  if (a.ntr <= 0) return;
  const TileView &tv = m.tile;
  t.q = q;
  t.ids = tv.ids;
  t.nx = tv.nx;
  t.ny = tv.ny;
  t.tiles_x = (tv.nx + tv.tw - 1) / tv.tw;
  t.nch = (lanes + tv.lx - 1) / tv.lx;
  t.work = t.tiles_x * ((tv.ny + tv.th - 1) / tv.th) * t.nch;
  t.nc = m.nc;
  t.L = m.L;
  t.per_block = a.ntr;
  t.lx = tv.lx;
  t.swz = lc.swizzle;
  t.a = a;
  t.d = d;
}

bool stage_shares_launch(const MeshView &m, const Launch &lc, int terms, int ntr) {
  if (ntr <= 0 || (terms & T_VDEL4)) return false;
  StageArgs a{};
  a.ntr = ntr;
  const int N = stage_levels(m, lc);
  StageLaunch p;
  TileLaunch t;
  stage_launch(m, lc, N, HexCoef{}, a, DiagOut{}, p, t);
  return stage_one_launch(N, p, t);
}

void launch_stage_hex(const MeshView &m, const Launch &lc, const HexCoef &q, const StageArgs &a,
                      const DiagOut &d, bool emit, hipStream_t s, const PreOut *pre) {
  TimerScope ts("tend", s);
  const int N = stage_levels(m, lc);
  OMEGA_REQUIRE(!pre || emit, "stage launch: the VJP rows come with the diagnostics");
  StageLaunch p;
  TileLaunch t;
  stage_launch(m, lc, N, q, a, d, p, t);
  const dim3 grid(p.tiles), block(p.lx * p.rows);
  const bool v4 = a.terms & T_VDEL4;
  if (v4) {
    p.x = a.vn.in;
    p.y = d.vdel2_e;
    hipLaunchKernelGGL((N == 2 ? k_stage_lap<2, false, false> : k_stage_lap<1, false, false>), grid,
                       block, 0, s, p);
    p.x = d.vdel2_e;
    p.y = d.vdel4_e;
    const StageFn k = N == 2 ? (emit ? k_stage_lap<2, true, true> : k_stage_lap<2, true, false>)
                             : (emit ? k_stage_lap<1, true, true> : k_stage_lap<1, true, false>);
    hipLaunchKernelGGL(k, grid, block, 0, s, p);
    p.x = d.vdel4_e;
  }
  const bool v2 = a.terms & T_VDEL2, d2 = a.terms & T_TDEL2, d4 = a.terms & T_TDEL4;
  if (pre) p.pre = *pre;
  const StageFn k = pre      ? (N == 2 ? pick_pre<2>(v2, v4) : pick_pre<1>(v2, v4))
                    : N == 2 ? (emit ? pick_mom<2, true>(v2, v4) : pick_mom<2, false>(v2, v4))
                             : (emit ? pick_mom<1, true>(v2, v4) : pick_mom<1, false>(v2, v4));
  if (a.ntr > 0 && !v4 && launch_stage_both(N, m.tile.lx, p, t, emit, pre != nullptr, s)) return;
  hipLaunchKernelGGL(k, grid, block, 0, s, p);
  if (a.ntr > 0) {
    // one block takes all tracers of its tile, keeping the tile's thicknesses
    // and velocities (6.3 against 7.5 ms per step at nx=512, 4 tracers);
    // where the tiles alone leave the chip short of blocks each tracer has
    // its own
    if (t.work < kFewTiles) t.per_block = 1;
    hipLaunchKernelGGL(pick_tile(N, m.tile.lx, d2, d4, emit),
                       dim3(t.work, (a.ntr + t.per_block - 1) / t.per_block), dim3(kTileThreads), 0,
                       s, t);
  }
  OMEGA_HIP_CHECK(hipGetLastError());
}

// The momentum body without its update: one launch instead of two, and the
// adjoint's PV pass then reads the edges-on-edge sums instead of forming them
// (step adjoint at nx=256, 64 layers, 1 tracer: 2286 -> 2272 us).  The tracers'
// Laplacian comes along in the same launch (6-step gradient at 1920 cells, 20
// layers: 1600 -> 1557 us) but is not worth a tile launch of its own, nor with
// two levels per lane one in which a block takes all tracers of its tile: us
// per tendency VJP with tracer del4, 64 layers, 102 against 105 at 2304 cells,
// 2 tracers, but 107, 115, 134 against 106, 113, 127 at 4096 cells, 1, 2 and 4.
bool launch_stage_rows(const MeshView &m, const Launch &lc, const HexCoef &q, StageArgs a,
                       const DiagOut &d, const PreOut &pre, hipStream_t s) {
  a.epi = EPI_NONE;
  a.base_from_tend = 0;
  // only tracer del4 needs a diagnostic of the tracers
  if (!(a.terms & T_TDEL4)) a.ntr = 0;
  if (a.ntr > 0) {
    StageLaunch p;
    TileLaunch t;
    const int N = stage_levels(m, lc);
    stage_launch(m, lc, N, q, a, d, p, t);
    if ((a.terms & T_VDEL4) || !stage_one_launch(N, p, t)) return false;
    if (N == 2 && t.work >= kFewTiles) return false;
  }
  launch_stage_hex(m, lc, q, a, d, true, s, &pre);
  return true;
}

namespace {
using BatchMomFn = void (*)(const StageLaunch *, const int *);
using BatchTileFn = void (*)(const TileLaunch *, const int *);

template <int N, bool EMIT> BatchMomFn pick_batch_mom(const StageKind &k) {
  if (k.v2 == kAny) return k_batch_mom<N, kAny, EMIT>;
  return k.v2 ? k_batch_mom<N, 1, EMIT> : k_batch_mom<N, 0, EMIT>;
}
template <int N, int LX> BatchTileFn pick_batch_shape(int d2, bool d4, bool emit) {
  if (!d4) return d2 ? k_batch_tile<N, LX, 1, false, false> : k_batch_tile<N, LX, 0, false, false>;
  if (emit) return d2 ? k_batch_tile<N, LX, 1, true, true> : k_batch_tile<N, LX, 0, true, true>;
  return d2 ? k_batch_tile<N, LX, 1, true, false> : k_batch_tile<N, LX, 0, true, false>;
}
template <int N> BatchTileFn pick_batch_tile(const StageKind &k, bool emit) {
  if (k.lx == 4) return pick_batch_shape<N, 4>(k.d2, k.d4, emit);
  if (k.lx == 2) return pick_batch_shape<N, 2>(k.d2, k.d4, emit);
  if (k.lx == 1) return pick_batch_shape<N, 1>(k.d2, k.d4, emit);
  if (!k.d4) return k_batch_tile<N, kAny, kAny, false, false>;
  return emit ? k_batch_tile<N, kAny, kAny, true, true> : k_batch_tile<N, kAny, kAny, true, false>;
}
} // namespace

void launch_stage_batch(const StageKind &k, const StageLaunch *desc, const int *who, int n, bool emit,
                        hipStream_t s) {
  TimerScope ts("batch_tend", s);
  const BatchMomFn f = k.N == 2 ? (emit ? pick_batch_mom<2, true>(k) : pick_batch_mom<2, false>(k))
                                : (emit ? pick_batch_mom<1, true>(k) : pick_batch_mom<1, false>(k));
  hipLaunchKernelGGL(f, dim3(n), dim3(256), 0, s, desc, who);
  OMEGA_HIP_CHECK(hipGetLastError());
}

void launch_tile_batch(const StageKind &k, const TileLaunch *desc, const int *who, int n, bool emit,
                       hipStream_t s) {
  TimerScope ts("batch_tracers", s);
  const BatchTileFn f = k.N == 2 ? pick_batch_tile<2>(k, emit) : pick_batch_tile<1>(k, emit);
  hipLaunchKernelGGL(f, dim3(n), dim3(kTileThreads), 0, s, desc, who);
  OMEGA_HIP_CHECK(hipGetLastError());
}

} // namespace omega_hip
