// Momentum, thickness and tracers of a stage in one launch, for models too
// small to fill the GPU with either: the first blocks run the momentum body,
// the others the tracer tiles, side by side instead of one after the other.
#include "stage_blocks.hpp"

namespace omega_hip {

namespace {

using namespace stage;

// what else a stage leaves: nothing, its input's diagnostics, or those and
// the tendency VJP's rows
enum Leave { kNothing, kDiag, kPre };

template <int N, int LX, int TW, int TH, bool V2, bool D2, bool D4, Leave E>
__global__ void __launch_bounds__(256)
    __attribute__((amdgpu_waves_per_eu(N == 2 ? 2 : E == kPre ? 3 : 4)))
    k_stage_both(StageLaunch p, TileLaunch t) {
  const int b = (int)blockIdx.x;
  if (b < p.tiles) {
    stage_mom<N, V2, false, E != kNothing, E == kPre>(p, b);
  } else {
    // tiles of all tracers of a group, then the next group
    using R = TileRows<N, LX, TW, TH, D4>;
    __shared__ double h[R::ROWS], ratio[R::ROWS], lap[R::LAPS];
    __shared__ int ids[R::PLACES];
    const int w = b - p.tiles, group = uniform(w / t.work);
    stage_tile<N, LX, TW, TH, D2, D4, E != kNothing>(t, w - group * t.work, group * t.per_block, h,
                                                     ratio, lap, ids);
  }
}

template <int N, int LX, int TW, int TH, bool V2, Leave E> auto pick4(bool d2, bool d4) {
  if (d4)
    return d2 ? k_stage_both<N, LX, TW, TH, V2, true, true, E>
              : k_stage_both<N, LX, TW, TH, V2, false, true, E>;
  return d2 ? k_stage_both<N, LX, TW, TH, V2, true, false, E>
            : k_stage_both<N, LX, TW, TH, V2, false, false, E>;
}
template <int N, int LX, int TW, int TH, Leave E> auto pick3(bool v2, bool d2, bool d4) {
  return v2 ? pick4<N, LX, TW, TH, true, E>(d2, d4) : pick4<N, LX, TW, TH, false, E>(d2, d4);
}
template <int N, Leave E> auto pick2(int lx, bool v2, bool d2, bool d4) {
  if (lx == 4) return pick3<N, 4, 8, 8, E>(v2, d2, d4);
  if (lx == 2) return pick3<N, 2, 16, 8, E>(v2, d2, d4);
  return pick3<N, 1, 16, 16, E>(v2, d2, d4);
}
template <int N> auto pick(int lx, bool v2, bool d2, bool d4, Leave e) {
  return e == kPre    ? pick2<N, kPre>(lx, v2, d2, d4)
         : e == kDiag ? pick2<N, kDiag>(lx, v2, d2, d4)
                      : pick2<N, kNothing>(lx, v2, d2, d4);
}

} // namespace

namespace {
// blocks of the tracers: tiles times groups of per_block tracers
int tile_blocks(const TileLaunch &t, int &per_block) {
  per_block = t.work < kFewTiles ? 1 : t.per_block;
  return t.work * ((t.a.ntr + per_block - 1) / per_block);
}
} // namespace

// Both bodies hold the momentum's registers here: 2 blocks per CU with two
// levels per lane, 4 with one, on 256 CUs.  Up to two rounds of those one
// launch is faster (us per RK4 step, 64 layers, 1 tracer: 49 -> 37 at 576
// cells, 74 -> 58 at 2304, 80 -> 80 at 4096 where it is two rounds; one
// layer, 196608 cells, LSRK5: 97 -> 83 at one and a half), beyond them the
// tracers miss the waves they have alone (142 -> 151 at 9216 cells).
bool stage_one_launch(int N, const StageLaunch &p0, const TileLaunch &t) {
  int per_block;
  StageLaunch p = p0;
  whole_blocks(p);
  return p.tiles + tile_blocks(t, per_block) <= (N == 2 ? 1024 : 2048);
}

bool launch_stage_both(int N, int lx, const StageLaunch &p0, const TileLaunch &t0, bool emit, bool pre,
                       hipStream_t s) {
  if (!stage_one_launch(N, p0, t0)) return false;
  StageLaunch p = p0;
  whole_blocks(p);
  TileLaunch t = t0;
  const int blocks = p.tiles + tile_blocks(t0, t.per_block), terms = p.a.terms;
  const bool v2 = terms & T_VDEL2, d2 = terms & T_TDEL2, d4 = terms & T_TDEL4;
  const Leave e = pre ? kPre : emit ? kDiag : kNothing;
  hipLaunchKernelGGL(N == 2 ? pick<2>(lx, v2, d2, d4, e) : pick<1>(lx, v2, d2, d4, e),
                     dim3(blocks), dim3(256), 0, s, p, t);
  OMEGA_HIP_CHECK(hipGetLastError());
  return true;
}

} // namespace omega_hip
