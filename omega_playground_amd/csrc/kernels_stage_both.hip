// Momentum, thickness and tracers of a stage in one launch, for models too
// small to fill the GPU with either: the first blocks run the momentum body,
// the others the tracer tiles, side by side instead of one after the other.
#include "stage_blocks.hpp"

namespace omega_hip {

namespace {

using namespace stage;

template <int N, int LX, int TW, int TH, bool V2, bool D2, bool D4, bool EMIT>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(N == 1 ? 4 : 2)))
    k_stage_both(StageLaunch p, TileLaunch t) {
  const int b = (int)blockIdx.x;
  if (b < p.tiles) {
    stage_mom<N, V2, false, EMIT>(p, b);
  } else {
    // tiles of all tracers of a group, then the next group
    const int w = b - p.tiles, group = uniform(w / t.work);
    stage_tile<N, LX, TW, TH, D2, D4, EMIT>(t, w - group * t.work, group * t.per_block);
  }
}

template <int N, int LX, int TW, int TH, bool V2, bool EMIT> auto pick4(bool d2, bool d4) {
  if (d4)
    return d2 ? k_stage_both<N, LX, TW, TH, V2, true, true, EMIT>
              : k_stage_both<N, LX, TW, TH, V2, false, true, EMIT>;
  return d2 ? k_stage_both<N, LX, TW, TH, V2, true, false, EMIT>
            : k_stage_both<N, LX, TW, TH, V2, false, false, EMIT>;
}
template <int N, int LX, int TW, int TH> auto pick3(bool v2, bool d2, bool d4, bool emit) {
  if (v2) return emit ? pick4<N, LX, TW, TH, true, true>(d2, d4) : pick4<N, LX, TW, TH, true, false>(d2, d4);
  return emit ? pick4<N, LX, TW, TH, false, true>(d2, d4) : pick4<N, LX, TW, TH, false, false>(d2, d4);
}
template <int N> auto pick2(int lx, bool v2, bool d2, bool d4, bool emit) {
  if (lx == 4) return pick3<N, 4, 8, 8>(v2, d2, d4, emit);
  if (lx == 2) return pick3<N, 2, 16, 8>(v2, d2, d4, emit);
  return pick3<N, 1, 16, 16>(v2, d2, d4, emit);
}

} // namespace

bool launch_stage_both(int N, int lx, const StageLaunch &p, const TileLaunch &t0, bool emit,
                       hipStream_t s) {
  const StageArgs &a = p.a;
  TileLaunch t = t0;
  if (t.work < kFewTiles) t.per_block = 1;
  const int groups = (a.ntr + t.per_block - 1) / t.per_block;
  // Both bodies hold the momentum's registers here: 2 blocks per CU with two
  // levels per lane, 4 with one, on 256 CUs.  Up to two rounds of those one
  // launch is faster (us per RK4 step, 64 layers, 1 tracer: 49 -> 37 at 576
  // cells, 74 -> 58 at 2304, 80 -> 80 at 4096 where it is two rounds; one
  // layer, 196608 cells, LSRK5: 97 -> 83 at one and a half), beyond them the
  // tracers miss the waves they have alone (142 -> 151 at 9216 cells).
  if (p.tiles + t.work * groups > (N == 2 ? 1024 : 2048)) return false;
  const bool v2 = a.terms & T_VDEL2, d2 = a.terms & T_TDEL2, d4 = a.terms & T_TDEL4;
  hipLaunchKernelGGL(N == 2 ? pick2<2>(lx, v2, d2, d4, emit) : pick2<1>(lx, v2, d2, d4, emit),
                     dim3(p.tiles + t.work * groups), dim3(256), 0, s, p, t);
  OMEGA_HIP_CHECK(hipGetLastError());
  return true;
}

} // namespace omega_hip
