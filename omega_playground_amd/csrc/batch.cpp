// Ensembles (no reference counterpart): independent members -- each its own
// mesh, layer count, tracer count, coefficients and time step -- advanced
// together.  Members on the stage kernels without stored diagnostics
// (kernels_stage.hip) have one momentum and one tracer launch per stage and
// number of levels per lane (16 mixed members, 64 layers at most, LSRK5: 2.05
// -> 0.97 ms per step against the launches below).  For the others every stage
// phase (diagnostics, momentum del4 pre-pass, tendency + update) is one launch
// over all members' blocks, driven by a
// table of per-member descriptors built once per (step parity, stage); the
// step can be captured in a HIP graph.  The stage updates are the fused
// epilogues of the single-model steppers (rk4.cpp:28-104, lsrk.cpp:36-89),
// so each member advances bit for bit as it would alone.
#include <algorithm>
#include <cstdlib>
#include <fstream>
#include <map>
#include <sstream>

#include "batch.hpp"
#include "objects.hpp"
#include "stage_launch.hpp"

using namespace omega_hip;

struct omega_batch_s {
  int kind = OMEGA_STEPPER_LSRK;
  int nstages = 5;
  std::vector<Real> rka, rkb, rkc;
  struct Member {
    omega_model_s *M;
    omega_state_s *S;
    double dt;
    int cur0 = 0;                    // state buffer at parity 0
    DBuf<Real> acc[3], p1[3], p2[3]; // RK4
    DBuf<Real> tend[3];              // LSRK
    uint64_t gen = 0;                // model configuration the tables hold
    omega_model_s::DiagSet diag;     // where an earlier member has the same model
  };
  std::vector<std::unique_ptr<Member>> mem;
  int N = 2;         // levels per lane
  int threads = 256; // threads per block
  int per_cu = 0;    // persistent grid: blocks per CU (0: one block per entry)
  bool built = false;
  int parity = 0;
  // one table over all members; member kinds share each launch
  int nblocks = 0; // entries of a stage's first launches, ntable in the table
  int ntable = 0;
  int kinds = 0; // bit 0 general-kernel members, bit 1 pattern-specialised
  int tset = 0;  // term set compiled into the pair tendency launch (0: none)
  bool any_vdel4 = false;
  DBuf<int> blk;
  DBuf<BatchMember> desc; // [parity][stage][member]
  // members on the stage kernels without stored diagnostics, by the levels per
  // lane of their launches; the tables above hold the others
  struct Group {
    StageKind kind;
    std::vector<int> members;
    int nmom = 0, ntile = 0;     // blocks of the two launches
    DBuf<int> wmom, wtile;       // member (of the group) of each block, -1: none
    DBuf<StageLaunch> mom;       // [parity][stage][member]
    DBuf<TileLaunch> tile;
  };
  std::vector<std::unique_ptr<Group>> groups;
  // where there are both, the groups' launches run beside the others' on a
  // stream of the batch's own, from fork to join
  hipStream_t side = nullptr;
  hipEvent_t fork = nullptr, join = nullptr;
  bool use_graph = false;
  std::map<int, hipGraphExec_t> graphs;
  // omega_batch_adjoint_run's stacked mesh, model, stepper and states, kept
  // for the next call within kKeepBytes, and what they were built for
  std::shared_ptr<void> stacked;
  struct StackedFor {
    uint64_t mesh = 0;
    int M = 0, ntr = 0, terms = 0;
    omega_params params{};
  } stacked_for;

  ~omega_batch_s() {
    drop_graphs();
    if (side) {
      (void)hipStreamSynchronize(side);
      (void)hipStreamDestroy(side);
    }
    for (hipEvent_t e : {fork, join})
      if (e) (void)hipEventDestroy(e);
  }
  void drop_graphs() { destroy_graphs(graphs); }
};

namespace {

// Blocks of the persistent grid (0: one block per table entry).
int persistent_blocks(const omega_batch_s *B) {
  if (B->per_cu <= 0) return 0;
  static int cus = 0;
  if (!cus) {
    int dev = 0;
    OMEGA_HIP_CHECK(hipGetDevice(&dev));
    OMEGA_HIP_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  }
  return B->per_cu * cus;
}

bool odd_flip(const omega_batch_s *B) {
  return B->kind == OMEGA_STEPPER_LSRK && (B->nstages % 2 == 1);
}

// Buffers of state field f at buffer index c (allocating the second buffer).
Real *state_buf(omega_state_s *S, int c, int f) {
  if (c != S->cur) return S->alt(f);
  return S->ptr(f);
}

// Which members run the stage kernels without stored diagnostics (their
// coefficients in coef), in launches of their own beside those of the others.
//
// Where there are others and all members together are less than one round of
// resident blocks (512, of 512 cells and levels), the others' launches take
// them along at no cost, and a member of a few blocks next to them stays on
// one XCD; us per LSRK5 step, a general member of 144 cells, 8 layers, with 16
// lattice members of 576 cells, 16 layers: 295 so, 331 in launches of their
// own (147000 cells and levels); 4 general members of 2304 cells, 16 layers
// with 8 lattice members of 256 cells, 16 layers 394 and 397 (180000), of 1024
// cells, 32 layers 685 and 437 (410000).
std::vector<char> grouped_members(const omega_batch_s *B, std::vector<HexCoef> &coef) {
  const size_t nm = B->mem.size();
  std::vector<char> in(nm, 0);
  coef.resize(nm);
  size_t work = 0;
  bool others = false;
  for (size_t i = 0; i < nm; ++i) {
    const omega_model_s *M = B->mem[i]->M;
    in[i] = !(M->terms & T_VDEL4) && M->stage_coef(coef[i]);
    others = others || !in[i];
    work += (size_t)M->mesh->dm.host.ncells * M->mesh->dm.host.nlayers;
  }
  if (others && work < 512 * 512) std::fill(in.begin(), in.end(), 0);
  return in;
}

// Where member i's diagnostics go: to its model's buffers, or, if an earlier
// member has the same model, to buffers of its own (the launches step both).
DiagOut member_diag(omega_batch_s *B, int i) {
  omega_model_s *M = B->mem[i]->M;
  DiagOut d = M->diag();
  bool shared = false;
  for (int j = 0; j < i; ++j) shared = shared || B->mem[j]->M == M;
  if (!shared) return d;
  auto own = [](DBuf<Real> &b, const DBuf<Real> &like) {
    if (b.n != like.n) b.alloc(like.n);
    return b.p;
  };
  omega_model_s::DiagSet &s = B->mem[i]->diag;
  d.rvort_v = own(s.rvort_v, M->rvort_v);
  d.inv_thick_v = own(s.inv_thick_v, M->inv_thick_v);
  d.ke_c = own(s.ke_c, M->ke_c);
  d.div_c = own(s.div_c, M->div_c);
  d.trdel2_c = own(s.trdel2_c, M->trdel2_c);
  d.vdel2_e = own(s.vdel2_e, M->vdel2_e);
  d.vdel2_rv_v = own(s.vdel2_rv_v, M->vdel2_rv_v);
  d.vdel2_div_c = own(s.vdel2_div_c, M->vdel2_div_c);
  return d;
}

void build_tables(omega_batch_s *B) {
  OMEGA_REQUIRE(!B->mem.empty(), "batch: no members");
  // a build that fails leaves neither tables to step with nor graphs that
  // read the ones freed below
  B->built = false;
  B->drop_graphs();
  const int nm = (int)B->mem.size(), ns = B->nstages, N = B->N, T = B->threads;
  std::vector<int> blk;
  std::vector<BatchMember> geo(nm);
  std::vector<int> own(nm, -1); // group of a member on the stage kernels
  std::vector<HexCoef> coef;
  const std::vector<char> grouped = grouped_members(B, coef);
  B->groups.clear();
  B->any_vdel4 = false;
  for (int i = 0; i < nm; ++i) {
    auto &mb = *B->mem[i];
    omega_model_s *M = mb.M;
    omega_state_s *S = mb.S;
    const HostMesh &hm = M->mesh->dm.host;
    OMEGA_REQUIRE(N == 1 || hm.nlayers % 2 == 0,
                  "batch: two levels per lane need an even layer count in every member");
    M->mesh->dm.upload();
    if (M->terms & T_VDEL4) ensure_vdel4(M);
    for (int f = 0; f < 3; ++f) (void)S->alt(f);
    if (B->kind == OMEGA_STEPPER_RK4) {
      ensure3(mb.acc, S);
      ensure3(mb.p1, S);
      ensure3(mb.p2, S);
    } else {
      ensure3(mb.tend, S);
    }
    mb.cur0 = S->cur;
    mb.gen = M->gen;
    if (grouped[i]) {
      const MeshView mv = M->view();
      const bool v2 = M->terms & T_VDEL2, d2 = M->terms & T_TDEL2, d4 = M->terms & T_TDEL4;
      StageKind k{stage_levels(mv, M->lc), v2, mv.tile.lx, d2, d4};
      size_t j = 0;
      while (j < B->groups.size() && B->groups[j]->kind.N != k.N) ++j;
      if (j == B->groups.size()) {
        B->groups.push_back(std::make_unique<omega_batch_s::Group>());
        B->groups[j]->kind = k;
      }
      StageKind &g = B->groups[j]->kind;
      if (g.v2 != k.v2) g.v2 = kAny;
      if (g.lx != k.lx || g.d2 != k.d2 || g.d4 != k.d4) {
        g.lx = g.d2 = kAny;
        g.d4 = g.d4 || k.d4;
      }
      B->groups[j]->members.push_back(i);
      own[i] = (int)j;
      continue;
    }
    BatchMember &g = geo[i];
    // 16 or 32 layers run the pattern kernels with several cells per
    // wavefront, which needs two levels per lane
    g.hex = hex_usable(M->mesh->dm.view(), M->lc) && !general_only(M) &&
                    (hm.nlayers % 64 == 0 || N == 2)
                ? 1
                : 0;
    if (g.hex) {
      // one row of lanes covers 64 levels (or all 16 / 32); the pair form
      // (64-level rows, N = 2) needs an even row count, which every
      // admissible block size gives
      const int span = hm.nlayers % 64 == 0 ? 64 : hm.nlayers;
      g.lx = span / N;
      g.rows = std::max(1, T / g.lx);
      g.chunks = hm.nlayers / span;
    } else {
      int lanes = (hm.nlayers + N - 1) / N;
      if (lanes > 64) lanes = 64;
      int lx = 1;
      while (lx < lanes) lx <<= 1;
      g.lx = lx;
      g.rows = std::max(1, T / lx);
      g.chunks = (hm.nlayers + lx * N - 1) / (lx * N);
    }
    g.block0 = (int)blk.size();
    const int nb = ((hm.ncells + g.rows - 1) / g.rows) * g.chunks;
    blk.insert(blk.end(), nb, i);
    const bool do_vn = !M->params.disable_vn_tendency;
    const int ntr = M->params.ntracers;
    const bool need_diag = do_vn || ((M->terms & T_TDEL4) && ntr > 0);
    g.dterms = need_diag ? (do_vn ? M->terms : (M->terms & T_TDEL4)) : 0;
    g.vdel4 = do_vn && (M->terms & T_VDEL4);
    B->any_vdel4 = B->any_vdel4 || g.vdel4;
  }
  B->nblocks = B->ntable = (int)blk.size();
  B->kinds = 0;
  for (int i = 0; i < nm; ++i)
    if (own[i] < 0) B->kinds |= geo[i].hex ? 2 : 1;
  // the members' term set, compiled into the tendency launch when they all
  // share it (the 64k-layer members' pair operators also need the
  // shared-coefficient, 32-bit-offset forms and the vertex-union records)
  B->tset = 0;
  if (B->kinds == 2 && N == 2) {
    int ts = 0;
    bool ok = true;
    for (int i = 0; i < nm && ok; ++i) {
      if (own[i] >= 0) continue;
      omega_model_s *M = B->mem[i]->M;
      const MeshView v = M->view();
      const ModelCoef c = M->coef();
      const bool pair = M->mesh->dm.host.nlayers % 64 == 0;
      ok = v.term_sets && (!pair || (v.coef_uni && c.uniform && v.off32 && v.hexu_ok)) &&
           !M->params.disable_h_tendency && !M->params.disable_vn_tendency &&
           term_set_batch(M->terms) && (ts == 0 || ts == M->terms);
      ts = M->terms;
    }
    if (ok) B->tset = ts;
  }
  // entries of the groups' launches
  struct Tables {
    std::vector<StageLaunch> mom;
    std::vector<TileLaunch> tile;
    std::vector<int> wmom, wtile;
  };
  std::vector<Tables> gt(B->groups.size());
  std::vector<int> place(nm, 0);
  for (size_t j = 0; j < gt.size(); ++j) {
    const std::vector<int> &mem = B->groups[j]->members;
    gt[j].mom.resize((size_t)2 * ns * mem.size());
    gt[j].tile.resize((size_t)2 * ns * mem.size());
    for (size_t q = 0; q < mem.size(); ++q) place[mem[q]] = (int)q;
  }
  std::vector<DiagOut> diag(nm);
  for (int i = 0; i < nm; ++i) diag[i] = member_diag(B, i);
  std::vector<BatchMember> tab((size_t)2 * ns * nm);
  for (int p = 0; p < 2; ++p)
    for (int s = 0; s < ns; ++s)
      for (int i = 0; i < nm; ++i) {
        auto &mb = *B->mem[i];
        omega_model_s *M = mb.M;
        omega_state_s *S = mb.S;
        BatchMember g = geo[i];
        g.m = M->view();
        g.mc = M->coef();
        g.d = diag[i];
        StageArgs a{};
        a.terms = M->terms;
        a.do_h = !M->params.disable_h_tendency;
        a.do_vn = !M->params.disable_vn_tendency;
        a.ntr = M->params.ntracers;
        const double dt = mb.dt;
        if (B->kind == OMEGA_STEPPER_RK4) {
          // rk4_fused_step's buffer rotation
          const int c = mb.cur0;
          Real *Y[3], *A[3], *P1[3], *P2[3];
          for (int f = 0; f < 3; ++f) {
            Y[f] = state_buf(S, c, f);
            A[f] = mb.acc[f].p;
            P1[f] = mb.p1[f].p;
            P2[f] = mb.p2[f].p;
          }
          a.base_from_tend = 0;
          a.db = dt * B->rkb[s];
          a.da = s < 3 ? dt * B->rka[s] : 0.0;
          Real **in = s == 0 ? Y : (s == 2 ? P2 : P1);
          Real **out = s == 0 ? P1 : (s == 1 ? P2 : (s == 2 ? P1 : Y));
          a.epi = s == 0 ? EPI_RK4_FIRST : (s == 3 ? EPI_RK4_LAST : EPI_RK4_MID);
          a.h = fio(in[0], nullptr, A[0], Y[0], out[0]);
          a.vn = fio(in[1], nullptr, A[1], Y[1], out[1]);
          a.tr = fio(in[2], nullptr, A[2], Y[2], out[2]);
        } else {
          // lsrk_fused_step: stage s reads buffer (cur0 ^ parity ^ s) and
          // writes the other one
          const int steps_parity = odd_flip(B) ? p : 0;
          const int cin = (mb.cur0 ^ steps_parity ^ (s & 1)) & 1;
          a.epi = EPI_LSRK;
          a.a = B->rka[s];
          a.base_from_tend = B->rka[s] != 0.0;
          a.db = dt * B->rkb[s];
          Real *in[3], *out[3];
          for (int f = 0; f < 3; ++f) {
            in[f] = state_buf(S, cin, f);
            out[f] = state_buf(S, 1 - cin, f);
          }
          a.h = fio(in[0], mb.tend[0].p, nullptr, nullptr, out[0]);
          a.vn = fio(in[1], mb.tend[1].p, nullptr, nullptr, out[1]);
          a.tr = fio(in[2], mb.tend[2].p, nullptr, nullptr, out[2]);
        }
        if (own[i] >= 0) {
          Tables &T = gt[own[i]];
          const size_t ng = B->groups[own[i]]->members.size();
          const size_t at = ((size_t)p * ns + s) * ng + place[i];
          stage_launch(g.m, M->lc, B->groups[own[i]]->kind.N, coef[i], a, g.d, T.mom[at], T.tile[at]);
          whole_blocks(T.mom[at]);
          continue;
        }
        g.a = a;
        tab[((size_t)p * ns + s) * nm + i] = g;
      }
  for (size_t j = 0; j < gt.size(); ++j) {
    omega_batch_s::Group &G = *B->groups[j];
    // Each member's entries start at a multiple of 8, so that its share of
    // every XCD is the one of a launch of its own (one range over all members
    // left the XCD of the many-tracer ones behind: 16 mixed members, 2.4
    // million cells and levels, 1 to 4 tracers, 1231 -> 1012 us per step); most
    // tracers per tile first, so that the last blocks are short ones.
    Tables &T = gt[j];
    const size_t ng = G.members.size();
    std::vector<int> order(ng);
    for (size_t q = 0; q < ng; ++q) order[q] = (int)q;
    std::stable_sort(order.begin(), order.end(), [&](int x, int y) {
      return B->mem[G.members[x]]->M->params.ntracers > B->mem[G.members[y]]->M->params.ntracers;
    });
    for (int q : order) {
      T.wmom.resize((T.wmom.size() + 7) / 8 * 8, -1);
      T.wtile.resize((T.wtile.size() + 7) / 8 * 8, -1);
      for (size_t t = q; t < T.mom.size(); t += ng) {
        T.mom[t].block0 = (int)T.wmom.size();
        T.tile[t].block0 = (int)T.wtile.size();
      }
      T.wmom.insert(T.wmom.end(), T.mom[q].tiles, q);
      T.wtile.insert(T.wtile.end(), T.tile[q].work, q);
      B->nblocks += T.mom[q].tiles;
    }
    G.nmom = (int)gt[j].wmom.size();
    G.ntile = (int)gt[j].wtile.size();
    G.wmom.upload(gt[j].wmom);
    G.wtile.upload(gt[j].wtile);
    G.mom.upload(gt[j].mom);
    G.tile.upload(gt[j].tile);
  }
  B->blk.upload(blk);
  if (B->desc.n != tab.size()) B->desc.alloc(tab.size());
  OMEGA_HIP_CHECK(hipMemcpy(B->desc.p, tab.data(), tab.size() * sizeof(BatchMember),
                            hipMemcpyHostToDevice));
  if (!B->groups.empty() && B->ntable) {
    if (!B->fork) OMEGA_HIP_CHECK(hipEventCreateWithFlags(&B->fork, hipEventDisableTiming));
    if (!B->join) OMEGA_HIP_CHECK(hipEventCreateWithFlags(&B->join, hipEventDisableTiming));
    if (!B->side) OMEGA_HIP_CHECK(hipStreamCreateWithFlags(&B->side, hipStreamNonBlocking));
  }
  B->parity = 0;
  B->built = true;
}

// The tables hold buffer addresses for the states' current buffer parity
// and each member's model configuration; a member stepped on its own in
// between, or a model setting changed since (terms, f_vertex, launch shape,
// kernel forms: the model's configuration generation), forces a rebuild.
void ensure_tables(omega_batch_s *B) {
  bool ok = B->built;
  if (ok)
    for (auto &mbp : B->mem) {
      const auto &mb = *mbp;
      const int expect = odd_flip(B) ? (mb.cur0 ^ B->parity) : mb.cur0;
      if (mb.S->cur != expect || mb.gen != mb.M->gen) ok = false;
    }
  if (!ok) build_tables(B);
}

void step_launches(omega_batch_s *B, int parity, hipStream_t s) {
  const int nm = (int)B->mem.size();
  if (B->kind == OMEGA_STEPPER_LSRK)
    for (auto &mb : B->mem) {
      // the stage-0 input buffer of this parity is the state's current one
      omega_state_s *S = mb->S;
      const int cin = (mb->cur0 ^ (odd_flip(B) ? parity : 0)) & 1;
      const int keep = S->cur;
      S->cur = cin;
      carry_extra_tracers(mb->M, S, s);
      S->cur = keep;
    }
  const int pers = persistent_blocks(B), n = B->ntable;
  const int *g = B->blk.p;
  // Members are independent for the whole step, so the groups' launches do not
  // wait for the others' (us per LSRK5 step, a general member of 144 cells, 8
  // layers, with 16 lattice members of 1024 cells, 32 layers: 502 one after the
  // other, 388 so; of 2304 cells, 64 layers: 1136 and 850).
  const bool both = !B->groups.empty() && n;
  const hipStream_t gs = both ? B->side : s;
  if (both) {
    OMEGA_HIP_CHECK(hipEventRecord(B->fork, s));
    OMEGA_HIP_CHECK(hipStreamWaitEvent(gs, B->fork, 0));
  }
  for (int st = 0; st < B->nstages; ++st)
    for (auto &gp : B->groups) {
      // the last stage leaves its input's diagnostics in the models' buffers
      const omega_batch_s::Group &G = *gp;
      const size_t at = ((size_t)parity * B->nstages + st) * G.members.size();
      const bool emit = st + 1 == B->nstages;
      launch_stage_batch(G.kind, G.mom.p + at, G.wmom.p, G.nmom, emit, gs);
      if (G.ntile) launch_tile_batch(G.kind, G.tile.p + at, G.wtile.p, G.ntile, emit, gs);
    }
  for (int st = 0; st < B->nstages && n; ++st) {
    const BatchMember *d = B->desc.p + ((size_t)parity * B->nstages + st) * nm;
    launch_batch_diag(d, g, n, B->threads, B->N, pers, B->kinds, s);
    if (B->any_vdel4) launch_batch_vdel4(d, g, n, B->threads, B->N, pers, s);
    launch_batch_tend(d, g, n, B->threads, B->N, pers, B->kinds, B->tset, s);
  }
  if (both) {
    OMEGA_HIP_CHECK(hipEventRecord(B->join, gs));
    OMEGA_HIP_CHECK(hipStreamWaitEvent(s, B->join, 0));
  }
}

void batch_step(omega_batch_s *B, hipStream_t s) {
  ensure_tables(B);
  const int p = B->parity;
  if (B->use_graph && !stream_capturing(s)) {
    auto it = B->graphs.find(p);
    if (it == B->graphs.end()) {
      hipStream_t cs = capture_stream();
      hipGraph_t g;
      OMEGA_HIP_CHECK(hipStreamBeginCapture(cs, hipStreamCaptureModeThreadLocal));
      try {
        step_launches(B, p, cs);
      } catch (...) {
        hipGraph_t dummy;
        (void)hipStreamEndCapture(cs, &dummy);
        throw;
      }
      OMEGA_HIP_CHECK(hipStreamEndCapture(cs, &g));
      hipGraphExec_t ex;
      OMEGA_HIP_CHECK(hipGraphInstantiate(&ex, g, nullptr, nullptr, 0));
      OMEGA_HIP_CHECK(hipGraphDestroy(g));
      it = B->graphs.emplace(p, ex).first;
    }
    OMEGA_HIP_CHECK(hipGraphLaunch(it->second, s));
  } else {
    step_launches(B, p, s);
  }
  if (odd_flip(B)) {
    for (auto &mb : B->mem) mb->S->cur = 1 - mb->S->cur;
    B->parity ^= 1;
  }
}

double time_steps(omega_batch_s *B, int reps, hipStream_t s) {
  hipEvent_t a, b;
  OMEGA_HIP_CHECK(hipEventCreate(&a));
  OMEGA_HIP_CHECK(hipEventCreate(&b));
  batch_step(B, s); // warm-up (and graph capture)
  OMEGA_HIP_CHECK(hipEventRecord(a, s));
  for (int i = 0; i < reps; ++i) batch_step(B, s);
  OMEGA_HIP_CHECK(hipEventRecord(b, s));
  OMEGA_HIP_CHECK(hipEventSynchronize(b));
  float ms = 0;
  OMEGA_HIP_CHECK(hipEventElapsedTime(&ms, a, b));
  (void)hipEventDestroy(a);
  (void)hipEventDestroy(b);
  return ms / std::max(reps, 1);
}

} // namespace

extern "C" {

int omega_batch_create(int kind, int nstages, omega_batch_t *out) {
  return guarded([&] {
    OMEGA_REQUIRE(out, "null argument");
    OMEGA_REQUIRE(kind == OMEGA_STEPPER_RK4 || kind == OMEGA_STEPPER_LSRK, "bad stepper kind");
    OMEGA_REQUIRE(kind == OMEGA_STEPPER_RK4 || nstages >= 1, "nstages must be >= 1");
    auto B = std::make_unique<omega_batch_s>();
    B->kind = kind;
    B->nstages = kind == OMEGA_STEPPER_RK4 ? 4 : nstages;
    stepper_coefficients(kind, B->nstages, B->rka, B->rkb, B->rkc);
    *out = B.release();
  });
}

int omega_batch_destroy(omega_batch_t B) {
  return guarded([&] { delete B; });
}

int omega_batch_add(omega_batch_t B, omega_model_t M, omega_state_t S, double dt, int *index) {
  return guarded([&] {
    OMEGA_REQUIRE(B && M, "null argument");
    check_state(M, S, "batch member");
    OMEGA_REQUIRE(M->add_fn == nullptr,
                  "batch: members cannot have an additional-tendency hook");
    OMEGA_REQUIRE(!M->linear, "batch: linear models step on their own (omega_stepper_*)");
    for (auto &mb : B->mem)
      OMEGA_REQUIRE(mb->S != S, "batch: a state can belong to one member only");
    // two levels per lane need an even layer count in every member
    if (M->mesh->dm.host.nlayers % 2 != 0) B->N = 1;
    auto mb = std::make_unique<omega_batch_s::Member>();
    mb->M = M;
    mb->S = S;
    mb->dt = dt;
    B->mem.push_back(std::move(mb));
    B->built = false;
    if (index) *index = (int)B->mem.size() - 1;
  });
}

int omega_batch_step(omega_batch_t B, omega_stream_t stream) {
  return guarded([&] {
    OMEGA_REQUIRE(B, "null batch");
    batch_step(B, as_stream(stream));
  });
}

int omega_batch_run(omega_batch_t B, int nsteps, omega_stream_t stream) {
  return guarded([&] {
    OMEGA_REQUIRE(B, "null batch");
    OMEGA_REQUIRE(nsteps >= 0, "nsteps must be >= 0");
    for (int i = 0; i < nsteps; ++i) batch_step(B, as_stream(stream));
  });
}

int omega_batch_set_graph(omega_batch_t B, int enable) {
  return guarded([&] {
    OMEGA_REQUIRE(B, "null batch");
    B->use_graph = enable != 0;
  });
}

int omega_batch_set_launch(omega_batch_t B, int threads, int levels_per_thread) {
  return guarded([&] {
    OMEGA_REQUIRE(B, "null batch");
    OMEGA_REQUIRE(threads == 64 || threads == 128 || threads == 256,
                  "threads must be 64, 128 or 256");
    OMEGA_REQUIRE(levels_per_thread == 1 || levels_per_thread == 2,
                  "levels_per_thread must be 1 or 2");
    B->threads = threads;
    B->N = levels_per_thread;
    B->built = false;
  });
}

int omega_batch_get_launch(omega_batch_t B, int *threads, int *levels_per_thread) {
  return guarded([&] {
    OMEGA_REQUIRE(B, "null batch");
    if (threads) *threads = B->threads;
    if (levels_per_thread) *levels_per_thread = B->N;
  });
}

// Times `reps` steps for every launch shape the ensemble admits -- levels
// per lane (2, 1), threads per block (256, 128, 64: the cells per block of
// every member) and the grid (one block per table entry, or a persistent
// grid of 4, 8 or 16 blocks per CU) -- and keeps the fastest.  The members'
// states are restored afterwards, so the ensemble continues from where it
// was.  With OMEGA_TUNE_CACHE naming a file, a choice recorded there for
// the same ensemble signature (stepper, and per member: cells, layers,
// tracers, terms, kernel kind) is applied without timing, and a new choice
// is appended to it.  Where every member has the launches of its group none
// of it applies: the setting stays, is timed once and not recorded.
int omega_batch_autotune(omega_batch_t B, int reps, double *best_ms, omega_stream_t stream) {
  return guarded([&] {
    OMEGA_REQUIRE(B && !B->mem.empty(), "batch: no members");
    hipStream_t s = as_stream(stream);
    reps = std::max(1, reps);
    bool even_layers = true;
    for (auto &mb : B->mem) even_layers = even_layers && mb->M->mesh->dm.host.nlayers % 2 == 0;
    // the ensemble's signature for the tuning cache
    // (stored: with the kind that a member on the stage kernels would have on
    // the others, as in records from before they had one of their own)
    std::string sig = std::to_string(B->kind) + "/" + std::to_string(B->nstages), stored = sig;
    bool shapes = false; // some member runs the launches that have them
    std::vector<HexCoef> coef;
    const std::vector<char> in = grouped_members(B, coef);
    for (size_t i = 0; i < in.size(); ++i) {
      const auto &mb = B->mem[i];
      const HostMesh &hm = mb->M->mesh->dm.host;
      const bool hx = hex_usable(mb->M->mesh->dm.view(), mb->M->lc) && !general_only(mb->M);
      shapes = shapes || !in[i];
      const std::string member = ";" + std::to_string(hm.ncells) + ":" +
                                 std::to_string(hm.nlayers) + ":" +
                                 std::to_string(mb->M->params.ntracers) + ":" +
                                 std::to_string(mb->M->terms) + ":";
      sig += member + (in[i] ? "s" : hx ? "h" : "g");
      stored += member + (hx ? "h" : "g");
    }
    const char *cache = std::getenv("OMEGA_TUNE_CACHE");
    auto recorded = [&](const std::string &wanted) {
      std::ifstream in(cache);
      std::string line;
      while (std::getline(in, line)) {
        std::istringstream ls(line);
        std::string key;
        int n = 0, t = 0, pc = -1;
        double ms = -1;
        if (!(ls >> key >> n >> t >> pc >> ms) || key != wanted) continue;
        if ((n == 1 || (n == 2 && even_layers)) && (t == 64 || t == 128 || t == 256) && pc >= 0) {
          B->N = n;
          B->threads = t;
          B->per_cu = pc;
          B->built = false;
          if (best_ms) *best_ms = ms;
          return true;
        }
      }
      return false;
    };
    if (cache && *cache && (recorded(sig) || recorded(stored))) return;
    // save every member's state
    std::vector<std::array<DBuf<Real>, 3>> saved(B->mem.size());
    std::vector<int> cur(B->mem.size());
    for (size_t i = 0; i < B->mem.size(); ++i) {
      omega_state_s *S = B->mem[i]->S;
      cur[i] = S->cur;
      for (int f = 0; f < 3; ++f) {
        saved[i][f].alloc(S->n[f]);
        if (S->n[f])
          OMEGA_HIP_CHECK(hipMemcpyAsync(saved[i][f].p, S->ptr(f), S->n[f] * sizeof(Real),
                                         hipMemcpyDeviceToDevice, s));
      }
    }
    double best = -1;
    int bestN = B->N, bestT = B->threads, bestP = B->per_cu;
    if (!shapes) best = time_steps(B, reps, s);
    for (int N : {2, 1}) {
      if (!shapes || (N == 2 && !even_layers)) continue;
      for (int T : {256, 128, 64})
        for (int P : {0, 4, 8, 16}) {
          B->N = N;
          B->threads = T;
          B->per_cu = P;
          B->built = false;
          const double ms = time_steps(B, reps, s);
          if (best < 0 || ms < best) {
            best = ms;
            bestN = N;
            bestT = T;
            bestP = P;
          }
        }
    }
    B->N = bestN;
    B->threads = bestT;
    B->per_cu = bestP;
    B->built = false;
    // restore the states
    for (size_t i = 0; i < B->mem.size(); ++i) {
      omega_state_s *S = B->mem[i]->S;
      S->cur = cur[i];
      for (int f = 0; f < 3; ++f)
        if (S->n[f])
          OMEGA_HIP_CHECK(hipMemcpyAsync(S->ptr(f), saved[i][f].p, S->n[f] * sizeof(Real),
                                         hipMemcpyDeviceToDevice, s));
    }
    OMEGA_HIP_CHECK(hipStreamSynchronize(s));
    if (shapes && cache && *cache) {
      std::ofstream out(cache, std::ios::app);
      if (out) out << sig << " " << bestN << " " << bestT << " " << bestP << " " << best << "\n";
    }
    if (best_ms) *best_ms = best;
  });
}

int omega_batch_set_persistent(omega_batch_t B, int blocks_per_cu) {
  return guarded([&] {
    OMEGA_REQUIRE(B, "null batch");
    OMEGA_REQUIRE(blocks_per_cu >= 0 && blocks_per_cu <= 64, "blocks_per_cu must be in 0..64");
    B->per_cu = blocks_per_cu;
  });
}

int omega_batch_get_persistent(omega_batch_t B, int *blocks_per_cu) {
  return guarded([&] {
    OMEGA_REQUIRE(B && blocks_per_cu, "null argument");
    *blocks_per_cu = B->per_cu;
  });
}

int omega_batch_info(omega_batch_t B, int *nmembers, int64_t *blocks_per_launch,
                     int64_t *cell_layers) {
  return guarded([&] {
    OMEGA_REQUIRE(B, "null batch");
    if (!B->built && !B->mem.empty()) build_tables(B);
    if (nmembers) *nmembers = (int)B->mem.size();
    if (blocks_per_launch) *blocks_per_launch = B->nblocks;
    if (cell_layers) {
      int64_t n = 0;
      for (auto &mb : B->mem)
        n += (int64_t)mb->M->mesh->dm.host.ncells * mb->M->mesh->dm.host.nlayers;
      *cell_layers = n;
    }
  });
}

} // extern "C"

// ---------------------------------------------------------------------------
// Ensemble adjoint.  No operator couples one layer to another, so members
// that share a mesh, layer and tracer counts and coefficients are the
// layers of one model: member m occupies layers [m*L, (m+1)*L) of a
// stacked model with M*L layers.  The stacked model runs the checkpointed
// adjoint once, so every stage of the forward, recompute and reverse sweeps
// is one launch per kernel for the whole ensemble, the per-level arithmetic
// is that of each member alone, and the gradients of the shared
// coefficients are summed over all members by the same reductions.
// ---------------------------------------------------------------------------
namespace {

void ok(int rc) {
  if (rc != OMEGA_OK) throw Error(rc, g_last_error);
}

bool same_params(const omega_params &a, const omega_params &b) {
  return a.f0 == b.f0 && a.grav == b.grav && a.drag_coeff == b.drag_coeff &&
         a.visc_del2 == b.visc_del2 && a.visc_del4 == b.visc_del4 &&
         a.eddy_diff2 == b.eddy_diff2 && a.eddy_diff4 == b.eddy_diff4 &&
         a.ntracers == b.ntracers && a.disable_h_tendency == b.disable_h_tendency &&
         a.disable_vn_tendency == b.disable_vn_tendency;
}

// Vertex by vertex only where one of them varies: comparing equal constants took
// 7 us of the 1.1 ms of 4 steps of 8 members at 1024 cells, 16 layers.
bool same_f(const omega_model_s *a, const omega_model_s *b) {
  if (a->f_uniform && b->f_uniform) return a == b || a->f_value == b->f_value;
  return a == b || a->f_h == b->f_h;
}

// Rows of width n*L (member m at column m*L) of the stacked state <-> rows of
// width L of the members' states, all fields of up to kMany members a launch.
void stack_fields(omega_state_s *big, const std::vector<omega_state_s *> &mem, int L, bool to_big,
                  hipStream_t s) {
  const int M = (int)mem.size();
  for (int m0 = 0; m0 < M; m0 += StackArgs::kMany) {
    StackArgs a{};
    a.count = std::min(StackArgs::kMany, M - m0);
    a.first = m0;
    a.L = L;
    a.wide = M * L;
    a.to_big = to_big;
    for (int f = 0; f < 3; ++f) {
      a.n[f] = mem[m0]->n[f];
      a.big[f] = big->ptr(f);
      for (int i = 0; i < a.count; ++i) a.mem[i][f] = mem[m0 + i]->ptr(f);
    }
    launch_stack(a, s);
  }
}

struct Owned {
  omega_mesh_s *mesh = nullptr;
  omega_model_s *model = nullptr;
  omega_stepper_s *st = nullptr;
  omega_state_s *y = nullptr, *obs = nullptr, *grad = nullptr;
  int64_t bytes = 0; // device memory of all of it
  ~Owned() {
    (void)omega_state_destroy(grad);
    (void)omega_state_destroy(obs);
    (void)omega_state_destroy(y);
    (void)omega_stepper_destroy(st);
    (void)omega_model_destroy(model);
    delete mesh;
  }
};

} // namespace

extern "C" {

int omega_batch_adjoint_run(omega_batch_t B, double t0, int nsteps, int n_snapshots,
                            int64_t byte_cap, const omega_state_t *obs, const double *weights,
                            double *J, omega_state_t *grads, double *param_grad,
                            omega_stream_t stream) {
  return guarded([&] {
    OMEGA_REQUIRE(B && obs && weights && J && grads, "null argument");
    const int M = (int)B->mem.size();
    OMEGA_REQUIRE(M >= 1, "batch adjoint: the batch has no members");
    const omega_model_s *M0 = B->mem[0]->M;
    const omega_mesh_s *mesh0 = M0->mesh;
    const HostMesh &h0 = mesh0->dm.host;
    const int L = h0.nlayers, ntr = M0->params.ntracers;
    const double dt = B->mem[0]->dt;
    for (int m = 0; m < M; ++m) {
      const auto &mb = *B->mem[m];
      OMEGA_REQUIRE(mb.M->mesh == mesh0,
                    "batch adjoint: all members must share one mesh (layers are stacked)");
      OMEGA_REQUIRE(same_params(mb.M->params, M0->params) && mb.M->terms == M0->terms,
                    "batch adjoint: members must share the model parameters and terms");
      OMEGA_REQUIRE(same_f(mb.M, M0),
                    "batch adjoint: members must share the Coriolis parameter of every vertex");
      OMEGA_REQUIRE(mb.dt == dt, "batch adjoint: members must share dt");
      OMEGA_REQUIRE(!mb.M->add_fn, "batch adjoint: members must not have an additional tendency");
      OMEGA_REQUIRE(mb.S->ntr == ntr, "batch adjoint: member state tracer count differs");
      OMEGA_REQUIRE(obs[m] && obs[m]->mesh == mesh0 && obs[m]->ntr == ntr,
                    "batch adjoint: observation state does not match its member");
      OMEGA_REQUIRE(grads[m] && grads[m]->mesh == mesh0 && grads[m]->ntr == ntr,
                    "batch adjoint: gradient state does not match its member");
    }
    for (int e = 0; e < h0.nedges; ++e)
      OMEGA_REQUIRE(h0.max_level_edge_top[e] >= L,
                    "batch adjoint: stacking needs every layer active on every edge");
    OMEGA_REQUIRE((int64_t)M * L <= (1 << 20), "batch adjoint: too many stacked layers");
    hipStream_t s = as_stream(stream);

    // stacked mesh, model, stepper and states: built once for a set of members
    // and kept with the batch (their host build, allocations and frees were
    // 20 of the 21 ms of 4 steps of 8 members at 1024 cells, 16 layers)
    const omega_batch_s::StackedFor &sf = B->stacked_for;
    std::shared_ptr<Owned> o = std::static_pointer_cast<Owned>(B->stacked);
    B->stacked.reset(); // a call that fails leaves none behind
    int64_t start = device_bytes();
    if (!o || sf.mesh != mesh0->uid || sf.M != M || sf.ntr != ntr || sf.terms != M0->terms ||
        !same_params(sf.params, M0->params)) {
      o.reset();
      start = device_bytes();
      o = std::make_shared<Owned>();
      o->mesh = new omega_mesh_s();
      o->mesh->dm.host = h0;
      HostMesh &hb = o->mesh->dm.host;
      hb.nlayers = M * L;
      for (auto *v : {&hb.max_level_cell, &hb.max_level_edge_bot, &hb.max_level_edge_top,
                      &hb.max_level_vertex_bot, &hb.max_level_vertex_top})
        for (int &x : *v)
          if (x >= L) x = M * L;
      o->mesh->dm.build_device(mesh0->dm.ordering);
      ok(omega_model_create(o->mesh, &M0->params, &o->model));
      o->model->terms = M0->terms;
      ok(omega_stepper_create(o->model, B->kind, B->nstages, &o->st));
      ok(omega_state_create(o->mesh, ntr, &o->y));
      ok(omega_state_create(o->mesh, ntr, &o->obs));
      ok(omega_state_create(o->mesh, ntr, &o->grad));
    }
    if (!same_f(o->model, M0)) model_set_f(o->model, M0->f_h); // same numbering
    std::vector<omega_state_s *> members(M), wanted(obs, obs + M), out(grads, grads + M);
    for (int m = 0; m < M; ++m) members[m] = B->mem[m]->S;
    stack_fields(o->y, members, L, true, s);
    stack_fields(o->obs, wanted, L, true, s);
    // ensemble-mean misfit
    const double w[3] = {weights[0] / M, weights[1] / M, weights[2] / M};
    ok(omega_adjoint_run(o->st, t0, dt, nsteps, n_snapshots, byte_cap, o->y, o->obs, w, J, o->grad,
                         param_grad, stream));
    stack_fields(o->grad, out, L, false, s);
    OMEGA_HIP_CHECK(hipStreamSynchronize(s));
    // this call allocates for the stacked objects alone, and they only grow
    o->bytes += device_bytes() - start;
    if (o->bytes > kKeepBytes) {
      // without the snapshots it may do
      start = device_bytes();
      o->st->adj_run.reset();
      o->bytes += device_bytes() - start;
    }
    if (o->bytes <= kKeepBytes) {
      B->stacked = o;
      B->stacked_for.mesh = mesh0->uid;
      B->stacked_for.M = M;
      B->stacked_for.ntr = ntr;
      B->stacked_for.terms = M0->terms;
      B->stacked_for.params = M0->params;
    }
  });
}

} // extern "C"
