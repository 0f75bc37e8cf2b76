// Checks of the library's host side that need no GPU: the program stands in
// for the HIP runtime (memory is host memory, a launch is noted and not run),
// so that what the host code allocates, keeps, launches and does after a
// failing call can be looked at.  Built and run by tests/test_host_side.py.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <fstream>
#include <functional>
#include <iterator>
#include <map>
#include <set>
#include <string>
#include <vector>

#include <unistd.h>

#include "batch.hpp"
#include "stage_launch.hpp"

using namespace omega_hip;

#define CHECK(cond)                                                     \
  do {                                                                  \
    if (!(cond)) {                                                      \
      std::printf("%s:%d: %s\n", __FILE__, __LINE__, #cond);            \
      std::exit(1);                                                     \
    }                                                                   \
  } while (0)

// ---------------------------------------------------------------------------
// The HIP runtime this program runs on
// ---------------------------------------------------------------------------
namespace fake {
std::map<void *, size_t> live; // device allocations
size_t bytes = 0;
int fail_after = -1; // allocations until one fails, -1: none does

struct Launched {
  dim3 grid, block;
  hipStream_t stream;
  std::vector<char> arg; // of its first argument, as many bytes as were asked for
  template <class T> T at() const {
    T x;
    std::memcpy(static_cast<void *>(&x), arg.data(), sizeof(T));
    return x;
  }
};
size_t arg_bytes = 0;
std::vector<Launched> launches;
std::map<hipGraphExec_t, int> graphs; // live executables and their replays
// streams that wait for another's work so far, with the number of launches
// before each wait
struct Wait {
  hipStream_t stream, on;
  size_t at;
};
std::vector<Wait> waits;
std::map<hipEvent_t, hipStream_t> events;
int streams = 0;
} // namespace fake

extern "C" {
hipError_t hipMalloc(void **p, size_t n) {
  if (fake::fail_after == 0) return hipErrorOutOfMemory;
  if (fake::fail_after > 0) --fake::fail_after;
  *p = std::calloc(1, n); // pages are taken when they are first written
  if (!*p) return hipErrorOutOfMemory;
  fake::live[*p] = n;
  fake::bytes += n;
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  if (!p) return hipSuccess;
  CHECK(fake::live.count(p));
  fake::bytes -= fake::live[p];
  fake::live.erase(p);
  std::free(p);
  return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemset(void *p, int v, size_t n) {
  if (v || !fake::live.count(p)) std::memset(p, v, n);
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void *, dim3 grid, dim3 block, void **args, size_t, hipStream_t s) {
  const char *a = static_cast<const char *>(args[0]);
  fake::launches.push_back({grid, block, s, std::vector<char>(a, a + fake::arg_bytes)});
  return hipSuccess;
}
static fake::Launched pushed;
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t, hipStream_t s) {
  pushed = {grid, block, s, {}};
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *shared, hipStream_t *s) {
  *grid = pushed.grid;
  *block = pushed.block;
  *shared = 0;
  *s = pushed.stream;
  return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "no GPU here"; }
hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { return *v = 256, hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *s) {
  return *s = hipStreamCaptureStatusNone, hipSuccess;
}
static char *handle() {
  static char *next = nullptr;
  return ++next;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
  ++fake::streams;
  return *s = reinterpret_cast<hipStream_t>(handle()), hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return --fake::streams, hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
  CHECK(fake::events.count(e));
  fake::waits.push_back({s, fake::events[e], fake::launches.size()});
  return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) { return *g = nullptr, hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t, hipGraphNode_t *, char *, size_t) {
  *e = reinterpret_cast<hipGraphExec_t>(handle());
  fake::graphs[*e] = 0;
  return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t e) {
  CHECK(fake::graphs.erase(e));
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t) {
  CHECK(fake::graphs.count(e));
  ++fake::graphs[e];
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) { return *e = reinterpret_cast<hipEvent_t>(handle()), hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { return fake::events.erase(e), hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { return fake::events[e] = s, hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { return *ms = 1, hipSuccess; }
}

// Tables of a lattice whose rows have as many levels as 24-bit byte strides
// hold, and one more: 8 bytes a level in a row, 24 in a cell's three edges.
static void tall() {
  for (int L : {64, 699050, 699051, 2097151, 2097152}) {
    DeviceMesh dm;
    build_planar_hex(dm.host, 6, 4, 1.0, L);
    dm.build_device(OMEGA_ORDER_HILBERT);
    std::printf("L %d off32 %d stage %d\n", L, (int)dm.off32, (int)dm.stage_ok);
    CHECK(dm.hex_ok && dm.coef_uni);
    CHECK(dm.off32 == (8.0 * L < 1 << 24));
    CHECK(dm.stage_ok == (24.0 * L < 1 << 24));
  }
}

static void ok(int rc) {
  if (rc != OMEGA_OK) std::printf("%s\n", omega_last_error());
  CHECK(rc == OMEGA_OK);
}

// An ensemble of lattice members for the stage kernels, and its parts
struct Ensemble {
  omega_mesh_t mesh = nullptr;
  std::vector<omega_model_t> models;
  std::vector<omega_state_t> states;
  omega_batch_t batch = nullptr;

  Ensemble(int members, int nx, int ny, int L, omega_params p, int kind) {
    ok(omega_mesh_create_planar_hex(nx, ny, 1e4, L, OMEGA_ORDER_HILBERT, &mesh));
    ok(omega_batch_create(kind, 5, &batch));
    for (int i = 0; i < members; ++i) {
      omega_model_t m;
      omega_state_t s;
      ok(omega_model_create(mesh, &p, &m));
      ok(omega_state_create(mesh, p.ntracers, &s));
      ok(omega_batch_add(batch, m, s, 10.0, nullptr));
      models.push_back(m);
      states.push_back(s);
    }
  }
  ~Ensemble() {
    ok(omega_batch_destroy(batch));
    for (auto s : states) ok(omega_state_destroy(s));
    for (auto m : models) ok(omega_model_destroy(m));
    ok(omega_mesh_destroy(mesh));
  }
  static omega_params params(int ntr) {
    omega_params p{};
    p.f0 = 1e-4;
    p.grav = 9.81;
    p.ntracers = ntr;
    return p;
  }
};

// The launches of f, with as many bytes of their first arguments
template <class F> static std::vector<fake::Launched> launched(size_t arg_bytes, F &&f) {
  fake::launches.clear();
  fake::arg_bytes = arg_bytes;
  f();
  fake::arg_bytes = 0;
  return fake::launches;
}

// A step whose tables cannot be rebuilt fails and leaves no graph of the old
// ones; the step after it does all of its work.
static void rebuild() {
  for (int graph : {0, 1})
    for (int fail = 0;; ++fail) {
      Ensemble e(2, 6, 4, 8, Ensemble::params(1), OMEGA_STEPPER_RK4);
      ok(omega_batch_set_graph(e.batch, graph));
      const size_t want = launched(0, [&] { ok(omega_batch_step(e.batch, nullptr)); }).size();
      fake::launches.clear();
      ok(omega_model_set_terms(e.models[1], 7 + 8)); // the tables are now out of date
      fake::fail_after = fail;
      const bool failed = omega_batch_step(e.batch, nullptr) != OMEGA_OK;
      fake::fail_after = -1;
      std::printf("graph %d, allocation %d fails: %d\n", graph, fail, (int)failed);
      if (!failed) {
        CHECK(fake::launches.size() == want && fail > 0);
        break;
      }
      CHECK(fake::graphs.empty());
      fake::launches.clear();
      ok(omega_batch_step(e.batch, nullptr));
      CHECK(fake::launches.size() == want);
    }
}

// What adjoint runs keep between calls is within its bound, 1 GiB for a
// stepper and for an ensemble.
constexpr size_t kBound = size_t(1) << 30;
static const double weights[3] = {1, 0, 1};

static void keep_stepper() {
  for (int kind : {OMEGA_STEPPER_RK4, OMEGA_STEPPER_LSRK})
    for (int L : {64, 108, 114, 120, 140}) {
      // the first call's snapshots are too many to keep
      omega_mesh_t mesh;
      omega_model_t model;
      omega_stepper_t st;
      omega_state_t y, obs, grad;
      const omega_params p = Ensemble::params(0);
      ok(omega_mesh_create_planar_hex(256, 256, 1e4, L, OMEGA_ORDER_HILBERT, &mesh));
      ok(omega_model_create(mesh, &p, &model));
      ok(omega_stepper_create(model, kind, 5, &st));
      for (omega_state_t *s : {&y, &obs, &grad}) ok(omega_state_create(mesh, 0, s));
      size_t held[2];
      for (int snaps : {12, 1}) {
        double J;
        ok(omega_adjoint_run(st, 0.0, 1.0, 12, snaps, 0, y, obs, weights, &J, grad, nullptr, nullptr));
        held[snaps == 1] = fake::bytes;
      }
      std::printf("kind %d, %d levels: %zu bytes kept\n", kind, L, held[1] - held[0]);
      CHECK(held[1] - held[0] <= kBound);
      CHECK(L > 64 || held[1] > held[0]);
      for (omega_state_t s : {y, obs, grad}) ok(omega_state_destroy(s));
      ok(omega_stepper_destroy(st));
      ok(omega_model_destroy(model));
      ok(omega_mesh_destroy(mesh));
      CHECK(fake::bytes == 0);
    }
}

static void keep_ensemble() {
  for (int kind : {OMEGA_STEPPER_RK4, OMEGA_STEPPER_LSRK})
    for (int ntr : {1, 4})
      for (int L : {8, 24, 32, 40, 56, 64}) {
        omega_params p = Ensemble::params(ntr);
        p.visc_del4 = 1;
        p.eddy_diff4 = 1;
        Ensemble e(4, 64, 64, L, p, kind);
        std::vector<omega_state_t> obs(4), grads(4);
        for (int i = 0; i < 4; ++i) {
          ok(omega_state_create(e.mesh, ntr, &obs[i]));
          ok(omega_state_create(e.mesh, ntr, &grads[i]));
        }
        const size_t before = fake::bytes;
        double J;
        for (int call = 0; call < 2; ++call)
          ok(omega_batch_adjoint_run(e.batch, 0.0, 20, 20, 0, obs.data(), weights, &J, grads.data(),
                                     nullptr, nullptr));
        std::printf("kind %d, %d tracers, %d levels: %zu bytes kept\n", kind, ntr, L,
                    fake::bytes - before);
        CHECK(fake::bytes - before <= kBound);
        CHECK(L > 8 || fake::bytes > before);
        for (int i = 0; i < 4; ++i) {
          ok(omega_state_destroy(obs[i]));
          ok(omega_state_destroy(grads[i]));
        }
      }
  CHECK(fake::bytes == 0);
}

// The block order set with omega_model_set_launch reaches the stage kernels,
// a model's own and an ensemble's.
static void block_order() {
  Ensemble e(1, 128, 128, 64, Ensemble::params(2), OMEGA_STEPPER_RK4);
  omega_state_t tend;
  ok(omega_state_create(e.mesh, 2, &tend));
  for (int order : {1, 0}) {
    ok(omega_model_set_launch(e.models[0], 0, 0, order, -1));
    const auto own = launched(std::max(sizeof(StageLaunch), sizeof(TileLaunch)), [&] {
      ok(omega_model_compute_tendency(e.models[0], tend, e.states[0], 0.0, OMEGA_ADD_REPLACE, nullptr));
    });
    const auto batch = launched(sizeof(void *), [&] { ok(omega_batch_step(e.batch, nullptr)); });
    CHECK(own.size() == 2 && batch.size() == 8); // momentum, tracers
    CHECK(own[0].at<StageLaunch>().swz == order);
    CHECK(own[1].at<TileLaunch>().swz == order);
    CHECK(batch[0].at<const StageLaunch *>()->swz == order);
    CHECK(batch[1].at<const TileLaunch *>()->swz == order);
  }
  ok(omega_state_destroy(tend));
}

// Cells per block, set or tuned, leave no wavefronts idle where a kernel has
// 256 threads in any case (models small enough for one launch, ensembles);
// where momentum has a launch of its own the block is as large as they ask.
static void tuned_cells() {
  for (int nx : {16, 128})
    for (int L : {64, 60, 7})
      for (int rows : {0, 4, 2}) {
        Ensemble e(1, nx, nx, L, Ensemble::params(2), OMEGA_STEPPER_RK4);
        omega_state_t tend;
        ok(omega_state_create(e.mesh, 2, &tend));
        ok(omega_model_set_launch(e.models[0], rows, 0, -1, -1));
        const auto own = launched(sizeof(StageLaunch), [&] {
          ok(omega_model_compute_tendency(e.models[0], tend, e.states[0], 0.0, OMEGA_ADD_REPLACE, nullptr));
        });
        const auto batch = launched(sizeof(void *), [&] { ok(omega_batch_step(e.batch, nullptr)); });
        const StageLaunch p = own[0].at<StageLaunch>(), q = *batch[0].at<const StageLaunch *>();
        const bool one = own.size() == 1;
        std::printf("%d x %d cells, %d levels, rows %d: %zu launches, %d x %d of %u threads; ensemble %d x %d\n",
                    nx, nx, L, rows, own.size(), p.lx, p.rows, own[0].block.x, q.lx, q.rows);
        CHECK(one == (nx == 16 || L == 7));
        CHECK((int)own[0].block.x == (one ? 256 : p.lx * p.rows));
        if (one) CHECK(p.rows == 256 / p.lx);
        else CHECK(p.rows == (rows ? rows : 256 / p.lx));
        CHECK(batch[0].block.x == 256 && q.rows == 256 / q.lx);
        for (const StageLaunch &x : {p, q}) CHECK(x.tiles >= 1 && (x.tiles / x.ncb) * x.ncb == x.tiles &&
                                                  x.ncb * x.rows >= x.nc && (x.ncb - 1) * x.rows < x.nc);
        ok(omega_state_destroy(tend));
      }
}

// Bit 5 of the kernel flags is set exactly where a tendency launches the
// stage kernels (no diagnostics launch), whatever else is said.
static void reports() {
  struct Case {
    const char *what;
    int L, stage;
    std::function<void(omega_params &)> params;
    std::function<void(omega_model_t)> set;
  };
  auto none = [](auto) {};
  auto f = [](omega_model_t m) {
    std::vector<double> f((size_t)16 * 16 * 2, 1e-4);
    f[3] = 2e-4;
    ok(omega_model_set_f_vertex(m, f.data()));
  };
  const std::vector<Case> cases = {
      {"default", 64, 1, [](omega_params &) {}, none},
      {"any layer count", 7, 1, [](omega_params &) {}, none},
      {"every term", 64, 1, [](omega_params &p) { p.visc_del2 = p.visc_del4 = p.eddy_diff2 = p.eddy_diff4 = 1; }, none},
      {"forms", 64, 0, [](omega_params &) {}, [](omega_model_t m) { ok(omega_model_set_kernel_forms(m, 3)); }},
      {"variant", 64, 0, [](omega_params &) {}, [](omega_model_t m) { ok(omega_model_set_variant(m, 1)); }},
      {"no PV term", 64, 0, [](omega_params &) {}, [](omega_model_t m) { ok(omega_model_set_terms(m, 6)); }},
      {"drag", 64, 0, [](omega_params &) {}, [](omega_model_t m) { ok(omega_model_set_terms(m, 128 + 7)); }},
      {"f per vertex", 64, 0, [](omega_params &) {}, f},
      {"a tendency off", 64, 0, [](omega_params &p) { p.disable_vn_tendency = 1; }, none},
  };
  for (const Case &c : cases) {
    omega_params p = Ensemble::params(1);
    c.params(p);
    Ensemble e(1, 16, 16, c.L, p, OMEGA_STEPPER_RK4);
    c.set(e.models[0]);
    int flags;
    ok(omega_model_kernel_flags(e.models[0], &flags));
    omega_state_t tend;
    ok(omega_state_create(e.mesh, 1, &tend));
    ok(omega_timing_enable(1));
    ok(omega_timing_reset());
    ok(omega_model_compute_tendency(e.models[0], tend, e.states[0], 0.0, OMEGA_ADD_REPLACE, nullptr));
    double ms;
    int64_t diag = 0, tends = 0;
    ok(omega_timing_read("diag", &ms, &diag));
    ok(omega_timing_read("tend", &ms, &tends));
    ok(omega_timing_enable(0));
    std::printf("%s: flags %d, %d diagnostics launches\n", c.what, flags, (int)diag);
    CHECK(tends == 1);
    CHECK(((flags >> 5) & 1) == c.stage);
    if (!p.disable_vn_tendency) CHECK((diag == 0) == (c.stage == 1));
    ok(omega_state_destroy(tend));
  }
}

static std::string contents(const std::string &path) {
  std::ifstream in(path);
  return std::string(std::istreambuf_iterator<char>(in), {});
}

// The tuners time shapes that change what runs and nothing else, and their
// records tell the stage kernels from the others; records of the others are
// still read where there is none of the stage kernels.
static void tuning() {
  char dir[] = "/tmp/omega_tuning_XXXXXX";
  CHECK(mkdtemp(dir));
  const std::string cache = std::string(dir) + "/cache";
  setenv("OMEGA_TUNE_CACHE", cache.c_str(), 1);
  // cells, levels, shapes to time: levels per lane, and cells per block and
  // block order where momentum has a launch of its own
  struct Size {
    int nx, L, launches, shapes;
  };
  for (const Size &c : {Size{16, 64, 1, 2}, Size{16, 7, 1, 1}, Size{128, 64, 2, 12}}) {
    for (const char *forms : {"s", "h", ""}) {
      std::remove(cache.c_str());
      Ensemble e(1, c.nx, c.nx, c.L, Ensemble::params(2), OMEGA_STEPPER_RK4);
      const std::string key = "model;" + std::to_string(c.nx * c.nx) + ":" + std::to_string(c.L) + ":2:7:";
      const std::string old = c.L == 64 ? "h" : "g";
      // another family's record comes first in the file
      if (*forms) std::ofstream(cache) << key << old << " 4 1 0 9.5 -1\n";
      if (*forms == 's') std::ofstream(cache, std::ios::app) << key << "s 2 1 1 0.5 -1\n";
      double ms = 0;
      const auto n = launched(0, [&] { ok(omega_model_autotune(e.models[0], e.states[0], 3, &ms, nullptr)); });
      std::printf("%d x %d cells, %d levels, records '%s': %zu launches, %g ms\n%s", c.nx, c.nx, c.L, forms,
                  n.size(), ms, contents(cache).c_str());
      int rows, lpt, order;
      ok(omega_model_get_launch(e.models[0], &rows, &lpt, &order, nullptr));
      if (*forms == 's') CHECK(n.empty() && ms == 0.5 && rows == 2 && order == 1);
      else if (*forms) CHECK(n.empty() && ms == 9.5 && rows == 4 && order == 0);
      else {
        CHECK((int)n.size() == c.shapes * c.launches * (1 + 3));
        CHECK(contents(cache).rfind(key + "s ", 0) == 0);
      }
    }
  }
  // an ensemble of such members alone: nothing to choose
  std::remove(cache.c_str());
  {
    Ensemble e(3, 16, 16, 64, Ensemble::params(2), OMEGA_STEPPER_RK4);
    ok(omega_batch_set_launch(e.batch, 128, 1));
    double ms = 0;
    const auto n = launched(0, [&] { ok(omega_batch_autotune(e.batch, 3, &ms, nullptr)); });
    int threads, lpt;
    ok(omega_batch_get_launch(e.batch, &threads, &lpt));
    std::printf("ensemble: %zu launches, %g ms, %d threads\n", n.size(), ms, threads);
    CHECK(n.size() == 4 * 2 * (1 + 3) && ms > 0 && threads == 128 && lpt == 1);
    CHECK(contents(cache).empty());
  }
  // with a member on the other kernels: every shape
  {
    Ensemble e(3, 128, 128, 64, Ensemble::params(2), OMEGA_STEPPER_RK4);
    ok(omega_model_set_kernel_forms(e.models[1], 3));
    const auto n = launched(0, [&] { ok(omega_batch_autotune(e.batch, 3, nullptr, nullptr)); });
    CHECK(n.size() == 24 * 4 * (2 + 2) * (1 + 3));
    CHECK(contents(cache).rfind("0/4;16384:64:2:7:s;16384:64:2:7:h;16384:64:2:7:s ", 0) == 0);
  }
  std::remove(cache.c_str());
  CHECK(rmdir(dir) == 0);
  unsetenv("OMEGA_TUNE_CACHE");
}

// An ensemble's stage is two launches for all its members of even layer counts
// and two for those of odd ones, whatever their terms, layers and tiles.
static void few_launches() {
  omega_batch_t batch;
  ok(omega_batch_create(OMEGA_STEPPER_RK4, 4, &batch));
  std::vector<omega_mesh_t> meshes;
  std::vector<omega_model_t> models;
  std::vector<omega_state_t> states;
  auto add = [&](int L, int ntr, int terms) {
    omega_mesh_t mesh;
    omega_model_t m;
    omega_state_t s;
    const omega_params p = Ensemble::params(ntr);
    ok(omega_mesh_create_planar_hex(10, 8, 1e4, L, OMEGA_ORDER_HILBERT, &mesh));
    ok(omega_model_create(mesh, &p, &m));
    ok(omega_model_set_terms(m, terms));
    ok(omega_state_create(mesh, ntr, &s));
    ok(omega_batch_add(batch, m, s, 10.0, nullptr));
    meshes.push_back(mesh);
    models.push_back(m);
    states.push_back(s);
  };
  for (int L : {2, 4, 8, 64})
    for (int terms : {7, 15, 39, 47, 71, 79, 103, 111}) add(L, 1 + L % 3, terms);
  size_t n = launched(0, [&] { ok(omega_batch_step(batch, nullptr)); }).size();
  std::printf("even layer counts: %zu launches a step\n", n);
  CHECK(n == 4 * 2);
  for (int L : {1, 5})
    for (int terms : {7, 111}) add(L, 2, terms);
  n = launched(0, [&] { ok(omega_batch_step(batch, nullptr)); }).size();
  std::printf("and odd ones: %zu launches a step\n", n);
  CHECK(n == 4 * 4);
  ok(omega_batch_destroy(batch));
  for (auto s : states) ok(omega_state_destroy(s));
  for (auto m : models) ok(omega_model_destroy(m));
  for (auto m : meshes) ok(omega_mesh_destroy(m));
}

// Next to others small members run the others' kernels: no launches more.
// Members on the stage kernels do not wait for those on the others: their
// launches run on a stream of the batch's, which starts after what came before
// the step and ends before what comes after it.
static void side_by_side() {
  const int streams = fake::streams;
  {
    Ensemble e(3, 16, 16, 64, Ensemble::params(1), OMEGA_STEPPER_RK4);
    ok(omega_model_set_kernel_forms(e.models[1], 3));
    CHECK(launched(0, [&] { ok(omega_batch_step(e.batch, nullptr)); }).size() == 4 * 2);
  }
  {
    Ensemble e(3, 128, 128, 64, Ensemble::params(1), OMEGA_STEPPER_RK4);
    const hipStream_t s = reinterpret_cast<hipStream_t>(handle());
    fake::waits.clear();
    for (const auto &l : launched(0, [&] { ok(omega_batch_step(e.batch, reinterpret_cast<omega_stream_t>(s))); }))
      CHECK(l.stream == s);
    CHECK(fake::waits.empty());
    ok(omega_model_set_kernel_forms(e.models[1], 3));
    const auto n = launched(0, [&] { ok(omega_batch_step(e.batch, reinterpret_cast<omega_stream_t>(s))); });
    CHECK(n.size() == 4 * (2 + 2) && fake::waits.size() == 2);
    const auto &from = fake::waits[0], &to = fake::waits[1];
    CHECK(from.on == s && from.stream != s && from.at == 0);
    CHECK(to.on == from.stream && to.stream == s && to.at == n.size());
    size_t side = 0;
    for (const auto &l : n) side += l.stream == from.stream;
    CHECK(side == 4 * 2);
  }
  CHECK(fake::streams == streams);
}

// Members of one model have diagnostics of their own: no two members of a
// launch write the same rows.
static void one_model() {
  for (int terms : {7, 7 + 16}) { // the stage kernels' ensemble launches, the others'
    omega_mesh_t mesh;
    omega_model_t model;
    omega_batch_t batch;
    std::vector<omega_state_t> states(3);
    const omega_params p = Ensemble::params(1);
    ok(omega_mesh_create_planar_hex(12, 10, 1e4, 64, OMEGA_ORDER_HILBERT, &mesh));
    ok(omega_model_create(mesh, &p, &model));
    ok(omega_model_set_terms(model, terms));
    ok(omega_batch_create(OMEGA_STEPPER_RK4, 4, &batch));
    for (auto &s : states) {
      ok(omega_state_create(mesh, 1, &s));
      ok(omega_batch_add(batch, model, s, 10.0, nullptr));
    }
    const auto n = launched(sizeof(void *), [&] { ok(omega_batch_step(batch, nullptr)); });
    std::set<const double *> rows;
    for (int i = 0; i < 3; ++i) {
      const DiagOut &d = terms == 7 ? n[6].at<const StageLaunch *>()[i].d : n[0].at<const BatchMember *>()[i].d;
      for (const double *x : {d.rvort_v, d.inv_thick_v, d.ke_c, d.div_c, d.trdel2_c}) CHECK(x && rows.insert(x).second);
      if (terms != 7)
        for (const double *x : {d.vdel2_e, d.vdel2_rv_v, d.vdel2_div_c}) CHECK(x && rows.insert(x).second);
    }
    ok(omega_batch_destroy(batch));
    for (auto s : states) ok(omega_state_destroy(s));
    ok(omega_model_destroy(model));
    ok(omega_mesh_destroy(mesh));
    CHECK(fake::bytes == 0);
  }
}

// A tendency VJP with tracer del4 takes its diagnostics from the stage kernels
// where their launch has a block for each tracer of a tile, and without del4
// at any size.
static void vjp_rows() {
  struct Case {
    int nx, L, ntr, terms, diag;
  };
  for (const Case &c : {Case{48, 64, 2, 79, 0}, Case{64, 64, 1, 79, 1}, Case{64, 64, 9, 79, 1},
                        Case{64, 64, 9, 15, 0}, Case{80, 25, 4, 79, 0}, Case{128, 64, 2, 79, 1},
                        Case{128, 64, 2, 15, 0}}) {
    Ensemble e(1, c.nx, c.nx, c.L, Ensemble::params(c.ntr), OMEGA_STEPPER_RK4);
    ok(omega_model_set_terms(e.models[0], c.terms));
    omega_state_t cot[2];
    for (auto &s : cot) ok(omega_state_create(e.mesh, c.ntr, &s));
    ok(omega_timing_enable(1));
    ok(omega_timing_reset());
    ok(omega_model_tendency_vjp(e.models[0], e.states[0], cot[0], cot[1], nullptr, nullptr));
    double ms;
    int64_t diag = 0;
    ok(omega_timing_read("diag", &ms, &diag));
    ok(omega_timing_enable(0));
    std::printf("%d x %d cells, %d levels, %d tracers, terms %d: %d\n", c.nx, c.nx, c.L, c.ntr, c.terms,
                (int)diag);
    CHECK(diag == c.diag);
    for (auto &s : cot) ok(omega_state_destroy(s));
  }
}

int main(int argc, char **argv) {
  const std::map<std::string, std::function<void()>> checks = {{"tall", tall}, {"rebuild", rebuild},
                                                              {"keep_stepper", keep_stepper},
                                                              {"keep_ensemble", keep_ensemble},
                                                              {"block_order", block_order},
                                                              {"tuned_cells", tuned_cells},
                                                              {"reports", reports},
                                                              {"tuning", tuning},
                                                              {"few_launches", few_launches},
                                                              {"side_by_side", side_by_side},
                                                              {"one_model", one_model},
                                                              {"vjp_rows", vjp_rows}};
  CHECK(argc == 2 && checks.count(argv[1]));
  checks.at(argv[1])();
  std::printf("%s ok\n", argv[1]);
}
