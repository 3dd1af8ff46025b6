// Graph bookkeeping of the uniform mesh: the source file itself, with the HIP calls
// it makes and the kernel launches replaced below.  A step is what launch_advance_time
// enqueues; a graph is the number of steps captured into it.
//
// usage: mesh_host_check; prints what is wrong and exits 1.
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "../../exahype-engine_amd/csrc/mesh.cpp"

namespace {
bool capturing = false;
int captured = 0, steps = 0, graphs = 0, execs = 0, launches = 0, most_steps = 1000;
hipError_t last_error = hipSuccess;

#define CHECK(cond)                                             \
  do {                                                          \
    if (!(cond)) {                                              \
      std::printf("line %d: %s\n", __LINE__, #cond);            \
      std::exit(1);                                             \
    }                                                           \
  } while (0)
}  // namespace

extern "C" {
hipError_t hipFree(void* p) { return std::free(p), hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { return std::memcpy(d, s, n), hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  return std::memcpy(d, s, n), hipSuccess;
}
hipError_t hipMemset(void* d, int v, size_t n) { return std::memset(d, v, n), hipSuccess; }
hipError_t hipGetLastError() {
  const hipError_t e = last_error;
  last_error = hipSuccess;
  return e;
}
const char* hipGetErrorString(hipError_t) { return ""; }
hipError_t hipEventCreate(hipEvent_t*) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t*, unsigned) { return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { return *ms = 0, hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return *s = reinterpret_cast<hipStream_t>(1), hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) {
  capturing = true;
  captured = 0;
  return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) {
  capturing = false;
  graphs++;
  *g = reinterpret_cast<hipGraph_t>(size_t(captured));
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t g, hipGraphNode_t*, char*, size_t) {
  if (int(reinterpret_cast<size_t>(g)) > most_steps) return last_error = hipErrorOutOfMemory;
  execs++;
  *e = reinterpret_cast<hipGraphExec_t>(g);
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t) {
  steps += int(reinterpret_cast<size_t>(e));
  launches++;
  return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t) { return graphs--, hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return execs--, hipSuccess; }
int roctxRangePushA(const char*) { return 0; }
int roctxRangePop() { return 0; }
}

namespace exa {
static KernelCfg cfg;
const KernelCfg& ctx_cfg(const exa_ctx*) { return cfg; }
void set_error(const std::string&) {}
hipError_t device_malloc(void** p, size_t n) { return *p = std::calloc(1, n), hipSuccess; }
static int enqueue() { return static_cast<int>(hipGetLastError()); }
int launch_advance_time(hipStream_t, double*, int, double*, int) {
  (capturing ? captured : steps)++;
  return enqueue();
}
int launch_predictor(const KernelCfg&, hipStream_t, long, const double*, const double*, const double*, double*, double*,
                     double*, int*, const LaunchOpts&) {
  return enqueue();
}
int launch_riemann(const KernelCfg&, hipStream_t, long, const int*, const double*, double*, const LaunchOpts&) {
  return enqueue();
}
int launch_corrector(const KernelCfg&, hipStream_t, long, double*, double*, const double*, const double*, const double*,
                     double*, const LaunchOpts&) {
  return enqueue();
}
int launch_corrector_riemann(const KernelCfg&, hipStream_t, long, int, double*, const double*, const double*,
                             const double*, const double*, double*, const LaunchOpts&) {
  return enqueue();
}
int launch_stable_dt(const KernelCfg&, hipStream_t, long, const double*, const double*, double*, const LaunchOpts&) {
  return enqueue();
}
int launch_dt_reduce(hipStream_t, double*, double*) { return enqueue(); }
int launch_dt_slots_init(hipStream_t, double*, long) { return enqueue(); }
bool corrector_riemann_supported(const KernelCfg&) { return true; }
bool predictor_f32_faces_supported(const KernelCfg&) { return false; }
bool predictor_supports_range(const KernelCfg&) { return false; }
bool boundary_supported(const KernelCfg&) { return false; }
int observables_blocks(long) { return 1; }
int launch_observables(const KernelCfg&, hipStream_t, long, double, const double*, double*, double*) { return 0; }
int launch_probe(const KernelCfg&, hipStream_t, int, double, const double*, int, const double*, double*) { return 0; }
int launch_halo_pack(const KernelCfg&, hipStream_t, int, int, const double*, const double*, double*, double*) { return 0; }
int launch_density_wave(hipStream_t, long, int, int, int, int, double, const double*, const double*, double*) { return 0; }
int launch_entropy_wave(hipStream_t, long, int, int, int, int, double, const double*, double, double*) { return 0; }
int launch_boundary_mesh(const KernelCfg&, hipStream_t, int, double, const BcKinds&, const double*, double*, double*,
                         const double*) {
  return 0;
}
}  // namespace exa

int main() {
  exa::cfg.dim = 2, exa::cfg.order = 3, exa::cfg.nvar = 5;
  exa::cfg.cfl = 0.9, exa::cfg.pnpm = 0.1;
  for (bool room : {true, false}) {
    exa_mesh* m = nullptr;
    CHECK(!exa_mesh_create_uniform(&m, reinterpret_cast<exa_ctx*>(&exa::cfg), 3, 1.0 / 3));
    // without room the graph of several steps cannot be instantiated: steps one by one, nothing left behind
    most_steps = room ? 1000 : 1;
    for (int n : {19, 8, 7, 19, 16}) {
      steps = launches = 0;
      CHECK(!exa_mesh_run(m, n, 1) && steps == n);
      CHECK(launches <= n && (room || launches == n));
      CHECK(graphs == execs && execs <= 2);
    }
    most_steps = 1000;
    steps = launches = 0;
    CHECK(!exa_mesh_run(m, 17, 1) && steps == 17 && launches == 3);
    // a change of the step drops both graphs
    CHECK(!exa_mesh_set_fused(m, 0) && graphs == 0 && execs == 0);
    steps = launches = 0;
    CHECK(!exa_mesh_run(m, 9, 1) && !exa_mesh_run(m, 9, 1) && steps == 18 && graphs == 2);
    exa_mesh_destroy(m);
    CHECK(graphs == 0 && execs == 0);
    // a first capture that cannot be instantiated is an error, and leaves nothing either
    CHECK(!exa_mesh_create_uniform(&m, reinterpret_cast<exa_ctx*>(&exa::cfg), 3, 1.0 / 3));
    most_steps = 0;
    CHECK(exa_mesh_run(m, 3, 1) == EXA_ERR_HIP && exa_mesh_run(m, 3, 1) == EXA_ERR_HIP && graphs == 0);
    most_steps = 1000;
    steps = 0;
    CHECK(!exa_mesh_run(m, 3, 1) && steps == 3 && graphs == 1);
    exa_mesh_destroy(m);
    CHECK(graphs == 0 && execs == 0);
  }
  std::puts("ok");
  return 0;
}
