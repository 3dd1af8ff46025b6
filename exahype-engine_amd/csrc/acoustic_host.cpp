// Host driver of the linear acoustic mesh and its discrete adjoint
// (exa_acoustic_* of include/exahype_amd.h).
//
// Forward step (order of the reference's fused linear ADER-DG step,
// ExaHyPE/exahype/solvers/ADERDGSolver.cpp:887-947 prediction, 1764-1823
// Riemann, 1190-1256 face integrals + update):
//   ac_predict (update)  predictor + volume integral + volume part of the update
//   ac_corrector         Riemann + face integrals + face part of the update
//   ac_receivers         p at the receivers
// Point source: getPointSources / deltaDistribution
// (generic/c/3d/deltaDistribution.cpph:37-146) for a pressure source with a
// Ricker time function.  The moments are separable, PSi[n][node] =
// f(t_n) * g[node] with g = phi(x_ref) / (W_node h^3), so the device needs g
// and, per step, B numbers: sigma_0 = dt sum_t w_t f(t_t) (added to level 0
// and removed by the volume integral, spaceTimePredictorLinear.cpph:111-131,482-503),
// f(t) (level 1, :133-140) and the time derivatives of the interpolant of f
// at the time nodes (levels 2..B-1, :141-178).
//
// Adjoint with checkpointing: states are stored every `every` steps on the
// forward sweep; the backward sweep recomputes each segment from its
// checkpoint, then runs the transposed step backwards through it.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>
#include <mutex>
#include <string>
#include <utility>
#include <vector>

#include "../../include/exahype_amd.h"
#include "engine.h"
#include "trace.h"

namespace exa {
const KernelCfg& ctx_cfg(const exa_ctx* c);
}

struct exa_acoustic {
  exa::KernelCfg k{};
  exa::Tables tab{};
  int n = 0, B = 0, N = 0, F = 0;
  long nc = 0;
  double h = 0, dt = 0;
  int step = 0;  // host mirror of the device step counter
  hipStream_t stream = nullptr;
  double *d_u = nullptr, *d_mat = nullptr, *d_qb = nullptr;
  double *d_qb2 = nullptr, *d_rec_p = nullptr;  // fused steps: the other face buffer, p at the receivers' cells
  double *d_ubar = nullptr, *d_fbar = nullptr, *d_fbar2 = nullptr, *d_gc = nullptr;
  // gradient: checkpoints, the states of a segment behind its checkpoint, and the
  // faces of its steps (optional)
  double *d_ck = nullptr, *d_seg = nullptr, *d_segq = nullptr;
  long ck_cap = 0, seg_cap = 0, segq_cap = 0;  // doubles
  int* d_step = nullptr;
  std::vector<double> mat;  // host copy of (rho, c) per cell
  // source
  bool has_src = false;
  double src_x[3] = {0, 0, 0}, amp = 0, f0 = 0, t0 = 0;
  long src_cell = -1;
  double* d_src_g = nullptr;
  double* d_src_tab = nullptr;
  int src_tab_steps = 0;  // steps covered by d_src_tab
  // receivers
  int nrec = 0;
  int* d_rcell = nullptr;
  int *d_rstart = nullptr, *d_rorder = nullptr;  // receivers by cell [nc + 1], [nrec]
  double* d_rw = nullptr;
  double* d_rec = nullptr;
  long rec_cap = 0;  // doubles
  double* d_res = nullptr;
  long res_cap = 0;
  double ms[3] = {0, 0, 0};
  // per-kernel timing of exa_acoustic_run (HIP events on the launch stream)
  bool timing = false;
  std::vector<hipEvent_t> ev;
  int timed_steps = 0;
  int pred_variant = 0;  // forward predictor: 0 x-line form, 1 node form
  // optional buffers kept between calls
  int device = 0;
  size_t device_bytes = 0;  // its memory
  bool idle = false;        // in the list of meshes that keep some
  exa_acoustic* next_idle = nullptr;
};

namespace {

int fail(hipError_t e, const char* what) {
  (void)hipGetLastError();  // reported here: not by the next launch
  exa::set_error(std::string(what) + ": " + hipGetErrorString(e));
  return EXA_ERR_HIP;
}

int argerr(const char* what) {
  exa::set_error(what);
  return EXA_ERR_ARG;
}

#define HIP_OK(expr, what)                       \
  do {                                           \
    hipError_t _e = (expr);                      \
    if (_e != hipSuccess) return fail(_e, what); \
  } while (0)

#define RC_OK(expr)          \
  do {                       \
    const int _rc = (expr);  \
    if (_rc) return _rc;     \
  } while (0)

int status(int rc, const char* what) {
  if (rc == -1) {
    exa::set_error(std::string(what) + ": order not compiled into this library");
    return EXA_ERR_UNSUPPORTED;
  }
  if (rc != 0) return fail(static_cast<hipError_t>(rc), what);
  return EXA_OK;
}

double lagrange(const double* x, int B, int k, double s) {
  double r = 1.0;
  for (int m = 0; m < B; m++)
    if (m != k) r *= (s - x[m]) / (x[k] - x[m]);
  return r;
}

double ricker(double t, double f0, double t0) {
  const double pi = 3.14159265358979323846;
  const double a = pi * pi * f0 * f0 * (t - t0) * (t - t0);
  return (1.0 - 2.0 * a) * std::exp(-a);
}

long locate(const exa_acoustic* ac, const double* p, double* xi) {
  int ic[3];
  for (int d = 0; d < 3; d++) {
    ic[d] = static_cast<int>(std::floor(p[d] / ac->h));
    if (ic[d] < 0) ic[d] = 0;
    if (ic[d] >= ac->n) ic[d] = ac->n - 1;
    if (xi) xi[d] = (p[d] - ic[d] * ac->h) / ac->h;
  }
  return (long(ic[2]) * ac->n + ic[1]) * ac->n + ic[0];
}

// Frees what a mesh holds only to save time: the fused steps' and the gradient's buffers.
void free_optional(exa_acoustic* ac) {
  for (double** p : {&ac->d_qb2, &ac->d_rec_p, &ac->d_ck, &ac->d_seg, &ac->d_segq}) {
    if (*p) (void)hipFree(*p);
    *p = nullptr;
  }
  ac->ck_cap = ac->seg_cap = ac->segq_cap = 0;
}

size_t optional_bytes(const exa_acoustic* ac) {
  const long doubles = (ac->d_qb2 ? ac->nc * 6 * ac->F * 4 : 0) + (ac->d_rec_p ? long(ac->nrec) * ac->N : 0) +
                       ac->ck_cap + ac->seg_cap + ac->segq_cap;
  return sizeof(double) * size_t(doubles);
}

// Allocating and freeing its optional buffers costs a gradient 6 % at 27^3 of order 4
// (40 steps) and 40 % at 13^3, so a mesh keeps them for its next call: all meshes of
// a device together at most an eighth of its memory, and what idle meshes keep is
// freed as soon as the library cannot allocate something (device_malloc).
std::mutex idle_mutex;
exa_acoustic* idle_meshes = nullptr;  // no call in flight, some buffers kept

void unlink_idle(exa_acoustic* ac) {  // idle_mutex held
  if (!ac->idle) return;
  exa_acoustic** p = &idle_meshes;
  while (*p != ac) p = &(*p)->next_idle;
  *p = ac->next_idle;
  ac->idle = false;
}

// A call that may use or free the optional buffers of its mesh.
class Call {
 public:
  explicit Call(exa_acoustic* ac) : ac_(ac) {
    std::lock_guard<std::mutex> lock(idle_mutex);
    unlink_idle(ac);
  }
  ~Call() {
    std::lock_guard<std::mutex> lock(idle_mutex);
    size_t kept = optional_bytes(ac_);
    if (kept == 0) return;
    for (const exa_acoustic* m = idle_meshes; m; m = m->next_idle)
      if (m->device == ac_->device) kept += optional_bytes(m);
    if (kept > ac_->device_bytes / 8) {
      free_optional(ac_);
      return;
    }
    ac_->next_idle = idle_meshes;
    ac_->idle = true;
    idle_meshes = ac_;
  }
  Call(const Call&) = delete;
  Call& operator=(const Call&) = delete;

 private:
  exa_acoustic* ac_;
};

// hipMalloc of what a call cannot do without; before it uses an optional buffer
template <typename T>
hipError_t allocate(exa_acoustic* ac, T** p, size_t n) {
  hipError_t e = exa::device_malloc(p, sizeof(T) * n);
  if (e == hipSuccess) return e;
  (void)hipGetLastError();
  free_optional(ac);
  e = hipMalloc(p, sizeof(T) * n);
  if (e != hipSuccess) *p = nullptr;
  return e;
}
// of what it can: false (and no error left) without memory for it
bool try_allocate(double** p, size_t n) {
  if (exa::device_malloc(p, sizeof(double) * n) == hipSuccess) return true;
  (void)hipGetLastError();
  *p = nullptr;
  return false;
}

int grow(exa_acoustic* ac, double** p, long* cap, long need) {
  if (*cap >= need) return EXA_OK;
  if (*p) (void)hipFree(*p);
  *p = nullptr;
  *cap = 0;
  HIP_OK(allocate(ac, p, need), "hipMalloc");
  *cap = need;
  return EXA_OK;
}
bool try_grow(double** p, long* cap, long need) {
  if (*cap >= need) return true;
  if (*p) (void)hipFree(*p);
  *p = nullptr;
  *cap = 0;
  if (!try_allocate(p, need)) return false;
  *cap = need;
  return true;
}

// Time factors of the source for steps [0, steps).
int ensure_source_table(exa_acoustic* ac, int steps) {
  if (!ac->has_src || steps <= ac->src_tab_steps) return EXA_OK;
  const int B = ac->B;
  const double* w = ac->tab.w;
  const double* x = ac->tab.x;
  const double* dudx = ac->tab.dudx;
  const double* F0 = ac->tab.F0;
  const int cap = steps + 64;
  const int SW = ac->k.split_ck ? B + 1 : B;  // row width
  std::vector<double> tabh(size_t(cap) * SW);
  std::vector<double> fn(B + 1), psd(B), tmp(B);
  for (int k = 0; k < cap; k++) {
    const double t = k * ac->dt;
    for (int m = 0; m < B + 1; m++) {
      const double tm = (m == 0) ? t : ac->dt * x[m - 1] + t;
      fn[m] = ac->amp * ricker(tm, ac->f0, ac->t0);
    }
    double sum = 0.0;
    for (int m = 1; m < B + 1; m++) sum += w[m - 1] * fn[m];
    double* row = &tabh[size_t(k) * SW];
    if (ac->k.split_ck) {
      // split predictor (fusedSPTVI_linear_split_ck_cpp.template:179-199, 313-331):
      // {dt sum_t w_t f_t, s_0 .. s_{B-1}}, s_k = derPS_k . f at the Gauss time
      // nodes, derPS_0 = FLCoeff, derPS_{k+1}[j] = sum_i derPS_k[i] dudx[i][j]
      row[0] = ac->dt * sum;
      std::vector<double> der(F0, F0 + B), nxt(B);
      for (int q = 0; q < B; q++) {
        double v = 0.0;
        for (int j = 0; j < B; j++) v += der[j] * fn[j + 1];
        row[1 + q] = v;
        for (int j = 0; j < B; j++) {
          double acc = 0.0;
          for (int i = 0; i < B; i++) acc += der[i] * dudx[i * B + j];
          nxt[j] = acc;
        }
        der = nxt;
      }
      continue;
    }
    row[0] = ac->dt * sum;
    if (B > 1) row[1] = fn[0];
    for (int m = 0; m < B; m++) psd[m] = fn[m + 1];
    const double invDt = 1.0 / ac->dt;
    for (int i = 2; i < B; i++) {
      for (int tt = 0; tt < B; tt++) {
        double s = 0.0;
        for (int q = 0; q < B; q++) s += psd[q] * dudx[tt * B + q] * invDt;
        tmp[tt] = s;
      }
      double v = 0.0;
      for (int tt = 0; tt < B; tt++) v += tmp[tt] * F0[tt];
      row[i] = v;
      psd = tmp;
    }
  }
  if (ac->d_src_tab) (void)hipFree(ac->d_src_tab);
  ac->d_src_tab = nullptr;
  ac->src_tab_steps = 0;
  HIP_OK(allocate(ac, &ac->d_src_tab, tabh.size()), "hipMalloc(source table)");
  HIP_OK(hipMemcpy(ac->d_src_tab, tabh.data(), sizeof(double) * tabh.size(), hipMemcpyHostToDevice),
         "upload source table");
  ac->src_tab_steps = cap;
  return EXA_OK;
}

exa::AcousticArgs args(exa_acoustic* ac, double* u) {
  exa::AcousticArgs a;
  a.ncells = ac->nc;
  a.n = ac->n;
  a.h = ac->h;
  a.dt = ac->dt;
  a.tab = ac->k.tab;
  a.u = u;
  a.mat = ac->d_mat;
  a.qb = ac->d_qb;
  a.src_cell = ac->has_src ? ac->src_cell : -1;
  a.src_g = ac->d_src_g;
  a.src_tab = ac->d_src_tab;
  a.step_ptr = ac->d_step;
  a.nrec = ac->nrec;
  a.rcell = ac->d_rcell;
  a.rw = ac->d_rw;
  a.ubar = ac->d_ubar;
  a.fbar = ac->d_fbar;
  a.u_out = u;
  a.qb_out = ac->d_qb;
  a.rstart = ac->d_rstart;
  a.rorder = ac->d_rorder;
  a.gc = ac->d_gc;
  a.pred_variant = ac->pred_variant;
  a.split_ck = ac->k.split_ck;
  return a;
}

// Buffers of one gradient, grown on demand.  Where they do not fit beside what earlier
// calls left, that goes first.  The faces of a segment's steps are kept (and not
// formed a second time) when they fit a quarter of what is free.
int gradient_buffers(exa_acoustic* ac, size_t su, size_t sq, int nck, int seg) {
  auto states = [&] {
    return try_grow(&ac->d_ck, &ac->ck_cap, long(su) * nck) && try_grow(&ac->d_seg, &ac->seg_cap, long(su) * seg);
  };
  if (!states()) {
    free_optional(ac);
    if (!states()) {
      free_optional(ac);
      return fail(hipErrorOutOfMemory, "hipMalloc(checkpoints)");
    }
  }
  const long faces = long(sq) * (seg + 1);
  if (ac->segq_cap < faces) {
    size_t free = 0, total = 0;
    HIP_OK(hipMemGetInfo(&free, &total), "memory");
    if (sizeof(double) * size_t(faces) <= free / 4) (void)try_grow(&ac->d_segq, &ac->segq_cap, faces);
  }
  return EXA_OK;
}

// one forward step from u to u_out (step index `step`, or the device counter if < 0);
// receivers recorded into rec[(step - rec_base) * nrec + r] when rec != nullptr; the
// step's faces in qb (nullptr: the mesh's face buffer)
int enqueue_forward(exa_acoustic* ac, double* u, double* u_out, int step, double* rec, hipEvent_t* ev = nullptr,
                    double* qb = nullptr) {
  exa::TraceRange tr("exa.acoustic.step");
  exa::AcousticArgs a = args(ac, u);
  a.u_out = u_out;
  if (qb) a.qb = a.qb_out = qb;
  a.step_override = step;
  const int o = ac->k.order;
  if (ev) HIP_OK(hipEventRecord(ev[0], ac->stream), "event");
  RC_OK(status(exa::launch_acoustic(exa::kAcPredictUpdate, o, a, ac->stream), "acoustic predictor"));
  if (ev) HIP_OK(hipEventRecord(ev[1], ac->stream), "event");
  a.u = u_out;
  RC_OK(status(exa::launch_acoustic(exa::kAcCorrector, o, a, ac->stream), "acoustic corrector"));
  if (ev) HIP_OK(hipEventRecord(ev[2], ac->stream), "event");
  if (rec && ac->nrec > 0) {
    a.rec = rec;
    RC_OK(status(exa::launch_acoustic(exa::kAcReceivers, o, a, ac->stream), "acoustic receivers"));
  }
  return EXA_OK;
}

// The buffers of the fused steps; false: steps in two kernels, for want of memory or
// because a face buffer too large to keep takes as long to allocate as some six
// steps gain by it.
bool fused_buffers(exa_acoustic* ac, bool receive, int nsteps) {
  if (!ac->d_qb2 && nsteps < 16 && sizeof(double) * ac->nc * 6 * ac->F * 4 > ac->device_bytes / 8) return false;
  struct {
    double** p;
    long n;
  } const need[] = {{&ac->d_qb2, ac->nc * 6 * ac->F * 4}, {&ac->d_rec_p, receive ? long(ac->nrec) * ac->N : 0}};
  for (const auto& b : need) {
    if (*b.p || b.n == 0) continue;
    if (!try_allocate(b.p, b.n)) return false;
  }
  return true;
}

// nsteps forward steps on d_u from step s0, receivers as enqueue_forward: the
// corrector of a step and the predictor of the next run as one kernel where the
// order has one and there is memory for its second face buffer.
int enqueue_forward_steps(exa_acoustic* ac, int s0, int nsteps, double* rec) {
  const bool receive = rec && ac->nrec > 0;
  if (nsteps < 2 || ac->pred_variant != 0 || !exa::acoustic_steps_fused(ac->k.order) || !fused_buffers(ac, receive, nsteps)) {
    for (int i = 0; i < nsteps; i++) RC_OK(enqueue_forward(ac, ac->d_u, ac->d_u, s0 + i, rec));
    return EXA_OK;
  }
  exa::TraceRange tr("exa.acoustic.steps");
  const int o = ac->k.order;
  exa::AcousticArgs a = args(ac, ac->d_u);
  a.step_override = s0;
  RC_OK(status(exa::launch_acoustic(exa::kAcPredictUpdate, o, a, ac->stream), "acoustic predictor"));
  for (int i = 1; i < nsteps; i++) {
    a = args(ac, ac->d_u);
    a.qb_out = ac->d_qb2;
    a.step_override = s0 + i;
    a.rec_p = receive ? ac->d_rec_p : nullptr;
    RC_OK(status(exa::launch_acoustic(exa::kAcStep, o, a, ac->stream), "acoustic step"));
    std::swap(ac->d_qb, ac->d_qb2);
    if (receive) {
      a.step_override = s0 + i - 1;
      a.rec = rec;
      RC_OK(status(exa::launch_acoustic(exa::kAcReceivers, o, a, ac->stream), "acoustic receivers"));
    }
  }
  a = args(ac, ac->d_u);
  a.step_override = s0 + nsteps - 1;
  RC_OK(status(exa::launch_acoustic(exa::kAcCorrector, o, a, ac->stream), "acoustic corrector"));
  if (receive) {
    a.rec = rec;
    RC_OK(status(exa::launch_acoustic(exa::kAcReceivers, o, a, ac->stream), "acoustic receivers"));
  }
  return EXA_OK;
}

void free_acoustic(exa_acoustic* ac) {
  {
    std::lock_guard<std::mutex> lock(idle_mutex);
    unlink_idle(ac);
  }
  double* bufs[] = {ac->d_ck,    ac->d_seg,   ac->d_segq,  ac->d_qb2,   ac->d_rec_p, ac->d_u,     ac->d_mat,   ac->d_qb,     ac->d_ubar,  ac->d_fbar, ac->d_fbar2,
                    ac->d_gc,    ac->d_src_g, ac->d_src_tab, ac->d_rw,   ac->d_rec,  ac->d_res};
  for (double* b : bufs)
    if (b) (void)hipFree(b);
  if (ac->d_step) (void)hipFree(ac->d_step);
  for (int* p : {ac->d_rcell, ac->d_rstart, ac->d_rorder})
    if (p) (void)hipFree(p);
  for (hipEvent_t e : ac->ev) (void)hipEventDestroy(e);
  if (ac->stream) (void)hipStreamDestroy(ac->stream);
  delete ac;
}

int upload_material(exa_acoustic* ac) {
  HIP_OK(hipMemcpyAsync(ac->d_mat, ac->mat.data(), sizeof(double) * ac->mat.size(), hipMemcpyHostToDevice,
                        ac->stream),
         "upload material");
  HIP_OK(hipStreamSynchronize(ac->stream), "sync");
  return EXA_OK;
}

int set_step(exa_acoustic* ac, int step) {
  ac->step = step;
  HIP_OK(hipMemcpyAsync(ac->d_step, &ac->step, sizeof(int), hipMemcpyHostToDevice, ac->stream), "set step");
  HIP_OK(hipStreamSynchronize(ac->stream), "sync");
  return EXA_OK;
}

}  // namespace

namespace exa {
hipError_t device_malloc(void** p, size_t bytes) {
  hipError_t e = hipMalloc(p, bytes);
  if (e == hipSuccess) return e;
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess) return e;
  bool freed = false;
  {
    std::lock_guard<std::mutex> lock(idle_mutex);
    for (exa_acoustic *m = idle_meshes, *next; m; m = next) {
      next = m->next_idle;
      if (m->device != device) continue;
      free_optional(m);
      unlink_idle(m);
      freed = true;
    }
  }
  if (!freed) return e;
  (void)hipGetLastError();  // the one above
  return hipMalloc(p, bytes);
}
}  // namespace exa

extern "C" {

int exa_acoustic_create(exa_acoustic** out, exa_ctx* ctx, int n, double h) {
  if (!out || !ctx || n < 1 || !(h > 0)) return argerr("exa_acoustic_create: invalid argument");
  *out = nullptr;
  const exa::KernelCfg& k = exa::ctx_cfg(ctx);
  if (k.pde.id != EXA_PDE_ACOUSTIC || k.dim != 3 || k.nvar != 4 || k.npar != 2 || k.precision != EXA_PREC_FP64) {
    exa::set_error("exa_acoustic_create: context must be 3D EXA_PDE_ACOUSTIC, 4 variables, 2 parameters, FP64");
    return EXA_ERR_ARG;
  }
  if (!exa::acoustic_order_supported(k.order)) {
    exa::set_error("exa_acoustic_create: order not compiled into this library");
    return EXA_ERR_UNSUPPORTED;
  }
  exa_acoustic* ac = new exa_acoustic;
  ac->k = k;
  exa::build_tables(k.order, &ac->tab);
  ac->n = n;
  ac->h = h;
  ac->B = k.order + 1;
  ac->N = ac->B * ac->B * ac->B;
  ac->F = ac->B * ac->B;
  ac->nc = long(n) * n * n;
  ac->mat.assign(size_t(2) * ac->nc, 1.0);
  const size_t su = size_t(ac->nc) * ac->N * 4, sq = size_t(ac->nc) * 6 * ac->F * 4;
  size_t free = 0;
  hipError_t e = hipGetDevice(&ac->device);
  if (e == hipSuccess) e = hipMemGetInfo(&free, &ac->device_bytes);
  if (e == hipSuccess) e = hipStreamCreateWithFlags(&ac->stream, hipStreamNonBlocking);
  if (e == hipSuccess) e = exa::device_malloc(&ac->d_u, sizeof(double) * su);
  if (e == hipSuccess) e = exa::device_malloc(&ac->d_mat, sizeof(double) * 2 * ac->nc);
  if (e == hipSuccess) e = exa::device_malloc(&ac->d_qb, sizeof(double) * sq);
  if (e == hipSuccess) e = exa::device_malloc(&ac->d_step, sizeof(int));
  if (e == hipSuccess) e = exa::device_malloc(&ac->d_src_g, sizeof(double) * ac->N);
  if (e == hipSuccess) e = hipMemsetAsync(ac->d_u, 0, sizeof(double) * su, ac->stream);
  if (e != hipSuccess) {
    free_acoustic(ac);
    return fail(e, "exa_acoustic_create");
  }
  int rc = upload_material(ac);
  if (!rc) rc = set_step(ac, 0);
  if (!rc) rc = exa_acoustic_set_dt(ac, 0.0);
  if (rc) {
    free_acoustic(ac);
    return rc;
  }
  *out = ac;
  return EXA_OK;
}

int exa_acoustic_destroy(exa_acoustic* ac) {
  if (!ac) return EXA_OK;
  if (ac->stream) (void)hipStreamSynchronize(ac->stream);
  free_acoustic(ac);
  return EXA_OK;
}

long exa_acoustic_ncells(const exa_acoustic* ac) { return ac ? ac->nc : 0; }

int exa_acoustic_set_solution(exa_acoustic* ac, const double* luh) {
  if (!ac || !luh) return argerr("exa_acoustic_set_solution: NULL argument");
  const int N = ac->N;
  std::vector<double> u(size_t(ac->nc) * N * 4);
  std::vector<double> mat(size_t(2) * ac->nc);
  for (long c = 0; c < ac->nc; c++) {
    const double* q = luh + size_t(c) * N * 6;
    const double rho = q[4], cc = q[5];
    for (int nd = 0; nd < N; nd++) {
      const double* qn = q + size_t(nd) * 6;
      if (qn[4] != rho || qn[5] != cc) {
        exa::set_error("exa_acoustic_set_solution: rho and c must be constant within a cell");
        return EXA_ERR_UNSUPPORTED;
      }
      for (int v = 0; v < 4; v++) u[(size_t(c) * N + nd) * 4 + v] = qn[v];
    }
    if (!(rho > 0)) return argerr("exa_acoustic_set_solution: rho must be positive");
    mat[2 * c] = rho;
    mat[2 * c + 1] = cc;
  }
  ac->mat = mat;
  HIP_OK(hipMemcpyAsync(ac->d_u, u.data(), sizeof(double) * u.size(), hipMemcpyHostToDevice, ac->stream),
         "set_solution");
  return upload_material(ac);
}

int exa_acoustic_get_solution(exa_acoustic* ac, double* luh) {
  if (!ac || !luh) return argerr("exa_acoustic_get_solution: NULL argument");
  const int N = ac->N;
  std::vector<double> u(size_t(ac->nc) * N * 4);
  HIP_OK(hipMemcpyAsync(u.data(), ac->d_u, sizeof(double) * u.size(), hipMemcpyDeviceToHost, ac->stream),
         "get_solution");
  HIP_OK(hipStreamSynchronize(ac->stream), "sync");
  for (long c = 0; c < ac->nc; c++)
    for (int nd = 0; nd < N; nd++) {
      double* q = luh + (size_t(c) * N + nd) * 6;
      for (int v = 0; v < 4; v++) q[v] = u[(size_t(c) * N + nd) * 4 + v];
      q[4] = ac->mat[2 * c];
      q[5] = ac->mat[2 * c + 1];
    }
  return EXA_OK;
}

int exa_acoustic_set_material(exa_acoustic* ac, const double* rho, const double* c) {
  if (!ac) return argerr("exa_acoustic_set_material: NULL acoustic");
  for (long i = 0; i < ac->nc; i++) {
    if (rho) {
      if (!(rho[i] > 0)) return argerr("exa_acoustic_set_material: rho must be positive");
      ac->mat[2 * i] = rho[i];
    }
    if (c) ac->mat[2 * i + 1] = c[i];
  }
  return upload_material(ac);
}

int exa_acoustic_get_material(exa_acoustic* ac, double* rho, double* c) {
  if (!ac) return argerr("exa_acoustic_get_material: NULL acoustic");
  for (long i = 0; i < ac->nc; i++) {
    if (rho) rho[i] = ac->mat[2 * i];
    if (c) c[i] = ac->mat[2 * i + 1];
  }
  return EXA_OK;
}

int exa_acoustic_set_dt(exa_acoustic* ac, double dt) {
  if (!ac) return argerr("exa_acoustic_set_dt: NULL acoustic");
  if (!(dt > 0)) {
    double cmax = 0.0;
    for (long i = 0; i < ac->nc; i++) cmax = std::fmax(cmax, std::fabs(ac->mat[2 * i + 1]));
    if (!(cmax > 0)) return argerr("exa_acoustic_set_dt: wave speed is zero everywhere");
    dt = ac->k.cfl * ac->k.pnpm / (3.0 * (cmax / ac->h));
  }
  ac->dt = dt;
  ac->src_tab_steps = 0;  // the source table depends on dt
  return EXA_OK;
}

int exa_acoustic_set_step(exa_acoustic* ac, int step) {
  if (!ac || step < 0) return argerr("exa_acoustic_set_step: invalid argument");
  return set_step(ac, step);
}

int exa_acoustic_time(exa_acoustic* ac, int* step, double* t, double* dt) {
  if (!ac) return argerr("exa_acoustic_time: NULL acoustic");
  if (step) *step = ac->step;
  if (t) *t = ac->step * ac->dt;
  if (dt) *dt = ac->dt;
  return EXA_OK;
}

int exa_acoustic_set_source(exa_acoustic* ac, const double* x, double amp, double f0, double t0) {
  if (!ac) return argerr("exa_acoustic_set_source: NULL acoustic");
  if (amp == 0.0 || !x) {
    ac->has_src = false;
    ac->src_cell = -1;
    return EXA_OK;
  }
  const double L = ac->n * ac->h;
  for (int d = 0; d < 3; d++)
    if (!(x[d] >= 0 && x[d] <= L)) return argerr("exa_acoustic_set_source: source outside the domain");
  ac->has_src = true;
  for (int d = 0; d < 3; d++) ac->src_x[d] = x[d];
  ac->amp = amp;
  ac->f0 = f0;
  ac->t0 = t0;
  ac->src_cell = locate(ac, x, nullptr);
  const long c = ac->src_cell;
  const long ix = c % ac->n, iy = (c / ac->n) % ac->n, iz = c / (long(ac->n) * ac->n);
  const double centre[3] = {(ix + 0.5) * ac->h, (iy + 0.5) * ac->h, (iz + 0.5) * ac->h};
  double xr[3];
  for (int d = 0; d < 3; d++) xr[d] = (x[d] - centre[d]) / ac->h + 0.5;
  const int B = ac->B;
  const double* w = ac->tab.w;
  std::vector<double> g(ac->N);
  for (int i = 0; i < B; i++)
    for (int j = 0; j < B; j++)
      for (int kk = 0; kk < B; kk++) {
        const double basis = lagrange(ac->tab.x, B, kk, xr[0]) * lagrange(ac->tab.x, B, j, xr[1]) *
                             lagrange(ac->tab.x, B, i, xr[2]);
        const double winv = 1.0 / (w[kk] * ac->h * w[j] * ac->h * w[i] * ac->h);
        g[(i * B + j) * B + kk] = winv * basis;
      }
  HIP_OK(hipMemcpy(ac->d_src_g, g.data(), sizeof(double) * g.size(), hipMemcpyHostToDevice), "upload source");
  ac->src_tab_steps = 0;
  return EXA_OK;
}

int exa_acoustic_set_receivers(exa_acoustic* ac, int nrec, const double* xr) {
  if (!ac || nrec < 0 || (nrec > 0 && !xr)) return argerr("exa_acoustic_set_receivers: invalid argument");
  const Call call(ac);
  for (int* p : {ac->d_rcell, ac->d_rstart, ac->d_rorder})
    if (p) (void)hipFree(p);
  if (ac->d_rw) (void)hipFree(ac->d_rw);
  ac->d_rcell = ac->d_rstart = ac->d_rorder = nullptr;
  if (ac->d_rec_p) (void)hipFree(ac->d_rec_p);
  ac->d_rec_p = nullptr;
  ac->d_rw = nullptr;
  ac->nrec = 0;
  if (nrec == 0) return EXA_OK;
  const int B = ac->B, N = ac->N;
  std::vector<int> cells(nrec);
  std::vector<double> wts(size_t(nrec) * N);
  for (int r = 0; r < nrec; r++) {
    double xi[3];
    cells[r] = static_cast<int>(locate(ac, xr + 3 * r, xi));
    double phi[3][exa::kMaxBasis];
    for (int d = 0; d < 3; d++)
      for (int kk = 0; kk < B; kk++) phi[d][kk] = lagrange(ac->tab.x, B, kk, xi[d]);
    for (int z = 0; z < B; z++)
      for (int y = 0; y < B; y++)
        for (int x = 0; x < B; x++) wts[size_t(r) * N + (z * B + y) * B + x] = phi[0][x] * phi[1][y] * phi[2][z];
  }
  // by cell, each cell's receivers in their order
  std::vector<int> start(size_t(ac->nc) + 1, 0), order(nrec);
  for (int r = 0; r < nrec; r++) start[cells[r] + 1]++;
  for (long c = 0; c < ac->nc; c++) start[c + 1] += start[c];
  std::vector<int> at(start.begin(), start.end() - 1);
  for (int r = 0; r < nrec; r++) order[at[cells[r]]++] = r;
  HIP_OK(allocate(ac, &ac->d_rstart, start.size()), "hipMalloc(receivers)");
  HIP_OK(allocate(ac, &ac->d_rorder, nrec), "hipMalloc(receivers)");
  HIP_OK(hipMemcpy(ac->d_rstart, start.data(), sizeof(int) * start.size(), hipMemcpyHostToDevice), "upload receivers");
  HIP_OK(hipMemcpy(ac->d_rorder, order.data(), sizeof(int) * nrec, hipMemcpyHostToDevice), "upload receivers");
  HIP_OK(allocate(ac, &ac->d_rcell, nrec), "hipMalloc(receivers)");
  HIP_OK(allocate(ac, &ac->d_rw, wts.size()), "hipMalloc(receivers)");
  HIP_OK(hipMemcpy(ac->d_rcell, cells.data(), sizeof(int) * nrec, hipMemcpyHostToDevice), "upload receivers");
  HIP_OK(hipMemcpy(ac->d_rw, wts.data(), sizeof(double) * wts.size(), hipMemcpyHostToDevice), "upload receivers");
  ac->nrec = nrec;
  return EXA_OK;
}

int exa_acoustic_run(exa_acoustic* ac, int nsteps, int use_graph, double* rec) {
  if (!ac || nsteps < 0) return argerr("exa_acoustic_run: invalid argument");
  if (nsteps == 0) return EXA_OK;
  const Call call(ac);
  const int s0 = ac->step;
  RC_OK(ensure_source_table(ac, s0 + nsteps));
  RC_OK(grow(ac, &ac->d_rec, &ac->rec_cap, long(nsteps) * (ac->nrec > 0 ? ac->nrec : 1)));
  hipEvent_t e0 = nullptr, e1 = nullptr;
  HIP_OK(hipEventCreate(&e0), "event");
  HIP_OK(hipEventCreate(&e1), "event");
  HIP_OK(hipEventRecord(e0, ac->stream), "event");
  int rc = EXA_OK;
  if (use_graph) {
    // one captured step reading the device step counter; receivers go to
    // d_rec + (step - s0) * nrec through the base pointer of this run
    exa::AcousticArgs a = args(ac, ac->d_u);
    a.rec = ac->d_rec - long(s0) * ac->nrec;
    hipGraph_t g = nullptr;
    hipGraphExec_t ge = nullptr;
    HIP_OK(hipStreamBeginCapture(ac->stream, hipStreamCaptureModeThreadLocal), "begin capture");
    const int o = ac->k.order;
    rc = status(exa::launch_acoustic(exa::kAcPredictUpdate, o, a, ac->stream), "acoustic predictor");
    if (!rc) rc = status(exa::launch_acoustic(exa::kAcCorrector, o, a, ac->stream), "acoustic corrector");
    if (!rc && ac->nrec > 0) rc = status(exa::launch_acoustic(exa::kAcReceivers, o, a, ac->stream), "receivers");
    if (!rc) rc = status(exa::launch_acoustic_advance(ac->d_step, ac->stream), "advance");
    const hipError_t e = hipStreamEndCapture(ac->stream, &g);
    if (!rc && e != hipSuccess) rc = fail(e, "end capture");
    if (!rc) {
      const hipError_t ei = hipGraphInstantiate(&ge, g, nullptr, nullptr, 0);
      if (ei != hipSuccess) rc = fail(ei, "instantiate");
    }
    for (int i = 0; !rc && i < nsteps; i++) {
      const hipError_t el = hipGraphLaunch(ge, ac->stream);
      if (el != hipSuccess) rc = fail(el, "graph launch");
    }
    (void)hipStreamSynchronize(ac->stream);
    if (ge) (void)hipGraphExecDestroy(ge);
    if (g) (void)hipGraphDestroy(g);
  } else {
    if (ac->timing) {
      while (ac->ev.size() < size_t(3) * nsteps) {
        hipEvent_t e = nullptr;
        HIP_OK(hipEventCreate(&e), "event create");
        ac->ev.push_back(e);
      }
      ac->timed_steps = nsteps;
    }
    double* rec_base = ac->d_rec - long(s0) * ac->nrec;
    if (!ac->timing)
      rc = enqueue_forward_steps(ac, s0, nsteps, rec_base);
    else  // predictor and corrector apart, to time each
      for (int i = 0; !rc && i < nsteps; i++)
        rc = enqueue_forward(ac, ac->d_u, ac->d_u, s0 + i, rec_base, &ac->ev[size_t(3) * i]);
  }
  if (!rc) {
    const hipError_t e = hipEventRecord(e1, ac->stream);
    if (e != hipSuccess) rc = fail(e, "event");
  }
  if (!rc) {
    const hipError_t e = hipEventSynchronize(e1);
    if (e != hipSuccess) rc = fail(e, "sync");
  }
  float ms = 0;
  if (!rc) (void)hipEventElapsedTime(&ms, e0, e1);
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  if (rc) return rc;
  ac->ms[0] = ms;
  ac->ms[1] = ac->ms[2] = 0;
  RC_OK(set_step(ac, s0 + nsteps));
  if (rec && ac->nrec > 0)
    HIP_OK(hipMemcpy(rec, ac->d_rec, sizeof(double) * nsteps * ac->nrec, hipMemcpyDeviceToHost), "receivers");
  return EXA_OK;
}

int exa_acoustic_misfit_gradient(exa_acoustic* ac, int nsteps, int every, const double* obs, double* J,
                                 double* grad_c) {
  if (!ac || nsteps < 1 || every < 1 || !obs || !J || !grad_c)
    return argerr("exa_acoustic_misfit_gradient: invalid argument");
  if (ac->nrec < 1) return argerr("exa_acoustic_misfit_gradient: no receivers");
  if (ac->k.split_ck) {
    exa::set_error("exa_acoustic_misfit_gradient: the adjoint transposes the generic predictor (context dialect "
                   "EXA_DIALECT_SPLIT_CK)");
    return EXA_ERR_UNSUPPORTED;
  }
  const Call call(ac);
  const int s0 = ac->step, K = nsteps, R = ac->nrec, o = ac->k.order;
  const int nck = (K + every - 1) / every;
  const int seg = (every < K ? every : K) - 1;  // states of a segment besides its checkpoint
  const size_t su = size_t(ac->nc) * ac->N * 4, sq = size_t(ac->nc) * 6 * ac->F * 4;
  RC_OK(ensure_source_table(ac, s0 + K));
  RC_OK(grow(ac, &ac->d_rec, &ac->rec_cap, long(K) * R));
  RC_OK(grow(ac, &ac->d_res, &ac->res_cap, long(K) * R));
  struct {
    double** p;
    size_t n;
  } const adjoint[] = {{&ac->d_ubar, su}, {&ac->d_fbar, sq}, {&ac->d_fbar2, sq}, {&ac->d_gc, size_t(ac->nc)}};
  for (const auto& b : adjoint)  // each by itself: an earlier call may have got only some of them
    if (!*b.p) HIP_OK(allocate(ac, b.p, b.n), "hipMalloc(adjoint)");
  RC_OK(gradient_buffers(ac, su, sq, nck, seg));
  double *d_ck = ac->d_ck, *d_seg = ac->d_seg;
  double* d_segq = ac->segq_cap >= long(sq) * (seg + 1) ? ac->d_segq : nullptr;
  std::vector<hipEvent_t> ev(2 + 3 * nck, nullptr);
  int rc = EXA_OK;
  for (auto& e : ev)
    if (!rc && hipEventCreate(&e) != hipSuccess) rc = fail(hipErrorUnknown, "event");
  double* rec_base = ac->d_rec - long(s0) * R;
  // forward sweep with checkpoints
  if (!rc && hipEventRecord(ev[0], ac->stream) != hipSuccess) rc = fail(hipErrorUnknown, "event");
  exa::TraceRange tr_fwd("exa.acoustic.adjoint.forward");
  // states k0 .. of segment j (k0 = j every): the checkpoint, then d_seg; their steps' faces
  auto state = [&](int j, int k) { return k == j * every ? d_ck + su * j : d_seg + su * (k - j * every - 1); };
  auto faces = [&](int j, int k) { return d_segq ? d_segq + sq * (k - j * every) : nullptr; };
  for (int j = 0; !rc && j < nck; j++) {
    const int k0 = j * every;
    const hipError_t e = hipMemcpyAsync(d_ck + su * j, ac->d_u, sizeof(double) * su, hipMemcpyDeviceToDevice,
                                        ac->stream);
    if (e != hipSuccess) rc = fail(e, "checkpoint");
    if (!rc && j + 1 < nck) rc = enqueue_forward_steps(ac, s0 + k0, every, rec_base);
    // the backward sweep starts in the last segment: keep its states
    for (int k = k0; !rc && j + 1 == nck && k < K; k++)
      rc = enqueue_forward(ac, state(j, k), k + 1 < K ? state(j, k + 1) : ac->d_u, s0 + k, rec_base, nullptr,
                           faces(j, k));
  }
  if (!rc && hipEventRecord(ev[1], ac->stream) != hipSuccess) rc = fail(hipErrorUnknown, "event");
  std::vector<double> rec(size_t(K) * R), res(size_t(K) * R);
  if (!rc) {
    const hipError_t e = hipMemcpyAsync(rec.data(), ac->d_rec, sizeof(double) * rec.size(), hipMemcpyDeviceToHost,
                                        ac->stream);
    if (e != hipSuccess) rc = fail(e, "receivers");
    else if (hipStreamSynchronize(ac->stream) != hipSuccess) rc = fail(hipErrorUnknown, "sync");
  }
  double Jv = 0.0;
  for (size_t i = 0; i < rec.size(); i++) {
    res[i] = rec[i] - obs[i];
    Jv += 0.5 * res[i] * res[i];
  }
  if (!rc) {
    hipError_t e = hipMemcpyAsync(ac->d_res, res.data(), sizeof(double) * res.size(), hipMemcpyHostToDevice,
                                  ac->stream);
    if (e == hipSuccess) e = hipMemsetAsync(ac->d_ubar, 0, sizeof(double) * su, ac->stream);
    if (e == hipSuccess) e = hipMemsetAsync(ac->d_gc, 0, sizeof(double) * ac->nc, ac->stream);
    if (e != hipSuccess) rc = fail(e, "adjoint init");
  }
  // backward sweep, segment by segment
  exa::TraceRange tr_bwd("exa.acoustic.adjoint.backward");
  for (int j = nck - 1; !rc && j >= 0; j--) {
    const int k0 = j * every, k1 = (k0 + every < K) ? k0 + every : K;
    (void)hipEventRecord(ev[2 + 3 * j], ac->stream);
    for (int k = k0; !rc && j + 1 < nck && k < k1 - 1; k++)
      rc = enqueue_forward(ac, state(j, k), state(j, k + 1), s0 + k, nullptr, nullptr, faces(j, k));
    (void)hipEventRecord(ev[3 + 3 * j], ac->stream);
    for (int k = k1 - 1; !rc && k >= k0; k--) {
      exa::AcousticArgs a = args(ac, state(j, k));
      a.step_override = s0 + k;
      if (d_segq) a.qb = a.qb_out = faces(j, k);
      if (k == K - 1) {
        rc = status(exa::launch_acoustic_receivers_adj(o, a, ac->d_res + long(k) * R, ac->stream), "receiver adjoint");
        if (!rc) rc = status(exa::launch_acoustic(exa::kAcFbar, o, a, ac->stream), "adjoint fbar");
      }
      // the faces are there from the segment's steps, all but its last one's
      if (!rc && (!d_segq || (k == k1 - 1 && j + 1 < nck)))
        rc = status(exa::launch_acoustic(exa::kAcPredictFaces, o, a, ac->stream), "acoustic faces");
      if (k > 0) a.res_prev = ac->d_res + long(k - 1) * R;
      a.fbar_out = ac->d_fbar2;
      if (!rc) rc = status(exa::launch_acoustic(exa::kAcAdjoint, o, a, ac->stream), "adjoint step");
      std::swap(ac->d_fbar, ac->d_fbar2);
    }
    (void)hipEventRecord(ev[4 + 3 * j], ac->stream);
  }
  if (!rc) {
    const hipError_t e = hipMemcpyAsync(grad_c, ac->d_gc, sizeof(double) * ac->nc, hipMemcpyDeviceToHost, ac->stream);
    if (e != hipSuccess) rc = fail(e, "gradient");
    else if (hipStreamSynchronize(ac->stream) != hipSuccess) rc = fail(hipErrorUnknown, "sync");
  }
  if (!rc) {
    float f = 0;
    (void)hipEventElapsedTime(&f, ev[0], ev[1]);
    ac->ms[0] = f;
    ac->ms[1] = ac->ms[2] = 0;
    for (int j = 0; j < nck; j++) {
      float a1 = 0, a2 = 0;
      (void)hipEventElapsedTime(&a1, ev[2 + 3 * j], ev[3 + 3 * j]);
      (void)hipEventElapsedTime(&a2, ev[3 + 3 * j], ev[4 + 3 * j]);
      ac->ms[1] += a1;
      ac->ms[2] += a2;
    }
  }
  (void)hipStreamSynchronize(ac->stream);
  for (auto& e : ev)
    if (e) (void)hipEventDestroy(e);
  if (rc) return rc;
  *J = Jv;
  return set_step(ac, s0 + K);
}

int exa_acoustic_set_timing(exa_acoustic* ac, int enabled) {
  if (!ac) return argerr("exa_acoustic_set_timing: NULL acoustic");
  ac->timing = enabled != 0;
  ac->timed_steps = 0;
  return EXA_OK;
}

int exa_acoustic_set_predictor(exa_acoustic* ac, int variant) {
  if (!ac) return argerr("exa_acoustic_set_predictor: NULL acoustic");
  if (variant != 0 && variant != 1) return argerr("exa_acoustic_set_predictor: variant must be 0 (x-line) or 1 (node)");
  if (variant == 1 && ac->k.split_ck) {
    exa::set_error("exa_acoustic_set_predictor: the split Cauchy-Kowalevski predictor has the x-line form only");
    return EXA_ERR_UNSUPPORTED;
  }
  ac->pred_variant = variant;
  return EXA_OK;
}

int exa_acoustic_phase_times(exa_acoustic* ac, double* ms_predictor, double* ms_corrector, int* nsteps) {
  if (!ac) return argerr("exa_acoustic_phase_times: NULL acoustic");
  double a = 0, b = 0;
  for (int i = 0; i < ac->timed_steps; i++) {
    float x = 0, y = 0;
    HIP_OK(hipEventElapsedTime(&x, ac->ev[size_t(3) * i], ac->ev[size_t(3) * i + 1]), "elapsed");
    HIP_OK(hipEventElapsedTime(&y, ac->ev[size_t(3) * i + 1], ac->ev[size_t(3) * i + 2]), "elapsed");
    a += x;
    b += y;
  }
  if (ms_predictor) *ms_predictor = a;
  if (ms_corrector) *ms_corrector = b;
  if (nsteps) *nsteps = ac->timed_steps;
  return EXA_OK;
}

int exa_acoustic_last_times(exa_acoustic* ac, double* ms_forward, double* ms_recompute, double* ms_adjoint) {
  if (!ac) return argerr("exa_acoustic_last_times: NULL acoustic");
  if (ms_forward) *ms_forward = ac->ms[0];
  if (ms_recompute) *ms_recompute = ac->ms[1];
  if (ms_adjoint) *ms_adjoint = ac->ms[2];
  return EXA_OK;
}

}  // extern "C"
