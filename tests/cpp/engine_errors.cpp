// The serving engine (csrc/server.cpp) on the CPU, with the HIP runtime and the
// library's kernels replaced by stand-ins that record what each request's
// systems have been through: its inputs, matrix, descriptor, set-up, starts and
// turns.  An allocation of the engine is made to fail in turn; the run that meets it
// may end in an error, and no later launch may then reach a slot whose descriptor
// was not uploaded, a system not set up or started, or a gradient without its turn.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <set>

#include "batched.h"
#include "mg.h"

namespace admfem {
struct Server;
Server *server_create(const admfem_server_opts &o);
void server_free(Server *sv);
int server_add_topology(Server *sv, System *s, double jitter);
int64_t server_submit(Server *sv, const admfem_request &r);
void server_run(Server *sv, double timeout);
void server_result(Server *sv, int64_t id, admfem_result &out);

static long calls = 0, fail_at = -1, bad = 0;
static void check(bool ok, const char *what) {
  if (!ok) {
    bad++;
    printf("allocation %ld: %s\n", fail_at, what);
  }
}
static bool fails() { return calls++ == fail_at; }

// what a slot's system has been through (by the address of its right-hand side)
struct Slot { bool up = false, running = false; };
static Slot slots[8];
static std::set<const void *> with_inputs, with_matrix, with_turn;

void set_error(const std::string &) {}
void *device_alloc(size_t bytes, int &device) {
  device = 0;
  if (fails()) throw OutOfMemory{{ADMFEM_ERR_HIP, "out of memory"}};
  return calloc(1, bytes + 256);
}
void device_free(void *p, size_t, int) { free(p); }
void release_device_memory() {}

static MgPlan the_plan;
const MgPlan *mg_plan(System &, hipStream_t) { return &the_plan; }
void mg_allow_lds(const MgPlan &) {}
size_t mg_tail_lds(const MgPlan &) { return 0; }
size_t mg_setup_lds(const MgPlan &) { return 0; }
size_t mg_grid_floats(const MgPlan &) { return 64; }
void mg_grid_layout(const MgPlan &, float *, MgSys &) {}
void mg_parts(MgSys &, int, bool, double *) {}
void mg_stages(const MgPlan &, int npad, int (&n)[MG_STAGES]) {
  for (int &v : n) v = 0;
  n[MGS_ROWS] = n[MGS_GALERKIN] = npad / 256 + 1;
}
static void valid(const MgSys &d, int slot, const char *who) {
  check(slot >= 0 && slot < 8, "a launch on no slot");
  check(d.b && with_matrix.count(d.b), who);
}
void mg_batch_setup(const MgBatch &B, const MgSys *D, hipStream_t) {
  for (int k = 0; k < B.nsys; k++) {
    valid(D[B.list[k]], B.list[k], "set up without its descriptor or matrix");
    slots[B.list[k]].up = true;
  }
}
void mg_batch_start(const MgBatch &B, const MgSys *D, MgScal *S, double, int, hipStream_t) {
  for (int k = 0; k < B.nsys; k++) {
    const int s = B.list[k];
    valid(D[s], s, "started without its descriptor or matrix");
    check(slots[s].up, "started and not set up");
    slots[s].running = true;
    S[s] = MgScal{};
  }
}
void mg_batch_iterations(const MgBatch &B, const MgSys *D, MgScal *S, int, MgScal *host,
                         hipStream_t) {
  for (int k = 0; k < B.nsys; k++) {
    const int s = B.list[k];
    valid(D[s], s, "iterated without its descriptor or matrix");
    check(slots[s].up && slots[s].running, "iterated and not started");
    S[s].a.it += 4;  // (a solve takes two chunks)
    if (S[s].a.it >= 8) S[s].a.status = S[s].checked = 1;
    host[s] = S[s];
  }
}
void batch_maps(int, int, const int *, const int *, const int *, int, int2 *, hipStream_t) {}
void serve_inputs(const ServeIn *j, int n, int, hipStream_t) {
  for (int k = 0; k < n; k++) with_inputs.insert(j[k].dst[0]);
}
void launch_assemble_to(const System &, const double2 *, const admfem_problem &p, const SellOut &o,
                        hipStream_t) {
  check(with_inputs.count(p.kappa), "assembled without its inputs");
  with_matrix.insert(o.rhs);
  with_turn.erase(o.rhs);
}
void serve_turn(const ServeTurn *j, int n, int, hipStream_t) {
  for (int k = 0; k < n; k++) with_turn.insert(j[k].u);
}
void serve_outputs(const ServeOut *, int, int, hipStream_t) {}
void launch_kappa_gradient_to(const System &, const double2 *, const double *u, const double *,
                              double, double *, hipStream_t) {
  check(with_turn.count(u), "a gradient without its turn");
  with_turn.erase(u);
}
// (the Jacobi-PCG side is not reached)
void batch_init(const BSys *, BScal *, int, int, double, double, int, hipStream_t) { abort(); }
void batch_final(const BSys *, const BScal *, int, int, double *, hipStream_t) { abort(); }
void batch_scale(const System &, const double *, const double *, double *, float *, hipStream_t) { abort(); }
void batch_iterations(const int2 *, int, const int *, int, const BSys *, BScal *, int, hipStream_t) { abort(); }
void batch_spmv_repeat(const int2 *, int, const BSys *, const BScal *, int, hipStream_t) { abort(); }
void batch_map(int, const int *, const int *, int, int, int2 *, hipStream_t) { abort(); }
void launch_loss(const System &, const double *, const int *, const double *, int, double *, double *, hipStream_t) { abort(); }
void launch_scatter(const int *, const double *, double *, int, hipStream_t) { abort(); }
void launch_perm_coords(int, const int *, const double *, double *, double *, double2 *, hipStream_t) { abort(); }
void synth_inputs(const System &, const double *, const double *, unsigned long, double, const SynField &, const SynField *, double *, double *, double2 *, double *, double *, double *, hipStream_t) { abort(); }
void cg_solve(System &, const double *, double *, const admfem_solve_opts &, admfem_solve_stats &, hipStream_t) { abort(); }
}  // namespace admfem

using namespace admfem;

// the HIP calls that the engine makes
hipError_t hipMalloc(void **p, size_t n) {
  if (fails()) return hipErrorOutOfMemory;
  *p = calloc(1, n + 256);
  return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
  if (fails()) return hipErrorOutOfMemory;
  *p = calloc(1, n + 256);
  return hipSuccess;
}
hipError_t hipFree(void *p) { free(p); return hipSuccess; }
hipError_t hipHostFree(void *p) { free(p); return hipSuccess; }
hipError_t hipMemGetInfo(size_t *a, size_t *b) { *a = *b = (size_t)1 << 30; return hipSuccess; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemset(void *d, int v, size_t n) { memset(d, v, n); return hipSuccess; }
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) { memset(d, v, n); return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { *s = nullptr; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { abort(); }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *) { abort(); }
hipError_t hipGraphInstantiate(hipGraphExec_t *, hipGraph_t, hipGraphNode_t *, char *, size_t) { abort(); }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { abort(); }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { *e = nullptr; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { *e = nullptr; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *, hipEvent_t, hipEvent_t) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "refused"; }

// One engine with its k-th allocation (from the first run on) refused: three
// requests, a run that may fail, three more, a run that may not.  Returns the
// allocations made.
static long scenario(long k) {
  constexpr int N = 300, NPAD = 320, NG = 900;
  Mesh m;
  m.nnode = N;
  m.ngauss = NG;
  System s;
  s.mesh = &m;
  s.n = N;
  s.npad = NPAD;
  s.row_bd.assign(N, -1);
  s.slice_ptr = {0, 64 * 7 * 5};
  m.perm.resize(N);
  for (int i = 0; i < N; i++) m.perm[i] = i;
  for (Slot &q : slots) q = Slot{};
  with_inputs.clear();
  with_matrix.clear();
  with_turn.clear();
  fail_at = -1;
  admfem_server_opts o{};
  o.hbm_budget_bytes = 1 << 24;
  o.max_active = 8;
  o.rtol = 1e-8;
  o.max_iter = 1000;
  Server *sv = server_create(o);
  const int t = server_add_topology(sv, &s, 0.0);
  std::vector<double> a(NG), u(N), g(NG);
  int idx = 0;
  admfem_request r{};
  r.topo = t;
  r.source = ADMFEM_SRC_DEVICE;
  r.kappa = r.f = r.obs_val = a.data();
  r.obs_idx = &idx;
  r.nobs = 1;
  r.grad_out = g.data();
  for (int i = 0; i < 3; i++) server_submit(sv, r);
  calls = 0;
  fail_at = k;
  bool failed = false;
  try {
    server_run(sv, 1e9);
  } catch (const Error &) {
    failed = true;
  }
  const long made = calls;
  fail_at = -1 - k;  // (none from here on; printed by check)
  for (int i = 0; i < 3; i++) server_submit(sv, r);
  try {
    server_run(sv, 1e9);
  } catch (const Error &) {
    check(false, "a run after a failed one failed as well");
  }
  for (int i = 0; i < 6; i++) {
    admfem_result res{};
    server_result(sv, i, res);
    check(res.done, "a request is left over");
    check(res.status == ADMFEM_OK || (failed && i < 3), "a request failed for no reason");
  }
  server_free(sv);
  return made;
}

int main() {
  the_plan.ok = true;
  const long made = scenario(-1);
  check(made > 0, "no allocation in a run");
  for (long k = 0; k < made; k++) scenario(k);
  printf("%ld allocations refused in turn, %ld faults\n", made, bad);
  return bad ? 1 : 0;
}
