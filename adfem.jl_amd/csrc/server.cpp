// Serving engine: continuous batching of forward+adjoint requests on one GPU.
//
// A request runs the reference's pipeline for its own coefficients
// (assemble -> Dirichlet -> u = K^-1 F -> L -> lambda = K^-1 dL/du ->
// dL/dkappa).  The engine admits arrived requests while their device memory
// fits the HBM budget (an arena that grows to the budget by what waits, so
// admission rarely and release never calls hipMalloc/hipFree), advances every admitted system with
// one batched launch per CG step (batched.hip), and moves systems that
// converge to their next phase at the chunk boundaries, where finished
// requests release their memory to the waiting queue.
#include <algorithm>
#include <array>
#include <chrono>
#include <cmath>
#include <map>
#include <random>
#include <thread>
#include <unordered_set>

#include "batched.h"
#include "mg.h"

namespace admfem {

namespace {

constexpr size_t ALIGN = 256;
inline size_t up(size_t v) { return (v + ALIGN - 1) / ALIGN * ALIGN; }

// Best-fit allocator over device segments, coalescing on free.  `cap` bounds
// the segments' total; they are allocated as requests need them (the bytes
// of every waiting request at once), not all at creation: an arena of the
// whole budget cost its allocation at every start, and the driver clears what
// a process gives back: an engine made and closed for 64 requests in a loop,
// with a budget of 8 GiB, waited 180 ms in hipFree once the card's free memory
// had gone round.
struct Arena {
  size_t cap = 0, used = 0, peak = 0, held = 0;
  std::map<char *, size_t> segs;   // segment -> size
  std::map<char *, size_t> free_;  // block -> size
  void init(size_t bytes) {
    cap = up(bytes);
    size_t avail = 0, total = 0;
    HIPCHECK(hipMemGetInfo(&avail, &total));
    if (cap > avail) {  // (what the library keeps for later buffers is free, too)
      release_device_memory();
      HIPCHECK(hipMemGetInfo(&avail, &total));
    }
    REQUIRE(cap <= avail, ADMFEM_ERR_HIP, "the HBM budget exceeds the free device memory");
  }
  ~Arena() {
    for (auto &s : segs) (void)hipFree(s.first);
  }
  // A new segment of `want` bytes if the budget has room, else of `bytes`,
  // after giving back unused segments when it must.  False: no room now.
  bool grow(size_t bytes, size_t want) {
    if (held + bytes > cap)
      for (auto it = segs.begin(); it != segs.end();) {
        auto f = free_.find(it->first);
        if (f == free_.end() || f->second != it->second) {
          ++it;
          continue;
        }
        (void)hipFree(it->first);
        held -= it->second;
        free_.erase(f);
        it = segs.erase(it);
      }
    if (held + bytes > cap) return false;
    const size_t size = std::max(bytes, std::min(want, cap - held));
    char *p = nullptr;
    if (hipMalloc(&p, size) != hipSuccess) {
      (void)hipGetLastError();
      release_device_memory();
      if (hipMalloc(&p, size) != hipSuccess) {
        (void)hipGetLastError();
        return false;
      }
    }
    segs[p] = size;
    free_[p] = size;
    held += size;
    return true;
  }
  // (want 0: only from the segments there are)
  bool alloc(size_t bytes, size_t want, char *&out) {
    bytes = up(bytes);
    for (int tries = 0; tries < 2; tries++) {
      auto best = free_.end();
      for (auto it = free_.begin(); it != free_.end(); ++it)
        if (it->second >= bytes && (best == free_.end() || it->second < best->second)) best = it;
      if (best == free_.end()) {
        if (tries || !want || !grow(bytes, up(want))) return false;
        continue;
      }
      out = best->first;
      const size_t rest = best->second - bytes;
      free_.erase(best);
      if (rest) free_[out + bytes] = rest;
      used += bytes;
      peak = std::max(peak, used);
      return true;
    }
    return false;
  }
  void release(char *p, size_t bytes) {
    bytes = up(bytes);
    used -= bytes;
    auto it = free_.emplace(p, bytes).first;
    auto nx = std::next(it);
    // (a segment's first block never joins the block before it)
    if (nx != free_.end() && it->first + it->second == nx->first && !segs.count(nx->first)) {
      it->second += nx->second;
      free_.erase(nx);
    }
    if (it != free_.begin() && !segs.count(it->first)) {
      auto pv = std::prev(it);
      if (pv->first + pv->second == it->first) {
        pv->second += it->second;
        free_.erase(it);
      }
    }
  }
};

struct Topo {
  System *sys;
  const MgPlan *plan;        // multigrid CG's grids, or null: Jacobi-PCG
  double jitter;
  int nblk;                  // batched blocks of 256 rows
  std::vector<int> interior; // user ids of interior nodes
};

enum { Q_WAIT = 0, Q_FWD = 1, Q_ADJ = 2, Q_DONE = 3 };

struct Req {
  admfem_request r;
  admfem_result res{};
  int state = Q_WAIT;
  bool mg = false;           // multigrid CG (else Jacobi-PCG)
  int slot = -1;
  char *mem = nullptr;       // its memory in the arena
  size_t bytes = 0;          // how much (of the layout it was admitted with)
  // device buffers (inside the arena)
  double2 *xy;
  double *x, *y, *kappa, *f, *uprev, *b, *sv64, *diag64, *dsq, *xa, *xb, *u64, *lam64,
      *grad, *obsv, *loss2, *part, *stage;
  float *sv32, *ysa, *ysb, *ra, *rb, *pa, *pb, *qa, *qb;
  // multigrid CG: FP64 x, r, q, two directions; FP32 vectors; the grids
  double *mgx, *mgr, *mgr1, *mgq, *mgp0, *mgp1;
  float *sq, *minv, *z, *rs, *x0, *t, *ts, *grid;
  float2 *wrq;
  int *obsi;
  int nobs = 0;
  std::vector<int> h_obs;  // synthetic observation indices, kept until the request is done
};

double now_s(std::chrono::steady_clock::time_point t0) {
  return std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
}

}  // namespace

// small kernels of the engine (batched.hip)
void launch_perm_coords(int n, const int *iperm, const double *coords_user, double *x,
                        double *y, double2 *xy, hipStream_t st);

struct Server {
  admfem_server_opts o{};
  hipStream_t st = nullptr;
  Arena arena;
  std::vector<Topo> topos;
  std::vector<Req> reqs;
  int max_slots = 0;
  std::vector<int> free_slots;
  DevBuf<BSys> d_desc;
  DevBuf<BScal> d_scal;
  BScal *h_scal = nullptr;       // pinned mirror
  double *h_loss = nullptr;      // pinned, per slot: loss and bad-index flag
  BSys *h_desc = nullptr;        // pinned staging of the descriptors
  // multigrid requests: descriptors and states by slot, their pinned staging
  // and mirror, and the maps of the batch, of the set-ups and of the starts
  DevBuf<MgSys> d_mg;
  DevBuf<MgScal> d_mgs;
  MgSys *h_mg = nullptr;
  MgScal *h_mgs = nullptr;
  std::vector<int> starts;       // multigrid requests whose solve is to start
  DevBuf<double> d_loss;         // per slot: loss and bad-index flag
  // the requests whose inputs, turn or outputs go out together: pinned and
  // device job lists (rewritten only after the stream has passed them)
  template <class T> struct Jobs {
    T *h = nullptr;
    DevBuf<T> d;
    int n = 0, longest = 0;
    void alloc(int cap) {
      HIPCHECK(hipHostMalloc((void **)&h, sizeof(T) * cap, hipHostMallocDefault));
      d.alloc(cap);
    }
    void add(const T &job, int len) {
      h[n++] = job;
      longest = std::max(longest, len);
    }
    template <class F> void flush(F launch, hipStream_t st) {
      if (!n) return;
      HIPCHECK(hipMemcpyAsync(d.p, h, sizeof(T) * n, hipMemcpyHostToDevice, st));
      launch(d.p, n, longest, st);
      clear();
    }
    void clear() { n = longest = 0; }
    ~Jobs() {
      if (h) (void)hipHostFree(h);
    }
  };
  Jobs<ServeIn> jobs_in;
  Jobs<ServeTurn> jobs_turn;
  Jobs<ServeOut> jobs_out;
  static constexpr int MG_BATCH_SUM = 128;  // partials summed by the wide kernels
  int *h_list = nullptr;         // pinned staging: the batch's slots, then
                                 // their first logical blocks (list_cap each)
  size_t map_cap = 0, list_cap = 0;
  DevBuf<int2> d_map;
  DevBuf<int> d_list;            // slots [list_cap], first blocks [list_cap + 1]
  bool started = false;
  bool use_graph = false;
  std::chrono::steady_clock::time_point t0;
  // stats
  int64_t steps = 0, iters = 0, batch_sum = 0;
  int peak_active = 0;
  double wall = 0;

  ~Server() {
    drop_graphs();
    if (h_scal) (void)hipHostFree(h_scal);
    if (h_loss) (void)hipHostFree(h_loss);
    if (h_desc) (void)hipHostFree(h_desc);
    if (h_mg) (void)hipHostFree(h_mg);
    if (h_mgs) (void)hipHostFree(h_mgs);
    if (h_list) (void)hipHostFree(h_list);
    if (st) (void)hipStreamDestroy(st);
  }

  // ------------------------------------------------------------ layout
  // (pl: the plan of a request that runs on multigrid CG, else null)
  static size_t layout(const System &s, const MgPlan *pl, Req *q, char *base, int nobs) {
    const Mesh &m = *s.mesh;
    const size_t np = s.npad, ng = m.ngauss, ns = std::max<size_t>(1, s.slice_ptr.back());
    const size_t nblk = (np + BATCH_NT - 1) / BATCH_NT;
    const size_t nv = s.degree == 2 ? (size_t)m.nnode : np;  // vertices (coordinates)
    size_t off = 0;
    auto take = [&](size_t bytes) {
      size_t o = off;
      off += up(bytes);
      return base ? (void *)(base + o) : nullptr;
    };
    auto D = [&](size_t n) { return (double *)take(n * sizeof(double)); };
    auto F = [&](size_t n) { return (float *)take(n * sizeof(float)); };
    double *x = D(nv), *y = D(nv), *kappa = D(ng), *f = D(ng), *uprev = D(np), *b = D(np),
           *sv64 = D(ns), *diag64 = D(np), *dsq = D(np),
           *u64 = D(np), *lam64 = D(np), *grad = D(ng), *obsv = D(nobs + 1),
           *part = D(pl ? 5 * nblk + 6 : 4 * nblk), *stage = D(2 * np);
    double2 *xy = (double2 *)take(nv * sizeof(double2));
    float *sv32 = F(ns);
    if (pl) {
      double *mgx = D(np), *mgr = D(np), *mgr1 = D(np), *mgq = D(np), *mgp0 = D(np), *mgp1 = D(np);
      float *sq = F(np), *minv = F(np), *z = F(np), *rs = F(np), *x0 = F(np), *t = F(np),
            *ts = F(np), *grid = F(mg_grid_floats(*pl));
      float2 *wrq = (float2 *)take(np * sizeof(float2));
      if (q) {
        q->wrq = wrq;
        q->mgx = mgx; q->mgr = mgr; q->mgr1 = mgr1; q->mgq = mgq; q->mgp0 = mgp0; q->mgp1 = mgp1;
        q->sq = sq; q->minv = minv; q->z = z; q->rs = rs; q->x0 = x0; q->t = t; q->ts = ts;
        q->grid = grid;
      }
    } else {
      double *xa = D(np), *xb = D(np);
      float *ysa = F(np), *ysb = F(np), *ra = F(np), *rb = F(np), *pa = F(np), *pb = F(np),
            *qa = F(np), *qb = F(np);
      if (q) {
        q->xa = xa; q->xb = xb; q->ysa = ysa; q->ysb = ysb;
        q->ra = ra; q->rb = rb; q->pa = pa; q->pb = pb; q->qa = qa; q->qb = qb;
      }
    }
    int *obsi = (int *)take((nobs + 1) * sizeof(int));
    if (q) {
      q->x = x; q->y = y; q->xy = xy; q->kappa = kappa; q->f = f; q->uprev = uprev; q->b = b;
      q->sv64 = sv64; q->diag64 = diag64; q->dsq = dsq;
      q->u64 = u64; q->lam64 = lam64; q->grad = grad; q->obsv = obsv;
      q->part = part; q->stage = stage; q->sv32 = sv32; q->obsi = obsi;
    }
    return off;
  }
  // The solver of a request about to be admitted.  Multigrid CG's memory is 1.2 to
  // 1.5 times Jacobi-PCG's (P1 of side 511: 114.5 against 94.2 MB; 32: 0.57 against
  // 0.39), so a budget may hold the request with Jacobi-PCG alone.
  void size_up(Req &q, bool jacobi) {
    q.nobs = nobs_of(q);
    q.mg = topos[q.r.topo].plan && o.mode == ADMFEM_MODE_BATCHED && !jacobi;
    if (q.mg && bytes_of(q) > arena.cap) q.mg = false;
  }
  size_t bytes_of(const Req &q) const {
    const Topo &T = topos[q.r.topo];
    return layout(*T.sys, q.mg ? T.plan : nullptr, nullptr, nullptr, q.nobs);
  }

  int nobs_of(const Req &q) const {
    if (q.r.source == ADMFEM_SRC_SYNTH)
      return std::max<int>(1, (int)topos[q.r.topo].interior.size() / 100);
    return q.r.nobs;
  }

  // ------------------------------------------------------------ phases
  void write_desc(Req &q, const double *b) {
    const System &s = *topos[q.r.topo].sys;
    // staged in pinned memory: the copy is asynchronous, and a slot's entry
    // is rewritten only after the stream has drained its previous request
    BSys &d = h_desc[q.slot];
    d = BSys{};
    d.sp = s.d_slice_ptr.p;
    d.sc = s.d_sell_col.p;
    d.sd = s.d_sell_d16.p;
    d.row_bd = s.d_row_bd.p;
    d.sv64 = q.sv64;
    d.diag64 = q.diag64;
    d.sv32 = q.sv32;
    d.dsq = q.dsq;
    d.b = b;
    d.x[0] = q.xa;
    d.x[1] = q.xb;
    d.ys[0] = q.ysa;
    d.ys[1] = q.ysb;
    d.r[0] = q.ra;
    d.r[1] = q.rb;
    d.p[0] = q.pa;
    d.p[1] = q.pb;
    d.q[0] = q.qa;
    d.q[1] = q.qb;
    d.part = q.part;
    d.n = s.n;
    d.npad = s.npad;
    d.nblk = topos[q.r.topo].nblk;
    HIPCHECK(hipMemcpyAsync(d_desc.p + q.slot, &d, sizeof(BSys), hipMemcpyHostToDevice, st));
  }

  void write_mg_desc(Req &q) {
    const Topo &T = topos[q.r.topo];
    const System &s = *T.sys;
    MgSys &d = h_mg[q.slot];
    d = MgSys{};
    d.sp = s.d_slice_ptr.p;
    d.sc = s.d_sell_col.p;
    d.sd = s.d_sell_d16.p;
    d.row_bd = s.d_row_bd.p;
    d.sv64 = q.sv64;
    d.diag = q.diag64;
    d.sv32 = q.sv32;
    d.dsq = q.dsq;
    d.sq = q.sq;
    d.minv = q.minv;
    d.b = q.b;
    d.x = q.mgx;
    d.r[0] = q.mgr;
    d.r[1] = q.mgr1;
    d.q = q.mgq;
    d.p[0] = q.mgp0;
    d.p[1] = q.mgp1;
    d.z = q.z;
    d.rs = q.rs;
    d.x0 = q.x0;
    d.t = q.t;
    d.ts = q.ts;
    d.wrq = q.wrq;
    d.n = s.n;
    d.npad = s.npad;
    mg_parts(d, T.nblk, T.nblk > MG_BATCH_SUM, q.part);
    mg_grid_layout(*T.plan, q.grid, d);
  }

  // The descriptors of new requests, in one copy: of the slots between them
  // too, whose descriptors are what they were (or nobody's).
  void upload_mg_descs(const std::vector<int> &reqs_) {
    int lo = max_slots, hi = -1;
    for (int i : reqs_) {
      lo = std::min(lo, reqs[i].slot);
      hi = std::max(hi, reqs[i].slot);
    }
    HIPCHECK(hipMemcpyAsync(d_mg.p + lo, h_mg + lo, sizeof(MgSys) * (hi - lo + 1),
                            hipMemcpyHostToDevice, st));
  }

  // The block maps of a set of multigrid requests, in buffers of the set's own
  // (rewritten only after the stream has passed their last use).
  struct MgSet {
    int *h = nullptr;          // pinned: slots, offsets, prefixes
    size_t h_cap = 0;
    DevBuf<int> d;
    DevBuf<int2> map;
    MgBatch batch;
    std::vector<std::pair<int, int>> slots;  // (slot, topology): what the maps
                                             // were made for
    ~MgSet() {
      if (h) (void)hipHostFree(h);
    }
  };
  void build_set(MgSet &B, const std::vector<int> &reqs_) {
    std::vector<std::pair<int, int>> slots;
    for (int i : reqs_) slots.emplace_back(reqs[i].slot, reqs[i].r.topo);
    if (slots == B.slots) return;
    const int ns = (int)reqs_.size();
    std::vector<std::array<int, MG_STAGES>> nblk(ns);
    MgBatch b;
    b.nsys = ns;
    for (int a = 0; a < ns; a++) {
      const Topo &T = topos[reqs[reqs_[a]].r.topo];
      int v[MG_STAGES];
      mg_stages(*T.plan, T.sys->npad, v);
      std::copy(v, v + MG_STAGES, nblk[a].begin());
      b.tail = std::max(b.tail, T.plan->tail);
      b.tail_lds = std::max(b.tail_lds, mg_tail_lds(*T.plan));
      b.setup_lds = std::max(b.setup_lds, mg_setup_lds(*T.plan));
      b.reduce = b.reduce || T.nblk > MG_BATCH_SUM;
    }
    std::vector<int> used;
    for (int q = 0; q < MG_STAGES; q++)
      for (int a = 0; a < ns; a++)
        if (nblk[a][q]) {
          used.push_back(q);
          break;
        }
    const int nu = (int)used.size();
    const size_t need = (size_t)ns + nu + (size_t)nu * (ns + 1);
    if (need > B.h_cap) {
      if (B.h) HIPCHECK(hipHostFree(B.h));
      B.h = nullptr;
      B.h_cap = std::max(need, 2 * B.h_cap);
      HIPCHECK(hipHostMalloc((void **)&B.h, sizeof(int) * B.h_cap, hipHostMallocDefault));
      B.d.alloc(B.h_cap);
    }
    int total = 0;
    for (int a = 0; a < ns; a++) B.h[a] = reqs[reqs_[a]].slot;
    for (int u = 0; u < nu; u++) {
      int *pref = B.h + ns + nu + (size_t)u * (ns + 1);
      int acc = 0;
      for (int a = 0; a < ns; a++) {
        pref[a] = acc;
        acc += nblk[a][used[u]];
      }
      pref[ns] = acc;
      B.h[ns + u] = total;
      b.nmap[used[u]] = acc;
      total += acc;
    }
    if ((size_t)total > B.map.n) B.map.alloc(std::max((size_t)total, 2 * B.map.n));
    for (int u = 0; u < nu; u++) b.map[used[u]] = B.map.p + B.h[ns + u];
    b.list = B.d.p;
    HIPCHECK(hipMemcpyAsync(B.d.p, B.h, sizeof(int) * need, hipMemcpyHostToDevice, st));
    batch_maps(ns, nu, B.d.p, B.d.p + ns + nu, B.d.p + ns, total, B.map.p, st);
    B.batch = b;
    B.slots = slots;
  }

  void inputs(Req &q) {
    const Topo &T = topos[q.r.topo];
    const System &s = *T.sys;
    const Mesh &m = *s.mesh;
    const admfem_request &r = q.r;
    const bool heat = r.kind == 1;
    if (r.source == ADMFEM_SRC_SYNTH) {
      std::mt19937_64 rng(r.seed);
      std::normal_distribution<double> nrm(0.0, 1.0 / 0.1);
      std::uniform_real_distribution<double> ph(0.0, 2.0 * M_PI);
      SynField kf{}, uf{};
      kf.nmodes = uf.nmodes = 32;
      kf.scale = uf.scale = std::sqrt(2.0 / 32.0);
      for (int j = 0; j < 32; j++) {
        kf.wx[j] = nrm(rng);
        kf.wy[j] = nrm(rng);
        kf.phi[j] = ph(rng);
      }
      for (int j = 0; j < 32; j++) {
        uf.wx[j] = nrm(rng);
        uf.wy[j] = nrm(rng);
        uf.phi[j] = ph(rng);
      }
      synth_inputs(s, m.x.p, m.y.p, r.seed, T.jitter, kf, heat ? &uf : nullptr, q.x, q.y,
                   q.xy, q.kappa, q.f, q.uprev, st);
      // observations: 1% of the interior nodes, obs_val = 0; the indices'
      // host copy lives with the request (no wait for the copy here)
      std::vector<int> &idx = q.h_obs;
      idx.clear();
      std::unordered_set<int> seen;
      std::uniform_int_distribution<size_t> pick(0, T.interior.size() - 1);
      while ((int)idx.size() < q.nobs) {
        int u = T.interior[pick(rng)];
        if (seen.insert(u).second) idx.push_back(u);
      }
      HIPCHECK(hipMemcpyAsync(q.obsi, idx.data(), sizeof(int) * q.nobs, hipMemcpyHostToDevice, st));
      HIPCHECK(hipMemsetAsync(q.obsv, 0, sizeof(double) * q.nobs, st));
      return;
    }
    const hipMemcpyKind kind =
        r.source == ADMFEM_SRC_HOST ? hipMemcpyHostToDevice : hipMemcpyDeviceToDevice;
    // (the inputs' presence was checked by server_submit)
    // user-order inputs are staged, then permuted to the internal order
    const int nn = m.nnode;  // vertices
    if (r.coords) {
      HIPCHECK(hipMemcpyAsync(q.stage, r.coords, sizeof(double) * 2 * nn, kind, st));
      launch_perm_coords(nn, m.d_iperm.p, q.stage, q.x, q.y, q.xy, st);
    } else {
      q.xy = m.xy.p;  // (only read)
    }
    if (r.source == ADMFEM_SRC_DEVICE) {  // with the other requests'
      jobs_in.add(ServeIn{{r.kappa, r.f, r.obs_val, heat ? r.u_prev : nullptr},
                          {q.kappa, q.f, q.obsv, q.uprev},
                          {(int)m.ngauss, (int)m.ngauss, r.nobs, heat ? s.n : 0},
                          s.d_uperm(), r.obs_idx, q.obsi, r.nobs},
                  std::max({(int)m.ngauss, s.n, r.nobs}));
      return;
    }
    HIPCHECK(hipMemcpyAsync(q.kappa, r.kappa, sizeof(double) * m.ngauss, kind, st));
    HIPCHECK(hipMemcpyAsync(q.f, r.f, sizeof(double) * m.ngauss, kind, st));
    if (heat) {
      HIPCHECK(hipMemcpyAsync(q.stage, r.u_prev, sizeof(double) * s.n, kind, st));
      launch_scatter(s.d_uperm(), q.stage, q.uprev, s.n, st);
    }
    if (r.nobs) {
      HIPCHECK(hipMemcpyAsync(q.obsi, r.obs_idx, sizeof(int) * r.nobs, kind, st));
      HIPCHECK(hipMemcpyAsync(q.obsv, r.obs_val, sizeof(double) * r.nobs, kind, st));
    }
    if (r.source == ADMFEM_SRC_HOST) HIPCHECK(hipStreamSynchronize(st));
  }

  admfem_problem problem(const Req &q) const {
    admfem_problem p{};
    const bool heat = q.r.kind == 1;
    p.kappa = q.kappa;
    p.f = q.f;
    p.u_prev = heat ? q.uprev : nullptr;
    p.lap_coef = heat ? q.r.dt : 1.0;
    p.mass_coef = heat ? 1.0 : 0.0;
    p.src_coef = heat ? q.r.dt : 1.0;
    return p;
  }

  void assemble(Req &q) {
    const System &s = *topos[q.r.topo].sys;
    admfem_problem p = problem(q);
    // FP64 matrix and rhs; the FP32 scaled matrix of the inner iteration
    launch_assemble_to(s, q.xy, p, SellOut{q.sv64, q.diag64, q.b}, st);
    if (!q.mg) batch_scale(s, q.sv64, q.diag64, q.dsq, q.sv32, st);
  }

  void start_cg(Req &q) {
    const double d = o.replace_delta > 0 ? o.replace_delta : REPLACE_DELTA;
    batch_init(d_desc.p, d_scal.p, q.slot, topos[q.r.topo].nblk, o.rtol * o.rtol, d * d,
               o.max_iter, st);
  }

  // waiting: bytes of the requests waiting with this one, which a new segment
  // is made for (0: make none)
  bool admit(Req &q, double t, size_t waiting, bool jacobi = false) {
    const Topo &T = topos[q.r.topo];
    if (free_slots.empty()) return false;
    size_up(q, jacobi);
    size_t bytes = bytes_of(q);
    if (bytes > arena.cap) {
      q.state = Q_DONE;
      q.res.done = 1;
      q.res.status = ADMFEM_ERR_BUDGET;
      q.res.t_done = t;
      return true;
    }
    char *mem;
    if (!arena.alloc(bytes, waiting ? std::max(bytes, waiting) : 0, mem)) {
      if (!waiting || arena.used) return false;  // when some request has finished
      if (q.mg) return admit(q, t, waiting, true);
      q.state = Q_DONE;              // the card's memory is gone
      q.res.done = 1;
      q.res.status = ADMFEM_ERR_BUDGET;
      q.res.t_done = t;
      return true;
    }
    q.mem = mem;
    q.bytes = bytes;
    q.res.device_bytes = (double)bytes;
    layout(*T.sys, q.mg ? T.plan : nullptr, &q, mem, q.nobs);
    q.slot = free_slots.back();
    q.loss2 = d_loss.p + 2 * q.slot;
    free_slots.pop_back();
    q.res.t_admit = t;
    return attempt(q, [&] { inputs(q); });
  }

  // A step of a request's admission.  When it fails the request fails alone:
  // its memory and slot go back to the queue, the requests behind it are
  // admitted as usual.
  template <class F> bool attempt(Req &q, F step) {
    try {
      step();
    } catch (const Error &e) {
      (void)hipStreamSynchronize(st);
      set_error(e.msg);
      fail(q, e.code == ADMFEM_ERR_HIP ? ADMFEM_ERR_HIP : ADMFEM_ERR_ARG);
      return true;
    }
    q.state = Q_FWD;
    return true;
  }

  // an admitted request's matrix and start, behind its inputs
  void prepare(Req &q) {
    attempt(q, [&] {
      assemble(q);
      if (q.mg) {
        write_mg_desc(q);  // set up and started with the batch's others
      } else {
        write_desc(q, q.b);
        start_cg(q);
      }
    });
  }
  void flush_inputs() {
    jobs_in.flush(serve_inputs, st);
  }

  // A solve that multigrid CG ended without a solution starts over with
  // Jacobi-PCG, which need not fail (and if it does, the status is its own), and
  // the request stays there.  The matrix and the right-hand side are where they
  // were (the caller's inputs may be gone by now); Jacobi-PCG's vectors take the
  // place of the others.
  void to_jacobi(Req &q) {
    const System &s = *topos[q.r.topo].sys;
    const size_t np = s.npad;
    q.mg = false;
    q.xa = q.mgx;
    q.xb = q.mgr;
    float **const v[] = {&q.ysa, &q.ysb, &q.ra, &q.rb, &q.pa, &q.pb, &q.qa, &q.qb};
    float *const at[] = {q.sq, q.minv, q.z, q.rs, q.x0, q.t, (float *)q.wrq, (float *)q.wrq + np};
    for (int k = 0; k < 8; k++) *v[k] = at[k];
    batch_scale(s, q.sv64, q.diag64, q.dsq, q.sv32, st);
    write_desc(q, q.b);
    start_cg(q);
  }

  void release(Req &q) {
    arena.release(q.mem, q.bytes);
    free_slots.push_back(q.slot);
    q.slot = -1;
  }

  // forward solve finished: u, loss, dL/du; start the adjoint solve
  void to_adjoint(Req &q, int it) {
    const System &s = *topos[q.r.topo].sys;
    q.res.iters_fwd = it;
    if (!q.mg) batch_final(d_desc.p, d_scal.p, q.slot, s.npad, q.u64, st);
    jobs_turn.add(ServeTurn{q.mg ? q.mgx : nullptr, q.obsv, s.d_uperm(), q.obsi, q.u64, q.b,
                            q.loss2, s.n, s.npad, q.nobs},  // (g overwrites b)
                  s.npad);
    q.state = Q_ADJ;
  }

  // adjoint solve finished: the gradient is enqueued, and the solution's way
  // to the caller's order with the other requests'
  void finish(Req &q, int it) {
    const System &s = *topos[q.r.topo].sys;
    q.res.iters_adj = it;
    if (!q.mg) batch_final(d_desc.p, d_scal.p, q.slot, s.npad, q.lam64, st);
    admfem_problem p = problem(q);
    launch_kappa_gradient_to(s, q.xy, q.u64, q.mg ? q.mgx : q.lam64, p.lap_coef, q.grad, st);
    if (q.r.u_out) jobs_out.add(ServeOut{s.d_uiperm(), q.u64, q.stage, s.n}, s.n);
  }

  // The outputs of the requests that finished at one chunk boundary, their
  // losses to the slots' pinned staging in one copy; complete() finishes them
  // once the stream has drained.
  void copy_outputs(const std::vector<int> &done) {
    jobs_out.flush(serve_outputs, st);
    int lo = max_slots, hi = -1;
    for (int i : done) {
      Req &q = reqs[i];
      const System &s = *topos[q.r.topo].sys;
      lo = std::min(lo, q.slot);
      hi = std::max(hi, q.slot);
      if (q.r.u_out)
        HIPCHECK(hipMemcpyAsync(q.r.u_out, q.stage, sizeof(double) * s.n, hipMemcpyDeviceToHost,
                                st));
      if (q.r.grad_out)
        HIPCHECK(hipMemcpyAsync(q.r.grad_out, q.grad, sizeof(double) * s.mesh->ngauss,
                                hipMemcpyDeviceToHost, st));
    }
    if (hi >= lo)
      HIPCHECK(hipMemcpyAsync(h_loss + 2 * lo, d_loss.p + 2 * lo,
                              2 * sizeof(double) * (hi - lo + 1), hipMemcpyDeviceToHost, st));
  }

  // after the stream has drained: a finished request's loss and status, its
  // memory and slot back to the queue
  void complete(Req &q) {
    std::vector<int>().swap(q.h_obs);
    const double *l2 = h_loss + 2 * q.slot;
    q.res.loss = l2[0];
    if (l2[1] != 0.0 && q.res.status == ADMFEM_OK) q.res.status = ADMFEM_ERR_ARG;
    q.res.t_done = now_s(t0);
    q.res.done = 1;
    q.state = Q_DONE;
    release(q);
  }

  void fail(Req &q, int code) {
    HIPCHECK(hipStreamSynchronize(st));
    q.res.status = code;
    q.res.done = 1;
    q.res.t_done = now_s(t0);
    q.state = Q_DONE;
    release(q);
  }

  static int code_of(int status) {
    switch (status) {
      case 1: return ADMFEM_OK;
      case 3: return ADMFEM_ERR_NAN;
      case 4: return ADMFEM_ERR_BREAKDOWN;
      default: return ADMFEM_ERR_NOT_CONVERGED;
    }
  }

  // ------------------------------------------------------------ batched run
  // Device map of gmap grid blocks and host/device lists for nlist systems;
  // growing them drops the captured graphs (they point at the old buffers).
  void ensure_map(size_t gmap, size_t nlist) {
    if (gmap > map_cap) {
      map_cap = std::max(gmap, 2 * map_cap);
      d_map.alloc(map_cap);
      drop_graphs();
    }
    if (nlist > list_cap) {
      if (h_list) HIPCHECK(hipHostFree(h_list));
      list_cap = std::max(nlist, 2 * list_cap);
      HIPCHECK(hipHostMalloc((void **)&h_list, sizeof(int) * (2 * list_cap + 1),
                             hipHostMallocDefault));
      d_list.alloc(2 * list_cap + 1);
      drop_graphs();
    }
  }

  // Uploads the slots of `slots` (padded to glist with `pad`) and their
  // first logical blocks, and expands the block map on the device.
  void upload_batch(const std::vector<std::pair<int, int>> &slots, size_t glist, int pad,
                    size_t nmap, size_t gmap) {
    int *pref = h_list + list_cap;
    int acc = 0;
    for (size_t a = 0; a < slots.size(); a++) {
      h_list[a] = slots[a].first;
      pref[a] = acc;
      acc += slots[a].second;
    }
    pref[slots.size()] = acc;
    for (size_t a = slots.size(); a < glist; a++) h_list[a] = pad;
    HIPCHECK(hipMemcpyAsync(d_list.p, h_list, sizeof(int) * glist, hipMemcpyHostToDevice, st));
    HIPCHECK(hipMemcpyAsync(d_list.p + list_cap, pref, sizeof(int) * (slots.size() + 1),
                            hipMemcpyHostToDevice, st));
    batch_map((int)slots.size(), d_list.p, d_list.p + list_cap, (int)nmap, (int)gmap, d_map.p,
              st);
  }

  // One CG chunk for a (map size, list size) bucket, captured once as a HIP
  // graph of kernel nodes only and replayed for every batch of that size.
  std::map<std::pair<int, int>, hipGraphExec_t> graphs;
  void drop_graphs() {
    for (auto &g : graphs) (void)hipGraphExecDestroy(g.second);
    graphs.clear();
  }
  static int bucket(size_t v) {
    size_t b = 64;
    while (b < v) b <<= 1;
    return (int)b;
  }
  void launch_chunk(int nmap, int nlist, int chunk) {
    auto key = std::make_pair(nmap, nlist);
    auto it = graphs.find(key);
    if (it == graphs.end()) {
      hipGraph_t g;
      HIPCHECK(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
      batch_iterations(d_map.p, nmap, d_list.p, nlist, d_desc.p, d_scal.p, chunk, st);
      HIPCHECK(hipStreamEndCapture(st, &g));
      hipGraphExec_t ex;
      HIPCHECK(hipGraphInstantiate(&ex, g, nullptr, nullptr, 0));
      HIPCHECK(hipGraphDestroy(g));
      it = graphs.emplace(key, ex).first;
    }
    HIPCHECK(hipGraphLaunch(it->second, st));
  }

  // What an error that ends a run leaves half done (inputs on no list any more,
  // descriptors not uploaded, systems not set up) is not taken up again: the
  // admitted requests fail with it, and the next run serves the waiting ones.
  void abandon(int code) {
    (void)hipStreamSynchronize(st);
    (void)hipGetLastError();
    starts.clear();
    jobs_in.clear();
    jobs_turn.clear();
    jobs_out.clear();
    for (Req &q : reqs) {
      if (q.slot < 0) continue;
      q.res.status = code;
      q.res.done = 1;
      q.res.t_done = now_s(t0);
      q.state = Q_DONE;
      std::vector<int>().swap(q.h_obs);
      release(q);
    }
  }

  void run_batched(double timeout) {
    try {
      serve_batched(timeout);
    } catch (const Error &e) {
      abandon(e.code);
      throw;
    } catch (...) {
      abandon(ADMFEM_ERR_ARG);
      throw;
    }
  }

  void serve_batched(double timeout) {
    const int chunk = o.chunk > 0 ? (o.chunk + REPLACE_EVERY - 1) / REPLACE_EVERY * REPLACE_EVERY
                                  : 2 * REPLACE_EVERY;
    std::vector<int> order(reqs.size());
    for (size_t i = 0; i < reqs.size(); i++) order[i] = (int)i;
    std::stable_sort(order.begin(), order.end(), [&](int a, int b) {
      return reqs[a].r.arrival < reqs[b].r.arrival;
    });
    size_t next = 0;  // first request (in arrival order) not yet admitted
    while (next < order.size() && reqs[order[next]].state != Q_WAIT) next++;
    // (a solve is 8 to 12 iterations; 64 a chunk on 8 requests of 64^2: 1.7 -> 3.0 ms,
    // 512: 21.8)
    const int mg_chunk = o.chunk > 0 ? std::min(o.chunk, 4) : 4;
    std::vector<int> active;
    for (size_t i = 0; i < reqs.size(); i++)
      if (reqs[i].state == Q_FWD || reqs[i].state == Q_ADJ) active.push_back((int)i);
    std::vector<int> admitted, fresh, jac, mgr;  // fresh: multigrid requests to be set up
    MgSet set_fresh, set_starts, set_mg;
    // requests whose last work (outputs, loss) is enqueued, and an event
    // behind that work: they complete once it has passed -- waited for
    // while the next chunk runs, so the host bookkeeping overlaps it
    std::vector<int> done, failed;
    struct Ev {
      hipEvent_t e = nullptr;
      ~Ev() {
        if (e) (void)hipEventDestroy(e);
      }
    } ev;
    HIPCHECK(hipEventCreateWithFlags(&ev.e, hipEventDisableTiming));
    hipEvent_t ev_done = ev.e;
    auto settle = [&]() {
      for (int i : done) complete(reqs[i]);
      for (int i : failed) {
        Req &q = reqs[i];
        std::vector<int>().swap(q.h_obs);
        q.res.done = 1;
        q.res.t_done = now_s(t0);
        q.state = Q_DONE;
        release(q);
      }
      done.clear();
      failed.clear();
    };
    auto flush = [&]() {
      if (done.empty() && failed.empty()) return;
      HIPCHECK(hipEventSynchronize(ev_done));
      settle();
    };
    for (;;) {
      double t = now_s(t0);
      if (t > timeout) break;
      // admit arrived requests, FIFO, while memory and slots allow
      admitted.clear();
      while (next < order.size() &&
             (o.max_active <= 0 || (int)(active.size() + admitted.size()) < o.max_active)) {
        Req &q = reqs[order[next]];
        if (q.r.arrival > t) break;
        if (!admit(q, t, 0)) {
          size_t waiting = 0;  // of the arrived requests that there is a slot for
          for (size_t k = next, n = 0; k < order.size() && n < free_slots.size(); k++, n++) {
            Req &w = reqs[order[k]];
            if (w.r.arrival > t) break;
            size_up(w, false);
            const size_t bytes = bytes_of(w);
            if (bytes <= arena.cap) waiting += up(bytes);
          }
          if (!waiting || !admit(q, t, waiting)) break;
        }
        if (q.state != Q_DONE) admitted.push_back(order[next]);
        next++;
      }
      flush_inputs();
      for (int i : admitted) {
        prepare(reqs[i]);
        if (reqs[i].state == Q_DONE) continue;
        active.push_back(i);
        if (reqs[i].mg) {
          fresh.push_back(i);
          starts.push_back(i);
        }
      }
      peak_active = std::max(peak_active, (int)active.size());
      if (active.empty()) {
        if (!done.empty() || !failed.empty()) {  // their slots may admit the next ones
          flush();
          continue;
        }
        if (next >= order.size()) break;
        double wait = reqs[order[next]].r.arrival - now_s(t0);
        if (wait > 0) std::this_thread::sleep_for(std::chrono::duration<double>(std::min(wait, 0.01)));
        continue;
      }
      jac.clear();
      mgr.clear();
      for (int i : active) (reqs[i].mg ? mgr : jac).push_back(i);
      if (!fresh.empty()) {
        upload_mg_descs(fresh);
        build_set(set_fresh, fresh);
        mg_batch_setup(set_fresh.batch, d_mg.p, st);
        fresh.clear();
      }
      if (!starts.empty()) {
        build_set(set_starts, starts);
        mg_batch_start(set_starts.batch, d_mg.p, d_mgs.p, o.rtol * o.rtol,
                       std::min(MG_GIVE_UP, std::max(1, o.max_iter / MG_PRODUCTS)), st);
        starts.clear();
      }
      if (!mgr.empty()) {
        build_set(set_mg, mgr);
        mg_batch_iterations(set_mg.batch, d_mg.p, d_mgs.p, mg_chunk, h_mgs, st);
      }
      if (!jac.empty()) {
        // block map over the Jacobi-PCG systems; with graphs, both grids are
        // padded to power-of-two buckets with entries that do no work (map:
        // system -1, list: the never-running dummy slot)
        size_t nmap = 0;
        for (int i : jac) nmap += topos[reqs[i].r.topo].nblk;
        const size_t gmap = use_graph ? (size_t)bucket(nmap) : nmap;
        const size_t glist = use_graph ? (size_t)bucket(jac.size()) : jac.size();
        ensure_map(gmap, glist);
        std::vector<std::pair<int, int>> slots(jac.size());
        for (size_t a = 0; a < jac.size(); a++) {
          const Req &q = reqs[jac[a]];
          slots[a] = std::make_pair(q.slot, topos[q.r.topo].nblk);
        }
        upload_batch(slots, glist, max_slots, nmap, gmap);  // padding: the dummy slot
        if (use_graph)
          launch_chunk((int)gmap, (int)glist, chunk);
        else
          batch_iterations(d_map.p, (int)nmap, d_list.p, (int)jac.size(), d_desc.p, d_scal.p,
                           chunk, st);
        HIPCHECK(hipMemcpyAsync(h_scal, d_scal.p, sizeof(BScal) * max_slots,
                                hipMemcpyDeviceToHost, st));
      }
      steps += 1;
      iters += jac.empty() ? mg_chunk : chunk;
      batch_sum += (int64_t)active.size();
      flush();  // the previous chunk's finished requests, while this one runs
      HIPCHECK(hipStreamSynchronize(st));
      // phase changes; requests that finished or failed complete once their
      // enqueued work has passed
      std::vector<int> still, turned;
      for (int i : active) {
        Req &q = reqs[i];
        // where the solve stands: status (0 run, 1 converged, else failed),
        // products with A, true residual and right-hand side norms squared
        struct { int status, it; double rr, bb; } sc;
        if (q.mg) {
          const MgScal &v = h_mgs[q.slot];
          sc = {v.checked ? v.a.status : 0, MG_PRODUCTS * v.a.it, v.rr_true, v.bb};
        } else {
          const BScal &v = h_scal[q.slot];
          sc = {v.status, v.it, v.rr, v.bb};
        }
        if (sc.status == 0) {
          still.push_back(i);
          continue;
        }
        if (sc.status != 1 && q.mg) {
          to_jacobi(q);
          still.push_back(i);
          continue;
        }
        if (sc.status != 1) {
          if (q.state == Q_FWD) q.res.iters_fwd = sc.it;
          else q.res.iters_adj = sc.it;
          q.res.status = code_of(sc.status);
          failed.push_back(i);
          continue;
        }
        if (q.state == Q_FWD) {
          q.res.relres_fwd = sc.bb > 0 ? std::sqrt(sc.rr / sc.bb) : 0.0;
          to_adjoint(q, sc.it);
          turned.push_back(i);
          still.push_back(i);
        } else {
          q.res.relres_adj = sc.bb > 0 ? std::sqrt(sc.rr / sc.bb) : 0.0;
          finish(q, sc.it);
          done.push_back(i);
        }
      }
      jobs_turn.flush(serve_turn, st);
      for (int i : turned) {
        if (reqs[i].mg) starts.push_back(i);
        else start_cg(reqs[i]);
      }
      copy_outputs(done);
      if (!done.empty() || !failed.empty()) HIPCHECK(hipEventRecord(ev_done, st));
      active.swap(still);
    }
    flush();
    wall = now_s(t0);
  }

  // ------------------------------------------------------------ sequential
  void run_seq(double timeout) {
    std::vector<int> order(reqs.size());
    for (size_t i = 0; i < reqs.size(); i++) order[i] = (int)i;
    std::stable_sort(order.begin(), order.end(), [&](int a, int b) {
      return reqs[a].r.arrival < reqs[b].r.arrival;
    });
    for (int i : order) {
      Req &q = reqs[i];
      if (q.state != Q_WAIT) continue;
      double t = now_s(t0);
      if (t > timeout) break;
      if (q.r.arrival > t)
        std::this_thread::sleep_for(std::chrono::duration<double>(q.r.arrival - t));
      t = now_s(t0);
      System &s = *topos[q.r.topo].sys;
      q.nobs = nobs_of(q);
      size_t bytes = bytes_of(q);
      char *mem;
      if (bytes > arena.cap || !arena.alloc(bytes, bytes, mem)) {
        q.res.status = ADMFEM_ERR_BUDGET;
        q.res.done = 1;
        q.state = Q_DONE;
        continue;
      }
      q.mem = mem;
      q.res.device_bytes = (double)bytes;
      layout(s, nullptr, &q, mem, q.nobs);
      q.slot = 0;
      q.loss2 = d_loss.p;
      q.res.t_admit = t;
      peak_active = std::max(peak_active, 1);
      try {
        serve_seq(q, s);
      } catch (const Error &e) {
        (void)hipStreamSynchronize(st);
        set_error(e.msg);
        q.res.status = e.code == ADMFEM_ERR_HIP ? ADMFEM_ERR_HIP : ADMFEM_ERR_ARG;
      }
      q.res.t_done = now_s(t0);
      q.res.done = 1;
      q.state = Q_DONE;
      arena.release(q.mem, bytes);
    }
    wall = now_s(t0);
  }

  // One request on the FP64 single-system path, on the topology's own solver
  // buffers (the request's arena range holds its inputs and outputs).
  void serve_seq(Req &q, System &s) {
    inputs(q);
    flush_inputs();
    admfem_problem p = problem(q);
    s.a_version++;
    s.mass = p.mass_coef != 0.0;
    launch_assemble_to(s, q.xy, p, SellOut{s.d_sell_val.p, s.d_diag.p, s.rhs.p},
                       st);
    admfem_solve_opts so{ADMFEM_PREC_FP64, o.max_iter, o.rtol, 0, 0.0};
    admfem_solve_stats s0{}, s1{};
    cg_solve(s, s.rhs.p, q.u64, so, s0, st);
    launch_loss(s, q.u64, q.obsi, q.obsv, q.nobs, q.b, q.loss2, st);
    cg_solve(s, q.b, q.lam64, so, s1, st);
    q.res.iters_fwd = s0.iterations;
    q.res.iters_adj = s1.iterations;
    q.res.relres_fwd = s0.rel_residual;
    q.res.relres_adj = s1.rel_residual;
    iters += s0.iterations + s1.iterations;
    steps += 1;
    batch_sum += 1;
    q.res.status = s0.status != ADMFEM_OK ? s0.status : s1.status;
    if (q.res.status != ADMFEM_OK) {
      HIPCHECK(hipStreamSynchronize(st));
      return;
    }
    const Mesh &m = *s.mesh;
    launch_kappa_gradient_to(s, q.xy, q.u64, q.lam64, p.lap_coef, q.grad, st);
    if (q.r.u_out) {
      launch_scatter(s.d_uiperm(), q.u64, q.stage, s.n, st);
      HIPCHECK(hipMemcpyAsync(q.r.u_out, q.stage, sizeof(double) * s.n, hipMemcpyDeviceToHost,
                              st));
    }
    if (q.r.grad_out)
      HIPCHECK(hipMemcpyAsync(q.r.grad_out, q.grad, sizeof(double) * m.ngauss,
                              hipMemcpyDeviceToHost, st));
    double l2[2];
    HIPCHECK(hipMemcpyAsync(l2, q.loss2, sizeof(l2), hipMemcpyDeviceToHost, st));
    HIPCHECK(hipStreamSynchronize(st));
    q.res.loss = l2[0];
    if (l2[1] != 0.0) q.res.status = ADMFEM_ERR_ARG;  // bad or repeated obs index
  }
};

// Instrumentation: the batched CG step kernel over a batch of synthetic
// Poisson systems.  The scalars it reads (alpha = beta = 0, it, status) stay
// as batch_init left them, so every launch reads the same buffers, does its
// full work and writes the same values to the other buffers.
double server_spmv_repeat(Server *sv, const int *topos, int nsys, int repeat,
                          hipStream_t st, double *seconds) {
  REQUIRE(nsys <= (int)sv->free_slots.size(), ADMFEM_ERR_ARG, "more systems than free slots");
  for (int i = 0; i < nsys; i++)
    REQUIRE(topos[i] >= 0 && topos[i] < (int)sv->topos.size(), ADMFEM_ERR_ARG,
            "bad topology id");
  std::vector<Req> qs(nsys);
  int admitted = 0;
  double bytes = 0.0;
  hipEvent_t ev[2] = {nullptr, nullptr};
  auto cleanup = [&] {
    (void)hipStreamSynchronize(st);
    (void)hipStreamSynchronize(sv->st);
    for (int i = 0; i < admitted; i++) sv->release(qs[i]);
    for (hipEvent_t e : ev)
      if (e) (void)hipEventDestroy(e);
  };
  try {
    size_t nmap = 0;
    for (int i = 0; i < nsys; i++) {
      Req &q = qs[i];
      q.r = admfem_request{};
      q.r.topo = topos[i];
      q.r.source = ADMFEM_SRC_SYNTH;
      q.r.seed = (unsigned long long)i;
      const bool ok = sv->admit(q, 0.0, (size_t)1 << 30, true);
      if (ok && q.state == Q_FWD) sv->prepare(q);
      REQUIRE(ok && q.state == Q_FWD, ADMFEM_ERR_BUDGET, "batch does not fit the budget");
      admitted++;
      nmap += sv->topos[q.r.topo].nblk;
      const System &s = *sv->topos[q.r.topo].sys;
      // one CG iteration of the canonical CSR form: the SpMV's
      // nnz (s + 4) + 4 (n + 1) + 2 n s plus 6 n s of vector updates (s = 4)
      bytes += (double)s.nnz * 8.0 + 4.0 * (s.n + 1) + 8.0 * s.n * 4.0;
    }
    sv->ensure_map(nmap, (size_t)nsys);
    std::vector<std::pair<int, int>> slots(nsys);
    for (int i = 0; i < nsys; i++)
      slots[i] = std::make_pair(qs[i].slot, sv->topos[qs[i].r.topo].nblk);
    sv->upload_batch(slots, (size_t)nsys, sv->max_slots, nmap, nmap);
    HIPCHECK(hipStreamSynchronize(sv->st));
    HIPCHECK(hipEventCreate(&ev[0]));
    HIPCHECK(hipEventCreate(&ev[1]));
    HIPCHECK(hipEventRecord(ev[0], st));
    batch_spmv_repeat(sv->d_map.p, (int)nmap, sv->d_desc.p, sv->d_scal.p, repeat, st);
    HIPCHECK(hipEventRecord(ev[1], st));
    HIPCHECK(hipEventSynchronize(ev[1]));
    float ms = 0.0f;
    HIPCHECK(hipEventElapsedTime(&ms, ev[0], ev[1]));
    *seconds = repeat > 0 ? 1e-3 * ms / repeat : 0.0;
  } catch (...) {
    cleanup();
    throw;
  }
  cleanup();
  return bytes;
}

// ---------------------------------------------------------------- C-ABI glue
Server *server_create(const admfem_server_opts &o) {
  REQUIRE(o.hbm_budget_bytes > 0, ADMFEM_ERR_ARG, "budget must be positive");
  REQUIRE(o.rtol > 0 && o.max_iter > 0, ADMFEM_ERR_ARG, "bad rtol / max_iter");
  REQUIRE(o.mode == ADMFEM_MODE_BATCHED || o.mode == ADMFEM_MODE_SEQ_FP64, ADMFEM_ERR_ARG,
          "bad mode");
  Server *sv = new Server();
  try {
    sv->o = o;
    HIPCHECK(hipStreamCreateWithFlags(&sv->st, hipStreamNonBlocking));
    sv->arena.init((size_t)o.hbm_budget_bytes);
    sv->max_slots = o.max_active > 0 ? o.max_active : 1024;
    for (int i = sv->max_slots - 1; i >= 0; i--) sv->free_slots.push_back(i);
    sv->use_graph = o.use_graph != 0;
    // one extra slot: the dummy the padded graph launches point at; its
    // status is never "running", so every kernel skips it
    sv->d_desc.alloc(sv->max_slots + 1);
    sv->d_scal.alloc(sv->max_slots + 1);
    HIPCHECK(hipMemset(sv->d_desc.p, 0, sv->d_desc.bytes()));
    HIPCHECK(hipMemset(sv->d_scal.p, 0, sv->d_scal.bytes()));
    sv->d_mg.alloc(sv->max_slots);
    sv->d_loss.alloc(2 * (size_t)sv->max_slots);
    sv->jobs_in.alloc(sv->max_slots);
    sv->jobs_turn.alloc(sv->max_slots);
    sv->jobs_out.alloc(sv->max_slots);
    sv->d_mgs.alloc(sv->max_slots);
    HIPCHECK(hipHostMalloc((void **)&sv->h_mg, sizeof(MgSys) * sv->max_slots,
                           hipHostMallocDefault));
    HIPCHECK(hipHostMalloc((void **)&sv->h_mgs, sizeof(MgScal) * sv->max_slots,
                           hipHostMallocDefault));
    BScal dummy{};
    dummy.status = 99;
    HIPCHECK(hipMemcpy(sv->d_scal.p + sv->max_slots, &dummy, sizeof(BScal),
                       hipMemcpyHostToDevice));
    HIPCHECK(hipHostMalloc((void **)&sv->h_scal, sizeof(BScal) * sv->max_slots,
                           hipHostMallocDefault));
    HIPCHECK(hipHostMalloc((void **)&sv->h_loss, 2 * sizeof(double) * sv->max_slots,
                           hipHostMallocDefault));
    HIPCHECK(hipHostMalloc((void **)&sv->h_desc, sizeof(BSys) * sv->max_slots,
                           hipHostMallocDefault));
  } catch (...) {
    delete sv;
    throw;
  }
  return sv;
}

void server_free(Server *sv) { delete sv; }

int server_add_topology(Server *sv, System *s, double jitter) {
  Topo T;
  T.sys = s;
  T.jitter = jitter;
  T.nblk = (s->npad + BATCH_NT - 1) / BATCH_NT;
  T.plan = nullptr;
  if (s->n >= MG_MIN_ROWS && sv->o.mode == ADMFEM_MODE_BATCHED) {
    try {
      T.plan = mg_plan(*s, sv->st);
      if (T.plan) mg_allow_lds(*T.plan);
    } catch (const OutOfMemory &) {  // (Jacobi-PCG needs none)
      release_device_memory();
    }
  }
  for (int u = 0; u < s->n; u++)
    if (s->row_bd[s->uperm()[u]] < 0) T.interior.push_back(u);
  REQUIRE(!T.interior.empty(), ADMFEM_ERR_ARG, "topology has no interior node");
  sv->topos.push_back(std::move(T));
  return (int)sv->topos.size() - 1;
}

int64_t server_submit(Server *sv, const admfem_request &r) {
  REQUIRE(r.topo >= 0 && r.topo < (int)sv->topos.size(), ADMFEM_ERR_ARG, "bad topology id");
  REQUIRE(r.kind == 0 || r.kind == 1, ADMFEM_ERR_ARG, "bad request kind");
  REQUIRE(r.source >= 0 && r.source <= 2, ADMFEM_ERR_ARG, "bad request source");
  REQUIRE(r.kind == 0 || r.dt > 0, ADMFEM_ERR_ARG, "heat step needs dt > 0");
  REQUIRE(r.nobs >= 0, ADMFEM_ERR_ARG, "bad nobs");
  if (r.source != ADMFEM_SRC_SYNTH) {
    // every input the request reads is checked here, before it can hold a
    // slot or arena memory
    REQUIRE(r.kappa && r.f, ADMFEM_ERR_ARG, "request needs kappa and f");
    REQUIRE(r.kind == 0 || r.u_prev, ADMFEM_ERR_ARG, "heat step needs u_prev");
    REQUIRE(r.nobs == 0 || (r.obs_idx && r.obs_val), ADMFEM_ERR_ARG,
            "observations need obs_idx and obs_val");
    if (r.source == ADMFEM_SRC_HOST && r.nobs > 0) {
      // host indices: range and distinctness checked now (device indices
      // are checked by the loss kernel, which fails the request)
      const int n = sv->topos[r.topo].sys->n;
      std::vector<int> idx(r.obs_idx, r.obs_idx + r.nobs);
      for (int v : idx)
        REQUIRE(v >= 0 && v < n, ADMFEM_ERR_ARG, "observation index out of range [0, n)");
      std::sort(idx.begin(), idx.end());
      REQUIRE(std::adjacent_find(idx.begin(), idx.end()) == idx.end(), ADMFEM_ERR_ARG,
              "observation indices must be distinct");
    }
  }
  Req q;
  q.r = r;
  q.res.t_arrival = r.arrival;
  sv->reqs.push_back(q);
  return (int64_t)sv->reqs.size() - 1;
}

void server_run(Server *sv, double timeout) {
  if (!sv->started) {
    sv->started = true;
    sv->t0 = std::chrono::steady_clock::now();
  }
  if (sv->o.mode == ADMFEM_MODE_BATCHED) sv->run_batched(timeout);
  else sv->run_seq(timeout);
}

void server_result(Server *sv, int64_t id, admfem_result &out) {
  REQUIRE(id >= 0 && id < (int64_t)sv->reqs.size(), ADMFEM_ERR_ARG, "bad request id");
  out = sv->reqs[id].res;
}

void server_stats(Server *sv, double *s) {
  int done = 0, failed = 0;
  for (auto &q : sv->reqs)
    if (q.res.done) {
      done++;
      if (q.res.status != ADMFEM_OK) failed++;
    }
  s[0] = done;
  s[1] = sv->wall;
  s[2] = (double)sv->arena.peak;
  s[3] = sv->peak_active;
  s[4] = (double)sv->steps;
  s[5] = (double)sv->iters;
  s[6] = failed;
  s[7] = sv->steps ? (double)sv->batch_sum / sv->steps : 0.0;
}

}  // namespace admfem
