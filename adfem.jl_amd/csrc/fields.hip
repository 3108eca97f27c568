// Nodal fields <-> Gauss points, and the matrix-free Laplace term, for P1
// (P2 meshes dispatch to p2.hip, except FemToGaussPoints, which maps vertex
// values with the linear functions for either degree):
//   FemToGaussPointsMfem / DofToGaussPointsMfem (deps/MFEM/FemToGaussPoints/
//     FemToGaussPointsMfem.h:6-33, DofToGaussPoints/DofToGaussPointsMfem.h:
//     6-32): out[g] = sum_r u[node_r] h_r(g)
//   FemGradMfem (deps/MFEM/FemGrad/FemGradMfem.h:8-41):
//     out[g] = (sum_r u[node_r] dh_r/dx, sum_r u[node_r] dh_r/dy)
//   ComputeLaplaceTermMfem (deps/MFEM/ComputeLaplaceTermMfem/
//     ComputeLaplaceTermMfem.h:4-39): out = K(nu) u without forming K.
// Fields are in the user's node order, Gauss arrays in the user's element
// order (g = nq e + k).  Forward maps to Gauss points run one thread per
// element.  The maps to the nodes have one writer per output and no
// atomics: a gather over the node's incident elements, or, where deriving an
// element's geometry anew at each of its nodes costs more than passing its
// terms through memory, a pass over the elements and a pass over the nodes.
#include <type_traits>

#include "geom.h"

namespace admfem {

namespace {

struct Tri {
  double x[3], y[3];
};

__device__ __forceinline__ Tri load_tri(const int *__restrict__ conn, int nelem, int e,
                                        const double *__restrict__ x,
                                        const double *__restrict__ y) {
  Tri t;
#pragma unroll
  for (int k = 0; k < 3; k++) {
    const int v = conn[(size_t)k * nelem + e];
    t.x[k] = x[v];
    t.y[k] = y[v];
  }
  return t;
}

// Forward maps: one thread per element and an XCD's blocks one range of
// elements; the values leave by way of LDS, in consecutive stores.  With one
// thread per Gauss point the three of an element fetched its vertices and ids
// three times, and every XCD all of the vertices (700^2, 3 points: to the Gauss
// points 15.4 -> 14.1 us, gradients 23.7 -> 19.9; 29 with each element's
// thread storing its own).
template <int NQ>
__global__ void __launch_bounds__(256)
    to_gauss_kernel(int nelem, QuadRule rule, const int *__restrict__ conn_user,
                    const double *__restrict__ u, double *__restrict__ out) {
#pragma clang fp contract(off)
  __shared__ double sh[256 * NQ];
  const int e0 = xcd_block(blockIdx.x, gridDim.x) * 256, e = e0 + threadIdx.x;
  if (e < nelem) {
    const double u0 = u[conn_user[e]], u1 = u[conn_user[(size_t)nelem + e]],
                 u2 = u[conn_user[2 * (size_t)nelem + e]];
#pragma unroll
    for (int k = 0; k < NQ; k++)
      sh[NQ * threadIdx.x + k] = u0 * shape(0, rule.xi[k], rule.eta[k]) +
                                 u1 * shape(1, rule.xi[k], rule.eta[k]) +
                                 u2 * shape(2, rule.xi[k], rule.eta[k]);
  }
  __syncthreads();
  const int ng = NQ * min(256, nelem - e0);
  double *o = out + (size_t)NQ * e0;
#pragma unroll
  for (int k = 0; k < NQ; k++) {
    const int g = k * 256 + threadIdx.x;
    if (g < ng) o[g] = sh[g];
  }
}

// Vertices of element e (xy: internal order).
__device__ __forceinline__ void load_xy(const int *__restrict__ conn, int nelem, int e,
                                        const double2 *__restrict__ xy, double2 (&v)[3]) {
#pragma unroll
  for (int q = 0; q < 3; q++) v[q] = xy[conn[(size_t)q * nelem + e]];
}

// out16: out is 16-byte aligned (one store per Gauss point)
template <int NQ>
__global__ void __launch_bounds__(256)
    fem_grad_kernel(int nelem, const int *__restrict__ conn, const int *__restrict__ conn_user,
                    const double2 *__restrict__ xy, const double *__restrict__ u,
                    double *__restrict__ out, bool out16) {
#pragma clang fp contract(off)
  __shared__ double sx[256], sy[256];
  const int e0 = xcd_block(blockIdx.x, gridDim.x) * 256, e = e0 + threadIdx.x;
  if (e < nelem) {
    double2 v[3];
    load_xy(conn, nelem, e, xy, v);
    double hx[3], hy[3], gx = 0.0, gy = 0.0;
    elem_grads(v[0].x, v[0].y, v[1].x, v[1].y, v[2].x, v[2].y, hx, hy);
#pragma unroll
    for (int r = 0; r < 3; r++) {
      const double ur = u[conn_user[(size_t)r * nelem + e]];
      gx += ur * hx[r];
      gy += ur * hy[r];
    }
    sx[threadIdx.x] = gx;
    sy[threadIdx.x] = gy;
  }
  __syncthreads();
  const int ng = NQ * min(256, nelem - e0);
  double *o = out + 2 * (size_t)NQ * e0;
#pragma unroll
  for (int k = 0; k < NQ; k++) {
    const int g = k * 256 + threadIdx.x;
    if (g >= ng) continue;
    const double gx = sx[g / NQ], gy = sy[g / NQ];
    if (out16) {
      reinterpret_cast<double2 *>(o)[g] = make_double2(gx, gy);
    } else {
      o[2 * g] = gx;
      o[2 * g + 1] = gy;
    }
  }
}

// Per node: the transposes of the two maps above.
enum { NODE_TO_GAUSS_T = 0, NODE_GRAD_T = 1 };

template <int OP, int NQ>
__global__ void __launch_bounds__(256) node_gather_kernel(int n, int nelem, QuadRule rule, const int *__restrict__ conn,
                                   const int *__restrict__ conn_user,
                                   const double *__restrict__ x, const double *__restrict__ y,
                                   const int *__restrict__ n2e_ptr,
                                   const int *__restrict__ n2e_elem,
                                   const uint32_t *__restrict__ slots,
                                   const int *__restrict__ iperm,
                                   const double *__restrict__ in,   // Gauss array
                                   double *__restrict__ out_user) {
  const int r = xcd_block(blockIdx.x, gridDim.x) * 256 + threadIdx.x;
  if (r >= n) return;
  double acc = 0.0;
  const int t1 = n2e_ptr[r + 1];
  // unrolled over incidences so that their loads overlap
#pragma unroll 4
  for (int t = n2e_ptr[r]; t < t1; t++) {
    const int e = n2e_elem[t];
    const int p = (int)(slots[t] & 3u);
    if (OP == NODE_TO_GAUSS_T) {
#pragma unroll
      for (int k = 0; k < NQ; k++)
        acc += in[(size_t)NQ * e + k] * shape(p, rule.xi[k], rule.eta[k]);
    } else {
      const Tri tr = load_tri(conn, nelem, e, x, y);
      double gx[3], gy[3];
      elem_grads(tr.x[0], tr.y[0], tr.x[1], tr.y[1], tr.x[2], tr.y[2], gx, gy);
#pragma unroll
      for (int k = 0; k < NQ; k++) {
        const size_t g = (size_t)NQ * e + k;
        acc += in[2 * g] * gx[p] + in[2 * g + 1] * gy[p];
      }
    }
  }
  out_user[iperm[r]] = acc;
}

// The two passes of K(nu) u and of fem_grad's transpose.  Element e's term of
// its vertex p goes to c[p nelem + e]; the node pass sums each node's terms
// in ascending element order.  Both are bound by memory: the element pass
// streams the Gauss arrays once (the one-pass gather met each element's
// values and vertex ids six times, in the nodes' order) and the node pass
// reads one scattered double per incidence.  K(nu) u: 9.6 -> 6.3 us at 64^2,
// 64 -> 37 us at 700^2; fem_grad's transpose at 700^2: 55 -> 30 us.
// K(nu)'s transpose for the gradient (KIND 2) also takes the gradient in nu,
// w_g grad(in) . grad(u) (ComputeLaplaceTermMfemGrad; the term is linear in nu),
// from the element's vertices in hand: 55 -> 33 us at 700^2 for the two.  The
// weights come from the area (8 bytes an element instead of 24; K(nu) u's element
// pass 26 -> 22 us).
enum { TERM_GRAD_T = 0, TERM_LAPLACE = 1, TERM_LAPLACE_GRAD = 2 };
template <int KIND, int NQ>
__global__ void __launch_bounds__(256)
    elem_terms_kernel(int nelem, QuadRule rule, const int *__restrict__ conn,
                      const int *__restrict__ conn_user, const double2 *__restrict__ xy,
                      const double *__restrict__ area,
                      const double *__restrict__ in,  // field, or (TERM_GRAD_T) Gauss array (x, y)
                      const double *nu, double *__restrict__ c, const double *__restrict__ u,
                      double *gnu) {  // (gnu may be nu)
  const int e = xcd_block(blockIdx.x, gridDim.x) * 256 + threadIdx.x;
  if (e >= nelem) return;
  double2 v[3];
  load_xy(conn, nelem, e, xy, v);
  double gx[3], gy[3], sx = 0.0, sy = 0.0;
  elem_grads(v[0].x, v[0].y, v[1].x, v[1].y, v[2].x, v[2].y, gx, gy);
  if (KIND != TERM_GRAD_T) {  // sum_k nu_k w_k grad phi_p . grad u_e
    double ux = 0.0, uy = 0.0;
#pragma unroll
    for (int q = 0; q < 3; q++) {
      const int w = conn_user[(size_t)q * nelem + e];
      const double uq = in[w];
      sx += gx[q] * uq;
      sy += gy[q] * uq;
      if (KIND == TERM_LAPLACE_GRAD) {
        const double vq = u[w];
        ux += gx[q] * vq;
        uy += gy[q] * vq;
      }
    }
    const double a = area[e];
    double cw = 0.0, nk[NQ];
#pragma unroll
    for (int k = 0; k < NQ; k++) nk[k] = nu[(size_t)NQ * e + k];
#pragma unroll
    for (int k = 0; k < NQ; k++) {
      const double wk = gauss_weight(rule.w[k], a);
      cw += nk[k] * wk;
      if (KIND == TERM_LAPLACE_GRAD) gnu[(size_t)NQ * e + k] = wk * (sx * ux + sy * uy);
    }
    sx *= cw;
    sy *= cw;
  } else {
#pragma unroll
    for (int k = 0; k < NQ; k++) {
      const size_t g = (size_t)NQ * e + k;
      sx += in[2 * g];
      sy += in[2 * g + 1];
    }
  }
#pragma unroll
  for (int p = 0; p < 3; p++) c[(size_t)p * nelem + e] = sx * gx[p] + sy * gy[p];
}

__global__ void __launch_bounds__(256)
    node_sum_kernel(int n, int nelem, const int *__restrict__ n2e_ptr,
                    const int *__restrict__ n2e_elem, const uint32_t *__restrict__ slots,
                    const int *__restrict__ iperm, const double *__restrict__ c,
                    double *__restrict__ out_user) {
  const int r = xcd_block(blockIdx.x, gridDim.x) * 256 + threadIdx.x;
  if (r >= n) return;
  const int t1 = n2e_ptr[r + 1];
  double acc = 0.0;
  int t = n2e_ptr[r];
  for (; t + 2 < t1; t += 3) {  // three terms' loads in flight
    double v[3];
#pragma unroll
    for (int k = 0; k < 3; k++) v[k] = c[(size_t)(slots[t + k] & 3u) * nelem + n2e_elem[t + k]];
#pragma unroll
    for (int k = 0; k < 3; k++) acc += v[k];
  }
  for (; t < t1; t++) acc += c[(size_t)(slots[t] & 3u) * nelem + n2e_elem[t]];
  out_user[iperm[r]] = acc;
}

// ComputeLaplaceTermMfemGrad's nu part alone.
template <int NQ>
__global__ void __launch_bounds__(256)
    laplace_term_nu_grad_kernel(int nelem, QuadRule rule, const int *__restrict__ conn,
                                const int *__restrict__ conn_user,
                                const double2 *__restrict__ xy, const double *__restrict__ area,
                                const double *__restrict__ go, const double *__restrict__ u,
                                double *__restrict__ gnu) {
  const int e = xcd_block(blockIdx.x, gridDim.x) * 256 + threadIdx.x;
  if (e >= nelem) return;
  double2 v[3];
  load_xy(conn, nelem, e, xy, v);
  double gx[3], gy[3], ax = 0.0, ay = 0.0, bx = 0.0, by = 0.0;
  elem_grads(v[0].x, v[0].y, v[1].x, v[1].y, v[2].x, v[2].y, gx, gy);
#pragma unroll
  for (int q = 0; q < 3; q++) {
    const int w = conn_user[(size_t)q * nelem + e];
    ax += gx[q] * go[w];
    ay += gy[q] * go[w];
    bx += gx[q] * u[w];
    by += gy[q] * u[w];
  }
  const double a = area[e];
#pragma unroll
  for (int k = 0; k < NQ; k++)
    gnu[(size_t)NQ * e + k] = gauss_weight(rule.w[k], a) * (ax * bx + ay * by);
}

inline unsigned nb(int64_t n, int bs) { return (unsigned)((n + bs - 1) / bs); }

// go(Gauss points of the rule, a compile-time constant)
template <class F>
void by_rule(const Mesh &m, F go) {
  if (m.rule.nq == 3) go(std::integral_constant<int, 3>{});
  else if (m.rule.nq == 6) go(std::integral_constant<int, 6>{});
  else go(std::integral_constant<int, 1>{});
  HIPCHECK(hipGetLastError());
}

template <int OP>
void node_gather(const Mesh &m, const double *in, double *out_user, hipStream_t st) {
  by_rule(m, [&](auto nq) {
    node_gather_kernel<OP, nq()><<<nb(m.nnode, 256), 256, 0, st>>>(
        m.nnode, m.nelem, m.rule, m.conn.p, m.conn_user.p, m.x.p, m.y.p, m.d_n2e_ptr.p,
        m.d_n2e_elem.p, m.d_slots_full.p, m.d_iperm.p, in, out_user);
  });
}

template <int KIND>
void two_pass(const Mesh &m, const double *in, const double *nu, double *out_user, double *c,
              const double *u, double *gnu, hipStream_t st) {
  by_rule(m, [&](auto nq) {
    elem_terms_kernel<KIND, nq()><<<nb(m.nelem, 256), 256, 0, st>>>(
        m.nelem, m.rule, m.conn.p, m.conn_user.p, m.xy.p, m.area.p, in, nu, c, u, gnu);
  });
  node_sum_kernel<<<nb(m.nnode, 256), 256, 0, st>>>(m.nnode, m.nelem, m.d_n2e_ptr.p,
                                                    m.d_n2e_elem.p, m.d_slots_full.p,
                                                    m.d_iperm.p, c, out_user);
  HIPCHECK(hipGetLastError());
}

// fem_grad's transpose takes the two passes from here on: below, the second
// launch costs what the passes save (one pass / two: 200^2 7.0 / 7.7 us,
// 250^2 8.5 / 8.8, 360^2 14.1 / 12.1, 700^2 55 / 32).
constexpr int GRAD_T_TWO_PASS = 100000;

}  // namespace

void launch_to_gauss(const Mesh &m, const double *u, double *out, hipStream_t st) {
  by_rule(m, [&](auto nq) {
    to_gauss_kernel<nq()><<<nb(m.nelem, 256), 256, 0, st>>>(m.nelem, m.rule, m.conn_user.p, u,
                                                            out);
  });
}

void launch_to_gauss_grad(const Mesh &m, const double *grad_out, double *grad_u,
                          hipStream_t st) {
  node_gather<NODE_TO_GAUSS_T>(m, grad_out, grad_u, st);
}

void launch_dof_to_gauss(const Mesh &m, const double *u, double *out, hipStream_t st) {
  if (m.degree == 2) return launch_p2_dof_to_gauss(m, u, out, st);
  launch_to_gauss(m, u, out, st);
}

void launch_dof_to_gauss_grad(const Mesh &m, const double *grad_out, double *grad_u,
                              hipStream_t st) {
  if (m.degree == 2) return launch_p2_dof_to_gauss_grad(m, grad_out, grad_u, st);
  launch_to_gauss_grad(m, grad_out, grad_u, st);
}

void launch_fem_grad(const Mesh &m, const double *u, double *out, hipStream_t st) {
  if (m.degree == 2) return launch_p2_fem_grad(m, u, out, st);
  by_rule(m, [&](auto nq) {
    fem_grad_kernel<nq()><<<nb(m.nelem, 256), 256, 0, st>>>(
        m.nelem, m.conn.p, m.conn_user.p, m.xy.p, u, out, ((uintptr_t)out & 15) == 0);
  });
}

void launch_fem_grad_grad(const Mesh &m, const double *grad_out, double *grad_u, double *work,
                          hipStream_t st) {
  if (m.degree == 2) return launch_p2_fem_grad_grad(m, grad_out, grad_u, work, st);
  if (work && m.nnode >= GRAD_T_TWO_PASS)
    two_pass<TERM_GRAD_T>(m, grad_out, nullptr, grad_u, work, nullptr, nullptr, st);
  else
    node_gather<NODE_GRAD_T>(m, grad_out, grad_u, st);
}

// A caller without scratch gets a stream-ordered temporary (10 us on the host,
// 20 to 30 when the stream has drained since the last one).
static void laplace_term(const Mesh &m, const double *v, const double *nu, double *out,
                         double *work, const double *u, double *gnu, hipStream_t st) {
  double *c = work;
  if (!work)
    HIPCHECK(hipMallocAsync((void **)&c, sizeof(double) * (m.degree == 2 ? 6 : 3) * m.nelem, st));
  if (m.degree == 2) {
    launch_p2_laplace_term(m, v, nu, out, c, st);
    if (gnu) launch_p2_laplace_term_nu_grad(m, v, u, gnu, st);
  } else if (gnu) {
    two_pass<TERM_LAPLACE_GRAD>(m, v, nu, out, c, u, gnu, st);
  } else {
    two_pass<TERM_LAPLACE>(m, v, nu, out, c, nullptr, nullptr, st);
  }
  if (!work) HIPCHECK(hipFreeAsync(c, st));
}

void launch_laplace_term(const Mesh &m, const double *u, const double *nu, double *out,
                         double *work, hipStream_t st) {
  laplace_term(m, u, nu, out, work, nullptr, nullptr, st);
}

void launch_laplace_term_grad(const Mesh &m, const double *grad_out, const double *u,
                              const double *nu, double *grad_u, double *grad_nu, double *work,
                              hipStream_t st) {
  if (grad_u) return laplace_term(m, grad_out, nu, grad_u, work, u, grad_nu, st);
  if (!grad_nu) return;
  if (m.degree == 2) return launch_p2_laplace_term_nu_grad(m, grad_out, u, grad_nu, st);
  by_rule(m, [&](auto nq) {
    laplace_term_nu_grad_kernel<nq()><<<nb(m.nelem, 256), 256, 0, st>>>(
        m.nelem, m.rule, m.conn.p, m.conn_user.p, m.xy.p, m.area.p, grad_out, u, grad_nu);
  });
}

}  // namespace admfem
