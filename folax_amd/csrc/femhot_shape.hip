// Shape sensitivities: g_x = (dR/dX)^T w, the VJP of the assembled residual with respect to the node
// coordinates, as the reference's adjoint shape derivative contracts it
// (fol/responses/fe_response.py:312-332: jacrev(ComputeElement[1], argnums=0) with the element adjoint,
// assembled per node component at :365-406), and the Gauss-point side of responses.
//
// At a Gauss point w . r is wdet q(grad u, grad w) with q = grad w : P(grad u) (less the body force's
// work).  Moving node b by dX changes wdet by wdet dN_b . dX and a gradient G by -(G dX) (x) dN_b, so
//   d(wdet q)/dX_b = wdet (q I - G_u^T dq/dG_u - G_w^T dq/dG_w) dN_b,
// with the same stresses the residual VJP forms: one pass per element, where differentiating the element
// routine along each of its N x D coordinates took N x D passes.
#include "femhot_launch.h"

namespace femhot {

struct ShapeArgs {
  const double *coords;
  const int *conn;
  long long Ne;
  const void *field, *u, *w;
  const void *wphi;  // optional (Ne, G): weights times an integrand whose own shape derivative is added
  void *gx;          // (Nn, 3) added with atomics, or
  void *corner;      // (Ne, N, D): each corner's part, summed per node by k_corner_gather
  unsigned flags;
  PhysParams pp;
};

// One lane per element.  The corner buffer costs one write and one read of N x D values per element;
// adding into the nodes with atomics instead goes at about 24 G adds/s (23^3 x 6 tetrahedra in FP64: 36 us
// with atomics and one pass per coordinate, 9.7 us here and 6 us for the gather).
template <class R, int ET, int PH, int NGP>
__global__ __launch_bounds__(128) void k_shape_vjp(ShapeArgs A) {
  using E = Elem<R, ET, PH>;
  constexpr int N = E::N, D = E::D, P = E::P, G = RuleSize<ET, NGP>::G;
  const long long e = (long long)blockIdx.x * 128 + threadIdx.x;
  if (e >= A.Ne) return;
  int nodes[N];
  load_conn<N>(A.conn, e, nodes);
  E el;
  load_geometry<R, ET, PH>(A.coords, nodes, el);
  const R *F = reinterpret_cast<const R *>(A.field);
  const R *U = reinterpret_cast<const R *>(A.u);
  const R *W = reinterpret_cast<const R *>(A.w);
  const R *phi = reinterpret_cast<const R *>(A.wphi);
  el.elemental = (A.flags & FEMHOT_ELEMENT_FIELD) != 0;
  el.de = el.elemental ? F[e] : R(0);
  R w[E::NL], gx[N][D];
#pragma unroll
  for (int a = 0; a < N; ++a) {
    el.d[a] = el.elemental ? el.de : F[nodes[a]];
#pragma unroll
    for (int c = 0; c < P; ++c) {
      el.u[a * P + c] = U[(size_t)nodes[a] * P + c];
      w[a * P + c] = W[(size_t)nodes[a] * P + c];
    }
#pragma unroll
    for (int i = 0; i < D; ++i) gx[a][i] = R(0);
  }
#pragma unroll 1
  for (int g = 0; g < G; ++g) {
    GP<R, ET> gp;
    gp_geometry<R, ET, NGP>(g, el.x, gp);
    const R eg = field_gp<R, N>(el.d, el.de, el.elemental, gp.Nv);
    R Gu[P][D], Gw[P][D], Au[P][D], Aw[P][D];  // gradients, and dq/dG_u, dq/dG_w
#pragma unroll
    for (int c = 0; c < P; ++c)
#pragma unroll
      for (int j = 0; j < D; ++j) {
        R s = R(0), t = R(0);
#pragma unroll
        for (int a = 0; a < N; ++a) {
          s += el.u[a * P + c] * gp.DN[a][j];
          t += w[a * P + c] * gp.DN[a][j];
        }
        Gu[c][j] = s;
        Gw[c][j] = t;
      }
    R q = R(0);
    if constexpr (PH == THERMAL) {
      R Tg = R(0);
#pragma unroll
      for (int a = 0; a < N; ++a) Tg += gp.Nv[a] * el.u[a];
      const R k = eg * (R(1) + R(A.pp.beta) * powc(Tg, R(A.pp.c)));
#pragma unroll
      for (int j = 0; j < D; ++j) {
        Au[0][j] = k * Gw[0][j];
        Aw[0][j] = k * Gu[0][j];
      }
    } else if constexpr (PH == MECH) {
      R Su[D][D], Sw[D][D];
      lin_stress<R, D>(Gu, A.pp, Su);
      lin_stress<R, D>(Gw, A.pp, Sw);
      scale_sym<R, D>(Sw, eg, Au);
      scale_sym<R, D>(Su, eg, Aw);
    } else {
      NHState<R, D> st;
      nh_state<R, D>(Gu, R(A.pp.kap1), R(A.pp.mu1), st);
      R X[D][D], dS[D][D];  // sym(F^T Gw) and its stress
#pragma unroll
      for (int i = 0; i < D; ++i)
#pragma unroll
        for (int j = 0; j < D; ++j) {
          R s = R(0);
#pragma unroll
          for (int k = 0; k < D; ++k) s += st.F[k][i] * Gw[k][j] + st.F[k][j] * Gw[k][i];
          X[i][j] = R(0.5) * s;
        }
      nh_tangent_apply<R, D>(st, R(A.pp.kap1), R(A.pp.mu1), X, dS);
#pragma unroll
      for (int i = 0; i < D; ++i)
#pragma unroll
        for (int j = 0; j < D; ++j) {
          R m = R(0), p = R(0);
#pragma unroll
          for (int k = 0; k < D; ++k) {
            m += st.F[i][k] * dS[k][j] + Gw[i][k] * st.S[k][j];
            p += st.F[i][k] * st.S[k][j];
          }
          Au[i][j] = eg * m;
          Aw[i][j] = eg * p;
        }
    }
#pragma unroll
    for (int c = 0; c < P; ++c) {
#pragma unroll
      for (int j = 0; j < D; ++j) q += Gw[c][j] * Aw[c][j];
      if (A.pp.has_body) {
        R wg = R(0);
#pragma unroll
        for (int a = 0; a < N; ++a) wg += gp.Nv[a] * w[a * P + c];
        q -= R(A.pp.body[c]) * wg;
      }
    }
    // M = wdet q I + (w detJ phi) I - wdet (G_u^T A_u + G_w^T A_w); g_x(b) += M dN_b
    const R dg = gp.wdet * q + (phi ? phi[e * G + g] : R(0));
    R M[D][D];
#pragma unroll
    for (int i = 0; i < D; ++i)
#pragma unroll
      for (int j = 0; j < D; ++j) {
        R s = R(0);
#pragma unroll
        for (int c = 0; c < P; ++c) s += Gu[c][i] * Au[c][j] + Gw[c][i] * Aw[c][j];
        M[i][j] = (i == j ? dg : R(0)) - gp.wdet * s;
      }
#pragma unroll
    for (int b = 0; b < N; ++b)
#pragma unroll
      for (int i = 0; i < D; ++i)
#pragma unroll
        for (int j = 0; j < D; ++j) gx[b][i] += M[i][j] * gp.DN[b][j];
  }
  if (A.corner) {
    R *o = reinterpret_cast<R *>(A.corner) + e * (N * D);
#pragma unroll
    for (int a = 0; a < N; ++a)
#pragma unroll
      for (int i = 0; i < D; ++i) o[a * D + i] = gx[a][i];
  } else {
    R *o = reinterpret_cast<R *>(A.gx);
#pragma unroll
    for (int a = 0; a < N; ++a)
#pragma unroll
      for (int i = 0; i < D; ++i) unsafeAtomicAdd(o + (size_t)nodes[a] * 3 + i, gx[a][i]);
  }
}

constexpr int GATHER_U = 8;  // corners per step of the node gathers: two dependent loads each, so latency-bound
                             // (23^3 x 6 tetrahedra FP64: one at a time 12.1 us, eight 6.0)

// g_x of every node from its corners, in element order: three lanes per node, so a corner's D values are
// read as one run (the third component of plane elements is zero).
template <class R, int D>
__global__ __launch_bounds__(256) void k_corner_gather(long long nn, const int *off, const int *list, const R *corner,
                                                       R *gx) {
  const long long t = (long long)blockIdx.x * 256 + threadIdx.x;
  if (t >= 3 * nn) return;
  const long long node = t / 3;
  const int i = (int)(t - 3 * node);
  R s = R(0);
  const int k1 = off[node + 1];
  if (i < D)
    for (int k = off[node]; k < k1; k += GATHER_U) {  // GATHER_U corners' loads in flight, summed in order
      long long at[GATHER_U];
      R v[GATHER_U];
#pragma unroll
      for (int j = 0; j < GATHER_U; ++j) at[j] = (long long)list[min(k + j, k1 - 1)] * D + i;
#pragma unroll
      for (int j = 0; j < GATHER_U; ++j) v[j] = corner[at[j]];
#pragma unroll
      for (int j = 0; j < GATHER_U; ++j) s += k + j < k1 ? v[j] : R(-0.0);
    }
  gx[t] = s;
}

template <int ET> static int launch_shape(int dtype, int ph, int ngp, dim3 grid, hipStream_t s, const ShapeArgs &A) {
  return dispatch_r_ph_ngp(dtype, ph, ngp, [&](auto rp, auto phc, auto ngpc) -> int {
    using R = std::remove_pointer_t<decltype(rp)>;
    constexpr int PH = decltype(phc)::value, NGP = decltype(ngpc)::value;
    hipLaunchKernelGGL((k_shape_vjp<R, ET, PH, NGP>), grid, dim3(128), 0, s, A);
    FH_HIP(hipGetLastError());
    return FEMHOT_OK;
  });
}

// The incidence lists; *ready false when they are not built and `s` is being captured (they are uploaded
// with blocking copies).
static int incidence_for(Ctx *c, hipStream_t s, bool *ready) {
  *ready = true;
  if (c->d_ne_off) return FEMHOT_OK;
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  FH_HIP(hipStreamIsCapturing(s, &cs));
  *ready = cs == hipStreamCaptureStatusNone;
  return *ready ? ensure_incidence(c) : FEMHOT_OK;
}

static int shape_vjp(Ctx *c, int dtype, const void *field, const void *u, const void *w, const void *wphi,
                     void *scratch, void *g_x, unsigned flags, hipStream_t s) {
  int rc;
  bool ready = false;
  if (scratch && (rc = incidence_for(c, s, &ready))) return rc;
  if (!ready) {
    scratch = nullptr;
    rc = dtype == FEMHOT_F32 ? fill<float>((float *)g_x, 3 * c->Nn, 3 * c->Nn, 1, 0.f, s)
                             : fill<double>((double *)g_x, 3 * c->Nn, 3 * c->Nn, 1, 0.0, s);
    if (rc) return rc;
  }
  ShapeArgs A{};
  A.coords = c->d_coords64;
  A.conn = c->d_conn;
  A.Ne = c->Ne;
  A.field = field;
  A.u = u;
  A.w = w;
  A.wphi = wphi;
  A.gx = g_x;
  A.corner = scratch;
  A.flags = flags & FEMHOT_ELEMENT_FIELD;
  A.pp = c->pp;
  const dim3 grid((unsigned)((c->Ne + 127) / 128));
  switch (c->et) {
    case QUAD4: rc = launch_shape<QUAD4>(dtype, c->ph, c->ngp, grid, s, A); break;
    case HEX8: rc = launch_shape<HEX8>(dtype, c->ph, c->ngp, grid, s, A); break;
    default: rc = launch_shape<TET4>(dtype, c->ph, c->ngp, grid, s, A); break;
  }
  if (rc || !scratch) return rc;
  const dim3 gg((unsigned)((3 * c->Nn + 255) / 256));
  auto gather = [&](auto zero) {
    using R = decltype(zero);
    if (c->dim == 2)
      hipLaunchKernelGGL((k_corner_gather<R, 2>), gg, dim3(256), 0, s, c->Nn, c->d_ne_off, c->d_ne_list,
                         (const R *)scratch, (R *)g_x);
    else
      hipLaunchKernelGGL((k_corner_gather<R, 3>), gg, dim3(256), 0, s, c->Nn, c->d_ne_off, c->d_ne_list,
                         (const R *)scratch, (R *)g_x);
  };
  if (dtype == FEMHOT_F32)
    gather(0.0f);
  else
    gather(0.0);
  FH_HIP(hipGetLastError());
  return FEMHOT_OK;
}

}  // namespace femhot

using namespace femhot;

extern "C" int femhot_residual_shape_vjp(femhot_ctx *h, int dtype, const void *field, const void *u, const void *w,
                                         void *g_x, unsigned flags, void *stream) {
  FH_CHECK_ARG(h && field && u && w && g_x, FEMHOT_ERR_ARG, "null argument");
  FH_CHECK_ARG(dtype == FEMHOT_F32 || dtype == FEMHOT_F64, FEMHOT_ERR_ARG, "dtype must be FEMHOT_F32 or FEMHOT_F64");
  return shape_vjp(&h->c, dtype, field, u, w, nullptr, nullptr, g_x, flags, (hipStream_t)stream);
}

extern "C" int femhot_shape_gradient(femhot_ctx *h, int dtype, const void *field, const void *u, const void *w,
                                     const void *wphi, void *scratch, void *g_x, unsigned flags, void *stream) {
  FH_CHECK_ARG(h && field && u && w && g_x && scratch, FEMHOT_ERR_ARG, "null argument");
  FH_CHECK_ARG(dtype == FEMHOT_F32 || dtype == FEMHOT_F64, FEMHOT_ERR_ARG, "dtype must be FEMHOT_F32 or FEMHOT_F64");
  return shape_vjp(&h->c, dtype, field, u, w, wphi, scratch, g_x, flags, (hipStream_t)stream);
}

// ---------------------------------------------------------------------------------------------
// Gauss-point geometry of every element: the integration data a response integrand needs
// (fol/responses/fe_response.py:92-113 evaluates its formula at each Gauss point with weight w detJ,
// field N.d and state N.u; its shape gradient needs d(detJ)/dX = detJ dN/dx).
// ---------------------------------------------------------------------------------------------
namespace femhot {

struct GPDataArgs {
  const double *coords;
  const int *conn;
  long long Ne;
  void *N, *wdet, *dndx;
};

template <class R, int ET, int NGP>
__global__ __launch_bounds__(128) void k_gp_data(GPDataArgs A) {
  constexpr int N = ElemT<ET>::N, D = ElemT<ET>::D, G = RuleSize<ET, NGP>::G;
  const long long e = (long long)blockIdx.x * 128 + threadIdx.x;
  if (e >= A.Ne) return;
  int nodes[N];
  load_conn<N>(A.conn, e, nodes);
  R x[N][D];
  double x0[D];
#pragma unroll
  for (int i = 0; i < D; ++i) x0[i] = A.coords[(size_t)nodes[0] * 3 + i];
#pragma unroll
  for (int a = 0; a < N; ++a)
#pragma unroll
    for (int i = 0; i < D; ++i) x[a][i] = R(A.coords[(size_t)nodes[a] * 3 + i] - x0[i]);
  R *Wd = reinterpret_cast<R *>(A.wdet) + e * G;
  R *Dn = reinterpret_cast<R *>(A.dndx) + e * G * N * D;
  R *Nt = reinterpret_cast<R *>(A.N);
#pragma unroll 1
  for (int g = 0; g < G; ++g) {
    GP<R, ET> gp;
    gp_geometry<R, ET, NGP>(g, x, gp);
    if (Wd) Wd[g] = gp.wdet;
    if (Dn)
#pragma unroll
      for (int a = 0; a < N; ++a)
#pragma unroll
        for (int j = 0; j < D; ++j) Dn[(g * N + a) * D + j] = gp.DN[a][j];
    if (Nt && e == 0)
#pragma unroll
      for (int a = 0; a < N; ++a) Nt[g * N + a] = gp.Nv[a];
  }
}

template <int ET> static int launch_gp_data(int dtype, int ngp, dim3 grid, hipStream_t s, const GPDataArgs &A) {
  auto go = [&](auto rp) -> int {
    using R = std::remove_pointer_t<decltype(rp)>;
    if (ngp == 1)
      hipLaunchKernelGGL((k_gp_data<R, ET, 1>), grid, dim3(128), 0, s, A);
    else if (ngp == 2)
      hipLaunchKernelGGL((k_gp_data<R, ET, 2>), grid, dim3(128), 0, s, A);
    else
      hipLaunchKernelGGL((k_gp_data<R, ET, 3>), grid, dim3(128), 0, s, A);
    FH_HIP(hipGetLastError());
    return FEMHOT_OK;
  };
  return dtype == FEMHOT_F32 ? go((float *)nullptr) : go((double *)nullptr);
}

}  // namespace femhot

extern "C" int femhot_gauss_point_data(femhot_ctx *h, int dtype, void *N, void *wdetJ, void *dNdx, void *stream) {
  FH_CHECK_ARG(h, FEMHOT_ERR_ARG, "null context");
  FH_CHECK_ARG(dtype == FEMHOT_F32 || dtype == FEMHOT_F64, FEMHOT_ERR_ARG, "dtype must be FEMHOT_F32 or FEMHOT_F64");
  FH_CHECK_ARG(N || wdetJ || dNdx, FEMHOT_ERR_ARG, "no output requested");
  Ctx *c = &h->c;
  GPDataArgs A{};
  A.coords = c->d_coords64;
  A.conn = c->d_conn;
  A.Ne = c->Ne;
  A.N = N;
  A.wdet = wdetJ;
  A.dndx = dNdx;
  const dim3 grid((unsigned)((c->Ne + 127) / 128));
  hipStream_t s = (hipStream_t)stream;
  switch (c->et) {
    case QUAD4: return launch_gp_data<QUAD4>(dtype, c->ngp, grid, s, A);
    case HEX8: return launch_gp_data<HEX8>(dtype, c->ngp, grid, s, A);
    default: return launch_gp_data<TET4>(dtype, c->ngp, grid, s, A);
  }
}

// ---------------------------------------------------------------------------------------------
// Responses: nodal values at the Gauss points, and Gauss-point terms back to the nodes (the two sides of
// fol/responses/fe_response.py:92-113 and 271-272 around a response's formula).
// ---------------------------------------------------------------------------------------------
namespace femhot {

struct GPValueArgs {
  const int *conn;
  long long Ne;
  const void *d, *u;
  void *gd, *gu;  // (Ne, G), (P, Ne, G)
};

// N.d and N.u at every Gauss point, one lane per element (a latency-bound gather; writes are runs of G).
template <class R, int ET, int NGP, int P> __global__ __launch_bounds__(128) void k_gp_values(GPValueArgs A) {
  constexpr int N = ElemT<ET>::N, G = RuleSize<ET, NGP>::G;
  const long long e = (long long)blockIdx.x * 128 + threadIdx.x;
  if (e >= A.Ne) return;
  int nodes[N];
  load_conn<N>(A.conn, e, nodes);
  R d[N], u[N][P];
#pragma unroll
  for (int a = 0; a < N; ++a) {
    d[a] = reinterpret_cast<const R *>(A.d)[nodes[a]];
#pragma unroll
    for (int c = 0; c < P; ++c) u[a][c] = reinterpret_cast<const R *>(A.u)[(size_t)nodes[a] * P + c];
  }
#pragma unroll 1
  for (int g = 0; g < G; ++g) {
    double x, y, z, w;
    gauss_point<ET, NGP>(g, x, y, z, w);
    R Nv[N], dN[N][ElemT<ET>::D];
    shape<ET, R>(x, y, z, Nv, dN);
    R s = R(0), t[P];
#pragma unroll
    for (int c = 0; c < P; ++c) t[c] = R(0);
#pragma unroll
    for (int a = 0; a < N; ++a) {
      s += Nv[a] * d[a];
#pragma unroll
      for (int c = 0; c < P; ++c) t[c] += Nv[a] * u[a][c];
    }
    reinterpret_cast<R *>(A.gd)[e * G + g] = s;
#pragma unroll
    for (int c = 0; c < P; ++c) reinterpret_cast<R *>(A.gu)[((long long)c * A.Ne + e) * G + g] = t[c];
  }
}

// out(node, c) = sum over the node's corners of sum_g N_a(g) q(c, e, g), in element order; one lane per node.
template <class R, int ET, int NGP>
__global__ __launch_bounds__(256) void k_gp_gather(long long nn, long long Ne, int nc, const int *off, const int *list,
                                                   const R *q, R *out, int accumulate) {
  constexpr int N = ElemT<ET>::N, G = RuleSize<ET, NGP>::G;
  __shared__ R Nt[N * G];  // shape values, a's row of G
  if ((int)threadIdx.x < G) {
    double x, y, z, w;
    gauss_point<ET, NGP>((int)threadIdx.x, x, y, z, w);
    R Nv[N], dN[N][ElemT<ET>::D];
    shape<ET, R>(x, y, z, Nv, dN);
#pragma unroll
    for (int a = 0; a < N; ++a) Nt[a * G + threadIdx.x] = Nv[a];
  }
  __syncthreads();
  const long long t = (long long)blockIdx.x * 256 + threadIdx.x;
  if (t >= nn * nc) return;
  const long long node = t / nc;
  const int c = (int)(t - node * nc);
  R s = R(0);
  const int k1 = off[node + 1];
  constexpr int U = G == 1 ? GATHER_U : 2;
  for (int k = off[node]; k < k1; k += U) {
    int ea[U];
    R v[U];
#pragma unroll
    for (int j = 0; j < U; ++j) ea[j] = list[min(k + j, k1 - 1)];
#pragma unroll
    for (int j = 0; j < U; ++j) {
      const int e = ea[j] / N, a = ea[j] - e * N;
      const R *p = q + ((long long)c * Ne + e) * G;
      R t = R(0);
#pragma unroll
      for (int g = 0; g < G; ++g) t += Nt[a * G + g] * p[g];
      v[j] = t;
    }
#pragma unroll
    for (int j = 0; j < U; ++j) s += k + j < k1 ? v[j] : R(-0.0);
  }
  out[t] = accumulate ? out[t] + s : s;
}

// Calls f(R*, ET, NGP)
template <class F> static int dispatch_gp(int dtype, int et, int ngp, F &&f) {
  using std::integral_constant;
  auto with_rule = [&](auto rp, auto etc) -> int {
    if (ngp == 1) return f(rp, etc, integral_constant<int, 1>{});
    if (ngp == 2) return f(rp, etc, integral_constant<int, 2>{});
    return f(rp, etc, integral_constant<int, 3>{});
  };
  auto with_type = [&](auto rp) -> int {
    if (et == QUAD4) return with_rule(rp, integral_constant<int, QUAD4>{});
    if (et == HEX8) return with_rule(rp, integral_constant<int, HEX8>{});
    return with_rule(rp, integral_constant<int, TET4>{});
  };
  return dtype == FEMHOT_F32 ? with_type((float *)nullptr) : with_type((double *)nullptr);
}

}  // namespace femhot

extern "C" int femhot_gauss_point_values(femhot_ctx *h, int dtype, const void *field, const void *u, void *gp_field,
                                         void *gp_u, void *stream) {
  FH_CHECK_ARG(h && field && u && gp_field && gp_u, FEMHOT_ERR_ARG, "null argument");
  FH_CHECK_ARG(dtype == FEMHOT_F32 || dtype == FEMHOT_F64, FEMHOT_ERR_ARG, "dtype must be FEMHOT_F32 or FEMHOT_F64");
  Ctx *c = &h->c;
  GPValueArgs A{c->d_conn, c->Ne, field, u, gp_field, gp_u};
  const dim3 grid((unsigned)((c->Ne + 127) / 128));
  return dispatch_gp(dtype, c->et, c->ngp, [&](auto rp, auto etc, auto ngpc) -> int {
    using R = std::remove_pointer_t<decltype(rp)>;
    constexpr int ET = decltype(etc)::value, NGP = decltype(ngpc)::value;
    if (c->ndpn == 1)
      hipLaunchKernelGGL((k_gp_values<R, ET, NGP, 1>), grid, dim3(128), 0, (hipStream_t)stream, A);
    else
      hipLaunchKernelGGL((k_gp_values<R, ET, NGP, ElemT<ET>::D>), grid, dim3(128), 0, (hipStream_t)stream, A);
    FH_HIP(hipGetLastError());
    return FEMHOT_OK;
  });
}

extern "C" int femhot_incidence(femhot_ctx *h) {
  FH_CHECK_ARG(h, FEMHOT_ERR_ARG, "null context");
  return ensure_incidence(&h->c);
}

extern "C" int femhot_gauss_point_gather(femhot_ctx *h, int dtype, int ncomp, const void *q, void *out,
                                         unsigned flags, void *stream) {
  FH_CHECK_ARG(h && q && out, FEMHOT_ERR_ARG, "null argument");
  FH_CHECK_ARG(dtype == FEMHOT_F32 || dtype == FEMHOT_F64, FEMHOT_ERR_ARG, "dtype must be FEMHOT_F32 or FEMHOT_F64");
  FH_CHECK_ARG(ncomp >= 1 && ncomp <= 3, FEMHOT_ERR_SHAPE, "one to three components");
  Ctx *c = &h->c;
  hipStream_t s = (hipStream_t)stream;
  bool ready = false;
  if (int rc = incidence_for(c, s, &ready)) return rc;
  FH_CHECK_ARG(ready, FEMHOT_ERR_ARG, "call femhot_incidence before capturing the gather");
  const dim3 grid((unsigned)((c->Nn * ncomp + 255) / 256));
  return dispatch_gp(dtype, c->et, c->ngp, [&](auto rp, auto etc, auto ngpc) -> int {
    using R = std::remove_pointer_t<decltype(rp)>;
    hipLaunchKernelGGL((k_gp_gather<R, decltype(etc)::value, decltype(ngpc)::value>), grid, dim3(256), 0, s, c->Nn,
                       c->Ne, ncomp, c->d_ne_off, c->d_ne_list, (const R *)q, (R *)out,
                       (flags & FEMHOT_ACCUMULATE) ? 1 : 0);
    FH_HIP(hipGetLastError());
    return FEMHOT_OK;
  });
}
