// Row-owner assembly of the tangent on the CSR pattern, thermal and linear-elastic physics
// (the element tangents of fe_loss.py:264-318, BC-masked as fe_loss.py:191-207).
//
// One 64-lane workgroup owns node i: the P rows of i (P * P * deg consecutive values, deg = number
// of neighbours of i including i) are summed from i's incident elements in a fixed order and each
// value is written once, so the assembly needs no zero fill, no atomics and no colouring, and reads
// and writes every CSR value exactly once.  Per batch of up to EB incident elements:
//   1. lane (element s, Gauss point g) computes the geometry of g and stages dN/dx of all N nodes
//      and the Gauss factor f_g in LDS;
//   2. lane (element s, node b) forms block (a, b) of the element tangent (a = local index of i in
//      s), Dirichlet-masked, stores it in LDS and sets its bit in the mask of its column k (the
//      position of node b among i's neighbours, from the slot table);
//   3. lane per output value (row c, column k, component d; CPW columns per round, so a lane keeps its row
//      and component) adds the blocks of the lanes in column k's mask, in lane order (element order,
//      then b), to its register accumulator.
// Columns are taken KW at a time; one window covers every node of hexahedral and tetrahedral meshes
// of ordinary valence, and a wider node repeats the batches once per window.
//
// Blocks.  Thermal: K_ab = sum_g f_g dN_a . dN_b, f_g = wdetJ k0_g (1 + beta T_g^c), the Picard
// matrix of thermal.py:31-40.  Linear elastic: with M_ab = sum_g f_g dN_a (x) dN_b and f_g = wdetJ E_g,
//   K_ab[c][c] = c2 M[c][c] + c4 sum_{j != c} M[j][j],   K_ab[c][d] = c3 M[c][d] + c4 M[d][c] (c != d),
// which is B_a^T D B_b for the isotropic D of mechanical.py:60-82 (c2 = D_00, c3 = D_01, c4 = D_33 in
// 3-D; f2, f2nu, f2sh of plane stress in 2-D).  Both element tangents are symmetric, so
// FEMHOT_TRANSPOSE leaves them unchanged.
//
// Residual (A.R): formed in the same pass from the blocks, so a call that wants both reads the mesh and the
// fields once and needs no second kernel, workspace or plan.  Linear elastic in FP64, with the residual through the chunk
// kernel and here: tetrahedra 40^3 x 6 158 and 140 us, quads 200 x 200 46 and 38.  On elastic quads the gather of u and the
// store of the residual cost a sixth of the tangent at every size, so from about 500 x 500 the separate kernel would be
// faster once its plan is built (700 x 700: 433 and 447).
#pragma once
#include "femhot_kernels.h"

namespace femhot {

// Shape function value and local gradient of node a (unrolled callers make a a constant).
template <int ET, class R>
__device__ __forceinline__ void shape_node(int a, double x, double y, double z, R &Na, R (&dn)[ElemT<ET>::D]) {
  if constexpr (ET == QUAD4) {
    const double sx = (a == 1 || a == 2) ? 1.0 : -1.0, sy = (a >= 2) ? 1.0 : -1.0;
    Na = R(0.25 * (1.0 + sx * x) * (1.0 + sy * y));
    dn[0] = R(0.25 * sx * (1.0 + sy * y));
    dn[1] = R(0.25 * sy * (1.0 + sx * x));
  } else if constexpr (ET == HEX8) {
    const int q = a & 3;
    const double sx = (q == 1 || q == 2) ? 1.0 : -1.0, sy = (q >= 2) ? 1.0 : -1.0, sz = (a >= 4) ? 1.0 : -1.0;
    const double px = 1.0 + sx * x, py = 1.0 + sy * y, pz = 1.0 + sz * z;
    Na = R(0.125 * px * py * pz);
    dn[0] = R(0.125 * sx * py * pz);
    dn[1] = R(0.125 * sy * px * pz);
    dn[2] = R(0.125 * sz * px * py);
  } else {
    Na = R(a == 0 ? 1.0 - (x + y + z) : a == 1 ? x : a == 2 ? y : z);
    dn[0] = R(a == 0 ? -1.0 : a == 1 ? 1.0 : 0.0);
    dn[1] = R(a == 0 ? -1.0 : a == 2 ? 1.0 : 0.0);
    dn[2] = R(a == 0 ? -1.0 : a == 3 ? 1.0 : 0.0);
  }
}

// Whether the lanes of an element form the moments of its coordinates together: HEX8 beyond the one-point rule, whose
// only Gauss-point lane needs three of the seven (30^3 thermal FP32 tangent: 24.8 us together, 22.7 alone).
template <int ET, int NGP> constexpr bool rows_moments() { return ET == HEX8 && NGP > 1; }

// Inverse Jacobian of Gauss point g of one element for the row-owner staging, with the shape function
// values there: the arithmetic of gp_geometry (coordinates relative to node 0, J = sum_a x_a (x)
// dN_a/dxi, inverse by cofactors), returning wdetJ.  xs: the element's node coordinates (N x 3, FP64).
// HEX8 takes the trilinear modes of femhot_physics.h instead: J from the moments of the coordinates
// (adds only, then 4 terms per entry), and the pair (8 J)^-1 with stage_gradients' 8 dN/dxi.
template <class R, int ET, int NGP>
__device__ __forceinline__ R gp_inverse(int g, const double *xs, R (&Nv)[ElemT<ET>::N],
                                        R (&inv)[ElemT<ET>::D][ElemT<ET>::D]) {
  constexpr int N = ElemT<ET>::N, D = ElemT<ET>::D;
  double xi, eta, zeta, w;
  gauss_point<ET, NGP>(g, xi, eta, zeta, w);
  if constexpr (ET == HEX8) {  // xs holds the coordinates' moments (rows_moments) or the coordinates
    R J[3][3];  // 8 J
    const R X = R(xi), Y = R(eta), Z = R(zeta), XY = R(xi * eta), XZ = R(xi * zeta), YZ = R(eta * zeta);
    constexpr int lane_of[8] = {0, 1, 3, 4, 2, 5, 7, 6};  // the lane that holds moment m
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      R m[8];
      if constexpr (rows_moments<ET, NGP>()) {
        m[0] = R(0);
#pragma unroll
        for (int k = 1; k < 8; ++k) m[k] = R(xs[lane_of[k] * 3 + i]);
      } else {
        R col[8];
        col[0] = R(0);
#pragma unroll
        for (int a = 1; a < 8; ++a) col[a] = R(xs[a * 3 + i] - xs[i]);
        hex8_moments<R>(col, m);
      }
      hex8_dxi<R>(m, X, Y, Z, XY, XZ, YZ, J[i]);
    }
#pragma unroll
    for (int a = 0; a < 8; ++a) {
      R dn[3];
      shape_node<ET, R>(a, xi, eta, zeta, Nv[a], dn);
    }
    const R c00 = J[1][1] * J[2][2] - J[1][2] * J[2][1];
    const R c01 = J[1][2] * J[2][0] - J[1][0] * J[2][2];
    const R c02 = J[1][0] * J[2][1] - J[1][1] * J[2][0];
    const R det8 = J[0][0] * c00 + J[0][1] * c01 + J[0][2] * c02;
    const R id = recip(det8);
    inv[0][0] = c00 * id;
    inv[1][0] = c01 * id;
    inv[2][0] = c02 * id;
    inv[0][1] = (J[0][2] * J[2][1] - J[0][1] * J[2][2]) * id;
    inv[1][1] = (J[0][0] * J[2][2] - J[0][2] * J[2][0]) * id;
    inv[2][1] = (J[0][1] * J[2][0] - J[0][0] * J[2][1]) * id;
    inv[0][2] = (J[0][1] * J[1][2] - J[0][2] * J[1][1]) * id;
    inv[1][2] = (J[0][2] * J[1][0] - J[0][0] * J[1][2]) * id;
    inv[2][2] = (J[0][0] * J[1][1] - J[0][1] * J[1][0]) * id;
    return R(w * (1.0 / 512.0)) * det8;
  }
  double x0[D];
#pragma unroll
  for (int i = 0; i < D; ++i) x0[i] = xs[i];
  R J[D][D];
  {
    R dn[D];
    shape_node<ET, R>(0, xi, eta, zeta, Nv[0], dn);
  }
#pragma unroll
  for (int a = 1; a < N; ++a) {
    R xa[D], dn[D];
#pragma unroll
    for (int i = 0; i < D; ++i) xa[i] = R(xs[a * 3 + i] - x0[i]);
    shape_node<ET, R>(a, xi, eta, zeta, Nv[a], dn);
    if constexpr (ET == TET4) {
#pragma unroll
      for (int i = 0; i < D; ++i) J[i][a - 1] = xa[i];
    } else {
#pragma unroll
      for (int i = 0; i < D; ++i)
#pragma unroll
        for (int k = 0; k < D; ++k) J[i][k] = (a == 1) ? xa[i] * dn[k] : J[i][k] + xa[i] * dn[k];
    }
  }
  R det;
  if constexpr (D == 2) {
    det = J[0][0] * J[1][1] - J[0][1] * J[1][0];
    const R id = recip(det);
    inv[0][0] = J[1][1] * id;
    inv[0][1] = -J[0][1] * id;
    inv[1][0] = -J[1][0] * id;
    inv[1][1] = J[0][0] * id;
  } else {
    const R c00 = J[1][1] * J[2][2] - J[1][2] * J[2][1];
    const R c01 = J[1][2] * J[2][0] - J[1][0] * J[2][2];
    const R c02 = J[1][0] * J[2][1] - J[1][1] * J[2][0];
    det = J[0][0] * c00 + J[0][1] * c01 + J[0][2] * c02;
    const R id = recip(det);
    inv[0][0] = c00 * id;
    inv[1][0] = c01 * id;
    inv[2][0] = c02 * id;
    inv[0][1] = (J[0][2] * J[2][1] - J[0][1] * J[2][2]) * id;
    inv[1][1] = (J[0][0] * J[2][2] - J[0][2] * J[2][0]) * id;
    inv[2][1] = (J[0][1] * J[2][0] - J[0][0] * J[2][1]) * id;
    inv[0][2] = (J[0][1] * J[1][2] - J[0][2] * J[1][1]) * id;
    inv[1][2] = (J[0][2] * J[1][0] - J[0][0] * J[1][2]) * id;
    inv[2][2] = (J[0][0] * J[1][1] - J[0][1] * J[1][0]) * id;
  }
  return R(w) * det;
}

// dN_b/dx = dN_b/dxi . inv(J) of every node at Gauss point g, stored at st[b * D + j] (TET4: the
// rows of inv(J), node 0 minus their sum, as gp_geometry; HEX8: (8 dN_b/dxi) . inv(8 J), from the
// node signs).
template <class R, int ET, int NGP>
__device__ __forceinline__ void stage_gradients(int g, const R (&inv)[ElemT<ET>::D][ElemT<ET>::D], R *st) {
  constexpr int N = ElemT<ET>::N, D = ElemT<ET>::D;
  if constexpr (ET == HEX8) {
    double xi, eta, zeta, w;
    gauss_point<ET, NGP>(g, xi, eta, zeta, w);
    const R X = R(xi), Y = R(eta), Z = R(zeta);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      const int q = b & 3;
      const R sx = (q == 1 || q == 2) ? R(1) : R(-1), sy = q >= 2 ? R(1) : R(-1), sz = b >= 4 ? R(1) : R(-1);
      const R px = R(1) + sx * X, py = R(1) + sy * Y, pz = R(1) + sz * Z;
      const R sh[3] = {sx * (py * pz), sy * (px * pz), sz * (px * py)};
#pragma unroll
      for (int j = 0; j < 3; ++j) st[b * 3 + j] = (sh[0] * inv[0][j] + sh[1] * inv[1][j]) + sh[2] * inv[2][j];
    }
  } else if constexpr (ET == TET4) {
#pragma unroll
    for (int j = 0; j < D; ++j) {
      st[1 * D + j] = inv[0][j];
      st[2 * D + j] = inv[1][j];
      st[3 * D + j] = inv[2][j];
      st[j] = -((inv[0][j] + inv[1][j]) + inv[2][j]);
    }
  } else {
    double xi, eta, zeta, w;
    gauss_point<ET, NGP>(g, xi, eta, zeta, w);
#pragma unroll
    for (int b = 0; b < N; ++b) {
      R Nb, dn[D];
      shape_node<ET, R>(b, xi, eta, zeta, Nb, dn);
#pragma unroll
      for (int j = 0; j < D; ++j) {
        R s = dn[0] * inv[0][j];
#pragma unroll
        for (int k = 1; k < D; ++k) s += dn[k] * inv[k][j];
        st[b * D + j] = s;
      }
    }
  }
}

// Coordinate of a HEX8 node -> moment of the element's coordinates (hex8_moments' sums, in its order), across
// the 8 lanes that hold the element's nodes 0..7: coordinates relative to node 0, then one butterfly per
// reference direction with DPP register moves.  Lane b ends with the moment whose sign product is that of
// the directions in which node b lies on the + side: moment lane_of^-1 of gp_inverse.  Formed
// once per element where every Gauss-point lane formed all of them (93 FP64 adds each).
template <int CTRL, int BANKS> __device__ __forceinline__ double rows_dpp_into(double old, double v) {
  const int lo = __builtin_amdgcn_update_dpp(__double2loint(old), __double2loint(v), CTRL, 0xf, BANKS, false);
  const int hi = __builtin_amdgcn_update_dpp(__double2hiint(old), __double2hiint(v), CTRL, 0xf, BANKS, false);
  return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double hex8_lane_moment(double v, int b) {
  // node 0's value: lane 0 of the lower and lane 8 of the upper half of each row of 16 (row_newbcast)
  double ref = lane_dpp<0x150, 0x3>(v);
  ref = rows_dpp_into<0x158, 0xc>(ref, v);
  v -= ref;
  const double sx = (b & 3) == 1 || (b & 3) == 2 ? -1.0 : 1.0, sy = (b & 3) >= 2 ? -1.0 : 1.0, sz = b >= 4 ? -1.0 : 1.0;
  // the lane on the - side adds its partner, the one on the + side subtracts it (products by +-1 are exact)
  v = __builtin_fma(sx, lane_dpp<0xB1>(v), v);  // b ^ 1 (quad_perm [1,0,3,2])
  v = __builtin_fma(sy, lane_dpp<0x1B>(v), v);  // b ^ 3 (quad_perm [3,2,1,0])
  double up = lane_dpp<0x104, 0x5>(v);    // b ^ 4: row_shl:4 into banks 0 and 2,
  up = rows_dpp_into<0x114, 0xa>(up, v);  // row_shr:4 into banks 1 and 3
  return __builtin_fma(sz, up, v);
}

template <int ET, int NGP, int N, int P> struct RowsShape {
  static constexpr int G = RuleSize<ET, NGP>::G;
  static constexpr int CPW = 64 / (P * P);                         // columns per round of the output stage
  static constexpr int EB = (64 / G < 64 / N) ? 64 / G : 64 / N;  // incident elements per batch
  static constexpr int KW = (P == 3) ? 28 : 64;                    // neighbour columns per window
  static constexpr int OR = (KW + CPW - 1) / CPW;                  // output values per lane per window
};

// CS[k] = first block of column k: exclusive prefix sums of the columns' lane counts, by DPP register moves.
template <int KW>
__device__ __forceinline__ void rows_column_starts(int lane, int kw, const unsigned long long *MK, int *CS) {
  int pc = lane < kw ? __popcll(MK[lane]) : 0;
  pc += __builtin_amdgcn_update_dpp(0, pc, 0x111, 0xf, 0xf, true);  // row_shr:1, 2, 4, 8: sums in rows of 16
  pc += __builtin_amdgcn_update_dpp(0, pc, 0x112, 0xf, 0xf, true);
  pc += __builtin_amdgcn_update_dpp(0, pc, 0x114, 0xf, 0xf, true);
  pc += __builtin_amdgcn_update_dpp(0, pc, 0x118, 0xf, 0xf, true);
  pc += __builtin_amdgcn_update_dpp(0, pc, 0x142, 0xa, 0xf, false);  // row_bcast:15 into rows 1 and 3
  pc += __builtin_amdgcn_update_dpp(0, pc, 0x143, 0xc, 0xf, false);  // row_bcast:31 into rows 2 and 3
  if (lane < kw) CS[lane + 1] = pc;
  if (lane == 0) CS[0] = 0;
}

// Output stage: a lane owns row oc, component od and column kk of each round's CPW, and adds the column's
// blocks in lane order.  The first four blocks of every round are loaded together, so their LDS latency is
// paid once and not once a round (S reaches 3 blocks past the last); the sums stop at the column's end
// by branches, for a select costs three instructions an entry.  With two dofs per node the rounds go one at a time and
// those past the node's columns are left out: a window has four, and the 9 neighbours of a quadrilateral's node fill one,
// so loads for all four cost instructions and registers alone (300 x 300 elastic one-point tangent: FP64 54.0 us with 94
// VGPRs, 48.5 with 78 and six waves per SIMD; FP32 41.0 and 35.5.  Hexahedra fill all four of theirs, and the test
// costs their 64^3 call 392 us against 385).
template <class R, int N> __device__ __forceinline__ R rows_sum_four(int n, const R (&x)[N], R sum) {
  if (n > 0) {
    sum += x[0];
    if (n > 1) {
      asm volatile("" ::: "memory");  // keeps these branches
      sum += x[1];
      if (n > 2) {
        asm volatile("" ::: "memory");
        sum += x[2];
        if (n > 3) {
          asm volatile("" ::: "memory");
          sum += x[3];
        }
      }
    }
  }
  return sum;
}
template <class R, int P, int CPW, int OR>
__device__ __forceinline__ void rows_add_columns(int kw, int oc, int kk, int od, const R *S, const int *CS,
                                                 R (&acc)[OR]) {
  constexpr int T = P == 2 ? 1 : OR;  // rounds whose loads are issued together
#pragma unroll
  for (int r0 = 0; r0 < OR; r0 += T) {
    if (P == 2 && r0 * CPW >= kw) continue;
    int lo[T], n[T];
    R x[T][4];
#pragma unroll
    for (int r = 0; r < T; ++r) {
      const int k = (r0 + r) * CPW + kk;
      const bool own = k < kw && oc < P;
      lo[r] = own ? CS[k] : 0;
      n[r] = own ? CS[k + 1] - lo[r] : 0;
    }
#pragma unroll
    for (int r = 0; r < T; ++r)
#pragma unroll
      for (int q = 0; q < 4; ++q) x[r][q] = S[(lo[r] + q) * (P * P) + oc * P + od];
#pragma unroll
    for (int r = 0; r < T; ++r) {
      R sum = rows_sum_four(n[r], x[r], R(0));
      for (int i = 4; i < n[r]; i += 4) {
        R y[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) y[q] = S[(lo[r] + i + q) * (P * P) + oc * P + od];
        sum = rows_sum_four(n[r] - i, y, sum);
      }
      acc[r0 + r] += sum;
    }
  }
}
template <class R, int P, int CPW, int OR>
__device__ __forceinline__ void rows_write(int kw, int k0, int deg, int oc, int kk, int od, bool accumulate,
                                           const R (&acc)[OR], R *V) {
#pragma unroll
  for (int r = 0; r < OR; ++r) {
    if (P == 2 && r * CPW >= kw) continue;  // (as rows_add_columns)
    const int k = r * CPW + kk;
    if (k >= kw || oc >= P) continue;
    R *v = V + oc * P * deg + (k0 + k) * P + od;
    *v = accumulate ? *v + acc[r] : acc[r];
  }
}

// K (u - u_i) of the output lanes' values of one window: DU = the columns' u_b - u_i.
template <class R, int P, int CPW, int OR>
__device__ __forceinline__ R rows_apply(int kw, int oc, int kk, int od, const R *DU, const R (&acc)[OR]) {
  R s = R(0);
#pragma unroll
  for (int r = 0; r < OR; ++r) {
    if (P == 2 && r * CPW >= kw) continue;  // (as rows_add_columns)
    const int k = r * CPW + kk;
    if (k < kw && oc < P) s += acc[r] * DU[k * P + od];
  }
  return s;
}

// v of lane l (the same in all lanes) in all lanes.
__device__ __forceinline__ float rows_lane(float v, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
__device__ __forceinline__ double rows_lane(double v, int l) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l), __builtin_amdgcn_readlane(__double2loint(v), l));
}
// Sums over lanes 0..31 and 32..63, valid in lanes 31 and 63 (wave_sum_to_last without its last step).
__device__ __forceinline__ float rows_from_15(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x142, 0xa, 0xf, false));
}
__device__ __forceinline__ double rows_from_15(double v) { return dpp_f64<0x142, 0xa>(v); }
template <class R> __device__ __forceinline__ R rows_half_sums(R v) {
  v += lane_dpp<0xB1>(v);
  v += lane_dpp<0x4E>(v);
  v += lane_dpp<0x141>(v);
  v += lane_dpp<0x140>(v);
  return v + rows_from_15(v);
}

// The owned node's residual, masked as fe_loss.py:191-207: the output lanes' shares of K (u - u_i) (SHARES;
// lane / G is the component) and, with lanes, each lane's own res, summed in a fixed order.  S: 64 values of scratch;
// with one or two components those of each are the wave or a half of it, and register moves do (tangent and residual, 300 x
// 300 quads, through scratch and by moves: thermal FP32 49.3 and 43.5 us, FP64 89.9 and 83.2, elastic FP32 62.2 and 59.9).
template <class R, int P, int G, bool SHARES>
__device__ __forceinline__ void rows_write_residual(R share, const R (&res)[P], bool lanes, unsigned dm,
                                                    bool accumulate, R *S, R *out) {
  constexpr int LPC = P == 1 ? 64 : P == 2 ? 32 : 16;  // lanes per component
  static_assert(P == 3 || !SHARES || G == LPC, "a component's shares fill its lanes");
  const int lane = threadIdx.x, c = lane / LPC;
  const bool writer = (lane & (LPC - 1)) == LPC - 1 && c < P;
  R x = R(0);
  if constexpr (SHARES && P == 1) {
    x = wave_sum_to_last(share);
  } else if constexpr (SHARES && P == 2) {
    x = rows_half_sums(share);
  } else if constexpr (SHARES) {
    S[lane] = share;
    __syncthreads();
    for (int m = lane & 15; c < P && m < G; m += 16) x += S[c * G + m];
    x += lane_dpp<0xB1>(x);
    x += lane_dpp<0x4E>(x);
    x += lane_dpp<0x141>(x);
    x += lane_dpp<0x140>(x);
  }
  const bool masked = (dm >> c) & 1;
  if (lanes) {
#pragma unroll
    for (int k = 0; k < P; ++k) {
      const R s = rows_lane(wave_sum_to_last(res[k]), 63);
      x += c == k ? s : R(0);
    }
  }
  if (writer) {
    if (!accumulate)
      out[c] = masked ? R(0) : x;
    else if (!masked)
      out[c] += x;
  }
}

// Waves per SIMD the compiler must fit: 3 for linear elasticity (130 VGPRs at most, at the 27-point rule of HEX8, no spills);
// the thermal instantiations keep the compiler's own choice (the powc of k(T) would spill), except that FP64 tetrahedra at
// four points, whose choice is 3, take 4 with 4 spilled registers (24^3 x 6, tangent: 32.0 us at 3 waves, 29.5 at 4).
template <class R, int ET, int PH, int NGP> constexpr int rows_min_waves() {
  if (PH == MECH) return 3;
  return ET == TET4 && NGP == 2 && sizeof(R) == 8 ? 4 : 1;
}

template <class R, int ET, int PH, int NGP>
__global__ __launch_bounds__(64, (rows_min_waves<R, ET, PH, NGP>())) void k_tangent_rows(TArgs A) {
  static_assert(PH != NEOHOOKE, "row-owner assembly covers thermal and linear elasticity");
  using E = Elem<R, ET, PH>;
  constexpr int N = E::N, D = E::D, P = E::P;
  using SH = RowsShape<ET, NGP, N, P>;
  constexpr int G = SH::G, EB = SH::EB, KW = SH::KW, OR = SH::OR, CPW = SH::CPW;
  constexpr int UNR = G <= 8 ? G : 1;
  constexpr int ST = N * D + 1;  // staged values per (element, Gauss point): dN/dx of N nodes, f_g
  constexpr int SW = (EB * G * ST > 64 * P * P) ? EB * G * ST : 64 * P * P;
  // LDS: S holds the staged geometry, then the 64 lanes' P x P blocks.  The node data of step 0
  // (coordinates XS, field FS, thermal solution US of lane (s, b) = node b of incident element s)
  // sits at the end of the same space: step 1 reads all of it before it writes the geometry (each
  // lane's writes depend on its reads, and the workgroup is one wave), so the two never overlap in
  // time and the workgroup needs no extra LDS.
  constexpr int XW = (64 * 3 * 8 + 2 * 64 * (int)sizeof(R)) / (int)sizeof(R);  // a multiple of 4
  // (the output stage reads up to 3 blocks past a column's last: 4 more blocks stay in bounds)
  constexpr int SB = SW > (64 + 4) * P * P ? SW : (64 + 4) * P * P;
  constexpr int SX = ((SB > XW ? SB : XW) + 3) & ~3;  // so XS starts 16-byte aligned
  __shared__ __align__(16) R S[SX];
  __shared__ unsigned long long MK[KW];
  __shared__ int CS[KW + 1];
  __shared__ R DU[KW * P];  // u_b - u_i of the window's columns
  double *XS = reinterpret_cast<double *>(S + SX - XW);
  R *FS = reinterpret_cast<R *>(XS + 64 * 3);
  R *US = FS + 64;
  const int lane = threadIdx.x;
  // Workgroups go to the 8 XCDs in turn, and nodes with nearby ids share elements: XCD x takes the
  // x-th eighth of the nodes in order, so its workgroups find their neighbours' element data in
  // its own L2 (a bijection of workgroup ids onto nodes)
  const long long per = gridDim.x / 8, rem = gridDim.x % 8;
  const long long xcd = blockIdx.x % 8, q = blockIdx.x / 8;
  const long long node = xcd * per + (xcd < rem ? xcd : rem) + q;
  const int off0 = A.ne_off[node], cnt = A.ne_off[node + 1] - off0;
  const long long rp = A.row_ptr[node * P];
  const int deg = (int)((A.row_ptr[node * P + 1] - rp) / P);
  // the Dirichlet mask in lanes 0..P-1, a bit mask where it is needed (read as a scalar it would be waited
  // for before the first element is fetched)
  const int dmv = lane < P ? A.dmask[node * P + lane] : 0;
  const bool elemental = (A.flags & FEMHOT_ELEMENT_FIELD) != 0;
  const bool accumulate = (A.flags & FEMHOT_ACCUMULATE) != 0;
  const R *F = reinterpret_cast<const R *>(A.field);
  const R *U = reinterpret_cast<const R *>(A.u);
  R *V = reinterpret_cast<R *>(A.vals) + rp;
  const int s2 = lane / N, b2 = lane - s2 * N;  // lane (element, node) of steps 0 and 2
  const int s1 = lane / G, g1 = lane - s1 * G;  // lane (element, Gauss point) of step 1
  // lane of the output stage: row oc, column kk of a round's CPW, component od (row by row, so a round
  // writes P runs of CPW * P values); lanes past P rows idle
  const int oc = lane / (CPW * P), kk = (lane - oc * CPW * P) / P, od = lane - oc * CPW * P - kk * P;
  // The residual of these physics is K u (Picard K for thermal) less the body force, and the rows of K sum to
  // zero, so with du_b = u_b - u_i it is sum K_ab du_b: an FMA per value in the output lanes.
  const bool want_r = A.R != nullptr;
  R res[P], ui[P], share = R(0);
#pragma unroll
  for (int c = 0; c < P; ++c) {
    res[c] = R(0);
    ui[c] = want_r ? U[node * P + c] : R(0);
  }
  for (int k0 = 0; k0 < deg; k0 += KW) {
    const bool first = want_r && k0 == 0;
    const int kw = min(KW, deg - k0);
    R acc[OR];
#pragma unroll
    for (int r = 0; r < OR; ++r) acc[r] = R(0);
    for (int base = 0; base < cnt; base += EB) {
      const int nb = min(EB, cnt - base);
      // 0. lane (s, b) fetches node b of incident element s: coordinates, field and (thermal)
      //    solution to LDS; its column among the owned node's neighbours stays in a register
      int a2 = 0, col = -1;
      double xc[3] = {0.0, 0.0, 0.0};
      if (s2 < nb) {
        const int ea = A.ne_list[off0 + base + s2];
        const int e = ea / N;
        a2 = ea - e * N;
        col = A.slot[((size_t)e * N + a2) * N + b2];
        const int nd = A.conn[(size_t)e * N + b2];
#pragma unroll
        for (int i = 0; i < 3; ++i) xc[i] = A.coords[(size_t)nd * 3 + i];
        FS[lane] = elemental ? F[e] : F[nd];
        if constexpr (PH == THERMAL) US[lane] = U[nd];
        if (want_r && col >= k0 && col < k0 + kw) {
#pragma unroll
          for (int c = 0; c < P; ++c) DU[(col - k0) * P + c] = U[(size_t)nd * P + c] - ui[c];
        }
      }
#pragma unroll
      for (int i = 0; i < 3; ++i) XS[lane * 3 + i] = rows_moments<ET, NGP>() ? hex8_lane_moment(xc[i], b2) : xc[i];
      for (int t = lane; t < kw; t += 64) MK[t] = 0ull;
      __syncthreads();
      // the lanes of each column of the window, as a bit mask
      if (col >= k0 && col < k0 + kw) atomicOr(&MK[col - k0], 1ull << lane);
      if (s1 < nb) {  // 1. geometry of (element, Gauss point) pairs
        const int n0 = s1 * N;
        R *st = S + lane * ST;
        R Nv[N], inv[D][D];
        const R wdet = gp_inverse<R, ET, NGP>(g1, XS + n0 * 3, Nv, inv);
        if (first && A.pp.has_body) {  // this lane's point of the owned node's body force
          const int a1 = A.ne_list[off0 + base + s1] % N;
          R na = Nv[0];
#pragma unroll
          for (int b = 1; b < N; ++b) na = b == a1 ? Nv[b] : na;
#pragma unroll
          for (int c = 0; c < P; ++c) res[c] -= (wdet * na) * R(A.pp.body[c]);
        }
        R eg;
        if (elemental) {
          eg = FS[n0];
        } else {
          eg = R(-0.0);
#pragma unroll
          for (int b = 0; b < N; ++b) eg += Nv[b] * FS[n0 + b];
        }
        R f = wdet * eg;
        if constexpr (PH == THERMAL) {
          R Tg = R(-0.0);
#pragma unroll
          for (int b = 0; b < N; ++b) Tg += Nv[b] * US[n0 + b];
          f *= R(1) + R(A.pp.beta) * powc(Tg, R(A.pp.c));
        }
        // inv(J) and f make a round trip through this lane's own staging slot, and the Gauss point
        // index an opaque copy, so the compiler keeps neither the Jacobian step's values nor its
        // shape derivatives live into the gradient step (fewer registers, more waves per SIMD)
#pragma unroll
        for (int i = 0; i < D; ++i)
#pragma unroll
          for (int j = 0; j < D; ++j) st[i * D + j] = inv[i][j];
        st[N * D] = f;
        asm volatile("" ::: "memory");
        int go = g1;
        asm volatile("" : "+v"(go));
        R iv[D][D];
#pragma unroll
        for (int i = 0; i < D; ++i)
#pragma unroll
          for (int j = 0; j < D; ++j) iv[i][j] = st[i * D + j];
        stage_gradients<R, ET, NGP>(go, iv, st);
      }
      __syncthreads();
      rows_column_starts<KW>(lane, kw, MK, CS);  // blocks are stored column by column, lanes in order
      const unsigned dm = (unsigned)__ballot(dmv != 0);
      R K[P * P];
      {  // 2. block (a, b) of each incident element's tangent (lanes past the batch's elements form one that
         // is not stored, from whatever their slots hold)
        const int a = a2, b = b2, sb = 64 / N > EB ? min(s2, EB - 1) : s2;
        R M[D][D];
#pragma unroll
        for (int p = 0; p < D; ++p)
#pragma unroll
          for (int q = 0; q < D; ++q) M[p][q] = R(-0.0);
        R t = R(-0.0);
#pragma unroll UNR
        for (int g = 0; g < G; ++g) {
          const R *st = S + (sb * G + g) * ST;
          const R f = st[N * D];
          R fa[D], db[D];
#pragma unroll
          for (int j = 0; j < D; ++j) {
            fa[j] = f * st[a * D + j];
            db[j] = st[b * D + j];
          }
          if constexpr (PH == THERMAL) {
#pragma unroll
            for (int j = 0; j < D; ++j) t += fa[j] * db[j];
          } else {
#pragma unroll
            for (int p = 0; p < D; ++p)
#pragma unroll
              for (int q = 0; q < D; ++q) M[p][q] += fa[p] * db[q];
          }
        }
        if constexpr (PH == THERMAL) {
          K[0] = t;
        } else {
          const R c2 = R(D == 3 ? A.pp.c2 : A.pp.f2), c3 = R(D == 3 ? A.pp.c3 : A.pp.f2nu),
                  c4 = R(D == 3 ? A.pp.c4 : A.pp.f2sh);
#pragma unroll
          for (int c = 0; c < D; ++c)
#pragma unroll
            for (int d = 0; d < D; ++d) {
              if (c == d) {
                R o = M[(c + 1) % D][(c + 1) % D];
                if constexpr (D == 3) o += M[(c + 2) % D][(c + 2) % D];
                K[c * P + d] = c2 * M[c][c] + c4 * o;
              } else {
                K[c * P + d] = c3 * M[c][d] + c4 * M[d][c];
              }
            }
        }
        // a Dirichlet row keeps only the element diagonal (fe_loss.py:191-207); dm is the same for
        // the whole workgroup, so free nodes skip this
        if (dm) {
          asm volatile("" ::: "memory");  // keeps this a branch: the selects would run for every node
#pragma unroll
          for (int c = 0; c < P; ++c)
#pragma unroll
            for (int d = 0; d < P; ++d)
              if ((dm >> c & 1) && !(b == a && d == c)) K[c * P + d] = R(0);
        }
      }
      __syncthreads();  // every lane has read the staged geometry: the space takes the blocks
      if (col >= k0 && col < k0 + kw) {
        const int k = col - k0;
        const int dst = CS[k] + __popcll(MK[k] & ((1ull << lane) - 1ull));
#pragma unroll
        for (int i = 0; i < P * P; ++i) S[dst * P * P + i] = K[i];
      }
      __syncthreads();
      rows_add_columns<R, P, CPW, OR>(kw, oc, kk, od, S, CS, acc);  // 3. each output sums its column's blocks
      __syncthreads();  // before the next batch overwrites the blocks and the masks
    }
    if (want_r) (P == 1 ? res[0] : share) += rows_apply<R, P, CPW, OR>(kw, oc, kk, od, DU, acc);
    __syncthreads();  // before the next window's DU
    rows_write<R, P, CPW, OR>(kw, k0, deg, oc, kk, od, accumulate, acc, V);
  }
  if (want_r)  // (one dof per node: every lane's share and body force in one sum over the wave)
    rows_write_residual<R, P, CPW * P, P != 1>(share, res, P == 1 || A.pp.has_body, (unsigned)__ballot(dmv != 0), accumulate, S,
                                             reinterpret_cast<R *>(A.R) + node * P);
}

}  // namespace femhot
