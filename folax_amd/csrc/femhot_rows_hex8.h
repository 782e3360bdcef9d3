// Row-owner tangent assembly for HEX8 at the 2x2x2 rule (see femhot_rows.h for the assembly itself: one
// 64-lane workgroup per node, its incident elements' blocks summed per column in a fixed order).
//
// The 8 lanes of an element are its 8 nodes and its 8 Gauss points at once: with the Gauss coordinates
// +-s, s = 1/sqrt(3), the trilinear shape functions are products of 2 x 2 matrices, one per reference
// direction, so every map between nodal and Gauss-point values is three butterflies between the lanes
// whose node (point) lies across that direction:
//   B: v + g p   (interpolation; g = (1 - s) / (1 + s), times 1 + s)
//   D: the difference quotient across the direction (s v - s p from nodes to points, s (v + p) back)
// with v the lane's own value and p its partner's.  J, the field, the temperature and the displacement
// gradient come from the nodes by them, and the blocks sum_g f dN_a (x) dN_b of all 8 nodes b go back
// by the transposed ones.  Nothing is staged in LDS (the general kernel stages 25 values per Gauss
// point and reads 56 back per lane, which kept its LDS busy for half its time and allowed 3 waves
// per SIMD), and each of the blocks' 9 entries costs 29 instructions.  A lane's partners are lane ^ 1, ^ 3
// and ^ 7, one DPP move per 32 bits: lanes 4..7 hold the upper nodes in the order 7, 6, 5, 4.
//
// Bound: vector issue (5 waves per SIMD, 722 instructions a node: 198 M of them are 357 us at the clock it
// runs at) and, close behind, the memory round trips of a wave: kernel arguments, incidence list, connectivity,
// coordinates.  HEX8 64^3 FP64, tangent and residual of the linear-elastic box with its boundary
// conditions: 669 us through the general kernel (its tangent 565), 495 with the butterflies and the residual
// through the chunk kernel, 447 with the residual formed here, 405 with lane moves that keep no old
// value, 392 with the signs, the determinant and c4 taken out of the butterflies, the residual summed in the
// output lanes and the list of blocks found while the coordinates arrive.  A loop over nodes in a wave with the next
// node's connectivity fetched ahead was slower (484: its registers leave 3 waves per SIMD).  The values are
// stored after the residual's shares are formed (389).
// The residual is 35 us of the 389.
#pragma once
#include "femhot_rows.h"

namespace femhot {

template <int DIR, class T> __device__ __forceinline__ T hex8_across(T v) {
  return lane_dpp<DIR == 0 ? 0xB1 : DIR == 1 ? 0x1B : 0x141>(v);  // quad_perm [1,0,3,2], [3,2,1,0], row_half_mirror
}

constexpr double HEX8_S = 0.57735026918962576451;  // 1/sqrt(3)
constexpr double HEX8_G = (1.0 - HEX8_S) / (1.0 + HEX8_S);

// Node values -> their derivatives along the reference directions at the lane's point, over (1 + s)^2 / 8,
// each times the lane's sign along its direction: the Jacobian J' of these has (J')^-1 = diag(signs) J^-1,
// whose rows carry the signs that the way back (hex8_node_sum) needs, so none is ever multiplied in.
template <class R> __device__ __forceinline__ void hex8_point_gradient(R v, R (&o)[3]) {
  const R g = R(HEX8_G);
  const R px = hex8_across<0>(v), u = v - px, w = v + g * px;
  const R yu = u + g * hex8_across<1>(u), pw = hex8_across<1>(w), dw = w - pw, bw = w + g * pw;
  o[0] = yu + g * hex8_across<2>(yu);
  o[1] = dw + g * hex8_across<2>(dw);
  o[2] = bw - hex8_across<2>(bw);
}
// Node values -> the value at the lane's point, over (1 + s)^3 / 8.
template <class R> __device__ __forceinline__ R hex8_point_value(R v) {
  const R g = R(HEX8_G);
  v += g * hex8_across<0>(v);
  v += g * hex8_across<1>(v);
  return v + g * hex8_across<2>(v);
}
// sum over the points of sum_k q_k dN_b/dxi_k for the lane's node b, over (1 + s)^2 / 8; q_k carries the
// lane's sign along k.
template <class R> __device__ __forceinline__ R hex8_node_sum(R q0, R q1, R q2) {
  const R g = R(HEX8_G);
  const R u0 = q0 - hex8_across<0>(q0), u1 = q1 + g * hex8_across<0>(q1), u2 = q2 + g * hex8_across<0>(q2);
  const R w0 = (u0 + g * hex8_across<1>(u0)) + (u1 - hex8_across<1>(u1)), w2 = u2 + g * hex8_across<1>(u2);
  return (w0 + g * hex8_across<2>(w0)) + (w2 - hex8_across<2>(w2));
}

// Waves per SIMD the compiler must fit, by measurement at 64^3 (us with the residual): thermal FP64 272 at 4 waves (2
// spilled registers), 315 at 3 (none), 433 at 5 (the general power of k(T) spills more); thermal FP32 141 at 8, 149 at 7;
// linear elastic FP64 5 (4: 450, 6: 700), FP32 4 or more alike (270); Neo-Hookean FP64 1211 at 2 (7 spilled), 1650 at 1,
// FP32 4 or 5 alike (585).
template <class R, int PH> constexpr int rows_hex8_waves() {
  if (sizeof(R) == 4) return PH == THERMAL ? 8 : 4;
  return PH == NEOHOOKE ? 2 : PH == THERMAL ? 4 : 5;
}

template <class R, int PH>
__global__ __launch_bounds__(64, (rows_hex8_waves<R, PH>())) void k_tangent_rows_hex8(TArgs A) {
  constexpr int N = 8, D = 3, P = PH == THERMAL ? 1 : 3;
  using SH = RowsShape<HEX8, 2, N, P>;
  constexpr int EB = 8, KW = SH::KW, OR = SH::OR, CPW = SH::CPW;
  __shared__ __align__(16) R S[(64 + 4) * P * P];  // the lanes' blocks, column by column (4 of padding)
  __shared__ unsigned long long MK[KW];
  __shared__ int CS[KW + 1];
  __shared__ R DU[PH == NEOHOOKE ? 1 : KW * P];  // u_b - u_i of the window's columns
  const int lane = threadIdx.x;
  const bool elemental = (A.flags & FEMHOT_ELEMENT_FIELD) != 0;
  const bool accumulate = (A.flags & FEMHOT_ACCUMULATE) != 0;
  const R *F = reinterpret_cast<const R *>(A.field);
  const R *U = reinterpret_cast<const R *>(A.u);
  const int s = lane / 8, j = lane % 8, b = j < 4 ? j : 11 - j;  // the lane's node and Gauss point
  const int ix = ((b & 3) == 1 || (b & 3) == 2) ? 1 : 0, iy = (b & 3) >= 2 ? 1 : 0, iz = b >= 4 ? 1 : 0;
  const R sgn = ((ix + iy + iz) & 1) ? R(1) : R(-1);  // the product of the lane's signs
  const int oc = lane / (CPW * P), kk = (lane - oc * CPW * P) / P, od = lane - oc * CPW * P - kk * P;
  const R g = R(HEX8_G);
  const long long per = gridDim.x / 8, rem = gridDim.x % 8;  // XCD x takes the x-th eighth of the nodes
  const long long xcd = blockIdx.x % 8, qn = blockIdx.x / 8;
  const long long node = xcd * per + (xcd < rem ? xcd : rem) + qn;
  const int off0 = A.ne_off[node], cnt = A.ne_off[node + 1] - off0;
  const long long rp = A.row_ptr[node * P];
  const int deg = (int)((A.row_ptr[node * P + 1] - rp) / P);
  const int dmv = lane < P ? A.dmask[node * P + lane] : 0;  // (a bit mask where it is needed)
  R *V = reinterpret_cast<R *>(A.vals) + rp;
  // The residual beside the tangent: sum K_ab (u_b - u_i) for the linear physics (see femhot_rows.h), the
  // stress times dN_a at the lane's point for Neo-Hookean, less the body force N_a b at that point.
  const bool want_r = A.R != nullptr;
  R res[P], ui[P], share = R(0);
#pragma unroll
  for (int c = 0; c < P; ++c) res[c] = ui[c] = R(0);
  if (PH != NEOHOOKE && want_r) {
#pragma unroll
    for (int c = 0; c < P; ++c) ui[c] = U[node * P + c];
  }
  for (int k0 = 0; k0 < deg; k0 += KW) {
    const bool first = want_r && k0 == 0;
    const int kw = min(KW, deg - k0);
    R acc[OR];
#pragma unroll
    for (int r = 0; r < OR; ++r) acc[r] = R(0);
    for (int base = 0; base < cnt; base += EB) {
      const int nb = min(EB, cnt - base);
      int a = 0, col = -1;
      double xc[D] = {0.0, 0.0, 0.0};
      R fd = R(0), ud[P];
#pragma unroll
      for (int c = 0; c < P; ++c) ud[c] = R(0);
      if (s < nb) {
        const unsigned ea = A.ne_list[off0 + base + s];  // element * 8 + local node
        a = ea % N;
        col = A.slot[(size_t)ea * N + b];
        const unsigned nd = A.conn[(size_t)(ea - a) + b], nd3 = 3 * nd;  // (at most 2^26 nodes)
#pragma unroll
        for (int i = 0; i < D; ++i) xc[i] = A.coords[nd3 + i];
        fd = F[elemental ? ea / N : nd];
        if (PH != MECH || want_r) {
#pragma unroll
          for (int c = 0; c < P; ++c) ud[c] = U[nd * P + c];
        }
      }
      for (int t = lane; t < kw; t += 64) MK[t] = 0ull;
      __syncthreads();
      // the lane's place among its column's blocks, found while the coordinates are on their way
      const bool in = col >= k0 && col < k0 + kw;
      int dst = 0;
      if (in) atomicOr(&MK[col - k0], 1ull << lane);
      __syncthreads();
      rows_column_starts<KW>(lane, kw, MK, CS);
      __syncthreads();
      if (in) dst = CS[col - k0] + __popcll(MK[col - k0] & ((1ull << lane) - 1ull));
      // J' = 8 J / (1 + s)^2 and its inverse
      R J[D][D];
#pragma unroll
      for (int i = 0; i < D; ++i) {
        double ref = lane_dpp<0x150, 0x3>(xc[i]);  // node 0 of the element
        ref = rows_dpp_into<0x158, 0xc>(ref, xc[i]);
        hex8_point_gradient<R>(R(xc[i] - ref), J[i]);
      }
      const R c00 = J[1][1] * J[2][2] - J[1][2] * J[2][1];
      const R c01 = J[1][2] * J[2][0] - J[1][0] * J[2][2];
      const R c02 = J[1][0] * J[2][1] - J[1][1] * J[2][0];
      const R det = J[0][0] * c00 + J[0][1] * c01 + J[0][2] * c02;
      const R id = recip(det);
      R iv[D][D];  // the cofactors: det J' times its inverse
      iv[0][0] = c00;
      iv[1][0] = c01;
      iv[2][0] = c02;
      iv[0][1] = J[0][2] * J[2][1] - J[0][1] * J[2][2];
      iv[1][1] = J[0][0] * J[2][2] - J[0][2] * J[2][0];
      iv[2][1] = J[0][1] * J[2][0] - J[0][0] * J[2][1];
      iv[0][2] = J[0][1] * J[1][2] - J[0][2] * J[1][1];
      iv[1][2] = J[0][2] * J[1][0] - J[0][0] * J[1][2];
      iv[2][2] = J[0][0] * J[1][1] - J[0][1] * J[1][0];
      if (PH != NEOHOOKE && want_r && in) {
#pragma unroll
        for (int c = 0; c < P; ++c) DU[(col - k0) * P + c] = ud[c] - ui[c];
      }
      constexpr double a1 = 1.0 + HEX8_S, a3 = a1 * a1 * a1 / 8.0;
      constexpr double aw = a3 * a3 / 8.0;  // det J = ((1 + s)^2 / 8)^3 det J' over the signs
      const R fe = elemental ? fd : R(a3) * hex8_point_value<R>(fd);
      // dN_a/dx of the owned node a times det J' (the factors of J' and of the shape gradients cancel)
      const int ax = ((a & 3) == 1 || (a & 3) == 2) ? 1 : 0, ay = (a & 3) >= 2 ? 1 : 0, az = a >= 4 ? 1 : 0;
      const R rx = ax == ix ? R(1) : g, ry = ay == iy ? R(1) : g, rz = az == iz ? R(1) : g;
      if (first && A.pp.has_body && s < nb) {
        const R na = (R(a3 * aw) * sgn) * det * (rx * (ry * rz));
#pragma unroll
        for (int c = 0; c < P; ++c) res[c] -= na * R(A.pp.body[c]);
      }
      const R sh[3] = {ax == ix ? ry * rz : -(ry * rz), ay == iy ? rx * rz : -(rx * rz),
                       az == iz ? rx * ry : -(rx * ry)};
      R dNa[D];
#pragma unroll
      for (int q = 0; q < D; ++q) dNa[q] = (sh[0] * iv[0][q] + sh[1] * iv[1][q]) + sh[2] * iv[2][q];
      R f = (R(aw) * sgn) * (fe * id);  // w det J times the field, over (det J')^2 of the two gradients
      R K[P * P];
      if constexpr (PH == THERMAL) {
        f *= R(1) + R(A.pp.beta) * powc(R(a3) * hex8_point_value<R>(ud[0]), R(A.pp.c));
        R q[D];
#pragma unroll
        for (int k = 0; k < D; ++k) q[k] = f * ((dNa[0] * iv[k][0] + dNa[1] * iv[k][1]) + dNa[2] * iv[k][2]);
        K[0] = hex8_node_sum<R>(q[0], q[1], q[2]);
      } else if constexpr (PH == MECH) {
        R fa[D], M[D][D];  // c4 times the moments
        f *= R(A.pp.c4);
#pragma unroll
        for (int i = 0; i < D; ++i) fa[i] = f * dNa[i];
#pragma unroll
        for (int q = 0; q < D; ++q) {
#pragma unroll
          for (int p = 0; p < D; ++p)
            M[p][q] = hex8_node_sum<R>(fa[p] * iv[0][q], fa[p] * iv[1][q], fa[p] * iv[2][q]);
        }
        const R r2 = R(A.r2), r3 = R(A.r3), tr = M[0][0] + M[1][1] + M[2][2];
#pragma unroll
        for (int c = 0; c < D; ++c)
#pragma unroll
          for (int d = 0; d < D; ++d) K[c * P + d] = c == d ? r2 * M[c][c] + tr : r3 * M[c][d] + M[d][c];
      } else {
        f *= det * det;
#pragma unroll
        for (int i = 0; i < D; ++i) {
          dNa[i] *= id;
#pragma unroll
          for (int q = 0; q < D; ++q) iv[i][q] *= id;
        }
        R H[D][D];
#pragma unroll
        for (int i = 0; i < D; ++i) {
          R h[D];
          hex8_point_gradient<R>(ud[i], h);
#pragma unroll
          for (int q = 0; q < D; ++q) H[i][q] = (h[0] * iv[0][q] + h[1] * iv[1][q]) + h[2] * iv[2][q];
        }
        NHState<R, D> st;
        nh_state<R, D>(H, R(A.pp.kap1), R(A.pp.mu1), st);
        R Sa[D];  // S dN_a
#pragma unroll
        for (int i = 0; i < D; ++i) Sa[i] = (st.S[i][0] * dNa[0] + st.S[i][1] * dNa[1]) + st.S[i][2] * dNa[2];
        if (first && s < nb) {
#pragma unroll
          for (int c = 0; c < D; ++c)
            res[c] += f * ((st.F[c][0] * Sa[0] + st.F[c][1] * Sa[1]) + st.F[c][2] * Sa[2]);
        }
#pragma unroll
        for (int c = 0; c < D; ++c) {  // the stress change of a unit displacement (a, c): F dS + dF S
          R X[D][D], dS[D][D];
#pragma unroll
          for (int p = 0; p < D; ++p)
#pragma unroll
            for (int q = 0; q < D; ++q) X[p][q] = R(0.5) * (st.F[c][p] * dNa[q] + st.F[c][q] * dNa[p]);
          nh_tangent_apply<R, D>(st, R(A.pp.kap1), R(A.pp.mu1), X, dS);
#pragma unroll
          for (int d = 0; d < D; ++d) {
            R w[D], q[D];
#pragma unroll
            for (int i = 0; i < D; ++i) {
              const R m = (st.F[d][0] * dS[0][i] + st.F[d][1] * dS[1][i]) + st.F[d][2] * dS[2][i];
              w[i] = f * (c == d ? m + Sa[i] : m);
            }
#pragma unroll
            for (int k = 0; k < D; ++k) q[k] = (w[0] * iv[k][0] + w[1] * iv[k][1]) + w[2] * iv[k][2];
            K[c * P + d] = hex8_node_sum<R>(q[0], q[1], q[2]);
          }
        }
      }
      const unsigned dm = (unsigned)__ballot(dmv != 0);
      if (dm) {  // a Dirichlet row keeps only the element diagonal (fe_loss.py:191-207)
        asm volatile("" ::: "memory");  // keeps this a branch: the selects would run for every node
#pragma unroll
        for (int c = 0; c < P; ++c)
#pragma unroll
          for (int d = 0; d < P; ++d)
            if ((dm >> c & 1) && !(b == a && d == c)) K[c * P + d] = R(0);
      }
      if (in) {
#pragma unroll
        for (int i = 0; i < P * P; ++i) S[dst * P * P + i] = K[i];
      }
      __syncthreads();
      rows_add_columns<R, P, CPW, OR>(kw, oc, kk, od, S, CS, acc);
      __syncthreads();  // before the next batch overwrites the blocks and the masks
    }
    if constexpr (PH != NEOHOOKE) {
      if (want_r) share += rows_apply<R, P, CPW, OR>(kw, oc, kk, od, DU, acc);
      __syncthreads();  // before the next window's DU
    }
    rows_write<R, P, CPW, OR>(kw, k0, deg, oc, kk, od, accumulate, acc, V);
  }
  if (want_r)
    rows_write_residual<R, P, CPW * P, PH != NEOHOOKE>(share, res, PH == NEOHOOKE || A.pp.has_body,
                                                       (unsigned)__ballot(dmv != 0), accumulate, S,
                                                       reinterpret_cast<R *>(A.R) + node * P);
}

}  // namespace femhot
