// Jacobi-preconditioned conjugate gradients on the assembled CSR tangent.
//
// Reference: fol/solvers/fe_solver.py:60-78 (LinearSolve: BiCGSTAB / direct solve of K du = -R)
// and fe_linear_residual_based_solver.py:15-22.  The reference has no CG; with the reference's
// BC treatment (Dirichlet rows zeroed except the diagonal, R_D = 0) the Dirichlet unknowns stay
// zero and the iteration runs on the SPD free block, so CG applies to the matrix as assembled.
//
// Design: an iteration is three stream-ordered kernels with no host round trip; the host reads the
// residual norm only every `check` iterations.  Dot products are reduced without atomics: every
// reducing kernel runs a fixed grid of NBR workgroups (grid-stride loops) and writes one FP64
// partial per workgroup; the kernel that needs the scalar sums the NBR partials itself, in a fixed
// order, in its prologue.  (One device-scope atomic per wave onto a single address serialises: on
// an 823,875-row system that alone cost ~10 ms per iteration.)  Results are bitwise reproducible.
// FP32 mode keeps the matrix and vectors in FP32, accumulates every dot product in FP64, and wraps
// the FP32 solves in FP64 iterative refinement r = b - A x with the FP64 matrix.
#include <cmath>

#include "femhot_pcg_tile.h"

namespace femhot {

constexpr int NBR = 1024;  // workgroups of every reducing kernel (one FP64 partial each)

// Sum over the workgroup; the result is returned to every thread (blockDim.x == 256).
__device__ __forceinline__ double block_sum256(double v) {
  __shared__ double red[4];
  v = wave_sum(v);
  __syncthreads();  // red may still be read by a previous call
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  return (red[0] + red[1]) + (red[2] + red[3]);
}

// Sum of the NBR partials, in a fixed order, returned to every thread.
__device__ __forceinline__ double sum_partials(const double *part) {
  double v = 0.0;
#pragma unroll
  for (int k = 0; k < NBR / 256; ++k) v += part[k * 256 + threadIdx.x];
  return block_sum256(v);
}

// Both SpMV kernels take `rev`: the workgroups then walk the tiles from the last to the first.  Consecutive
// iterations alternate, so a sweep starts on the part of the matrix that the sweep before left in the
// 256 MB memory-side cache, where a forward sweep each time finds its beginning gone.  An iteration, always forward
// -> alternating: HEX8 64^3, 518 MB of FP64 values, 158.7 -> 147.1 us, 259 MB of FP32 values 97.9 -> 87.6; 52^3 FP64,
// 281 MB, 88.4 -> 79.0; 40^3, 127 MB, 42.0 both ways.  A matrix that the L2 caches hold together is always walked forward:
// turned round, a tile comes to another XCD, whose L2 has not seen it (any-pattern solve, HEX8 20^3 elastic, 24 MB
// with its columns, 20.1 -> 21.1; thermal 40^3, 22 MB, 21.1 -> 22.2; 42 MB 25.0 both ways).  Partials are stored by tile, so
// the sums, and the iterates, are the same.
//
// y = A x, LPR lanes per row, one pass (grid = rows * LPR / 256).  Each lane first loads up to U = 8
// of its row's (column, value) pairs, then gathers x for all of them, so a row costs three dependent
// memory round trips whatever its length up to 8 * LPR (longer rows continue in a loop).  When part
// is set, part[block] = this workgroup's share of x.y (FP64).
template <class T, int LPR>
__global__ __launch_bounds__(256) void k_spmv(long long nrows, const long long *__restrict__ rp,
                                              const int *__restrict__ ci, const T *__restrict__ v,
                                              const T *__restrict__ x, T *__restrict__ y, double *part,
                                              const int *stop, int rev) {
  if (stop && *stop) return;  // a device-side solve that has stopped (uniform over the grid)
  constexpr int U = 8;
  const unsigned tile = rev ? gridDim.x - 1 - blockIdx.x : blockIdx.x;
  const long long row = ((long long)tile * 256 + threadIdx.x) / LPR;
  const int lane = (int)(threadIdx.x % LPR);
  double d = 0.0;
  if (row < nrows) {
    const long long b = rp[row], e = rp[row + 1];
    int cols[U];
    T vals[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const long long k = b + lane + (long long)u * LPR;
      const bool in = k < e;
      cols[u] = in ? ci[k] : (int)row;
      vals[u] = in ? v[k] : T(0);
    }
    // accumulated in the arithmetic type (FP32 only in the mixed solve's inner iterations)
    T s = T(0);
#pragma unroll
    for (int u = 0; u < U; ++u) s += vals[u] * x[cols[u]];
    for (long long k = b + lane + (long long)U * LPR; k < e; k += LPR) s += v[k] * x[ci[k]];
#pragma unroll
    for (int off = LPR / 2; off >= 1; off >>= 1) s += __shfl_xor(s, off, LPR);
    if (lane == 0) {
      y[row] = s;
      d = (double)x[row] * (double)s;
    }
  }
  if (part) {
    const double t = block_sum256(d);
    if (threadIdx.x == 0) part[tile] = t;
  }
}

// y = A x on a node-blocked pattern: P dofs per node, and every dof row of node i lists the same
// neighbours m, each as the P consecutive columns P*m .. P*m+P-1 (the pattern ensure_pattern builds).
// LPN lanes per node; a lane takes every LPN-th neighbour and reads its column index once for the
// whole P x P block (the other P*P-1 indices of the block are implied), then the P x values of the
// neighbour as one contiguous block.  Index traffic drops from 4 to 4/(P*P) bytes per nonzero.
// When part is set, part[block] = this workgroup's share of x.y (FP64).
template <class T, int P, int LPN>
__global__ __launch_bounds__(256) void k_spmv_node(long long nnodes, const long long *__restrict__ rp,
                                                   const int *__restrict__ ci, const T *__restrict__ v,
                                                   const T *__restrict__ x, T *__restrict__ y, double *part,
                                                   const int *stop, int rev) {
  if (stop && *stop) return;
  constexpr int U = 4;
  const unsigned tile = rev ? gridDim.x - 1 - blockIdx.x : blockIdx.x;
  const long long node = ((long long)tile * 256 + threadIdx.x) / LPN;
  const int lane = (int)(threadIdx.x % LPN);
  double d = 0.0;
  if (node < nnodes) {
    long long rb[P];
#pragma unroll
    for (int c = 0; c < P; ++c) rb[c] = rp[node * P + c];
    const int deg = (int)((rp[node * P + 1] - rb[0]) / P);
    // accumulated in the arithmetic type: FP32 for the inner iterations of the mixed solve (whose
    // FP64 outer refinement recomputes the residual), FP64 otherwise
    T s[P];
#pragma unroll
    for (int c = 0; c < P; ++c) s[c] = T(0);
    // slots past the node's last neighbour re-read that neighbour (deg >= 1 inside the loop) and skip
    // the add: unconditional loads let each row's P consecutive values merge into one wide load
    for (int k0 = lane; k0 < deg; k0 += U * LPN) {
      int col[U];
      T vv[U][P][P];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const long long k = min(k0 + u * LPN, deg - 1);
        col[u] = ci[rb[0] + P * k];
#pragma unroll
        for (int c = 0; c < P; ++c)
#pragma unroll
          for (int e = 0; e < P; ++e) vv[u][c][e] = v[rb[c] + P * k + e];
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        T xv[P];
#pragma unroll
        for (int e = 0; e < P; ++e) xv[e] = x[col[u] + e];
        if (k0 + u * LPN < deg) {
#pragma unroll
          for (int c = 0; c < P; ++c)
#pragma unroll
            for (int e = 0; e < P; ++e) s[c] += vv[u][c][e] * xv[e];
        }
      }
    }
#pragma unroll
    for (int c = 0; c < P; ++c)
#pragma unroll
      for (int off = LPN / 2; off >= 1; off >>= 1) s[c] += __shfl_xor(s[c], off, LPN);
    if (lane == 0) {
#pragma unroll
      for (int c = 0; c < P; ++c) {
        y[node * P + c] = s[c];
        d += (double)x[node * P + c] * (double)s[c];
      }
    }
  }
  if (part) {
    const double t = block_sum256(d);
    if (threadIdx.x == 0) part[tile] = t;
  }
}

// out[0] = sum of part[0 .. n) in a fixed order (one workgroup of 1024; four independent
// accumulators per thread keep four loads in flight).
__global__ __launch_bounds__(1024) void k_sum_parts(const double *part, long long n, double *out,
                                                    const int *stop) {
  if (stop && *stop) return;
  __shared__ double red[16];
  double a0 = 0.0, a1 = 0.0, a2 = 0.0, a3 = 0.0;
  long long i = threadIdx.x;
  for (; i + 3 * 1024 < n; i += 4 * 1024) {
    a0 += part[i];
    a1 += part[i + 1024];
    a2 += part[i + 2 * 1024];
    a3 += part[i + 3 * 1024];
  }
  for (; i < n; i += 1024) a0 += part[i];
  double v = wave_sum((a0 + a1) + (a2 + a3));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int k = 0; k < 16; ++k) t += red[k];
    out[0] = t;
  }
}

template <class T>
__global__ void k_diag_inv(long long nrows, const long long *rp, const int *ci, const double *v, T *dinv) {
  const long long r = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= nrows) return;
  long long lo = rp[r], hi = rp[r + 1];
  double dv = 0.0;
  while (lo < hi) {
    const long long mid = (lo + hi) >> 1;
    if (ci[mid] < r)
      lo = mid + 1;
    else
      hi = mid;
  }
  if (lo < rp[r + 1] && ci[lo] == r) dv = v[lo];
  dinv[r] = (T)(dv != 0.0 ? 1.0 / dv : 1.0);
}

// The same on the context's own pattern, whose diagonal offsets are known: one value per row is read
// instead of a binary search over the row's column indices.
template <class T>
__global__ void k_diag_inv_pos(long long nrows, const long long *rp, const int *doff, const double *v, T *dinv) {
  const long long r = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= nrows) return;
  const double dv = doff[r] >= 0 ? v[rp[r] + doff[r]] : 0.0;
  dinv[r] = (T)(dv != 0.0 ? 1.0 / dv : 1.0);
}

template <class T> __global__ void k_cast(long long n, const double *a, T *b) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const long long st = (long long)gridDim.x * blockDim.x;
  for (long long k = i; k < n; k += st) b[k] = (T)a[k];
}

// r = b - r (r holds A x on entry); p = Dinv r; partials of r.Dinv r and r.r
template <class T>
__global__ __launch_bounds__(256) void k_init(long long n, const double *b, T *r, T *p, const T *dinv, double *rz_part,
                                              double *rr_part) {
  double rz = 0.0, rr = 0.0;
  for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long long)gridDim.x * 256) {
    const double ri = b[i] - (double)r[i];
    const T rt = (T)ri;
    r[i] = rt;
    const T z = rt * dinv[i];
    p[i] = z;
    rz += (double)rt * (double)z;
    rr += (double)rt * (double)rt;
  }
  rz = block_sum256(rz);
  rr = block_sum256(rr);
  if (threadIdx.x == 0) rz_part[blockIdx.x] = rz, rr_part[blockIdx.x] = rr;
}

// alpha = (r.z) / (p.Ap); x += alpha p; r -= alpha q; partials of the new r.z and r.r.  The
// thread's first element is loaded before the partial sums, so its loads overlap their latency.
template <class T>
__global__ __launch_bounds__(256) void k_update_xr(long long n, T *x, T *r, const T *p, const T *q, const T *dinv,
                                                   const double *rz_part, const double *pap, double *rz_next,
                                                   double *rr_next, const int *stop) {
  if (stop && *stop) return;
  const long long i0 = (long long)blockIdx.x * 256 + threadIdx.x, st = (long long)gridDim.x * 256;
  const long long j0 = i0 < n ? i0 : 0;  // n >= 1: index 0 is in bounds
  const T x0 = x[j0], p0 = p[j0], r0 = r[j0], q0 = q[j0], d0 = dinv[j0];
  const double alpha = sum_partials(rz_part) / pap[0];
  double rz = 0.0, rr = 0.0;
  auto step = [&](long long i, T xi, T pi, T rv, T qi, T di) {
    x[i] = (T)((double)xi + alpha * (double)pi);
    const T ri = (T)((double)rv - alpha * (double)qi);
    r[i] = ri;
    const T z = ri * di;
    rz += (double)ri * (double)z;
    rr += (double)ri * (double)ri;
  };
  if (i0 < n) step(i0, x0, p0, r0, q0, d0);
  for (long long i = i0 + st; i < n; i += st) step(i, x[i], p[i], r[i], q[i], dinv[i]);
  rz = block_sum256(rz);
  rr = block_sum256(rr);
  if (threadIdx.x == 0) rz_next[blockIdx.x] = rz, rr_next[blockIdx.x] = rr;
}

// beta = (r.z)_new / (r.z)_old; p = Dinv r + beta p (first element loaded before the partial sums)
template <class T>
__global__ __launch_bounds__(256) void k_update_p(long long n, T *p, const T *r, const T *dinv, const double *rz_new,
                                                  const double *rz_old, const int *stop) {
  if (stop && *stop) return;
  const long long i0 = (long long)blockIdx.x * 256 + threadIdx.x, st = (long long)gridDim.x * 256;
  const long long j0 = i0 < n ? i0 : 0;  // n >= 1: index 0 is in bounds
  const T r0 = r[j0], d0 = dinv[j0], p0 = p[j0];
  const double beta = sum_partials(rz_new) / sum_partials(rz_old);
  if (i0 < n) p[i0] = (T)((double)(r0 * d0) + beta * (double)p0);
  for (long long i = i0 + st; i < n; i += st) p[i] = (T)((double)(r[i] * dinv[i]) + beta * (double)p[i]);
}

template <class T> __global__ void k_axpy_to64(long long n, const T *d, double *x) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) x[i] += (double)d[i];
}

// Lanes per row: the smallest power of two (4..64) whose eight loads per lane cover an average row.
static int lanes_per_row(long long nnz, long long n) {
  const double avg = n ? (double)nnz / (double)n : 1.0;
  int l = 4;
  while (l < 64 && 8.0 * l < avg) l *= 2;
  return l;
}

// How an SpMV is launched: row-wise CSR with `lanes` lanes per row, or node-blocked (P = 2 or 3 dofs
// per node) with `lanes` lanes per node.  blocks = workgroups of 256 = number of x.y partials.
struct SpmvPlan {
  int P = 1;  // 1: row-wise CSR kernel
  int lanes = 4;
  unsigned blocks = 1;
};

static SpmvPlan spmv_plan(long long n, long long nnz, int P, bool node_blocked) {
  SpmvPlan sp;
  if (node_blocked && (P == 2 || P == 3) && n % P == 0) {
    const long long nodes = n / P;
    const double deg = nodes ? (double)nnz / (double)(P * P * nodes) : 1.0;  // neighbours per node
    int l = 2;
    while (l < 16 && 4.0 * l < deg) l *= 2;
    sp.P = P;
    sp.lanes = l;
    sp.blocks = (unsigned)((nodes * l + 255) / 256);
  } else {
    sp.lanes = lanes_per_row(nnz, n);
    sp.blocks = (unsigned)((n * sp.lanes + 255) / 256);
  }
  return sp;
}

// Whether consecutive sweeps of a matrix of T alternate: values and columns beyond the 8 L2 caches of 4 MB.
template <class T> static bool spmv_alternates(long long nnz) { return nnz * (long long)(sizeof(T) + sizeof(int)) > (32LL << 20); }

template <class T, int P>
static void spmv_node_launch(long long nodes, const long long *rp, const int *ci, const T *v, const T *x, T *y,
                             double *part, const SpmvPlan &sp, hipStream_t s, const int *stop, int rev) {
  const dim3 grid(sp.blocks);
  switch (sp.lanes) {
    case 2: hipLaunchKernelGGL((k_spmv_node<T, P, 2>), grid, dim3(256), 0, s, nodes, rp, ci, v, x, y, part, stop, rev); break;
    case 4: hipLaunchKernelGGL((k_spmv_node<T, P, 4>), grid, dim3(256), 0, s, nodes, rp, ci, v, x, y, part, stop, rev); break;
    case 8: hipLaunchKernelGGL((k_spmv_node<T, P, 8>), grid, dim3(256), 0, s, nodes, rp, ci, v, x, y, part, stop, rev); break;
    default: hipLaunchKernelGGL((k_spmv_node<T, P, 16>), grid, dim3(256), 0, s, nodes, rp, ci, v, x, y, part, stop, rev); break;
  }
}

template <class T>
static void spmv_launch(long long n, const long long *rp, const int *ci, const T *v, const T *x, T *y, double *part,
                        const SpmvPlan &sp, hipStream_t s, const int *stop = nullptr, int rev = 0) {
  if (sp.P == 3) return spmv_node_launch<T, 3>(n / 3, rp, ci, v, x, y, part, sp, s, stop, rev);
  if (sp.P == 2) return spmv_node_launch<T, 2>(n / 2, rp, ci, v, x, y, part, sp, s, stop, rev);
  const dim3 grid(sp.blocks);
  switch (sp.lanes) {
    case 4: hipLaunchKernelGGL((k_spmv<T, 4>), grid, dim3(256), 0, s, n, rp, ci, v, x, y, part, stop, rev); break;
    case 8: hipLaunchKernelGGL((k_spmv<T, 8>), grid, dim3(256), 0, s, n, rp, ci, v, x, y, part, stop, rev); break;
    case 16: hipLaunchKernelGGL((k_spmv<T, 16>), grid, dim3(256), 0, s, n, rp, ci, v, x, y, part, stop, rev); break;
    case 32: hipLaunchKernelGGL((k_spmv<T, 32>), grid, dim3(256), 0, s, n, rp, ci, v, x, y, part, stop, rev); break;
    default: hipLaunchKernelGGL((k_spmv<T, 64>), grid, dim3(256), 0, s, n, rp, ci, v, x, y, part, stop, rev); break;
  }
}

// Host sum (fixed order) of NBR partials copied to pinned memory.
static int host_sum_partials(Ctx *c, const double *part, hipStream_t s, double *out) {
  FH_HIP(hipMemcpyAsync(c->h_pinned, part, NBR * sizeof(double), hipMemcpyDeviceToHost, s));
  FH_HIP(hipStreamSynchronize(s));
  double t = 0.0;
  for (int k = 0; k < NBR; ++k) t += c->h_pinned[k];
  *out = t;
  return FEMHOT_OK;
}

// Jacobi-PCG in type T on (rp, ci, v) for A x = b (b in FP64), x in T.  Partials in sc (3 x NBR
// doubles: r.z for two parities, r.r), pap_part (one per SpMV workgroup) and pap (the summed p.Ap).
// Returns iterations; *relres = ||r||/||b|| at exit (as tracked by the recurrence).
template <class T>
static int pcg_core(Ctx *c, long long n, const long long *rp, const int *ci, const T *v, const double *b, T *x,
                    T *r, T *p, T *q, T *dinv, double *sc, double *pap_part, double *pap, double bnorm, double tol,
                    int maxiter, int check, const SpmvPlan &sp, hipStream_t s, int *iters_out, double *relres,
                    bool *converged) {
  const dim3 grid(NBR);
  double *rz[2] = {sc, sc + NBR}, *rrp = sc + 2 * NBR;
  const unsigned nsp = sp.blocks;
  spmv_launch<T>(n, rp, ci, v, x, r, nullptr, sp, s);  // r = A x
  hipLaunchKernelGGL((k_init<T>), grid, dim3(256), 0, s, n, b, r, p, dinv, rz[0], rrp);
  double rr = 0.0;
  int rc = host_sum_partials(c, rrp, s, &rr);
  if (rc) return rc;
  *converged = false;
  *relres = bnorm > 0 ? std::sqrt(rr) / bnorm : 0.0;
  if (bnorm == 0.0 || *relres <= tol) {
    *converged = true;
    *iters_out = 0;
    return FEMHOT_OK;
  }
  int k = 0;
  const bool alt = spmv_alternates<T>(c->nnz);
  while (k < maxiter) {
    const int par = k & 1;
    spmv_launch<T>(n, rp, ci, v, p, q, pap_part, sp, s, nullptr, alt ? par : 0);
    hipLaunchKernelGGL(k_sum_parts, dim3(1), dim3(1024), 0, s, pap_part, (long long)nsp, pap, (const int *)nullptr);
    hipLaunchKernelGGL((k_update_xr<T>), grid, dim3(256), 0, s, n, x, r, p, q, dinv, rz[par], pap, rz[1 - par], rrp,
                       (const int *)nullptr);
    hipLaunchKernelGGL((k_update_p<T>), grid, dim3(256), 0, s, n, p, r, dinv, rz[1 - par], rz[par],
                       (const int *)nullptr);
    ++k;
    if (k % check == 0 || k == maxiter) {
      rc = host_sum_partials(c, rrp, s, &rr);
      if (rc) return rc;
      *relres = std::sqrt(std::max(rr, 0.0)) / bnorm;
      if (!(std::isfinite(rr))) {
        set_error("femhot_pcg: non-finite residual");
        *iters_out = k;
        return FEMHOT_ERR_NONFINITE;
      }
      if (*relres <= tol) {
        *converged = true;
        break;
      }
    }
  }
  FH_HIP(hipGetLastError());
  *iters_out = k;
  return FEMHOT_OK;
}

// How a system is cut for the tile kernels: G workgroups of 512 threads, `lpn` lanes per node, S nodes per
// group of lanes.  ok only on the context's pattern, for systems whose rows fit: at most 4 neighbour
// blocks per lane, the S x 4 blocks of a lane within the register file, one workgroup per CU, a
// workgroup's columns within TILE_RANGE ids and its vectors within LDS.
struct TilePlan {
  bool ok = false;
  int lpn = 4, S = 1, G = 0, cap = 0;
  size_t lds = 0;
};

static int device_cus() {
  static int cus = 0;
  if (!cus) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
      cus = 256;
  }
  return cus;
}

// Most nodes per lane group: S x 4 x P x P values of T within about 150 registers.
template <class T> constexpr int tile_max_s(int P) { return P == 1 ? 8 : P == 2 ? 4 : sizeof(T) == 4 ? 4 : 2; }

// Calls f(integral_constant P, LPN, S) for a plan (S within what tile_plan chooses for P and T).
template <class T, class F> static int tile_dispatch(int P, const TilePlan &tp, F &&f) {
  using std::integral_constant;
  auto with_s = [&](auto p, auto l) -> int {
    constexpr int MAXS = tile_max_s<T>(decltype(p)::value);
    if constexpr (MAXS >= 8)
      if (tp.S == 8) return f(p, l, integral_constant<int, 8>{});
    if constexpr (MAXS >= 4)
      if (tp.S == 4) return f(p, l, integral_constant<int, 4>{});
    if constexpr (MAXS >= 2)
      if (tp.S == 2) return f(p, l, integral_constant<int, 2>{});
    return f(p, l, integral_constant<int, 1>{});
  };
  auto with_l = [&](auto p) -> int {
    return tp.lpn == 4 ? with_s(p, integral_constant<int, 4>{}) : with_s(p, integral_constant<int, 8>{});
  };
  if (P == 1) return with_l(integral_constant<int, 1>{});
  if (P == 2) return with_l(integral_constant<int, 2>{});
  return with_l(integral_constant<int, 3>{});
}

template <class T> static TilePlan tile_plan(const Ctx *c) {
  TilePlan tp;
  if (c->max_deg < 1 || c->max_deg > 8 * TILE_U) return tp;
  tp.lpn = c->max_deg <= 4 * TILE_U ? 4 : 8;
  const int P = c->ndpn, npw = TILE_T / tp.lpn;
  const int max_s = tile_max_s<T>(P);
  const int most = std::min(device_cus(), 256);
  auto groups = [&](int s) { return (c->Nn + (long long)npw * s - 1) / ((long long)npw * s); };
  if (groups(max_s) > most) return tp;
  // One workgroup needs no exchange, and is taken while its passes stay few (quads 20 x 20 conduction in FP64:
  // 2.6 us an iteration with S = 4 in one workgroup, 4.0 in four with S = 1; 40 x 40: 5.5 with S = 8 in two,
  // 4.0 with S = 2 in seven).  Otherwise few workgroups, but not at the cost of passes where a node's block is
  // large: from S = 1 (3 dofs per node) or 2 up to the first S that leaves at most 128 workgroups (quads
  // 128 x 128: 7.4 us with 130, 6.1 with 65; tetrahedra 20^3 mixed: 6.1 with S = 1, 7.7 with S = 4), else up
  // to the first that fits the device.
  int s = P == 3 ? 1 : 2;
  if (groups(std::min(4, max_s)) == 1) {
    s = 1;
    while (groups(s) > 1) s *= 2;
  } else {
    if (P == 1)
      while (s < max_s && groups(s) > 128) s *= 2;
    while (groups(s) > most) s *= 2;
  }
  tp.S = s;
  tp.G = (int)groups(s);
  const long long range = std::min<long long>(c->Nn, (long long)npw * s + 2LL * c->bandwidth);
  if (range > TILE_RANGE) return tp;
  tp.cap = (int)std::min<long long>(range, (long long)TILE_T * TILE_U * s);
  tile_dispatch<T>(P, tp, [&](auto p, auto l, auto sc) {
    tp.lds = Tile<T, decltype(p)::value, decltype(l)::value, decltype(sc)::value>::lds(tp.cap);
    return 0;
  });
  static size_t lim = 0;
  if (!lim) {
    int dev = 0, v = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess || v <= 0)
      v = 64 * 1024;
    lim = (size_t)v - 2048;  // less the kernel's static LDS
  }
  tp.ok = tp.lds <= lim;
  return tp;
}

static size_t r256(size_t b) { return (b + 255) & ~size_t(255); }
template <class T> static size_t tile_ws_bytes(const Ctx *c, const TilePlan &tp) {
  return 3 * r256(sizeof(T) * c->Ndof) + r256(sizeof(double) * 8 * tp.G) + 2 * r256(sizeof(PcgState));
}

// Workspace of an FP64 solve on this context, host-checked or enqueued, on the context's pattern or any
// other: the most that any of their forms takes, so the first call of one kind sizes it for all of them and a
// later call of another kind neither allocates under a capture nor frees what a captured graph uses.  Each
// piece is 256-byte aligned.
static size_t pcg_ws_bytes(const Ctx *c) {
  const size_t vec64 = r256(sizeof(double) * c->Ndof), state = r256(sizeof(PcgState));
  size_t need = 0;
  for (const bool node_blocked : {false, true}) {  // launched: partials, 5 vectors, the state
    const size_t nsp = spmv_plan(c->Ndof, c->nnz, c->ndpn, node_blocked).blocks;
    need = std::max(need, r256(3 * NBR * sizeof(double)) + r256(NBR * sizeof(double)) + r256(nsp * sizeof(double)) +
                              r256(8 * sizeof(double)) + 5 * vec64 + state);
  }
  const TilePlan tp = tile_plan<double>(c);
  if (tp.ok)  // in one launch; one launch per phase: 6 vectors, partials, the state
    need = std::max({need, tile_ws_bytes<double>(c, tp), 6 * vec64 + r256(sizeof(double) * 8 * tp.G) + state});
  return need;
}

// One resident solve (k_pcg_resident), synchronised: *st the final state; *ran false when it could not be
// launched or a wait between its workgroups ran out (x is then the initial guess again).
template <class T>
static int tile_solve(Ctx *c, const TilePlan &tp, void *ws, const long long *rp, const int *ci, const double *vals,
                      const double *b, T *x, double bnorm, double tol, int maxiter, int check, hipStream_t s,
                      PcgState *st, bool *ran) {
  char *w = (char *)ws;
  auto take = [&](size_t bytes) {
    char *p = w;
    w += r256(bytes);
    return (void *)p;
  };
  TileArgs A{};
  A.nodes = c->Nn;
  A.rp = rp;
  A.ci = ci;
  A.vals = vals;
  A.doff = c->d_diag_off;
  A.b = b;
  A.x = x;
  A.z[0] = take(sizeof(T) * c->Ndof);
  A.z[1] = take(sizeof(T) * c->Ndof);
  A.x0 = take(sizeof(T) * c->Ndof);
  A.pa = (double *)take(sizeof(double) * 8 * tp.G);
  A.pc = A.pa + 6 * tp.G;
  A.st = (PcgState *)take(sizeof(PcgState));
  A.fail = (int *)(A.st + 1);
  (void)take(sizeof(PcgState));
  A.G = tp.G;
  A.bw = c->bandwidth;
  A.cap = tp.cap;
  A.bnorm = bnorm;
  A.tol = tol;
  A.maxiter = maxiter;
  A.check = check;
  A.looks = c->tile_looks;
  const long long nc = std::max<long long>(c->Ndof, 8LL * tp.G);
  hipLaunchKernelGGL((k_tile_clear<T>), dim3((unsigned)((nc + 255) / 256)), dim3(256), 0, s, A, c->Ndof);
  *ran = false;
  int rc = tile_dispatch<T>(c->ndpn, tp, [&](auto p, auto l, auto sc) -> int {
    auto k = k_pcg_resident<T, decltype(p)::value, decltype(l)::value, decltype(sc)::value>;
    if (tp.G == 1) {
      hipLaunchKernelGGL(k, dim3(1), dim3(TILE_T), tp.lds, s, A);
      *ran = hipGetLastError() == hipSuccess;
    } else {
      // cooperative: the runtime starts it only with every workgroup resident
      void *args[] = {&A};
      *ran = hipLaunchCooperativeKernel((const void *)k, dim3(tp.G), dim3(TILE_T), args, (unsigned)tp.lds, s) == hipSuccess;
      (void)hipGetLastError();
    }
    return FEMHOT_OK;
  });
  if (rc) return rc;
  if (!*ran) {
    c->tile_gave_up = true;
    return FEMHOT_OK;
  }
  struct Out {
    PcgState st;
    int fail;
  };
  Out *o = (Out *)c->h_pinned;
  FH_HIP(hipMemcpyAsync(o, A.st, sizeof(PcgState) + sizeof(int), hipMemcpyDeviceToHost, s));
  FH_HIP(hipStreamSynchronize(s));
  *ran = !o->fail && o->st.status != 0;
  *st = o->st;
  if (!*ran) {
    c->tile_gave_up = true;
    FH_HIP(hipMemcpyAsync(x, A.x0, sizeof(T) * c->Ndof, hipMemcpyDeviceToDevice, s));
  }
  return FEMHOT_OK;
}

// Sum (fixed order) of NBR partials by one workgroup of 1024 threads.
__device__ __forceinline__ double sum_nbr_1024(const double *part) {
  __shared__ double red[16];
  double v = part[threadIdx.x];
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  double t = 0.0;
  for (int k = 0; k < 16; ++k) t += red[k];
  return t;
}

// ||b||^2 and the initial ||r||^2 from their partials; converged at once when b = 0 or r is small enough.
// A nonzero *outer (the enclosing Newton solve has finished this load step, or failed) stops the solve
// before its first iteration with status 4.
__global__ __launch_bounds__(1024) void k_pcg_start(const double *bb_part, const double *rr_part, double tol2,
                                                    int maxiter, const int *outer, PcgState *st) {
  const double bb = sum_nbr_1024(bb_part);
  const double rr = sum_nbr_1024(rr_part);
  if (threadIdx.x == 0) {
    st->bnorm2 = bb;
    st->rr = rr;
    st->iters = 0;
    st->status = (outer && *outer)              ? 4
                 : !(rr == rr && rr < INFINITY) ? 2
                 : (bb == 0.0 || rr <= tol2 * bb) ? 1
                                                  : (maxiter <= 0 ? 3 : 0);
  }
}

// After one iteration's x, r update: count it, sum ||r||^2, stop on convergence, a non-finite residual or
// the iteration budget
__global__ __launch_bounds__(1024) void k_pcg_check(const double *rr_part, double tol2, int maxiter, PcgState *st) {
  if (st->status) return;
  const double rr = sum_nbr_1024(rr_part);
  if (threadIdx.x == 0) {
    const int it = st->iters + 1;
    st->iters = it;
    st->rr = rr;
    st->status = !(rr == rr && rr < INFINITY) ? 2 : rr <= tol2 * st->bnorm2 ? 1 : (it >= maxiter ? 3 : 0);
  }
}

__global__ void k_pcg_finish(const PcgState *st, int *iters, double *rel_res, int *status) {
  if (threadIdx.x == 0) {
    if (iters) *iters = st->iters;
    if (rel_res) *rel_res = st->bnorm2 > 0.0 ? sqrt(st->rr / st->bnorm2) : 0.0;
    if (status) *status = st->status;
  }
}

// part[block] = this workgroup's share of a.b
__global__ __launch_bounds__(256) void k_dot64(long long n, const double *a, const double *b, double *part) {
  double v = 0.0;
  for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long long)gridDim.x * 256)
    v += a[i] * b[i];
  v = block_sum256(v);
  if (threadIdx.x == 0) part[blockIdx.x] = v;
}

// r = b - A x (FP64); part[block] = this workgroup's share of ||r||^2
__global__ __launch_bounds__(256) void k_resid64(long long n, const double *b, const double *ax, double *r,
                                                 double *part) {
  double v = 0.0;
  for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long long)gridDim.x * 256) {
    const double ri = b[i] - ax[i];
    r[i] = ri;
    v += ri * ri;
  }
  v = block_sum256(v);
  if (threadIdx.x == 0) part[blockIdx.x] = v;
}

}  // namespace femhot

using namespace femhot;

extern "C" int femhot_spmv(femhot_ctx *h, const long long *row_ptr, const int *col_idx, const double *vals,
                           const double *x, double *y, void *stream) {
  FH_CHECK_ARG(h && row_ptr && col_idx && vals && x && y, FEMHOT_ERR_ARG, "null argument");
  Ctx *c = &h->c;
  int rc = ensure_pattern(c);
  if (rc) return rc;
  spmv_launch<double>(c->Ndof, row_ptr, col_idx, vals, x, y, nullptr, spmv_plan(c->Ndof, c->nnz, 1, false),
                      (hipStream_t)stream);
  FH_HIP(hipGetLastError());
  return FEMHOT_OK;
}

// femhot_pcg, also for the linear solves inside another call (which do not try a one-launch solve again after
// one has given up).
static int pcg_call(femhot_ctx *h, int mode, const long long *row_ptr, const int *col_idx, const double *vals,
                    const double *b, double *x, double tol, int maxiter, int *iters, double *rel_res, void *stream) {
  FH_CHECK_ARG(h && row_ptr && col_idx && vals && b && x, FEMHOT_ERR_ARG, "null argument");
  const bool node_blocked = (mode & FEMHOT_PCG_CONTEXT_PATTERN) != 0;
  mode &= ~FEMHOT_PCG_CONTEXT_PATTERN;
  FH_CHECK_ARG(mode == FEMHOT_F64 || mode == FEMHOT_F32, FEMHOT_ERR_ARG,
               "mode must be FEMHOT_F64 or FEMHOT_F32 (| FEMHOT_PCG_CONTEXT_PATTERN)");
  FH_CHECK_ARG(tol > 0 && maxiter > 0, FEMHOT_ERR_ARG, "tol and maxiter must be positive");
  Ctx *c = &h->c;
  int rc = ensure_pattern(c);
  if (rc) return rc;
  hipStream_t s = (hipStream_t)stream;
  const long long n = c->Ndof, nnz = c->nnz;
  const dim3 grid((unsigned)((n + 255) / 256));
  const int check = 10;
  const size_t vec64 = sizeof(double) * n, vec32 = sizeof(float) * n;
  const SpmvPlan sp = spmv_plan(n, nnz, c->ndpn, node_blocked);
  const size_t nsp = sp.blocks;
  // systems the tile kernels hold are solved in one launch (mixed: one launch per inner solve)
  TilePlan tp;
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  FH_HIP(hipStreamIsCapturing(s, &cs));
  if (node_blocked && cs == hipStreamCaptureStatusNone && !c->tile_gave_up)
    tp = mode == FEMHOT_F64 ? tile_plan<double>(c) : tile_plan<float>(c);
  // FP32 mode keeps an FP32 matrix and 5 FP32 vectors, and the resident solve's buffers, beside the FP64 part
  const size_t tile_bytes = mode == FEMHOT_F32 && tp.ok ? tile_ws_bytes<float>(c, tp) : 0;
  rc = ensure_workspace(c, pcg_ws_bytes(c) + (mode == FEMHOT_F32 ? tile_bytes + 5 * r256(vec32) + r256(sizeof(float) * nnz)
                                                                 : 0));
  if (rc) return rc;
  if (tp.ok && mode == FEMHOT_F64) {
    PcgState st{};
    bool ran = false;
    rc = tile_solve<double>(c, tp, c->d_ws, row_ptr, col_idx, vals, b, x, -1.0, tol, maxiter, check, s, &st, &ran);
    if (rc) return rc;
    if (ran) {
      if (iters) *iters = st.iters;
      if (st.status == 2) {
        set_error("femhot_pcg: non-finite residual");
        return FEMHOT_ERR_NONFINITE;
      }
      if (rel_res) *rel_res = st.bnorm2 > 0.0 ? std::sqrt(std::max(st.rr, 0.0) / st.bnorm2) : 0.0;
      if (st.status != 1) {
        set_error("femhot_pcg: maximum iterations reached");
        return FEMHOT_ERR_NOT_CONVERGED;
      }
      return FEMHOT_OK;
    }
  }
  char *ws = (char *)c->d_ws;
  auto take = [&](size_t bytes) {
    char *p = ws;
    ws += (bytes + 255) & ~size_t(255);
    return (void *)p;
  };
  void *tile_ws = mode == FEMHOT_F32 && tp.ok ? take(tile_bytes) : nullptr;
  double *sc = (double *)take(3 * NBR * sizeof(double));
  double *aux = (double *)take(NBR * sizeof(double));
  double *pap_part = (double *)take(nsp * sizeof(double));
  double *pap = (double *)take(8 * sizeof(double));
  double *r64 = (double *)take(vec64), *p64 = (double *)take(vec64), *q64 = (double *)take(vec64);
  double *dinv64 = (double *)take(vec64), *ax64 = (double *)take(vec64);
  // ||b||
  hipLaunchKernelGGL(k_dot64, dim3(NBR), dim3(256), 0, s, n, b, b, aux);
  double bb = 0.0;
  rc = host_sum_partials(c, aux, s, &bb);
  if (rc) return rc;
  const double bnorm = std::sqrt(bb);
  if (node_blocked)
    hipLaunchKernelGGL((k_diag_inv_pos<double>), grid, dim3(256), 0, s, n, row_ptr, c->d_diag_off, vals, dinv64);
  else
    hipLaunchKernelGGL((k_diag_inv<double>), grid, dim3(256), 0, s, n, row_ptr, col_idx, vals, dinv64);
  int it = 0;
  double rel = 0.0;
  bool conv = false;
  if (mode == FEMHOT_F64) {
    rc = pcg_core<double>(c, n, row_ptr, col_idx, vals, b, x, r64, p64, q64, dinv64, sc, pap_part, pap, bnorm, tol,
                          maxiter, check, sp, s, &it, &rel, &conv);
    if (rc) return rc;
  } else {
    float *v32 = (float *)take(sizeof(float) * nnz);
    float *x32 = (float *)take(vec32), *r32 = (float *)take(vec32), *p32 = (float *)take(vec32);
    float *q32 = (float *)take(vec32), *dinv32 = (float *)take(vec32);
    bool cast_done = false;
    auto cast = [&] {  // the FP32 matrix and diagonal of the launched kernels (the tile kernels convert as they load)
      if (cast_done) return;
      cast_done = true;
      const unsigned cg = (unsigned)std::min<long long>((nnz + 255) / 256, 65536);
      hipLaunchKernelGGL((k_cast<float>), dim3(cg), dim3(256), 0, s, nnz, vals, v32);
      if (node_blocked)
        hipLaunchKernelGGL((k_diag_inv_pos<float>), grid, dim3(256), 0, s, n, row_ptr, c->d_diag_off, vals, dinv32);
      else
        hipLaunchKernelGGL((k_diag_inv<float>), grid, dim3(256), 0, s, n, row_ptr, col_idx, vals, dinv32);
    };
    // outer FP64 refinement: r = b - A x; solve A d = r in FP32 to inner_tol; x += d
    const double inner_tol = 1e-4;
    int outer = 0;
    while (true) {
      spmv_launch<double>(n, row_ptr, col_idx, vals, x, ax64, nullptr, sp, s);
      hipLaunchKernelGGL(k_resid64, dim3(NBR), dim3(256), 0, s, n, b, ax64, r64, aux);
      double r2 = 0.0;
      rc = host_sum_partials(c, aux, s, &r2);
      if (rc) return rc;
      rel = bnorm > 0 ? std::sqrt(r2) / bnorm : 0.0;
      if (!std::isfinite(rel)) {
        set_error("femhot_pcg: non-finite residual");
        return FEMHOT_ERR_NONFINITE;
      }
      if (rel <= tol) {
        conv = true;
        break;
      }
      if (it >= maxiter || outer >= 50) break;
      FH_CHECK_ARG(fill<float>(x32, n, n, 1, 0.0f, s) == FEMHOT_OK, FEMHOT_ERR_HIP, "fill failed");
      int k_in = 0;
      double rel_in = 0.0;
      bool cin = false;
      // inner solve on the FP64 residual r64 (FP32 iterates, FP64 dot products)
      const double tol_in = std::max(inner_tol, 0.5 * tol / std::max(rel, 1e-300));
      bool ran = false;
      if (tile_ws) {
        PcgState st{};
        rc = tile_solve<float>(c, tp, tile_ws, row_ptr, col_idx, vals, r64, x32, bnorm * rel, tol_in, maxiter - it,
                               check, s, &st, &ran);
        if (rc) return rc;
        k_in = st.iters;
        if (ran && st.status == 2) {
          set_error("femhot_pcg: non-finite residual");
          if (iters) *iters = it + k_in;
          return FEMHOT_ERR_NONFINITE;
        }
        if (!ran) tile_ws = nullptr;  // the further inner solves do not try again
      }
      if (!ran) cast();
      if (!ran)
        rc = pcg_core<float>(c, n, row_ptr, col_idx, v32, r64, x32, r32, p32, q32, dinv32, sc, pap_part, pap, bnorm * rel,
                             tol_in, maxiter - it, check, sp, s, &k_in, &rel_in, &cin);
      if (rc) return rc;
      it += std::max(k_in, 1);
      hipLaunchKernelGGL((k_axpy_to64<float>), grid, dim3(256), 0, s, n, x32, x);
      ++outer;
    }
  }
  FH_HIP(hipGetLastError());
  if (iters) *iters = it;
  if (rel_res) *rel_res = rel;
  if (!conv) {
    set_error("femhot_pcg: maximum iterations reached");
    return FEMHOT_ERR_NOT_CONVERGED;
  }
  return FEMHOT_OK;
}

extern "C" int femhot_pcg(femhot_ctx *h, int mode, const long long *row_ptr, const int *col_idx, const double *vals,
                          const double *b, double *x, double tol, int maxiter, int *iters, double *rel_res,
                          void *stream) {
  if (h) h->c.tile_gave_up = false;
  return pcg_call(h, mode, row_ptr, col_idx, vals, b, x, tol, maxiter, iters, rel_res, stream);
}

extern "C" int femhot_pcg_wait_limit(femhot_ctx *h, int looks) {
  FH_CHECK_ARG(h && looks >= 0, FEMHOT_ERR_ARG, "femhot_pcg_wait_limit: a context and looks >= 0");
  h->c.tile_looks = looks;
  return FEMHOT_OK;
}

static int pcg_async_core(Ctx *c, bool node_blocked, const long long *row_ptr, const int *col_idx,
                          const double *vals, const double *b, double *x, double tol, int iterations,
                          const int *outer, const PcgState **state_out, int *iters, double *rel_res, int *status,
                          hipStream_t s);

extern "C" int femhot_pcg_async(femhot_ctx *h, int mode, const long long *row_ptr, const int *col_idx,
                                const double *vals, const double *b, double *x, double tol, int iterations,
                                int *iters, double *rel_res, int *status, void *stream) {
  FH_CHECK_ARG(h && row_ptr && col_idx && vals && b && x, FEMHOT_ERR_ARG, "femhot_pcg_async: null argument");
  const bool node_blocked = (mode & FEMHOT_PCG_CONTEXT_PATTERN) != 0;
  mode &= ~FEMHOT_PCG_CONTEXT_PATTERN;
  FH_CHECK_ARG(mode == FEMHOT_F64, FEMHOT_ERR_ARG, "femhot_pcg_async: mode must be FEMHOT_F64 (| FEMHOT_PCG_CONTEXT_PATTERN)");
  FH_CHECK_ARG(tol > 0 && iterations > 0, FEMHOT_ERR_ARG, "femhot_pcg_async: tol and iterations must be positive");
  Ctx *c = &h->c;
  FH_CHECK_ARG(c->have_pattern, FEMHOT_ERR_ARG,
               "femhot_pcg_async: build the context's pattern first (femhot_pattern or one tangent call)");
  return pcg_async_core(c, node_blocked, row_ptr, col_idx, vals, b, x, tol, iterations, nullptr, nullptr, iters,
                        rel_res, status, (hipStream_t)stream);
}

// The enqueued solve of femhot_pcg_async.  outer: a device flag that, when nonzero as the solve starts,
// skips it (status 4; the Newton driver's end-of-step flag); *state_out: where the solver state lives
// until the next solve on this context.
static int pcg_async_core(Ctx *c, bool node_blocked, const long long *row_ptr, const int *col_idx,
                          const double *vals, const double *b, double *x, double tol, int iterations,
                          const int *outer, const PcgState **state_out, int *iters, double *rel_res, int *status,
                          hipStream_t s) {
  const long long n = c->Ndof, nnz = c->nnz;
  const dim3 grid((unsigned)((n + 255) / 256)), nbr(NBR);
  const size_t vec64 = sizeof(double) * n;
  const SpmvPlan sp = spmv_plan(n, nnz, c->ndpn, node_blocked);
  const size_t nsp = sp.blocks;
  const size_t need = pcg_ws_bytes(c);
  if (c->ws_bytes < need) {  // sized once; never inside a graph capture
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    FH_HIP(hipStreamIsCapturing(s, &cs));
    FH_CHECK_ARG(cs == hipStreamCaptureStatusNone, FEMHOT_ERR_ARG,
                 "femhot_pcg_async: the solver workspace is not sized; make one uncaptured call (or femhot_pcg) on "
                 "this context first, so captured calls allocate nothing");
    int rc = ensure_workspace(c, need);
    if (rc) return rc;
  }
  char *ws = (char *)c->d_ws;
  auto take = [&](size_t bytes) {
    char *p = ws;
    ws += (bytes + 255) & ~size_t(255);
    return (void *)p;
  };
  const TilePlan tp = node_blocked ? tile_plan<double>(c) : TilePlan{};
  if (tp.ok) {  // the phases of the resident solve, one launch each: its bits, and a graph can hold them
    TileVecs V;
    V.r = (double *)take(vec64);
    V.z = (double *)take(vec64);
    V.dinv = (double *)take(vec64);
    V.q = (double *)take(vec64);
    V.p[0] = (double *)take(vec64);
    V.p[1] = (double *)take(vec64);
    TileArgs A{};
    A.nodes = c->Nn;
    A.rp = row_ptr;
    A.ci = col_idx;
    A.vals = vals;
    A.doff = c->d_diag_off;
    A.b = b;
    A.x = x;
    A.pa = (double *)take(sizeof(double) * 8 * tp.G);
    A.pc = A.pa + 6 * tp.G;
    A.st = (PcgState *)take(sizeof(PcgState));
    A.G = tp.G;
    A.tol = tol;
    A.maxiter = iterations;
    int rc = tile_dispatch<double>(c->ndpn, tp, [&](auto p, auto l, auto sc) -> int {
      constexpr int P = decltype(p)::value, LPN = decltype(l)::value, S = decltype(sc)::value;
      const dim3 g(tp.G), t(TILE_T);
      // Workgroups that make 4 or 8 passes wait for memory as often, with at most two waves per SIMD: with one
      // dof per node a workgroup per pass and a kernel for p.q are faster (us an iteration: quads 300 x 300
      // 18.6 -> 15.6, hexahedra 38^3 21.5 -> 16.7, 48^3 25.2 -> 24.8), with two, whose passes hold four times
      // the values, slower (quads 350 x 350 26.5 -> 28.8); one workgroup alone has too few passes to gain.
      constexpr bool may_split = P == 1 && S >= 4;
      [[maybe_unused]] const long long passes = (c->Nn * LPN + TILE_T - 1) / TILE_T;
      hipLaunchKernelGGL((k_tile_init<P, LPN, S>), g, t, 0, s, A, V);
      for (int k = 0; k < iterations; ++k) {
        bool split = false;
        if constexpr (may_split)
          if ((split = tp.G > 1)) {
            hipLaunchKernelGGL((k_tile_pass<P, LPN>), dim3((unsigned)passes), t, 0, s, A, V, k, outer);
            hipLaunchKernelGGL((k_tile_dot<P, LPN, S>), g, t, 0, s, A, V, k & 1);
          }
        if (!split) hipLaunchKernelGGL((k_tile_spmv<P, LPN, S>), g, t, 0, s, A, V, k, outer);
        hipLaunchKernelGGL((k_tile_update<P, LPN, S>), g, t, 0, s, A, V, k & 1);
      }
      hipLaunchKernelGGL(k_tile_test, dim3(1), t, 0, s, A, iterations);
      hipLaunchKernelGGL(k_pcg_finish, dim3(1), dim3(64), 0, s, A.st, iters, rel_res, status);
      FH_HIP(hipGetLastError());
      return FEMHOT_OK;
    });
    if (state_out) *state_out = A.st;
    return rc;
  }
  double *sc = (double *)take(3 * NBR * sizeof(double));
  double *aux = (double *)take(NBR * sizeof(double));
  double *pap_part = (double *)take(nsp * sizeof(double));
  double *pap = (double *)take(8 * sizeof(double));
  double *r = (double *)take(vec64), *p = (double *)take(vec64), *q = (double *)take(vec64);
  double *dinv = (double *)take(vec64);
  (void)take(vec64);
  PcgState *st = (PcgState *)take(sizeof(PcgState));
  const int *stop = &st->status;
  double *rz[2] = {sc, sc + NBR}, *rrp = sc + 2 * NBR;
  const double tol2 = tol * tol;
  hipLaunchKernelGGL(k_dot64, nbr, dim3(256), 0, s, n, b, b, aux);
  if (node_blocked)
    hipLaunchKernelGGL((k_diag_inv_pos<double>), grid, dim3(256), 0, s, n, row_ptr, c->d_diag_off, vals, dinv);
  else
    hipLaunchKernelGGL((k_diag_inv<double>), grid, dim3(256), 0, s, n, row_ptr, col_idx, vals, dinv);
  spmv_launch<double>(n, row_ptr, col_idx, vals, x, r, nullptr, sp, s);  // r = A x
  hipLaunchKernelGGL((k_init<double>), nbr, dim3(256), 0, s, n, b, r, p, dinv, rz[0], rrp);
  hipLaunchKernelGGL(k_pcg_start, dim3(1), dim3(1024), 0, s, aux, rrp, tol2, iterations, outer, st);
  const bool alt = spmv_alternates<double>(c->nnz);
  for (int k = 0; k < iterations; ++k) {  // the same kernels as femhot_pcg; a stopped solve skips them
    const int par = k & 1;
    spmv_launch<double>(n, row_ptr, col_idx, vals, p, q, pap_part, sp, s, stop, alt ? par : 0);
    hipLaunchKernelGGL(k_sum_parts, dim3(1), dim3(1024), 0, s, pap_part, (long long)nsp, pap, stop);
    hipLaunchKernelGGL((k_update_xr<double>), nbr, dim3(256), 0, s, n, x, r, p, q, dinv, rz[par], pap, rz[1 - par],
                       rrp, stop);
    hipLaunchKernelGGL(k_pcg_check, dim3(1), dim3(1024), 0, s, rrp, tol2, iterations, st);
    hipLaunchKernelGGL((k_update_p<double>), nbr, dim3(256), 0, s, n, p, r, dinv, rz[1 - par], rz[par], stop);
  }
  hipLaunchKernelGGL(k_pcg_finish, dim3(1), dim3(64), 0, s, st, iters, rel_res, status);
  FH_HIP(hipGetLastError());
  if (state_out) *state_out = st;
  return FEMHOT_OK;
}

// ------------------------------------------------------------------------------------------
// Load-stepped Newton-Raphson driver (fol/solvers/fe_nonlinear_residual_based_solver.py:76-170)
// ------------------------------------------------------------------------------------------

// Dirichlet dofs of u set to scale * value (ApplyDirichletBCOnDofVector, fe_loss.py:91-92 with the
// load increment of the nonlinear solver).
__global__ void k_apply_dirichlet(long long n, double *u, const uint8_t *dmask, const double *dval, double scale) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n && dmask[i]) u[i] = scale * dval[i];
}
__global__ void k_newton_rhs(long long n, const double *R, double *b, double *du) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) {
    b[i] = -R[i];
    du[i] = 0.0;
  }
}
__global__ void k_add64(long long n, double *u, const double *du) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) u[i] += du[i];
}

extern "C" int femhot_newton(femhot_ctx *h, int mode, const double *field, double *u, unsigned flags,
                             int load_steps, int max_iter, double abs_tol, double rel_tol, double lin_tol,
                             int lin_maxiter, double *history, int *steps, void *stream) {
  FH_CHECK_ARG(h && field && u, FEMHOT_ERR_ARG, "femhot_newton: null argument");
  FH_CHECK_ARG(mode == FEMHOT_F64 || mode == FEMHOT_F32, FEMHOT_ERR_ARG,
               "femhot_newton: mode must be FEMHOT_F64 or FEMHOT_F32");
  FH_CHECK_ARG(load_steps > 0 && max_iter > 0 && lin_tol > 0 && lin_maxiter > 0, FEMHOT_ERR_ARG,
               "femhot_newton: load_steps, max_iter, lin_tol and lin_maxiter must be positive");
  FH_CHECK_ARG((flags & ~(FEMHOT_ELEMENT_FIELD | FEMHOT_SCATTER_COLOUR | FEMHOT_SCATTER_CHUNK | FEMHOT_SCATTER_ROWS)) ==
                   0,
               FEMHOT_ERR_ARG,
               "femhot_newton: flags may hold FEMHOT_ELEMENT_FIELD and FEMHOT_SCATTER_{COLOUR,CHUNK,ROWS} only");
  Ctx *c = &h->c;
  c->tile_gave_up = false;
  int rc = ensure_pattern(c);
  if (rc) return rc;
  hipStream_t s = (hipStream_t)stream;
  const long long n = c->Ndof, nnz = c->nnz;
  auto up = [](size_t b) { return (b + 255) & ~size_t(255); };
  const size_t need = up(sizeof(double) * std::max<long long>(nnz, 1)) + 4 * up(sizeof(double) * n) +
                      up(sizeof(double) * NBR);
  if (c->newton_ws.bytes < need) {
    FH_HIP(hipStreamSynchronize(s));
    if (c->newton_ws.ptr) FH_HIP(hipFree(c->newton_ws.ptr));
    c->newton_ws.ptr = nullptr;
    c->newton_ws.bytes = 0;
    c->newton_dval_ready = false;
    FH_HIP(hipMalloc(&c->newton_ws.ptr, need));
    c->newton_ws.bytes = need;
  }
  char *ws = (char *)c->newton_ws.ptr;
  auto take = [&](size_t bytes) {
    char *p = ws;
    ws += up(bytes);
    return (void *)p;
  };
  double *vals = (double *)take(sizeof(double) * std::max<long long>(nnz, 1));
  double *R = (double *)take(sizeof(double) * n), *b = (double *)take(sizeof(double) * n);
  double *du = (double *)take(sizeof(double) * n), *dval = (double *)take(sizeof(double) * n);
  double *part = (double *)take(sizeof(double) * NBR);
  if (!c->newton_dval_ready) {  // Dirichlet values as a dense dof vector (the last entry of a repeated dof wins)
    std::vector<double> hv((size_t)n, 0.0);
    for (size_t k = 0; k < c->h_dir_idx.size(); ++k) hv[(size_t)c->h_dir_idx[k]] = c->h_dir_val[k];
    FH_HIP(hipStreamSynchronize(s));
    FH_HIP(hipMemcpy(dval, hv.data(), sizeof(double) * n, hipMemcpyHostToDevice));
    c->newton_dval_ready = true;
  }
  if (history)
    for (long long k = 0; k < 2LL * load_steps * max_iter; ++k) history[k] = std::nan("");
  const dim3 grid((unsigned)((n + 255) / 256));
  for (int step = 1; step <= load_steps; ++step) {
    hipLaunchKernelGGL(k_apply_dirichlet, grid, dim3(256), 0, s, n, u, c->d_dmask, dval,
                       (double)step / load_steps);
    int it = 1;
    for (;; ++it) {
      rc = femhot_tangent_csr(h, FEMHOT_F64, field, u, vals, R, flags, stream);
      if (rc) return rc;
      hipLaunchKernelGGL(k_dot64, dim3(NBR), dim3(256), 0, s, n, R, R, part);
      double rr = 0.0;
      if ((rc = host_sum_partials(c, part, s, &rr))) return rc;
      const double res_norm = std::sqrt(rr);
      if (std::isnan(res_norm)) {
        if (steps) steps[step - 1] = it;
        set_error("femhot_newton: residual norm contains NaN values");
        return FEMHOT_ERR_NONFINITE;
      }
      hipLaunchKernelGGL(k_newton_rhs, grid, dim3(256), 0, s, n, R, b, du);
      int lit = 0;
      double lrel = 0.0;
      rc = pcg_call(h, mode | FEMHOT_PCG_CONTEXT_PATTERN, c->d_row_ptr, c->d_col_idx, vals, b, du, lin_tol,
                    lin_maxiter, &lit, &lrel, stream);
      if (rc && rc != FEMHOT_ERR_NOT_CONVERGED) return rc;  // an unconverged solve continues with its iterate
      hipLaunchKernelGGL(k_dot64, dim3(NBR), dim3(256), 0, s, n, du, du, part);
      double dd = 0.0;
      if ((rc = host_sum_partials(c, part, s, &dd))) return rc;
      const double du_norm = std::sqrt(dd);
      if (history) {
        history[2LL * ((long long)(step - 1) * max_iter + (it - 1))] = res_norm;
        history[2LL * ((long long)(step - 1) * max_iter + (it - 1)) + 1] = du_norm;
      }
      if (res_norm < abs_tol || du_norm < rel_tol || it == max_iter) break;
      hipLaunchKernelGGL(k_add64, grid, dim3(256), 0, s, n, u, du);
    }
    if (steps) steps[step - 1] = it;
  }
  FH_HIP(hipGetLastError());
  FH_HIP(hipStreamSynchronize(s));
  return FEMHOT_OK;
}

// ------------------------------------------------------------------------------------------
// The same load-stepped Newton solve with every decision on the device: nothing waits for the host,
// so a whole nonlinear solve can be captured into a HIP graph.
// ------------------------------------------------------------------------------------------

struct NewtonState {
  int halt;    // this load step has ended (or the solve failed): the guarded kernels return
  int failed;  // a NaN residual norm or a non-finite linear solve: every later kernel returns
  double res_norm;
};

__global__ void k_newton_init(NewtonState *st, double *history, long long n_hist, int *steps, int load_steps) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i == 0) {
    st->halt = 0;
    st->failed = 0;
    st->res_norm = 0.0;
  }
  if (history && i < n_hist) history[i] = __builtin_nan("");
  if (steps && i < load_steps) steps[i] = 0;
}
__global__ void k_newton_begin_step(NewtonState *st) { st->halt = st->failed; }
__global__ void k_apply_dirichlet_if(long long n, double *u, const uint8_t *dmask, const double *dval, double scale,
                                     const int *failed) {
  if (*failed) return;
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n && dmask[i]) u[i] = scale * dval[i];
}
__global__ void k_newton_rhs_if(long long n, const double *R, double *b, double *du, const int *halt) {
  if (*halt) return;
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) {
    b[i] = -R[i];
    du[i] = 0.0;
  }
}
__global__ void k_add64_if(long long n, double *u, const double *du, const int *halt) {
  if (*halt) return;
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) u[i] += du[i];
}
// ||R|| of this iteration (from k_dot64's partials) into the state and the history; a NaN ends the solve
__global__ __launch_bounds__(1024) void k_newton_res(const double *part, NewtonState *st, double *hist,
                                                     int *step_iters, int it) {
  if (st->halt) return;
  const double rn = sqrt(sum_nbr_1024(part));
  if (threadIdx.x == 0) {
    st->res_norm = rn;
    if (hist) hist[0] = rn;
    if (rn != rn) {
      st->failed = 1;
      st->halt = 1;
      if (step_iters) *step_iters = it;
    }
  }
}
// ||du|| after the linear solve; the load step ends when ||R|| < abs_tol, ||du|| < rel_tol or at max_iter
// (the update of that last iteration is not applied), the solve when the linear solve was non-finite
__global__ __launch_bounds__(1024) void k_newton_du(const double *part, NewtonState *st, const PcgState *ps,
                                                    double *hist, int *step_iters, int it, int max_iter,
                                                    double abs_tol, double rel_tol) {
  if (st->halt) return;
  const double dn = sqrt(sum_nbr_1024(part));
  if (threadIdx.x == 0) {
    if (ps->status == 2) {
      st->failed = 1;
      st->halt = 1;
      if (step_iters) *step_iters = it;
      return;
    }
    if (hist) hist[1] = dn;
    if (st->res_norm < abs_tol || dn < rel_tol || it == max_iter) {
      st->halt = 1;
      if (step_iters) *step_iters = it;
    }
  }
}
__global__ void k_newton_finish(const NewtonState *st, int *status) {
  if (threadIdx.x == 0 && status) *status = st->failed ? FEMHOT_ERR_NONFINITE : FEMHOT_OK;
}

extern "C" int femhot_newton_async(femhot_ctx *h, const double *field, double *u, unsigned flags, int load_steps,
                                   int max_iter, double abs_tol, double rel_tol, double lin_tol, int lin_iterations,
                                   double *history, int *steps, int *status, void *stream) {
  FH_CHECK_ARG(h && field && u, FEMHOT_ERR_ARG, "femhot_newton_async: null argument");
  FH_CHECK_ARG(load_steps > 0 && max_iter > 0 && lin_tol > 0 && lin_iterations > 0, FEMHOT_ERR_ARG,
               "femhot_newton_async: load_steps, max_iter, lin_tol and lin_iterations must be positive");
  FH_CHECK_ARG((flags & ~(FEMHOT_ELEMENT_FIELD | FEMHOT_SCATTER_COLOUR | FEMHOT_SCATTER_CHUNK | FEMHOT_SCATTER_ROWS)) ==
                   0,
               FEMHOT_ERR_ARG,
               "femhot_newton_async: flags may hold FEMHOT_ELEMENT_FIELD and FEMHOT_SCATTER_{COLOUR,CHUNK,ROWS} only");
  Ctx *c = &h->c;
  hipStream_t s = (hipStream_t)stream;
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  FH_HIP(hipStreamIsCapturing(s, &cs));
  const bool capturing = cs != hipStreamCaptureStatusNone;
  auto up = [](size_t b) { return (b + 255) & ~size_t(255); };
  const long long n = c->Ndof;
  // the workspace of femhot_newton followed by the solve's state
  const size_t need = up(sizeof(double) * std::max<long long>(c->nnz, 1)) + 4 * up(sizeof(double) * n) +
                      up(sizeof(double) * NBR) + up(sizeof(NewtonState));
  if (!c->have_pattern || c->newton_ws.bytes < need || !c->newton_dval_ready ||
      c->ws_bytes < pcg_ws_bytes(c)) {
    FH_CHECK_ARG(!capturing, FEMHOT_ERR_ARG,
                 "femhot_newton_async: make one uncaptured call on this context first (it builds the pattern and sizes "
                 "the workspaces), so captured calls allocate nothing");
    int rc = ensure_pattern(c);
    if (rc) return rc;
    const size_t need_now = up(sizeof(double) * std::max<long long>(c->nnz, 1)) + 4 * up(sizeof(double) * n) +
                            up(sizeof(double) * NBR) + up(sizeof(NewtonState));
    if (c->newton_ws.bytes < need_now) {
      FH_HIP(hipStreamSynchronize(s));
      if (c->newton_ws.ptr) FH_HIP(hipFree(c->newton_ws.ptr));
      c->newton_ws.ptr = nullptr;
      c->newton_ws.bytes = 0;
      c->newton_dval_ready = false;
      FH_HIP(hipMalloc(&c->newton_ws.ptr, need_now));
      c->newton_ws.bytes = need_now;
    }
    if ((rc = ensure_workspace(c, pcg_ws_bytes(c)))) return rc;
  }
  char *ws = (char *)c->newton_ws.ptr;
  auto take = [&](size_t bytes) {
    char *p = ws;
    ws += up(bytes);
    return (void *)p;
  };
  double *vals = (double *)take(sizeof(double) * std::max<long long>(c->nnz, 1));
  double *R = (double *)take(sizeof(double) * n), *b = (double *)take(sizeof(double) * n);
  double *du = (double *)take(sizeof(double) * n), *dval = (double *)take(sizeof(double) * n);
  double *part = (double *)take(sizeof(double) * NBR);
  NewtonState *st = (NewtonState *)take(sizeof(NewtonState));
  if (!c->newton_dval_ready) {  // Dirichlet values as a dense dof vector (the last entry of a repeated dof wins)
    std::vector<double> hv((size_t)n, 0.0);
    for (size_t k = 0; k < c->h_dir_idx.size(); ++k) hv[(size_t)c->h_dir_idx[k]] = c->h_dir_val[k];
    FH_HIP(hipStreamSynchronize(s));
    FH_HIP(hipMemcpy(dval, hv.data(), sizeof(double) * n, hipMemcpyHostToDevice));
    c->newton_dval_ready = true;
  }
  const long long n_hist = 2LL * load_steps * max_iter;
  const dim3 grid((unsigned)((n + 255) / 256));
  const long long n_init = std::max<long long>({n_hist, (long long)load_steps, 1});
  hipLaunchKernelGGL(k_newton_init, dim3((unsigned)((n_init + 255) / 256)), dim3(256), 0, s, st, history, n_hist,
                     steps, load_steps);
  const int *halt = &st->halt, *failed = &st->failed;
  for (int step = 1; step <= load_steps; ++step) {
    hipLaunchKernelGGL(k_apply_dirichlet_if, grid, dim3(256), 0, s, n, u, c->d_dmask, dval, (double)step / load_steps,
                       failed);
    hipLaunchKernelGGL(k_newton_begin_step, dim3(1), dim3(1), 0, s, st);
    int *step_iters = steps ? steps + (step - 1) : nullptr;
    for (int it = 1; it <= max_iter; ++it) {
      double *hist = history ? history + 2LL * ((long long)(step - 1) * max_iter + (it - 1)) : nullptr;
      // the tangent and residual are assembled whatever the flags say (their outputs are this call's
      // workspace; u only changes through the guarded update below)
      int rc = femhot_tangent_csr(h, FEMHOT_F64, field, u, vals, R, flags, stream);
      if (rc) return rc;
      hipLaunchKernelGGL(k_dot64, dim3(NBR), dim3(256), 0, s, n, R, R, part);
      hipLaunchKernelGGL(k_newton_res, dim3(1), dim3(1024), 0, s, part, st, hist, step_iters, it);
      hipLaunchKernelGGL(k_newton_rhs_if, grid, dim3(256), 0, s, n, R, b, du, halt);
      const PcgState *ps = nullptr;
      rc = pcg_async_core(c, true, c->d_row_ptr, c->d_col_idx, vals, b, du, lin_tol, lin_iterations, halt, &ps,
                          nullptr, nullptr, nullptr, s);
      if (rc) return rc;
      hipLaunchKernelGGL(k_dot64, dim3(NBR), dim3(256), 0, s, n, du, du, part);
      hipLaunchKernelGGL(k_newton_du, dim3(1), dim3(1024), 0, s, part, st, ps, hist, step_iters, it, max_iter, abs_tol,
                         rel_tol);
      hipLaunchKernelGGL(k_add64_if, grid, dim3(256), 0, s, n, u, du, halt);
    }
  }
  hipLaunchKernelGGL(k_newton_finish, dim3(1), dim3(64), 0, s, st, status);
  FH_HIP(hipGetLastError());
  return FEMHOT_OK;
}
