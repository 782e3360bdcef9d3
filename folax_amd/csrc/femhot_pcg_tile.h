// Jacobi-PCG of small and medium systems on the context's own pattern (P dofs per node, every dof row of
// a node listing the same neighbours as P x P blocks): G workgroups of 512 threads, each owning a run
// of nodes, LPN lanes per node, U = 4 neighbour blocks per lane, S nodes per group of lanes.  Two forms
// with the same node-to-lane mapping, the same arithmetic and the same summation orders, so that their
// iterates are equal bit for bit:
//
//  * k_pcg_resident: the whole solve in one launch (cooperative when G > 1).  A launched iteration costs
//    four kernels of 2-5 us each whatever the system's size (16-18 us up to 10,000 dofs).  Here the
//    matrix stays in registers, the search direction of every node the workgroup's rows touch stays in
//    LDS, and an iteration exchanges only z and the partial dot products: two hops through memory.
//  * k_tile_init / k_tile_spmv (or k_tile_pass, k_tile_dot) / k_tile_update: one launch per phase, for
//    callers that capture solves into a graph, where a cooperative launch does not belong.  Bound by the
//    launches: two an iteration and 2-5 us each up to 60,000 dofs.  A captured iteration against the five
//    kernels of larger systems, which these sizes took before: quads 40 x 40 conduction 15.1 -> 8.9 us,
//    300 x 300 18.4 -> 15.6, hexahedra 20^3 elastic 18.5 -> 11.4, 45^3 conduction 23.5 -> 21.2.
//
// Exchange.  Values are published with agent-scope stores into slots that hold a sentinel (a NaN with all
// bits set) until then, and read by polling until the sentinel is gone: the value is its own flag, no
// fence and no second message.  Slots alternate by the iteration's parity; an owner resets a slot after
// every reader has consumed it (it has passed the next exchange) and waits for that store before it
// publishes to the exchange that precedes the slot's reuse.  Polls are bounded: a workgroup that waits
// too long raises `fail` and leaves, after which every other one's waits end too, and the caller solves with the
// launched kernels.  A workgroup may give up just as the others converge and store their parts of x, so the
// start vector is kept (x0) and put back first.
//
// p of a neighbour is formed by its readers as z + beta p (as by its owner: one FMA, the same bits), so
// the exchange that sums r.z also carries the vector the SpMV needs.
#pragma once
#include "femhot_kernels.h"

namespace femhot {

constexpr int TILE_U = 4;       // neighbour blocks per lane
constexpr int TILE_T = 512;     // threads per workgroup
constexpr int TILE_RANGE = 65536;  // most node ids between the first and last column of a workgroup's rows

// Solver state shared by the forms: status 0 running, 1 converged, 2 non-finite residual, 3 iteration
// budget spent, 4 skipped (an enclosing solve has ended).
struct PcgState {
  int status;
  int iters;
  double bnorm2;
  double rr;
};

struct TileArgs {
  long long nodes;
  const long long *rp;
  const int *ci;
  const double *vals;
  const int *doff;  // offset of each row's diagonal within the row, -1 for an empty row
  const double *b;
  void *x;          // initial guess in, solution out (T)
  void *x0;         // the initial guess, kept by k_tile_clear (T)
  void *z[2];       // published z by parity (n, T)
  double *pa;       // (2 parities, 3, G): r.z, r.r, b.b
  double *pc;       // (2 parities, G): p.Ap
  int G, bw, cap;   // workgroups, largest |column node - row node|, LDS nodes per workgroup
  double bnorm;     // < 0: the solve takes ||b|| itself
  double tol;
  int maxiter, check;
  int looks;        // before a wait gives up
  PcgState *st;
  int *fail;
};

template <class T> struct TileBits;
template <> struct TileBits<double> { using U = unsigned long long; };
template <> struct TileBits<float> { using U = unsigned int; };

template <class T> __device__ __forceinline__ void tile_publish(T *p, T v) {
  using U = typename TileBits<T>::U;
  U b = __builtin_bit_cast(U, v != v ? T(__builtin_nan("")) : v);
  __hip_atomic_store(reinterpret_cast<U *>(p), b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class T> __device__ __forceinline__ void tile_reset(T *p) {
  using U = typename TileBits<T>::U;
  __hip_atomic_store(reinterpret_cast<U *>(p), ~U(0), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class T> __device__ __forceinline__ typename TileBits<T>::U tile_peek(const T *p) {
  using U = typename TileBits<T>::U;
  return __hip_atomic_load(reinterpret_cast<const U *>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// The value published at p; `seen` may hold an earlier look at it.  Gives up (bad) after `looks` looks, and at
// once where this lane has given up before.
template <class T>
__device__ __forceinline__ T tile_wait(const T *p, typename TileBits<T>::U seen, int looks, int &bad) {
  using U = typename TileBits<T>::U;
  for (int n = 0; seen == ~U(0); ++n) {
    if (bad || n >= looks) {
      bad = 1;
      return T(0);
    }
    seen = tile_peek(p);
  }
  return __builtin_bit_cast(T, seen);
}
// Every store of this wave has reached the memory other workgroups read.
__device__ __forceinline__ void tile_stores_done() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// Sum over each aligned group of N lanes (4, 8 or 16), held by all of them: quad_perm [1,0,3,2] and
// [2,3,0,1], then row_half_mirror and row_mirror, which pair lanes of equal sums.
template <int N, class T> __device__ __forceinline__ T tile_lane_sum(T v) {
  v += lane_dpp<0xB1>(v);
  v += lane_dpp<0x4E>(v);
  if constexpr (N >= 8) v += lane_dpp<0x141>(v);
  if constexpr (N >= 16) v += lane_dpp<0x140>(v);
  return v;
}

// Sum over the workgroup's threads, returned to every thread; `red` (one double per wave) must not be in
// use.
__device__ __forceinline__ double tile_block_sum(double v, double *red) {
  static_assert(TILE_T / 64 == 8, "the waves' sums are added over 8 lanes");
  v = wave_sum_to_last(v);
  if ((threadIdx.x & 63) == 63) red[threadIdx.x >> 6] = v;
  __syncthreads();
  return tile_lane_sum<8>(red[threadIdx.x & 7]);
}

// Two sums behind one barrier.
__device__ __forceinline__ void tile_block_sum2(double &a, double &b, double *ra, double *rb) {
  a = wave_sum_to_last(a);
  b = wave_sum_to_last(b);
  if ((threadIdx.x & 63) == 63) {
    ra[threadIdx.x >> 6] = a;
    rb[threadIdx.x >> 6] = b;
  }
  __syncthreads();
  a = tile_lane_sum<8>(ra[threadIdx.x & 7]);
  b = tile_lane_sum<8>(rb[threadIdx.x & 7]);
}

// One lane's blocks of a node's rows: values, and the columns as node ids (the node itself past its last
// neighbour, with zero values).
template <class T, int P, int LPN>
__device__ __forceinline__ void tile_load(const TileArgs &A, long long node, int lane, T (&v)[TILE_U][P][P],
                                          int (&col)[TILE_U]) {
#pragma unroll
  for (int u = 0; u < TILE_U; ++u) {
    col[u] = (int)node;
#pragma unroll
    for (int c = 0; c < P; ++c)
#pragma unroll
      for (int e = 0; e < P; ++e) v[u][c][e] = T(0);
  }
  if (node >= A.nodes) return;
  long long rb[P];
#pragma unroll
  for (int c = 0; c < P; ++c) rb[c] = A.rp[node * P + c];
  const int deg = (int)((A.rp[node * P + 1] - rb[0]) / P);
#pragma unroll
  for (int u = 0; u < TILE_U; ++u) {
    const int k = lane + u * LPN;
    if (k < deg) {
      col[u] = A.ci[rb[0] + (long long)P * k] / P;
#pragma unroll
      for (int c = 0; c < P; ++c)
#pragma unroll
        for (int e = 0; e < P; ++e) v[u][c][e] = (T)A.vals[rb[c] + (long long)P * k + e];
    }
  }
}

// s += block . x, and the sum over the node's lanes (every lane holds it)
template <class T, int P>
__device__ __forceinline__ void tile_block(const T (&v)[P][P], const T (&x)[P], T (&s)[P]) {
#pragma unroll
  for (int c = 0; c < P; ++c)
#pragma unroll
    for (int e = 0; e < P; ++e) s[c] = __builtin_elementwise_fma(v[c][e], x[e], s[c]);
}
template <class T, int P, int LPN> __device__ __forceinline__ T tile_row(T (&s)[P], int lane) {
#pragma unroll
  for (int c = 0; c < P; ++c) s[c] = tile_lane_sum<LPN>(s[c]);
  T q = s[0];  // lane c of the node keeps component c
#pragma unroll
  for (int c = 1; c < P; ++c) q = lane == c ? s[c] : q;
  return q;
}
template <class T> __device__ __forceinline__ T tile_axpy(double a, T x, T y) {
  return (T)__builtin_fma(a, (double)x, (double)y);
}
template <class T> __device__ __forceinline__ T tile_dinv(const TileArgs &A, long long row) {
  const int o = A.doff[row];
  const double d = o >= 0 ? A.vals[A.rp[row] + o] : 0.0;
  return (T)(d != 0.0 ? 1.0 / d : 1.0);
}

template <class T, int P, int LPN, int S> struct Tile {
  static constexpr int NPW = TILE_T / LPN;  // nodes per pass
  static constexpr int NPB = NPW * S;       // nodes per workgroup
  // LDS of k_pcg_resident in bytes: p of the touched nodes, their ids, the rank table, the own dofs' x, r
  // and 1/diagonal
  static size_t lds(int cap) {
    return (size_t)cap * P * sizeof(T) + (size_t)cap * sizeof(int) + TILE_RANGE / 32 * (sizeof(unsigned) + 2) +
           3 * (size_t)NPB * P * sizeof(T) + 64;
  }
};

// The solve of A x = b in one launch.  What bounds it is the latency of its exchanges (about 1.3 us a hop
// between XCDs), then the LDS gathers of the SpMV; the matrix is read once.  512 threads at 256 VGPRs
// (one workgroup per CU) hold S x 4 blocks per lane; 1024 threads at 128 VGPRs spilled.  One iteration,
// four launched kernels -> here: quads 40 x 40 conduction FP64 17 -> 4.0 us, hexahedra 17 x 13 x 11 elastic
// FP64 18 -> 5.5 us, 43 x 37 x 29 mixed (its FP32 matrix, 46 MB, in 196 workgroups' registers) 22 -> 7.8 us.
template <class T, int P, int LPN, int S>
__global__ __launch_bounds__(TILE_T) void k_pcg_resident(TileArgs A) {
  using G_ = Tile<T, P, LPN, S>;
  constexpr int NPW = G_::NPW, NPB = G_::NPB;
  extern __shared__ __align__(16) unsigned char tile_smem[];
  __shared__ double red[7][TILE_T / 64];
  __shared__ int bad_s;
  T *const pl = reinterpret_cast<T *>(tile_smem);           // (cap, P) search direction
  T *const xs = pl + (size_t)A.cap * P;                     // own dofs
  T *const rs = xs + NPB * P;
  T *const ds = rs + NPB * P;
  int *const list = reinterpret_cast<int *>(ds + NPB * P);  // (cap) node ids, ascending
  unsigned *const bits = reinterpret_cast<unsigned *>(list + A.cap);
  unsigned short *const rank = reinterpret_cast<unsigned short *>(bits + TILE_RANGE / 32);
  const int tid = threadIdx.x, lane = tid % LPN, grp = tid / LPN, wg = blockIdx.x, G = A.G;
  const long long n0 = (long long)wg * NPB;
  T *const X = reinterpret_cast<T *>(A.x);
  const bool solo = G == 1;
  if (tid == 0) bad_s = 0;
  // the matrix, and the nodes its columns name: a bit per node id, the rank of a bit its place in LDS
  T v[S][TILE_U][P][P];
  int col[S][TILE_U];
  const long long base = max(0LL, n0 - A.bw), end = min(A.nodes, n0 + NPB + A.bw);
  const int words = (int)((end - base + 31) / 32);
  for (int w = tid; w < words; w += TILE_T) bits[w] = 0u;
  __syncthreads();
#pragma unroll
  for (int s = 0; s < S; ++s) {
    const long long node = n0 + s * NPW + grp;
    tile_load<T, P, LPN>(A, node, lane, v[s], col[s]);
    if (node < A.nodes) {
#pragma unroll
      for (int u = 0; u < TILE_U; ++u) {
        const int o = (int)(col[s][u] - base);
        atomicOr(&bits[o >> 5], 1u << (o & 31));
      }
    }
  }
  __syncthreads();
  int count;
  {  // exclusive prefix sums of the words' bit counts (WPT words per thread), then the id list
    constexpr int WPT = TILE_RANGE / 32 / TILE_T;
    __shared__ int wsum[TILE_T / 64];
    int mine = 0;
#pragma unroll
    for (int k = 0; k < WPT; ++k) mine += WPT * tid + k < words ? __popc(bits[WPT * tid + k]) : 0;
    int inc = mine;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int y = __shfl_up(inc, o);
      if ((tid & 63) >= o) inc += y;
    }
    if ((tid & 63) == 63) wsum[tid >> 6] = inc;
    __syncthreads();
    int at = inc - mine;
    count = 0;
    for (int k = 0; k < TILE_T / 64; ++k) {
      if (k < (tid >> 6)) at += wsum[k];
      count += wsum[k];
    }
    for (int k = WPT * tid; k < min(WPT * tid + WPT, words); ++k) {
      rank[k] = (unsigned short)at;
      for (unsigned m = bits[k]; m; m &= m - 1) list[at++] = (int)(base + (long long)k * 32 + __builtin_ctz(m));
    }
  }
  __syncthreads();
  auto place = [&](int c) {
    const int o = (int)(c - base);
    return (int)rank[o >> 5] + __popc(bits[o >> 5] & ((1u << (o & 31)) - 1u));
  };
  unsigned at[S][TILE_U / 2];  // two LDS places per register
  unsigned own[(S + 1) / 2];
#pragma unroll
  for (int s = 0; s < (S + 1) / 2; ++s) own[s] = 0u;
#pragma unroll
  for (int s = 0; s < S; ++s) {
    const long long node = n0 + s * NPW + grp;
    const bool in = node < A.nodes;
#pragma unroll
    for (int h = 0; h < TILE_U / 2; ++h)
      at[s][h] = in ? (unsigned)place(col[s][2 * h]) | (unsigned)place(col[s][2 * h + 1]) << 16 : 0u;
    own[s / 2] |= (in ? (unsigned)place((int)node) : 0u) << (16 * (s & 1));
  }
  // q of this lane's own dof of pass s, from the vector in pl
  auto spmv = [&](int s) {
    T sum[P];
#pragma unroll
    for (int c = 0; c < P; ++c) sum[c] = T(0);
#pragma unroll
    for (int u = 0; u < TILE_U; ++u) {
      const int o = (int)((at[s][u / 2] >> (16 * (u & 1))) & 0xffffu) * P;
      T xv[P];
#pragma unroll
      for (int e = 0; e < P; ++e) xv[e] = pl[o + e];
      tile_block<T, P>(v[s][u], xv, sum);
    }
    return tile_row<T, P, LPN>(sum, lane);
  };
  // r = b - A x, z = r / diagonal
  const int nh = count * P;
  for (int i = tid; i < nh; i += TILE_T) pl[i] = X[(long long)list[i / P] * P + i % P];
  __syncthreads();
  double rz = 0.0, rr = 0.0, bb = 0.0;
#pragma unroll
  for (int s = 0; s < S; ++s) {
    const T q = spmv(s);
    const long long node = n0 + s * NPW + grp;
    if (lane < P && node < A.nodes) {
      const long long row = node * P + lane;
      const int o = (s * NPW + grp) * P + lane;
      const double bi = A.b[row];
      const T d = tile_dinv<T>(A, row), r = (T)(bi - (double)q), z = r * d;
      xs[o] = X[row];
      rs[o] = r;
      ds[o] = d;
      rz = __builtin_fma((double)r, (double)z, rz);
      rr = __builtin_fma((double)r, (double)r, rr);
      bb = __builtin_fma(bi, bi, bb);
      if (!solo) tile_publish<T>(reinterpret_cast<T *>(A.z[0]) + row, z);
    }
  }
  double trz = rz, trr = rr, tbb = tile_block_sum(bb, red[2]);
  tile_block_sum2(trz, trr, red[0], red[1]);
  if (!solo && tid == 0) {
    tile_publish<double>(A.pa + wg, trz);
    tile_publish<double>(A.pa + G + wg, trr);
    tile_publish<double>(A.pa + 2 * G + wg, tbb);
  }
  for (int i = tid; i < nh; i += TILE_T) pl[i] = T(0);  // (every lane's SpMV reads precede the sums' barriers)
  __syncthreads();
  // the z this thread brings to LDS first (up to ZN values; further ones go through `list`)
  constexpr int ZN = 4;
  int zo[ZN];
#pragma unroll
  for (int j = 0; j < ZN; ++j) {
    const int i = min(tid + j * TILE_T, nh - 1);
    zo[j] = list[i / P] * P + i % P;
  }
  double rz_old = 0.0, bnorm = 0.0;
  int status = 0, k = 0, next = min(A.check, A.maxiter), bad = 0;
  for (;; ++k) {
    const int par = k & 1;
    const T *const zk = reinterpret_cast<const T *>(A.z[par]);
    typename TileBits<T>::U seen[ZN];
    // exchange A: r.z, r.r (and b.b) and z of the touched nodes, all looked at together (z was published
    // before the sums)
    if (!solo) {
      const double *pa = A.pa + (size_t)par * 3 * G;
      double pz = 0.0, pr = 0.0, pb = 0.0;
      unsigned long long s0 = 0, s1 = 0;
      if (tid < G) {
        s0 = tile_peek<double>(pa + tid);
        s1 = tile_peek<double>(pa + G + tid);
      }
#pragma unroll
      for (int j = 0; j < ZN; ++j) seen[j] = tile_peek<T>(zk + zo[j]);
      if (tid < G) {
        pz = tile_wait<double>(pa + tid, s0, A.looks, bad);
        pr = tile_wait<double>(pa + G + tid, s1, A.looks, bad);
        if (k == 0) pb = tile_wait<double>(pa + 2 * G + tid, ~0ull, A.looks, bad);
      }
      if (bad) bad_s = 1;
      if (k == 0) tbb = tile_block_sum(pb, red[2]);
      trz = pz;
      trr = pr;
      tile_block_sum2(trz, trr, red[0], red[1]);
      if (bad_s) break;
    }
    // the tests of the host-checked solve: at the start, every `check` iterations and at the last
    if (k == 0) {
      bnorm = A.bnorm >= 0.0 ? A.bnorm : sqrt(tbb);
      if (bnorm == 0.0 || sqrt(trr) / bnorm <= A.tol) status = 1;
    } else if (k == next) {
      next = min(next + A.check, A.maxiter);
      if (!(trr == trr && trr < INFINITY))
        status = 2;
      else if (sqrt(trr > 0.0 ? trr : 0.0) / bnorm <= A.tol)
        status = 1;
      else if (k == A.maxiter)
        status = 3;
    }
    if (status) break;
    const double beta = k ? trz / rz_old : 0.0;
    rz_old = trz;
    if (solo) {
#pragma unroll
      for (int s = 0; s < S; ++s) {
        const int g = s * NPW + grp, o = g * P + lane;
        if (lane < P && n0 + g < A.nodes) {
          const int pi = (int)((own[s / 2] >> (16 * (s & 1))) & 0xffffu) * P + lane;
          pl[pi] = tile_axpy<T>(beta, pl[pi], rs[o] * ds[o]);
        }
      }
    } else {
      if (tid == 0 && k > 0) tile_reset<double>(A.pc + (size_t)(1 - par) * G + wg);  // read by all before A
#pragma unroll
      for (int j = 0; j < ZN; ++j) {
        const int i = tid + j * TILE_T;
        if (i < nh) pl[i] = tile_axpy<T>(beta, pl[i], tile_wait<T>(zk + zo[j], seen[j], A.looks, bad));
      }
      for (int i0 = tid + ZN * TILE_T; i0 < nh; i0 += ZN * TILE_T) {
        const T *zr[ZN];
#pragma unroll
        for (int j = 0; j < ZN; ++j) {
          const int i = min(i0 + j * TILE_T, nh - 1);
          zr[j] = zk + (list[i / P] * P + i % P);
          seen[j] = tile_peek<T>(zr[j]);
        }
#pragma unroll
        for (int j = 0; j < ZN; ++j) {
          const int i = i0 + j * TILE_T;
          if (i < nh) pl[i] = tile_axpy<T>(beta, pl[i], tile_wait<T>(zr[j], seen[j], A.looks, bad));
        }
      }
    }
    __syncthreads();  // (a wait that ran out here is raised at exchange C: bad_s has readers until this barrier)
    T q[S];
    double pq = 0.0;
#pragma unroll
    for (int s = 0; s < S; ++s) {
      q[s] = spmv(s);
      const int g = s * NPW + grp;
      if (lane < P && n0 + g < A.nodes) {
        const int pi = (int)((own[s / 2] >> (16 * (s & 1))) & 0xffffu) * P + lane;
        pq = __builtin_fma((double)pl[pi], (double)q[s], pq);
      }
    }
    if (!solo) tile_stores_done();  // resets of the last phase precede this exchange
    double tpq = tile_block_sum(pq, red[3]);
    if (!solo) {  // exchange C: p.Ap
      double *pc = A.pc + (size_t)par * G;
      if (tid == 0) tile_publish<double>(pc + wg, tpq);
      double pp = 0.0;
      if (tid < G) pp = tile_wait<double>(pc + tid, ~0ull, A.looks, bad);
      if (bad) bad_s = 1;
      tpq = tile_block_sum(pp, red[4]);
      if (bad_s) break;
    }
    const double alpha = trz / tpq;
    rz = rr = 0.0;
    T *const zn = reinterpret_cast<T *>(A.z[1 - par]);
    T *const zp = reinterpret_cast<T *>(A.z[par]);
#pragma unroll
    for (int s = 0; s < S; ++s) {
      const int g = s * NPW + grp, o = g * P + lane;
      if (lane < P && n0 + g < A.nodes) {
        const int pi = (int)((own[s / 2] >> (16 * (s & 1))) & 0xffffu) * P + lane;
        const T r = tile_axpy<T>(-alpha, q[s], rs[o]), z = r * ds[o];
        if (!solo) tile_publish<T>(zn + (n0 + g) * P + lane, z);
        rs[o] = r;
        xs[o] = tile_axpy<T>(alpha, pl[pi], xs[o]);
        rz = __builtin_fma((double)r, (double)z, rz);
        rr = __builtin_fma((double)r, (double)r, rr);
        // every workgroup has read z of this iteration (it published p.Ap)
        if (!solo) tile_reset<T>(zp + (n0 + g) * P + lane);
      }
    }
    trz = rz;
    trr = rr;
    tile_block_sum2(trz, trr, red[5], red[6]);
    if (!solo && tid == 0) {
      double *pn = A.pa + (size_t)(1 - par) * 3 * G, *po = A.pa + (size_t)par * 3 * G;
      tile_publish<double>(pn + wg, trz);
      tile_publish<double>(pn + G + wg, trr);
      tile_reset<double>(po + wg);
      tile_reset<double>(po + G + wg);
    }
  }
  if (status == 0) {  // a wait ran out
    if (tid == 0) *A.fail = 1;
    return;
  }
#pragma unroll
  for (int s = 0; s < S; ++s) {
    const int g = s * NPW + grp;
    if (lane < P && n0 + g < A.nodes && k > 0) X[(n0 + g) * P + lane] = xs[g * P + lane];
  }
  if (wg == 0 && tid == 0) {
    A.st->status = status;
    A.st->iters = k;
    A.st->bnorm2 = A.bnorm >= 0.0 ? A.bnorm * A.bnorm : tbb;
    A.st->rr = trr;
  }
}

// Slots of the exchanges to the sentinel, the failure flag and the state cleared, x kept.
template <class T> __global__ __launch_bounds__(256) void k_tile_clear(TileArgs A, long long n) {
  using U = typename TileBits<T>::U;
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i < n) {
    reinterpret_cast<U *>(A.z[0])[i] = ~U(0);
    reinterpret_cast<U *>(A.z[1])[i] = ~U(0);
    reinterpret_cast<T *>(A.x0)[i] = reinterpret_cast<const T *>(A.x)[i];
  }
  if (i < 6 * A.G) reinterpret_cast<unsigned long long *>(A.pa)[i] = ~0ull;
  if (i < 2 * A.G) reinterpret_cast<unsigned long long *>(A.pc)[i] = ~0ull;
  if (i == 0) {
    *A.fail = 0;
    A.st->status = 0;
    A.st->iters = 0;
    A.st->bnorm2 = 0.0;
    A.st->rr = 0.0;
  }
}

// ---- the launched form (FP64) ---------------------------------------------------------------------
struct TileVecs {
  double *r, *z, *dinv, *q, *p[2];
};

// Sum of the G workgroups' partials, in the order of k_pcg_resident.
__device__ __forceinline__ double tile_sum_slots(const double *part, int G, double *red) {
  return tile_block_sum((int)threadIdx.x < G ? part[threadIdx.x] : 0.0, red);
}

template <int P, int LPN, int S, bool INIT>
__device__ __forceinline__ void tile_rows(const TileArgs &A, const TileVecs &V, int par, double beta, double (&q)[S],
                                          double (&own)[S]) {
  using G_ = Tile<double, P, LPN, S>;
  const int lane = threadIdx.x % LPN, grp = threadIdx.x / LPN;
  const long long n0 = (long long)blockIdx.x * G_::NPB;
  const double *X = reinterpret_cast<const double *>(A.x);
#pragma unroll
  for (int s = 0; s < S; ++s) {
    const long long node = n0 + s * G_::NPW + grp;
    double v[TILE_U][P][P], sum[P];
    int col[TILE_U];
    tile_load<double, P, LPN>(A, node, lane, v, col);
#pragma unroll
    for (int c = 0; c < P; ++c) sum[c] = 0.0;
#pragma unroll
    for (int u = 0; u < TILE_U; ++u) {
      const long long m = node < A.nodes ? col[u] : 0;
      double xv[P];
#pragma unroll
      for (int e = 0; e < P; ++e)
        xv[e] = INIT ? X[m * P + e] : tile_axpy<double>(beta, V.p[par][m * P + e], V.z[m * P + e]);
      tile_block<double, P>(v[u], xv, sum);
    }
    q[s] = tile_row<double, P, LPN>(sum, lane);
    own[s] = 0.0;
    if (!INIT && lane < P && node < A.nodes) {
      const long long row = node * P + lane;
      own[s] = tile_axpy<double>(beta, V.p[par][row], V.z[row]);
      V.p[1 - par][row] = own[s];
    }
  }
}

// r = b - A x, z, p = 0 and the first partials (parity 0)
template <int P, int LPN, int S> __global__ __launch_bounds__(TILE_T) void k_tile_init(TileArgs A, TileVecs V) {
  using G_ = Tile<double, P, LPN, S>;
  __shared__ double red[3][TILE_T / 64];
  const int lane = threadIdx.x % LPN, grp = threadIdx.x / LPN;
  double q[S], own[S], rz = 0.0, rr = 0.0, bb = 0.0;
  tile_rows<P, LPN, S, true>(A, V, 0, 0.0, q, own);
#pragma unroll
  for (int s = 0; s < S; ++s) {
    const long long node = (long long)blockIdx.x * G_::NPB + s * G_::NPW + grp;
    if (lane < P && node < A.nodes) {
      const long long row = node * P + lane;
      const double bi = A.b[row], d = tile_dinv<double>(A, row), r = bi - q[s], z = r * d;
      V.dinv[row] = d;
      V.r[row] = r;
      V.z[row] = z;
      V.p[0][row] = 0.0;
      rz = __builtin_fma(r, z, rz);
      rr = __builtin_fma(r, r, rr);
      bb = __builtin_fma(bi, bi, bb);
    }
  }
  rz = tile_block_sum(rz, red[0]);
  rr = tile_block_sum(rr, red[1]);
  bb = tile_block_sum(bb, red[2]);
  if (threadIdx.x == 0) {
    A.pa[blockIdx.x] = rz;
    A.pa[A.G + blockIdx.x] = rr;
    A.pa[2 * A.G + blockIdx.x] = bb;
  }
}

// The test of the enqueued solve, after `it` iterations.
__device__ __forceinline__ int tile_status(const TileArgs &A, double rr, double bb, int it) {
  if (!(rr == rr && rr < INFINITY)) return 2;
  if ((it == 0 && bb == 0.0) || rr <= A.tol * A.tol * bb) return 1;
  return it >= A.maxiter ? 3 : 0;
}

// Opens iteration k: every workgroup makes the test that precedes it (workgroup 0 records it; a workgroup that finds
// its record already there reads the decision it would make) and takes beta.  False: the solve has ended, for the
// whole workgroup: one thread reads the record, which may change between two waves' reads.  A kernel of its own for
// the test cost 2-3 us an iteration.
__device__ __forceinline__ bool tile_open(const TileArgs &A, int k, const int *outer, double (*red)[TILE_T / 64],
                                          double &beta) {
  __shared__ int ended;
  if (threadIdx.x == 0) ended = k > 0 ? A.st->status : 0;
  const int par = k & 1;
  const double *now = A.pa + (size_t)par * 3 * A.G, *before = A.pa + (size_t)(1 - par) * 3 * A.G;
  const double rr = tile_sum_slots(now + A.G, A.G, red[0]);  // (its barrier shows `ended` to all)
  if (ended) return false;
  const double bb = k == 0 ? tile_sum_slots(now + 2 * A.G, A.G, red[1]) : A.st->bnorm2;
  const int status = k == 0 && outer && *outer ? 4 : tile_status(A, rr, bb, k);
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    if (k == 0) A.st->bnorm2 = bb;
    A.st->rr = rr;
    A.st->iters = k;
    A.st->status = status;
  }
  if (status) return false;
  beta = k == 0 ? 0.0 : tile_sum_slots(now, A.G, red[2]) / tile_sum_slots(before, A.G, red[3]);
  return true;
}

// This workgroup's sums of a b and of b b over its dofs, in the order of k_pcg_resident (a thread's S products, then
// the workgroup's), from LDS, where the dofs are brought by all lanes: LPN - P of LPN lanes own none.
template <int P, int LPN, int S, bool BOTH>
__device__ __forceinline__ void tile_products(const TileArgs &A, const double *a, const double *b, double &ab,
                                              double &bb) {
  using G_ = Tile<double, P, LPN, S>;
  const int lane = threadIdx.x % LPN, grp = threadIdx.x / LPN;
  ab = bb = 0.0;
#pragma unroll
  for (int s = 0; s < S; ++s) {
    const int g = s * G_::NPW + grp;
    if (lane < P && (long long)blockIdx.x * G_::NPB + g < A.nodes) {
      ab = __builtin_fma(b[g * P + lane], a[g * P + lane], ab);
      if (BOTH) bb = __builtin_fma(b[g * P + lane], b[g * P + lane], bb);
    }
  }
}

// Iteration k: p = z + beta p (p[par] -> p[1 - par]), q = A p, partials of p.q
template <int P, int LPN, int S>
__global__ __launch_bounds__(TILE_T) void k_tile_spmv(TileArgs A, TileVecs V, int k, const int *outer) {
  using G_ = Tile<double, P, LPN, S>;
  __shared__ double red[5][TILE_T / 64];
  const int lane = threadIdx.x % LPN, grp = threadIdx.x / LPN;
  double beta;
  if (!tile_open(A, k, outer, red, beta)) return;
  double q[S], own[S], pq = 0.0;
  tile_rows<P, LPN, S, false>(A, V, k & 1, beta, q, own);
#pragma unroll
  for (int s = 0; s < S; ++s) {
    const long long node = (long long)blockIdx.x * G_::NPB + s * G_::NPW + grp;
    if (lane < P && node < A.nodes) {
      V.q[node * P + lane] = q[s];
      pq = __builtin_fma(own[s], q[s], pq);
    }
  }
  pq = tile_block_sum(pq, red[4]);
  if (threadIdx.x == 0) A.pc[blockIdx.x] = pq;
}

// The same in two kernels: a workgroup per pass, then the partials of p.q.  For many passes of one dof per node
// (see pcg_async_core).
template <int P, int LPN>
__global__ __launch_bounds__(TILE_T) void k_tile_pass(TileArgs A, TileVecs V, int k, const int *outer) {
  __shared__ double red[4][TILE_T / 64];
  const int lane = threadIdx.x % LPN, grp = threadIdx.x / LPN;
  double beta;
  if (!tile_open(A, k, outer, red, beta)) return;
  double q[1], own[1];
  tile_rows<P, LPN, 1, false>(A, V, k & 1, beta, q, own);
  const long long node = (long long)blockIdx.x * (TILE_T / LPN) + grp;
  if (lane < P && node < A.nodes) V.q[node * P + lane] = q[0];
}
template <int P, int LPN, int S> __global__ __launch_bounds__(TILE_T) void k_tile_dot(TileArgs A, TileVecs V, int par) {
  constexpr int N = Tile<double, P, LPN, S>::NPB * P;
  if (A.st->status) return;
  __shared__ double red[TILE_T / 64], p[N], q[N];
  const long long r0 = (long long)blockIdx.x * N, n = A.nodes * P;
#pragma unroll
  for (int i = threadIdx.x; i < N; i += TILE_T) {
    p[i] = r0 + i < n ? V.p[1 - par][r0 + i] : 0.0;
    q[i] = r0 + i < n ? V.q[r0 + i] : 0.0;
  }
  __syncthreads();
  double pq, unused;
  tile_products<P, LPN, S, false>(A, q, p, pq, unused);
  pq = tile_block_sum(pq, red);
  if (threadIdx.x == 0) A.pc[blockIdx.x] = pq;
}

// x += alpha p, r -= alpha q, z, partials of parity 1 - par
template <int P, int LPN, int S>
__global__ __launch_bounds__(TILE_T) void k_tile_update(TileArgs A, TileVecs V, int par) {
  constexpr int N = Tile<double, P, LPN, S>::NPB * P, K = (N + TILE_T - 1) / TILE_T;
  if (A.st->status) return;
  __shared__ double red[4][TILE_T / 64], rl[N], zl[N];
  const double top = tile_sum_slots(A.pa + (size_t)par * 3 * A.G, A.G, red[0]);
  const double alpha = top / tile_sum_slots(A.pc, A.G, red[1]);
  double *X = reinterpret_cast<double *>(A.x), x[K], r[K], z[K];
  const long long r0 = (long long)blockIdx.x * N, n = A.nodes * P;
#pragma unroll
  for (int j = 0; j < K; ++j) {  // (all loads before the first store, which they might alias)
    const int i = threadIdx.x + j * TILE_T;
    const long long row = min(r0 + min(i, N - 1), n - 1);
    x[j] = tile_axpy<double>(alpha, V.p[1 - par][row], X[row]);
    r[j] = tile_axpy<double>(-alpha, V.q[row], V.r[row]);
    z[j] = r[j] * V.dinv[row];
  }
#pragma unroll
  for (int j = 0; j < K; ++j) {
    const int i = threadIdx.x + j * TILE_T;
    if (i < N) {
      rl[i] = r[j];
      zl[i] = z[j];
      if (r0 + i < n) {
        X[r0 + i] = x[j];
        V.r[r0 + i] = r[j];
        V.z[r0 + i] = z[j];
      }
    }
  }
  __syncthreads();
  double rz, rr;
  tile_products<P, LPN, S, true>(A, zl, rl, rz, rr);
  rz = tile_block_sum(rz, red[2]);
  rr = tile_block_sum(rr, red[3]);
  if (threadIdx.x == 0) {
    A.pa[(size_t)(1 - par) * 3 * A.G + blockIdx.x] = rz;
    A.pa[(size_t)(1 - par) * 3 * A.G + A.G + blockIdx.x] = rr;
  }
}

// The test after the last iteration
static __global__ __launch_bounds__(TILE_T) void k_tile_test(TileArgs A, int it) {
  if (A.st->status) return;
  __shared__ double red[TILE_T / 64];
  const double rr = tile_sum_slots(A.pa + (size_t)(it & 1) * 3 * A.G + A.G, A.G, red);
  if (threadIdx.x == 0) {
    A.st->rr = rr;
    A.st->iters = it;
    A.st->status = tile_status(A, rr, A.st->bnorm2, it);
  }
}

}  // namespace femhot
