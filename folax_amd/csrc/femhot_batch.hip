// Whole training-loss calls: the Dirichlet values set, the residual or energies of a batch, and the scalar
// loss, in one entry point (fol/loss_functions/fe_loss.py:91-100, 250-262), and the scaling of their
// gradients.  A training step on a small or medium mesh is bound by its launches and the host work
// around them, not by the element kernels; these entry points leave 4-5 launches to a forward pass and
// 1-2 to a backward pass, where torch's operators around the kernels took about 25 in all.  Forward and
// backward of quads 128 x 128 x 64 thermal FP32: 284 -> 167 us; quads 10 x 10 elastic FP64: 281 -> 155;
// hexahedra 48^3 x 16 Neo-Hookean FP32: 785 -> 354 (the forward residual is kept as the gradient, so the
// backward pass no longer runs the element kernel again).
#include <algorithm>

#include "femhot_kernels.h"

namespace femhot {

constexpr int BATCH_PARTS = 256;  // partial sums of the squared residual

// full = u with the Dirichlet dofs at their values; one sample per blockIdx.y.  HBM-bound (read u, write
// full).
template <class R>
__global__ __launch_bounds__(256) void k_full_dofs(long long n, const R *u, long long us, R *full,
                                                   const uint8_t *dmask, const double *dval) {
  u += (long long)blockIdx.y * us;
  full += (long long)blockIdx.y * n;
  for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long long)gridDim.x * 256)
    full[i] = dmask[i] ? (R)dval[i] : u[i];
}

// FP64 sums of the squares of v, one per workgroup, then the half of their sum (fixed orders).
template <class R> __global__ __launch_bounds__(256) void k_square_parts(long long n, const R *v, double *part) {
  __shared__ double red[4];
  double s = 0.0;
  const long long st = (long long)gridDim.x * 256;
  long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  for (; i + 3 * st < n; i += 4 * st) {  // four loads in flight
    const double a = (double)v[i], b = (double)v[i + st], c = (double)v[i + 2 * st], d = (double)v[i + 3 * st];
    s += a * a;
    s += b * b;
    s += c * c;
    s += d * d;
  }
  for (; i < n; i += st) s += (double)v[i] * (double)v[i];
  s = wave_sum(s);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) part[blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
}
template <class R> __global__ __launch_bounds__(256) void k_half_sum(const double *part, int n, R *loss) {
  __shared__ double red[4];
  double s = (int)threadIdx.x < n ? part[threadIdx.x] : 0.0;
  s = wave_sum(s);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) loss[0] = (R)(0.5 * ((red[0] + red[1]) + (red[2] + red[3])));
}

// mean, min and max over the samples of the energies summed over each sample's segments
template <class R>
__global__ __launch_bounds__(256) void k_batch_stats(int batch, int nseg, const double *energy, R *mean, R *low,
                                                     R *high) {
  __shared__ double rs[4], rl[4], rh[4];
  double s = 0.0, lo = INFINITY, hi = -INFINITY;
  bool nan = false;
  for (int b = threadIdx.x; b < batch; b += 256) {
    double e = 0.0;
    for (int k = 0; k < nseg; ++k) e += energy[(long long)b * nseg + k];
    s += e;
    lo = e < lo ? e : lo;
    hi = e > hi ? e : hi;
    nan = nan || e != e;
  }
  nan = __syncthreads_or(nan);  // as torch.min and torch.max, a NaN is the result
  s = wave_sum(s);
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    const double l = __shfl_xor(lo, off), h = __shfl_xor(hi, off);
    lo = l < lo ? l : lo;
    hi = h > hi ? h : hi;
  }
  if ((threadIdx.x & 63) == 0) rs[threadIdx.x >> 6] = s, rl[threadIdx.x >> 6] = lo, rh[threadIdx.x >> 6] = hi;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int k = 1; k < 4; ++k) {
      rl[0] = rl[k] < rl[0] ? rl[k] : rl[0];
      rh[0] = rh[k] > rh[0] ? rh[k] : rh[0];
    }
    mean[0] = (R)(((rs[0] + rs[1]) + (rs[2] + rs[3])) / batch);
    low[0] = nan ? (R)NAN : (R)rl[0];
    high[0] = nan ? (R)NAN : (R)rh[0];
  }
}

// dst = src * (factor * g), g on the device
template <class R>
__global__ __launch_bounds__(256) void k_scale(long long n, const R *src, const R *g, double factor, R *dst) {
  const R f = (R)(factor * (double)g[0]);
  for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long long)gridDim.x * 256)
    dst[i] = src[i] * f;
}

template <class R>
static int full_dofs(Ctx *c, int batch, const void *u, long long us, void *full, hipStream_t s) {
  const unsigned per = (unsigned)std::min<long long>((c->Ndof + 1023) / 1024, 4096);
  hipLaunchKernelGGL((k_full_dofs<R>), dim3(per, batch), dim3(256), 0, s, c->Ndof, (const R *)u,
                     batch > 1 ? us : c->Ndof, (R *)full, c->d_dmask, c->d_dval64);
  FH_HIP(hipGetLastError());
  return FEMHOT_OK;
}

static int check_batch(const Ctx *c, int dtype, int batch, const void *field, const void *u, long long us) {
  FH_CHECK_ARG(dtype == FEMHOT_F32 || dtype == FEMHOT_F64, FEMHOT_ERR_ARG, "dtype must be F32 or F64");
  FH_CHECK_ARG(batch >= 1 && batch <= 65535, FEMHOT_ERR_SHAPE, "batch must be in [1, 65535]");
  FH_CHECK_ARG(field && u, FEMHOT_ERR_ARG, "null field/u");
  FH_CHECK_ARG(batch == 1 || us >= c->Ndof, FEMHOT_ERR_SHAPE, "input stride smaller than n_dofs");
  return FEMHOT_OK;
}

}  // namespace femhot

using namespace femhot;

extern "C" int femhot_batch_residual_norm(femhot_ctx *h, int dtype, int batch, const void *field, long long fs,
                                          const void *u, long long us, void *full, void *R, void *loss,
                                          double *scratch, unsigned flags, void *stream) {
  FH_CHECK_ARG(h && full && R && loss && scratch, FEMHOT_ERR_ARG, "null argument");
  Ctx *c = &h->c;
  hipStream_t s = (hipStream_t)stream;
  int rc = check_batch(c, dtype, batch, field, u, us);
  if (rc) return rc;
  rc = dtype == FEMHOT_F32 ? full_dofs<float>(c, batch, u, us, full, s) : full_dofs<double>(c, batch, u, us, full, s);
  if (rc) return rc;
  if ((rc = femhot_residual(h, dtype, batch, field, fs, full, c->Ndof, R, c->Ndof, nullptr,
                            (flags & ~FEMHOT_ACCUMULATE) | FEMHOT_MASK_DIRICHLET, stream)))
    return rc;
  const long long n = c->Ndof * batch;
  const int parts = (int)std::min<long long>(BATCH_PARTS, (n + 2047) / 2048);
  if (dtype == FEMHOT_F32) {
    hipLaunchKernelGGL((k_square_parts<float>), dim3(parts), dim3(256), 0, s, n, (const float *)R, scratch);
    hipLaunchKernelGGL((k_half_sum<float>), dim3(1), dim3(256), 0, s, scratch, parts, (float *)loss);
  } else {
    hipLaunchKernelGGL((k_square_parts<double>), dim3(parts), dim3(256), 0, s, n, (const double *)R, scratch);
    hipLaunchKernelGGL((k_half_sum<double>), dim3(1), dim3(256), 0, s, scratch, parts, (double *)loss);
  }
  FH_HIP(hipGetLastError());
  return FEMHOT_OK;
}

extern "C" int femhot_batch_loss(femhot_ctx *h, int dtype, int batch, const void *field, long long fs, const void *u,
                                 long long us, void *full, void *R, double *energy, void *mean, void *low, void *high,
                                 unsigned flags, void *stream) {
  FH_CHECK_ARG(h && full && energy && mean && low && high, FEMHOT_ERR_ARG, "null argument");
  Ctx *c = &h->c;
  hipStream_t s = (hipStream_t)stream;
  int rc = check_batch(c, dtype, batch, field, u, us);
  if (rc) return rc;
  rc = dtype == FEMHOT_F32 ? full_dofs<float>(c, batch, u, us, full, s) : full_dofs<double>(c, batch, u, us, full, s);
  if (rc) return rc;
  if ((rc = femhot_residual(h, dtype, batch, field, fs, full, c->Ndof, R, c->Ndof, energy,
                            (flags & ~FEMHOT_ACCUMULATE) | FEMHOT_MASK_DIRICHLET, stream)))
    return rc;
  if (dtype == FEMHOT_F32)
    hipLaunchKernelGGL((k_batch_stats<float>), dim3(1), dim3(256), 0, s, batch, c->nseg, energy, (float *)mean,
                       (float *)low, (float *)high);
  else
    hipLaunchKernelGGL((k_batch_stats<double>), dim3(1), dim3(256), 0, s, batch, c->nseg, energy, (double *)mean,
                       (double *)low, (double *)high);
  FH_HIP(hipGetLastError());
  return FEMHOT_OK;
}

extern "C" int femhot_scale(int dtype, long long n, const void *src, const void *g, double factor, void *dst,
                            void *stream) {
  FH_CHECK_ARG(dtype == FEMHOT_F32 || dtype == FEMHOT_F64, FEMHOT_ERR_ARG, "dtype must be F32 or F64");
  FH_CHECK_ARG(src && g && dst && n >= 0, FEMHOT_ERR_ARG, "null argument");
  if (!n) return FEMHOT_OK;
  hipStream_t s = (hipStream_t)stream;
  const dim3 grid((unsigned)std::min<long long>((n + 1023) / 1024, 8192));
  if (dtype == FEMHOT_F32)
    hipLaunchKernelGGL((k_scale<float>), grid, dim3(256), 0, s, n, (const float *)src, (const float *)g, factor,
                       (float *)dst);
  else
    hipLaunchKernelGGL((k_scale<double>), grid, dim3(256), 0, s, n, (const double *)src, (const double *)g, factor,
                       (double *)dst);
  FH_HIP(hipGetLastError());
  return FEMHOT_OK;
}
