// Vector kernels of the solvers: BLAS-1 updates, deterministic reductions, constraint
// helpers and the geometric multigrid transfers.
//
// Reductions are two-stage with a fixed grid, so a dot product gives the same bits on
// every run (the reference's MPI_Allreduce-based dots are deterministic for a fixed
// rank count too).
#pragma once

#include "device.hpp"
#include "grid.hpp"
#include "host_scalars.hpp"

#include <algorithm>
#include <cmath>

namespace ppf
{
  constexpr int reduce_threads = 256;
  constexpr int reduce_blocks  = 1024;

  template <typename T>
  __device__ PPF_INLINE double
  wave_sum(double v)
  {
    for (int off = warpSize / 2; off > 0; off /= 2)
      v += __shfl_down(v, off, warpSize);
    return v;
  }

  /// Block-level sum of one double per thread; valid in thread 0.
  __device__ PPF_INLINE double
  block_sum(double v)
  {
    __shared__ double partial[reduce_threads / 32];
    v             = wave_sum<double>(v);
    const int lane = threadIdx.x % warpSize;
    const int wave = threadIdx.x / warpSize;
    if (lane == 0)
      partial[wave] = v;
    __syncthreads();
    double r = 0.0;
    if (threadIdx.x == 0)
      for (int w = 0; w < int(blockDim.x) / warpSize; ++w)
        r += partial[w];
    return r;
  }

  /// Block-level maximum of one double per thread; valid in thread 0.
  __device__ PPF_INLINE double
  block_max(double v)
  {
    __shared__ double partial[reduce_threads / 32];
    for (int o = warpSize / 2; o > 0; o /= 2)
      v = fmax(v, __shfl_xor(v, o));
    const int lane = threadIdx.x % warpSize;
    const int wave = threadIdx.x / warpSize;
    if (lane == 0)
      partial[wave] = v;
    __syncthreads();
    double r = 0.0;
    if (threadIdx.x == 0)
      for (int w = 0; w < int(blockDim.x) / warpSize; ++w)
        r = fmax(r, partial[w]);
    return r;
  }

  /// Vectors to compare: one pair per field of a block.
  template <typename T>
  struct ComparedFields
  {
    const T *a[PPF_MAX_FIELDS];
    const T *b[PPF_MAX_FIELDS];
  };

  /// Per-block max |a - b| (NaN or infinite counted as +inf) and max |b| of a field, into
  /// partial[i] and partial[all + i] for block i of all.  Grid: x over the vectors, y the fields.
  template <typename T>
  __global__ void __launch_bounds__(reduce_threads)
  max_diff_partial_kernel(double *__restrict__ partial, const ComparedFields<T> f, int64_t n)
  {
    const T *__restrict__ a = f.a[blockIdx.y];
    const T *__restrict__ b = f.b[blockIdx.y];
    double d = 0.0, m = 0.0;
    for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
         i += int64_t(gridDim.x) * blockDim.x)
      {
        const double e = fabs(double(a[i]) - double(b[i]));
        d              = e <= d ? d : (e == e && e < INFINITY ? e : INFINITY);
        m              = fmax(m, fabs(double(b[i])));
      }
    d = block_max(d);
    __syncthreads();
    m = block_max(m);
    if (threadIdx.x == 0)
      {
        const int i = int(blockIdx.x + gridDim.x * blockIdx.y);
        partial[i]  = d;
        partial[int(gridDim.x * gridDim.y) + i] = m;
      }
  }

  /// 16 bytes of a vector, at any element's address (block vectors and lattice planes of odd
  /// length start at no better alignment; global memory takes such loads).
  template <typename T>
  struct Pack
  {
    static constexpr int n = 16 / int(sizeof(T));
    typedef T            type __attribute__((vector_size(16), aligned(sizeof(T))));
  };

  template <typename T>
  __global__ void
  fill_kernel(T *__restrict__ x, T value, int64_t n)
  {
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n)
      x[i] = value;
  }

  /// dst = src converted; a no-op once *halt is set (halt may be null).
  template <typename T, typename U>
  __global__ void
  convert_kernel(T *__restrict__ dst, const U *__restrict__ src, int64_t n, const int *halt)
  {
    if (halt && *reinterpret_cast<const volatile int *>(halt))
      return;
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n)
      dst[i] = T(src[i]);
  }

  /// y = a*x + b*y, 16 bytes per thread (one FP32 element per thread reached 3.4 TB/s at
  /// 257^3 nodes).  b = 0 overwrites y without reading it (y may hold anything, NaN included).
  template <typename T>
  __global__ void
  axpby_kernel(T *__restrict__ y, T a, const T *__restrict__ x, T b, int64_t n)
  {
    using P         = typename Pack<T>::type;
    const int64_t i = (int64_t(blockIdx.x) * blockDim.x + threadIdx.x) * Pack<T>::n;
    if (i + Pack<T>::n <= n)
      {
        const P xv = *reinterpret_cast<const P *>(x + i);
        P      *yp = reinterpret_cast<P *>(y + i);
        *yp = b == T(0) ? a * xv : a * xv + b * *yp;
      }
    else
      for (int64_t k = i; k < n; ++k)
        y[k] = b == T(0) ? a * x[k] : a * x[k] + b * y[k];
  }

  /// y = b*y (in place; one array, so no aliasing of restrict-qualified operands)
  template <typename T>
  __global__ void
  scale_kernel(T *__restrict__ y, T b, int64_t n)
  {
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n)
      y[i] = b * y[i];
  }

  /// z = x - y
  template <typename T>
  __global__ void
  sub_kernel(T *__restrict__ z, const T *__restrict__ x, const T *__restrict__ y, int64_t n)
  {
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n)
      z[i] = x[i] - y[i];
  }

  /// y = d .* x (diagonal preconditioner application)
  template <typename T>
  __global__ void
  diag_mult_kernel(T *__restrict__ y, const T *__restrict__ d, const T *__restrict__ x,
                   int64_t n)
  {
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n)
      y[i] = d[i] * x[i];
  }

  /// inv = 1/d with zero entries mapped to 1 (reference mf_operator.cc:98-100,245-255).
  template <typename T>
  __global__ void
  invert_diagonal_kernel(T *__restrict__ inv, const T *__restrict__ d, int64_t n)
  {
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n)
      inv[i] = d[i] == T(0) ? T(1) : T(1) / d[i];
  }

  /// Start vector of the eigenvalue estimate: splitmix64 of the index, uniform in
  /// [-0.5, 0.5) (integer mixing and exact 53-bit scaling: the same values as on a CPU).
  template <typename T>
  __global__ void
  splitmix_fill_kernel(T *__restrict__ x, int64_t n)
  {
    for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
         i += int64_t(gridDim.x) * blockDim.x)
      {
        uint64_t z = uint64_t(i) + 0x9e3779b97f4a7c15ull;
        z          = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
        z          = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
        z ^= z >> 31;
        x[i] = T(double(z >> 11) * (1.0 / 9007199254740992.0) - 0.5);
      }
  }

  /// Stage 1 of a dot product: one partial per block (grid-stride, fixed grid).
  template <typename T>
  __global__ void __launch_bounds__(reduce_threads)
  dot_partial_kernel(double *__restrict__ partial, const T *__restrict__ x,
                     const T *__restrict__ y, int64_t n)
  {
    double s = 0.0;
    for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
         i += int64_t(gridDim.x) * blockDim.x)
      s += double(x[i]) * double(y[i]);
    s = block_sum(s);
    if (threadIdx.x == 0)
      partial[blockIdx.x] = s;
  }

  /// Stage 2: sums `count` partials in a fixed order into out[slot].
  __global__ void __launch_bounds__(reduce_threads)
  reduce_partials_kernel(double *__restrict__ out, const double *__restrict__ partial,
                         int count)
  {
    double s = 0.0;
    for (int i = threadIdx.x; i < count; i += blockDim.x)
      s += partial[i];
    s = block_sum(s);
    if (threadIdx.x == 0)
      out[0] = s;
  }

  // ---------------------------------------------------- device-side CG scalars
  //
  // Small CG loops (eigenvalue estimates, coarse-grid solves) keep their scalars in
  // device memory: dot products land in slots, alpha and beta are formed in the update
  // kernels with the same expressions the host loop uses, and the host reads the slots
  // once per estimate or every few coarse iterations instead of three times per step.

  /// Iteration i of the eigenvalue estimate is valid if rz and pAp stayed positive up
  /// to and including i (the host loop stops at the first that does not).
  __device__ inline bool
  eig_valid(const double *rz, const double *pap, int i)
  {
    for (int j = 0; j <= i; ++j)
      if (!(rz[j] > 0.0) || !(pap[j] > 0.0))
        return false;
    return true;
  }

  /// r = (-alpha) ap + r with alpha = rz_i / pAp_i, if iteration i is valid.
  template <typename T>
  __global__ void
  eig_r_update_kernel(T *__restrict__ r, const T *__restrict__ ap, const double *rz,
                      const double *pap, int i, int64_t n)
  {
    if (!eig_valid(rz, pap, i))
      return;
    const double  alpha = rz[i] / pap[i];
    const int64_t k     = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (k < n)
      r[k] = T(-alpha) * ap[k] + T(1) * r[k];
  }

  /// p = z + beta p with beta = rz_{i+1} / rz_i, if iteration i is valid.
  template <typename T>
  __global__ void
  eig_p_update_kernel(T *__restrict__ p, const T *__restrict__ z, const double *rz,
                      const double *pap, int i, int64_t n)
  {
    if (!eig_valid(rz, pap, i))
      return;
    const double  beta = rz[i + 1] / rz[i];
    const int64_t k    = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (k < n)
      p[k] = T(1) * z[k] + T(beta) * p[k];
  }

  /// Slots of the coarse CG: |r0|^2, rz (two parities), pAp, |r|^2; flag[0] = done.
  enum CoarseSlot : int
  {
    cs_r0sq = 0,
    cs_rz   = 1,
    cs_pap  = 3,
    cs_rr   = 4
  };

  __global__ void
  coarse_cg_start_kernel(const double *s, int *flag)
  {
    flag[0] = s[cs_r0sq] > 0.0 ? 0 : 1;
  }

  /// x = alpha p + x, r = (-alpha) ap + r with alpha = rz / pAp, unless done.
  __global__ void
  coarse_cg_xr_kernel(double *__restrict__ x, double *__restrict__ r, const double *__restrict__ p,
                      const double *__restrict__ ap, const double *s, const int *flag, int par,
                      int64_t n)
  {
    if (flag[0])
      return;
    const double  alpha = s[cs_rz + par] / s[cs_pap];
    const int64_t k     = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (k < n)
      {
        x[k] = alpha * p[k] + 1.0 * x[k];
        r[k] = (-alpha) * ap[k] + 1.0 * r[k];
      }
  }

  /// Marks the solve done once |r| <= tol |r0|.
  __global__ void
  coarse_cg_check_kernel(const double *s, int *flag, double tol)
  {
    if (!flag[0] && std::sqrt(s[cs_rr]) <= tol * std::sqrt(s[cs_r0sq]))
      flag[0] = 1;
  }

  /// p = z + beta p with beta = rz_new / rz, unless done.
  __global__ void
  coarse_cg_p_kernel(double *__restrict__ p, const double *__restrict__ z, const double *s,
                     const int *flag, int par, int64_t n)
  {
    if (flag[0])
      return;
    const double  beta = s[cs_rz + (par ^ 1)] / s[cs_rz + par];
    const int64_t k    = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (k < n)
      p[k] = 1.0 * z[k] + beta * p[k];
  }

  // ---------------------------------------------------------------- CG iteration
  //
  // A step is: operator application, d.Ad partial sums (by the operator's own launch where
  // that takes them), cg_step_kernel, and either cg_turn_kernel (no preconditioner: h = g) or
  // reduce_to_host_kernel, preconditioner, g.h partial sums and cg_direction_kernel.  Sums
  // that only the device needs have no kernel that finishes them: every workgroup of the
  // kernel that uses a dot product adds the few hundred partial sums itself, in one fixed
  // order (8 kB from L2; a reduction kernel of its own costs a launch, about 5 us of a 45 us
  // step at 140k nodes).  The residual norm goes to pinned host memory, which the host polls,
  // so that no copy or stream synchronization ends a step.

  /// Workgroups (and partial sums) of the kernels below for vectors of length n: one element
  /// per thread until every compute unit has a workgroup (with four, 66k elements used 65 of
  /// them: cg_step_kernel 5.7 us, now 4.1), then four elements per thread, since each
  /// workgroup adds all partial sums (a CG step on 417k elements: 34.6 us with 407
  /// workgroups, 35.1 us with 1024).
  inline unsigned int
  cg_grid(int64_t n)
  {
    const int64_t one = (n + reduce_threads - 1) / reduce_threads, four = (n + 1023) / 1024;
    return unsigned(std::min<int64_t>(
      std::max<int64_t>({four, std::min<int64_t>(one, 256), int64_t(1)}), reduce_blocks));
  }

  /// Sum of one double per thread in every thread of the block.
  __device__ PPF_INLINE double
  block_total(double v)
  {
    __shared__ double total;
    v = block_sum(v);
    if (threadIdx.x == 0)
      total = v;
    __syncthreads();
    v = total;
    __syncthreads();
    return v;
  }

  /// Sum of `count` partial sums, the same bits in every thread of every block.
  __device__ PPF_INLINE double
  sum_partials(const double *__restrict__ partial, int count)
  {
    double s = 0.0;
    for (int i = threadIdx.x; i < count; i += reduce_threads)
      s += partial[i];
    return block_total(s);
  }

  /// Sends a scalar to the polling host.
  __device__ PPF_INLINE void
  tell_host(HostScalar *to, double value, unsigned int tag, bool flag)
  {
    *reinterpret_cast<volatile double *>(&to->value) = value;
    __threadfence_system();
    *reinterpret_cast<volatile unsigned int *>(&to->word) = (tag << 1) | (flag ? 1u : 0u);
  }

  /// Sums `count` partials and tells the host.
  __global__ void __launch_bounds__(reduce_threads)
  reduce_to_host_kernel(HostScalar *to, const double *__restrict__ partial, int count,
                        unsigned int tag)
  {
    const double s = sum_partials(partial, count);
    if (threadIdx.x == 0)
      tell_host(to, s, tag, false);
  }

  /// Tells the host the maxima of both halves of 2 * count partials; launched as one workgroup.
  __global__ void __launch_bounds__(reduce_threads)
  max_to_host_kernel(HostScalar *first, unsigned int first_tag, HostScalar *second,
                     unsigned int second_tag, const double *__restrict__ partial, int count)
  {
    double d = 0.0, m = 0.0;
    for (int i = threadIdx.x; i < count; i += reduce_threads)
      {
        d = fmax(d, partial[i]);
        m = fmax(m, partial[count + i]);
      }
    d = block_max(d);
    __syncthreads();
    m = block_max(m);
    if (threadIdx.x == 0)
      {
        tell_host(first, d, first_tag, false);
        tell_host(second, m, second_tag, false);
      }
  }

  /// Per-block partial sums of x.y; nothing once *done is set (done may be null).
  template <typename T>
  __global__ void __launch_bounds__(reduce_threads)
  cg_dot_kernel(double *__restrict__ partial, const double *__restrict__ x,
                const T *__restrict__ y, int64_t n, const int *done)
  {
    if (done && *done)
      return;
    double s = 0.0;
    for (int64_t i = int64_t(blockIdx.x) * reduce_threads + threadIdx.x; i < n;
         i += int64_t(gridDim.x) * reduce_threads)
      s += x[i] * double(y[i]);
    s = block_sum(s);
    if (threadIdx.x == 0)
      partial[blockIdx.x] = s;
  }

  /// x += alpha d, g += alpha Ad with alpha = s[cur] / (d.Ad), and partial sums of g.g; the
  /// new g also goes to `gt` (the preconditioner's copy, in its precision) unless null.
  template <typename T>
  __global__ void __launch_bounds__(reduce_threads)
  cg_step_kernel(double *__restrict__ partial_gg, double *__restrict__ x,
                 double *__restrict__ g, T *__restrict__ gt, const double *__restrict__ d,
                 const double *__restrict__ ad, const double *__restrict__ s, int cur,
                 const double *__restrict__ partial_dad, int count, int64_t n, const int *done)
  {
    if (done && *done)
      return;
    const double alpha = s[cur] / sum_partials(partial_dad, count);
    double       acc   = 0.0;
    for (int64_t i = int64_t(blockIdx.x) * reduce_threads + threadIdx.x; i < n;
         i += int64_t(gridDim.x) * reduce_threads)
      {
        x[i] += alpha * d[i];
        const double gi = g[i] + alpha * ad[i];
        g[i]            = gi;
        if (gt)
          gt[i] = T(gi);
        acc += gi * gi;
      }
    acc = block_sum(acc);
    if (threadIdx.x == 0)
      partial_gg[blockIdx.x] = acc;
  }

  /// *done holds the tag of the scalar with which a CG iteration ended, 0 before.  Whether the
  /// cg_turn_kernel launch with scalar `tag` follows that end: not if it is the launch that
  /// sets *done, whose waves read the word while workgroup 0 stores it.  Either value they find
  /// then takes all of them into the sums below, with barriers, and out by their result.
  PPF_HD PPF_INLINE bool
  cg_ended_before(int done, unsigned int tag)
  {
    return done != 0 && (unsigned int) done != tag;
  }

  /// Unpreconditioned end of a step: gg = g.g (also the next g.h); if |g| <= tol (or it is
  /// not a number) *done is set and d stays, else d = -g + (gg / s[cur]) d and s[1 - cur] =
  /// gg.  Tells the host gg and whether the iteration is done.
  __global__ void __launch_bounds__(reduce_threads)
  cg_turn_kernel(double *__restrict__ d, const double *__restrict__ g, double *__restrict__ s,
                 int cur, const double *__restrict__ partial_gg, int count, int64_t n,
                 double tol, int *done, HostScalar *to, unsigned int tag)
  {
    if (cg_ended_before(__hip_atomic_load(done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT), tag))
      return;
    const double gg  = sum_partials(partial_gg, count);
    const bool   end = !(std::sqrt(gg) > tol);
    if (blockIdx.x == 0 && threadIdx.x == 0)
      {
        tell_host(to, gg, tag, end);
        if (end)
          __hip_atomic_store(done, int(tag), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    if (end)
      return;
    const double beta = gg / s[cur];
    if (blockIdx.x == 0 && threadIdx.x == 0)
      s[1 - cur] = gg;
    for (int64_t i = int64_t(blockIdx.x) * reduce_threads + threadIdx.x; i < n;
         i += int64_t(gridDim.x) * reduce_threads)
      d[i] = -g[i] + beta * d[i];
  }

  /// d = -h + beta d with beta = (g.h) / s[cur] from the partial sums of g.h, which becomes
  /// s[1 - cur]; with `first` set d = -h.
  template <typename T>
  __global__ void __launch_bounds__(reduce_threads)
  cg_direction_kernel(double *__restrict__ d, const T *__restrict__ h, double *__restrict__ s,
                      int cur, const double *__restrict__ partial_gh, int count, int64_t n,
                      int first)
  {
    const double gh   = sum_partials(partial_gh, count);
    const double beta = first ? 0.0 : gh / s[cur];
    if (blockIdx.x == 0 && threadIdx.x == 0)
      s[1 - cur] = gh;
    for (int64_t i = int64_t(blockIdx.x) * reduce_threads + threadIdx.x; i < n;
         i += int64_t(gridDim.x) * reduce_threads)
      d[i] = first ? -double(h[i]) : -double(h[i]) + beta * d[i];
  }

  /// BiCGStab scalars in device slots: 0 rho, 1 alpha, 2 omega, 3 r.rbar, 4 rbar.v,
  /// 5 t.r, 6 t.t, 7 beta.  One thread; `op` 0: beta = (r.rbar) alpha / (rho omega),
  /// rho = r.rbar; 1: alpha = rho / (rbar.v); 2: omega = (t.r) / (t.t), 0 when t.t is
  /// below the smallest normal double.
  __global__ void
  bicgstab_scalar_kernel(double *s, int op)
  {
    if (op == 0)
      {
        s[7] = s[3] * s[1] / (s[0] * s[2]);
        s[0] = s[3];
      }
    else if (op == 1)
      s[1] = s[0] / s[4];
    else
      s[2] = s[6] < 2.2250738585072014e-308 ? 0.0 : s[5] / s[6];
  }

  /// p = beta p + r - beta omega v (beta = s[7], omega = s[2]).
  __global__ void
  bicgstab_p_kernel(double *__restrict__ p, const double *__restrict__ r,
                    const double *__restrict__ v, const double *__restrict__ s, int64_t n)
  {
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n)
      p[i] = (s[7] * p[i] + r[i]) - s[7] * s[2] * v[i];
  }

  /// y += sign s[k] x.
  __global__ void
  axpy_slot_kernel(double *__restrict__ y, const double *__restrict__ x,
                   const double *__restrict__ s, int k, double sign, int64_t n)
  {
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n)
      y[i] += (sign * s[k]) * x[i];
  }

  /// y += sign s[k] x, with per-block partial sums of y.y (grid-stride).
  __global__ void __launch_bounds__(reduce_threads)
  axpy_slot_norm_kernel(double *__restrict__ partial, double *__restrict__ y,
                        const double *__restrict__ x, const double *__restrict__ s, int k,
                        double sign, int64_t n)
  {
    const double a   = sign * s[k];
    double       acc = 0.0;
    for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
         i += int64_t(gridDim.x) * blockDim.x)
      {
        const double yi = y[i] + a * x[i];
        y[i]            = yi;
        acc += yi * yi;
      }
    acc = block_sum(acc);
    if (threadIdx.x == 0)
      partial[blockIdx.x] = acc;
  }

  /// x += alpha y + omega z (alpha = s[1], omega = s[2]).
  __global__ void
  bicgstab_x_kernel(double *__restrict__ x, const double *__restrict__ y,
                    const double *__restrict__ z, const double *__restrict__ s, int64_t n)
  {
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n)
      x[i] += s[1] * y[i] + s[2] * z[i];
  }

  /// First Chebyshev step from x = 0 (A x = 0): d = c2 P^{-1} b, x = d.  Same values as
  /// chebyshev_step_kernel with x = ax = 0, without reading or clearing them.
  template <typename T>
  __global__ void
  chebyshev_first_zero_kernel(T *__restrict__ x, T *__restrict__ d, const T *__restrict__ b,
                              const T *__restrict__ inv_diag, T c2, int64_t n)
  {
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n)
      return;
    const T di = c2 * inv_diag[i] * b[i];
    d[i]       = di;
    x[i]       = di;
  }

  /// Chebyshev step (Varga / Saad 12.1 recurrence as used by deal.II's
  /// PreconditionChebyshev): d = c1 * d + c2 * P^{-1} (b - A x);  x += d.
  /// With `first` set, d = c2 * P^{-1}(b - A x).
  template <typename T>
  __global__ void
  chebyshev_step_kernel(T *__restrict__ x, T *__restrict__ d, const T *__restrict__ b,
                        const T *__restrict__ ax, const T *__restrict__ inv_diag, T c1,
                        T c2, int first, int64_t n)
  {
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n)
      return;
    const T r  = b[i] - ax[i];
    const T di = first ? c2 * inv_diag[i] * r : c1 * d[i] + c2 * inv_diag[i] * r;
    d[i]       = di;
    x[i] += di;
  }

  // Inverse diagonal by node class.  For constant-coefficient split operators (the
  // Poisson and level operators) the diagonal is a function of each axis' node class
  // only: 0 odd (Q2), 1 even interior (or periodic), 2 lower and 3 upper non-periodic
  // boundary.  The smoother then reads a 4^dim table per field instead of a diagonal
  // array (one stream fewer per step).  The table is checked node by node against the
  // computed diagonal whenever it is rebuilt; where any node differs the kernels read
  // the diagonal array as before (the flag is read once per thread, no host sync).

  /// Lattice of a diagonal table: nodes and periodicity per axis, fields, degree.
  struct ClassGrid
  {
    int     n[3];
    int     periodic[3];
    int     degree;
    int     dim;
    int     n_fields;
    int64_t n_nodes;
  };

  constexpr int diag_classes = 64;

  /// Node class of the inverse-diagonal tables along one axis of n nodes.
  PPF_HD PPF_INLINE int
  line_class(int degree, int i, int n, int periodic)
  {
    if (!periodic && i == 0)
      return 2;
    if (!periodic && i == n - 1)
      return 3;
    return (degree == 2 && (i & 1)) ? 0 : 1;
  }

  PPF_HD PPF_INLINE int
  axis_class(const ClassGrid &g, int d, int i)
  {
    return d < g.dim ? line_class(g.degree, i, g.n[d], g.periodic[d]) : 1;
  }

  /// Representative coordinate of class c along axis d, -1 if the class does not occur.
  PPF_HD PPF_INLINE int
  class_representative(const ClassGrid &g, int d, int c)
  {
    if (d >= g.dim)
      return c == 1 ? 0 : -1;
    const int n = g.n[d];
    int       i = -1;
    if (c == 0)
      i = (g.degree == 2 && n >= 2) ? 1 : -1;
    else if (c == 1)
      i = g.periodic[d] ? 0 : (g.degree == 2 ? 2 : 1);
    else if (c == 2)
      i = g.periodic[d] ? -1 : 0;
    else
      i = (g.periodic[d] || n < 2) ? -1 : n - 1;
    return (i >= 0 && i < n && axis_class(g, d, i) == c) ? i : -1;
  }

  /// table[f * 64 + class] from the diagonal at one node of each occurring class; one
  /// workgroup of n_fields * 64 threads; sets *ok = 1.
  template <typename T>
  __global__ void
  diag_table_build_kernel(T *__restrict__ table, int *__restrict__ ok,
                          const T *__restrict__ inv_diag, const ClassGrid g)
  {
    const int t = threadIdx.x;
    if (t == 0)
      *ok = 1;
    if (t >= g.n_fields * diag_classes)
      return;
    const int f = t / diag_classes, c = t % diag_classes;
    const int i0 = class_representative(g, 0, c & 3);
    const int i1 = class_representative(g, 1, (c >> 2) & 3);
    const int i2 = class_representative(g, 2, c >> 4);
    T         v  = T(0);
    if (i0 >= 0 && i1 >= 0 && i2 >= 0)
      v = inv_diag[f * g.n_nodes + i0 + int64_t(g.n[0]) * (i1 + int64_t(g.n[1]) * i2)];
    table[t] = v;
  }

  PPF_HD PPF_INLINE int
  node_class(const ClassGrid &g, int i0, int i1, int i2)
  {
    return axis_class(g, 0, i0) + 4 * axis_class(g, 1, i1) + 16 * axis_class(g, 2, i2);
  }

  /// Clears *ok where a node's diagonal differs from its class entry.  Grid: x over the
  /// n0 * n1 plane, y over n2, z over the fields.
  template <typename T>
  __global__ void
  diag_table_check_kernel(int *__restrict__ ok, const T *__restrict__ table,
                          const T *__restrict__ inv_diag, const ClassGrid g)
  {
    const unsigned int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= unsigned(g.n[0]) * unsigned(g.n[1]))
      return;
    const int     i0 = int(r % unsigned(g.n[0])), i1 = int(r / unsigned(g.n[0]));
    const int     i2 = int(blockIdx.y), f = int(blockIdx.z);
    const int64_t i  = f * g.n_nodes + int64_t(i2) * g.n[0] * g.n[1] + r;
    if (inv_diag[i] != table[f * diag_classes + node_class(g, i0, i1, i2)])
      *ok = 0;
  }

  /// chebyshev_step_kernel / chebyshev_first_zero_kernel (first_zero set) with the
  /// inverse diagonal taken from the class table when *ok.  A thread takes 16 consecutive
  /// bytes of every array: with one FP32 element per thread the seven streams of a step ran
  /// at 4.2 TB/s (257^3 nodes).  Grid: x over the n0 * n1 plane, y over n2, z over the fields.
  template <typename T>
  __global__ void
  chebyshev_table_kernel(T *__restrict__ x, T *__restrict__ d, const T *__restrict__ b,
                         const T *__restrict__ ax, const T *__restrict__ inv_diag,
                         const T *__restrict__ table, const int *__restrict__ ok, T c1, T c2,
                         int first, int first_zero, const ClassGrid g)
  {
    constexpr int      N = Pack<T>::n;
    using P              = typename Pack<T>::type;
    const unsigned int n0 = unsigned(g.n[0]), plane = n0 * unsigned(g.n[1]);
    const unsigned int r = (blockIdx.x * blockDim.x + threadIdx.x) * N;
    if (r >= plane)
      return;
    const int     i2 = int(blockIdx.y), f = int(blockIdx.z);
    const int64_t i  = f * g.n_nodes + int64_t(i2) * plane + r;
    const bool    by_class = *ok != 0, whole = r + N <= plane;
    const int     count = whole ? N : int(plane - r);
    P             bv {}, av {}, dv {}, xv {}, inv {};
    const auto    load = [&](P &to, const T *from) {
      if (whole)
        to = *reinterpret_cast<const P *>(from + i);
      else
        for (int k = 0; k < count; ++k)
          to[k] = from[i + k];
    };
    const auto store = [&](T *to, const P &v) {
      if (whole)
        *reinterpret_cast<P *>(to + i) = v;
      else
        for (int k = 0; k < count; ++k)
          to[i + k] = v[k];
    };
    load(bv, b);
    if (!first_zero)
      {
        load(av, ax);
        load(xv, x);
        if (!first)
          load(dv, d);
      }
    if (by_class)
      {
        int       i1 = int(r / n0), i0 = int(r - unsigned(i1) * n0);
        const T  *t  = table + f * diag_classes + 16 * axis_class(g, 2, i2);
#pragma unroll
        for (int k = 0; k < N; ++k)
          {
            inv[k] = t[axis_class(g, 0, i0) + 4 * axis_class(g, 1, i1)];
            if (++i0 == g.n[0])
              {
                i0 = 0;
                ++i1;
              }
          }
      }
    else
      load(inv, inv_diag);
    P di;
    if (first_zero)
      di = c2 * inv * bv;
    else
      {
        const P rr = bv - av;
        di         = first ? c2 * inv * rr : c1 * dv + c2 * inv * rr;
      }
    store(d, di);
    store(x, first_zero ? di : xv + di);
  }

  /// NaN/Inf probe of entry 0 (reference problem.cc:453-469 checks one entry per field).
  template <typename T>
  __global__ void
  finite_probe_kernel(int *__restrict__ flag, const T *__restrict__ x)
  {
    if (threadIdx.x == 0 && blockIdx.x == 0)
      flag[0] = isfinite(double(x[0])) ? 0 : 1;
  }

  /// Entry-0 NaN/Inf probe of every field at once: writes the index of the first field
  /// whose entry 0 is not finite, or -1.
  struct ProbeFields
  {
    const double *ptr[PPF_MAX_FIELDS];
    int           n;
  };

  /// Probe of entry 0 of every field.  Writes (tag << 5) | (bad + 1) to *result, where
  /// bad is the first field whose entry 0 is not finite (-1: none), in one store so that
  /// a host polling the word sees the tag and the result together.  When a field is bad
  /// and halt is given, sets *halt so that the launches carrying the flag that follow on
  /// the stream do nothing.
  __global__ void
  finite_probe_fields_kernel(int *__restrict__ result, const ProbeFields fields,
                             int *__restrict__ halt, unsigned int hmask, int tag)
  {
    if (threadIdx.x == 0 && blockIdx.x == 0)
      {
        int bad = -1;
        for (int f = 0; f < fields.n && f < PPF_MAX_FIELDS; ++f)
          if (bad < 0 && !isfinite(fields.ptr[f][0]))
            bad = f;
        if (bad >= 0 && halt)
          for (int i = 0; i < 32; ++i)
            if ((hmask >> i) & 1u)
              halt[i] = 1;
        *reinterpret_cast<volatile int *>(result) = (tag << 5) | (bad + 1);
      }
  }

  /// Output diagnostics: partial sums of u^2 over deal.II's full node set (periodic
  /// images counted with their multiplicity) and of u * jxw (images carry jxw = 0).
  template <int dim, int degree, typename T>
  __global__ void __launch_bounds__(reduce_threads)
  norms_partial_kernel(double *__restrict__ partial, const GridDesc g, const T *__restrict__ u)
  {
    double s2 = 0.0, si = 0.0;
    for (int64_t node = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; node < g.n_nodes;
         node += int64_t(gridDim.x) * blockDim.x)
      {
        int i[3];
        i[0] = int(node % g.nodes[0]);
        i[1] = int((node / g.nodes[0]) % g.nodes[1]);
        i[2] = dim == 3 ? int(node / (int64_t(g.nodes[0]) * g.nodes[1])) : 0;
        double mult = 1.0;
        for (int d = 0; d < dim; ++d)
          if (g.periodic[d] && i[d] == 0)
            mult *= 2.0;
        const double v = double(u[node]);
        s2 += mult * v * v;
        si += v * lumped_mass<dim, degree>(g, i);
      }
    s2 = block_sum(s2);
    __syncthreads();
    si = block_sum(si);
    if (threadIdx.x == 0)
      {
        partial[blockIdx.x]             = s2;
        partial[gridDim.x + blockIdx.x] = si;
      }
  }

  /// dst[idx[k]] = vals[k] for k < count.
  template <typename T>
  __global__ void
  scatter_kernel(T *__restrict__ dst, const int64_t *__restrict__ idx, const T *__restrict__ vals,
                 int64_t count)
  {
    const int64_t k = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (k < count)
      dst[idx[k]] = vals[k];
  }

  /// dst = value at non-Dirichlet nodes, g at Dirichlet nodes.
  template <int dim, typename T>
  __global__ void
  dirichlet_compose_kernel(T *__restrict__ dst, const GridDesc g, const T *__restrict__ gvals,
                           unsigned int mask, T value, int keep_interior)
  {
    const int64_t node = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (node >= g.n_nodes)
      return;
    int i[3];
    i[0] = int(node % g.nodes[0]);
    i[1] = int((node / g.nodes[0]) % g.nodes[1]);
    i[2] = dim == 3 ? int(node / (int64_t(g.nodes[0]) * g.nodes[1])) : 0;
    if (is_dirichlet<dim>(g, i, mask))
      dst[node] = gvals[node];
    else if (!keep_interior)
      dst[node] = value;
  }

  /// Zeroes the Dirichlet nodes of x (homogeneous level constraints).
  template <int dim, typename T>
  __global__ void
  zero_dirichlet_kernel(T *__restrict__ x, const GridDesc g, unsigned int mask)
  {
    const int64_t node = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (node >= g.n_nodes)
      return;
    int i[3];
    i[0] = int(node % g.nodes[0]);
    i[1] = int((node / g.nodes[0]) % g.nodes[1]);
    i[2] = dim == 3 ? int(node / (int64_t(g.nodes[0]) * g.nodes[1])) : 0;
    if (is_dirichlet<dim>(g, i, mask))
      x[node] = T(0);
  }

  // ------------------------------------------------------------------ transfers
  //
  // Nested uniform grids: the fine grid has twice the cells per direction.  Fine lattice
  // coordinate I sits at coarse lattice position I/2.  Prolongation evaluates the coarse
  // Q_p function at the fine nodes (exact embedding; this is the interpolation that
  // deal.II's MGTransferGlobalCoarsening uses for h-coarsening); restriction is its
  // transpose.  1-D weights:
  //   p = 1: even I -> coarse I/2 (1); odd I -> (I-1)/2, (I+1)/2 (1/2, 1/2)
  //   p = 2: even I -> coarse I/2 (1); odd I in coarse cell c = I/4 at xi = 1/4 or 3/4
  //          -> local nodes (0,1,2) with (3/8, 3/4, -1/8) or (-1/8, 3/4, 3/8).

  /// Both transfers run in one launch each: a thread owns an (x, y) column of the output
  /// lattice (flattened, so that no lane idles at a ragged width) and sums the x and y taps
  /// of a plane in registers before the z taps, which needs no intermediate lattices.  (A
  /// pass per axis moved the fine vector three times: at 257^3 FP32 the restriction took
  /// about 100 us and the prolongation 130 us.)  Every output takes a fixed number of taps.
  /// One that does not occur or lies outside a non-periodic lattice has weight zero and the
  /// position of one that counts: a NaN or an infinity reaches only the outputs that take it.

  /// Taps of the restriction along one axis at coarse coordinate J: fine positions and
  /// weights, in the order 2J (always there), 2J - 1, 2J + 1, 2J - 3, 2J + 3.
  template <int degree>
  constexpr int restrict_taps = degree == 1 ? 3 : 5;

  PPF_HD constexpr int
  restrict_offset(int k)
  {
    return k == 0 ? 0 : (k == 1 ? -1 : (k == 2 ? 1 : (k == 3 ? -3 : 3)));
  }

  template <int degree>
  PPF_HD constexpr double
  restrict_weight(int k, bool even)
  {
    if (k == 0)
      return 1.0;
    if (degree == 1)
      return 0.5;
    return k < 3 ? (even ? 3.0 / 8.0 : 3.0 / 4.0) : (even ? -1.0 / 8.0 : 0.0);
  }

  template <int degree, typename T>
  PPF_HD PPF_INLINE void
  restrict_axis(int J, int n, int periodic, int (&pos)[restrict_taps<degree>],
                T (&w)[restrict_taps<degree>])
  {
    const bool even = degree == 2 && (J & 1) == 0;
#pragma unroll
    for (int k = 0; k < restrict_taps<degree>; ++k)
      {
        int  i  = 2 * J + restrict_offset(k);
        bool ok = true;
        if (periodic) // a finer periodic lattice has at least 2 cells: one wrap suffices
          i = i < 0 ? i + n : (i >= n ? i - n : i);
        else
          ok = i >= 0 && i < n;
        const double weight = ok ? restrict_weight<degree>(k, even) : 0.0;
        pos[k]              = weight != 0.0 ? i : 2 * J;
        w[k]                = T(weight);
      }
  }

  /// Coarse planes a thread of restrict_kernel owns (even: the tap pattern in z is that of
  /// an even first plane).
  template <int dim>
  constexpr int restrict_planes = dim == 3 ? 4 : 1;
  constexpr int transfer_threads = 256;

  /// Launch grid of a transfer between the lattices gc and gf: the x-y plane of `out` (either),
  /// `groups` groups of its planes.  Both kernels index a plane of both lattices with 32 bits;
  /// the fine one is the larger, also where the launch runs over the coarse one.
  inline dim3
  transfer_grid(const GridDesc &out, const GridDesc &gc, const GridDesc &gf, int groups)
  {
    for (const GridDesc *g : {&gc, &gf})
      if (int64_t(g->nodes[0]) * g->nodes[1] >= (int64_t(1) << 31) || g->nodes[2] > 65535)
        throw Error(status_unsupported, "transfer: lattice too large for one launch");
    return dim3(grid_for(int64_t(out.nodes[0]) * out.nodes[1], transfer_threads),
                unsigned(groups));
  }

  /// coarse = P^T fine (transposed 1-D weights per axis), zero at the coarse Dirichlet nodes.
  /// Grid: x over the coarse plane, y over groups of restrict_planes planes.
  template <int dim, int degree, typename T>
  __global__ void __launch_bounds__(transfer_threads)
  restrict_kernel(T *__restrict__ coarse, const T *__restrict__ fine, const GridDesc gc,
                  const GridDesc gf, unsigned int mask)
  {
    constexpr int      K = restrict_taps<degree>, ZC = restrict_planes<dim>;
    const unsigned int c0 = unsigned(gc.nodes[0]), q = blockIdx.x * transfer_threads + threadIdx.x;
    if (q >= c0 * unsigned(gc.nodes[1]))
      return;
    const int J1 = int(q / c0), J0 = int(q - unsigned(J1) * c0);
    int       px[K], py[K];
    T         wx[K], wy[K];
    restrict_axis<degree>(J0, gf.nodes[0], gf.periodic[0], px, wx);
    restrict_axis<degree>(J1, gf.nodes[1], gf.periodic[1], py, wy);
#pragma unroll
    for (int k = 0; k < K; ++k)
      py[k] *= gf.nodes[0];
    const int64_t fine_plane = int64_t(gf.nodes[0]) * gf.nodes[1];
    const int64_t coarse_plane = int64_t(c0) * gc.nodes[1];
    const auto    plane_sum = [&](int64_t p) {
      const T *f = fine + p * fine_plane;
      T        v[K][K];
#pragma unroll
      for (int j = 0; j < K; ++j)
#pragma unroll
        for (int i = 0; i < K; ++i)
          v[j][i] = f[py[j] + px[i]];
      T sum = T(0);
#pragma unroll
      for (int j = 0; j < K; ++j)
        {
          T line = T(0);
#pragma unroll
          for (int i = 0; i < K; ++i)
            line = fma(wx[i], v[j][i], line);
          sum = fma(wy[j], line, sum);
        }
      return sum;
    };
    if constexpr (dim == 2)
      {
        const int c[3] = {J0, J1, 0};
        coarse[q]      = is_dirichlet<2>(gc, c, mask) ? T(0) : plane_sum(0);
      }
    else
      {
        const int z0 = int(blockIdx.y) * ZC, n2 = gf.nodes[2];
        T         acc[ZC];
#pragma unroll
        for (int j = 0; j < ZC; ++j)
          acc[j] = T(0);
        // fine planes 2 z0 + t that some owned plane takes
        constexpr int first = degree == 1 ? -1 : -3, last = 2 * ZC - 2 + (degree == 1 ? 1 : 3);
#pragma unroll
        for (int t = first; t <= last; ++t)
          {
            int  p  = 2 * z0 + t;
            bool ok = true;
            if (gf.periodic[2])
              p = p < 0 ? p + n2 : (p >= n2 ? p - n2 : p);
            ok = p >= 0 && p < n2;
            if (ok)
              {
                const T s = plane_sum(p);
#pragma unroll
                for (int j = 0; j < ZC; ++j)
#pragma unroll
                  for (int k = 0; k < K; ++k)
                    if (restrict_offset(k) == t - 2 * j &&
                        restrict_weight<degree>(k, j % 2 == 0) != 0.0)
                      acc[j] = fma(T(restrict_weight<degree>(k, j % 2 == 0)), s, acc[j]);
              }
          }
#pragma unroll
        for (int j = 0; j < ZC; ++j)
          if (z0 + j < gc.nodes[2])
            {
              const int c[3] = {J0, J1, z0 + j};
              coarse[(z0 + j) * coarse_plane + q] = is_dirichlet<3>(gc, c, mask) ? T(0) : acc[j];
            }
      }
  }

  /// Taps of the prolongation along one axis at fine coordinate I: coarse positions
  /// b .. b + degree of its coarse cell and their weights (an even I is a coarse node).
  template <int degree, typename T>
  PPF_HD PPF_INLINE void
  prolong_axis(int I, int n, int periodic, int (&pos)[degree + 1], T (&w)[degree + 1])
  {
    const int b = degree * (I / (2 * degree)), r = I % (2 * degree);
#pragma unroll
    for (int k = 0; k <= degree; ++k)
      {
        double v;
        if (degree == 1)
          v = r == 0 ? (k == 0 ? 1.0 : 0.0) : 0.5;
        else if ((r & 1) == 0)
          v = k == r / 2 ? 1.0 : 0.0;
        else
          v = k == 1 ? 3.0 / 4.0 : ((k == 0) == (r == 1) ? 3.0 / 8.0 : -1.0 / 8.0);
        // weight zero only where I is the coarse node b + r / 2
        const int i = b + (v != 0.0 ? k : r / 2);
        pos[k]      = i >= n && periodic ? i - n : i;
        w[k]        = T(v);
      }
  }

  /// fine += P coarse, fine Dirichlet nodes untouched.  A thread owns the 2 * degree fine
  /// planes of one coarse layer.  Grid: x over the fine plane, y over the coarse layers (and
  /// the closing plane of a non-periodic axis).
  template <int dim, int degree, typename T>
  __global__ void __launch_bounds__(transfer_threads)
  prolongate_add_kernel(T *__restrict__ fine, const T *__restrict__ coarse, const GridDesc gc,
                        const GridDesc gf, unsigned int mask)
  {
    constexpr int      K = degree + 1, ZC = dim == 3 ? 2 * degree : 1;
    const unsigned int f0 = unsigned(gf.nodes[0]), q = blockIdx.x * transfer_threads + threadIdx.x;
    if (q >= f0 * unsigned(gf.nodes[1]))
      return;
    const int I1 = int(q / f0), I0 = int(q - unsigned(I1) * f0);
    int       px[K], py[K];
    T         wx[K], wy[K];
    prolong_axis<degree>(I0, gc.nodes[0], gc.periodic[0], px, wx);
    prolong_axis<degree>(I1, gc.nodes[1], gc.periodic[1], py, wy);
#pragma unroll
    for (int k = 0; k < K; ++k)
      py[k] *= gc.nodes[0];
    const int64_t fine_plane = int64_t(f0) * gf.nodes[1];
    const int64_t coarse_plane = int64_t(gc.nodes[0]) * gc.nodes[1];
    constexpr int NP = dim == 3 ? K : 1;
    const int     layer = int(blockIdx.y);
    T             old[ZC], v[NP][K][K], s[NP];
#pragma unroll
    for (int j = 0; j < ZC; ++j)
      old[j] = fine[min(ZC * layer + j, dim == 3 ? gf.nodes[2] - 1 : 0) * fine_plane + q];
#pragma unroll
    for (int p = 0; p < NP; ++p)
      {
        int z = degree * layer + p;
        if (dim == 3)
          z = z >= gc.nodes[2] ? (gc.periodic[2] ? z - gc.nodes[2] : gc.nodes[2] - 1) : z;
        const T *c = coarse + (dim == 3 ? z : 0) * coarse_plane;
#pragma unroll
        for (int j = 0; j < K; ++j)
#pragma unroll
          for (int i = 0; i < K; ++i)
            v[p][j][i] = c[py[j] + px[i]];
      }
#pragma unroll
    for (int p = 0; p < NP; ++p)
      {
        s[p] = T(0);
#pragma unroll
        for (int j = 0; j < K; ++j)
          {
            T line = T(0);
#pragma unroll
            for (int i = 0; i < K; ++i)
              line = fma(wx[i], v[p][j][i], line);
            s[p] = fma(wy[j], line, s[p]);
          }
      }
#pragma unroll
    for (int j = 0; j < ZC; ++j)
      {
        const int I2   = ZC * layer + j;
        const int c[3] = {I0, I1, dim == 3 ? I2 : 0};
        if ((dim == 3 && I2 >= gf.nodes[2]) || is_dirichlet<dim>(gf, c, mask))
          continue;
        T sum;
        if constexpr (dim == 2)
          sum = s[0];
        else if constexpr (degree == 1)
          sum = j == 0 ? s[0] : T(0.5) * (s[0] + s[1]);
        else if (j % 2 == 0)
          sum = s[j / 2];
        else
          sum = fma(T(j == 1 ? 3.0 / 8.0 : -1.0 / 8.0), s[0],
                    fma(T(3.0 / 4.0), s[1], T(j == 1 ? -1.0 / 8.0 : 3.0 / 8.0) * s[2]));
        fine[(dim == 3 ? I2 : 0) * fine_plane + q] = old[j] + sum;
      }
  }

  /// Nodal injection fine -> coarse (coarse lattice J = fine lattice stride*J, stride a
  /// power of two); transfers non-operand fields to the levels
  /// (reference group_solution_handler.h:356-417).
  template <int dim, typename T, typename U>
  __global__ void
  inject_kernel(T *__restrict__ coarse, const GridDesc gc, const U *__restrict__ fine,
                const GridDesc gf, int stride)
  {
    const int64_t node = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (node >= gc.n_nodes)
      return;
    const int j0 = int(node % gc.nodes[0]);
    const int j1 = int((node / gc.nodes[0]) % gc.nodes[1]);
    const int j2 = dim == 3 ? int(node / (int64_t(gc.nodes[0]) * gc.nodes[1])) : 0;
    coarse[node] = T(fine[node_index(gf, stride * j0, stride * j1, stride * j2)]);
  }
} // namespace ppf
