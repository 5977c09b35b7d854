// Davidson vector kernels (included by sigma.hip inside its anonymous
// namespace): reductions, the fused Gram-Schmidt and Olsen steps, the
// subspace matrix and the Ritz rotation.  All are bound by memory at large n
// and by launches at small n, so each reads its vectors as few times as its
// data dependences allow and takes as few kernels.  One Davidson iteration's
// vector work with 20 vectors of 801,444: 1.13 -> 0.43 ms, with 6 of 13,752:
// 318 -> 125 to 141 us.
constexpr int RB = 256, RMAXB = 512;  // threads, most workgroups of a reduction

// 16-byte accesses to vectors that are only 8-byte aligned
typedef double dbl2v __attribute__((ext_vector_type(2), aligned(8)));

// sum over the workgroup in a fixed order, the same value in every thread
template <int N>
__device__ inline void block_sum(double (&s)[N], double* sh) {
#pragma unroll
  for (int q = 0; q < N; ++q) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s[q] += __shfl_xor(s[q], o);
    if ((threadIdx.x & 63) == 0) sh[q * (RB / 64) + (threadIdx.x >> 6)] = s[q];
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < N; ++q) {
    s[q] = 0.0;
#pragma unroll
    for (int w = 0; w < RB / 64; ++w) s[q] += sh[q * (RB / 64) + w];
  }
}
// the sums of N partial lists of np values, RMAXB apart (every workgroup adds
// them itself: no kernel between a reduction and the step that uses it)
template <int N>
__device__ inline void sum_partials(const double* __restrict__ part, int np, double (&s)[N], double* sh) {
#pragma unroll
  for (int q = 0; q < N; ++q) {
    s[q] = 0.0;
    for (int i = threadIdx.x; i < np; i += RB) s[q] += part[q * RMAXB + i];
  }
  block_sum<N>(s, sh);
}
// f(i, x pairs or a single last element) over this workgroup's share of n
template <class F2, class F1>
__device__ inline void over_vector(int64_t n, F2&& pair, F1&& single) {
  const int64_t n2 = n >> 1;
  for (int64_t i = (int64_t)blockIdx.x * RB + threadIdx.x; i < n2; i += (int64_t)gridDim.x * RB) pair(2 * i);
  if ((n & 1) && blockIdx.x == 0 && threadIdx.x == 0) single(n - 1);
}

// partials of <x, y> (and, with z, of <x, z>)
template <bool TWO>
__global__ __launch_bounds__(RB) void k_dot_partial(const double* __restrict__ x, const double* __restrict__ y,
                                                    const double* __restrict__ z, int64_t n, double* __restrict__ part) {
  __shared__ double sh[2 * RB / 64];
  double s[2] = {0.0, 0.0};
  over_vector(
      n,
      [&](int64_t i) {
        const dbl2v a = *(const dbl2v*)(x + i), b = *(const dbl2v*)(y + i);
        s[0] += a[0] * b[0];
        s[0] += a[1] * b[1];
        if (TWO) {
          const dbl2v c = *(const dbl2v*)(z + i);
          s[1] += a[0] * c[0];
          s[1] += a[1] * c[1];
        }
      },
      [&](int64_t i) {
        s[0] += x[i] * y[i];
        if (TWO) s[1] += x[i] * z[i];
      });
  block_sum<2>(s, sh);
  if (threadIdx.x == 0) {
    part[blockIdx.x] = s[0];
    if (TWO) part[RMAXB + blockIdx.x] = s[1];
  }
}
// out[0] = sum of np partials; out may be page-locked host memory
__global__ __launch_bounds__(RB) void k_sum_partial(const double* __restrict__ part, int np, double* __restrict__ out) {
  __shared__ double sh[RB / 64];
  double s[1];
  sum_partials<1>(part, np, s, sh);
  if (threadIdx.x == 0) out[0] = s[0];
}
// One step of the Gram-Schmidt loop with the dot products of the next: from
// the partials of <r, r> and <r, b> of the current r,
//   r <- r / |r| - <r / |r|, b> b,
// and the partials of the new <r, r> and, unless next is null, <r, next>.
// One kernel per subspace vector where normalise, dot, axpy took six.
__global__ __launch_bounds__(RB) void k_gs_step(double* __restrict__ r, const double* __restrict__ b,
                                                const double* __restrict__ next, int64_t n,
                                                const double* __restrict__ pin, int np, double* __restrict__ pout) {
  __shared__ double sh[2 * RB / 64];
  double d[2];
  sum_partials<2>(pin, np, d, sh);
  const double a = 1.0 / sqrt(d[0]), f = -(d[1] * a);
  __syncthreads();  // sh is used again below
  double s[2] = {0.0, 0.0};
  over_vector(
      n,
      [&](int64_t i) {
        const dbl2v x = *(const dbl2v*)(r + i) * a + *(const dbl2v*)(b + i) * f;
        *(dbl2v*)(r + i) = x;
        s[0] += x[0] * x[0];
        s[0] += x[1] * x[1];
        if (next) {
          const dbl2v c = *(const dbl2v*)(next + i);
          s[1] += x[0] * c[0];
          s[1] += x[1] * c[1];
        }
      },
      [&](int64_t i) {
        const double x = r[i] * a + b[i] * f;
        r[i] = x;
        s[0] += x * x;
        if (next) s[1] += x * next[i];
      });
  block_sum<2>(s, sh);
  if (threadIdx.x == 0) {
    pout[blockIdx.x] = s[0];
    pout[RMAXB + blockIdx.x] = s[1];
  }
}
// x /= sqrt(sum of the partials) if that sum is above floor
__global__ __launch_bounds__(RB) void k_scal_rsqrt(const double* __restrict__ part, int np, double floor,
                                                   double* __restrict__ x, int64_t n) {
  __shared__ double sh[RB / 64];
  double d[1];
  sum_partials<1>(part, np, d, sh);
  if (!(d[0] > floor)) return;
  const double a = 1.0 / sqrt(d[0]);
  over_vector(n, [&](int64_t i) { *(dbl2v*)(x + i) *= a; }, [&](int64_t i) { x[i] *= a; });
}

__global__ void k_axpy(double a, const double* __restrict__ x, double* __restrict__ y, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    y[i] += a * x[i];
}
__global__ void k_scal(double a, double* __restrict__ x, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    x[i] *= a;
}
// (x, d) -> x / (e - d + shift) where e - d is not tiny (linear.C:27-47)
__device__ inline double preconditioned(double x, double d, double e, double shift) {
  const double den = e - d;
  return fabs(den) > 1e-12 ? x / (den + shift) : x;
}
__global__ void k_precond(double* __restrict__ x, const double* __restrict__ d, double e, double shift, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    x[i] = preconditioned(x[i], d[i], e, shift);
}
// Olsen's step (linear.C:50-60) in two kernels: the partials of <C~, r> and
// <C, C~> with C~ = precond(C), kept in work, then r <- precond(r - ratio C)
__global__ __launch_bounds__(RB) void k_olsen_dots(const double* __restrict__ r, const double* __restrict__ c,
                                                   const double* __restrict__ d, double e, double shift,
                                                   double* __restrict__ work, int64_t n, double* __restrict__ part) {
  __shared__ double sh[2 * RB / 64];
  double s[2] = {0.0, 0.0};
  for (int64_t i = (int64_t)blockIdx.x * RB + threadIdx.x; i < n; i += (int64_t)gridDim.x * RB) {
    const double ci = c[i], t = preconditioned(ci, d[i], e, shift);
    work[i] = t;
    s[0] += t * r[i];
    s[1] += ci * t;
  }
  block_sum<2>(s, sh);
  if (threadIdx.x == 0) {
    part[blockIdx.x] = s[0];
    part[RMAXB + blockIdx.x] = s[1];
  }
}
__global__ __launch_bounds__(RB) void k_olsen_step(double* __restrict__ r, const double* __restrict__ c,
                                                   const double* __restrict__ d, double e, double shift, int64_t n,
                                                   const double* __restrict__ part, int np) {
  __shared__ double sh[2 * RB / 64];
  double s[2];
  sum_partials<2>(part, np, s, sh);
  const double a = -(s[0] / s[1]);
  for (int64_t i = (int64_t)blockIdx.x * RB + threadIdx.x; i < n; i += (int64_t)gridDim.x * RB)
    r[i] = preconditioned(r[i] + a * c[i], d[i], e, shift);
}
__global__ void k_copy(const double* __restrict__ x, double* __restrict__ y, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    y[i] = x[i];
}

// Gram matrix tile of two vector sets (mx, my <= GMAX vectors of length n,
// stride ld): G(i, j) = sum_x X_i[x] Y_j[x] on the matrix cores, K = x.  A
// wavefront takes 16 x at a time (lane (li, lk): x = 4 lk + e of vector li, so
// four lanes read a vector's 128 bytes), accumulates the whole 32 x 32 tile
// and the workgroup's waves are summed in LDS; partials go out as
// part[(i my + j) nblk + block], contiguous for the ordered sum.  Larger sets
// (up to GRAM_MAX vectors) run as GMAX x GMAX tiles.
constexpr int GMAX = 32, GBLK = 512, GRAM_MAX = 128;
__global__ __launch_bounds__(256) void k_gram_partial(const double* __restrict__ X, const double* __restrict__ Y, int mx,
                                                      int my, int64_t n, int64_t ld, double* __restrict__ part) {
  __shared__ double sh[4][16 * 16];
  const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4, w = threadIdx.x >> 6;
  const int bx = mx > 16 ? 2 : 1, by = my > 16 ? 2 : 1;
  dbl4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = dbl4{0.0, 0.0, 0.0, 0.0};
  // a vector past the set reads the set's last one (its results are not kept)
  const double* xp[2];
  const double* yp[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    xp[i] = X + (int64_t)min(16 * i + li, mx - 1) * ld + 4 * lk;
    yp[i] = Y + (int64_t)min(16 * i + li, my - 1) * ld + 4 * lk;
  }
  const int64_t full = n & ~(int64_t)15;
  for (int64_t x0 = ((int64_t)blockIdx.x * 4 + w) * 16; x0 < full; x0 += (int64_t)gridDim.x * 64) {
    dbl2v a[2][2], b[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        if (i < bx) a[i][h] = *(const dbl2v*)(xp[i] + x0 + 2 * h);
        if (i < by) b[i][h] = *(const dbl2v*)(yp[i] + x0 + 2 * h);
      }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int e = 0; e < 2; ++e)
#pragma unroll
        for (int i = 0; i < 2; ++i)
          if (i < bx)
#pragma unroll
            for (int j = 0; j < 2; ++j)
              if (j < by) acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i][h][e], b[j][h][e], acc[i][j], 0, 0, 0);
  }
  if (full < n && blockIdx.x == 0 && w == 0)  // the last n mod 16
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const bool in = full + 4 * lk + e < n;
      double a[2], b[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        a[i] = in ? xp[i][full + e] : 0.0;
        b[i] = in ? yp[i][full + e] : 0.0;
      }
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i], b[j], acc[i][j], 0, 0, 0);
    }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      if (i >= bx || j >= by) continue;
      __syncthreads();
#pragma unroll
      for (int e = 0; e < 4; ++e) sh[w][(lk + 4 * e) * 16 + li] = acc[i][j][e];
      __syncthreads();
      const int r = 16 * i + threadIdx.x / 16, c = 16 * j + threadIdx.x % 16;
      if (r < mx && c < my) {
        double s = 0.0;
#pragma unroll
        for (int q = 0; q < 4; ++q) s += sh[q][threadIdx.x];
        part[(int64_t)(r * my + c) * gridDim.x + blockIdx.x] = s;
      }
    }
}
// out[i ldo + j] = ordered sum of the tile's partials, one wavefront per
// element; out may be page-locked host memory
__global__ __launch_bounds__(256) void k_gram_sum(const double* __restrict__ part, int nblk, int mx, int my,
                                                  double* __restrict__ out, int ldo) {
  const int pidx = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (pidx >= mx * my) return;
  double s = 0.0;
  for (int b = lane; b < nblk; b += 64) s += part[(int64_t)pidx * nblk + b];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
  if (lane == 0) out[(int64_t)(pidx / my) * ldo + pidx % my] = s;
}
// Y_j[x] (+)= sum_{i < m} coef[j ldc + i] X_i[x] for j < mo (m, mo <= GMAX);
// accumulate = 0 overwrites Y.  A thread keeps a pair of x of every X vector
// in registers, so X is read and Y written once; the coefficients of a result
// are contiguous and uniform (scalar loads of several at a time: one load
// each, with i as the slow index, took twice the time of the vectors).
template <int MB>  // m <= 4 MB
__global__ __launch_bounds__(256) void k_lincomb(const double* __restrict__ X, int m, int64_t n, int64_t ld,
                                                 const double* __restrict__ coef, int ldc, int mo,
                                                 double* __restrict__ Y, int64_t ldy, int accumulate) {
  const int64_t np = (n + 1) >> 1;
  for (int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x; p < np; p += (int64_t)gridDim.x * 256) {
    const int64_t x = 2 * p;
    const bool two = x + 1 < n;
    dbl2 xv[4 * MB];
#pragma unroll
    for (int i = 0; i < 4 * MB; ++i) {
      const double* q = X + (int64_t)min(i, m - 1) * ld + x;
      if (two) {
        const dbl2v t = *(const dbl2v*)q;
        xv[i] = dbl2{t[0], t[1]};
      } else {
        xv[i] = dbl2{*q, 0.0};
      }
    }
    for (int j = 0; j < mo; ++j) {
      const double* cj = coef + (int64_t)j * ldc;
      dbl2 s = {0.0, 0.0};
#pragma unroll
      for (int i = 0; i < 4 * MB; ++i)
        if (i < 4 * MB - 4 || i < m) s += xv[i] * cj[i];
      double* y = Y + (int64_t)j * ldy + x;
      if (accumulate) {
        s[0] += y[0];
        if (two) s[1] += y[1];
      }
      if (two)
        *(dbl2v*)y = dbl2v{s[0], s[1]};
      else
        y[0] = s[0];
    }
  }
}
