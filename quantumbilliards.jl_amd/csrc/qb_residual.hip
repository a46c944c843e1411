// Residual check of Beyn eigenpairs: y = T(lambda) phi for a batch of
// assembled matrices (one candidate eigenvalue and density per matrix),
// with the absolute column sums (opnorm(T, 1)) and row sums (opnorm(T, Inf))
// of each matrix.  Replaces the mul!(y, Tbufs[j], phi) / opnorm loop of
// residual_and_norm_select (beyn.jl:557-593) and of
// imag_k_check_EXPERIMENTAL (beyn.jl:666-687).
//
// k_gemv_part streams the N x N complex128 matrices once, column-major: a
// workgroup owns 256 rows and one of `nsplit` column chunks; lanes read
// consecutive rows of a column (coalesced), the chunk of phi is staged in LDS.
// Partial products, row sums of a chunk and column sums of a wave's 64 rows go to
// buffers that k_norms adds up in a fixed order, one workgroup per candidate, so
// the result does not depend on launch order and five numbers per candidate leave
// the device.  What bounds it: the one pass over T, 4.1 TB/s (520 us for 32
// matrices of N = 2050; k_norms 55).  Column sums in a pass of their own and all
// partial sums added on the host took 810 us and about 1.7 ms.
#include "qb_internal.h"
#include "qb_linalg.h"

// v[u] summed over the wave, u < 4: lane l returns the sum of v[l / 16].
__device__ __forceinline__ double wave_sum4(const double* v, int lane) {
  const bool hi = lane & 32, up = lane & 16;
  double a = hi ? v[2] : v[0], b = hi ? v[3] : v[1];
  a += __shfl_xor(hi ? v[0] : v[2], 32);
  b += __shfl_xor(hi ? v[1] : v[3], 32);
  double c = up ? b : a;
  c += __shfl_xor(up ? a : b, 16);
  for (int off = 8; off >= 1; off >>= 1) c += __shfl_xor(c, off);
  return c;
}

__global__ void __launch_bounds__(256) k_gemv_part(const cd* __restrict__ T,
                                                   const cd* __restrict__ phi,
                                                   cd* __restrict__ part,
                                                   double* __restrict__ rowabs,
                                                   double* __restrict__ colabs, int64_t N,
                                                   int64_t chunk, int nb) {
  __shared__ cd ph[256];
  const int b = blockIdx.z, s = blockIdx.y, lane = threadIdx.x & 63;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const cd* Tb = T + (int64_t)b * N * N;
  const cd* pb = phi + (int64_t)b * N;
  // column sums of this wave's 64 rows
  double* cw = colabs + (((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * nb + b) * N;
  const int64_t j0 = (int64_t)s * chunk;
  const int64_t j1 = (j0 + chunk < N) ? j0 + chunk : N;
  const bool ok = i < N;
  double ar = 0, ai = 0, sa = 0;
  for (int64_t jb = j0; jb < j1; jb += 256) {
    __syncthreads();
    if (jb + threadIdx.x < j1) ph[threadIdx.x] = pb[jb + threadIdx.x];
    __syncthreads();
    const int m = (j1 - jb < 256) ? (int)(j1 - jb) : 256;
    const cd* col = Tb + (ok ? i : N - 1) + jb * N;
    for (int q = 0; q < m; q += 4) {  // columns past the end repeat the last, with weight 0
      cd t[4];
      double a[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) t[u] = col[(int64_t)(q + u < m ? q + u : m - 1) * N];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        a[u] = 0;
        if (!ok || q + u >= m) continue;
        const cd p = ph[q + u];
        ar += t[u].re * p.re - t[u].im * p.im;
        ai += t[u].re * p.im + t[u].im * p.re;
        a[u] = hypot(t[u].re, t[u].im);
        sa += a[u];
      }
      const double c = wave_sum4(a, lane);
      if ((lane & 15) == 0 && q + (lane >> 4) < m) cw[jb + q + (lane >> 4)] = c;
    }
  }
  if (ok) {
    const int64_t o = ((int64_t)s * nb + b) * N + i;
    part[o] = cd{ar, ai};
    rowabs[o] = sa;
  }
}

// out[b][0..4]: ||y||_2, ||y||_1, ||y||_inf, largest column sum, largest row sum.
__global__ void __launch_bounds__(1024) k_norms(const cd* __restrict__ part,
                                                const double* __restrict__ rowabs,
                                                const double* __restrict__ colabs, int64_t N, int nb,
                                                int nsplit, int nrow, double* __restrict__ out) {
  __shared__ double red[5][16];
  const int b = blockIdx.x, tid = threadIdx.x;
  double v[5] = {0, 0, 0, 0, 0};
  for (int64_t i = tid; i < N; i += 1024) {
    double yr = 0, yi = 0, ra = 0, ca = 0;
    for (int s = 0; s < nsplit; ++s) {
      const int64_t o = ((int64_t)s * nb + b) * N + i;
      yr += part[o].re;
      yi += part[o].im;
      ra += rowabs[o];
    }
#pragma unroll 8
    for (int w = 0; w < nrow; ++w) ca += colabs[((int64_t)w * nb + b) * N + i];
    const double a = hypot(yr, yi);
    v[0] += a * a;
    v[1] += a;
    v[2] = fmax(v[2], a);
    v[3] = fmax(v[3], ca);
    v[4] = fmax(v[4], ra);
  }
  for (int off = 32; off >= 1; off >>= 1)
    for (int c = 0; c < 5; ++c) {
      const double o = __shfl_xor(v[c], off);
      v[c] = c < 2 ? v[c] + o : fmax(v[c], o);
    }
  if ((tid & 63) == 0)
    for (int c = 0; c < 5; ++c) red[c][tid >> 6] = v[c];
  __syncthreads();
  if (tid < 5) {
    double x = red[tid][0];
    for (int w = 1; w < 16; ++w) x = tid < 2 ? x + red[tid][w] : fmax(x, red[tid][w]);
    out[5 * b + tid] = tid == 0 ? sqrt(x) : x;
  }
}

size_t qb_gemv_norms_bytes(int64_t N, int nb, int nsplit) {
  const int64_t nrow = (N + 255) / 256 * 4;
  return (size_t)nb * N * (nsplit * (sizeof(cd) + sizeof(double)) + nrow * sizeof(double));
}

int qb_gemv_norms(qb_ctx* ctx, const cd* T, const cd* phi, int64_t N, int nb, int nsplit,
                  void* work, double* out) {
  if (N <= 0 || nb <= 0) return QB_OK;
  const int64_t chunk = (N + nsplit - 1) / nsplit;
  const unsigned rows = (unsigned)((N + 255) / 256);
  cd* part = (cd*)work;
  double* rowabs = (double*)(part + (int64_t)nsplit * nb * N);
  double* colabs = rowabs + (int64_t)nsplit * nb * N;
  int slot = qb_prof_begin(ctx, QB_K_OTHER, 8.0 * (double)N * N * nb, 16.0 * (double)N * N * nb);
  hipLaunchKernelGGL(k_gemv_part, dim3(rows, (unsigned)nsplit, (unsigned)nb), dim3(256), 0,
                     ctx->stream, T, phi, part, rowabs, colabs, N, chunk, nb);
  QB_HIP(ctx, hipGetLastError());
  // waves wholly past row N write zeros: nrow counts them
  hipLaunchKernelGGL(k_norms, dim3((unsigned)nb), dim3(1024), 0, ctx->stream, part, rowabs, colabs,
                     N, nb, nsplit, (int)rows * 4, out);
  qb_prof_end(ctx, slot);
  QB_HIP(ctx, hipGetLastError());
  return QB_OK;
}
