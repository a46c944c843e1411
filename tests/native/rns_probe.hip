// Test-only wrapper of the int8 residue GEMM (qb_rns.hip): host operands,
// column-major per matrix, C[b] -= A[b] B[b] with inner dimension K = 512.
#include "../../quantumbilliards.jl_amd/csrc/qb_linalg.h"

extern "C" int qbt_rns_sub(qb_ctx* ctx, int M, int N, int K, const cd* A, const cd* B, cd* C,
                           int batch, int iters, double* ms_slice, double* ms_gemm) {
  const size_t na = (size_t)M * K * batch, nb = (size_t)K * N * batch, nc = (size_t)M * N * batch;
  cd *dA = nullptr, *dB = nullptr, *dC = nullptr;
  QbRns h;
  hipEvent_t e[3];
  int rc = K == 512 ? qb_rns_open(ctx, &h, M, N, batch) : QB_E_ARG;
  if (rc) return rc;
  bool ok = hipMalloc((void**)&dA, na * sizeof(cd)) == hipSuccess &&
            hipMalloc((void**)&dB, nb * sizeof(cd)) == hipSuccess &&
            hipMalloc((void**)&dC, nc * sizeof(cd)) == hipSuccess;
  ok = ok && hipMemcpy(dA, A, na * sizeof(cd), hipMemcpyHostToDevice) == hipSuccess &&
       hipMemcpy(dB, B, nb * sizeof(cd), hipMemcpyHostToDevice) == hipSuccess &&
       hipMemcpy(dC, C, nc * sizeof(cd), hipMemcpyHostToDevice) == hipSuccess;
  for (auto& v : e) ok = ok && hipEventCreate(&v) == hipSuccess;
  if (ok) {
    rc = qb_rns_set_a(ctx, &h, M, dA, M, (int64_t)M * K);
    if (!rc) rc = qb_rns_sub(ctx, &h, N, dB, K, (int64_t)K * N, dC, M, (int64_t)M * N);
    ok = !rc && hipStreamSynchronize(ctx->stream) == hipSuccess &&
         hipMemcpy(C, dC, nc * sizeof(cd), hipMemcpyDeviceToHost) == hipSuccess;
  }
  if (ok && iters > 0) {  // timing: set_a, then set_a + sub, per call
    (void)hipEventRecord(e[0], ctx->stream);
    for (int i = 0; i < iters; ++i) (void)qb_rns_set_a(ctx, &h, M, dA, M, (int64_t)M * K);
    (void)hipEventRecord(e[1], ctx->stream);
    for (int i = 0; i < iters; ++i)
      (void)qb_rns_sub(ctx, &h, N, dB, K, (int64_t)K * N, dC, M, (int64_t)M * N);
    (void)hipEventRecord(e[2], ctx->stream);
    ok = hipEventSynchronize(e[2]) == hipSuccess;
    float a = 0, b = 0;
    (void)hipEventElapsedTime(&a, e[0], e[1]);
    (void)hipEventElapsedTime(&b, e[1], e[2]);
    *ms_slice = a / iters;
    *ms_gemm = b / iters;
  }
  for (auto& v : e) (void)hipEventDestroy(v);
  (void)hipFree(dA);
  (void)hipFree(dB);
  (void)hipFree(dC);
  qb_rns_close(ctx, &h);
  return rc ? rc : ok ? QB_OK : QB_E_HIP;
}
