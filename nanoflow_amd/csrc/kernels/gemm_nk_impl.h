#pragma once
// bf16 GEMMs on k-contiguous weights ([N][K], the orientation a checkpoint holds), with an optional
// activation in the epilogue: what the layer-stack pipeline's projections run on.  Same tiles, split-K
// plans and kernels as the fp16 entries.
#include "gemm_impl.h"

// bias: one row of N elements added to every row of the product (null: none)
template <class E>
static int gemm_nk_entry(const char* who, const uint16_t* A, const uint16_t* B, const uint16_t* bias, uint16_t* D, int M, int N,
                         int K, void* workspace, size_t workspace_bytes, nf_stream_t stream) {
  int rc = check_gemm_args(who, A, B, D, M, N, K);
  if (rc) return rc;
  NF_REQUIRE((uintptr_t)bias % 8 == 0, "%s: the bias must be 8-byte aligned", who);
  const float beta = bias ? 1.f : 0.f;
  const int ldc = bias ? 0 : N;
  if (M == 0) return NF_OK;
  hipStream_t s = (hipStream_t)stream;
  int k_per = 0;
  const int shares = M <= kTallRows ? splitk_plan(M, N, K, &k_per) : 1;
  const bool aligned = (uintptr_t)workspace % 16 == 0, given = shares > 1 && workspace && workspace_bytes >= (size_t)shares * M * N * sizeof(float);
  NF_REQUIRE(!given || aligned, "%s: the workspace must be 16-byte aligned", who);  // whatever runs
  if (rows_pay(M, N, K) && !(given && narrow_and_deep(M, N, K))) return dispatch_rows<E, false>(A, B, bias, D, M, N, K, 1.f, beta, ldc, s);
  if (workspace && aligned && M > kTallRows) {
    const MidPlan mid = mid_split_plan(M, N, K, kMidBytes);
    if (mid.shares > 1 && workspace_bytes >= (size_t)mid.shares * M * N * sizeof(float))
      return launch_mid<E, true>(mid, A, B, bias, D, M, N, K, 1.f, beta, ldc, static_cast<float*>(workspace), s);
  }
  if (!given) return dispatch_plain<E, true>(A, B, bias, D, M, N, K, 1.f, beta, ldc, s);
  float* P = static_cast<float*>(workspace);
  if (M <= 64) return launch_splitk_64<E>(A, B, bias, D, M, N, K, 1.f, beta, ldc, shares, k_per, P, true, s);
  if (M > 256) return launch_splitk<E, 320, 128, 2, 2, true>(A, B, bias, D, M, N, K, 1.f, beta, ldc, shares, k_per, P, s);
  return launch_splitk<E, 128, 128, 2, 4, true>(A, B, bias, D, M, N, K, 1.f, beta, ldc, shares, k_per, P, s);
}
