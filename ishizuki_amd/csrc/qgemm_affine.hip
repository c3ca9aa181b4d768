// MLX affine packs (2, 4, 6 and 8 bits, groups of 64 and 128) times any number of rows (qgemm.h).
#include "qgemm.h"

namespace ishz {

template <int BITS, int GS, bool BF16S>
static int affine_rows(const void *x, int dt, int M, int K, const uint32_t *codes, const void *scales, const void *biases,
                       int N, void *y, void *ws, hipStream_t st) {
  using F = QAffine<BITS, GS, BF16S>;
  const QLayout l = qgemm_layout(M, K, N, true, 4);
  float *X = (float *)((char *)ws + l.X), *rs = (float *)((char *)ws + l.rs);
  int rc = launch_qimage<F>(x, dt, M, K, ws, X, rs, st);
  if (rc) return rc;
  const int S = qgemm_splits(M, K, N, 4, gemv_num_cu());
  const Out o{y, dt, dt == ISHZ_DT_BF16 ? rs : nullptr};
  float *part = S > 1 ? (float *)((char *)ws + l.part) : nullptr;
  const QPlain<typename F::Args> p{{codes, (const uint16_t *)scales, (const uint16_t *)biases, K}, M, N, o, part};
  if ((rc = launch_qgemm<F>(p, M, K, N, 1, S, ws, X, st)) || S == 1) return rc;
  const size_t n = (size_t)M * N;
  hipLaunchKernelGGL(vgemm_sum_kernel, dim3((unsigned)std::min<size_t>((n + 255) / 256, 2048)), dim3(256), 0, st, part, S, n, N, o);
  ISHZ_LAUNCH_CHECK("many-row matmul sum launch");
  return ISHZ_OK;
}

}  // namespace ishz

using namespace ishz;

// Workspace: x rotated in its own dtype, then what qgemm_layout says.
static size_t affine_rot_bytes(int M, int K) { return q256((size_t)M * K * 2); }

extern "C" size_t ishz_affine_rows_workspace_size(int M, int K, int N) {
  if (M <= 0 || K <= 0 || N <= 0 || K % 256) return 0;
  return affine_rot_bytes(M, K) + qgemm_layout(M, K, N, true, 4).bytes;
}

extern "C" int ishz_affine_linear_rows(const void *x, int x_dtype, int M, int K, const float *signs, int block,
                                       const uint32_t *codes, const void *scales, const void *biases, int scale_dtype, int N,
                                       int bits, int group, void *y, void *workspace, size_t workspace_bytes,
                                       ishz_stream_t stream) {
  if (x_dtype != ISHZ_DT_F16 && x_dtype != ISHZ_DT_BF16) return decline("many rows: activations must be fp16 or bf16");
  if (scale_dtype != ISHZ_DT_F16 && scale_dtype != ISHZ_DT_BF16) return decline("scales must be fp16 or bf16");
  if (bits != 2 && bits != 4 && bits != 6 && bits != 8) return decline("many rows: packs of 2, 4, 6 and 8 bits");
  if (group != 64 && group != 128) return decline("many rows: groups of 64 and 128");
  if (M < 1 || N < 1 || K <= 0 || K % 256) return decline("many rows: K a multiple of 256");
  if (block > 0 && ((block & (block - 1)) || block > 4096 || K % block)) return decline("bad Hadamard block");
  if (!x || !codes || !scales || !biases || !y) return einval("null pointer");
  if (!lds_loadable(codes) || !lds_loadable(workspace) || (uintptr_t)scales % 4 || (uintptr_t)biases % 4)
    return decline("many rows: codes and workspace aligned to 16 bytes, scales and biases to 4");
  if (M > QROWS_MAX) return decline("many rows: more row blocks than a grid holds");
  if (block > 0 && !one_rotation(M, K, block)) return decline("many rows: more to rotate than a launch holds");
  if (!workspace || workspace_bytes < ishz_affine_rows_workspace_size(M, K, N))
    return einval("workspace too small (ishz_affine_rows_workspace_size)");
  hipStream_t st = S(stream);
  const void *xr = x;
  if (block > 0) {
    const int rc = ishz_hadamard(x, x_dtype, M, K, block, signs, 0, workspace, stream);
    if (rc) return rc;
    xr = workspace;
  }
  void *ws = (char *)workspace + affine_rot_bytes(M, K);
#define ISHZ_ROWS(B)                                                                                                        \
  case B:                                                                                                                   \
    if (group == 64)                                                                                                        \
      return scale_dtype == ISHZ_DT_BF16 ? affine_rows<B, 64, true>(xr, x_dtype, M, K, codes, scales, biases, N, y, ws, st)   \
                                         : affine_rows<B, 64, false>(xr, x_dtype, M, K, codes, scales, biases, N, y, ws, st); \
    return scale_dtype == ISHZ_DT_BF16 ? affine_rows<B, 128, true>(xr, x_dtype, M, K, codes, scales, biases, N, y, ws, st)    \
                                       : affine_rows<B, 128, false>(xr, x_dtype, M, K, codes, scales, biases, N, y, ws, st);
  switch (bits) {
    ISHZ_ROWS(2)
    ISHZ_ROWS(4)
    ISHZ_ROWS(6)
    ISHZ_ROWS(8)
  }
#undef ISHZ_ROWS
  return decline("many rows: packs of 2, 4, 6 and 8 bits");
}
