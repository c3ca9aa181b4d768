// GGML matmul of 5..16 rows with sixteen rows per MFMA (wgemm.h): Q4_K, Q6_K, IQ2_XS.
#include "wgemm.h"

#define ISHZ_TABLE_QUAL static __device__
#include "ggml_grids.inc"
#include "ggml_tables.h"

namespace ishz {

// From five rows on: up to four, vgemm.h's diagonal A costs one set of MFMAs too and decodes with fewer
// instructions (17408x5120, 4 rows: Q4_K 16.6 us there, 19.7 here; Q6_K and IQ2_XS within 6 %).
// Q4_K keeps it up to eight rows too where it splits a long K and a CU's share is large (5120x25600, 125
// tile steps a CU, 8 rows: 26.3 us there, 26.7-27.3 here; 1024x8192, 8 steps: 13.1 and 9.0); Q6_K and
// IQ2_XS are faster here at that shape too (46.8 and 43.1, 31.4 and 27.2).
bool ggml_wgemm_takes(uint32_t type, int M, int K, int N) {
  int T;
  const int cus = gemv_num_cu();
  if (type == ISHZ_GGML_Q4_K && M <= 8 && K % 256 == 0 && (size_t)((N + 15) / 16) * (K / 256) >= (size_t)64 * cus &&
      vgemm_splits(M, K, N, cus, T) > 1)
    return false;
  return M > 4 && M <= 16 && K % 256 == 0 && (type == ISHZ_GGML_Q4_K || type == ISHZ_GGML_Q6_K || type == ISHZ_GGML_IQ2_XS);
}
size_t ggml_wgemm_part_bytes(int M, int K, int N, int cus) { return wgemm_part_bytes(M, K, N, cus); }
int ggml_wgemm(uint32_t type, const void *x, int M, int K, const void *w, int N, const Out &y, void *ws, size_t ws_bytes,
               hipStream_t st) {
  switch (type) {
  case ISHZ_GGML_Q4_K: return wgemm<WQ4_K>(x, M, K, w, N, y, ws, ws_bytes, st);
  case ISHZ_GGML_Q6_K: return wgemm<WQ6_K>(x, M, K, w, N, y, ws, ws_bytes, st);
  default: return wgemm<WIQ2_XS>(x, M, K, w, N, y, ws, ws_bytes, st);
  }
}
}  // namespace ishz
