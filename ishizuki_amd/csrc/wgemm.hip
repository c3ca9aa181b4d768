// GGML matmul of 5..16 rows with sixteen rows per MFMA (wgemm.h): Q4_K, Q6_K, IQ2_XS.
#include "wgemm.h"

#define ISHZ_TABLE_QUAL static __device__
#include "ggml_grids.inc"
#include "ggml_tables.h"

namespace ishz {

// From five rows on: up to four, vgemm.h's diagonal A costs one set of MFMAs too and decodes with fewer
// instructions (17408x5120, 4 rows: Q4_K 16.6 us there, 19.7 here; Q6_K and IQ2_XS within 6 %).
// Where a long K is split the two are level from five rows on (Q4_K 5120x25600, 5 to 8 rows: 24.9-25.2 us here,
// 24.5-25.5 there; 2048x32768 18.3-18.9 and 19.4-20.6), and without a workspace, where neither splits, this one
// is ahead (32.2-36.3 us against 41.0-43.1).
bool ggml_wgemm_takes(uint32_t type, int M, int K) {
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
