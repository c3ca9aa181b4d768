// IQ2_XS's LDS tables, built from the codebook of ggml_grids.inc (included first, into this unit).
#pragma once
#include "common.h"

namespace ishz {

// IQ2_XS grid entries as fp16 (values 8, 25, 43), either in the permuted pair order of the GEMV
// (x0,x2,x1,x3,...) or in natural order for the MFMA B operand; with `sgn`, also the 128 sign
// patterns of ksigns (index | parity << 7) as natural-order fp16 sign-bit masks (the GEMV computes
// its masks in registers).
template <bool PERM>
DEV void build_iq2xs_tables(u4 *grid, u4 *sgn) {
  for (int e = threadIdx.x; e < 512 + (sgn ? 128 : 0); e += blockDim.x) {
    if (e < 512) {
      const uint64_t v = ishz_iq2xs_grid[e];
      uint32_t hv[8];
#pragma unroll
      for (int j = 0; j < 8; j++) hv[j] = f2h((float)((v >> (8 * j)) & 0xff));
      grid[e] = PERM ? u4{hv[0] | hv[2] << 16, hv[1] | hv[3] << 16, hv[4] | hv[6] << 16,
                          hv[5] | hv[7] << 16}
                     : u4{hv[0] | hv[1] << 16, hv[2] | hv[3] << 16, hv[4] | hv[5] << 16,
                          hv[6] | hv[7] << 16};
    } else {
      const int i = e - 512;
      const uint32_t s = (uint32_t)i | (uint32_t)(__builtin_popcount(i) & 1) << 7;
      auto bit = [&](int j) { return ((s >> j) & 1u) << 15; };
      sgn[i] = u4{bit(0) | bit(1) << 16, bit(2) | bit(3) << 16, bit(4) | bit(5) << 16, bit(6) | bit(7) << 16};
    }
  }
}

DEV void build_iq2xs_tables_perm(u4 *grid, u4 *sgn) { build_iq2xs_tables<true>(grid, sgn); }
DEV void build_iq2xs_tables_nat(u4 *grid, u4 *sgn) { build_iq2xs_tables<false>(grid, sgn); }

}  // namespace ishz
