// EXL3 trellis weights times any number of rows (qgemm.h).
#include "exl3_fmt.h"
#include "qgemm.h"

namespace ishz {

// A wave's 16 K tiles x 2 column tiles of a step are 1024 bytes per bit: adjacent column tiles of one
// K tile are contiguous, so whole 16-byte pieces go straight to the wave's own LDS, a step ahead, and
// each lane reads its window of every tile there. The weights decode to fp16 exactly: no scale, the
// MFMAs add into the sums. An MFMA takes two K tiles: k slots 0..3 of lane group g are rows
// 2 g + {0, 1, 8, 9} of the first, 4..7 of the second (the order the trellis decodes them in).
template <int KA, bool HALF, int CB>
struct QExl3 {
  using TR = Trellis<KA, HALF>;
  using T32 = Trellis32<KA, HALF>;
  static constexpr bool SCALED = false;
  static constexpr int MT_MAX = 8, OCC = 3, W = TR::WORDS, NTC = QNT, PIECES = 4 * NTC * W, PTK = NTC * W / 4;
  static constexpr int WOPS = (PIECES + 63) / 64 / NTC, WQ = 0;
  static size_t lds_bytes(int) { return (size_t)4 * 2 * PIECES * 16; }
  struct Args {
    const uint32_t *trellis;
    int tiles_n;
  };
  struct Ctx {
    uint32_t *buf;  // this wave's two steps
    const uint32_t *src;
    int lane, p0;
    typename T32::Win wn;
    DEV Ctx(const Args &a, char *extra, int wave, int lane_, int c0, int N, int)
        : buf((uint32_t *)extra + wave * 2 * PIECES * 4), src(a.trellis + (size_t)(min(c0, N - 16 * NTC) / 16) * W), lane(lane_),
          p0(8 * (4 * (lane_ & 7) + (lane_ >> 4)) + 4 * ((lane_ >> 3) & 1)), wn(T32::window(p0)) {}
  };
  struct Raw {
    int buf;
  };
  template <int NT>
  static DEV void fetch(const Args &a, const Ctx &c, int j, int buf) {
    static_assert(NT == NTC, "a step's bytes");
#pragma unroll
    for (int i = 0; i < (PIECES + 63) / 64; i++) {
      const int q = i * 64 + c.lane;
      if (PIECES % 64 == 0 || q < PIECES)
        load16_to_lds(c.src + ((size_t)(16 * j + q / PTK) * a.tiles_n) * W + (q % PTK) * 4, c.buf + ((buf & 1) * PIECES + i * 64) * 4);
    }
  }
  template <int NT>
  static DEV Raw raw(const Ctx &, int j, int) {
    return {j & 1};
  }
  static DEV u2 decode4(const uint32_t *tile, const Ctx &c) {
    if constexpr (T32::FITS) {
      const uint32_t win = __builtin_amdgcn_alignbit(tile[c.wn.ja], tile[c.wn.jb], c.wn.amt);
      uint32_t s[4];
#pragma unroll
      for (int i = 0; i < 4; i++) s[i] = __builtin_amdgcn_ubfe(win, T32::field(i), 16);
      return u2{exl3_decode2<CB>(s[0], s[1]), exl3_decode2<CB>(s[2], s[3])};
    } else {
      return TR::decode4(tile, c.p0, CB);
    }
  }
  template <int QB>
  static DEV void decode(const Raw &r, int q, u4 *B, const Ctx &c, int col) {
#pragma unroll
    for (int b = 0; b < QB; b++) {
      const uint32_t *t = c.buf + r.buf * PIECES * 4 + (2 * (q * QB + b) * NTC + col) * W;
      const u2 lo = decode4(t, c), hi = decode4(t + NTC * W, c);
      B[b] = u4{lo.x, lo.y, hi.x, hi.y};
    }
  }
  // Run r: half r % 2 of K tile r / 2; its word i belongs to lane group i.
  static DEV void place(u4 *step, int r, u4 v) {
    uint32_t *d = (uint32_t *)(step + (r >> 2) * 4) + ((r >> 1) & 1) * 2 + (r & 1);
#pragma unroll
    for (int i = 0; i < 4; i++) d[4 * i] = v[i];
  }
};

template <int KA, bool HALF, int CB>
static int exl3_rows(const void *xr, int dt, int M, int K, const int16_t *trellis, int N, void *ws, const QLayout &l, float *part,
                     int S, hipStream_t st) {
  using F = QExl3<KA, HALF, CB>;
  const int rc = launch_qimage<F>(xr, dt, M, K, ws, nullptr, (float *)((char *)ws + l.rs), st);
  if (rc) return rc;
  const QPlain<typename F::Args> p{{(const uint32_t *)trellis, N / 16}, M, N, Out{nullptr, 0, nullptr}, part};
  return launch_qgemm<F>(p, M, K, N, 1, S, ws, nullptr, st);
}

// part [S][M][N] = the K parts of xr (rotated, fp16 or bf16) . W; *rs: the bf16 rows' factors.
int exl3_rows_core(const void *xr, int dt, int M, int K, const int16_t *trellis, int N, int bits2, int cb, void *ws, float *part,
                   int S, const float **rs, hipStream_t st) {
  const QLayout l = qgemm_layout(M, K, N, false, qgemm_mt(8, M));
  *rs = dt == ISHZ_DT_BF16 ? (const float *)((char *)ws + l.rs) : nullptr;
#define ISHZ_E3(KA)                                                                                     \
  switch (cb) {                                                                                          \
  case 0: return exl3_rows<KA, false, 0>(xr, dt, M, K, trellis, N, ws, l, part, S, st);                   \
  case 1: return exl3_rows<KA, false, 1>(xr, dt, M, K, trellis, N, ws, l, part, S, st);                   \
  default: return exl3_rows<KA, false, 2>(xr, dt, M, K, trellis, N, ws, l, part, S, st);                  \
  }
  switch (bits2) {
  case 2: ISHZ_E3(1)
  case 3: return exl3_rows<1, true, 2>(xr, dt, M, K, trellis, N, ws, l, part, S, st);
  case 4: ISHZ_E3(2)
  case 5: return exl3_rows<2, true, 2>(xr, dt, M, K, trellis, N, ws, l, part, S, st);
  case 6: ISHZ_E3(3)
  case 7: return exl3_rows<3, true, 2>(xr, dt, M, K, trellis, N, ws, l, part, S, st);
  case 8: ISHZ_E3(4)
  case 10: ISHZ_E3(5)
  case 12: ISHZ_E3(6)
  case 14: ISHZ_E3(7)
  case 16: ISHZ_E3(8)
  }
#undef ISHZ_E3
  return decline("EXL3 rate");
}

}  // namespace ishz
