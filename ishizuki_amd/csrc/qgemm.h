// Matrix product of many activation rows with packed weights, y[M][N] = x[M][K] . W[N][K]^T: prompts
// (more than 16 rows), where the streaming kernels would read and decode the weights again for every
// sixteen rows.
//
// Bound: instruction issue, the matrix cores beside the decode and the scaling. A workgroup (4 waves) owns
// up to 16 MT rows of x and 64 NT columns; a wave holds 16 NT of the columns for all of the rows, so every
// weight is decoded by one wave of one workgroup per 16 MT rows, straight from its packed words into
// MFMA B operands, and each 16x16x32 MFMA multiplies sixteen rows (the verify kernel's diagonal A takes
// four). 17408x5120: 2-bit affine with the rotation, 300 rows 716 -> 99 us (19 calls of 16 rows
// before; 105-108 over three weights in turn), 4-bit affine, 512 rows 170 us (537 TFLOP/s); EXL3 2-bit, 128
// rows 275 -> 59 us (64-66 over three weights).
//
// x comes as an image (qimage_kernel): one row per token, each 256-step of it reordered into the A
// operands of its 8 MFMAs (16 bytes per lane group g, at piece 4 b + g of the step), so a wave moves
// an operand into LDS with one load of sixteen rows' 64-byte runs; rows may be gathered in any order
// (routed experts). A chunk is two MFMAs' worth (K = 64) of every row; three or four are in LDS, and the
// weights come a step ahead, all by direct-to-LDS loads: a register load in the loop made the compiler
// wait for every load under way once a step, the prefetched chunks too (it does not count direct
// loads), so the waits here are counted by hand.
//
// Scales (affine packs). B holds exact small integers and the fp32 scale multiplies C: a chunk's two MFMAs
// share one scale per column (a lane's C column is its own weight row). The biases go through one fp32 MFMA
// 16x16x4 a step on the image's four fp32 sums of x, so nothing is narrowed on the way: the same
// exact products, fp32 sums, as the kernels for up to 16 rows.
//
// A format F provides:
//   Args, Ctx (per-wave constants), Raw (a column tile's step in registers)
//   void fetch<NT>(args, ctx, j, buf)    a step's weights of the wave's NT column tiles into its LDS, WOPS
//                                        loads per tile at least, issued at chunk WQ of the step before
//   Raw raw<NT>(ctx, j, c)               column tile c's share of lane group g, read from there
//   void decode<QB>(raw, q, B[QB], ctx, c)   the B operands of chunk q (MFMAs QB q .. QB q + QB - 1)
//   SCALED                               weights in groups of 64, each with a scale and a bias; else the MFMAs
//                                        add straight into the sums
//   float scale(raw, q), bias(raw)       the scale of chunk q, and the bias of lane group g's 64 weights
//   void place(step, r, v)               where the image holds values 8 r .. 8 r + 7 of a step
//   OCC                                  workgroups of 64 rows a CU is to hold (registers). 6-bit packs with fp16
//                                        scales spill three registers at three, which is ahead all the
//                                        same: 17408x5120, 300 / 512 rows 124 / 193 us against 135 / 211 at two
//                                        (64 rows 53 against 52; 4096x4096, 64 / 300 rows 28 / 43 against 26 / 41)
//   MT_MAX                               8 where the decode outweighs the products (see qgemm_mt), else 4
#pragma once
#include <algorithm>

#include "affine_fmt.h"
#include "affine_nbit.h"
#include "common.h"

namespace ishz {

int gemv_num_cu();
__global__ void vgemm_sum_kernel(const float *__restrict__ part, int S, size_t n, int N, Out y);

// 16 or 4 bytes per lane straight into LDS, lane after lane from `lds` (uniform). Functions of their own:
// the builtin takes no template-dependent argument.
DEV void load16_to_lds(const void *src, void *lds) {
  __builtin_amdgcn_global_load_lds(src, (__attribute__((address_space(3))) void *)lds, 16, 0, 0);
}
DEV void load4_to_lds(const void *src, void *lds) {
  __builtin_amdgcn_global_load_lds(src, (__attribute__((address_space(3))) void *)lds, 4, 0, 0);
}

// ------------------------------------------------------------------------------- the x image
// One workgroup per row: bf16 rows scaled to fp16 by a power of two (see act_prepare), then every
// run of eight values moved to its place in the A operands, and the sums of x that the format's
// biases multiply. Bound by latency, as act_half_kernel: a thread's loads are all in flight at once.
template <class F>
__global__ __launch_bounds__(1024) void qimage_kernel(const uint16_t *__restrict__ x, int bf16, int K,
                                                      u4 *__restrict__ img, float *__restrict__ X, float *__restrict__ rs) {
  __shared__ uint32_t wmax[16];
  constexpr int U = 4;
  const int n8 = K / 8, nt = blockDim.x;  // K a multiple of 256: whole waves hold whole steps
  const uint8_t *src = (const uint8_t *)(x + (size_t)blockIdx.x * K);
  img += (size_t)blockIdx.x * n8;
  X += (size_t)blockIdx.x * (K / 256) * 4;
  u4 v[U];
  auto load = [&](int i0) {
#pragma unroll
    for (int u = 0; u < U; u++) v[u] = ld16<2>(src + 16 * (size_t)min(i0 + u * nt, n8 - 1));
  };
  float down = 1.0f;
  if (bf16) {
    uint32_t m = 0;
    for (int i0 = threadIdx.x; i0 < n8; i0 += U * nt) {
      load(i0);
#pragma unroll
      for (int u = 0; u < U; u++) m = bf16_absmax(v[u], m);
    }
    const int e = bf16_row_exponent(block_absmax(m, wmax));
    down = ldexpf(1.0f, -e);
    if (threadIdx.x == 0) rs[blockIdx.x] = ldexpf(1.0f, e);
  }
  for (int i0 = threadIdx.x; i0 < n8; i0 += U * nt) {
    if (!bf16 || n8 > U * nt) load(i0);
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int q = i0 + u * nt;
      if (q >= n8) break;  // whole groups of 32 lanes leave together
      const u4 h = bf16 ? bf16_to_half8(v[u], down) : v[u];
      F::place(img + (q & ~31), q & 31, h);
      if constexpr (F::SCALED) {  // the sum of each 64 values
        float s = 0.0f;
#pragma unroll
        for (int e = 0; e < 4; e++) s = dot2(h[e], 0x3C003C00u, s);
        s += ISHZ_DPP(s, 0xB1);
        s += ISHZ_DPP(s, 0x4E);
        s += ISHZ_DPP(s, 0x141);
        if ((q & 7) == 0) X[q >> 3] = s;
      }
    }
  }
}

// ------------------------------------------------------------------------------- the product
// At most N vector-memory operations of this wave still under way, its LDS reads done, then the
// workgroup's barrier. (__syncthreads would wait for every load, the prefetched ones too.)
#define ISHZ_WAIT_BARRIER(N) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory")

// Row block y of mb takes row tiles block_tile0(n, mb, y) .. block_tile0(n, mb, y + 1) - 1 of n, dealt evenly:
// quotient plus remainder, as n * y leaves 32 bits at about 1.5 million rows.
__host__ __device__ constexpr int block_tile0(int n, int mb, int y) { return n / mb * y + (y < n % mb ? y : n % mb); }
constexpr int QROWS_MAX = 65535 * 64;  // rows of one call: the row blocks of 64 a grid holds
static_assert(block_tile0(QROWS_MAX / 16, 65535, 65535) == QROWS_MAX / 16 && block_tile0(QROWS_MAX / 16, 32768, 32767) == QROWS_MAX / 16 - 7,
              "the last blocks of the largest call");
static_assert(block_tile0(9, 2, 1) == 5 && block_tile0(7, 2, 1) == 4 && block_tile0(5, 5, 3) == 3, "no block over ceil(n / mb)");
// Whether the rotation of M rows of K values, 512 to a workgroup (or one larger Hadamard block), is one launch:
// less than 2^32 threads, workgroups of 256. The rotations have no loop over workgroups.
constexpr bool one_rotation(int M, int K, int block = 128) {
  const size_t per = block > 128 ? block : 512;
  return ((size_t)M * K + per - 1) / per < (size_t)1 << 24;
}

// A problem P: bool group(z, Group &); int count(g) rows of x, rows(g) weight rows; size_t src(g, i)
// the image row of row i; F::Args weights(g); Row row(g, i), what is to be known of output row i; void
// put(g, row, c, v, part) one output (of part blockIdx.x % S of K), or void put2(g, row, o, v0, v1), column o = n of
// the wave's first column tile and of its second.
template <class F, class P, int MT, int NT>
__global__ __launch_bounds__(256, MT == 4 ? F::OCC : 2) void qgemm_kernel(P p, const u4 *__restrict__ img, const float *__restrict__ X, int K, int S) {
  constexpr bool RAGGED = requires { P::RAGGED; };
  constexpr int QB = 2, NB = MT == 4 ? 3 : 4, CPS = 8 / QB;  // MFMAs per chunk, chunks in LDS, chunks per step
  static_assert(MT % 4 == 0, "four waves stage the row tiles");
  static_assert(F::WQ + NB - 1 < CPS, "a step's weights are requested before its first chunk of x, whose wait covers them");
  extern __shared__ __align__(16) u4 qlds[];
  typename P::Group gp;
  if (!p.group(blockIdx.z, gp)) return;
  const int lane = threadIdx.x & 63, wave = wave_id(), n = lane & 15, g = lane >> 4;
  const int count = p.count(gp), N = p.rows(gp), steps = K / 256;
  // row tiles dealt evenly to the workgroups of a column block
  const int mtiles = (count + 15) / 16, mb = (mtiles + MT - 1) / MT;
  if ((int)blockIdx.y >= mb) return;
  const int part = blockIdx.x % S, c0 = (blockIdx.x / S * 4 + wave) * 16 * NT;
  const int jb = part * steps / S, je = (part + 1) * steps / S;  // this part's steps of K
  u4 *abuf = qlds;                                  // [NB][MT][QB][64]
  float *xbuf = (float *)(abuf + NB * MT * QB * 64);     // [2][MT][64], SCALED
  char *extra = (char *)(xbuf + 2 * F::SCALED * MT * 64);
  const auto w = p.weights(gp);
  const typename F::Ctx ctx(w, extra, wave, lane, c0, N, NT);

  for (int y = blockIdx.y; y < mb; y += gridDim.y) {  // (one pass where the grid covers every row)
    const int t0 = block_tile0(mtiles, mb, y), mt = block_tile0(mtiles, mb, y + 1) - t0;
    const u4 *abase[MT / 4];
    const float *xbase[MT / 4];
#pragma unroll
    for (int tt = 0; tt < MT / 4; tt++) {
      const size_t s = p.src(gp, min(16 * (t0 + wave + 4 * tt) + n, count - 1));
      abase[tt] = img + s * (K / 8) + g;
      xbase[tt] = X + s * steps * 4 + g;
    }
    // chunk c of every row tile (and with a step's first chunk its sums) into buffer c % NB; past the end
    // the last one again, so that the number of loads under way is always known
    const int cend = je * CPS - 1;
    auto stage = [&](int c) {
      const int cc = min(c, cend);
      u4 *dst = abuf + ((c % NB) * MT + wave) * QB * 64;
#pragma unroll
      for (int tt = 0; tt < MT / 4; tt++)
#pragma unroll
        for (int b = 0; b < QB; b++) load16_to_lds(abase[tt] + (cc * QB + b) * 4, dst + (4 * tt * QB + b) * 64);
      if (F::SCALED && c % CPS == 0)
#pragma unroll
        for (int tt = 0; tt < MT / 4; tt++)
          load4_to_lds(xbase[tt] + cc / CPS * 4, xbuf + (((c / CPS) & 1) * MT + wave + 4 * tt) * 64);
    };

    f4 acc[MT][NT];
#pragma unroll
    for (int t = 0; t < MT; t++)
#pragma unroll
      for (int c = 0; c < NT; c++) acc[t][c] = f4{0, 0, 0, 0};
    F::template fetch<NT>(w, ctx, jb, jb);
#pragma unroll
    for (int d = 0; d < NB - 1; d++) stage(jb * CPS + d);
    typename F::Raw cur[NT];
    for (int j = jb; j < je; j++) {
#pragma unroll
      for (int q = 0; q < CPS; q++) {
        // Chunk c = CPS j + q is here and the buffer of chunk c - 1 is free. Loads issued after c's own
        // iteration c - (NB - 1): the chunks of the NB - 2 iterations since, with a step's sums among them
        // where one began, and the weights of the step after next (issued at q = 0).
        constexpr int D = NB - 1;
        auto pending = [](int q) constexpr {
          int v = 0;
          for (int i = 1; i < NB - 1; i++) {  // iteration c - i staged chunk c - i + D
            v += MT * QB / 4;
            if ((q - i + D + 8 * CPS) % CPS == 0) v += F::SCALED * MT / 4;
            if ((q - i + 8 * CPS) % CPS == F::WQ) v += F::WOPS * NT;
          }
          return v;
        };
        if (q == 0) ISHZ_WAIT_BARRIER(pending(0));
        else if (q == 1) ISHZ_WAIT_BARRIER(pending(1));
        else if (q == 2) ISHZ_WAIT_BARRIER(pending(2));
        else ISHZ_WAIT_BARRIER(pending(3));
        stage(j * CPS + q + D);
        if (q == F::WQ) F::template fetch<NT>(w, ctx, min(j + 1, je - 1), j + 1);
        if (q == 0)
#pragma unroll
          for (int c = 0; c < NT; c++) cur[c] = F::template raw<NT>(ctx, j, c);
        const u4 *ab = abuf + ((j * CPS + q) % NB) * MT * QB * 64 + lane;
        h8 AA[2][QB];
#pragma unroll
        for (int b = 0; b < QB; b++) AA[0][b] = as_h8(ab[b * 64]);
        u4 B[NT][QB];
#pragma unroll
        for (int c = 0; c < NT; c++) F::template decode<QB>(cur[c], q, B[c], ctx, c);
        float sc[NT];
        if constexpr (F::SCALED)
#pragma unroll
          for (int c = 0; c < NT; c++) sc[c] = F::scale(cur[c], q);
        // tile t's operands are read a tile ahead; RAGGED: pairs of tiles past the workgroup's rows are left
        // out (groups of any size; the branches cost a plain product 3 %)
#pragma unroll
        for (int t = 0; t < MT; t++) {
          if (RAGGED && t % 2 == 0 && t >= mt) break;
          const h8 *A = AA[t & 1];
          if (t + 1 < MT)
#pragma unroll
            for (int b = 0; b < QB; b++) AA[(t + 1) & 1][b] = as_h8(ab[((t + 1) * QB + b) * 64]);
          __builtin_amdgcn_sched_barrier(0);
          f4 T[NT];
#pragma unroll
          for (int b = 0; b < QB; b++)
#pragma unroll
            for (int c = 0; c < NT; c++) {
              f4 &o = F::SCALED ? T[c] : acc[t][c];
              o = mfma32(A[b], as_h8(B[c][b]), F::SCALED && b == 0 ? f4{0, 0, 0, 0} : o);
            }
          if constexpr (F::SCALED)
#pragma unroll
            for (int c = 0; c < NT; c++)
#pragma unroll
              for (int e = 0; e < 4; e++) acc[t][c][e] = fmaf(sc[c], T[c][e], acc[t][c][e]);
        }
      }
      if constexpr (F::SCALED) {
        const float *xb = xbuf + (j & 1) * MT * 64 + lane;
        float bv[NT];
#pragma unroll
        for (int c = 0; c < NT; c++) bv[c] = F::bias(cur[c]);
#pragma unroll
        for (int t = 0; t < MT; t++) {
          if (RAGGED && t % 2 == 0 && t >= mt) break;
#pragma unroll
          for (int c = 0; c < NT; c++) acc[t][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(xb[t * 64], bv[c], acc[t][c], 0, 0, 0);
        }
      }
    }
    ISHZ_WAIT_BARRIER(0);  // nothing still on its way to LDS when the workgroup ends
    // every output row's place and factor first (loads for the gathered problems), then the stores. The loads end
    // here: to the compiler one of them could be under way still in the next pass, and it put a wait for every
    // load, the prefetched chunks too, into each step of K (MoE down, by chance of the registers).
    typename P::Row at[MT][4];
#pragma unroll
    for (int t = 0; t < MT; t++)
#pragma unroll
      for (int e = 0; e < 4; e++) at[t][e] = p.row(gp, min(16 * (t0 + t) + 4 * g + e, count - 1));
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
#pragma unroll
    for (int t = 0; t < MT; t++) {
      if (t >= mt) break;
#pragma unroll
      for (int e = 0; e < 4; e++) {
        if (16 * (t0 + t) + 4 * g + e >= count) continue;
        if constexpr (requires { p.put2(gp, at[0][0], 0, 0.0f, 0.0f); }) {  // the wave's two column tiles go together
          p.put2(gp, at[t][e], c0 / 2 + n, acc[t][0][e], acc[t][1][e]);
        } else {
#pragma unroll
          for (int c = 0; c < NT; c++)
            if (c0 + 16 * c + n < N) p.put(gp, at[t][e], c0 + 16 * c + n, acc[t][c][e], part);
        }
      }
    }
  }
}

// ------------------------------------------------------------------------------- the plain problem
// One matrix, rows 0 .. M - 1 of the image. With S > 1 the parts' products go to part [S][M][N] (fp32).
template <class A>
struct QPlain {
  A w;
  int M, N;
  Out y;
  float *part;
  struct Group {};
  DEV bool group(int, Group &) const { return true; }
  DEV int count(const Group &) const { return M; }
  DEV int rows(const Group &) const { return N; }
  DEV size_t src(const Group &, int i) const { return i; }
  DEV A weights(const Group &) const { return w; }
  typedef int Row;
  DEV Row row(const Group &, int i) const { return i; }
  DEV void put(const Group &, Row i, int c, float v, int s) const {
    if (part) part[((size_t)s * M + i) * N + c] = v;
    else y.put((size_t)i * N + c, i, v);
  }
};

constexpr int QNT = 2;  // column tiles per wave: 128 columns a workgroup

// Workspace: the image, its sums, the bf16 rows' factors, then the K parts.
struct QLayout {
  size_t X, rs, part, bytes;
};
inline size_t q256(size_t b) { return (b + 255) / 256 * 256; }
// Row tiles of a workgroup: eight for the formats whose decode costs most beside it (EXL3) once there are
// that many rows, else four, which leaves LDS and registers for three workgroups a CU instead of two.
inline int qgemm_mt(int mt_max, int M) { return mt_max == 8 && M > 64 ? 8 : 4; }
// Parts of K: none once every CU has a workgroup; below that enough to fill the CUs, at least four
// steps a part and at most 16.
inline int qgemm_splits(int M, int K, int N, int mt, int cus) {
  const int blocks = (N + 64 * QNT - 1) / (64 * QNT) * ((M + 16 * mt - 1) / (16 * mt));
  if (blocks >= cus) return 1;
  return std::max(1, std::min({2 * cus / blocks, K / 256 / 4, 16}));
}
inline QLayout qgemm_layout(int M, int K, int N, bool scaled, int mt) {
  QLayout l;
  const int S = qgemm_splits(M, K, N, mt, gemv_num_cu());
  l.X = q256((size_t)M * K * 2);
  l.rs = l.X + q256((size_t)M * (K / 256) * scaled * 16);
  l.part = l.rs + q256((size_t)M * 4);
  l.bytes = l.part + (S > 1 ? q256((size_t)S * M * N * 4) : 0);
  return l;
}

template <class F>
static int launch_qimage(const void *x, int dt, int M, int K, void *img, float *X, float *rs, hipStream_t st) {
  const int nt = std::min(1024, K / 8);
  hipLaunchKernelGGL((qimage_kernel<F>), dim3(M), dim3((nt + 63) / 64 * 64), 0, st, (const uint16_t *)x, dt == ISHZ_DT_BF16, K,
                     (u4 *)img, X, rs);
  ISHZ_LAUNCH_CHECK("activation image launch");
  return ISHZ_OK;
}

template <class F, class P, int MT>
static int launch_qgemm_mt(const P &p, int mmax, int mbs, int K, int N, int groups, int S, const void *img, const float *X, hipStream_t st) {
  const size_t lds = (size_t)(MT == 4 ? 3 : 4) * MT * 2 * 64 * 16 + (size_t)2 * F::SCALED * MT * 64 * 4 + F::lds_bytes(QNT);
  hipLaunchKernelGGL((qgemm_kernel<F, P, MT, QNT>),
                     dim3((N + 64 * QNT - 1) / (64 * QNT) * S, mbs ? mbs : (mmax + 16 * MT - 1) / (16 * MT), groups), dim3(256), lds, st, p,
                     (const u4 *)img, X, K, S);
  ISHZ_LAUNCH_CHECK("many-row matmul launch");
  return ISHZ_OK;
}
// mmax: the most rows a group can have; mbs: the row blocks to launch where few groups will have that many
// (0: all; a workgroup takes every mbs-th block).
template <class F, class P>
static int launch_qgemm(const P &p, int mmax, int K, int N, int groups, int S, const void *img, const float *X, hipStream_t st,
                        int mbs = 0) {
  if constexpr (F::MT_MAX == 8)
    if (qgemm_mt(8, mmax) == 8) return launch_qgemm_mt<F, P, 8>(p, mmax, mbs, K, N, groups, S, img, X, st);
  return launch_qgemm_mt<F, P, 4>(p, mmax, mbs, K, N, groups, S, img, X, st);
}

// ------------------------------------------------------------------------------- MLX affine packs
// Even widths. Lane (n, g) loads group 4 j + g of row n; a 4x4 transpose of words between the lane groups
// (two row swaps per pair of registers) leaves lane group g with words g WPL .. of all four groups,
// sixteen codes of each: the four lane groups of an MFMA then share one scale. Codes become exact
// fp16 integers: masked under the exponent of 1024, and 1024 taken off again.
DEV void transpose4(uint32_t &a, uint32_t &b, uint32_t &c, uint32_t &d) {
  const auto p = __builtin_amdgcn_permlane32_swap(a, c, false, false), q = __builtin_amdgcn_permlane32_swap(b, d, false, false);
  const auto r = __builtin_amdgcn_permlane16_swap(p[0], q[0], false, false), s = __builtin_amdgcn_permlane16_swap(p[1], q[1], false, false);
  a = r[0], b = r[1], c = s[0], d = s[1];
}
DEV uint32_t pk_fma(uint32_t t, float m, float a) {  // halves t * m + a (exact here)
  const _Float16 mh = (_Float16)m, ah = (_Float16)a;
  return as_u32(__builtin_elementwise_fma(as_h2(t), h2{mh, mh}, h2{ah, ah}));
}

template <int BITS, int GS, bool BF16S>
struct QAffine {
  static constexpr bool SCALED = true;
  static constexpr int WPL = BITS / 2, MT_MAX = 4, OCC = BITS == 8 ? 2 : 3, WOPS = WPL + 1;
  // a wave's step of weights in LDS (read into registers with the step's first chunk, so the next step's
  // loads follow from the second one on), per column tile: 16 rows of 32 BITS bytes of codes, then the
  // rows' scales and biases of the step (8 bytes each; 4 for groups of 128)
  static constexpr int TILE = 512 * BITS + 256, WQ = 1;
  static size_t lds_bytes(int nt) { return (size_t)4 * nt * TILE; }
  // Args: anything with AffRow arow(row)
  struct Args {
    const uint32_t *codes;
    const uint16_t *scales, *biases;
    int K;
    DEV AffRow arow(int row) const {
      return {codes + (size_t)row * (K * BITS / 32), scales + (size_t)row * (K / GS), biases + (size_t)row * (K / GS)};
    }
  };
  struct Ctx {
    char *buf;
    int lane, c0, N;
    uint32_t mg;
    template <class A>
    DEV Ctx(const A &, char *extra, int wave, int lane_, int c0_, int N_, int nt)
          : buf(extra + wave * nt * TILE), lane(lane_), c0(c0_), N(N_), mg(vconst(0x64006400u)) {}
  };
  struct Raw {
    uint32_t w[4 * WPL];
    uint32_t s[2];
    uint32_t b;
  };
  static DEV float ld_s(uint32_t v) { return BF16S ? __builtin_bit_cast(float, v << 16) : h2f(v); }
  template <int NT, class A>
  static DEV void fetch(const A &a, const Ctx &c, int j, int) {
#pragma unroll
    for (int t = 0; t < NT; t++) {
      char *dst = c.buf + t * TILE;
#pragma unroll
      for (int i = 0; i < WPL; i++) {
        const int q = i * 64 + c.lane, row = min(c.c0 + 16 * t + q / (2 * BITS), c.N - 1);
        load16_to_lds(a.arow(row).codes + j * 8 * BITS + (q % (2 * BITS)) * 4, dst + i * 1024);
      }
      // lanes 0..31 the scales, 32..63 the biases: dword l % 2 of row l / 2 (groups of 128: one dword)
      const int l = c.lane & 31, row = min(c.c0 + 16 * t + (l >> 1), c.N - 1);
      const AffRow ar = a.arow(row);
      const uint16_t *p = (c.lane < 32 ? ar.scales : ar.biases) + j * (256 / GS) + (GS == 64 ? 2 * (l & 1) : 0);
      load4_to_lds(p, dst + 512 * BITS);
    }
  }
  template <int NT>
  static DEV Raw raw(const Ctx &c, int, int t) {
    const char *src = c.buf + t * TILE;
    const int n = c.lane & 15, g = c.lane >> 4;
    Raw r;
#pragma unroll
    for (int i = 0; i < WPL; i++) {
      const u4 v = *(const u4 *)(src + n * 32 * BITS + g * 8 * BITS + 16 * i);
      r.w[4 * i] = v.x, r.w[4 * i + 1] = v.y, r.w[4 * i + 2] = v.z, r.w[4 * i + 3] = v.w;
    }
    const u2 s = *(const u2 *)(src + 512 * BITS + 8 * n);
    r.s[0] = s.x, r.s[1] = s.y;
    r.b = *(const uint16_t *)(src + 512 * BITS + 128 + 8 * n + 2 * (GS == 64 ? g : g / 2));
    return r;
  }
  static DEV float scale(const Raw &r, int s) {
    const int i = GS == 64 ? s : s / 2;
    return ld_s((r.s[i >> 1] >> (16 * (i & 1))) & 0xffffu);
  }
  static DEV float bias(const Raw &r) { return ld_s(r.b); }
  template <int QB>
  static DEV void decode(Raw &r, int q, u4 *B, const Ctx &c, int) {
    if (q == 0)
#pragma unroll
      for (int x = 0; x < WPL; x++) transpose4(r.w[x], r.w[WPL + x], r.w[2 * WPL + x], r.w[3 * WPL + x]);
    const uint32_t mg = c.mg;
#pragma unroll
    for (int t = 0; t < QB / 2; t++) {
      const uint32_t *w = r.w + (q * (QB / 2) + t) * WPL;
      if constexpr (BITS == 2) {
        const uint32_t a = w[0], a10 = a >> 10;
        B[2 * t] = u4{pk_fma(and_or(a, 0x00030003u, mg), 1.0f, -1024.0f), pk_fma(and_or(a, 0x000C000Cu, mg), 0.25f, -256.0f),
                      pk_fma(and_or(a, 0x00300030u, mg), 0.0625f, -64.0f), pk_fma(and_or(a, 0x00C000C0u, mg), 0.015625f, -16.0f)};
        B[2 * t + 1] = u4{pk_fma(and_or(a, 0x03000300u, mg), 0.00390625f, -4.0f), pk_fma(and_or(a10, 0x00030003u, mg), 1.0f, -1024.0f),
                          pk_fma(and_or(a10, 0x000C000Cu, mg), 0.25f, -256.0f), pk_fma(and_or(a10, 0x00300030u, mg), 0.0625f, -64.0f)};
      } else {
#pragma unroll
        for (int s = 0; s < 2; s++)
#pragma unroll
          for (int i = 0; i < 4; i++) {
            uint32_t v;
            if constexpr (BITS == 4) {
              v = and_or(w[s] >> (4 * i), 0x000F000Fu, mg);
            } else if constexpr (BITS == 8) {
              v = and_or(w[2 * s + (i >> 1)] >> (8 * (i & 1)), 0x00FF00FFu, mg);
            } else {  // 6 bits: codes 2 j, 2 j + 1 of the sixteen are 12 bits of the three words
              const int o = 12 * (4 * s + i), wi = o >> 5, sh = o & 31;
              const uint32_t win = sh + 12 <= 32 ? w[wi] >> sh : __builtin_amdgcn_alignbit(w[wi + 1], w[wi], sh);
              v = ((win >> 6) & 63u) << 16 | and_or(win, 63u, mg);
            }
            B[2 * t + s][i] = pk_fma(v, 1.0f, -1024.0f);
          }
      }
    }
  }
  // Image: run r of eight values of the step is group r / 8, lane group (r / 2) % 4, MFMA 2 (r / 8) + r % 2;
  // 2 bits: a word's pairs are values p and p + 8, so neighbouring runs interleave.
  static DEV void place(u4 *step, int r, u4 v) {
    const int s = r & 1, dst = (2 * (r >> 3) + s) * 4 + ((r >> 1) & 3);
    if constexpr (BITS == 2) {
      const uint32_t k0 = s ? v.z : v.x, k1 = s ? v.w : v.y, o0 = s ? v.x : v.z, o1 = s ? v.y : v.w;
      const uint32_t p0 = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)o0, 0xB1, 0xf, 0xf, true);  // lane ^ 1
      const uint32_t p1 = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)o1, 0xB1, 0xf, 0xf, true);
      // this lane's MFMA s: values 4 s .. 4 s + 3 of the even run (lo) beside those of the odd one (hi)
      const uint32_t l0 = s ? p0 : k0, l1 = s ? p1 : k1, h0 = s ? k0 : p0, h1 = s ? k1 : p1;
      v = u4{(l0 & 0xffffu) | h0 << 16, (l0 >> 16) | (h0 & 0xffff0000u), (l1 & 0xffffu) | h1 << 16, (l1 >> 16) | (h1 & 0xffff0000u)};
    } else if constexpr (BITS == 4) {
      v = u4{(v.x & 0xffffu) | (v.z << 16), (v.x >> 16) | (v.z & 0xffff0000u), (v.y & 0xffffu) | (v.w << 16), (v.y >> 16) | (v.w & 0xffff0000u)};
    } else if constexpr (BITS == 8) {
      v = perm0213(v);
    }
    step[dst] = v;
  }
};

}  // namespace ishz
