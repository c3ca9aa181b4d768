// Streaming MFMA GEMM for 2..16 rows over GGML super-blocks, sixteen rows per MFMA.
//
// The sub-scales of these formats are small integers, so a weight is d * (s q), s q an exact fp16 integer
// (|s q| <= 2048), or d * (s_hi q + s_lo q) with two such terms (Q6_K). Lane (n, g) decodes quarter g of
// row n's super-block with its own sub-scales folded in (one packed fp16 op per two weights), so
// all four lane groups of an MFMA 16x16x32 share the row's d, eight MFMAs (sixteen for Q6_K) run in one
// chain, and A holds sixteen rows of x. The verify kernel it takes over from (vgemm.h) keeps the lane
// groups' scales apart with a diagonal A: four rows an MFMA, the epilogue once per sub-unit and quad
// of rows. A min (Q4_K) is a small integer too: its term is the same chain with the sub-block's min as
// every weight, scaled by dmin.
//
// x lies in LDS as it lies in memory (rows 16 bytes apart in the banks), copied there by direct-to-LDS
// loads behind the first weights: the codes are decoded in natural order, a lane's eight weights of an
// MFMA being eight consecutive x of a row. Long rows come in chunks of K.
//
// 17408x5120 on MI355X, us against vgemm.h: 16 rows Q4_K 43.7 -> 22.4, Q6_K 52.7 -> 36.6, IQ2_XS 49.6 -> 21.7;
// 8 rows 22.0 -> 19.9, 34.8 -> 31.7, 26.4 -> 19.0; the time hardly grows with the rows.
//
// Work split as vgemm.h: a workgroup owns T tiles of 16 weight rows and one of S parts of K; its (tile,
// step) items go to its waves round robin (whole tiles once there are as many as waves).
#pragma once
#include "ggml_formats.h"
#include "qgemm.h"
#include "vgemm.h"

namespace ishz {

DEV u4 pk_mul4(u4 v, uint32_t m) {
  u4 o;
#pragma unroll
  for (int i = 0; i < 4; i++) o[i] = as_u32(as_h2(v[i]) * as_h2(m));
  return o;
}
DEV u4 pk_fma4(u4 v, uint32_t m, uint32_t a) {
  u4 o;
#pragma unroll
  for (int i = 0; i < 4; i++) o[i] = as_u32(__builtin_elementwise_fma(as_h2(v[i]), as_h2(m), as_h2(a)));
  return o;
}
DEV uint32_t h2_of(float v) {  // v (exact in fp16) in both halves
  const uint32_t h = f2h(v);
  return h | h << 16;
}

// Bytes 2 i, 2 i + 1 of v under the fp16 exponent of 1024: 1024 + byte in both halves.
template <int I>
DEV uint32_t bytes_1024(uint32_t v, uint32_t mg) {
  return __builtin_amdgcn_perm(v, mg, I ? 0x01070106u : 0x01050104u);
}

// A format: the verify format F (its loads and tables) with
//   NSPLIT                  operands per eight weights (1, or 2: each weight's two terms)
//   void wdecode(r, g, B[8 NSPLIT], mg, tabs)   s q, natural order
//   int wk(g, b)            where in the step the eight weights of MFMA b begin
//   float wscale(r)         d
//   MINS; uint32_t wmin(r, g, s), float wdmin(r)   the min of the MFMAs 4 s .. 4 s + 3, in both halves; -dmin
struct WQ4_K : FQ4_K {
  static constexpr int NSPLIT = 1;
  static constexpr bool MINS = true;
  static DEV void wdecode(const VRaw &r, int g, u4 *B, uint32_t mg, const u4 *) {
    const uint32_t q[8] = {r.q0.x, r.q0.y, r.q0.z, r.q0.w, r.q1.x, r.q1.y, r.q1.z, r.q1.w};
#pragma unroll
    for (int s = 0; s < 2; s++) {  // low nibbles 1024 + q, high ones 1024 + 16 q
      int sc, m;
      q4k_scale_min(r.h.y, r.h.z, r.h.w, 2 * g + s, sc, m);
      const uint32_t k = h2_of((float)sc * (s ? 0.0625f : 1.0f)), a = h2_of((float)sc * (s ? -64.0f : -1024.0f));
#pragma unroll
      for (int b = 0; b < 4; b++) {
        const uint32_t x = q[2 * b] & (s ? 0xF0F0F0F0u : 0x0F0F0F0Fu), y = q[2 * b + 1] & (s ? 0xF0F0F0F0u : 0x0F0F0F0Fu);
        B[4 * s + b] = pk_fma4(u4{bytes_1024<0>(x, mg), bytes_1024<1>(x, mg), bytes_1024<0>(y, mg), bytes_1024<1>(y, mg)}, k, a);
      }
    }
  }
  static DEV int wk(int g, int b) { return 64 * g + 8 * b; }
  static DEV float wscale(const VRaw &r) { return h2f(r.h.x & 0xffff); }
  static DEV uint32_t wmin(const VRaw &r, int g, int s) {
    int sc, m;
    q4k_scale_min(r.h.y, r.h.z, r.h.w, 2 * g + s, sc, m);
    return h2_of((float)m);
  }
  static DEV float wdmin(const VRaw &r) { return -h2f(r.h.x >> 16); }
};

struct WQ6_K : FQ6_K {
  static constexpr int NSPLIT = 2;
  static constexpr bool MINS = false;
  static DEV void wdecode(const VRaw &r, int g, u4 *B, uint32_t mg, const u4 *) {
    const uint32_t one = h2_of(1.0f), off = h2_of(-1056.0f);
#pragma unroll
    for (int s = 0; s < 4; s++) {
      const int bi = 8 * (g >> 1) + (g & 1) + 2 * s;  // the sub-scale, 16 hi + lo
      const int sc = (int8_t)(r.sc[bi >> 2] >> (8 * (bi & 3)));
      const uint32_t hi = h2_of((float)(sc & ~15)), lo = h2_of((float)(sc & 15));
#pragma unroll
      for (int h = 0; h < 2; h++) {
        uint32_t c[2];
#pragma unroll
        for (int t = 0; t < 2; t++) {  // four codes as bytes: a nibble of ql, two bits of qh
          const uint32_t l = (s & 1 ? r.ql1 : r.ql0)[2 * h + t], u = r.qh[2 * h + t];
          c[t] = and_or(s >= 2 ? l >> 4 : l, 0x0F0F0F0Fu, (s == 0 ? u << 4 : s == 1 ? u << 2 : s == 2 ? u : u >> 2) & 0x30303030u);
        }
        const u4 v = pk_fma4(u4{bytes_1024<0>(c[0], mg), bytes_1024<1>(c[0], mg), bytes_1024<0>(c[1], mg), bytes_1024<1>(c[1], mg)},
                             one, off);  // code - 32
        B[2 * (2 * s + h)] = pk_mul4(v, hi);
        B[2 * (2 * s + h) + 1] = pk_mul4(v, lo);
      }
    }
  }
  static DEV int wk(int g, int b) { return 128 * (g >> 1) + 16 * (g & 1) + 32 * (b >> 1) + 8 * (b & 1); }
  static DEV float wscale(const VRaw &r) { return h2f(r.d); }
};

struct WIQ2_XS : FIQ2_XS {
  static constexpr int NSPLIT = 1;
  static constexpr bool MINS = false;
  static DEV void wdecode(const VRaw &r, int, u4 *B, uint32_t mg, const u4 *tabs) {
    vdecode(r, B, mg, tabs, tabs + 512);
#pragma unroll
    for (int s = 0; s < 4; s++) {  // d (0.5 + nibble) / 4 = (d / 8)(2 nibble + 1), times a grid value up to 43
      const uint32_t k = h2_of((float)(2 * ((r.sc >> (4 * s)) & 15) + 1));
      B[2 * s] = pk_mul4(B[2 * s], k);
      B[2 * s + 1] = pk_mul4(B[2 * s + 1], k);
    }
  }
  static DEV int wk(int g, int b) { return 64 * g + 8 * b; }
  static DEV float wscale(const VRaw &r) { return 0.125f * h2f(r.d); }
};

// A problem P: vgemm.h's.
template <class F, class P, int D, int NW>
__global__ __launch_bounds__(64 * NW) void wgemm_kernel(P p, int K, int Kc, int T, int S) {
  typedef typename P::Group Group;
  Group gp;
  extern __shared__ __align__(16) u4 wlds[];
  if constexpr (requires { p.prologue(); }) p.prologue();  // every thread; ends with a barrier
  if (!p.group(blockIdx.y, gp)) return;
  const int lane = threadIdx.x & 63, wave = wave_id(), n = lane & 15, G = lane >> 4;
  const int N = p.rows(gp), ntiles = (N + 15) / 16;
  const int tb = (blockIdx.x / S) * T, te = min(tb + T, ntiles);
  if (tb >= te) return;
  const int split = blockIdx.x % S, ksteps = K / 256;
  const int kb = split * ksteps / S * 256, ke = (split + 1) * ksteps / S * 256, ntl = te - tb;
  const bool whole = T >= NW;  // a wave takes whole tiles; else the tiles' steps are dealt to the waves
  const int RW = Kc / 8 + 1;                      // 16-byte words of a row of x
  const int count = p.count(gp), R = min(16, count);
  float *outb = (float *)(wlds + R * RW);         // [tile][16 tokens][16 rows]
  f4 *accb = (f4 *)(outb + T * 256);              // [wave][tile][64], dealt steps only
  u4 *tabs = (u4 *)(accb + (whole ? 0 : NW * T * 64));
  const uint32_t mg = vconst(0x64006400u);
  for (int c0 = 0; c0 < count; c0 += 16) {
    const int M = min(16, count - c0);
    for (int kc0 = kb; kc0 < ke; kc0 += Kc) {
      const int klen = min(Kc, ke - kc0), steps = klen / 256;
      // item k of the wave: tile wave + NW (k / steps), step k % steps, or item wave + NW k of the
      // workgroup's (tile, step) sequence
      const int items = ntl * steps;
      const int cnt = whole ? (ntl > wave ? (ntl - wave + NW - 1) / NW : 0) * steps
                            : (items > wave ? (items - wave + NW - 1) / NW : 0);
      struct Cur {
        int tl, j;
      };
      auto next = [&](Cur c) {
        if (whole) {
          if (++c.j == steps) {
            c.j = 0;
            c.tl += NW;
          }
        } else {
          c.j += NW;
          while (c.j >= steps) {
            c.j -= steps;
            c.tl++;
          }
        }
        return c;
      };
      const Cur first = whole ? Cur{wave, 0} : Cur{wave / steps, wave % steps};
      typedef typename F::VRaw Raw;
      auto load = [&](const Cur &c, Raw &o) {
        const int row = min((tb + c.tl) * 16 + n, N - 1);
        o = F::vload(p.wrow(gp, row) + (size_t)(kc0 / 256) * F::VSTEP_BYTES, c.j, G);
      };
      Cur lc = first, cc = first;
      int lk = 0;  // past the wave's last item it is loaded again and dropped
      Raw ring[D];
      auto load_next = [&](Raw &o) {
        load(lc, o);
        if (lk < cnt - 1) {
          lc = next(lc);
          lk++;
        }
      };
      if (cnt > 0) {
#pragma unroll
        for (int d = 0; d < D - 1; d++) load_next(ring[d]);
      }
      for (int m = wave; m < M; m += NW) {
        const uint16_t *src = p.xrow(gp, c0 + m) + kc0 + 8 * lane;
        u4 *dst = wlds + m * RW;
        for (int k = 0; k < klen; k += 512, src += 512, dst += 64)
          if (k + 8 * lane < klen) load16_to_lds(src, dst);
      }
      if (c0 == 0 && kc0 == kb) F::vtables(tabs);
      if (kc0 == kb) {
        if (whole)
          for (int i = threadIdx.x; i < ntl * 256; i += 64 * NW) outb[i] = 0.0f;
        else
          for (int i = threadIdx.x; i < NW * T * 64; i += 64 * NW) accb[i] = f4{0, 0, 0, 0};
      }
      __syncthreads();  // (waits for the loads into LDS)

      const u4 *xr = wlds + min(n, M - 1) * RW;
      f4 acc = f4{0, 0, 0, 0};
      for (int k0 = 0; k0 < cnt; k0 += D) {
#pragma unroll
        for (int d = 0; d < D; d++) {
          if (k0 + d >= cnt) break;
          load_next(ring[(d + D - 1) % D]);
          const Raw &o = ring[d];
          h8 A[8];
#pragma unroll
          for (int b = 0; b < 8; b++) A[b] = as_h8(xr[(256 * cc.j + F::wk(G, b)) / 8]);
          u4 B[8 * F::NSPLIT];
          F::wdecode(o, G, B, mg, tabs);
          f4 C = f4{0, 0, 0, 0};
#pragma unroll
          for (int b = 0; b < 8; b++)
#pragma unroll
            for (int h = 0; h < F::NSPLIT; h++) C = mfma32(A[b], as_h8(B[b * F::NSPLIT + h]), C);
          if constexpr (F::MINS) {
            f4 m = f4{0, 0, 0, 0};
#pragma unroll
            for (int b = 0; b < 8; b++) {
              const uint32_t v = F::wmin(o, G, b >> 2);
              m = mfma32(A[b], as_h8(u4{v, v, v, v}), m);
            }
            const float dm = F::wdmin(o);
#pragma unroll
            for (int e = 0; e < 4; e++) acc[e] = fmaf(dm, m[e], acc[e]);
          }
          const float sc = F::wscale(o);
#pragma unroll
          for (int e = 0; e < 4; e++) acc[e] = fmaf(sc, C[e], acc[e]);
          const int tl = cc.tl;
          cc = next(cc);
          if (k0 + d + 1 == cnt || cc.tl != tl) {  // the wave's last item of the tile
            if (whole) {
#pragma unroll
              for (int e = 0; e < 4; e++) outb[tl * 256 + (4 * G + e) * 16 + n] += acc[e];
            } else {
              accb[(wave * T + tl) * 64 + lane] += acc;
            }
            acc = f4{0, 0, 0, 0};
          }
        }
      }
      __syncthreads();  // parts in LDS; x is free for the next chunk
    }
    if (!whole) {  // the waves' parts, in wave order
      for (int i = threadIdx.x; i < ntl * 64; i += 64 * NW) {
        const int tl = i >> 6, l = i & 63;
        f4 v = accb[tl * 64 + l];
        for (int w = 1; w < NW; w++) v += accb[(w * T + tl) * 64 + l];
#pragma unroll
        for (int e = 0; e < 4; e++) outb[tl * 256 + (4 * (l >> 4) + e) * 16 + (l & 15)] = v[e];
      }
      __syncthreads();
    }
    p.finish(gp, c0, M, tb, te, outb);
    __syncthreads();
  }
}

// LDS of a workgroup: R rows of Kc values, T tiles.
template <class F, int NW>
static size_t wgemm_lds(int R, int Kc, int T) {
  return (size_t)R * (Kc * 2 + 16) + (size_t)T * 1024 + (T >= NW ? 0 : (size_t)NW * T * 1024) + F::tab_bytes();
}
// rmax: the most rows a group has. The chunk of K: the part divided into the fewest equal chunks that fit.
// Ring depth 2 and eight waves: depth 3 and 10, 12 or 16 waves measured within 5 % or slower
// (17408x5120, 16 rows: Q4_K 22.5 us against 23.1 / 23.4 / 21.9 / 24.0, Q6_K 36.9 against 39.5 / 37.6 / 36.2 / 50.6).
template <class F, class P, int D = 2, int NW = 8>
static int launch_wgemm(const P &p, int rmax, int K, int rows, int groups, int T, int S, hipStream_t st) {
  const int steps = (K / 256 + S - 1) / S, R = std::min(16, rmax);
  int nc = 1;
  while (nc < steps && wgemm_lds<F, NW>(R, (steps + nc - 1) / nc * 256, T) > 150 * 1024) nc++;
  const int Kc = (steps + nc - 1) / nc * 256;
  const size_t lds = wgemm_lds<F, NW>(R, Kc, T);
  if (lds > 150 * 1024) return decline("verify x does not fit in LDS");
  hipLaunchKernelGGL((wgemm_kernel<F, P, D, NW>), dim3(((rows + 15) / 16 + T - 1) / T * S, groups), dim3(64 * NW), lds, st, p, K, Kc,
                     T, S);
  ISHZ_LAUNCH_CHECK("verify launch");
  return ISHZ_OK;
}

// Tiles per workgroup T and parts of K S: one workgroup per CU, the split with the fewest (tile, step)
// items in the fullest one; parts (a sum launch of about 3 us) only where they take more than a
// fifth off. Up to 16 tiles a workgroup.
inline int wgemm_tiles(int N, int S, int cus) { return std::min(16, std::max(1, ((N + 15) / 16 * S + cus - 1) / cus)); }
inline int wgemm_splits(int K, int N, int cus, int &T) {
  const int ntiles = (N + 15) / 16, steps = K / 256;
  auto items = [&](int S) {
    const int t = wgemm_tiles(N, S, cus);
    const int rounds = ((ntiles + t - 1) / t * S + cus - 1) / cus;
    return rounds * t * ((steps + S - 1) / S);
  };
  int best = 1;
  for (int S = 2; S <= 8 && S <= steps / 4; S++)
    if (items(S) * 5 < items(1) * 4 && items(S) < items(best)) best = S;
  T = wgemm_tiles(N, best, cus);
  return best;
}
inline size_t wgemm_part_bytes(int M, int K, int N, int cus) {
  int T;
  const int S = wgemm_splits(K, N, cus, T);
  return S > 1 ? (size_t)S * M * N * 4 : 0;
}

// y[M][N] = x[M][K] . W^T, M <= 16, x fp16 (or bf16's image, see act_prepare). ws: room for the K parts, else K
// is not split.
template <class F>
static int wgemm(const void *x, int M, int K, const void *w, int N, const Out &y, void *ws, size_t ws_bytes, hipStream_t st) {
  int T, rc;
  int S = wgemm_splits(K, N, gemv_num_cu(), T);
  if (S > 1 && (!ws || ws_bytes < (size_t)S * M * N * 4)) {
    S = 1;
    T = wgemm_tiles(N, 1, gemv_num_cu());
  }
  float *part = S > 1 ? (float *)ws : nullptr;
  const VPlain p{(const uint16_t *)x, (const uint8_t *)w, (size_t)(K / F::BS) * F::TS, M, K, N, y, part, S};
  if ((rc = launch_wgemm<F>(p, M, K, N, 1, T, S, st)) || S == 1) return rc;
  const size_t n = (size_t)M * N;
  hipLaunchKernelGGL(vgemm_sum_kernel, dim3((unsigned)std::min<size_t>((n + 255) / 256, 2048)), dim3(256), 0, st, part, S, n, N, y);
  ISHZ_LAUNCH_CHECK("verify sum launch");
  return ISHZ_OK;
}

}  // namespace ishz
