// Prompt-pass GEMM on packed int8 weights (gfx950 MFMA), the reference's dense numerics for
// many rows (app/kernels.py:46-49: dequantise, then GEMM):
//   y[m, n] = fp16( sum_k x[m, k] * fp16(q[n, k] * s[n]) )      fp32 accumulation
//   EPI_STORE: y (+ res as an fp16 add);  EPI_SILU: rows interleaved (w1 row j at 2j, w3 row j
//   at 2j + 1), mm[m, j] = fp16(fp16(silu(y[m, 2j])) * y[m, 2j + 1]) (app/kernels.py:171-180);
//   EPI_ROPE: y is the q | k | v projection; the interleaved pairs of the q and k heads are
//   rotated by the RoPE table at the row's position and q goes to its buffer, k and v into the
//   cache slot (app/kernels.py:78-107: the same fp16 input, fp32 rotation and rounding as the
//   rope_kv kernel).
//
// Weights use the lane-ordered packed layout of gemv_fused.hip: chunk (tile, c) = 16 rows x
// 64 bytes stored so that lane l's 16 bytes are row l & 15, k = 64c + 16 (l >> 4) .. +15.  The
// row-major variant (RM) reads the same 16 bytes straight from an [N, K] int8 matrix (the
// layout int8_mm receives, app/kernels.py:40-49): the DMA lands them in LDS in the same lane
// order, so everything after the load is shared.
//
// Tiles and main loop: gemm_core.h.  At few rows the former kernel (128 x 128 tiles, two stages) left
// most CUs idle and waited 0.6 us for each 64-wide chunk; deeper rings and smaller tiles took, in us
// (M = 154; N, K): (5120, 3072) 36.5 -> 17.1, (3072, 3072) 30.4 -> 16.4, (16384, 3072) 39.4 -> 27.7,
// (3072, 8192) 91.6 -> 35.7.  At 2048 rows it is bound
// by the products, the conversion and the LDS reads together: (3072, 3072) 46.6 -> 42.5,
// (16384, 3072) 197 -> 192, (3072, 8192) 110 -> 102 (1.01 PFLOP/s); at 4096 rows (3072, 3072) 81.9 -> 77.8,
// (5120, 3072) 132.9 -> 130.4, (16384, 3072) 487 -> 405, (3072, 8192) 208.2 -> 207.9.
//
// Block order is XCD-aware: the row blocks that share a weight tile get block ids that are
// equal modulo 8, so they run on one XCD and re-read the tile from its L2.
#include "gemm_core.h"

namespace ecd {

enum { GEPI_STORE = 0, GEPI_SILU = 1, GEPI_ROPE = 2 };

// Operands of the RoPE + cache-write epilogue: row m is batch item m / S at position pos[m];
// rope [L, HD] fp32 holds (cos, sin) of pair i at columns 2i, 2i + 1.
struct RopeOut {
  const float* rope;
  const int64_t* pos;
  f16* q;   // [M, Hq * HD]
  f16* kc;  // [B, Hk, L, HD]
  f16* vc;
  int S, Hq, Hk, L, HD;
};

// 128 x 128 with two stages, three workgroups per CU: their waves hide each other's loads and conversions,
// where GemmTile reads ahead.  (Its products add k in another order: the other tiles agree bit for bit, with this one
// in all but 0.1% of the values, and either is 2.07e-4 from float64.)  Wave w owns features 32 w .. + 31 of all 128 rows as 2 x 8 tiles of
// v_mfma_f32_16x16x32_f16.  For launches of more than two workgroups per CU whose 256 x 128 tiles end in a half empty
// round; us at 4096 rows, best of the other tiles -> this: (3072, 3072) 90.0 -> 79.7, (5120, 3072) 140 -> 132,
// (3072, 8192) 218 -> 210.  (32x32x16 products in the same loop: 87.9, 145, 223.)
template <bool RM>
struct GemmTile3 : GemmTile<true, RM, 4, 1, 1, 4, 2> {
  using G = GemmTile<true, RM, 4, 1, 1, 4, 2>;
  static __device__ __forceinline__ void run(f16* lds, const f16* __restrict__ x, long ldx,
                                             const int8_t* __restrict__ wp, const f16* __restrict__ sc, int M,
                                             int N, int K, int n0, int m0) {
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nch = K >> 6, ntiles = (N + 15) >> 4;
    const int t0 = min(n0 / 16, ntiles - 1);
    const char* wb = (const char*)wp + (long)t0 * 16 * K;
    const f16* xb = x;
    uint32_t woff[2], xoff[4];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int t = min(n0 / 16 + wv + 4 * j, ntiles - 1);
      woff[j] = RM ? (uint32_t)((min(16 * t + (lane & 15), N - 1) - 16 * t0) * (long)K + 16 * (lane >> 4))
                   : (uint32_t)((t - t0) * (16L * K)) + 16 * lane;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int r = 8 * (wv + 4 * j) + (lane >> 3);
      xoff[j] = (uint32_t)(min(m0 + r, M - 1) * ldx * 2 + 16 * ((lane & 7) ^ (r & 7)));
    }
    const uint32_t lds0 = lds_addr(lds) + wv * 1024;
    auto load = [&](int st) {
      const uint32_t sa = lds0 + st * (G::STG * 2);
      static_for<0, 2>([&](auto J) { lds_dma16_at<4096 * J.value>(wb, woff[J.value], sa); });
      static_for<0, 4>([&](auto J) { lds_dma16_at<G::LW * 2 + 4096 * J.value>(xb, xoff[J.value], sa); });
      wb += RM ? 64 : 1024;
      xb += 64;
    };
    f16 scale[2];
    f32x4 acc[2][8];
#pragma unroll
    for (int ft = 0; ft < 2; ++ft) {
      scale[ft] = sc[min(n0 + 32 * wv + 16 * ft + (lane & 15), N - 1)];
#pragma unroll
      for (int rt = 0; rt < 8; ++rt) acc[ft][rt] = (f32x4){0.f, 0.f, 0.f, 0.f};
    }
    load(0);
    for (int c = 0; c < nch; ++c) {
      wait_vm_lgkm0<0>();  // this wave's loads of chunk c, and its reads of chunk c - 1
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_barrier();  // chunk c complete; the stage of chunk c - 1 is free
      asm volatile("" ::: "memory");
      if (c + 1 < nch) load((c + 1) & 1);
      const f16* st = lds + (c & 1) * G::STG;
      f16x8 w[2][2];
#pragma unroll
      for (int ft = 0; ft < 2; ++ft) {
        i8x16_to_f16(*(const u32x4*)(st + (2 * wv + ft) * 512 + 8 * lane), w[ft][0], w[ft][1]);
        w[ft][0] = w[ft][0] * scale[ft];
        w[ft][1] = w[ft][1] * scale[ft];
      }
#pragma unroll
      for (int rt = 0; rt < 8; ++rt) {
        const f16* xr = st + G::LW + (16 * rt + (lane & 15)) * 64;
        f16x8 xv[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) xv[h] = *(const f16x8*)(xr + 8 * ((2 * (lane >> 4) + h) ^ (lane & 7)));
#pragma unroll
        for (int ft = 0; ft < 2; ++ft)
#pragma unroll
          for (int h = 0; h < 2; ++h)
            acc[ft][rt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w[ft][h], xv[h], acc[ft][rt], 0, 0, 0);
      }
    }
    __syncthreads();
#pragma unroll
    for (int ft = 0; ft < 2; ++ft)
#pragma unroll
      for (int rt = 0; rt < 8; ++rt) {
        const int nl = 32 * wv + 16 * ft + 4 * (lane >> 4);
        f16x4 yv;
#pragma unroll
        for (int j = 0; j < 4; ++j) yv[j] = (f16)acc[ft][rt][j];
        *(f16x4*)(lds + G::piece(16 * rt + (lane & 15), nl >> 3) + (nl & 4)) = yv;
      }
    __syncthreads();
  }
};

template <int EPI, bool RM, int WN, int WM, int FT, int RT, int NS, bool BIG>
__global__ __launch_bounds__(64 * WN * WM, 2) void gemm_i8p_kernel(
    const f16* __restrict__ x, long ldx, const int8_t* __restrict__ wp,
    const f16* __restrict__ s, const f16* __restrict__ res, long ldr, f16* __restrict__ y, long ldy,
    int M, int N, int K, int nfb, int nmb, RopeOut ro) {
  using G = GemmTile<true, RM, WN, WM, FT, RT, NS>;
  __shared__ __align__(16) f16 lds[G::LDS_HALFS];
  int fb, mb;
  G::block(nfb, nmb, fb, mb);
  const int n0 = fb * G::BN, m0 = mb * G::BM;
  const RowMap rm = {0, 0, -1, 0, 0, 1, {0, 0, 0, 0, 0, 0, 0, 0}};  // plain rows
  if constexpr (NS == 2)
    GemmTile3<RM>::run(lds, x, ldx, wp, s, M, N, K, n0, m0);
  else
    G::template run<false, BIG>(lds, x, ldx, wp, s, nullptr, M, N, K, n0, m0, rm);
  constexpr int U = G::U;
  const int p = threadIdx.x % G::PR, nb = n0 + 8 * p;
  if (nb >= N) return;
  const bool full = nb + 7 < N;
  // GEPI_ROPE (HD % 4 == 0): heads and offsets of the piece's two groups of 4 features
  int hh[2], hd[2];
  if constexpr (EPI == GEPI_ROPE) {
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      hh[q] = (nb + 4 * q) / ro.HD;
      hd[q] = nb + 4 * q - hh[q] * ro.HD;
    }
  }
#pragma unroll 1
  for (int r0 = threadIdx.x / G::PR; r0 < G::BM; r0 += G::RS * U) {
    if (m0 + r0 >= M) break;
    f16x8 v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = *(const f16x8*)(lds + G::piece(r0 + G::RS * u, p));
    if constexpr (EPI == GEPI_STORE) {
      f16x8 rv[U];
      if (res && full) {
#pragma unroll
        for (int u = 0; u < U; ++u)
          rv[u] = *(const f16x8u*)(res + (long)min(m0 + r0 + G::RS * u, M - 1) * ldr + nb);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int m = m0 + r0 + G::RS * u;
        if (m >= M) break;
        if (full)
          *(f16x8u*)(y + (long)m * ldy + nb) = res ? v[u] + rv[u] : v[u];
        else
          store_tail(y + (long)m * ldy + nb, res ? res + (long)m * ldr + nb : nullptr, v[u], N - nb);
      }
    } else if constexpr (EPI == GEPI_ROPE) {
      long pr[U];
      f32x4 cs[U][2];
#pragma unroll
      for (int u = 0; u < U; ++u) pr[u] = ro.pos[min(m0 + r0 + G::RS * u, M - 1)];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const long pc = pr[u] < 0 ? 0 : (pr[u] >= ro.L ? ro.L - 1 : pr[u]);
#pragma unroll
        for (int q = 0; q < 2; ++q) cs[u][q] = *(const f32x4*)(ro.rope + pc * ro.HD + hd[q]);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int m = m0 + r0 + G::RS * u;
        if (m >= M) break;
        const bool pval = pr[u] >= 0 && pr[u] < ro.L;
        const int bi = m / ro.S;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          if (nb + 4 * q >= N) break;
          const int h = hh[q], d = hd[q];
          f16x4 o = q ? __builtin_shufflevector(v[u], v[u], 4, 5, 6, 7)
                      : __builtin_shufflevector(v[u], v[u], 0, 1, 2, 3);
          if (h < ro.Hq + ro.Hk) {
            const f32x4 c = cs[u][q];
            const float x0 = (float)o[0], x1 = (float)o[1], x2 = (float)o[2], x3 = (float)o[3];
            o[0] = (f16)(x0 * c[0] - x1 * c[1]);
            o[1] = (f16)(x1 * c[0] + x0 * c[1]);
            o[2] = (f16)(x2 * c[2] - x3 * c[3]);
            o[3] = (f16)(x3 * c[2] + x2 * c[3]);
          }
          if (h < ro.Hq) {
            *(f16x4*)(ro.q + ((long)m * ro.Hq + h) * ro.HD + d) = o;
          } else if (pval) {
            const int kh = h < ro.Hq + ro.Hk ? h - ro.Hq : h - ro.Hq - ro.Hk;
            f16* dst = h < ro.Hq + ro.Hk ? ro.kc : ro.vc;
            *(f16x4*)(dst + (((long)bi * ro.Hk + kh) * ro.L + pr[u]) * ro.HD + d) = o;
          }
        }
      }
    } else {  // pairs (a_j, b_j) with j = nb / 2 ..; N even
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int m = m0 + r0 + G::RS * u;
        if (m >= M) break;
        const f16x4 o = silu_mul4(v[u]);
        f16* dst = y + (long)m * ldy + (nb >> 1);
        if (full) {
          *(f16x4u*)dst = o;
        } else {
#pragma unroll
          for (int q = 0; q < 4; ++q)
            if (nb + 2 * q < N) dst[q] = o[q];
        }
      }
    }
  }
}

template <int EPI, bool RM, int WN, int WM, int FT, int RT, int NS, bool BIG = false>
static int launch_cfg(const f16* x, long ldx, const int8_t* wp, const f16* s, const f16* res,
                      long ldr, f16* y, long ldy, int M, int N, int K, hipStream_t st,
                      const RopeOut& ro) {
  constexpr int BN = 32 * WN * FT, BM = 32 * WM * RT;
  const int nfb = (N + BN - 1) / BN, nmb = (M + BM - 1) / BM;
  const long blocks = (long)nfb * nmb;
  if (blocks > 0x7FFFFFFFL) return ECD_ENOTSUP;
  if constexpr (!BIG)
    if (!w_offsets_fit(BN, K >> 6))
      return launch_cfg<EPI, RM, 2, 2, 1, 1, 12, true>(x, ldx, wp, s, res, ldr, y, ldy, M, N, K, st, ro);
  hipLaunchKernelGGL((gemm_i8p_kernel<EPI, RM, WN, WM, FT, RT, NS, BIG>), dim3((unsigned)blocks),
                     dim3(64 * WN * WM), 0, st, x, ldx, wp, s, res, ldr, y, ldy, M, N, K, nfb, nmb, ro);
  return ecd_launch_status();
}

// The tiles (features x rows, LDS stages).  A launch takes ceil(blocks / 256) rounds, a round about K / 64
// chunk times plus a fill and an epilogue; in ns, measured over K = 3072 and 8192 with 40 to 2048
// workgroups; a chunk takes longer when all CUs load at once (`full`: 256 workgroups) than with at
// most LIGHT of them (`light`).  One feature tile per wave everywhere: with two, the conversion of twice the
// weights between the same products made every shape 15 to 25% slower.
constexpr Tile TILES[4] = {
    {256, 128, 580, 920, 2500},  // 1: 8 waves of 32 x 128, 3 stages
    {128, 128, 385, 570, 1200},  // 2: 4 waves of 32 x 128, 3 stages (two workgroups per CU)
    {64, 128, 300, 370, 800},    // 3: 4 waves of 32 x 64, 7 stages
    {64, 64, 255, 280, 600},     // 4: 4 waves of 32 x 32, 12 stages
};

// 5: GemmTile3, from its third workgroup per CU up to three full rounds of 768; there only tile 1 is ever faster,
// where its last round of 256 is nearly full (beyond, tile 1 always: (16384, 3072) at 3072 rows 296 us, at 4096 405,
// tile 5 310 and 455).  A round of 768 takes 1550 ns a chunk, a last one of b workgroups 270 + 1260 b / 768; of tile 1
// a round takes 980, a last one 520 + 460 b / 256.
constexpr int THREE_PER_CU = 5;
static bool three_per_cu(int M, int N, int nch) {
  const long rows = (M + 127) / 128, b5 = (N + 127) / 128 * rows, b1 = (N + 255) / 256 * rows;
  if (b5 <= 2 * 256 || b5 > 3 * 768 || !w_offsets_fit(128, nch)) return false;
  const long last = b5 % 768;
  const long e5 = b5 / 768 * (nch * 1550L + 2500) + (last ? nch * (270 + 1260 * last / 768) + 2500 : 0);
  const long e1 = b1 / 256 * (nch * 980L + 2500) + (b1 % 256 ? nch * (520 + 460 * (b1 % 256) / 256) + 2500 : 0);
  return e5 < e1;
}

// The tile of the shortest estimate.  (Of 18 prompt shapes of few rows measured with every tile it is the fastest or
// within 3% of it, of 137 shapes of 300 to 4096 rows within 2%.)
static int default_tile(int M, int N, int K) {
  long est = 0;
  return three_per_cu(M, N, K >> 6) ? THREE_PER_CU : 1 + best_tile(TILES, 4, M, N, K >> 6, 1, &est);
}

// K split over gridDim.y: fp32 partial sums [gridDim.y][M, N]
template <int WN, int WM, int FT, int RT, int NS>
__global__ __launch_bounds__(64 * WN * WM, 2) void gemm_i8p_partial_kernel(
    const f16* __restrict__ x, long ldx, const int8_t* __restrict__ wp, const f16* __restrict__ s,
    float* __restrict__ ws, int M, int N, int K, int nfb, int nmb) {
  using G = GemmTile<true, false, WN, WM, FT, RT, NS>;
  __shared__ __align__(16) f16 lds[G::LDS_HALFS];
  int fb, mb;
  G::block(nfb, nmb, fb, mb);
  const RowMap rm = {0, 0, -1, 0, 0, 1, {0, 0, 0, 0, 0, 0, 0, 0}};  // plain rows
  const int z = blockIdx.y, c0 = (K >> 6) * z / gridDim.y, c1 = (K >> 6) * (z + 1) / gridDim.y;
  G::template run<true>(lds, x, ldx, wp, s, nullptr, M, N, K, fb * G::BN, mb * G::BM, rm, c0, c1 - c0,
                        ws + (long)z * M * N);
}

template <int WN, int WM, int FT, int RT, int NS>
static int launch_partial(const f16* x, long ldx, const int8_t* wp, const f16* s, float* ws, int M, int N, int K,
                          int ks, hipStream_t st) {
  const int nfb = (N + 32 * WN * FT - 1) / (32 * WN * FT), nmb = (M + 32 * WM * RT - 1) / (32 * WM * RT);
  if ((long)nfb * nmb > 0x7FFFFFFFL || !w_offsets_fit(32 * WN * FT, K >> 6)) return ECD_ENOTSUP;
  hipLaunchKernelGGL((gemm_i8p_partial_kernel<WN, WM, FT, RT, NS>), dim3((unsigned)(nfb * nmb), ks),
                     dim3(64 * WN * WM), 0, st, x, ldx, wp, s, ws, M, N, K, nfb, nmb);
  return ecd_launch_status();
}

template <int EPI, bool RM = false>
static int launch_gemm(const f16* x, long ldx, const int8_t* wp, const f16* s, const f16* res,
                       long ldr, f16* y, long ldy, int M, int N, int K, hipStream_t st,
                       RopeOut ro = RopeOut{}, int cfg = 0) {
#define I8_CFG(I, ...)                                                                            \
  case I:                                                                                         \
    return launch_cfg<EPI, RM, __VA_ARGS__>(x, ldx, wp, s, res, ldr, y, ldy, M, N, K, st, ro)
  switch (cfg ? cfg : default_tile(M, N, K)) {
    I8_CFG(1, 8, 1, 1, 4, 3);
    I8_CFG(2, 4, 1, 1, 4, 3);
    I8_CFG(3, 2, 2, 1, 2, 7);
    I8_CFG(4, 2, 2, 1, 1, 12);
    I8_CFG(5, 4, 1, 1, 4, 2);
    default: return ECD_EINVAL;
  }
#undef I8_CFG
}

static bool al16(const void* p) { return ((uintptr_t)p & 15) == 0; }

// the per-lane byte offsets of the x loads are 32-bit: the x buffer must stay below 2 GiB
static bool x_offsets_fit(int M, long ldx) { return (long)M * ldx * 2 < 0x7FFFFFFFL; }

// The dense-numerics GEMM on a row-major [N, K] int8 weight (int8_mm with more than 16 rows).
// Returns 1 without launching when the operands do not fit the kernel (the caller then runs
// its own path).
int gemm_i8_rowmajor(const f16* x, long ldx, const int8_t* w, const f16* s, const f16* res,
                     long ldr, f16* y, long ldy, int M, int N, int K, hipStream_t st) {
  if ((K % 64) || (ldx % 8) || !al16(x) || !al16(w) || !x_offsets_fit(M, ldx) ||
      16L * K >= 0x7FFFFFFFL)
    return 1;
  return launch_gemm<GEPI_STORE, true>(x, ldx, w, s, res, ldr, y, ldy, M, N, K, st);
}

}  // namespace ecd

using namespace ecd;

extern "C" {

int ecd_gemm_i8p(const void* x, long ldx, const void* wp, const void* s, const void* res,
                 long ldr, void* y, long ldy, int M, int N, int K, void* stream) {
  if (!x || !wp || !s || !y || M <= 0 || N <= 0 || K <= 0 || (K % 64) || ldx < K || (ldx % 8) ||
      !al16(x) || !al16(wp) || ldy < N || (res && ldr < N))
    return ECD_EINVAL;
  if (!x_offsets_fit(M, ldx)) return ECD_ENOTSUP;
  return launch_gemm<GEPI_STORE>((const f16*)x, ldx, (const int8_t*)wp, (const f16*)s,
                                 (const f16*)res, ldr, (f16*)y, ldy, M, N, K, (hipStream_t)stream);
}

int ecd_gemm_i8p_tile(int M, int N, int K) {
  return M > 0 && N > 0 && K > 0 && K % 64 == 0 ? default_tile(M, N, K) : 0;
}

int ecd_gemm_i8p_tuned(const void* x, long ldx, const void* w, const void* s, const void* res, long ldr, void* y,
                       long ldy, int M, int N, int K, int rowmajor, int cfg, void* stream) {
  if (!x || !w || !s || !y || M <= 0 || N <= 0 || K <= 0 || (K % 64) || ldx < K || (ldx % 8) || !al16(x) ||
      !al16(w) || ldy < N || (res && ldr < N) || cfg < 0 || cfg > 5)
    return ECD_EINVAL;
  if (!x_offsets_fit(M, ldx) || (rowmajor && 16L * K >= 0x7FFFFFFFL)) return ECD_ENOTSUP;
  const f16 *xh = (const f16*)x, *sh = (const f16*)s, *rh = (const f16*)res;
  const int8_t* wh = (const int8_t*)w;
  const hipStream_t st = (hipStream_t)stream;
  if (rowmajor)
    return launch_gemm<GEPI_STORE, true>(xh, ldx, wh, sh, rh, ldr, (f16*)y, ldy, M, N, K, st, RopeOut{}, cfg);
  return launch_gemm<GEPI_STORE>(xh, ldx, wh, sh, rh, ldr, (f16*)y, ldy, M, N, K, st, RopeOut{}, cfg);
}

int ecd_gemm_i8p_rope(const void* x, long ldx, const void* wp, const void* s, const float* rope,
                      const int64_t* pos, void* q, void* kc, void* vc, int M, int S, int Hq,
                      int Hk, int L, int HD, int K, void* stream) {
  if (!x || !wp || !s || !rope || !pos || !q || !kc || !vc || M <= 0 || S <= 0 || Hq <= 0 ||
      Hk <= 0 || (Hq % Hk) || L <= 0 || HD <= 0 || (HD % 4) || K <= 0 || (K % 64) || ldx < K ||
      (ldx % 8) || !al16(x) || !al16(wp) || ((uintptr_t)q & 7) || ((uintptr_t)kc & 7) ||
      ((uintptr_t)vc & 7) || ((uintptr_t)rope & 15))
    return ECD_EINVAL;
  if (!x_offsets_fit(M, ldx)) return ECD_ENOTSUP;
  const RopeOut ro{rope, pos, (f16*)q, (f16*)kc, (f16*)vc, S, Hq, Hk, L, HD};
  return launch_gemm<GEPI_ROPE>((const f16*)x, ldx, (const int8_t*)wp, (const f16*)s, nullptr, 0,
                                nullptr, 0, M, (Hq + 2 * Hk) * HD, K, (hipStream_t)stream, ro);
}

int ecd_gemm_i8p_silu(const void* x, long ldx, const void* wp, const void* s, void* mm,
                      long ldm, int M, int F, int K, void* stream) {
  if (!x || !wp || !s || !mm || M <= 0 || F <= 0 || (F % 2) || K <= 0 || (K % 64) || ldx < K ||
      (ldx % 8) || !al16(x) || !al16(wp) || ldm < F || (ldm % 2) || ((uintptr_t)mm & 3))
    return ECD_EINVAL;
  if (!x_offsets_fit(M, ldx)) return ECD_ENOTSUP;
  return launch_gemm<GEPI_SILU>((const f16*)x, ldx, (const int8_t*)wp, (const f16*)s, nullptr,
                                0, (f16*)mm, ldm, M, 2 * F, K, (hipStream_t)stream);
}

int ecd_gemm_i8p_splits(int M, int N, int K) {
  if (M <= 0 || N <= 0 || K <= 0 || (K % 64) || (N % 64) || !w_offsets_fit(TILES[2].bn, K >> 6)) return 1;
  return split_ways(TILES, 4, TILES + 2, 2, M, N, K >> 6);
}

int ecd_gemm_i8p_partial(const void* x, long ldx, const void* wp, const void* s, float* ws, int M, int N, int K,
                         int ks, void* stream) {
  if (!x || !wp || !s || !ws || M <= 0 || N <= 0 || K <= 0 || (K % 64) || (N % 64) || ldx < K || (ldx % 8) ||
      ks < 1 || ks > SPLIT_MAX || ks > K / 64 || !al16(x) || !al16(wp) || !al16(ws))
    return ECD_EINVAL;
  if (!x_offsets_fit(M, ldx)) return ECD_ENOTSUP;
  long est = 0;
  const f16 *xh = (const f16*)x, *sh = (const f16*)s;
  const int8_t* wh = (const int8_t*)wp;
  const hipStream_t st = (hipStream_t)stream;
  if (best_tile(TILES + 2, 2, M, N, K >> 6, ks, &est) == 0)
    return launch_partial<2, 2, 1, 2, 7>(xh, ldx, wh, sh, ws, M, N, K, ks, st);
  return launch_partial<2, 2, 1, 1, 12>(xh, ldx, wh, sh, ws, M, N, K, ks, st);
}

}  // extern "C"
