// fp16-weight GEMM on gfx950 MFMA for the dense layers of the codec's flow-matching estimator
// (the nn.Linear layers and the k = 3 Conv1d-as-GEMM of app/heartcodec/models/transformer.py),
// with torch's F.linear numerics: fp32 accumulation, fp32 bias, one fp16 rounding.
//   EPI_STORE: y = fp16(acc + bias); if alpha != 1, y = fp16(y * alpha); then y = fp16(y + res).
//   EPI_SILU:  weight rows interleaved (gate row j at 2j, up row j at 2j + 1),
//              mm[m, j] = fp16(fp16(silu(g)) * u) with g, u the fp16 GEMM outputs (LlamaMLP,
//              transformer.py:178-181).
//   EPI_PRELU: y = fp16(acc + bias), then nn.PReLU with one slope a: y < 0 -> fp16(a * y), then
//              y = fp16(y + res) (the conv -> PReLU (-> + x) steps of the codec's waveform
//              decoder, app/heartcodec/models/sq_codec.py:149-168).
//
// Packed weights: 16-row tiles x 64-wide K chunks of 2 KB, two 1 KB halves h; lane l's 16 bytes
// of half h hold row l & 15, k = 64c + 16 (l >> 4) + 8h .. +7 (ecd_pack_f16), so one 16-byte
// LDS read is an MFMA A fragment.  The activations x are the B operand.
//
// Tiles and main loop: gemm_core.h.
//
// Block order is XCD-aware: the row blocks that share a weight tile get block ids equal modulo 8,
// so they run on one XCD and share its L2 (feature blocks in whole groups of 8; the grid has
// exactly one workgroup per output tile, so narrow outputs launch no empty workgroups).
#include "gemm_core.h"

namespace ecd {

enum { F16_STORE = 0, F16_SILU = 1, F16_PRELU = 2, F16_ROPE = 3 };

// Output of the q | k | v projection with RoPE (F16_ROPE): features [0, D) are q, [D, 2D) k,
// [2D, 3D) v, D = H * HD, rows m = b * T + t.  q and k pairs (2i, 2i + 1) are rotated by
// tab[t, i] = (cos, sin) (fp16); q goes to rows [M, D], k and v to [B, H, T, HD].
struct RopeOut {
  const f16* tab;
  f16 *q, *k, *v;
  int T, H, HD;
};

template <int EPI, int WN, int WM, int FT, int RT, int NS, bool BIG>
__global__ __launch_bounds__(64 * WN * WM, 2) void gemm_f16w_kernel(
    const f16* __restrict__ x, long ldx, const f16* __restrict__ wp,
    const float* __restrict__ bias, float alpha, const f16* res, long ldr,
    f16* y, long ldy, int M, int N, int K, int nfb, int nmb, RowMap rm,
    RopeOut ro) {
  using G = GemmTile<false, false, WN, WM, FT, RT, NS>;
  __shared__ __align__(16) f16 lds[G::LDS_HALFS];
  int fb, mb;
  G::block(nfb, nmb, fb, mb);
  const int n0 = fb * G::BN, m0 = mb * G::BM;
  G::template run<false, BIG>(lds, x, ldx, wp, nullptr, bias, M, N, K, n0, m0, rm);
  constexpr int U = G::U;
  const int p = threadIdx.x % G::PR, nb = n0 + 8 * p;
  if (nb >= N) return;
  const bool full = nb + 7 < N;
  // F16_ROPE (HD % 4 == 0): sections (q, k, v), heads and offsets of the piece's two groups of 4 features
  const int D = ro.H * ro.HD;
  int sec[2], hh[2], hd[2];
  if constexpr (EPI == F16_ROPE) {
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int n = nb + 4 * q;
      sec[q] = n >= 2 * D ? 2 : (n >= D ? 1 : 0);
      hh[q] = (n - sec[q] * D) / ro.HD;
      hd[q] = n - sec[q] * D - hh[q] * ro.HD;
    }
  }
#pragma unroll 1
  for (int r0 = threadIdx.x / G::PR; r0 < G::BM; r0 += G::RS * U) {
    if (m0 + r0 >= M) break;
    f16x8 v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = *(const f16x8*)(lds + G::piece(r0 + G::RS * u, p));
    if constexpr (EPI == F16_STORE || EPI == F16_PRELU) {
      long m[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int mm = min(m0 + r0 + G::RS * u, M - 1);
        m[u] = rm.ypad >= 0 ? seq_row(mm, rm.T, rm.ypad) : mm;
      }
      f16x8 rv[U];
      if (res && full) {
#pragma unroll
        for (int u = 0; u < U; ++u) rv[u] = *(const f16x8u*)(res + m[u] * ldr + nb);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (m0 + r0 + G::RS * u >= M) break;
        if constexpr (EPI == F16_PRELU) {  // alpha: the slope
#pragma unroll
          for (int j = 0; j < 8; ++j)
            if ((float)v[u][j] < 0.f) v[u][j] = (f16)((float)v[u][j] * alpha);
        } else if (alpha != 1.0f) {
#pragma unroll
          for (int j = 0; j < 8; ++j) v[u][j] = (f16)((float)v[u][j] * alpha);
        }
        if (full)
          *(f16x8u*)(y + m[u] * ldy + nb) = res ? v[u] + rv[u] : v[u];
        else
          store_tail(y + m[u] * ldy + nb, res ? res + m[u] * ldr + nb : nullptr, v[u], N - nb);
      }
    } else if constexpr (EPI == F16_ROPE) {
      int rb[U], t[U];
      f16x4 cs[U][2];  // pairs d / 2, d / 2 + 1
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int mm = min(m0 + r0 + G::RS * u, M - 1);
        rb[u] = mm / ro.T;
        t[u] = mm - rb[u] * ro.T;
#pragma unroll
        for (int q = 0; q < 2; ++q) cs[u][q] = *(const f16x4*)(ro.tab + (long)t[u] * ro.HD + hd[q]);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int mm = m0 + r0 + G::RS * u;
        if (mm >= M) break;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          if (nb + 4 * q >= N) break;
          f16x4 o = q ? __builtin_shufflevector(v[u], v[u], 4, 5, 6, 7)
                      : __builtin_shufflevector(v[u], v[u], 0, 1, 2, 3);
          if (sec[q] < 2) {
            const f16x4 c = cs[u][q];
            f16 o0, o1, o2, o3;
            rope_pair_f16((float)o[0], (float)o[1], (float)c[0], (float)c[1], o0, o1);
            rope_pair_f16((float)o[2], (float)o[3], (float)c[2], (float)c[3], o2, o3);
            o = (f16x4){o0, o1, o2, o3};
          }
          f16* dst = sec[q] == 0 ? ro.q + (long)mm * D + hh[q] * ro.HD + hd[q]
                                 : (sec[q] == 1 ? ro.k : ro.v) +
                                       (((long)rb[u] * ro.H + hh[q]) * ro.T + t[u]) * ro.HD + hd[q];
          *(f16x4*)dst = o;
        }
      }
    } else {  // pairs (a_j, b_j) with j = nb / 2 ..; N even
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int mm = m0 + r0 + G::RS * u;
        if (mm >= M) break;
        const f16x4 o = silu_mul4(v[u]);
        f16* dst = y + (long)mm * ldy + (nb >> 1);
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

// Pack fp16 w [N, K] into lane-ordered 16 x 64 tiles of 2 KB (two 1 KB halves); with
// `interleave` (N even) packed row 2j is source row j and 2j + 1 is source row N/2 + j.
__global__ __launch_bounds__(256) void pack_f16_kernel(const f16* __restrict__ w, int N, int K,
                                                       int interleave, f16* __restrict__ out) {
  const int nch = K >> 6;
  const long ntiles = (N + 15) >> 4;
  const long idx = (long)blockIdx.x * 256 + threadIdx.x;
  if (idx >= ntiles * nch * 128) return;
  const int l = (int)(idx & 63);
  const int h = (int)((idx >> 6) & 1);
  const long tc = idx >> 7;
  const int c = (int)(tc % nch);
  const long tile = tc / nch;
  const long r = tile * 16 + (l & 15);
  u32x4 v = (u32x4){0u, 0u, 0u, 0u};
  if (r < N) {
    const long src = interleave ? ((r & 1) ? (N >> 1) + (r >> 1) : (r >> 1)) : r;
    v = *(const u32x4*)(w + src * K + 64L * c + 16 * (l >> 4) + 8 * h);
  }
  *(u32x4*)(out + (tile * nch + c) * 1024 + 512 * h + 8 * l) = v;
}

template <int EPI, int WN, int WM, int FT, int RT, int NS, bool BIG = false>
static int launch_cfg(const f16* x, long ldx, const f16* wp, const float* bias, float alpha,
                      const f16* res, long ldr, f16* y, long ldy, int M, int N, int K,
                      const RowMap& rm, const RopeOut& ro, hipStream_t st) {
  constexpr int BN = 32 * WN * FT, BM = 32 * WM * RT;
  const int nfb = (N + BN - 1) / BN;
  const int nmb = (M + BM - 1) / BM;
  const long blocks = (long)nfb * nmb;
  if (blocks > 0x7FFFFFFFL) return ECD_ENOTSUP;
  if constexpr (!BIG)
    if (!w_offsets_fit(BN, K >> 6))
      return launch_cfg<EPI, 2, 2, 1, 1, 8, true>(x, ldx, wp, bias, alpha, res, ldr, y, ldy, M, N, K, rm, ro, st);
  hipLaunchKernelGGL((gemm_f16w_kernel<EPI, WN, WM, FT, RT, NS, BIG>), dim3((unsigned)blocks),
                     dim3(64 * WN * WM), 0, st, x, ldx, wp, bias, alpha, res, ldr, y, ldy, M, N, K,
                     nfb, nmb, rm, ro);
  return ecd_launch_status();
}

// The tiles (features x rows, LDS stages).  1 to 8 leave room for one workgroup per CU: a launch takes
// ceil(blocks / 256) rounds, a round about K / 64 chunk times plus a fill and an epilogue.  In ns,
// measured over K = 1536 .. 8192; a chunk takes longer when all CUs load at once (`full`: 256 workgroups)
// than with at most LIGHT of them (`light`).
constexpr Tile TILES[8] = {
    {256, 256, 1300, 1550, 5000},  // 1: 8 waves of 64 x 128, 2 stages
    {256, 192, 1190, 1450, 3500},  // 2: 8 waves of 64 x 96, 2 stages
    {256, 128, 750, 870, 2500},    // 3: 8 waves of 64 x 64, 3 stages
    {128, 192, 660, 800, 3000},    // 4: 8 waves of 32 x 96, 3 stages
    {128, 128, 440, 670, 1200},    // 5: 8 waves of 32 x 64, 4 stages
    {128, 64, 280, 420, 800},      // 6: 4 waves of 64 x 32, 5 stages
    {64, 128, 280, 420, 800},      // 7: 4 waves of 32 x 64, 5 stages
    {64, 64, 200, 260, 600},       // 8: 4 waves of 32 x 32, 8 stages
};
// 9: 128 x 128, 8 waves, 2 stages; 10: 64 x 128, 8 waves, 2 stages: several workgroups per CU, for the
// waveform decoder's convolutions of at most 128 channels over many rows, whose few chunks leave the
// fill and the stores to be hidden by other workgroups (476160 rows, 128 channels, us for K = 896 / 128:
// tile 9 213 / 43, 5 228 / 62, 3 270 / 79; 1.4 M rows, 64 channels, K = 448 / 64: tile 10 274 / 69,
// 9 295 / 91, 7 322 / 134).
constexpr int MANY_ROWS = 16384;
// Tile 10 also for short K (at most 8 chunks), where the fill of a deep ring is most of the time: up to one round of it,
// and up to two where the 128 x 128 tiles need a second as well.  us, best of the others -> tile 10 (before this main
// loop): 8000 x 256 x 256 6.70 -> 5.33 (6.11), 4500 x 256 x 256 6.37 -> 4.98 (5.81), 16000 x 128 x 128 5.89 -> 4.82
// (5.63), 2000 x 1024 x 512 7.81 -> 6.54 (7.45), 3000 x 512 x 512 7.58 -> 6.25 (7.23), 20000 x 192 x 256 11.9 -> 8.9
// (12.1), 1 x 256 x 256 4.40 -> 4.25 (3.80); with K = 1024 2000 x 1024 11.8 -> 13.0.
constexpr int SHORT_K = 512;

// Library default per shape (N counts output features before the SiLU pairing): the tile of the
// shortest estimate.  (Of 29 shapes measured with every tile it is the fastest or within 10% of it.)
static int default_cfg(int M, int N, int K) {
  if (M >= MANY_ROWS && N <= 128) return N <= 64 ? 10 : 9;
  const long b10 = (long)((N + 63) / 64) * ((M + 127) / 128);
  if (K <= SHORT_K && (b10 <= 256 || (b10 <= 512 && (long)((N + 127) / 128) * ((M + 127) / 128) > 256))) return 10;
  long est = 0;
  return 1 + best_tile(TILES, 8, M, N, K >> 6, 1, &est);
}

// K split over gridDim.y: fp32 partial sums [gridDim.y][M, N]
template <int WN, int WM, int FT, int RT, int NS>
__global__ __launch_bounds__(64 * WN * WM, 2) void gemm_f16w_partial_kernel(
    const f16* __restrict__ x, long ldx, const f16* __restrict__ wp, float* __restrict__ ws, int M, int N,
    int K, int nfb, int nmb) {
  using G = GemmTile<false, false, WN, WM, FT, RT, NS>;
  __shared__ __align__(16) f16 lds[G::LDS_HALFS];
  int fb, mb;
  G::block(nfb, nmb, fb, mb);
  const RowMap rm = {0, 0, -1, 0, 0, 1, {0, 0, 0, 0, 0, 0, 0, 0}};  // plain rows
  const int z = blockIdx.y, c0 = (K >> 6) * z / gridDim.y, c1 = (K >> 6) * (z + 1) / gridDim.y;
  G::template run<true>(lds, x, ldx, wp, nullptr, nullptr, M, N, K, fb * G::BN, mb * G::BM, rm, c0, c1 - c0,
                        ws + (long)z * M * N);
}

template <int EPI>
static int launch_f16(int cfg, const f16* x, long ldx, const f16* wp, const float* bias,
                      float alpha, const f16* res, long ldr, f16* y, long ldy, int M, int N,
                      int K, const RowMap& rm, const RopeOut& ro, hipStream_t st) {
  if (cfg == 0) cfg = default_cfg(M, N, K);
#define F16_CFG(I, ...)                                                                       \
  case I:                                                                                     \
    return launch_cfg<EPI, __VA_ARGS__>(x, ldx, wp, bias, alpha, res, ldr, y, ldy, M, N, K, rm, \
                                        ro, st)
  switch ((cfg - 1) % 10 + 1) {
    F16_CFG(1, 4, 2, 2, 4, 2);
    F16_CFG(2, 4, 2, 2, 3, 2);
    F16_CFG(3, 4, 2, 2, 2, 3);
    F16_CFG(4, 4, 2, 1, 3, 3);
    F16_CFG(5, 4, 2, 1, 2, 4);
    F16_CFG(6, 2, 2, 2, 1, 5);
    F16_CFG(7, 2, 2, 1, 2, 5);
    F16_CFG(8, 2, 2, 1, 1, 8);
    F16_CFG(9, 4, 2, 1, 2, 2);
    F16_CFG(10, 2, 4, 1, 1, 2);
    default: return ECD_EINVAL;
  }
#undef F16_CFG
}

template <int WN, int WM, int FT, int RT, int NS>
static int launch_partial(const f16* x, long ldx, const f16* wp, float* ws, int M, int N, int K, int ks,
                          hipStream_t st) {
  const int nfb = (N + 32 * WN * FT - 1) / (32 * WN * FT), nmb = (M + 32 * WM * RT - 1) / (32 * WM * RT);
  if ((long)nfb * nmb > 0x7FFFFFFFL || !w_offsets_fit(32 * WN * FT, K >> 6)) return ECD_ENOTSUP;
  hipLaunchKernelGGL((gemm_f16w_partial_kernel<WN, WM, FT, RT, NS>), dim3((unsigned)(nfb * nmb), ks),
                     dim3(64 * WN * WM), 0, st, x, ldx, wp, ws, M, N, K, nfb, nmb);
  return ecd_launch_status();
}

static int launch_epi(int epi, int cfg, const f16* x, long ldx, const f16* wp, const float* bias,
                      float alpha, const f16* res, long ldr, f16* y, long ldy, int M, int N, int K,
                      const RowMap& rm, hipStream_t st) {
  const RopeOut ro = {nullptr, nullptr, nullptr, nullptr, 1, 1, 4};
  if (epi == F16_SILU)
    return launch_f16<F16_SILU>(cfg, x, ldx, wp, nullptr, 1.0f, nullptr, 0, y, ldy, M, N, K, rm,
                                ro, st);
  if (epi == F16_PRELU)
    return launch_f16<F16_PRELU>(cfg, x, ldx, wp, bias, alpha, res, ldr, y, ldy, M, N, K, rm, ro,
                                 st);
  return launch_f16<F16_STORE>(cfg, x, ldx, wp, bias, alpha, res, ldr, y, ldy, M, N, K, rm, ro,
                               st);
}

static bool al16(const void* p) { return ((uintptr_t)p & 15) == 0; }

// the per-lane byte offsets of the x loads are 32-bit: the x buffer must stay below 2 GiB
static bool x_offsets_fit(int M, long ldx) { return (long)M * ldx * 2 < 0x7FFFFFFFL; }

}  // namespace ecd

using namespace ecd;

extern "C" {

long ecd_packed_bytes_f16(int N, int K) { return (long)((N + 15) / 16) * 16 * (long)K * 2; }

int ecd_pack_f16(const void* w, int N, int K, int interleave, void* out, void* stream) {
  if (!w || !out || N <= 0 || K <= 0 || (K % 64) || (interleave && (N & 1)) || !al16(w) ||
      !al16(out))
    return ECD_EINVAL;
  const long total = (long)((N + 15) / 16) * (K / 64) * 128;
  hipLaunchKernelGGL(pack_f16_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0,
                     (hipStream_t)stream, (const f16*)w, N, K, interleave, (f16*)out);
  return ecd_launch_status();
}

int ecd_gemm_f16p_tuned(const void* x, long ldx, const void* wp, const float* bias, float alpha,
                        const void* res, long ldr, void* y, long ldy, int M, int N, int K,
                        int epi, int cfg, void* stream) {
  if (!x || !wp || !y || M <= 0 || N <= 0 || K <= 0 || (K % 64) || ldx < K || (ldx % 8) ||
      !al16(x) || !al16(wp) || cfg < 0 || cfg > 16 || epi < 0 || epi > 2)
    return ECD_EINVAL;
  const bool silu = epi == F16_SILU;
  if (silu) {
    if ((N % 2) || ldy < N / 2 || (ldy % 2) || ((uintptr_t)y & 3) || bias || res || alpha != 1.0f)
      return ECD_EINVAL;
  } else if (ldy < N || (res && ldr < N)) {
    return ECD_EINVAL;
  }
  if (!x_offsets_fit(M, ldx)) return ECD_ENOTSUP;
  const RowMap rm = {0, 0, -1, 0, 0, 1, {0, 0, 0, 0, 0, 0, 0, 0}};
  return launch_epi(epi, cfg, (const f16*)x, ldx, (const f16*)wp, bias, alpha, (const f16*)res,
                    ldr, (f16*)y, ldy, M, N, K, rm, (hipStream_t)stream);
}

int ecd_gemm_f16p_rope(const void* x, long ldx, const void* wp, const float* bias,
                       const void* tab, void* q, void* k, void* v, int M, int T, int H, int HD,
                       int K, void* stream) {
  const long N = 3L * H * HD;
  if (!x || !wp || !tab || !q || !k || !v || M <= 0 || T <= 0 || M % T || H <= 0 || HD <= 0 ||
      (HD % 4) || N > 0x7FFFFFFFL || K <= 0 || (K % 64) || ldx < K || (ldx % 8) || !al16(x) ||
      !al16(wp) || ((uintptr_t)tab & 7) || ((uintptr_t)q & 7) || ((uintptr_t)k & 7) ||
      ((uintptr_t)v & 7))
    return ECD_EINVAL;
  if (!x_offsets_fit(M, ldx)) return ECD_ENOTSUP;
  const RowMap rm = {0, 0, -1, 0, 0, 1, {0, 0, 0, 0, 0, 0, 0, 0}};
  const RopeOut ro = {(const f16*)tab, (f16*)q, (f16*)k, (f16*)v, T, H, HD};
  return launch_f16<F16_ROPE>(0, (const f16*)x, ldx, (const f16*)wp, bias, 1.0f, nullptr, 0,
                              nullptr, 0, M, (int)N, K, rm, ro, (hipStream_t)stream);
}

int ecd_gemm_f16p_conv_tuned(const void* x, long ldx, const void* wp, const float* bias,
                             float alpha, const void* res, long ldr, void* y, long ldy, int M,
                             int N, int K, int T, int xpad, int ypad, const int* offsets, int k,
                             int rep, int epi, int cfg, void* stream) {
  if (!x || !wp || !y || M <= 0 || N <= 0 || K <= 0 || (K % 64) || (ldx % 8) || !al16(x) ||
      !al16(wp) || epi < 0 || epi > 2 || epi == F16_SILU || cfg < 0 || cfg > 16 || T <= 0 ||
      M % T || k < 0 || k > 8 ||
      (k && (!offsets || K % (64 * k) || xpad < 0)) || (!k && ldx < K) || ldy < N ||
      (res && ldr < N) || ypad < -1 || (rep != 1 && rep != 2) || (rep == 2 && (!k || T % 2)))
    return ECD_EINVAL;
  RowMap rm = {T, xpad, ypad, k ? K / (64 * k) : 0, k, rep, {0, 0, 0, 0, 0, 0, 0, 0}};
  if (k) {
    if (ldx < K / k) return ECD_EINVAL;
    for (int j = 0; j < k; ++j) {
      // source rows stay in the pad rows: shift o (or o >> 1 and (o + 1) >> 1 with a repeat)
      const int lo = rep == 2 ? offsets[j] >> 1 : offsets[j];
      const int hi = rep == 2 ? (offsets[j] + 1) >> 1 : offsets[j];
      if (lo < -xpad || hi > xpad) return ECD_EINVAL;
      rm.off[j] = offsets[j];
    }
  }
  const long tin = rep == 2 ? T / 2 : T;  // source rows per sequence
  const long xrows = k ? (long)(M / T) * (tin + xpad) + xpad : M;  // + the rows after the last
  if (!x_offsets_fit((int)min(xrows, 0x7FFFFFFFL), ldx)) return ECD_ENOTSUP;
  return launch_epi(epi, cfg, (const f16*)x, ldx, (const f16*)wp, bias, alpha, (const f16*)res,
                    ldr, (f16*)y, ldy, M, N, K, rm, (hipStream_t)stream);
}

int ecd_gemm_f16p_conv(const void* x, long ldx, const void* wp, const float* bias, float alpha,
                       const void* res, long ldr, void* y, long ldy, int M, int N, int K, int T,
                       int xpad, int ypad, const int* offsets, int k, int rep, int epi,
                       void* stream) {
  return ecd_gemm_f16p_conv_tuned(x, ldx, wp, bias, alpha, res, ldr, y, ldy, M, N, K, T, xpad,
                                  ypad, offsets, k, rep, epi, 0, stream);
}

int ecd_gemm_f16p(const void* x, long ldx, const void* wp, const float* bias, float alpha,
                  const void* res, long ldr, void* y, long ldy, int M, int N, int K,
                  void* stream) {
  return ecd_gemm_f16p_tuned(x, ldx, wp, bias, alpha, res, ldr, y, ldy, M, N, K, 0, 0, stream);
}

int ecd_gemm_f16p_prelu(const void* x, long ldx, const void* wp, const float* bias, float slope,
                        const void* res, long ldr, void* y, long ldy, int M, int N, int K,
                        void* stream) {
  return ecd_gemm_f16p_tuned(x, ldx, wp, bias, slope, res, ldr, y, ldy, M, N, K, F16_PRELU, 0,
                             stream);
}

int ecd_gemm_f16p_splits(int M, int N, int K) {
  if (M <= 0 || N <= 0 || K <= 0 || (K % 64) || (N % 64) || !w_offsets_fit(TILES[6].bn, K >> 6)) return 1;
  return split_ways(TILES, 8, TILES + 6, 2, M, N, K >> 6);
}

int ecd_gemm_f16p_partial(const void* x, long ldx, const void* wp, float* ws, int M, int N, int K, int ks,
                          void* stream) {
  if (!x || !wp || !ws || M <= 0 || N <= 0 || K <= 0 || (K % 64) || (N % 64) || ldx < K || (ldx % 8) ||
      ks < 1 || ks > SPLIT_MAX || ks > K / 64 || !al16(x) || !al16(wp) || !al16(ws))
    return ECD_EINVAL;
  if (!x_offsets_fit(M, ldx)) return ECD_ENOTSUP;
  long est = 0;
  const f16 *xh = (const f16*)x, *wh = (const f16*)wp;
  const hipStream_t st = (hipStream_t)stream;
  if (best_tile(TILES + 6, 2, M, N, K >> 6, ks, &est) == 0)
    return launch_partial<2, 2, 1, 2, 5>(xh, ldx, wh, ws, M, N, K, ks, st);
  return launch_partial<2, 2, 1, 1, 8>(xh, ldx, wh, ws, M, N, K, ks, st);
}

int ecd_gemm_f16p_silu(const void* x, long ldx, const void* wp, void* mm, long ldm, int M, int F,
                       int K, void* stream) {
  if (F <= 0) return ECD_EINVAL;
  return ecd_gemm_f16p_tuned(x, ldx, wp, nullptr, 1.0f, nullptr, 0, mm, ldm, M, 2 * F, K, 1, 0,
                             stream);
}

}  // extern "C"
