// The waveform decoder's 64-channel stages on gfx950, each as one pass over the samples
// (app/heartcodec/models/sq_codec.py:120-168, :380-526): a residual unit (dilated causal conv k = 7 ->
// PReLU -> 1x1 conv -> PReLU -> + x), and the PostProcessor's 2x repeat + conv + PReLU together with
// the final conv to one channel.
//
// As GEMMs over implicit taps (gemm_f16.hip) these stages are bound by the loads: with 64 output
// channels every x row is fetched once per tap through the CU's 57 B/clock vector memory path, and
// each conv writes its activation and reads it back.  Here a workgroup loads the window of x rows that
// its tile needs once (LDS DMA, the next tile's window in flight while this one is computed), holds the
// weights in registers for all its tiles (a wave owns 32 output channels: 28 + 4 fragments of
// v_mfma_f32_32x32x16_f16, 128 registers), and keeps the intermediate activation in LDS, rounded to fp16
// exactly where the stored one was.  Persistent workgroups of four waves, two per CU, so that one's barriers
// and memory phases lie under the other's products (one of eight waves: 154 and 194 us).  At the
// decoder's 2 x 714240 rows: a unit 141 us (two GEMMs: 307; its 366 MB at the 5 TB/s of a large copy: 73, its
// products 45), post + final 184 us (two GEMMs: 641; 188 MB: 38, products 90).  What is left is the wait
// between dependent phases of a tile.
//
// Numerics: fp32 sums, fp32 bias, one fp16 rounding, PReLU and residual add on fp16 values, as the
// GEMM epilogues; the conv's products are summed in the same k order as there.
#include "gemm_core.h"

namespace ecd {

constexpr int CU_C = 64;          // channels
constexpr int CU_K = 7;           // taps of the wide convs
constexpr int CU_KS = CU_K * 4;   // their k-steps of 16
constexpr int CU_W = 4;           // waves per workgroup: 2 halves of the channels x 2 row groups

__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_s_waitcnt((15) | (7 << 4) | (3 << 14));  // lgkmcnt(0); vmcnt is not waited for
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// fragment of a packed [N, 64 n] weight: 32-row tile t32, k-step ks (chunk ks >> 2)
__device__ __forceinline__ f16x8 w_frag(const f16* w, int nch, int t32, int ks, int lane) {
  return *(const f16x8*)(w + ((long)(2 * t32 + ((lane >> 4) & 1)) * nch + (ks >> 2)) * 1024 +
                         (lane >> 5) * 512 + (16 * (ks & 3) + (lane & 15)) * 8);
}

// element address (halfs) of 16-byte piece p of row r of a 64-channel LDS tile
__device__ __forceinline__ int row_piece(int r, int p) { return r * CU_C + 8 * (p ^ x_swz(r)); }

// DMA of window rows 0 .. 32 N - 1 (CU_W waves, 8 rows per instruction): row r comes from source row
// min(r, last) of `src`
template <int N>
__device__ __forceinline__ void load_window(const f16* src, int last, const f16* win, int wv, int lane) {
  const uint32_t sa = lds_addr(win) + wv * 1024;
  static_for<0, N>([&](auto J) {
    const int r = 8 * (wv + CU_W * J.value) + (lane >> 3);
    lds_dma16_at<CU_W * J.value * 1024>(src, (uint32_t)(min(r, last) * (CU_C * 2) + 16 * ((lane & 7) ^ x_swz(r))), sa);
  });
}

// fp16(acc + bias) -> PReLU of group g (4 channels) of a 32 x 32 tile
__device__ __forceinline__ f16x4 bias_prelu(const f32x16& acc, int g, const f32x4& b, float a) {
  f16x4 v;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    v[j] = (f16)(acc[4 * g + j] + b[j]);
    if ((float)v[j] < 0.f) v[j] = (f16)((float)v[j] * a);
  }
  return v;
}

constexpr int RU_BM = 32 * CU_W;            // rows per tile
constexpr int RU_WIN = 6;                   // window DMA instructions per wave: 192 rows >= 128 + 6 * 10

// One residual unit, x -> y (different buffers of the same padded layout: `pad` zero rows before
// each of S sequences of T rows; y's pad rows are not written).  6 dil <= min(pad, 64).
__global__ __launch_bounds__(64 * CU_W, 2) void codec_unit64_kernel(
    const f16* __restrict__ x, f16* __restrict__ y, const f16* __restrict__ w1,
    const float* __restrict__ b1, float a1, const f16* __restrict__ w2, const float* __restrict__ b2,
    float a2, int T, int pad, int dil, int tps, int ntiles) {
  __shared__ __align__(16) f16 win[2][8 * CU_W * RU_WIN * CU_C];
  __shared__ __align__(16) f16 hs[RU_BM * CU_C];
  __shared__ __align__(16) float bs[2 * CU_C];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = wv & 1, wm = wv >> 1;  // 32 channels, 64 rows
  if (tid < CU_C) {
    bs[tid] = b1[tid];
    bs[CU_C + tid] = b2[tid];
  }
  f16x8 f1[CU_KS], f2[4];
  static_for<0, CU_KS>([&](auto I) { f1[I.value] = w_frag(w1, CU_K, wn, I.value, lane); });
  static_for<0, 4>([&](auto I) { f2[I.value] = w_frag(w2, 1, wn, I.value, lane); });

  auto load = [&](int tile, int buf) {
    const int b = tile / tps, t0 = (tile - b * tps) * RU_BM;
    load_window<RU_WIN>(x + ((long)b * (T + pad) + pad + t0 - 6 * dil) * CU_C, T - 1 - t0 + 6 * dil, win[buf],
                        wv, lane);
  };
  int tile = blockIdx.x, buf = 0;
  wait_vm0();  // the weights; from here on the outstanding operations are counted
  if (tile < ntiles) load(tile, 0);
  bool whole = false;  // the previous tile stored all its rows: 4 store instructions behind its DMA
  for (; tile < ntiles; tile += gridDim.x, buf ^= 1) {
    asm volatile("" ::: "memory");  // (the stores stay before the wait that counts them)
    if (whole) wait_vm<4>(); else wait_vm0();
    lds_barrier();  // this tile's window complete; every wave is done with the previous tile
    const int nt = tile + (int)gridDim.x;
    if (nt < ntiles) load(nt, buf ^ 1);
    const f16* w = win[buf];
    const int b = tile / tps, t0 = (tile - b * tps) * RU_BM;

    f32x16 acc[2] = {(f32x16)(0.f), (f32x16)(0.f)};
    static_for<0, CU_K>([&](auto J) {
      const int r = wm * 64 + (lane & 31) + J.value * dil;  // row + 32 has the same swizzle
      static_for<0, 4>([&](auto S) {
        const f16* p = w + row_piece(r, 2 * S.value + (lane >> 5));
        const f16x8 x0 = *(const f16x8*)p, x1 = *(const f16x8*)(p + 32 * CU_C);
        acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f1[4 * J.value + S.value], x0, acc[0], 0, 0, 0);
        acc[1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f1[4 * J.value + S.value], x1, acc[1], 0, 0, 0);
      });
    });
    auto stage = [&](int bo, float a) {
      static_for<0, 4>([&](auto G) {
        const int nl = wn * 32 + 8 * G.value + 4 * (lane >> 5);
        const f32x4 bv = *(const f32x4*)(bs + bo + nl);
        static_for<0, 2>([&](auto R) {
          const int r = wm * 64 + R.value * 32 + (lane & 31);
          *(f16x4*)(hs + row_piece(r, nl >> 3) + (nl & 4)) = bias_prelu(acc[R.value], G.value, bv, a);
        });
      });
    };
    stage(0, a1);
    lds_barrier();  // h complete
    acc[0] = (f32x16)(0.f);
    acc[1] = (f32x16)(0.f);
    static_for<0, 4>([&](auto S) {
      const f16* p = hs + row_piece(wm * 64 + (lane & 31), 2 * S.value + (lane >> 5));
      const f16x8 x0 = *(const f16x8*)p, x1 = *(const f16x8*)(p + 32 * CU_C);
      acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f2[S.value], x0, acc[0], 0, 0, 0);
      acc[1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f2[S.value], x1, acc[1], 0, 0, 0);
    });
    lds_barrier();  // h consumed
    stage(CU_C, a2);
    lds_barrier();
    f16* yo = y + ((long)b * (T + pad) + pad + t0) * CU_C;
    whole = t0 + RU_BM <= T;
    f16x8 v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int r = (tid >> 3) + 8 * CU_W * k, p = tid & 7;
      v[k] = *(const f16x8*)(hs + row_piece(r, p)) + *(const f16x8*)(w + row_piece(r + 6 * dil, p));
    }
    if (whole) {
#pragma unroll
      for (int k = 0; k < 4; ++k) *(f16x8*)(yo + (tid + 64 * CU_W * k) * 8) = v[k];
    } else {
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (t0 + (tid >> 3) + 8 * CU_W * k < T) *(f16x8*)(yo + (tid + 64 * CU_W * k) * 8) = v[k];
    }
  }
}

constexpr int PF_U = 32 * CU_W;      // samples of the wide conv per tile, the first 6 history
constexpr int PF_T = PF_U / 2 - 3;   // source rows per tile
constexpr int PF_WIN = 3;            // window DMA instructions per wave: 96 rows >= 61 + 6

// PostProcessor and final conv: u[s] = prelu(conv7 over x[s >> 1]) for samples s = 0 .. 2T - 1 (the nearest
// 2x repeat: output s, tap o reads source row (s + o) >> 1), out[s] = fp16(sum_j wf_j . u[s - 6 + j] + bf),
// u zero before the sequence.  Even and odd samples are separate row tiles that share their source rows:
// source row t - 3 + h feeds even taps 2h, 2h + 1 and odd taps 2h - 1, 2h.  The final conv has one output
// channel: its 7 taps are the features of one product over the 64 channels, P[j][s] = wf_j . u[s] (4
// products per 32 rows instead of 28), and out[s] sums P[j][s - 6 + j] in fp32.
__global__ __launch_bounds__(64 * CU_W, 2) void codec_post_final_kernel(
    const f16* __restrict__ x, const f16* __restrict__ w1, const float* __restrict__ b1, float a1,
    const f16* __restrict__ wf, const float* __restrict__ bf, f16* __restrict__ y, int T, int pad, int tps,
    int ntiles) {
  __shared__ __align__(16) f16 win[2][8 * CU_W * PF_WIN * CU_C];
  __shared__ __align__(16) f16 us[PF_U * CU_C];
  __shared__ __align__(16) float ps[PF_U * 8];
  __shared__ __align__(16) float bs[CU_C];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = wv & 1, wm = wv >> 1;  // 32 channels, 32 source rows (64 samples)
  if (tid < CU_C) bs[tid] = b1[tid];
  const float bias = bf[0];
  f16x8 f1[CU_KS], ff[4];
  static_for<0, CU_KS>([&](auto I) { f1[I.value] = w_frag(w1, CU_K, wn, I.value, lane); });
  // feature j of P is row 0 of chunk j of the packed final weight
  static_for<0, 4>([&](auto S) {
    ff[S.value] = *(const f16x8*)(wf + min(lane & 31, CU_K - 1) * 1024 + (lane >> 5) * 512 + 128 * S.value);
    if ((lane & 31) >= CU_K) ff[S.value] = (f16x8)(f16)0.f;
  });
  auto load = [&](int tile, int buf) {
    const int b = tile / tps, t0 = (tile - b * tps) * PF_T;
    load_window<PF_WIN>(x + ((long)b * (T + pad) + pad + t0 - 6) * CU_C, T - 1 - t0 + 6, win[buf], wv, lane);
  };
  int tile = blockIdx.x, buf = 0;
  wait_vm0();
  if (tile < ntiles) load(tile, 0);
  bool stored = false;  // this wave stored (one instruction) behind its DMA
  for (; tile < ntiles; tile += gridDim.x, buf ^= 1) {
    asm volatile("" ::: "memory");
    if (stored) wait_vm<1>(); else wait_vm0();
    lds_barrier();
    const int nt = tile + (int)gridDim.x;
    if (nt < ntiles) load(nt, buf ^ 1);
    const f16* w = win[buf];
    const int b = tile / tps, t0 = (tile - b * tps) * PF_T;

    // source row of local row l: t0 - 3 + l; window row l + h is source row t - 3 + h
    const int l = wm * 32 + (lane & 31);
    f32x16 acc[2] = {(f32x16)(0.f), (f32x16)(0.f)};  // even, odd samples
    static_for<0, 4>([&](auto H) {
      constexpr int h = decltype(H)::value;
      f16x8 xf[4];
      static_for<0, 4>([&](auto S) {
        xf[S.value] = *(const f16x8*)(w + row_piece(l + h, 2 * S.value + (lane >> 5)));
      });
      static_for<0, 2>([&](auto E) {  // the first, then the second tap of each parity
        constexpr int te = 2 * h + decltype(E)::value, to = te - 1;
        static_for<0, 4>([&](auto S) {
          if constexpr (te < CU_K)
            acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f1[4 * (te < CU_K ? te : 0) + S.value], xf[S.value],
                                                           acc[0], 0, 0, 0);
          if constexpr (to >= 0)
            acc[1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f1[4 * (to < 0 ? 0 : to) + S.value], xf[S.value],
                                                           acc[1], 0, 0, 0);
        });
      });
    });
    const bool before = t0 - 3 + l < 0;  // samples before the sequence are zero
    static_for<0, 4>([&](auto G) {
      const int nl = wn * 32 + 8 * G.value + 4 * (lane >> 5);
      const f32x4 bv = *(const f32x4*)(bs + nl);
      static_for<0, 2>([&](auto R) {
        f16x4 v = bias_prelu(acc[R.value], G.value, bv, a1);
        if (before) v = (f16x4)(f16)0.f;
        *(f16x4*)(us + row_piece(2 * l + R.value, nl >> 3) + (nl & 4)) = v;
      });
    });
    lds_barrier();
    f32x16 pa = (f32x16)(0.f);
    static_for<0, 4>([&](auto S) {
      const f16x8 u = *(const f16x8*)(us + row_piece(wv * 32 + (lane & 31), 2 * S.value + (lane >> 5)));
      pa = __builtin_amdgcn_mfma_f32_32x32x16_f16(ff[S.value], u, pa, 0, 0, 0);
    });
    *(f32x4*)(ps + (wv * 32 + (lane & 31)) * 8 + 4 * (lane >> 5)) = (f32x4){pa[0], pa[1], pa[2], pa[3]};
    lds_barrier();
    const int s = 2 * t0 + tid;
    stored = wv < CU_W / 2 && t0 + PF_T <= T;  // (samples 0 .. 2 PF_T - 1 lie in the first half of the waves)
    if (tid < 2 * PF_T && s < 2 * T) {
      float o = 0.f;
#pragma unroll
      for (int j = 0; j < CU_K; ++j) o += ps[(tid + j) * 8 + j];
      y[(long)b * 2 * T + s] = (f16)(o + bias);
    }
  }
}

static int persistent_blocks(int ntiles) {
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
    cus = 256;
  return ntiles < 2 * cus ? ntiles : 2 * cus;
}

static bool al(const void* p, int n) { return ((uintptr_t)p & (n - 1)) == 0; }

}  // namespace ecd

using namespace ecd;

extern "C" {

int ecd_codec_unit64(const void* x, void* y, const void* w1, const float* b1, float a1, const void* w2,
                     const float* b2, float a2, int S, int T, int pad, int dil, void* stream) {
  if (!x || !y || x == y || !w1 || !b1 || !w2 || !b2 || S <= 0 || T <= 0 || dil <= 0 || pad < 0 ||
      6L * dil > pad || 6L * dil > 64 || !al(x, 16) || !al(y, 16) || !al(w1, 16) || !al(w2, 16))
    return ECD_EINVAL;
  const int tps = (T + RU_BM - 1) / RU_BM;
  const long ntiles = (long)S * tps;
  if (ntiles > 0x3FFFFFFFL) return ECD_ENOTSUP;
  hipLaunchKernelGGL(codec_unit64_kernel, dim3(persistent_blocks((int)ntiles)), dim3(64 * CU_W), 0,
                     (hipStream_t)stream, (const f16*)x, (f16*)y, (const f16*)w1, b1, a1, (const f16*)w2, b2,
                     a2, T, pad, dil, tps, (int)ntiles);
  return ecd_launch_status();
}

int ecd_codec_post_final(const void* x, const void* w1, const float* b1, float a1, const void* wf,
                         const float* bf, void* y, int S, int T, int pad, void* stream) {
  if (!x || !y || !w1 || !b1 || !wf || !bf || S <= 0 || T <= 0 || T > 0x3FFFFFFF || pad < 6 || !al(x, 16) ||
      !al(y, 2) || !al(w1, 16) || !al(wf, 16))
    return ECD_EINVAL;
  const int tps = (T + PF_T - 1) / PF_T;
  const long ntiles = (long)S * tps;
  if (ntiles > 0x3FFFFFFFL) return ECD_ENOTSUP;
  hipLaunchKernelGGL(codec_post_final_kernel, dim3(persistent_blocks((int)ntiles)), dim3(64 * CU_W), 0,
                     (hipStream_t)stream, (const f16*)x, (const f16*)w1, b1, a1, (const f16*)wf, bf, (f16*)y, T,
                     pad, tps, (int)ntiles);
  return ecd_launch_status();
}

}  // extern "C"
