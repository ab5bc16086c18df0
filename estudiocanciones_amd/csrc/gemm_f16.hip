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
// Tiling (template): NW = WN x WM waves; wave (wn, wm) owns FT 32-feature tiles and RT 32-row tiles
// of v_mfma_f32_32x32x16_f16, so a block covers BN = 32 WN FT features x BM = 32 WM RT rows.  (At
// one wave per SIMD independent 32x32x16 products issued back to back reach 2.14 PFLOP/s on this
// chip, 16x16x32 ones 1.86.)  K advances in 64-wide chunks that go straight from global memory into
// an NS-stage LDS ring (LDS DMA, no register staging); x rows are stored with their 16-byte pieces
// XOR-swizzled by row (piece p of row r at position p ^ ((r >> 1) & 7)), so that the 16 rows that a
// ds_read_b128 serves at a time lie in distinct banks (no conflicts counted).
//
// What bounds it: a CU takes about 57 bytes per clock through its vector memory path (measured, L2
// hits), so a block tile needs a high ratio of products to bytes: 128 x 128 needs 575 clocks of
// loads for 512 of MFMA per chunk, 256 x 256 1150 for 2048.  Loads that miss L2 take 1 to 2 us, so a
// small tile needs many chunks in flight: NS is what the LDS holds.  Fragments are read half a chunk
// ahead, interleaved with the products; each DMA takes three instructions (computing every address
// on the scalar unit took twelve, and the issue slots of a third of the loop).  The output goes through
// LDS (see the epilogue).  us before -> now, M = 1488 (N, K): (4608, 1536) 31.8 -> 25.7, (8192, 1536)
// 56.3 -> 41.5, (1536, 1536) 16.6 -> 14.1, (1536, 4096) 36.3 -> 28.2, (9216, 3072) 102 -> 80,
// (16384, 3072) 182 -> 145, (3072, 8192) 111 -> 84; M = 187: (4608, 1536) 19.8 -> 9.9,
// (1536, 4096) 26.1 -> 14.4, (3072, 8192) 99.7 -> 36.8; 8192^3 0.90 -> 1.21 PFLOP/s.
//
// Block order is XCD-aware: the row blocks that share a weight tile get block ids equal modulo 8,
// so they run on one XCD and share its L2 (feature blocks in whole groups of 8; the grid has
// exactly one workgroup per output tile, so narrow outputs launch no empty workgroups).
#include "common.h"

namespace ecd {

enum { F16_STORE = 0, F16_SILU = 1, F16_PRELU = 2, F16_ROPE = 3 };

// wait until at most N vector-memory operations of this wave are outstanding and its LDS
// operations are done (lgkmcnt 0)
template <int N>
__device__ __forceinline__ void wait_vm_lgkm0() {
  static_assert(N >= 0 && N < 64, "vmcnt is 6 bits");
  __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | ((N >> 4) << 14));
}

// wait for this wave's DMA of one chunk while the `later` chunks issued after it (uniform,
// 0 .. MAXL) stay in flight; PER instructions per chunk; LGKM: also drain LDS operations
template <int PER, int MAXL, bool LGKM>
__device__ __forceinline__ void wait_chunk(int later) {
  if constexpr (MAXL >= 1) {
    if (later < MAXL) {
      wait_chunk<PER, MAXL - 1, LGKM>(later);
      return;
    }
  }
  if constexpr (LGKM) wait_vm_lgkm0<MAXL * PER>(); else wait_vm<MAXL * PER>();
}

template <int I>
struct IC {
  static constexpr int value = I;
};
// f(IC<B>{}), .., f(IC<E - 1>{})
template <int B, int E, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (B < E) {
    f(IC<B>{});
    static_for<B + 1, E>(f);
  }
}

// The fragments of half a 64-wide chunk, two k-steps of v_mfma_f32_32x32x16_f16: lane l holds
// feature (or row) l & 31 of a 32-wide tile, k = 16 s + 8 (l >> 5) .. + 7 of step s.
template <int FT, int RT>
struct Frags {
  f16x8 w[2][FT], x[2][RT];
};

// Row layouts of a convolution as a GEMM over implicit tap columns (the waveform decoder):
// row m = b * T + t of the GEMM.  With k > 0, x is time-major with xpad zero rows before each
// sequence and row m's K index j * C + c (C = 64 cpt) reads x row b (T + xpad) + xpad + t + off[j]
// (the tap offsets move the chunk's DMA base; the pad rows supply the zeros of the padding).
// With ypad >= 0, y and res rows are b (T + ypad) + ypad + t.  T = 0: plain rows throughout.
struct RowMap {
  int T, xpad, ypad, cpt, k, rep;
  int off[8];
};

// Output of the q | k | v projection with RoPE (F16_ROPE): features [0, D) are q, [D, 2D) k,
// [2D, 3D) v, D = H * HD, rows m = b * T + t.  q and k pairs (2i, 2i + 1) are rotated by
// tab[t, i] = (cos, sin) (fp16); q goes to rows [M, D], k and v to [B, H, T, HD].
struct RopeOut {
  const f16* tab;
  f16 *q, *k, *v;
  int T, H, HD;
};

__device__ __forceinline__ long seq_row(int m, int T, int pad) {
  const int b = m / T;
  return (long)b * (T + pad) + pad + (m - b * T);
}

// piece p of x row r lies at position p ^ x_swz(r) of its 128 bytes
__device__ __forceinline__ int x_swz(int r) { return (r >> 1) & 7; }

template <int EPI, int WN, int WM, int FT, int RT, int NS>
__global__ __launch_bounds__(64 * WN * WM, 2) void gemm_f16w_kernel(
    const f16* __restrict__ x, long ldx, const f16* __restrict__ wp,
    const float* __restrict__ bias, float alpha, const f16* res, long ldr,
    f16* y, long ldy, int M, int N, int K, int nfb, int nmb, RowMap rm,
    RopeOut ro) {
  constexpr int NW = WN * WM;           // waves
  constexpr int BN = 32 * WN * FT;      // features per block
  constexpr int BM = 32 * WM * RT;      // rows per block
  constexpr int WI = BN / 8 / NW;       // weight DMA instructions per wave per chunk (1 KB each)
  constexpr int XI = BM / 8 / NW;       // x DMA instructions per wave per chunk (8 rows each)
  constexpr int PER_CHUNK = WI + XI;
  static_assert(WI * 8 * NW == BN && XI * 8 * NW == BM, "whole DMA instructions per wave");
  static_assert(NS >= 2 && PER_CHUNK * (NS - 1) < 64, "vmcnt range");
  constexpr int LW = BN * 64, LX = BM * 64, STG = LW + LX;  // halfs per stage
  __shared__ __align__(16) f16 lds[NS * STG];

  // feature blocks in full groups of 8 share XCDs with their row blocks; the remaining
  // nfb % 8 feature blocks (all of them when nfb < 8) are laid out row-major after them
  const int b = blockIdx.x;
  const int full = nfb & ~7;
  int fb, mb;
  if (b < full * nmb) {
    const int grp8 = b / (8 * nmb);
    const int rem = b - grp8 * 8 * nmb;
    mb = rem >> 3;
    fb = grp8 * 8 + (rem & 7);
  } else {
    const int rem = b - full * nmb;
    const int tw = nfb - full;
    mb = rem / tw;
    fb = full + (rem - mb * tw);
  }

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = wv % WN, wm = wv / WN;
  const int n0 = fb * BN;
  const int m0 = mb * BM;
  const int nch = K >> 6;
  const int ntiles = (N + 15) >> 4;
  const long tile_bytes = (long)nch * 2048;

  // DMA sources: weight instruction j of this wave is tile t = i >> 1, half h = i & 1 with
  // i = wv + NW j (tiles past N re-read the last tile; their results are never stored); x
  // instruction j covers rows 8 i .. 8 i + 7, i = wv + NW j (rows past M re-read row M - 1).
  // Every address is a uniform base, advanced per chunk, plus a per-lane offset.
  const int t0 = min(n0 / 16, ntiles - 1);
  const char* wb = (const char*)wp + (long)t0 * tile_bytes;
  uint32_t woff[WI];
#pragma unroll
  for (int j = 0; j < WI; ++j) {
    const int i = wv + NW * j;
    woff[j] = (uint32_t)((min(n0 / 16 + (i >> 1), ntiles - 1) - t0) * tile_bytes) + 1024 * (i & 1) + 16 * lane;
  }
  // with a 2x row-repeat (rm.rep == 2) output step t reads source row (t + o) >> 1 for tap o:
  // (t >> 1) + (o >> 1) for even o, ((t + 1) >> 1) + (o >> 1) for odd o -- two lane rows
  uint32_t xoff[XI], xoff1[XI];
#pragma unroll
  for (int j = 0; j < XI; ++j) {
    const int i = wv + NW * j;
    const int xpiece = (lane & 7) ^ x_swz(8 * i + (lane >> 3));
    const int row = min(m0 + 8 * i + (lane >> 3), M - 1);
    long xr = row, xr1 = row;
    if (rm.k && rm.rep == 2) {
      const int b = row / rm.T, t = row - b * rm.T;
      const long base = (long)b * (rm.T / 2 + rm.xpad) + rm.xpad;
      xr = base + (t >> 1);
      xr1 = base + ((t + 1) >> 1);
    } else if (rm.k) {
      xr = xr1 = seq_row(row, rm.T, rm.xpad);
    }
    xoff[j] = (uint32_t)(xr * ldx * 2 + 16 * xpiece);
    xoff1[j] = (uint32_t)(xr1 * ldx * 2 + 16 * xpiece);
  }
  // x base of the next chunk to load: plain K offset 64 c, or tap j = c / cpt shifted by off[j]
  // rows (by off[j] >> 1 with a 2x row-repeat, odd taps reading the second set of lane rows)
  const f16* xb = x;
  int tap = 0, tc = 0;
  bool odd = false;
  auto set_tap = [&]() {
    const int o = rm.off[tap];
    odd = rm.rep == 2 && (o & 1);
    xb = x + (long)(rm.rep == 2 ? (o >> 1) : o) * ldx;
  };
  if (rm.k) set_tap();
  auto next_chunk = [&]() {
    xb += 64;
    wb += 2048;
    if (rm.k && ++tc == rm.cpt) {
      tc = 0;
      ++tap;
      if (tap < rm.k) set_tap();
    }
  };
  // DMA instruction J of the next chunk into the stage at LDS byte address `sa` (this wave's first
  // KB of it): weights first, then x rows
  auto dma = [&](auto J, uint32_t sa) {
    constexpr int j = decltype(J)::value;
    if constexpr (j < WI)
      lds_dma16_at<NW * j * 1024>(wb, woff[j], sa);
    else
      lds_dma16_at<LW * 2 + NW * (j - WI) * 1024>(xb, odd ? xoff1[j - WI] : xoff[j - WI], sa);
  };
  const uint32_t lds0 = lds_addr(lds) + wv * 1024;

  f32x16 acc[FT][RT];
  static_for<0, FT * RT>([&](auto I) {
    acc[I.value / RT][I.value % RT] = (f32x16)(0.f);
  });

  // fragment addresses within a stage (halfs): a 32-feature tile is two packed 16-row tiles, octet
  // o = 2 s + (lane >> 5) of k-step s lies in half o & 1 = lane >> 5 at 16-byte unit 16 s + row
  const int wfo = (wn * FT * 2 + ((lane >> 4) & 1)) * 1024 + (lane >> 5) * 512 + (lane & 15) * 8;
  int xfo[4];
  static_for<0, 4>([&](auto S) {
    xfo[S.value] = LW + (wm * RT * 32 + (lane & 31)) * 64 +
                   8 * ((2 * S.value + (lane >> 5)) ^ x_swz(lane & 31));
  });

  // read I of a half chunk's fragments (k-steps 2 H and 2 H + 1), k-step by k-step
  constexpr int NM = 2 * FT * RT, NR = 2 * (FT + RT);
  auto read1 = [&](auto I, auto H, const f16* base, Frags<FT, RT>& f) {
    constexpr int s = decltype(I)::value / (FT + RT), i = decltype(I)::value % (FT + RT);
    constexpr int ks = 2 * decltype(H)::value + s;
    if constexpr (i < FT)
      f.w[s][i] = *(const f16x8*)(base + wfo + 128 * ks + i * 2048);
    else
      f.x[s][i - FT] = *(const f16x8*)(base + xfo[ks] + (i - FT) * 2048);
  };
  // the products of a half chunk, interleaved with the reads of the next half chunk's fragments
  // (in the first half of the products, so that they have landed at its end) and, with LOAD, the
  // loads of a later chunk
  auto half = [&](const Frags<FT, RT>& f, auto H, const f16* base, Frags<FT, RT>& nf, auto LOAD,
                  uint32_t sa) {
    constexpr int RH = NM / 2;
    static_for<0, NM>([&](auto I) {
      constexpr int m = decltype(I)::value, s = m / (FT * RT), ft = m % (FT * RT) / RT, rt = m % RT;
      acc[ft][rt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.w[s][ft], f.x[s][rt], acc[ft][rt], 0, 0, 0);
      if constexpr (decltype(LOAD)::value)
        static_for<m * PER_CHUNK / NM, (m + 1) * PER_CHUNK / NM>([&](auto J) { dma(J, sa); });
      if constexpr (m < RH)
        static_for<m * NR / RH, (m + 1) * NR / RH>([&](auto J) { read1(J, H, base, nf); });
      __builtin_amdgcn_sched_barrier(0);
    });
  };

  for (int s = 0; s < NS; ++s)
    if (s < nch) {
      static_for<0, PER_CHUNK>([&](auto J) { dma(J, lds0 + s * (STG * 2)); });
      next_chunk();
    }
  wait_chunk<PER_CHUNK, NS - 1, false>(min(NS - 1, nch - 1));
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  Frags<FT, RT> fa, fc;
  static_for<0, NR>([&](auto I) { read1(I, IC<0>{}, lds, fa); });

  // Chunk c: its first half while its second half is read; then, with chunk c + 1 landed for this
  // wave (later ones may fly) and its own reads of chunk c done, a barrier that publishes the one and
  // frees the stage of the other; then the second half while chunk c + 1's first half is read and
  // chunk c + NS loaded into the stage left free.
  int c = 0, st = 0;  // st: stage of chunk c
  for (; c < nch - NS; ++c) {
    half(fa, IC<1>{}, lds + st * STG, fc, IC<0>{}, 0);
    wait_vm_lgkm0<(NS - 2) * PER_CHUNK>();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    const int sn = st + 1 == NS ? 0 : st + 1;
    half(fc, IC<0>{}, lds + sn * STG, fa, IC<1>{}, lds0 + st * (STG * 2));
    next_chunk();
    st = sn;
  }
  for (; c < nch; ++c) {
    half(fa, IC<1>{}, lds + st * STG, fc, IC<0>{}, 0);
    if (c + 1 < nch) {
      wait_chunk<PER_CHUNK, NS - 2, true>(min(NS - 2, nch - 2 - c));
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
    }
    // (behind the last chunk the reads return a stage's old contents, never used)
    const int sn = st + 1 == NS ? 0 : st + 1;
    half(fc, IC<0>{}, lds + sn * STG, fa, IC<0>{}, 0);
    st = sn;
  }

  // Epilogue.  A lane holds features 8 g + 4 (lane >> 5) .. + 3 (g < 4) of row lane & 31 of each of
  // its tiles.  The rounded sums go through LDS (the stages are free once every wave has read its last
  // fragments), so that a short loop finishes them in 16-byte pieces of consecutive features and
  // writes whole row segments.  Unrolled over the accumulators, with 8-byte stores to 32 rows per
  // instruction, the same work took about 1.1 us per 32 x 32 tile of a wave, most of it instruction
  // fetch (the code runs once per workgroup).
  constexpr int PR = BN / 8;                       // 16-byte pieces per row
  constexpr int SM = PR < 16 ? PR - 1 : 15;
  auto piece = [](int r, int p) { return (r * PR + (p ^ (r & SM))) * 8; };  // in halfs
  static_assert(NS * STG >= BM * BN, "the output tile fits the stages");
  __syncthreads();
  static_for<0, 4 * FT>([&](auto I) {
    constexpr int ft = decltype(I)::value >> 2, g = decltype(I)::value & 3;
    const int nl = (wn * FT + ft) * 32 + 8 * g + 4 * (lane >> 5);
    f32x4 bv = (f32x4){0.f, 0.f, 0.f, 0.f};
    if (bias) {
#pragma unroll
      for (int r = 0; r < 4; ++r) bv[r] = bias[min(n0 + nl + r, N - 1)];
    }
    static_for<0, RT>([&](auto R) {
      constexpr int rt = decltype(R)::value;
      const int r = (wm * RT + rt) * 32 + (lane & 31);
      f16x4 yv;
#pragma unroll
      for (int j = 0; j < 4; ++j) yv[j] = (f16)(acc[ft][rt][4 * g + j] + bv[j]);
      *(f16x4*)(lds + piece(r, nl >> 3) + (nl & 4)) = yv;
    });
  });
  __syncthreads();
  // 16-byte rows of y (and res) take one store per piece
  const bool vec = ((ldy & 7) == 0) && (((uintptr_t)y & 15) == 0) &&
                   (!res || (((ldr & 7) == 0) && (((uintptr_t)res & 15) == 0)));
#pragma unroll 1
  for (int i = tid; i < BM * PR; i += 64 * NW) {
    const int r = i / PR, p = i - r * PR;
    const int mm = m0 + r, nb = n0 + 8 * p;
    if (mm >= M || nb >= N) continue;
    f16x8 v = *(const f16x8*)(lds + piece(r, p));
    if constexpr (EPI == F16_STORE || EPI == F16_PRELU) {
      const long m = rm.ypad >= 0 ? seq_row(mm, rm.T, rm.ypad) : mm;
      if constexpr (EPI == F16_PRELU) {  // alpha: the slope
#pragma unroll
        for (int j = 0; j < 8; ++j)
          if ((float)v[j] < 0.f) v[j] = (f16)((float)v[j] * alpha);
      } else if (alpha != 1.0f) {
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = (f16)((float)v[j] * alpha);
      }
      if (vec && nb + 7 < N) {
        if (res) v = v + *(const f16x8*)(res + m * ldr + nb);
        *(f16x8*)(y + m * ldy + nb) = v;
      } else {
        for (int j = 0; j < 8 && nb + j < N; ++j) {
          f16 o = v[0];
          if (res) o = o + res[m * ldr + nb + j];
          y[m * ldy + nb + j] = o;
          v = __builtin_shufflevector(v, v, 1, 2, 3, 4, 5, 6, 7, 0);
        }
      }
    } else if constexpr (EPI == F16_ROPE) {
      // sections q, k, v; 4 features never straddle a head (HD % 4 == 0)
      const int D = ro.H * ro.HD;
      const int rb = mm / ro.T, t = mm - rb * ro.T;
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int n = nb + 4 * q;
        if (n >= N) break;
        const int sec = n >= 2 * D ? 2 : (n >= D ? 1 : 0);
        const int hc = n - sec * D, hh = hc / ro.HD, d = hc - hh * ro.HD;
        f16x4 o = q ? __builtin_shufflevector(v, v, 4, 5, 6, 7) : __builtin_shufflevector(v, v, 0, 1, 2, 3);
        if (sec < 2) {
          const f16x4 cs = *(const f16x4*)(ro.tab + (long)t * ro.HD + d);  // pairs d/2, d/2 + 1
          f16 o0, o1, o2, o3;
          rope_pair_f16((float)o[0], (float)o[1], (float)cs[0], (float)cs[1], o0, o1);
          rope_pair_f16((float)o[2], (float)o[3], (float)cs[2], (float)cs[3], o2, o3);
          o = (f16x4){o0, o1, o2, o3};
        }
        f16* dst = sec == 0 ? ro.q + (long)mm * D + hc
                            : (sec == 1 ? ro.k : ro.v) + (((long)rb * ro.H + hh) * ro.T + t) * ro.HD + d;
        *(f16x4*)dst = o;
      }
    } else {  // pairs (a_j, b_j) with j = nb / 2 ..; N even
      f16x2 o[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const float a = (float)v[2 * q];
        const f16 s = (f16)(a / (1.0f + expf(-a))) * v[2 * q + 1];
        o[q >> 1][q & 1] = s;
      }
      f16* dst = y + (long)mm * ldy + (nb >> 1);
      if (nb + 7 < N && ((ldy & 3) == 0) && (((uintptr_t)y & 7) == 0)) {
        *(f16x4*)dst = (f16x4){o[0].x, o[0].y, o[1].x, o[1].y};
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (nb + 2 * q < N) dst[q] = o[q >> 1][q & 1];
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

template <int EPI, int WN, int WM, int FT, int RT, int NS>
static int launch_cfg(const f16* x, long ldx, const f16* wp, const float* bias, float alpha,
                      const f16* res, long ldr, f16* y, long ldy, int M, int N, int K,
                      const RowMap& rm, const RopeOut& ro, hipStream_t st) {
  constexpr int BN = 32 * WN * FT, BM = 32 * WM * RT;
  const int nfb = (N + BN - 1) / BN;
  const int nmb = (M + BM - 1) / BM;
  const long blocks = (long)nfb * nmb;
  if (blocks > 0x7FFFFFFFL) return ECD_ENOTSUP;
  hipLaunchKernelGGL((gemm_f16w_kernel<EPI, WN, WM, FT, RT, NS>), dim3((unsigned)blocks),
                     dim3(64 * WN * WM), 0, st, x, ldx, wp, bias, alpha, res, ldr, y, ldy, M, N, K,
                     nfb, nmb, rm, ro);
  return ecd_launch_status();
}

// The tiles (features x rows, LDS stages).  1 to 8 leave room for one workgroup per CU: a launch takes
// ceil(blocks / 256) rounds, a round about K / 64 chunk times plus a fill and an epilogue; both in ns,
// measured over K = 1536 .. 8192 with 100 to 256 workgroups.
struct Tile {
  int bn, bm, chunk, edge;
};
constexpr Tile TILES[8] = {
    {256, 256, 1550, 4500},  // 1: 8 waves of 64 x 128, 2 stages
    {256, 192, 1450, 3500},  // 2: 8 waves of 64 x 96, 2 stages
    {256, 128, 850, 2500},   // 3: 8 waves of 64 x 64, 3 stages
    {128, 192, 620, 3000},   // 4: 8 waves of 32 x 96, 3 stages
    {128, 128, 440, 1200},   // 5: 8 waves of 32 x 64, 4 stages
    {128, 64, 300, 800},     // 6: 4 waves of 64 x 32, 5 stages
    {64, 128, 300, 800},     // 7: 4 waves of 32 x 64, 5 stages
    {64, 64, 220, 600},      // 8: 4 waves of 32 x 32, 8 stages
};
// 9: 128 x 128, 8 waves, 2 stages; 10: 64 x 128, 8 waves, 2 stages: several workgroups per CU, for the
// waveform decoder's convolutions of at most 128 channels over many rows, whose few chunks leave the
// fill and the stores to be hidden by other workgroups (476160 rows, 128 channels, us for K = 896 / 128:
// tile 9 213 / 43, 5 228 / 62, 3 270 / 79; 1.4 M rows, 64 channels, K = 448 / 64: tile 10 274 / 69,
// 9 295 / 91, 7 322 / 134).
constexpr int MANY_ROWS = 16384;

// Library default per shape (N counts output features before the SiLU pairing): the tile of the
// shortest estimate.  (Of 29 shapes measured with every tile it is the fastest or within 10% of it.)
static int default_cfg(int M, int N, int K) {
  if (M >= MANY_ROWS && N <= 128) return N <= 64 ? 10 : 9;
  int best = 1;
  long tb = 0;
  for (int i = 0; i < 8; ++i) {
    const Tile& t = TILES[i];
    const long blocks = (long)((N + t.bn - 1) / t.bn) * ((M + t.bm - 1) / t.bm);
    const long est = (blocks + 255) / 256 * ((long)(K >> 6) * t.chunk + t.edge);
    if (i == 0 || est < tb) {
      best = i + 1;
      tb = est;
    }
  }
  return best;
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

int ecd_gemm_f16p_silu(const void* x, long ldx, const void* wp, void* mm, long ldm, int M, int F,
                       int K, void* stream) {
  if (F <= 0) return ECD_EINVAL;
  return ecd_gemm_f16p_tuned(x, ldx, wp, nullptr, 1.0f, nullptr, 0, mm, ldm, M, 2 * F, K, 1, 0,
                             stream);
}

}  // extern "C"
