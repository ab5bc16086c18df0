// The MFMA GEMM main loop shared by the fp16-weight GEMM (gemm_f16.hip) and the int8-weight GEMM
// (gemm_i8.hip): one workgroup computes a BN x BM (features x rows) tile of x @ w^T and leaves the
// rounded fp16 sums in LDS for an epilogue to finish.
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
//
// int8 weights (W8) take half the LDS and load bytes; their 16-byte units (16 consecutive k of one
// feature) are read half a chunk ahead like the other fragments and dequantised, fp16(q * s), between
// the products of the half chunk before the one that uses them, so no product waits for the conversion.
#pragma once
#include "common.h"

namespace ecd {

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

__device__ __forceinline__ long seq_row(int m, int T, int pad) {
  const int b = m / T;
  return (long)b * (T + pad) + pad + (m - b * T);
}

// Vectors in rows of any alignment (one instruction all the same: global memory takes dwordx2 and dwordx4 at
// any address).  With 2-byte stores wherever a row was not 16-byte aligned, us -> now: fp16 1488 x 1536 x 1536 in
// rows of 1540 21.7 -> 14.1, 1488 x 1021 x 512 12.9 -> 8.0; int8 400 x 8197 x 3072 39.4 -> 32.7, 2048 x 8197 x
// 3072 150 -> 123.
typedef f16x8 f16x8u __attribute__((aligned(2)));
typedef f16x4 f16x4u __attribute__((aligned(2)));
typedef f16x2 f16x2u __attribute__((aligned(2)));

// y[0 .. n - 1] = v (+ res), n < 8: the piece that holds the end of a row
__device__ __forceinline__ void store_tail(f16* y, const f16* res, f16x8 v, int n) {
  if (n & 4) {
    const f16x4 o = __builtin_shufflevector(v, v, 0, 1, 2, 3);
    *(f16x4u*)y = res ? o + *(const f16x4u*)res : o;
    v = __builtin_shufflevector(v, v, 4, 5, 6, 7, 0, 1, 2, 3);
  }
  const int n4 = n & 4;
  if (n & 2) {
    const f16x2 o = __builtin_shufflevector(v, v, 0, 1);
    *(f16x2u*)(y + n4) = res ? o + *(const f16x2u*)(res + n4) : o;
    v = __builtin_shufflevector(v, v, 2, 3, 4, 5, 6, 7, 0, 1);
  }
  const int n6 = n & 6;
  if (n & 1) y[n6] = res ? v[0] + res[n6] : v[0];
}

// piece p of x row r lies at position p ^ x_swz(r) of its 128 bytes
__device__ __forceinline__ int x_swz(int r) { return (r >> 1) & 7; }


// fp16(silu(a)) * b for 4 interleaved pairs (a, b).  The sigmoid by the exp2 and reciprocal instructions (1 ulp
// of fp32 each): for every finite fp16 a the rounded result is the nearest fp16, which expf and an IEEE division miss
// once (a = -2.7246); with those the SiLU epilogue of a 256 x 128 tile took about 5 us.
__device__ __forceinline__ f16x4 silu_mul4(const f16x8& v) {
  f16x4 o;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const float a = (float)v[2 * q];
    const float e = __builtin_amdgcn_exp2f(a * -1.44269504088896341f);
    o[q] = (f16)(a * __builtin_amdgcn_rcpf(1.0f + e)) * v[2 * q + 1];
  }
  return o;
}

// A tile (features x rows) with its measured times in ns: a 64-wide chunk with at most LIGHT workgroups and
// with 256 (one per CU, all loading), and the fill and epilogue of a round.
struct Tile {
  int bn, bm, light, full, edge;
};
constexpr int LIGHT = 144;

// Estimate of a launch over nch chunks, K split `ks` ways: rounds of 256 workgroups (also for a tile of which two fit a
// CU: their rounds run at the same time, each chunk twice as long).
inline long tile_estimate(const Tile& t, int M, int N, int nch, int ks) {
  const long blocks = (long)((N + t.bn - 1) / t.bn) * ((M + t.bm - 1) / t.bm) * ks;
  const long load = blocks <= LIGHT ? 0 : (blocks >= 256 ? 256 - LIGHT : blocks - LIGHT);
  const long chunk = t.light + (t.full - t.light) * load / (256 - LIGHT);
  return (blocks + 255) / 256 * ((long)((nch + ks - 1) / ks) * chunk + t.edge);
}

// The loads' weight offsets are 32-bit from a workgroup's first feature: its bn features of K 16-bit values
// (int8 weights: half of that) must stay below 4 GiB.  A K for which even 64 features do not fit runs on 64 x 64 tiles
// with a base of its own for every load (GemmTile::run's BIG).
inline bool w_offsets_fit(int bn, int nch) { return (long)bn * nch * 128 <= 0xFFFFFFFFL; }

// The tile of the shortest estimate (0-based) among those whose weight offsets fit, and that estimate.
inline int best_tile(const Tile* t, int n, int M, int N, int nch, int ks, long* est) {
  int best = n - 1;
  *est = 0x7FFFFFFFFFFFFFFFL;
  for (int i = 0; i < n; ++i) {
    const long e = tile_estimate(t[i], M, N, nch, ks);
    if (w_offsets_fit(t[i].bn, nch) && e < *est) {
      best = i;
      *est = e;
    }
  }
  return best;
}

// Ways to split K for a product of few rows whose consumer adds fp32 partial sums (1: do not).  A split
// launch fills CUs that the tiles of one leave idle, at most one workgroup per CU; the ks M N floats that it
// writes and the consumer reads are taken at 2 ps each, its larger edges at 0.5 us.  (Its sums group K by the ways, so above
// 64 rows the bits of a row depend on how many rows the call has; the decode attention's split is by rows too.)  Product and
// consuming norm, us, one way -> the rule's ways (best of 1..8):
//   fp16 weights  187 x 1536 x 1536   11.4 -> 10.1 (2)  10.1 | 187 x 1536 x 4096   17.4 -> 12.3 (3)  12.3
//                 187 x 3072 x 8192   40.9 -> 28.5 (2)  28.5 | 187 x 3072 x 3072   16.5 -> 16.5 (1)  15.4
//                  24 x 3072 x 8192   33.8 -> 18.3 (5)  18.1 | 372 x 1536 x 4096   19.1 -> 16.4 (2)  15.4
//                 372 x 3072 x 8192   55.8 -> 55.8 (1)  45.2 | 744 x 1536 x 4096   25.0 -> 25.0 (1)  25.0
//   int8 weights   77 x 3072 x 8192   40.7 -> 21.1 (5)  19.6 | 154 x 3072 x 8192   41.1 -> 28.2 (2)  28.2
//                  77 x 3072 x 3072   19.5 -> 14.1 (5)  13.6 | 154 x 3072 x 3072   20.1 -> 16.6 (2)  16.6
//                 512 x 3072 x 8192   50.2 -> 50.2 (1)  50.2 | 256 x 3072 x 8192   42.5 -> 30.1 (2)  30.1
constexpr int SPLIT_MAX = 8;
inline int split_ways(const Tile* t, int n, const Tile* small, int nsmall, int M, int N, int nch) {
  long best = 0;
  best_tile(t, n, M, N, nch, 1, &best);
  int ks = 1;
  for (int k = 2; k <= SPLIT_MAX && k * 2 <= nch; ++k)
    for (int i = 0; i < nsmall; ++i) {
      const long blocks = (long)((N + small[i].bn - 1) / small[i].bn) * ((M + small[i].bm - 1) / small[i].bm) * k;
      if (blocks > 256) continue;
      const long e = tile_estimate(small[i], M, N, nch, k) + (long)k * M * N / 500 + 500;
      if (e < best) {
        best = e;
        ks = k;
      }
    }
  return ks;
}

template <bool W8, bool RM, int WN, int WM, int FT, int RT, int NS>
struct GemmTile {
  static constexpr int NW = WN * WM;           // waves
  static constexpr int BN = 32 * WN * FT;      // features per block
  static constexpr int BM = 32 * WM * RT;      // rows per block
  static constexpr int WPT = W8 ? 1 : 2;       // KB of weights per 16 features and chunk
  static constexpr int WI = BN / 16 * WPT / NW;  // weight DMA instructions per wave per chunk (1 KB each)
  static constexpr int XI = BM / 8 / NW;       // x DMA instructions per wave per chunk (8 rows each)
  static constexpr int PER_CHUNK = WI + XI;
  static_assert(WI * NW * 16 == BN * WPT && XI * 8 * NW == BM, "whole DMA instructions per wave");
  static_assert(NS >= 2 && PER_CHUNK * (NS - 1) < 64, "vmcnt range");
  static constexpr int LW = BN * (W8 ? 32 : 64), LX = BM * 64, STG = LW + LX;  // halfs per stage

  static constexpr int LDS_HALFS = NS * STG;
  static constexpr int PR = BN / 8;            // 16-byte pieces per output row
  static_assert(NS * STG >= BM * BN, "the output tile fits the stages");
  // piece p of output row r in LDS, in halfs
  static __device__ __forceinline__ int piece(int r, int p) {
    constexpr int SM = PR < 16 ? PR - 1 : 15;
    return (r * PR + (p ^ (r & SM))) * 8;
  }

  // An epilogue's thread keeps one piece p of the row (whatever depends on the feature is formed once) and
  // takes rows threadIdx.x / PR + RS k, U at a time, so that the loads of U rows are in flight together.
  static constexpr int RS = 64 * NW / PR;
  static_assert(64 * NW % PR == 0 && BM % RS == 0, "whole rows per pass");
  static constexpr int U = BM / RS < 4 ? BM / RS : (BM / RS % 4 == 0 ? 4 : (BM / RS % 3 == 0 ? 3 : 2));
  static_assert(BM / RS % U == 0, "whole batches of rows");

  // Block b of the XCD-aware order -> (feature block, row block)
  static __device__ __forceinline__ void block(int nfb, int nmb, int& fb, int& mb) {
    // feature blocks in full groups of 8 share XCDs with their row blocks; the remaining
    // nfb % 8 feature blocks (all of them when nfb < 8) are laid out row-major after them
    const int b = blockIdx.x;
    const int full = nfb & ~7;
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

  }

  // The tile at features n0, rows m0: the fp16 sums (plus bias) of feature n0 + 8 p + j and row m0 + r
  // end at lds[piece(r, p) + j].  sc: the per-feature scales of int8 weights.  RM: w is a row-major
  // [N, K] int8 matrix instead of packed tiles.  Ends with a barrier.
  // PART: only K chunks c0 .. c0 + cn - 1 (plain rows), whose fp32 sums go to part [M, N] (N % 4 == 0)
  // instead, straight from the registers.
  // BIG: weights whose offsets from the first feature pass 32 bits; each DMA instruction keeps its own base.
  template <bool PART = false, bool BIG = false>
  static __device__ __forceinline__ void run(f16* lds, const f16* __restrict__ x, long ldx,
                                             const void* __restrict__ wp, const f16* __restrict__ sc,
                                             const float* __restrict__ bias, int M, int N, int K,
                                             int n0, int m0, const RowMap& rm, int c0 = 0, int cn = 0,
                                             float* __restrict__ part = nullptr) {
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wn = wv % WN, wm = wv / WN;
    const int nch = PART ? cn : K >> 6;
    const int ntiles = (N + 15) >> 4;
    const long tile_bytes = RM ? 16L * K : (long)(K >> 6) * (1024 * WPT);

    // DMA sources: weight instruction j of this wave is tile t = i >> 1, half h = i & 1 (int8: tile i) with
    // i = wv + NW j (tiles past N re-read the last tile; their results are never stored); x
    // instruction j covers rows 8 i .. 8 i + 7, i = wv + NW j (rows past M re-read row M - 1).
    // Every address is a uniform base, advanced per chunk, plus a per-lane offset.
    const int t0 = min(n0 / 16, ntiles - 1);
    const char* wb = (const char*)wp + (long)t0 * tile_bytes;
    uint32_t woff[WI];
    const char* wbig[BIG ? WI : 1];
#pragma unroll
    for (int j = 0; j < WI; ++j) {
      const int i = wv + NW * j;
      const int t = min(n0 / 16 + (W8 ? i : i >> 1), ntiles - 1);
      if constexpr (BIG) {
        wbig[j] = (const char*)wp + (long)t * tile_bytes + (W8 ? 0 : 1024 * (i & 1));
        woff[j] = RM ? (uint32_t)((min(16 * t + (lane & 15), N - 1) - 16 * t) * (long)K + 16 * (lane >> 4)) : 16 * lane;
      } else if constexpr (RM)  // the same lane order from rows of w: row lane & 15 (past N: the last), unit lane >> 4
        woff[j] = (uint32_t)((min(16 * t + (lane & 15), N - 1) - 16 * t0) * (long)K + 16 * (lane >> 4));
      else
        woff[j] = (uint32_t)((t - t0) * tile_bytes) + (W8 ? 0 : 1024 * (i & 1)) + 16 * lane;
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
    if constexpr (PART) {
      xb += c0 * 64L;
      wb += (long)c0 * (RM ? 64 : 1024 * WPT);
    }
    auto next_chunk = [&]() {
      xb += 64;
      wb += RM ? 64 : 1024 * WPT;
      if constexpr (BIG) {
#pragma unroll
        for (int j = 0; j < WI; ++j) wbig[j] += RM ? 64 : 1024 * WPT;
      }
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
        lds_dma16_at<NW * j * 1024>(BIG ? wbig[BIG ? j : 0] : wb, woff[j], sa);
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
    // (int8: unit 2 h + (lane >> 5) of half chunk h, whose first and last 8 codes are the two k-steps)
    const int wfo = W8 ? (wn * FT * 2 + ((lane >> 4) & 1)) * 512 + (lane >> 5) * 128 + (lane & 15) * 8
                       : (wn * FT * 2 + ((lane >> 4) & 1)) * 1024 + (lane >> 5) * 512 + (lane & 15) * 8;
    int xfo[4];
    static_for<0, 4>([&](auto S) {
      xfo[S.value] = LW + (wm * RT * 32 + (lane & 31)) * 64 +
                     8 * ((W8 ? 4 * (S.value >> 1) + 2 * (lane >> 5) + (S.value & 1) : 2 * S.value + (lane >> 5)) ^
                          x_swz(lane & 31));
    });

    // read I of half chunk H's fragments (k-steps 2 H and 2 H + 1): weights, then x rows
    constexpr int NM = 2 * FT * RT, NRW = W8 ? FT : 2 * FT, NR = NRW + 2 * RT;
    u32x4 raw[W8 ? FT : 1];  // int8 codes of the next half chunk
    f16 scale[W8 ? FT : 1];
    if constexpr (W8) {
#pragma unroll
      for (int ft = 0; ft < FT; ++ft) scale[ft] = sc[min(n0 + (wn * FT + ft) * 32 + (lane & 31), N - 1)];
    }
    auto read1 = [&](auto I, auto H, const f16* base, Frags<FT, RT>& f) {
      constexpr int i = decltype(I)::value, h = decltype(H)::value;
      if constexpr (i < NRW) {
        if constexpr (W8)
          raw[i] = *(const u32x4*)(base + wfo + 256 * h + i * 1024);
        else
          f.w[i / FT][i % FT] = *(const f16x8*)(base + wfo + 128 * (2 * h + i / FT) + (i % FT) * 2048);
      } else {
        constexpr int k = i - NRW, s = k / RT, rt = k % RT;
        f.x[s][rt] = *(const f16x8*)(base + xfo[2 * h + s] + rt * 2048);
      }
    };
    // the conversion of feature tile T
    auto dequant_tile = [&](auto T, Frags<FT, RT>& f) {
      constexpr int ft = decltype(T)::value;
      f16x8 a, c;
      i8x16_to_f16(raw[ft], a, c);
      f.w[0][ft] = a * scale[ft];
      f.w[1][ft] = c * scale[ft];
    };
    // piece T of the conversion: 4 codes of feature tile T / 4
    auto dequant = [&](auto T, Frags<FT, RT>& f) {
      constexpr int ft = decltype(T)::value >> 2, q = decltype(T)::value & 3;
      f16x2 lo, hi;
      i8x4_to_f16(raw[ft][q], lo, hi);
      const f16x2 s2 = {scale[ft], scale[ft]};
      lo = lo * s2;
      hi = hi * s2;
      f16x8& w = f.w[q >> 1][ft];
      w[4 * (q & 1)] = lo.x;
      w[4 * (q & 1) + 1] = lo.y;
      w[4 * (q & 1) + 2] = hi.x;
      w[4 * (q & 1) + 3] = hi.y;
    };
    // the products of a half chunk, interleaved with the reads of the next half chunk's fragments, DMA
    // instructions D0 .. D1 - 1 of a later chunk and, behind the reads, the dequantisation
    auto half = [&](const Frags<FT, RT>& f, auto H, const f16* base, Frags<FT, RT>& nf, auto D0,
                    auto D1, uint32_t sa) {
      constexpr int RH = W8 ? NM / 2 : NM;
      static_for<0, NM>([&](auto I) {
        constexpr int m = decltype(I)::value, s = m / (FT * RT), ft = m % (FT * RT) / RT, rt = m % RT;
        acc[ft][rt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.w[s][ft], f.x[s][rt], acc[ft][rt], 0, 0, 0);
        // few products: no conversion (and its wait) ahead of one.  (With many the compiler's own order is
        // better: 2048 rows (3072, 3072) 42.5 us without this line, 50.8 with it.)
        if constexpr (W8 && RT < 4) __builtin_amdgcn_sched_barrier(0);
        constexpr int d0 = decltype(D0)::value, nd = decltype(D1)::value - d0;
        static_for<d0 + m * nd / NM, d0 + (m + 1) * nd / NM>([&](auto J) { dma(J, sa); });
        if constexpr (m < RH)
          static_for<m * NR / RH, (m + 1) * NR / RH>([&](auto J) { read1(J, H, base, nf); });
        if constexpr (W8 && m >= RH)
          static_for<(m - RH) * 4 * FT / (NM - RH), (m - RH + 1) * 4 * FT / (NM - RH)>(
              [&](auto T) { dequant(T, nf); });
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
    if constexpr (W8) static_for<0, FT>([&](auto T) { dequant_tile(T, fa); });

    // Each pass of the loop: with chunk c + 1 landed for this wave (later ones may fly) and its own reads of
    // chunk c done, a barrier that publishes the one and frees the stage of the other; then chunk c's second
    // half while chunk c + 1's first half is read, and chunk c + 1's first half while its second is read.
    // Chunk c + NS is loaded into the stage left free, spread over both halves; over the first alone with two
    // stages, where it is needed soonest, and with int8 weights, whose conversion fills the second.
    constexpr int DS = NS > 2 && !W8 ? (PER_CHUNK + 1) / 2 : PER_CHUNK;
    int c = 0, st = 0;  // st: stage of chunk c
    half(fa, IC<1>{}, lds, fc, IC<0>{}, IC<0>{}, 0);
    for (; c < nch - NS; ++c) {
      wait_vm_lgkm0<(NS - 2) * PER_CHUNK>();
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      const int sn = st + 1 == NS ? 0 : st + 1;
      const f16* base = lds + sn * STG;
      const uint32_t sa = lds0 + st * (STG * 2);
      half(fc, IC<0>{}, base, fa, IC<0>{}, IC<DS>{}, sa);
      half(fa, IC<1>{}, base, fc, IC<DS>{}, IC<PER_CHUNK>{}, sa);
      next_chunk();
      st = sn;
    }
    for (; c < nch - 1; ++c) {
      wait_chunk<PER_CHUNK, NS - 2, true>(min(NS - 2, nch - 2 - c));
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      const int sn = st + 1 == NS ? 0 : st + 1;
      const f16* base = lds + sn * STG;
      half(fc, IC<0>{}, base, fa, IC<0>{}, IC<0>{}, 0);
      half(fa, IC<1>{}, base, fc, IC<0>{}, IC<0>{}, 0);
      st = sn;
    }
    half(fc, IC<0>{}, lds, fa, IC<0>{}, IC<0>{}, 0);  // (its reads are never used)

    if constexpr (PART) {
      static_for<0, 4 * FT>([&](auto I) {
        constexpr int ft = decltype(I)::value >> 2, g = decltype(I)::value & 3;
        const int n = n0 + (wn * FT + ft) * 32 + 8 * g + 4 * (lane >> 5);
        static_for<0, RT>([&](auto R) {
          constexpr int rt = decltype(R)::value;
          const int m = m0 + (wm * RT + rt) * 32 + (lane & 31);
          if (m < M && n < N)
            *(f32x4*)(part + (long)m * N + n) = (f32x4){acc[ft][rt][4 * g], acc[ft][rt][4 * g + 1],
                                                        acc[ft][rt][4 * g + 2], acc[ft][rt][4 * g + 3]};
        });
      });
      return;
    }
    // Epilogue.  A lane holds features 8 g + 4 (lane >> 5) .. + 3 (g < 4) of row lane & 31 of each of
    // its tiles.  The rounded sums go through LDS (the stages are free once every wave has read its last
    // fragments), so that a short loop finishes them in 16-byte pieces of consecutive features and
    // writes whole row segments.  Unrolled over the accumulators, with 8-byte stores to 32 rows per
    // instruction, the same work took about 1.1 us per 32 x 32 tile of a wave, most of it instruction
    // fetch (the code runs once per workgroup).
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
  }
};

}  // namespace ecd
