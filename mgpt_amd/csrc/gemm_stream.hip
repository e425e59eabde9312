// gemm_stream.hip -- grouped expert GEMMs whose weights are the larger
// operand: bf16 weights under few rows per expert (decode steps, short
// prompts), and fp8 weights at every row count the decode kernel does not
// take.
//
// Same contract as gemm_dma.hip (A = expert-contiguous bf16 rows [rows][K],
// B = packed weights [E][Npad][K], bf16 or e4m3 with per-output-channel
// scales; gate/up, down and SwiGLU-backward epilogues) and the same frame:
// a persistent block per CU (two of 64-row tiles) walks BM x BN tiles in an order
// that shares operand panels within an XCD, operands go HBM -> LDS by untracked
// 1 KB loads, waves of 64 features x BM/2 tokens run
// v_mfma_f32_32x32x16_bf16 on D = W . X^T.  What differs:
//  * The ring holds ST stages, each a whole 64-column slab (BM rows of A, BN
//    rows of B), ST - 1 slabs ahead.  With fp8 weights a slab is 48 KB (BM =
//    256) instead of 64 KB, so both operands lead by two slabs in 144 KB; the
//    64 x 128 tiles take 24 KB (bf16) or 16 KB (fp8) a slab and a ring of 72 or
//    80 KB, so that two blocks share a CU: one's start, epilogue and last slabs
//    are covered by the other's stream, with 96 to 128 KB of loads in flight a CU.
//    (One block with twice the ring, us of the forward: 96 experts of C = H = 512,
//    48 tokens, bf16 65 / 50 with two; 512 experts, 71 tokens, k = 6, H = 1376, fp8
//    400 / 266; the 24-token step below 64 / 61; no shape slower.)
//  * A k-step ks contracts columns 16ks .. 16ks+15 of the slab, lane half h
//    columns 16ks + 8h .. +7, as in the other bf16 products (the same sums, bit
//    for bit); the packed fp8 rows keep a lane's weights of two k-steps in one
//    16-byte LDS read (fp8_col); they become bf16 in registers (exact).  fp8 rows are 64
//    bytes: 16-byte chunk c of row r sits at slot c ^ ((r >> 2) & 3), which
//    spreads the 16 lanes served together over all banks.
//  * Scales and biases are applied after the contraction from scalar loads (a
//    vector load would wait for the ring's loads as well).
//  * Few rows take 64 x 128 tiles (4 waves): the narrower they are, the more
//    evenly a step's few tiles spread over the CUs (16 experts of H = 2816:
//    704 gate/up tiles are 2.75 rounds, 352 of 256 columns 1.4, paid as 2).
//
// Measured on MI355X, stage times, against the register-staged 32 x 256 (bf16, fp8) and
// 128 x 128 (fp8) tiles used before, gate/up + down us: bf16, C = 1024, H = 2816, E =
// 16, k = 2: 1 token 33 + 38 -> 12 + 19, 24 tokens 47 + 60 -> 34 + 26, 300 tokens 67 +
// 61 -> 36 + 28; C = 2048, H = 1408, E = 64, k = 8 (1.1 GB of weights): 64 tokens 190 +
// 107 -> 160 + 67 (4.9 TB/s), 400 tokens 305 + 196 -> 175 + 82.  fp8, the latter layer:
// 600 tokens 202 + 138 -> 117 + 64, 1999 tokens 345 + 226 -> 194 + 114 (950 TFLOP/s in
// gate/up), 4096 tokens 555 + 390 -> 343 + 216.
#include <type_traits>

#include "gemm_ring.hpp"

namespace mgpt {
namespace {

// e4m3 byte pair (low or high half of a dword) -> two bf16 in one dword.
template <bool HI>
__device__ __forceinline__ uint32_t e4m3x2_to_bf16x2(uint32_t packed) {
  typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
  const bf16x2_t v = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8((int)packed, 1.0f, HI);
  uint32_t r;
  __builtin_memcpy(&r, &v, 4);
  return r;
}

__device__ __forceinline__ bf16x8 fp8x8_to_bf16x8(uint32_t lo, uint32_t hi) {
  const uint32_t w[4] = {e4m3x2_to_bf16x2<false>(lo), e4m3x2_to_bf16x2<true>(lo),
                         e4m3x2_to_bf16x2<false>(hi), e4m3x2_to_bf16x2<true>(hi)};
  bf16x8 r;
  __builtin_memcpy(&r, w, 16);
  return r;
}

// acc = acc * scale + bias, per output feature (register v of a 32x32 tile
// holds feature 8*(v/4) + 4*lhalf + v%4 of the tile, a token per lane);
// scale null: 1, bias null: none.  An array's 32 values are requested at once (8
// at a time in the 256-row tiles, which run at the register limit).
template <typename W>
__device__ __forceinline__ void affine(f32x16 (&acc)[W::TN][W::TM], int j, const float* scale,
                                       const float* bias, int lhalf) {
  constexpr int kBatch = W::TM >= 4 ? 8 : 32;
  auto each = [&](const float* p, int f0, auto op) __attribute__((always_inline)) {
    typedef const __attribute__((address_space(4))) float* cptr;   // scalar loads
    const cptr u = (cptr)(uintptr_t)(p + f0);
    float t[kBatch];
#pragma unroll
    for (int f = 0; f < kBatch; ++f) t[f] = u[f];
#pragma unroll
    for (int f = 0; f < kBatch; ++f) {
      if (f & 4) continue;   // the other half's
      const int v = (f0 + f) / 8 * 4 + f % 4;
      const float x = lhalf ? t[f + 4] : t[f];
#pragma unroll
      for (int i = 0; i < W::TM; ++i) acc[j][i][v] = op(acc[j][i][v], x);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
#pragma unroll
  for (int f0 = 0; f0 < 32; f0 += kBatch) {
    if (scale) each(scale, f0, [](float a, float x) { return a * x; });
    if (bias) each(bias, f0, [](float a, float x) { return a + x; });
  }
}

template <int EPI, typename WT, int NW, int BM, int BN, int ST, bool kSave>
__global__ __launch_bounds__(NW * 64) void gemm_stream_kernel(
    const bf16_t* __restrict__ A, const WT* __restrict__ B, const float* __restrict__ wscale,
    const float* __restrict__ bias0, const float* __restrict__ bias1,
    const int32_t* __restrict__ counts, int E, int K, int Npad, int nbx,
    int n_store, int bias_ld, bf16_t* out, int ldo, bf16_t* save, int save_ld) {
  using W = Waves<NW, BM, BN>;
  constexpr int kTN = W::TN, kTM = W::TM;
  constexpr bool kFp8 = sizeof(WT) == 1;
  constexpr int kARow = 128, kBRow = 64 * (int)sizeof(WT);   // LDS bytes per row of a slab
  constexpr int kABytes = BM * kARow, kBBytes = BN * kBRow;
  constexpr int kStage = kABytes + kBBytes;
  constexpr int kDA = kABytes / 1024 / NW, kDB = kBBytes / 1024 / NW, kD = kDA + kDB;   // loads per wave
  constexpr int kBPer = 1024 / kBRow;                         // B rows per load
  __shared__ __attribute__((aligned(1024))) char smem[ST * kStage];

  const int G = gridDim.x;
  const int KT = K / 64;
  int e_base = 0;
  if (gridDim.y > 1) {   // a group of 64 experts per grid row
    const int g0 = (int)blockIdx.y * kMaxExperts;
    E = min(kMaxExperts, E - g0);
    e_base = g0;
    B += (size_t)g0 * Npad * K;
    if (wscale) wscale += (size_t)g0 * Npad;
    if (bias0) bias0 += (size_t)g0 * bias_ld;
    if (bias1) bias1 += (size_t)g0 * bias_ld;
  }
  SegScan<BM> sc;
  sc.init(counts, E, e_base);
  // Which tiles an XCD (own L2) takes.  256-row tiles: contiguous runs of each round,
  // which share operand panels; an eighth of a round that does not fill the grid, and
  // every other group from the other end, so that the last rounds even out.  64-row
  // tiles share little beyond the (at most four) m-tiles of a weight panel, so runs of
  // four tiles are dealt to the XCDs in turn.
  constexpr int kRun = 4;
  const int in_xcd = blockIdx.x / kNumXcd;
  int xcd = blockIdx.x % kNumXcd, t = blockIdx.x;
  if (blockIdx.y & 1) xcd = kNumXcd - 1 - xcd;
  if (BM <= 64) {
    if (G % (kRun * kNumXcd) == 0) t = (in_xcd / kRun * kNumXcd + xcd) * kRun + in_xcd % kRun;
  } else if (G % kNumXcd == 0) {
    const int items = sc.tm * nbx, run = min(G, items + kNumXcd - 1) / kNumXcd;
    t = in_xcd < run ? xcd * run + in_xcd : items;
  }
  Tile cur;
  if (!locate_tile<BN>(sc, E, nbx, t, &cur)) return;

  const int tid = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid / kWave), lane = lane_id();
  const int wn = w % W::WN, wm = w / W::WN;
  const int lrow = lane & 31, lhalf = lane >> 5;

  // Loads of a slab: wave w fills A rows w*BM/NW .. and B rows w*BN/NW ..  Lane
  // offsets from the tile's first row; A chunk c of row r at slot c ^ ((r >>
  // 1) & 7), B likewise (bf16) or c ^ ((r >> 2) & 3) of 64-byte rows (fp8).
  uint32_t a_off[kDA], b_off[kDB];
  int a_row[kDA];
#pragma unroll
  for (int i = 0; i < kDA; ++i) {
    a_row[i] = (w * kDA + i) * 8 + lane / 8;
    a_off[i] = (uint32_t)(((lane % 8) ^ ((a_row[i] >> 1) & 7)) * 16);
  }
#pragma unroll
  for (int i = 0; i < kDB; ++i) {
    const int r = (w * kDB + i) * kBPer + lane / (kBRow / 16), s = lane % (kBRow / 16);
    b_off[i] = (uint32_t)r * (uint32_t)(K * (int)sizeof(WT)) +
               (uint32_t)((kFp8 ? s ^ ((r >> 2) & 3) : s ^ ((r >> 1) & 7)) * 16);
  }
  const uint32_t lds_a = (uint32_t)(uintptr_t)(lds_char*)smem + (uint32_t)(w * kDA * 1024);
  const uint32_t lds_b = (uint32_t)(uintptr_t)(lds_char*)smem + (uint32_t)(kABytes + w * kDB * 1024);

  // Cursor over slabs (tile dtl, slab dkt, ring stage dstage).  Past the
  // end of the block's work it repeats the last slab (in bounds, into a freed
  // stage), so every slab issues the same loads and waits the same way.
  Tile dtl = cur;
  int dt = t, dkt = 0, dstage = 0;
  bool dvalid = true;
  const char *dga, *dgb;
  uint32_t ga_off[kDA];
  auto enter_item = [&]() __attribute__((always_inline)) {
    dga = reinterpret_cast<const char*>(A + (size_t)dtl.row0 * K);
    dgb = reinterpret_cast<const char*>(B + ((size_t)dtl.expert * Npad + dtl.n0) * K);
    // (few rows: those past the segment re-read its last one, in L1)
    const int rows = dtl.row_end - dtl.row0;
#pragma unroll
    for (int i = 0; i < kDA; ++i)
      ga_off[i] = a_off[i] + (uint32_t)(BM <= 64 ? min(a_row[i], rows - 1) : a_row[i]) * (uint32_t)(K * 2);
  };
  enter_item();
  const char *ua, *ub;   // the slab being issued
  uint32_t uda, udb;
  auto next_slab = [&]() __attribute__((always_inline)) {
    ua = dga + (size_t)dkt * kARow;
    ub = dgb + (size_t)dkt * kBRow;
    uda = lds_a + (uint32_t)(dstage * kStage);
    udb = lds_b + (uint32_t)(dstage * kStage);
    dstage = dstage + 1 == ST ? 0 : dstage + 1;
    if (dvalid && ++dkt == KT) {
      dt += G;
      Tile nx;
      dvalid = locate_tile<BN>(sc, E, nbx, dt, &nx);
      if (dvalid) {
        dtl = nx;
        dkt = 0;
      } else {
        --dkt;
      }
    }
  };
  int item_of_offs = t;   // the item that ga_off belongs to
  auto issue = [&](int d0, int d1) __attribute__((always_inline)) {
#pragma unroll
    for (int d = d0; d < d1; ++d) {
      if (d < kDA)
        dma16(ua + ga_off[d], uda + d * 1024);
      else
        dma16(ub + b_off[d - kDA], udb + (d - kDA) * 1024);
    }
  };
  // after the last loads of a slab: the offsets of the next one's item
  auto settle = [&]() __attribute__((always_inline)) {
    if (dvalid && dt != item_of_offs) {
      item_of_offs = dt;
      enter_item();
    }
  };
  auto quarter = [&](int q) __attribute__((always_inline)) { issue(q * kD / 4, (q + 1) * kD / 4); };
  auto slab_wait = [&]() __attribute__((always_inline)) {
    slab_barrier<(ST - 2) * kD>();
    settle();
    next_slab();
  };

  const int swz = (lrow >> 1) & 7, swz4 = (lrow >> 2) & 3;
  const char* x_base = smem + (wm * W::WTM + lrow) * kARow;
  const char* w_base = smem + kABytes + (wn * W::WTN + lrow) * kBRow;
  bf16x8 xf[2][kTM];
  bf16x8 wf[2][kFp8 ? 1 : kTN];   // bf16 weights by k-step
  uint4 wr[2][kFp8 ? kTN : 1];    // fp8 weights by pair of k-steps
  auto frags = [&](int stage, int ks) __attribute__((always_inline)) {
    const int cofs = ((2 * ks + lhalf) ^ swz) << 4;
#pragma unroll
    for (int i = 0; i < kTM; ++i)
      xf[ks & 1][i] = *reinterpret_cast<const bf16x8*>(x_base + stage * kStage + i * 32 * kARow + cofs);
    if constexpr (kFp8) {
      if ((ks & 1) == 0) {
        const int c4 = ((2 * lhalf + ks / 2) ^ swz4) << 4;
#pragma unroll
        for (int j = 0; j < kTN; ++j)
          wr[(ks >> 1) & 1][j] =
              *reinterpret_cast<const uint4*>(w_base + stage * kStage + j * 32 * kBRow + c4);
      }
    } else {
#pragma unroll
      for (int j = 0; j < kTN; ++j)
        wf[ks & 1][j] =
            *reinterpret_cast<const bf16x8*>(w_base + stage * kStage + j * 32 * kBRow + cofs);
    }
  };

#pragma unroll
  for (int s = 0; s < ST - 1; ++s) {
    settle();
    next_slab();
    issue(0, kD);
  }
  slab_wait();
  quarter(0);
  int stage = 0;
  frags(0, 0);

  for (;;) {
    Tile nxt;
    const bool have_next = locate_tile<BN>(sc, E, nbx, t + G, &nxt);
    f32x16 acc[kTN][kTM];
#pragma unroll
    for (int j = 0; j < kTN; ++j)
#pragma unroll
      for (int i = 0; i < kTM; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[j][i][v] = 0.0f;

    // the k loop for MT live 32-token sub-tiles of this wave (as gemm_dma's)
    auto kloop = [&](auto mt_c) __attribute__((always_inline)) {
      constexpr int MT = decltype(mt_c)::value;
      constexpr int kMfma = kTN * MT;
      for (int kt = 0; kt < KT; ++kt) {
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
          if (ks < 3) {
            quarter(ks + 1);
            frags(stage, ks + 1);
          } else {
            stage = stage + 1 == ST ? 0 : stage + 1;
            slab_wait();
            quarter(0);
            frags(stage, 0);
          }
#pragma unroll
          for (int j = 0; j < kTN; ++j) {
            if constexpr (MT > 0) {
              bf16x8 wv;
              if constexpr (kFp8) {
                const uint4 r = wr[(ks >> 1) & 1][j];
                wv = (ks & 1) ? fp8x8_to_bf16x8(r.z, r.w) : fp8x8_to_bf16x8(r.x, r.y);
              } else {
                wv = wf[ks & 1][j];
              }
#pragma unroll
              for (int i = 0; i < MT; ++i)
                acc[j][i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wv, xf[ks & 1][i], acc[j][i], 0, 0, 0);
            }
          }
          constexpr int kReads = kTM + (kFp8 ? (1) : kTN);
          constexpr int kPairs = kReads < kMfma ? kReads : kMfma;
#pragma unroll
          for (int q = 0; q < kPairs; ++q) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);   // one MFMA
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);   // one LDS read
          }
        }
      }
    };
    const int wrows = cur.row_end - (cur.row0 + wm * W::WTM);
    const int mt_live = wrows <= 0 ? 0 : min(kTM, (wrows + 31) / 32);
    if constexpr (kTM == 4) {
      switch (mt_live) {
        case 0: kloop(IntC<0>{}); break;
        case 1: kloop(IntC<1>{}); break;
        case 2: kloop(IntC<2>{}); break;
        case 3: kloop(IntC<3>{}); break;
        default: kloop(IntC<4>{}); break;
      }
    } else if constexpr (kTM == 2) {
      if (mt_live == 0) kloop(IntC<0>{});
      else if (mt_live == 1) kloop(IntC<1>{});
      else kloop(IntC<2>{});
    } else {
      if (mt_live == 0) kloop(IntC<0>{});
      else kloop(IntC<1>{});
    }
    if (mt_live > 0) {
      // the lane recomputed rather than kept live across the k loop (the 256-
      // row tiles run at the register limit)
      int lane_now;
      asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(lane_now));
      const int lrow = lane_now & 31, lhalf = lane_now >> 5;
      const size_t e = cur.expert;
      const int nw = cur.n0 + wn * W::WTN;
      if constexpr (EPI == kEpiGateUp) {
        const int hb = nw / 2;   // [32 gate | 32 up] of units hb .. hb+31
        affine<W>(acc, 0, kFp8 ? wscale + e * Npad + nw : nullptr, bias0 + e * bias_ld + hb, lhalf);
        affine<W>(acc, 1, kFp8 ? wscale + e * Npad + nw + 32 : nullptr, bias1 + e * bias_ld + hb, lhalf);
      } else if constexpr (EPI == kEpiDown) {
#pragma unroll
        for (int j = 0; j < kTN; ++j)
          if (kFp8 || bias0)
            affine<W>(acc, j, kFp8 ? wscale + e * Npad + nw + 32 * j : nullptr,
                      bias0 ? bias0 + e * bias_ld + nw + 32 * j : nullptr, lhalf);
      }
      store_tile<EPI, W, kSave, true>(acc, cur, wn, wm, lrow, lhalf, n_store, out, ldo, save, save_ld);
    }
    if (!have_next) break;
    t += G;
    cur = nxt;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the repeated tail loads
}

}  // namespace

// Persistent launch, one block per CU (two of the small tiles).  Tiles of 64 rows x 128 features
// (small) or 256 x 256.  save: the training pre-activations (gate/up: written;
// SwiGLU backward: read, bf16 weights only).  K % 64 == 0, Npad % 256 == 0,
// n_store % 64 == 0; A has 256 rows of slack.
template <int EPI, typename WT>
hipError_t launch_gemm_stream(const bf16_t* A, const WT* B, const float* wscale, const float* bias0,
                              const float* bias1, const int32_t* counts, int E, int K, int Npad,
                              int n_store, int bias_ld, bf16_t* out, int ldo, size_t rows, bool small,
                              int num_cus, bf16_t* save, int save_ld, hipStream_t stream) {
  constexpr bool kFp8 = sizeof(WT) == 1;
  if (rows == 0) return hipSuccess;
  if (E <= 0 || E > kMaxExpertsWide || K % 64 || Npad % 256 || n_store % 64 || num_cus <= 0 ||
      ldo % 8 || (reinterpret_cast<uintptr_t>(out) & 15) ||
      (save && (save_ld % 8 || (reinterpret_cast<uintptr_t>(save) & 15))) ||
      (EPI == kEpiSwigluBwd && !save) || (kFp8 && (save || !wscale)))
    return hipErrorInvalidValue;
  const int BM = small ? 64 : 256, BN = small ? 128 : 256;
  const int nt = EPI == kEpiGateUp ? Npad / BN : (n_store + BN - 1) / BN;
  // More than 64 experts: one launch, a group of 64 per grid row (as in
  // gemm_dma.hip; us of gate/up + down, E = 128, C = 512, H = 256, 16 rows an expert 16 +
  // 11, E = 256, C = 512, H = 512, 24 rows 63 + 34; with a launch a group and one block a
  // CU 28 + 22 and 91 + 57).
  const int groups = (E + kMaxExperts - 1) / kMaxExperts;
  // at most this many tiles (an expert with rows has one more than its whole
  // ones at most)
  const long tiles = ((long)(rows / BM) + (long)std::min<size_t>(std::min(E, kMaxExperts), rows)) * nt;
  const int grid = (int)std::min<long>((tiles + 31) / 32 * 32, small ? 2 * num_cus : num_cus);
  auto launch = [&](auto kernel, int threads) {
    hipLaunchKernelGGL(kernel, dim3(grid, groups), dim3(threads), 0, stream, A, B, wscale, bias0, bias1,
                       counts, E, K, Npad, nt, n_store, bias_ld, out, ldo, save, save_ld);
  };
  if constexpr (kFp8) {
    if (small)
      launch(gemm_stream_kernel<EPI, fp8_t, 4, 64, 128, 5, false>, 256);
    else
      launch(gemm_stream_kernel<EPI, fp8_t, 8, 256, 256, 3, false>, 512);
  } else {
    if (!small) return hipErrorInvalidValue;   // gemm_dma.hip's
    if constexpr (EPI == kEpiGateUp) {
      if (save)
        launch(gemm_stream_kernel<EPI, bf16_t, 4, 64, 128, 3, true>, 256);
      else
        launch(gemm_stream_kernel<EPI, bf16_t, 4, 64, 128, 3, false>, 256);
    } else {
      launch(gemm_stream_kernel<EPI, bf16_t, 4, 64, 128, 3, false>, 256);
    }
  }
  return hipGetLastError();
}

#define MGPT_INST_STREAM(EPI, WT)                                                                   \
  template hipError_t launch_gemm_stream<EPI, WT>(                                                  \
      const bf16_t*, const WT*, const float*, const float*, const float*, const int32_t*, int, int, \
      int, int, int, bf16_t*, int, size_t, bool, int, bf16_t*, int, hipStream_t);
MGPT_INST_STREAM(kEpiGateUp, bf16_t)
MGPT_INST_STREAM(kEpiDown, bf16_t)
MGPT_INST_STREAM(kEpiSwigluBwd, bf16_t)
MGPT_INST_STREAM(kEpiGateUp, fp8_t)
MGPT_INST_STREAM(kEpiDown, fp8_t)

}  // namespace mgpt
