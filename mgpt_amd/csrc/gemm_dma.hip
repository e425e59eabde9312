// gemm_dma.hip -- bf16 grouped expert GEMMs, direct-to-LDS pipeline.
//
// Same contract as gemm.hip's grouped_gemm_kernel for the bf16 x bf16 case
// (A = expert-contiguous activations [rows][K], B = packed weights
// [E][Npad][K], K contiguous; gate/up epilogue with SwiGLU or down epilogue
// with bias), built for the large prefill-shaped segments that dominate the
// MoE layer's time.
//
// CDNA4 design (choices measured on MI355X):
//  * Persistent: one 512-thread block per CU walks the 256 x 256 output
//    tiles; the blocks of one XCD take consecutive tiles of an order that
//    groups 4 token blocks x all feature blocks, so they share operand
//    panels in their XCD's L2.  Tile lookup is a per-wave register scan of
//    the expert counts (no LDS, no barrier).
//  * 8 waves (2 per SIMD) each own 64 output features x 128 tokens: 2 x 4
//    tiles of v_mfma_f32_32x32x16_bf16.  Issue is in order within a wave, so
//    one wave's MFMAs cover the other's LDS and barrier waits.
//  * The MFMA computes D = W . X^T (weights as the row operand), so each
//    lane holds 4 consecutive output features of one token: the epilogue
//    writes 8-byte vectors.
//  * Operands move HBM -> LDS with global_load_lds_dwordx4 (1 KB per wave
//    instruction; no staging registers, no ds_write) into a ring of five
//    32 KB units (activations or weights of a 64-column slab) that runs
//    across tile boundaries.  The loads are inline asm the compiler does not
//    track, with explicit vmcnt waits: for the builtin it inserts vmcnt(0)
//    before LDS reads, which serialises the ring.
//  * Fragments are read one k-step ahead of the MFMAs, interleaved with
//    them (sched_group_barrier), across slab boundaries.
//  * LDS rows are 128 B (64 bf16); K-chunk c of row r sits at slot
//    c ^ ((r >> 1) & 7): gfx950's LDS has 64 banks, so the 16 lanes served
//    together (16 rows of one logical chunk) hit 16 distinct bank groups.
//  * SwiGLU in the epilogue uses the hardware exp/reciprocal (well inside
//    the bf16 tolerance).
#include <type_traits>

#include "gemm_ring.hpp"

namespace mgpt {
namespace {

constexpr int kBN = 256;   // features per tile

// The accumulators of a work item start from the biases of its features
// (the same for every token), or from zero for split-K parts (the reduce
// kernel adds the bias), the SwiGLU backward and a down product without
// bias.  Register v of a 32x32 tile holds feature 8*(v/4) + 4*(lane/32) +
// v%4.  The biases are read at wave-uniform addresses (scalar loads): a
// vector load would make the compiler wait for the ring's DMA loads, which
// it does not track, as well.
template <int EPI, int NW>
__device__ __forceinline__ void init_acc(f32x16 (&acc)[Waves<NW>::TN][Waves<NW>::TM],
                                         const Work& wk, int wn, int lhalf,
                                         const float* __restrict__ bias0,
                                         const float* __restrict__ bias1, int bias_ld) {
  using W = Waves<NW>;
  const bool has_bias = EPI != kEpiSwigluBwd && wk.sidx < 0 && bias0 != nullptr;
#pragma unroll
  for (int j = 0; j < W::TN; ++j) {
    f32x16 b;
    if (has_bias) {
      const float* src;
      if constexpr (EPI == kEpiGateUp) {
        // packed rows: each 64 of them are [32 gate | 32 up] of hidden units hb..hb+31
        const int hb = (wk.tile.n0 + wn * W::WTN) / 2 + 32 * (j / 2);
        src = ((j & 1) ? bias1 : bias0) + (size_t)wk.tile.expert * bias_ld + hb;
      } else {
        src = bias0 + (size_t)wk.tile.expert * bias_ld + wk.tile.n0 + wn * W::WTN + 32 * j;
      }
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const float4 v = *reinterpret_cast<const float4*>(src + 8 * g + 4 * lhalf);
        b[4 * g] = v.x;
        b[4 * g + 1] = v.y;
        b[4 * g + 2] = v.z;
        b[4 * g + 3] = v.w;
      }
    } else {
#pragma unroll
      for (int v = 0; v < 16; ++v) b[v] = 0.0f;
    }
    // The wait for these loads happens here, at the item's start: past this
    // point the values count as computed, so sub-tiles that no MFMA
    // touches (MT < 4) do not make the epilogue wait for the loads and,
    // with them, for the ring's DMA.
    if constexpr (EPI != kEpiSwigluBwd) asm volatile("" : "+v"(b));
#pragma unroll
    for (int i = 0; i < W::TM; ++i) acc[j][i] = b;
    // one feature group at a time: keeps the scheduler from hoisting all
    // TN * 32 scalar loads together (SGPR pressure)
    __builtin_amdgcn_sched_barrier(0);
  }
}

constexpr int kPartialFloats = 256 * 256;   // of one split work item

// ---------------------------------------------------------------------------
// Split ring.  LDS holds 5 units of 32 KB, a unit being the 256 activation
// rows or the 256 weight rows of one 64-column slab (128-byte rows, as in
// the whole design).  Units are loaded in the order A0 B0 A1 B1 ...; slab s
// reads units 2s and 2s+1, and barrier B_s frees the two units of slab s-1
// and refills them with units 2s+3 (weights of slab s+1) and 2s+4
// (activations of slab s+2): the activations are requested two slabs ahead
// and the weights one (a 2-stage ring of 64 KB slabs manages one for both).
// More than 64 experts: `group` of them (at most 64) per grid row; kTurn: every other
// row takes its tiles from the other end, so that the rows' last rounds even out over
// the XCDs (an instance of its own: the kernel runs at the register limit, and the
// turn cost launches of one row 1%).
template <int EPI, int NW, bool kSave, bool kTurn>
__global__ __launch_bounds__(NW * 64) void gemm_ring5_kernel(
    const bf16_t* __restrict__ A, const bf16_t* __restrict__ B, const float* __restrict__ bias0,
    const float* __restrict__ bias1, const int32_t* __restrict__ counts, int E, int group, int K,
    int Npad, int n_store, int bias_ld, bf16_t* out, int ldo, float* __restrict__ partials,
    bf16_t* save, int save_ld) {
  using W = Waves<NW>;
  constexpr int kTN = W::TN, kTM = W::TM;
  constexpr int kUnits = 5;
  constexpr int kRowBytes = 128;
  constexpr int kUnit = 256 * kRowBytes;           // 32 KB
  constexpr int kDmaPerWave = kUnit / 1024 / NW;   // 1 KB loads per wave and unit
  constexpr int kWaveRows = 256 / NW;              // unit rows each wave loads
  __shared__ __attribute__((aligned(1024))) char smem[kUnits * kUnit];

  const int nbx = Npad / kBN;
  const int G = gridDim.x;
  const int KT = K / 64;
  int e_base = 0;
  if (gridDim.y > 1) {
    const int g0 = (int)blockIdx.y * group;
    E = min(group, E - g0);
    e_base = g0;
    B += (size_t)g0 * Npad * K;
    if (bias0) bias0 += (size_t)g0 * bias_ld;
    if (bias1) bias1 += (size_t)g0 * bias_ld;
  }
  SegScan<256> sc;
  sc.init(counts, E, e_base);
  SplitPlan plan;
  plan.init(sc.tm * nbx, G, KT, partials != nullptr);
  int t = (G % kNumXcd == 0) ? (blockIdx.x % kNumXcd) * (G / kNumXcd) + blockIdx.x / kNumXcd
                             : blockIdx.x;
  if (kTurn && (blockIdx.y & 1)) t = G - 1 - t;
  // (a down product that does not fill the grid: an eighth of its items per XCD)
  if (EPI == kEpiDown && plan.items < G && G % kNumXcd == 0) {
    const int run = (plan.items + kNumXcd - 1) / kNumXcd, in_xcd = (int)blockIdx.x / kNumXcd;
    t = in_xcd < run ? (int)(blockIdx.x % kNumXcd) * run + in_xcd : plan.items;
  }
  Work cur;
  if (!locate_work(sc, plan, E, nbx, KT, t, &cur)) return;

  const int tid = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid / kWave), lane = lane_id();
  const int wn = w % W::WN, wm = w / W::WN;
  const int lrow = lane & 31, lhalf = lane >> 5;
  const size_t row_bytes_g = (size_t)K * 2;

  // DMA of a unit: wave w fills its kWaveRows rows in blocks of 8 rows;
  // lane l covers row r = 8i + l/8, slot l%8 = chunk ^ ((r >> 1) & 7)
  // (kWaveRows is a multiple of 16, so the slot depends on i & 1 only).
  uint32_t lane_off[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = i * 8 + lane / 8;
    lane_off[i] = (uint32_t)(lane / 8) * (uint32_t)row_bytes_g +
                  (uint32_t)((((lane % 8) ^ ((r >> 1) & 7))) * 16);
  }
  const uint32_t lds_base = (uint32_t)(uintptr_t)(lds_char*)smem + (uint32_t)(w * kDmaPerWave * 1024);
  auto abase = [&](const Tile& tl) -> const char* {
    return reinterpret_cast<const char*>(A + ((size_t)tl.row0 + kWaveRows * w) * K);
  };
  auto bbase = [&](const Tile& tl) -> const char* {
    return reinterpret_cast<const char*>(B + ((size_t)tl.expert * Npad + tl.n0 + kWaveRows * w) * K);
  };

  // Cursor over units: (work item dwk, slab dkt, operand dop), ring slot
  // dslot.
  Work dwk = cur;
  int dt = t, dkt = cur.k0, dop = 0, dslot = 0;
  bool dvalid = true;
  const char* dga = abase(cur.tile);
  const char* dgb = bbase(cur.tile);
  const char* dlast = dga;
  // Source and ring slot of the next unit.  Past the end of the block's
  // work it repeats the last real unit (in bounds, into a freed slot), so
  // every slab issues the same loads and waits the same way.
  auto next_unit = [&](const char*& g, uint32_t& dst) __attribute__((always_inline)) {
    if (dvalid) dlast = (dop ? dgb : dga) + (size_t)dkt * kRowBytes;
    g = dlast;
    dst = lds_base + (uint32_t)(dslot * kUnit);
    dslot = dslot + 1 == kUnits ? 0 : dslot + 1;
    if (dop == 0) {
      dop = 1;
    } else {
      dop = 0;
      if (dvalid && ++dkt == dwk.k1) {
        dt += G;
        dvalid = locate_work(sc, plan, E, nbx, KT, dt, &dwk);
        if (dvalid) {
          dkt = dwk.k0;
          dga = abase(dwk.tile);
          dgb = bbase(dwk.tile);
        }
      }
    }
  };
  auto dma_loads = [&](const char* g, uint32_t dst, int i0, int n) __attribute__((always_inline)) {
#pragma unroll
    for (int i = i0; i < i0 + n; ++i)
      dma16(g + (size_t)(i * 8) * row_bytes_g + lane_off[i & 1], dst + i * 1024);
  };
  // The two units refilled after barrier B_s (weights of slab s+1, then
  // activations of slab s+2, into the slots of slab s-1) are issued a
  // quarter at a time in the four MFMA segments that follow, so that the
  // loads queue behind MFMAs instead of 64 of them reaching the load unit
  // together at the barrier.  B_s waits for units 2s and 2s+1 with the four
  // loads of unit 2s+2 still allowed in flight.
  const char* ug[2];
  uint32_t ud[2];
  auto quarter = [&](int q) __attribute__((always_inline)) {
    dma_loads(ug[q >> 1], ud[q >> 1], (q & 1) * (kDmaPerWave / 2), kDmaPerWave / 2);
  };
  auto slab_wait = [&]() __attribute__((always_inline)) {
    slab_barrier<kDmaPerWave>();
    next_unit(ug[0], ud[0]);
    next_unit(ug[1], ud[1]);
  };

  const int x_row = (wm * W::WTM + lrow) * kRowBytes;
  const int w_row = (wn * W::WTN + lrow) * kRowBytes;
  const int swz = (lrow >> 1) & 7;
  bf16x8 xf[2][kTM], wf[2][kTN];
  // k-step ks of the slab whose activation unit is in ring slot `aslot`
  // (its weight unit follows in the next slot)
  auto frags = [&](int aslot, int ks, bf16x8 (&xs)[kTM], bf16x8 (&ws)[kTN])
      __attribute__((always_inline)) {
    const int bslot = aslot + 1 == kUnits ? 0 : aslot + 1;
    const char* sa = smem + aslot * kUnit + x_row;
    const char* sb = smem + bslot * kUnit + w_row;
    const int cofs = (((ks * 2 + lhalf) ^ swz) << 4);
#pragma unroll
    for (int i = 0; i < kTM; ++i)
      xs[i] = *reinterpret_cast<const bf16x8*>(sa + i * 32 * kRowBytes + cofs);
#pragma unroll
    for (int j = 0; j < kTN; ++j)
      ws[j] = *reinterpret_cast<const bf16x8*>(sb + j * 32 * kRowBytes + cofs);
  };

  // Prologue: units 0, 1, 2 (A0 B0 A1), then B_0 and the first quarter.
  for (int u = 0; u < 3; ++u) {
    const char* g;
    uint32_t dst;
    next_unit(g, dst);
    dma_loads(g, dst, 0, kDmaPerWave);
  }
  slab_wait();
  quarter(0);
  frags(0, 0, xf[0], wf[0]);
  int aslot = 0;

  for (;;) {
    Work nxt;
    const bool have_next = locate_work(sc, plan, E, nbx, KT, t + G, &nxt);
    f32x16 acc[kTN][kTM];
    init_acc<EPI, NW>(acc, cur, wn, lhalf, bias0, bias1, bias_ld);

    // The k loop for MT live 32-token sub-tiles of this wave (the rest of
    // its 128 tokens lie past the segment: their MFMAs would only multiply
    // padding rows, which costs time and, the chip being power-limited,
    // clock).  Loads, fragment reads and barriers are the same for all MT.
    auto kloop = [&](auto mt_c) __attribute__((always_inline)) {
      constexpr int MT = decltype(mt_c)::value;
      constexpr int kReads = kTM + kTN, kMfma = kTN * MT;
      constexpr int kPairs = kReads < kMfma ? kReads : kMfma;
      for (int kt = cur.k0; kt < cur.k1; ++kt) {
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
          if (ks + 1 < 4) {
            quarter(ks + 1);
            frags(aslot, ks + 1, xf[(ks + 1) & 1], wf[(ks + 1) & 1]);
          } else {
            // next slab; after the block's last slab this reads stale units
            // whose values are never used (one code path keeps the
            // compiler's LDS wait counting exact)
            aslot += 2;
            if (aslot >= kUnits) aslot -= kUnits;
            slab_wait();
            quarter(0);
            frags(aslot, 0, xf[0], wf[0]);
          }
#pragma unroll
          for (int j = 0; j < kTN; ++j)
#pragma unroll
            for (int i = 0; i < MT; ++i)
              acc[j][i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[ks & 1][j], xf[ks & 1][i],
                                                                  acc[j][i], 0, 0, 0);
#pragma unroll
          for (int q = 0; q < kPairs; ++q) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);   // one MFMA
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);   // one LDS read
          }
          if constexpr (kMfma > kPairs) __builtin_amdgcn_sched_group_barrier(0x008, kMfma - kPairs, 0);
          if constexpr (kReads > kPairs) __builtin_amdgcn_sched_group_barrier(0x100, kReads - kPairs, 0);
        }
      }
    };
    const int wrows = cur.tile.row_end - (cur.tile.row0 + wm * W::WTM);
    const int mt_live = wrows <= 0 ? 0 : min(kTM, (wrows + 31) / 32);
    static_assert(kTM == 4, "sub-tile dispatch below");
    switch (mt_live) {
      case 0: kloop(IntC<0>{}); break;
      case 1: kloop(IntC<1>{}); break;
      case 2: kloop(IntC<2>{}); break;
      case 3: kloop(IntC<3>{}); break;
      default: kloop(IntC<4>{}); break;
    }
    mfma_drain<W>();
    if (cur.sidx < 0) {
      // The lane's row and half recomputed here rather than kept live from
      // the start: the kernel runs at the register limit, and a value held
      // across the k loop gets spilled (its reload then waits for the
      // ring's DMA loads as well).
      int lane_now;
      asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0"
                   : "=v"(lane_now));
      store_tile<EPI, W, kSave>(acc, cur.tile, wn, wm, lane_now & 31, lane_now >> 5, n_store,
                                 out, ldo, save, save_ld);
    } else {
      float4* P = reinterpret_cast<float4*>(partials + (size_t)cur.sidx * kPartialFloats) + tid;
#pragma unroll
      for (int j = 0; j < kTN; ++j) {
#pragma unroll
        for (int i = 0; i < kTM; ++i) {
          const f32x16 a = acc_fetch<W>(acc[j][i]);
#pragma unroll
          for (int v4 = 0; v4 < 4; ++v4)
            P[((j * kTM + i) * 4 + v4) * W::kThreads] =
                make_float4(a[4 * v4], a[4 * v4 + 1], a[4 * v4 + 2], a[4 * v4 + 3]);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if (!have_next) break;
    t += G;
    cur = nxt;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the repeated tail loads
}


#ifndef MGPT_RING_WAVES
#define MGPT_RING_WAVES 8
#endif
constexpr int kRingWaves = MGPT_RING_WAVES;

}  // namespace

// Persistent launch: one block per CU (the kernel walks the tiles itself).
// max_mtiles bounds sum_e ceil(count_e / 256); it only caps the grid.
// partials (num_cus * kPartialFloats floats, or null to disable) holds the
// split last round; the reduce kernel that follows exits at once when the
// counts leave nothing to split.  save (gate/up only, and only without
// partials) also stores the pre-activations g + b_g, u + b_u as bf16 in the
// packed column order, save[row][n] with leading dimension save_ld.
// SWIGLU_BWD (no partials) reads those pre-activations from save and writes
// d(gate), d(up) to out in the same layout (out may equal save).  DOWN
// adds no bias when bias0 is null.  Measured on MI355X (cfg3 shapes, skewed
// counts): the split 5-unit ring (gate/up 1035, down 871 TFLOP/s) beats a
// 2-slab ring of 64 KB slabs (1034, 827) and 32-column slabs (4 x 32: 938,
// 724; 5 x 32 with 2 per barrier: 970, 786), whose 64-byte row segments
// double the DMA cost; a ping-pong schedule of the two waves of a SIMD
// (934) and weights loaded straight into registers in fragment order (990)
// did not help either.
template <int EPI>
hipError_t launch_gemm_dma(const bf16_t* A, const bf16_t* B, const float* bias0,
                           const float* bias1, const int32_t* counts, int E, int K, int Npad,
                           int n_store, int bias_ld, bf16_t* out, int ldo, int max_mtiles,
                           float* partials, int num_cus, bf16_t* save, int save_ld,
                           hipStream_t stream) {
  if (max_mtiles <= 0) return hipSuccess;
  if (E <= 0 || E > kMaxExpertsWide) return hipErrorInvalidValue;
  // 16-byte output vectors: ldo and the output base must keep 8-element alignment
  if (K % 64 != 0 || Npad % kBN != 0 || n_store % 64 != 0 || num_cus <= 0 || ldo % 8 != 0 ||
      (reinterpret_cast<uintptr_t>(out) & 15) != 0)
    return hipErrorInvalidValue;
  if (save && (EPI == kEpiDown || partials || save_ld % 8 != 0 ||
               (reinterpret_cast<uintptr_t>(save) & 15) != 0))
    return hipErrorInvalidValue;
  if (EPI == kEpiSwigluBwd && !save) return hipErrorInvalidValue;
  // the accumulators start from the biases, read as 16-byte vectors
  if (((reinterpret_cast<uintptr_t>(bias0) | reinterpret_cast<uintptr_t>(bias1)) & 15) != 0 ||
      bias_ld % 4 != 0)
    return hipErrorInvalidValue;
  if (K / 64 < kMinSplitSlabs) partials = nullptr;   // no split, no reduce launch
  const int tiles = max_mtiles * (Npad / kBN);
  // More than 64 experts: equal groups of up to 64, the weights and biases from the
  // group's first expert on; the rows come in expert order, so each group's follow the
  // earlier groups'.  One launch takes all groups as rows of its grid, so that
  // the CUs that a group's last round leaves idle go on with the next group;
  // that round is then not split (us of gate/up + down on MI355X with a launch
  // and a split reduction per group, so, and every other group turned: E = 128, C =
  // 1024, H = 704, 511 rows an expert 238 + 163, 235 + 158, 237 + 137; E = 256, C = 768, H =
  // 512, 200 rows 192 + 107 -> 151 + 94).
  const int groups = (E + kMaxExperts - 1) / kMaxExperts;
  if (groups > 1) partials = nullptr;
  // (with split tiles every CU has work, also where there are fewer tiles)
  const int grid = partials || tiles >= num_cus ? num_cus : tiles;
  // the gate/up epilogue's pre-activation stores are compiled only into
  // the training instance (fewer live registers in the inference one)
  auto launch = [&](auto save_c) {
    auto go = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3(grid, groups), dim3(kRingWaves * kWave), 0, stream, A, B, bias0,
                         bias1, counts, E, (E + groups - 1) / groups, K, Npad, n_store, bias_ld, out, ldo,
                         partials, save, save_ld);
    };
    if (groups > 1)
      go(gemm_ring5_kernel<EPI, kRingWaves, decltype(save_c)::value, true>);
    else
      go(gemm_ring5_kernel<EPI, kRingWaves, decltype(save_c)::value, false>);
  };
  if constexpr (EPI == kEpiGateUp) {
    if (save)
      launch(std::true_type{});
    else
      launch(std::false_type{});
  } else {
    launch(std::false_type{});
  }
  if constexpr (EPI != kEpiSwigluBwd) {
    if (partials)
      hipLaunchKernelGGL((gemm_split_reduce_kernel<EPI, Waves<kRingWaves>>), dim3(8 * grid),
                         dim3(256), 0, stream, partials, bias0, bias1, counts, E, 0, K, Npad / kBN,
                         n_store, bias_ld, out, ldo, grid);
  }
  return hipGetLastError();
}

template hipError_t launch_gemm_dma<kEpiGateUp>(const bf16_t*, const bf16_t*, const float*,
                                                const float*, const int32_t*, int, int, int, int,
                                                int, bf16_t*, int, int, float*, int, bf16_t*, int,
                                                hipStream_t);
template hipError_t launch_gemm_dma<kEpiDown>(const bf16_t*, const bf16_t*, const float*,
                                              const float*, const int32_t*, int, int, int, int,
                                              int, bf16_t*, int, int, float*, int, bf16_t*, int,
                                              hipStream_t);
template hipError_t launch_gemm_dma<kEpiSwigluBwd>(const bf16_t*, const bf16_t*, const float*,
                                                   const float*, const int32_t*, int, int, int,
                                                   int, int, bf16_t*, int, int, float*, int,
                                                   bf16_t*, int, hipStream_t);

}  // namespace mgpt
