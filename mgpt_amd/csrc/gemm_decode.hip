// gemm_decode.hip -- fp8-weight grouped expert GEMMs for decode shapes.
//
// Few tokens per expert (a decode step: N = 64 tokens, k = 8, E = 64 gives
// about 8 rows per expert) make the expert GEMMs a weight stream: every
// weight byte is used by at most 32 rows, so the bound is HBM bandwidth,
// not MFMA.  This kernel is built for that bound:
//  * Work items are (expert m-tile of <= 32 rows, 64, 128 or 256 output features);
//    two persistent blocks per CU (one of 256 features) walk them, so that one
//    block's start, epilogue and waits are covered by the other's stream, each
//    with a direct-to-LDS ring across item boundaries (a stage: the item's weight
//    rows x 128 fp8 columns and 32 activation rows x 128 columns).  The loads are inline asm the
//    compiler does not track, with explicit waits (as in gemm_dma.hip); a lane's
//    addresses are formed once an item and stepped by additions.
//  * Each wave owns 64 features (a [32 gate | 32 up] pair for gate/up) x the 32
//    token rows: two v_mfma_f32_32x32x16_bf16 per 16 columns, the fp8 weights
//    converted to bf16 in registers (exact: every e4m3 value is a bf16 value);
//    the per-output-channel scale is applied in the epilogue.  A stage's LDS
//    reads are all issued before its first MFMA.  Few tokens are bound by this
//    chain (launch, routing, then a stage's reads, conversions and barrier), not
//    by HBM; address arithmetic and reads waited for one by one had made a stage
//    0.85 us where the weights take 0.4 (E = 64, C = 2048, H = 1408, 1 token:
//    gate/up 22.2 -> 16.6 us, down 15.1 -> 10.8; 64 tokens, HBM-bound at 5.5
//    TB/s: 69.8 -> 66.8, 37.4 -> 36.0).
//  * K order within a stage: lane half h holds k = 64h + 8*ks + e for k-step
//    ks (element e) in both operands, so a lane's weights for the stage are
//    64 contiguous bytes of its row (four 16-byte LDS reads).
// Same contract as gemm.hip's grouped_gemm_kernel (A = expert-contiguous
// activations [rows][K], B = fp8 weights in stage tiles
// [E][Npad/256][K/128][256][128] (pack.hip: tile_fp8_kernel) with scales
// [E][Npad], SwiGLU or bias epilogue).
#include <algorithm>
#include <cmath>

#include "common.hpp"

namespace mgpt {
namespace {

constexpr int kDBM = 32;                     // token rows per item
constexpr int kDBK = 128;                    // columns per stage
constexpr int kTileN = 256;                  // features per tile of the weights' layout
constexpr int blocks_per_cu(int nw) { return nw == 4 ? 1 : 2; }   // nw waves a block
constexpr int kDmaW = 64 * kDBK / 1024;      // 8 weight blocks per wave (64 features) and stage

typedef __attribute__((address_space(3))) char lds_char;

__device__ __forceinline__ void dma16(const void* g, uint32_t lds) {
  asm volatile("global_load_lds_dwordx4 %0, off" ::"v"(g), "{m0}"(lds) : "memory");
}
// The same for the weight stream, with the non-temporal hint: every weight
// byte is read once per step, and a decode step's weights (hundreds of MB)
// would otherwise push the activations, the router's operands and the
// combine's rows out of the caches.  Measured at cfg5 (graph-replayed
// steps): gate/up 74.1 -> 64.7 us, down 39.7 -> 35.6 us.
__device__ __forceinline__ void dma16_stream(const void* g, uint32_t lds) {
  asm volatile("global_load_lds_dwordx4 %0, off nt" ::"v"(g), "{m0}"(lds) : "memory");
}

template <int N>
__device__ __forceinline__ void stage_barrier() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

__device__ __forceinline__ float uniform_load(const float* p) {
  return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(*p)));
}

// e4m3 byte pair (low or high half of a dword) -> two bf16 in one dword.
template <bool HI>
__device__ __forceinline__ uint32_t e4m3x2_to_bf16x2(uint32_t packed) {
  typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
  bf16x2_t v = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8((int)packed, 1.0f, HI);
  uint32_t r;
  __builtin_memcpy(&r, &v, 4);
  return r;
}

// 8 fp8 weights (two dwords) -> a bf16x8 MFMA operand.
__device__ __forceinline__ bf16x8 fp8x8_to_bf16x8(uint32_t lo, uint32_t hi) {
  const uint32_t w[4] = {e4m3x2_to_bf16x2<false>(lo), e4m3x2_to_bf16x2<true>(lo),
                         e4m3x2_to_bf16x2<false>(hi), e4m3x2_to_bf16x2<true>(hi)};
  bf16x8 r;
  __builtin_memcpy(&r, w, 16);
  return r;
}

__device__ __forceinline__ float silu_mul_fast(float g, float u) {
  return g * u * __builtin_amdgcn_rcpf(1.0f + __expf(-g));
}

__device__ __forceinline__ uint2 pack4_bf16(float a, float b, float c, float d) {
  typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
  bf16x2_t lo = {(__bf16)a, (__bf16)b}, hi = {(__bf16)c, (__bf16)d};
  uint2 r;
  __builtin_memcpy(&r.x, &lo, 4);
  __builtin_memcpy(&r.y, &hi, 4);
  return r;
}

struct DItem {
  int expert, row0, row_end, n0;
};

// Per-wave register scan of the expert counts in 32-row m-tiles (lane e =
// expert e, E <= 64): items are m-tiles x feature blocks, feature-major
// within an m-tile.
struct DScan {
  int cnt, rows_incl, tiles_incl, tiles_excl, tm;
  __device__ __forceinline__ void init(const int32_t* counts, int E) {   // global or LDS
    const int l = lane_id();
    cnt = (l < E) ? counts[l] : 0;
    const int tiles = (cnt + kDBM - 1) / kDBM;
    rows_incl = wave_incl_scan(cnt);
    tiles_incl = wave_incl_scan(tiles);
    tiles_excl = tiles_incl - tiles;
    tm = __builtin_amdgcn_readlane(tiles_incl, kWave - 1);
  }
  __device__ __forceinline__ bool locate(int E, int nbx, int bn, int v, DItem* out) const {
    if (v >= tm * nbx) return false;
    const int mt = v / nbx;
    const int l = lane_id();
    const bool mine = (l < E) && (mt >= tiles_excl) && (mt < tiles_incl);
    const unsigned long long m = __ballot(mine);
    const int owner = __builtin_amdgcn_readfirstlane(__ffsll((long long)m) - 1);
    out->expert = owner;
    // The expert's T x nbx items in runs of eight feature blocks, row tiles next: the
    // hardware deals blocks round-robin to the eight XCDs (each with its own L2), so
    // the T items that read the same weights run on one XCD at about the same time.
    const int T = __builtin_amdgcn_readlane(tiles_incl - tiles_excl, owner);
    const int u = v - __builtin_amdgcn_readlane(tiles_excl, owner) * nbx;
    int tile = 0, n = u;
    if (T > 1) {
      const int run = u / (kNumXcd * T), left = u - run * (kNumXcd * T);
      const int g = min(kNumXcd, nbx - run * kNumXcd);
      tile = left / g;
      n = run * kNumXcd + left - tile * g;
    }
    out->row0 = __builtin_amdgcn_readlane(rows_incl - cnt, owner) + tile * kDBM;
    out->row_end = __builtin_amdgcn_readlane(rows_incl, owner);
    out->n0 = n * bn;
    return true;
  }
};

// The routing of at most 512 flat ids (nflat = N * k), computed by each
// block of the gathering gate/up kernel instead of a separate permute
// launch: per-expert counts, expert-major slots in
// flat order within each expert (the permute's assignment, dispatch.hip),
// and the slot -> token map s_tok.  Ids outside [0, E) get no slot, as in
// the permute.  With publish set the block also writes counts, perm and
// slot_of for the down GEMM, the combine and the caller.  All threads call
// it; wave 0 does the work.
constexpr int kGatherFlat = kRouterTokens * kMaxTopK;
__device__ __forceinline__ void decode_rank(const int32_t* __restrict__ topk_idx, int nflat,
                                            int k, int E, int* s_cnt, int* s_base, int* s_run,
                                            int* s_tok, bool publish,
                                            int32_t* __restrict__ counts,
                                            int32_t* __restrict__ perm,
                                            int32_t* __restrict__ slot_of) {
  const int tid = threadIdx.x;
  if (tid < kWave) {
    const int l = tid;
    constexpr int kIdPerLane = kGatherFlat / kWave;
    int ids[kIdPerLane];
#pragma unroll
    for (int u = 0; u < kIdPerLane; ++u) {
      const int f = u * kWave + l;
      ids[u] = f < nflat ? topk_idx[f] : -1;
    }
    s_cnt[l] = 0;
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int u = 0; u < kIdPerLane; ++u)
      if (ids[u] >= 0 && ids[u] < E) atomicAdd(&s_cnt[ids[u]], 1);
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    const int cnt = l < E ? s_cnt[l] : 0;
    s_base[l] = wave_incl_scan(cnt) - cnt;
    s_run[l] = 0;
    if (publish && l < E) counts[l] = cnt;
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    const unsigned long long lt = (l == 0) ? 0ull : (~0ull >> (kWave - l));
#pragma unroll
    for (int u = 0; u < kIdPerLane; ++u) {
      const int f0 = u * kWave;
      if (f0 >= nflat) break;
      const int f = f0 + l;
      int e = ids[u];
      const bool valid = e >= 0 && e < E;
      if (!valid) e = 0;
      unsigned long long match = __ballot(valid);
#pragma unroll
      for (int bit = 0; bit < 6; ++bit) {
        const unsigned long long on = __ballot(valid && ((e >> bit) & 1));
        match &= ((e >> bit) & 1) ? on : ~on;
      }
      if (valid) {
        const int run = s_run[e];
        const int slot = s_base[e] + run + __popcll(match & lt);
        s_tok[slot] = f / k;
        if (publish) {
          perm[slot] = f;
          slot_of[f] = slot;
        }
        // the highest lane of each expert group advances the running count
        if ((match >> l) == 1ull) s_run[e] = run + __popcll(match);
      }
    }
  }
  __syncthreads();
}

// GATHER (gate/up of at most 512 flat ids, bf16 rows): the activation rows
// come straight from the caller's x through s_tok instead of from the
// gathered copy A, and the routing is computed in the block (decode_rank).
template <int EPI, bool GATHER, typename XT, int NW>
__global__ __launch_bounds__(NW * 64) void gemm_decode_kernel(
    const XT* __restrict__ A, const fp8_t* __restrict__ B, const float* __restrict__ wscale,
    const float* __restrict__ bias0, const float* __restrict__ bias1,
    const int32_t* __restrict__ counts, int E, int K, int Npad, int n_store, int bias_ld,
    bf16_t* __restrict__ out, int ldo, const int32_t* __restrict__ topk_idx, int nflat, int k,
    int32_t* __restrict__ counts_out, int32_t* __restrict__ perm,
    int32_t* __restrict__ slot_of) {
  // Activation rows of XT (bf16, or the caller's fp32 rows when gathering):
  // kRowB bytes per stage row, staged as they are and converted to bf16 when
  // the fragments are read.
  constexpr int kXS = (int)sizeof(XT);
  constexpr int BN = 64 * NW;                  // features per item
  constexpr int kWBytes = BN * kDBK;
  constexpr int kAB = kDBM * kDBK * kXS;       // activation bytes per stage
  constexpr int kStage = kWBytes + kAB;
  constexpr int kDA = kAB / 1024 / NW;         // activation blocks per wave
  constexpr int kDm = kDmaW + kDA;             // loads per wave and stage
  constexpr int kRowB = kDBK * kXS;            // LDS bytes per activation row
  constexpr int kRowsPerBlk = 1024 / kRowB;
  constexpr int kChunks = kRowB / 16;          // 16-byte chunks per row
  static_assert(kXS == 2 || kXS == 4, "bf16 or fp32 rows");
  // ring depth: what LDS holds and the wait counter can count (63 loads)
  constexpr int kLds = (160 * 1024 / blocks_per_cu(NW) - (GATHER ? kGatherFlat * 4 + 1024 : 0)) / kStage;
  constexpr int kCnt = 63 / kDm + 2;
  constexpr int kDStages = kLds < kCnt ? kLds : kCnt;
  static_assert(kDStages >= 2, "ring depth");
  __shared__ __attribute__((aligned(1024))) char smem[kDStages * kStage];
  __shared__ int s_tok[GATHER ? kGatherFlat : 1];
  __shared__ int s_cnt[GATHER ? kMaxExperts : 1], s_base[GATHER ? kMaxExperts : 1],
      s_run[GATHER ? kMaxExperts : 1];
  const int nbx = (n_store + BN - 1) / BN;
  const int G = gridDim.x;
  const int32_t* cnts = counts;
  if constexpr (GATHER) {
    decode_rank(topk_idx, nflat, k, E, s_cnt, s_base, s_run, s_tok, blockIdx.x == 0, counts_out,
                perm, slot_of);
    cnts = s_cnt;
  }
  DScan sc;
  sc.init(cnts, E);
  int v = blockIdx.x;
  DItem cur;
  if (!sc.locate(E, nbx, BN, v, &cur)) return;

  const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave);
  const int lane = lane_id();
  const int lrow = lane & 31, lhalf = lane >> 5;
  const int KT = K / kDBK;
  const size_t tiles_n = Npad / kTileN;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_char*)smem;

  // DMA lane mapping.  Weights: 128-byte rows, wave w fills rows 64w ..
  // 64w+63 in 8 blocks of 8 rows; lane l covers row 8i + l/8, slot l%8 =
  // chunk ^ ((row >> 1) & 7).  Activations: kRowB-byte rows (256 for bf16,
  // 512 for fp32), wave w fills kDA blocks of kRowsPerBlk rows; lane l covers row kRowsPerBlk*i + l/kChunks, slot
  // l%kChunks = chunk ^ (row & (kChunks - 1)).  Activation rows past the
  // item's last token re-read that token (in bounds, never stored).
  // Weights are in the tiled layout [E][Npad/256][K/128][256][128]: a
  // stage's are one contiguous block, rows 128 bytes apart.
  const size_t arow_g = (size_t)K * kXS;    // bytes per activation row
  uint32_t woff[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = i * 8 + lane / 8;
    woff[i] = (uint32_t)(lane / 8) * (uint32_t)kDBK + (uint32_t)(((lane % 8) ^ ((r >> 1) & 7)) * 16);
  }

  // DMA cursor: item dv at stage column block dkt, STAGES-1 stages ahead, with
  // this lane's addresses of the stage (a row of weights 8i + lane / 8 is 1024 i
  // bytes on; the addresses are formed once an item and stepped per stage: a
  // stage's arithmetic is 64-bit adds only).
  DItem dit = cur;
  int dv = v, dkt = 0, dstage = 0;
  bool dvalid = true;
  int ahead = 0;   // stages issued and not yet waited for
  const char* wp[2];
  const char* ap[kDA];
  auto enter_item = [&]() __attribute__((always_inline)) {
    const char* wg = reinterpret_cast<const char*>(B) +
                     ((size_t)dit.expert * tiles_n + dit.n0 / kTileN) * KT * (size_t)(kTileN * kDBK) +
                     (size_t)(dit.n0 % kTileN + 64 * w) * kDBK;
    wp[0] = wg + woff[0];
    wp[1] = wg + woff[1];
#pragma unroll
    for (int i = 0; i < kDA; ++i) {
      const int r = (w * kDA + i) * kRowsPerBlk + lane / kChunks;   // activation row in the tile
      const int tok = min(dit.row0 + r, dit.row_end - 1);           // a slot
      const int src_row = GATHER ? s_tok[tok] : tok;
      ap[i] = reinterpret_cast<const char*>(A) + (size_t)src_row * arow_g +
              (((lane % kChunks) ^ (r & (kChunks - 1))) << 4);
    }
  };
  enter_item();
  auto advance = [&]() __attribute__((always_inline)) {
    if (dvalid) {
      const uint32_t st = lds0 + (uint32_t)(dstage * kStage);
#pragma unroll
      for (int i = 0; i < kDmaW; ++i)
        dma16_stream(wp[i & 1] + 1024 * i, st + (uint32_t)((w * kDmaW + i) * 1024));
#pragma unroll
      for (int i = 0; i < kDA; ++i) dma16(ap[i], st + (uint32_t)(kWBytes + (w * kDA + i) * 1024));
      wp[0] += kTileN * kDBK;
      wp[1] += kTileN * kDBK;
#pragma unroll
      for (int i = 0; i < kDA; ++i) ap[i] += kRowB;
      ++ahead;
    }
    dstage = dstage + 1 == kDStages ? 0 : dstage + 1;
    if (++dkt == KT) {
      dkt = 0;
      dv += G;
      if (dvalid) dvalid = sc.locate(E, nbx, BN, dv, &dit);
      if (dvalid) enter_item();
    }
  };
  // Barrier before consuming stage c: it landed, with the stages issued
  // after it (`ahead` once c is counted) possibly in flight; every wave is
  // done with stage c-1, which the DMA issued right after refills.
  auto next_stage_barrier = [&]() __attribute__((always_inline)) {
    --ahead;
    if (ahead >= kDStages - 2) stage_barrier<(kDStages - 2) * kDm>();
    else stage_barrier<0>();
    advance();
  };

  // Fragment reads.  Weights (A operand): this wave's rows 64w + 32j + lrow,
  // bytes 64*lhalf .. +63 of the stage row = chunks 4*lhalf .. +3.
  // Activations (B operand): token row lrow, k-step ks = chunk 8*lhalf + ks.
  const int wswz = (lrow >> 1) & 7;
  auto wfrag = [&](const char* st, int j, int q) -> uint4 {   // q = chunk pair index 0..3
    const int row = 64 * w + 32 * j + lrow;
    const int chunk = 4 * lhalf + q;
    return *reinterpret_cast<const uint4*>(st + row * kDBK + ((chunk ^ wswz) << 4));
  };
  struct ARaw {
    uint4 v[kXS / 2];
  };
  auto aread = [&](const char* st, int ks) -> ARaw {
    const int c = 8 * lhalf + ks;   // columns 8c .. 8c+7 of the stage
    const char* row = st + kWBytes + lrow * kRowB;
    ARaw r;
    if constexpr (kXS == 2) {
      r.v[0] = *reinterpret_cast<const uint4*>(row + ((c ^ (lrow & 15)) << 4));
    } else {
      r.v[0] = *reinterpret_cast<const uint4*>(row + (((2 * c) ^ (lrow & 31)) << 4));
      r.v[kXS / 2 - 1] = *reinterpret_cast<const uint4*>(row + (((2 * c + 1) ^ (lrow & 31)) << 4));
    }
    return r;
  };
  auto abf16 = [&](const ARaw& r) -> bf16x8 {
    if constexpr (kXS == 2) {
      return __builtin_bit_cast(bf16x8, r.v[0]);
    } else {
      // two 16-byte chunks of fp32 rounded to bf16 by v_cvt_pk_bf16_f32
      // (nearest even, fp32 denormals kept: the rounding f32_to_bf16 does in
      // software for the permute's gather, at 4 instructions a fragment)
      typedef float f32x8 __attribute__((ext_vector_type(8)));
      return __builtin_convertvector(__builtin_bit_cast(f32x8, r), bf16x8);
    }
  };

#pragma unroll
  for (int s = 0; s < kDStages - 1; ++s) advance();
  next_stage_barrier();
  int cstage = 0;

  for (;;) {
    DItem nxt;
    const bool have_next = sc.locate(E, nbx, BN, v + G, &nxt);
    f32x16 acc[2];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[j][e] = 0.0f;
    for (int kt = 0; kt < KT; ++kt) {
      const char* st = smem + cstage * kStage;
      // every LDS read of the stage first (one wave a SIMD: nothing else hides
      // their latency), then 8 k-steps: weights as 4 chunks of 16 fp8 per row
      // (2 k-steps each)
      uint4 wv[2][4];
      ARaw av[8];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        wv[0][q] = wfrag(st, 0, q);
        wv[1][q] = wfrag(st, 1, q);
        av[2 * q] = aread(st, 2 * q);
        av[2 * q + 1] = aread(st, 2 * q + 1);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int ks = 0; ks < 8; ++ks) {
        const uint4 w0 = wv[0][ks / 2], w1 = wv[1][ks / 2];
        const bf16x8 b = abf16(av[ks]);
        const bf16x8 a0 = (ks & 1) ? fp8x8_to_bf16x8(w0.z, w0.w) : fp8x8_to_bf16x8(w0.x, w0.y);
        const bf16x8 a1 = (ks & 1) ? fp8x8_to_bf16x8(w1.z, w1.w) : fp8x8_to_bf16x8(w1.x, w1.y);
        acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a0, b, acc[0], 0, 0, 0);
        acc[1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a1, b, acc[1], 0, 0, 0);
      }
      cstage = cstage + 1 == kDStages ? 0 : cstage + 1;
      // next stage (after the block's last one this waits for nothing new)
      next_stage_barrier();
    }

    // Epilogue.  Register e of a 32x32 tile holds feature row
    // 8*(e/4) + 4*(lane/32) + e%4 and token column lane%32.
    const int row = cur.row0 + lrow;
    const float* sc_e = wscale + (size_t)cur.expert * Npad;
    if constexpr (EPI == kEpiGateUp) {
      // rows 64w .. 64w+31 gate, 64w+32 .. +63 up of hidden units hb .. hb+31
      const int p0 = cur.n0 + 64 * w;            // packed row of gate unit 0
      const int hb = p0 / 2;
      const float* bgp = bias0 + (size_t)cur.expert * bias_ld + hb;
      const float* bup = bias1 + (size_t)cur.expert * bias_ld + hb;
      if (row < cur.row_end) {
        bf16_t* orow = out + (size_t)row * ldo + hb + 4 * lhalf;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          float o[4];
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const int f = 8 * g + q;   // feature within the 32 (lane half 0)
            const float sg0 = uniform_load(sc_e + p0 + f), sg1 = uniform_load(sc_e + p0 + f + 4);
            const float su0 = uniform_load(sc_e + p0 + 32 + f), su1 = uniform_load(sc_e + p0 + 32 + f + 4);
            const float bg0 = uniform_load(bgp + f), bg1 = uniform_load(bgp + f + 4);
            const float bu0 = uniform_load(bup + f), bu1 = uniform_load(bup + f + 4);
            const float gv = acc[0][4 * g + q] * (lhalf ? sg1 : sg0) + (lhalf ? bg1 : bg0);
            const float uv = acc[1][4 * g + q] * (lhalf ? su1 : su0) + (lhalf ? bu1 : bu0);
            o[q] = silu_mul_fast(gv, uv);
          }
          *reinterpret_cast<uint2*>(orow + 8 * g) = pack4_bf16(o[0], o[1], o[2], o[3]);
        }
      }
    } else {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int cb = cur.n0 + 64 * w + 32 * j;
        if (cb >= n_store || row >= cur.row_end) continue;
        const float* bdp = bias0 + (size_t)cur.expert * bias_ld + cb;
        bf16_t* orow = out + (size_t)row * ldo + cb + 4 * lhalf;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          float o[4];
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const int f = 8 * g + q;
            const float s0 = uniform_load(sc_e + cb + f), s1 = uniform_load(sc_e + cb + f + 4);
            const float b0 = uniform_load(bdp + f), b1 = uniform_load(bdp + f + 4);
            o[q] = acc[j][4 * g + q] * (lhalf ? s1 : s0) + (lhalf ? b1 : b0);
          }
          *reinterpret_cast<uint2*>(orow + 8 * g) = pack4_bf16(o[0], o[1], o[2], o[3]);
        }
      }
    }
    if (!have_next) break;
    v += G;
    cur = nxt;
  }
}

// Persistent launch.  Requires K % 128 == 0, Npad % 256 ==
// 0 and n_store % 64 == 0; rows: all rows of the E segments.
template <int EPI, bool GATHER, typename XT>
hipError_t launch_decode(const XT* A, const fp8_t* B, const float* wscale, const float* bias0,
                         const float* bias1, const int32_t* counts, int E, int K, int Npad,
                         int n_store, int bias_ld, bf16_t* out, int ldo, int rows,
                         const int32_t* topk_idx, int k, int32_t* counts_out, int32_t* perm,
                         int32_t* slot_of, hipStream_t stream) {
  if (rows <= 0) return hipSuccess;
  if (K % kDBK != 0 || Npad % kTileN != 0 || n_store % 64 != 0) return hipErrorInvalidValue;
  static int num_cus = 0;
  if (num_cus == 0) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&num_cus, hipDeviceAttributeMultiprocessorCount, dev);
    if (e != hipSuccess || num_cus <= 0) num_cus = 256;
  }
  // An item of 64 features (one wave) where those give no CU more than one.  us on
  // MI355X for 256 features and one block a CU / 128 / 64: down, E = 64, C = 2048, H =
  // 1408, 1 token 15.2 / 12.0 / 10.8 (256 items of 64), 64 tokens 36.9 / 36.0 / 40.1
  // (2048); E = 16, C = 1024, H = 2816, 37 tokens 23.3 / 19.8 / 16.3 (256); gate/up of the
  // former, 1 token 20.1 / 16.6 / 17.4 (352), 64 tokens 67.1 / 66.8 / 79.6 (2816).
  const long est = (long)rows <= 16L * E ? std::min<long>(E, rows) : rows / 32 + E;
  const bool narrow = est * ((n_store + 63) / 64) <= num_cus;
  // Else 128 features.  fp32 rows leave two blocks' rings two stages each, so they
  // take 256 features and one block a CU where those fill one round of the CUs by more
  // than half, or a last round, by the experts to expect under an even routing (and
  // one and a half standard deviations more).  us of gate/up for 256 / 128: E = 32, C
  // = 2048, H = 1024, k = 8: 1 token (a quarter of a round) 24 / 20, 4 (0.65) 26 / 29, 40
  // (1) 28 / 31; E = 16, C = 1024, H = 2816, k = 2: 10 (1.03) 29 / 26, 37 (1.4) 28 / 28;
  // E = 64, C = 2048, H = 1408, k = 8: 40 (2.75) 67 / 77.
  bool wide = false;
  if (sizeof(XT) == 4) {
    const double per_tile = (double)((n_store + 255) / 256) / num_cus;   // rounds
    const double p = 1.0 - std::exp(-(double)rows / E);
    const double rounds = E * p * per_tile;
    const double most = std::ceil(std::min((double)E, E * p + 1.5 * std::sqrt(E * p * (1.0 - p))) * per_tile);
    wide = most < 1.33 * rounds || (most == 1.0 && rounds > 0.5);
  } else if (rows >= 4L * E && K >= 1024) {
    // bf16 rows, one row tile an expert or two: items of 128 features read the rows'
    // stages twice as often, which costs more than their finer last round saves where a
    // CU has much to contract (twice that for one tile) and the 256-feature items nearly
    // fill their rounds (and an expert has eight feature blocks, so that its row tiles
    // share an XCD).  us of the forward for 128 / 256: E = 64, C = 4096, H = 2048, k = 8,
    // 288 tokens 487 / 406; E = 32, C = 2048, H = 4096, k = 4, 352 tokens 270 / 228; E = 32,
    // C = 4096, H = 1024, k = 2, 992 tokens 206 / 193; E = 64, C = 1024, H = 4096, k = 4, 448
    // tokens 225 / 206; where the rule keeps 128, gate/up alone: E = 16, C = 1024, H = 2816,
    // k = 2, 352 tokens 33 / 39; E = 64, C = 2048, H = 512, k = 4, 832 tokens 57 / 66; E =
    // 64, C = 2048, H = 1408, k = 8, 240 tokens 83 / 88.
    const int tiles = rows > 32L * E ? 2 : 1;
    const int nb = (n_store + 255) / 256;
    const double rounds = (double)tiles * E * nb / num_cus;
    wide = nb >= 8 && rounds * K >= 8192.0 / tiles && rounds > 0.9 * std::ceil(rounds);
  }
  auto launch = [&](auto kernel, int NW) {
    const long items = (long)(rows / 32 + std::min(E, rows)) * ((n_store + 64 * NW - 1) / (64 * NW));
    hipLaunchKernelGGL(kernel, dim3((unsigned)std::min<long>(items, blocks_per_cu(NW) * num_cus)),
                       dim3(64 * NW), 0, stream, A, B, wscale, bias0, bias1, counts, E, K, Npad, n_store,
                       bias_ld, out, ldo, topk_idx, rows, k, counts_out, perm, slot_of);
  };
  if (narrow)
    launch(gemm_decode_kernel<EPI, GATHER, XT, 1>, 1);
  else if (wide)
    launch(gemm_decode_kernel<EPI, GATHER, XT, 4>, 4);
  else
    launch(gemm_decode_kernel<EPI, GATHER, XT, 2>, 2);
  return hipGetLastError();
}

}  // namespace

template <int EPI>
hipError_t launch_gemm_decode(const bf16_t* A, const fp8_t* B, const float* wscale,
                              const float* bias0, const float* bias1, const int32_t* counts, int E,
                              int K, int Npad, int n_store, int bias_ld, bf16_t* out, int ldo,
                              int rows, hipStream_t stream) {
  return launch_decode<EPI, false, bf16_t>(A, B, wscale, bias0, bias1, counts, E, K, Npad, n_store,
                                   bias_ld, out, ldo, rows, nullptr, 0, nullptr, nullptr, nullptr,
                                   stream);
}

template hipError_t launch_gemm_decode<kEpiGateUp>(const bf16_t*, const fp8_t*, const float*,
                                                   const float*, const float*, const int32_t*, int,
                                                   int, int, int, int, bf16_t*, int, int,
                                                   hipStream_t);
template hipError_t launch_gemm_decode<kEpiDown>(const bf16_t*, const fp8_t*, const float*,
                                                 const float*, const float*, const int32_t*, int,
                                                 int, int, int, int, bf16_t*, int, int,
                                                 hipStream_t);

// The gate/up GEMM of at most 512 flat ids (nflat = N * k) with the
// caller's rows x [N][K] (bf16, or fp32 rounded to bf16 as the permute
// would): routes the ids itself (the permute's
// counts, perm and slot_of, written by block 0) and reads the activation
// rows from x, so no permute kernel runs and no gathered copy is written.
template <typename XT>
hipError_t launch_gemm_decode_gather(const XT* x, const fp8_t* B, const float* wscale,
                                     const float* bias0, const float* bias1, const int32_t* topk_idx,
                                     int nflat, int k, int E, int K, int Npad, int n_store,
                                     int bias_ld, bf16_t* out, int ldo, int32_t* counts, int32_t* perm, int32_t* slot_of,
                                     hipStream_t stream) {
  if (nflat > kGatherFlat || E > kMaxExperts || k < 1) return hipErrorInvalidValue;
  return launch_decode<kEpiGateUp, true, XT>(x, B, wscale, bias0, bias1, nullptr, E, K, Npad, n_store,
                                         bias_ld, out, ldo, nflat, topk_idx, k, counts, perm,
                                         slot_of, stream);
}
template hipError_t launch_gemm_decode_gather<bf16_t>(const bf16_t*, const fp8_t*, const float*,
                                                       const float*, const float*, const int32_t*,
                                                       int, int, int, int, int, int, int, bf16_t*,
                                                       int, int32_t*, int32_t*, int32_t*,
                                                       hipStream_t);
template hipError_t launch_gemm_decode_gather<float>(const float*, const fp8_t*, const float*,
                                                      const float*, const float*, const int32_t*,
                                                      int, int, int, int, int, int, int, bf16_t*,
                                                      int, int32_t*, int32_t*, int32_t*,
                                                      hipStream_t);

}  // namespace mgpt
