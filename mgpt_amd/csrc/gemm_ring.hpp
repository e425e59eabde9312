// gemm_ring.hpp -- what the direct-to-LDS grouped GEMMs (gemm_dma.hip,
// gemm_stream.hip) share: the wave layout, the tile order over the experts'
// segments, the split of a persistent launch's last round, the epilogues and
// the reduction of split tiles.
#pragma once

#include "common.hpp"

namespace mgpt {
namespace {

// Wave layout of a block on a tile of BM tokens x BN features: NW waves as WN
// (features) x WM (tokens); each wave owns a WTN x WTM tile of TN x TM 32x32
// MFMA tiles.
template <int NW, int BM = 256, int BN = 256>
struct Waves {
  static constexpr int kWaves = NW, kBM = BM, kBN = BN;
  static constexpr int kThreads = NW * kWave;
  static constexpr int WN = NW == 8 ? 4 : 2, WM = 2;
  static constexpr int WTN = BN / WN, WTM = BM / WM;
  static constexpr int TN = WTN / 32, TM = WTM / 32;
  static_assert(WN * WM == NW, "wave layout");
  static constexpr bool kAgpr = TN * TM > 8;   // accumulators beyond the VGPRs
};

typedef __attribute__((address_space(3))) char lds_char;

template <int V>
struct IntC {
  static constexpr int value = V;
};

// One 1 KB direct-to-LDS load: lane l's 16 bytes at g land at LDS address
// lds + 16*l.  Written as inline asm so that the compiler does not track it:
// for the builtin it places a vmcnt(0) wait before every LDS read that it
// cannot prove disjoint from the DMA, which serialises the ring.  The
// kernel waits for the DMA itself (slab_barrier); M0 is an input operand.
__device__ __forceinline__ void dma16(const void* g, uint32_t lds) {
  asm volatile("global_load_lds_dwordx4 %0, off" ::"v"(g), "{m0}"(lds) : "memory");
}

// Start of a slab: this wave's DMA of the slab has landed (at most N of its
// later DMA loads still in flight) and its own LDS reads are complete; then
// meet the other waves.  Inline asm, because the compiler treats the
// builtin s_waitcnt as a hint it may relax (it dropped the lgkmcnt(0) that
// protects the stage the next DMA overwrites), and the memory clobber keeps
// LDS accesses from moving across it.
template <int N>
__device__ __forceinline__ void slab_barrier() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

// A float read at a wave-uniform address, forced into an SGPR (so the
// compiler emits a scalar load).
__device__ __forceinline__ float uniform_load(const float* p) {
  return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(*p)));
}

// silu(g) * u and the sigmoid, by the hardware reciprocal (1 ulp) or divided.
// The reciprocal form multiplies g by u first, so a product past fp32's range
// (|g u| > 3.4e38) gives infinity, or NaN where the reciprocal is 0; the divided
// one makes g small first.
__device__ __forceinline__ float silu_mul_fast(float g, float u) {
  return g * u * __builtin_amdgcn_rcpf(1.0f + __expf(-g));
}
__device__ __forceinline__ float silu_mul(float g, float u) { return (g / (1.0f + __expf(-g))) * u; }

// Four floats -> four bf16 (round to nearest even) in 8 bytes.
__device__ __forceinline__ uint2 pack4_bf16(float a, float b, float c, float d) {
  typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
  bf16x2_t lo = {(__bf16)a, (__bf16)b}, hi = {(__bf16)c, (__bf16)d};
  uint2 r;
  __builtin_memcpy(&r.x, &lo, 4);
  __builtin_memcpy(&r.y, &hi, 4);
  return r;
}

struct Tile {
  int expert, row0, row_end, n0;
};

constexpr int kGroupM = 4;   // m-tiles per group of the tile order

// Per-expert segment bookkeeping, computed once per wave from counts[] (lane
// e holds expert e_base + e of the block's group of E <= 64 experts; more
// experts take a grid row, or a launch, per group, whose rows start after the
// earlier groups' rows), so that locating a tile needs no memory access and no
// barrier.
template <int BM>
struct SegScan {
  // (the exclusive counts are recomputed where needed: the kernel runs at
  // the register limit, and these live in every lane throughout)
  int cnt, rows_incl, tiles_incl, tm;
  __device__ __forceinline__ int tiles_excl() const { return tiles_incl - (cnt + BM - 1) / BM; }
  __device__ __forceinline__ void init(const int32_t* __restrict__ counts, int E, int e_base) {
    const int l = lane_id();
    cnt = (l < E) ? counts[e_base + l] : 0;
    const int tiles = (cnt + BM - 1) / BM;
    int before = 0;   // rows of the experts before the group
    if (e_base > 0) {
      for (int e = l; e < e_base; e += kWave) before += counts[e];
      before = __builtin_amdgcn_readfirstlane(__shfl(wave_incl_scan(before), kWave - 1, kWave));
    }
    rows_incl = wave_incl_scan(cnt) + before;
    tiles_incl = wave_incl_scan(tiles);
    tm = __builtin_amdgcn_readfirstlane(__shfl(tiles_incl, kWave - 1, kWave));   // all m-tiles
  }
};

// Tile of linear index v, or false past the last one.  Tiles are ordered in
// groups of kGroupM m-tiles (token blocks, over all experts' segments) x all
// n-tiles, m fastest, so that any 32 consecutive indices cover about 4 token
// blocks x 8 feature blocks: the 32 blocks of one XCD (see the remap in the
// kernel) then share 12 operand panels in that XCD's L2 instead of ~23.
template <int BN = 256, int BM>
__device__ __forceinline__ bool locate_tile(const SegScan<BM>& sc, int E, int nbx, int v, Tile* out) {
  if (v >= sc.tm * nbx) return false;
  const int g = v / (kGroupM * nbx);
  const int gsize = min(kGroupM, sc.tm - g * kGroupM);
  const int idx = v - g * kGroupM * nbx;
  const int mt = g * kGroupM + idx % gsize;
  const int l = lane_id();
  const int texcl = sc.tiles_excl();
  const bool mine = (l < E) && (mt >= texcl) && (mt < sc.tiles_incl);
  const unsigned long long m = __ballot(mine);
  const int owner = __ffsll((long long)m) - 1;   // exists: mt < tm
  out->expert = __builtin_amdgcn_readfirstlane(owner);
  out->row0 = __builtin_amdgcn_readfirstlane(
      __shfl((sc.rows_incl - sc.cnt) + (mt - texcl) * BM, owner, kWave));
  out->row_end = __builtin_amdgcn_readfirstlane(__shfl(sc.rows_incl, owner, kWave));
  out->n0 = (idx / gsize) * BN;
  return true;
}

// The accumulators of one 32 x 32 tile as VGPR values.  With 4 waves on a
// 256 x 256 tile (256 accumulators per lane) the accumulators live in AGPRs; reading
// them through v_accvgpr_read one tile at a time stops the compiler from
// copying all 256 into VGPRs at the loop exit (which spills).  The caller
// has waited out the MFMA result latency (mfma_drain).
template <typename W>
__device__ __forceinline__ f32x16 acc_fetch(const f32x16& a) {
  if constexpr (!W::kAgpr) {
    return a;
  } else {
    f32x16 r;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      float x;
      asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(x) : "a"(a[v]));
      r[v] = x;
    }
    return r;
  }
}

template <typename W>
__device__ __forceinline__ void mfma_drain() {
  if constexpr (W::kAgpr) asm volatile("s_nop 15\n\ts_nop 15\n\ts_nop 15\n\ts_nop 15" ::: "memory");
}

// Stores the 32 outputs (features base .. base+31) of one token that a lane
// pair (l, l+32) holds as quads: q[g] of lane l are features 8g..8g+3, of lane
// l+32 features 8g+4..8g+7 (bf16 pairs).  Swapping two quads across the pair
// leaves lane l with the whole 8-feature groups 0 and 2 and lane l+32 with 1
// and 3, so each lane writes 16-byte vectors and a store covers 32 bytes of
// each of the 32 token rows (instead of 16).  The swap is gfx950's
// v_permlane32_swap (a VALU op, no LDS round trip): swap(a, b) gives lane
// l < 32 the pair (a[l], a[l+32]) and lane l >= 32 (b[l-32], b[l]), which
// with (a, b) = (q[0], q[1]) is each lane's 8-feature group as it is stored.
// Every lane of the pair must run this (it exchanges registers); `store`
// gates the memory writes.
__device__ __forceinline__ void store_group32(bf16_t* base, const uint2 (&q)[4], int lhalf,
                                              bool store) {
  const auto ax = __builtin_amdgcn_permlane32_swap(q[0].x, q[1].x, false, false);
  const auto ay = __builtin_amdgcn_permlane32_swap(q[0].y, q[1].y, false, false);
  const auto bx = __builtin_amdgcn_permlane32_swap(q[2].x, q[3].x, false, false);
  const auto by = __builtin_amdgcn_permlane32_swap(q[2].y, q[3].y, false, false);
  const uint4 w0 = make_uint4(ax[0], ay[0], ax[1], ay[1]);
  const uint4 w1 = make_uint4(bx[0], by[0], bx[1], by[1]);
  if (store) {
    *reinterpret_cast<uint4*>(base + 8 * lhalf) = w0;
    *reinterpret_cast<uint4*>(base + 16 + 8 * lhalf) = w1;
  }
}

// The inverse of store_group32: loads the 32 bf16 values (features base ..
// base+31) of one token as two 16-byte vectors per lane (lane half h takes
// features 8h..8h+7 and 16+8h..16+8h+7) and swaps quads with the partner
// lane, so that q[g] of lane half h holds features 8g+4h .. 8g+4h+3, the
// accumulator layout.  Rows past the segment read zeros (no access); every
// lane of the pair runs the swaps.
__device__ __forceinline__ void load_group32(const bf16_t* base, uint2 (&q)[4], int lhalf,
                                             bool load) {
  uint4 w0 = make_uint4(0u, 0u, 0u, 0u), w1 = w0;
  if (load) {
    w0 = *reinterpret_cast<const uint4*>(base + 8 * lhalf);
    w1 = *reinterpret_cast<const uint4*>(base + 16 + 8 * lhalf);
  }
  const auto s0 = __builtin_amdgcn_permlane32_swap(w0.x, w0.z, false, false);
  const auto s1 = __builtin_amdgcn_permlane32_swap(w0.y, w0.w, false, false);
  const auto s2 = __builtin_amdgcn_permlane32_swap(w1.x, w1.z, false, false);
  const auto s3 = __builtin_amdgcn_permlane32_swap(w1.y, w1.w, false, false);
  q[0] = make_uint2(s0[0], s1[0]);
  q[1] = make_uint2(s0[1], s1[1]);
  q[2] = make_uint2(s2[0], s3[0]);
  q[3] = make_uint2(s2[1], s3[1]);
}

// Epilogue straight from the accumulators of a wave's WTN-feature x
// WTM-token tile.  Register v of a 32x32 tile holds feature row
// 8*(v/4) + 4*(lane/32) + v%4 (four consecutive features per group v/4) and
// token column lane%32.  Biases are read at wave-uniform addresses (scalar
// loads): a vector load here would make the compiler wait for the DMA loads
// it does not track as well.  kStream (gemm_stream.hip): one sub-tile at a
// time, and silu and the sigmoid divided.
template <int EPI, typename W, bool kSave, bool kStream = false>
__device__ __forceinline__ void store_tile(const f32x16 (&acc)[W::TN][W::TM],
                                           const Tile& cur, int wn, int wm, int lrow, int lhalf,
                                           int n_store, bf16_t* out, int ldo, bf16_t* save,
                                           int save_ld) {
  const int tok_base = cur.row0 + wm * W::WTM + lrow;
  if constexpr (EPI == kEpiGateUp) {
    // each 64 packed rows of the wave are one [32 gate | 32 up] group
#pragma unroll
    for (int gi = 0; gi < W::TN / 2; ++gi) {
      const int hb = (cur.n0 + wn * W::WTN) / 2 + 32 * gi;
#pragma unroll
      for (int i = 0; i < W::TM; ++i) {
        const int row = tok_base + i * 32;
        const f32x16 ga = acc_fetch<W>(acc[2 * gi][i]);
        const f32x16 ua = acc_fetch<W>(acc[2 * gi + 1][i]);
        auto act = [](float gv, float uv) { return kStream ? silu_mul(gv, uv) : silu_mul_fast(gv, uv); };
        uint2 q[4];
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const int v = 4 * g;
          q[g] = pack4_bf16(act(ga[v + 0], ua[v + 0]), act(ga[v + 1], ua[v + 1]),
                            act(ga[v + 2], ua[v + 2]), act(ga[v + 3], ua[v + 3]));
        }
        store_group32(out + (size_t)row * ldo + hb, q, lhalf, row < cur.row_end);
        if constexpr (kSave) {
          // pre-activations for the backward pass, in the packed column order
          const int pc = cur.n0 + wn * W::WTN + 64 * gi;
          uint2 sg[4], su[4];
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            const int v = 4 * g;
            sg[g] = pack4_bf16(ga[v], ga[v + 1], ga[v + 2], ga[v + 3]);
            su[g] = pack4_bf16(ua[v], ua[v + 1], ua[v + 2], ua[v + 3]);
          }
          store_group32(save + (size_t)row * save_ld + pc, sg, lhalf, row < cur.row_end);
          store_group32(save + (size_t)row * save_ld + pc + 32, su, lhalf, row < cur.row_end);
        }
        if constexpr (kStream) __builtin_amdgcn_sched_barrier(0);   // one sub-tile at a time
      }
      // one column group at a time: keeps the scheduler from hoisting every
      // accumulator read (TN * TM * 16 values) ahead of the stores
      __builtin_amdgcn_sched_barrier(0);
    }
  } else if constexpr (EPI == kEpiSwigluBwd) {
    // The features are hidden units h and the accumulators d(act)[row][h];
    // save holds the pre-activations g, u of h at its packed columns (32 gate
    // then 32 up per 32 units), and d(gate), d(up) overwrite them there.
#pragma unroll
    for (int j = 0; j < W::TN; ++j) {
      const int hb = cur.n0 + wn * W::WTN + j * 32;
      if (hb >= n_store) continue;
      const int pc = packed_gate_col(hb);
      // the g and u loads of two 32-token sub-tiles at a time, as 16-byte
      // vectors: half the memory round trips of one at a time, within the
      // register budget (four at a time spill)
      constexpr int kPair = W::TM < 2 ? 1 : 2;
#pragma unroll
      for (int i2 = 0; i2 < W::TM; i2 += kPair) {
        uint2 gq[kPair][4], uq[kPair][4];
#pragma unroll
        for (int ii = 0; ii < kPair; ++ii) {
          const int row = tok_base + (i2 + ii) * 32;
          const bool ok = row < cur.row_end;
          const bf16_t* src = save + (size_t)row * save_ld + pc;
          load_group32(src, gq[ii], lhalf, ok);
          load_group32(src + 32, uq[ii], lhalf, ok);
        }
#pragma unroll
        for (int ii = 0; ii < kPair; ++ii) {
          const int i = i2 + ii;
          const int row = tok_base + i * 32;
          const bool ok = row < cur.row_end;
          const f32x16 a = acc_fetch<W>(acc[j][i]);
          uint2 dq[4], uqo[4];
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            float dg[4], du[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              const uint32_t gw = q < 2 ? gq[ii][g].x : gq[ii][g].y;
              const uint32_t uw = q < 2 ? uq[ii][g].x : uq[ii][g].y;
              const float gv = __uint_as_float((q & 1) ? (gw & 0xFFFF0000u) : (gw << 16));
              const float uv = __uint_as_float((q & 1) ? (uw & 0xFFFF0000u) : (uw << 16));
              const float d = a[4 * g + q];
              const float den = 1.0f + __expf(-gv);
              const float sig = kStream ? 1.0f / den : __builtin_amdgcn_rcpf(den);
              du[q] = d * (gv * sig);
              dg[q] = (d * uv) * (sig * (1.0f + gv * (1.0f - sig)));
            }
            dq[g] = pack4_bf16(dg[0], dg[1], dg[2], dg[3]);
            uqo[g] = pack4_bf16(du[0], du[1], du[2], du[3]);
          }
          store_group32(out + (size_t)row * ldo + pc, dq, lhalf, ok);
          store_group32(out + (size_t)row * ldo + pc + 32, uqo, lhalf, ok);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  } else {
#pragma unroll
    for (int j = 0; j < W::TN; ++j) {
      const int cb = cur.n0 + wn * W::WTN + j * 32;
      if (cb >= n_store) continue;   // n_store is a multiple of 64
#pragma unroll
      for (int i = 0; i < W::TM; ++i) {
        const int row = tok_base + i * 32;
        const f32x16 a = acc_fetch<W>(acc[j][i]);
        uint2 q[4];
#pragma unroll
        for (int g = 0; g < 4; ++g)
          q[g] = pack4_bf16(a[4 * g + 0], a[4 * g + 1], a[4 * g + 2], a[4 * g + 3]);
        store_group32(out + (size_t)row * ldo + cb, q, lhalf, row < cur.row_end);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
}

// Work items of a persistent launch over T tiles with G blocks: the
// ceil(T/G)-th round would leave most blocks idle when T % G is small, so
// the tiles of that last round are split along K into s parts (s <= 8,
// G/(T % G) of them), each a work item of its own whose fp32 partial sums
// go to a workspace; gemm_split_reduce_kernel adds the parts in order and
// runs the epilogue.  All tiles of the full rounds are whole items.  A
// split item writes a 256 KB fp32 partial tile and the reduce kernel reads
// them back, a cost that only a long K amortises: 256-row tiles of fewer
// than kMinSplitSlabs 64-column slabs stay whole.  Measured on MI355X at the
// cfg3 shapes (skewed counts): gate/up (K = 1024, 16 slabs) 0.426 ms whole
// vs 0.439 split; down (K = 2816, 44 slabs) 0.214 split vs 0.246 whole.  A launch
// without a full round splits from three parts on: two save little or nothing, and
// the CUs that they keep busy cost the power-limited chip clock in the products around
// (us of gate/up + down, the latter whole / in two: E = 16, C = 1024, H = 1536, 3200
// tokens 58 + 44 / 59 + 52; C = 256, H = 2816, 12000 tokens 92 + 65 / 101 + 64; E = 32, C =
// 512, 4096 tokens H = 2048 51 + 49 / 57 + 50, H = 2816 90 + 75 / 91 + 66).
constexpr int kMinSplitSlabs = 24;
struct SplitPlan {
  int full, rem, s, items;
  __device__ __forceinline__ void init(int T, int G, int KT, bool enable) {
    full = (T / G) * G;
    rem = T - full;
    s = 1;
    if (enable && rem > 0 && KT >= kMinSplitSlabs) {
      s = min(min(G / rem, 8), KT);
      if (s < (full > 0 ? 2 : 3)) s = 1;
    }
    items = s > 1 ? full + rem * s : T;
  }
};

struct Work {
  Tile tile;
  int k0, k1;   // slab range
  int sidx;     // partial-sum slot, or -1 for a whole tile
};

template <int BN = 256, int BM>
__device__ __forceinline__ bool locate_work(const SegScan<BM>& sc, const SplitPlan& pl, int E,
                                            int nbx, int KT, int v, Work* wk) {
  if (v >= pl.items) return false;
  int tv;
  if (pl.s == 1 || v < pl.full) {
    tv = v;
    wk->k0 = 0;
    wk->k1 = KT;
    wk->sidx = -1;
  } else {
    const int u = v - pl.full;
    const int part = u % pl.s;
    tv = pl.full + u / pl.s;
    wk->k0 = part * KT / pl.s;
    wk->k1 = (part + 1) * KT / pl.s;
    wk->sidx = u;
  }
  return locate_tile<BN>(sc, E, nbx, tv, &wk->tile);
}


// Partial sums of one work item, a whole BM x BN fp32 tile, stored as
// [TN*TM*4 float4 slots q][threads] so that every store and load is a
// coalesced row.  q = (j * kTM + i) * 4 + v4 holds acc[j][i][4v4 ..].

// Sums the s partial tiles of each split tile in order and applies the
// epilogue, one output quad (4 features of one token) per thread and
// iteration: the s float4 loads of a quad are independent, so each thread
// keeps them all in flight, and the quads of all split tiles are spread over
// the whole grid.  The (GEMM thread, slot) -> (token, feature) mapping is
// the one store_tile applies to the GEMM's accumulators.
template <int EPI, typename W>
__global__ __launch_bounds__(256) void gemm_split_reduce_kernel(
    const float* __restrict__ partials, const float* __restrict__ bias0,
    const float* __restrict__ bias1, const int32_t* __restrict__ counts, int E, int e_base, int K,
    int nbx, int n_store, int bias_ld, bf16_t* __restrict__ out, int ldo, int G) {
  constexpr int kPartialFloats = W::kBM * W::kBN;
  constexpr int kTM = W::TM, kT = W::kThreads;
  constexpr bool kGU = EPI == kEpiGateUp;
  // quads per tile: gate/up pairs two slots (gate j, up j+1) into one quad
  constexpr int kQuads = kT * W::TN * kTM * 4 / (kGU ? 2 : 1);
  const int KT = K / 64;
  SegScan<W::kBM> sc;
  sc.init(counts, E, e_base);
  SplitPlan plan;
  plan.init(sc.tm * nbx, G, KT, true);
  if (plan.s == 1) return;
  const int total = plan.rem * kQuads;
  // kQuads is a multiple of 256, so r (and the tile) is uniform per block
  for (int u = blockIdx.x * 256 + threadIdx.x; u < total; u += gridDim.x * 256) {
    const int r = u / kQuads, uq = u % kQuads;
    Tile tile;
    if (!locate_tile<W::kBN>(sc, E, nbx, plan.full + r, &tile)) return;
    const int tid = uq % kT, qq = uq / kT;
    const int w = tid / kWave, lane = tid % kWave;
    const int wn = w % W::WN, wm = w / W::WN, lrow = lane & 31, lhalf = lane >> 5;
    const int g = qq % 4, i = (qq / 4) % kTM, j = qq / (4 * kTM);   // j: column group (pair)
    const int row = tile.row0 + wm * W::WTM + lrow + i * 32;
    if (row >= tile.row_end) continue;
    const float4* P = reinterpret_cast<const float4*>(partials + (size_t)r * plan.s * kPartialFloats) + tid;
    if constexpr (kGU) {
      const int qg = ((2 * j) * kTM + i) * 4 + g, qu = ((2 * j + 1) * kTM + i) * 4 + g;
      float4 ga = make_float4(0.f, 0.f, 0.f, 0.f), ua = ga;
      for (int p = 0; p < plan.s; ++p) {
        const float4 x = P[(size_t)p * (kPartialFloats / 4) + qg * kT];
        const float4 y = P[(size_t)p * (kPartialFloats / 4) + qu * kT];
        ga.x += x.x; ga.y += x.y; ga.z += x.z; ga.w += x.w;
        ua.x += y.x; ua.y += y.y; ua.z += y.z; ua.w += y.w;
      }
      const int hb = (tile.n0 + wn * W::WTN) / 2 + 32 * j;
      const int f = hb + 8 * g + 4 * lhalf;
      const float* bg = bias0 + (size_t)tile.expert * bias_ld + f;
      const float* bu = bias1 + (size_t)tile.expert * bias_ld + f;
      *reinterpret_cast<uint2*>(out + (size_t)row * ldo + f) =
          pack4_bf16(silu_mul_fast(ga.x + bg[0], ua.x + bu[0]),
                     silu_mul_fast(ga.y + bg[1], ua.y + bu[1]),
                     silu_mul_fast(ga.z + bg[2], ua.z + bu[2]),
                     silu_mul_fast(ga.w + bg[3], ua.w + bu[3]));
    } else {
      const int cb = tile.n0 + wn * W::WTN + j * 32;
      if (cb >= n_store) continue;
      const int q = (j * kTM + i) * 4 + g;
      float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
      for (int p = 0; p < plan.s; ++p) {
        const float4 x = P[(size_t)p * (kPartialFloats / 4) + q * kT];
        a.x += x.x; a.y += x.y; a.z += x.z; a.w += x.w;
      }
      const int f = cb + 8 * g + 4 * lhalf;
      float b[4] = {0.0f, 0.0f, 0.0f, 0.0f};
      if (bias0) {
        const float* bp = bias0 + (size_t)tile.expert * bias_ld + f;
        b[0] = bp[0]; b[1] = bp[1]; b[2] = bp[2]; b[3] = bp[3];
      }
      *reinterpret_cast<uint2*>(out + (size_t)row * ldo + f) =
          pack4_bf16(a.x + b[0], a.y + b[1], a.z + b[2], a.w + b[3]);
    }
  }
}

}  // namespace
}  // namespace mgpt
