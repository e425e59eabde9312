// gemm_f32.hip -- fp32 grouped expert products on CDNA4 matrix cores: the
// forward's and the data gradients' C = A . B^T, and the weight gradients'
// D = P^T . Q.
//
// Same contracts as gemm.hip's grouped_gemm_kernel (A = expert-contiguous
// rows [rows][K], B = packed weights [E][Npad][K]) and wgrad.hip's kernels
// (P, Q row-major, contracted over each expert's rows), for fp32.
//
// v_mfma_f32_32x32x2_f32 takes 64 cycles for two operand registers, so the
// operands' paths are wide enough by far, and what bounds these products at
// the engine's own sizes (cfg1: 0.5 GFLOP a product, 128 to 1024 columns) is
// latency and CUs without work; at large ones it is the matrix rate.  So the
// tiles are small, and the four waves of a small tile share its contraction
// (added in wave order: deterministic).
//
// Measured on MI355X against the register-staged 64 x 128 tiles (whose down
// product split K over the CUs for few tokens) and the transposing 256 x 256
// weight-gradient tiles used before, us, stage times with their 2-5 us event
// gap (cfg1 rows: 1024 tokens, C = 128, H = 512, E = 8, k = 2; large: 4096
// tokens, C = 512, H = 2048, E = 8, k = 2, where gate/up reaches 110 of the
// 157 TFLOP/s fp32 peak):
//
//            gate/up      down        d(act)   dX    dW_down  dW_gate/up
//   cfg1   17.4 -> 17.6  15.5 -> 9.3   12.4   14.4    16.4      13.0
//   large   349 -> 314    235 -> 171    208    329     175       334
//
// whole training steps 608 -> 150 us (cfg1, its parameter load included, where 220 of
// the 458 us saved are pack.hip's) and 2680 -> 1810 us.
#include <algorithm>

#include "common.hpp"

namespace mgpt {
namespace {

constexpr int kWT = 64;   // wave tile, both dimensions

// The m-tile of BM rows `mtile` belongs to, found by every wave for itself
// (a scan of the counts 64 experts at a time; no LDS, no barrier).
template <int BM>
__device__ __forceinline__ bool locate_rows(const int32_t* __restrict__ counts, int E, int mtile,
                                            TileInfo* out) {
  const int l = lane_id();
  int rows_carry = 0, tiles_carry = 0;
  for (int e0 = 0; e0 < E; e0 += kWave) {
    const int e = e0 + l;
    const int cnt = e < E ? counts[e] : 0;
    const int tiles = (cnt + BM - 1) / BM;
    const int rows_incl = wave_incl_scan(cnt) + rows_carry;
    const int tiles_incl = wave_incl_scan(tiles) + tiles_carry;
    const unsigned long long m = __ballot(mtile >= tiles_incl - tiles && mtile < tiles_incl);
    if (m) {
      const int owner = __ffsll((long long)m) - 1;
      out->expert = e0 + owner;
      out->row0 = __builtin_amdgcn_readlane(rows_incl - cnt + (mtile - tiles_incl + tiles) * BM, owner);
      out->row_end = __builtin_amdgcn_readlane(rows_incl, owner);
      return true;
    }
    rows_carry = __builtin_amdgcn_readlane(rows_incl, kWave - 1);
    tiles_carry = __builtin_amdgcn_readlane(tiles_incl, kWave - 1);
  }
  return false;
}

// Rows of the experts before e, and e's own.
__device__ __forceinline__ void locate_expert(const int32_t* __restrict__ counts, int e, int* seg0,
                                              int* cnt) {
  int before = 0;
  for (int i = lane_id(); i < e; i += kWave) before += counts[i];
  *seg0 = __builtin_amdgcn_readfirstlane(wave_sum(before));
  *cnt = counts[e];
}

// One tile row (TN tiles) of the four waves of a KS = 4 block added in wave
// order: wave w ends with registers 4w .. 4w+3 of every tile.  Ends with all
// writes done but other waves perhaps still reading.
template <int TN>
__device__ __forceinline__ void add_waves(const f32x16 (&acc)[TN], float4* red, int w, int lane,
                                          float (&sum)[TN][4]) {
#pragma unroll
  for (int j = 0; j < TN; ++j)
#pragma unroll
    for (int q = 0; q < 4; ++q)   // [wave][tile, register quad][lane]
      red[(w * TN * 4 + j * 4 + q) * kWave + lane] =
          make_float4(acc[j][4 * q], acc[j][4 * q + 1], acc[j][4 * q + 2], acc[j][4 * q + 3]);
  __syncthreads();
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    float4 s = red[(j * 4 + w) * kWave + lane];
#pragma unroll
    for (int p = 1; p < 4; ++p) {
      const float4 x = red[(p * TN * 4 + j * 4 + w) * kWave + lane];
      s.x += x.x; s.y += x.y; s.z += x.z; s.w += x.w;
    }
    sum[j][0] = s.x;
    sum[j][1] = s.y;
    sum[j][2] = s.z;
    sum[j][3] = s.w;
  }
}

struct GemmArgs {
  const float *A, *B, *bias0, *bias1;
  const int32_t* counts;
  int E, K, Npad, n_store, bias_ld;
  float* out;
  int ldo;
  float* aux;
  int aux_ld;
};

// Epilogue of registers 4*vb .. 4*vb + NV - 1 of the TN MFMA tiles (columns n
// + 32j ..) of one 32-row tile.  Register v of a tile holds row 8*(v/4) +
// 4*(lane/32) + v%4 and column lane%32.
template <int EPI, int TN, int NV>
__device__ __forceinline__ void emit(const GemmArgs& g, int e, int row_t, int row_end, int n,
                                     int lrow, int lhalf, int vb, const float (&d)[TN][NV]) {
  auto row_of = [&](int v) { return row_t + 8 * (vb + v / 4) + 4 * lhalf + (v % 4); };
  if constexpr (EPI == kEpiGateUp) {
    static_assert(EPI != kEpiGateUp || TN == 2, "a gate and an up tile");
    const int hcol = n / 2 + lrow, prow = n + lrow;
    const float bg = g.bias0[(size_t)e * g.bias_ld + hcol];
    const float bu = g.bias1[(size_t)e * g.bias_ld + hcol];
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const int row = row_of(v);
      if (row >= row_end) continue;
      const float gv = d[0][v] + bg, uv = d[TN - 1][v] + bu;
      g.out[(size_t)row * g.ldo + hcol] = (gv / (1.0f + expf(-gv))) * uv;
      if (g.aux) {
        g.aux[(size_t)row * g.aux_ld + prow] = gv;
        g.aux[(size_t)row * g.aux_ld + prow + 32] = uv;
      }
    }
  } else {
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int col = n + 32 * j + lrow;
      const float b = EPI == kEpiDown && g.bias0 ? g.bias0[(size_t)e * g.bias_ld + col] : 0.0f;
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        const int row = row_of(v);
        if (row >= row_end) continue;
        if constexpr (EPI == kEpiDown) {
          g.out[(size_t)row * g.ldo + col] = d[j][v] + b;
        } else {
          const int pc = packed_gate_col(col);
          const float gv = g.aux[(size_t)row * g.aux_ld + pc];
          const float uv = g.aux[(size_t)row * g.aux_ld + pc + 32];
          const float sig = 1.0f / (1.0f + expf(-gv));
          g.out[(size_t)row * g.ldo + pc] = (d[j][v] * uv) * (sig * (1.0f + gv * (1.0f - sig)));
          g.out[(size_t)row * g.ldo + pc + 32] = d[j][v] * (gv * sig);
        }
      }
    }
  }
}

typedef __attribute__((address_space(3))) char lds_char;

// One 1 KB direct-to-LDS load (lane l's 16 bytes land at lds + 16*l).  The
// compiler does not track it: the kernel waits itself.
__device__ __forceinline__ void dma16(const void* g, uint32_t lds) {
  asm volatile("global_load_lds_dwordx4 %0, off" ::"v"(g), "{m0}"(lds) : "memory");
}

// All but this wave's newest N loads have landed and its LDS reads are done;
// then meet the other waves.
template <int N>
__device__ __forceinline__ void wait_barrier() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

// Block tile BM x BN by four waves: WM x WN of them each with a tile of its
// own or, with WM * WN = 1, all four on the block's one tile, each taking a
// quarter of every slab's columns (the parts are added in wave order through
// LDS at the end: deterministic).
//
// Operands go straight into an LDS ring of ST slabs (32 columns: 128-byte
// rows, the A rows and then the B rows; 16-byte chunk c of row r at slot
// c ^ ((r >> 1) & 7), so that the 16 lanes served together hit distinct
// banks), ST - 1 slabs ahead.  A lane reads its row's columns 8q + 4h .. +3
// (h its half) as one 16-byte vector for four k-steps, k-step x pairing
// column 8q + x with 8q + 4 + x in both operands.  A slab is 4096 cycles of
// MFMAs for a 64 x 64 wave tile, so one barrier a slab and 16 bytes a cycle
// and CU of LDS reads leave the matrix rate as the bound of large products;
// small ones are latency (launch, counts, the first slabs) and what CUs they
// reach.
// Rows past the segment read the slack after it; past the last slab the loads
// repeat it (in bounds, into a slab that is no longer read).
template <int EPI, int BM, int BN, int WM, int WN, int ST>
__global__ __launch_bounds__(256) void gemm_f32_kernel(GemmArgs g) {
  constexpr bool kSplit = WM * WN == 1;
  static_assert(kSplit || WM * WN == 4, "4 waves");
  constexpr int TM = BM / WM / 32, TN = BN / WN / 32;
  static_assert(EPI != kEpiGateUp || TN == 2, "gate/up pairs");
  constexpr int kSlab = (BM + BN) * 128;
  constexpr int D = kSlab / 1024 / 4;   // loads per wave and slab
  constexpr int kRed = kSplit ? 4 * TN * 4 * kWave * 16 : 0;
  __shared__ __attribute__((aligned(1024))) char smem[ST * kSlab > kRed ? ST * kSlab : kRed];
  // each XCD (own L2) takes a contiguous run of tiles, n fastest (the
  // hardware deals workgroups round-robin to the XCDs)
  const int nbx = gridDim.x, total = nbx * gridDim.y;
  int bid = blockIdx.y * nbx + blockIdx.x;
  const int per = total / kNumXcd;
  if (bid < per * kNumXcd) bid = (bid % kNumXcd) * per + bid / kNumXcd;
  TileInfo ti;
  if (!locate_rows<BM>(g.counts, g.E, bid / nbx, &ti)) return;
  const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave), lane = lane_id();
  const int lrow = lane & 31, lhalf = lane >> 5;
  const int wm = kSplit ? 0 : w / WN, wn = kSplit ? 0 : w % WN;
  const int K = g.K, KT = K / 32, n0 = (bid % nbx) * BN;

  // this wave's D groups of 8 rows; lane l loads chunk (l % 8) ^ ((r >> 1) & 7)
  // of row r = l / 8 of the group into slot l % 8
  const char* src[D];
#pragma unroll
  for (int i = 0; i < D; ++i) {
    const int r = (w * D + i) * 8 + lane / 8;
    const float* row = r < BM ? g.A + (size_t)(ti.row0 + r) * K
                              : g.B + ((size_t)ti.expert * g.Npad + n0 + (r - BM)) * K;
    src[i] = reinterpret_cast<const char*>(row) + (((lane % 8) ^ ((r >> 1) & 7)) << 4);
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_char*)smem + (uint32_t)(w * D * 1024);
  auto issue = [&](int kt) __attribute__((always_inline)) {
    const uint32_t dst = lds0 + (uint32_t)(kt % ST * kSlab);
    const size_t off = (size_t)min(kt, KT - 1) * 128;
#pragma unroll
    for (int i = 0; i < D; ++i) dma16(src[i] + off, dst + i * 1024);
  };

  f32x16 acc[TM][TN];
#pragma unroll
  for (int t = 0; t < TM * TN; ++t)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[t / TN][t % TN][v] = 0.0f;
  const int swz = (lrow >> 1) & 7;
  auto frags = [&](const char* sl, int q, f32x4 (&a)[TM], f32x4 (&b)[TN]) __attribute__((always_inline)) {
    const int ofs = lrow * 128 + (((2 * q + lhalf) ^ swz) << 4);
#pragma unroll
    for (int i = 0; i < TM; ++i)
      a[i] = *reinterpret_cast<const f32x4*>(sl + (wm * TM + i) * 32 * 128 + ofs);
#pragma unroll
    for (int j = 0; j < TN; ++j)
      b[j] = *reinterpret_cast<const f32x4*>(sl + (BM + (wn * TN + j) * 32) * 128 + ofs);
  };
  auto mfmas = [&](const f32x4 (&a)[TM], const f32x4 (&b)[TN]) __attribute__((always_inline)) {
#pragma unroll
    for (int x = 0; x < 4; ++x)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i][x], b[j][x], acc[i][j], 0, 0, 0);
  };

#pragma unroll
  for (int s = 0; s < ST - 1; ++s) issue(s);
  for (int kt = 0; kt < KT; ++kt) {
    wait_barrier<(ST - 2) * D>();   // slab kt is there, and slab kt - 1 read by all
    issue(kt + ST - 1);
    const char* sl = smem + kt % ST * kSlab;
    if constexpr (kSplit) {
      f32x4 a[TM], b[TN];
      frags(sl, w, a, b);
      mfmas(a, b);
    } else {
      f32x4 a[2][TM], b[2][TN];
      frags(sl, 0, a[0], b[0]);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        if (q < 3) frags(sl, q + 1, a[(q + 1) & 1], b[(q + 1) & 1]);
        mfmas(a[q & 1], b[q & 1]);
      }
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the repeated tail loads

  const int row_w = ti.row0 + wm * TM * 32, n_w = n0 + wn * TN * 32;
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    if constexpr (kSplit) {
      float sum[TN][4];
      __syncthreads();   // every wave is done with the ring (and the last tile row's sums)
      add_waves<TN>(acc[i], reinterpret_cast<float4*>(smem), w, lane, sum);
      emit<EPI, TN, 4>(g, ti.expert, row_w + 32 * i, ti.row_end, n_w, lrow, lhalf, w, sum);
    } else {
      float d[TN][16];
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) d[j][v] = acc[i][j][v];
      if (EPI == kEpiGateUp || n_w < g.n_store)   // n_store is a multiple of 64
        emit<EPI, TN, 16>(g, ti.expert, row_w + 32 * i, ti.row_end, n_w, lrow, lhalf, 0, d);
    }
  }
}

struct WgArgs {
  const float *P, *Q;
  int ldp, p_valid, ldq, q_valid;
  const int32_t* counts;
  float *out0, *out1;
  int ldo;
  size_t out_estride;
  int i_store, j_store;
  float *bias0, *bias1;
  size_t bias_estride;
  int Iy, Jx, store;
};

// Registers 4*vb .. 4*vb+NV-1 of tile row ti for both column tiles: D rows
// i = i0 + 2 * m + ti (m the MFMA row) and columns 2 * lrow, 2 * lrow + 1 of
// the 64-column tile, added to the gradient or stored.
template <int MODE, int NV>
__device__ __forceinline__ void wg_emit(const WgArgs& g, int e, int i0, int ti, int j0, int lrow,
                                        int lhalf, int vb, const float (&d)[2][NV]) {
  const int j = j0 + 2 * lrow;
  float* ob = g.out0;
  int col = j;
  if constexpr (MODE == 1) {   // 32 gate columns, then the 32 up ones
    ob = ((j >> 5) & 1) ? g.out1 : g.out0;
    col = (j >> 6) * 32 + (j & 31);
  }
  if (col >= g.j_store) return;
  const bool two = col + 1 < g.j_store;
  ob += (size_t)e * g.out_estride + col;
  const bool vec = two && (g.ldo & 1) == 0 && (reinterpret_cast<uintptr_t>(ob) & 7) == 0;
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    const int i = i0 + 2 * (8 * (vb + v / 4) + 4 * lhalf + (v % 4)) + ti;
    if (i >= g.i_store) continue;
    float* o = ob + (size_t)i * g.ldo;
    float2 r = make_float2(d[0][v], d[1][v]);
    if (vec) {
      if (!g.store) {
        const float2 old = *reinterpret_cast<const float2*>(o);
        r.x = old.x + r.x;
        r.y = old.y + r.y;
      }
      *reinterpret_cast<float2*>(o) = r;
    } else {
      o[0] = g.store ? r.x : o[0] + r.x;
      if (two) o[1] = g.store ? r.y : o[1] + r.y;
    }
  }
}

// D_e = P_e^T . Q_e: the contraction runs over rows, and an fp32 MFMA operand
// is one value per lane (feature lane%32 of row lane/32 of the pair), so
// row-major operands feed it as they are.  A lane loads two neighbouring
// columns of its row (8 bytes, 256 bytes a row and half-wave): the even
// columns make fragment 0, the odd ones fragment 1.  A wave step is 16 rows
// (16 loads, 32 MFMAs); the next step's loads are in flight meanwhile.
// Grid: (column tiles, row tiles, experts); an expert's blocks leave at once
// when it has no rows.  The blocks of the first row tile also sum Q's
// columns for the bias gradient.
template <int MODE, int KS>
__global__ __launch_bounds__(256, 2) void wgrad_f32_kernel(WgArgs g) {
  constexpr int WB = KS == 4 ? 1 : 2;
  __shared__ float4 red[KS == 4 ? 4 * 8 * kWave : 1];
  const int e = blockIdx.z;
  int seg0, cnt;
  locate_expert(g.counts, e, &seg0, &cnt);
  if (cnt <= 0) return;
  const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave), lane = lane_id();
  const int lrow = lane & 31, lhalf = lane >> 5;
  const int kw = KS == 4 ? w : 0;
  const int ty = blockIdx.y * WB + (KS == 4 ? 0 : w >> 1), tx = blockIdx.x * WB + (KS == 4 ? 0 : w & 1);
  if (KS == 1 && (ty >= g.Iy || tx >= g.Jx)) return;
  const int i0 = ty * kWT, j0 = tx * kWT;
  // (columns past the operand's read its last pair; they are not stored)
  const float* pp = g.P + (size_t)seg0 * g.ldp + min(i0 + 2 * lrow, g.p_valid - 2);
  const float* pq = g.Q + (size_t)seg0 * g.ldq + min(j0 + 2 * lrow, g.q_valid - 2);
  const bool do_bias = ty == 0 && g.bias0 != nullptr;

  f32x16 acc[2][2];
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[t / 2][t % 2][v] = 0.0f;
  float bs0 = 0.0f, bs1 = 0.0f;
  auto load = [&](int s, float2 (&fp)[8], float2 (&fq)[8]) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int r = min(16 * s + 2 * u + lhalf, cnt - 1);
      fp[u] = *reinterpret_cast<const float2*>(pp + (size_t)r * g.ldp);
      fq[u] = *reinterpret_cast<const float2*>(pq + (size_t)r * g.ldq);
    }
  };
  // rows past the expert's last one count as zeros (in both operands)
  auto mfmas = [&](int s, const float2 (&fp)[8], const float2 (&fq)[8])
      __attribute__((always_inline)) {
    const int live = cnt - 16 * s - lhalf;
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const bool ok = 2 * u < live;
      const float p0 = ok ? fp[u].x : 0.0f, p1 = ok ? fp[u].y : 0.0f;
      const float q0 = ok ? fq[u].x : 0.0f, q1 = ok ? fq[u].y : 0.0f;
      acc[0][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(p0, q0, acc[0][0], 0, 0, 0);
      acc[0][1] = __builtin_amdgcn_mfma_f32_32x32x2f32(p0, q1, acc[0][1], 0, 0, 0);
      acc[1][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(p1, q0, acc[1][0], 0, 0, 0);
      acc[1][1] = __builtin_amdgcn_mfma_f32_32x32x2f32(p1, q1, acc[1][1], 0, 0, 0);
      if (do_bias) {
        bs0 += q0;
        bs1 += q1;
      }
    }
  };
  const int KC = (cnt + 15) / 16;
  float2 p0[8], q0[8], p1[8], q1[8];
  const int steps = kw < KC ? (KC - kw + KS - 1) / KS : 0;
  if (steps > 0) load(kw, p0, q0);
  for (int s = 0; s + 1 < steps; s += 2) {
    const int c = kw + s * KS;
    load(c + KS, p1, q1);
    __builtin_amdgcn_sched_barrier(0);
    mfmas(c, p0, q0);
    __builtin_amdgcn_sched_barrier(0);
    load(kw + min(s + 2, steps - 1) * KS, p0, q0);
    __builtin_amdgcn_sched_barrier(0);
    mfmas(c + KS, p1, q1);
    __builtin_amdgcn_sched_barrier(0);
  }
  if (steps & 1) mfmas(kw + (steps - 1) * KS, p0, q0);

#pragma unroll
  for (int ti = 0; ti < 2; ++ti) {
    if constexpr (KS == 4) {
      float sum[2][4];
      if (ti) __syncthreads();
      add_waves<2>(acc[ti], red, w, lane, sum);
      wg_emit<MODE, 4>(g, e, i0, ti, j0, lrow, lhalf, w, sum);
    } else {
      float d[2][16];
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) d[j][v] = acc[ti][j][v];
      wg_emit<MODE, 16>(g, e, i0, ti, j0, lrow, lhalf, 0, d);
    }
  }
  if (!do_bias) return;   // uniform per wave, and per block when KS = 4
  bs0 += __shfl_xor(bs0, 32, kWave);
  bs1 += __shfl_xor(bs1, 32, kWave);
  if constexpr (KS == 4) {
    float* rb = reinterpret_cast<float*>(red);
    __syncthreads();   // every wave has read the sums
    if (lhalf == 0) {
      rb[w * 64 + 2 * lrow] = bs0;
      rb[w * 64 + 2 * lrow + 1] = bs1;
    }
    __syncthreads();
    if (w != 0) return;
    bs0 = ((rb[2 * lrow] + rb[64 + 2 * lrow]) + rb[128 + 2 * lrow]) + rb[192 + 2 * lrow];
    bs1 = ((rb[2 * lrow + 1] + rb[65 + 2 * lrow]) + rb[129 + 2 * lrow]) + rb[193 + 2 * lrow];
  }
  if (lhalf != 0) return;
  const int j = j0 + 2 * lrow;
  float* bb = g.bias0;
  int col = j;
  if constexpr (MODE == 1) {
    bb = ((j >> 5) & 1) ? g.bias1 : g.bias0;
    col = (j >> 6) * 32 + (j & 31);
  }
  bb += (size_t)e * g.bias_estride + col;
  if (col < g.j_store) bb[0] = g.store ? bs0 : bb[0] + bs0;
  if (col + 1 < g.j_store) bb[1] = g.store ? bs1 : bb[1] + bs1;
}

}  // namespace

// C = A . B^T with the epilogues of gemm.hip over `rows` rows in E segments
// (K % 64 == 0, Npad % 128 == 0, n_store % 64 == 0; A has at least 128 rows
// of slack).  The tile: smaller ones win until there are many per CU, then
// the operand traffic of small tiles does not fit L2 (t = 64 x 128 tiles per
// CU; us for 64 x 128 / 32 x 64 / 32 x 32): gate/up t = 2: 61 / 54, t = 5.5:
// 77 / 82, t = 16: 314 / 362; down t = 2: 208 / 169 / 168, t = 4: 473 / 454 /
// 500, t = 16: 2661 / 2941 / 3091; d(act) t = 2.7: 67 / 51 / 50, t = 8: 244 /
// 208 / 217, t = 11: 498 / 512 / 554.
template <int EPI>
hipError_t launch_gemm_f32(const float* A, const float* B, const float* bias0, const float* bias1,
                           const int32_t* counts, int E, int K, int Npad, int n_store, int bias_ld,
                           float* out, int ldo, size_t rows, float* aux, int aux_ld, int num_cus,
                           hipStream_t stream) {
  if (rows == 0) return hipSuccess;
  if (E <= 0 || E > kMaxExpertsWide || K % 64 || Npad % 128 || n_store % 64 ||
      (EPI == kEpiSwigluBwd && !aux))
    return hipErrorInvalidValue;
  const GemmArgs g = {A, B, bias0, bias1, counts, E, K, Npad, n_store, bias_ld, out, ldo, aux, aux_ld};
  const int cols = EPI == kEpiGateUp ? Npad : n_store;
  // tiles of TM x TN MFMA tiles over the rows (without the surplus of ragged
  // segments) and columns
  auto tiles = [&](int wm, int wn) { return (long)((rows + wm - 1) / wm) * ((cols + wn - 1) / wn); };
  auto launch = [&](auto kernel, int wm, int wn) {
    hipLaunchKernelGGL(kernel, dim3((cols + wn - 1) / wn, (unsigned)((rows + wm - 1) / wm + E)),
                       dim3(256), 0, stream, g);
  };
  const long t = tiles(64, 128);
  if (t >= (EPI == kEpiGateUp ? 4L : 10L) * num_cus)
    launch(gemm_f32_kernel<EPI, 64, 128, 2, 2, 3>, 64, 128);
  else if (EPI == kEpiGateUp || t >= 3L * num_cus)
    launch(gemm_f32_kernel<EPI, 32, 64, 1, 1, 3>, 32, 64);
  else if constexpr (EPI != kEpiGateUp)
    launch(gemm_f32_kernel<EPI, 32, 32, 1, 1, 4>, 32, 32);
  return hipGetLastError();
}

// launch_wgrad's product for fp32 (see wgrad.hip).  A tile a wave only from
// six 128 x 128 blocks per CU on (us for KS = 1 / 4 at t blocks per CU: t = 2:
// 183 / 175, t = 5.5: 501 / 500, t = 11: 910 / 977, t = 16: 2934 / 3109).
template <int MODE>
hipError_t launch_wgrad_f32(const float* P, int ldp, int p_valid, const float* Q, int ldq,
                            int q_valid, const int32_t* counts, int E, float* out0, float* out1,
                            int ldo, size_t out_estride, int i_store, int j_store, float* bias0,
                            float* bias1, size_t bias_estride, int num_cus, bool store,
                            hipStream_t stream) {
  if (E <= 0 || E > kMaxExpertsWide || p_valid < 2 || q_valid < 2 || p_valid % 2 || q_valid % 2 ||
      ldp % 2 || ldq % 2 || ((reinterpret_cast<uintptr_t>(P) | reinterpret_cast<uintptr_t>(Q)) & 7))
    return hipErrorInvalidValue;
  if (i_store <= 0) return hipSuccess;
  const int Iy = (i_store + kWT - 1) / kWT, Jx = (q_valid + kWT - 1) / kWT;
  const WgArgs g = {P,       Q,       ldp,   p_valid, ldq,          q_valid, counts, out0, out1, ldo,
                    out_estride, i_store, j_store, bias0, bias1, bias_estride, Iy, Jx, (int)store};
  const int by = (Iy + 1) / 2, bx = (Jx + 1) / 2;
  if ((long)by * bx * E >= 6L * num_cus)
    hipLaunchKernelGGL((wgrad_f32_kernel<MODE, 1>), dim3(bx, by, E), dim3(256), 0, stream, g);
  else
    hipLaunchKernelGGL((wgrad_f32_kernel<MODE, 4>), dim3(Jx, Iy, E), dim3(256), 0, stream, g);
  return hipGetLastError();
}

#define MGPT_INST_F32(EPI)                                                                       \
  template hipError_t launch_gemm_f32<EPI>(const float*, const float*, const float*, const float*, \
                                           const int32_t*, int, int, int, int, int, float*, int,   \
                                           size_t, float*, int, int, hipStream_t);
MGPT_INST_F32(kEpiGateUp)
MGPT_INST_F32(kEpiDown)
MGPT_INST_F32(kEpiSwigluBwd)
#define MGPT_INST_WG32(MODE)                                                                       \
  template hipError_t launch_wgrad_f32<MODE>(const float*, int, int, const float*, int, int,       \
                                             const int32_t*, int, float*, float*, int, size_t, int, \
                                             int, float*, float*, size_t, int, bool, hipStream_t);
MGPT_INST_WG32(0)
MGPT_INST_WG32(1)

}  // namespace mgpt
