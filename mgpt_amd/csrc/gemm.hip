// gemm.hip -- grouped bf16 expert GEMMs with register-staged 128 x 128 tiles,
// the alternative to gemm_dma.hip's 256 x 256 ones for large segments that
// MGPT_MOE_GEMM_TILE=128 selects.
//
// Reference: per expert e with count_e > 0, SwiGLU::forward_into
// (layers/SwiGLU.cpp:23-50): g = X_e W_g + b_g, u = X_e W_u + b_u,
// h = silu(g) * u (utils/Tensor.cpp:1986-2004), y_e = h W_d + b_d, run by a
// host loop over experts (layers/MoELayer.cpp:94-118).  Here each product is
// one launch over all experts: the rows of X are expert-contiguous segments
// (dispatch.hip), the grid covers an upper bound of m-tiles, and each block
// finds its expert from the device-side counts (common.hpp find_tile).
//
// Operands: A = activations [rows][K] (bf16, K contiguous);
// B = packed weights [E][Npad][K] (K contiguous, so both MFMA operands are
// read as 16-byte K-runs); C = A . B^T.  Tiles: block BM x BN x BK with 4
// waves in a WM x WN grid; each wave owns (BM/WM) x (BN/WN) made of 32x32
// MFMA tiles: v_mfma_f32_32x32x16_bf16.  Global -> register -> LDS double buffering: the next K-slab is
// fetched while the current one feeds the MFMAs; one barrier per slab.
//
// Epilogues: GATEUP (B rows interleaved in 64-row groups [32 gate | 32 up]
// for the same 32 hidden units, so a wave's two adjacent 32x32 tiles hold
// g and u of the same (row, h) in the same lane) computes
// h = silu(g + b_g) * (u + b_u) and stores bf16 h, and, when
// `aux` is given, also the pre-activations g, u in the interleaved layout
// (aux[row][packed column], the caches of layers/SwiGLU.cpp:30-31 that the
// backward pass reads);
// DOWN stores o = acc + b_d in the activation dtype (no bias if bias0 is
// null);
// SWIGLU_BWD treats the product as d(act)[row][h] and applies the CPU
// swiglu_backward of utils/Tensor.cpp:2006-2030 with the saved g, u read
// from aux: sig = 1/(1+exp(-g)), d_up = d*(g*sig),
// d_gate = (d*u)*(sig*(1+g*(1-sig))), written to out in the interleaved
// layout (out may equal aux: each element is read before it is written by
// the same thread).
#include <algorithm>
#include <type_traits>

#include "common.hpp"

namespace mgpt {

namespace {

constexpr int kSlab = 64;   // K columns per slab

struct alignas(16) U4 {
  uint32_t x, y, z, w;
};
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

template <int BM, int BN, int WM, int WN, int EPI>
__global__ __launch_bounds__(256) void grouped_gemm_kernel(
    const bf16_t* __restrict__ A, const bf16_t* __restrict__ B, const float* __restrict__ bias0, const float* __restrict__ bias1,
    const int32_t* __restrict__ counts, int E, int K, int Npad, int n_store, int bias_ld,
    bf16_t* out, int ldo, bf16_t* aux, int aux_ld) {
  constexpr int BK = kSlab;
  constexpr int PAD = 16 / 2;
  constexpr int LDK = BK + PAD;
  constexpr int WTM = BM / WM, WTN = BN / WN;
  constexpr int TM = WTM / 32, TN = WTN / 32;
  static_assert(WM * WN == 4, "4 waves");
  static_assert(TM >= 1 && TN >= 1, "wave tile >= 32x32");
  static_assert(EPI != kEpiGateUp || (TN % 2 == 0), "gate/up pairs");
  // 16-byte chunks per K-slab row, and per-thread chunk counts.
  constexpr int A_CPR = BK * 2 / 16;             // 8
  constexpr int B_CPR = BK * 2 / 16;             // 8
  constexpr int A_CH = BM * A_CPR / 256;
  constexpr int B_CH = BN * B_CPR / 256;
  static_assert(A_CH >= 1 && B_CH >= 1, "tile too small for 256 threads");

  __shared__ __attribute__((aligned(16))) bf16_t sA[2][BM][LDK];
  __shared__ __attribute__((aligned(16))) bf16_t sB[2][BN][LDK];

  // XCD-aware order: the hardware deals consecutive workgroups round-robin
  // to the 8 XCDs (each with its own L2); remap so each XCD receives a
  // contiguous run of tiles, n fastest, so concurrently resident blocks on
  // one XCD share their A (activation) tile and neighbouring B tiles.
  const int nbx = gridDim.x;
  const int total = nbx * gridDim.y;
  int bid = blockIdx.y * nbx + blockIdx.x;
  const int per = total / kNumXcd;
  if (bid < per * kNumXcd) bid = (bid % kNumXcd) * per + bid / kNumXcd;
  const int mtile = bid / nbx;
  TileInfo ti;
  if (!find_tile<BM>(counts, E, mtile, &ti)) return;
  const int e = ti.expert;
  const int n0 = (bid % nbx) * BN;
  const int tid = threadIdx.x;
  const int w = tid / kWave, lane = lane_id();
  const int wm = w / WN, wn = w % WN;

  const bf16_t* Ablk = A + (size_t)ti.row0 * K;
  const bf16_t* Bblk = B + ((size_t)e * Npad + n0) * K;

  U4 ra[A_CH], rb[B_CH];
  auto gload = [&](int kt) __attribute__((always_inline)) {
    const char* abase = reinterpret_cast<const char*>(Ablk + (size_t)kt * BK);
    const char* bbase = reinterpret_cast<const char*>(Bblk + (size_t)kt * BK);
#pragma unroll
    for (int i = 0; i < A_CH; ++i) {
      const int q = tid + 256 * i;
      const int r = q / A_CPR, c = q % A_CPR;
      const u32x4 v = *reinterpret_cast<const u32x4*>(abase + (size_t)r * K * 2 + c * 16);
      ra[i].x = v.x; ra[i].y = v.y; ra[i].z = v.z; ra[i].w = v.w;
    }
#pragma unroll
    for (int i = 0; i < B_CH; ++i) {
      const int q = tid + 256 * i;
      const int r = q / B_CPR, c = q % B_CPR;
      const u32x4 v = *reinterpret_cast<const u32x4*>(bbase + (size_t)r * K * 2 + c * 16);
      rb[i].x = v.x; rb[i].y = v.y; rb[i].z = v.z; rb[i].w = v.w;
    }
  };
  auto sstore = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < A_CH; ++i) {
      const int q = tid + 256 * i;
      const int r = q / A_CPR, c = q % A_CPR;
      *reinterpret_cast<U4*>(reinterpret_cast<char*>(&sA[buf][r][0]) + c * 16) = ra[i];
    }
#pragma unroll
    for (int i = 0; i < B_CH; ++i) {
      const int q = tid + 256 * i;
      const int r = q / B_CPR, c = q % B_CPR;
      *reinterpret_cast<U4*>(reinterpret_cast<char*>(&sB[buf][r][0]) + c * 16) = rb[i];
    }
  };

  f32x16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;

  const int KT = K / BK;
  gload(0);
  sstore(0);
  __syncthreads();
  const int lrow = lane & 31, lhalf = lane >> 5;
  for (int kt = 0; kt < KT; ++kt) {
    const int cur = kt & 1;
    if (kt + 1 < KT) gload(kt + 1);
    {
      // Fragments of k-step ks+1 are read from LDS while the MFMAs of
      // k-step ks run.
      constexpr int KS = BK / 16;
      bf16x8 af[2][TM], bfr[2][TN];
      auto lds_frags = [&](int ks, bf16x8 (&a)[TM], bf16x8 (&b)[TN]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
          a[i] = *reinterpret_cast<const bf16x8*>(
              &sA[cur][wm * WTM + i * 32 + lrow][ks * 16 + lhalf * 8]);
#pragma unroll
        for (int j = 0; j < TN; ++j)
          b[j] = *reinterpret_cast<const bf16x8*>(
              &sB[cur][wn * WTN + j * 32 + lrow][ks * 16 + lhalf * 8]);
      };
      lds_frags(0, af[0], bfr[0]);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        if (ks + 1 < KS) lds_frags(ks + 1, af[(ks + 1) & 1], bfr[(ks + 1) & 1]);
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[ks & 1][i], bfr[ks & 1][j],
                                                                acc[i][j], 0, 0, 0);
      }
    }
    if (kt + 1 < KT) sstore(cur ^ 1);
    __syncthreads();
  }

  // Epilogue.  Accumulator register v of a 32x32 tile holds row
  // 8*(v/4) + 4*(lane/32) + v%4 and column lane%32.
  const int row_base = ti.row0 + wm * WTM;
  if constexpr (EPI == kEpiGateUp) {
#pragma unroll
    for (int q = 0; q < TN / 2; ++q) {
      const int prow = n0 + wn * WTN + q * 64 + lrow;   // packed row of the gate column
      const int hcol = (n0 + wn * WTN) / 2 + q * 32 + lrow;
      const float bg = bias0[(size_t)e * bias_ld + hcol];
      const float bu = bias1[(size_t)e * bias_ld + hcol];
#pragma unroll
      for (int i = 0; i < TM; ++i) {
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int row = row_base + i * 32 + 8 * (v / 4) + 4 * lhalf + (v % 4);
          if (row < ti.row_end) {
            float g = acc[i][2 * q][v];
            float u = acc[i][2 * q + 1][v];
            g = g + bg;
            u = u + bu;
            const float ex = __expf(-g);
            const float hv = (g / (1.0f + ex)) * u;
            store_act(out + (size_t)row * ldo + hcol, hv);
            if (aux) {
              store_act(aux + (size_t)row * aux_ld + prow, g);
              store_act(aux + (size_t)row * aux_ld + prow + 32, u);
            }
          }
        }
      }
    }
  } else if constexpr (EPI == kEpiSwigluBwd) {
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int h = n0 + wn * WTN + j * 32 + lrow;
      if (h >= n_store) continue;
      const int pc = packed_gate_col(h);
#pragma unroll
      for (int i = 0; i < TM; ++i) {
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int row = row_base + i * 32 + 8 * (v / 4) + 4 * lhalf + (v % 4);
          if (row < ti.row_end) {
            const float d = acc[i][j][v];
            const float g = to_f32(aux[(size_t)row * aux_ld + pc]);
            const float u = to_f32(aux[(size_t)row * aux_ld + pc + 32]);
            const float ex = __expf(-g);
            const float sig = 1.0f / (1.0f + ex);
            const float d_up = d * (g * sig);
            const float d_gate = (d * u) * (sig * (1.0f + g * (1.0f - sig)));
            store_act(out + (size_t)row * ldo + pc, d_gate);
            store_act(out + (size_t)row * ldo + pc + 32, d_up);
          }
        }
      }
    }
  } else {
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int col = n0 + wn * WTN + j * 32 + lrow;
      if (col >= n_store) continue;
      const float b = bias0 ? bias0[(size_t)e * bias_ld + col] : 0.0f;
#pragma unroll
      for (int i = 0; i < TM; ++i) {
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int row = row_base + i * 32 + 8 * (v / 4) + 4 * lhalf + (v % 4);
          if (row < ti.row_end) {
            store_act(out + (size_t)row * ldo + col, acc[i][j][v] + b);
          }
        }
      }
    }
  }
}

}  // namespace

// Host launcher.  max_mtiles must bound sum_e ceil(count_e / BM) (the
// caller uses ceil(A / BM) + E); surplus blocks exit after find_tile.
// aux / aux_ld: the pre-activation save of GATEUP (null: none) or the saved
// pre-activations SWIGLU_BWD reads (required).
// DOWN and SWIGLU_BWD cover only the n-tiles that hold stored columns
// (n_store; Npad is the weights' row stride).
template <int BM, int BN, int WM, int WN, int EPI>
hipError_t launch_grouped_gemm(const bf16_t* A, const bf16_t* B, const float* bias0,
                               const float* bias1, const int32_t* counts, int E, int K, int Npad,
                               int n_store, int bias_ld, bf16_t* out, int ldo, int max_mtiles,
                               bf16_t* aux, int aux_ld, hipStream_t stream) {
  if (max_mtiles <= 0) return hipSuccess;
  if (EPI == kEpiSwigluBwd && aux == nullptr) return hipErrorInvalidValue;
  const int ntiles = EPI == kEpiGateUp ? Npad / BN : std::min(Npad / BN, (n_store + BN - 1) / BN);
  hipLaunchKernelGGL((grouped_gemm_kernel<BM, BN, WM, WN, EPI>),
                     dim3(ntiles, max_mtiles), dim3(256), 0, stream, A, B, bias0, bias1,
                     counts, E, K, Npad, n_store, bias_ld, out, ldo, aux, aux_ld);
  return hipGetLastError();
}

#define MGPT_INST_GEMM(EPI)                                                                  \
  template hipError_t launch_grouped_gemm<128, 128, 2, 2, EPI>(                              \
      const bf16_t*, const bf16_t*, const float*, const float*, const int32_t*, int, int, int, \
      int, int, bf16_t*, int, int, bf16_t*, int, hipStream_t);
MGPT_INST_GEMM(kEpiGateUp)
MGPT_INST_GEMM(kEpiDown)
MGPT_INST_GEMM(kEpiSwigluBwd)

}  // namespace mgpt
