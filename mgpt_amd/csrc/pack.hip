// pack.hip -- weight packing: reference layout fp32 -> GEMM layouts.
//
// The reference stores a Linear weight as W[in][out] row-major
// (layers/LinearLayer.cpp:15-21).  The grouped GEMMs want each output
// channel's K-run contiguous (B[n][k]), so the weights are transposed at
// load time through 64x64 LDS tiles (coalesced on both sides), converted
// to the compute type, and, for gate/up, interleaved in 64-row groups
// [32 gate rows | 32 up rows] of the same 32 hidden units.  A training step
// loads its parameters again after every optimizer step, so fp32 and bf16
// weights take one launch per 64 experts that reads each parameter once and
// writes the forward's and the backward's layouts.  fp8 weights (inference)
// are first packed as fp32 and then quantised row by row: per output channel,
// scale = amax / 448 (1 for an all-zero channel) and q = e4m3(w / scale),
// round-to-nearest-even, saturating at +-448, zero encoded as +0.
#include <algorithm>

#include "common.hpp"

namespace mgpt {
namespace {

// dst row of source column n: gate/up interleave (mode 1) or identity (0).
__device__ __forceinline__ int dst_row(int n, int mode, int off) {
  return mode ? (n / 32) * 64 + (n % 32) + off : n;
}

// src [Kin][Nout] fp32 (leading dim Nout) -> dst[dst_row(n)][k] (leading dim
// ldd), fp32: the rows of fp8 weights before their quantisation.
__global__ __launch_bounds__(256) void pack_transpose_kernel(const float* __restrict__ src, int Kin,
                                                             int Nout, float* __restrict__ dst,
                                                             int ldd, int mode, int off) {
  __shared__ float tile[64][65];
  const int k0 = blockIdx.y * 64, n0 = blockIdx.x * 64;
  const int tx = threadIdx.x % 64, ty = threadIdx.x / 64;
  for (int r = ty; r < 64; r += 4) {
    const int k = k0 + r, n = n0 + tx;
    tile[r][tx] = (k < Kin && n < Nout) ? src[(size_t)k * Nout + n] : 0.0f;
  }
  __syncthreads();
  for (int r = ty; r < 64; r += 4) {
    const int n = n0 + r, k = k0 + tx;
    if (n < Nout && k < Kin) dst[(size_t)dst_row(n, mode, off) * ldd + k] = tile[tx][r];
  }
}

// OCP E4M3FN encode, nearest-even, saturating to 448.
__device__ __forceinline__ uint8_t f32_to_e4m3(float v) {
  const uint32_t sign = (__float_as_uint(v) >> 31) & 1u;
  const float a = fabsf(v);
  uint32_t code;
  if (!(a < 448.0f)) {
    code = 0x7E;
  } else if (a < 0x1p-6f) {
    code = (uint32_t)rintf(a * 512.0f);          // subnormal grid m * 2^-9 (m = 8 is 2^-6)
  } else {
    uint32_t b = __float_as_uint(a);
    uint32_t q = b >> 20;                          // exponent + top 3 mantissa bits
    const uint32_t rem = b & 0xFFFFFu;
    q += (rem > 0x80000u) || (rem == 0x80000u && (q & 1u));
    const int ex = (int)(q >> 3) - 127 + 7;
    code = ((uint32_t)ex << 3) | (q & 7u);
    if (code > 0x7E) code = 0x7E;
  }
  return (uint8_t)(code | ((sign && code) ? 0x80u : 0u));
}

// Row-wise quantisation of src [rows][K] fp32 -> q [rows][K] e4m3 (columns at
// fp8_col), scale[rows].
__global__ __launch_bounds__(256) void quantize_rows_kernel(const float* __restrict__ src, int K,
                                                            uint8_t* __restrict__ q,
                                                            float* __restrict__ scale) {
  __shared__ float s_red[4];
  const size_t r = blockIdx.x;
  const float* row = src + r * K;
  float m = 0.0f;
  for (int k = threadIdx.x; k < K; k += 256) m = fmaxf(m, fabsf(row[k]));
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) m = fmaxf(m, __shfl_xor(m, d, kWave));
  if (lane_id() == 0) s_red[threadIdx.x / kWave] = m;
  __syncthreads();
  const float amax = fmaxf(fmaxf(s_red[0], s_red[1]), fmaxf(s_red[2], s_red[3]));
  const float s = amax > 0.0f ? amax / 448.0f : 1.0f;
  for (int k = threadIdx.x; k < K; k += 256) q[r * K + fp8_col(k)] = f32_to_e4m3(row[k] / s);
  if (threadIdx.x == 0) scale[r] = s;
}

// dst[i][0..n) = src[i][0..n), zero elsewhere up to ldd (bias padding).
__global__ void pad_rows_kernel(const float* __restrict__ src, int n, float* __restrict__ dst,
                                int ldd) {
  const int i = threadIdx.x + blockIdx.x * blockDim.x;
  if (i < ldd) dst[i] = i < n ? src[i] : 0.0f;
}

// Eight values as DT at a 16-byte aligned address.
__device__ __forceinline__ void put8(float* p, const float (&v)[8]) {
  *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
  *reinterpret_cast<float4*>(p + 4) = make_float4(v[4], v[5], v[6], v[7]);
}
__device__ __forceinline__ void put8(bf16_t* p, const float (&v)[8]) {
  *reinterpret_cast<uint4*>(p) = make_uint4(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]),
                                            pack_bf16x2(v[4], v[5]), pack_bf16x2(v[6], v[7]));
}

// Every layout of an expert's weights from one read of its fp32 parameters
// (blockIdx.y = expert): the forward's transposed operands, the padded
// biases and, with wgub set, the backward's operands, which keep the
// parameters' own orientation.  HBM-bound: 4 bytes read and 2 (bf16, forward
// only) or 4 (with the backward's) written an element.  A block takes two
// 64 x 64 tiles through LDS, the gate and up tile of the same place (so that
// a row of wgub, [32 gate | 32 up] twice, is one 256-byte run of bf16) or two
// W_down tiles side by side; rows of the transposed side are 128-byte runs.
// The tiles cover the padding of the contiguous dimension (zeros there);
// rows past the parameters' are left as they are (cleared at allocation).
// Measured on MI355X, training steps that load their parameters: cfg3
// through the fused block (16 experts, C = 1024, H = 2816, bf16) 3.74 -> 2.83
// ms, cfg1 (8 experts, C = 128, H = 512, fp32) 0.607 -> 0.385 ms, against one
// launch per tensor (715 + 207 us of kernels at cfg3) and transposes of the
// forward packs in the backward (222 us).
template <typename DT>
__global__ __launch_bounds__(256) void pack_experts_kernel(ExpertParams src, ExpertPacks<DT> out,
                                                           int Cx, int C, int H, int Hp, int Cp,
                                                           int Hq, int gu_units, int d_units) {
  __shared__ float tile[2][64][65];
  const int e = blockIdx.y, tid = threadIdx.x;
  int u = blockIdx.x;
  const float* const* P = src.p[e];
  if (u >= gu_units + d_units) {   // the biases
    for (int i = tid; i < Hp; i += 256) {
      out.bg[(size_t)e * Hp + i] = i < H ? P[1][i] : 0.0f;
      out.bu[(size_t)e * Hp + i] = i < H ? P[3][i] : 0.0f;
    }
    for (int i = tid; i < Cp; i += 256) out.bd[(size_t)e * Cp + i] = i < Cx ? P[5][i] : 0.0f;
    return;
  }
  // Tile t of the pair: rows r0.., columns n0[t].. of src_t [rows][cols].
  const bool down = u >= gu_units;
  if (down) u -= gu_units;
  const int rows = down ? H : Cx, cols = down ? Cx : H;
  const int nx = down ? (Cx + 127) / 128 : (H + 63) / 64;
  const int r0 = (u / nx) * 64, c0 = (u % nx) * (down ? 128 : 64);
  const int dc = down ? 64 : 0;   // column step from the first tile to the second
  const int q = tid % 16;
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const float* s = down ? P[4] : P[2 * t];
    const int c = c0 + t * dc + 4 * q;
    // 16-byte loads where the rows keep the alignment
    const bool vec = (cols & 3) == 0 && (reinterpret_cast<uintptr_t>(s) & 15) == 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int lr = 16 * i + tid / 16, r = r0 + lr;
      float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      if (r < rows) {
        const float* g = s + (size_t)r * cols + c;
        if (vec) {
          if (c < cols) v = *reinterpret_cast<const float4*>(g);
        } else {
          if (c < cols) v.x = g[0];
          if (c + 1 < cols) v.y = g[1];
          if (c + 2 < cols) v.z = g[2];
          if (c + 3 < cols) v.w = g[3];
        }
      }
      float* d = &tile[t][lr][4 * q];
      d[0] = v.x;
      d[1] = v.y;
      d[2] = v.z;
      d[3] = v.w;
    }
  }
  __syncthreads();
  // transposed: source column n becomes a row, its 64 source rows a run
#pragma unroll
  for (int t = 0; t < 2; ++t) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int ln = 32 * i + tid / 8, n = c0 + t * dc + ln, k8 = (tid % 8) * 8;
      if (n >= cols) continue;
      float v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = tile[t][k8 + j][ln];
      if (down)
        put8(out.wd + ((size_t)e * Cp + n) * Hp + r0 + k8, v);
      else
        put8(out.wgu + ((size_t)e * 2 * Hp + dst_row(n, 1, 32 * t)) * C + r0 + k8, v);
    }
  }
  if (!out.wgub) return;
  // as they are: rows of 128 values, 8 per thread
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int lr = 16 * i + tid / 16, r = r0 + lr;
    if (r >= rows) continue;
    const int g4 = q / 4;   // 32-value group of the row
    const int t = down ? g4 / 2 : g4 & 1;
    const int ln = (down ? (g4 & 1) : (g4 >> 1)) * 32 + (q % 4) * 8;
    float v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = tile[t][lr][ln + j];
    if (down) {
      const int c = c0 + 64 * t + ln;
      if (c < C) put8(out.wdb + ((size_t)e * Hq + r) * C + c, v);
    } else {
      put8(out.wgub + ((size_t)e * Cp + r) * 2 * Hp + 2 * c0 + 8 * q, v);
    }
  }
}

// Every layout of the router's parameters: [G][C][RE] (G = ceil(E/RE), the
// fused kernels), and where the pointers are set [E][C] (split decode
// router), column quads [C/4][E][4] (one-launch decode router) and [G*RE][C]
// (the backward), zero over the columns c >= Cx of a padded width and the
// experts past E; and the bias.
__global__ __launch_bounds__(256) void pack_router_kernel(const float* __restrict__ wr,
                                                          const float* __restrict__ br, int Cx,
                                                          int C, int E, int RE,
                                                          float* __restrict__ wr_g,
                                                          float* __restrict__ wr1,
                                                          float* __restrict__ wr4,
                                                          float* __restrict__ wrt,
                                                          float* __restrict__ br_out, int total) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < E) br_out[i] = br[i];
  if (i >= total) return;
  const int j = i % RE, c = (i / RE) % C, g = i / (RE * C);
  const int e = g * RE + j;
  const float v = (e < E && c < Cx) ? wr[(size_t)c * E + e] : 0.0f;
  wr_g[i] = v;
  if (wrt) wrt[(size_t)e * C + c] = v;
  if (e >= E) return;
  if (wr1) wr1[(size_t)e * C + c] = v;
  if (wr4) wr4[((size_t)(c / 4) * E + e) * 4 + c % 4] = v;
}

// dst[r][0..ncopy) = src[r][0..ncopy), dst[r][ncopy..nfill) = 0: a row block
// moved between a caller's width and the library's zero-padded width.
template <typename T>
__global__ __launch_bounds__(256) void copy_cols_kernel(const T* __restrict__ src, int lds,
                                                        T* __restrict__ dst, int ldd, int ncopy,
                                                        int nfill, int rows) {
  const int c = blockIdx.x * 256 + threadIdx.x;
  if (c >= nfill) return;
  for (size_t r = blockIdx.y; r < (size_t)rows; r += gridDim.y)
    dst[r * ldd + c] = c < ncopy ? src[r * lds + c] : T(0);
}

// fp8 weights [E][Npad][K] (columns at fp8_col) -> the decode stream's tiles
// [E][Npad/256][K/128][256][128]: every 256-row x 128-column stage the decode
// GEMM loads is one contiguous 32 KB block, columns in their own order.  One
// thread per 16-byte chunk.
__global__ __launch_bounds__(256) void tile_fp8_kernel(const uint8_t* __restrict__ src, int Npad,
                                                       int K, size_t chunks,
                                                       uint4* __restrict__ dst) {
  const size_t q = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (q >= chunks) return;
  const size_t row_chunks = (size_t)K / 16;
  const size_t row = q / row_chunks;               // e * Npad + n
  const int c16 = (int)(q % row_chunks);
  const size_t e = row / Npad;
  const int n = (int)(row % Npad);
  const int KT = K / 128;
  const size_t tile = (e * (size_t)(Npad / 256) + n / 256) * KT + c16 / 8;
  const uint8_t* r = src + row * K;
  const uint2 lo = *reinterpret_cast<const uint2*>(r + fp8_col(16 * c16));
  const uint2 hi = *reinterpret_cast<const uint2*>(r + fp8_col(16 * c16 + 8));
  dst[(tile * 256 + n % 256) * 8 + c16 % 8] = make_uint4(lo.x, lo.y, hi.x, hi.y);
}

// dst_j[r][c] += src[off_j + r * lds_j + c]: the handle's gradients added
// into the caller's (Tensor::add_grad, one rounded add per element), a batch
// of tensors per launch (blockIdx.y = tensor).
__global__ __launch_bounds__(256) void add_jobs_kernel(const float* __restrict__ src,
                                                       AddJobs jobs) {
  const int j = blockIdx.y;
  const int cols = jobs.cols[j];
  const size_t total = (size_t)jobs.rows[j] * cols;
  float* __restrict__ dst = jobs.dst[j];
  const float* __restrict__ s = src + jobs.off[j];
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (size_t)gridDim.x * 256) {
    const size_t r = i / cols, c = i % cols;
    dst[i] = dst[i] + s[r * jobs.lds[j] + c];
  }
}

}  // namespace

hipError_t launch_add_jobs(const float* src, const AddJobs& jobs, size_t max_elems,
                           hipStream_t stream) {
  if (jobs.n <= 0) return hipSuccess;
  const unsigned gx = (unsigned)std::min<size_t>((max_elems + 255) / 256, 1024);
  hipLaunchKernelGGL(add_jobs_kernel, dim3(std::max(gx, 1u), jobs.n), dim3(256), 0, stream, src,
                     jobs);
  return hipGetLastError();
}

hipError_t launch_tile_fp8(const uint8_t* src, int E, int Npad, int K, uint8_t* dst,
                           hipStream_t stream) {
  if (Npad % 256 != 0 || K % 128 != 0) return hipErrorInvalidValue;
  const size_t chunks = (size_t)E * Npad * (K / 16);
  hipLaunchKernelGGL(tile_fp8_kernel, dim3((unsigned)((chunks + 255) / 256)), dim3(256), 0, stream,
                     src, Npad, K, chunks, reinterpret_cast<uint4*>(dst));
  return hipGetLastError();
}

// RE experts per wave group (router_experts_per_wave(E)); Cx <= C: the
// caller's width.  wr1, wr4 (C % 4 == 0) and wrt may be null.
hipError_t launch_pack_router(const float* wr, const float* br, int Cx, int C, int E, int RE,
                              float* wr_g, float* wr1, float* wr4, float* wrt, float* br_out,
                              hipStream_t stream) {
  if (wr4 && C % 4) return hipErrorInvalidValue;
  const int total = ((E + RE - 1) / RE) * C * RE;   // >= E
  hipLaunchKernelGGL(pack_router_kernel, dim3((total + 255) / 256), dim3(256), 0, stream, wr, br,
                     Cx, C, E, RE, wr_g, wr1, wr4, wrt, br_out, total);
  return hipGetLastError();
}

// n <= kMaxExperts experts (see pack_experts_kernel); C, Hp and Hq multiples
// of 64, the destinations 16-byte aligned.
template <typename DT>
hipError_t launch_pack_experts(const ExpertParams& src, int n, const ExpertPacks<DT>& out, int Cx,
                               int C, int H, int Hp, int Cp, int Hq, hipStream_t stream) {
  if (n <= 0) return hipSuccess;
  if (n > kMaxExperts || C % 64 || Hp % 64 || Hq % 64 || !out.wgub != !out.wdb)
    return hipErrorInvalidValue;
  const int gu_units = ((Cx + 63) / 64) * ((H + 63) / 64);
  const int d_units = ((H + 63) / 64) * ((Cx + 127) / 128);
  hipLaunchKernelGGL(pack_experts_kernel<DT>, dim3(gu_units + d_units + 1, n), dim3(256), 0,
                     stream, src, out, Cx, C, H, Hp, Cp, Hq, gu_units, d_units);
  return hipGetLastError();
}
template hipError_t launch_pack_experts<float>(const ExpertParams&, int, const ExpertPacks<float>&,
                                               int, int, int, int, int, int, hipStream_t);
template hipError_t launch_pack_experts<bf16_t>(const ExpertParams&, int,
                                                const ExpertPacks<bf16_t>&, int, int, int, int,
                                                int, int, hipStream_t);

// rows x nfill block: copy ncopy columns, zero the rest (pad), or copy
// ncopy = nfill columns of a wider source (unpad).
template <typename T>
hipError_t launch_copy_cols(const T* src, int lds, T* dst, int ldd, int rows, int ncopy, int nfill,
                            hipStream_t stream) {
  if (rows <= 0 || nfill <= 0) return hipSuccess;
  hipLaunchKernelGGL(copy_cols_kernel<T>, dim3((nfill + 255) / 256, std::min(rows, 16384)),
                     dim3(256), 0, stream, src, lds, dst, ldd, ncopy, nfill, rows);
  return hipGetLastError();
}
template hipError_t launch_copy_cols<float>(const float*, int, float*, int, int, int, int,
                                            hipStream_t);
template hipError_t launch_copy_cols<bf16_t>(const bf16_t*, int, bf16_t*, int, int, int, int,
                                             hipStream_t);

hipError_t launch_pack_transpose(const float* src, int Kin, int Nout, float* dst, int ldd,
                                 int mode, int off, hipStream_t stream) {
  dim3 grid((Nout + 63) / 64, (Kin + 63) / 64);
  hipLaunchKernelGGL(pack_transpose_kernel, grid, dim3(256), 0, stream, src, Kin, Nout, dst, ldd,
                     mode, off);
  return hipGetLastError();
}

hipError_t launch_quantize_rows(const float* src, int rows, int K, uint8_t* q, float* scale,
                                hipStream_t stream) {
  hipLaunchKernelGGL(quantize_rows_kernel, dim3(rows), dim3(256), 0, stream, src, K, q, scale);
  return hipGetLastError();
}

hipError_t launch_pad_row(const float* src, int n, float* dst, int ldd, hipStream_t stream) {
  hipLaunchKernelGGL(pad_rows_kernel, dim3((ldd + 255) / 256), dim3(256), 0, stream, src, n, dst,
                     ldd);
  return hipGetLastError();
}

}  // namespace mgpt
