// Row kernels around the training path of GridSelfAttention (src/deepfold3/model/attention.py:211-257)
// at 128 channels in 4 heads: the pair-bias projection with its backward, and the output gate
// o * sigmoid(g) with its backward. All are bound by the bytes of their [B, N, N, 128] operands;
// each reads and writes every operand once.
#include <algorithm>

#include "capi.h"
#include "common.h"

namespace {

constexpr int kGC = 128;  // channels of a token
constexpr int kGH = 4;    // heads

// A thread takes one 16-byte piece of a token: LPT lanes per token.
template <class TC>
struct Piece {
  static constexpr int VEC = 16 / sizeof(TC);
  static constexpr int LPT = kGC / VEC;       // 16 (bf16), 32 (fp32)
  static constexpr int TPB = 256 / LPT;       // tokens per pass of a block
  static constexpr int TILE = 64;             // tokens per block iteration
};

// pb[b][h][p] = sum_c x[b][p][c] w[h][c], in fp32 from the products to the result. The weights
// stay in registers, a token's sums are reduced over its lanes, and the tile's results go
// through LDS so that each head's row is written in 256-byte runs. A GEMM of 4 columns leaves
// 12 of a 16-wide MFMA's columns empty and its result needs a second pass into the head-major
// fp32 order: library product and copies 25 us, this kernel 12 us at 384 x 384 tokens in bf16.
template <class TC>
__global__ __launch_bounds__(256) void grid_bias_fwd_kernel(const TC* __restrict__ x, const TC* __restrict__ w,
                                                            float* __restrict__ pb, int B, long NN) {
  using P = Piece<TC>;
  __shared__ float t[kGH][P::TILE];
  const int sub = threadIdx.x % P::LPT, tok = threadIdx.x / P::LPT;
  float wr[kGH][P::VEC];
#pragma unroll
  for (int h = 0; h < kGH; ++h) load16<TC>(w + h * kGC + sub * P::VEC, wr[h]);
  const long M = (long)B * NN;
  for (long m0 = (long)blockIdx.x * P::TILE; m0 < M; m0 += (long)gridDim.x * P::TILE) {
    const int lim = (int)min((long)P::TILE, M - m0);
    float v[P::TILE / P::TPB][P::VEC];
#pragma unroll
    for (int u = 0; u < P::TILE / P::TPB; ++u)
      load16<TC>(x + (m0 + min(tok + u * P::TPB, lim - 1)) * kGC + sub * P::VEC, v[u]);
#pragma unroll
    for (int u = 0; u < P::TILE / P::TPB; ++u) {
      float s[kGH];
#pragma unroll
      for (int h = 0; h < kGH; ++h) {
        s[h] = 0.f;
#pragma unroll
        for (int e = 0; e < P::VEC; ++e) s[h] = fmaf(v[u][e], wr[h][e], s[h]);
#pragma unroll
        for (int o = P::LPT / 2; o > 0; o >>= 1) s[h] += __shfl_xor(s[h], o, 64);
      }
      if (sub < kGH) t[sub][tok + u * P::TPB] = sub == 0 ? s[0] : (sub == 1 ? s[1] : (sub == 2 ? s[2] : s[3]));
    }
    __syncthreads();
    const int h = threadIdx.x / P::TILE, i = threadIdx.x % P::TILE;  // 4 x 64
    if (i < lim) {
      const long m = m0 + i;
      const long b = m / NN;
      pb[(b * kGH + h) * NN + (m - b * NN)] = t[h][i];
    }
    __syncthreads();
  }
}

// dx[b][p][c] = sum_h dpb[b][h][p] w[h][c] and, per block, the partial dw[h][c] = sum_p
// dpb[b][h][p] x[b][p][c]: one read of x, one write of dx, fp32 sums. Two library products
// (K = 4 and, split over tokens, an output of 4 rows) with the copies between the two orders
// take 95 us at 384 x 384 tokens in bf16, this kernel 19 us and its reduction 5 us.
template <class TC>
__global__ __launch_bounds__(256) void grid_bias_bwd_kernel(const TC* __restrict__ x, const TC* __restrict__ w,
                                                            const float* __restrict__ dpb, TC* __restrict__ dx,
                                                            float* __restrict__ part, int B, long NN) {
  using P = Piece<TC>;
  __shared__ float t[kGH][P::TILE];
  __shared__ float red[4][kGH][kGC];  // [wave]
  const int sub = threadIdx.x % P::LPT, tok = threadIdx.x / P::LPT;
  float wr[kGH][P::VEC], acc[kGH][P::VEC];
#pragma unroll
  for (int h = 0; h < kGH; ++h) {
    load16<TC>(w + h * kGC + sub * P::VEC, wr[h]);
#pragma unroll
    for (int e = 0; e < P::VEC; ++e) acc[h][e] = 0.f;
  }
  const long M = (long)B * NN;
  for (long m0 = (long)blockIdx.x * P::TILE; m0 < M; m0 += (long)gridDim.x * P::TILE) {
    const int lim = (int)min((long)P::TILE, M - m0);
    {
      const int h = threadIdx.x / P::TILE, i = threadIdx.x % P::TILE;
      const long m = m0 + min(i, lim - 1);
      const long b = m / NN;
      const float d = dpb[(b * kGH + h) * NN + (m - b * NN)];
      t[h][i] = i < lim ? d : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < P::TILE / P::TPB; ++u) {
      const int i = tok + u * P::TPB;
      float v[P::VEC], y[P::VEC], d[kGH];
      load16<TC>(x + (m0 + min(i, lim - 1)) * kGC + sub * P::VEC, v);
#pragma unroll
      for (int h = 0; h < kGH; ++h) d[h] = t[h][i];
#pragma unroll
      for (int e = 0; e < P::VEC; ++e) {
        y[e] = 0.f;
#pragma unroll
        for (int h = 0; h < kGH; ++h) {
          y[e] = fmaf(d[h], wr[h][e], y[e]);
          acc[h][e] = fmaf(d[h], i < lim ? v[e] : 0.f, acc[h][e]);
        }
      }
      if (i < lim) store_vec<TC, P::VEC>(dx + (m0 + i) * kGC + sub * P::VEC, y);
    }
    __syncthreads();
  }
#pragma unroll
  for (int h = 0; h < kGH; ++h)
#pragma unroll
    for (int e = 0; e < P::VEC; ++e) {
#pragma unroll
      for (int o = P::LPT; o < 64; o <<= 1) acc[h][e] += __shfl_xor(acc[h][e], o, 64);
      if (lane_id() < P::LPT) red[wave_id()][h][sub * P::VEC + e] = acc[h][e];
    }
  __syncthreads();
  for (int i = threadIdx.x; i < kGH * kGC; i += 256) {
    const float* r = &red[0][0][0] + i;
    part[(size_t)blockIdx.x * kGH * kGC + i] =
        (r[0] + r[kGH * kGC]) + (r[2 * kGH * kGC] + r[3 * kGH * kGC]);
  }
}

// dw[i] = sum over the blocks of part[block][i], in a fixed order: a block sums 16 outputs,
// 16 threads each.
__global__ __launch_bounds__(256) void grid_bias_dw_kernel(const float* __restrict__ part, int blocks,
                                                           float* __restrict__ dw) {
  __shared__ float r[16][16];
  const int i = threadIdx.x % 16, k = threadIdx.x / 16;
  float s = 0.f;
#pragma unroll 8
  for (int g = k; g < blocks; g += 16) s += part[(size_t)g * kGH * kGC + blockIdx.x * 16 + i];
  r[k][i] = s;
  __syncthreads();
  if (k == 0) {
    for (int j = 1; j < 16; ++j) s += r[j][i];
    dw[blockIdx.x * 16 + i] = s;
  }
}

// Blocks of the backward's token loop (also the rows of its partial sums): two per CU keep the
// partial sums small; fewer for short inputs.
int grid_bias_blocks(long M) { return (int)std::min<long>((M + 63) / 64, 512); }

// out = o * sigmoid(g); g in rows of ldg elements.
template <class TC>
__global__ __launch_bounds__(256) void grid_gate_fwd_kernel(const TC* __restrict__ o, const TC* __restrict__ g,
                                                            long ldg, TC* __restrict__ out, long M) {
  using P = Piece<TC>;
  const int sub = threadIdx.x % P::LPT;
  for (long m = (long)blockIdx.x * P::TPB + threadIdx.x / P::LPT; m < M; m += (long)gridDim.x * P::TPB) {
    float a[P::VEC], b[P::VEC];
    load16<TC>(o + m * kGC + sub * P::VEC, a);
    load16<TC>(g + m * ldg + sub * P::VEC, b);
#pragma unroll
    for (int e = 0; e < P::VEC; ++e) a[e] *= sigmoidf_(b[e]);
    store_vec<TC, P::VEC>(out + m * kGC + sub * P::VEC, a);
  }
}

// d_o = dout sigmoid(g), dg = dout o sigmoid(g) (1 - sigmoid(g)); g and dg in rows of ldg and
// lddg elements. One pass of five operands: 31 us at 384 x 384 tokens in bf16 against 58 us
// for two products and the sigmoid's backward.
template <class TC>
__global__ __launch_bounds__(256) void grid_gate_bwd_kernel(const TC* __restrict__ dout, const TC* __restrict__ o,
                                                            const TC* __restrict__ g, long ldg, TC* __restrict__ d_o,
                                                            TC* __restrict__ dg, long lddg, long M) {
  using P = Piece<TC>;
  const int sub = threadIdx.x % P::LPT;
  for (long m = (long)blockIdx.x * P::TPB + threadIdx.x / P::LPT; m < M; m += (long)gridDim.x * P::TPB) {
    float a[P::VEC], b[P::VEC], c[P::VEC];
    load16<TC>(dout + m * kGC + sub * P::VEC, a);
    load16<TC>(o + m * kGC + sub * P::VEC, b);
    load16<TC>(g + m * ldg + sub * P::VEC, c);
#pragma unroll
    for (int e = 0; e < P::VEC; ++e) {
      const float sg = sigmoidf_(c[e]);
      const float d = a[e] * sg;
      c[e] = d * b[e] * (1.f - sg);
      a[e] = d;
    }
    store_vec<TC, P::VEC>(d_o + m * kGC + sub * P::VEC, a);
    store_vec<TC, P::VEC>(dg + m * lddg + sub * P::VEC, c);
  }
}

int check_common(const char* fn, long M, int C, int dtype) {
  PF_REQUIRE(M > 0, PF_ERR_INVALID_ARG, "%s: no tokens", fn);
  PF_REQUIRE(C == kGC, PF_ERR_UNSUPPORTED, "%s: C=%d (built: C=%d)", fn, C, kGC);
  PF_REQUIRE(dtype == PF_F32 || dtype == PF_BF16, PF_ERR_UNSUPPORTED, "%s: dtype %d", fn, dtype);
  return PF_OK;
}

template <class TC>
unsigned gate_grid(long M) {
  return (unsigned)std::min<long>((M + Piece<TC>::TPB - 1) / Piece<TC>::TPB, 16384);
}

}  // namespace

extern "C" {

int pf_grid_bias_fwd(const void* x, const void* w, int dtype, int B, int N, int C, int H, float* out, void* stream) {
  PF_REQUIRE(x && w && out, PF_ERR_INVALID_ARG, "pf_grid_bias_fwd: null pointer");
  PF_REQUIRE(B > 0 && N > 0, PF_ERR_INVALID_ARG, "pf_grid_bias_fwd: B=%d N=%d", B, N);
  const long NN = (long)N * N;
  if (int e = check_common("pf_grid_bias_fwd", B * NN, C, dtype)) return e;
  PF_REQUIRE(H == kGH, PF_ERR_UNSUPPORTED, "pf_grid_bias_fwd: H=%d (built: H=%d)", H, kGH);
  PF_REQUIRE(pf::aligned16(x) && pf::aligned16(w), PF_ERR_ALIGNMENT, "pf_grid_bias_fwd: unaligned pointer");
  hipStream_t s = pf::as_stream(stream);
  const unsigned grid = (unsigned)std::min<long>((B * NN + 63) / 64, 4096);
  if (dtype == PF_F32)
    grid_bias_fwd_kernel<float><<<grid, 256, 0, s>>>((const float*)x, (const float*)w, out, B, NN);
  else
    grid_bias_fwd_kernel<bf16><<<grid, 256, 0, s>>>((const bf16*)x, (const bf16*)w, out, B, NN);
  return pf::check_launch("pf_grid_bias_fwd");
}

size_t pf_grid_bias_bwd_workspace_bytes(int B, int N, int C, int H) {
  if (B <= 0 || N <= 0 || C != kGC || H != kGH) return 0;
  return (size_t)grid_bias_blocks((long)B * N * N) * kGH * kGC * sizeof(float);
}

int pf_grid_bias_bwd(const void* x, const void* w, const float* dout, int dtype, int B, int N, int C, int H, void* dx,
                     float* dw, void* workspace, size_t workspace_bytes, void* stream) {
  PF_REQUIRE(x && w && dout && dx && dw && workspace, PF_ERR_INVALID_ARG, "pf_grid_bias_bwd: null pointer");
  PF_REQUIRE(B > 0 && N > 0, PF_ERR_INVALID_ARG, "pf_grid_bias_bwd: B=%d N=%d", B, N);
  const long NN = (long)N * N;
  if (int e = check_common("pf_grid_bias_bwd", B * NN, C, dtype)) return e;
  PF_REQUIRE(H == kGH, PF_ERR_UNSUPPORTED, "pf_grid_bias_bwd: H=%d (built: H=%d)", H, kGH);
  PF_REQUIRE(pf::aligned16(x) && pf::aligned16(w) && pf::aligned16(dx) && pf::aligned16(workspace), PF_ERR_ALIGNMENT,
             "pf_grid_bias_bwd: unaligned pointer");
  const size_t need = pf_grid_bias_bwd_workspace_bytes(B, N, C, H);
  PF_REQUIRE(workspace_bytes >= need, PF_ERR_WORKSPACE, "pf_grid_bias_bwd: workspace %zu < %zu bytes",
             workspace_bytes, need);
  hipStream_t s = pf::as_stream(stream);
  const int blocks = grid_bias_blocks(B * NN);
  float* part = static_cast<float*>(workspace);
  if (dtype == PF_F32)
    grid_bias_bwd_kernel<float><<<blocks, 256, 0, s>>>((const float*)x, (const float*)w, dout, (float*)dx, part, B, NN);
  else
    grid_bias_bwd_kernel<bf16><<<blocks, 256, 0, s>>>((const bf16*)x, (const bf16*)w, dout, (bf16*)dx, part, B, NN);
  if (int e = pf::check_launch("pf_grid_bias_bwd")) return e;
  grid_bias_dw_kernel<<<kGH * kGC / 16, 256, 0, s>>>(part, blocks, dw);
  return pf::check_launch("pf_grid_bias_bwd dw");
}

int pf_grid_gate_fwd(const void* o, const void* g, long ldg, int dtype, void* out, long M, int C, void* stream) {
  PF_REQUIRE(o && g && out, PF_ERR_INVALID_ARG, "pf_grid_gate_fwd: null pointer");
  if (int e = check_common("pf_grid_gate_fwd", M, C, dtype)) return e;
  const long vec = dtype == PF_F32 ? 4 : 8;
  PF_REQUIRE(pf::aligned16(o) && pf::aligned16(g) && pf::aligned16(out) && ldg >= C && ldg % vec == 0,
             PF_ERR_ALIGNMENT, "pf_grid_gate_fwd: rows must be 16-byte aligned");
  hipStream_t s = pf::as_stream(stream);
  if (dtype == PF_F32)
    grid_gate_fwd_kernel<float><<<gate_grid<float>(M), 256, 0, s>>>((const float*)o, (const float*)g, ldg,
                                                                    (float*)out, M);
  else
    grid_gate_fwd_kernel<bf16><<<gate_grid<bf16>(M), 256, 0, s>>>((const bf16*)o, (const bf16*)g, ldg, (bf16*)out, M);
  return pf::check_launch("pf_grid_gate_fwd");
}

int pf_grid_gate_bwd(const void* dout, const void* o, const void* g, long ldg, int dtype, void* d_o, void* dg,
                     long lddg, long M, int C, void* stream) {
  PF_REQUIRE(dout && o && g && d_o && dg, PF_ERR_INVALID_ARG, "pf_grid_gate_bwd: null pointer");
  if (int e = check_common("pf_grid_gate_bwd", M, C, dtype)) return e;
  const long vec = dtype == PF_F32 ? 4 : 8;
  PF_REQUIRE(pf::aligned16(dout) && pf::aligned16(o) && pf::aligned16(g) && pf::aligned16(d_o) && pf::aligned16(dg) &&
                 ldg >= C && lddg >= C && ldg % vec == 0 && lddg % vec == 0,
             PF_ERR_ALIGNMENT, "pf_grid_gate_bwd: rows must be 16-byte aligned");
  hipStream_t s = pf::as_stream(stream);
  if (dtype == PF_F32)
    grid_gate_bwd_kernel<float><<<gate_grid<float>(M), 256, 0, s>>>((const float*)dout, (const float*)o,
                                                                    (const float*)g, ldg, (float*)d_o, (float*)dg,
                                                                    lddg, M);
  else
    grid_gate_bwd_kernel<bf16><<<gate_grid<bf16>(M), 256, 0, s>>>((const bf16*)dout, (const bf16*)o, (const bf16*)g,
                                                                  ldg, (bf16*)d_o, (bf16*)dg, lddg, M);
  return pf::check_launch("pf_grid_gate_bwd");
}

}  // extern "C"
