// Weight gradient of a linear over token-major operands: out [Co][Ci] = sum_t gy[t][co] x[t][ci]
// with t in the hundreds of thousands (the pair track's tokens), bf16 operands, fp32 sums.
//
// The contraction runs over the slow axis of both operands, so an MFMA operand (8 consecutive
// tokens of one channel per lane) is a transpose away from memory. It needs no LDS: a lane
// loads 2 (gy) or 4 (x) neighbouring channels of 8 tokens and pairs the tokens' halves with one
// v_perm_b32 per fragment register; lane r's channel m then is row (or column) r of fragment m,
// so the channels of a result are interleaved, 2 r + m and 4 c + n, which the store undoes.
//
// A block sums a 128 x 128 tile of the result over one chunk of tokens: wave w takes channels
// 64 (w & 1) .. +64 of the tile's gy columns, all of its x columns and every fourth 16-token
// step, two steps of loads in flight; the four waves of a half are added through LDS, the
// chunks by a second kernel, both in a fixed order. Blocks of one chunk run on one XCD, which
// reads a chunk that several tiles share once. Bytes bound it (gy and x once, 256 KB of partial
// sums per CU). At 147456 tokens: 512 x 128 38 us and 128 x 128 22 us with the sum over
// chunks (their bytes: 36 and 15); a batched library product over token chunks and its sum
// take 70 and 41 us. At 40000 tokens 20 and 19 us against 49 and 41.
#include <algorithm>

#include "capi.h"
#include "common.h"

namespace {

constexpr int kWgTile = 128;
constexpr int kWgNT = 512;
constexpr int kWgDepth = 2;  // 16-token steps of loads in flight per wave

typedef unsigned u32x2_t __attribute__((ext_vector_type(2)));

// Token chunks: about one block per CU over all tiles, a multiple of the eight XCDs.
int wg_chunks(long M, int tiles) {
  const int n = std::max(8, pf::cu_count() / tiles / 8 * 8);
  return (int)std::min<long>(n, std::max<long>(8, (M + 63) / 64 / 8 * 8));
}

__global__ __launch_bounds__(kWgNT, 2) void weight_grad_kernel(const bf16* __restrict__ gy, const bf16* __restrict__ x,
                                                               int M, int Co, int Ci, int chunk,
                                                               float* __restrict__ part) {
  __shared__ __attribute__((aligned(16))) f32x4 red[4][32 * 64];  // [slot][register quad][lane]
  const int tiles_i = Ci / kWgTile;
  const int tiles = (Co / kWgTile) * tiles_i;
  // chunk c's tiles take the blocks 8 tiles (c / 8) + 8 tile + c % 8: one XCD
  const int id = blockIdx.x;
  const int c = id / (8 * tiles) * 8 + (id & 7);
  const int tile = id / 8 % tiles;
  const int w = wave_id(), l = lane_id();
  const int hh = l >> 5, r = l & 31;
  const int half = w & 1, tg = w >> 1;
  const int co0 = tile / tiles_i * kWgTile + 64 * half;
  const int ci0 = tile % tiles_i * kWgTile;
  const int t0 = c * chunk;
  const int nt = __builtin_amdgcn_readfirstlane(max(0, min(chunk, M - t0)));
  const int steps = (nt + 63) / 64;  // of this wave: 16-token steps tg, tg + 4, ..
  int go[8], xo[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    go[j] = ((16 * tg + 8 * hh + j) * Co + co0 + 2 * r) * 2;
    xo[j] = ((16 * tg + 8 * hh + j) * Ci + ci0 + 4 * r) * 2;
  }

  unsigned gb[kWgDepth][8];
  u32x2_t xb[kWgDepth][8];
  auto issue = [&](int s, int k) __attribute__((always_inline)) {
    // 64 tokens of the chunk; rows past its end read as zeros
    // (readfirstlane: the clamp is a vector instruction, a resource must be scalar)
    const int left = __builtin_amdgcn_readfirstlane(max(0, min(64, nt - 64 * s)));
    const long t = left > 0 ? t0 + 64 * s : 0;
    const auto rg = buf_rsrc(gy + t * Co, left * Co * 2);
    const auto rx = buf_rsrc(x + t * Ci, left * Ci * 2);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      gb[k][j] = __builtin_amdgcn_raw_buffer_load_b32(rg, go[j], 0, 0);
      xb[k][j] = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_raw_buffer_load_b64(rx, xo[j], 0, 0));
    }
  };
  auto pair = [](unsigned lo, unsigned hi, int m) __attribute__((always_inline)) {
    return __builtin_amdgcn_perm(hi, lo, m ? 0x07060302u : 0x05040100u);
  };
  f32x16 acc[2][4] = {};
#pragma unroll
  for (int k = 0; k < kWgDepth; ++k) issue(k, k);
  for (int s = 0; s < steps; s += kWgDepth) {
#pragma unroll
    for (int k = 0; k < kWgDepth; ++k) {
      bf16x8 a[2], b[4];
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        u32x4 f;
#pragma unroll
        for (int d = 0; d < 4; ++d) f[d] = pair(gb[k][2 * d], gb[k][2 * d + 1], m);
        a[m] = __builtin_bit_cast(bf16x8, f);
      }
#pragma unroll
      for (int n = 0; n < 4; ++n) {
        u32x4 f;
#pragma unroll
        for (int d = 0; d < 4; ++d) f[d] = pair(xb[k][2 * d][n >> 1], xb[k][2 * d + 1][n >> 1], n & 1);
        b[n] = __builtin_bit_cast(bf16x8, f);
      }
      issue(s + k + kWgDepth, k);
#pragma unroll
      for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int n = 0; n < 4; ++n) acc[m][n] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[m], b[n], acc[m][n], 0, 0, 0);
    }
  }
  // (0 + 2) + (1 + 3) over the token groups
  auto put = [&](f32x4* dst) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < 32; ++q) {
      const f32x16& v = acc[q >> 4][(q >> 2) & 3];
      dst[q * 64 + l] = f32x4{v[4 * (q & 3)], v[4 * (q & 3) + 1], v[4 * (q & 3) + 2], v[4 * (q & 3) + 3]};
    }
  };
  auto add = [&](const f32x4* src) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < 32; ++q) {
      const f32x4 v = src[q * 64 + l];
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[q >> 4][(q >> 2) & 3][4 * (q & 3) + e] += v[e];
    }
  };
  if (tg >= 2) put(red[w - 4]);
  __syncthreads();
  if (tg < 2) add(red[w]);
  __syncthreads();
  if (tg == 1) put(red[half]);
  __syncthreads();
  if (tg != 0) return;
  add(red[half]);
  float* out = part + (size_t)c * Co * Ci;
#pragma unroll
  for (int m = 0; m < 2; ++m)
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      const int row = 8 * (q >> 2) + 4 * hh + (q & 3);
      const f32x4 v = {acc[m][0][q], acc[m][1][q], acc[m][2][q], acc[m][3][q]};
      *reinterpret_cast<f32x4*>(out + (size_t)(co0 + 2 * row + m) * Ci + ci0 + 4 * r) = v;
    }
}

// out = sum over chunks of part[chunk], in a fixed order: a block sums 16 vectors of four, 16
// threads each.
__global__ __launch_bounds__(256) void weight_grad_reduce_kernel(const f32x4* __restrict__ part, long n4, int chunks,
                                                                 f32x4* __restrict__ out) {
  __shared__ f32x4 r[16][16];
  const int i = threadIdx.x % 16, k = threadIdx.x / 16;
  const long o = (long)blockIdx.x * 16 + i;
  f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int g = k; g < chunks; g += 16) s += part[(size_t)g * n4 + o];
  r[k][i] = s;
  __syncthreads();
  if (k == 0) {
#pragma unroll
    for (int j = 1; j < 16; ++j) s += r[j][i];
    out[o] = s;
  }
}

}  // namespace

extern "C" {

size_t pf_weight_grad_workspace_bytes(long M, int Co, int Ci) {
  if (M <= 0 || Co <= 0 || Ci <= 0 || Co % kWgTile || Ci % kWgTile) return 0;
  return (size_t)wg_chunks(M, (Co / kWgTile) * (Ci / kWgTile)) * Co * Ci * sizeof(float);
}

int pf_weight_grad(const void* gy, const void* x, long M, int Co, int Ci, int dtype, float* out, void* workspace,
                   size_t workspace_bytes, void* stream) {
  PF_REQUIRE(gy && x && out && workspace, PF_ERR_INVALID_ARG, "pf_weight_grad: null pointer");
  PF_REQUIRE(M > 0 && Co > 0 && Ci > 0, PF_ERR_INVALID_ARG, "pf_weight_grad: M=%ld Co=%d Ci=%d", M, Co, Ci);
  PF_REQUIRE(dtype == PF_BF16 && Co % kWgTile == 0 && Ci % kWgTile == 0, PF_ERR_UNSUPPORTED,
             "pf_weight_grad: dtype %d Co=%d Ci=%d (built: bf16, multiples of %d)", dtype, Co, Ci, kWgTile);
  PF_REQUIRE(pf::aligned16(gy) && pf::aligned16(x) && pf::aligned16(out) && pf::aligned16(workspace), PF_ERR_ALIGNMENT,
             "pf_weight_grad: pointers must be 16-byte aligned");
  const int tiles = (Co / kWgTile) * (Ci / kWgTile);
  const int chunks = wg_chunks(M, tiles);
  const long chunk = (M + chunks - 1) / chunks;
  PF_REQUIRE(M < (1L << 31) - 65536 && (long)chunks * tiles < (1L << 31) && std::max(Co, Ci) < (1 << 20),
             PF_ERR_UNSUPPORTED, "pf_weight_grad: M=%ld Co=%d Ci=%d too large", M, Co, Ci);
  const size_t need = pf_weight_grad_workspace_bytes(M, Co, Ci);
  PF_REQUIRE(workspace_bytes >= need, PF_ERR_WORKSPACE, "pf_weight_grad: workspace %zu < %zu bytes", workspace_bytes,
             need);
  hipStream_t s = pf::as_stream(stream);
  weight_grad_kernel<<<chunks * tiles, kWgNT, 0, s>>>((const bf16*)gy, (const bf16*)x, (int)M, Co, Ci, (int)chunk,
                                                      static_cast<float*>(workspace));
  if (int e = pf::check_launch("pf_weight_grad")) return e;
  const long n4 = (long)Co * Ci / 4;
  weight_grad_reduce_kernel<<<(unsigned)(n4 / 16), 256, 0, s>>>(static_cast<const f32x4*>(workspace), n4, chunks,
                                                               reinterpret_cast<f32x4*>(out));
  return pf::check_launch("pf_weight_grad sum");
}

}  // extern "C"
