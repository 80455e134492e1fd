// Row-wise RMSNorm with an optional fused residual add, and the SwiGLU product, for the decoder
// layers of the serving path (the roles of vLLM's fused_add_rms_norm and silu_and_mul around the
// attention backend).  Both keep the rounding points of the torch expressions they replace, so a
// row computed here differs from torch's only where torch's own reduction order would.
#include <algorithm>

#include "common.h"
#include "runtime.h"

namespace lkv {
namespace {

constexpr int kNormThreads = 256;
constexpr int kNormMaxHidden = 16384;  // 8 chunks of 8 elements per thread
constexpr int kNormMaxChunks = kNormMaxHidden / (kNormThreads * 8);

struct NormParams {
  const uint16_t* x;
  int64_t x_stride;
  uint16_t* residual;
  int64_t res_stride;
  const uint16_t* w;
  uint16_t* out;
  int64_t out_stride;
  int32_t hidden;
  float eps;
};

__device__ inline void unpack8(uint4 u, float (&f)[8]) {
  f[0] = bf16_lo(u.x);
  f[1] = bf16_hi(u.x);
  f[2] = bf16_lo(u.y);
  f[3] = bf16_hi(u.y);
  f[4] = bf16_lo(u.z);
  f[5] = bf16_hi(u.z);
  f[6] = bf16_lo(u.w);
  f[7] = bf16_hi(u.w);
}

__device__ inline uint4 pack8(const float (&f)[8]) {
  return make_uint4(pack_bf16x2(f[0], f[1]), pack_bf16x2(f[2], f[3]), pack_bf16x2(f[4], f[5]), pack_bf16x2(f[6], f[7]));
}

// One workgroup per row; thread t owns the 8-element chunks t, t + 256, ... (kChunks of them).  With kAdd
// the row is residual := bf16(residual + x) first (torch's bf16 add) and the normalised row is that sum.
// Then, as transformers' LlamaRMSNorm: h = float(row); r = rsqrt(sum(h^2) * (1 / hidden) + eps);
// out = bf16(w * bf16(h * r)).
// Bound by HBM: every load (x, residual and the weights) is issued before the first use, with no branch
// between them (a chunk past the row rereads the last one), so a row costs one memory round trip.  x and
// the residual are streams (read once; the residual's next reader comes a projection later) and take
// non-temporal accesses; the output stays cached for the projection that reads it next.  4096 rows of
// 4096 with a residual: 22.6 us = 5.9 TB/s (25.4 with cached accesses, 27.3 with a branch around each
// chunk's loads).
template <bool kAdd, int kChunks>
__global__ __launch_bounds__(kNormThreads) void rmsnorm_kernel(const NormParams p) {
  __shared__ float part[kNormThreads / 64];
  const int row = blockIdx.x;
  const int chunks = p.hidden >> 3;
  const uint4* x = reinterpret_cast<const uint4*>(p.x + row * p.x_stride);
  uint4* res = kAdd ? reinterpret_cast<uint4*>(p.residual + row * p.res_stride) : nullptr;
  const uint4* w = reinterpret_cast<const uint4*>(p.w);
  uint4 xv[kChunks], rv[kChunks], wv[kChunks];
#pragma unroll
  for (int k = 0; k < kChunks; ++k) {
    const int c = min(static_cast<int>(threadIdx.x) + k * kNormThreads, chunks - 1);
    xv[k] = load_nt(x + c);
    if (kAdd) rv[k] = load_nt(res + c);
  }
#pragma unroll
  for (int k = 0; k < kChunks; ++k) wv[k] = w[min(static_cast<int>(threadIdx.x) + k * kNormThreads, chunks - 1)];
  float ss = 0.f;
#pragma unroll
  for (int k = 0; k < kChunks; ++k) {
    const int c = threadIdx.x + k * kNormThreads;
    if (c < chunks) {
      float v[8];
      unpack8(xv[k], v);
      if (kAdd) {
        float r[8];
        unpack8(rv[k], r);
#pragma unroll
        for (int j = 0; j < 8; ++j) r[j] += v[j];
        xv[k] = pack8(r);
        __builtin_nontemporal_store(__builtin_bit_cast(u32x4, xv[k]), reinterpret_cast<u32x4*>(res + c));
        unpack8(xv[k], v);
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) ss = __builtin_fmaf(v[j], v[j], ss);
    }
  }
  // row sum: within the wave (DPP through the shuffle builtins), then across the 4 waves
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) ss += __shfl_xor(ss, off);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = ss;
  __syncthreads();
  const float total = (part[0] + part[1]) + (part[2] + part[3]);
  const float r = rsqrtf(total * (1.f / static_cast<float>(p.hidden)) + p.eps);
  uint4* out = reinterpret_cast<uint4*>(p.out + row * p.out_stride);
#pragma unroll
  for (int k = 0; k < kChunks; ++k) {
    const int c = threadIdx.x + k * kNormThreads;
    if (c < chunks) {
      float h[8], wf[8];
      unpack8(xv[k], h);
#pragma unroll
      for (int j = 0; j < 8; ++j) h[j] *= r;
      unpack8(pack8(h), h);  // h.to(bf16)
      unpack8(wv[k], wf);
#pragma unroll
      for (int j = 0; j < 8; ++j) h[j] = wf[j] * h[j];
      out[c] = pack8(h);
    }
  }
}

// out = bf16(bf16(silu(gate)) * up), silu(g) = g / (1 + e^-g) in fp32 (v_exp_f32 and v_rcp_f32; the bf16
// result is that of torch's correctly rounded expf and division for all 65,536 gate values); grid
// (column groups, rows), one 8-element chunk per thread (4096 rows of 14336: 1 chunk and non-temporal loads
// 52.4 us = 6.7 TB/s, 2 chunks 56.8, 4 chunks 55.1, cached loads 61-66 us).

__device__ inline float silu(float g) {
  if (g < -80.f) return g / (1.f + expf(-g));  // (1 / (1 + e^-g) is near or below the normal range)
  // e^x = 2^hi (1 + lo ln 2), hi + lo = x log2(e): the rounding of the product x log2(e) alone would reach
  // 2^-18 of e^x; the reciprocal takes one Newton step (both arguments finite: x >= -80)
  const float x = -fminf(g, 80.f);
  const float hi = x * kLog2e, lo = __builtin_fmaf(x, kLog2e, -hi);
  const float e = fast_exp2(hi);
  const float d = 1.f + __builtin_fmaf(e, lo * kLn2, e);
  const float r = __builtin_amdgcn_rcpf(d);
  return g * __builtin_fmaf(__builtin_fmaf(-d, r, 1.f), r, r);
}

__global__ __launch_bounds__(256) void silu_mul_kernel(const uint16_t* gate, int64_t g_stride, const uint16_t* up,
                                                       int64_t u_stride, uint16_t* out, int64_t o_stride, int32_t rows,
                                                       int32_t width) {
  const int c = blockIdx.x * 256 + threadIdx.x;
  if (c >= width >> 3) return;
  for (int64_t row = blockIdx.y; row < rows; row += gridDim.y) {
    const uint4 gv = load_nt(reinterpret_cast<const uint4*>(gate + row * g_stride) + c);
    const uint4 uv = load_nt(reinterpret_cast<const uint4*>(up + row * u_stride) + c);
    float g[8], u[8];
    unpack8(gv, g);
    unpack8(uv, u);
#pragma unroll
    for (int j = 0; j < 8; ++j) g[j] = silu(g[j]);
    unpack8(pack8(g), g);  // silu's bf16 result
#pragma unroll
    for (int j = 0; j < 8; ++j) g[j] *= u[j];
    reinterpret_cast<uint4*>(out + row * o_stride)[c] = pack8(g);
  }
}

// The RMSNorm instance that holds a row of `hidden` elements.
template <bool kAdd>
void launch_rmsnorm(const NormParams& p, int32_t rows, hipStream_t s) {
  const int chunks = (p.hidden + kNormThreads * 8 - 1) / (kNormThreads * 8);
  if (chunks <= 1)
    rmsnorm_kernel<kAdd, 1><<<rows, kNormThreads, 0, s>>>(p);
  else if (chunks <= 2)
    rmsnorm_kernel<kAdd, 2><<<rows, kNormThreads, 0, s>>>(p);
  else if (chunks <= 4)
    rmsnorm_kernel<kAdd, 4><<<rows, kNormThreads, 0, s>>>(p);
  else
    rmsnorm_kernel<kAdd, kNormMaxChunks><<<rows, kNormThreads, 0, s>>>(p);
}

}  // namespace
}  // namespace lkv

extern "C" int32_t lkv_rmsnorm(const lkv_rmsnorm_args* a, lkv_stream_t stream) {
  using namespace lkv;
  LKV_REQUIRE(a != nullptr, "null args");
  LKV_REQUIRE(a->struct_size == static_cast<int32_t>(sizeof(lkv_rmsnorm_args)),
              "lkv_rmsnorm_args size mismatch (caller %d, library %d)", a->struct_size,
              static_cast<int32_t>(sizeof(lkv_rmsnorm_args)));
  LKV_REQUIRE(a->rows >= 0, "rows must be non-negative");
  LKV_REQUIRE(a->hidden > 0 && a->hidden % 8 == 0 && a->hidden <= kNormMaxHidden,
              "hidden must be a positive multiple of 8 up to %d, got %d", kNormMaxHidden, a->hidden);
  LKV_REQUIRE(a->x != nullptr && a->weight != nullptr && a->out != nullptr, "null x/weight/out");
  const uintptr_t align = reinterpret_cast<uintptr_t>(a->x) | reinterpret_cast<uintptr_t>(a->weight) |
                          reinterpret_cast<uintptr_t>(a->out) | reinterpret_cast<uintptr_t>(a->residual);
  LKV_REQUIRE((align & 15) == 0, "rows must be 16-byte aligned");
  LKV_REQUIRE((a->x_stride | a->out_stride | a->residual_stride) % 8 == 0, "row strides must be multiples of 8 elements");
  if (a->rows == 0) return LKV_OK;
  NormParams p;
  p.x = static_cast<const uint16_t*>(a->x);
  p.x_stride = a->x_stride;
  p.residual = static_cast<uint16_t*>(a->residual);
  p.res_stride = a->residual_stride;
  p.w = static_cast<const uint16_t*>(a->weight);
  p.out = static_cast<uint16_t*>(a->out);
  p.out_stride = a->out_stride;
  p.hidden = a->hidden;
  p.eps = a->eps;
  hipStream_t s = as_stream(stream);
  if (a->residual != nullptr)
    launch_rmsnorm<true>(p, a->rows, s);
  else
    launch_rmsnorm<false>(p, a->rows, s);
  return check_launch("lkv_rmsnorm");
}

extern "C" int32_t lkv_silu_mul(const void* gate, int64_t gate_stride, const void* up, int64_t up_stride, void* out,
                                int64_t out_stride, int32_t rows, int32_t width, lkv_stream_t stream) {
  using namespace lkv;
  LKV_REQUIRE(gate != nullptr && up != nullptr && out != nullptr, "null gate/up/out");
  LKV_REQUIRE(rows >= 0 && width > 0 && width % 8 == 0, "width must be a positive multiple of 8");
  const uintptr_t align = reinterpret_cast<uintptr_t>(gate) | reinterpret_cast<uintptr_t>(up) | reinterpret_cast<uintptr_t>(out);
  LKV_REQUIRE((align & 15) == 0, "rows must be 16-byte aligned");
  LKV_REQUIRE((gate_stride | up_stride | out_stride) % 8 == 0, "row strides must be multiples of 8 elements");
  if (rows == 0) return LKV_OK;
  const dim3 grid(static_cast<unsigned>((width / 8 + 255) / 256),
                  static_cast<unsigned>(std::min(rows, 65535)));
  silu_mul_kernel<<<grid, 256, 0, as_stream(stream)>>>(
      static_cast<const uint16_t*>(gate), gate_stride, static_cast<const uint16_t*>(up), up_stride,
      static_cast<uint16_t*>(out), out_stride, rows, width);
  return check_launch("lkv_silu_mul");
}
