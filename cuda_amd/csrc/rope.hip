// RoPE + prefill for gfx950: the fused_rope_flash_attention entry point.
//
// O = softmax(rope(Q) rope(K)^T * scale [+ causal]) V with the rotate-half
// RoPE of the reference (fused_rope_flash_attention_kernel.cuh:60-70,98-108;
// tests/_utils.py:75-94): for position s and dim c,
//   x'[c] = x[c] cos[s][c] + r[c] sin[s][c],  r = [-x[D/2:], x[:D/2]],
// with fp32 tables cos / sin [S, D].
//
// q and k are rotated once, in one launch, in the input dtype (the operand
// precision of the prefill kernels): k into the caller's workspace, 16-bit q
// into the output buffer o, whose rows each prefill workgroup reads as Q before
// it writes them as O, float32 q into the workspace too. The pass is bound by
// memory (q and k read and written once); it lets head dim 128 run on the 64-row
// kernel, which has no registers to rotate in: 32/8 heads x 4096 x 128, causal,
// bf16 138 -> 125 us, 8192 keys 509 -> 465. (The reference rotates both inside
// its attention loop.)
// One thread rotates dims c .. c+7 of the first half together with their
// partners c+D/2 .. c+D/2+7, at one position for `group` heads: the position's
// 128 bytes of cos and sin stay in registers, loads and stores are 16 bytes.
#include <algorithm>

#include "common.h"
#include "launch.h"

namespace ca {
namespace {

// 8 consecutive elements as floats, and back (rounded to the type)
template <typename Tr>
struct Elem {
  using vec8 = typename Tr::vec8;
  static __device__ __forceinline__ void ld(const void* p, size_t i, float (&x)[8]) {
    const vec8 v = *(const vec8*)((const uint16_t*)p + i);
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = (float)v[e];
  }
  static __device__ __forceinline__ void st(void* p, size_t i, const float (&x)[8]) {
    vec8 v;
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
      const typename Tr::vec2 w = Tr::pack2(x[e], x[e + 1]);
      v[e] = w[0];
      v[e + 1] = w[1];
    }
    *(vec8*)((uint16_t*)p + i) = v;
  }
};
template <>
struct Elem<F32> {
  static __device__ __forceinline__ void ld(const void* p, size_t i, float (&x)[8]) {
    *(f32x4*)x = *(const f32x4*)((const float*)p + i);
    *(f32x4*)(x + 4) = *(const f32x4*)((const float*)p + i + 4);
  }
  static __device__ __forceinline__ void st(void* p, size_t i, const float (&x)[8]) {
    *(f32x4*)((float*)p + i) = *(const f32x4*)x;
    *(f32x4*)((float*)p + i + 4) = *(const f32x4*)(x + 4);
  }
};

// Heads 0 .. nq - 1 are q's, nq .. n_heads - 1 k's ([heads, S, D]); block y takes
// `group` of them, block x 256 / (D / 16) positions.
template <typename Tr, int D>
__global__ __launch_bounds__(256) void rope_kernel(const void* __restrict__ q, void* qr,
                                                   const void* __restrict__ k, void* __restrict__ kr,
                                                   const float* __restrict__ cos_tab,
                                                   const float* __restrict__ sin_tab, int nq,
                                                   int n_heads, int group, int S) {
  constexpr int H = D / 2;
  constexpr int L = H / 8;  // threads per row
  const int s = (int)blockIdx.x * (256 / L) + (int)threadIdx.x / L;
  if (s >= S) return;
  const int c = 8 * ((int)threadIdx.x % L);
  float ca[8], cb[8], sa[8], sb[8];
  const size_t tab = (size_t)s * D + c;
  Elem<F32>::ld(cos_tab, tab, ca);
  Elem<F32>::ld(cos_tab, tab + H, cb);
  Elem<F32>::ld(sin_tab, tab, sa);
  Elem<F32>::ld(sin_tab, tab + H, sb);
  const int h0 = (int)blockIdx.y * group, h1 = min(h0 + group, n_heads);
#pragma unroll 2
  for (int h = h0; h < h1; ++h) {
    const bool is_q = h < nq;
    const void* x = is_q ? q : k;
    void* y = is_q ? qr : kr;
    const size_t row = ((size_t)(is_q ? h : h - nq) * S + s) * D + c;
    float a[8], b[8], lo[8], hi[8];
    Elem<Tr>::ld(x, row, a);
    Elem<Tr>::ld(x, row + H, b);
    // x'[c] = a cos[c] - b sin[c];  x'[c + H] = b cos[c + H] + a sin[c + H]
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      lo[e] = a[e] * ca[e] - b[e] * sa[e];
      hi[e] = b[e] * cb[e] + a[e] * sb[e];
    }
    Elem<Tr>::st(y, row, lo);
    Elem<Tr>::st(y, row + H, hi);
  }
}

template <typename Tr, int D>
hipError_t rope_t(const void* q, void* qr, const void* k, void* kr, const float* cos_tab,
                  const float* sin_tab, long long nq, long long nk, int S, hipStream_t stream) {
  constexpr int kPos = 256 / (D / 16);
  const long long gx = (S + kPos - 1) / kPos, heads = nq + nk;
  if (gx == 0 || heads == 0) return hipSuccess;
  // as many heads per thread as leave about 8 blocks per CU; grid y is 16-bit
  const long long fill = std::max(1LL, std::min(16LL, gx * heads / (8LL * std::max(device_cus(), 1))));
  const long long group = std::max(fill, (heads + 65534) / 65535);
  if (heads > 0x7fffffffLL - group) return hipErrorInvalidValue;
  hipLaunchKernelGGL((rope_kernel<Tr, D>), dim3((unsigned)gx, (unsigned)((heads + group - 1) / group)),
                     dim3(256), 0, stream, q, qr, k, kr, cos_tab, sin_tab, (int)nq, (int)heads,
                     (int)group, S);
  return hipGetLastError();
}

hipError_t rope(int dtype, int D, const void* q, void* qr, const void* k, void* kr,
                const float* cos_tab, const float* sin_tab, long long nq, long long nk, int S,
                hipStream_t stream) {
#define CA_ROPE_CASE(TR)                                                                 \
  return D == 64 ? rope_t<TR, 64>(q, qr, k, kr, cos_tab, sin_tab, nq, nk, S, stream)     \
                 : rope_t<TR, 128>(q, qr, k, kr, cos_tab, sin_tab, nq, nk, S, stream);
  if (dtype == kDtypeBF16) { CA_ROPE_CASE(BF16) }
  if (dtype == kDtypeF16) { CA_ROPE_CASE(F16) }
  if (dtype == kDtypeF32) { CA_ROPE_CASE(F32) }
#undef CA_ROPE_CASE
  return hipErrorInvalidValue;
}

size_t elem_bytes(int dtype) { return dtype == kDtypeF32 ? 4 : 2; }

}  // namespace

// float32: rotated q, then k (256-byte aligned); 16-bit: rotated k only (q goes
// through the output buffer).
size_t rope_workspace_bytes(int dtype, int B, int Hq, int Hkv, int S, int D) {
  const size_t qb = (size_t)B * Hq * S * D * elem_bytes(dtype);
  const size_t kb = (size_t)B * Hkv * S * D * elem_bytes(dtype);
  return dtype == kDtypeF32 ? ((qb + 255) & ~(size_t)255) + kb : kb;
}

hipError_t launch_rope_prefill(int dtype, const void* q, const void* k, const void* v,
                               const float* cos_tab, const float* sin_tab, void* o, int B, int Hq,
                               int Hkv, int S, int D, float scale, bool causal, void* ws,
                               hipStream_t stream) {
  const size_t qb = (size_t)B * Hq * S * D * elem_bytes(dtype);
  void* qr = dtype == kDtypeF32 ? ws : o;
  void* kr = dtype == kDtypeF32 ? (char*)ws + ((qb + 255) & ~(size_t)255) : ws;
  const hipError_t e = rope(dtype, D, q, qr, k, kr, cos_tab, sin_tab, (long long)B * Hq,
                            (long long)B * Hkv, S, stream);
  if (e != hipSuccess) return e;
  return launch_prefill(dtype, qr, kr, v, o, nullptr, B, Hq, Hkv, S, D, scale, causal, stream);
}

}  // namespace ca
