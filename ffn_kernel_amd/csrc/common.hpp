// Shared device/host helpers for the gfx950 kernels of libffnk.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stddef.h>

namespace ffnk {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;
typedef __attribute__((ext_vector_type(16))) float f32x16_t;

constexpr int kWave = 64;

__host__ __device__ constexpr int64_t cdiv64(int64_t a, int64_t b) { return (a + b - 1) / b; }
__host__ __device__ constexpr int cdiv(int a, int b) { return (a + b - 1) / b; }
__host__ __device__ constexpr int64_t round_up64(int64_t a, int64_t b) { return cdiv64(a, b) * b; }

// fp32 -> bf16, round to nearest even (NaN stays NaN).
__device__ __forceinline__ uint16_t f2bf(float f) {
  __bf16 b = static_cast<__bf16>(f);
  return __builtin_bit_cast(uint16_t, b);
}

__device__ __forceinline__ float bf2f(uint16_t v) {
  return __builtin_bit_cast(float, static_cast<uint32_t>(v) << 16);
}

// Two fp32 -> packed pair of bf16 (lo in bits 0..15).
__device__ __forceinline__ uint32_t pack2bf(float lo, float hi) {
  typedef __attribute__((ext_vector_type(2))) float f32x2_t;
  typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2_t;
  const f32x2_t v = {lo, hi};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));  // one v_cvt_pk_bf16_f32
}

// silu(g) * u in fp32: g * sigmoid(g) * u.
__device__ __forceinline__ float swiglu(float g, float u) {
  // v_exp_f32 and v_rcp_f32 are each good to 1 ulp, far inside the bf16 rounding of the result;
  // an IEEE division would cost about ten more instructions per element of the epilogue.
  const float s = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(g * -1.44269504088896341f));
  return g * s * u;
}

// SwiGLU backward on eight bf16 values: o1 = dh * t3 * silu'(t1), o3 = dh * silu(t1), oh = silu(t1) * t3.
// silu'(t) = s + t s (1 - s), s = sigmoid(t), in fp32 (the derivative term sketched in the reference's README.md:159-172 is not this one).
// The division is a correctly rounded one, unlike swiglu()'s: forward + backward at M = 4096, d = 4096, h = 14336 takes 3436 us with it,
// 3428 with v_rcp_f32 (runs of one side differ by 0.3 %).
__device__ __forceinline__ void swiglu_bwd(const uint4& t1, const uint4& t3, const uint4& dh, uint4* o1, uint4* o3, uint4* oh) {
  auto word = [](const uint4& v, int i) { return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w; };
  auto set = [](uint4* v, int i, uint32_t w) { (i == 0 ? v->x : i == 1 ? v->y : i == 2 ? v->z : v->w) = w; };
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float r1[2], r3[2], rh[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      auto value = [&](const uint4& v) { return __builtin_bit_cast(float, e == 0 ? word(v, i) << 16 : word(v, i) & 0xffff0000u); };
      const float a = value(t1), b = value(t3), d = value(dh);
      const float s = 1.0f / (1.0f + __expf(-a)), silu = a * s;
      r1[e] = d * b * (s + silu * (1.0f - s));
      r3[e] = d * silu;
      rh[e] = silu * b;
    }
    set(o1, i, pack2bf(r1[0], r1[1]));
    set(o3, i, pack2bf(r3[0], r3[1]));
    set(oh, i, pack2bf(rh[0], rh[1]));
  }
}

// p[0] + p[stride] + ... + p[(n - 1) * stride], in that order.  The loads of up to four terms are in flight together: one
// after the other, a reduce pass over few workgroups is n memory round trips long.  Over 13000 drawn calls with partials a call
// gains 0.2 - 0.4 us with two or three K ranges, 0.5 - 0.7 with four to seven and 1.4 with eight and more (MaskedLinear at
// M = 65 ... 512 0.9, 3.1 and 9.3 %, at M <= 64 2.0 and 4.9 %; MaskedFFN 0 - 3 %), unsplit calls nothing.
__device__ __forceinline__ float4 sum_partials(const float* p, int64_t stride, int n) {
  float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
  auto term = [&](int k) { return *reinterpret_cast<const float4*>(p + (int64_t)k * stride); };
  auto add = [&](const float4 v) { s.x += v.x; s.y += v.y; s.z += v.z; s.w += v.w; };
  int k = 0;
  for (; k + 4 <= n; k += 4) {
    const float4 a = term(k), b = term(k + 1), c = term(k + 2), d = term(k + 3);
    add(a); add(b); add(c); add(d);
  }
  if (n - k == 3) {
    const float4 a = term(k), b = term(k + 1), c = term(k + 2);
    add(a); add(b); add(c);
  } else if (n - k == 2) {
    const float4 a = term(k), b = term(k + 1);
    add(a); add(b);
  } else if (n - k == 1) {
    add(term(k));
  }
  return s;
}

// The weight streams' first workgroups: those of the visual rows, or of the text rows where there are no others.  A modality
// without rows takes up half of the launch, and its workgroups, which end at once, would fill the chip ahead of the ones
// with work: MaskedFFN d = 4096, h = 14336, text rows only, M = 5 ... 8 71.6 -> 62.5 us, M = 36 ... 48 81-86 -> 71.5.
__device__ __forceinline__ int first_group(int n_vis) {
#if defined(__HIP_DEVICE_COMPILE__)
  n_vis = __builtin_amdgcn_readfirstlane(n_vis);  // (uniform, which the compiler cannot see: the weights' addresses stay scalar)
#endif
  return n_vis == 0 ? 1 : 0;
}

// Workspace carving: every sub-buffer starts on a 256-byte boundary.
constexpr size_t kWsAlign = 256;
__host__ __device__ constexpr size_t ws_align(size_t n) { return (n + kWsAlign - 1) / kWsAlign * kWsAlign; }

}  // namespace ffnk
