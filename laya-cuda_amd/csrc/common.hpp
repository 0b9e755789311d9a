// Shared device helpers for the gfx950 (CDNA4) encoder kernels.
#pragma once

#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <cstddef>

namespace laya {

// Kernel-level timing on request: when the host has set `launch_timing` on this thread, the next
// LAYA_LAUNCH records that event pair from the kernel's own dispatch (hipExtLaunchKernel: start
// and end of the kernel, the interval a kernel trace reports, without the extra stream packets of
// hipEventRecord around the launch) and clears it.  Never set while a stream is being captured.
struct LaunchTiming {
  hipEvent_t start = nullptr, stop = nullptr;
};
inline thread_local LaunchTiming launch_timing;

#define LAYA_LAUNCH(kernel, grid, block, lds, stream, ...)                                          \
  do {                                                                                              \
    if (::laya::launch_timing.start) {                                                              \
      hipExtLaunchKernelGGL(kernel, grid, block, lds, stream, ::laya::launch_timing.start,          \
                            ::laya::launch_timing.stop, 0, __VA_ARGS__);                            \
      ::laya::launch_timing = ::laya::LaunchTiming{};                                              \
    } else {                                                                                        \
      hipLaunchKernelGGL(kernel, grid, block, lds, stream, __VA_ARGS__);                            \
    }                                                                                               \
  } while (0)

// 16-bit MFMA operand types.  Storage in HBM is raw 16-bit; arithmetic is always fp32.
typedef __bf16 bf16;
typedef _Float16 f16;

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef int i32x4 __attribute__((ext_vector_type(4)));

constexpr int kWave = 64;

template <typename T> struct Vec8;
template <> struct Vec8<bf16> { typedef bf16x8 type; };
template <> struct Vec8<f16> { typedef f16x8 type; };
template <typename T> struct Vec4;
template <> struct Vec4<bf16> { typedef bf16x4 type; };
template <> struct Vec4<f16> { typedef f16x4 type; };

// D = A(32x16) * B(16x32) + C, fp32 accumulate.  Lane l supplies row/col l%32 and the 8
// consecutive k-slots of group l/32; the accumulator's element r of lane l is
// C[8*(r/4) + 4*(l/32) + r%4][l%32].
__device__ __forceinline__ f32x16 mfma32(bf16x8 a, bf16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x16 mfma32(f16x8 a, f16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}
// D = A(16x32) * B(32x16) + C; element r of lane l is C[4*(l/16) + r][l%16].
__device__ __forceinline__ f32x4 mfma16(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mfma16(f16x8 a, f16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

// Direct global -> LDS load (global_load_lds_dwordx4): the wave's 64 lanes each fetch 16 bytes from
// their own address `g` and the hardware writes them, lane by lane, to the 1 KB of LDS starting at
// byte address `lds` (wave-uniform; M0 holds it).  Issued from inline assembly: the compiler's own
// form makes its wait-counter model assume that each such load may overwrite any LDS a pending
// read targets, so it drains every LDS read before each load.  Here a load's destination is read
// only after publish_stage below, which waits for the loads explicitly.  The {m0} operand lets the
// compiler write M0 and know it is live; one s_nop separates that write from the LDS DMA.
__device__ __forceinline__ void lds_load16(const void* g, unsigned lds) {
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(g), "{m0}"(lds));
}
// The same direct load through a buffer resource (buffer_load_dwordx4 ... offen lds): lane l fetches
// 16 bytes at resource base + voffset(l) + soffset and the hardware writes them to LDS byte address
// lds + 16 l (lds wave-uniform, in M0).  Loads past the resource's byte range return zeros.
// soffset must be wave-uniform; readfirstlane puts it in an SGPR where the compiler computed it with
// vector instructions (integer division of uniform values), and folds away where it already is one.
__device__ __forceinline__ void lds_load16_buffer(i32x4 rsrc, unsigned voffset, unsigned soffset, unsigned lds) {
  soffset = __builtin_amdgcn_readfirstlane(soffset);
  asm volatile("s_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds" ::"v"(voffset), "s"(rsrc), "s"(soffset),
               "{m0}"(lds));
}
// 128-bit buffer resource of `bytes` bytes at `base` (raw buffer: stride 0, byte offsets), wave-uniform.
__device__ __forceinline__ i32x4 buffer_resource(const void* base, unsigned bytes) {
  const uint64_t p = reinterpret_cast<uint64_t>(base);
  i32x4 r;
  r[0] = __builtin_amdgcn_readfirstlane(static_cast<int>(p & 0xffffffffu));
  r[1] = __builtin_amdgcn_readfirstlane(static_cast<int>((p >> 32) & 0xffffu));
  r[2] = __builtin_amdgcn_readfirstlane(static_cast<int>(bytes));
  r[3] = 0x00020000;  // dword 3 of a raw gfx9 buffer resource: 32-bit data format
  return r;
}
// Stores that write through the XCD's L2 (sc1).  A kernel's end writes its dirty L2 lines back, since
// the next kernel's workgroups read them from other XCDs; written through as they are made, the
// lines are clean by then.  16-byte form through a buffer resource, 4- and 8-byte forms as relaxed
// device-scope stores.  512 x 3,072 x 768 on the few-row GEMM: 8.6 -> 8.2 us; but a kernel that has little
// else to wait for pays for them (the paired-key attention: 9.4 -> 11.3 us).
// store_through16: the resource must be the same in all lanes (a row's, say, with the row index from
// readfirstlane) and cover every lane's 16 bytes: a lane past its range stores nothing, without an error.
constexpr int kWriteThrough = 16;  // sc1 in the cache-policy operand of the gfx950 buffer builtins
__device__ __forceinline__ void store_through16(__amdgpu_buffer_rsrc_t r, unsigned voffset, f32x4 v) {
  typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), r, voffset, 0, kWriteThrough);
}
template <typename V>
__device__ __forceinline__ void store_through(void* p, V v) {
  static_assert(sizeof(V) == 4 || sizeof(V) == 8, "4- or 8-byte values");
  if constexpr (sizeof(V) == 4) {
    __hip_atomic_store(static_cast<unsigned*>(p), __builtin_bit_cast(unsigned, v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  } else {
    __hip_atomic_store(static_cast<unsigned long long*>(p), __builtin_bit_cast(unsigned long long, v), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
  }
}
// Byte address of an LDS object, as M0 wants it.
__device__ __forceinline__ unsigned lds_address(const void* p) {
  typedef __attribute__((address_space(3))) const void* LdsPtr;
  return static_cast<unsigned>(reinterpret_cast<uintptr_t>((LdsPtr)p));
}
// Publishes LDS written by direct loads: wait for this wave's memory operations up to the
// s_waitcnt immediate `kWait`, then one workgroup barrier.  s_waitcnt and s_barrier are intrinsics
// without memory semantics in LLVM IR, so the empty asm with a memory clobber keeps the compiler
// from moving the following LDS reads above them; it emits no instruction.
template <int kWait>
__device__ __forceinline__ void publish_stage() {
  __builtin_amdgcn_s_waitcnt(kWait);
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}
// s_waitcnt immediate (gfx9 layout: vmcnt bits 3:0 and 15:14, expcnt 6:4, lgkmcnt 11:8) that waits
// until at most `vm` vector memory operations are outstanding and every LDS access has completed.
constexpr int waitcnt_vm(int vm) { return (vm & 15) | ((vm >> 4) << 14) | (7 << 4); }
// s_waitcnt immediate that waits until at most `vm` vector memory operations are outstanding and
// leaves LDS accesses in flight.
constexpr int waitcnt_vm_only(int vm) { return (vm & 15) | ((vm >> 4) << 14) | (7 << 4) | (15 << 8); }
// s_waitcnt immediate that waits for every LDS access (lgkmcnt 0) and no vector memory operation.
constexpr int waitcnt_lgkm0_keep_vm() { return 15 | (3 << 14) | (7 << 4); }

template <typename T> __device__ __forceinline__ T to_half(float v) { return static_cast<T>(v); }
template <typename T> __device__ __forceinline__ float to_float(T v) { return static_cast<float>(v); }

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d, kWave);
  return v;
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) v = fmaxf(v, __shfl_xor(v, d, kWave));
  return v;
}

// Exact-erf GELU, computed in fp32 with the device libm's erff (the fp32 decision head).
__device__ __forceinline__ float gelu(float v) { return 0.5f * v * (1.0f + erff(v * 0.7071067811865475f)); }

// Exact-erf GELU for values rounded to 16 bits right after (the FFN-up GEMM epilogue).  With
// q = Phi(-|x|), GELU(x) = x Phi(x) is x (1 - q) for x >= 0 and x q for x < 0, i.e. max(x, 0) - |x| q:
// one max and one FMA, and large negative inputs never subtract nearly equal numbers.  -log2 q is
// smooth, so q is the exp2 of a polynomial: degree 8 in |x|, a weighted least-squares fit with the
// weights moved to the largest errors, over [0, 5.5] with the constant term pinned to q(0) = 1/2; its
// leading coefficient is positive, so q falls to 0 beyond (7: 1.2e-12, the true 1.3e-12; 20: 0).
// In fp32: absolute error at most 2.5e-7, 2.6e-8 rms on N(0, 1), relative error at most 6e-5 down to
// |GELU| = 1e-5, against 3.3e-7, 5.4e-8 and 1e-3 for the rational form below.  An exponential and ten
// VALU operations where that takes a reciprocal more: the epilogue of a 65536 x 4096 GEMM runs this
// 268M times (585 -> 551 us).
__device__ __forceinline__ float gelu16(float x) {
  const float ax = fabsf(x);
  float p = __builtin_fmaf(ax, 8.8822900e-07f, -1.4745427506568376e-05f);
  p = __builtin_fmaf(ax, p, 6.223141099326313e-05f);
  p = __builtin_fmaf(ax, p, 4.555389459710568e-04f);
  p = __builtin_fmaf(ax, p, -7.509920746088028e-03f);
  p = __builtin_fmaf(ax, p, 5.283201485872269e-02f);
  p = __builtin_fmaf(ax, p, 4.590853750705719e-01f);
  p = __builtin_fmaf(ax, p, 1.1511214971542358f);
  p = __builtin_fmaf(ax, p, 1.0f);
  return __builtin_fmaf(-ax, __builtin_amdgcn_exp2f(-p), fmaxf(x, 0.f));
}

// The same function by a rational approximation: less exact and dearer, kept for the GeGLU epilogues because
// of one test.  The small ModernBERT fixture's weights (std 0.15) amplify bf16 rounding to 0.14 in its logits,
// two of its options are 0.23 apart, and with gelu16 in GeGLU the rounding falls so that the bf16 run
// decides the other way (logits within the test's tolerance either way; fp16 is not affected).  With erfc
// from Abramowitz & Stegun, Handbook of Mathematical Functions, formula 7.1.26:
//   erfc(z) = t (a1 + t (a2 + t (a3 + t (a4 + t a5)))) exp(-z^2),  t = 1 / (1 + p z),  z >= 0,
// absolute error <= 1.5e-7 (far below the 2^-11 relative rounding of fp16 that follows).
// With q = Phi(-|x|) = erfc(|x|/sqrt(2))/2, GELU(x) = x Phi(x) is x (1 - q) for x >= 0 and x q for
// x < 0, i.e. max(x, 0) - |x| q: one max and one FMA instead of a compare, a select and two
// products, and large negative inputs never subtract nearly equal numbers.  The 1/sqrt(2) is folded
// into p and the 1/2 into the a_i, so a value costs one reciprocal, one exp2 and nine VALU
// operations instead of the libm erff's range reduction.
__device__ __forceinline__ float gelu16_rational(float x) {
  const float ax = fabsf(x);
  const float t = __builtin_amdgcn_rcpf(__builtin_fmaf(0.3275911f * 0.7071067811865475f, ax, 1.0f));
  float poly = __builtin_fmaf(t, 0.5f * 1.061405429f, 0.5f * -1.453152027f);
  poly = __builtin_fmaf(t, poly, 0.5f * 1.421413741f);
  poly = __builtin_fmaf(t, poly, 0.5f * -0.284496736f);
  poly = __builtin_fmaf(t, poly, 0.5f * 0.254829592f);
  // exp(-z^2) = exp2(-x^2 log2(e) / 2)
  const float q = t * poly * __builtin_amdgcn_exp2f(x * x * (-0.5f * 1.4426950408889634f));
  return __builtin_fmaf(-ax, q, fmaxf(x, 0.f));
}

}  // namespace laya
