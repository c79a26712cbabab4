// s2s_device.h - device helpers shared by the kernel files: raw buffer access,
// LDS copies and barriers, cross-lane sums, the GELU.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

typedef float f16v __attribute__((ext_vector_type(16)));

#define MFMA32(a, b, c) __builtin_amdgcn_mfma_f32_32x32x2f32((a), (b), (c), 0, 0, 0)

typedef unsigned v4u __attribute__((ext_vector_type(4)));

// Raw buffer access: a load whose byte offset lies past the resource's size
// returns zero and such a store is dropped, so tile edges (rows past M, columns
// past the group) need no branches, and every wave issues the same number of
// memory instructions on every path - which lets the compiler count them
// exactly in its s_waitcnt instead of draining the queue.
#define BUF_OOB 0x7ffffff0
// The size is capped below BUF_OOB, so that offset stays out of range even
// for a resource based inside a larger buffer (whose own offsets stay small).
#define BUF_MAX_BYTES 0x7fff0000u
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf_rsrc(const void *p, size_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), (short)0,
                                             (int)(bytes < BUF_MAX_BYTES ? bytes : BUF_MAX_BYTES),
                                             0x00020000);
}
__device__ __forceinline__ float4 buf_load4(__amdgpu_buffer_rsrc_t r, int off) {
    return __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
}
__device__ __forceinline__ float buf_load1(__amdgpu_buffer_rsrc_t r, int off) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
}
__device__ __forceinline__ void buf_store1(__amdgpu_buffer_rsrc_t r, int off, float v) {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, off, 0, 0);
}
__device__ __forceinline__ void buf_store4(__amdgpu_buffer_rsrc_t r, int off, float4 v) {
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4u, v), r, off, 0, 0);
}
// The same with a wave-uniform part of the offset in the instruction's SGPR
// offset (only for accesses known to be in range: the bounds check is not
// meant to be relied on for that part).
__device__ __forceinline__ float4 buf_load4s(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
    return __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0));
}
__device__ __forceinline__ void buf_store1s(__amdgpu_buffer_rsrc_t r, int voff, int soff, float v) {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, voff, soff, 0);
}
__device__ __forceinline__ void buf_store4s(__amdgpu_buffer_rsrc_t r, int voff, int soff, float4 v) {
    const v4u d = __builtin_bit_cast(v4u, v);
    __builtin_amdgcn_raw_buffer_store_b128(d, r, voff, soff, 0);
    // A VALU write of the data registers right behind a 16-byte store can
    // reach memory in its place: the compiler leaves a wait state there for
    // stores without an SGPR offset only, and with one, two workgroups per CU
    // stored the next value's first dword in the last lanes now and then. The
    // data stays in use until after the nop.
    asm volatile("s_nop 1" : : "v"(d));
}
typedef unsigned v2u __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void buf_store2(__amdgpu_buffer_rsrc_t r, int off, float2 v) {
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(v2u, v), r, off, 0, 0);
}


// The erf GELU, 0.5 v (1 + erf(v/sqrt2)) = v * Phi(v), evaluated through the
// complementary error function so that one branch-free formula covers every v:
// with t = |v|/sqrt2, erfc(t) = exp(-t^2) * erfcx(t), and the scaled function
// erfcx is smooth and bounded on [0, inf), so it is u times a degree-4
// polynomial in u = 1/(1 + 0.478 t) (u in (0, 1]; the substitution of
// Abramowitz & Stegun 7.1.26 with a refitted p). The five coefficients
// (halved, so the result is erfc(t)/2 directly) are a fit of erfcx on
// t in [0, 9] weighted by what an error costs the GELU (|v| exp(-t^2) / 2),
// iterated toward equal ripple against scipy.special.erfcx: 4.3e-8 absolute
// on the GELU in exact arithmetic, below float32 rounding. With q = erfc(t)/2,
// Phi(v) is 1 - q for v > 0 and q otherwise, so v Phi(v) = max(v, 0) - |v| q:
// one max and one fused multiply-add, and the negative side keeps its
// relative accuracy instead of cancelling in 1 + erf. Evaluated in float32
// the absolute error against the exact GELU is below 2.6e-7 on [-12, 12], the
// same as the erff form's rounding. One reciprocal, one exp2 and 11 other
// VALU operations, with no divergent branch (a library erff evaluates two
// polynomial branches when a wavefront holds both small and large arguments).
__device__ __forceinline__ float gelu_erf(float v) {
    // u = 1 / (1 + 0.478 |v| / sqrt2)
    const float u = __builtin_amdgcn_rcpf(fmaf(fabsf(v), 0.33799704f, 1.0f));
    float p = -0.10729234942429587f;
    p = fmaf(p, u, 0.34028711412207455f);
    p = fmaf(p, u, -0.05061983683614841f);
    p = fmaf(p, u, 0.18978627981436072f);
    p = fmaf(p, u, 0.12783743829594208f);
    // exp(-t^2) = 2^(v^2 * (-log2(e) / 2)); q = erfc(t) / 2
    const float q = u * p * __builtin_amdgcn_exp2f(v * v * -0.72134752044448170368f);
    // max(v, 0) as one v_max_f32: fmaxf (and every builtin the compiler
    // recognises as a max) adds a NaN-quieting max(v, v) in front of it (a
    // NaN in v still gives a NaN through the fma)
    float m;
    asm("v_max_f32 %0, 0, %1" : "=v"(m) : "v"(v));
    return fmaf(-fabsf(v), q, m);
}

typedef float f4v __attribute__((ext_vector_type(4)));
#define MFMA16(a, b, c) __builtin_amdgcn_mfma_f32_16x16x4f32((a), (b), (c), 0, 0, 0)

// Direct global -> LDS copy (gfx950 buffer_load_dwordx4 ... lds): lane l of the
// wave writes its 16 bytes at lds + 16*l, so one instruction moves a contiguous
// 1 KiB chunk without staging it in VGPRs. Out-of-range offsets write zeros.
__device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t r, float *lds, int off) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void *)lds, 16,
                                             off, 0, 0, 0);
}
// ... with a wave-uniform part of the offset in the instruction's SGPR offset
// (only for copies whose whole offset is in range: the range check sees the
// per-lane part alone)
__device__ __forceinline__ void dma16s(__amdgpu_buffer_rsrc_t r, float *lds, int voff, int soff) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void *)lds, 16,
                                             voff, soff, 0, 0);
}
// s_waitcnt vmcnt(n) alone (gfx9 encoding: vmcnt in bits 3:0 and 15:14,
// expcnt and lgkmcnt left at their maxima).
#define WAIT_VMCNT(n) __builtin_amdgcn_s_waitcnt((((n) & 15) | (((n) >> 4) << 14)) | 0x0F70)
// A workgroup barrier for LDS traffic only: this wave's LDS writes retired
// (lgkmcnt(0)), then s_barrier, with compiler fences on both sides. Unlike
// __syncthreads() it does not drain outstanding global stores (its release
// fence does), so a task's output stores and the next task's copies stay in
// flight across it. Data copied into LDS by DMA is covered by a WAIT_VMCNT
// before the barrier.
__device__ __forceinline__ void lds_sync() {
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0xC07F);
    __builtin_amdgcn_s_barrier();
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

// Sum over the 16 lanes of a DPP row, every lane receiving the total: four
// DPP moves on the VALU (quad_perm [1,0,3,2], quad_perm [2,3,0,1],
// row_half_mirror, row_mirror) instead of LDS-routed lane shuffles.
#define DPP_ADD(v, ctrl)                                                                       \
    ((v) + __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, (v)), \
                                                              (ctrl), 0xF, 0xF, true)))
__device__ __forceinline__ float row16_sum(float v) {
    v = DPP_ADD(v, 0xB1);
    v = DPP_ADD(v, 0x4E);
    v = DPP_ADD(v, 0x141);
    v = DPP_ADD(v, 0x140);
    return v;
}

// Two sums over the four 16-lane rows at once: lane j of row 0 (lanes 0-15)
// gets a[j] + a[j+16] + a[j+32] + a[j+48], lane j of row 1 the same sum of b
// (rows 2 and 3 repeat rows 0 and 1). v_permlane16_swap(a, b) leaves rows
// (a0, b0, a2, b2) in a and (a1, b1, a3, b3) in b, so a + b holds the pair
// sums of a in rows 0 and 2 and of b in rows 1 and 3; v_permlane32_swap(c, d)
// with d a copy of c leaves rows (c0, c1, c0, c1) in c and (c2, c3, c2, c3) in
// d (gfx950). The order is (x0 + x1) + (x2 + x3) for both. Inline assembly:
// the compiler's builtins for these swaps have added one result to itself
// instead of to the other one; the s_nop covers the VALU-write-then-permlane
// hazard.
__device__ __forceinline__ float xrow_sum2(float a, float b) {
    asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(a), "+v"(b));
    float c = a + b;
    float d = c;
    asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(c), "+v"(d));
    return c + d;
}

// The two 32-lane halves of a wave exchanged on the VALU (gfx950
// v_permlane32_swap with both operands a copy of x): `lo` gets lanes 0-31 of x
// in both halves, `hi` lanes 32-63, so lo + hi (or max(lo, hi)) combines lane
// l with lane l ^ 32 in every lane. Inline assembly for the reason above.
__device__ __forceinline__ void halves(float x, float &lo, float &hi) {
    lo = x;
    hi = x;
    asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(lo), "+v"(hi));
}
__device__ __forceinline__ float half_sum(float x) {
    float lo, hi;
    halves(x, lo, hi);
    return lo + hi;
}
__device__ __forceinline__ float half_max(float x) {
    float lo, hi;
    halves(x, lo, hi);
    return fmaxf(lo, hi);
}
