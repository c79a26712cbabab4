// s2s_split.hip - fp32 contractions on the f16 matrix cores, by splitting.
//
// An fp32 operand x is scaled by a power of two and written as hi + lo, hi =
// f16(x) and lo = f16(x - hi): 22 bits of it, and a product a b as the three
// products hi hi + hi lo + lo hi, each exact in the MFMA's fp32 accumulation
// (the lo lo term is 2^-22 of it and below). v_mfma_f32_16x16x32_f16 takes 32 k
// where the fp32 v_mfma_f32_16x16x4f32 takes 4 in twice the time; under pure MFMA
// load three of them make 3.8 times the fp32 rate on random operands (1,789 / 3
// against 155 TFLOP/s) and 4.9 times on zeros, the chip's clock making the
// difference. The error is no larger than the fp32 MFMA's, whose accumulator
// rounds once per 4 k: on K = 192 dot products of unit normals, rms 1.63e-7 of the
// result's rms against 2.47e-7, at K = 384 2.24e-7 against 3.56e-7.
//
// The scales keep f16's exponent range out of the way. A weight row is scaled
// at upload so that its largest element lies in [2^14, 2^15); an activation row
// (a token's, a pixel's) by 2^(14 - floor(log2 B)), B its largest magnitude or a
// bound of it. What f16 drops is 2^-39 of B, so an element down to 2^-14 of it
// keeps its 22 bits, and below that a sum still keeps its largest terms'. Where
// values that owe each other nothing would share a scale (the pixels of a conv's
// tile, the tokens of a window) each has its own. The products are scaled back in
// fp32, exactly (powers of two), before the bias.
//
// A operand tiles live in LDS in MFMA fragment order: per (row block of 16,
// k step of 32, part) 1 KiB, lane l = 16 q + r holding row r, k = 8 q .. 8 q + 7,
// so every operand read is one linear ds_read_b128. Weights are packed in the
// same order per wave and stream from L2 through registers, each wave reading
// only its own columns (33-39 TB/s measured with every CU reading the same
// 737 KB).
//
// MFMA 16x16x32 f16 lane layout (checked on the device): lane l supplies
// A[l%16][8(l/16) .. + 7] and B[l%16][the same k]; accumulator register i of
// lane l holds D[4(l/16) + i][l%16], rows from A, columns from B. With A =
// weights and B = tokens a lane holds one token and 4 consecutive columns.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <type_traits>
#include <vector>

#include "s2s_device.h"
#include "s2s_kernels.h"

typedef _Float16 h8v __attribute__((ext_vector_type(8)));
typedef _Float16 h4v __attribute__((ext_vector_type(4)));
#define MFMA16H(a, b, c) __builtin_amdgcn_mfma_f32_16x16x32_f16((a), (b), (c), 0, 0, 0)

namespace {

// 2^(14 - floor(log2 b)) for a bound b >= 0 (the exponent clamped so that the
// scale and its inverse are normal), and that inverse
__device__ __forceinline__ int bound_exp(float b) {
    return max((int)(__builtin_bit_cast(unsigned, b) >> 23), 15);
}
__device__ __forceinline__ float exp_scale(int e) { return __builtin_bit_cast(float, (268 - e) << 23); }
__device__ __forceinline__ float exp_unscale(int e) { return __builtin_bit_cast(float, (e - 14) << 23); }

// hi and lo of 4 values. Values and residuals pass through fp32 registers (the
// empty asm). Left to itself the compiler folds a scaling into the conversions
// (v_fma_mixlo_f16 rounds once where the packed conversion of the rounded
// product rounds twice, so the stored hi could differ from the one subtracted),
// and those issue at a quarter of the rate: measured 3.7 ns against 1.9 for
// v_fma_mix_f32 or the packed conversion and 1.2 for v_fma_f32.
__device__ __forceinline__ void split4(f4v v, h4v &hi, h4v &lo) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float x = v[i];
        asm("" : "+v"(x));
        v[i] = x;
        hi[i] = (_Float16)x;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float r = fmaf((float)hi[i], -1.0f, v[i]);
        asm("" : "+v"(r));
        lo[i] = (_Float16)r;
    }
}

#define DPP_MAX(v, ctrl)                                                                         \
    fmaxf((v), __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, (v)), \
                                                                  (ctrl), 0xF, 0xF, true)))
__device__ __forceinline__ float row16_max(float v) {
    v = DPP_MAX(v, 0xB1);
    v = DPP_MAX(v, 0x4E);
    v = DPP_MAX(v, 0x141);
    v = DPP_MAX(v, 0x140);
    return v;
}
// The maximum over lanes j, j+16, j+32, j+48, in every lane (xrow_sum2's swaps).
__device__ __forceinline__ float xrow_max(float a) {
    float b = a;
    asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(a), "+v"(b));
    float c = fmaxf(a, b);
    float d = c;
    asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(c), "+v"(d));
    return fmaxf(c, d);
}

// ... and the sum.
__device__ __forceinline__ float xrow_sum(float a) {
    float b = a;
    asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(a), "+v"(b));
    float c = a + b;
    float d = c;
    asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(c), "+v"(d));
    return c + d;
}

constexpr int FRAG = 1024;  // bytes of one fragment

// Byte offset within a fragment of row r's 8 k of group q (k = 8 q ..), of k step
// ks. The row's slot is permuted by q and the parity of ks, within 128 bytes, so
// that a wave writing a few rows' contiguous columns (operand tiles are loaded
// so) spreads over the banks: unpermuted, the 8 groups of two k steps are 8-way
// conflicts.
__device__ __forceinline__ int frag_slot(int ks, int q, int r) {
    return (q * 16 + (r ^ (q | (ks & 1) << 2))) * 16;
}
// Byte offset in a row block's fragments of the hi part of columns 16 T + 4 q ..
// + 3 of row j: where an output column tile T lands as the next contraction's
// operand (the lo part FRAG further on, row block rb 2 KS rb FRAG).
__device__ __forceinline__ int frag_col(int T, int j, int q) {
    return (T >> 1) * 2 * FRAG + frag_slot(T >> 1, (T & 1) * 2 + (q >> 1), j) + (q & 1) * 8;
}

}  // namespace

// ---------------------------------------------------------------------------
// k_token_mlp: the token half of a Swin block in one kernel,
//   x1  = x + LN1(o Wproj^T + b),  out = x1 + LN2(GELU(x1 W1^T + b1) W2^T + b2),
// reading the attention output o and the block input x once and writing the
// block output once, and x1 once each way through the output's rows (the three
// GEMMs it replaces moved 600 MB per block at 264 x 264 x 180 where this moves
// 244).
//
// A workgroup's 4 waves own 16 TN output columns each (C <= 64 TN), all of
// them the task's rows: RB row blocks of 16 tokens, at most 3, sized so that
// the two operand tiles (P0: o, then x1; P1: one C-wide chunk of the hidden
// layer) let two workgroups run per CU. The hidden layer is made and consumed
// C columns at a time, fc2's accumulators kept across the chunks.
//
// Weights stream through a register ring of WD k steps, refilled as consumed,
// through GEMM and task boundaries (every task walks the same stream). The row
// scales: o's from the row's maximum, x1's from the bound max|x| + sqrt(C)
// max|ln_w| + max|ln_b| (a normalised value is at most sqrt(C)), the hidden
// layer's from bound(x1) max_j sum_k |W1[j][k]| + max(b1, 0.17) (GELU(v) lies in
// [-0.17, max(v, 0)]). The hidden layer's is shared by its units: a stage of one
// block is 3.0e-7 of its rms from 64 bits (fp32 GEMMs 6.9e-7), with one fc1 row 2^12
// times the others 4.7e-7, 2^16 2.9e-6.
//
// A bound that a value passes by more than a factor of two would be an infinite
// hi, so the variance E[v^2] - mean^2 must not cancel: Wproj, W2 and their biases
// are uploaded less their mean over the output columns (in 64 bits, rounded once),
// which takes each row's mean off v, and a LayerNorm is the same without it. As
// given, rows of 180 whose mean is 2,000 times their deviation normalise to 870
// (emulated) and come out as NaN, and an fp32 GEMM loses the mean's digits of v.
//
// Every task of a launch has RB row blocks (the launcher's choice), workgroup b
// taking tasks b, b + gridDim.x, ...; the next task's rows are loaded while this
// one's last epilogue runs. MI355X: 69,696 tokens x 180 in 104-106 us where the
// three GEMMs took 228 (22.6 GFLOP as three f16 products each: 41 us of MFMA at
// the rate real data reaches, the rest VALU, which does not overlap MFMA on a
// SIMD, operand reads and barriers); 2,880 tokens 15 us against 3 launches of
// about 11.
// ---------------------------------------------------------------------------
namespace {

template <int TN, int RB> struct TokCfg {
    static constexpr int CP = 64 * TN;                // padded width
    static constexpr int KS = 2 * TN;                 // k steps per GEMM
    // weight ring, k steps (a divisor of KS); with three row blocks of 180 the
    // registers go to the operand prefetch instead of a third step (126 -> 119
    // us at 69,696 tokens), with fewer the ring is what hides L2's latency. 120
    // wide, 69,696 and 2,880 tokens: 59.3 and 7.8 us, with a ring of two steps
    // 60.0 and 8.4, without the prefetch 61.0 and 8.0; 60 wide 23.8 and 4.2,
    // with a ring of one step 24.6 and 4.6, without the prefetch 23.9 and 4.2
    static constexpr int WD = TN == 3 ? (RB == 3 ? 2 : 3) : (TN == 2 ? 4 : 2);
    static constexpr bool PRE = TN < 3 || RB == 3;  // operands read a k step ahead
};

template <int TN, int RB> struct TokState {
    h8v w[TokCfg<TN, RB>::WD][TN][2];  // the weight ring
    int wpos;                      // next k step of the stream to load
};

template <int TN, int RB>
__device__ __forceinline__ void tok_load(TokState<TN, RB> &s, int slot, __amdgpu_buffer_rsrc_t rw, int wbase,
                                         int lane) {
#pragma unroll
    for (int t = 0; t < TN; ++t)
#pragma unroll
        for (int p = 0; p < 2; ++p)
            s.w[slot][t][p] = __builtin_bit_cast(
                h8v, __builtin_amdgcn_raw_buffer_load_b128(rw, lane * 16,
                                                           wbase + ((s.wpos * TN + t) * 2 + p) * FRAG, 0));
    ++s.wpos;
}

// acc += tile (RB row blocks, KS k steps) x the stream's next KS k steps
template <int TN, int RB, bool TAIL>
__device__ __forceinline__ void tok_gemm(f4v (&acc)[RB][TN], const char *tile, TokState<TN, RB> &s,
                                         __amdgpu_buffer_rsrc_t rw, int wbase, int lane, int steps) {
    using K = TokCfg<TN, RB>;
    h8v a[2][RB][2];  // this k step's operands and the next one's
    const int fr0 = frag_slot(0, lane >> 4, lane & 15), fr1 = frag_slot(1, lane >> 4, lane & 15);
    auto read = [&](int ks) __attribute__((always_inline)) {
#pragma unroll
        for (int p = 1; p >= 0; --p)
#pragma unroll
            for (int rb = 0; rb < RB; ++rb)
                a[ks & 1][rb][p] = *reinterpret_cast<const h8v *>(tile + ((rb * K::KS + ks) * 2 + p) * FRAG + (ks & 1 ? fr1 : fr0));
    };
    read(0);
#pragma unroll
    for (int ks = 0; ks < K::KS; ++ks) {
        const int slot = ks % K::WD;
        if (K::PRE && ks + 1 < K::KS) read(ks + 1);
        if (!K::PRE && ks) read(ks);
#pragma unroll
        for (int m = 0; m < 3; ++m)
#pragma unroll
            for (int rb = 0; rb < RB; ++rb)
#pragma unroll
                for (int t = 0; t < TN; ++t)
                    acc[rb][t] = MFMA16H(s.w[slot][t][m == 1], a[ks & 1][rb][m == 0], acc[rb][t]);
        if (!TAIL || s.wpos < steps) tok_load<TN, RB>(s, slot, rw, wbase, lane);
        // (without it the compiler hoists later steps' operand reads and spills)
        __builtin_amdgcn_sched_barrier(0);
    }
}

}  // namespace

template <int TN, int RB> __global__ __launch_bounds__(256, 2) void k_token_mlp(TokMlpArgs g) {
    using K = TokCfg<TN, RB>;
    constexpr int KS = K::KS, CP = K::CP;
    __shared__ __attribute__((aligned(16))) char P0[RB * KS * 2 * FRAG];
    __shared__ __attribute__((aligned(16))) char P1[RB * KS * 2 * FRAG];
    // per row: 4 waves' (sum, sum of squares) of LN2; LN1's, the 4 waves' max
    // |x| and o's row unscale lie in P1, which is free until the first chunk
    __shared__ __attribute__((aligned(16))) float red2[RB * 16][8];
    __shared__ __attribute__((aligned(16))) float lnp[4 * CP];  // LN1, LN2 weights and biases
    float(*const red1)[8] = reinterpret_cast<float(*)[8]>(P1);
    float(*const redm)[4] = reinterpret_cast<float(*)[4]>(P1 + RB * 512);
    float *const osc = reinterpret_cast<float *>(P1 + RB * 768);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int j = lane & 15, q = lane >> 4;
    const int C = g.C;
    const size_t plane = (size_t)g.M * C * 4;
    const int steps = (1 + 2 * g.chunks) * KS;
    const __amdgpu_buffer_rsrc_t rw = buf_rsrc(g.w, (size_t)4 * steps * TN * 2 * FRAG);
    const int wbase = wave * steps * TN * 2 * FRAG;
    const __amdgpu_buffer_rsrc_t rp = buf_rsrc(g.prm, (size_t)(8 + 2 * g.chunks) * CP * 4);
    const float inv_c = g.inv_c;

    for (int i = tid; i < CP; i += 256)
        reinterpret_cast<float4 *>(lnp)[i] = buf_load4(rp, 16 * i);

    TokState<TN, RB> st;

    // o rows of a task: wave w takes rows 4w .. 4w + 3 of each row block, 16
    // lanes a row, lane c float4s c, c + 16, ...
    float4 oa[RB][TN];
    f4v xn[RB][TN];  // the residual x at this lane's output columns
    int ooff[TN], off[TN], foff[TN];  // o's loads, this lane's output columns, their fragments
#pragma unroll
    for (int t = 0; t < TN; ++t) {
        const int f = j + 16 * t;
        ooff[t] = 4 * f < C ? ((4 * wave + q) * C + 4 * f) * 4 : BUF_OOB;
        const int c = 16 * (wave * TN + t) + 4 * q;
        off[t] = c < C ? (j * C + c) * 4 : BUF_OOB;
        foff[t] = frag_col(wave * TN + t, j, q);
    }
    const int osto = (j >> 3) * 2 * FRAG + frag_slot(j >> 3, (j >> 1) & 3, 4 * wave + q) + (j & 1) * 8;
    const int nrb = g.M / 16;
    auto load_rows = [&](int r0) __attribute__((always_inline)) {
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
            const __amdgpu_buffer_rsrc_t r = buf_rsrc(g.o, r0 + rb < nrb ? plane : 0);
#pragma unroll
            for (int i = 0; i < TN; ++i) oa[rb][i] = buf_load4s(r, ooff[i], (r0 + rb) * 16 * C * 4);
        }
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
            const __amdgpu_buffer_rsrc_t r = buf_rsrc(g.x, r0 + rb < nrb ? plane : 0);
#pragma unroll
            for (int t = 0; t < TN; ++t)
                xn[rb][t] = __builtin_bit_cast(f4v, buf_load4s(r, off[t], (r0 + rb) * 16 * C * 4));
        }
    };
    // the parameter row `a`'s values at this lane's columns of tile t
    auto prm4 = [&](int a, int t) __attribute__((always_inline)) {
        return __builtin_bit_cast(f4v, buf_load4s(rp, 16 * q, (a * CP + 16 * (wave * TN + t)) * 4));
    };
    auto store_frag = [&](char *tile, int rb, int t, f4v v) __attribute__((always_inline)) {
        h4v hi, lo;
        split4(v, hi, lo);
        char *d = tile + foff[t] + rb * KS * 2 * FRAG;
        *reinterpret_cast<h4v *>(d) = hi;
        *reinterpret_cast<h4v *>(d + FRAG) = lo;
    };

    load_rows(blockIdx.x * RB);
    // as many dropped stores as a task's output has: the loop is entered with
    // the same queue (o's loads, then stores) as it loops back with, so that
    // the wait for o does not wait for the stores
#pragma unroll
    for (int i = 0; i < RB * TN; ++i) buf_store4(buf_rsrc(g.out, 0), 16 * i, make_float4(0.f, 0.f, 0.f, 0.f));
#pragma unroll 1
    for (int r0 = blockIdx.x * RB; r0 < nrb; r0 += gridDim.x * RB) {
        // (a row block past the end reads zeros and stores nothing)
        auto plane_of = [&](const float *p, int rb) __attribute__((always_inline)) {
            return buf_rsrc(p, r0 + rb < nrb ? plane : 0);
        };
        st.wpos = 0;
#pragma unroll
        for (int s = 0; s < K::WD; ++s) tok_load<TN, RB>(st, s, rw, wbase, lane);
        __builtin_amdgcn_sched_barrier(0);
        // ---- o into P0 ----
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
            float m = 0.f;
#pragma unroll
            for (int i = 0; i < TN; ++i) {
                const float4 v = oa[rb][i];
                m = fmaxf(m, fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
            }
            const int e = bound_exp(row16_max(m));
            const float sc = exp_scale(e);
            const int r = 4 * wave + q;
            if (j == 0) osc[rb * 16 + r] = exp_unscale(e);
#pragma unroll
            for (int i = 0; i < TN; ++i) {
                h4v hi, lo;
                split4(__builtin_bit_cast(f4v, oa[rb][i]) * sc, hi, lo);
                char *d = P0 + osto + (rb * KS * 2 + 4 * i) * FRAG;
                *reinterpret_cast<h4v *>(d) = hi;
                *reinterpret_cast<h4v *>(d + FRAG) = lo;
            }
        }
        f4v x1[RB][TN];
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
#pragma unroll
            for (int t = 0; t < TN; ++t) x1[rb][t] = xn[rb][t];
        lds_sync();

        // ---- proj, LN1, residual ----
        f4v acc[RB][TN];
        f4v cs[TN], b[TN];  // the GEMM's column unscales and biases, loaded ahead of it
        auto load_cb = [&](int a) __attribute__((always_inline)) {
#pragma unroll
            for (int t = 0; t < TN; ++t) {
                cs[t] = prm4(a, t);
                b[t] = prm4(a + 1, t);
            }
        };
        load_cb(4);
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
#pragma unroll
            for (int t = 0; t < TN; ++t) acc[rb][t] = f4v{0.f, 0.f, 0.f, 0.f};
        tok_gemm<TN, RB, false>(acc, P0, st, rw, wbase, lane, steps);

        // v = acc scaled back + bias, its row sums (and max |x1|'s part) to
        // LDS; after the barrier the rows' mean and 1/std
        float mean[RB], rstd[RB];
        auto norm_stats = [&](float(*red)[8], const float (&un)[RB]) __attribute__((always_inline)) {
#pragma unroll
            for (int rb = 0; rb < RB; ++rb) {
                float s1 = 0.f, s2 = 0.f;
#pragma unroll
                for (int t = 0; t < TN; ++t)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const float v = fmaf(acc[rb][t][i] * cs[t][i], un[rb], b[t][i]);
                        acc[rb][t][i] = v;
                        s1 += v;
                        s2 = fmaf(v, v, s2);
                    }
                const float s = xrow_sum2(s1, s2);
                if (lane < 32) red[rb * 16 + j][2 * wave + q] = s;
            }
        };
        auto norm_finish = [&](const float(*red)[8]) __attribute__((always_inline)) {
#pragma unroll
            for (int rb = 0; rb < RB; ++rb) {
                const float4 u = *reinterpret_cast<const float4 *>(&red[rb * 16 + j][0]);
                const float4 v = *reinterpret_cast<const float4 *>(&red[rb * 16 + j][4]);
                const float m = ((u.x + u.z) + (v.x + v.z)) * inv_c;
                const float var = fmaxf(((u.y + u.w) + (v.y + v.w)) * inv_c - m * m, 0.f);
                rstd[rb] = __builtin_amdgcn_rsqf(var + 1e-5f);
                mean[rb] = m * rstd[rb];
            }
        };
        auto load_ln = [&](int a, f4v(&lw)[TN], f4v(&lb)[TN]) __attribute__((always_inline)) {
#pragma unroll
            for (int t = 0; t < TN; ++t) {
                const float *d = lnp + a * CP + 16 * (wave * TN + t) + 4 * q;
                lw[t] = *reinterpret_cast<const f4v *>(d);
                lb[t] = *reinterpret_cast<const f4v *>(d + CP);
            }
        };
        float un[RB];
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) un[rb] = osc[rb * 16 + j];
        norm_stats(red1, un);
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
            float m = 0.f;
#pragma unroll
            for (int t = 0; t < TN; ++t)
#pragma unroll
                for (int i = 0; i < 4; ++i) m = fmaxf(m, fabsf(x1[rb][t][i]));
            m = xrow_max(m);
            if (lane < 16) redm[rb * 16 + j][wave] = m;
        }
        lds_sync();
        norm_finish(red1);
        float hsc[RB];  // the hidden rows' scale (its inverse into un)
        {
            f4v lw[TN], lb[TN];
            load_ln(0, lw, lb);
            float hun[RB];
#pragma unroll
            for (int rb = 0; rb < RB; ++rb) {
                const float4 m4 = *reinterpret_cast<const float4 *>(&redm[rb * 16 + j][0]);
                const float bx = fmaxf(fmaxf(m4.x, m4.y), fmaxf(m4.z, m4.w)) + g.ln1_bound;
                const int e = bound_exp(bx);
                const int eh = bound_exp(fmaf(bx, g.fc1_l1, g.fc1_bmax));
                const float sc = exp_scale(e);
                un[rb] = exp_unscale(e);
                hsc[rb] = exp_scale(eh);
                hun[rb] = exp_unscale(eh);
#pragma unroll
                for (int t = 0; t < TN; ++t) {
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        x1[rb][t][i] += fmaf(fmaf(acc[rb][t][i], rstd[rb], -mean[rb]), lw[t][i], lb[t][i]);
                    store_frag(P0, rb, t, x1[rb][t] * sc);
                    // (kept in the output until LN2: its registers are
                    // wanted in the MLP loop)
                    buf_store4s(plane_of(g.out, rb), off[t], (r0 + rb) * 16 * C * 4, __builtin_bit_cast(float4, x1[rb][t]));
                }
            }
            lds_sync();

            // ---- the MLP, a C-wide chunk of the hidden layer at a time ----
            f4v acc2[RB][TN];
#pragma unroll
            for (int rb = 0; rb < RB; ++rb)
#pragma unroll
                for (int t = 0; t < TN; ++t) acc2[rb][t] = f4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
            for (int h = 0; h < g.chunks; ++h) {
#pragma unroll
                for (int rb = 0; rb < RB; ++rb)
#pragma unroll
                    for (int t = 0; t < TN; ++t) acc[rb][t] = f4v{0.f, 0.f, 0.f, 0.f};
                load_cb(8 + 2 * h);
                tok_gemm<TN, RB, false>(acc, P0, st, rw, wbase, lane, steps);
                if (h) lds_sync();  // every wave is past the last chunk's fc2
#pragma unroll
                for (int rb = 0; rb < RB; ++rb)
#pragma unroll
                    for (int t = 0; t < TN; ++t) {
                        f4v v;
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            v[i] = gelu_erf(fmaf(acc[rb][t][i] * cs[t][i], un[rb], b[t][i])) * hsc[rb];
                        store_frag(P1, rb, t, v);
                    }
                lds_sync();
                load_cb(6);  // (used after the last chunk)
                if (h + 1 == g.chunks)
#pragma unroll
                    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
                        for (int t = 0; t < TN; ++t)
                            x1[rb][t] = __builtin_bit_cast(f4v, buf_load4s(plane_of(g.out, rb), off[t], (r0 + rb) * 16 * C * 4));
                tok_gemm<TN, RB, true>(acc2, P1, st, rw, wbase, lane, steps);
            }
#pragma unroll
            for (int rb = 0; rb < RB; ++rb) {
                un[rb] = hun[rb];
#pragma unroll
                for (int t = 0; t < TN; ++t) acc[rb][t] = acc2[rb][t];
            }
        }
        load_rows(r0 + gridDim.x * RB);
        norm_stats(red2, un);
        lds_sync();
        norm_finish(red2);
        f4v lw[TN], lb[TN];
        load_ln(2, lw, lb);
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
#pragma unroll
            for (int t = 0; t < TN; ++t) {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    x1[rb][t][i] += fmaf(fmaf(acc[rb][t][i], rstd[rb], -mean[rb]), lw[t][i], lb[t][i]);
                buf_store4s(plane_of(g.out, rb), off[t], (r0 + rb) * 16 * C * 4, __builtin_bit_cast(float4, x1[rb][t]));
            }
    }
}

// ---------------------------------------------------------------------------
// k_qkv_attn: a block's qkv projection and window attention in one kernel, for
// 6 heads of 30 and 6 heads of 10 (every released checkpoint). An item is a
// window and a group of its heads (two of 30, all six of 10): 64 tokens, 60 q, 60
// k and 60 v columns. Per item a workgroup
//   - loads the window's token rows (the block's shifted-window order, with
//     torch.roll's wrap), an item ahead, scales and splits them into LDS;
//   - multiplies them by the group's q|k|v weights, streamed from L2 through
//     registers: each wave owns three 16-column tiles, two of q or k (weights
//     as the MFMA's A operand: a lane holds a token's consecutive columns) and
//     one of v (tokens as A: a lane holds a column's consecutive tokens);
//   - normalises q and k (a head's columns are in one wave, so the norm is one
//     reduction over the lanes), splits q, k and v and writes them over the
//     token tile as the operands of the two attention products;
//   - S^T = K Q^T, the CPB bias, the shift mask and the softmax with a lane
//     holding one query, then O^T = V^T P^T with P straight from the registers
//     (the k slots of that product are numbered as S^T's accumulator rows, so
//     P needs no exchange between lanes); row HD of V^T is ones, so that row of
//     O^T is the softmax denominator.
// Head columns are padded to whole tiles: 30 to 32, 10 to 16. The scales: x's
// rows from their maximum; q and k are unit vectors (2^14); the probabilities
// are at most 1 (2^14, in the exponent's argument); v from the bound max|x|
// max_j sum_k |Wv[j][k]| + max|bv|, over the window or token by token (VSPAN).
//
// Items go to workgroups as window w on XCD w % 8, a window's groups one after
// another, so they read its rows through one L2. MI355X, 69,696 tokens x 180: 80
// us (77-83; the fp32 MFMA form with the weights in registers took 146); 2,880 tokens
// 13.4 (19.9). 6 heads of 10: 5,184 tokens 13.7 us and 526,592 296, where the
// qkv GEMM and the attention as two kernels took 20.6 and 355. With three
// workgroups per CU (168 registers) the form of 30 spills 76 registers.
// ---------------------------------------------------------------------------
typedef float f16acc __attribute__((ext_vector_type(16)));
#define MFMA32H(a, b, c) __builtin_amdgcn_mfma_f32_32x32x16_f16((a), (b), (c), 0, 0, 0)

namespace {

template <int HD> struct QaCfg {
    static constexpr int NW = HD > 16 ? 4 : 6;       // waves
    static constexpr int NG = HD > 16 ? 3 : 1;       // head groups
    static constexpr int GH = 6 / NG;                // heads per group
    static constexpr int C = 6 * HD;
    static constexpr int TF = (C + 63) / 64;         // float4s of a row per lane of 16
    static constexpr int KS = 2 * TF;                // k steps of the projection
    static constexpr int DS = HD > 16 ? 2 : 1;       // k steps of q . k
    static constexpr int VR = HD > 16 ? 32 : 16;     // rows of a v operand
    static constexpr int QB = DS * 2 * FRAG;         // bytes of 32 queries of a head
    static constexpr int VB = 2 * VR * 32;           // bytes of 16 keys of a head's v, both parts
    static constexpr int HB = 4 * QB + 4 * VB;       // bytes of a head: q, k, v
    static constexpr int TILE = 4 * KS * 2 * FRAG;   // bytes of the token tile
    static constexpr int BUF = GH * HB > TILE ? GH * HB : TILE;
};
// Tokens of a window share v's scale while their bounds lie within 2^VSPAN of each
// other, as they do in real images. Further apart each has its own, and the
// probabilities take what it lies below the largest, since a query that sees only
// small tokens is owed their precision: an output is then at most 1.8e-5 of sum P |v|
// off at any distance (in fp32 2.7e-5). With a shared scale it was that at 2^10
// too, 2.6e-5 at 2^20 and 0.8 at 2^40. At 264 x 264 windows that all spread take 86
// us against 84 (heads of 30) and 56 against 54 (of 10).
constexpr int VSPAN = 6;

}  // namespace

template <int HD> __global__ __launch_bounds__(64 * QaCfg<HD>::NW, 2) void k_qkv_attn(QkvAttnArgs g) {
    using K = QaCfg<HD>;
    constexpr int KS = K::KS, C = K::C, NW = K::NW, TF = K::TF, DS = K::DS, NT = 64 * NW;
    constexpr int SUM_E = 4 * (HD / 8) + (HD % 8) % 4, SUM_HH = (HD % 8) / 4;
    constexpr int NST = (64 + NT / 16 - 1) / (NT / 16);  // output stores per thread
    __shared__ __attribute__((aligned(16))) char buf[K::BUF];
    __shared__ __attribute__((aligned(16))) float xun[64];  // the rows' unscale
    __shared__ __attribute__((aligned(16))) float xmx[64];  // the rows' max |x|
    // v's scale per token, and what it lies below the largest token's (wide windows)
    __shared__ __attribute__((aligned(16))) float vsc[64], vlow[64];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int j = lane & 15, q = lane >> 4;
    const int r = lane & 31, hh = lane >> 5;
    const int shift = g.shift;
    const __amdgpu_buffer_rsrc_t rx = buf_rsrc(g.x, (size_t)g.hp * g.wp * C * 4);
    const __amdgpu_buffer_rsrc_t ro = buf_rsrc(g.out, (size_t)g.hp * g.wp * C * 4);
    const __amdgpu_buffer_rsrc_t rw = buf_rsrc(g.w, (size_t)K::NG * NW * KS * 6 * FRAG);
    const __amdgpu_buffer_rsrc_t rp = buf_rsrc(g.prm, (size_t)K::NG * NW * 3 * 32 * 4);

    // items of this XCD: window xcd + 8 (i / NG), group i % NG
    const int xcd = blockIdx.x & 7;
    const int nitem = ((g.nw - xcd + 7) >> 3) * K::NG, istep = gridDim.x >> 3;

    // x rows of an item: wave w < 4 takes tokens 16 rb + 4 w + q, 16 lanes a row
    float4 xa[4][TF];
    auto load_x = [&](int it) __attribute__((always_inline)) {
        const int wi = xcd + 8 * (it / K::NG);
        const int wh = wi / g.nww, ww = wi - wh * g.nww;
        const bool on = it < nitem;
#pragma unroll
        for (int rb = 0; rb < 4; ++rb) {
            const int t = 16 * rb + 4 * wave + q;
            int y = 8 * wh + (t >> 3) + shift;
            if (y >= g.hp) y -= g.hp;
            int x = 8 * ww + (t & 7) + shift;
            if (x >= g.wp) x -= g.wp;
            const int o = ((y * g.wp + x) * C + 4 * j) * 4;
#pragma unroll
            for (int i = 0; i < TF; ++i) xa[rb][i] = buf_load4(rx, on && 4 * (j + 16 * i) < C ? o + 256 * i : BUF_OOB);
        }
    };
    h8v w[2][3][2];
    int wbase = 0;
    auto load_w = [&](int ks) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < 3; ++t)
#pragma unroll
            for (int p = 0; p < 2; ++p)
                w[ks & 1][t][p] = __builtin_bit_cast(
                    h8v, __builtin_amdgcn_raw_buffer_load_b128(rw, lane * 16, wbase + ((ks * 3 + t) * 2 + p) * FRAG, 0));
    };

    const int fr0 = frag_slot(0, q, j), fr1 = frag_slot(1, q, j);
    const int osto = (j >> 3) * 2 * FRAG + frag_slot(j >> 3, (j >> 1) & 3, 4 * (wave & 3) + q) + (j & 1) * 8;

    int it = blockIdx.x >> 3;
    if (wave < 4) load_x(it);
#pragma unroll 1
    for (; it < nitem; it += istep) {
        const int hg = it % K::NG;
        const int wi = xcd + 8 * (it / K::NG);
        const int wh = wi / g.nww, ww = wi - wh * g.nww;
        wbase = (hg * NW + wave) * KS * 6 * FRAG;
        load_w(0);
        load_w(1);
        // the tiles' column unscales and biases: q and k tiles as the lane's 4
        // columns, the v tile as its one
        f4v cs[2], bi[2];
        float csv, biv;
        {
            const int pb = (hg * NW + wave) * 96 * 4;
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                cs[t] = __builtin_bit_cast(f4v, buf_load4s(rp, 16 * q, pb + t * 128));
                bi[t] = __builtin_bit_cast(f4v, buf_load4s(rp, 16 * q, pb + t * 128 + 64));
            }
            csv = buf_load1(rp, pb + 256 + 4 * j);
            biv = buf_load1(rp, pb + 320 + 4 * j);
        }
        // ---- x into the token tile ----
        if (wave < 4) {
#pragma unroll
            for (int rb = 0; rb < 4; ++rb) {
                float m = 0.f;
#pragma unroll
                for (int i = 0; i < TF; ++i) {
                    const float4 v = xa[rb][i];
                    m = fmaxf(m, fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
                }
                m = row16_max(m);
                const int e = bound_exp(m);
                const float sc = exp_scale(e);
                if (j == 0) {
                    xun[16 * rb + 4 * wave + q] = exp_unscale(e);
                    xmx[16 * rb + 4 * wave + q] = m;
                }
#pragma unroll
                for (int i = 0; i < TF; ++i) {
                    h4v hi, lo;
                    split4(__builtin_bit_cast(f4v, xa[rb][i]) * sc, hi, lo);
                    char *d = buf + osto + (rb * KS * 2 + 4 * i) * FRAG;
                    *reinterpret_cast<h4v *>(d) = hi;
                    *reinterpret_cast<h4v *>(d + FRAG) = lo;
                }
            }
        }
        lds_sync();

        // ---- q | k | v ----
        f4v acc[4][3];
#pragma unroll
        for (int rb = 0; rb < 4; ++rb)
#pragma unroll
            for (int t = 0; t < 3; ++t) acc[rb][t] = f4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            h8v a[4][2];
#pragma unroll
            for (int p = 1; p >= 0; --p)
#pragma unroll
                for (int rb = 0; rb < 4; ++rb)
                    a[rb][p] = *reinterpret_cast<const h8v *>(buf + ((rb * KS + ks) * 2 + p) * FRAG + (ks & 1 ? fr1 : fr0));
#pragma unroll
            for (int m = 0; m < 3; ++m)
#pragma unroll
                for (int rb = 0; rb < 4; ++rb) {
#pragma unroll
                    for (int t = 0; t < 2; ++t)
                        acc[rb][t] = MFMA16H(w[ks & 1][t][m == 1], a[rb][m == 0], acc[rb][t]);
                    acc[rb][2] = MFMA16H(a[rb][m == 0], w[ks & 1][2][m == 1], acc[rb][2]);
                }
            if (ks + 2 < KS) load_w(ks + 2);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (wave < 4) load_x(it + istep);
        // v's scale, from the bound of |v| of the window's largest row, or of each
        // token's own where the rows lie further apart than 2^VSPAN (`wide`)
        const float vb = fmaf(xmx[lane], g.v_l1, g.v_bmax);
        const int ev = __builtin_amdgcn_readfirstlane(bound_exp(xrow_max(row16_max(vb))));
        const bool wide = ev - __builtin_amdgcn_readfirstlane(bound_exp(-xrow_max(row16_max(-vb)))) > VSPAN;
        if (wave == 0) {
            const int et = wide ? max(bound_exp(vb), ev - 60) : ev;
            vsc[lane] = exp_scale(et);
            vlow[lane] = __builtin_bit_cast(float, (127 + et - ev) << 23);
        }
        lds_sync();  // every wave has read the token tile
        {
            // q and k: unit vectors times 2^14. A head of 30 has both tiles
            // (q in waves 0-1, k in waves 2-3), a head of 10 one of each
            char *dq[2];
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const int head = DS == 2 ? (wave & 1) : wave;
                const int isk = DS == 2 ? (wave >> 1) : t;
                const int st = DS == 2 ? t : 0;
                dq[t] = buf + head * K::HB + isk * 2 * K::QB + st * 2 * FRAG + ((q >> 1) * 32 + j) * 16 + (q & 1) * 8;
            }
#pragma unroll
            for (int rb = 0; rb < 4; ++rb) {
                const float un = xun[16 * rb + j];
                float ss[2];
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    ss[t] = 0.f;
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const float v = fmaf(acc[rb][t][i] * cs[t][i], un, bi[t][i]);
                        acc[rb][t][i] = v;
                        ss[t] = fmaf(v, v, ss[t]);
                    }
                }
                if (DS == 2) ss[0] = ss[1] = xrow_sum(ss[0] + ss[1]);
                else {
                    ss[0] = xrow_sum(ss[0]);
                    ss[1] = xrow_sum(ss[1]);
                }
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const float n = 16384.f * __builtin_amdgcn_rsqf(fmaxf(ss[t], 1e-24f));
                    h4v hi, lo;
                    split4(acc[rb][t] * n, hi, lo);
                    char *d = dq[t] + (rb >> 1) * K::QB + (rb & 1) * 256;
                    *reinterpret_cast<h4v *>(d) = hi;
                    *reinterpret_cast<h4v *>(d + FRAG) = lo;
                }
            }
            // v: row d, 16 keys 16 rb .. a fragment, the ones row at d = HD
            const int vh = DS == 2 ? (wave >> 1) : wave, d = DS == 2 ? 16 * (wave & 1) + j : j;
            char *dv = buf + vh * K::HB + 4 * K::QB + ((q & 1) * K::VR + d) * 16 + (q >> 1) * 8;
#pragma unroll
            for (int rb = 0; rb < 4; ++rb) {
                const f4v un = *reinterpret_cast<const f4v *>(&xun[16 * rb + 4 * q]);
                const f4v sc = *reinterpret_cast<const f4v *>(&vsc[16 * rb + 4 * q]);
                f4v v;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    v[i] = fmaf(acc[rb][2][i] * csv, un[i], biv) * sc[i];
                    v[i] = d == HD ? 1.0f : v[i];
                }
                h4v hi, lo;
                split4(v, hi, lo);
                *reinterpret_cast<h4v *>(dv + rb * K::VB) = hi;
                *reinterpret_cast<h4v *>(dv + rb * K::VB + K::VB / 2) = lo;
            }
        }
        lds_sync();

        // ---- attention: this wave's head, 32 queries at a time ----
#pragma unroll
        for (int jb = 0; jb < 3 - DS; ++jb) {
            const int hl = DS == 2 ? (wave >> 1) : wave, qt = DS == 2 ? (wave & 1) : jb;
            const int head = hg * K::GH + hl, qtok = 32 * qt + r;
            char *const hb = buf + hl * K::HB;
            const float *cp = g.cpbt + ((size_t)head * 64 + qtok) * 64 + 4 * hh;
            f4v cb[2][4];
#pragma unroll
            for (int kt = 0; kt < 2; ++kt)
#pragma unroll
                for (int a = 0; a < 4; ++a) cb[kt][a] = *reinterpret_cast<const f4v *>(cp + 32 * kt + 8 * a);
            // logit scale x log2(e), the two 2^14 taken out
            const float ls = ATTN_LOG2E * __expf(fminf(g.logit_scale[head], 4.605170185988092f)) * (1.0f / 268435456.0f);
            h8v qf[DS][2];
#pragma unroll
            for (int s = 0; s < DS; ++s)
#pragma unroll
                for (int p = 0; p < 2; ++p)
                    qf[s][p] = *reinterpret_cast<const h8v *>(hb + qt * K::QB + (s * 2 + p) * FRAG + lane * 16);
            f16acc sa[2];
#pragma unroll
            for (int kt = 0; kt < 2; ++kt) {
                h8v kf[DS][2];
#pragma unroll
                for (int s = 0; s < DS; ++s)
#pragma unroll
                    for (int p = 0; p < 2; ++p)
                        kf[s][p] = *reinterpret_cast<const h8v *>(hb + (2 + kt) * K::QB + (s * 2 + p) * FRAG + lane * 16);
#pragma unroll
                for (int e = 0; e < 16; ++e) sa[kt][e] = 0.f;
#pragma unroll
                for (int m = 0; m < 3; ++m)
#pragma unroll
                    for (int s = 0; s < DS; ++s) sa[kt] = MFMA32H(kf[s][m == 1], qf[s][m == 0], sa[kt]);
            }
#pragma unroll
            for (int kt = 0; kt < 2; ++kt)
#pragma unroll
                for (int e = 0; e < 16; ++e) sa[kt][e] = fmaf(sa[kt][e], ls, cb[kt][e >> 2][e & 3]);
            // shift mask (last window row / column of a shifted block)
            const bool ey = shift && (wh * 8 + 8 >= g.hp);
            const bool ex = shift && (ww * 8 + 8 >= g.wp);
            if (ey || ex) {
                const bool qy = (qtok >> 3) < 8 - shift;
                const bool qx = (qtok & 7) < 8 - shift;
#pragma unroll
                for (int kt = 0; kt < 2; ++kt)
#pragma unroll
                    for (int e = 0; e < 16; ++e) {
                        const int krw = 4 * kt + (e >> 2);
                        const int kcl = 4 * hh + (e & 3);
                        const bool dy = ey && ((krw < 8 - shift) != qy);
                        const bool dx = ex && ((kcl < 8 - shift) != qx);
                        if (dy || dx) sa[kt][e] -= 100.f * ATTN_LOG2E;
                    }
            }
            float mx = -INFINITY;
#pragma unroll
            for (int kt = 0; kt < 2; ++kt)
#pragma unroll
                for (int e = 0; e < 16; ++e) mx = fmaxf(mx, sa[kt][e]);
            mx = half_max(mx);
            f16acc o;
#pragma unroll
            for (int e = 0; e < 16; ++e) o[e] = 0.f;
            const char *vb = hb + 4 * K::QB + (hh * K::VR + (r & (K::VR - 1))) * 16;
            // o += V^T P^T, P from its value at sa[kt][e]
            auto pv = [&](auto prob) __attribute__((always_inline)) {
#pragma unroll
                for (int kt = 0; kt < 2; ++kt)
#pragma unroll
                    for (int s = 0; s < 2; ++s) {
                        const h8v vh = *reinterpret_cast<const h8v *>(vb + (2 * kt + s) * K::VB);
                        const h8v vl = *reinterpret_cast<const h8v *>(vb + (2 * kt + s) * K::VB + K::VB / 2);
                        h4v ph[2], pl[2];
#pragma unroll
                        for (int a = 0; a < 2; ++a) {
                            f4v p;
#pragma unroll
                            for (int b = 0; b < 4; ++b) p[b] = prob(sa[kt][8 * s + 4 * a + b]);
                            split4(p, ph[a], pl[a]);
                        }
                        const h8v p8 = __builtin_shufflevector(ph[0], ph[1], 0, 1, 2, 3, 4, 5, 6, 7);
                        const h8v l8 = __builtin_shufflevector(pl[0], pl[1], 0, 1, 2, 3, 4, 5, 6, 7);
                        o = MFMA32H(vh, l8, o);
                        o = MFMA32H(vl, p8, o);
                        o = MFMA32H(vh, p8, o);
                    }
            };
            float inv = exp_unscale(ev);
            if (!wide) {
                mx -= 14.0f;  // (probabilities times 2^14)
                pv([&](float v) __attribute__((always_inline)) { return __builtin_amdgcn_exp2f(v - mx); });
                float lo, hi;
                halves(o[SUM_E], lo, hi);
                inv /= SUM_HH ? hi : lo;
            } else {
                // the small tokens' v is held larger by 1 / vlow: the probabilities
                // times vlow, scaled anew by the query's largest such product, and
                // the denominator summed from the probabilities themselves
                float sum = 0.f, pm = 0.f;
#pragma unroll
                for (int kt = 0; kt < 2; ++kt)
#pragma unroll
                    for (int a = 0; a < 4; ++a) {
                        const f4v low = *reinterpret_cast<const f4v *>(&vlow[32 * kt + 8 * a + 4 * hh]);
#pragma unroll
                        for (int b = 0; b < 4; ++b) {
                            const float p = __builtin_amdgcn_exp2f(sa[kt][4 * a + b] - mx);
                            sum += p;
                            sa[kt][4 * a + b] = p * low[b];
                            pm = fmaxf(pm, p * low[b]);
                        }
                    }
                const int ep = bound_exp(half_max(pm));
                const float sc = exp_scale(ep);
                pv([&](float v) __attribute__((always_inline)) { return v * sc; });
                inv *= exp_unscale(ep) / half_sum(sum);
            }
            // O over this wave's own q operands, [32][HD] floats
            float *orow = reinterpret_cast<float *>(hb + qt * K::QB) + r * HD;
#pragma unroll
            for (int e = 0; e < 16; e += 2) {
                const int dd = 8 * (e >> 2) + 4 * hh + (e & 3);
                if (dd < HD) *reinterpret_cast<float2 *>(orow + dd) = make_float2(o[e] * inv, o[e + 1] * inv);
            }
        }
        lds_sync();
        // ---- out: 16 lanes a token, lane c float4 c of its 60 floats ----
        float4 ov[NST];
#pragma unroll
        for (int u = 0; u < NST; ++u) {
            const int t = min(u * (NT / 16) + (tid >> 4), 63), c4 = min(j, 14);
            float2 p[2];
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const int f = 2 * c4 + k, hl = f / (HD / 2), d2 = f - hl * (HD / 2);
                p[k] = *reinterpret_cast<const float2 *>(buf + hl * K::HB + (t >> 5) * K::QB + ((t & 31) * HD + 2 * d2) * 4);
            }
            ov[u] = make_float4(p[0].x, p[0].y, p[1].x, p[1].y);
        }
        lds_sync();  // every wave has read the buffer: the next token tile may land
#pragma unroll
        for (int u = 0; u < NST; ++u) {
            const int t = u * (NT / 16) + (tid >> 4);
            int y = 8 * wh + (t >> 3) + shift;
            if (y >= g.hp) y -= g.hp;
            int x = 8 * ww + (t & 7) + shift;
            if (x >= g.wp) x -= g.wp;
            buf_store4(ro, t < 64 && j < 15 ? ((y * g.wp + x) * C + hg * 60 + 4 * j) * 4 : BUF_OOB, ov[u]);
        }
    }
}

// ---------------------------------------------------------------------------
// k_split_conv: 3x3 stride-1 zero-pad-1 convolution of a channel-last plane, cin
// and cout at most 192, as one implicit GEMM on the split: + bias, then the
// residual or LeakyReLU.
//
// A workgroup makes a tile of 8 pixels by 2 RBT rows, RBT = RB 4 / WC row blocks
// of 2 x 8 pixels: WC waves side by side in the output columns (16 TN each), 4 /
// WC groups of waves below one another, RB row blocks each. The tile's halo is
// loaded a tile ahead, 16 lanes a pixel, each pixel scaled by its largest
// magnitude, split and kept in LDS as [k step][part][q][pixel], so that a tap is
// an offset; a tap's products are scaled back as they are added to the output's
// sum, a lane's products all being of one pixel, so what a pixel holds bears on
// its own footprint only, as in fp32. The nine taps' weights stream from L2
// through a register ring as in k_token_mlp. On a plane of few tiles CS workgroups
// (blockIdx.y) share one, each with its part of every wave's column tiles: a
// workgroup streams all of its columns' weights, 1.3 MB at 180 wide and 12 us
// through one CU's cache, however few its pixels. The pixel slots are permuted within
// 8 by q and the parity of the k step, for the writes' banks (frag_slot).
//
// Tiles go to workgroups in plane order within each XCD, so that halos are shared
// in its L2. MI355X: 264 x 264 x 180 in 127-137 us, where F(4x4,3x3) Winograd (a
// quarter of the multiply-adds, in fp32, and 560 MB of transform planes) took 176;
// 40 x 72 x 180 20.1 (31.7); 544 x 968 x 60 162 (338); 64 -> 64 at 1952 x 2592 1.29
// ms where the fp32 implicit GEMM took 3.1. 81 us of the first are MFMA issue at
// the clock the kernel runs at. One workgroup per CU with six row blocks per wave
// and operands read ahead: 138 us.
// ---------------------------------------------------------------------------
namespace {

template <int KSC, int TN, int RB, int WC> struct ConvCfg {
    static constexpr int RBT = RB * 4 / WC;
    static constexpr int TH = 2 * RBT;                    // tile rows
    static constexpr int NPIX = (TH + 2) * 10;            // halo pixels
    static constexpr int NP = (NPIX + 7) / 8 * 8;
    static constexpr int NV = KSC / 2;                    // float4s of a pixel per lane of 16
    static constexpr int NG = (NPIX + 15) / 16;           // pixels per 16 lanes
    static constexpr int STEP = 4 * NP * 16;              // bytes of a k step's part
};

}  // namespace

template <int KSC, int TN, int RB, int WC, int CS> __global__ __launch_bounds__(256, 2) void k_split_conv(SplitConvArgs g) {
    using K = ConvCfg<KSC, TN, RB, WC>;
    constexpr int NT = TN / CS;  // this workgroup's column tiles per wave, from n0
    const int n0 = CS > 1 ? blockIdx.y * NT : 0;
    __shared__ __attribute__((aligned(16))) char buf[2 * KSC * K::STEP];
    __shared__ float pun[K::NP];  // the pixels' unscale x 2^-15
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int j = lane & 15, q = lane >> 4;
    const int cw = wave % WC, rw = wave / WC;
    const __amdgpu_buffer_rsrc_t rw_ = buf_rsrc(g.w, (size_t)WC * (9 * KSC * TN * 2 * FRAG + 64 * TN));
    const int wbase = cw * 9 * KSC * TN * 2 * FRAG;
    const int tx = (g.W + 7) / 8, ty = (g.H + K::TH - 1) / K::TH, nt = tx * ty;
    // tiles of this XCD: a contiguous eighth
    const int xcd = blockIdx.x & 7;
    const int t0 = (int)((unsigned)nt * xcd / 8), t1 = (int)((unsigned)nt * (xcd + 1) / 8);
    const int istep = gridDim.x >> 3;

    // (an opaque copy per use: hoisted out of the tile loop, the addresses made
    // from it would not fit the registers)
    auto tid_of = [&]() __attribute__((always_inline)) {
        int i = tid;
        asm("" : "+v"(i));
        return i;
    };
    float4 v[K::NG][K::NV];
    auto load_tile = [&](int t) __attribute__((always_inline)) {
        const int by = t / tx, y0 = by * K::TH - 1, x0 = (t - by * tx) * 8 - 1;
        // a resource based at the tile's first row (the plane may pass 2 GiB)
        const size_t row = (size_t)g.W * g.cin * 4;
        const int ti = tid_of();
        const int yb = max(y0, 0);
        const __amdgpu_buffer_rsrc_t r = buf_rsrc(g.in + (size_t)yb * g.W * g.cin, t < t1 ? (size_t)(g.H - yb) * row : 0);
#pragma unroll
        for (int i = 0; i < K::NG; ++i) {
            const int pix = (ti >> 4) + 16 * i, f = ti & 15, py = pix / 10, y = y0 + py, x = x0 + pix - 10 * py;
            const bool in = pix < K::NPIX && y >= 0 && y < g.H && x >= 0 && x < g.W;
            const int o = (((y - yb) * g.W + x) * g.cin + 4 * f) * 4;
#pragma unroll
            for (int u = 0; u < K::NV; ++u) v[i][u] = buf_load4(r, in && 4 * (f + 16 * u) < g.cin ? o + 256 * u : BUF_OOB);
        }
    };

    int t = t0 + (blockIdx.x >> 3);
    load_tile(t);
#pragma unroll 1
    for (; t < t1; t += istep) {
        // ---- the pixels' scales, and their split into LDS ----
        lds_sync();  // every wave is past the last tile's reads
        const int ti = tid_of();
#pragma unroll
        for (int i = 0; i < K::NG; ++i) {
            const int pix = (ti >> 4) + 16 * i, f = ti & 15;
            f4v p[K::NV];
            float m = 0.f;
#pragma unroll
            for (int u = 0; u < K::NV; ++u) {
                p[u] = __builtin_bit_cast(f4v, v[i][u]);
#pragma unroll
                for (int b = 0; b < 4; ++b) m = fmaxf(m, fabsf(p[u][b]));
            }
            m = row16_max(m);
            const int e = bound_exp(m);
            float sc = exp_scale(e), un = exp_unscale(e) * 0x1p-15f;
            if (m == INFINITY) {
                // its infinities (as 1) and NaNs alone count, its sums times
                // infinity
                sc = 16384.f;
                un = INFINITY;
#pragma unroll
                for (int u = 0; u < K::NV; ++u)
#pragma unroll
                    for (int b = 0; b < 4; ++b) {
                        const float x = p[u][b];
                        p[u][b] = fabsf(x) == INFINITY ? copysignf(1.f, x) : x != x ? x : 0.f;
                    }
            }
            if (16 * (i + 1) > K::NPIX && pix >= K::NPIX) continue;
            if (f == 0) pun[pix] = un;
#pragma unroll
            for (int u = 0; u < K::NV; ++u) {
                h4v hi, lo;
                split4(p[u] * sc, hi, lo);
                const int ks = 2 * u + (f >> 3), qf = (f >> 1) & 3;
                char *d = buf + 2 * ks * K::STEP + (qf * K::NP + (pix ^ (qf | (ks & 1) << 2))) * 16 + (f & 1) * 8;
                *reinterpret_cast<h4v *>(d) = hi;
                *reinterpret_cast<h4v *>(d + K::STEP) = lo;
            }
        }
        lds_sync();
        load_tile(t + istep);

        // ---- nine taps ----
        h8v w[2][NT][2];
        int wpos = wbase + n0 * 2 * FRAG;
        auto load_w = [&](int slot) __attribute__((always_inline)) {
#pragma unroll
            for (int n = 0; n < NT; ++n)
#pragma unroll
                for (int p = 0; p < 2; ++p)
                    w[slot][n][p] = __builtin_bit_cast(
                        h8v, __builtin_amdgcn_raw_buffer_load_b128(rw_, lane * 16, wpos + (n * 2 + p) * FRAG, 0));
            wpos += TN * 2 * FRAG;
        };
        load_w(0);
        load_w(1);
        // each tap is summed by itself, then scaled back and added: also a ninth
        // as long a chain of roundings at the sum's full size (largest error of
        // a 180-wide conv of unit normals against 64 bits 9.5e-7; 2.0e-6 with a
        // row of three taps in one chain, and an image 7.6e-8 off, now 6.3e-8)
        f4v tot[RB][NT];
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
#pragma unroll
            for (int n = 0; n < NT; ++n) tot[rb][n] = f4v{0.f, 0.f, 0.f, 0.f};
        const int pix0 = (2 * RB * rw + (j >> 3)) * 10 + (j & 7);
        int tap = 0;
#pragma unroll 1
        for (int dy = 0; dy < 3; ++dy)
#pragma unroll 1
            for (int dx = 0; dx < 3; ++dx, ++tap) {
                const char *ad[RB][2];
                float un[RB];
                f4v acc[RB][NT];
#pragma unroll
                for (int rb = 0; rb < RB; ++rb) {
                    const int pix = pix0 + (2 * rb + dy) * 10 + dx;
                    ad[rb][0] = buf + (q * K::NP + (pix ^ q)) * 16;
                    ad[rb][1] = buf + (q * K::NP + (pix ^ (q | 4))) * 16;
                    un[rb] = pun[pix];
#pragma unroll
                    for (int n = 0; n < NT; ++n) acc[rb][n] = f4v{0.f, 0.f, 0.f, 0.f};
                }
#pragma unroll
                for (int ks = 0; ks < KSC; ++ks) {
                    h8v a[RB][2];
#pragma unroll
                    for (int p = 1; p >= 0; --p)
#pragma unroll
                        for (int rb = 0; rb < RB; ++rb)
                            a[rb][p] = *reinterpret_cast<const h8v *>(ad[rb][ks & 1] + (2 * ks + p) * K::STEP);
#pragma unroll
                    for (int mm = 0; mm < 3; ++mm)
#pragma unroll
                        for (int rb = 0; rb < RB; ++rb)
#pragma unroll
                            for (int n = 0; n < NT; ++n)
                                acc[rb][n] = MFMA16H(w[ks & 1][n][mm == 1], a[rb][mm == 0], acc[rb][n]);
                    if (ks < KSC - 2 || tap < 8) load_w(ks & 1);
                    __builtin_amdgcn_sched_barrier(0);
                }
#pragma unroll
                for (int rb = 0; rb < RB; ++rb)
#pragma unroll
                    for (int n = 0; n < NT; ++n)
#pragma unroll
                        for (int i = 0; i < 4; ++i) tot[rb][n][i] = fmaf(acc[rb][n][i], un[rb], tot[rb][n][i]);
            }

        // ---- epilogue: lane (j, q) holds pixel j of each row block ----
        const int by = t / tx, x = (t - by * tx) * 8 + (j & 7);
        const int yt = by * K::TH;
        const __amdgpu_buffer_rsrc_t ro = buf_rsrc(g.out + (size_t)yt * g.W * g.cout, (size_t)(g.H - yt) * g.W * g.cout * 4);
        const __amdgpu_buffer_rsrc_t rr =
            buf_rsrc(g.res + (g.res ? (size_t)yt * g.W * g.cout : 0), g.res ? (size_t)(g.H - yt) * g.W * g.cout * 4 : 0);
#pragma unroll
        for (int n = 0; n < NT; ++n) {
            const int c = 16 * (cw * TN + n0 + n) + 4 * q;
            const f4v cs = __builtin_bit_cast(f4v, buf_load4(rw_, WC * 9 * KSC * TN * 2 * FRAG + 4 * c));
            const f4v b = __builtin_bit_cast(f4v, buf_load4(buf_rsrc(g.bias, g.bias ? (size_t)g.cout * 4 : 0), c * 4));
#pragma unroll
            for (int rb = 0; rb < RB; ++rb) {
                const int y = 2 * (RB * rw + rb) + (j >> 3);
                const int off = x < g.W && yt + y < g.H && c < g.cout ? ((y * g.W + x) * g.cout + c) * 4 : BUF_OOB;
                const f4v r = __builtin_bit_cast(f4v, buf_load4(rr, off));
                f4v o;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    o[i] = fmaf(tot[rb][n][i], cs[i], b[i]) + r[i];
                    if (g.lrelu) o[i] = o[i] >= 0.f ? o[i] : o[i] * g.slope;
                }
                buf_store4(ro, off, __builtin_bit_cast(float4, o));
            }
        }
    }
}

// ---- host side ------------------------------------------------------------

namespace {

uint16_t f16_bits(float f) {
    // round to nearest even; |f| < 2^15 by the scaling
    uint32_t x;
    memcpy(&x, &f, 4);
    const uint32_t sign = (x >> 16) & 0x8000u;
    const uint32_t a = x & 0x7fffffffu;
    if (a > 0x7f800000u) return (uint16_t)(sign | 0x7e00u);
    if (a >= 0x47800000u) return (uint16_t)(sign | 0x7c00u);
    if (a < 0x38800000u) {
        // subnormal: units of 2^-24 (the fp32 addition rounds to them)
        float m;
        memcpy(&m, &a, 4);
        const float r = m + 0.5f;
        uint32_t y;
        memcpy(&y, &r, 4);
        return (uint16_t)(sign | (y - 0x3f000000u));
    }
    const uint32_t r = a + 0xfffu + ((a >> 13) & 1u);
    return (uint16_t)(sign | ((r - 0x38000000u) >> 13));
}
float f16_value(uint16_t h) {
    const uint32_t e = (h >> 10) & 31, m = h & 0x3ffu, sign = (uint32_t)(h & 0x8000u) << 16;
    uint32_t x;
    if (e == 0) {
        const float v = (float)m * 5.9604644775390625e-8f;  // 2^-24 units
        memcpy(&x, &v, 4);
    } else {
        x = e == 31 ? 0x7f800000u | m << 13 : (e + 112) << 23 | m << 13;
    }
    x |= sign;
    float v;
    memcpy(&v, &x, 4);
    return v;
}

}  // namespace

float split_row_scale(const float *w, int n) {
    float m = 0.f;
    for (int i = 0; i < n; ++i) m = std::max(m, std::fabs(w[i]));
    if (!(m > 0.f) || !std::isfinite(m)) return 1.f;
    int e;
    (void)frexpf(m, &e);  // m = f 2^e, f in [0.5, 1)
    return ldexpf(1.f, std::min(std::max(15 - e, -126), 126));
}

void split_pack_step(const float *const *rows, const float *scale, int k0, int kn, uint16_t *dst) {
    for (int l = 0; l < 64; ++l) {
        const float *row = rows[l & 15];
        const float sc = scale[l & 15];
        for (int i = 0; i < 8; ++i) {
            const int k = k0 + 8 * (l >> 4) + i;
            const float v = row && k < kn ? row[k] * sc : 0.f;
            const uint16_t hi = f16_bits(v);
            dst[l * 8 + i] = hi;
            dst[512 + l * 8 + i] = f16_bits(v - f16_value(hi));
        }
    }
}

bool token_mlp_takes(int C, int ratio) { return C % 4 == 0 && C <= 192 && ratio >= 1; }
static int tok_tn(int C) { return (C + 63) / 64; }
size_t token_mlp_weight_floats(int C, int ratio) {
    const int tn = tok_tn(C);
    return (size_t)4 * (1 + 2 * ratio) * 2 * tn * tn * 2 * (FRAG / 4);
}
size_t token_mlp_param_floats(int C, int ratio) { return (size_t)(8 + 2 * ratio) * 64 * tok_tn(C); }

// [C][K] weights less each k's mean over the C columns.
static std::vector<float> centred(const float *w, int C, int K) {
    std::vector<double> mean(K, 0.0);
    for (int c = 0; c < C; ++c)
        for (int k = 0; k < K; ++k) mean[k] += w[(size_t)c * K + k];
    std::vector<float> out((size_t)C * K);
    for (int c = 0; c < C; ++c)
        for (int k = 0; k < K; ++k) out[(size_t)c * K + k] = (float)(w[(size_t)c * K + k] - mean[k] / C);
    return out;
}

void token_mlp_pack(const TokMlpWeights &h, int C, int ratio, float *w, float *prm, float *ln1_bound,
                    float *fc1_l1, float *fc1_bmax) {
    const int tn = tok_tn(C), CP = 64 * tn, ks = 2 * tn;
    uint16_t *dst = reinterpret_cast<uint16_t *>(w);
    std::fill(prm, prm + token_mlp_param_floats(C, ratio), 0.f);
    std::vector<float> sp(C), s2(C), s1((size_t)ratio * C);
    const std::vector<float> wproj = centred(h.wproj, C, C), w2 = centred(h.w2, C, ratio * C);
    const std::vector<float> bproj = centred(h.bproj, C, 1), b2 = centred(h.b2, C, 1);
    for (int c = 0; c < C; ++c) {
        sp[c] = split_row_scale(&wproj[(size_t)c * C], C);
        s2[c] = split_row_scale(&w2[(size_t)c * ratio * C], ratio * C);
        prm[c] = h.n1w[c];
        prm[CP + c] = h.n1b[c];
        prm[2 * CP + c] = h.n2w[c];
        prm[3 * CP + c] = h.n2b[c];
        prm[4 * CP + c] = 1.f / sp[c];
        prm[5 * CP + c] = bproj[c];
        prm[6 * CP + c] = 1.f / s2[c];
        prm[7 * CP + c] = b2[c];
    }
    float l1 = 0.f, bmax = 0.17f, nw = 0.f, nb = 0.f;
    for (int o = 0; o < ratio * C; ++o) {
        const float *row = h.w1 + (size_t)o * C;
        s1[o] = split_row_scale(row, C);
        const int ch = o / C, c = o % C;
        prm[(8 + 2 * ch) * CP + c] = 1.f / s1[o];
        prm[(9 + 2 * ch) * CP + c] = h.b1[o];
        double a = 0.0;
        for (int k = 0; k < C; ++k) a += std::fabs((double)row[k]);
        l1 = std::max(l1, (float)a);
        bmax = std::max(bmax, h.b1[o]);
    }
    for (int c = 0; c < C; ++c) {
        nw = std::max(nw, std::fabs(h.n1w[c]));
        nb = std::max(nb, std::fabs(h.n1b[c]));
    }
    *ln1_bound = sqrtf((float)C) * nw + nb;
    *fc1_l1 = l1;
    *fc1_bmax = bmax;
    // the stream of each wave: proj, then per chunk fc1 and fc2
    for (int wave = 0; wave < 4; ++wave)
        for (int gm = 0; gm < 1 + 2 * ratio; ++gm)
            for (int s = 0; s < ks; ++s)
                for (int t = 0; t < tn; ++t, dst += FRAG) {
                    const float *rows[16];
                    float sc[16];
                    const int ch = (gm - 1) / 2;
                    for (int r = 0; r < 16; ++r) {
                        const int c = 16 * (wave * tn + t) + r;
                        rows[r] = nullptr;
                        sc[r] = 0.f;
                        if (c >= C) continue;
                        if (gm == 0) {
                            rows[r] = &wproj[(size_t)c * C];
                            sc[r] = sp[c];
                        } else if (gm % 2 == 1) {
                            rows[r] = h.w1 + ((size_t)ch * C + c) * C;
                            sc[r] = s1[(size_t)ch * C + c];
                        } else {
                            rows[r] = &w2[(size_t)c * ratio * C + (size_t)ch * C];
                            sc[r] = s2[c];
                        }
                    }
                    split_pack_step(rows, sc, 32 * s, C, dst);
                }
}

// Workgroups that run at once (by registers and LDS).
static int tok_slots(int C) { return cu_count() * (tok_tn(C) > 1 ? 2 : 4); }
// Row blocks per task: the count whose rounds over those slots take least, a
// round costing its row blocks plus a constant of about one (its weight stream,
// barriers and latencies).
int token_mlp_row_blocks(int M, int C) {
    const int nrb = M / 16, slots = tok_slots(C);
    int best = 1;
    long best_cost = 0;
    for (int rb = 1; rb <= 3; ++rb) {
        const int tasks = (nrb + rb - 1) / rb;
        const long cost = (long)((tasks + slots - 1) / slots) * (rb + 1);
        if (rb == 1 || cost <= best_cost) {
            best = rb;
            best_cost = cost;
        }
    }
    return best;
}

unsigned token_mlp_grid(int M, int C) {
    const int rb = token_mlp_row_blocks(M, C), tasks = (M / 16 + rb - 1) / rb;
    return (unsigned)std::max(1, std::min(tasks, tok_slots(C)));
}

template <int TN> static void tok_launch(const TokMlpArgs &g, int rb, dim3 grid, hipStream_t st) {
    switch (rb) {
    case 1: hipLaunchKernelGGL((k_token_mlp<TN, 1>), grid, dim3(256), 0, st, g); break;
    case 2: hipLaunchKernelGGL((k_token_mlp<TN, 2>), grid, dim3(256), 0, st, g); break;
    default: hipLaunchKernelGGL((k_token_mlp<TN, 3>), grid, dim3(256), 0, st, g); break;
    }
}

hipError_t launch_token_mlp(const TokMlpArgs &g, hipStream_t st) {
    if (g.M <= 0 || g.M % 16 || !token_mlp_takes(g.C, g.chunks)) return hipErrorInvalidValue;
    const dim3 grid(token_mlp_grid(g.M, g.C));
    const int rb = token_mlp_row_blocks(g.M, g.C);
    switch (tok_tn(g.C)) {
    case 1: tok_launch<1>(g, rb, grid, st); break;
    case 2: tok_launch<2>(g, rb, grid, st); break;
    default: tok_launch<3>(g, rb, grid, st); break;
    }
    return hipGetLastError();
}

size_t qkv_attn_weight_floats(int hd) { return (size_t)(hd == 30 ? 3 * 4 * 6 : 6 * 2) * 6 * (FRAG / 4); }
size_t qkv_attn_param_floats(int hd) { return (size_t)(hd == 30 ? 12 : 6) * 96; }

void qkv_attn_pack(const float *wqkv, const float *bqkv, int hd, float *w, float *prm, float *v_l1, float *v_bmax) {
    const int c = 6 * hd, ks = c > 64 ? 6 : 2, nw = hd == 30 ? 4 : 6, ng = hd == 30 ? 3 : 1;
    uint16_t *dst = reinterpret_cast<uint16_t *>(w);
    // the qkv row of column n of tile t of wave wv, group g; -1: padding
    auto row_of = [&](int g, int wv, int t, int n) {
        int seg, head, d;
        if (hd == 30) {
            seg = t == 2 ? 2 : wv >> 1;
            head = 2 * g + (t == 2 ? wv >> 1 : wv & 1);
            d = 16 * (t == 2 ? wv & 1 : t) + n;
        } else {
            seg = t;
            head = wv;
            d = n;
        }
        return d < hd ? seg * c + head * hd + d : -1;
    };
    for (int g = 0; g < ng; ++g)
        for (int wv = 0; wv < nw; ++wv) {
            float sc[3][16];
            const float *rows[3][16];
            for (int t = 0; t < 3; ++t)
                for (int n = 0; n < 16; ++n) {
                    const int r = row_of(g, wv, t, n);
                    rows[t][n] = r < 0 ? nullptr : wqkv + (size_t)r * c;
                    sc[t][n] = r < 0 ? 1.f : split_row_scale(rows[t][n], c);
                    float *p = prm + ((size_t)(g * nw + wv) * 3 + t) * 32;
                    p[n] = 1.f / sc[t][n];
                    p[16 + n] = r < 0 ? 0.f : bqkv[r];
                }
            for (int s = 0; s < ks; ++s)
                for (int t = 0; t < 3; ++t, dst += FRAG) split_pack_step(rows[t], sc[t], 32 * s, c, dst);
        }
    float l1 = 0.f, bm = 0.f;
    for (int n = 0; n < c; ++n) {
        double a = 0.0;
        for (int k = 0; k < c; ++k) a += std::fabs((double)wqkv[(size_t)(2 * c + n) * c + k]);
        l1 = std::max(l1, (float)a);
        bm = std::max(bm, std::fabs(bqkv[2 * c + n]));
    }
    *v_l1 = l1;
    *v_bmax = bm;
}

// Workgroups: whole XCDs' worth of slots (a multiple of 8), at most two per CU,
// no more than the items.
unsigned qkv_attention_grid(int hp, int wp, int hd) {
    const int nw = (hp / 8) * (wp / 8), ng = hd == 30 ? 3 : 1;
    const int per_xcd = ((nw + 7) / 8) * ng;
    const int slots = std::max(1, cu_count() * 2 / 8);
    return 8u * (unsigned)std::min(per_xcd, slots);
}

hipError_t launch_qkv_attention(const QkvAttnArgs &g0, int hd, hipStream_t st) {
    if (g0.hp <= 0 || g0.wp <= 0 || g0.hp % 8 || g0.wp % 8 || g0.shift < 0 || g0.shift >= 8 || !qkv_attn_fused(6, hd))
        return hipErrorInvalidValue;
    QkvAttnArgs g = g0;
    g.nww = g.wp / 8;
    g.nw = (g.hp / 8) * g.nww;
    const dim3 grid(qkv_attention_grid(g.hp, g.wp, hd));
    if (hd == 30)
        hipLaunchKernelGGL(k_qkv_attn<30>, grid, dim3(64 * QaCfg<30>::NW), 0, st, g);
    else
        hipLaunchKernelGGL(k_qkv_attn<10>, grid, dim3(64 * QaCfg<10>::NW), 0, st, g);
    return hipGetLastError();
}

// k_split_conv's shapes: waves side by side and column tiles per wave by cout,
// k steps per tap by cin (both padded to 64).
static int conv_tn(int cout) { return cout <= 64 ? 2 : (cout + 63) / 64; }
static int conv_wc(int cout) { return cout <= 64 ? 2 : 4; }
static int conv_ks(int cin) { return 2 * ((cin + 63) / 64); }
bool split_conv_takes(int cin, int cout) {
    const int a = (cin + 63) / 64, b = (cout + 63) / 64;
    return cin % 4 == 0 && cout % 4 == 0 && cin > 0 && cout > 0 && a <= 3 && (b == 1 || b == a);
}
size_t split_conv_weight_floats(int cin, int cout) {
    // the fragments, then the columns' unscale
    return (size_t)conv_wc(cout) * conv_tn(cout) * (9 * conv_ks(cin) * 2 * (FRAG / 4) + 16);
}
void split_conv_pack(const float *w, int cin, int cout, float *out) {
    const int wc = conv_wc(cout), tn = conv_tn(cout), ks = conv_ks(cin);
    uint16_t *dst = reinterpret_cast<uint16_t *>(out);
    std::vector<float> tapw((size_t)9 * cout * cin);
    for (int o = 0; o < cout; ++o)
        for (int c = 0; c < cin; ++c)
            for (int t = 0; t < 9; ++t) tapw[((size_t)t * cout + o) * cin + c] = w[((size_t)o * cin + c) * 9 + t];
    std::vector<float> scale(16 * wc * tn, 1.f);
    for (int o = 0; o < cout; ++o) scale[o] = split_row_scale(w + (size_t)o * cin * 9, cin * 9);
    for (int g = 0; g < wc; ++g)
        for (int t = 0; t < 9; ++t)
            for (int s = 0; s < ks; ++s)
                for (int n = 0; n < tn; ++n, dst += FRAG) {
                    const float *rows[16];
                    for (int r = 0; r < 16; ++r) {
                        const int o = 16 * (g * tn + n) + r;
                        rows[r] = o < cout ? &tapw[((size_t)t * cout + o) * cin] : nullptr;
                    }
                    split_pack_step(rows, &scale[16 * (g * tn + n)], 32 * s, cin, dst);
                }
    // (the pixels' unscale holds 2^-15 of it, so that a sum stays near its value)
    float *un = reinterpret_cast<float *>(dst);
    for (float sc : scale) *un++ = 32768.f / sc;
}

// Row blocks per wave: the count whose rounds over two workgroups per CU take
// least, a tile costing its row blocks plus its halo rows and a constant; at
// most what two workgroups' registers and LDS hold.
static int conv_rb_max(int cin, int cout) {
    const int a = (cin + 63) / 64;
    return cout <= 64 ? (a == 1 ? 4 : a == 2 ? 3 : 2) : (a == 2 ? 4 : 3);
}
int split_conv_row_blocks(int H, int W, int cin, int cout) {
    const int wr = 4 / conv_wc(cout), slots = 2 * cu_count();
    int best = 1;
    double best_cost = 0;
    for (int rb = 1; rb <= conv_rb_max(cin, cout); ++rb) {
        const int th = 2 * rb * wr;
        const long tiles = (long)((W + 7) / 8) * ((H + th - 1) / th);
        const double cost = (double)((tiles + slots - 1) / slots) * (rb + 0.5);
        if (rb == 1 || cost <= best_cost) {
            best = rb;
            best_cost = cost;
        }
    }
    return best;
}

static long conv_tiles(int H, int W, int cout, int rb) {
    const int th = 2 * rb * 4 / conv_wc(cout);
    return (long)((W + 7) / 8) * ((H + th - 1) / th);
}
// Workgroups that share a tile's columns: all the column tiles of a wave apart
// while the one-row-block tiles alone leave half the CUs without one (180 wide:
// 4 tiles 15.2 -> 9.4 us, 96 tiles 15.9 -> 12.6; at 180 and 224 tiles no gain).
static int conv_split(int H, int W, int cin, int cout) {
    return split_conv_row_blocks(H, W, cin, cout) == 1 && conv_tiles(H, W, cout, 1) <= cu_count() / 2 ? conv_tn(cout) : 1;
}
dim3 split_conv_grid(int H, int W, int cin, int cout) {
    const long nt = conv_tiles(H, W, cout, split_conv_row_blocks(H, W, cin, cout));
    return dim3(8u * (unsigned)std::min<long>((nt + 7) / 8, std::max(1, cu_count() / 4)),
                (unsigned)conv_split(H, W, cin, cout));
}

template <int KSC, int TN, int WC, int RBM>
static void conv_launch(const SplitConvArgs &g, int rb, dim3 grid, hipStream_t st) {
    if (rb != RBM) {
        if constexpr (RBM > 1) conv_launch<KSC, TN, WC, RBM - 1>(g, rb, grid, st);
        return;
    }
    if constexpr (RBM == 1) {
        if (grid.y > 1) {
            hipLaunchKernelGGL((k_split_conv<KSC, TN, 1, WC, TN>), grid, dim3(256), 0, st, g);
            return;
        }
    }
    hipLaunchKernelGGL((k_split_conv<KSC, TN, RBM, WC, 1>), grid, dim3(256), 0, st, g);
}

hipError_t launch_split_conv(const SplitConvArgs &g, hipStream_t st) {
    if (g.H <= 0 || g.W <= 0 || !split_conv_takes(g.cin, g.cout)) return hipErrorInvalidValue;
    const int rb = split_conv_row_blocks(g.H, g.W, g.cin, g.cout);
    const dim3 grid = split_conv_grid(g.H, g.W, g.cin, g.cout);
    const int a = (g.cin + 63) / 64;
    if (g.cout <= 64) {
        if (a == 1) conv_launch<2, 2, 2, 4>(g, rb, grid, st);
        else if (a == 2) conv_launch<4, 2, 2, 3>(g, rb, grid, st);
        else conv_launch<6, 2, 2, 2>(g, rb, grid, st);
    } else if (a == 2) {
        conv_launch<4, 2, 4, 4>(g, rb, grid, st);
    } else {
        conv_launch<6, 3, 4, 3>(g, rb, grid, st);
    }
    return hipGetLastError();
}
