// Shared device helpers for the gfx950 (CDNA4) kernels: element types, wave64
// reductions, MFMA wrappers and the layout of a cache page.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

typedef _Float16 f16;
typedef __bf16 bf16;

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

#define WAVE 64
#define PAGE 64   // tokens of a cache page

// dtype codes of the C interface
enum { DT_F32 = 0, DT_F16 = 1, DT_BF16 = 2 };

// status codes of the C interface (0 = launched)
enum { LI_OK = 0, LI_BAD_ARG = 1, LI_UNSUPPORTED = 2, LI_HIP_ERROR = 3 };

template <class T> struct Vec;
template <> struct Vec<f16> { typedef f16x8 v8; typedef f16x4 v4; typedef f16x2 v2; };
template <> struct Vec<bf16> { typedef bf16x8 v8; typedef bf16x4 v4; typedef bf16x2 v2; };

template <class T> __device__ __forceinline__ float to_f32(T v) { return (float)v; }
template <class T> __device__ __forceinline__ T from_f32(float v) { return (T)v; }

__device__ __forceinline__ f32x16 mfma32(f16x8 a, f16x8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x16 mfma32(bf16x8 a, bf16x8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ float dot2(f16x2 a, f16x2 b, float c) { return __builtin_amdgcn_fdot2(a, b, c, false); }
__device__ __forceinline__ float dot2(bf16x2 a, bf16x2 b, float c) {
    return __builtin_amdgcn_fdot2_f32_bf16(a, b, c, false);
}

// 16 bytes that a launch reads once (a matrix's fragment in a decode step, a page of the cache): marked as not to be kept, so that
// they pass the caches without pushing anything out.  Bound by memory: a launch that only streams 8, 32, 128, 256 MB (of 2 GB in
// turn) takes 3.2, 6.6, 23.2, 44.1 us with ordinary loads and 2.7, 6.2, 21.6, 40.2 with these; 16 steps of batch 8 on 8,192 tokens
// (8B shape) 88.0 -> 79.8 ms, 24 of batch 1 82.4 -> 75.8.  Models whose matrices would fit the 256 MB cache gain as much (2 layers
// 2,048 wide with their head, batch 1: 5.69 -> 5.20 ms, 4.95 -> 4.47).  Not for what several workgroups read (a prompt's W), and not
// where an instruction takes half lines whose other halves the next one takes (float32 rows of W: 25.1 -> 25.4 ms a request).
template <class V> __device__ __forceinline__ V load_once(const void* p) {
    return __builtin_bit_cast(V, __builtin_nontemporal_load((const f32x4*)p));
}

// Values of other lanes by the vector unit alone: swaps of half waves and of rows of 16 lanes, moves within a row.  (__shfl is a
// round trip through the LDS unit, some 50 ns each in a chain that nothing runs beside: a wave's sum is six of them.  The same lanes
// are added in the same order, a + b for b + a, so the bits are the same; where a product is summed, wave_sum_product keeps the
// multiply-add that the compiler makes of a product and a __shfl.  Requests: Dopivik, batch 1, 6.89 -> 6.77 ms, Manirax 14.2 -> 14.05, 8B
// chat 75.8 -> 75.5; batches of 4 and more the same.)  Every lane of the wave must be active.
template <int CTRL> __device__ __forceinline__ float row_move(float v) {           // a move within every row of 16 lanes
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
#define ROW_ROR(n) (0x120 + (n))
#define QUAD_SWAP2 0x4E                                // lanes 2, 3, 0, 1 of every four
#define QUAD_SWAP1 0xB1                                // lanes 1, 0, 3, 2
struct LanePair { float lo, hi; };
__device__ __forceinline__ LanePair halves(float v) {  // the values of this lane's place in the lower and the upper half wave
    auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return LanePair{__uint_as_float(p[0]), __uint_as_float(p[1])};
}
__device__ __forceinline__ LanePair quarters(float v) { // and in the first and second 16 lanes of its half
    auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return LanePair{__uint_as_float(p[0]), __uint_as_float(p[1])};
}
__device__ __forceinline__ float sum_halves(float v) { const LanePair p = halves(v); return p.lo + p.hi; }        // v + that of lane ^ 32
__device__ __forceinline__ float sum_quarters(float v) { const LanePair p = quarters(v); return p.lo + p.hi; }    // v + that of lane ^ 16
__device__ __forceinline__ float max_halves(float v) { const LanePair p = halves(v); return fmaxf(p.lo, p.hi); }
__device__ __forceinline__ float max_quarters(float v) { const LanePair p = quarters(v); return fmaxf(p.lo, p.hi); }

// Sums over the 16 lanes of a row, over a half wave and over the wave, every lane's the same.
__device__ __forceinline__ float row_sum(float v) {
    v += row_move<ROW_ROR(8)>(v);
    v += row_move<ROW_ROR(4)>(v);                      // (a row repeats every 8 lanes by now: 4 back is 4 on)
    v += row_move<QUAD_SWAP2>(v);
    return v + row_move<QUAD_SWAP1>(v);
}
__device__ __forceinline__ float half_sum(float v) { return row_sum(sum_quarters(v)); }
__device__ __forceinline__ float wave_sum(float v) { return half_sum(sum_halves(v)); }
// wave_sum of a * b with the first addition and the lane's own product one multiply-add: a rounding less.  (The other half's
// product is rounded, so the two halves' results may differ in their last bit.)
__device__ __forceinline__ float wave_sum_product(float a, float b) {
    const LanePair p = halves(a * b);
    return half_sum(fmaf(a, b, (threadIdx.x & 32) ? p.lo : p.hi));
}
__device__ __forceinline__ float wave_max(float v) {
    v = max_quarters(max_halves(v));
    v = fmaxf(v, row_move<ROW_ROR(8)>(v));
    v = fmaxf(v, row_move<ROW_ROR(4)>(v));
    v = fmaxf(v, row_move<QUAD_SWAP2>(v));
    return fmaxf(v, row_move<QUAD_SWAP1>(v));
}

// A wave's choice among pairs (value, index): `take(value, index)` compares another lane's pair with this lane's `v`, `i` and
// takes it over if it is the better one.  Lane 0 compares its own with those of lanes 32, 16, 8, 4, 2 and 1 on, in this order; where `take`
// orders all pairs (no value is no number), every lane ends with the same one.
template <class F> __device__ __forceinline__ void wave_choice(float& v, int& i, F take) {
    const auto moved = [&](auto move) { take(move(v), __float_as_int(move(__int_as_float(i)))); };
    const LanePair hv = halves(v), hi = halves(__int_as_float(i));
    v = hv.lo; i = __float_as_int(hi.lo);
    take(hv.hi, __float_as_int(hi.hi));
    const LanePair qv = quarters(v), qi = quarters(__int_as_float(i));
    v = qv.lo; i = __float_as_int(qi.lo);
    take(qv.hi, __float_as_int(qi.hi));
    moved([](float x) { return row_move<ROW_ROR(8)>(x); });
    moved([](float x) { return row_move<ROW_ROR(12)>(x); });
    moved([](float x) { return row_move<QUAD_SWAP2>(x); });
    moved([](float x) { return row_move<QUAD_SWAP1>(x); });
}

// Sum over a block of up to 1024 threads; `scratch` holds 16 floats of LDS.  (All sixteen are read at once, the waves' added in
// their order: a loop over as many as there are waits for one after the other.  Up to 4, 8 and 16 of them: sixteen additions and choices for
// every workgroup were a chain that many rows felt, RMS norm of 300 rows of 8,192 with its launch 5.1 us by the loop, 5.3, now 5.1, of 2,000 rows 16.8, 17.0
// and 16.7; 1 row of 4,096 3.1, 2.9 and 2.8.)
__device__ __forceinline__ float sum_of_waves(float v, float* scratch) {       // v: a wave's number, in its lane 0
    const int w = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
    __syncthreads();
    if ((threadIdx.x & 63) == 0) scratch[w] = v;
    __syncthreads();
    float s[16], t = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = scratch[i];
#pragma unroll
    for (int i = 0; i < 4; ++i) t = i < nw ? t + s[i] : t;
    if (nw > 4) {
#pragma unroll
        for (int i = 4; i < 8; ++i) t = i < nw ? t + s[i] : t;
    }
    if (nw > 8) {
#pragma unroll
        for (int i = 8; i < 16; ++i) t = i < nw ? t + s[i] : t;
    }
    return t;
}
__device__ __forceinline__ float block_sum(float v, float* scratch) { return sum_of_waves(wave_sum(v), scratch); }
__device__ __forceinline__ float block_max(float v, float* scratch) {
    v = wave_max(v);
    const int w = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
    __syncthreads();
    if ((threadIdx.x & 63) == 0) scratch[w] = v;
    __syncthreads();
    float t = scratch[0];
    for (int i = 1; i < nw; ++i) t = fmaxf(t, scratch[i]);
    return t;
}

// Rows gathered from a table: threads of a workgroup take four elements each; a row of the few tokens of a decode step is
// shared by as many workgroups as it takes (an element at a time by one workgroup, which waited for memory 16 times a row
// of 4,096: 4,096 wide, bfloat16, with its launch, 1 row 3.9 -> 1.2 us, 8 rows 6.4 -> 1.7; with positions 9.7 -> 2.0 and 14.0 -> 2.4).
#define GATHER_THREADS 256
static inline dim3 gather_grid(int n_tokens, int d) {
    return dim3(n_tokens, n_tokens < 256 ? (d + 4 * GATHER_THREADS - 1) / (4 * GATHER_THREADS) : 1);
}
// For this thread's elements of a row of d: quad(i) for four from i on, or, where the rows do not allow a load for four, one(i),
// neighbouring elements by neighbouring threads (514 wide, 4,000 rows 4.2 us, four to a thread 6.3)
template <class Q, class E> __device__ __forceinline__ void gather_row(int d, bool quads, Q quad, E one) {
    const int at = blockIdx.y * GATHER_THREADS + threadIdx.x, step = GATHER_THREADS * gridDim.y;
    if (quads) for (int i = 4 * at; i < d; i += 4 * step) quad(i);
    else for (int i = at; i < d; i += step) one(i);
}
template <class T> struct alignas(4 * sizeof(T)) Quad { T v[4]; };
template <class T> __device__ __forceinline__ f32x4 quad_of(const T* p) {       // four elements, one load
    const Quad<T> q = *(const Quad<T>*)p;
    return f32x4{to_f32(q.v[0]), to_f32(q.v[1]), to_f32(q.v[2]), to_f32(q.v[3])};
}

// A power of two near 1 / (8 rms) for a row whose root mean square is `rms`: what the rows of a residual
// stream are multiplied by before they are rounded to float16 on their way from one product to the norm
// inside the next (gemm.hip, RowsOut), so that they lie in the middle of that type's range whatever the
// model's own scale.  An element is at most sqrt(width) times the rms, so a row that has grown a hundredfold
// since the rms was taken still fits.
__device__ __forceinline__ float row_scale_for(float rms) {
    int e;
    frexpf(fminf(fmaxf(rms, 1e-30f), 1e30f), &e);        // rms = m 2^e, 0.5 <= m < 1
    return ldexpf(0.125f, -e);
}

// The gate's activation: silu(x) = x / (1 + exp(-x)) (include/kernels_cpu.hpp:186) or the tanh form of
// gelu that the reference computes, 0.5 x (1 + tanh(sqrt(2 / pi) (x + 0.044715 x^3)))
// (include/kernels_cpu.hpp:179-184).
__device__ __forceinline__ float gate_activation(float g, bool gelu) {
    if (gelu) return 0.5f * g * (1.f + tanhf(0.7978845608028654f * (g + 0.044715f * g * g * g)));
    return g / (1.f + expf(-g));
}

// The activations of feed-forwards without a gate.  act: 0 gelu (erf), 1 gelu (tanh), 2 silu, 3 the square of relu.
__device__ __forceinline__ float plain_activation(float z, int act) {
    if (act == 3) { const float r = fmaxf(z, 0.f); return r * r; }
    if (act == 2) return z / (1.f + expf(-z));
    if (act == 1) return gate_activation(z, true);
    return 0.5f * z * (1.f + erff(z * 0.70710678118654752f));
}

// A score's soft cap, c tanh(x / c), with a = 2 log2(e) / c beside c: tanh z = 1 - 2 / (e^(2z) + 1) by the hardware's
// 2^x and reciprocal (an error of some 1e-7 c; for large |x| the exponential becomes infinite or 0 and the result +-c).
__device__ __forceinline__ float soft_cap(float x, float c, float a) {
    return c - 2.f * c * __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(x * a) + 1.f);
}

// ---------------------------------------------------------------------------
// Layout of a cache page.  A page holds PAGE (64) tokens of one layer for all
// KV heads.  Keys and values are stored in the order in which a wave's lanes
// feed them to the 32x32x16 matrix instruction, so that attention reads every
// operand as one contiguous 1 KiB load per wave, with no transposition in LDS.
//
// Keys (operand A of S^T = K Q^T, rows = tokens, inner index = head dim):
//   [kv head][token block b = t/32][step s = d/16][lane = 32*((d%16)/8) + t%32][d%8]
// Values (operand A of O^T = V^T P^T, rows = head dim, inner index = tokens, in the
// order in which the score accumulators hold the tokens):
//   [kv head][dim block d/32][token group t/16][lane = 32*((t%8)/4) + d%32][4*((t%16)/8) + t%4]
// The value part of a page is padded to a multiple of 32 in the head dim.
// ---------------------------------------------------------------------------
__host__ __device__ __forceinline__ int round_up(int a, int b) { return (a + b - 1) / b * b; }

__host__ __device__ __forceinline__ int64_t k_head_elems(int hd) { return (int64_t)PAGE * hd; }
__host__ __device__ __forceinline__ int64_t v_head_elems(int hd) { return (int64_t)PAGE * round_up(hd, 32); }

__host__ __device__ __forceinline__ int k_offset(int t, int d, int hd) {
    const int b = t >> 5, s = d >> 4, lane = (((d & 15) >> 3) << 5) + (t & 31);
    return ((b * (hd >> 4) + s) * 64 + lane) * 8 + (d & 7);
}
__host__ __device__ __forceinline__ int v_offset(int t, int d, int hd) {
    (void)hd;
    const int db = d >> 5, tj = t >> 4, u = t & 15;
    const int lane = (((u & 7) >> 2) << 5) + (d & 31);
    const int idx = ((u >> 3) << 2) + (u & 3);
    return ((db * (PAGE / 16) + tj) * 64 + lane) * 8 + idx;
}

#define LI_CHECK_LAUNCH()                                        \
    do {                                                         \
        hipError_t e_ = hipGetLastError();                       \
        if (e_ != hipSuccess) return LI_HIP_ERROR;               \
    } while (0)
