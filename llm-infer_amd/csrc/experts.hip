// Routed experts, token by token on the experts that were chosen and nothing else, with no wait for the host.
//
// A step's work is its pairs (token, chosen expert), sorted by expert: `counts` [E] pairs an expert, which begin at
// `offsets` [E]; `row_of` [P] the token of every pair, ascending within an expert; `slot_of` [T, top] where a token's
// pairs lie (-1: none) beside their weights `weights` [T, top], experts ascending.  Then every expert's two products run
// on its own pairs' rows (experts_gemv here for few pairs an expert; gemm_wreg's pairs mode for many), and a token's
// result is the weighted sum of its pairs' rows, in the order of the experts (in the pass that adds a sub-layer's
// normed output, or pair_sum here).  Everything is planned on the device: a step can be recorded whatever was chosen.
// Router logits, the choice, the weights and all sums are float32.
#include "gemm_common.h"

__device__ __forceinline__ f32x4 mfma16(f16x8 a, f16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mfma16(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

struct Pairs {
    int* counts;        // [E]
    int* offsets;       // [E]
    int* row_of;        // [P]
    int* slot_of;       // [T, top]
};

// The pairs of expert e (workgroup e), from `chosen` [n = T * top]: what lies before expert e is counted too, so every
// workgroup knows its own offset and none waits for another.  A wave takes a run of the pairs, 64 at a time; twice: how
// many there are, then where each goes.  Pairs that name no expert (-1) lie nowhere.  With weights [T, top] a pair's weight goes
// to weight_of [P] beside row_of.
#define SORT_WAVES 16

__global__ __launch_bounds__(64 * SORT_WAVES) void sort_pairs_kernel(const int* __restrict__ chosen, int n, int top, Pairs p,
                                                                     const float* __restrict__ weights, float* __restrict__ weight_of) {
    __shared__ int eq[SORT_WAVES], lt[SORT_WAVES];
    const int e = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int per = (n + 64 * SORT_WAVES - 1) / (64 * SORT_WAVES) * 64, lo = wave * per, hi = min(n, lo + per);
    int mine = 0, before = 0;
#pragma unroll 4
    for (int i0 = lo; i0 < hi; i0 += 64) {
        const int v = i0 + lane < hi ? chosen[i0 + lane] : -1;
        mine += __builtin_popcountll(__builtin_amdgcn_ballot_w64(v == e));
        before += __builtin_popcountll(__builtin_amdgcn_ballot_w64(v >= 0 && v < e));
    }
    if (lane == 0) { eq[wave] = mine; lt[wave] = before; }
    __syncthreads();
    int at = 0, total = 0, offset = 0;
#pragma unroll
    for (int w = 0; w < SORT_WAVES; ++w) {
        if (w < wave) at += eq[w];
        total += eq[w];
        offset += lt[w];
    }
    at += offset;
#pragma unroll 4
    for (int i0 = lo; i0 < hi; i0 += 64) {
        const int i = i0 + lane, v = i < hi ? chosen[i] : -2;
        const uint64_t mask = __builtin_amdgcn_ballot_w64(v == e);
        if (v == e) {
            const int s = at + __builtin_popcountll(mask & ((1ull << lane) - 1));
            p.row_of[s] = i / top;
            p.slot_of[i] = s;
            if (weights) weight_of[s] = weights[i];
        }
        if (e == 0 && v == -1) p.slot_of[i] = -1;
        at += __builtin_popcountll(mask);
    }
    if (threadIdx.x == 0) { p.counts[e] = total; p.offsets[e] = offset; }
}

// The pairs of dense routing weights [T, cols] (0: not chosen; the first n_experts columns), to be sorted as above: chosen
// [T, top] the experts of the first `top` weights of a token that are not 0, ascending, -1 behind them; weights [T, top] beside
// it, 0 behind them.  GROUP lanes a token (a power of two), so that eight tokens of eight experts share a wave and a row is read
// in one piece; a row is read once.  With the sort, one call after another: 16,384 tokens 41 us at 8 experts, 100 at 128, 94 at
// 256 (a workgroup an expert that read every row of all experts before its own 138, 2,313 and 7,045); up to 4,096 tokens the
// host's launches, 24 us (at 8 experts 39, at 256 1,489).
template <int GROUP>
__global__ __launch_bounds__(256) void list_pairs_kernel(const float* __restrict__ dense, int cols, int n_tokens, int n_experts, int top,
                                                         int* __restrict__ chosen, float* __restrict__ weights) {
    const int lane = threadIdx.x & 63, i0 = lane % GROUP, first = lane - i0;
    const int64_t t = (int64_t)blockIdx.x * (256 / GROUP) + threadIdx.x / GROUP;
    const bool have = t < n_tokens;
    const float* w = dense + (have ? t : 0) * cols;
    int rank = 0;
    for (int c0 = 0; c0 < n_experts; c0 += GROUP) {
        const float v = have && c0 + i0 < n_experts ? w[c0 + i0] : 0.f;
        uint64_t mask = __builtin_amdgcn_ballot_w64(v != 0.f) >> first;
        if (GROUP < 64) mask &= (1ull << (GROUP & 63)) - 1;
        const int at = rank + __builtin_popcountll(mask & ((1ull << i0) - 1));
        if (v != 0.f && at < top) {
            chosen[t * top + at] = c0 + i0;
            weights[t * top + at] = v;
        }
        rank += __builtin_popcountll(mask);
    }
    if (have)
        for (int j = rank + i0; j < top; j += GROUP) { chosen[t * top + j] = -1; weights[t * top + j] = 0.f; }
}

extern "C" int li_pairs_of_weights(const float* dense, int cols, int n_tokens, int top, int n_experts, int* chosen, int* counts,
                                   int* offsets, int* row_of, int* slot_of, float* weights, float* weight_of, hipStream_t stream) {
    if (n_tokens <= 0) return LI_OK;
    if (!dense || cols < n_experts || top < 1 || n_experts < 1 || !chosen || !counts || !offsets || !row_of || !slot_of || !weights || !weight_of)
        return LI_BAD_ARG;
    if ((int64_t)n_tokens * top > 0x7fffffff) return LI_UNSUPPORTED;
#define GO(GROUP) list_pairs_kernel<GROUP><<<(n_tokens + 256 / GROUP - 1) / (256 / GROUP), 256, 0, stream>>>(dense, cols, n_tokens, n_experts, top, chosen, weights)
    if (n_experts <= 8) GO(8); else if (n_experts <= 16) GO(16); else if (n_experts <= 32) GO(32); else GO(64);
#undef GO
    LI_CHECK_LAUNCH();
    sort_pairs_kernel<<<n_experts, 64 * SORT_WAVES, 0, stream>>>(chosen, n_tokens * top, top, Pairs{counts, offsets, row_of, slot_of}, weights,
                                                                 weight_of);
    LI_CHECK_LAUNCH();
    return LI_OK;
}

extern "C" int li_sort_pairs(const int* chosen, int n, int top, int n_experts, int* counts, int* offsets, int* row_of,
                             int* slot_of, hipStream_t stream) {
    if (n <= 0) return LI_OK;
    if (top < 1 || n % top || n_experts < 1 || !chosen || !counts || !offsets || !row_of || !slot_of) return LI_BAD_ARG;
    sort_pairs_kernel<<<n_experts, 64 * SORT_WAVES, 0, stream>>>(chosen, n, top, Pairs{counts, offsets, row_of, slot_of}, nullptr, nullptr);
    LI_CHECK_LAUNCH();
    return LI_OK;
}

// ---------------------------------------------------------------------------
// The router, 16 tokens at a time, in two launches: logits z = W h + b against the tiled 16-bit matrix W [n, K] on the matrix
// cores, then the choice.  W is the sum of `parts` 16-bit matrices one behind the other (each of n rows rounded up to 16: the
// rounding of W and the roundings of what is left, one matrix where the file's own numbers are 16-bit), so products are those of
// a float32 W, summed in float32.  For a tile of 16 rows of W `kw` waves share K, sixteen waves for all tiles where there are no
// more tiles than that.  Each is a workgroup of its own: one workgroup of them all is bound by what a CU takes in (W and X,
// 0.2 to 0.5 MB for 16 x 4,096).  us in a recorded chain, one launch with a workgroup for 16 tokens and these two, 8 tokens:
// 16 x 4,096 in one part 8.4 -> 5.8, in three 15.3 -> 6.5, 64 x 4,096 18.3 -> 8.6 and 42.8 -> 13.2, 8 x 2,048 6.7 -> 5.2 and 9.6 -> 5.8;
// 600 tokens x 16 x 4,096 13.4 -> 10.7 and 22.5 -> 12.5.  Where nearly every CU has a workgroup of 16 tokens anyway, one launch
// does it all after all (router_one_kernel; the same values): us in one launch and in two, with the sort, in one part and in three, 4,096
// tokens x 16 x 4,096 19.5, 21.0 and 28.3, 29.7, x 64 x 4,096 46.5, 48.9 and 81.1, 83.5, x 8 x 2,048 17.0, 18.6 and 21.7, 22.3, x 256 x 4,096 109, 111
// and 248, 250; 3,584 18.5, 19.4 and 27.6, 28.0, 44.1, 45.7 and 79.3, 80.9, x 512 x 2,048 119, 111 and 257, 232; 3,328 18.7, 19.1 and 27.3, 26.9;
// 4,112 28.7, 22.7 and 46.6, 31.5; 8,192 35.7, 33.9 and 52.6, 49.2, 88.6, 90.2 and 158, 160.
// ---------------------------------------------------------------------------
#define ROUTER_WAVES 16
#define ROUTER_MAX 512

static __host__ __device__ __forceinline__ int router_share(int tiles) { return tiles >= ROUTER_WAVES ? 1 : ROUTER_WAVES / tiles; }

// sums [token / 16][tile * kw + share][lane][4]: a share's accumulators, element q of a lane the output 4 (lane / 16) + q of the
// tile and the token lane % 16
template <class T>
__global__ __launch_bounds__(64) void router_sums_kernel(const T* __restrict__ X, const T* __restrict__ Wt, float* __restrict__ sums,
                                                         int parts, int n_tokens, int K, int tiles, int kw) {
    typedef typename Vec<T>::v8 v8;
    constexpr int U = 8, AHEAD = 3;                        // batches of loads on their way together
    const int lane = threadIdx.x, r = lane & 15, g = lane >> 4, t0 = blockIdx.x * 16;
    const int steps = K >> 5, tile = blockIdx.y / kw, share = blockIdx.y % kw;
    const int per = (steps + kw - 1) / kw, s_begin = share * per, s_end = min(steps, s_begin + per);
    const int batches = s_end > s_begin ? (s_end - s_begin + U - 1) / U : 0, total = parts * batches;
    const bool have = t0 + r < n_tokens;
    const T* xrow = X + (int64_t)(have ? t0 + r : t0) * K + 8 * g;
    v8 a[AHEAD][U], b[AHEAD][U];
    auto load = [&](int i, v8 (&av)[U], v8 (&bv)[U]) {     // the parts one after the other, K ascending in each
        const int pt = i / batches, s0 = s_begin + i % batches * U;
        const T* wt = Wt + ((int64_t)(pt * tiles + tile) * steps * 64 + lane) * 8;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const v8 zero = {};
            const bool in = s0 + u < s_end;
            av[u] = in ? *(const v8*)(wt + (int64_t)(s0 + u) * 512) : zero;
            bv[u] = in && have ? *(const v8*)(xrow + (s0 + u) * 32) : zero;
        }
    };
#pragma unroll
    for (int k = 0; k < AHEAD; ++k) if (k < total) load(k, a[k], b[k]);
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int i = 0; i < total; i += AHEAD) {
#pragma unroll
        for (int k = 0; k < AHEAD; ++k) {
            if (i + k >= total) break;
#pragma unroll
            for (int u = 0; u < U; ++u) acc = mfma16(a[k][u], b[k][u], acc);
            if (i + k + AHEAD < total) load(i + k + AHEAD, a[k], b[k]);
        }
    }
    *(f32x4*)(sums + (((int64_t)blockIdx.x * gridDim.y + blockIdx.y) * 64 + lane) * 4) = acc;
}

// The choice for a wave's token t, whose logits zs its lanes hold (output c * 64 + lane in zs[c], -infinity beyond n): the `top` largest (the
// first of equals), their weights the softmax over them alone times `scale`.  chosen and weights [T, top], experts ascending; `picked`
// (may be null) receives the chosen experts too, from token t0 on.
template <int NC>
__device__ __forceinline__ void choose(const float (&zs)[NC], int t, int t0, int n, int top, float scale, int* __restrict__ chosen,
                                       float* __restrict__ weights, int* picked) {
    const int lane = threadIdx.x & 63;
    float mx = 0.f, sum = 0.f;
    uint32_t taken = 0;                                // bit c: this lane's output c * 64 + lane is chosen
    for (int k = 0; k < top; ++k) {
        float best = -INFINITY; int bi = 0x7fffffff;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            const int i = c * 64 + lane;
            if (i < n && !(taken >> c & 1) && (zs[c] > best || bi == 0x7fffffff)) { best = zs[c]; bi = i; }
        }
        wave_choice(best, bi, [&](float ob, int oi) {
            if (oi != 0x7fffffff && (bi == 0x7fffffff || ob > best || (ob == best && oi < bi))) { best = ob; bi = oi; }
        });
        bi = __builtin_amdgcn_readfirstlane(bi);       // (one choice for the wave, also where logits are no numbers)
        best = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(best)));
        if (k == 0) mx = best;
        sum += expf(best - mx);
        if ((bi & 63) == lane) taken |= 1u << (bi >> 6);
    }
    int rank = 0;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        const bool mine = taken >> c & 1;
        const uint64_t mask = __builtin_amdgcn_ballot_w64(mine);
        if (mine) {
            const int64_t at = (int64_t)t * top + rank + __builtin_popcountll(mask & ((1ull << lane) - 1));
            chosen[at] = c * 64 + lane;
            if (picked) picked[at - (int64_t)t0 * top] = c * 64 + lane;
            weights[at] = expf(zs[c] - mx) / sum * scale;
        }
        rank += __builtin_popcountll(mask);
    }
}

// Everything in one launch, 16 tokens a workgroup: the waves share W's tiles, and K where there are fewer tiles than waves, as above.
template <class T, int NC>
__global__ __launch_bounds__(64 * ROUTER_WAVES) void router_one_kernel(const T* __restrict__ X, const T* __restrict__ Wt,
                                                                       const float* __restrict__ bias, int parts, int n_tokens, int K,
                                                                       int n, int top, float scale, int* __restrict__ chosen,
                                                                       float* __restrict__ weights) {
    typedef typename Vec<T>::v8 v8;
    constexpr int U = 8;
    extern __shared__ float z[];                           // [16][n]
    __shared__ float part[ROUTER_WAVES][64][4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, g = lane >> 4;
    const int t0 = blockIdx.x * 16, steps = K >> 5, tiles = (n + 15) >> 4;
    const int kw = router_share(tiles), at_once = ROUTER_WAVES / kw;              // tiles that are worked on at a time
    const int share = wave % kw, per = (steps + kw - 1) / kw, s_begin = share * per, s_end = min(steps, s_begin + per);
    const bool have = t0 + r < n_tokens;
    const T* xrow = X + (int64_t)(have ? t0 + r : t0) * K + 8 * g;
    for (int first = 0; first < tiles; first += at_once) {
        const int tile = first + wave / kw;
        const bool on = wave / kw < at_once && tile < tiles;
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
        if (on) {
            for (int pt = 0; pt < parts; ++pt) {
                const T* wt = Wt + ((int64_t)(pt * tiles + tile) * steps * 64 + lane) * 8;
                for (int s0 = s_begin; s0 < s_end; s0 += U) {
                    v8 a[U], b[U];
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        const v8 zero = {};
                        const bool in = s0 + u < s_end;
                        a[u] = in ? *(const v8*)(wt + (int64_t)(s0 + u) * 512) : zero;
                        b[u] = in && have ? *(const v8*)(xrow + (s0 + u) * 32) : zero;
                    }
#pragma unroll
                    for (int u = 0; u < U; ++u) acc = mfma16(a[u], b[u], acc);
                }
            }
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) part[wave][lane][q] = acc[q];
        __syncthreads();
        if (on && share == 0) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                float v = part[wave][lane][q];
                for (int k = 1; k < kw; ++k) v += part[wave + k][lane][q];
                const int j = tile * 16 + 4 * g + q;
                if (j < n) z[r * n + j] = v + (bias ? bias[j] : 0.f);
            }
        }
        __syncthreads();
    }
    const int t = t0 + wave;
    if (t >= n_tokens) return;                             // (a wave's token, the same for all its lanes)
    float zs[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) zs[c] = c * 64 + lane < n ? z[wave * n + c * 64 + lane] : -INFINITY;
    choose<NC>(zs, t, t0, n, top, scale, chosen, weights, nullptr);
}

// The second launch, a wave a token: its logits are the shares' sums in ascending order.  With one workgroup (up to 16 tokens) it
// also sorts the pairs.
// NC: outputs in groups of 64 that a wave holds, ceil(n / 64) rounded up to 1 or 8.
template <int NC>
__global__ __launch_bounds__(64 * ROUTER_WAVES) void router_kernel(const float* __restrict__ sums, const float* __restrict__ bias,
                                                                   int n_tokens, int n, int kw, int top, float scale,
                                                                   int* __restrict__ chosen, float* __restrict__ weights, Pairs p) {
    constexpr int SHARES = NC == 1 ? ROUTER_WAVES : 3;     // kw at the most: n > 64 has five tiles or more
    extern __shared__ int picked[];                        // [16][top]: the chosen experts, for the sort
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int t0 = blockIdx.x * 16, tiles = (n + 15) >> 4;
    const int t = t0 + wave;
    if (t < n_tokens) {                                    // (a wave's token, the same for all its lanes)
        float zs[NC];
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            const int j = min(c * 64 + lane, n - 1);
            const float* at = sums + (((int64_t)blockIdx.x * tiles + (j >> 4)) * kw * 64 + ((j >> 2) & 3) * 16 + wave) * 4 + (j & 3);
            const float own = bias ? bias[j] : 0.f;
            float v[SHARES];
#pragma unroll
            for (int k = 0; k < SHARES; ++k) v[k] = at[(int64_t)min(k, kw - 1) * 256];
            float z = v[0];
#pragma unroll
            for (int k = 1; k < SHARES; ++k) z = k < kw ? z + v[k] : z;
            zs[c] = c * 64 + lane < n ? z + own : -INFINITY;
        }
        choose<NC>(zs, t, t0, n, top, scale, chosen, weights, picked);
    }
    if (gridDim.x == 1 && p.counts) {
        __syncthreads();
        const int pairs = n_tokens * top;
        // a wave an expert: up to 16 * top pairs, 64 at a time
        for (int e = wave; e < n; e += ROUTER_WAVES) {
            int before = 0, total = 0;
            for (int i0 = 0; i0 < pairs; i0 += 64) {
                const int v = i0 + lane < pairs ? picked[i0 + lane] : 0x7fffffff;
                before += __builtin_popcountll(__builtin_amdgcn_ballot_w64(v < e));
                total += __builtin_popcountll(__builtin_amdgcn_ballot_w64(v == e));
            }
            int at = before;
            for (int i0 = 0; i0 < pairs && total; i0 += 64) {
                const bool mine = i0 + lane < pairs && picked[i0 + lane] == e;
                const uint64_t mask = __builtin_amdgcn_ballot_w64(mine);
                if (mine) {
                    const int s = at + __builtin_popcountll(mask & ((1ull << lane) - 1));
                    p.row_of[s] = (i0 + lane) / top;
                    p.slot_of[i0 + lane] = s;
                }
                at += __builtin_popcountll(mask);
            }
            if (lane == 0) { p.counts[e] = total; p.offsets[e] = before; }
        }
    }
}

// float32 numbers of workspace that li_router wants; 0: one launch, without any (workgroups of 16 tokens for 7/8 of the 256 CUs and more, but
// not for more than all of them; figures above).
extern "C" int64_t li_router_sums(int n_tokens, int n) {
    const int blocks = (n_tokens + 15) / 16, tiles = (n + 15) / 16;
    if (n < 1 || (blocks > 224 && blocks <= 256)) return 0;
    return (int64_t)blocks * tiles * router_share(tiles) * 256;
}

// counts (and the other three) not null with up to 16 tokens: the pairs are sorted too.  sums: li_router_sums of them.
extern "C" int li_router(const void* X, const void* Wt, int dt, const float* bias, int parts, int n_tokens, int K, int n, int top, float scale,
                         int* chosen, float* weights, int* counts, int* offsets, int* row_of, int* slot_of, float* sums, hipStream_t stream) {
    if (n_tokens <= 0) return LI_OK;
    if (!X || !Wt || !chosen || !weights || n < 1 || top < 1 || top > n || parts < 1 || parts > 3 || (dt != DT_F16 && dt != DT_BF16)) return LI_BAD_ARG;
    // (n + top: what this entry takes; LDS would hold more, 64 bytes an output or a choice.  The caller has a path for the others)
    if (n > ROUTER_MAX || n + top > 640 || K < 32 || K % 32 || ((uintptr_t)X & 15) || ((uintptr_t)Wt & 15) || ((uintptr_t)sums & 15)) return LI_UNSUPPORTED;
    if (counts && (n_tokens > 16 || !offsets || !row_of || !slot_of || !sums)) return LI_BAD_ARG;
    const Pairs p{counts, offsets, row_of, slot_of};
    const int blocks = (n_tokens + 15) / 16, tiles = (n + 15) / 16, kw = router_share(tiles);
    if (!sums) {
        const size_t lds = (size_t)16 * n * sizeof(float);
#define GO(T, NC) router_one_kernel<T, NC><<<blocks, 64 * ROUTER_WAVES, lds, stream>>>((const T*)X, (const T*)Wt, bias, parts, n_tokens, K, n, top, scale, chosen, weights)
        if (dt == DT_F16) { if (n <= 64) GO(f16, 1); else GO(f16, 8); }
        else { if (n <= 64) GO(bf16, 1); else GO(bf16, 8); }
#undef GO
        LI_CHECK_LAUNCH();
        return LI_OK;
    }
    dim3 grid(blocks, tiles * kw);
    if (dt == DT_F16) router_sums_kernel<f16><<<grid, 64, 0, stream>>>((const f16*)X, (const f16*)Wt, sums, parts, n_tokens, K, tiles, kw);
    else router_sums_kernel<bf16><<<grid, 64, 0, stream>>>((const bf16*)X, (const bf16*)Wt, sums, parts, n_tokens, K, tiles, kw);
    const size_t lds = (size_t)16 * top * sizeof(int);
    if (n <= 64) router_kernel<1><<<blocks, 64 * ROUTER_WAVES, lds, stream>>>(sums, bias, n_tokens, n, kw, top, scale, chosen, weights, p);
    else router_kernel<8><<<blocks, 64 * ROUTER_WAVES, lds, stream>>>(sums, bias, n_tokens, n, kw, top, scale, chosen, weights, p);
    LI_CHECK_LAUNCH();
    return LI_OK;
}

// ---------------------------------------------------------------------------
// An expert's product on its own pairs' rows, few of them: C[pair] = epilogue(W_e X[row_of[pair]]) for the pairs of
// the blockIdx.y-th expert that has any (row_of null: X[pair]).  gemv_tiled's structure: a workgroup takes 16 rows of W_e
// for the whole of K, its KW waves share K; 16 MT pairs at a time (W is read again, from the caches, for the next ones; only the
// last time past them).  us, 16 experts, up 7,168 x 4,096, all reads of W past the caches, none, and so: 8 pairs each 157, 163, 157; a
// quarter of the experts with 32 each 106, 94, 90; one with 64, 8 in the mean 181, 177, 168; 64 experts of 1,536 x 2,048, 10 each 98, 100,
// 98, a quarter with 32 each 53, 46, 46.
// ---------------------------------------------------------------------------
template <class T, int MT, int KW>
__global__ __launch_bounds__(64 * KW, 4) void experts_gemv_kernel(const T* __restrict__ X, const T* __restrict__ Wt, int K,
                                                               int64_t w_stride, Epilogue e, int n_experts,
                                                               const int* __restrict__ counts, const int* __restrict__ offsets,
                                                               const int* __restrict__ row_of) {
    typedef typename Vec<T>::v8 v8;
    constexpr int U = MT == 1 ? 8 : 4;
    __shared__ float part[KW][MT][64][4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, g = lane >> 4;
    int expert = -1, nth = blockIdx.y;
    for (int e0 = 0; e0 < n_experts; e0 += 64) {
        uint64_t any = __builtin_amdgcn_ballot_w64(e0 + lane < n_experts && counts[min(e0 + lane, n_experts - 1)] > 0);
        const int here = __builtin_popcountll(any);
        if (nth < here) {
            for (int i = 0; i < nth; ++i) any &= any - 1;
            expert = e0 + __builtin_ctzll(any);
            break;
        }
        nth -= here;
    }
    if (expert < 0) return;
    const int count = counts[expert], row0 = offsets[expert];
    Wt += expert * w_stride;
    const int tile = blockIdx.x, steps = K >> 5;
    const int per = (steps + KW - 1) / KW, s_begin = wave * per, s_end = min(steps, s_begin + per);
    const T* wt = Wt + ((int64_t)tile * steps * 64 + lane) * 8;
    e.M = row0 + count;
    for (int r0 = 0; r0 < count; r0 += 16 * MT) {
        bool have[MT];
        const T* xrow[MT];
        f32x4 acc[MT];
#pragma unroll
        for (int j = 0; j < MT; ++j) {
            have[j] = r0 + 16 * j + r < count;
            const int pair = row0 + (have[j] ? r0 + 16 * j + r : 0);
            xrow[j] = X + (int64_t)(row_of ? row_of[pair] : pair) * K + 8 * g;
            acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
        auto product = [&](auto last) {
            for (int s0 = s_begin; s0 < s_end; s0 += U) {
                v8 a[U], b[U][MT];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const bool in = s0 + u < s_end;
                    const v8 z = {};
                    const T* from = wt + (int64_t)(s0 + u) * 512;
                    a[u] = !in ? z : decltype(last)::value ? load_once<v8>(from) : *(const v8*)from;
#pragma unroll
                    for (int j = 0; j < MT; ++j) b[u][j] = in && have[j] ? *(const v8*)(xrow[j] + (s0 + u) * 32) : z;
                }
#pragma unroll
                for (int u = 0; u < U; ++u)
#pragma unroll
                    for (int j = 0; j < MT; ++j) acc[j] = mfma16(a[u], b[u][j], acc[j]);
            }
        };
        if (r0 + 16 * MT >= count) product(std::true_type{}); else product(std::false_type{});
        if (r0) __syncthreads();                           // wave 0 has read the sums of the pairs before
#pragma unroll
        for (int j = 0; j < MT; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q) part[wave][j][lane][q] = acc[j][q];
        __syncthreads();
        if (wave == 0) {
#pragma unroll
            for (int j = 0; j < MT; ++j) {
                float v[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    v[q] = part[0][j][lane][q];
                    for (int w = 1; w < KW; ++w) v[q] += part[w][j][lane][q];
                }
                if (have[j]) epilogue4_base(e, row0 + r0 + 16 * j + r, tile * 16 + 4 * g, v);
            }
        }
    }
}

// mode: EPI_STORE or EPI_SWIGLU.  Wt: the experts' tiled matrices [N, K] one behind the other, w_stride elements apart.
extern "C" int li_experts_gemv(const void* X, const void* Wt, int dt, void* C, int out_dt, int mode, int n_pairs, int N, int K,
                               int64_t w_stride, int n_experts, const int* counts, const int* offsets, const int* row_of,
                               hipStream_t stream) {
    int rc = check_common(X, Wt, C, n_pairs, N, K, mode, out_dt);
    if (rc) return rc;
    if ((dt != DT_F16 && dt != DT_BF16) || (mode != EPI_STORE && mode != EPI_SWIGLU) || !counts || !offsets || n_experts < 1) return LI_BAD_ARG;
    if (K % 32 || ((uintptr_t)X & 15) || ((uintptr_t)Wt & 15) || w_stride % 8) return LI_UNSUPPORTED;
    if (n_pairs == 0) return LI_OK;
    Epilogue e;
    rc = make_epilogue(e, C, mode, out_dt, n_pairs, N, nullptr);
    if (rc) return rc;
    dim3 grid((N + 15) / 16, min(n_experts, n_pairs));
#define GO(T, MT, KW)                                                                                                             \
    experts_gemv_kernel<T, MT, KW><<<grid, 64 * KW, 0, stream>>>((const T*)X, (const T*)Wt, K, w_stride, e, n_experts, counts, offsets, row_of)
#define BY_K(T, MT) do { if (K >= 2048) GO(T, MT, 8); else GO(T, MT, 4); } while (0)
#define BY_M(T) do { if (n_pairs <= 8 * n_experts) BY_K(T, 1); else BY_K(T, 2); } while (0)
    if (dt == DT_F16) BY_M(f16); else BY_M(bf16);
#undef BY_M
#undef BY_K
#undef GO
    LI_CHECK_LAUNCH();
    return LI_OK;
}

// ---------------------------------------------------------------------------
// out[t] (+)= sum over j < top of weights[t][j] * rows[slot_of[t][j]], in the order of j.
// ---------------------------------------------------------------------------
__global__ void pair_sum_kernel(const float* __restrict__ rows, const int* __restrict__ slot_of, const float* __restrict__ weights,
                                int top, int width, float* __restrict__ out, int add) {
    const int64_t t = blockIdx.x;
    for (int i = blockIdx.y * blockDim.x + threadIdx.x; i < width; i += gridDim.y * blockDim.x) {
        float v = add ? out[t * width + i] : 0.f;
        for (int j = 0; j < top; ++j) {
            const int s = slot_of[t * top + j];
            if (s >= 0) v += weights[t * top + j] * rows[(int64_t)s * width + i];
        }
        out[t * width + i] = v;
    }
}

extern "C" int li_pair_sum(const float* rows, const int* slot_of, const float* weights, int n_tokens, int top, int width, float* out,
                           int add, hipStream_t stream) {
    if (n_tokens <= 0 || width <= 0) return LI_OK;
    if (!rows || !slot_of || !weights || !out || top < 1) return LI_BAD_ARG;
    dim3 grid(n_tokens, n_tokens >= 1024 ? 1 : (width + 1023) / 1024);
    pair_sum_kernel<<<grid, 256, 0, stream>>>(rows, slot_of, weights, top, width, out, add);
    LI_CHECK_LAUNCH();
    return LI_OK;
}
