// Matrix products of float32 operands  C[M, N] = X[M, K] . W[N, K]^T  on the matrix cores, for the 32-bit path.
//
// v_mfma_f32_16x16x4_f32 adds its products one after the other in ascending k, each as a fused multiply-add rounded to
// nearest, subnormal numbers kept: an accumulator that takes k in ascending order is bit for bit the chain of fmaf that
// gemm_fma runs (compared on an MI355X, operands, products and sums below 2^-126 among them).  The kernels here sum as gemm_fma does, chains
// over 256 consecutive k that are added up in ascending order, so a result depends neither on the kernel nor on the batch,
// and a call that these do not take (K no multiple of 16, an address that is not 16-byte aligned) gives the same numbers
// through gemm_fma.
//
//   gemv_f32   few rows of X: W from memory straight into operand A, the waves of a workgroup take chains in turn
//   gemm_f32   many rows: tiles of W and X through LDS
//   gemm_f32_chains   rows between: smaller tiles, whose chains the waves of a workgroup take in turn
//
// The operands lie row-major, so a lane fetches four consecutive k of its row with one 16-byte load; what instruction j
// wants instead is k = 4 j + lane / 16.  gemv_f32 turns one into the other in registers, by four swaps of half waves and
// of quarters (v_permlane32_swap, v_permlane16_swap) for four instructions; gemm_f32 on the way into LDS;
// gemm_f32_chains reads LDS word by word.
#include "gemm_common.h"

#define CHAIN 256                       // consecutive k of one chain of multiply-adds (as in gemm_fma)
#define F32_TILES ((1 << 24) - 8)       // tiles of gemm_f32's grid, in one dimension: a launch has fewer than 2^32 threads in each

__device__ __forceinline__ f32x4 mfma16_f32(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

__device__ __forceinline__ void swap32(float& x, float& y) {      // x's upper half wave <-> y's lower half wave
    auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(y), false, false);
    x = __uint_as_float(p[0]);
    y = __uint_as_float(p[1]);
}
__device__ __forceinline__ void swap16(float& x, float& y) {      // the same within either half
    auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(y), false, false);
    x = __uint_as_float(p[0]);
    y = __uint_as_float(p[1]);
}
// Lane l holds k = 4 (l / 16) .. + 3 of a row; afterwards element j holds k = 4 j + l / 16.
__device__ __forceinline__ void to_operand16(f32x4& v) {
    float a = v[0], b = v[1], c = v[2], d = v[3];
    swap32(a, c);
    swap32(b, d);
    swap16(a, b);
    swap16(c, d);
    v = f32x4{a, b, c, d};
}

// ===========================================================================
// gemv_f32: 16 NT rows of W, 16 MT rows of X, KW waves.  Wave w takes the chains w, w + KW, ... and leaves each
// finished one in LDS, where a wave per 16 x 16 tile adds them up in ascending order: K is shared by the waves and the sum
// is still taken in one order.  Bound by the stream of W: 128,256 x 2,048 at 3 rows 180 us, 5.8 TB/s (gemm_fma: 942 us);
// 16,384 x 2,048 27 us, 5.0 TB/s (222); short products end a few us after their stream (2,048 x 2,048 9.7 us, 201 before;
// 2,048 x 8,192 29, 862 before), and with a workgroup on half the CUs the matrix instructions take as long as the stream.
// U steps of 16 k whose loads go out together: 4, so that eight waves fit a SIMD (with 16 the first of these takes 187 us, the
// second 37).
// HALF (at most 8 rows of X): 8 rows of W a workgroup, and wave w takes pairs of neighbouring chains, 2 w and 2 w + 1, then those
// 2 KW on.  The lanes of r < 8 hold the first chain of a pair, the others the second of the same rows, and likewise the columns
// of X: of the 16 x 16 sums the two diagonal quarters are the two chains, each in its order.  Twice the workgroups and no
// instruction more: 2,048 x 2,048 9.8 -> 7.6 us at 3 rows, 2,048 x 8,192 29.0 -> 19.6 (8 rows 32.5 -> 24.0); 4,096 x 4,096 17.5
// and 18.3, where every CU has its workgroup without it.
// WHOLE (K a multiple of a wave's chain, or pair of them): a chain's sixteen steps under no condition, U of them on their way and the
// next one asked for as soon as a step's registers are free, in the order that is written (left to itself the compiler asked for two steps
// and waited for them, and a step's condition was a branch).  A wave's loads are then what a step waits for, so it pays where a wave has one chain
// or a CU one workgroup; else four steps at a time in more waves are as fast.  us at 1, 3 and 8 rows, before and now: 2,048 x 2,048 7.3 -> 6.1, 7.5 ->
// 6.2, 7.7 -> 6.9; 2,048 x 8,192 18.5 -> 15.9, 19.5 -> 16.8, 23.8 -> 20.4; 3,072 x 2,048 9.9 -> 8.0, 10.0 -> 8.3, 10.2 -> 9.0; 16,384 x 2,048
// 28.1 -> 24.8, 27.6 -> 25.7, 30.8 -> 29.4; 4,096 x 14,336 53.6 -> 45.2, 55.5 -> 46.4, 61.7 -> 51.9; but 28,672 x 4,096 at 4 rows 88.3 and 89.6.
// ===========================================================================
template <int NT, int MT, int KW, int U, bool HALF = false, bool WHOLE = false>
__global__ __launch_bounds__(64 * KW) void gemv_f32_kernel(const float* __restrict__ X, const float* __restrict__ W, int K, Epilogue e) {
    __shared__ f32x4 part[KW][NT * MT][64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 15, g = lane >> 4;
    constexpr int ROWS = HALF ? 8 : 16, CL = HALF ? 2 : 1;               // rows of W, and of X, of a tile; chains of one accumulator
    const int n0 = blockIdx.x * ROWS * NT, m0 = blockIdx.y * ROWS * MT;
    const int row = HALF ? r & 7 : r, later = HALF ? r >> 3 : 0;         // (HALF: lanes of r >= 8 hold the same rows in the next chain)
    const float *wp[NT], *xp[MT];                    // rows beyond the last are the last again, and not stored
#pragma unroll
    for (int t = 0; t < NT; ++t) wp[t] = W + (int64_t)min(n0 + 16 * t + row, e.N - 1) * K + 4 * g;
#pragma unroll
    for (int j = 0; j < MT; ++j) xp[j] = X + (int64_t)min(m0 + 16 * j + row, e.M - 1) * K + 4 * g;
    const int chains = (K + CHAIN - 1) / CHAIN;
    constexpr int OWN = (NT * MT + KW - 1) / KW;     // tiles whose sums this wave adds up
    f32x4 total[OWN];
#pragma unroll
    for (int o = 0; o < OWN; ++o) total[o] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int c0 = 0; c0 < chains; c0 += KW * CL) {
        const int c = c0 + wave * CL;
        if (c < chains) {
            f32x4 acc[NT][MT];
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int j = 0; j < MT; ++j) acc[t][j] = f32x4{0.f, 0.f, 0.f, 0.f};
            // (HALF: the first chain of a pair is whole, the second may be short or missing; what it has no steps for it takes
            // from the row's end, and that is not added)
            const int k0 = c * CHAIN, steps = min(CHAIN, K - k0) >> 4;
            const int mine = HALF && later ? max(0, min(CHAIN, K - k0 - CHAIN)) >> 4 : steps;
            const int from = HALF && later ? min(k0 + CHAIN, K - 16) : k0;
            if constexpr (WHOLE) {
                constexpr int STEPS = CHAIN / 16;
                f32x4 a[U][NT], b[U][MT];
                const float *wc[NT], *xc[MT];
#pragma unroll
                for (int t = 0; t < NT; ++t) wc[t] = wp[t] + from;
#pragma unroll
                for (int j = 0; j < MT; ++j) xc[j] = xp[j] + from;
                auto fetch = [&](int s) {
#pragma unroll
                    for (int t = 0; t < NT; ++t) a[s % U][t] = *(const f32x4*)(wc[t] + 16 * s);
#pragma unroll
                    for (int j = 0; j < MT; ++j) b[s % U][j] = *(const f32x4*)(xc[j] + 16 * s);
                };
#pragma unroll
                for (int s = 0; s < U; ++s) fetch(s);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int s = 0; s < STEPS; ++s) {
                    const int u = s % U;
#pragma unroll
                    for (int t = 0; t < NT; ++t) to_operand16(a[u][t]);
#pragma unroll
                    for (int j = 0; j < MT; ++j) to_operand16(b[u][j]);
#pragma unroll
                    for (int i = 0; i < 4; ++i)
#pragma unroll
                        for (int t = 0; t < NT; ++t)
#pragma unroll
                            for (int j = 0; j < MT; ++j) acc[t][j] = mfma16_f32(a[u][t][i], b[u][j][i], acc[t][j]);
                    __builtin_amdgcn_sched_barrier(0);
                    if (s + U < STEPS) fetch(s + U);
                    __builtin_amdgcn_sched_barrier(0);
                }
            } else
            for (int s0 = 0; s0 < steps; s0 += U) {
                f32x4 a[U][NT], b[U][MT];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int k = from + 16 * max(0, min(s0 + u, mine - 1));      // (a step that is not there: the last again, unused)
#pragma unroll
                    for (int t = 0; t < NT; ++t) a[u][t] = *(const f32x4*)(wp[t] + k);
#pragma unroll
                    for (int j = 0; j < MT; ++j) b[u][j] = *(const f32x4*)(xp[j] + k);
                }
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    if (s0 + u < steps) {
                        if (HALF && s0 + u >= mine) a[u][0] = b[u][0] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                        for (int t = 0; t < NT; ++t) to_operand16(a[u][t]);
#pragma unroll
                        for (int j = 0; j < MT; ++j) to_operand16(b[u][j]);
#pragma unroll
                        for (int i = 0; i < 4; ++i)
#pragma unroll
                            for (int t = 0; t < NT; ++t)
#pragma unroll
                                for (int j = 0; j < MT; ++j) acc[t][j] = mfma16_f32(a[u][t][i], b[u][j][i], acc[t][j]);
                    }
                }
            }
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int j = 0; j < MT; ++j) part[wave][t * MT + j][lane] = acc[t][j];
        }
        __syncthreads();
        const int have = min(KW, (chains - c0 + CL - 1) / CL);
#pragma unroll
        for (int o = 0; o < OWN; ++o) {
            const int q = wave + o * KW;
            if (q < NT * MT)
                for (int w = 0; w < have; ++w) {
                    total[o] += part[w][q][lane];
                    // rows 4 g + q (g < 2) of column r (r < 8): the second chain's sums lie 40 lanes on
                    if (HALF && c0 + 2 * w + 1 < chains) total[o] += part[w][q][(lane + 40) & 63];
                }
        }
        __syncthreads();
    }
#pragma unroll
    for (int o = 0; o < OWN; ++o) {
        const int q = wave + o * KW;
        if (q < NT * MT) {
            const float v[4] = {total[o][0], total[o][1], total[o][2], total[o][3]};
            if (!HALF || (r < 8 && g < 2)) epilogue4(e, m0 + 16 * (q % MT) + r, n0 + 16 * (q / MT) + 4 * g, v);
        }
    }
}

// ===========================================================================
// gemm_f32: 64 rows of W x 64 rows of X, 4 waves of 32 x 32 (four sums of 16 x 16, which do not wait for each other), 32 of K a
// stage, three stages in LDS.  While a stage is multiplied out of registers, the operands of the next are read from LDS,
// the one after that is written to LDS and the third is on its way from memory, so that a workgroup alone on its CU
// keeps the matrix cores busy.  In LDS the sixteen k of a step lie as the instructions want them (k = 4 j + g at 4 g + j), dealt
// out as they are written: swapped in registers as gemv_f32 does it, they cost a third of the matrix
// instructions' own time.  Rows are 36 floats apart, which keeps the 16-byte reads of a quarter wave on different banks.
// Bound by the matrix instructions (32 cycles each): 28,672 x 4,096 at 2,048 rows 3.99 ms, 121 TFLOP/s, the matrix cores busy three
// quarters of the time, LDS a quarter (a third of that bank conflicts of the writes), waves waiting for LDS 4% of theirs.  Few
// tiles: a tile's own instructions one after another, at 400 rows 2,048 x 2,048 27 of 41 us (gemm_fma: 233); 16,384 x 2,048
// 259 us (1,076).
// ===========================================================================
__global__ __launch_bounds__(256, 2) void gemm_f32_kernel(const float* __restrict__ X, const float* __restrict__ W, int K, int tiles_m, int tiles, Epilogue e) {
    constexpr int BK = 32, LD = BK + 4, ST = 2 * 64 * LD;              // a stage in LDS: rows of W, then rows of X
    __shared__ f32x4 lds4[3 * ST / 4];
    float* lds = (float*)lds4;
    // workgroups go round the eight XCDs: each XCD takes a run of tiles, the rows of X fastest, so that a tile of W is
    // fetched into one L2
    const int id = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    if (id >= tiles) return;
    const int n0 = id / tiles_m * 64, m0 = id % tiles_m * 64;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r = lane & 15, g = lane >> 4;
    const int wn = (wave & 1) * 32, wm = (wave >> 1) * 32;
    f32x4 acc[2][2], total[2][2];
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i >> 1][i & 1] = total[i >> 1][i & 1] = f32x4{0.f, 0.f, 0.f, 0.f};
    // this thread fetches four of the first and of the second sixteen k of a row of W and of X: a wave then writes to sixteen
    // rows of LDS at a time, each on banks of its own
    const int row = tid >> 2, kc = (tid & 3) * 4;
    const float *wp = W + (int64_t)min(n0 + row, e.N - 1) * K, *xp = X + (int64_t)min(m0 + row, e.M - 1) * K;
    f32x4 st[4];
    auto fetch = [&](int k0) {                       // (what lies beyond K is the row's end again, and not multiplied)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int k = min(k0 + 16 * u + kc, K - 4);
            st[u] = *(const f32x4*)(wp + k);
            st[2 + u] = *(const f32x4*)(xp + k);
        }
    };
    const int put_at = row * LD + (tid & 3);
    auto put = [&](int at) {
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int q = 0; q < 4; ++q) lds[4 * at + put_at + 64 * (c >> 1) * LD + 16 * (c & 1) + 4 * q] = st[c][q];
    };
    const int w_at = (wn + r) * (LD / 4) + g, x_at = (64 + wm + r) * (LD / 4) + g;
    f32x4 op[2][2][4];                               // [stage's parity][sixteen of K][two blocks of W, two of X]
    auto operands = [&](f32x4 (&o)[2][4], int at) {                  // (`at`: in pieces of 16 bytes)
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                o[u][i] = lds4[at + w_at + 4 * i * LD + 4 * u];
                o[u][2 + i] = lds4[at + x_at + 4 * i * LD + 4 * u];
            }
    };
    auto multiply = [&](f32x4 (&o)[4]) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[i >> 1][i & 1] = mfma16_f32(o[i >> 1][q], o[2 + (i & 1)][q], acc[i >> 1][i & 1]);
    };
    fetch(0);
    put(0);
    fetch(BK);
    put(ST / 4);
    fetch(2 * BK);
    __syncthreads();
    operands(op[0], 0);
    int next = ST / 4, after = 2 * ST / 4, spent = 0;        // the stages in LDS: the next one, the one that is written now, the last one
    for (int k0 = 0; k0 < K; k0 += 2 * BK) {
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const int k = k0 + b * BK;
            if (k >= K) break;
            if (k && k % CHAIN == 0) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    total[i >> 1][i & 1] += acc[i >> 1][i & 1];
                    acc[i >> 1][i & 1] = f32x4{0.f, 0.f, 0.f, 0.f};
                }
            }
            operands(op[b ^ 1], next);
            multiply(op[b][0]);
            put(after);
            fetch(k + 3 * BK);
            // the order of the instructions: an operand's read, a write or a load under every matrix instruction
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x200, 2, 0);
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            }
            if (k + 16 < K) multiply(op[b][1]);
            __syncthreads();
            const int t = next;
            next = after;
            after = spent;
            spent = t;
        }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const f32x4 t = total[i >> 1][i & 1] + acc[i >> 1][i & 1];
        const float v[4] = {t[0], t[1], t[2], t[3]};
        epilogue4(e, m0 + wm + 16 * (i & 1) + r, n0 + wn + 16 * (i >> 1) + 4 * g, v);
    }
}

// ===========================================================================
// gemm_f32_chains: 32 rows of W x 32 rows of X, KW waves that take the chains of K in turn (wave w: w, w + KW, ...), each for the whole
// tile (four sums of 16 x 16), and add the finished ones up in ascending order through LDS, as gemv_f32 does: a quarter of gemm_f32's
// tile and a quarter of its serial chain.
// A wave brings 32 of K of its 64 rows, a stage, into LDS of its own by global_load_lds, in units of 8 rows x 128 bytes (whole lines);
// nobody else reads it, so there is no barrier but at the chains' ends.  Two stages in LDS and one in registers: a stage is read while the one
// before it is multiplied, and the one two on is fetched into its place.
// Operands are read word by word (lane (r, g) wants k = 4 j + g of row r; two blocks of 16 rows an instruction); chunk c of 16 bytes of row r lies
// at place c ^ (r / 2 % 8), so that the sixteen rows are on different banks.
// Bound by the rows it fetches (32 bytes a cycle and CU at the matrix cores' rate; it gets 12 to 13 TB/s in all) where there are many tiles, by a
// tile's own 7 us of instructions at K = 2,048 where there are few.  us, before (gemv_f32 up to 64 or 128 rows, gemm_f32) and now: 32 rows x 2,048 x
// 2,048 15.2 and 13.3, x 2,048 x 8,192 57.1 and 46.2, x 6,144 x 4,096 55.9 and 29.1; 64 rows 23.9 and 13.2, 91.4 and 43.5, 85.5 and 45.4; 200 rows
// 45.2 and 23.0, 174 and 77.6, 149 and 118; 375 rows 45.9 and 34.2, 174 and 118, 226 and 183.  Stages read in the first third of the
// one before, so that the next is fetched earlier: 14% slower; one stage in LDS and three workgroups a CU: a third slower; two waves a workgroup: 10 to 60%.
// ===========================================================================
template <int KW>
__global__ __launch_bounds__(64 * KW, 2) void gemm_f32_chains_kernel(const float* __restrict__ X, const float* __restrict__ W, int K, int tiles_m, int tiles,
                                                                    Epilogue e) {
    constexpr int STAGE = 8 * 1024, STAGES = CHAIN / 32, OWN = 4 / KW;
    static_assert(KW == 2 || KW == 4, "the four blocks are dealt to the waves");
    extern __shared__ __attribute__((aligned(1024))) unsigned char f32_smem[];       // KW x (two stages), then KW x (four blocks of sums)
    const int id = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);           // (as gemm_f32)
    if (id >= tiles) return;
    const int n0 = id / tiles_m * 32, m0 = id % tiles_m * 32;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 15, g = lane >> 4;
    const int chains = K / CHAIN;                                                     // (K is a multiple of a chain)
    const int mine = (chains - wave + KW - 1) / KW, all = mine * STAGES;             // this wave's chains and stages
    unsigned char* region = f32_smem + wave * 2 * STAGE;
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)region;
    const uint32_t sums = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)f32_smem + KW * 2 * STAGE + lane * 16;
    // unit q < 4: rows 8 q .. of W, then of X; lane 8 p + c brings chunk c ^ (row / 2 % 8) of row 8 q + p (rows beyond the last: the last)
    const float* from[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        const int p = lane >> 3, row = 8 * (q & 3) + p, chunk = (lane & 7) ^ ((row >> 1) & 7);
        from[q] = (q < 4 ? W + (int64_t)min(n0 + row, e.N - 1) * K : X + (int64_t)min(m0 + row, e.M - 1) * K) + 4 * chunk;
    }
    auto fetch = [&](int t) {                        // stage t of this wave into place t % 2 (t beyond the last: the last again, unused)
        const int s = min(t, all - 1), k = (wave + KW * (s / STAGES)) * CHAIN + s % STAGES * 32;
#pragma unroll
        for (int q = 0; q < 8; ++q)
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(from[q] + k),
                                             (__attribute__((address_space(3))) void*)(region + (t & 1) * STAGE + q * 1024), 16, 0, 0);
    };
    uint32_t at[8];                                  // chunk c of row r of a block; the next block lies 2 KiB on
#pragma unroll
    for (int c = 0; c < 8; ++c) at[c] = lds0 + (r >> 3) * 1024 + (r & 7) * 128 + ((c ^ (r >> 1)) * 16) + 4 * g;
    f32x2 a[2][8], b[2][8];                          // [stage's parity][chunk]: both blocks of W, both of X
#define READ(SET, C)                                                                                                             \
    do {                                                                                                                        \
        asm volatile("ds_read2st64_b32 %0, %1 offset0:0 offset1:8" : "=v"(a[SET][C]) : "v"(at[C] + (SET) * STAGE) : "memory");   \
        asm volatile("ds_read2st64_b32 %0, %1 offset0:16 offset1:24" : "=v"(b[SET][C]) : "v"(at[C] + (SET) * STAGE) : "memory"); \
    } while (0)
    f32x4 acc[2][2], total[OWN];
#pragma unroll
    for (int o = 0; o < OWN; ++o) total[o] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (all > 0) {
        fetch(0);
        fetch(1);
        __builtin_amdgcn_s_waitcnt(0x0F78);                                           // vmcnt(8): stage 0 has landed
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int c = 0; c < 8; ++c) READ(0, c);
        __builtin_amdgcn_s_waitcnt(0xC07F);                                           // lgkmcnt(0)
        __builtin_amdgcn_sched_barrier(0);
        fetch(2);
    }
    for (int c0 = 0; c0 < chains; c0 += KW) {
        const int t0 = c0 / KW * STAGES;
        if (c0 + wave < chains) {
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[i >> 1][i & 1] = f32x4{0.f, 0.f, 0.f, 0.f};
            for (int t = t0; t < t0 + STAGES; t += 2) {
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    __builtin_amdgcn_sched_barrier(0);
                    __builtin_amdgcn_s_waitcnt(0x0F78);                               // vmcnt(8): stage t + u + 1 has landed
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int c = 0; c < 8; ++c) {
                        READ(u ^ 1, c);
#pragma unroll
                        for (int i = 0; i < 4; ++i) acc[i >> 1][i & 1] = mfma16_f32(a[u][c][i >> 1], b[u][c][i & 1], acc[i >> 1][i & 1]);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    __builtin_amdgcn_s_waitcnt(0xC07F);                               // lgkmcnt(0)
                    __builtin_amdgcn_sched_barrier(0);
                    fetch(t + u + 3);                // the next stage is in registers: its place is free
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            // (the compiler does not know that the stores below read what a matrix instruction writes: 19 cycles after the last one)
            asm volatile("s_nop 15\n\ts_nop 7" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < 4; ++i)
                asm volatile("ds_write_b128 %0, %1 offset:%2" ::"v"(sums + wave * 4096), "v"(acc[i >> 1][i & 1]), "n"(i * 1024) : "memory");
        }
        __builtin_amdgcn_s_waitcnt(0xC07F);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        const int have = min(KW, chains - c0);
#pragma unroll
        for (int o = 0; o < OWN; ++o) {
            f32x4 part[KW];
#pragma unroll
            for (int w = 0; w < KW; ++w)
                asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(part[w]) : "v"(sums + (wave + o * KW) * 1024), "n"(w * 4096) : "memory");
            __builtin_amdgcn_s_waitcnt(0xC07F);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int w = 0; w < KW; ++w)
                if (w < have) total[o] += part[w];
        }
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);              // nothing is in flight into LDS when the workgroup ends
#pragma unroll
    for (int o = 0; o < OWN; ++o) {
        const int q = wave + o * KW;
        const float v[4] = {total[o][0], total[o][1], total[o][2], total[o][3]};
        epilogue4(e, m0 + 16 * (q & 1) + r, n0 + 16 * (q >> 1) + 4 * g, v);
    }
#undef READ
}

// ===========================================================================
// C interface
// ===========================================================================
// kind: 0 = by the sizes, 1 = gemv_f32 (at most 128 rows), 2 = gemm_f32, 3 = gemm_f32_chains (whole chains only).
extern "C" int li_gemm_f32(const float* X, const float* W, void* C, int out_dt, int mode, int M, int N, int K, int kind,
                           const RopeStore* rs, hipStream_t stream) {
    int rc = check_common(X, W, C, M, N, K, mode, out_dt);
    if (rc) return rc;
    if (K % 16 != 0 || (((uintptr_t)X | (uintptr_t)W) & 15) || kind < 0 || kind > 3 || (kind == 1 && M > 128) || (kind == 3 && K % CHAIN)) return LI_UNSUPPORTED;
    if (M == 0) return LI_OK;
    Epilogue e;
    rc = make_epilogue(e, C, mode, out_dt, M, N, rs);
    if (rc) return rc;
    const int chains = (K + CHAIN - 1) / CHAIN, blocks = (N + 15) / 16;
    // Whole chains: gemv_f32 up to 16 rows (20: 3,072 x 2,048 at 17 rows 14.0 us, gemm_f32_chains 14.7, at 24 rows 15.2 and 14.7), fewer against many
    // rows of W (6,144 x 4,096 at 9 and 16 rows 29.0 and 28.0, 33.7 and 28.3, at 8 rows 28.9 and 28.1; but 8,192 x 512 6.9 and 7.9).  Beyond, an
    // estimate of both in us, fitted to 2,348 products of 21 to 1,000 rows, 320 to 28,672 rows of W and K of 256 to 8,192: rounds of 256 tiles (one that is
    // not full counts for nearly a whole one), each as long as its K for gemm_f32, and for gemm_f32_chains as the chains of its busiest wave and all
    // of them.  What it names takes 0.2% more than the faster one in the mean, 15% at most; by the rounds alone, with K = 2,048 in mind, it was 3%, where four
    // waves do not share K evenly most (677 rows x 1,024 x 512 13.9 and 16.7, 195 x 28,672 x 1,536 204 and 231, 200 x 8,192 x 256 15.7 and 26.2).
    // Else gemv_f32 has its workgroups by the rows of W alone, gemm_f32 fills the chip only where both sides have enough
    // rows.  us at 64 rows of X: 2,048 x 2,048 25 against 41, 2,048 x 8,192 89 against 160, but 16,384 x 2,048 71 against 49; at
    // 32 rows 16,384 x 2,048 46 against 49
    auto rounds = [&](int side, double last) {
        const int64_t tiles = (int64_t)((M + side - 1) / side) * ((N + side - 1) / side);
        return last * ((tiles + 255) / 256) + (1 - last) * tiles / 256;
    };
    if (kind == 0 && K % CHAIN == 0) {
        const double whole = rounds(64, 0.9) * (1.4 + 0.0156 * K) + 2.7 + 0.004 * K;
        const double shared = (rounds(32, 0.85) + 0.2) * (0.55 + 2.0 * ((chains + 3) / 4) + 0.62 * chains) + 4.4;
        if (M <= 8 || (M <= 20 && (blocks < 384 || chains < 8))) kind = 1;
        else kind = shared < whole && (int64_t)((M + 31) / 32) * ((N + 31) / 32) <= F32_TILES ? 3 : 2;
    } else if (kind == 0) kind = M <= 32 || (M <= 64 && blocks < 1024) || (M <= 128 && blocks <= 256) ? 1 : 2;
    if (kind == 1) {
        const int mt = M <= 16 ? 1 : (M <= 32 ? 2 : 4), nt = M > 8 && blocks >= 1024 ? 2 : 1;
        // sixteen waves where half the CUs have no workgroup (2,048 x 8,192 at 3 rows, whole blocks: 28 against 32 us), else eight; two
        // blocks of W a wave where there are workgroups enough (28,672 x 4,096 at 32 rows: 164 against 169 us)
        const int kw = chains <= 4 ? 4 : (mt == 1 && chains >= 16 && blocks <= 256 ? 16 : 8);
        // up to 128 blocks and 8 rows: half blocks, so that every CU has a workgroup, a wave for each pair of chains.  Beyond 256 blocks with two
        // chains and more a wave, half blocks where the rows are few (us of whole and half ones at 1, 2, 4 and 8 rows: 5,120 x 4,096 24.6 and 19.3,
        // 23.4 and 20.1, 25.2 and 22.4, 28.0 and 26.8; 8,192 x 4,096 29.2 and 26.7, 27.7 and 26.2, 28.0 and 28.9, 30.2 and 36.7; 28,672 x 4,096 88.9
        // and 78.7, 84.2 and 81.5, 88.6 and 92.4; but with pairs that eight waves do not share evenly 2 rows x 8,192 x 14,336 89 and 96, x 11,008 x 5,120 50
        // and 52)
        const bool pairs_whole = K % (2 * CHAIN) == 0;
        const bool few = K % (16 * CHAIN) == 0 && blocks > 256 && (M <= 2 || (M <= 4 && blocks <= 384));
        if (few || (M <= 8 && blocks <= 128)) {
            const int pairs = (chains + 1) / 2, waves = pairs <= 4 ? 4 : pairs <= 8 || few ? 8 : 16;
            const unsigned grid = (N + 7) / 8;
#define HALVES(KW)                                                                                                   \
    do {                                                                                                            \
        if (pairs_whole) gemv_f32_kernel<1, 1, KW, 8, true, true><<<grid, 64 * KW, 0, stream>>>(X, W, K, e);        \
        else gemv_f32_kernel<1, 1, KW, 8, true><<<grid, 64 * KW, 0, stream>>>(X, W, K, e);                          \
    } while (0)
            if (waves == 4) HALVES(4); else if (waves == 8) HALVES(8); else HALVES(16);
#undef HALVES
            LI_CHECK_LAUNCH();
            return LI_OK;
        }
        // one block of W and of X: whole chains where a wave has one of them, or a CU one workgroup
        if (nt == 1 && mt == 1 && K % CHAIN == 0 && (chains <= kw || blocks <= 256)) {
            const unsigned grid = blocks;
            if (kw == 4) gemv_f32_kernel<1, 1, 4, 8, false, true><<<grid, 256, 0, stream>>>(X, W, K, e);
            else if (kw == 8) gemv_f32_kernel<1, 1, 8, 8, false, true><<<grid, 512, 0, stream>>>(X, W, K, e);
            else gemv_f32_kernel<1, 1, 16, 8, false, true><<<grid, 1024, 0, stream>>>(X, W, K, e);
            LI_CHECK_LAUNCH();
            return LI_OK;
        }
#define GO(NT, MT, KW, U)                                                                                                       \
    if (nt == NT && mt == MT && kw == KW) {                                                                                     \
        gemv_f32_kernel<NT, MT, KW, U><<<dim3((blocks + NT - 1) / NT, (M + 16 * MT - 1) / (16 * MT)), 64 * KW, 0, stream>>>(X, W, K, e);                             \
        LI_CHECK_LAUNCH();                                                                                                      \
        return LI_OK;                                                                                                           \
    }
        GO(1, 1, 4, 4) GO(1, 1, 8, 4) GO(1, 1, 16, 4) GO(1, 2, 4, 8) GO(1, 2, 8, 8) GO(1, 4, 4, 4) GO(1, 4, 8, 4)
        GO(2, 1, 4, 4) GO(2, 1, 8, 4) GO(2, 2, 4, 4) GO(2, 2, 8, 4) GO(2, 4, 4, 4) GO(2, 4, 8, 4)
#undef GO
        return LI_UNSUPPORTED;
    }
    if (kind == 3) {
        constexpr int KW = 4, LDS = KW * (2 * 8192 + 4096);
        const int tiles_m = (M + 31) / 32;
        const int64_t tiles = (int64_t)tiles_m * ((N + 31) / 32);
        if (tiles > F32_TILES) return LI_UNSUPPORTED;
        static bool allowed = false;               // more than 64 KiB of LDS is asked for once
        if (!allowed) {
            if (hipFuncSetAttribute((const void*)gemm_f32_chains_kernel<KW>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS) != hipSuccess) return LI_HIP_ERROR;
            allowed = true;
        }
        gemm_f32_chains_kernel<KW><<<(int)((tiles + 7) / 8 * 8), 64 * KW, LDS, stream>>>(X, W, K, tiles_m, (int)tiles, e);
        LI_CHECK_LAUNCH();
        return LI_OK;
    }
    const int tiles_m = (M + 63) / 64;
    const int64_t tiles = (int64_t)tiles_m * ((N + 63) / 64);
    if (tiles > F32_TILES) return LI_UNSUPPORTED;
    gemm_f32_kernel<<<(int)((tiles + 7) / 8 * 8), 256, 0, stream>>>(X, W, K, tiles_m, (int)tiles, e);
    LI_CHECK_LAUNCH();
    return LI_OK;
}
