// The selective state-space recurrence of a prompt on the matrix cores (the token-by-token kernels and the formula: hybrid.hip).
// A sequence's tokens are cut into chunks of 64.  With l_t the sum of log a up to and with token t of a chunk, S the state before it
// and S' the one after it,
//   y_t = exp(l_t) C_t S + sum over s <= t of exp(l_t - l_s) dt_s (C_t . B_s) x_s + D x_t
//   S'  = exp(l_64) S + sum over t of exp(l_64 - l_t) dt_t B_t x_t^T
// so that all of it but the walk over the chunks' states is products of matrices.  They are float32 products
// (v_mfma_f32_16x16x4_f32), every exponent is at most 0, and the sums l_t, whose differences are taken, are 64-bit numbers (in 32
// bits the results were ten times as far off): operands, sums and decays are as exact as in the token-by-token form.
//   ssm_scores      C_t . B_s of a chunk, once for all heads of a group
//   ssm_chunk_state what a chunk adds to a head's state, and its whole decay
//   ssm_combine     (hybrid.hip) the walk: the state before every chunk where its contribution was
//   ssm_chunk_out   y
// An instruction's four k are one of each group of 16 lanes; a lane holds four consecutive k of a row in one 16-byte load, so
// instruction j of four takes k = 4 g + j from group g, in both operands (the order of K is free).
// Bound by the chunks' states, written twice and read twice (128 heads of 128 x 64: 4 MB a chunk), then by the matrix
// instructions.  128 heads of 128 x 64, us in segments on the vector units and so: 300 tokens 187 and 81, 2,000 tokens 745 and 288,
// four sequences of 300 to 700 905 and 329, 8,000 tokens 2,645 and 1,280.
#include "common.h"

#define SSM_CHUNK 64

__device__ __forceinline__ f32x4 mfma16_f32(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

struct SsmChunks {
    const float* xbc;            // [T, xbc_stride]: x [P, dv] | B [G, N] | C [G, N]
    const float* proj;           // [T, proj_stride], the raw step sizes from column dt_col on
    const float* dt_bias;        // [P]
    const float* A_log;          // [P]
    const float* D;              // [P] or null
    const int* seq_qstart;
    const int* seg_seq;          // [chunks] its sequence, first token and tokens
    const int* seg_t0;
    const int* seg_n;
    float* scores;               // [chunks, G, 64, 64]; [t][s] for s up to the end of t's tile of 16
    float* seg_state;            // [chunks, P, N, dv]
    float* seg_decay;            // [chunks, P]
    float* y;                    // [T, P dv]
    int xbc_stride, proj_stride, dt_col, P, G, N, dv;
};

// exp of a 64-bit number, in 32 bits: what the exponent loses when it is rounded is a factor of its own.
__device__ __forceinline__ float exp_of(double v) {
    const float hi = (float)v;
    return expf(hi) * (1.f + (float)(v - (double)hi));
}

// Lane t: dt_t (0 beyond the chunk's tokens) and l_t.
__device__ __forceinline__ void chunk_decays(const SsmChunks& c, int64_t q0, int n, int h, float& dt, double& l) {
    const int lane = threadIdx.x & 63;
    const float raw = c.proj[(q0 + min(lane, n - 1)) * c.proj_stride + c.dt_col + h] + c.dt_bias[h];
    dt = lane < n ? (raw > 20.f ? raw : log1pf(expf(raw))) : 0.f;
    l = -(double)expf(c.A_log[h]) * (double)dt;
#pragma unroll
    for (int o = 1; o < WAVE; o <<= 1) {
        const double v = __shfl_up(l, o, WAVE);
        if (lane >= o) l += v;
    }
}

__global__ __launch_bounds__(256) void ssm_scores_kernel(SsmChunks c) {
    const int seg = blockIdx.x, grp = blockIdx.y, lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, g = lane >> 4;
    const int n = c.seg_n[seg];
    const int64_t q0 = c.seq_qstart[c.seg_seq[seg]] + c.seg_t0[seg];
    const float* b0 = c.xbc + c.P * c.dv + grp * c.N + 4 * g;
    const float* crow = b0 + c.G * c.N + (q0 + min(16 * wave + r, n - 1)) * c.xbc_stride;
    const float* brow[4];
    f32x4 acc[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        brow[s] = b0 + (q0 + min(16 * s + r, n - 1)) * c.xbc_stride;
        acc[s] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    for (int k = 0; k < c.N; k += 16) {
        const f32x4 a = *(const f32x4*)(crow + k);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            if (s > wave) continue;                  // (later tokens: not read)
            const f32x4 b = *(const f32x4*)(brow[s] + k);
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[s] = mfma16_f32(a[j], b[j], acc[s]);
        }
    }
    float* out = c.scores + (((int64_t)seg * c.G + grp) * SSM_CHUNK + 16 * wave + 4 * g) * SSM_CHUNK + r;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        if (s > wave) continue;
#pragma unroll
        for (int q = 0; q < 4; ++q) out[q * SSM_CHUNK + 16 * s] = acc[s][q];
    }
}

// A workgroup a chunk, head and 64 columns of dv; its waves take the tiles of 16 rows of N in turn, TW each.
template <int TW>
__global__ __launch_bounds__(256) void ssm_chunk_state_kernel(SsmChunks c) {
    const int seg = blockIdx.x, h = blockIdx.y, dv0 = blockIdx.z * 64;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, g = lane >> 4;
    const int n = c.seg_n[seg], n_tiles = c.N >> 4;
    const int64_t q0 = c.seq_qstart[c.seg_seq[seg]] + c.seg_t0[seg];
    float dt;
    double l;
    chunk_decays(c, q0, n, h, dt, l);
    const double last = __shfl(l, WAVE - 1, WAVE);
    const float weight = exp_of(last - l) * dt;
    if (threadIdx.x == 0 && blockIdx.z == 0) c.seg_decay[(int64_t)seg * c.P + h] = exp_of(last);
    const float* x0 = c.xbc + (int64_t)h * c.dv + dv0 + r;
    const float* b0 = c.xbc + c.P * c.dv + h / (c.P / c.G) * c.N + r;
    f32x4 acc[TW][4];
#pragma unroll
    for (int i = 0; i < TW; ++i)
#pragma unroll
        for (int d = 0; d < 4; ++d) acc[i][d] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int b = 0; b < 4; ++b) {
        if (16 * b >= n) break;
        float x[4][4], bb[TW][4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int t = 16 * b + 4 * g + j;
            const int64_t at = (q0 + min(t, n - 1)) * c.xbc_stride;
            const float w = __shfl(weight, t, WAVE);
#pragma unroll
            for (int d = 0; d < 4; ++d) x[d][j] = dv0 + 16 * d < c.dv ? x0[at + 16 * d] * w : 0.f;
#pragma unroll
            for (int i = 0; i < TW; ++i) bb[i][j] = wave + 4 * i < n_tiles ? b0[at + 16 * (wave + 4 * i)] : 0.f;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int i = 0; i < TW; ++i)
#pragma unroll
                for (int d = 0; d < 4; ++d) acc[i][d] = mfma16_f32(bb[i][j], x[d][j], acc[i][d]);
    }
#pragma unroll
    for (int i = 0; i < TW; ++i) {
        if (wave + 4 * i >= n_tiles) continue;
        float* out = c.seg_state + (((int64_t)seg * c.P + h) * c.N + 16 * (wave + 4 * i) + 4 * g) * c.dv + dv0 + r;
#pragma unroll
        for (int d = 0; d < 4; ++d)
            if (dv0 + 16 * d < c.dv)
#pragma unroll
                for (int q = 0; q < 4; ++q) out[(int64_t)q * c.dv + 16 * d] = acc[i][d][q];
    }
}

// A workgroup a chunk, head and 64 columns of dv, 16 columns a wave.
__global__ __launch_bounds__(256) void ssm_chunk_out_kernel(SsmChunks c) {
    constexpr int LD = SSM_CHUNK + 4;
    __shared__ f32x4 decayed4[SSM_CHUNK * LD / 4];           // [t][s]: scores x exp(l_t - l_s) dt_s
    float* decayed = (float*)decayed4;
    const int seg = blockIdx.x, h = blockIdx.y;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, g = lane >> 4;
    const int n = c.seg_n[seg], grp = h / (c.P / c.G), inner = c.P * c.dv;
    const int64_t q0 = c.seq_qstart[c.seg_seq[seg]] + c.seg_t0[seg];
    float dt;
    double l;
    chunk_decays(c, q0, n, h, dt, l);
    const float* score = c.scores + (((int64_t)seg * c.G + grp) * SSM_CHUNK + 16 * wave) * SSM_CHUNK + lane;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int t = 16 * wave + i;
        const double lt = __shfl(l, t, WAVE);
        decayed[t * LD + lane] = lane <= t ? score[i * SSM_CHUNK] * exp_of(lt - l) * dt : 0.f;
    }
    __syncthreads();
    const int col = blockIdx.z * 64 + 16 * wave;
    if (col >= c.dv) return;
    const int64_t xcol = (int64_t)h * c.dv + col + r;
    const float* crow[4];
    f32x4 acc[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        crow[t] = c.xbc + inner + c.G * c.N + grp * c.N + 4 * g + (q0 + min(16 * t + r, n - 1)) * c.xbc_stride;
        acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    const float* S = c.seg_state + (((int64_t)seg * c.P + h) * c.N + 4 * g) * c.dv + col + r;
#pragma unroll 2
    for (int k = 0; k < c.N; k += 16) {
        f32x4 a[4];
        float s[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) s[j] = S[(int64_t)(k + j) * c.dv];
#pragma unroll
        for (int t = 0; t < 4; ++t) a[t] = *(const f32x4*)(crow[t] + k);
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int t = 0; t < 4; ++t) acc[t] = mfma16_f32(a[t][j], s[j], acc[t]);
    }
    const float decay = exp_of(l);
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[t][q] *= __shfl(decay, 16 * t + 4 * g + q, WAVE);
#pragma unroll
    for (int b = 0; b < 4; ++b) {
        if (16 * b >= n) break;
        float x[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) x[j] = c.xbc[(q0 + min(16 * b + 4 * g + j, n - 1)) * c.xbc_stride + xcol];
#pragma unroll
        for (int t = b; t < 4; ++t) {
            const f32x4 m = *(const f32x4*)(decayed + (16 * t + r) * LD + 16 * b + 4 * g);
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[t] = mfma16_f32(m[j], x[j], acc[t]);
        }
    }
    const float dh = c.D ? c.D[h] : 0.f;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int at = 16 * t + 4 * g + q;
            if (at < n) c.y[(q0 + at) * inner + xcol] = acc[t][q] + dh * c.xbc[(q0 + at) * c.xbc_stride + xcol];
        }
}

extern "C" int li_ssm_combine(float* state, const int* seq_slot, const int* seq_seg0, const int* seq_nseg, float* seg_state,
                              const float* seg_decay, int n_seqs, int P, int64_t per_head, hipStream_t stream);

// Sequences in chunks of at most 64 tokens (seg_*, as li_ssm_scan_segments takes segments).  N and dv multiples of 16, N at most 256;
// xbc 16-byte aligned with rows of a multiple of 4.  scores [chunks, G, 64, 64], seg_state [chunks, P, N, dv], seg_decay
// [chunks, P]: scratch memory of the caller.
extern "C" int li_ssm_chunks(const float* xbc, int xbc_stride, const float* proj, int proj_stride, int dt_col, const float* dt_bias,
                             const float* A_log, const float* D, float* state, const int* seq_slot, const int* seq_qstart, float* y,
                             int n_seqs, int P, int G, int N, int dv, const int* seg_seq, const int* seg_t0, const int* seg_n,
                             const int* seq_seg0, const int* seq_nseg, int n_segs, float* scores, float* seg_state, float* seg_decay,
                             hipStream_t stream) {
    if (n_seqs <= 0 || n_segs <= 0) return LI_OK;
    if (P <= 0 || G <= 0 || P % G || N <= 0 || dv <= 0 || !seq_qstart || !scores || !seg_state || !seg_decay) return LI_BAD_ARG;
    if (N > 256 || N % 16 || dv % 16 || xbc_stride % 4 || (uintptr_t)xbc % 16 || P > 65535 || G > 65535) return LI_UNSUPPORTED;
    const SsmChunks c{xbc, proj, dt_bias, A_log, D, seq_qstart, seg_seq, seg_t0, seg_n, scores, seg_state, seg_decay, y,
                      xbc_stride, proj_stride, dt_col, P, G, N, dv};
    const dim3 grid(n_segs, P, (dv + 63) / 64);
    ssm_scores_kernel<<<dim3(n_segs, G), 256, 0, stream>>>(c);
    if (N <= 64) ssm_chunk_state_kernel<1><<<grid, 256, 0, stream>>>(c);
    else if (N <= 128) ssm_chunk_state_kernel<2><<<grid, 256, 0, stream>>>(c);
    else ssm_chunk_state_kernel<4><<<grid, 256, 0, stream>>>(c);
    const int rc = li_ssm_combine(state, seq_slot, seq_seg0, seq_nseg, seg_state, seg_decay, n_seqs, P, (int64_t)N * dv, stream);
    if (rc) return rc;
    ssm_chunk_out_kernel<<<grid, 256, 0, stream>>>(c);
    LI_CHECK_LAUNCH();
    return LI_OK;
}
