// Embedding gather, RMSNorm, rotation of q/k with the write into the paged
// cache, and the per-step bookkeeping kernel of decoding.  One kernel for each,
// every size taken at run time.
#include "common.h"

#include <chrono>

// ---------------------------------------------------------------------------
// x[t, :] = float(table[token[t], :])          (src/model/model.cpp:101-118)
// ---------------------------------------------------------------------------
template <class T>
__global__ void embed_kernel(const T* __restrict__ table, const int* __restrict__ tokens,
                             float* __restrict__ x, int d, int vocab) {
    const int t = blockIdx.x;
    int tok = tokens[t];
    tok = tok < 0 ? 0 : (tok >= vocab ? vocab - 1 : tok);   // ids are checked on the host; never read outside
    const T* row = table + (int64_t)tok * d;
    float* out = x + (int64_t)t * d;
    const bool whole = (d & 3) == 0 && (((uintptr_t)table | (uintptr_t)x) & 15) == 0;
    gather_row(d, whole, [&](int i) { *(f32x4*)(out + i) = quad_of(row + i); }, [&](int i) { out[i] = to_f32(row[i]); });
}

extern "C" int li_embed(const void* table, int table_dt, const int* tokens, float* x,
                        int n_tokens, int d, int vocab, hipStream_t stream) {
    if (n_tokens <= 0) return LI_OK;
    if (d <= 0 || vocab <= 0) return LI_BAD_ARG;
    dim3 grid = gather_grid(n_tokens, d), block(GATHER_THREADS);
    if (table_dt == DT_F32) embed_kernel<float><<<grid, block, 0, stream>>>((const float*)table, tokens, x, d, vocab);
    else if (table_dt == DT_F16) embed_kernel<f16><<<grid, block, 0, stream>>>((const f16*)table, tokens, x, d, vocab);
    else if (table_dt == DT_BF16) embed_kernel<bf16><<<grid, block, 0, stream>>>((const bf16*)table, tokens, x, d, vocab);
    else return LI_BAD_ARG;
    LI_CHECK_LAUNCH();
    return LI_OK;
}

// ---------------------------------------------------------------------------
// out[r, :] = x[row(r), :] / sqrt(mean(x^2) + eps) * w     (include/kernels_cpu.hpp:43-54)
// Sum of squares, root and scaling in float32; `rows` (may be null) picks rows.
// ---------------------------------------------------------------------------
// `row_scale` (may be null): row_scale_for(rms) of the first 16 rows, for a product that will add into these
// rows and hand them on in float16 (gemm.hip, RowsOut).
template <class TO>
__global__ void rmsnorm_kernel(const float* __restrict__ x, const float* __restrict__ w,
                               const int* __restrict__ rows, TO* __restrict__ out, int d, float eps,
                               float* __restrict__ row_scale) {
    __shared__ float scratch[16];
    const int r = blockIdx.x;
    const float* xr = x + (int64_t)(rows ? rows[r] : r) * d;
    TO* o = out + (int64_t)r * d;
    float ss = 0.f;
    for (int i = threadIdx.x; i < d; i += blockDim.x) { const float v = xr[i]; ss += v * v; }
    ss = block_sum(ss, scratch);
    const float rms = sqrtf(ss / (float)d + eps);
    if (row_scale && threadIdx.x == 0 && r < 16) row_scale[r] = row_scale_for(rms);
    for (int i = threadIdx.x; i < d; i += blockDim.x) o[i] = from_f32<TO>(xr[i] / rms * w[i]);
}

// The same for rows of up to 4 * V * blockDim.x elements (d a multiple of 4, 16-byte aligned
// pointers): the row and its weights are read once, in 16-byte pieces that stay in registers.
template <class TO, int V>
__global__ void rmsnorm_vec_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                   const int* __restrict__ rows, TO* __restrict__ out, int d, float eps,
                                   float* __restrict__ row_scale) {
    struct alignas(4 * sizeof(TO)) Out4 { TO v[4]; };
    __shared__ float scratch[16];
    const int r = blockIdx.x, n4 = d >> 2;
    const f32x4* xr = (const f32x4*)(x + (int64_t)(rows ? rows[r] : r) * d);
    const f32x4* w4 = (const f32x4*)w;
    Out4* o = (Out4*)(out + (int64_t)r * d);
    f32x4 xv[V], wv[V];
#pragma unroll
    for (int j = 0; j < V; ++j) {
        const int i = threadIdx.x + j * blockDim.x;
        xv[j] = i < n4 ? xr[i] : f32x4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int j = 0; j < V; ++j) {
        const int i = threadIdx.x + j * blockDim.x;
        wv[j] = i < n4 ? w4[i] : f32x4{0.f, 0.f, 0.f, 0.f};
    }
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < V; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) ss += xv[j][q] * xv[j][q];
    ss = block_sum(ss, scratch);
    const float rms = sqrtf(ss / (float)d + eps);
    if (row_scale && threadIdx.x == 0 && r < 16) row_scale[r] = row_scale_for(rms);
#pragma unroll
    for (int j = 0; j < V; ++j) {
        const int i = threadIdx.x + j * blockDim.x;
        if (i < n4) {
            Out4 t;
#pragma unroll
            for (int q = 0; q < 4; ++q) t.v[q] = from_f32<TO>(xv[j][q] / rms * wv[j][q]);
            o[i] = t;
        }
    }
}

extern "C" int li_rmsnorm(const float* x, const float* w, const int* rows, void* out, int out_dt,
                          int n_rows, int d, float eps, float* row_scale, hipStream_t stream) {
    if (n_rows <= 0) return LI_OK;
    if (d <= 0) return LI_BAD_ARG;
    if (out_dt != DT_F32 && out_dt != DT_F16 && out_dt != DT_BF16) return LI_BAD_ARG;
    dim3 grid(n_rows);
    const bool vec = d % 4 == 0 && d <= 8192 && !(((uintptr_t)x | (uintptr_t)w | (uintptr_t)out) & 15);
    if (vec) {
        const int n4 = d / 4;
        const int threads = n4 <= 64 ? 64 : (n4 <= 256 ? 128 : (n4 <= 1024 ? 256 : 512));
        const bool two = n4 <= 2 * threads;
#define GO(TO)                                                                                             \
    do {                                                                                                   \
        if (two) rmsnorm_vec_kernel<TO, 2><<<grid, threads, 0, stream>>>(x, w, rows, (TO*)out, d, eps, row_scale); \
        else rmsnorm_vec_kernel<TO, 4><<<grid, threads, 0, stream>>>(x, w, rows, (TO*)out, d, eps, row_scale);     \
    } while (0)
        if (out_dt == DT_F32) GO(float); else if (out_dt == DT_F16) GO(f16); else GO(bf16);
#undef GO
    } else {
        dim3 block(d >= 2048 ? 512 : (d >= 512 ? 256 : 64));
        if (out_dt == DT_F32) rmsnorm_kernel<float><<<grid, block, 0, stream>>>(x, w, rows, (float*)out, d, eps, row_scale);
        else if (out_dt == DT_F16) rmsnorm_kernel<f16><<<grid, block, 0, stream>>>(x, w, rows, (f16*)out, d, eps, row_scale);
        else rmsnorm_kernel<bf16><<<grid, block, 0, stream>>>(x, w, rows, (bf16*)out, d, eps, row_scale);
    }
    LI_CHECK_LAUNCH();
    return LI_OK;
}

// ---------------------------------------------------------------------------
// Rotation of q and k by position, and the write of k and v into the cache.
//   qkv   [T, row_stride] float32: q heads, then k heads, then v heads of one token
//   q_out [T, H, hd]
//   pages: k_pages/v_pages of this layer, page = page_table[slot, pos / PAGE]
// Rotation (include/kernels_cpu.hpp:82-100): pair (a, b) <- (a cos - b sin, a sin + b cos),
// angle = pos * inv_freq[j]; adjacent pairing rotates (2j, 2j+1), half pairing
// (j, j + rotary_dim/2).  Dimensions at and beyond rotary_dim pass unchanged.
// Keys are stored after the rotation (src/model/block.cpp:141-148).
// ---------------------------------------------------------------------------
template <class T>
__global__ void rope_store_kernel(const float* __restrict__ qkv, int row_stride,
                                  const float* __restrict__ inv_freq, int rotary_dim, int half_pairing,
                                  const int* __restrict__ pos, const int* __restrict__ tok_slot,
                                  const int* __restrict__ page_table, int max_pages, int64_t page_stride,
                                  T* __restrict__ q_out, T* __restrict__ k_pages, T* __restrict__ v_pages,
                                  int H, int K, int hd, int kv_round) {
    const int t = blockIdx.x;
    const int p = pos[t];
    const int half = hd >> 1;
    const int n_pairs = (H + 2 * K) * half;
    const float* row = qkv + (int64_t)t * row_stride;
    int64_t page = 0;
    if (K > 0) page = page_table[(int64_t)tok_slot[t] * max_pages + p / PAGE];
    const int tp = p % PAGE;
    for (int i = blockIdx.y * blockDim.x + threadIdx.x; i < n_pairs; i += blockDim.x * gridDim.y) {
        const int head = i / half, j = i - head * half;
        int d0, d1;
        bool rotate = false;
        if (2 * j < rotary_dim) {
            rotate = true;
            if (half_pairing) { d0 = j; d1 = j + (rotary_dim >> 1); }
            else { d0 = 2 * j; d1 = 2 * j + 1; }
        } else { d0 = 2 * j; d1 = 2 * j + 1; }
        float a = row[head * hd + d0], b = row[head * hd + d1];
        if (rotate && head < H + K) {
            float s, c;
            sincosf((float)p * inv_freq[j], &s, &c);
            const float ra = a * c - b * s, rb = a * s + b * c;
            a = ra; b = rb;
        }
        if (head >= H && kv_round != DT_F32) {
            // what goes into the cache takes a 16-bit type's values on its way (block.cpp:145-148)
            if (kv_round == DT_F16) { a = (float)(f16)a; b = (float)(f16)b; }
            else { a = (float)(bf16)a; b = (float)(bf16)b; }
        }
        if (head < H) {
            T* q = q_out + ((int64_t)t * H + head) * hd;
            q[d0] = from_f32<T>(a); q[d1] = from_f32<T>(b);
        } else if (head < H + K) {
            T* kp = k_pages + page * page_stride + (int64_t)(head - H) * k_head_elems(hd);
            kp[k_offset(tp, d0, hd)] = from_f32<T>(a); kp[k_offset(tp, d1, hd)] = from_f32<T>(b);
        } else {
            T* vp = v_pages + page * page_stride + (int64_t)(head - H - K) * v_head_elems(hd);
            vp[v_offset(tp, d0, hd)] = from_f32<T>(a); vp[v_offset(tp, d1, hd)] = from_f32<T>(b);
        }
    }
}

extern "C" int li_rope_store(const float* qkv, int row_stride, const float* inv_freq, int rotary_dim,
                             int half_pairing, const int* pos, const int* tok_slot, const int* page_table,
                             int max_pages, int64_t page_stride, void* q_out, void* k_pages, void* v_pages, int dt,
                             int n_tokens, int H, int K, int hd, int kv_round, hipStream_t stream) {
    if (n_tokens <= 0) return LI_OK;
    if (kv_round < DT_F32 || kv_round > DT_BF16) return LI_BAD_ARG;
    if (hd <= 0 || (hd & 1) || H <= 0 || K < 0 || rotary_dim < 0 || rotary_dim > hd || (rotary_dim & 1) ||
        row_stride < (H + 2 * K) * hd)
        return LI_BAD_ARG;
    if (K > 0 && (hd % 16 != 0)) return LI_UNSUPPORTED;
    // few tokens: a token's pairs over several workgroups, since a thread's pairs come one after the other (a sine and cosine each;
    // 3 tokens of 32 + 16 heads of 64: 6.8 -> 5.0 us)
    const int64_t n_pairs = (int64_t)(H + 2 * K) * (hd / 2);
    dim3 grid(n_tokens, n_tokens < 256 ? (unsigned)((n_pairs + 255) / 256 < 64 ? (n_pairs + 255) / 256 : 64) : 1u), block(256);
#define LAUNCH(T)                                                                                        \
    rope_store_kernel<T><<<grid, block, 0, stream>>>(qkv, row_stride, inv_freq, rotary_dim, half_pairing, \
                                                     pos, tok_slot, page_table, max_pages, page_stride, (T*)q_out, \
                                                     (T*)k_pages, (T*)v_pages, H, K, hd, kv_round)
    if (dt == DT_F32) LAUNCH(float);
    else if (dt == DT_F16) LAUNCH(f16);
    else if (dt == DT_BF16) LAUNCH(bf16);
    else return LI_BAD_ARG;
#undef LAUNCH
    LI_CHECK_LAUNCH();
    return LI_OK;
}

// cos and sin of pos[t] * inv_freq[j] for the tokens of a step: [T, n_freq, 2] float32.  The angles
// are the same in every layer, so a step computes them once.
__global__ void rope_table_kernel(const float* __restrict__ inv_freq, const int* __restrict__ pos,
                                  float* __restrict__ out, int n_tokens, int n_freq) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n_tokens * n_freq) return;
    const int t = i / n_freq, j = i - t * n_freq;
    float s, c;
    sincosf((float)pos[t] * inv_freq[j], &s, &c);
    out[2 * i] = c;
    out[2 * i + 1] = s;
}

extern "C" int li_rope_table(const float* inv_freq, const int* pos, float* out, int n_tokens, int n_freq,
                             hipStream_t stream) {
    if (n_tokens <= 0 || n_freq <= 0) return LI_OK;
    const int n = n_tokens * n_freq;
    rope_table_kernel<<<(n + 255) / 256, 256, 0, stream>>>(inv_freq, pos, out, n_tokens, n_freq);
    LI_CHECK_LAUNCH();
    return LI_OK;
}

// ---------------------------------------------------------------------------
// Bookkeeping of one decode step, on the device so that a captured step can be
// replayed: each sequence's new token gets the position lens[slot], the
// sequence's context grows by one.  A row on `scratch_slot` is an idle row of a
// step that runs more rows than there are live sequences: position 0, a context
// of one token, and no length is changed.  With `cos_sin` (may be null) the same
// kernel fills the table of rotation angles of the step, [n, n_freq, 2] = cos and
// sin of pos * inv_freq as rope_table_kernel does, so that a step needs no
// second small kernel before its first layer.
// ---------------------------------------------------------------------------
// What the step before chose, for the host (ring null: not wanted): row i's token and the number of this step in one word of page-locked memory,
// written past the caches, so that neither order nor a flag is needed; the host polls for the number.  `steps`: one counter a row, all of them `rows`
// advanced by every step.
struct TokensOut {
    const int* tokens;
    unsigned* steps;
    unsigned long long* ring;                        // [TOKEN_RING][rows]
    int rows;
};
enum { TOKEN_RING = 4 };

__global__ void decode_prepare_kernel(const int* __restrict__ seq_slot, int* __restrict__ lens,
                                      int* __restrict__ pos, int* __restrict__ ctx, int n, int scratch_slot,
                                      const float* __restrict__ inv_freq, float* __restrict__ cos_sin, int n_freq, TokensOut out) {
    // one workgroup a row: thread 0 does the bookkeeping, all threads the row's angles
    const int i = blockIdx.x;
    const int s = seq_slot[i];
    if (out.ring) {
        if (threadIdx.x == 0) {
            const unsigned step = out.steps[i] + 1;
            out.steps[i] = step;
            __hip_atomic_store(out.ring + (int64_t)(step % TOKEN_RING) * out.rows + i, (unsigned long long)step << 32 | (unsigned)out.tokens[i],
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
        if (i == 0)
            for (int j = n + threadIdx.x; j < out.rows; j += blockDim.x) out.steps[j] += 1;
    }
    const int l = s == scratch_slot ? 0 : lens[s];
    __syncthreads();                                  // every thread has read the length before it changes
    if (threadIdx.x == 0) {
        pos[i] = l;
        ctx[i] = l + 1;
        if (s != scratch_slot) lens[s] = l + 1;
    }
    if (cos_sin)
        for (int j = threadIdx.x; j < n_freq; j += blockDim.x) {
            float sn, cs;
            sincosf((float)l * inv_freq[j], &sn, &cs);
            cos_sin[2 * ((int64_t)i * n_freq + j)] = cs;
            cos_sin[2 * ((int64_t)i * n_freq + j) + 1] = sn;
        }
}

extern "C" int li_decode_prepare(const int* seq_slot, int* lens, int* pos, int* ctx, int n, int scratch_slot,
                                 const float* inv_freq, float* cos_sin, int n_freq, const int* tokens, unsigned* steps,
                                 unsigned long long* ring, int rows, hipStream_t stream) {
    if (n <= 0) return LI_OK;
    if (cos_sin && (!inv_freq || n_freq <= 0)) return LI_BAD_ARG;
    if (ring && (!tokens || !steps || rows < n || ((uintptr_t)ring & 7))) return LI_BAD_ARG;
    // the device's address of the ring, which has to be page-locked memory
    if (ring && hipHostGetDevicePointer((void**)&ring, ring, 0) != hipSuccess) return LI_BAD_ARG;
    decode_prepare_kernel<<<n, 64, 0, stream>>>(seq_slot, lens, pos, ctx, n, scratch_slot, inv_freq, cos_sin, n_freq,
                                                TokensOut{tokens, steps, ring, rows});
    LI_CHECK_LAUNCH();
    return LI_OK;
}

// Waits on the host until the first n rows of `ring` bear step number `step`, at most `micros`; their tokens go to `out`.  1: not yet.
extern "C" int li_wait_tokens(const unsigned long long* ring, int rows, int n, unsigned step, int* out, int64_t micros) {
    const unsigned long long* p = ring + (int64_t)(step % TOKEN_RING) * rows;
    const auto until = std::chrono::steady_clock::now() + std::chrono::microseconds(micros);
    for (int i = 0, spins = 0; i < n;) {
        const unsigned long long v = __atomic_load_n(p + i, __ATOMIC_ACQUIRE);
        if ((unsigned)(v >> 32) == step) {
            out[i++] = (int)(unsigned)v;
            continue;
        }
        if (++spins % 64 == 0 && std::chrono::steady_clock::now() >= until) return 1;
#if !defined(__HIP_DEVICE_COMPILE__)
        __builtin_ia32_pause();
#endif
    }
    return LI_OK;
}

// ---------------------------------------------------------------------------
// Bookkeeping of the cache between steps: single words of its tables (page tables, lengths, sampling state) and pages
// to be cleared, both listed in the kernel's own arguments, so that nothing is uploaded and the host does not wait.
// Bound by the launch.  A page-table update by index and row tensors was three uploads from pageable memory and two kernels, each
// upload waiting for all work before it: with 48 live sequences every other decode step paid 0.1 ms for that.
// ---------------------------------------------------------------------------
enum { EDIT_WORDS = 896 };                       // 3.5 KiB of arguments; a launch takes 4

struct CacheEdits {
    int n0, n1, n_pages;
    int data[EDIT_WORDS];                        // (word, value) pairs of dst0, those of dst1, pages
};

enum { CLEAR_BLOCK = 256 * 16 * 8 };             // bytes that a workgroup clears: eight stores a thread

__global__ __launch_bounds__(256) void cache_edit_kernel(int* __restrict__ dst0, int* __restrict__ dst1,
                                                         uint4* __restrict__ pages, int64_t page_bytes, int per_page,
                                                         const CacheEdits e) {
    if (blockIdx.x == 0) {
        for (int i = threadIdx.x; i < e.n0; i += 256) dst0[e.data[2 * i]] = e.data[2 * i + 1];
        const int* d = e.data + 2 * e.n0;
        for (int i = threadIdx.x; i < e.n1; i += 256) dst1[d[2 * i]] = d[2 * i + 1];
        return;
    }
    const int b = blockIdx.x - 1;
    uint4* p = pages + (int64_t)e.data[2 * (e.n0 + e.n1) + b / per_page] * (page_bytes / 16);
    const int64_t from = (int64_t)(b % per_page) * (CLEAR_BLOCK / 16);
    const int64_t to = min(from + CLEAR_BLOCK / 16, page_bytes / 16);
    for (int64_t i = from + threadIdx.x; i < to; i += 256) p[i] = make_uint4(0, 0, 0, 0);
}

// words: n0 pairs for dst0, n1 pairs for dst1, n_pages pages of page_bytes bytes each behind `pages`.
extern "C" int li_cache_edit(int* dst0, int n0, int* dst1, int n1, void* pages, int64_t page_bytes, int n_pages,
                             const int* words, hipStream_t stream) {
    if (n0 < 0 || n1 < 0 || n_pages < 0 || 2 * ((int64_t)n0 + n1) + n_pages > EDIT_WORDS) return LI_BAD_ARG;
    if (n0 + n1 + n_pages == 0) return LI_OK;
    if ((n0 && !dst0) || (n1 && !dst1) || (n_pages && (!pages || page_bytes <= 0 || page_bytes % 16 || (uintptr_t)pages % 16))) return LI_BAD_ARG;
    CacheEdits e;
    e.n0 = n0, e.n1 = n1, e.n_pages = n_pages;
    for (int i = 0; i < 2 * (n0 + n1) + n_pages; i++) e.data[i] = words[i];
    const int64_t per_page = n_pages ? (page_bytes + CLEAR_BLOCK - 1) / CLEAR_BLOCK : 1;
    if (1 + n_pages * per_page > 0x7fffffff) return LI_UNSUPPORTED;
    cache_edit_kernel<<<(unsigned)(1 + n_pages * per_page), 256, 0, stream>>>(dst0, dst1, (uint4*)pages, page_bytes, (int)per_page, e);
    LI_CHECK_LAUNCH();
    return LI_OK;
}

// What a sequence keeps outside the pages starts at zero: one row of every table (group) of fixed-size state, for each of
// the group's entries.  One launch for all groups; an index fill for each was an upload and a kernel a group, 0.2 ms of host
// time a sequence in a model of four groups.
enum { CLEAR_GROUPS = 32 };

struct ClearGroup {
    char* row;                                   // the slot's row of the group's first entry
    int64_t entry_stride, row_bytes;
    int64_t entries;
};

struct ClearGroups {
    ClearGroup g[CLEAR_GROUPS];
};

template <class U> __device__ __forceinline__ void clear_units(char* p, int64_t bytes, U zero) {
    U* u = (U*)p;
    for (int64_t i = threadIdx.x; i < bytes / (int64_t)sizeof(U); i += 256) u[i] = zero;
}

__global__ __launch_bounds__(256) void clear_rows_kernel(const ClearGroups groups) {
    int g = 0, entry = blockIdx.y;
    while (entry >= groups.g[g].entries) entry -= (int)groups.g[g++].entries;
    const ClearGroup c = groups.g[g];
    const int64_t from = (int64_t)blockIdx.x * CLEAR_BLOCK;
    if (from >= c.row_bytes) return;
    char* p = c.row + entry * c.entry_stride + from;
    const int64_t n = min((int64_t)CLEAR_BLOCK, c.row_bytes - from);
    const uint64_t odd = (uint64_t)(uintptr_t)p | (uint64_t)n;
    if (odd % 16 == 0) clear_units<uint4>(p, n, make_uint4(0, 0, 0, 0));
    else if (odd % 4 == 0) clear_units<uint32_t>(p, n, 0u);
    else clear_units<uint8_t>(p, n, 0);
}

extern "C" int li_clear_rows(const ClearGroup* groups, int n, hipStream_t stream) {
    if (n < 0 || n > CLEAR_GROUPS) return LI_BAD_ARG;
    ClearGroups all = {};
    int64_t entries = 0, most = 0;
    for (int i = 0; i < n; i++) {
        if (!groups[i].row || groups[i].entries < 0 || groups[i].row_bytes < 0) return LI_BAD_ARG;
        all.g[i] = groups[i];
        entries += groups[i].entries;
        most = groups[i].row_bytes > most ? groups[i].row_bytes : most;
    }
    if (entries == 0 || most == 0) return LI_OK;
    if (entries > 65535 || most > (int64_t)CLEAR_BLOCK * 0x7fffffff) return LI_UNSUPPORTED;
    clear_rows_kernel<<<dim3((unsigned)((most + CLEAR_BLOCK - 1) / CLEAR_BLOCK), (unsigned)entries), 256, 0, stream>>>(all);
    LI_CHECK_LAUNCH();
    return LI_OK;
}

// out[i] = act(gate[i]) * up[i] for separate gate and up rows:  gu [T, 2F] float32 with
// gate_j at column 2j and up_j at column 2j+1  ->  h [T, F].  (src/model/block.cpp:203-214)
// act: gate_activation of common.h (silu, or the reference's gelu).
template <class T>
__global__ void swiglu_kernel(const float* __restrict__ gu, T* __restrict__ h, int64_t n, int gelu) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float g = gu[2 * i], u = gu[2 * i + 1];
    h[i] = from_f32<T>(gate_activation(g, gelu != 0) * u);
}

extern "C" int li_swiglu(const float* gu, void* h, int dt, int64_t n, int gelu, hipStream_t stream) {
    if (n <= 0) return LI_OK;
    dim3 grid((unsigned)((n + 255) / 256)), block(256);
    if (dt == DT_F32) swiglu_kernel<float><<<grid, block, 0, stream>>>(gu, (float*)h, n, gelu);
    else if (dt == DT_F16) swiglu_kernel<f16><<<grid, block, 0, stream>>>(gu, (f16*)h, n, gelu);
    else if (dt == DT_BF16) swiglu_kernel<bf16><<<grid, block, 0, stream>>>(gu, (bf16*)h, n, gelu);
    else return LI_BAD_ARG;
    LI_CHECK_LAUNCH();
    return LI_OK;
}
