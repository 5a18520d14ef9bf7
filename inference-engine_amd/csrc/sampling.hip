// Token sampling over the vocabulary (gfx950): Gumbel-max with Triton's Philox uniforms, greedy
// argmax at tau = 0.
//
// Semantics (qwen3-1.7b/kernels.py:1286-1370): token[b] = the first v maximizing
// logits[b, v] + tau * -log(-log(clamp(u[b, v], 1e-10, 1 - 1e-7))), u = tl.rand(seed, b * V + v):
// Philox4x32-10 on counter (b * V + v as int32, 0, 0, 0) and key (seed low word, seed high word),
// first output word x as int32, u = float(x < 0 ? -x - 1 : x) * 4.6566127342e-10. Then the
// device seed is incremented. At tau = 0 the noise term is 0 * finite, so no uniform is drawn.
//
// sample_partial_kernel, grid (cdiv(V, block), B), 256 threads: the best (value, index) of each
// block of a row's raw logits (sp_rounds), at tau != 0 with that entry's perturbed score.
// sample_gumbel_kernel (tau != 0), the same grid: the best score of each block. Small batches skip
// the first launch at tau != 0: each block finds its own best raw entry (sample_launch).
// sample_combine_kernel, grid B, one wave: the best over the row's blocks, and the seed increment
// (after every block has read the seed: the launches are stream-ordered).
//
// Greedy is bound by HBM and launch latency (B x V logits read once). With noise, drawing a uniform
// is what costs: Philox's 16 64-bit products take 16 cycles per wave each, 10 us for 32 x 151,936
// entries on the whole chip. So entries that cannot win draw none: the noise is at most SP_GMAX, and
// the best score of the row's block maxima (or of the block's own) bounds the winner's from below, so
// an entry whose logit plus tau SP_GMAX stays under it is out. Float addition and multiplication are monotonic:
// no winner is lost, whatever the logits. What is left is listed and drawn densely by the
// workgroup, the hardware's fast logarithm first and the exact score only where that one plus its
// error margin reaches the bound. 32 x 151,936 bf16, against every entry drawn with exact
// logarithms: next-token logits (a few candidates above a bulk) at tau 0.7 21.6 -> 12.7 us, logits
// without any candidates (all drawn) 21.7 -> 18.4. Merging the blocks by arrival counts in the
// second launch instead of the third one cost 1-3 us.
#include "ie_common.h"

namespace ie {

constexpr int SP_THREADS = 256;
constexpr int SP_VEC = 8;                                // entries per 16-byte bf16 load
constexpr int SP_PASS = SP_THREADS * SP_VEC;             // 2048 entries per load of a workgroup
constexpr int SP_ROUNDS = 2;                             // loads per thread, or 1
constexpr int64_t SP_MAX_VOCAB = 65535LL * 8192;         // at most (indices fit int32)
// No uniform's noise exceeds 15.95 (u <= 0.99999988) or falls below -3.14 (u >= 1e-10).
constexpr float SP_GMAX = 16.0f, SP_GMIN = -4.0f;
// Loads per thread for a batch of rows: blocks of 4096 entries while they give each CU four
// workgroups, else of 2048, for the latency of small batches (of 151,936 entries, us at tau 0 / 0.7:
// 32 rows 6.45 / 12.7 in blocks of 4096, 6.9 / 14.0 of 2048, 6.7 / 14.4 of 8192; 128 rows 12.2 /
// 27.3, 13.3 / 32.8 and 12.7 / 26.9; one row 4.8 / 8.9 of 2048 against 6.6 / 12.4 of 8192).
int sp_rounds(int64_t batch, int64_t vocab) {
    const int64_t blk = (int64_t)SP_PASS * SP_ROUNDS;
    return batch * ((vocab + blk - 1) / blk) >= 4 * device_cu_count() ? SP_ROUNDS : 1;
}
int64_t sp_blocks(int64_t batch, int64_t vocab) {
    const int64_t blk = (int64_t)SP_PASS * sp_rounds(batch, vocab);
    return (vocab + blk - 1) / blk;
}

struct Best {
    float v;
    int i;
};
// (a, b) ordered as the reference's argmax: larger value, then smaller index
__device__ __forceinline__ bool better(float av, int ai, float bv, int bi) {
    return av > bv || (av == bv && ai < bi);
}
__device__ __forceinline__ void take(Best& best, float v, int i) {
    if (better(v, i, best.v, best.i)) {
        best.v = v;
        best.i = i;
    }
}
__device__ __forceinline__ Best wave_best(Best b) {
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) {
        const float ov = __shfl_xor(b.v, m, IE_WAVE);
        const int oi = __shfl_xor(b.i, m, IE_WAVE);
        take(b, ov, oi);
    }
    return b;
}

// a ^ b ^ c in one instruction.
__device__ __forceinline__ uint32_t xor3(uint32_t a, uint32_t b, uint32_t c) {
    uint32_t d;
    asm("v_bitop3_b32 %0, %1, %2, %3 bitop3:0x96" : "=v"(d) : "v"(a), "v"(b), "s"(c));
    return d;
}
// Philox4x32-10, first output word, for counter (c0, 0, 0, 0) and key (k0, k1) (wave-uniform). One
// 64-bit product gives both halves (v_mad_u64_u32); the first two rounds' zero words fold away.
__device__ __forceinline__ uint32_t philox_first(uint32_t c0, uint32_t k0, uint32_t k1) {
    // rounds 1 and 2: (c0, 0, 0, 0) -> (k0, 0, h ^ k1, l) -> ...
    const uint64_t p1 = (uint64_t)0xD2511F53u * c0;
    uint32_t c2 = (uint32_t)(p1 >> 32) ^ k1, c3 = (uint32_t)p1, c1 = 0;
    c0 = k0;
#pragma unroll
    for (int r = 1; r < 10; ++r) {
        k0 += 0x9E3779B9u;
        k1 += 0xBB67AE85u;
        const uint64_t a = (uint64_t)0xD2511F53u * c0, b = (uint64_t)0xCD9E8D57u * c2;
        const uint32_t n0 = r == 1 ? (uint32_t)(b >> 32) ^ k0 : xor3((uint32_t)(b >> 32), c1, k0);
        c2 = r == 1 ? c3 ^ ((uint32_t)(a >> 32) ^ k1) : xor3((uint32_t)(a >> 32), c3, k1);
        c1 = (uint32_t)b;
        c3 = (uint32_t)a;
        c0 = n0;
    }
    return c0;
}

// The uniform of entry `offset` (b * V + v, int32 arithmetic as the reference).
__device__ __forceinline__ float uniform_of(uint32_t offset, uint32_t k0, uint32_t k1) {
    const int32_t w = (int32_t)philox_first(offset, k0, k1);
    const float u0 = (float)(w ^ (w >> 31)) * 4.6566127342e-10f;  // x < 0 ? -x - 1 : x
    return fminf(fmaxf(u0, 1e-10f), 0.99999988f);                 // clamp(u, 1e-10, 1 - 1e-7)
}
// The Gumbel-perturbed logit.
__device__ __forceinline__ float gumbel(float x, float tau, float u) {
#pragma clang fp contract(off)
    return x + tau * -logf(-logf(u));
}
// At least the noise of u: the hardware logarithm (1 ulp, near u = 1 an absolute error of some
// 2^-23 in log2 u, 0.08 % of it at 0.9999) with a margin of 0.05 in the outer one (5 % of t).
__device__ __forceinline__ float noise_bound(float u) {
    const float t = -0.69314718f * __builtin_amdgcn_logf(u);
    return u > 0.9999f ? SP_GMAX : 0.05f - 0.69314718f * __builtin_amdgcn_logf(t);
}

// Eight entries at any element alignment (16-byte loads all the same: the device takes them
// unaligned; rows of an odd vocabulary start anywhere).
template <typename T>
__device__ __forceinline__ void load8(const T* row, int64_t v, float (&x)[SP_VEC]);
template <>
__device__ __forceinline__ void load8<uint16_t>(const uint16_t* row, int64_t v, float (&x)[SP_VEC]) {
    uint4 w;
    __builtin_memcpy(&w, row + v, sizeof(w));
    const uint32_t ws[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        x[2 * j] = bf16lo(ws[j]);
        x[2 * j + 1] = bf16hi(ws[j]);
    }
}
template <>
__device__ __forceinline__ void load8<float>(const float* row, int64_t v, float (&x)[SP_VEC]) {
    float4 a, b;
    __builtin_memcpy(&a, row + v, sizeof(a));
    __builtin_memcpy(&b, row + v + 4, sizeof(b));
    x[0] = a.x; x[1] = a.y; x[2] = a.z; x[3] = a.w;
    x[4] = b.x; x[5] = b.y; x[6] = b.z; x[7] = b.w;
}

// The workgroup's entries: thread tid holds 8 consecutive ones per round, [base + (r * 256 + tid) * 8,
// +8); -inf past the row's end.
template <typename T, int ROUNDS>
__device__ __forceinline__ void load_entries(const T* row, int64_t base, int64_t V,
                                             float (&x)[ROUNDS][SP_VEC]) {
#pragma unroll
    for (int r = 0; r < ROUNDS; ++r) {
        const int64_t v0 = base + (int64_t)(r * SP_THREADS + threadIdx.x) * SP_VEC;
        if (v0 + SP_VEC <= V) {
            load8<T>(row, v0, x[r]);
        } else {
#pragma unroll
            for (int j = 0; j < SP_VEC; ++j) {
                float y = -INFINITY;
                if (v0 + j < V) {
                    if constexpr (sizeof(T) == 2) y = bf16_to_f32(row[v0 + j]);
                    else y = (float)row[v0 + j];
                }
                x[r][j] = y;
            }
        }
    }
}
// The best over the workgroup, in thread 0.
__device__ __forceinline__ Best block_best(Best best) {
    best = wave_best(best);
    __shared__ float s_v[SP_THREADS / IE_WAVE];
    __shared__ int s_i[SP_THREADS / IE_WAVE];
    const int tid = threadIdx.x;
    if ((tid & 63) == 0) {
        s_v[tid >> 6] = best.v;
        s_i[tid >> 6] = best.i;
    }
    __syncthreads();
    if (tid == 0) {
#pragma unroll
        for (int w = 1; w < SP_THREADS / IE_WAVE; ++w) take(best, s_v[w], s_i[w]);
    }
    return best;
}

// The thread's best raw entry.
template <int ROUNDS>
__device__ __forceinline__ Best raw_best(const float (&x)[ROUNDS][SP_VEC], int64_t base,
                                         int64_t V) {
    Best best = {-INFINITY, 0x7fffffff};
#pragma unroll
    for (int r = 0; r < ROUNDS; ++r)
#pragma unroll
        for (int j = 0; j < SP_VEC; ++j) {
            const int64_t v = base + (int64_t)(r * SP_THREADS + threadIdx.x) * SP_VEC + j;
            if (v < V) take(best, x[r][j], (int)v);
        }
    return best;
}

// grid (blocks, B), block 256: the best raw (value, index) of block bx of row by, to partial slot
// by * gridDim.x + bx; at tau != 0 the value is that entry's perturbed score, the bound the next
// launch starts from.
template <typename T, int ROUNDS>
__global__ __launch_bounds__(SP_THREADS) void sample_partial_kernel(
    const T* __restrict__ logits, int64_t ls, int64_t V, float tau,
    const int64_t* __restrict__ seed, float* __restrict__ pv, int* __restrict__ pi) {
    const int b = blockIdx.y;
    const int64_t base = (int64_t)blockIdx.x * (SP_PASS * ROUNDS);
    const int tid = threadIdx.x;
    const uint64_t sd = (uint64_t)seed[0];
    float x[ROUNDS][SP_VEC];
    load_entries<T, ROUNDS>(logits + b * ls, base, V, x);
    Best best = block_best(raw_best<ROUNDS>(x, base, V));
    if (tid == 0) {
        if (tau != 0.f && best.i != 0x7fffffff)
            best.v = gumbel(best.v, tau,
                            uniform_of((uint32_t)b * (uint32_t)V + (uint32_t)best.i, (uint32_t)sd,
                                       (uint32_t)(sd >> 32)));
        const int64_t slot = (int64_t)b * gridDim.x + blockIdx.x;
        pv[slot] = best.v;
        pi[slot] = best.i;
    }
}

// grid (blocks, B), block 256, at tau != 0: see the top. pv: sample_partial_kernel's scores, or null:
// each block then bounds its entries by the score of its own largest one; bv, bi: the best (score,
// index) per block.
template <typename T, int ROUNDS>
__global__ __launch_bounds__(SP_THREADS) void sample_gumbel_kernel(
    const T* __restrict__ logits, int64_t ls, int64_t V, float tau,
    const int64_t* __restrict__ seed, const float* __restrict__ pv,
    float* __restrict__ bv, int* __restrict__ bi) {
    const int b = blockIdx.y, nblk = gridDim.x;
    const T* row = logits + b * ls;
    const int64_t base = (int64_t)blockIdx.x * (SP_PASS * ROUNDS);
    const int tid = threadIdx.x, lane = tid & 63;
    const uint64_t sd = (uint64_t)seed[0];
    const uint32_t k0 = (uint32_t)sd, k1 = (uint32_t)(sd >> 32);
    const uint32_t row_off = (uint32_t)b * (uint32_t)V;
    float lb = -INFINITY;  // a score the row's best is at least
    if (pv)
        for (int j = lane; j < nblk; j += IE_WAVE) lb = fmaxf(lb, pv[(int64_t)b * nblk + j]);
    float x[ROUNDS][SP_VEC];
    load_entries<T, ROUNDS>(row, base, V, x);
    if (pv) {
        lb = wave_max(lb);
    } else {  // small batches: the block's own bound
        __shared__ float s_lb;
        const Best top = block_best(raw_best<ROUNDS>(x, base, V));
        if (tid == 0)
            s_lb = top.i == 0x7fffffff
                       ? -INFINITY
                       : gumbel(top.v, tau, uniform_of(row_off + (uint32_t)top.i, k0, k1));
        __syncthreads();
        lb = s_lb;
    }
    const float reach = fmaxf(tau * SP_GMAX, tau * SP_GMIN);
    uint32_t mask = 0;  // entries that may still win (those past the row's end may not)
#pragma unroll
    for (int r = 0; r < ROUNDS; ++r)
#pragma unroll
        for (int j = 0; j < SP_VEC; ++j) {
            const int64_t v = base + (int64_t)(r * SP_THREADS + tid) * SP_VEC + j;
            if (v < V && !(x[r][j] + reach < lb)) mask |= 1u << (r * SP_VEC + j);
        }
    // the workgroup's candidates, numbered thread by thread
    __shared__ int s_n[SP_THREADS / IE_WAVE];
    const int mine = __popc(mask), incl = wave_incl_scan_i(mine);
    if (lane == IE_WAVE - 1) s_n[tid >> 6] = incl;
    __syncthreads();
    int n = 0, at = incl - mine;
#pragma unroll
    for (int w = 0; w < SP_THREADS / IE_WAVE; ++w) {
        if (w < (tid >> 6)) at += s_n[w];
        n += s_n[w];
    }
    Best best = {-INFINITY, 0x7fffffff};
    constexpr int LIST = SP_PASS * ROUNDS * 3 / 4;
    __shared__ uint16_t s_list[LIST];
    if (n <= LIST) {  // uniform
        while (mask) {
            const int e = __ffs(mask) - 1;
            mask &= mask - 1;
            s_list[at++] = (uint16_t)(((e / SP_VEC) * SP_THREADS + tid) * SP_VEC + e % SP_VEC);
        }
        __syncthreads();
        for (int c = tid; c < n; c += SP_THREADS) {
            const int64_t v = base + s_list[c];
            float y;
            if constexpr (sizeof(T) == 2) y = bf16_to_f32(row[v]);
            else y = (float)row[v];
            const float u = uniform_of(row_off + (uint32_t)v, k0, k1);
            const float top = tau < 0.f ? INFINITY : y + tau * noise_bound(u);
            if (!(top < lb)) take(best, gumbel(y, tau, u), (int)v);
        }
    } else {
#pragma unroll
        for (int r = 0; r < ROUNDS; ++r)
#pragma unroll
            for (int j = 0; j < SP_VEC; ++j) {
                const int64_t v = base + (int64_t)(r * SP_THREADS + tid) * SP_VEC + j;
                const float u = uniform_of(row_off + (uint32_t)v, k0, k1);
                // tau < 0 (the noise's bound is from above only) takes the exact score
                const float top = tau < 0.f ? INFINITY : x[r][j] + tau * noise_bound(u);
                if (((mask >> (r * SP_VEC + j)) & 1) && !(top < lb))
                    take(best, gumbel(x[r][j], tau, u), (int)v);
            }
    }
    best = block_best(best);
    if (tid == 0) {
        const int64_t slot = (int64_t)b * nblk + blockIdx.x;
        bv[slot] = best.v;
        bi[slot] = best.i;
    }
}

// grid max(B, 1), block 64: token of row b = the best of its nblk partials; workgroup 0 also
// advances the seed.
__global__ __launch_bounds__(64) void sample_combine_kernel(const float* __restrict__ pv,
                                                           const int* __restrict__ pi, int nblk,
                                                           int B, int64_t* __restrict__ out,
                                                           int64_t os, int64_t* __restrict__ seed) {
    const int b = blockIdx.x, lane = threadIdx.x;
    if (b < B) {
        Best best = {-INFINITY, 0x7fffffff};
        const int64_t row = (int64_t)b * nblk;
        for (int j = lane; j < nblk; j += IE_WAVE) take(best, pv[row + j], pi[row + j]);
        best = wave_best(best);
        if (lane == 0) out[b * os] = best.i;
    }
    if (b == 0 && lane == 0) seed[0] += 1;
}

}  // namespace ie

using namespace ie;

// Per block of a row: the first launch's (value, index) and, at tau != 0, the second's (whose place
// does not depend on whether the first one ran). The size counts the smaller blocks whatever the
// batch: it then never falls as the batch grows, and a workspace made for the largest batch serves
// every smaller one (26 rows of 151,936 entries have 1,950 of the smaller blocks, 32 rows 1,216 of
// the larger).
extern "C" size_t ie_sample_workspace_size(int32_t batch, int64_t vocab) {
    if (batch <= 0 || vocab <= 0) return 0;
    return (size_t)batch * (size_t)((vocab + SP_PASS - 1) / SP_PASS) * 2 *
           (sizeof(float) + sizeof(int));
}

namespace {
template <typename T, int ROUNDS>
void sample_launch(const T* logits, int64_t ls, int32_t batch, int64_t vocab, float tau,
                   int64_t* seed, int64_t* out, int64_t os, void* workspace,
                   int64_t nblk, hipStream_t stream) {
    const size_t n = (size_t)batch * (size_t)nblk;
    float* pv = reinterpret_cast<float*>(workspace);
    int* pi = reinterpret_cast<int*>(pv + n);
    const dim3 grid((unsigned)nblk, (unsigned)batch);
    // A row's bound is worth its launch from about five 2,048-entry workgroups per CU (151,936
    // entries at tau 0.7, us in a graph / called back to back: 1 row 7.5 / 10.9 without it against
    // 8.8 / 14.0, 16 rows 11.5 / 11.6 against 10.9 / 14.0, 24 rows 14.0 / 14.4 against 12.6 / 14.0).
    const bool own = tau != 0.f && ROUNDS == 1 && batch * nblk <= 5 * device_cu_count();
    if (!own)
        hipLaunchKernelGGL((sample_partial_kernel<T, ROUNDS>), grid, dim3(SP_THREADS), 0, stream,
                           logits, ls, vocab, tau, (const int64_t*)seed, pv, pi);
    if (tau != 0.f) {
        float* bv = reinterpret_cast<float*>(pi + n);
        int* bi = reinterpret_cast<int*>(bv + n);
        hipLaunchKernelGGL((sample_gumbel_kernel<T, ROUNDS>), grid, dim3(SP_THREADS), 0, stream,
                           logits, ls, vocab, tau, (const int64_t*)seed,
                           own ? (const float*)nullptr : (const float*)pv, bv, bi);
        pv = bv;
        pi = bi;
    }
    hipLaunchKernelGGL(sample_combine_kernel, dim3((unsigned)batch), dim3(64), 0, stream, pv, pi,
                       (int)nblk, batch, out, os, seed);
}
template <typename T>
void sample_rounds(const void* logits, int64_t ls, int32_t batch, int64_t vocab, float tau,
                   int64_t* seed, int64_t* out, int64_t os, void* workspace, hipStream_t stream) {
    const int64_t nblk = sp_blocks(batch, vocab);
    if (sp_rounds(batch, vocab) == SP_ROUNDS)
        sample_launch<T, SP_ROUNDS>((const T*)logits, ls, batch, vocab, tau, seed, out, os,
                                    workspace, nblk, stream);
    else
        sample_launch<T, 1>((const T*)logits, ls, batch, vocab, tau, seed, out, os,
                            workspace, nblk, stream);
}
}  // namespace

extern "C" hipError_t ie_sample(const void* logits, int32_t logits_dtype, int64_t logits_stride_row,
                                int32_t batch, int64_t vocab, float tau, int64_t* seed,
                                int64_t* out, int64_t out_stride_row, void* workspace,
                                size_t workspace_bytes, hipStream_t stream) {
    IE_REQUIRE(batch >= 0 && vocab >= 0, "negative sizes");
    IE_REQUIRE(seed, "null pointer");
    IE_REQUIRE(logits_dtype == IE_DTYPE_BF16 || logits_dtype == IE_DTYPE_F32,
               "logits must be bf16 or fp32");
    IE_REQUIRE(vocab < (1LL << 31), "vocab must fit int32 indices");
    IE_REQUIRE(batch == 0 || vocab > 0, "empty vocabulary");
    if (batch == 0) {  // the seed advances all the same
        hipLaunchKernelGGL(sample_combine_kernel, dim3(1), dim3(64), 0, stream, nullptr, nullptr, 0,
                           0, out, out_stride_row, seed);
        return hipGetLastError();
    }
    IE_REQUIRE(logits && out && workspace, "null pointer");
    IE_REQUIRE(workspace_bytes >= ie_sample_workspace_size(batch, vocab), "workspace too small");
    IE_REQUIRE(vocab <= SP_MAX_VOCAB, "vocab too large");
    if (logits_dtype == IE_DTYPE_BF16)
        sample_rounds<uint16_t>(logits, logits_stride_row, batch, vocab, tau, seed, out,
                                out_stride_row, workspace, stream);
    else
        sample_rounds<float>(logits, logits_stride_row, batch, vocab, tau, seed, out,
                             out_stride_row, workspace, stream);
    return hipGetLastError();
}
