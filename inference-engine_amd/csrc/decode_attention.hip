// Split-K GQA decode attention over the int8 KV cache, for gfx950.
//
// Work split (same rule as qwen3-1.7b/kernels.py:20-70): every decoding sequence's tokens
// [0, cached_len + 1) are cut into pieces of `piece` tokens, piece = roundup(max(MIN_PIECE,
// cdiv(total_tokens, TARGET)), MIN_PIECE) with TARGET = CUs * WG_PER_CU / Hkv workgroups per KV
// head (when B <= TARGET the piece is grown until the pieces fit TARGET, see decode_piece). The
// pieces of all sequences form one work list; workgroup (w, kv head) takes entry w. The grid is
// (TARGET, Hkv) when B <= TARGET, else (TARGET + B, Hkv): it depends on shapes only, so the
// launch is graph-capturable, and each workgroup finds its (sequence, piece) on the device from
// cached_lens.
//
// One workgroup = W waves = one (sequence, piece, KV head) and all query heads of that KV head
// (GQA ratio 1 to 16), so every cached byte is read once whatever the ratio. What bounds it is the
// stream of int8 rows from HBM; the heads are the 16 columns of the MFMA tiles, so one head costs
// what 16 do.
//
// The stream goes global -> LDS without registers (buffer_load ... lds, 16 bytes per lane): each
// wave owns two stages of 32 tokens (K 4 KB, V 4 KB, scales 256 B), block j + 2 is requested as
// soon as block j's reads are done, and no barrier runs in the loop. Eight waves per CU keep up to
// 132 KB in flight. A lane may fetch its 16 bytes from any address but they land at consecutive
// LDS places, so K's bank spreading (16-byte chunk c of token t at place c ^ (t & 7)) is done in
// the global addresses; every group of 8 lanes still reads one whole 128-byte row.
//
// Per block and wave, v_mfma_f32_16x16x32_f16:
//   S (32 tokens x 16 heads) = K . Q^T   A = K rows (lane (r, g): token r, channels 16 g ... and
//                                        64 + 16 g ...), B = Q^T, 8 MFMAs
//   online softmax in base 2             a lane holds head r's scores of 8 tokens
//   O^T (128 channels x 16 heads) += V^T . P^T   A: lane (r, g) holds channels 8 r ... 8 r + 7 of
//                                        the 8 tokens whose P it holds (bytes of 8 rows paired by
//                                        permutes), B = P straight from the score registers, 8 MFMAs
// int8 -> fp16 by byte permute into the fp16 pattern 0x64xx (= 1024 + byte) after flipping the
// sign bit, i.e. 1152 + x, then -1152: exact. q is scaled by a power of two per head so that it
// is exact in fp16; P * v_scale goes to fp16 under a wave-wide power of two chosen from the V
// scales. The waves are merged at the end (log-sum-exp through LDS), then either the output is
// written (one piece) or fp32 partials (m, l, acc) go to the workspace and the sequence's last
// piece to finish merges them (the reference's combine kernel, kernels.py:216-264, folded into
// the same launch).
//
// Measured in graphs of 20 calls of the fused form, cache streamed from HBM, against a kernel
// that loaded rows into registers and took one query-head pair per workgroup with dot products:
// 16/8 heads B=1 ctx 128 11.8 -> 7.2 us, B=8 ctx 512-1024 14.6 -> 10.0, B=16 ctx 4096 29.7 -> 27.3,
// B=32 ctx 128-4096 33.4 -> 31.1 (4.7 TB/s), B=64 ctx 4096 86.7 -> 86.0 (6.45 TB/s: the stream),
// B=256 ctx 1024 91.2 -> 91.6; 32/8 B=32 ctx 128-4096 61.9 -> 32.7, 40/8 84.5 -> 32.8, 64/4
// 99.6 -> 22.7, 64/8 B=12 ctx 5001-8190 95.8 -> 34.7.
#include <mutex>

#include "ie_common.h"
#include "kv_math.h"

// Launch shape: 8 waves per CU (what the stages leave room for in LDS), as 4-wave workgroups, 2
// per CU, while the batch fits their per-head target, else 2-wave (4 per CU) or one-wave
// workgroups (8 per CU), whose targets are twice and four times as large (decode_waves): every
// sequence keeps a fitted piece in one resident round (B=256 ctx=1024, 16/8 heads: one-wave
// workgroups 91.6 us against 121.6 for 2-wave ones, whose 384 entries per head take two rounds).

namespace ie {

typedef _Float16 half2_t __attribute__((ext_vector_type(2)));

constexpr int DA_WAVES_PER_CU = 8;
constexpr int DA_MIN_PIECE = 128;
constexpr int DA_MAX_SPLITS = 1024;  // per-KV-head workgroup target, at most
constexpr int DA_D = 128;
constexpr int DA_MAX_WORK = 1 << 22;  // work entries per head, at most (the merge's 32-bit offsets)
constexpr uint32_t K64 = 0x64646464u;

// Workgroup target per unit (a KV head in a launch; see decode_units for work lists) of workgroups
// of `waves` waves: one resident round.
int decode_target(int units, int waves) {
    return std::min(DA_MAX_SPLITS, std::max(1, device_cu_count() * (DA_WAVES_PER_CU / waves) /
                                                   std::max(1, units)));
}
// Waves per workgroup for a batch: the largest workgroup whose target holds the batch, else
// the smallest.
int decode_waves(int batch, int units) {
    for (int w = 4; w > 1; w /= 2)
        if (batch <= decode_target(units, w)) return w;
    return 1;
}
// Units a work list is taken to be made for: KV heads x query-head pairs per KV head, the KV heads at
// ratios 1 and 2; with IE_PLAN_LAUNCH_UNITS, what the launch is cut for (list_units).
int decode_units(int hq, int hkv) { return hkv * ((hq / std::max(1, hkv) + 1) / 2); }


// Piece size for this step; wave-uniform, every lane returns it. The reference's rule
// (kernels.py:20-37) gives p0 = roundup(max(128, cdiv(total, target)), 128), but every sequence
// rounds its own split count up, so its pieces can number up to target + nd and spill past the
// one resident wave of workgroups that target sizes. When nd <= target the piece is instead the
// smallest multiple of 128, at least p0, whose pieces number at most target: a binary search,
// since the count falls as the piece grows and is nd at the longest sequence's length.
// n0: this lane's n_b of the first 64 sequences (0 past nd).
__device__ int decode_piece(const int32_t* __restrict__ cached_lens, int nd, int target, int n0) {
    const int lane = threadIdx.x & 63;
    auto n_of = [&](int b0) { return b0 == 0 ? n0 : (b0 + lane < nd ? cached_lens[b0 + lane] + 1 : 0); };
    int total = 0, longest = 0;
    for (int b0 = 0; b0 < nd; b0 += 64) {
        const int n = n_of(b0);
        total += wave_sum_i(n);
        longest = max(longest, (int)wave_max((float)n));
    }
    const int k0 = max(1, cdiv_i(cdiv_i(total, target), DA_MIN_PIECE));
    if (nd > target) return k0 * DA_MIN_PIECE;
    auto pieces = [&](int k) {
        const Divisor p = divisor(k * DA_MIN_PIECE);
        int c = 0;
        for (int b0 = 0; b0 < nd; b0 += 64) c += wave_sum_i(div_ceil(n_of(b0), p));
        return c;
    };
    int lo = k0, hi = max(k0, cdiv_i(longest, DA_MIN_PIECE));  // pieces(hi) <= nd <= target
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (pieces(mid) <= target) hi = mid;
        else lo = mid + 1;
    }
    return lo * DA_MIN_PIECE;
}

struct Work {
    int b, split, needed, piece;
};

// Entry `w` of the work list (kernels.py:40-70); needed == 0 for idle workgroups. `raw0`: this
// lane's cached_lens entry of the first 64 sequences, loaded by the caller bounded by the batch
// size instead of num_decoding, so that it shares one memory round trip with num_decoding.
__device__ Work decode_assign(const int32_t* __restrict__ cached_lens, int nd, int w, int target,
                              int raw0) {
    const int lane = threadIdx.x & 63;
    const int n0 = lane < nd ? raw0 + 1 : 0;
    Work r{0, 0, 0, decode_piece(cached_lens, nd, target, n0)};
    int before = 0;
    for (int b0 = 0; b0 < nd; b0 += 64) {
        const int b = b0 + lane;
        const int s = b < nd ? cdiv_i(b0 == 0 ? n0 : cached_lens[b] + 1, r.piece) : 0;
        const int incl = wave_incl_scan_i(s) + before;
        const int excl = incl - s;
        const unsigned long long hit = __ballot(s > 0 && excl <= w && w < incl);
        if (hit) {
            const int src = __ffsll((long long)hit) - 1;  // wave-uniform
            r.b = b0 + src;
            r.split = w - __builtin_amdgcn_readlane(excl, src);
            r.needed = __builtin_amdgcn_readlane(s, src);
            return r;
        }
        before = __builtin_amdgcn_readlane(incl, 63);
    }
    return r;
}

__device__ __forceinline__ int uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }
__device__ __forceinline__ half2_t as_h2(uint32_t u) { return __builtin_bit_cast(half2_t, u); }
__device__ __forceinline__ float exp2_safe(float x) { return __builtin_amdgcn_exp2f(x); }

struct DecodeArgs {
    const uint16_t* q;
    int64_t q_sb, q_sh;
    ie_kv_cache c;
    const int32_t* cached_lens;
    const int32_t* slot_ids;
    const int32_t* num_decoding;
    float scale_log2;  // softmax scale * log2(e)
    uint16_t* out;
    int64_t o_sb, o_sh;
    float* part_acc;     // [Hq, nwork, 128]: work entry w's partial output for query head h
    float* part_m;       // [Hq, nwork]
    float* part_l;       // [Hq, nwork]
    uint32_t* arrivals;  // [B, Hkv]: pieces of the sequence done; 0 between calls
    // The work list precomputed for this step (ie_decode_attention_plan: row w = (b, split,
    // needed, piece) of workgroup index w), or null: every workgroup derives its entry itself.
    const int32_t* plan;
    int target, nwork, hq, hkv;
    int ratio;    // query heads per KV head (GQA ratio, 1 ... 16)
    int batch;    // rows of q / cached_lens (num_decoding[0] <= batch)
    int out_vec;  // out rows take 8-byte stores
    // The fused form (ie_decode_attention_rope): q holds the QKV projection's raw rows, and the
    // launch does fused_rope_kv_decode's work itself: q normed, rotated and scaled by the
    // calibration as that kernel computes it, and the new token's K/V row quantized and written
    // to the cache by the piece that ends at it.
    const uint16_t* k_new;
    int64_t k_sb, k_sh;
    const uint16_t* v_new;
    int64_t v_sb, v_sh;
    const uint16_t* q_norm;
    const uint16_t* k_norm;
    const uint16_t* cos;
    const uint16_t* sin;
    int64_t cos_sb, sin_sb;
    float eps;
};

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

constexpr int DA_TOK = 32;                      // tokens per block
constexpr int DA_V = 4096, DA_SC = 8192;        // byte offsets in a stage: V rows, then scales
constexpr int DA_STAGE = DA_SC + 2 * 4 * DA_TOK;
constexpr int DA_QROW = DA_D + 8;               // LDS row of q (bf16), padded by 16 bytes
constexpr int DA_OROW = DA_D + 4;               // LDS row of a wave's output (fp32), padded
constexpr float DA_SLACK = 3.0f;  // the running max moves when a score exceeds it by 2^3
// V scales served by the wave's exponent ve: [2^(5 - ve), 2^(12 - ve)); with p <= 2^(DA_SLACK + ve)
// the fp16 products stay below 2^15
constexpr int DA_VE_TOP = 12, DA_VE_WIN = 7;
static_assert(16 * DA_OROW * 4 <= 2 * DA_STAGE, "a wave's output overlays its stages");

constexpr int DA_DMAS = 9;  // loads per block: 4 K, 4 V, the scales

// eight int8 (two words) -> fp16, exactly
__device__ __forceinline__ half8_t da_cvt8(uint32_t x0, uint32_t x1) {
    const half2_t off = {(_Float16)1152.0f, (_Float16)1152.0f};
    x0 ^= 0x80808080u;
    x1 ^= 0x80808080u;
    const half2_t a = as_h2(__builtin_amdgcn_perm(K64, x0, 0x04010400u)) - off;
    const half2_t b = as_h2(__builtin_amdgcn_perm(K64, x0, 0x04030402u)) - off;
    const half2_t c = as_h2(__builtin_amdgcn_perm(K64, x1, 0x04010400u)) - off;
    const half2_t d = as_h2(__builtin_amdgcn_perm(K64, x1, 0x04030402u)) - off;
    return half8_t{a[0], a[1], b[0], b[1], c[0], c[1], d[0], d[1]};
}

struct DecodeState {
    f32x4_t acc[8];  // lane (r, g): head r, channel 32 g + 8 i + mm in acc[mm][i]
    float m, l;      // head r: running max - ve (all four g lanes), sum of p over the lane's tokens
    float ve;        // wave-uniform, an integer
    uint32_t vlo;    // bits of 2^(5 - ve)
};

// One block in LDS stage `st`, first token t0; MASKED: tokens at or past t_end do not count.
template <bool MASKED>
__device__ __forceinline__ void da_block(DecodeState& s, const half8_t (&qf)[4], float kmul,
                                         const uint8_t* st, int t0, int t_end, int l16, int g) {
    v4u k[2][2];
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) {
        const uint8_t* row = st + (16 * mt + l16) * DA_D;
#pragma unroll
        for (int c = 0; c < 2; ++c)
            k[mt][c] = *reinterpret_cast<const v4u*>(row + (((g + 4 * c) ^ (l16 & 7)) << 4));
    }
    f32x4_t ks[2], vs[2];
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) {
        ks[mt] = *reinterpret_cast<const f32x4_t*>(st + DA_SC + 4 * (16 * mt + 4 * g));
        vs[mt] = *reinterpret_cast<const f32x4_t*>(st + DA_SC + 4 * (DA_TOK + 16 * mt + 4 * g));
    }
    uint2 v[8];  // the lane's 8 tokens, channels 8 r ... 8 r + 7
#pragma unroll
    for (int u = 0; u < 8; ++u)
        v[u] = *reinterpret_cast<const uint2*>(
            st + DA_V + (16 * (u >> 2) + 4 * g + (u & 3)) * DA_D + 8 * l16);
    f32x4_t x[2];
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) {
        f32x4_t c = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k4 = 0; k4 < 4; ++k4)
            c = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                da_cvt8(k[mt][k4 >> 1][2 * (k4 & 1)], k[mt][k4 >> 1][2 * (k4 & 1) + 1]), qf[k4],
                c, 0, 0, 0);
        x[mt] = c * ks[mt];
    }
    if (MASKED) {
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const bool in = t0 + 16 * mt + 4 * g + i < t_end;
                x[mt][i] = in ? x[mt][i] : -INFINITY;
                vs[mt][i] = in ? vs[mt][i] : 0.0f;
            }
    }
    float mx = -INFINITY, vmax = 0.0f;
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            mx = fmaxf(mx, x[mt][i]);
            vmax = fmaxf(vmax, vs[mt][i]);
        }
    mx *= kmul;
    // The rare, wave-uniform branch: the running max moves (a score more than DA_SLACK above it),
    // or the V scales leave the window the exponent serves (one lane's above it, or all below).
    if (__ballot(mx - s.ve > s.m + DA_SLACK ||
                 __float_as_uint(vmax) >= s.vlo + ((uint32_t)DA_VE_WIN << 23)) ||
        !__ballot(__float_as_uint(vmax) >= s.vlo)) {
        const float vw = wave_max(vmax);
        const uint32_t vb = __float_as_uint(vw);
        if (vw > 0.0f && vb - s.vlo >= ((uint32_t)DA_VE_WIN << 23)) {
            const int ex = __builtin_amdgcn_frexp_expf(vw);  // vw in [2^(ex-1), 2^ex)
            const float ve = (float)(DA_VE_TOP - ex);
            const float d = ve - s.ve, r = ldexpf(1.0f, (int)d);
#pragma unroll
            for (int mm = 0; mm < 8; ++mm) s.acc[mm] *= r;
            s.l *= r;
            s.m -= d;  // -inf stays -inf
            s.ve = ve;
            s.vlo = (uint32_t)(ex - DA_VE_WIN + 127) << 23;
        }
        const float rm = max_xor32(max_xor16(mx)) - s.ve;
        if (rm > s.m + DA_SLACK) {
            const float alpha = exp2_safe(s.m - rm);  // m = -inf -> 0
#pragma unroll
            for (int mm = 0; mm < 8; ++mm) s.acc[mm] *= alpha;
            s.l *= alpha;
            s.m = rm;
        }
    }
    const float nms = s.m == -INFINITY ? 0.0f : -s.m;
    half8_t p;
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float e = exp2_safe(__builtin_fmaf(x[mt][i], kmul, nms));
            s.l += e;
            p[4 * mt + i] = (_Float16)(e * vs[mt][i]);
        }
    const half2_t off = {(_Float16)1152.0f, (_Float16)1152.0f};
#pragma unroll
    for (int w = 0; w < 2; ++w) {  // channels 8 r + 4 w ... + 3
        half2_t f[4][4];           // [channel][token pair]
#pragma unroll
        for (int u = 0; u < 8; u += 2) {
            const uint32_t xa = (w ? v[u].y : v[u].x) ^ 0x80808080u;
            const uint32_t xb = (w ? v[u + 1].y : v[u + 1].x) ^ 0x80808080u;
            const uint32_t t01 = __builtin_amdgcn_perm(xb, xa, 0x05010400u);
            const uint32_t t23 = __builtin_amdgcn_perm(xb, xa, 0x07030602u);
            f[0][u / 2] = as_h2(__builtin_amdgcn_perm(K64, t01, 0x04010400u)) - off;
            f[1][u / 2] = as_h2(__builtin_amdgcn_perm(K64, t01, 0x04030402u)) - off;
            f[2][u / 2] = as_h2(__builtin_amdgcn_perm(K64, t23, 0x04010400u)) - off;
            f[3][u / 2] = as_h2(__builtin_amdgcn_perm(K64, t23, 0x04030402u)) - off;
        }
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const half8_t a = {f[c][0][0], f[c][0][1], f[c][1][0], f[c][1][1],
                               f[c][2][0], f[c][2][1], f[c][3][0], f[c][3][1]};
            s.acc[4 * w + c] =
                __builtin_amdgcn_mfma_f32_16x16x32_f16(a, p, s.acc[4 * w + c], 0, 0, 0);
        }
    }
}

// grid (nwork, Hkv), block 64 W.
template <int W, bool ROPE>
__global__ __launch_bounds__(W * IE_WAVE) __attribute__((amdgpu_waves_per_eu(2, 2))) void
decode_attention_kernel(DecodeArgs a) {
    constexpr int THREADS = W * IE_WAVE;
    // q's rows of the fused form lie beside the stages; sixteen would cost a one-wave workgroup its
    // eighth place on the CU, so it has eight, and more lie over the second stage, which is then
    // requested after they are read
    constexpr int Q_ROWS = !ROPE ? 1 : W == 1 ? 8 : 16;
    const bool q_over = ROPE && W == 1 && a.ratio > Q_ROWS;
    static_assert(16 * DA_QROW * 2 <= DA_STAGE, "q's rows fit a stage");
    __shared__ __attribute__((aligned(16))) uint8_t s_ring[W][2][DA_STAGE];
    __shared__ __attribute__((aligned(16))) uint16_t s_qrow[Q_ROWS][DA_QROW];
    __shared__ float s_m[W][16], s_l[W][16];
    uint16_t(*s_q)[DA_QROW] =
        q_over ? reinterpret_cast<uint16_t(*)[DA_QROW]>(s_ring[0][1]) : s_qrow;
    const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6);
    const int l16 = lane & 15, g = lane >> 4;
    // The first 64 sequences' lengths and cache slots, issued beside num_decoding: for them the
    // row to stream is known from registers once the work entry is found.
    const int raw0 = lane < a.batch ? a.cached_lens[lane] : 0;
    const int slot0 = lane < a.batch ? a.slot_ids[lane] : 0;
    const int nd = a.num_decoding[0];
    const int item = blockIdx.x, hk = blockIdx.y, R = a.ratio, qh0 = R * hk;
    Work wk;
    if (a.plan) {  // one 16-byte row, requested with the loads above
        const int4 r = *reinterpret_cast<const int4*>(a.plan + 4 * item);
        wk = Work{r.x, r.y, r.z, r.w};
    } else {
        wk = decode_assign(a.cached_lens, nd, item, a.target, raw0);
    }
    const int needed = uniform(wk.needed);
    if (needed == 0) return;
    const int b = uniform(wk.b), split = uniform(wk.split), piece = uniform(wk.piece);
    const int n_end =
        b < 64 ? __builtin_amdgcn_readlane(raw0, b) + 1 : uniform(a.cached_lens[b] + 1);
    const int slot = b < 64 ? __builtin_amdgcn_readlane(slot0, b) : uniform(a.slot_ids[b]);
    const int t_begin = split * piece, t_end = min(t_begin + piece, n_end);

    const v4u rk = rsrc_words(a.c.k + slot * a.c.stride_slot + hk * a.c.stride_head,
                           (uint32_t)t_end * DA_D);
    const v4u rv = rsrc_words(a.c.v + slot * a.c.stride_slot + hk * a.c.stride_head,
                           (uint32_t)t_end * DA_D);
    // lanes 0 ... 31: the block's K scales, lanes 32 ... 63 its V scales
    const float* sc = (lane < DA_TOK ? a.c.k_scale : a.c.v_scale) +
                      slot * a.c.scale_stride_slot + hk * a.c.scale_stride_head;
    uint8_t* ring = s_ring[wave][0];
    const uint32_t lds0 = lds_addr(ring);
    const int koff = (lane >> 3) * DA_D + (((lane & 7) ^ (lane >> 3)) << 4), voff = 16 * lane;
    auto issue = [&](int stage, int t0) {
        const uint32_t l = lds0 + stage * DA_STAGE;
#pragma unroll
        for (int i = 0; i < 4; ++i) dma16<true>(rk, t0 * DA_D + 1024 * i + koff, l + 1024 * i);
        dma4(sc + min(t0 + (lane & (DA_TOK - 1)), t_end - 1), l + DA_SC);
#pragma unroll
        for (int i = 0; i < 4; ++i)
            dma16<true>(rv, t0 * DA_D + 1024 * i + voff, l + DA_V + 1024 * i);
    };
    // this wave's blocks: w, w + W, ... of the piece's 32-token blocks
    const int nb = (t_end - t_begin + DA_TOK - 1) / DA_TOK;
    const int cw = wave < nb ? (nb - wave + W - 1) / W : 0;
    const int t_first = t_begin + wave * DA_TOK;

    // ---- q, and in the fused form the new token's K/V row ----
    const bool last = ROPE && split == needed - 1;
    const bool kv_wave = last && wave == (nb - 1) % W;  // the owner of the new token's block
    uint4 qraw[4];  // lane (r, g): head r, channels 16 g ... + 15 and 64 + 16 g ... + 15
    constexpr int RPW = 16 / W;  // query heads a wave norms and rotates, at most
    uint16_t rq1[RPW], rq2[RPW], rqw1 = 0, rqw2 = 0, rcs = 0, rsn = 0;
    uint16_t rk1 = 0, rk2 = 0, rkw1 = 0, rkw2 = 0, rv1 = 0, rv2 = 0;
    float rc1 = 0.f, rc2 = 0.f;
    if constexpr (ROPE) {
        const float* cal =
            a.c.k_calibration + slot * a.c.cal_stride_slot + hk * a.c.cal_stride_head;
#pragma unroll
        for (int i = 0; i < RPW; ++i) {
            const int h = min(wave + W * i, R - 1);
            const uint16_t* src = a.q + b * a.q_sb + (qh0 + h) * a.q_sh;
            rq1[i] = src[lane];
            rq2[i] = src[lane + 64];
        }
        rqw1 = a.q_norm[lane];
        rqw2 = a.q_norm[lane + 64];
        rcs = a.cos[b * a.cos_sb + lane];
        rsn = a.sin[b * a.sin_sb + lane];
        rc1 = cal[lane];
        rc2 = cal[lane + 64];
        if (kv_wave) {
            const uint16_t* kp = a.k_new + b * a.k_sb + hk * a.k_sh;
            const uint16_t* vp = a.v_new + b * a.v_sb + hk * a.v_sh;
            rk1 = kp[lane];
            rk2 = kp[lane + 64];
            rkw1 = a.k_norm[lane];
            rkw2 = a.k_norm[lane + 64];
            rv1 = vp[lane];
            rv2 = vp[lane + 64];
        }
    } else {
        const uint16_t* qp = a.q + b * a.q_sb + (qh0 + min(l16, R - 1)) * a.q_sh + 16 * g;
        qraw[0] = *reinterpret_cast<const uint4*>(qp);
        qraw[1] = *reinterpret_cast<const uint4*>(qp + 8);
        qraw[2] = *reinterpret_cast<const uint4*>(qp + 64);
        qraw[3] = *reinterpret_cast<const uint4*>(qp + 72);
    }
    __builtin_amdgcn_sched_barrier(0);
    if (cw > 0) issue(0, t_first);
    // q and the first block share a round trip; the second block is requested once q is here
    // (the compiler's wait for q drains what was requested before it)
    int32_t nk1 = 0, nk2 = 0, nv1 = 0, nv2 = 0;
    float nks = 0.f, nvs = 0.f;
    if constexpr (ROPE) {
        asm volatile("" :: "v"(rq1[0]), "v"(rc2) : "memory");
        if (!q_over && cw > 1) issue(1, t_first + W * DA_TOK);
        const float cs = bf16_to_f32(rcs), sn = bf16_to_f32(rsn);
#pragma unroll
        for (int i = 0; i < RPW; ++i) {
            const int h = wave + W * i;
            if (h >= R) break;
            float o1, o2;
            norm_rope_row(bf16_to_f32(rq1[i]), bf16_to_f32(rq2[i]), bf16_to_f32(rqw1),
                          bf16_to_f32(rqw2), cs, sn, a.eps, o1, o2);
            s_q[h][lane] = (uint16_t)f32_to_bf16_rne(o1 * rc1);
            s_q[h][lane + 64] = (uint16_t)f32_to_bf16_rne(o2 * rc2);
        }
        if (kv_wave) {  // fused_rope_kv_decode's arithmetic; column n_end - 1 of the cache
            const int64_t col = n_end - 1;
            const int64_t base =
                slot * a.c.stride_slot + hk * a.c.stride_head + col * a.c.stride_tok;
            const int64_t sidx = slot * a.c.scale_stride_slot + hk * a.c.scale_stride_head + col;
            float o1, o2;
            norm_rope_row(bf16_to_f32(rk1), bf16_to_f32(rk2), bf16_to_f32(rkw1),
                          bf16_to_f32(rkw2), cs, sn, a.eps, o1, o2);
            nks = quantize_row_wave(o1 / rc1, o2 / rc2, nk1, nk2);
            nvs = quantize_row_wave(bf16_to_f32(rv1), bf16_to_f32(rv2), nv1, nv2);
            a.c.k[base + lane] = (int8_t)nk1;
            a.c.k[base + lane + 64] = (int8_t)nk2;
            a.c.v[base + lane] = (int8_t)nv1;
            a.c.v[base + lane + 64] = (int8_t)nv2;
            if (lane == 0) {
                a.c.k_scale[sidx] = nks;
                a.c.v_scale[sidx] = nvs;
            }
        }
        __syncthreads();
        const uint16_t* qp = &s_q[min(l16, R - 1)][16 * g];
        qraw[0] = *reinterpret_cast<const uint4*>(qp);
        qraw[1] = *reinterpret_cast<const uint4*>(qp + 8);
        qraw[2] = *reinterpret_cast<const uint4*>(qp + 64);
        qraw[3] = *reinterpret_cast<const uint4*>(qp + 72);
        if (q_over && cw > 1) {
            lds_reads_done();
            issue(1, t_first + W * DA_TOK);
        }
    } else {
        asm volatile("" :: "v"(qraw[0].x), "v"(qraw[3].w) : "memory");
        if (cw > 1) issue(1, t_first + W * DA_TOK);
    }
    half8_t qf[4];
    float kmul;
    {
        float f[4][8], amax = 0.0f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t w[4] = {qraw[i].x, qraw[i].y, qraw[i].z, qraw[i].w};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                f[i][2 * j] = bf16lo(w[j]);
                f[i][2 * j + 1] = bf16hi(w[j]);
                amax = fmaxf(amax, fmaxf(fabsf(f[i][2 * j]), fabsf(f[i][2 * j + 1])));
            }
        }
        amax = max_xor32(max_xor16(amax));
        int e = 0;
        frexpf(amax, &e);
        const float scl = amax > 0.0f ? ldexpf(1.0f, 14 - e) : 1.0f;  // amax scl in [2^13, 2^14)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 8; ++j) qf[i][j] = (_Float16)(f[i][j] * scl);
        kmul = a.scale_log2 / scl;
    }

    DecodeState s;
#pragma unroll
    for (int mm = 0; mm < 8; ++mm) s.acc[mm] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    s.m = -INFINITY;
    s.l = 0.0f;
    s.ve = 0.0f;
    s.vlo = (uint32_t)(DA_VE_TOP - DA_VE_WIN + 127) << 23;
    for (int j = 0, t0 = t_first; j < cw; ++j, t0 += W * DA_TOK) {
        // block j is here once at most block j + 1's loads (if any) are outstanding
        if (j + 1 < cw) wait_vm<DA_DMAS>();
        else wait_vm<0>();
        uint8_t* st = ring + (j & 1) * DA_STAGE;
        if (t0 + DA_TOK <= t_end && !(kv_wave && j == cw - 1)) {
            da_block<false>(s, qf, kmul, st, t0, t_end, l16, g);
        } else {
            if (kv_wave) {  // the new token's row takes the place of the cache column's old bytes
                const int t = n_end - 1 - t0;
                uint8_t* kr = st + t * DA_D;
                kr[((((lane >> 4)) ^ (t & 7)) << 4) + l16] = (uint8_t)nk1;
                kr[((((lane >> 4) + 4) ^ (t & 7)) << 4) + l16] = (uint8_t)nk2;
                st[DA_V + t * DA_D + lane] = (uint8_t)nv1;
                st[DA_V + t * DA_D + lane + 64] = (uint8_t)nv2;
                if (lane == 0) {
                    reinterpret_cast<float*>(st + DA_SC)[t] = nks;
                    reinterpret_cast<float*>(st + DA_SC)[DA_TOK + t] = nvs;
                }
                lds_reads_done();
            }
            da_block<true>(s, qf, kmul, st, t0, t_end, l16, g);
        }
        if (j + 2 < cw) {  // every read of this stage has its data
            lds_reads_done();
            issue(j & 1, t0 + 2 * W * DA_TOK);
        }
    }

    // ---- merge the waves through LDS (each wave's output over its own, drained stages) ----
    s.l = sum_xor32(sum_xor16(s.l));
    float* so = reinterpret_cast<float*>(ring);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int q = 0; q < 2; ++q)
            *reinterpret_cast<f32x4_t*>(so + l16 * DA_OROW + 32 * g + 8 * i + 4 * q) =
                f32x4_t{s.acc[4 * q][i], s.acc[4 * q + 1][i], s.acc[4 * q + 2][i],
                        s.acc[4 * q + 3][i]};
    if (g == 0) {
        s_m[wave][l16] = s.m;
        s_l[wave][l16] = s.l;
    }
    __syncthreads();
    auto store_out = [&](int h, int d, f32x4_t y) {
        uint16_t* o = a.out + b * a.o_sb + (qh0 + h) * a.o_sh + d;
        if (a.out_vec) {
            *reinterpret_cast<uint2*>(o) = make_uint2(pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3]));
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) o[i] = (uint16_t)f32_to_bf16_rne(y[i]);
        }
    };
    // four channels of one head per thread and pass
    const int quads = R * (DA_D / 4);
    for (int q = tid; q < quads; q += THREADS) {
        const int h = q >> 5, d = 4 * (q & 31);
        float mx = -INFINITY;
#pragma unroll
        for (int w = 0; w < W; ++w) mx = fmaxf(mx, s_m[w][h]);
        f32x4_t num = {0.f, 0.f, 0.f, 0.f};
        float den = 0.0f;
#pragma unroll
        for (int w = 0; w < W; ++w) {
            const float mw = s_m[w][h];
            const float f = mw == -INFINITY ? 0.0f : exp2_safe(mw - mx);
            num += *reinterpret_cast<const f32x4_t*>(reinterpret_cast<const float*>(s_ring[w][0]) +
                                                     h * DA_OROW + d) * f;
            den += s_l[w][h] * f;
        }
        if (needed == 1) {
            store_out(h, d, num / den);
        } else {
            const int64_t row = (int64_t)(qh0 + h) * a.nwork + item;
            float* pa = a.part_acc + row * DA_D + d;
            st_dev64(pa, (uint64_t)__float_as_uint(num[0]) | ((uint64_t)__float_as_uint(num[1]) << 32));
            st_dev64(pa + 2, (uint64_t)__float_as_uint(num[2]) | ((uint64_t)__float_as_uint(num[3]) << 32));
            if (d == 0) {
                st_dev(a.part_m + row, mx);
                st_dev(a.part_l + row, den);
            }
        }
    }
    if (needed == 1) return;
    // A sequence of several pieces (consecutive work entries): each has published its partial with
    // device-coherent stores and counts itself in; the last to arrive merges them all
    // (kernels.py:216-264, in base 2, pieces in order) and resets the count for the next call.
    if (!arrive_last(a.arrivals + b * a.hkv + hk, needed)) return;
    for (int q = tid; q < quads; q += THREADS) {
        const int h = q >> 5, d = 4 * (q & 31);
        const int64_t row0 = (int64_t)(qh0 + h) * a.nwork + (item - split);
        // The wave's two heads from the sequence's first partial of the first one: 32-bit offsets
        // reach them whatever the head count and the batch (nwork < DA_MAX_WORK), where offsets into
        // all partials passed 4 GiB at 128 heads of 65,536 sequences. (8-byte loads from 64-bit
        // addresses instead: 64 pieces of 64/4 heads 26.1 us against 21.6.)
        const int h0 = uniform(h);
        const rsrc_t pr =
            make_rsrc(a.part_acc + ((int64_t)(qh0 + h0) * a.nwork + (item - split)) * DA_D,
                      (uint32_t)(a.nwork + needed) * (DA_D * 4));
        const uint32_t off0 = (uint32_t)((h - h0) * a.nwork * DA_D + d) * 4;
        constexpr int CB = 8;  // partials in flight: one round trip each batch
        f32x4_t av[CB];
        float pm[CB], pl[CB];
        auto load_batch = [&](int s0) {
#pragma unroll
            for (int v = 0; v < CB; ++v) {
                const bool in = s0 + v < needed;
                av[v] = __builtin_bit_cast(
                    f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(
                                 pr, in ? (int)(off0 + (s0 + v) * (DA_D * 4)) : -64, 0, CPOL_SC1));
                pm[v] = in ? ld_dev(a.part_m + row0 + s0 + v) : -INFINITY;
                pl[v] = in ? ld_dev(a.part_l + row0 + s0 + v) : 0.0f;
            }
        };
        load_batch(0);
        float mx = -INFINITY;
#pragma unroll
        for (int v = 0; v < CB; ++v) mx = fmaxf(mx, pm[v]);
        // the other maxima, one per lane of the head's 32 (a batch of CB at a time, as the partials:
        // 64 pieces of 64/4 heads, B=1 ctx 8190, 20.6 us against 19.1)
        if (needed > CB) {
            for (int s = CB + (q & 31); s < needed; s += 32)
                mx = fmaxf(mx, ld_dev(a.part_m + row0 + s));
            mx = max_xor16(max16(mx));
        }
        f32x4_t num = {0.f, 0.f, 0.f, 0.f};
        float den = 0.0f;
        for (int s0 = 0; s0 < needed; s0 += CB) {
            if (s0 > 0) load_batch(s0);
#pragma unroll
            for (int v = 0; v < CB; ++v) {
                const float f = pm[v] == -INFINITY ? 0.0f : exp2_safe(pm[v] - mx);
                num += av[v] * f;
                den += pl[v] * f;
            }
        }
        store_out(h, d, num / den);
    }
}

// grid (work entries), block 64: the decode kernel's work list, one entry per workgroup index w
// of its grid, computed by the same device code (decode_assign), written as
// rows[w] = (b, split, needed, piece).
__global__ __launch_bounds__(64) void decode_plan_kernel(const int32_t* __restrict__ cached_lens,
                                                         const int32_t* __restrict__ num_decoding,
                                                         int batch, int target,
                                                         int32_t* __restrict__ rows) {
    const int lane = threadIdx.x;
    const int raw0 = lane < batch ? cached_lens[lane] : 0;
    const int nd = num_decoding[0];
    const Work wk = decode_assign(cached_lens, nd, blockIdx.x, target, raw0);
    if (lane == 0) {
        int32_t* r = rows + 4 * blockIdx.x;
        r[0] = wk.b;
        r[1] = wk.split;
        r[2] = wk.needed;
        r[3] = wk.piece;
    }
}

// A decode step's per-step launch (ie_decode_step_prologue): the first ngather workgroups copy
// 512-element pieces of the embedding rows x[b] = embed[ids[b]] (zeros for an id outside
// [0, vocab)), one 16-byte load per lane; the next nrope ones the RoPE tables of positions
// cached_lens[0, batch) (64 entries each, rope_table_entry); the rest the work list, as
// decode_plan_kernel writes it.
__global__ __launch_bounds__(64) void decode_prologue_kernel(
    const int32_t* __restrict__ cached_lens, const int32_t* __restrict__ num_decoding, int batch,
    int target, int32_t* __restrict__ rows, const float* __restrict__ inv, int half,
    uint16_t* __restrict__ cosv, uint16_t* __restrict__ sinv, int nrope,
    const int64_t* __restrict__ ids, const uint16_t* __restrict__ embed, int64_t es,
    int64_t vocab, int dim, uint16_t* __restrict__ x, int64_t xs) {
    const int lane = threadIdx.x;
    const int pieces = (dim + 8 * IE_WAVE - 1) / (8 * IE_WAVE);
    const int ngather = batch * pieces;
    int w = blockIdx.x;
    if (w < ngather) {
        const int b = w / pieces, c = (w % pieces) * 8 * IE_WAVE + 8 * lane;
        if (c >= dim) return;  // dim a multiple of 8
        const int64_t id = ids[b];
        const bool ok = id >= 0 && id < vocab;
        const uint4 v = ok ? *reinterpret_cast<const uint4*>(embed + id * es + c)
                           : make_uint4(0u, 0u, 0u, 0u);
        *reinterpret_cast<uint4*>(x + (int64_t)b * xs + c) = v;
        return;
    }
    w -= ngather;
    if (w < nrope) {
        const int64_t i = (int64_t)w * IE_WAVE + lane;
        if (i < (int64_t)batch * half) rope_table_entry(cached_lens, inv, i, half, cosv, sinv);
        return;
    }
    w -= nrope;
    const int raw0 = lane < batch ? cached_lens[lane] : 0;
    const int nd = num_decoding[0];
    const Work wk = decode_assign(cached_lens, nd, w, target, raw0);
    if (lane == 0) {
        int32_t* r = rows + 4 * w;
        r[0] = wk.b;
        r[1] = wk.split;
        r[2] = wk.needed;
        r[3] = wk.piece;
    }
}

// Workspace: the arrival counts (one per sequence and KV head; zero on entry, and every call
// leaves them zero), then fp32 partials (acc, m, l) of every (query head, work entry): one per
// piece, since pieces never outnumber the decode launch's work entries per KV head. The count
// region has room for DA_COUNT_CAP sequences and DA_COUNT_HEADS query heads whatever the batch
// and the head count, so calls of any batch and head count up to those agree on where the
// counts are and their partials never land on them: one workspace serves them all. (Sized by
// the call's own head count, a call with fewer query heads would write partials over the count
// words of a later call with more sequences or heads.) A larger batch or head count gets a
// count region of its own size.
constexpr int DA_COUNT_CAP = 1024;
constexpr int DA_COUNT_HEADS = 128;
struct Layout {
    int waves, target, nwork;
    size_t arr_off, acc_off, m_off, l_off, bytes;
};

// The layout of a launch whose entries are cut for `units` units. The count region has a count per
// sequence and query head (a launch uses one per sequence and KV head), so every launch of a batch
// size finds its counts and partials at the same offsets; then the partial rows, one per query
// head and work entry.
static Layout layout_of(int batch, int hq, int waves, int target) {
    Layout L;
    L.waves = waves;
    L.target = target;
    L.nwork = batch <= target ? target : target + batch;
    const size_t rows = (size_t)hq * L.nwork;
    L.arr_off = 0;
    L.acc_off = ((size_t)std::max(batch, DA_COUNT_CAP) * std::max(hq, DA_COUNT_HEADS) *
                     sizeof(uint32_t) + 255) / 256 * 256;
    L.m_off = L.acc_off + rows * DA_D * sizeof(float);
    L.l_off = L.m_off + rows * sizeof(float);
    L.bytes = L.l_off + rows * sizeof(float);
    return L;
}
static Layout workspace_layout(int batch, int hq, int units) {
    batch = std::max(batch, 0);
    const int waves = decode_waves(batch, units);
    return layout_of(batch, hq, waves, decode_target(units, waves));
}
// What ie_decode_attention_workspace_size reserves: the larger of the grids of cdiv(hq, 2) units
// (ratio 2) and of min(8, cdiv(hq, 2)) units, which gives launches above ratio 2 their entries.
static Layout workspace_size_layout(int batch, int hq) {
    const int pairs = std::max(1, (hq + 1) / 2);
    const Layout a = workspace_layout(batch, hq, pairs);
    const Layout b = workspace_layout(batch, hq, std::min(8, pairs));
    return b.bytes > a.bytes ? b : a;
}

// The layout of a call. Ratios 1 and 2: the grid of their work lists (decode_units is Hkv). Above:
// the same rule per KV head, but the partials of all heads of an entry must fit the workspace of
// workspace_size_layout (and max_bytes, what the call may count on at most): where they do not,
// workgroups of twice the waves and half the entries, up to 8 waves (one per CU), then as many
// entries as fit (few KV heads only: at 8 the first rule always fits). At ratio 1 a batch can pass
// the largest target of Hkv units, which adds spare entries, while the workspace's fewer units still
// hold it without (16/16 heads B=129-256 on 256 CUs: 257-384 entries, 256 reserved): the entries
// reserved, then.
static Layout call_layout(int batch, int hq, int hkv, size_t max_bytes = SIZE_MAX) {
    const Layout own = workspace_layout(batch, hq, hkv);
    if (hq == 2 * hkv) return own;  // one of the two that the workspace is made for
    const Layout S = workspace_size_layout(batch, hq);
    // the widest workgroups of which every entry is resident (one-wave ones where none is): 12/4
    // heads B=300 have 341 entries a head, 5 rounds of 8-wave workgroups
    auto resident_waves = [&](int entries) {
        int w = 8;
        while (w > 1 && decode_target(hkv, w) < entries) w /= 2;
        return w;
    };
    if (hq < 2 * hkv)
        return own.bytes <= S.bytes ? own : layout_of(batch, hq, resident_waves(S.nwork), S.target);
    const size_t room = std::min(S.bytes, max_bytes), row = (DA_D + 2) * sizeof(float);
    const int fit = room > S.acc_off ? (int)((room - S.acc_off) / (hq * row)) : 0;
    auto entries = [&](int t) { return batch <= t ? t : t + batch; };
    int waves = own.waves, target = own.target;
    while (entries(target) > fit && waves < 8) target = decode_target(hkv, waves *= 2);
    if (entries(target) > fit) {
        target = std::max(1, batch <= fit ? fit : fit - batch);
        waves = resident_waves(entries(target));
    }
    return layout_of(batch, hq, waves, target);
}

// The num_units whose work list has a call's entries (a list depends on the batch and the target
// alone), or 0: none of the unit counts that a layout comes from gives that target.
static int list_units(int batch, int hq, int hkv) {
    if (hq == 2 * hkv) return hkv;
    const int target = call_layout(batch, hq, hkv).target, pairs = std::max(1, (hq + 1) / 2);
    for (int u : {hkv, 2 * hkv, 4 * hkv, 8 * hkv, std::min(8, pairs), pairs})
        if (workspace_layout(batch, hq, u).target == target) return u;
    return 0;
}

}  // namespace ie

using namespace ie;

extern "C" size_t ie_decode_attention_workspace_counts_bytes(int32_t batch,
                                                             int32_t num_q_heads) {
    if (num_q_heads <= 0) return 0;
    return layout_of(std::max(batch, 0), num_q_heads, 1, 1).acc_off;  // whatever the entries
}

extern "C" int32_t ie_decode_attention_max_splits(int32_t num_units) {
    return decode_target(num_units, 1);  // the largest target of any launch shape
}

extern "C" int32_t ie_decode_attention_target(int32_t batch, int32_t num_units) {
    if (batch <= 0 || num_units <= 0) return 0;
    return decode_target(num_units, decode_waves(batch, num_units));
}

extern "C" int32_t ie_decode_attention_units(int32_t batch, int32_t num_q_heads,
                                             int32_t num_kv_heads) {
    if (num_q_heads <= 0 || num_kv_heads <= 0 || num_q_heads % num_kv_heads) return 0;
    const int units = list_units(std::max(batch, 0), num_q_heads, num_kv_heads);
    return units ? units : decode_units(num_q_heads, num_kv_heads);
}

extern "C" size_t ie_decode_attention_workspace_size(int32_t batch, int32_t num_q_heads,
                                                     int32_t head_dim) {
    (void)head_dim;
    if (num_q_heads <= 0) return 0;
    return workspace_size_layout(batch, num_q_heads).bytes;
}

// q_rows16: q is read in 16-byte pieces (the plain form; the fused form reads q two bytes per
// lane, as fused_rope_kv_decode does).
static hipError_t check_decode(const ie_bf16* q, int32_t batch, int32_t num_q_heads,
                               const ie_kv_cache* cache, const int32_t* cached_lens,
                               const int32_t* slot_ids, const int32_t* num_decoding,
                               const ie_bf16* out, int64_t q_sb, int64_t q_sh, void* workspace,
                               size_t workspace_bytes, Layout* L, bool q_rows16 = true,
                               size_t max_bytes = SIZE_MAX) {
    hipError_t e = check_cache(cache);
    if (e != hipSuccess) return e;
    IE_REQUIRE(batch >= 0, "negative batch");
    IE_REQUIRE(num_q_heads > 0 && num_q_heads % cache->num_kv_heads == 0 &&
                   num_q_heads / cache->num_kv_heads <= 16,
               "num_q_heads must be num_kv_heads times a GQA ratio of 1 to 16");
    if (batch == 0) return hipSuccess;
    IE_REQUIRE(q && cached_lens && slot_ids && num_decoding && out, "null pointer");
    IE_REQUIRE(!q_rows16 ||
                   ((reinterpret_cast<uintptr_t>(q) & 15) == 0 && q_sb % 8 == 0 && q_sh % 8 == 0),
               "q rows must be 16-byte aligned with contiguous head_dim");
    *L = call_layout(batch, num_q_heads, (int)cache->num_kv_heads, max_bytes);
    IE_REQUIRE(L->nwork < DA_MAX_WORK, "batch too large");
    IE_REQUIRE(workspace != nullptr && workspace_bytes >= L->bytes, "workspace too small");
    IE_REQUIRE((reinterpret_cast<uintptr_t>(workspace) & 15) == 0, "workspace must be aligned");
    return hipSuccess;
}

// The arguments both forms share; the fused form's own fields stay null.
static DecodeArgs decode_args(const ie_bf16* q, int64_t q_stride_b, int64_t q_stride_h,
                              int32_t batch, int32_t num_q_heads, const ie_kv_cache* cache,
                              const int32_t* cached_lens, const int32_t* slot_ids,
                              const int32_t* num_decoding, float scale, ie_bf16* out,
                              int64_t out_stride_b, int64_t out_stride_h, void* workspace,
                              const Layout& L) {
    DecodeArgs a{};
    a.q = (const uint16_t*)q;
    a.q_sb = q_stride_b;
    a.q_sh = q_stride_h;
    a.c = *cache;
    a.cached_lens = cached_lens;
    a.slot_ids = slot_ids;
    a.num_decoding = num_decoding;
    a.scale_log2 = scale * 1.4426950408889634f;
    a.out = (uint16_t*)out;
    a.o_sb = out_stride_b;
    a.o_sh = out_stride_h;
    char* ws = (char*)workspace;
    a.part_acc = (float*)(ws + L.acc_off);
    a.part_m = (float*)(ws + L.m_off);
    a.part_l = (float*)(ws + L.l_off);
    a.arrivals = (uint32_t*)(ws + L.arr_off);
    a.target = L.target;
    a.nwork = L.nwork;
    a.hq = num_q_heads;
    a.hkv = (int)cache->num_kv_heads;
    a.ratio = num_q_heads / a.hkv;
    a.batch = batch;
    return a;
}

template <bool ROPE>
static hipError_t decode_launch(DecodeArgs& a, const Layout& L, hipStream_t stream) {
    // pieces number at most target + nd, and at most target when nd <= target (decode_piece):
    // with batch <= target the grid needs no spare workgroups, which would otherwise hold
    // resident slots while they find out that they are idle
    const dim3 grid((unsigned)L.nwork, (unsigned)a.hkv);
    a.out_vec = (reinterpret_cast<uintptr_t>(a.out) & 7) == 0 && a.o_sb % 4 == 0 && a.o_sh % 4 == 0;
    switch (L.waves) {
        case 8: hipLaunchKernelGGL((decode_attention_kernel<8, ROPE>), grid, dim3(512), 0, stream, a); break;
        case 4: hipLaunchKernelGGL((decode_attention_kernel<4, ROPE>), grid, dim3(256), 0, stream, a); break;
        case 2: hipLaunchKernelGGL((decode_attention_kernel<2, ROPE>), grid, dim3(128), 0, stream, a); break;
        default: hipLaunchKernelGGL((decode_attention_kernel<1, ROPE>), grid, dim3(64), 0, stream, a); break;
    }
    return hipGetLastError();
}

// A precomputed work list must cover the grid it is made for; it is read (*read) where that is the
// launch's.
static hipError_t check_plan(const int32_t* plan, int64_t plan_rows, int32_t batch, int32_t hq,
                             int32_t hkv, const Layout& L, bool* read) {
    IE_REQUIRE(plan != nullptr, "null plan");
    const bool launch = plan_rows >= IE_PLAN_LAUNCH_UNITS;
    const int units = launch ? ie_decode_attention_units(batch, hq, hkv) : decode_units(hq, hkv);
    if (launch) plan_rows -= IE_PLAN_LAUNCH_UNITS;
    IE_REQUIRE(plan_rows >= ie_decode_attention_grid(batch, units),
               "plan must hold ie_decode_attention_grid(batch, units) rows");
    IE_REQUIRE((reinterpret_cast<uintptr_t>(plan) & 15) == 0, "plan must be 16-byte aligned");
    *read = ie_decode_attention_target(batch, units) == L.target;
    return hipSuccess;
}

static hipError_t decode_plain(const ie_bf16* q, int64_t q_stride_b, int64_t q_stride_h,
                               int32_t batch, int32_t num_q_heads, const ie_kv_cache* cache,
                               const int32_t* cached_lens, const int32_t* slot_ids,
                               const int32_t* num_decoding, float scale, ie_bf16* out,
                               int64_t out_stride_b, int64_t out_stride_h, void* workspace,
                               size_t workspace_bytes, const int32_t* plan, int64_t plan_rows,
                               bool planned, hipStream_t stream, size_t max_bytes = SIZE_MAX) {
    Layout L{};
    hipError_t e = check_decode(q, batch, num_q_heads, cache, cached_lens, slot_ids, num_decoding,
                                out, q_stride_b, q_stride_h, workspace, workspace_bytes, &L, true,
                                max_bytes);
    if (e != hipSuccess || batch == 0) return e;
    bool read = false;
    if (planned && (e = check_plan(plan, plan_rows, batch, num_q_heads,
                                   (int32_t)cache->num_kv_heads, L, &read)) != hipSuccess)
        return e;
    DecodeArgs a = decode_args(q, q_stride_b, q_stride_h, batch, num_q_heads, cache, cached_lens,
                               slot_ids, num_decoding, scale, out, out_stride_b, out_stride_h,
                               workspace, L);
    a.plan = read ? plan : nullptr;
    return decode_launch<false>(a, L, stream);
}

extern "C" hipError_t ie_decode_attention(
    const ie_bf16* q, int64_t q_stride_b, int64_t q_stride_h, int32_t batch, int32_t num_q_heads,
    const ie_kv_cache* cache, const int32_t* cached_lens, const int32_t* slot_ids,
    const int32_t* num_decoding, float scale, ie_bf16* out, int64_t out_stride_b,
    int64_t out_stride_h, void* workspace, size_t workspace_bytes, hipStream_t stream) {
    return decode_plain(q, q_stride_b, q_stride_h, batch, num_q_heads, cache, cached_lens,
                        slot_ids, num_decoding, scale, out, out_stride_b, out_stride_h, workspace,
                        workspace_bytes, nullptr, 0, false, stream);
}

extern "C" hipError_t ie_decode_attention_planned(
    const ie_bf16* q, int64_t q_stride_b, int64_t q_stride_h, int32_t batch, int32_t num_q_heads,
    const ie_kv_cache* cache, const int32_t* cached_lens, const int32_t* slot_ids,
    const int32_t* num_decoding, const int32_t* plan, int64_t plan_rows, float scale,
    ie_bf16* out, int64_t out_stride_b, int64_t out_stride_h, void* workspace,
    size_t workspace_bytes, hipStream_t stream) {
    return decode_plain(q, q_stride_b, q_stride_h, batch, num_q_heads, cache, cached_lens,
                        slot_ids, num_decoding, scale, out, out_stride_b, out_stride_h, workspace,
                        workspace_bytes, plan, plan_rows, true, stream);
}

static hipError_t decode_rope(
    const ie_bf16* q, int64_t q_stride_b, int64_t q_stride_h, const ie_bf16* k,
    int64_t k_stride_b, int64_t k_stride_h, const ie_bf16* v, int64_t v_stride_b,
    int64_t v_stride_h, const ie_bf16* q_norm_weight, const ie_bf16* k_norm_weight,
    const ie_bf16* cos, int64_t cos_stride_b, const ie_bf16* sin, int64_t sin_stride_b,
    float eps, int32_t batch, int32_t num_q_heads, const ie_kv_cache* cache,
    const int32_t* cached_lens, const int32_t* slot_ids, const int32_t* num_decoding,
    const int32_t* plan, int64_t plan_rows, bool planned, float scale, ie_bf16* out,
    int64_t out_stride_b, int64_t out_stride_h, void* workspace, size_t workspace_bytes,
    hipStream_t stream) {
    Layout L{};
    hipError_t e = check_decode(q, batch, num_q_heads, cache, cached_lens, slot_ids, num_decoding,
                                out, q_stride_b, q_stride_h, workspace, workspace_bytes, &L,
                                false);
    if (e != hipSuccess || batch == 0) return e;
    IE_REQUIRE(k && v && q_norm_weight && k_norm_weight && cos && sin, "null pointer");
    bool read = false;
    if (planned && (e = check_plan(plan, plan_rows, batch, num_q_heads,
                                   (int32_t)cache->num_kv_heads, L, &read)) != hipSuccess)
        return e;
    DecodeArgs a = decode_args(q, q_stride_b, q_stride_h, batch, num_q_heads, cache, cached_lens,
                               slot_ids, num_decoding, scale, out, out_stride_b, out_stride_h,
                               workspace, L);
    a.plan = read ? plan : nullptr;
    a.k_new = (const uint16_t*)k;
    a.k_sb = k_stride_b;
    a.k_sh = k_stride_h;
    a.v_new = (const uint16_t*)v;
    a.v_sb = v_stride_b;
    a.v_sh = v_stride_h;
    a.q_norm = (const uint16_t*)q_norm_weight;
    a.k_norm = (const uint16_t*)k_norm_weight;
    a.cos = (const uint16_t*)cos;
    a.sin = (const uint16_t*)sin;
    a.cos_sb = cos_stride_b;
    a.sin_sb = sin_stride_b;
    a.eps = eps;
    return decode_launch<true>(a, L, stream);
}

extern "C" hipError_t ie_decode_attention_rope(
    const ie_bf16* q, int64_t q_stride_b, int64_t q_stride_h, const ie_bf16* k,
    int64_t k_stride_b, int64_t k_stride_h, const ie_bf16* v, int64_t v_stride_b,
    int64_t v_stride_h, const ie_bf16* q_norm_weight, const ie_bf16* k_norm_weight,
    const ie_bf16* cos, int64_t cos_stride_b, const ie_bf16* sin, int64_t sin_stride_b,
    float eps, int32_t batch, int32_t num_q_heads, const ie_kv_cache* cache,
    const int32_t* cached_lens, const int32_t* slot_ids, const int32_t* num_decoding,
    float scale, ie_bf16* out, int64_t out_stride_b, int64_t out_stride_h, void* workspace,
    size_t workspace_bytes, hipStream_t stream) {
    return decode_rope(q, q_stride_b, q_stride_h, k, k_stride_b, k_stride_h, v, v_stride_b,
                       v_stride_h, q_norm_weight, k_norm_weight, cos, cos_stride_b, sin,
                       sin_stride_b, eps, batch, num_q_heads, cache, cached_lens, slot_ids,
                       num_decoding, nullptr, 0, false, scale, out, out_stride_b, out_stride_h,
                       workspace, workspace_bytes, stream);
}

extern "C" hipError_t ie_decode_attention_rope_planned(
    const ie_bf16* q, int64_t q_stride_b, int64_t q_stride_h, const ie_bf16* k,
    int64_t k_stride_b, int64_t k_stride_h, const ie_bf16* v, int64_t v_stride_b,
    int64_t v_stride_h, const ie_bf16* q_norm_weight, const ie_bf16* k_norm_weight,
    const ie_bf16* cos, int64_t cos_stride_b, const ie_bf16* sin, int64_t sin_stride_b,
    float eps, int32_t batch, int32_t num_q_heads, const ie_kv_cache* cache,
    const int32_t* cached_lens, const int32_t* slot_ids, const int32_t* num_decoding,
    const int32_t* plan, int64_t plan_rows, float scale, ie_bf16* out, int64_t out_stride_b,
    int64_t out_stride_h, void* workspace, size_t workspace_bytes, hipStream_t stream) {
    return decode_rope(q, q_stride_b, q_stride_h, k, k_stride_b, k_stride_h, v, v_stride_b,
                       v_stride_h, q_norm_weight, k_norm_weight, cos, cos_stride_b, sin,
                       sin_stride_b, eps, batch, num_q_heads, cache, cached_lens, slot_ids,
                       num_decoding, plan, plan_rows, true, scale, out, out_stride_b,
                       out_stride_h, workspace, workspace_bytes, stream);
}

extern "C" int32_t ie_decode_attention_grid(int32_t batch, int32_t num_units) {
    if (batch <= 0 || num_units <= 0) return 0;
    const int target = ie_decode_attention_target(batch, num_units);
    return batch <= target ? target : target + batch;
}

extern "C" hipError_t ie_decode_step_prologue(
    const int32_t* cached_lens, const int32_t* num_decoding, int32_t batch, int32_t num_units,
    int32_t* rows, const float* inv_freq, int32_t half_dim, ie_bf16* cos_out, ie_bf16* sin_out,
    const int64_t* ids, const ie_bf16* embed, int64_t embed_stride, int64_t vocab,
    int32_t model_dim, ie_bf16* x, int64_t x_stride, hipStream_t stream) {
    IE_REQUIRE(batch >= 0 && num_units > 0 && half_dim > 0 && vocab > 0 && model_dim > 0,
               "bad sizes");
    if (batch == 0) return hipSuccess;
    IE_REQUIRE(cached_lens && num_decoding && rows && inv_freq && cos_out && sin_out && ids &&
                   embed && x,
               "null pointer");
    IE_REQUIRE(model_dim % 8 == 0 && embed_stride % 8 == 0 && x_stride % 8 == 0 &&
                   (reinterpret_cast<uintptr_t>(embed) & 15) == 0 &&
                   (reinterpret_cast<uintptr_t>(x) & 15) == 0,
               "embedding and x rows must be 16-byte aligned, model_dim a multiple of 8");
    const int target = ie_decode_attention_target(batch, num_units);
    const int nplan = ie_decode_attention_grid(batch, num_units);
    const int64_t nrope = ((int64_t)batch * half_dim + IE_WAVE - 1) / IE_WAVE;
    const int64_t ngather = (int64_t)batch * ((model_dim + 8 * IE_WAVE - 1) / (8 * IE_WAVE));
    IE_REQUIRE(nplan + nrope + ngather < (1LL << 31), "too many workgroups");
    hipLaunchKernelGGL(decode_prologue_kernel, dim3((unsigned)(ngather + nrope + nplan)),
                       dim3(IE_WAVE), 0, stream, cached_lens, num_decoding, batch, target,
                       rows, inv_freq, (int)half_dim, (uint16_t*)cos_out, (uint16_t*)sin_out,
                       (int)nrope, ids, (const uint16_t*)embed, embed_stride, vocab,
                       (int)model_dim, (uint16_t*)x, x_stride);
    return hipGetLastError();
}

extern "C" hipError_t ie_decode_attention_plan(const int32_t* cached_lens,
                                               const int32_t* num_decoding, int32_t batch,
                                               int32_t num_units, int32_t* rows,
                                               hipStream_t stream) {
    IE_REQUIRE(batch >= 0 && num_units > 0, "bad sizes");
    if (batch == 0) return hipSuccess;
    IE_REQUIRE(cached_lens && num_decoding && rows, "null pointer");
    const int target = ie_decode_attention_target(batch, num_units);
    hipLaunchKernelGGL(decode_plan_kernel, dim3((unsigned)ie_decode_attention_grid(batch, num_units)),
                       dim3(IE_WAVE), 0, stream, cached_lens, num_decoding, batch, target, rows);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------------------
// The entry point that allocates nothing: ie_decode_attention with its workspace in a static
// device array of DA_SCRATCH_BYTES, which every device the library runs on holds until the
// process ends (16 MiB: the arrival counts and partials of up to 1,024 sequences, the batches
// that share one count region). The array's name is only a host-side stand-in for the device copy, so
// its address on each device is looked up once, with that device current, and only that
// address is passed to the kernels. The array starts zeroed, as the workspace contract asks,
// and every call leaves the arrival counts zeroed again. All calls on one device share the array,
// so calls that overlap on one device (different streams, or threads without ordering) race.
// ---------------------------------------------------------------------------------------------
namespace {
constexpr size_t DA_SCRATCH_BYTES = size_t(16) << 20;
constexpr int DA_SCRATCH_DEVICES = 64;
__device__ __align__(256) unsigned char scratch[DA_SCRATCH_BYTES];
std::mutex scratch_mu;
void* scratch_ptr[DA_SCRATCH_DEVICES];

// This device's copy of `scratch` (resolved on the first call made with the device current).
hipError_t scratch_address(void** out) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    IE_REQUIRE(dev >= 0 && dev < DA_SCRATCH_DEVICES, "device index out of range");
    std::lock_guard<std::mutex> lock(scratch_mu);
    if (scratch_ptr[dev] == nullptr) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        IE_REQUIRE(p != nullptr, "no device address for the decode scratch");
        scratch_ptr[dev] = p;
    }
    *out = scratch_ptr[dev];
    return hipSuccess;
}
}  // namespace

extern "C" size_t ie_decode_attention_noalloc_max_bytes(void) { return DA_SCRATCH_BYTES; }

extern "C" hipError_t ie_decode_attention_noalloc(
    const ie_bf16* q, int64_t q_stride_b, int64_t q_stride_h, int32_t batch, int32_t num_q_heads,
    const ie_kv_cache* cache, const int32_t* cached_lens, const int32_t* slot_ids,
    const int32_t* num_decoding, float scale, ie_bf16* out, int64_t out_stride_b,
    int64_t out_stride_h, hipStream_t stream) {
    hipError_t e = check_cache(cache);
    if (e != hipSuccess) return e;
    IE_REQUIRE(batch >= 0, "negative batch");
    if (batch == 0) return hipSuccess;
    IE_REQUIRE(num_q_heads > 0 && num_q_heads % cache->num_kv_heads == 0 &&
                   num_q_heads / cache->num_kv_heads <= 16,
               "num_q_heads must be num_kv_heads times a GQA ratio of 1 to 16");
    const Layout L = call_layout(batch, num_q_heads, (int)cache->num_kv_heads, DA_SCRATCH_BYTES);
    IE_REQUIRE(batch <= DA_COUNT_CAP && num_q_heads <= DA_COUNT_HEADS &&
                   L.bytes <= DA_SCRATCH_BYTES,
               "batch too large for the no-alloc decode scratch (at most 1024 sequences and "
               "128 query heads in 16 MiB; use ie_decode_attention with a workspace)");
    void* ws = nullptr;
    e = scratch_address(&ws);
    if (e != hipSuccess) return e;
    return decode_plain(q, q_stride_b, q_stride_h, batch, num_q_heads, cache, cached_lens, slot_ids,
                        num_decoding, scale, out, out_stride_b, out_stride_h, ws, DA_SCRATCH_BYTES,
                        nullptr, 0, false, stream, DA_SCRATCH_BYTES);
}
