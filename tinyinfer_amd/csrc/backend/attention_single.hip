// Stand-alone paged GQA decode attention over caller-owned pools in the
// reference layout ([block][layer][slot][kv_width], paged_kv.cpp:53-56): the
// single-operation entry point mp_hip_paged_attention_decode.
//
// Every reduction that the reference CPU path performs sequentially
// (miniprefix/src/backend/cpu/llama_runner.cpp:85-93) runs in ONE lane in the
// same order, with multiply and add rounded separately (this file is
// compiled with -ffp-contract=off). Parallelism comes from independent
// outputs: tokens for scores, (head, d) for the PV sums. (The denominator's
// order is kept by ordered_sum.h with a whole wavefront.)
//
// Pages of 16 tokens with 64-wide heads take the kernels at the end of this
// file (except where attention_row_pays says otherwise, where out lies over q
// and where the values are not 16-byte aligned); other shapes the general
// kernel below.
#include "exact_math.h"
#include "kernels.h"
#include "layout.h"
#include "ordered_sum.h"

namespace mphip {
namespace {

constexpr int kWave = 64;

// Sequential float sum of n values (n a multiple of 4, 16-byte aligned) in
// the calling lane, in index order, starting from `sum`. Two blocks of
// sixteen ping-pong: one is read while the other is added.
__device__ __forceinline__ void sum_block(const float4 (&a)[4], float& sum) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        sum = sum + a[j].x;
        sum = sum + a[j].y;
        sum = sum + a[j].z;
        sum = sum + a[j].w;
    }
}

__device__ __forceinline__ float sequential_sum(const float* v, int n, float sum = 0.0f) {
    const float4* v4 = reinterpret_cast<const float4*>(v);
    const int n4 = n / 4;
    int i = 0;
    if (n4 >= 4) {
        float4 a[4], b[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) a[j] = v4[j];
        for (; i + 8 <= n4; i += 8) {
#pragma unroll
            for (int j = 0; j < 4; ++j) b[j] = v4[i + 4 + j];
            sum_block(a, sum);
            const int in = min(i + 8, n4 - 4);
#pragma unroll
            for (int j = 0; j < 4; ++j) a[j] = v4[in + j];
            sum_block(b, sum);
        }
        if (i + 4 <= n4) {  // `a` holds the block at i
            sum_block(a, sum);
            i += 4;
        }
    }
    for (; i < n4; ++i) {
        const float4 a = v4[i];
        sum = sum + a.x;
        sum = sum + a.y;
        sum = sum + a.z;
        sum = sum + a.w;
    }
    return sum;
}

// Block-wide float max of one value per thread (max is exact and
// order-free, so a tree is fine here).
__device__ __forceinline__ float block_max(float v, float* shared) {
    for (int o = kWave / 2; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
    const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    __syncthreads();
    if (lane == 0) shared[wave] = v;
    __syncthreads();
    float m = shared[0];
    for (int i = 1; i < (int)(blockDim.x / kWave); ++i) m = fmaxf(m, shared[i]);
    return m;
}

constexpr int kAttentionThreads = 256;
constexpr int kMaxGroup = 8;
constexpr int kMaxDim = 256;
constexpr int kLdsTable = 2048;

// One work-group per (row, kv head): the group's query heads share every K
// and V byte. Reference order per (row, head) (llama_runner.cpp:86-92):
//   s_t = (sum_d q_d k_td, sequential d) / sqrt(dim)
//   m   = max_t s_t
//   e_t = expf(s_t - m);  den = sum_t e_t, sequential t
//   out_d = sum_t (e_t/den) * v_td, sequential t
// Scores are parallel over t; the denominator runs in one lane per head and
// each (head, d) output chain in one lane, streaming V page by page with the
// next page's loads already in flight. BT is the page size (0: runtime).
struct AttentionRow {
    const float* q;
    const int32_t* table;
    int length;
    float* out;
};

struct AttentionGeometry {
    int layer, layers, block_tokens, kv_width, group, dim, kh;
};

template <int BT>
__device__ void attention_row(const AttentionRow& row, const float* __restrict__ keys,
                              const float* __restrict__ values, const AttentionGeometry& g,
                              float* scores_global) {
    __shared__ float qs[kMaxGroup * kMaxDim];
    __shared__ float lds_scores[kAttentionLdsScores];
    __shared__ int32_t lds_table[kLdsTable];
    __shared__ float reduce[kAttentionThreads / kWave];
    __shared__ float den_shared[kMaxGroup];
    __shared__ float max_shared[kMaxGroup];
    const int tid = threadIdx.x;
    const int bt = BT ? BT : g.block_tokens;
    const int length = row.length, group = g.group, dim = g.dim;
    const int pages = (length + bt - 1) / bt;
    // Score rows padded to a multiple of 16; the padding holds zeros, which
    // leave the sequential sums unchanged (x + 0 == x for the non-negative
    // running sums here).
    const int stride = (length + 15) & ~15;
    float* scores = group * stride <= kAttentionLdsScores ? lds_scores : scores_global;
    const int32_t* table = row.table;
    if (pages <= kLdsTable) {
        for (int i = tid; i < pages; i += kAttentionThreads) lds_table[i] = row.table[i];
        table = lds_table;
    }
    for (int i = tid; i < group * dim; i += kAttentionThreads) qs[i] = row.q[i];
    __syncthreads();
    const size_t layer_stride = (size_t)bt * g.kv_width;
    auto token_offset = [&](int t) -> size_t {
        const int page = t / bt, slot = t - page * bt;
        return ((size_t)table[page] * g.layers + g.layer) * layer_stride + (size_t)slot * g.kv_width +
               (size_t)g.kh * dim;
    };
    // Scores: one token per thread, `group` sequential dot products.
    float local_max[kMaxGroup];
    for (int h = 0; h < group; ++h) local_max[h] = -INFINITY;
    const float root = sqrtf((float)dim);
    for (int t = tid; t < length; t += kAttentionThreads) {
        const float* k = keys + token_offset(t);
        float s[kMaxGroup];
        for (int h = 0; h < group; ++h) s[h] = 0.0f;
        for (int d0 = 0; d0 < dim; d0 += 16) {
            float4 kv4[4];
#pragma unroll
            for (int j = 0; j < 4; ++j)
                kv4[j] = d0 + 4 * j < dim ? *reinterpret_cast<const float4*>(k + d0 + 4 * j)
                                          : make_float4(0.f, 0.f, 0.f, 0.f);
            for (int h = 0; h < group; ++h) {
                const float* qh = qs + h * dim + d0;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    if (d0 + 4 * j >= dim) break;
                    s[h] = s[h] + qh[4 * j + 0] * kv4[j].x;
                    s[h] = s[h] + qh[4 * j + 1] * kv4[j].y;
                    s[h] = s[h] + qh[4 * j + 2] * kv4[j].z;
                    s[h] = s[h] + qh[4 * j + 3] * kv4[j].w;
                }
            }
        }
        for (int h = 0; h < group; ++h) {
            const float score = s[h] / root;
            scores[h * stride + t] = score;
            local_max[h] = local_max[h] < score ? score : local_max[h];
        }
    }
    for (int h = 0; h < group; ++h) {
        const float m = block_max(local_max[h], reduce);
        if (tid == 0) max_shared[h] = m;
    }
    __syncthreads();
    for (int h = 0; h < group; ++h) {
        const float m = max_shared[h];
        for (int t = tid; t < stride; t += kAttentionThreads)
            scores[h * stride + t] = t < length ? ref_expf(scores[h * stride + t] - m) : 0.0f;
    }
    __syncthreads();
    if (tid < group) den_shared[tid] = sequential_sum(scores + tid * stride, stride);
    __syncthreads();
    for (int h = 0; h < group; ++h) {
        const float den = den_shared[h];
        for (int t = tid; t < length; t += kAttentionThreads)
            scores[h * stride + t] = scores[h * stride + t] / den;
    }
    __syncthreads();
    // PV chains: thread -> (head, d).
    for (int chain = tid; chain < group * dim; chain += kAttentionThreads) {
        const int h = chain / dim, d = chain % dim;
        const float* p = scores + h * stride;
        const float* vbase = values + (size_t)g.kh * dim + d;
        float total = 0.0f;
        if (BT) {
            // Page-structured stream: a page's BT loads are independent; the
            // next page is loaded while this one is summed.
            float bufa[BT ? BT : 1], bufb[BT ? BT : 1];
            auto load_page = [&](int page, float* buf) {
                if (page >= pages) return;
                const float* src = vbase + ((size_t)table[page] * g.layers + g.layer) * layer_stride;
                const int valid = min(BT, length - page * BT);
#pragma unroll
                for (int j = 0; j < BT; ++j) buf[j] = j < valid ? src[(size_t)j * g.kv_width] : 0.0f;
            };
            auto sum_page = [&](int page, const float* buf) {
                if (page >= pages) return;
                const float4* p4 = reinterpret_cast<const float4*>(p + page * BT);
                const int valid = min(BT, length - page * BT);
#pragma unroll
                for (int j4 = 0; j4 < BT / 4; ++j4) {
                    const float4 pv = p4[j4];
                    if (4 * j4 + 0 < valid) total = total + pv.x * buf[4 * j4 + 0];
                    if (4 * j4 + 1 < valid) total = total + pv.y * buf[4 * j4 + 1];
                    if (4 * j4 + 2 < valid) total = total + pv.z * buf[4 * j4 + 2];
                    if (4 * j4 + 3 < valid) total = total + pv.w * buf[4 * j4 + 3];
                }
            };
            load_page(0, bufa);
            load_page(1, bufb);
            for (int page = 0; page < pages; page += 2) {
                sum_page(page, bufa);
                load_page(page + 2, bufa);
                sum_page(page + 1, bufb);
                load_page(page + 3, bufb);
            }
        } else {
            for (int t = 0; t < length; ++t) total = total + p[t] * vbase[token_offset(t) - (size_t)g.kh * dim];
        }
        row.out[h * dim + d] = total;
    }
    __syncthreads();
}

template <int BT>
__global__ __launch_bounds__(kAttentionThreads) void attention_single_kernel(
    const float* __restrict__ q, const float* __restrict__ keys, const float* __restrict__ values,
    const int32_t* __restrict__ table, int length, int layer, int layers, int block_tokens,
    int heads, int kv_heads, int dim, float* __restrict__ out, float* scratch) {
    const int kh = blockIdx.y;
    const int group = heads / kv_heads;
    AttentionRow row;
    row.q = q + (size_t)kh * group * dim;
    row.table = table;
    row.length = length;
    row.out = out + (size_t)kh * group * dim;
    float* scores_global =
        scratch ? scratch + (size_t)kh * group * (size_t)((length + 15) & ~15) : nullptr;
    const AttentionGeometry g{layer, layers, block_tokens, kv_heads * dim, group, dim, kh};
    attention_row<BT>(row, keys, values, g, scores_global);
}

// ---------------------------------------------------------------------------
// Pages of 16 tokens, 64-wide heads.
//
// What bounds it: the output chains, one dependent add per token (6 cycles,
// 2.5 ns); around them whatever a launch leaves to few wavefronts; and the
// bytes one CU can read (about 15 of the 64 per clock it nominally takes,
// over scattered rows). So:
// - scores (parallel over tokens): in a kernel of their own over the whole
//   chip where the row has scratch, else in the row kernel;
// - the row kernel: one work-group per query head and 16 of its dims, so that
//   a CU streams a quarter of the head's V. Each forms e_t and p_t for itself
//   with all wavefronts and the denominator by ordered_sum (a fifth of its
//   chain). For the output one consumer wavefront (lane = d) only adds: seven
//   producer wavefronts stream V (a page of the 16 dims is one 16-byte load
//   per lane), form the products p_t v_td and hand them over through LDS.
//   Product and sum in one lane cost 9.5 cycles per token, the sum alone 6.
// Against one work-group per KV head for everything (attention_single_kernel,
// 9 query heads on 3 KV heads): 47.3 -> 17.4 us for 503 tokens, 1,695 -> 95 us
// for 16,640, of which the scores 7.5, e_t 5.4, the denominator 10.2, p_t 3.5
// and the output chains 62 us (9 cycles per token).
constexpr int kRowThreads = 512;
constexpr int kRowDim = 64;
constexpr int kRowPage = 16;
constexpr int kRowWindow = 18432;  // tokens whose e_t are held in LDS (72 KB)
constexpr int kRowWaves = kRowThreads / kWave;
constexpr int kRowHeld = kRowWindow / kRowThreads;  // tokens of a window per thread
constexpr int kSlice = 16;         // dims per work-group
constexpr int kProducers = kRowWaves - 1;
constexpr int kPerPhase = 2;       // pages per producer and phase
constexpr int kPhasePages = kPerPhase * kProducers;
constexpr int kAhead = 4;          // phases whose V is in flight
constexpr int kRingPad = 20;       // floats per dim of a page's products in LDS (16 tokens)
constexpr int kTilePad = 36;  // floats per token of a 32-dim half tile in LDS
constexpr int kScoreThreads = 256;

struct RowArgs {
    const float* q;
    const float* keys;
    const float* values;
    const int32_t* table;
    int length, layer, layers, heads, kv_heads;
    float* out;
    float* scores;  // [heads][round_up(length, 16)], or null: scores in the row kernel
};

__device__ __forceinline__ size_t row_page(const RowArgs& a, int block, int kvh) {
    return ((size_t)block * a.layers + a.layer) * (size_t)(kRowPage * kRowDim) * a.kv_heads + (size_t)kvh * kRowDim;
}

// The K rows of 64 consecutive tokens (t0.., clamped to the row's last one),
// one per lane: read as whole 128-byte pieces, turned through this
// wavefront's LDS tile, 32 dims at a time. Then fn(half) finds the lane's
// token's dims 32 half .. + 31 in `k`.
template <typename Fn>
__device__ __forceinline__ void key_rows(const RowArgs& a, int kvh, int t0, float* tile, Fn&& fn) {
    const int lane = threadIdx.x & 63;
    const size_t step = (size_t)kRowDim * a.kv_heads;
    float4 lo[8], hi[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int t = min(t0 + 8 * i + (lane >> 3), a.length - 1);
        const float* src = a.keys + row_page(a, a.table[t / kRowPage], kvh) + (size_t)(t % kRowPage) * step + 4 * (lane & 7);
        lo[i] = *reinterpret_cast<const float4*>(src);
        hi[i] = *reinterpret_cast<const float4*>(src + 32);
    }
    auto turn = [&](const float4 (&raw)[8], float4 (&k)[8]) {
#pragma unroll
        for (int i = 0; i < 8; ++i)
            *reinterpret_cast<float4*>(tile + (8 * i + (lane >> 3)) * kTilePad + 4 * (lane & 7)) = raw[i];
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int j = 0; j < 8; ++j) k[j] = *reinterpret_cast<const float4*>(tile + lane * kTilePad + 4 * j);
        __builtin_amdgcn_wave_barrier();
    };
    float4 k[8];
    turn(lo, k);
    fn(0, k);
    turn(hi, k);
    fn(1, k);
}

// s += q . k over 32 dims, in order.
__device__ __forceinline__ float dot_half(const float* q, const float4 (&k)[8], float s) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const float4 v = *reinterpret_cast<const float4*>(q + 4 * j);
        s = s + v.x * k[j].x;
        s = s + v.y * k[j].y;
        s = s + v.z * k[j].z;
        s = s + v.w * k[j].w;
    }
    return s;
}

// s_t of a KV head's query heads into a.scores: grid (256-token chunks, KV
// heads), a wavefront per 64 tokens.
template <int G>
__global__ __launch_bounds__(kScoreThreads) void attention_row_scores_kernel(RowArgs a) {
    __shared__ __align__(16) float tile_s[kScoreThreads / kWave][64 * kTilePad];
    __shared__ __align__(16) float q_s[G * kRowDim];
    const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave, kvh = blockIdx.y;
    for (int i = threadIdx.x; i < G * kRowDim; i += kScoreThreads) q_s[i] = a.q[(size_t)kvh * G * kRowDim + i];
    __syncthreads();
    const int t0 = blockIdx.x * kScoreThreads + wave * 64;
    if (t0 >= a.length) return;
    float s[G];
#pragma unroll
    for (int h = 0; h < G; ++h) s[h] = 0.0f;
    key_rows(a, kvh, t0, tile_s[wave], [&](int half, const float4 (&k)[8]) {
#pragma unroll
        for (int h = 0; h < G; ++h) s[h] = dot_half(q_s + h * kRowDim + 32 * half, k, s[h]);
    });
    const int stride = (a.length + 15) & ~15;
    if (t0 + lane < a.length)
#pragma unroll
        for (int h = 0; h < G; ++h) a.scores[(size_t)(kvh * G + h) * stride + t0 + lane] = s[h] / sqrtf((float)kRowDim);
}

// Orders this wavefront's LDS accesses before the barrier; global loads stay
// in flight.
__device__ __forceinline__ void lds_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xC07F);  // vmcnt 63, expcnt 7, lgkmcnt 0
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

__global__ __launch_bounds__(kRowThreads) void attention_row_kernel(RowArgs a) {
    // Scores in the kernel: a K tile per wavefront; later the products of two
    // phases: [phase parity][page][dim][token].
    constexpr int kTiles = kRowWaves * 64 * kTilePad, kPageRing = kSlice * kRingPad;
    constexpr int kRing = 2 * kPhasePages * kPageRing;
    __shared__ __align__(16) float work_s[kTiles > kRing ? kTiles : kRing];
    __shared__ __align__(16) float e_s[kRowWindow];  // s_t, e_t, then p_t of the window
    __shared__ int32_t table_s[kRowWindow / kRowPage];
    __shared__ __align__(16) float q_s[kRowDim];
    __shared__ uint64_t exp_tab[32];
    __shared__ float reduce_s[kRowWaves];
    __shared__ float den_s;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int head = blockIdx.x / (kRowDim / kSlice), d0 = blockIdx.x % (kRowDim / kSlice) * kSlice;
    const int kvh = head / (a.heads / a.kv_heads);
    const int length = a.length;
    const bool one_window = length <= kRowWindow;
    const float* scores = a.scores ? a.scores + (size_t)head * ((length + 15) & ~15) : nullptr;
    // This thread's tokens of window [u0, u0 + n): u0 + tid + 512 j.
    float held[kRowHeld];
    auto hold = [&](const float* src, int n) {
#pragma unroll
        for (int j = 0; j < kRowHeld; ++j)
            if (kRowThreads * j < n) held[j] = src[min(kRowThreads * j + tid, n - 1)];
    };
    auto load_table = [&](int u0, int n) {
        for (int i = tid; i < (n + kRowPage - 1) / kRowPage; i += kRowThreads) table_s[i] = a.table[u0 / kRowPage + i];
    };
    if (tid < 32) exp_tab[tid] = kExp2Table[tid];
    // m = max_t s_t (order-free). Without scratch the whole row fits the
    // window (the launcher's rule).
    float m = -INFINITY;
    auto raise = [&](int n) {
#pragma unroll
        for (int j = 0; j < kRowHeld; ++j)
            if (kRowThreads * j < n) m = fmaxf(m, held[j]);
    };
    if (scores) {
        for (int u0 = 0; u0 < length; u0 += kRowWindow) {
            const int n = min(kRowWindow, length - u0);
            hold(scores + u0, n);
            if (u0 == 0) load_table(0, n);
            raise(n);
        }
    } else {
        if (tid < kRowDim) q_s[tid] = a.q[(size_t)head * kRowDim + tid];
        load_table(0, length);
        __syncthreads();
        for (int t0 = wave * 64; t0 < length; t0 += kRowWaves * 64) {
            float s = 0.0f;
            key_rows(a, kvh, t0, work_s + wave * 64 * kTilePad,
                     [&](int half, const float4 (&k)[8]) { s = dot_half(q_s + 32 * half, k, s); });
            if (t0 + lane < length) e_s[t0 + lane] = s / sqrtf((float)kRowDim);
        }
        __syncthreads();
        hold(e_s, length);
        raise(length);
    }
    for (int o = kWave / 2; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
    if (lane == 0) reduce_s[wave] = m;
    __syncthreads();
    m = reduce_s[0];
#pragma unroll
    for (int i = 1; i < kRowWaves; ++i) m = fmaxf(m, reduce_s[i]);
    // e_t of the window's tokens [u0, u0 + n) into e_s, zeros up to a whole page.
    auto stage = [&](int u0, int n) {
        if (!one_window) hold(scores + u0, n);
#pragma unroll
        for (int j = 0; j < kRowHeld; ++j) {
            const int t = kRowThreads * j + tid;
            if (kRowThreads * j < n && t < ((n + 15) & ~15))
                e_s[t] = t < n ? ref_expf_select(held[j] - m, exp_tab) : 0.0f;
        }
    };
    float den = 0.0f;
    for (int u0 = 0; u0 < length; u0 += kRowWindow) {
        const int n = min(kRowWindow, length - u0);
        stage(u0, n);
        __syncthreads();
        if (wave == 0) den = ordered_sum(e_s, n, den);
        __syncthreads();
    }
    if (tid == 0) den_s = den;
    const size_t step = (size_t)kRowDim * a.kv_heads;
    float total = 0.0f;  // the consumer's chain, lane % 16 = d - d0
    for (int u0 = 0; u0 < length; u0 += kRowWindow) {
        const int n = min(kRowWindow, length - u0), pages = (n + kRowPage - 1) / kRowPage;
        if (!one_window) {
            stage(u0, n);
            load_table(u0, n);
        }
        __syncthreads();
        const float dn = den_s;
        // Whole turns of kAhead phases, so that every turn issues the same
        // loads and each wait counts the later ones; phases past the last
        // page hand over nothing.
        const int phases = (pages + kPhasePages - 1) / kPhasePages;
        const int turns = (phases + kAhead - 1) / kAhead;
        // Producer w - 1 takes pages phase * kPhasePages + kPerPhase * (w - 1)
        // + {0, 1} of the window; lane = (token, 4 dims).
        const int slot = lane >> 2;
        float4 v[kAhead][kPerPhase];
        auto load = [&](int phase, float4 (&d)[kPerPhase]) {
#pragma unroll
            for (int i = 0; i < kPerPhase; ++i) {
                const int page = min(phase * kPhasePages + kPerPhase * (wave - 1) + i, pages - 1);
                const int at = min(slot, n - 1 - page * kRowPage);  // no slot past the row's end is read
                d[i] = *reinterpret_cast<const float4*>(
                    a.values + row_page(a, __builtin_amdgcn_readfirstlane(table_s[page]), kvh) + (size_t)at * step + d0 +
                    4 * (lane & 3));
            }
        };
        if (wave > 0)
#pragma unroll
            for (int i = 0; i < kAhead; ++i) load(i, v[i]);
        // p_t = e_t / den
        for (int t = tid; t < pages * kRowPage; t += kRowThreads) e_s[t] = e_s[t] / dn;
        lds_barrier();
        // The products of phase ph are formed while those of phase ph - 1
        // are added; a barrier after each.
        if (wave > 0) {
            for (int turn = 0; turn < turns; ++turn) {
#pragma unroll
                for (int k = 0; k < kAhead; ++k) {
                    const int ph = turn * kAhead + k;
#pragma unroll
                    for (int i = 0; i < kPerPhase; ++i) {
                        const int in_phase = kPerPhase * (wave - 1) + i, t = (ph * kPhasePages + in_phase) * kRowPage + slot;
                        const float p = e_s[min(t, kRowWindow - 1)];
                        const float4 x = v[k][i];
                        // Past the row's end +0: the chain starts at +0, so it
                        // never is -0, and adding +0 leaves it as it is.
                        const bool in = t < n;
                        float* dst = work_s + ((ph & 1) * kPhasePages + in_phase) * kPageRing + 4 * (lane & 3) * kRingPad + slot;
                        dst[0] = in ? p * x.x : 0.0f;
                        dst[kRingPad] = in ? p * x.y : 0.0f;
                        dst[2 * kRingPad] = in ? p * x.z : 0.0f;
                        dst[3 * kRingPad] = in ? p * x.w : 0.0f;
                    }
                    load(ph + kAhead, v[k]);
                    lds_barrier();
                }
            }
        } else {
            __builtin_amdgcn_s_setprio(3);
            for (int ph = 0; ph < turns * kAhead; ++ph) {
                lds_barrier();
                // The phase's products, two pages in flight; past the last
                // page they are zeros.
                const float4* src = reinterpret_cast<const float4*>(work_s + (ph & 1) * kPhasePages * kPageRing +
                                                                    (lane & 15) * kRingPad);
                float4 x[2][4];
                auto read = [&](int w, float4 (&y)[4]) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) y[j] = src[w * (kPageRing / 4) + j];
                };
                if (ph * kPhasePages >= pages) continue;
                read(0, x[0]);
#pragma unroll
                for (int w = 0; w < kPhasePages; ++w) {
                    if (w + 1 < kPhasePages) read(w + 1, x[(w + 1) & 1]);
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        total = total + x[w & 1][j].x;
                        total = total + x[w & 1][j].y;
                        total = total + x[w & 1][j].z;
                        total = total + x[w & 1][j].w;
                    }
                }
            }
            __builtin_amdgcn_s_setprio(0);
        }
        __syncthreads();  // the next window rewrites e_s, table_s and the ring
    }
    if (wave == 0 && lane < kSlice) a.out[(size_t)head * kRowDim + d0 + lane] = total;
}

template <int G>
void launch_row(hipStream_t s, const RowArgs& a) {
    // In the row kernel the scores take 3.1 us at 64 tokens, 7.2 at 503 and
    // 12.2 at 1,024; read from the scratch 1.6 us after a launch of 6 to 7.5.
    if (a.scores)
        attention_row_scores_kernel<G><<<dim3((a.length + kScoreThreads - 1) / kScoreThreads, a.kv_heads), kScoreThreads, 0, s>>>(a);
    attention_row_kernel<<<a.heads * (kRowDim / kSlice), kRowThreads, 0, s>>>(a);
}

}  // namespace

hipError_t launch_attention_single(hipStream_t s, const float* q, const float* keys,
                                   const float* values, const int32_t* table, int length,
                                   int layer, int layers, int block_tokens, int heads,
                                   int kv_heads, int dim, float* out, float* scratch) {
    if (heads / kv_heads > kMaxGroup || dim > kMaxDim || dim % 4) return hipErrorInvalidValue;
    // The row kernel's work-groups of one head read the whole head's q and each
    // writes its own dims of out, so where the scores are formed there and out
    // lies over q, one would read what another has written. attention_single's
    // work-group reads its heads' q before it writes them, and no other
    // work-group touches them: such calls take it.
    const size_t width = (size_t)heads * dim;
    const bool over_q = (uintptr_t)out < (uintptr_t)(q + width) && (uintptr_t)q < (uintptr_t)(out + width);
    // The row kernel reads V in 16-byte pieces, the general kernel by floats.
    const bool aligned = (uintptr_t)values % 16 == 0;
    if (block_tokens == kRowPage && dim == kRowDim && aligned &&
        (scratch || (length <= kRowWindow && !over_q && attention_row_pays(heads, kv_heads, length)))) {
        const RowArgs a{q, keys, values, table, length, layer, layers, heads, kv_heads, out, scratch};
        switch (heads / kv_heads) {
        case 1: launch_row<1>(s, a); break;
        case 2: launch_row<2>(s, a); break;
        case 3: launch_row<3>(s, a); break;
        case 4: launch_row<4>(s, a); break;
        case 5: launch_row<5>(s, a); break;
        case 6: launch_row<6>(s, a); break;
        case 7: launch_row<7>(s, a); break;
        default: launch_row<8>(s, a); break;
        }
        return hipGetLastError();
    }
    const dim3 grid(1, kv_heads);
    if (block_tokens == 16)
        attention_single_kernel<16><<<grid, kAttentionThreads, 0, s>>>(q, keys, values, table, length, layer, layers, block_tokens, heads, kv_heads, dim, out, scratch);
    else
        attention_single_kernel<0><<<grid, kAttentionThreads, 0, s>>>(q, keys, values, table, length, layer, layers, block_tokens, heads, kv_heads, dim, out, scratch);
    return hipGetLastError();
}


}  // namespace mphip
