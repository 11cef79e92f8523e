// Prefill attention of the fast arithmetic mode on FP32 matrix cores
// (v_mfma_f32_16x16x4f32): for a block of up to 16 consecutive rows of one
// sequence's chunk and one KV head, the query heads' scores against each
// 16-token page and the weighted sum of its values, with a reference maximum
// (raised only when a score exceeds it by more than 16) and a denominator
// per row (flash attention). The reference computes each
// (row, head) with an explicit two-pass softmax and sequential sums
// (llama_runner.cpp:85-93); the order of the floating-point sums differs
// here, and a row's result depends only on the row (its query and keys),
// not on the block, the chunking, the batch or the heads computed beside it.
//
// One work-group per (work item, run of HG of the KV head's G query heads):
// wavefront w of eight walks pages w, w + 8, ... with its own running maxima
// and sums, and the eight results are combined in order through LDS. The
// page-to-wavefront map depends only on the page, so the order of the sums
// is a function of the row.
//
// Per wavefront and page both products are taken transposed, so that a
// lane's results all belong to one row. MFMA operand layout (gfx950): lane l
// supplies A[l%16][l/16] and B[l/16][l%16]; result register i of lane l is
// D[4(l/16)+i][l%16]. With c = l%16 and g = l/16:
//  - S^T = K Q^T: the contraction step (jj, e) takes dims 16jj + 4g + e, so
//    lane (c, g) feeds A from component e of the float4 K[key c][16jj+4g..]
//    and B from Q[row c][16jj+4g+e]: K is four 16-byte loads per lane, each
//    1 KB contiguous in the page's key order [d/4][slot][4]. Register i
//    returns S[row c][key 4g+i];
//  - p = exp(s - reference) in those registers: row c's maximum, sum and
//    rescaling are lane-local (the four lanes of a row meet only when a
//    maximum is raised, and at the end);
//  - O^T += V^T P^T: contraction step e takes keys 4g + e, so B is the
//    lane's own p register e, and A component e of the float4
//    V[keys 4g..4g+3][dim 16n+c] (four 16-byte loads in the page's value
//    order [slot/4][d][4]). Register i returns O[row c][dim 16n+4g+i].
// P never leaves its registers (no LDS in the page loop), and a page is 8
// loads instead of 32 four-byte ones; the next page's are in flight during
// this page's 32 HG MFMAs. Against four wavefronts of all heads with P through
// LDS and four-byte loads: 45.7 -> 13.4 us for 256 rows at position 768 (48
// items), 795 -> 656 us for 8 x 512 rows at position 8,192 (79.7 GFLOP: 0.77
// of the FP32 matrix peak).
// Keys past the row's position are masked; keys past the block's last
// position (the rest of the last page) are masked for every row and their
// values taken as zero, so stale slots take no part, whatever they hold.
#include "kernels.h"
#include "lanes.h"
#include "layout.h"

// The fast mode's own summation order: multiply-adds may be fused.
#pragma clang fp contract(fast)

namespace mphip {
namespace {

constexpr int kDim = 64;
constexpr int kPage = 16;
constexpr int kWaves = 8;  // wavefronts (= page streams) per work item, two per SIMD
// Work items up to which every one of two or three query heads has a
// work-group of its own: with few items the launch is bound by one
// work-group's walk over its pages (an idle chip), beyond by the matrix cores,
// and then one K/V load serves all heads. Apart against together with three
// heads: 73 vs 85 us at 384 items of about 1,300 tokens, 91 vs 92 at 480, 138
// vs 137 at 768, and 322 vs 303 on average over 768 items of up to 8,700
// tokens. With two (whole one-layer steps): 98 vs 126 at 64 items of 3,200
// tokens, 244 vs 245 at 512, 336 vs 339 at 768. Four heads are always apart:
// in pairs 269 vs 264 at 384 items of 1,500 tokens, 572 vs 557 at 1,024, 865
// vs 844 at 1,024 of 3,500; together 570 and 826 at the last two, but 281 at
// the first and 408 vs 367 at 384 of 3,500.
constexpr int kSplitItems = 512;
constexpr float kScale = 0.125f;  // 1/sqrt(64)
constexpr float kRescale = 16.0f;  // probabilities stay below e^16 before a rescale

typedef float f4 __attribute__((ext_vector_type(4)));

// Of the four lanes (c, 0..3) of a row: the same value in each.
__device__ __forceinline__ float row4_max(float v) {
    v = fmaxf(v, __shfl_xor(v, 16));
    return fmaxf(v, __shfl_xor(v, 32));
}
__device__ __forceinline__ float row4_sum(float v) {
    v += __shfl_xor(v, 16);
    return v + __shfl_xor(v, 32);
}

template <int G, int HG>
__global__ __launch_bounds__(kWaves * 64, 2) void fast_prefill_kernel(const float* __restrict__ qkv, int ldq,
                                                                      PagedKv kv, int layer,
                                                                      const int4* __restrict__ items, int count,
                                                                      int kv_heads, float* __restrict__ out, int ldo) {
    static_assert(G % HG == 0, "equal runs of heads");
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // Per wavefront: its output tiles (as held per lane), and per row the
    // reference maximum and denominator.
    __shared__ f4 o_s[kWaves][HG][4][64];
    __shared__ float2 ml_s[kWaves][HG][kPage];
    const int index = blockIdx.x / (G / HG), h0 = (blockIdx.x % (G / HG)) * HG;  // uniform per work-group
    if (index >= count) return;
    const int4 item = items[index];
    const int row0 = item.x, kvh = item.y % kv_heads, pos0 = item.z, nrows = item.w;
    const int32_t* table = kv.tables + (size_t)(item.y / kv_heads) * kv.table_stride;
    const int last = pos0 + nrows - 1;  // the block's last position
    const int pages = last / kPage + 1;
    const int c = lane & 15, g = lane >> 4;
    const int qrow = row0 + min(c, nrows - 1), qpos = min(pos0 + c, last);
    const int head0 = kvh * G + h0;
    const size_t head_base = (size_t)kvh * kPage * kDim + 4 * lane;
    auto load = [&](int block, f4 (&k)[4], f4 (&v)[4]) {
        const size_t base = kv_page_base(block, layer, kv.layers, kPage, kv.kv_width) + head_base;
#pragma unroll
        for (int j = 0; j < 4; ++j) k[j] = *reinterpret_cast<const f4*>(kv.keys + base + 256 * j);
        // Value float4 (slot group g, dim 16n + c).
        const size_t vbase = base - 4 * lane + 256 * g + 4 * c;
#pragma unroll
        for (int n = 0; n < 4; ++n) v[n] = *reinterpret_cast<const f4*>(kv.values + vbase + 64 * n);
    };
    f4 kn[4], vn[4];  // the next page
    int next_block = table[min(wave, pages - 1)];
    load(next_block, kn, vn);
    next_block = table[min(wave + kWaves, pages - 1)];
    // Q of row c, scaled by 1/8: q[h][jj] holds dims 16jj + 4g .. +3.
    f4 q[HG][4];
#pragma unroll
    for (int h = 0; h < HG; ++h)
#pragma unroll
        for (int j = 0; j < 4; ++j)
            q[h][j] = *reinterpret_cast<const f4*>(qkv + quad_index(qrow, (head0 + h) * kDim + 16 * j + 4 * g, ldq)) *
                      kScale;
    f4 o[HG][4];
    // Row c: running maximum, the value subtracted in the exponent (the
    // maximum, 0 while that is -inf), this lane's share of the sum.
    float mx[HG], rf[HG], ls[HG];
#pragma unroll
    for (int h = 0; h < HG; ++h) {
#pragma unroll
        for (int n = 0; n < 4; ++n) o[h][n] = f4{0.f, 0.f, 0.f, 0.f};
        mx[h] = -__builtin_inff();
        rf[h] = 0.0f;
        ls[h] = 0.0f;
    }
    // Page p goes to wavefront p % kWaves, whatever the block.
    for (int p = wave; p < pages; p += kWaves) {
        f4 k[4], v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            k[j] = kn[j];
            v[j] = vn[j];
        }
        if (p + kWaves < pages) {
            load(next_block, kn, vn);
            next_block = table[min(p + 2 * kWaves, pages - 1)];
        }
        if (p == pages - 1) {
            // Value slots past the block's last position: zero.
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (p * kPage + 4 * g + e > last)
#pragma unroll
                    for (int n = 0; n < 4; ++n) v[n][e] = 0.0f;
        }
        f4 s[HG];
#pragma unroll
        for (int h = 0; h < HG; ++h) s[h] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int h = 0; h < HG; ++h)
                    s[h] = __builtin_amdgcn_mfma_f32_16x16x4f32(k[j][e], q[h][j][e], s[h], 0, 0, 0);
        if (p * kPage + kPage - 1 > pos0) {  // some row's position lies before the page's end
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (p * kPage + 4 * g + i > qpos)
#pragma unroll
                    for (int h = 0; h < HG; ++h) s[h][i] = -__builtin_inff();
        }
        // Per row a reference maximum, raised (and the sums rescaled) only
        // when one of the row's scores exceeds it by more than kRescale, so
        // the probabilities stay below e^16 and most pages need no row
        // maximum at all. A row with no unmasked key yet in this wavefront's
        // pages keeps maximum -inf and sums 0. Each row's raises depend on
        // its own scores only.
        float pm[HG];
        bool need = false;
#pragma unroll
        for (int h = 0; h < HG; ++h) {
            pm[h] = fmaxf(fmaxf(s[h][0], s[h][1]), fmaxf(s[h][2], s[h][3]));
            need |= pm[h] > mx[h] + kRescale;
        }
        if (__builtin_amdgcn_ballot_w64(need)) {
#pragma unroll
            for (int h = 0; h < HG; ++h) {
                const float m = row4_max(pm[h]);
                if (m > mx[h] + kRescale) {  // the same in the row's four lanes
                    const float keep = __expf(mx[h] - m);  // 0 from maximum -inf
                    ls[h] *= keep;
#pragma unroll
                    for (int n = 0; n < 4; ++n) o[h][n] *= keep;
                    mx[h] = m;
                    rf[h] = m;
                }
            }
        }
#pragma unroll
        for (int h = 0; h < HG; ++h)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                s[h][i] = __expf(s[h][i] - rf[h]);  // masked: 0
                ls[h] += s[h][i];
            }
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int n = 0; n < 4; ++n)
#pragma unroll
                for (int h = 0; h < HG; ++h)
                    o[h][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[n][e], s[h][e], o[h][n], 0, 0, 0);
    }
    // A wavefront without pages holds maximum -inf, sums 0 and outputs 0,
    // and takes no part below.
#pragma unroll
    for (int h = 0; h < HG; ++h) {
        const float l = row4_sum(ls[h]);
        if (g == 0) ml_s[wave][h][c] = make_float2(mx[h], l);
#pragma unroll
        for (int n = 0; n < 4; ++n) o_s[wave][h][n][lane] = o[h][n];
    }
    __syncthreads();
    // The eight results in order, the (head, 16 dims) tiles dealt to the
    // wavefronts.
    for (int t = wave; t < HG * 4; t += kWaves) {
        const int h = t >> 2, n = t & 3;
        float2 ml[kWaves];
#pragma unroll
        for (int w = 0; w < kWaves; ++w) ml[w] = ml_s[w][h][c];
        float m = ml[0].x;
#pragma unroll
        for (int w = 1; w < kWaves; ++w) m = fmaxf(m, ml[w].x);  // finite: page 0 is wave 0's
        f4 sum = {0.f, 0.f, 0.f, 0.f};
        float l = 0.0f;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
            const float f = __expf(ml[w].x - m);
            l += ml[w].y * f;
            sum += o_s[w][h][n][lane] * f;
        }
        if (c < nrows)
            *reinterpret_cast<f4*>(out + quad_index(row0 + c, (head0 + h) * kDim + 16 * n + 4 * g, ldo)) = sum / l;
    }
}

template <int G, int HG>
void launch(hipStream_t s, const float* qkv, int ldq, const PagedKv& kv, int layer, const int4* items, int count,
            int kv_heads, float* out, int ldo) {
    fast_prefill_kernel<G, HG><<<count * (G / HG), kWaves * 64, 0, s>>>(qkv, ldq, kv, layer, items, count, kv_heads,
                                                                        out, ldo);
}

}  // namespace

bool fast_prefill_fits(int heads, int kv_heads, const PagedKv& kv) {
    const int G = kv_heads > 0 ? heads / kv_heads : 0;
    return kv.block_tokens == kPage && kv.kv_width == kv_heads * kDim && G >= 1 && G <= 4 && G * kv_heads == heads;
}

hipError_t launch_fast_prefill(hipStream_t s, const float* qkv, int ldq, int heads, int kv_heads, const PagedKv& kv,
                               int layer, const int32_t* items, int count, float* out, int ldo) {
    if (count <= 0) return hipSuccess;
    if (!fast_prefill_fits(heads, kv_heads, kv)) return hipErrorInvalidValue;
    const int4* it = reinterpret_cast<const int4*>(items);
    const bool split = count <= kSplitItems;
    switch (heads / kv_heads) {
    case 1: launch<1, 1>(s, qkv, ldq, kv, layer, it, count, kv_heads, out, ldo); break;
    case 2:
        if (split) launch<2, 1>(s, qkv, ldq, kv, layer, it, count, kv_heads, out, ldo);
        else launch<2, 2>(s, qkv, ldq, kv, layer, it, count, kv_heads, out, ldo);
        break;
    case 3:
        if (split) launch<3, 1>(s, qkv, ldq, kv, layer, it, count, kv_heads, out, ldo);
        else launch<3, 3>(s, qkv, ldq, kv, layer, it, count, kv_heads, out, ldo);
        break;
    default: launch<4, 1>(s, qkv, ldq, kv, layer, it, count, kv_heads, out, ldo); break;
    }
    return hipGetLastError();
}

}  // namespace mphip
