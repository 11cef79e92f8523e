// The float sum of non-negative values added one by one in index order (the
// softmax denominator of the reference, llama_runner.cpp:89-91), bit for bit,
// by a whole wavefront.
//
// One lane's chain costs 6 cycles per value. It need not be a chain: while
// the running sum s stays in one binade [2^k, 2^(k+1)), s is an integer S of
// units u = ulp, and rounding s + e to nearest-even moves S by a whole number
// that depends on e and, where e lies exactly between two multiples of u, on
// the parity of S. So a run of values acts on S as S += (S odd ? d1 : d0).
// Lane l gets (d0, d1) of its kRun consecutive values from two chains of its
// own, started at 2^k (S even) and 2^k + u (S odd); such pairs compose
// associatively, and a scan over the lanes gives every prefix. That holds as
// long as S stays below 2^23 (the sums only grow, so the last one tells).
// Where a lane's run leaves the binade, the lanes before it are taken, the
// run itself is added value by value, and the next block starts behind it: at
// most one such step per doubling of the sum. The first kFirst values, over
// which a softmax's sum doubles most often, are added one by one, and so is
// everything while the sum is zero, denormal, infinite or NaN.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mphip {

constexpr int kOrderedRun = 16;     // values per lane and block
constexpr int kOrderedFirst = 256;  // values added one by one at the start

// Lane l's pair composed with that of lane l - N of its 16-lane row (of the
// lanes below N, with the identity).
template <int N>
__device__ __forceinline__ void ordered_compose(int& d0, int& d1) {
    const int a0 = __builtin_amdgcn_update_dpp(0, d0, 0x110 + N, 0xf, 0xf, false);
    const int a1 = __builtin_amdgcn_update_dpp(0, d1, 0x110 + N, 0xf, 0xf, false);
    const int c0 = a0 + ((a0 & 1) ? d1 : d0);
    const int c1 = a1 + ((a1 & 1) ? d0 : d1);  // S odd before: S + a1 is odd when a1 is even
    d0 = c0;
    d1 = c1;
}

// sum + v[0] + v[1] + ... + v[n-1] in this order; v is in LDS, 16-byte
// aligned, and v[n .. n rounded up to 4) are zeros. Every lane of the
// (whole) wavefront passes the same arguments and gets the result.
__device__ __forceinline__ float ordered_sum(const float* v, int n, float sum) {
    const float4* v4 = reinterpret_cast<const float4*>(v);
    const int n4 = (n + 3) >> 2;
    const int lane = threadIdx.x & 63;
    constexpr int kQuads = kOrderedRun / 4;
    constexpr int kTop = 1 << 23;
    auto in_order = [&](int from, int to) {  // quads [from, to) of v, one by one
        int i = from;
        for (; i + 4 <= to; i += 4) {
            float4 a[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) a[j] = v4[i + j];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                sum = sum + a[j].x;
                sum = sum + a[j].y;
                sum = sum + a[j].z;
                sum = sum + a[j].w;
            }
        }
        for (; i < to; ++i) {
            const float4 a = v4[i];
            sum = sum + a.x;
            sum = sum + a.y;
            sum = sum + a.z;
            sum = sum + a.w;
        }
    };
    int at = min(n4, sum == 0.0f ? kOrderedFirst / 4 : 0);
    in_order(0, at);
    while (at < n4) {  // uniform: `sum` and `at` are the same in every lane
        const int bits = __builtin_amdgcn_readfirstlane(__float_as_int(sum));
        const int exponent = bits >> 23 & 255;  // the sum is never negative, but a NaN may have its sign set
        if (exponent == 0 || exponent >= 255) {
            const int to = exponent ? n4 : min(n4, at + kOrderedFirst / 4);
            in_order(at, to);
            at = to;
            continue;
        }
        const int base = bits & 0x7f800000;
        float4 a[kQuads];
#pragma unroll
        for (int j = 0; j < kQuads; ++j) {
            const int q = at + lane * kQuads + j;
            a[j] = q < n4 ? v4[q] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        }
        float even = __int_as_float(base), odd = __int_as_float(base + 1);
#pragma unroll
        for (int j = 0; j < kQuads; ++j) {
            even = even + a[j].x;
            odd = odd + a[j].x;
            even = even + a[j].y;
            odd = odd + a[j].y;
            even = even + a[j].z;
            odd = odd + a[j].z;
            even = even + a[j].w;
            odd = odd + a[j].w;
        }
        // Clamped so that 64 of them stay in 32 bits; a lane's pair at the
        // clamp leaves the binade wherever it starts (NaN bits as well).
        int d0 = min(__float_as_int(even) - base, 2 * kTop), d1 = min(__float_as_int(odd) - (base + 1), 2 * kTop);
        if (even != even) d0 = d1 = 2 * kTop;
        ordered_compose<1>(d0, d1);
        ordered_compose<2>(d0, d1);
        ordered_compose<4>(d0, d1);
        ordered_compose<8>(d0, d1);
        // The four rows in order; S before row r.
        int s = bits - base, before = s;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            if ((lane >> 4) == r) before = s;
            const int r0 = __builtin_amdgcn_readlane(d0, 16 * r + 15), r1 = __builtin_amdgcn_readlane(d1, 16 * r + 15);
            s += (s & 1) ? r1 : r0;
        }
        if (s < kTop) {
            sum = __int_as_float(base + s);
            at += 64 * kQuads;
            continue;
        }
        const int after = before + ((before & 1) ? d1 : d0);
        const int first = __ffsll((unsigned long long)__builtin_amdgcn_ballot_w64(after >= kTop)) - 1;
        if (first > 0) sum = __int_as_float(base + __builtin_amdgcn_readlane(after, first - 1));
        const int from = at + first * kQuads, to = min(n4, from + kQuads);
        in_order(from, to);
        at = to;
    }
    return sum;
}

}  // namespace mphip
