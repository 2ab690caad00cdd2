// The time split of the record scans (gdn_scan forward, wkv7_bwd_scan backward) when every
// chunk's state has to be stored.
//
// A scan's state after a chunk is affine in the state before it, X' = X M + U, and its
// value rows are independent, so a head's chunks form k segments (in the scan's order):
//  * the "ends" launch runs segment 0 from its true start, with its outputs, and segments
//    1 .. k-2 from zero and from the identity side by side, for their U_s and Phi_s alone;
//  * scan_chain forms X_{s+1} = X_s Phi_s + U_s for the segments' true starts;
//  * the "resume" launch runs segments 1 .. k-1 from those, with their outputs.
// A chunk is visited twice, which pays once the segments fill CUs that one workgroup per 64
// value rows of a head leaves idle (2 n / k ticks instead of n).
#pragma once

#include "wkv7_io.h"

namespace wkv7 {
namespace {

// The split's buffers (float32): X_1 [BH][N][N], U_s and Phi_s^T [][BH][N][N] for s >= 1
// (X_{s+1} replaces U_s), X and U [value][key].  y0, z: the no-saved-states split of gdn_scan.
struct ScanSplit {
    int m = 0, k = 0;  // chunks of each segment after the first, segments
    int m0 = 0;        // chunks of segment 0
    float *send0 = nullptr, *uend = nullptr, *phi = nullptr, *y0 = nullptr, *z = nullptr;
};
// X_s of segment s >= 1: X_1 in send0, X_s (s >= 2) in the U_{s-1} slot
__device__ __forceinline__ const float* seg_state(const ScanSplit& sp, int BH, int bh, int s, long NN) {
    return s == 1 ? sp.send0 + bh * NN : sp.uend + ((long)(s - 2) * BH + bh) * NN;
}

// x = h + m + l to float32's 24 bits (bf16 each), and the six products of two such operands
// that reach 2^-24 of the result.
struct Frag3 {
    uint4 h, m, l;
};
__device__ __forceinline__ void split3(float x0, float x1, uint32_t& h, uint32_t& m, uint32_t& l) {
    const uint32_t u0 = __float_as_uint(x0), u1 = __float_as_uint(x1);
    h = (u0 >> 16) | (u1 & 0xffff0000u);
    split2(x0 - __uint_as_float(u0 & 0xffff0000u), x1 - __uint_as_float(u1 & 0xffff0000u), m, l);
}
__device__ __forceinline__ Frag3 pack3(const float (&x)[8]) {
    Frag3 f;
    split3(x[0], x[1], f.h.x, f.m.x, f.l.x);
    split3(x[2], x[3], f.h.y, f.m.y, f.l.y);
    split3(x[4], x[5], f.h.z, f.m.z, f.l.z);
    split3(x[6], x[7], f.h.w, f.m.w, f.l.w);
    return f;
}
__device__ __forceinline__ f32x4_t mma3(f32x4_t acc, const Frag3& a, const Frag3& b) {
    acc = mma32(mma32(mma32(acc, a.l, b.h), a.h, b.l), a.m, b.m);
    return mma32(mma32(mma32(acc, a.m, b.h), a.h, b.m), a.h, b.h);
}

// X_{s+1} = X_s Phi_s + U_s, s = 1 .. steps, in place of U_s; after the last step also to
// sT when given ([key][value] when kv).  Workgroup (head, block of 16 value rows), one wave
// per key tile (X^T as the B operand from LDS, Phi^T as the A operand).  Every later segment
// starts from these states, so they are formed to float32 (three-way splits: two-way ones
// had put 2^-16 of X_s into each).  A step is a chain of latencies -- Phi's load, its split,
// KS x 6 MFMAs, an LDS turn -- so it is spread over N/16 x N/16 waves per head, Phi and U
// are loaded two steps ahead, and each wave splits its tile of X once for all of them.
template <int NK>
__global__ __launch_bounds__(4 * NK) void scan_chain(int BH, int steps, int kv, ScanSplit sp, float* __restrict__ sT) {
    constexpr int KS = NK / 32;
    __shared__ uint2 xs[2][3][KS][64][2];  // X's 16 rows, split, as the K=32 B operands
    const int bh = blockIdx.x, rb = blockIdx.y, tid = threadIdx.x;
    const int tj = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, q4 = lane >> 4, r16 = lane & 15;
    const long NN = (long)NK * NK, row = (long)(16 * rb + r16) * NK + 16 * tj + 4 * q4;
    struct Step {  // Phi_s[32ks + 4q4 + e (+16)][16tj + r16], U_s[16rb + r16][16tj + 4q4 ..]
        float4 p[KS][2], u;
    };
    auto load = [&](Step& x, int s) {
        const float* const P = sp.phi + ((long)(s - 1) * BH + bh) * NN + (long)(16 * tj + r16) * NK + 4 * q4;  // (transposed)
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            x.p[ks][0] = *reinterpret_cast<const float4*>(P + 32 * ks);
            x.p[ks][1] = *reinterpret_cast<const float4*>(P + 32 * ks + 16);
        }
        x.u = *reinterpret_cast<const float4*>(sp.uend + ((long)(s - 1) * BH + bh) * NN + row);
    };
    auto publish = [&](int buf, const float4& x) {  // X[16rb + r16][16tj + 4q4 ..] for every wave
        uint2 h, m, l;
        split3(x.x, x.y, h.x, m.x, l.x);
        split3(x.z, x.w, h.y, m.y, l.y);
        xs[buf][0][tj >> 1][lane][tj & 1] = h;
        xs[buf][1][tj >> 1][lane][tj & 1] = m;
        xs[buf][2][tj >> 1][lane][tj & 1] = l;
    };
    auto step = [&](const Step& c, int s) {
        f32x4_t acc = {c.u.x, c.u.y, c.u.z, c.u.w}, acc2 = zero4();
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            const float f[8] = {c.p[ks][0].x, c.p[ks][0].y, c.p[ks][0].z, c.p[ks][0].w,
                                c.p[ks][1].x, c.p[ks][1].y, c.p[ks][1].z, c.p[ks][1].w};
            const auto& x = xs[(s - 1) & 1];
            const Frag3 b = {cat(x[0][ks][lane][0], x[0][ks][lane][1]), cat(x[1][ks][lane][0], x[1][ks][lane][1]),
                             cat(x[2][ks][lane][0], x[2][ks][lane][1])};
            f32x4_t& t = ks & 1 ? acc2 : acc;  // (two chains)
            t = mma3(t, pack3(f), b);
        }
        acc += acc2;
        const float4 o = make_float4(acc[0], acc[1], acc[2], acc[3]);
        publish(s & 1, o);
        if (s < steps || !sT) {
            *reinterpret_cast<float4*>(sp.uend + ((long)(s - 1) * BH + bh) * NN + row) = o;
        } else if (!kv) {
            *reinterpret_cast<float4*>(sT + bh * NN + row) = o;
        } else {
#pragma unroll
            for (int e = 0; e < 4; e++) sT[bh * NN + (long)(16 * tj + 4 * q4 + e) * NK + 16 * rb + r16] = acc[e];
        }
        __syncthreads();
    };
    publish(0, *reinterpret_cast<const float4*>(sp.send0 + bh * NN + row));
    Step even, odd;  // (the even and the odd steps' operands)
    load(odd, 1);
    if (steps > 1) load(even, 2);
    __syncthreads();
    for (int s = 1; s <= steps; s += 2) {
        step(odd, s);
        if (s + 2 <= steps) load(odd, s + 2);
        if (s + 1 <= steps) {
            step(even, s + 1);
            if (s + 3 <= steps) load(even, s + 3);
        }
    }
}

// Workgroups per head and segment (each of N/16 waves / groups): all of a head's value rows in
// one when the segments fill the CUs that way (each workgroup moves the whole record into
// its LDS, so one group halves that traffic), else groups of 64 rows.
inline int scan_groups(long BH, int N, int segments, int cus) {
    return N / 64 > 1 && segments * BH * (N / 64) <= cus ? N / 64 : 1;
}
// Segments of the split with saved states (1: one pass), at most 9 of at least 4 chunks each:
// k - 1 workgroups per head and row group in each of its two launches, one per CU.  A split
// costs 2 n / k ticks, a chain of k - 2 steps and two more launches against n ticks, and its
// ticks are longer than one pass's: all of a head's rows in one workgroup where N/64 row groups
// per segment do not fit the CUs (128 keys: 4 to 5.5 us a tick against 2.2 with two groups,
// one pass 1.5 to 2), and more records and states through memory at once.  So at 128 keys it is
// cut as far as both row groups fit, and further only from 96 chunks on, where fewer chunks per
// segment weigh more.  Forward with saved states | backward, whole calls at B = 1 in us, one
// pass / k segments (MI355X, 256 CUs):
//   heads   16 chunks              24                     48                      64                      128
//    8      56/4: 53 | 59/4: 61    73/6: 61 | 73/6: 67    124/9: 83 | 123/9: 96   155/9: 86 | 149/9: 102  284/9: 124 | 279/9: 160
//    32     60/4: 60 | 77/4: 80    77/5: 68 | 105/5: 101  132/5: 103 | 187/5: 176 171/5: 126 | 249/5: 233 370/9: 240 | 481/9: 422
//    40     60/4: 68 | 90/4: 100   78/4: 88 | 118/4: 128  137/4: 127 | 218/4: 225 188/4: 168 | 290/4: 285 409/7: 293 | 562/7: 526
//    56     63/4: 87 | 106/4: 126  84/5: 100 | 147/5: 169 160/5: 167 | 278/5: 303 236/5: 210 | 365/5: 384 460/5: 372 | 703/5: 694
//    85     70/4: 104 | 142/4: 173 94/4: 135 | 206/4: 245 228/4: 228 | 385/4: 418 297/4: 287 | 501/4: 532 552/4: 533 | 932/4: 999
// (32 heads, 48 chunks: one group's 9 segments 116 | 191.)  The backward, whose own work beside
// the scan is larger, starts a little later.  The gated delta rule's calls lie within 3 % of
// these lines.  At 64 keys (one row group always, and calls of more than 28 chunks only) every
// split pays: 29 chunks 47/7: 36 | 43/7: 38 at 8 heads, 55/6: 47 | 69/6: 67 at 48.
inline int resume_segments(long BH, int N, int nchunk, int cus, bool back) {
    auto fit = [&](long groups) {
        const long k = cus / (groups * BH) + 1, m = k < 9 ? k : 9;
        return (int)(nchunk / 4 < m ? nchunk / 4 : m);
    };
    const int one = fit(1);  // with one workgroup per head and segment
    if (N == 64) return one >= 4 && nchunk > 28 ? one : 1;
    if (nchunk >= 96) return one >= (back ? 5 : 4) ? one : 1;
    const int all = fit(N / 64);  // with every row group
    const long room = cus / (N / 64 * BH) + 1;  // (before the chunks' and the most segments' limits)
    if (room >= 4) {
        const int from = room >= 9 ? 16 : room >= 5 ? 20 : 48;
        return all >= 4 && nchunk >= from + (back ? room == 4 ? 16 : 4 : 0) ? all : 1;
    }
    return !back && nchunk >= 64 && one >= 4 ? one : 1;
}
// Chunks of segment 0 and of each later one: the first launch takes max(m0, 4/3 m) ticks
// (two states on one record), the second m.
inline void resume_lengths(int n, int k, int& m0, int& m) {
    int best = 1 << 30;
    m0 = n, m = 0;
    for (int mm = 1; n - (k - 1) * mm >= 1; mm++) {
        const int r = n - (k - 1) * mm, a = 3 * r, b = 4 * mm, cost = (a > b ? a : b) + 3 * mm;
        if (cost < best) best = cost, m0 = r, m = mm;
    }
}
inline size_t resume_bytes(size_t BH, int N, int k) {
    return k < 2 ? 0 : BH * N * N * (1 + 2 * (size_t)(k - 2)) * sizeof(float);
}
inline ScanSplit resume_split(size_t BH, int N, int n, int k, float* base) {
    ScanSplit sp;
    const size_t NN = (size_t)N * N;
    sp.k = k;
    resume_lengths(n, k, sp.m0, sp.m);
    sp.send0 = base, sp.uend = base + BH * NN, sp.phi = sp.uend + (size_t)(k - 2) * BH * NN;
    return sp;
}

// A record's 1 KB fragment block: lane l's 16 bytes as two 8-byte halves 512 bytes apart (LDS
// serves 8-byte reads at twice the rate of 16-byte ones).
__device__ __forceinline__ void put_frag(uint8_t* blk, int lane, uint4 v) {
    reinterpret_cast<uint2*>(blk)[lane] = make_uint2(v.x, v.y);
    reinterpret_cast<uint2*>(blk)[64 + lane] = make_uint2(v.z, v.w);
}
__device__ __forceinline__ uint4 get_frag(const uint8_t* blk, int lane) {
    return cat(reinterpret_cast<const uint2*>(blk)[lane], reinterpret_cast<const uint2*>(blk)[64 + lane]);
}

// What a scan launch runs.
enum ScanMode {
    SCAN_ALL,     // every chunk of a head, in order
    SCAN_TILES,   // gdn_scan's split without saved states (all segments at once, y0 and z tiles)
    SCAN_ENDS,    // segments 0 .. k-2 of the split above
    SCAN_RESUME,  // segments 1 .. k-1
};

}  // namespace
}  // namespace wkv7
