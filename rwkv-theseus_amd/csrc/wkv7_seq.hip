// Step-serial WKV7 kernels for any head size 2..128 (the generic path: float32 token
// tensors, head sizes the chunked kernels do not cover, the exp decay mode).
//
// Every product is a plain float32 FMA, one step at a time.  What bounds a step is its
// dependency chain, not its arithmetic, so the state is spread thin: four keys of one value
// row per lane (G = NP/4 lanes share a row, NP = 32, 64 or 128 the padded head size), whose
// row sums are a few DPP adds, and 16 steps' vectors are staged in LDS at once, so the steps
// between two stagings run without a barrier.  (One lane per row, with the whole row in
// registers, a barrier per step and one wave per head, had taken 1.7 us a step.)
//
// Forward: value rows are independent, so a head's rows are split over workgroups.
//
// Backward: three passes, of which only the second is serial in time.
//  * The forward saved the state every CKPT steps.
//  * seq_grad_scan runs dL/dS alone backwards over time (rows independent, as the forward)
//    and keeps it at every CKPT-step segment's end, in the workspace.
//  * seq_backward forms each segment's gradients, all segments of all heads at once: it
//    replays the segment's 16 states into registers (4 floats per lane and step), then
//    steps dL/dS back through them.  Row sums (q, dv) are DPP adds; column sums (dr, dw, dk,
//    db, da) are added over the wave's rows by row swaps and over the waves through LDS, in
//    a fixed order, so results are deterministic (the reference uses fp32 atomicAdd,
//    kernels/wkv7_state.cu:68-72).
// Long sequences go through the last two in windows of segments (the workspace stays within
// kSeqWindowBytes); ds0 carries dL/dS from one window to the one before it.
//
// MODE picks the decay (MODE_RWKV / MODE_EXP, wkv7_common.h); `kv` != 0 means the
// caller's states (s0, sT, dsT, ds0) are stored [key][value] (GDN's layout) instead of
// [value][key].  Saved states always use [value][key].
#include "wkv7_common.h"
#include "wkv7_io.h"

#include <algorithm>
#include <type_traits>

namespace wkv7 {

// Sum over the G lanes that share a value row, left in all of them.
template <int G> __device__ __forceinline__ float row_lanes_sum(float x) {
    static_assert(G == 8 || G == 16 || G == 32, "lanes per row");
    if constexpr (G == 8) {
        x += dpp_move<0xb1>(x);
        x += dpp_move<0x4e>(x);
        return x + dpp_move<0x141>(x);  // (row_half_mirror: the other quad of the eight)
    } else {
        x = row_sum16(x);
        if constexpr (G == 32) {
            const uint32_t b = __float_as_uint(x);
            const auto p = __builtin_amdgcn_permlane16_swap(b, b, false, false);
            x = __uint_as_float(p[0]) + __uint_as_float(p[1]);
        }
        return x;
    }
}
// Row swaps that add two values over half the wave's rows each: of x and y, summed over the
// lane pairs 32 (16) apart, the lower lanes (even rows) get x's sum, the others y's.
__device__ __forceinline__ float fold32(float x, float y) {
    const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(y), false, false);
    return __uint_as_float(p[0]) + __uint_as_float(p[1]);
}
__device__ __forceinline__ float fold16(float x, float y) {
    const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(y), false, false);
    return __uint_as_float(p[0]) + __uint_as_float(p[1]);
}
__device__ __forceinline__ float dot4(const float (&s)[4], const float4& x) {
    return (s[0] * x.x + s[1] * x.y) + (s[2] * x.z + s[3] * x.w);
}
__device__ __forceinline__ float one_or(uint32_t m, float x) {  // x where the mask is set, else 1
    return __uint_as_float((__float_as_uint(x) & m) | (0x3f800000u & ~m));
}

// ---------------------------------------------------------------------------
// Forward: workgroup (head, block of RB value rows).
// ---------------------------------------------------------------------------
template <typename T, int NP, int MODE, int W>
__global__ __launch_bounds__(W) void seq_forward(
    int Tn, int H, int N, int kv, int bh0, int blocks, const T* __restrict__ r, const T* __restrict__ w,
    const T* __restrict__ k, const T* __restrict__ v, const T* __restrict__ a,
    const T* __restrict__ b, const float* s0, T* __restrict__ y,
    float* sT, float* __restrict__ ckpt) {
    constexpr int G = NP / 4, RB = W / G, M = CKPT * NP / W, MV = (CKPT * RB + W - 1) / W, YR = (CKPT + G - 1) / G;
    const int hd = blockIdx.x / blocks, bh = bh0 + hd, row0 = (blockIdx.x - hd * blocks) * RB;
    const int bb = bh / H, h = bh - bb * H, tid = threadIdx.x;
    const int kg = tid % G, rl = tid / G, i = row0 + rl, j0 = 4 * kg;
    const bool row = i < N;
    const long NN = (long)N * N, ncp = ckpt_count(Tn);
    __shared__ __attribute__((aligned(16))) float vec[2][5][CKPT][NP];  // r, d, k, a, b
    __shared__ float vrow[2][CKPT][RB];                                 // v of the block's rows

    // element (i, j) of a caller state: [value][key], or [key][value] when kv
    const long ei = kv ? 1 : N, ej = kv ? N : 1;
    float S[4];
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const bool ok = row && j0 + e < N;
        S[e] = keep(lane_mask(ok), s0[bh * NN + (ok ? i * ei + (j0 + e) * ej : 0)]);
    }
    // the 16 steps of a segment, loaded raw a segment ahead (clamped addresses, masked when
    // they go to LDS: steps past the end get d = 1 and zeros, which leave the state as it is,
    // with S a taken as zero there: an infinite state times a's zeros is not)
    float raw[5][M], rawv[MV];
    auto load = [&](int t0) {
#pragma unroll
        for (int m = 0; m < M; m++) {
            const int e = tid + W * m, u = e / NP, j = e % NP;
            const long o = ((long)(bb * (long)Tn + (t0 + u < Tn ? t0 + u : t0)) * H + h) * N + (j < N ? j : 0);
            raw[0][m] = io<T>::ld(r, o), raw[1][m] = io<T>::ld(w, o), raw[2][m] = io<T>::ld(k, o);
            raw[3][m] = io<T>::ld(a, o), raw[4][m] = io<T>::ld(b, o);
        }
#pragma unroll
        for (int m = 0; m < MV; m++) {
            const int e = tid + W * m, u = e / RB, ii = row0 + e % RB;
            rawv[m] = io<T>::ld(v, ((long)(bb * (long)Tn + (t0 + u < Tn && u < CKPT ? t0 + u : t0)) * H + h) * N +
                                       (ii < N ? ii : 0));
        }
    };
    auto stage = [&](int t0, int buf) {
#pragma unroll
        for (int m = 0; m < M; m++) {
            const int e = tid + W * m, u = e / NP, j = e % NP;
            const uint32_t ok = lane_mask(t0 + u < Tn && j < N);
            vec[buf][0][u][j] = keep(ok, raw[0][m]);
            vec[buf][1][u][j] = one_or(ok, decay_of<MODE>(raw[1][m]));
            vec[buf][2][u][j] = keep(ok, raw[2][m]);
            vec[buf][3][u][j] = keep(ok, raw[3][m]);
            vec[buf][4][u][j] = keep(ok, raw[4][m]);
        }
#pragma unroll
        for (int m = 0; m < MV; m++) {
            const int e = tid + W * m, u = e / RB, ii = e % RB;
            if (CKPT * RB % W == 0 || u < CKPT)
                vrow[buf][u][ii] = keep(lane_mask(t0 + u < Tn && row0 + ii < N), rawv[m]);
        }
    };
    auto save = [&](long c) {
#pragma unroll
        for (int e = 0; e < 4; e++)
            if (row && j0 + e < N) ckpt[(bh * ncp + c) * NN + (long)i * N + j0 + e] = S[e];
    };
    load(0);
    stage(0, 0);
    __syncthreads();
    for (int t0 = 0, buf = 0; t0 < Tn; t0 += CKPT, buf ^= 1) {
        const bool more = t0 + CKPT < Tn;
        if (more) load(t0 + CKPT);
        if (ckpt) save(t0 / CKPT);
        float ys[YR];
#pragma unroll
        for (int u = 0; u < CKPT; u++) {
            const float4 a4 = *reinterpret_cast<const float4*>(&vec[buf][3][u][j0]);
            const float4 d4 = *reinterpret_cast<const float4*>(&vec[buf][1][u][j0]);
            const float4 b4 = *reinterpret_cast<const float4*>(&vec[buf][4][u][j0]);
            const float4 k4 = *reinterpret_cast<const float4*>(&vec[buf][2][u][j0]);
            const float4 r4 = *reinterpret_cast<const float4*>(&vec[buf][0][u][j0]);
            const float vi = vrow[buf][u][rl];
            const float sa = keep(t0 + u < Tn ? ~0u : 0u, row_lanes_sum<G>(dot4(S, a4)));
            S[0] = S[0] * d4.x + (sa * b4.x + vi * k4.x);
            S[1] = S[1] * d4.y + (sa * b4.y + vi * k4.y);
            S[2] = S[2] * d4.z + (sa * b4.z + vi * k4.z);
            S[3] = S[3] * d4.w + (sa * b4.w + vi * k4.w);
            const float out = row_lanes_sum<G>(dot4(S, r4));
            // lane kg of the row keeps the outputs of steps kg, kg + G: one store per G steps
            if (u % G == 0) ys[u / G] = out;
            else ys[u / G] = kg == u % G ? out : ys[u / G];
        }
#pragma unroll
        for (int m = 0; m < YR; m++) {
            const int t = t0 + kg + G * m;
            if (row && kg + G * m < CKPT && t < Tn) io<T>::st(y, ((long)(bb * (long)Tn + t) * H + h) * N + i, ys[m]);
        }
        if (more) {
            stage(t0 + CKPT, buf ^ 1);  // (the other buffer: last read a segment ago, behind a barrier)
            __syncthreads();
        }
    }
    if (ckpt) save(ncp - 1);
#pragma unroll
    for (int e = 0; e < 4; e++)
        if (row && j0 + e < N) sT[bh * NN + i * ei + (j0 + e) * ej] = S[e];
}

// ---------------------------------------------------------------------------
// dL/dS alone, backwards over segments [c0, c1) (the last one first): gin -> gout, both in
// the caller's layout (gin may be null: zero), hbuf[bh][c - c0] = dL/dS at segment c's end
// ([NP][NP], padding included).  Workgroup (head, block of RB value rows).
// ---------------------------------------------------------------------------
template <typename T, int NP, int MODE, int W>
__global__ __launch_bounds__(W) void seq_grad_scan(
    int Tn, int H, int N, int kv, int bh0, int blocks, int c0, int c1, const T* __restrict__ r, const T* __restrict__ w,
    const T* __restrict__ a, const T* __restrict__ b, const T* __restrict__ dy, const float* gin, float* gout,
    float* __restrict__ hbuf) {
    constexpr int G = NP / 4, RB = W / G, M = CKPT * NP / W, MV = (CKPT * RB + W - 1) / W;
    const int hd = blockIdx.x / blocks, bh = bh0 + hd, row0 = (blockIdx.x - hd * blocks) * RB;
    const int bb = bh / H, h = bh - bb * H, tid = threadIdx.x;
    const int kg = tid % G, rl = tid / G, i = row0 + rl, j0 = 4 * kg;
    const bool row = i < N;
    const long NN = (long)N * N;
    __shared__ __attribute__((aligned(16))) float vec[2][4][CKPT][NP];  // r, d, a, b
    __shared__ float vrow[2][CKPT][RB];                                 // dy of the block's rows

    const long ei = kv ? 1 : N, ej = kv ? N : 1;
    float g[4] = {0.f, 0.f, 0.f, 0.f};
    if (gin) {
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const bool ok = row && j0 + e < N;
            g[e] = keep(lane_mask(ok), gin[bh * NN + (ok ? i * ei + (j0 + e) * ej : 0)]);
        }
    }
    float raw[4][M], rawv[MV];
    auto load = [&](int t0) {
#pragma unroll
        for (int m = 0; m < M; m++) {
            const int e = tid + W * m, u = e / NP, j = e % NP;
            const long o = ((long)(bb * (long)Tn + (t0 + u < Tn ? t0 + u : t0)) * H + h) * N + (j < N ? j : 0);
            raw[0][m] = io<T>::ld(r, o), raw[1][m] = io<T>::ld(w, o);
            raw[2][m] = io<T>::ld(a, o), raw[3][m] = io<T>::ld(b, o);
        }
#pragma unroll
        for (int m = 0; m < MV; m++) {
            const int e = tid + W * m, u = e / RB, ii = row0 + e % RB;
            rawv[m] = io<T>::ld(dy, ((long)(bb * (long)Tn + (t0 + u < Tn && u < CKPT ? t0 + u : t0)) * H + h) * N +
                                        (ii < N ? ii : 0));
        }
    };
    auto stage = [&](int t0, int buf) {
#pragma unroll
        for (int m = 0; m < M; m++) {
            const int e = tid + W * m, u = e / NP, j = e % NP;
            const uint32_t ok = lane_mask(t0 + u < Tn && j < N);
            vec[buf][0][u][j] = keep(ok, raw[0][m]);
            vec[buf][1][u][j] = one_or(ok, decay_of<MODE>(raw[1][m]));
            vec[buf][2][u][j] = keep(ok, raw[2][m]);
            vec[buf][3][u][j] = keep(ok, raw[3][m]);
        }
#pragma unroll
        for (int m = 0; m < MV; m++) {
            const int e = tid + W * m, u = e / RB, ii = e % RB;
            if (CKPT * RB % W == 0 || u < CKPT)
                vrow[buf][u][ii] = keep(lane_mask(t0 + u < Tn && row0 + ii < N), rawv[m]);
        }
    };
    load((c1 - 1) * CKPT);
    stage((c1 - 1) * CKPT, 0);
    __syncthreads();
    for (int c = c1 - 1, buf = 0; c >= c0; c--, buf ^= 1) {
        if (c > c0) load((c - 1) * CKPT);
        *reinterpret_cast<float4*>(hbuf + ((long)bh * (c1 - c0) + (c - c0)) * NP * NP + (long)i * NP + j0) =
            make_float4(g[0], g[1], g[2], g[3]);
#pragma unroll
        for (int u = CKPT - 1; u >= 0; u--) {
            const float4 r4 = *reinterpret_cast<const float4*>(&vec[buf][0][u][j0]);
            const float4 b4 = *reinterpret_cast<const float4*>(&vec[buf][3][u][j0]);
            const float4 d4 = *reinterpret_cast<const float4*>(&vec[buf][1][u][j0]);
            const float4 a4 = *reinterpret_cast<const float4*>(&vec[buf][2][u][j0]);
            const float dyi = vrow[buf][u][rl];
            g[0] += dyi * r4.x, g[1] += dyi * r4.y, g[2] += dyi * r4.z, g[3] += dyi * r4.w;
            const float q = keep(c * CKPT + u < Tn ? ~0u : 0u, row_lanes_sum<G>(dot4(g, b4)));  // (as the forward's S a)
            g[0] = g[0] * d4.x + q * a4.x;
            g[1] = g[1] * d4.y + q * a4.y;
            g[2] = g[2] * d4.z + q * a4.z;
            g[3] = g[3] * d4.w + q * a4.w;
        }
        if (c > c0) {
            stage((c - 1) * CKPT, buf ^ 1);
            __syncthreads();
        }
    }
#pragma unroll
    for (int e = 0; e < 4; e++)
        if (row && j0 + e < N) gout[bh * NN + i * ei + (j0 + e) * ej] = g[e];
}

// ---------------------------------------------------------------------------
// The gradients of segment c0 + blockIdx % nseg of head blockIdx / nseg, from the state at
// its start (saved) and dL/dS at its end (hbuf).  One workgroup holds RP = 4 W / NP value
// rows at a time (all of them up to NP = 64, 16 at 128: then PASSES row blocks in sequence,
// their column sums added in LDS).
// ---------------------------------------------------------------------------
// (NP = 128: 512 lanes, since the 128 registers of a 1024-lane workgroup spill there and its
// column sums would not fit LDS)
template <int NP> constexpr int seq_bwd_lanes() { return NP == 32 ? 256 : NP == 64 ? 1024 : 512; }
template <int NP> struct SeqBwdLds {
    static constexpr int W = seq_bwd_lanes<NP>(), WAVES = W / 64, RP = 4 * W / NP, PASSES = NP / RP;
    float r[CKPT][NP], d[CKPT][NP], f[CKPT][NP], k[CKPT][NP], a[CKPT][NP], b[CKPT][NP], dy[CKPT][NP], v[CKPT][NP];
    float sa[CKPT][RP];
    float part[2][WAVES][5 * NP];  // the waves' column sums of a step (double-buffered)
    float acc[PASSES > 1 ? CKPT : 1][PASSES > 1 ? 5 * NP : 1];
};
static_assert(sizeof(SeqBwdLds<32>) <= 163840 && sizeof(SeqBwdLds<64>) <= 163840 && sizeof(SeqBwdLds<128>) <= 163840,
              "LDS of a CU");
template <typename T, int NP, int MODE>
__global__ __launch_bounds__(seq_bwd_lanes<NP>()) void seq_backward(
    int Tn, int H, int N, int bh0, int c0, int nseg, const T* __restrict__ r, const T* __restrict__ w,
    const T* __restrict__ k, const T* __restrict__ v, const T* __restrict__ a,
    const T* __restrict__ b, const float* __restrict__ ckpt, const T* __restrict__ dy,
    T* __restrict__ dr, T* __restrict__ dw, T* __restrict__ dk, T* __restrict__ dv, T* __restrict__ da,
    T* __restrict__ db, const float* __restrict__ hbuf) {
    using Lds = SeqBwdLds<NP>;
    constexpr int W = Lds::W, G = NP / 4, RP = Lds::RP, PASSES = Lds::PASSES, WAVES = Lds::WAVES;
    constexpr int M = CKPT * NP / W, YR = (CKPT + G - 1) / G;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds_raw[];
    Lds& sm = *reinterpret_cast<Lds*>(lds_raw);
    const int hd = blockIdx.x / nseg, bh = bh0 + hd, cw = blockIdx.x - hd * nseg, c = c0 + cw;
    const int bb = bh / H, h = bh - bb * H, tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int kg = tid % G, rl = tid / G, j0 = 4 * kg, t0 = c * CKPT;
    const long NN = (long)N * N, ncp = ckpt_count(Tn);
    auto tok = [&](int u) { return ((long)(bb * (long)Tn + t0 + u) * H + h) * N; };
    {
        float x[8][M];
#pragma unroll
        for (int m = 0; m < M; m++) {
            const int e = tid + W * m, u = e / NP, j = e % NP;
            const long o = tok(t0 + u < Tn ? u : 0) + (j < N ? j : 0);
            x[0][m] = io<T>::ld(r, o), x[1][m] = io<T>::ld(w, o), x[2][m] = io<T>::ld(k, o), x[3][m] = io<T>::ld(a, o);
            x[4][m] = io<T>::ld(b, o), x[5][m] = io<T>::ld(dy, o), x[6][m] = io<T>::ld(v, o);
        }
#pragma unroll
        for (int m = 0; m < M; m++) {
            const int e = tid + W * m, u = e / NP, j = e % NP;
            const uint32_t ok = lane_mask(t0 + u < Tn && j < N);
            const float d = decay_of<MODE>(x[1][m]);
            sm.r[u][j] = keep(ok, x[0][m]);
            sm.d[u][j] = one_or(ok, d);
            sm.f[u][j] = keep(ok, dw_factor<MODE>(x[1][m], d));
            sm.k[u][j] = keep(ok, x[2][m]);
            sm.a[u][j] = keep(ok, x[3][m]);
            sm.b[u][j] = keep(ok, x[4][m]);
            sm.dy[u][j] = keep(ok, x[5][m]);
            sm.v[u][j] = keep(ok, x[6][m]);
        }
    }
    __syncthreads();
    // columns [5][NP] of a step (dr, dw, dk, db, da), summed over the waves by LW of them (2 of 4,
    // 5 of 16, all 8 at NP = 32, 64, 128) in turn; each column's lane is the same in every pass
    auto columns = [&](int u, int pass, const float (&part)[WAVES][5 * NP]) {
        constexpr int LW = 5 * NP / 64 > WAVES ? WAVES : 5 * NP / 64;  // waves at work per step
        const int first = (u * LW) % WAVES, slot = (wave - first + WAVES) % WAVES;
        if (slot >= LW) return;
        int ln = lane;  // (opaque: else every step's addresses are kept in registers over the passes)
        asm volatile("" : "+v"(ln));
        for (int col = 64 * slot + ln; col < 5 * NP; col += 64 * LW) {
            float s = 0.f;
#pragma unroll
            for (int x = 0; x < WAVES; x++) s += part[x][col];
            if constexpr (PASSES > 1) {
                if (pass > 0) s += sm.acc[u][col];
                if (pass + 1 < PASSES) {
                    sm.acc[u][col] = s;
                    continue;
                }
            }
            const int kind = col / NP, j = col % NP;
            if (j >= N || t0 + u >= Tn) continue;
            const long o = tok(u) + j;
            if (kind == 0) io<T>::st(dr, o, s);
            else if (kind == 1) io<T>::st(dw, o, s * sm.f[u][j]);
            else if (kind == 2) io<T>::st(dk, o, s);
            else if (kind == 3) io<T>::st(db, o, s);
            else io<T>::st(da, o, s);
        }
    };
#pragma unroll 1
    for (int pass = 0; pass < PASSES; pass++) {
        const int i = pass * RP + rl;
        const bool row = i < N;
        // (a wave whose rows straddle N: padded rows' products are masked, so that an
        // infinite input there -- zero times infinity -- adds nothing to the columns)
        const bool edge = __builtin_amdgcn_readfirstlane(pass * RP + (64 / G) * wave + 64 / G > N ? 1 : 0);
        const uint32_t rm = lane_mask(row);
        float S[CKPT + 1][4], g[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const bool ok = row && j0 + e < N;
            S[0][e] = keep(lane_mask(ok), ckpt[(bh * ncp + c) * NN + (ok ? (long)i * N + j0 + e : 0)]);
        }
        {
            const float4 x = *reinterpret_cast<const float4*>(hbuf + ((long)bh * nseg + cw) * NP * NP + (long)i * NP + j0);
            g[0] = x.x, g[1] = x.y, g[2] = x.z, g[3] = x.w;
        }
        // the segment's states
#pragma unroll
        for (int u = 0; u < CKPT; u++) {
            const float4 a4 = *reinterpret_cast<const float4*>(&sm.a[u][j0]);
            const float4 d4 = *reinterpret_cast<const float4*>(&sm.d[u][j0]);
            const float4 b4 = *reinterpret_cast<const float4*>(&sm.b[u][j0]);
            const float4 k4 = *reinterpret_cast<const float4*>(&sm.k[u][j0]);
            const float vi = sm.v[u][i];
            const float sa = row_lanes_sum<G>(dot4(S[u], a4));
            if (kg == 0) sm.sa[u][rl] = sa;  // (read back by this row's lanes only)
            S[u + 1][0] = S[u][0] * d4.x + (sa * b4.x + vi * k4.x);
            S[u + 1][1] = S[u][1] * d4.y + (sa * b4.y + vi * k4.y);
            S[u + 1][2] = S[u][2] * d4.z + (sa * b4.z + vi * k4.z);
            S[u + 1][3] = S[u][3] * d4.w + (sa * b4.w + vi * k4.w);
        }
        wave_lds_fence();
        // the adjoint, last step first
        float dvs[YR];
#pragma unroll
        for (int u = CKPT - 1; u >= 0; u--) {
            const float4 r4 = *reinterpret_cast<const float4*>(&sm.r[u][j0]);
            const float4 b4 = *reinterpret_cast<const float4*>(&sm.b[u][j0]);
            const float4 k4 = *reinterpret_cast<const float4*>(&sm.k[u][j0]);
            const float4 d4 = *reinterpret_cast<const float4*>(&sm.d[u][j0]);
            const float4 a4 = *reinterpret_cast<const float4*>(&sm.a[u][j0]);
            const float dyi = sm.dy[u][i], vi = sm.v[u][i], sa = sm.sa[u][rl];
            g[0] += dyi * r4.x, g[1] += dyi * r4.y, g[2] += dyi * r4.z, g[3] += dyi * r4.w;
            const float q = keep(t0 + u < Tn ? ~0u : 0u, row_lanes_sum<G>(dot4(g, b4)));  // (as seq_grad_scan's)
            const float dvi = row_lanes_sum<G>(dot4(g, k4));
            if (u % G == G - 1 || u == CKPT - 1) dvs[u / G] = dvi;
            else dvs[u / G] = kg == u % G ? dvi : dvs[u / G];
            float x[4][5];  // the row's part of dr, dw, dk, db, da of its four keys
#pragma unroll
            for (int e = 0; e < 4; e++) {
                x[e][0] = dyi * S[u + 1][e];
                x[e][1] = g[e] * S[u][e];
                x[e][2] = g[e] * vi;
                x[e][3] = g[e] * sa;
                x[e][4] = q * S[u][e];
            }
            if (edge) {
#pragma unroll
                for (int e = 0; e < 4; e++)
#pragma unroll
                    for (int n = 0; n < 5; n++) x[e][n] = keep(rm, x[e][n]);
            }
            float* const out = sm.part[u & 1][wave];
#pragma unroll
            for (int n = 0; n < 5; n++) {
                // over the rows of the wave's halves: lower lanes keep keys 0, 1, upper 2, 3
                const float p = fold32(x[0][n], x[2][n]), s = fold32(x[1][n], x[3][n]);
                const int up = 2 * (lane >> 5);
                if constexpr (G == 32) {
                    *reinterpret_cast<float2*>(&out[n * NP + j0 + up]) = make_float2(p, s);
                } else {
                    float z = fold16(p, s);  // even rows keep the first key of the two, odd rows the second
                    if constexpr (G == 8) z += dpp_move<0x128>(z);  // (row_ror:8: the row's two value rows)
                    out[n * NP + j0 + up + ((lane >> 4) & 1)] = z;
                }
            }
            g[0] = g[0] * d4.x + q * a4.x;
            g[1] = g[1] * d4.y + q * a4.y;
            g[2] = g[2] * d4.z + q * a4.z;
            g[3] = g[3] * d4.w + q * a4.w;
            // one barrier per step: a step's parts are summed while the next step writes the
            // other buffer, which everyone left before this barrier
            __syncthreads();
            columns(u, pass, sm.part[u & 1]);
        }
#pragma unroll
        for (int m = 0; m < YR; m++) {
            const int u = kg + G * m;
            if (row && u < CKPT && t0 + u < Tn) io<T>::st(dv, tok(u) + i, dvs[m]);
        }
    }
}

}  // namespace wkv7

// ---------------------------------------------------------------------------
// host launchers
// ---------------------------------------------------------------------------
#include "wkv7_launch.h"

namespace wkv7 {

namespace {

// dL/dS kept for at most this much at a time (at least one segment of every head)
constexpr size_t kSeqWindowBytes = (size_t)1 << 30;

int padded(int N) { return N <= 32 ? 32 : N <= 64 ? 64 : 128; }
int window_segments(int BH, int T, int N) {
    const size_t one = (size_t)BH * padded(N) * padded(N) * sizeof(float), fit = kSeqWindowBytes / one;
    const int nseg = (T + CKPT - 1) / CKPT;
    return fit < 1 ? 1 : fit < (size_t)nseg ? (int)fit : nseg;
}

// Lanes of a forward or scan workgroup: all of a head's rows (32 of 128) share one staging
// of the step vectors when there are heads enough to fill the chip that way; with few
// heads the rows go to four times as many smaller workgroups.
template <typename F> void by_width(int BH, int NP, F&& f) {
    if (NP > 32 && BH >= 256) f(std::integral_constant<int, 1024>());
    else f(std::integral_constant<int, 256>());
}
// f(first head, heads) in as few launches as the grid takes: at most 2^32 - 1 lanes along x.
template <typename F> void by_heads(int BH, int lanes_per_head, F&& f) {
    const unsigned most = 0xffffffffu / (unsigned)lanes_per_head;
    for (unsigned h = 0, n; h < (unsigned)BH; h += n) f((int)h, n = std::min((unsigned)BH - h, most));
}
template <typename F> void by_shape(int N, int dtype, int flags, F&& f) {
    auto mode = [&](auto t, auto np) {
        if (flags & FLAG_DECAY_EXP) f(t, np, std::integral_constant<int, MODE_EXP>());
        else f(t, np, std::integral_constant<int, MODE_RWKV>());
    };
    auto size = [&](auto t) {
        if (N <= 32) mode(t, std::integral_constant<int, 32>());
        else if (N <= 64) mode(t, std::integral_constant<int, 64>());
        else mode(t, std::integral_constant<int, 128>());
    };
    if (dtype == 0) size(bf16_t());
    else size(float());
}

}  // namespace

void launch_seq_forward(const Fwd& p) {
    by_shape(p.N, p.dtype, p.flags, [&](auto t, auto np, auto mode) {
        using T = decltype(t);
        constexpr int NP = decltype(np)::value, MODE = decltype(mode)::value;
        by_width(p.B * p.H, NP, [&](auto width) {
            constexpr int W = decltype(width)::value, WW = NP == 32 ? 256 : W, RB = 4 * WW / NP;
            const int blocks = (p.N + RB - 1) / RB;
            by_heads(p.B * p.H, blocks * WW, [&](int bh0, unsigned heads) {
                hipLaunchKernelGGL((seq_forward<T, NP, MODE, WW>), dim3(heads * blocks), dim3(WW), 0, p.stream, p.T,
                                   p.H, p.N, (p.flags & FLAG_STATE_KV) ? 1 : 0, bh0, blocks, (const T*)p.r,
                                   (const T*)p.w, (const T*)p.k, (const T*)p.v, (const T*)p.a, (const T*)p.b, p.s0,
                                   (T*)p.y, p.sT, p.ckpt);
            });
        });
    });
}

size_t seq_backward_workspace(int B, int T, int H, int N) {
    return (size_t)B * H * window_segments(B * H, T, N) * padded(N) * padded(N) * sizeof(float);
}

void launch_seq_backward(const Bwd& p) {
    by_shape(p.N, p.dtype, p.flags, [&](auto t, auto np, auto mode) {
        using T = decltype(t);
        constexpr int NP = decltype(np)::value, MODE = decltype(mode)::value;
        using Lds = SeqBwdLds<NP>;
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&seq_backward<T, NP, MODE>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)sizeof(Lds));
        const int BH = p.B * p.H, kv = (p.flags & FLAG_STATE_KV) ? 1 : 0;
        const int nseg = (p.T + CKPT - 1) / CKPT, win = window_segments(BH, p.T, p.N);
        for (int c1 = nseg; c1 > 0; c1 -= win) {
            const int c0 = c1 > win ? c1 - win : 0;
            by_width(BH, NP, [&](auto width) {
                constexpr int W = decltype(width)::value, WW = NP == 32 ? 256 : W, RB = 4 * WW / NP;
                // (every padded row runs: the segment kernel reads hbuf's padding too)
                const int blocks = NP / RB;
                by_heads(BH, blocks * WW, [&](int bh0, unsigned heads) {
                    hipLaunchKernelGGL((seq_grad_scan<T, NP, MODE, WW>), dim3(heads * blocks), dim3(WW), 0, p.stream,
                                       p.T, p.H, p.N, kv, bh0, blocks, c0, c1, (const T*)p.r, (const T*)p.w,
                                       (const T*)p.a, (const T*)p.b, (const T*)p.dy, c1 == nseg ? p.dsT : p.ds0,
                                       p.ds0, (float*)p.ws);
                });
            });
            by_heads(BH, (c1 - c0) * Lds::W, [&](int bh0, unsigned heads) {
                hipLaunchKernelGGL((seq_backward<T, NP, MODE>), dim3(heads * (c1 - c0)), dim3(Lds::W), sizeof(Lds),
                                   p.stream, p.T, p.H, p.N, bh0, c0, c1 - c0, (const T*)p.r, (const T*)p.w,
                                   (const T*)p.k, (const T*)p.v, (const T*)p.a, (const T*)p.b, p.ckpt, (const T*)p.dy,
                                   (T*)p.dr, (T*)p.dw, (T*)p.dk, (T*)p.dv, (T*)p.da, (T*)p.db, (const float*)p.ws);
            });
        }
    });
}

}  // namespace wkv7
