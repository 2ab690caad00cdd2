// WKV7 backward (bf16, head size 128, and 64 with few heads) and the gated delta rule's (head
// size 128) on the matrix cores, every chunk at once.
//
// The chunk form of the recurrence (kernels/wkv7_state.cu:12-79; operands A~, R~, B-, K-,
// B^, K^, Aab, Aak, Brb, Brk, Ti, P, P2 as in wkv7_chunk_fwd.hip, decays per key) gives,
// with H = dL/dS at a chunk's end, H' = H diag(e^{gL}), S0 the state at its start (a
// saved state) and dY its output gradient,
//   SA = Ti (A~ S0^T + Aak V),  Q = Ti^T (B^ H^T + Brb^T dY)
//   dV = K^ H^T + Aak^T Q + Brk^T dY
//   dK = e^{-g} o [V H' + triu_s(V Q^T) A~ + triu(V dY^T) R~]
//   dB = e^{-g} o [SA H' + triu_s(SA Q^T) A~ + triu(SA dY^T) R~]
//   dR = e^{g}  o [dY S0 + tril(dY SA^T) B- + tril(dY V^T) K-]
//   dA = e^{gp} o [Q S0 + tril_s(Q SA^T) B- + tril_s(Q V^T) K-]
//   H at the chunk's start = H diag(e^{gL}) + (H B^^T) P + dY^T P2
// and the log-decay gradient dlogd_t = sum_{s>=t} (r dR - b dB - k dK)_s +
// sum_{s>t} (a dA)_s + colsum(H_end o S_end) over the chunk's own steps: the gradients of
// the steps up to a boundary are those of the sequence cut there with dL/dS_end = H_end,
// so the carry from every later step is the column sum of H_end o S_end at the chunk's
// end (S_end: the next saved state).  dw = dlogd * (-e^{-1/2}) sig(w) (1 - sig(w)).
// (Checked in float64 against the oracle's step adjoint before the kernels.)
//
// Three kernels.  wkv7_bwd_prep (one wave per chunk, all at once) writes each chunk's
// record for the scan: B^ as the K=32 A operand over the keys, [P | P2] per 16-key tile
// as the A operand of the K=32 update, e^{gL} per key.  wkv7_bwd_scan walks each head's
// chunks backwards (fp32 H in registers, one wave per 16 of its value rows; a workgroup holds
// 64 rows, or all of a head's where time segments fill the CUs that way; records
// double-buffered in LDS by DMA as gdn_scan's), storing H at every chunk's end in the
// workspace and the first chunk's start as ds0, in one pass or cut in time (wkv7_scan.h).
// wkv7_bwd_chunk then forms every chunk's gradients independently (N/16 waves; wave w owns
// value rows 16w..16w+15 for SA, Q, dV and keys 16w..16w+15 for dK, dB, dR, dA, dw), with the
// chunk's matrices from wkv7_bwd_prep (the gated delta rule's gdn_bwd_chunk forms its own).
#include "wkv7_launch.h"
#include "wkv7_scan.h"

namespace wkv7 {
namespace {

constexpr int BC = 16;        // chunk length
constexpr int BNK = 128;      // the gated delta rule's head size here
constexpr int BKS = BNK / 32, BTJ = BNK / 16;
constexpr long BNN = (long)BNK * BNK;

// One chunk's record for the scan (byte offsets).
template <int NK> struct BwdRec {
    static constexpr int KS = NK / 32, TJ = NK / 16;
    static constexpr size_t BF = 0;                               // B^ [KS][hi, lo][64 lanes] uint4
    static constexpr size_t PP = BF + (size_t)KS * 2 * 64 * 16;   // [P | P2] [TJ][hi, lo][64] uint4
    static constexpr size_t EL = PP + (size_t)TJ * 2 * 64 * 16;   // e^{gL} [NK]
    static constexpr size_t BYTES = EL + (size_t)NK * 4;
    static constexpr int DMA_BLOCKS = (int)((BYTES + 1023) / 1024);
};
static_assert(BwdRec<128>::BYTES % 256 == 0 && BwdRec<64>::BYTES % 256 == 0, "record alignment");

__device__ __forceinline__ f32x4_t mm3(f32x4_t acc, uint4 xh, uint4 xl, uint4 yh, uint4 yl) {
    return mma32(mma32(mma32(acc, xh, yh), xh, yl), xl, yh);
}
// M^T of a D-layout tile, by the product M^T I on the K=16 instruction (I exact in bf16)
__device__ __forceinline__ f32x4_t transpose16(const f32x4_t& m, int lane) {
    f32x4_t id;
#pragma unroll
    for (int e = 0; e < 4; e++) id[e] = (4 * (lane >> 4) + e) == (lane & 15) ? 1.f : 0.f;
    const Pk pm = pk(m), pi = pk(id);
    return mma16(mma16(zero4(), pm.h, pi.h), pm.l, pi.h);
}
__device__ __forceinline__ float bf2f(const bf16_t* p, long i) { return io<bf16_t>::ld(p, i); }

// The chunk's 16x16 matrices for wkv7_bwd_chunk, packed split pairs (uint4 per lane).
enum { MAT_AAKT, MAT_AAK, MAT_BRB, MAT_BRK, MAT_TI, MAT_TIT, MATS };

// ---------------------------------------------------------------------------
// Records of chunk blockIdx.x of head blockIdx.y (one wave; lane (q4, r16): token r16's
// keys 32ks + 4q4 + e and 32ks + 16 + 4q4 + e, planes and order as wkv7_rec_prep).  Bound by
// its bytes (4 lanes of 2048 tokens, 32 heads of 128: 850 MB, 167 us at the rate of a copy;
// measured 185).
// ---------------------------------------------------------------------------
template <int NK>
__global__ __launch_bounds__(64, NK == 64 ? 4 : 3) void wkv7_bwd_prep(int Tn, int H, const bf16_t* __restrict__ r,
                                                    const bf16_t* __restrict__ w, const bf16_t* __restrict__ k,
                                                    const bf16_t* __restrict__ a, const bf16_t* __restrict__ b,
                                                    uint8_t* __restrict__ ws, uint4* __restrict__ mats) {
    using R = BwdRec<NK>;
    constexpr int KS = R::KS;
    constexpr int LA = NK + 20, LB = 36;  // rows (bf16) that spread over the banks
    const int c = blockIdx.x, bh = blockIdx.y, nchunk = gridDim.x;
    const int bb = bh / H, h = bh - bb * H;
    const int lane = threadIdx.x, q4 = lane >> 4, r16 = lane & 15;
    const int t0 = c * BC, L = min(BC, Tn - t0);
    const bool tv = r16 < L;
    const long row = (((long)bb * Tn + t0 + (tv ? r16 : 0)) * H + h) * (long)NK;  // (clamped: read by every lane)
    const uint32_t tm = lane_mask(tv);
    __shared__ __attribute__((aligned(16))) uint16_t pa[2][BC][LA], pb[2][BC][LB];  // hi, lo
    uint8_t* const rec = ws + ((size_t)bh * nchunk + c) * R::BYTES;
    auto ld8 = [&](const bf16_t* x, int c0) {
        const uint2 p = *reinterpret_cast<const uint2*>(x + row + c0), q = *reinterpret_cast<const uint2*>(x + row + c0 + 16);
        return keepu4(tm, cat(p, q));
    };
    auto f8 = [](uint4 x, float (&o)[8]) {
        const uint32_t u[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
        for (int i = 0; i < 4; i++) o[2 * i] = __uint_as_float(u[i] << 16), o[2 * i + 1] = __uint_as_float(u[i] & 0xffff0000u);
    };
    auto st8 = [&](uint16_t* pl, int ld, int k0, uint4 x) {
        uint16_t* const d = pl + r16 * ld + k0 + 4 * q4;
        *reinterpret_cast<uint2*>(d) = make_uint2(x.x, x.y);
        *reinterpret_cast<uint2*>(d + 16) = make_uint2(x.z, x.w);
    };
    f32x4_t Aab = zero4(), AabT = zero4(), BrbT = zero4(), Aak = zero4(), Brb = zero4(), Brk = zero4();
    float rt[KS][8];  // R~ of the lane's keys, kept for P2
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
        const int c0 = 32 * ks + 4 * q4;
        const uint4 xw = ld8(w, c0), xa = ld8(a, c0), xb = ld8(b, c0), xk = ld8(k, c0), xr = ld8(r, c0);
        // (one operand after another, as wkv7_rec_prep)
        float x[8], y[8], eA[8], eR[8], em[8], eh[8], eL[8];
        f8(xw, x);
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const float g = row_prefix_sum(tv ? log_decay(x[e]) : 0.f);
            const float gp = row_prev(g, 0.f), gL = row_last(g);
            em[e] = __expf(-g), eh[e] = __expf(gL - g), eA[e] = __expf(gp), eR[e] = __expf(g), eL[e] = __expf(gL);
        }
        if (r16 == 0) {
            float* el = reinterpret_cast<float*>(rec + R::EL);
            *reinterpret_cast<float4*>(el + c0) = make_float4(eL[0], eL[1], eL[2], eL[3]);
            *reinterpret_cast<float4*>(el + c0 + 16) = make_float4(eL[4], eL[5], eL[6], eL[7]);
        }
        __builtin_amdgcn_sched_barrier(0);
        auto scaled = [&](const float (&f)[8], uint4& hi, uint4& lo) {  // the split pair of x o f
#pragma unroll
            for (int e = 0; e < 8; e++) y[e] = x[e] * f[e];
            pack8(y, hi, lo);
        };
        uint4 ah, al, bh_, bl, rh, rl, hh, hl, kh, kl;
        f8(xa, x), scaled(eA, ah, al);
        st8(&pa[0][0][0], LA, 32 * ks, ah), st8(&pa[1][0][0], LA, 32 * ks, al);
        __builtin_amdgcn_sched_barrier(0);
        f8(xb, x), scaled(eh, hh, hl);
        uint8_t* bf = rec + R::BF + (size_t)(2 * ks) * 1024;
        put_frag(bf, lane, hh);
        put_frag(bf + 1024, lane, hl);
        scaled(em, bh_, bl);
        Aab = mm3(Aab, ah, al, bh_, bl);    // A~_rr . B-_cc
        AabT = mm3(AabT, bh_, bl, ah, al);  // B-_rr . A~_cc
        __builtin_amdgcn_sched_barrier(0);
        f8(xk, x), scaled(em, kh, kl);
        Aak = mm3(Aak, ah, al, kh, kl);
        __builtin_amdgcn_sched_barrier(0);
        f8(xr, x), scaled(eR, rh, rl);
#pragma unroll
        for (int e = 0; e < 8; e++) rt[ks][e] = y[e];
        BrbT = mm3(BrbT, bh_, bl, rh, rl);  // B-_rr . R~_cc
        Brb = mm3(Brb, rh, rl, bh_, bl);
        Brk = mm3(Brk, rh, rl, kh, kl);
        __builtin_amdgcn_sched_barrier(0);
    }
    const int cc = r16;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const int rr = 4 * q4 + e;
        Aab[e] = cc < rr ? Aab[e] : 0.f;
        AabT[e] = rr < cc ? AabT[e] : 0.f;
        BrbT[e] = rr <= cc ? BrbT[e] : 0.f;  // Brb[cc][rr]
        Aak[e] = cc < rr ? Aak[e] : 0.f;
        Brb[e] = cc <= rr ? Brb[e] : 0.f;
        Brk[e] = cc <= rr ? Brk[e] : 0.f;
    }
    uint4* const mt = mats + ((size_t)bh * nchunk + c) * (MATS * 64) + lane;
    auto put_mat = [&](int i, const Pk& m) { mt[64 * i] = cat(m.h, m.l); };
    put_mat(MAT_AAKT, pk(transpose16(Aak, lane))), put_mat(MAT_AAK, pk(Aak));
    put_mat(MAT_BRB, pk(Brb)), put_mat(MAT_BRK, pk(Brk));
    f32x4_t Ti, TiT;
    tri_inverse(Aab, AabT, lane, Ti, TiT);
    const Pk pTiT = pk(TiT), pBrbT = pk(BrbT);
    put_mat(MAT_TI, pk(Ti)), put_mat(MAT_TIT, pTiT);
    __syncthreads();  // A~
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
        Pk pP[2], p2[2];
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const int tj = 2 * ks + u;
            // D layout [t][j], t = 4q4 + e, j = 16tj + r16
            const Pk pA{ldtr(&pa[0][0][16 * tj], LA, lane), ldtr(&pa[1][0][16 * tj], LA, lane)};
            pP[u] = pk(mm16s(pTiT, pA));           // P = Ti A~
            f32x4_t rr4;                            // R~[t = r16][16tj + 4q4 + e]
#pragma unroll
            for (int e = 0; e < 4; e++) rr4[e] = rt[ks][4 * u + e];
            p2[u] = pk(rr4 + mm16s(pP[u], pBrbT));  // P2^T = R~^T + P^T Brb^T
        }
        // P2's tiles as P's lie, by transpose reads
        st8(&pb[0][0][0], LB, 0, cat(p2[0].h, p2[1].h)), st8(&pb[1][0][0], LB, 0, cat(p2[0].l, p2[1].l));
#pragma unroll
        for (int u = 0; u < 2; u++) {
            uint8_t* pp = rec + R::PP + (size_t)(2 * (2 * ks + u)) * 1024;
            put_frag(pp, lane, cat(pP[u].h, ldtr(&pb[0][0][16 * u], LB, lane)));
            put_frag(pp + 1024, lane, cat(pP[u].l, ldtr(&pb[1][0][16 * u], LB, lane)));
        }
    }
}

// ---------------------------------------------------------------------------
// Each head's chunks backwards: workgroup (segment * RGS + rg) * BH + bh of NW waves (4, or
// N/16: all of a head's rows), wave wv of row group rg keeps value rows
// i_own = 16 (NW rg + wv) + r16 of H as Ht[tj][e] = H[i_own][16tj + 4q4 + e].
// Per chunk: H is stored (the chunk kernel's H_end), U^T = B^ H^T over the keys, then
// H^T <- e^{gL} o H^T + [P^T | P2^T] [U^T; dY] on the K=32 instruction.  dY of dtype TI;
// dsT (may be null) and ds0 [key][value] when kv (GDN's layout), else [value][key]; H in
// the workspace always [value][key].  MODE: the time split's launches (ScanMode).
// ---------------------------------------------------------------------------
template <int NK, typename TI, ScanMode MODE>
__global__ __launch_bounds__(4 * NK) void wkv7_bwd_scan(int Tn, int H, int BH, int kv, const float* __restrict__ dsT,
                                                     const TI* __restrict__ dy, float* __restrict__ ds0,
                                                     float* __restrict__ hbuf, const uint8_t* __restrict__ ws,
                                                     ScanSplit sp) {
    using R = BwdRec<NK>;
    constexpr int KS = R::KS, TJ = R::TJ;
    constexpr long NN = (long)NK * NK;
    __shared__ __attribute__((aligned(1024))) uint8_t recs[2][R::DMA_BLOCKS * 1024];
    // workgroup (segment * row groups + rg) * BH + bh, NW waves each
    const int NW = max(1, __builtin_amdgcn_readfirstlane((int)(blockDim.x >> 6))), RGS = NK / 16 / NW;
    const int bh = blockIdx.x % BH, rest = blockIdx.x / BH, rg = rest % RGS, bb = bh / H, h = bh - bb * H;
    const int sgm = MODE == SCAN_ENDS ? rest / RGS : MODE == SCAN_RESUME ? 1 + rest / RGS : 0;
    const bool dual = MODE == SCAN_ENDS && sgm > 0;  // from zero and from the identity, no H stored
    const int tid = threadIdx.x, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63, q4 = lane >> 4, r16 = lane & 15;
    const int i_own = 16 * (NW * rg + wv) + r16;
    const int nchunk = (Tn + BC - 1) / BC;
    // this segment's chunks, chi - 1 down to clo (segment 0: the last m0 chunks)
    const int chi = MODE == SCAN_ALL || sgm == 0 ? nchunk : nchunk - sp.m0 - (sgm - 1) * sp.m;
    const int clo = MODE == SCAN_ALL ? 0 : max(0, sgm == 0 ? nchunk - sp.m0 : chi - sp.m);
    const i32x4_t rs = dma_rsrc(ws + (size_t)bh * nchunk * R::BYTES, (uint32_t)((size_t)nchunk * R::BYTES));
    auto fetch = [&](int c, int buf) {
        uint32_t so = (uint32_t)((size_t)c * R::BYTES);
        asm volatile("" : "+s"(so));
        const uint32_t base = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) uint8_t*)recs[buf];
        for (int j = wv; j < R::DMA_BLOCKS; j += NW) dma_kb(base + 1024 * j, rs, (uint32_t)(1024 * j + 16 * lane), so);
    };
    // dY[t0 + 4q4 + e][i_own], loaded a chunk ahead as raw element bits: rows past the end
    // read row t0, and the bits are widened and zeroed where they are used (dy_of), so
    // nothing waits on the loads until the chunk's closing wait
    auto load_dy = [&](int c, uint32_t (&o)[4]) {
        const int t0 = c * BC, L = min(BC, Tn - t0);
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int t = 4 * q4 + e, tc = t < L ? t : 0;
            const long i = (((long)bb * Tn + t0 + tc) * H + h) * NK + i_own;
            if constexpr (sizeof(TI) == 2) o[e] = reinterpret_cast<const uint16_t*>(dy)[i];
            else o[e] = reinterpret_cast<const uint32_t*>(dy)[i];
        }
    };
    auto dy_of = [&](int c, const uint32_t (&o)[4]) {
        const int L = min(BC, Tn - c * BC);
        f32x4_t d;
#pragma unroll
        for (int e = 0; e < 4; e++)
            d[e] = keep(lane_mask(4 * q4 + e < L), __uint_as_float(sizeof(TI) == 2 ? o[e] << 16 : o[e]));
        return d;
    };
    fetch(chi - 1, 0);
    f32x4_t Ht[TJ], Hp[TJ];  // (Hp: the identity run)
    const float* const start = MODE == SCAN_RESUME ? seg_state(sp, BH, bh, sgm, NN) : dsT;
#pragma unroll
    for (int tj = 0; tj < TJ; tj++) {
        if (dual || (MODE != SCAN_RESUME && !dsT)) {
            Ht[tj] = zero4();
        } else if (MODE != SCAN_RESUME && kv) {
#pragma unroll
            for (int e = 0; e < 4; e++) Ht[tj][e] = dsT[bh * NN + (long)(16 * tj + 4 * q4 + e) * NK + i_own];
        } else {
            const float4 x = *reinterpret_cast<const float4*>(start + (MODE == SCAN_RESUME ? 0 : bh * NN) +
                                                              (long)i_own * NK + 16 * tj + 4 * q4);
            Ht[tj] = f32x4_t{x.x, x.y, x.z, x.w};
        }
        if (MODE == SCAN_ENDS)
#pragma unroll
            for (int e = 0; e < 4; e++) Hp[tj][e] = i_own == 16 * tj + 4 * q4 + e ? 1.f : 0.f;
    }
    uint32_t dyn[4];
    load_dy(chi - 1, dyn);
    vm_wait0();
    f32x4_t dyc = dy_of(chi - 1, dyn);  // this chunk's dY (the next chunk's is formed after each chunk's wait)
    __syncthreads();
    // U^T [t][i_own] = sum_j B^[t][j] H[i_own][j]
    auto btimes = [&](const uint8_t* rec, const f32x4_t (&X)[TJ]) {
        f32x4_t u = zero4();
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            const float sv[8] = {X[2 * ks][0], X[2 * ks][1], X[2 * ks][2], X[2 * ks][3],
                                 X[2 * ks + 1][0], X[2 * ks + 1][1], X[2 * ks + 1][2], X[2 * ks + 1][3]};
            uint4 sh, sl;
            pack8(sv, sh, sl);
            const uint8_t* bf = rec + R::BF + (2 * ks) * 1024;
            u = mm3(u, get_frag(bf, lane), get_frag(bf + 1024, lane), sh, sl);
        }
        return u;
    };
    for (int c = chi - 1, it = 0; c >= clo; c--, it++) {
        if (c > clo) fetch(c - 1, (it + 1) & 1);
        const uint8_t* const rec = recs[it & 1];
        if (c > clo) load_dy(c - 1, dyn);
        // H at the chunk's end, stored after the next record's DMA and left in flight by the
        // closing wait (vmcnt(TJ): a vmcnt(0) there had waited for these stores every chunk)
        if (!dual) {
            float* const hout = hbuf + ((long)bh * nchunk + c) * NN + (long)i_own * NK + 4 * q4;
#pragma unroll
            for (int tj = 0; tj < TJ; tj++)
                *reinterpret_cast<float4*>(hout + 16 * tj) = make_float4(Ht[tj][0], Ht[tj][1], Ht[tj][2], Ht[tj][3]);
        }
        const f32x4_t u = btimes(rec, Ht);
        uint2 uh, ul, dh, dl, ph = {}, pl = {};
        pack4(u, uh, ul);
        pack4(dyc, dh, dl);  // (bf16 dY: dl = 0)
        if (dual) pack4(btimes(rec, Hp), ph, pl);
        const uint4 bhi = cat(uh, dh), blo = cat(ul, dl);
        const uint4 phi = cat(ph, make_uint2(0, 0)), plo = cat(pl, make_uint2(0, 0));  // (the identity run has no dY)
#pragma unroll
        for (int tj = 0; tj < TJ; tj++) {
            const uint8_t* pp = rec + R::PP + (2 * tj) * 1024;
            const uint4 ah = get_frag(pp, lane), al = get_frag(pp + 1024, lane);
            const f32x4_t eg = *reinterpret_cast<const f32x4_t*>(rec + R::EL + 4 * (16 * tj + 4 * q4));
            Ht[tj] = mma32(mma32(mma32(Ht[tj] * eg, ah, bhi), ah, blo), al, bhi);
            if (dual) Hp[tj] = mma32(mma32(mma32(Hp[tj] * eg, ah, phi), ah, plo), al, phi);
        }
        // the next record and the dY loads after it have landed (only the stores may not)
        if (dual) vm_wait0();
        else vm_wait_n<TJ>();
        // the next chunk's dY, formed here where its loads are known complete (formed at the
        // top of the loop, the compiler's own wait there, merged with the path into the loop,
        // would have waited for these stores too)
        if (c > clo) dyc = dy_of(c - 1, dyn);
        __syncthreads();
    }
    if (MODE == SCAN_ENDS) {  // X_1, or U_s and Phi_s
        const long o4 = ((dual ? (long)(sgm - 1) * BH : 0) + bh) * NN + (long)i_own * NK + 4 * q4;
        float* const dst = dual ? sp.uend : sp.send0;
#pragma unroll
        for (int tj = 0; tj < TJ; tj++) {
            *reinterpret_cast<float4*>(dst + o4 + 16 * tj) = make_float4(Ht[tj][0], Ht[tj][1], Ht[tj][2], Ht[tj][3]);
            if (dual)  // (transposed, as scan_chain reads it)
#pragma unroll
                for (int e = 0; e < 4; e++)
                    sp.phi[((long)(sgm - 1) * BH + bh) * NN + (long)(16 * tj + 4 * q4 + e) * NK + i_own] = Hp[tj][e];
        }
        return;
    }
    if (clo > 0) return;  // (only the segment of the first chunk ends the head)
#pragma unroll
    for (int tj = 0; tj < TJ; tj++) {
        if (kv) {
#pragma unroll
            for (int e = 0; e < 4; e++) ds0[bh * NN + (long)(16 * tj + 4 * q4 + e) * NK + i_own] = Ht[tj][e];
        } else {
            *reinterpret_cast<float4*>(ds0 + bh * NN + (long)i_own * NK + 16 * tj + 4 * q4) =
                make_float4(Ht[tj][0], Ht[tj][1], Ht[tj][2], Ht[tj][3]);
        }
    }
}

// ---------------------------------------------------------------------------
// The gradients of one chunk (4 NK lanes).  Workgroups map to (head, chunk) so that a
// head's consecutive chunks share an XCD (chunk c's S_end is chunk c + 1's S0 in L2).
// ---------------------------------------------------------------------------
// The operands every wave reads as K=32 A/B fragments over the keys or value rows are
// split into bf16 hi/lo once, by the wave that owns their 16 columns, and kept so in LDS
// (splitting them in every reader had been most of the kernel's VALU work).
template <int NK> struct SplitPlane {
    static constexpr int CLB = NK + 8;  // padded row (bf16)
    uint16_t h[BC][CLB], l[BC][CLB];
};
// a D-layout tile ([t][16 wv + c], rows t = 4q4 + e) into a split plane, 8-byte rows per lane
template <int NK> __device__ __forceinline__ void put_split(SplitPlane<NK>& P, const f32x4_t& d, int lane, int wv) {
    uint2 h, l;
    quad_rows_split(d, lane, h, l);  // (cross-lane: every lane takes part)
    const int tr = 4 * (lane >> 4) + (lane & 3), c = 16 * wv + 4 * ((lane >> 2) & 3);
    *reinterpret_cast<uint2*>(&P.h[tr][c]) = h;
    *reinterpret_cast<uint2*>(&P.l[tr][c]) = l;
}
// the K=32 fragment of row r16, columns 32ks + 4q4 .. +3 and 32ks + 16 + 4q4 .. +3
template <int NK>
__device__ __forceinline__ void get_split(const SplitPlane<NK>& P, int lane, int ks, uint4& h, uint4& l) {
    const int r = lane & 15, c = 32 * ks + 4 * (lane >> 4);
    const uint2 a = *reinterpret_cast<const uint2*>(&P.h[r][c]), b = *reinterpret_cast<const uint2*>(&P.h[r][c + 16]);
    const uint2 x = *reinterpret_cast<const uint2*>(&P.l[r][c]), y = *reinterpret_cast<const uint2*>(&P.l[r][c + 16]);
    h = make_uint4(a.x, a.y, b.x, b.y);
    l = make_uint4(x.x, x.y, y.x, y.y);
}
// the same fragment of a bf16 row in memory (exact: no lo part), zero when !ok (the row
// is read either way: the caller passes a valid one)
__device__ __forceinline__ uint4 bf16_frag(const bf16_t* row, int ks, int q4, bool ok) {
    const uint2 a = *reinterpret_cast<const uint2*>(row + 32 * ks + 4 * q4);
    const uint2 b = *reinterpret_cast<const uint2*>(row + 32 * ks + 16 + 4 * q4);
    return keepu4(lane_mask(ok), make_uint4(a.x, a.y, b.x, b.y));
}
// One half (hi or lo) of H_end or S0, [value row][key] without padding: each wave puts the 16
// value rows that it loaded and split and takes its 16 keys over all value rows with transpose
// reads.  8-byte piece c of row p lies at c ^ swz_state(p): the writes down 16 rows (16 lanes
// per cycle over 32 banks) and the transpose reads (32 lanes over 64 banks) meet no conflict at
// 128 keys.
template <int NK> __device__ __forceinline__ int state_at(int row, int col) {  // col a multiple of 4
    const int sw = NK == 64 ? swz<SwLane>(row) : 4 * (row & 7) + 2 * ((row >> 3) & 1) + ((row >> 2) & 1);
    return row * NK + (((col >> 2) ^ sw) << 2);
}
// row `row`'s keys as the K=32 operand holds them (slots 32ks + 4q4 + e, +16)
template <int NK> __device__ __forceinline__ void put_state(uint16_t* x, uint4 v, int row, int ks, int q4) {
    *reinterpret_cast<uint2*>(x + state_at<NK>(row, 32 * ks + 4 * q4)) = make_uint2(v.x, v.y);
    *reinterpret_cast<uint2*>(x + state_at<NK>(row, 32 * ks + 16 + 4 * q4)) = make_uint2(v.z, v.w);
}
// the K=32 operand of key 16 wv + r16 over the value rows (the same slots)
template <int NK> __device__ __forceinline__ uint4 get_state(const uint16_t* x, int ks, int wv, int lane) {
    const int row = 32 * ks + 4 * (lane >> 4) + ((lane & 15) >> 2), c = 16 * wv + 4 * (lane & 3);
    return cat(tr_at(x + state_at<NK>(row, c)), tr_at(x + state_at<NK>(row + 16, c)));
}
template <int NK> struct ChunkLds {
    union {
        struct {
            SplitPlane<NK> At, Bh, Kh;  // [t][j], written by the key owners
        };
        uint16_t st[NK * NK];  // (then) the states, one half after another
    };
    SplitPlane<NK> SA, Q;              // [t][i], written by the value-row owners
    uint16_t V[BC][NK + 8], dY[BC][NK + 8];  // as given (exact in bf16)
    float csum[NK / 16][NK];           // per wave: column sums of H_end o S_end over its 16 value rows
    uint4 M[8][64];                    // the masked Gram matrices, packed
};

// What bounds it: H_end, S_end and S0 (64 KB each at 128 keys, S_end mostly from L2) and the
// registers that hide their latency.  Measured at 4 lanes of 2048 tokens and 32 heads of 128
// (rocprofv3; 3.4 GB through HBM, 670 us at the rate of a copy), in this order: 1206 us when each
// wave formed all the chunk's matrices and Gram matrices itself and loaded its key columns
// from memory (232 registers, one workgroup per CU); 1080 with the matrices from
// wkv7_bwd_prep, the Gram matrices shared out and the key operands formed twice instead of
// held (116 registers, two workgroups per CU; the prep kernel 151 -> 183 us); 908 with the
// states turned through LDS, one half of the split pair after another (all four halves at
// once, 128 KB and one workgroup per CU, had been 1320 us).  The column sums from key columns
// of S_end instead of its rows spill (1466 us).  At 64 keys, one lane of 1021 tokens and 40
// heads: 58 -> 49 us.
//
// Saved states: [value][key] at NK = 128; at NK = 64 in the chunked kernels' tiled order
// (but for the last, final one).
template <int NK>
__global__ __launch_bounds__(4 * NK, 4) void wkv7_bwd_chunk(int Tn, int H, int BH, int per_xcd,
                                                      const bf16_t* __restrict__ r, const bf16_t* __restrict__ w,
                                                      const bf16_t* __restrict__ k, const bf16_t* __restrict__ v,
                                                      const bf16_t* __restrict__ a, const bf16_t* __restrict__ b,
                                                      const bf16_t* __restrict__ dy, const float* __restrict__ ckpt,
                                                      const float* __restrict__ hbuf, const uint4* __restrict__ mats,
                                                      bf16_t* __restrict__ dr,
                                                      bf16_t* __restrict__ dw, bf16_t* __restrict__ dk,
                                                      bf16_t* __restrict__ dv, bf16_t* __restrict__ da,
                                                      bf16_t* __restrict__ db) {
    constexpr int KS = NK / 32, TJ = NK / 16, CLB = NK + 8;
    constexpr long NN = (long)NK * NK;
    constexpr bool TILED = NK == 64;
    __shared__ __attribute__((aligned(16))) ChunkLds<NK> sm;
    const int nchunk = (Tn + BC - 1) / BC;
    const int job = (int)(blockIdx.x % 8) * per_xcd + (int)(blockIdx.x / 8);
    if (job >= nchunk * BH) return;  // (whole workgroup)
    const int bh = job / nchunk, c = job - bh * nchunk, bb = bh / H, h = bh - bb * H;
    const int tid = threadIdx.x, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63, q4 = lane >> 4, r16 = lane & 15;
    const int t0 = c * BC, L = min(BC, Tn - t0);
    const long tok0 = (long)bb * Tn + t0;
    const int col = 16 * wv + r16;  // the lane's key (dK ...) and value column (dV ...)
    auto at_tok = [&](int t) { return ((tok0 + t) * H + h) * (long)NK; };
    const long ncp = nchunk + 1;
    const float* const S0 = ckpt + ((long)bh * ncp + c) * NN;
    const float* const Se = S0 + NN;
    const float* const Hm = hbuf + ((long)bh * nchunk + c) * NN;
    const uint4* const mt = mats + (size_t)job * (MATS * 64) + lane;
    const int irow = 16 * wv + r16;  // value row of the row-strip loads

    // ---- the wave's value rows of H_end, S_end and S0 (keys 32ks + 4q4 + e, +16) ----
    float hr[KS][8], sr[KS][8];
    auto rows = [&](const float* M, bool tiled, float (&o)[KS][8]) {
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            // (tiled: tile (wv, 2ks) keeps this lane's four keys at its own float4)
            const long ox = TILED && tiled ? (wv * TJ + 2 * ks) * 256 + 4 * lane : (long)irow * NK + 32 * ks + 4 * q4;
            const long oy = ox + (TILED && tiled ? 256 : 16);
            const float4 x = *reinterpret_cast<const float4*>(M + ox), y = *reinterpret_cast<const float4*>(M + oy);
            o[ks][0] = x.x, o[ks][1] = x.y, o[ks][2] = x.z, o[ks][3] = x.w;
            o[ks][4] = y.x, o[ks][5] = y.y, o[ks][6] = y.z, o[ks][7] = y.w;
        }
    };
    rows(Hm, false, hr);
    rows(Se, c + 1 < nchunk, sr);
    {  // V and dY: eight bytes per thread, rows past the chunk's end zero
        const int t = tid / (NK / 4), cv = 4 * (tid % (NK / 4));
        const uint32_t m = lane_mask(t < L);
        const long o = at_tok(t < L ? t : 0) + cv;
        const uint2 x = *reinterpret_cast<const uint2*>(v + o), y = *reinterpret_cast<const uint2*>(dy + o);
        *reinterpret_cast<uint2*>(&sm.V[t][cv]) = make_uint2(x.x & m, x.y & m);
        *reinterpret_cast<uint2*>(&sm.dY[t][cv]) = make_uint2(y.x & m, y.y & m);
    }

    // ---- the chunk operands of the wave's keys in D layout ([t][col], t = 4q4 + e) ----
    // (formed here for the planes and again for the gradients: kept, they and the decays would
    // be 48 registers through the products between)
    float xr[4], xw[4], xk[4], xa[4], xb[4], eLj;
    f32x4_t eA, eR, eM;
    auto keys = [&]() {
        int q = q4;
        asm volatile("" : "+v"(q));  // (opaque: the second call is not merged with the first)
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int t = 4 * q + e;
            const bool ok = t < L;
            const long o = at_tok(ok ? t : 0) + col;  // (clamped: every lane loads)
            const float r_ = bf2f(r, o), w_ = bf2f(w, o), k_ = bf2f(k, o), a_ = bf2f(a, o), b_ = bf2f(b, o);
            const uint32_t m = lane_mask(ok);
            xr[e] = keep(m, r_), xw[e] = keep(m, w_), xk[e] = keep(m, k_), xa[e] = keep(m, a_), xb[e] = keep(m, b_);
        }
        float ld[4], p[4];
#pragma unroll
        for (int e = 0; e < 4; e++) ld[e] = (4 * q + e) < L ? log_decay(xw[e]) : 0.f;
        p[0] = ld[0], p[1] = p[0] + ld[1], p[2] = p[1] + ld[2], p[3] = p[2] + ld[3];
        // cumulative over the four lane groups (tokens 4q'..4q'+3 of the same key)
        const float T0 = __shfl(p[3], r16), T1 = __shfl(p[3], 16 + r16), T2 = __shfl(p[3], 32 + r16),
                    T3 = __shfl(p[3], 48 + r16);
        const float excl = (q > 0 ? T0 : 0.f) + (q > 1 ? T1 : 0.f) + (q > 2 ? T2 : 0.f);
        eLj = __expf(T0 + T1 + T2 + T3);
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const float g = excl + p[e], gp = e ? excl + p[e - 1] : excl;
            eA[e] = __expf(gp), eR[e] = __expf(g), eM[e] = __expf(-g);
        }
    };
    keys();
    {
        f32x4_t At, Bh, Kh;
#pragma unroll
        for (int e = 0; e < 4; e++)
            At[e] = xa[e] * eA[e], Bh[e] = xb[e] * eM[e] * eLj, Kh[e] = xk[e] * eM[e] * eLj;
        put_split(sm.At, At, lane, wv), put_split(sm.Bh, Bh, lane, wv), put_split(sm.Kh, Kh, lane, wv);
    }
    // the carry's partial column sums over this wave's value rows
#pragma unroll
    for (int ks = 0; ks < KS; ks++)
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const float s = row_sum16(hr[ks][e] * sr[ks][e]);
            if (r16 == 0) sm.csum[wv][32 * ks + (e < 4 ? 4 * q4 + e : 16 + 4 * q4 + e - 4)] = s;
        }
    uint4 Hh[KS], Hl[KS], Sh[KS], Sl[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ks++) pack8(hr[ks], Hh[ks], Hl[ks]);
    rows(S0, true, sr);
#pragma unroll
    for (int ks = 0; ks < KS; ks++) pack8(sr[ks], Sh[ks], Sl[ks]);
    __syncthreads();

    // ---- the wave's [t][i] products over the keys ----
    f32x4_t P1 = zero4(), P2 = zero4(), P3 = zero4();
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
        uint4 ah, al, hh, hl, xh, xl;
        get_split(sm.At, lane, ks, ah, al), get_split(sm.Bh, lane, ks, hh, hl), get_split(sm.Kh, lane, ks, xh, xl);
        P1 = mm3(P1, ah, al, Sh[ks], Sl[ks]);  // A~ S0^T
        P2 = mm3(P2, hh, hl, Hh[ks], Hl[ks]);  // B^ H^T
        P3 = mm3(P3, xh, xl, Hh[ks], Hl[ks]);  // K^ H^T
    }
    // ---- SA, Q, dV for the wave's value columns ----
    auto mat = [&](int i) {
        const uint4 m = mt[64 * i];
        return Pk{make_uint2(m.x, m.y), make_uint2(m.z, m.w)};
    };
    auto mx = [&](const Pk& A, uint2 B) { return mma16(mma16(zero4(), A.h, B), A.l, B); };  // (B exact)
    const uint2 hV = ldtr(&sm.V[0][16 * wv], CLB, lane), hY = ldtr(&sm.dY[0][16 * wv], CLB, lane);
    const f32x4_t SA = mm16s(mat(MAT_TIT), pk(P1 + mx(mat(MAT_AAKT), hV)));  // Ti (A~ S0^T + Aak V)
    const f32x4_t Q = mm16s(mat(MAT_TI), pk(P2 + mx(mat(MAT_BRB), hY)));     // Ti^T (B^ H^T + Brb^T dY)
    const f32x4_t dV = P3 + mm16s(mat(MAT_AAK), pk(Q)) + mx(mat(MAT_BRK), hY);
    put_split(sm.SA, SA, lane, wv), put_split(sm.Q, Q, lane, wv);
    {
        const int tr = 4 * q4 + (lane & 3);  // the row quad_rows_bf16 gives this lane
        const uint2 q = quad_rows_bf16(dV, lane);  // (cross-lane: every lane takes part)
        if (tr < L) *reinterpret_cast<uint2*>(dv + at_tok(tr) + 16 * wv + 4 * ((lane >> 2) & 3)) = q;
    }
    // ---- the products over the value rows ----
    f32x4_t VH = zero4(), SAH = zero4(), dYS = zero4(), QS = zero4();
    auto turn = [&](const uint4 (&x)[KS]) {
        __syncthreads();  // (the key planes or the half before are read)
#pragma unroll
        for (int ks = 0; ks < KS; ks++) put_state<NK>(sm.st, x[ks], irow, ks, q4);
        __syncthreads();  // (the first also: SA, Q, csum)
    };
    // acc += X m, acc2 += Y m with X exact in bf16 and Y = (h, l) (`low`: m is a lo half)
    auto over_rows = [&](const uint16_t* X, const SplitPlane<NK>& Y, bool low, f32x4_t& acc, f32x4_t& acc2) {
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            const uint4 m = get_state<NK>(sm.st, ks, wv, lane);
            acc = mma32(acc, fragp(X, CLB, r16, 32 * ks, lane), m);
            acc2 = mma32(acc2, fragp(&Y.h[0][0], CLB, r16, 32 * ks, lane), m);
            if (!low) acc2 = mma32(acc2, fragp(&Y.l[0][0], CLB, r16, 32 * ks, lane), m);
        }
    };
    turn(Hh), over_rows(&sm.V[0][0], sm.SA, false, VH, SAH);
    turn(Hl), over_rows(&sm.V[0][0], sm.SA, true, VH, SAH);
    turn(Sh), over_rows(&sm.dY[0][0], sm.Q, false, dYS, QS);
    turn(Sl), over_rows(&sm.dY[0][0], sm.Q, true, dYS, QS);

    // ---- the intra-chunk matrices' masked transposes M1..M8, shared out over the waves:
    // element [rr][cc] = X_rr . Y_cc over the value rows ----
    //   0 triu_s(V Q^T)^T   1 triu(V dY^T)^T   2 triu_s(SA Q^T)^T   3 triu(SA dY^T)^T
    //   4 tril(dY SA^T)^T   5 tril(dY V^T)^T   6 tril_s(Q SA^T)^T   7 tril_s(Q V^T)^T
    for (int j = wv; j < 8; j += TJ) {
        // (X, Y): (Q, V) (dY, V) (Q, SA) (dY, SA) (SA, dY) (V, dY) (SA, Q) (V, Q)
        const bool up = j < 4, tok = up ? (j & 1) == 0 : j >= 6;    // tok: Q, else dY
        const bool sa = up ? j >= 2 : (j & 1) == 0;                 // sa: SA, else V
        const uint16_t *gh = tok ? &sm.Q.h[0][0] : &sm.dY[0][0], *gl = tok ? &sm.Q.l[0][0] : nullptr;
        const uint16_t *fh = sa ? &sm.SA.h[0][0] : &sm.V[0][0], *fl = sa ? &sm.SA.l[0][0] : nullptr;
        const uint16_t *xh = up ? gh : fh, *xl = up ? gl : fl, *yh = up ? fh : gh, *yl = up ? fl : gl;
        f32x4_t G = zero4();
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            const uint4 X = fragp(xh, CLB, r16, 32 * ks, lane), Y = fragp(yh, CLB, r16, 32 * ks, lane);
            G = mma32(G, X, Y);
            if (yl) G = mma32(G, X, fragp(yl, CLB, r16, 32 * ks, lane));
            if (xl) G = mma32(G, fragp(xl, CLB, r16, 32 * ks, lane), Y);
        }
        const int strict = up ? (j & 1) == 0 : j >= 6;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int d = up ? 4 * q4 + e - r16 : r16 - (4 * q4 + e);
            G[e] = d >= strict ? G[e] : 0.f;
        }
        const Pk g = pk(G);
        sm.M[j][lane] = cat(g.h, g.l);
    }
    keys();
    __syncthreads();  // M

    // ---- dK, dB, dR, dA, dw for the wave's keys ----
    auto M = [&](int i) {
        const uint4 m = sm.M[i][lane];
        return Pk{make_uint2(m.x, m.y), make_uint2(m.z, m.w)};
    };
    f32x4_t gK, gB, gR, gA;
    {
        f32x4_t At, Rt;
#pragma unroll
        for (int e = 0; e < 4; e++) At[e] = xa[e] * eA[e], Rt[e] = xr[e] * eR[e];
        const Pk pAt = pk(At), pRt = pk(Rt);
        gK = eM * (VH * eLj + mm16s(M(0), pAt) + mm16s(M(1), pRt));
        gB = eM * (SAH * eLj + mm16s(M(2), pAt) + mm16s(M(3), pRt));
    }
    {
        f32x4_t Bm, Km;
#pragma unroll
        for (int e = 0; e < 4; e++) Bm[e] = xb[e] * eM[e], Km[e] = xk[e] * eM[e];
        const Pk pBm = pk(Bm), pKm = pk(Km);
        gR = eR * (dYS + mm16s(M(4), pBm) + mm16s(M(5), pKm));
        gA = eA * (QS + mm16s(M(6), pBm) + mm16s(M(7), pKm));
    }
    // dlogd_t = sum_{s>=t} (r dR - b dB - k dK)_s + sum_{s>t} (a dA)_s + carry
    float sx[4], sy[4];
    {
        float x[4], y[4];
#pragma unroll
        for (int e = 0; e < 4; e++) x[e] = xr[e] * gR[e] - xb[e] * gB[e] - xk[e] * gK[e], y[e] = xa[e] * gA[e];
        sx[3] = x[3], sy[3] = 0.f;
#pragma unroll
        for (int e = 2; e >= 0; e--) sx[e] = sx[e + 1] + x[e], sy[e] = sy[e + 1] + y[e + 1];
        const float ytot = sy[0] + y[0];
        const float X1 = __shfl(sx[0], 16 + r16), X2 = __shfl(sx[0], 32 + r16), X3 = __shfl(sx[0], 48 + r16);
        const float Y1 = __shfl(ytot, 16 + r16), Y2 = __shfl(ytot, 32 + r16), Y3 = __shfl(ytot, 48 + r16);
        const float xa_ = (q4 < 1 ? X1 : 0.f) + (q4 < 2 ? X2 : 0.f) + (q4 < 3 ? X3 : 0.f);
        const float ya_ = (q4 < 1 ? Y1 : 0.f) + (q4 < 2 ? Y2 : 0.f) + (q4 < 3 ? Y3 : 0.f);
        float carry = 0.f;
#pragma unroll
        for (int u = 0; u < TJ; u++) carry += sm.csum[u][col];
#pragma unroll
        for (int e = 0; e < 4; e++) sx[e] += xa_ + carry, sy[e] += ya_;
    }
    f32x4_t gW;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const float s = sigmoidf_(xw[e]);
        gW[e] = (sx[e] + sy[e]) * (-DECAY_SCALE) * s * (1.f - s);
    }
    const int tr = 4 * q4 + (lane & 3);
    const uint2 qk = quad_rows_bf16(gK, lane), qb = quad_rows_bf16(gB, lane), qr = quad_rows_bf16(gR, lane),
                qa = quad_rows_bf16(gA, lane), qw = quad_rows_bf16(gW, lane);
    if (tr < L) {
        const long o = at_tok(tr) + 16 * wv + 4 * ((lane >> 2) & 3);
        *reinterpret_cast<uint2*>(dk + o) = qk;
        *reinterpret_cast<uint2*>(db + o) = qb;
        *reinterpret_cast<uint2*>(dr + o) = qr;
        *reinterpret_cast<uint2*>(da + o) = qa;
        *reinterpret_cast<uint2*>(dw + o) = qw;
    }
}


// ---------------------------------------------------------------------------
// The gated delta rule's backward (GDN layers: one decay e^{g_t} per token and head,
// r = q/sqrt(N), a = k, b = -e^{g} beta k, v' = beta v; q and k as the forward used them: with
// qk_norm L2-normalised here again, and their gradients carried through the normalisation).
// With gamma the chunk's inclusive cumulative g, the per-key factors above become 16x16
// decay-ratio masks, every one of them e^{(a later gamma) - (an earlier one)} <= 1, so
// nothing overflows for any decay (as gdn_prep in the forward):
//   Aab[t][s] = -beta_s (k_t.k_s) e^{gm1_t - gm1_s} (s < t)   Aak = (k_t.k_s) e^{gm1_t - gam_s}
//   Brb[t][s] = -beta_s (r_t.k_s) e^{gam_t - gm1_s} (s <= t)  Brk = (r_t.k_s) e^{gam_t - gam_s}
//   A~ S0^T = e^{gm1_t} (k S0^T),  B^ H^T = -beta_t e^{gL - gm1_t} (k H^T),  K^ H^T = e^{gL - gam_t} (k H^T)
//   dK = e^{gL - gam_t} V'H + M1 k + M2 r,   dB = e^{gL - gam_t} SA H + M3 k + M4 r
//   dR = e^{gam_t} dY S0 + (M5 + M6) k,      dA = e^{gm1_t} Q S0 + (M7 + M8) k
// with M1 = triu_s(V'Q^T) e^{gm1_s - gam_t}, M2 = triu(V'dY^T) e^{gam_s - gam_t}, M3, M4 the
// same for SA, M5 = tril(dY SA^T) (-beta_s) e^{gam_t - gm1_s}, M6 = tril(dY V'^T)
// e^{gam_t - gam_s}, M7 = tril_s(Q SA^T) (-beta_s) e^{gm1_t - gm1_s}, M8 = tril_s(Q V'^T)
// e^{gm1_t - gam_s}; then dq = dR/sqrt(N), dk = dK + dA - e^{g} beta dB, dv = beta dV',
// dbeta = sum_i v dV' - e^{g} sum_j k dB, dg = sum_j dlogd - e^{g} beta sum_j k dB.
// (Checked in float64 against the oracle's exp-mode step adjoint, strong decays included,
// before the kernels.)  The reverse scan's records are the WKV7 ones (e^{gL} repeated
// per key), so wkv7_bwd_scan runs them unchanged.
// ---------------------------------------------------------------------------
template <typename TI>
__global__ __launch_bounds__(64) void gdn_bwd_prep(int Tn, int H, int qk_norm, const TI* __restrict__ q, const TI* __restrict__ k,
                                                   const float* __restrict__ g, const float* __restrict__ beta,
                                                   uint8_t* __restrict__ ws) {
    using R = BwdRec<BNK>;
    const int c = blockIdx.x, bh = blockIdx.y, nchunk = gridDim.x;
    const int bb = bh / H, h = bh - bb * H;
    const int lane = threadIdx.x, q4 = lane >> 4, r16 = lane & 15;
    const int t0 = c * BC, L = min(BC, Tn - t0);
    const long tok0 = (long)bb * Tn + t0;
    auto row = [&](int t) { return ((tok0 + t) * H + h) * (long)BNK; };
    const float rs = 1.f / __builtin_sqrtf((float)BNK);
    __shared__ float gsh[5][BC];  // gamma_t, gamma_{t-1}, beta_t, k_t's and q_t's norm factors (past the end: 0)
    const bool tv = r16 < L;
    const int tl = tv ? r16 : 0;  // (clamped: every lane loads)
    const float g_ = g[(tok0 + tl) * H + h], b_ = beta[(tok0 + tl) * H + h];
    const uint32_t tm = lane_mask(tv);
    const float gt = keep(tm, g_), bt = keep(tm, b_);
    const float gam = row_prefix_sum(gt), gm1 = row_prev(gam, 0.f), gL = row_last(gam);
    uint8_t* const rec = ws + ((size_t)bh * nchunk + c) * R::BYTES;
    float kr[BKS][8], qr[BKS][8], ssk = 0.f, ssq = 0.f;
#pragma unroll
    for (int ks = 0; ks < BKS; ks++) {
        const int c0 = 32 * ks + 4 * q4;
        const float4 ka = keep4(tm, ld4f(k + row(tl) + c0)), kb = keep4(tm, ld4f(k + row(tl) + c0 + 16));
        const float4 qa = keep4(tm, ld4f(q + row(tl) + c0)), qb = keep4(tm, ld4f(q + row(tl) + c0 + 16));
        const float kx[8] = {ka.x, ka.y, ka.z, ka.w, kb.x, kb.y, kb.z, kb.w};
        const float qx[8] = {qa.x, qa.y, qa.z, qa.w, qb.x, qb.y, qb.z, qb.w};
#pragma unroll
        for (int e = 0; e < 8; e++) {
            kr[ks][e] = kx[e], qr[ks][e] = qx[e];
            ssk += kx[e] * kx[e], ssq += qx[e] * qx[e];
        }
    }
    float nk = 1.f, nq = 1.f;  // the rows' L2-norm factors (gdn_prep's)
    if (qk_norm) {
        ssk += __shfl_xor(ssk, 16), ssq += __shfl_xor(ssq, 16);
        ssk += __shfl_xor(ssk, 32), ssq += __shfl_xor(ssq, 32);
        nk = __frsqrt_rn(ssk + 1e-6f), nq = __frsqrt_rn(ssq + 1e-6f);
    }
    if (q4 == 0) gsh[0][r16] = gam, gsh[1][r16] = gm1, gsh[2][r16] = bt, gsh[3][r16] = nk, gsh[4][r16] = nq;
    const float sb = -bt * __expf(gL - gm1);  // B^ = sb k for the lane's token
    f32x4_t KK = zero4(), KR = zero4();
#pragma unroll
    for (int ks = 0; ks < BKS; ks++) {
        float br8[8];
#pragma unroll
        for (int e = 0; e < 8; e++) kr[ks][e] *= nk, qr[ks][e] *= nq, br8[e] = kr[ks][e] * sb;
        uint4 kh, kl, qh, ql, bh_, bl;
        pack8(kr[ks], kh, kl), pack8(qr[ks], qh, ql), pack8(br8, bh_, bl);
        uint8_t* bf = rec + R::BF + (size_t)(2 * ks) * 1024;
        put_frag(bf, lane, bh_);
        put_frag(bf + 1024, lane, bl);
        KK = mm3(KK, kh, kl, kh, kl);  // k_rr . k_cc
        KR = mm3(KR, kh, kl, qh, ql);  // k_rr . q_cc
    }
    __syncthreads();  // gsh
    const int cc = r16;
    f32x4_t Aab, AabT, BrbT;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const int rr = 4 * q4 + e;
        const float gm1r = gsh[1][rr], br = gsh[2][rr];
        const float kk = KK[e], kq = KR[e] * rs;  // k_rr.k_cc, k_rr.r_cc
        Aab[e] = cc < rr ? -bt * kk * __expf(gm1r - gm1) : 0.f;    // Aab[rr][cc]
        AabT[e] = rr < cc ? -br * kk * __expf(gm1 - gm1r) : 0.f;   // Aab[cc][rr]
        BrbT[e] = rr <= cc ? -br * kq * __expf(gam - gm1r) : 0.f;  // Brb[cc][rr]
    }
    f32x4_t Ti, TiT;
    tri_inverse(Aab, AabT, lane, Ti, TiT);
    const Pk pTiT = pk(TiT), pBrbT = pk(BrbT);
    float ea[4], er[4];
    const TI *krow[4], *qrow[4];
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const int t = 4 * q4 + e;
        krow[e] = k + row(t < L ? t : 0) + r16;
        qrow[e] = q + row(t < L ? t : 0) + r16;
        ea[e] = t < L ? gsh[3][t] * __expf(gsh[1][t]) : 0.f;
        er[e] = t < L ? gsh[4][t] * rs * __expf(gsh[0][t]) : 0.f;
    }
#pragma unroll
    for (int tj = 0; tj < BTJ; tj++) {
        f32x4_t at, rt;  // A~, R~ in D layout [t][j], j = 16tj + r16
#pragma unroll
        for (int e = 0; e < 4; e++) at[e] = io<TI>::ld(krow[e], 16 * tj) * ea[e], rt[e] = io<TI>::ld(qrow[e], 16 * tj) * er[e];
        const f32x4_t Pt = mm16s(pTiT, pk(at));
        const Pk pP = pk(Pt);
        const Pk pP2 = pk(rt + mm16s(pBrbT, pP));
        uint8_t* pp = rec + R::PP + (size_t)(2 * tj) * 1024;
        put_frag(pp, lane, cat(pP.h, pP2.h));
        put_frag(pp + 1024, lane, cat(pP.l, pP2.l));
    }
    if (lane < BNK / 4) {
        const float egL = __expf(gL);
        reinterpret_cast<float4*>(rec + R::EL)[lane] = make_float4(egL, egL, egL, egL);
    }
}

// The value rows' operands V and dY [t][i]: bf16 as given (exact), fp32 split.
template <typename TI> struct RowPlane {
    static constexpr int HALVES = sizeof(TI) == 2 ? 1 : 2;
    uint16_t x[HALVES][BC][BNK + 8];
    __device__ __forceinline__ const uint16_t* hi() const { return &x[0][0][0]; }
    __device__ __forceinline__ const uint16_t* lo() const { return HALVES == 2 ? &x[HALVES - 1][0][0] : nullptr; }
};
template <typename TI> struct GdnChunkLds {
    union {
        struct {
            SplitPlane<BNK> K, R;  // k, q as given [t][j], written by the key owners
        };
        uint16_t st[BNK * BNK];    // (then) the states, one half after another
    };
    SplitPlane<BNK> SA, Q;         // [t][i], written by the value-row owners
    RowPlane<TI> V, dY;
    uint4 mat[MATS][64];           // the chunk's matrices, then the masked Gram matrices, packed
    float gam[BC], gm1[BC], beta[BC], fk[BC], fq[BC];  // (fk, fq: the norm factors)
    float csum[BTJ][BNK];
    float pv[BTJ][BC], pd[BTJ][BC], pk[BTJ][BC];  // per wave and token: sum v dV', sum dlogd, sum k dB
    float nk[BTJ][BC], nq[BTJ][BC];  // with qk_norm: sum k^2, sum q^2; then sum k dk, sum q dq of the normalised
};

// As wkv7_bwd_chunk, but for the chunk's matrices, which waves 0..2 form here (from two Gram
// matrices over the keys; the inverse by one wave, not by all eight), and with the exact bf16
// operands' zero lo parts left out.  One lane of 2048 tokens and 32 heads: 364 -> 300 us (the
// states, inputs and outputs at the rate of a copy: 130).  128 registers with 15 spilled; the
// inverse left out is 3 %, S_end's rows left out 9 %; other orders of the first loads or of
// the matrices spill 13 to 20 and measure within 3 %.
template <typename TI>
__global__ __launch_bounds__(512, sizeof(TI) == 2 ? 4 : 2) void gdn_bwd_chunk(
    int Tn, int H, int BH, int per_xcd, int qk_norm, const TI* __restrict__ q, const TI* __restrict__ k,
    const TI* __restrict__ v, const float* __restrict__ g, const float* __restrict__ beta, const TI* __restrict__ dy,
    const float* __restrict__ ckpt, const float* __restrict__ hbuf, TI* __restrict__ dq, TI* __restrict__ dk,
    TI* __restrict__ dv, float* __restrict__ dg, float* __restrict__ dbeta) {
    constexpr bool EXACT = sizeof(TI) == 2;  // (k, q, v and dY without a lo part)
    constexpr int CLB = BNK + 8;
    __shared__ __attribute__((aligned(16))) GdnChunkLds<TI> sm;
    const int nchunk = (Tn + BC - 1) / BC;
    const int job = (int)(blockIdx.x % 8) * per_xcd + (int)(blockIdx.x / 8);
    if (job >= nchunk * BH) return;  // (whole workgroup)
    const int bh = job / nchunk, c = job - bh * nchunk, bb = bh / H, h = bh - bb * H;
    const int tid = threadIdx.x, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63, q4 = lane >> 4, r16 = lane & 15;
    const int t0 = c * BC, L = min(BC, Tn - t0);
    const long tok0 = (long)bb * Tn + t0;
    const int col = 16 * wv + r16;
    const float rs = 1.f / __builtin_sqrtf((float)BNK);
    auto at_tok = [&](int t) { return ((tok0 + t) * H + h) * (long)BNK; };
    const long ncp = nchunk + 1;
    const float* const S0 = ckpt + ((long)bh * ncp + c) * BNN;
    const float* const Se = S0 + BNN;
    const float* const Hm = hbuf + ((long)bh * nchunk + c) * BNN;
    const int irow = 16 * wv + r16;
    // the token scalars (wave 0)
    if (wv == 0) {
        const bool tv = r16 < L;
        const int tl = tv ? r16 : 0;  // (clamped: every lane loads)
        const float g_ = g[(tok0 + tl) * H + h], b_ = beta[(tok0 + tl) * H + h];
        const float gt = keep(lane_mask(tv), g_), bt = keep(lane_mask(tv), b_);
        const float gam = row_prefix_sum(gt), gm1 = row_prev(gam, 0.f);
        if (q4 == 0) sm.gam[r16] = gam, sm.gm1[r16] = gm1, sm.beta[r16] = bt;
    }
    float hr[BKS][8], sr[BKS][8];
    auto rows = [&](const float* M, float (&o)[BKS][8]) {
#pragma unroll
        for (int ks = 0; ks < BKS; ks++) {
            const float4 x = *reinterpret_cast<const float4*>(M + (long)irow * BNK + 32 * ks + 4 * q4);
            const float4 y = *reinterpret_cast<const float4*>(M + (long)irow * BNK + 32 * ks + 16 + 4 * q4);
            o[ks][0] = x.x, o[ks][1] = x.y, o[ks][2] = x.z, o[ks][3] = x.w;
            o[ks][4] = y.x, o[ks][5] = y.y, o[ks][6] = y.z, o[ks][7] = y.w;
        }
    };
    rows(Hm, hr);
    rows(Se, sr);
    {  // V and dY: four elements per thread, rows past the chunk's end zero
        const int t = tid / (BNK / 4), cv = 4 * (tid % (BNK / 4));
        const uint32_t m = lane_mask(t < L);
        const long o = at_tok(t < L ? t : 0) + cv;
        auto put_row = [&](RowPlane<TI>& P, const TI* x) {
            if constexpr (EXACT) {
                const uint2 u = *reinterpret_cast<const uint2*>(x + o);
                *reinterpret_cast<uint2*>(&P.x[0][t][cv]) = make_uint2(u.x & m, u.y & m);
            } else {
                const float4 f = keep4(m, ld4f(x + o));
                uint2 hi, lo;
                pack4(f32x4_t{f.x, f.y, f.z, f.w}, hi, lo);
                *reinterpret_cast<uint2*>(&P.x[0][t][cv]) = hi;
                *reinterpret_cast<uint2*>(&P.x[RowPlane<TI>::HALVES - 1][t][cv]) = lo;
            }
        };
        put_row(sm.V, v), put_row(sm.dY, dy);
    }
    // an input's column of the wave in D layout ([t][col], t = 4q4 + e), zero past the chunk's end
    auto tile = [&](const TI* x) {
        int u = q4;
        asm volatile("" : "+v"(u));  // (opaque: a second reading is not merged with the first and held)
        f32x4_t o;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int t = 4 * u + e;
            const float f = io<TI>::ld(x, at_tok(t < L ? t : 0) + col);  // (clamped: every lane loads)
            o[e] = keep(lane_mask(t < L), f);
        }
        return o;
    };
    // (the planes hold k and q as given: their products are scaled below)
    {
        const f32x4_t kD = tile(k), qD = tile(q);
        if constexpr (EXACT) {
            const int tr = 4 * q4 + (lane & 3), cv = 16 * wv + 4 * ((lane >> 2) & 3);
            *reinterpret_cast<uint2*>(&sm.K.h[tr][cv]) = quad_rows_bf16(kD, lane);
            *reinterpret_cast<uint2*>(&sm.R.h[tr][cv]) = quad_rows_bf16(qD, lane);
        } else {
            put_split(sm.K, kD, lane, wv), put_split(sm.R, qD, lane, wv);
        }
        if (qk_norm) {
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const float sk = row_sum16(kD[e] * kD[e]), sq = row_sum16(qD[e] * qD[e]);
                if (r16 == 0) sm.nk[wv][4 * q4 + e] = sk, sm.nq[wv][4 * q4 + e] = sq;
            }
        }
    }
#pragma unroll
    for (int ks = 0; ks < BKS; ks++)
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const float s = row_sum16(hr[ks][e] * sr[ks][e]);
            if (r16 == 0) sm.csum[wv][32 * ks + (e < 4 ? 4 * q4 + e : 16 + 4 * q4 + e - 4)] = s;
        }
    uint4 Hh[BKS], Hl[BKS], Sh[BKS], Sl[BKS];
#pragma unroll
    for (int ks = 0; ks < BKS; ks++) pack8(hr[ks], Hh[ks], Hl[ks]);
    rows(S0, sr);
#pragma unroll
    for (int ks = 0; ks < BKS; ks++) pack8(sr[ks], Sh[ks], Sl[ks]);
    __syncthreads();

    // the norm factors x * rsqrt(sum x^2 + 1e-6) of column token r16, and of rows 4q4 + e by shuffle
    float fk = 1.f, fq = 1.f;
    if (qk_norm) {
        float sk = 0.f, sq = 0.f;
#pragma unroll
        for (int u = 0; u < BTJ; u++) sk += sm.nk[u][r16], sq += sm.nq[u][r16];
        fk = __frsqrt_rn(sk + 1e-6f), fq = __frsqrt_rn(sq + 1e-6f);
    }
    if (wv == 0 && q4 == 0) sm.fk[r16] = fk, sm.fq[r16] = fq;
    auto put_mat = [&](int i, const f32x4_t& x) {
        const Pk p = pk(x);
        sm.mat[i][lane] = cat(p.h, p.l);
    };
    auto mat = [&](int i) {
        const uint4 m = sm.mat[i][lane];
        return Pk{make_uint2(m.x, m.y), make_uint2(m.z, m.w)};
    };
    // the chunk's matrices, element [rr][cc] (rr = 4q4 + e, cc = r16): wave 0 the inverse, 1 Aak, 2 Brb and Brk
    if (wv < 3) {
        f32x4_t G = zero4();  // k_rr . k_cc; wave 2: q_rr . k_cc
        const SplitPlane<BNK>& X = wv == 2 ? sm.R : sm.K;
#pragma unroll
        for (int ks = 0; ks < BKS; ks++) {
            uint4 xh, xl, kh, kl;
            get_split(X, lane, ks, xh, xl), get_split(sm.K, lane, ks, kh, kl);
            G = EXACT ? mma32(G, xh, kh) : mm3(G, xh, xl, kh, kl);
        }
        const int cc = r16;
        const float gc = sm.gam[cc], gm1c = sm.gm1[cc], bc = sm.beta[cc];
        float gr[4], gm1r[4], br[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            gr[e] = sm.gam[4 * q4 + e], gm1r[e] = sm.gm1[4 * q4 + e], br[e] = sm.beta[4 * q4 + e];
            G[e] *= (wv == 2 ? rs * __shfl(fq, 4 * q4 + e) : __shfl(fk, 4 * q4 + e)) * fk;
        }
        f32x4_t a, b;
        if (wv == 0) {
            f32x4_t Ti, TiT;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int rr = 4 * q4 + e;
                a[e] = cc < rr ? -bc * G[e] * __expf(gm1r[e] - gm1c) : 0.f;
                b[e] = rr < cc ? -br[e] * G[e] * __expf(gm1c - gm1r[e]) : 0.f;
            }
            tri_inverse(a, b, lane, Ti, TiT);
            put_mat(MAT_TI, Ti), put_mat(MAT_TIT, TiT);
        } else if (wv == 1) {
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int rr = 4 * q4 + e;
                a[e] = cc < rr ? G[e] * __expf(gm1r[e] - gc) : 0.f;
                b[e] = rr < cc ? G[e] * __expf(gm1c - gr[e]) : 0.f;
            }
            put_mat(MAT_AAK, a), put_mat(MAT_AAKT, b);
        } else {
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int rr = 4 * q4 + e;
                a[e] = cc <= rr ? -bc * G[e] * __expf(gr[e] - gm1c) : 0.f;
                b[e] = cc <= rr ? G[e] * __expf(gr[e] - gc) : 0.f;
            }
            put_mat(MAT_BRB, a), put_mat(MAT_BRK, b);
        }
    }
    // the wave's products k S0^T, k H^T
    f32x4_t P1 = zero4(), kH = zero4();
#pragma unroll
    for (int ks = 0; ks < BKS; ks++) {
        uint4 kh, kl;
        get_split(sm.K, lane, ks, kh, kl);
        P1 = mma32(mma32(P1, kh, Sh[ks]), kh, Sl[ks]);
        kH = mma32(mma32(kH, kh, Hh[ks]), kh, Hl[ks]);
        if constexpr (!EXACT) P1 = mma32(P1, kl, Sh[ks]), kH = mma32(kH, kl, Hh[ks]);
    }
    __syncthreads();  // the matrices, the norm factors; (the key planes are read)

    auto put = [&](TI* dst, const f32x4_t& x) {
        if constexpr (EXACT) {
            const int tr = 4 * q4 + (lane & 3);
            const uint2 qv = quad_rows_bf16(x, lane);  // (cross-lane: every lane takes part)
            if (tr < L) *reinterpret_cast<uint2*>(dst + at_tok(tr) + 16 * wv + 4 * ((lane >> 2) & 3)) = qv;
        } else {
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (4 * q4 + e < L) dst[at_tok(4 * q4 + e) + col] = x[e];
        }
    };
    // ---- SA, Q, dV' for the wave's value columns ----
    {
        const float gL = sm.gam[BC - 1];
        f32x4_t P2, P3, vD, br;
        const f32x4_t vraw = tile(v), dyD = tile(dy);
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const float gre = sm.gam[4 * q4 + e], gm1e = sm.gm1[4 * q4 + e], f = sm.fk[4 * q4 + e];
            br[e] = sm.beta[4 * q4 + e];
            P1[e] *= f * __expf(gm1e);
            P2[e] = kH[e] * f * (-br[e] * __expf(gL - gm1e));
            P3[e] = kH[e] * f * __expf(gL - gre);
            vD[e] = br[e] * vraw[e];
        }
        const Pk pV = pk(vD), pdY = pk(dyD);
        const f32x4_t SA = mm16s(mat(MAT_TIT), pk(P1 + mm16s(mat(MAT_AAKT), pV)));
        const f32x4_t Q = mm16s(mat(MAT_TI), pk(P2 + mm16s(mat(MAT_BRB), pdY)));
        const f32x4_t dVp = P3 + mm16s(mat(MAT_AAK), pk(Q)) + mm16s(mat(MAT_BRK), pdY);
        put_split(sm.SA, SA, lane, wv), put_split(sm.Q, Q, lane, wv);
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const float s = row_sum16(vraw[e] * dVp[e]);
            if (r16 == 0) sm.pv[wv][4 * q4 + e] = s;
        }
        put(dv, br * dVp);
    }
    // ---- the products over the value rows (V as given: V' = beta V of its rows below) ----
    f32x4_t VH = zero4(), SAH = zero4(), dYS = zero4(), QS = zero4();
    auto turn = [&](const uint4 (&x)[BKS], bool first) {
        if (!first) __syncthreads();  // (the half before is read)
#pragma unroll
        for (int ks = 0; ks < BKS; ks++) put_state<BNK>(sm.st, x[ks], irow, ks, q4);
        __syncthreads();  // (the first also: SA, Q, csum, pv; the matrices are read)
    };
    // acc += X m, acc2 += Y m (`low`: m is a lo half)
    auto over_rows = [&](const RowPlane<TI>& X, const SplitPlane<BNK>& Y, bool low, f32x4_t& acc, f32x4_t& acc2) {
#pragma unroll
        for (int ks = 0; ks < BKS; ks++) {
            const uint4 m = get_state<BNK>(sm.st, ks, wv, lane);
            acc = mma32(acc, fragp(X.hi(), CLB, r16, 32 * ks, lane), m);
            if (!EXACT && !low) acc = mma32(acc, fragp(X.lo(), CLB, r16, 32 * ks, lane), m);
            acc2 = mma32(acc2, fragp(&Y.h[0][0], CLB, r16, 32 * ks, lane), m);
            if (!low) acc2 = mma32(acc2, fragp(&Y.l[0][0], CLB, r16, 32 * ks, lane), m);
        }
    };
    turn(Hh, true), over_rows(sm.V, sm.SA, false, VH, SAH);
    turn(Hl, false), over_rows(sm.V, sm.SA, true, VH, SAH);
    turn(Sh, false), over_rows(sm.dY, sm.Q, false, dYS, QS);
    turn(Sl, false), over_rows(sm.dY, sm.Q, true, dYS, QS);

    // ---- the intra-chunk matrices' masked transposes, shared out over waves 0..5: element
    // [rr][cc] of the sums X_rr . Y_cc over the value rows ----
    //   0 (Q, V')   1 (dY, V')   2 (Q, SA)   3 (dY, SA)   4 (SA, dY) + (V', dY)   5 (SA, Q) + (V', Q)
    if (wv < 6) {
        const int cc = r16;
        const float gc = sm.gam[cc], gm1c = sm.gm1[cc], bc = sm.beta[cc];
        float gr[4], gm1r[4], br[4];
#pragma unroll
        for (int e = 0; e < 4; e++) gr[e] = sm.gam[4 * q4 + e], gm1r[e] = sm.gm1[4 * q4 + e], br[e] = sm.beta[4 * q4 + e];
        auto gram = [&](const uint16_t* xh, const uint16_t* xl, const uint16_t* yh, const uint16_t* yl) {
            f32x4_t G = zero4();
#pragma unroll
            for (int ks = 0; ks < BKS; ks++) {
                const uint4 X = fragp(xh, CLB, r16, 32 * ks, lane), Y = fragp(yh, CLB, r16, 32 * ks, lane);
                G = mma32(G, X, Y);
                if (yl) G = mma32(G, X, fragp(yl, CLB, r16, 32 * ks, lane));
                if (xl) G = mma32(G, fragp(xl, CLB, r16, 32 * ks, lane), Y);
            }
            return G;
        };
        const bool tok = wv == 5 || (wv < 4 && wv % 2 == 0);  // with Q, else with dY
        const uint16_t *yh = tok ? &sm.Q.h[0][0] : sm.dY.hi(), *yl = tok ? &sm.Q.l[0][0] : sm.dY.lo();
        f32x4_t M;
        if (wv < 4) {
            const bool sa = wv >= 2;
            M = gram(yh, yl, sa ? &sm.SA.h[0][0] : sm.V.hi(), sa ? &sm.SA.l[0][0] : sm.V.lo());
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int d = 4 * q4 + e - cc;
                // triu_s: e^{gm1_rr - gam_cc}, triu: e^{gam_rr - gam_cc}
                const float f = (sa ? 1.f : bc) * __expf((tok ? gm1r[e] : gr[e]) - gc);
                M[e] = d >= (tok ? 1 : 0) ? M[e] * f : 0.f;
            }
        } else {
            const f32x4_t S = gram(&sm.SA.h[0][0], &sm.SA.l[0][0], yh, yl), V = gram(sm.V.hi(), sm.V.lo(), yh, yl);
            const float gcol = tok ? gm1c : gc;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int d = cc - (4 * q4 + e);
                M[e] = d >= (tok ? 1 : 0) ? br[e] * (V[e] * __expf(gcol - gr[e]) - S[e] * __expf(gcol - gm1r[e])) : 0.f;
            }
        }
        put_mat(wv, M);
    }
    // ---- dq, dk and the token sums for the wave's keys ----
    float gr[4], gm1r[4], br[4], nkr[4], nqr[4];
    const float gL = sm.gam[BC - 1];
    f32x4_t kD = tile(k), rD = tile(q);
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const int t = 4 * q4 + e;
        gr[e] = sm.gam[t], gm1r[e] = sm.gm1[t], br[e] = sm.beta[t], nkr[e] = sm.fk[t], nqr[e] = sm.fq[t];
        kD[e] *= nkr[e], rD[e] *= rs * nqr[e];
        VH[e] *= br[e];
    }
    __syncthreads();  // the Gram matrices
    const Pk pkD = pk(kD), prD = pk(rD);
    const f32x4_t tK = mm16s(mat(0), pkD) + mm16s(mat(1), prD);
    const f32x4_t tB = mm16s(mat(2), pkD) + mm16s(mat(3), prD);
    const f32x4_t tR = mm16s(mat(4), pkD), tA = mm16s(mat(5), pkD);
    f32x4_t gK, gB, gR, gA, egb;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const float fL = __expf(gL - gr[e]);
        gK[e] = fL * VH[e] + tK[e];
        gB[e] = fL * SAH[e] + tB[e];
        gR[e] = __expf(gr[e]) * dYS[e] + tR[e];
        gA[e] = __expf(gm1r[e]) * QS[e] + tA[e];
        egb[e] = __expf(gr[e] - gm1r[e]) * br[e];  // e^{g_t} beta_t
    }
    float sx[4], sy[4];
    {
        float x[4], y[4];
#pragma unroll
        for (int e = 0; e < 4; e++)
            x[e] = rD[e] * gR[e] + egb[e] * kD[e] * gB[e] - kD[e] * gK[e], y[e] = kD[e] * gA[e];
        sx[3] = x[3], sy[3] = 0.f;
#pragma unroll
        for (int e = 2; e >= 0; e--) sx[e] = sx[e + 1] + x[e], sy[e] = sy[e + 1] + y[e + 1];
        const float ytot = sy[0] + y[0];
        const float X1 = __shfl(sx[0], 16 + r16), X2 = __shfl(sx[0], 32 + r16), X3 = __shfl(sx[0], 48 + r16);
        const float Y1 = __shfl(ytot, 16 + r16), Y2 = __shfl(ytot, 32 + r16), Y3 = __shfl(ytot, 48 + r16);
        const float xa_ = (q4 < 1 ? X1 : 0.f) + (q4 < 2 ? X2 : 0.f) + (q4 < 3 ? X3 : 0.f);
        const float ya_ = (q4 < 1 ? Y1 : 0.f) + (q4 < 2 ? Y2 : 0.f) + (q4 < 3 ? Y3 : 0.f);
        float carry = 0.f;
#pragma unroll
        for (int u = 0; u < BTJ; u++) carry += sm.csum[u][col];
#pragma unroll
        for (int e = 0; e < 4; e++) sx[e] += xa_ + carry, sy[e] += ya_;
    }
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const float sd = row_sum16(sx[e] + sy[e]), skb = row_sum16(kD[e] * gB[e]);
        if (r16 == 0) sm.pd[wv][4 * q4 + e] = sd, sm.pk[wv][4 * q4 + e] = skb;
    }
    // gradients of q and k as the recurrence takes them; with qk_norm dx = n (dy - y (y . dy)) of
    // y = n x, the dot over the token's keys summed over the waves
    f32x4_t gq = gR * rs, gk = gK + gA - egb * gB;
    if (qk_norm) {
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const float sk = row_sum16(kD[e] * gk[e]), sq = row_sum16(rD[e] * gR[e]);  // (q . dq = r . dr)
            if (r16 == 0) sm.nk[wv][4 * q4 + e] = sk, sm.nq[wv][4 * q4 + e] = sq;
        }
    }
    __syncthreads();  // pd, pk, nk, nq
    if (qk_norm) {
        const float sn = __builtin_sqrtf((float)BNK);
#pragma unroll
        for (int e = 0; e < 4; e++) {
            float a = 0.f, b = 0.f;
#pragma unroll
            for (int u = 0; u < BTJ; u++) a += sm.nk[u][4 * q4 + e], b += sm.nq[u][4 * q4 + e];
            gk[e] = nkr[e] * (gk[e] - kD[e] * a);
            gq[e] = nqr[e] * (gq[e] - rD[e] * sn * b);
        }
    }
    put(dq, gq);
    put(dk, gk);
    if (wv == 0 && lane < L) {
        float spv = 0.f, spd = 0.f, spk = 0.f;
#pragma unroll
        for (int u = 0; u < BTJ; u++) spv += sm.pv[u][lane], spd += sm.pd[u][lane], spk += sm.pk[u][lane];
        const float eg = __expf(sm.gam[lane] - sm.gm1[lane]);
        const long o = (tok0 + lane) * H + h;
        dg[o] = spd - eg * sm.beta[lane] * spk;
        dbeta[o] = spv - eg * spk;
    }
}

}  // namespace

// Workspace: the scan's records, H = dL/dS at every chunk's end, (WKV7) the chunks' matrices, and
// the time split's buffers (cus = 0: without them).
template <int NK> static size_t bwd_records(size_t chunks) { return (chunks * BwdRec<NK>::BYTES + 255) / 256 * 256; }
static size_t mats_bytes(size_t chunks) { return chunks * MATS * 64 * sizeof(uint4); }
template <int NK> static size_t split_at(size_t chunks, bool mats) {
    return bwd_records<NK>(chunks) + chunks * NK * NK * sizeof(float) + (mats ? mats_bytes(chunks) : 0);
}
template <int NK> static size_t bwd_workspace(int B, int T, int H, int cus, bool mats) {
    const int n = (T + BC - 1) / BC;
    const size_t BH = (size_t)B * H;
    return split_at<NK>(BH * n, mats) + resume_bytes(BH, NK, resume_segments(BH, NK, n, cus, true));
}
size_t wkv7_rec_bwd_workspace(int B, int T, int H, int N, int cus) {
    return N == 64 ? bwd_workspace<64>(B, T, H, cus, true) : bwd_workspace<128>(B, T, H, cus, true);
}
// The reverse scan over the records at ws, in one pass or in as many time segments as cus and
// the ws_bytes behind the records, H and (mats) matrices allow.
template <int NK, typename TI>
static const float* scan_back(int T, int H, int BH, int kv, const float* dsT, const void* dy, float* ds0, void* ws,
                              size_t ws_bytes, bool mats, int cus, hipStream_t stream) {
    const int n = (T + BC - 1) / BC;
    const size_t chunks = (size_t)BH * n, at = split_at<NK>(chunks, mats);
    int k = resume_segments(BH, NK, n, cus, true);
    while (k >= 4 && at + resume_bytes(BH, NK, k) > ws_bytes) k--;
    if (k < 4) k = 1;
    const int rgs = k < 2 ? NK / 64 : scan_groups(BH, NK, k - 1, cus), lanes = 4 * NK / rgs;
    const uint8_t* const recs = static_cast<const uint8_t*>(ws);
    float* const hbuf = reinterpret_cast<float*>(static_cast<uint8_t*>(ws) + bwd_records<NK>(chunks));
    const TI* const y = static_cast<const TI*>(dy);
    if (k < 2) {
        hipLaunchKernelGGL((wkv7_bwd_scan<NK, TI, SCAN_ALL>), dim3(BH * rgs), dim3(lanes), 0, stream, T, H, BH, kv, dsT, y,
                           ds0, hbuf, recs, ScanSplit{});
        return hbuf;
    }
    const ScanSplit sp = resume_split(BH, NK, n, k, reinterpret_cast<float*>(static_cast<uint8_t*>(ws) + at));
    hipLaunchKernelGGL((wkv7_bwd_scan<NK, TI, SCAN_ENDS>), dim3((k - 1) * BH * rgs), dim3(lanes), 0, stream, T, H, BH, kv,
                       dsT, y, ds0, hbuf, recs, sp);
    hipLaunchKernelGGL((scan_chain<NK>), dim3(BH, NK / 16), dim3(4 * NK), 0, stream, BH, k - 2, kv, sp, nullptr);
    hipLaunchKernelGGL((wkv7_bwd_scan<NK, TI, SCAN_RESUME>), dim3((k - 1) * BH * rgs), dim3(lanes), 0, stream, T, H, BH, kv,
                       dsT, y, ds0, hbuf, recs, sp);
    return hbuf;
}

template <int NK> static void launch_rec_bwd(const Bwd& p, int cus) {
    const int nchunk = (p.T + BC - 1) / BC, BH = p.B * p.H;
    const bf16_t *r = static_cast<const bf16_t*>(p.r), *w = static_cast<const bf16_t*>(p.w),
                 *k = static_cast<const bf16_t*>(p.k), *v = static_cast<const bf16_t*>(p.v),
                 *a = static_cast<const bf16_t*>(p.a), *b = static_cast<const bf16_t*>(p.b),
                 *dy = static_cast<const bf16_t*>(p.dy);
    uint4* const mats = reinterpret_cast<uint4*>(static_cast<uint8_t*>(p.ws) + split_at<NK>((size_t)BH * nchunk, false));
    hipLaunchKernelGGL(wkv7_bwd_prep<NK>, dim3(nchunk, BH), dim3(64), 0, p.stream, p.T, p.H, r, w, k, a, b,
                       static_cast<uint8_t*>(p.ws), mats);
    const float* const hbuf = scan_back<NK, bf16_t>(p.T, p.H, BH, 0, p.dsT, dy, p.ds0, p.ws, p.ws_bytes, true, cus,
                                                  p.stream);
    const int jobs = nchunk * BH, per_xcd = (jobs + 7) / 8;
    hipLaunchKernelGGL(wkv7_bwd_chunk<NK>, dim3(8 * per_xcd), dim3(4 * NK), 0, p.stream, p.T, p.H, BH, per_xcd, r, w, k,
                       v, a, b, dy, p.ckpt, hbuf, mats, static_cast<bf16_t*>(p.dr), static_cast<bf16_t*>(p.dw),
                       static_cast<bf16_t*>(p.dk), static_cast<bf16_t*>(p.dv), static_cast<bf16_t*>(p.da),
                       static_cast<bf16_t*>(p.db));
}
void launch_wkv7_rec_backward(const Bwd& p, int cus) {
    if (p.N == 64) launch_rec_bwd<64>(p, cus);
    else launch_rec_bwd<128>(p, cus);
}

size_t gdn_backward_workspace(int B, int T, int H, int cus) { return bwd_workspace<BNK>(B, T, H, cus, false); }

template <typename TI>
static void launch_gdn_bwd(const GdnBwd& p) {
    const int nchunk = (p.T + BC - 1) / BC, BH = p.B * p.H;
    const TI *q = static_cast<const TI*>(p.q), *k = static_cast<const TI*>(p.k), *v = static_cast<const TI*>(p.v),
             *dout = static_cast<const TI*>(p.dout);
    hipLaunchKernelGGL(gdn_bwd_prep<TI>, dim3(nchunk, BH), dim3(64), 0, p.stream, p.T, p.H, p.qk_norm, q, k,
                       p.g, p.beta, static_cast<uint8_t*>(p.ws));
    const float* const hbuf = scan_back<BNK, TI>(p.T, p.H, BH, 1, p.dsT, dout, p.ds0, p.ws, p.ws_bytes, false, p.cus,
                                             p.stream);
    const int jobs = nchunk * BH, per_xcd = (jobs + 7) / 8;
    hipLaunchKernelGGL(gdn_bwd_chunk<TI>, dim3(8 * per_xcd), dim3(512), 0, p.stream, p.T, p.H, BH, per_xcd,
                       p.qk_norm, q, k, v, p.g, p.beta, dout, p.ckpt, hbuf, static_cast<TI*>(p.dq), static_cast<TI*>(p.dk),
                       static_cast<TI*>(p.dv), p.dg, p.dbeta);
}
void launch_gdn_backward(const GdnBwd& p) {
    if (p.dtype == 0) launch_gdn_bwd<bf16_t>(p);
    else launch_gdn_bwd<float>(p);
}

}  // namespace wkv7
