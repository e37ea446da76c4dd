// Window attention on F16 MFMA with fp32 accuracy: QK^T + relative-position
// bias + shift mask + softmax + PV for one (window, head) per block.
//
// The same operator as attn.hip (cpu.rs:772-844; hat.cu:246-316) on gfx950's
// 16-bit matrix path, whose peak is 16x the FP32 MFMA rate. VALU and MFMA work
// share a SIMD's issue time (measured: they hardly overlap, from one wave or
// from two), so the splits and exponentials below cost their full time. Every
// fp32 operand enters as two f16 parts and a product as three MFMA terms
// (common.h states the split's accuracy); q, k and v must lie inside f16's
// range, which the host sees to by folding powers of two into the qkv weights
// (qkv_scale), and networks whose bounds do not allow it run attn.hip.
//
// What bounds it: issue time, MFMA and VALU together. Per 32-key tile and wave
// at head_dim 24, 11 MFMAs of 32 cycles (5 for QK^T, 6 for PV), 16 exponentials
// and ~90 other VALU instructions; the three-part bf16 split that this replaced
// took 21 MFMAs and ~120. HAT-S 512 x 512 (1024 windows, 6 heads): SW 252.6 ->
// 178.2 us a launch, OCA 574 -> 383; HAT 512 x 512 OCA 664 -> 458; head_dim 30
// SW as whole items (two planes fit two blocks a CU; the bf16 planes did not).
// Those are scores near 0, where the softmax needs no maximum; by the online softmax,
// where attnx_flat says so, 512 x 512, q . k of 3 units or a table around -3 (base 0
// tried first, then all again: 333, 374; 634 to 769, 498 to 899): SW 225, 272; OCA
// 460, 530. Launches where both forms stand, 512 x 512: 197 and 211 us, OCA 396 and
// 422 (head_dim 24), 250 and 259, 470 and 490 (30).
// Parts of 288 keys for OCA at head_dim 24 spilled 34 registers (446 us), parts
// of 192 at 30 27 of them (154 us at 256 x 256 against 122).
//
// Layout (all per item, in LDS): K as two f16 planes [256 keys][KS] and V^T
// as two planes [D + 1][VS] whose key order is permuted within each 16 so
// that a lane's eight keys of one MFMA step are contiguous; row D of V^T is
// ones in the high plane and zeros in the other, so row D of O^T is the
// softmax denominator. The bias table of the head is kept in log2 units. Wave
// w owns queries [32w, 32w+32). Scores are computed transposed, S^T = K Q^T
// (A = a 32-key tile of K, B = the wave's q, split in registers): lane l holds
// 16 scores of query l%32, which after the softmax are split and used directly
// as the B operand of O^T += V^T P^T. Bias, mask, online softmax in base 2 and
// the output are those of attn.hip.
#include "common.h"

using namespace hatk;

// What the max-subtracted softmax adds to its base: P up to 2^(8 + 6), so that
// the smallest probabilities stay clear of f16's subnormals.
#define ATTNX_SAFE_UP 6.0f

template <int D>
struct AttnXShape {
    static constexpr int NK = 256;
    // K row stride in f16: 24 (48 B) and 40 (80 B) put the 16 rows a ds_read_b128
    // phase touches on distinct banks.
    static constexpr int KS = D == 24 ? 24 : 40;
    static constexpr int VS = NK + 8;  // V^T row stride (528 B: rows 4 banks apart)
    static constexpr int KPL = NK * KS, VPL = (D + 1) * VS;  // elements per plane
    static constexpr int TROWS = 961;
    static constexpr int LDS_BYTES = 2 * 2 * (KPL + VPL) + 4 * TROWS;
};

// Position of key k in the V^T planes: within each 16 keys, bits 2 and 3
// swap, so that lane half h's eight keys of an MFMA step (16s + 8a + 4h + t,
// a, t the slot's high bit and low two bits) are positions 16s + 8h .. +7.
__device__ __forceinline__ int vpos(int k) { return (k & ~12) | ((k & 4) << 1) | ((k & 8) >> 1); }

// Item staging: this thread's K and V units (attn_fetch's registers), split
// into the LDS planes; row D of V^T: ones (high plane), zeros; K dims D .. 31
// of D = 30 zeroed (the q operand is zero there; LDS that was never written
// could hold a NaN).
template <int D>
__device__ __forceinline__ void attnx_stash(unsigned short* Kp, unsigned short* Vp,
                                            const typename AttnShape<D, false>::vec (&ks)[AttnShape<D, false>::NE],
                                            const typename AttnShape<D, false>::vec (&vs)[AttnShape<D, false>::NE])
{
    using S = AttnShape<D, false>;
    using X = AttnXShape<D>;
    constexpr int PER_KEY = D / S::U;
#pragma unroll
    for (int i = 0; i < S::NE; ++i) {
        const int e = threadIdx.x + i * 512;
        if (e < S::NK * PER_KEY) {
            const int k = e / PER_KEY, d = (e - k * PER_KEY) * S::U;
            float kv[4], vv[4];
            if constexpr (S::U == 4) {
                kv[0] = ks[i].x, kv[1] = ks[i].y, kv[2] = ks[i].z, kv[3] = ks[i].w;
                vv[0] = vs[i].x, vv[1] = vs[i].y, vv[2] = vs[i].z, vv[3] = vs[i].w;
            } else {
                kv[0] = ks[i].x, kv[1] = ks[i].y, kv[2] = kv[3] = 0.f;
                vv[0] = vs[i].x, vv[1] = vs[i].y, vv[2] = vv[3] = 0.f;
            }
#pragma unroll
            for (int j = 0; j < S::U; j += 2) {
                unsigned k0, k1, v0, v1;
                split2_pk(kv[j], kv[j + 1], k0, k1);
                *(unsigned*)(Kp + 0 * X::KPL + k * X::KS + d + j) = k0;
                *(unsigned*)(Kp + 1 * X::KPL + k * X::KS + d + j) = k1;
                split2_pk(vv[j], vv[j + 1], v0, v1);
                const int pos = vpos(k);
                Vp[0 * X::VPL + (d + j) * X::VS + pos] = (unsigned short)v0;
                Vp[0 * X::VPL + (d + j + 1) * X::VS + pos] = (unsigned short)(v0 >> 16);
                Vp[1 * X::VPL + (d + j) * X::VS + pos] = (unsigned short)v1;
                Vp[1 * X::VPL + (d + j + 1) * X::VS + pos] = (unsigned short)(v1 >> 16);
            }
        }
    }
    for (int e = threadIdx.x; e < 2 * (S::NK / 2); e += 512) {
        const int pl = e / (S::NK / 2), k2 = e - pl * (S::NK / 2);
        *(unsigned*)(Vp + pl * X::VPL + D * X::VS + 2 * k2) = pl == 0 ? 0x3c003c00u : 0u;  // f16 1.0 pairs
    }
    if (D == 30) {
        for (int e = threadIdx.x; e < 2 * S::NK; e += 512) {
            const int pl = e / S::NK, k = e - pl * S::NK;
            *(unsigned*)(Kp + pl * X::KPL + k * X::KS + 30) = 0u;
        }
    }
}

// The lane's q, pre-scaled and split: qb[s][part] = dims 16s + 8h .. 16s + 8h
// + 7 of its query (zeros past D). For D = 24 the second step is packed (see
// AttnxKRows): qb[1][0] = dims 16..23 of part h.
template <int D>
__device__ __forceinline__ int attnx_query(const AttnArgs& p, int wi, int head, u32x4 (&qb)[2][2])
{
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform, in a scalar register
    const int ql = lane & 31, h = lane >> 5;
    const int q = wave * 32 + ql, qy = q >> 4, qx = q & 15;
    const int wy = wi / p.nx, wx = wi - (wi / p.nx) * p.nx;
    int y = wy * 16 + qy + p.shift, x = wx * 16 + qx + p.shift;
    if (y >= p.hp) y -= p.hp;
    if (x >= p.wp) x -= p.wp;
    const int qpix = y * p.wp + x;
    const float* Qg = p.qkv + (size_t)head * p.T * D + (size_t)qpix * D;
    float qv[2][8];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        if constexpr (D == 24) {
            // both halves of the packed second step hold dims 16..23
            const int d0 = s == 0 ? 8 * h : 16;
            const f32x4 a = *(const f32x4*)(Qg + d0), b = *(const f32x4*)(Qg + d0 + 4);
#pragma unroll
            for (int j = 0; j < 4; ++j) qv[s][j] = a[j], qv[s][4 + j] = b[j];
        } else {
            const int d0 = 16 * s + 8 * h;
#pragma unroll
            for (int j = 0; j < 8; j += 2) {
                const bool live = d0 + j + 2 <= D;
                const float2 v = *(const float2*)(live ? Qg + d0 + j : hat_zero_row);
                qv[s][j] = v.x;
                qv[s][j + 1] = v.y;
            }
        }
    }
#pragma unroll
    for (int s = 0; s < 2; ++s) {
#pragma unroll
        for (int j = 0; j < 8; ++j) qv[s][j] *= p.qscale;
        split2_x8(qv[s], qb[s]);
    }
    if constexpr (D == 24) qb[1][0] = h ? qb[1][1] : qb[1][0];
    return qpix;
}

// The lane's K rows for S^T = K Q^T over 32-key tiles of two planes [keys][KS]
// (A = 32 keys x 16 dims: lane l gives key l % 32, dims 8h .. 8h + 7 of the step).
// Step 0 (dims 0..15) is the three products of mfma3. For D = 24, step 1 has only
// dims 16..23, so each MFMA carries two products, one per lane half: [k1 | k1] .
// [q0 | q1], then [k0 | k0] . [q0 | q1] (half 0 | half 1), two MFMAs for the
// three products (k1 q1 comes along). For D = 30 step 1 is dims 16..31 (30, 31
// zero) as step 0.
template <int D, int KS, int KPL>
struct AttnxKRows {
    const unsigned short *r0, *r1;
    __device__ __forceinline__ void init(const unsigned short* Kp, int ql, int h)
    {
        r0 = Kp + ql * KS + 8 * h;
        r1 = Kp + ql * KS + 16 + (D == 24 ? 0 : 8 * h);
    }
    // s += K Q^T for the tile whose first key row is koff elements in
    __device__ __forceinline__ f32x16 qk(int koff, const u32x4 (&qb)[2][2], f32x16 s) const
    {
        const u32x4 k0[2] = {*(const u32x4*)(r0 + koff), *(const u32x4*)(r0 + KPL + koff)};
        const u32x4 k1[2] = {*(const u32x4*)(r1 + koff), *(const u32x4*)(r1 + KPL + koff)};
        s = mfma3(k0, qb[0], s);
        if constexpr (D == 24) {
            s = mfma_f16(k1[1], qb[1][0], s);
            return mfma_f16(k1[0], qb[1][0], s);
        } else {
            return mfma3(k1, qb[1], s);
        }
    }
};

// e = exp2(s) for a lane's 16 scores of its item's first 32 keys (in log2 units, the
// shift mask left out), and whether the base-0 pass is likely to stand
// (attnx_item_done): no score so large that a later one is likely to reach 2^16, and
// a share of the denominator that makes 96 of 256 keys. The pass is checked at its end whatever
// this says; what it decides is that scores of a wider spread, as trained networks
// have them, go to the SAFE form at once instead of after a whole base-0 pass. A
// limit of 12 let through waves that met 2^16 later (q . k of 3 units at head_dim
// 24: 244 us against 228). Wave-uniform.
__device__ __forceinline__ bool attnx_flat(const f32x16& s, float (&e)[16])
{
    float mx = s[0], sum = 0.0f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        e[i] = fast_exp2(s[i]);
        mx = fmaxf(mx, s[i]);
        sum += e[i];
    }
    return __all(sum >= 6.0f && mx <= 10.0f);
}

// The same from the largest score alone (of 16 keys, one of 576 / 18 for the same
// denominator; low: whether to ask for that): the OCA kernels have no registers for
// the probabilities.
__device__ __forceinline__ bool attnx_flat(const f32x16& s, bool low)
{
    float mx = s[0];
#pragma unroll
    for (int i = 1; i < 16; ++i) mx = fmaxf(mx, s[i]);
    return __all(mx <= 10.0f && (!low || mx >= -1.0f));
}

// O^T (with the softmax denominator in row D) of the lane's query over the
// item's 256 keys. SAFE: the online softmax (the running base raised when a
// score exceeds it by more than 8, in log2 units), as the reference subtracts
// the row maximum (cpu.rs:801-812). Otherwise the base is 0: P = exp2(s)
// straight from the scores, no maximum, no subtraction, no rescaling (16 VALU
// a tile fewer); the caller checks the result and runs the SAFE form instead
// when a sum could have overflowed or lost its range (see attnx_item_done), or
// when the first tile says so (attnx_flat: zeros are returned, which fail the check).
// Either way o / o[row D] is the softmax-weighted sum, the same quantity.
template <int D, bool MASKED, bool SAFE>
__device__ __forceinline__ f32x16 attnx_tiles(const AttnArgs& p, const unsigned char* lds, int wi,
                                              const u32x4 (&qb)[2][2])
{
    using X = AttnXShape<D>;
    constexpr int NKT = X::NK / 32;
    const unsigned short* Kp = (const unsigned short*)lds;
    const unsigned short* Vp = Kp + 2 * X::KPL;
    const float* Tb = (const float*)(Vp + 2 * X::VPL);

    const int wy = wi / p.nx, wx = wi - (wi / p.nx) * p.nx;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform, in a scalar register
    const int ql = lane & 31, h = lane >> 5;
    const int q = wave * 32 + ql;
    const int qy = q >> 4, qx = q & 15;
    const int sw_rbase = 960 - ((qy + 15) * 31 + qx + 15 - 4 * h);
    const float NEG = -100.0f * HAT_LOG2E;
    const bool mrow = MASKED && wy == p.ny - 1;
    const bool mcol = MASKED && wx == p.nx - 1;
    const bool r_lo = mrow && (qy & 8), r_hi = mrow && !(qy & 8);
    const bool c_lo = mcol && (qx & 8), c_hi = mcol && !(qx & 8);
    const float madd[2][2] = {{(r_lo || c_lo) ? NEG : 0.0f, (r_lo || c_hi) ? NEG : 0.0f},
                              {(r_hi || c_lo) ? NEG : 0.0f, (r_hi || c_hi) ? NEG : 0.0f}};
    static_assert(D < 32, "a spare V^T row is needed");

    // The lane's V^T row (dims past D read row D: their outputs are not used)
    // and K rows.
    const unsigned short* vrow = Vp + (ql < D ? ql : D) * X::VS + 8 * h;
    AttnxKRows<D, X::KS, X::KPL> kr;
    kr.init(Kp, ql, h);

    f32x16 o;
#pragma unroll
    for (int i = 0; i < 16; ++i) o[i] = 0.0f;
    float mrun = SAFE ? -INFINITY : 0.0f;

// unrolled: the K, V and bias addresses of every tile are immediate offsets
#pragma unroll
    for (int kt = 0; kt < NKT; ++kt) {
        // S^T = bias (+ mask) + K Q^T
        f32x16 s;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int key0 = kt * 32 + (i >> 2) * 8 + (i & 3);
            const int ky = key0 >> 4, kx = key0 & 15;
            float b = Tb[sw_rbase + (ky * 31 + kx)];
            if (MASKED && (SAFE || kt > 0)) b += madd[(ky >> 3) & 1][(kx >> 3) & 1];
            s[i] = b;
        }
        s = kr.qk(kt * 32 * X::KS, qb, s);
        float e[16];
        if (!SAFE && kt == 0) {
            if (!attnx_flat(s, e)) return o;
            if (MASKED) {
                // key rows 0 and 1; a masked probability is 2^-132 at most, 0 in f16
#pragma unroll
                for (int i = 0; i < 16; ++i) e[i] = madd[0][(i >> 2) & 1] == 0.0f ? e[i] : 0.0f;
            }
        }
        if constexpr (SAFE) {
            float mx = -INFINITY;
#pragma unroll
            for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s[i]);
            if (kt == 0 || __any(mx > mrun + 8.0f)) {  // wave-uniform
                mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
                const float mnew = fmaxf(mrun, mx);
                const float corr = fast_exp2(mrun - mnew);
#pragma unroll
                for (int i = 0; i < 16; ++i) o[i] *= corr;
                mrun = mnew;
            }
        }
        // O^T += V^T P^T, P = exp2(S - base): the B operand of step st is
        // registers 8st .. 8st+7, split.
#pragma unroll
        for (int st = 0; st < 2; ++st) {
            float pv[8];
#pragma unroll
            for (int j = 0; j < 8; ++j)
                pv[j] = !SAFE && kt == 0 ? e[8 * st + j]
                                         : fast_exp2(SAFE ? s[8 * st + j] - (mrun - ATTNX_SAFE_UP) : s[8 * st + j]);
            u32x4 pb[2], va[2];
            split2_x8(pv, pb);
#pragma unroll
            for (int pl = 0; pl < 2; ++pl) va[pl] = *(const u32x4*)(vrow + pl * X::VPL + kt * 32 + 16 * st);
            o = mfma3(va, pb, o);
        }
    }
    return o;
}

// Whether an item's base-0 pass (attnx_tiles with SAFE false) may stand, for
// every query of the wave: the denominator at least 32 and every accumulator
// finite. A probability that left f16's range is infinite, and with it the sum: a
// finite one means that none did. The lower end bounds what the subnormal parts of
// the probabilities lose, up to 2^-25 of each of at most 576: 5.4e-7 of the
// denominator were all of them to fall the same way, 1e-8 as roundings do. A window
// of 256 scores around 0 has denominator 256; with the row maximum subtracted
// (ATTNX_SAFE_UP above it) it lies in [2^6, 576 * 2^14]. Wave-uniform.
template <int D>
__device__ __forceinline__ bool attnx_item_done(const f32x16& o)
{
    constexpr int RH = (D % 8) / 4, RR = (D / 8) * 4 + D % 4;
    const int ql = threadIdx.x & 31;
    const float ltot = __shfl(o[RR], ql + 32 * RH, 64);
    bool ok = ltot >= 32.0f;
#pragma unroll
    for (int i = 0; i < 16; ++i) ok = ok && __builtin_isfinite(o[i]);
    return __all(ok);
}

// out[query][head * D + d] = O^T[d] / O^T[D] for the lane's query.
template <int D>
__device__ __forceinline__ void attnx_store(const AttnArgs& p, int head, int qpix, const f32x16& o)
{
    constexpr int RH = (D % 8) / 4, RR = (D / 8) * 4 + D % 4;
    const int lane = threadIdx.x & 63;
    const int ql = lane & 31, h = lane >> 5;
    const float ltot = __shfl(o[RR], ql + 32 * RH, 64);
    const float inv = 1.0f / ltot;
    float* orow = p.out + (size_t)qpix * p.C + head * D;
#pragma unroll
    for (int i4 = 0; i4 < 4; ++i4) {
        const int d0 = 8 * i4 + 4 * h;
        if (D % 4 == 0) {
            if (d0 + 3 < D)
                *(float4*)(orow + d0) = make_float4(o[i4 * 4] * inv, o[i4 * 4 + 1] * inv,
                                                    o[i4 * 4 + 2] * inv, o[i4 * 4 + 3] * inv);
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (d0 + j < D) orow[d0 + j] = o[i4 * 4 + j] * inv;
        }
    }
}

template <int D, bool MASKED>
__device__ __forceinline__ void attnx_compute(const AttnArgs& p, const unsigned char* lds, int wi, int head,
                                              const u32x4 (&qb)[2][2], int qpix)
{
    f32x16 o = attnx_tiles<D, MASKED, false>(p, lds, wi, qb);
    if (!attnx_item_done<D>(o)) {  // wave-uniform
        // the same LDS through an offset the compiler cannot see is zero, so
        // that it does not keep the first pass's loaded values for this one
        int z = 0;
        asm volatile("" : "+s"(z));
        o = attnx_tiles<D, MASKED, true>(p, lds + z, wi, qb);
    }
    attnx_store<D>(p, head, qpix, o);
}

template <int D>
__device__ __forceinline__ void attnx_item_kernel(const AttnArgs& p, unsigned char* lds)
{
    using S = AttnShape<D, false>;
    using X = AttnXShape<D>;
    // The CAB's gate, which only the tail after this launch needs, as a block of
    // its own ahead of the items (one more column of the grid), so that no item
    // waits behind it: with the first item in the same block, small planes waited
    // for it (HAT-S 64 x 64: 39.2 -> 13.3 us a launch; HAT 512 x 512, where the
    // gate outlasted the items: 337 -> 246).
    const int lead = p.with_gate || p.with_se ? 1 : 0;
    const int wi = (int)blockIdx.x - lead, head = blockIdx.y;
    if (wi < 0) {  // block-uniform
        static_assert(4 * CAB_GATE_LDS <= X::LDS_BYTES && 4 * SE_GATE_LDS <= X::LDS_BYTES,
                      "the gates' scratch fits the item LDS");
        if (head != 0) return;
        if (p.with_gate) cab_gate_body<8>(p.gate, (float*)lds);
        else se_gate_body<8>(p.se, (float*)lds);
        return;
    }
    unsigned short* Kp = (unsigned short*)lds;
    unsigned short* Vp = Kp + 2 * X::KPL;
    float* Tb = (float*)(Vp + 2 * X::VPL);
    u32x4 qb[2][2];
    int qpix;
    {
        typename S::vec ks[S::NE], vs[S::NE];
        attn_fetch<D, false>(p, wi, head, ks, vs);
        AttnTableRegs<D, false> tr;
        attn_table_load<D, false>(p, head, tr);
        qpix = attnx_query<D>(p, wi, head, qb);
        attnx_stash<D>(Kp, Vp, ks, vs);
        attn_table_store<D, false>(Tb, tr);
    }
    __syncthreads();
    if (p.shift > 0 && (wi / p.nx == p.ny - 1 || wi % p.nx == p.nx - 1))
        attnx_compute<D, true>(p, lds, wi, head, qb, qpix);
    else
        attnx_compute<D, false>(p, lds, wi, head, qb, qpix);
}

// ---------------------------------------------------------------------------
// OCA (overlapping cross-attention: 576 keys of the 24x24 unfold with padding
// 4, zero outside the plane, biased and unmasked; hat_arch.py:373-427,
// cpu.rs:852-900), one (window, head) item per block. The two planes of K and
// V^T of 576 keys and the table would need 120 KB of LDS (D = 30: 171), so an item
// runs as parts of NK keys (D = 24: three of 192, key rows 0-7, 8-15, 16-23; D = 30:
// six of 96) that share the softmax; each part is split into LDS between two
// barriers and computed, and the next part's fetch into registers is issued
// before the computing, so that its latency runs under this part's tiles. At
// most 80 KB of LDS and 128 VGPRs, so that two blocks share a CU and one's
// staging overlaps the other's MFMAs.

template <int D, int NK>
struct AttnXOcaShape {
    static constexpr int NKEYS = 576;
    static_assert(NKEYS % NK == 0 && NK % 32 == 0, "whole 32-key tiles, whole parts");
    static constexpr int NPART = NKEYS / NK;
    static constexpr int KS = D == 24 ? 24 : 40;
    static constexpr int VS = NK + 8;                 // V^T row stride: 16 rows of a phase on distinct banks
    static constexpr int KPL = NK * KS, VPL = (D + 1) * VS;
    static constexpr int TROWS = 1521;
    static constexpr int LDS_BYTES = 2 * 2 * (KPL + VPL) + 4 * TROWS;
    static constexpr int U = D % 4 == 0 ? 4 : 2;       // floats per staging unit
    static constexpr int NE = (NK * D / U + 511) / 512;
    using vec = typename pick_t<U == 4, float4, float2>::type;
};

// This thread's share of part `part` of item (wi, head): K and V units.
template <int D, int NK>
__device__ __forceinline__ void attnx_oca_fetch(const AttnArgs& p, int wi, int head, int part,
                                                typename AttnXOcaShape<D, NK>::vec (&ks)[AttnXOcaShape<D, NK>::NE],
                                                typename AttnXOcaShape<D, NK>::vec (&vs)[AttnXOcaShape<D, NK>::NE])
{
    using X = AttnXOcaShape<D, NK>;
    using vec = typename X::vec;
    constexpr int PER_KEY = D / X::U;
    const float* Kg = p.qkv + (size_t)(p.heads + head) * p.T * D;
    const float* Vg = p.qkv + (size_t)(2 * p.heads + head) * p.T * D;
#pragma unroll
    for (int i = 0; i < X::NE; ++i) {
        const int e = threadIdx.x + i * 512;
        vec kv{}, vv{};
        if (e < NK * PER_KEY) {
            const int kl = e / PER_KEY, d = (e - kl * PER_KEY) * X::U;
            const int pix = attn_key_pixel<true>(p, wi, part * NK + kl);
            if (pix >= 0) {
                kv = *(const vec*)(Kg + (size_t)pix * D + d);
                vv = *(const vec*)(Vg + (size_t)pix * D + d);
            }
        }
        ks[i] = kv;
        vs[i] = vv;
    }
}

template <int D, int NK>
__device__ __forceinline__ void attnx_oca_stash(unsigned short* Kp, unsigned short* Vp,
                                                const typename AttnXOcaShape<D, NK>::vec (&ks)[AttnXOcaShape<D, NK>::NE],
                                                const typename AttnXOcaShape<D, NK>::vec (&vs)[AttnXOcaShape<D, NK>::NE])
{
    using X = AttnXOcaShape<D, NK>;
    constexpr int PER_KEY = D / X::U;
#pragma unroll
    for (int i = 0; i < X::NE; ++i) {
        const int e = threadIdx.x + i * 512;
        if (e < NK * PER_KEY) {
            const int k = e / PER_KEY, d = (e - k * PER_KEY) * X::U;
            float kv[4], vv[4];
            if constexpr (X::U == 4) {
                kv[0] = ks[i].x, kv[1] = ks[i].y, kv[2] = ks[i].z, kv[3] = ks[i].w;
                vv[0] = vs[i].x, vv[1] = vs[i].y, vv[2] = vs[i].z, vv[3] = vs[i].w;
            } else {
                kv[0] = ks[i].x, kv[1] = ks[i].y, kv[2] = kv[3] = 0.f;
                vv[0] = vs[i].x, vv[1] = vs[i].y, vv[2] = vv[3] = 0.f;
            }
            const int pos = vpos(k);
#pragma unroll
            for (int j = 0; j < X::U; j += 2) {
                unsigned k0, k1, v0, v1;
                split2_pk(kv[j], kv[j + 1], k0, k1);
                *(unsigned*)(Kp + 0 * X::KPL + k * X::KS + d + j) = k0;
                *(unsigned*)(Kp + 1 * X::KPL + k * X::KS + d + j) = k1;
                split2_pk(vv[j], vv[j + 1], v0, v1);
                Vp[0 * X::VPL + (d + j) * X::VS + pos] = (unsigned short)v0;
                Vp[0 * X::VPL + (d + j + 1) * X::VS + pos] = (unsigned short)(v0 >> 16);
                Vp[1 * X::VPL + (d + j) * X::VS + pos] = (unsigned short)v1;
                Vp[1 * X::VPL + (d + j + 1) * X::VS + pos] = (unsigned short)(v1 >> 16);
            }
        }
    }
}

// Whether the scores of one 32-key tile of part 0 are attnx_flat.
template <int D, int NK>
__device__ __forceinline__ bool attnx_oca_ask(const unsigned char* lds, int kt, const u32x4 (&qb)[2][2])
{
    using X = AttnXOcaShape<D, NK>;
    const unsigned short* Kp = (const unsigned short*)lds;
    const float* Tb = (const float*)(Kp + 2 * X::KPL + 2 * X::VPL);
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));  // the addresses are not to be kept for the tiles
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform, in a scalar register
    const int ql = lane & 31, h = lane >> 5, q = wave * 32 + ql;
    AttnxKRows<D, X::KS, X::KPL> kr;
    kr.init(Kp, ql, h);
    f32x16 s;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int key = kt * 32 + (i >> 2) * 8 + (i & 3) + 4 * h;
        s[i] = Tb[600 - ((q >> 4) * 39 + (q & 15)) + key + 15 * (int)((unsigned)key / 24u)];
    }
    return attnx_flat(kr.qk(kt * 32 * X::KS, qb, s), true);
}

// One part's key tiles onto the running (o, mrun) of the item; SAFE as in attnx_tiles
// (without it the base stays 0 and mrun is not used). False: not SAFE, and the part's
// first tile was not attnx_flat (the item's first is asked on the low side too);
// nothing was done. A later part's first tile can turn a wave to SAFE in the middle
// of the item: base 0 is a maximum of ATTNX_SAFE_UP.
template <int D, int NK, bool SAFE>
__device__ __forceinline__ bool attnx_oca_compute(const unsigned char* lds, int part, const u32x4 (&qb)[2][2],
                                                  f32x16& o, float& mrun)
{
    using X = AttnXOcaShape<D, NK>;
    constexpr int NKT = NK / 32;
    const unsigned short* Kp = (const unsigned short*)lds;
    const unsigned short* Vp = Kp + 2 * X::KPL;
    const float* Tb = (const float*)(Vp + 2 * X::VPL);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform, in a scalar register
    const int ql = lane & 31, h = lane >> 5;
    const int q = wave * 32 + ql;
    const int qy = q >> 4, qx = q & 15;
    // idx = (ky*39 + kx) - (qy*39 + qx) + 600 on the rotated table (attn.hip)
    const int oca_base = 600 - (qy * 39 + qx);
    const unsigned short* vrow = Vp + (ql < D ? ql : D) * X::VS + 8 * h;
    AttnxKRows<D, X::KS, X::KPL> kr;
    kr.init(Kp, ql, h);
#pragma unroll 1
    for (int kt = 0; kt < NKT; ++kt) {
        f32x16 s;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int key = part * NK + kt * 32 + (i >> 2) * 8 + (i & 3) + 4 * h;
            const int ky = (int)((unsigned)key / 24u);
            s[i] = Tb[oca_base + key + 15 * ky];
        }
        s = kr.qk(kt * 32 * X::KS, qb, s);
        if (!SAFE && kt == 0 && !attnx_flat(s, part == 0)) return false;
        if constexpr (SAFE) {
            float mx = -INFINITY;
#pragma unroll
            for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s[i]);
            if (part == 0 && kt == 0) {
                mrun = fmaxf(mx, __shfl_xor(mx, 32, 64));  // o is zero
            } else if (__any(mx > mrun + 8.0f)) {  // wave-uniform
                mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
                const float mnew = fmaxf(mrun, mx);
                const float corr = fast_exp2(mrun - mnew);
#pragma unroll
                for (int i = 0; i < 16; ++i) o[i] *= corr;
                mrun = mnew;
            }
        }
#pragma unroll
        for (int st = 0; st < 2; ++st) {
            float pv[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) pv[j] = fast_exp2(SAFE ? s[8 * st + j] - (mrun - ATTNX_SAFE_UP) : s[8 * st + j]);
            u32x4 pb[2], va[2];
            split2_x8(pv, pb);
#pragma unroll
            for (int pl = 0; pl < 2; ++pl) va[pl] = *(const u32x4*)(vrow + pl * X::VPL + kt * 32 + 16 * st);
            o = mfma3(va, pb, o);
        }
    }
    return true;
}

template <int D, int NK>
__device__ __forceinline__ void attnx_oca_kernel(const AttnArgs& p, unsigned char* lds)
{
    using X = AttnXOcaShape<D, NK>;
    const int wi = blockIdx.x, head = blockIdx.y;
    unsigned short* Kp = (unsigned short*)lds;
    unsigned short* Vp = Kp + 2 * X::KPL;
    float* Tb = (float*)(Vp + 2 * X::VPL);
    // Written once (no part's staging touches them): row D of V^T (ones in the
    // high plane), K dims 30, 31 (D = 30).
    for (int e = threadIdx.x; e < 2 * (NK / 2); e += 512) {
        const int pl = e / (NK / 2), k2 = e - pl * (NK / 2);
        *(unsigned*)(Vp + pl * X::VPL + D * X::VS + 2 * k2) = pl == 0 ? 0x3c003c00u : 0u;  // f16 1.0 pairs
    }
    if (D == 30) {
        for (int e = threadIdx.x; e < 2 * NK; e += 512) {
            const int pl = e / NK, k = e - pl * NK;
            *(unsigned*)(Kp + pl * X::KPL + k * X::KS + 30) = 0u;
        }
    }
    const int lane = threadIdx.x & 63;
    const int ql = lane & 31, h = lane >> 5;
    constexpr int RH = (D % 8) / 4, RR = (D / 8) * 4 + D % 4;
    typename X::vec ks[X::NE], vs[X::NE];
    u32x4 qb[2][2];
    int qpix;
    {
        attnx_oca_fetch<D, NK>(p, wi, head, 0, ks, vs);
        AttnTableRegs<D, true> tr;
        attn_table_load<D, true>(p, head, tr);
        qpix = attnx_query<D>(p, wi, head, qb);
        attn_table_store<D, true>(Tb, tr);
    }
    f32x16 o;
#pragma unroll
    for (int i = 0; i < 16; ++i) o[i] = 0.0f;
    float mrun = 0.0f;
    bool safe = false;  // this wave's form (attnx_flat)
#pragma unroll 1
    for (int part = 0; part < X::NPART; ++part) {
        if (part > 0) __syncthreads();  // every read of the previous part's K and V is done
        attnx_oca_stash<D, NK>(Kp, Vp, ks, vs);
        __syncthreads();
        // In the plane's top windows part 0's first four rows of keys are padding,
        // which says nothing about the others: at head_dim 24, where a part has eight,
        // its first tile with others is asked as well (here, where the registers of
        // the next part's fetch are still free).
        if (NK > 4 * 24 && part == 0 && wi < p.nx) safe = !attnx_oca_ask<D, NK>(lds, 3, qb);
        // the next part's K and V in flight while this part's tiles run (the
        // registers are free once stashed; same-box with the bf16 split: OCA head_dim
        // 30 677 -> 661 us, head_dim 24 589 -> 585)
        if (part + 1 < X::NPART) attnx_oca_fetch<D, NK>(p, wi, head, part + 1, ks, vs);
        if (!safe) {
            safe = !attnx_oca_compute<D, NK, false>(lds, part, qb, o, mrun);
            mrun = ATTNX_SAFE_UP;  // what base 0 is as a maximum
        }
        if (safe) attnx_oca_compute<D, NK, true>(lds, part, qb, o, mrun);
    }
    // The parts are staged by the whole block, so the block redoes the item
    // with the max-subtracted softmax if any of its waves needs it.
    __shared__ int item_ok[8];
    const bool ok = attnx_item_done<D>(o);
    if (lane == 0) item_ok[threadIdx.x >> 6] = ok;
    __syncthreads();  // also: every read of the last part's K and V is done
    bool all_ok = true;
#pragma unroll
    for (int w = 0; w < 8; ++w) all_ok = all_ok && item_ok[w];
    if (!all_ok) {  // block-uniform
#pragma unroll
        for (int i = 0; i < 16; ++i) o[i] = 0.0f;
#pragma unroll 1
        for (int part = 0; part < X::NPART; ++part) {
            attnx_oca_fetch<D, NK>(p, wi, head, part, ks, vs);
            if (part > 0) __syncthreads();  // every read of the previous part's K and V is done
            attnx_oca_stash<D, NK>(Kp, Vp, ks, vs);
            __syncthreads();
            attnx_oca_compute<D, NK, true>(lds, part, qb, o, mrun);
        }
    }
    const float ltot = __shfl(o[RR], ql + 32 * RH, 64);
    const float inv = 1.0f / ltot;
    float* orow = p.out + (size_t)qpix * p.C + head * D;
#pragma unroll
    for (int i4 = 0; i4 < 4; ++i4) {
        const int d0 = 8 * i4 + 4 * h;
        if (D % 4 == 0) {
            if (d0 + 3 < D)
                *(float4*)(orow + d0) = make_float4(o[i4 * 4] * inv, o[i4 * 4 + 1] * inv,
                                                    o[i4 * 4 + 2] * inv, o[i4 * 4 + 3] * inv);
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (d0 + j < D) orow[d0 + j] = o[i4 * 4 + j] * inv;
        }
    }
}

#define ATTNX_OCA_INST(NAME, D, NK)                                                                 \
    extern "C" __global__ __launch_bounds__(512, 4) void NAME(AttnArgs p)                           \
    {                                                                                               \
        static_assert(AttnXOcaShape<D, NK>::LDS_BYTES <= 80 * 1024, "two blocks per CU");           \
        __shared__ __attribute__((aligned(16))) unsigned char lds[AttnXOcaShape<D, NK>::LDS_BYTES]; \
        attnx_oca_kernel<D, NK>(p, lds);                                                            \
    }

ATTNX_OCA_INST(hat_attnx_oca_d24, 24, 192)
ATTNX_OCA_INST(hat_attnx_oca_d30, 30, 96)

#define ATTNX_INST(NAME, D)                                                                  \
    extern "C" __global__ __launch_bounds__(512, 4) void NAME(AttnArgs p)                    \
    {                                                                                        \
        static_assert(AttnXShape<D>::LDS_BYTES <= 80 * 1024, "two blocks per CU");           \
        __shared__ __attribute__((aligned(16))) unsigned char lds[AttnXShape<D>::LDS_BYTES]; \
        attnx_item_kernel<D>(p, lds);                                                        \
    }

ATTNX_INST(hat_attnx_sw_d24, 24)
ATTNX_INST(hat_attnx_sw_d30, 30)
