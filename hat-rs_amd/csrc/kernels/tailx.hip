// The second half of a HAB (and of an OCAB), C = 144 and 180, on split-f16
// MFMA in one kernel (hat_arch.py HAB.forward / OCAB.forward; cpu.rs hab
// 1090-1166, ocab 983-1055; the reference GPU graph's proj, CAB conv2 and
// channel scale, adds, norm2, fc1 + GELU + fc2 and the next norm1,
// src/gpu.rs:469-588):
//
//   x'  = x + ao . Wp^T (+ nb(t1) . W2g^T, C = 144) (+ aux * gate * cscale,
//         C = 180) + bias
//   out = x' + fc2(gelu(fc1(LN2(x')))) + b2,  xn = LN_next(out) when asked
//
//   hat_habx_cab_ln, hat_habx180_hab_ln: the HAB's form; hat_habx, hat_habx180:
//   the OCAB's (no CAB, no next norm)
//
// ao is the attention output, nb(t1) the 3x3 neighbourhood of the folded CAB's
// conv1 output (k = tap*6 + ci, 54 values) and W2g / bias the gate-scaled conv2
// weights and combined bias written by the gate (hat_cab_gate's work); aux is
// the unfolded CAB's conv2 output. Products are the three-term split-f16 ones of
// common.h on v_mfma_f32_16x16x32_f16, weights as the A operand, tokens as B; a
// lane's four accumulators are four consecutive output channels of one token.
//
// Scales (powers of two, chosen on the host so that every operand lies inside
// f16's range): the projection's accumulators hold p.ps times the sum (the
// attention output comes scaled, the weights are), norm2's weight and bias leave
// its rows scaled, fc1's accumulators times p.h1 plus b1x are the hidden units
// times their scale, which GELU takes in its constants (gelu_scaled), and the
// output's accumulators hold p.ms times the result. Every scale comes out in a
// multiply-add that adds a bias.
//
// A block of 4 waves takes one 128-token row tile, 32 tokens a wave (each weight
// fragment read from LDS feeds two 16-token MFMA tiles), and streams its weights
// through two LDS buffers a stage at a time: stage s + 1 in flight while stage
// s's MFMAs run, a stage as many 32-k steps as a buffer holds (C = 144: two of
// the projection's or fc2's 144 rows, three of fc1's 96; C = 180: one of 192
// rows, or fc1's six of 32), so that the waves meet at a barrier about every
// hundred MFMAs each. Two blocks share a CU, so one block's reads and barriers
// overlap the other's MFMAs.
//
// x' is the projection's accumulators; norm2(x') is split once, into registers
// (72 or 96 of them: two f16 parts take what the fp32 value would), and is fc1's
// B operand for every part of the hidden layer: fc1's input columns are packed
// on the host in the order a lane holds x' (k-step ks of lane group g is the
// lane's tiles 2 ks and 2 ks + 1: channels 32 ks + 4 g + j and 32 ks + 16 + 4 g +
// j, j < 4), so no lane needs another's values. fc1's rows are packed so that
// its output tile t, row 4 g + r is unit 32 (t / 2) + 8 g + 4 (t % 2) + r of the
// part: fc2's 32-k step s finds units 32 s + 8 g .. +7 in tiles 2 s and 2 s + 1
// of lane group g, its weights in natural order. So neither x', norm2(x') nor
// the hidden layer leaves the registers.
//
// What bounds it: issue time (MFMA, GELU and the splits) and HBM about equally
// (HAT-S 512 x 512: 612 MB a launch, 110 us at the copy kernel's rate; 1350 MFMAs
// of 16 cycles a wave, 86 us). Measured against the six-product bf16 split, which
// walked the hidden layer with norm2(x') read back from memory and split again for
// every part: hat_habx_cab_ln 371.8 -> 250.8 us, hat_habx 324.7 -> 210.2 (HAT-S
// 512); hat_habx180_hab_ln 546 -> 375, hat_habx180 492 -> 304 (HAT 512);
// 50 -> 36 and 75 -> 50 at 64 x 64.
//
// Included after gemmx.hip (WcRows, split_pre2).

#define TX_WAVES 4
#define TX_ROWS (TX_WAVES * 32)

// Row statistics of a token over its C channels (C = 144: 36 per lane, 180:
// 45; NT = ceil(C / 16) tiles of which the last holds C % 16 real channels in
// lane group 0), the four lane groups of the token reducing with shuffles:
// two-pass mean, biased variance (cpu.rs:563-581); returns (mean, rstd).
template <int C>
__device__ __forceinline__ bool tx_live(int nt, int lg)
{
    constexpr int NT = (C + 15) / 16;
    return C % 16 == 0 || nt < NT - 1 || lg * 4 < C % 16;
}
template <int C>
__device__ __forceinline__ float2 tx_row_stats(const f32x4 (&v)[(C + 15) / 16], int lg, float eps)
{
    constexpr int NT = (C + 15) / 16;
    float s = 0.0f;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int j = 0; j < 4; ++j) s += v[nt][j];  // zeros past C
    s += __shfl_xor(s, 16, 64);
    s += __shfl_xor(s, 32, 64);
    const float mean = s / (float)C;
    float q = 0.0f;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float d = tx_live<C>(nt, lg) ? v[nt][j] - mean : 0.0f;
            q += d * d;
        }
    q += __shfl_xor(q, 16, 64);
    q += __shfl_xor(q, 32, 64);
    return make_float2(mean, 1.0f / sqrtf(q / (float)C + eps));
}

// v = acc * mi + b2 (Cs); out = v (amax_out: its largest magnitude too); with xn: xn = LN(v) by (nw, nb) = (Cs + 16 NT,
// Cs + 32 NT) (Cs zero past C).
template <int C>
__device__ __forceinline__ void tx_store_rows(const f32x4 (&acc)[2][(C + 15) / 16], const float* Cs, float mi, int mbase,
                                              int M, int lr, int lg, float eps, float* out, float* xn,
                                              unsigned* amax_out, unsigned* lds)
{
    constexpr int NT = (C + 15) / 16;
    float big = 0.0f;
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) {
        const int m = mbase + mt * 16 + lr;
        f32x4 v[NT];
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            const f32x4 b4 = *(const f32x4*)(Cs + nt * 16 + lg * 4);
#pragma unroll
            for (int j = 0; j < 4; ++j) v[nt][j] = __builtin_fmaf(acc[mt][nt][j], mi, b4[j]);
        }
        float2 st = make_float2(0.f, 0.f);
        if (xn) st = tx_row_stats<C>(v, lg, eps);
        if (m >= M) continue;
        if (amax_out) {
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                for (int j = 0; j < 4; ++j) big = finite_max(big, v[nt][j]);  // zeros past C
        }
        float* orow = out + (size_t)m * C + lg * 4;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
            if (tx_live<C>(nt, lg)) *(f32x4*)(orow + nt * 16) = v[nt];
        if (xn) {
            float* nrow = xn + (size_t)m * C + lg * 4;
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                const f32x4 w4 = *(const f32x4*)(Cs + 16 * NT + nt * 16 + lg * 4);
                const f32x4 b4 = *(const f32x4*)(Cs + 32 * NT + nt * 16 + lg * 4);
                f32x4 y;
#pragma unroll
                for (int j = 0; j < 4; ++j) y[j] = (v[nt][j] - st.x) * st.y * w4[j] + b4[j];
                if (tx_live<C>(nt, lg)) *(f32x4*)(nrow + nt * 16) = y;
            }
        }
    }
    if (amax_out) block_amax(amax_out, lds, big);
}

// The shape of a tail kernel: NT channel tiles, KS 32-k steps over the channels
// (HALF: the last one packed), the hidden layer in NP parts of HU units; the
// steps a stage holds: SP of the projection's (16 NT rows), S1 of fc1's (HU
// rows), S2 of fc2's (16 NT rows).
template <int C>
struct TailXShape {
    static constexpr int NT = (C + 15) / 16, ROWS = 16 * NT, KS = (C + 31) / 32;
    static constexpr bool HALF = C == 144;
    static constexpr int HU = tailx_hu(C), HT = HU / 16, NP = (2 * C + HU - 1) / HU, K2 = HU / 32;
    static constexpr int SP = C == 144 ? 2 : 1, S1 = C == 144 ? 3 : 6, S2 = C == 144 ? 2 : 1;
    static constexpr int STEP = 2 * ROWS * 32, STEP1 = 2 * HU * 32;  // elements of a step
    static constexpr int PART = KS * STEP1 + K2 * STEP;              // a part's fc1 and fc2 steps
    static constexpr int ceil_div(int a, int b) { return (a + b - 1) / b; }
    // 1 KB loads of n elements, the same number from every wave (the last ones
    // may read past the stage: the arrays end in TX_PAD elements of padding)
    static constexpr int loads(int n) { return ceil_div(ceil_div(n, 512), TX_WAVES) * TX_WAVES; }
    static constexpr int NLP = loads(SP * STEP), NL1 = loads(S1 * STEP1), NL2 = loads(S2 * STEP);
    static constexpr int BUF = (NLP > NL1 ? (NLP > NL2 ? NLP : NL2) : (NL1 > NL2 ? NL1 : NL2)) * 512;
    static_assert(HU % 32 == 0 && TX_PAD >= TX_WAVES * 512, "whole fc2 steps; padding for the last loads");
};

template <int C, bool CAB, bool HAB, bool LN>
__device__ __forceinline__ void habx_body(const TailXArgs& p)
{
    using S = TailXShape<C>;
    constexpr int NT = S::NT, KS = S::KS, HT = S::HT;
    // the projection's stages: its own steps, then (CAB) one of conv2's two
    constexpr int NPS = S::ceil_div(KS, S::SP) + (CAB ? 1 : 0);
    constexpr int PB = NPS & 1;  // the MLP's first stage's buffer
    static_assert(!CAB || S::SP == 2, "conv2's two steps are one stage");
    constexpr int F1 = S::ceil_div(KS, S::S1), F2 = S::ceil_div(S::K2, S::S2);
    static_assert((F1 + F2) % 2 == 0, "a part leaves the buffers' parity as it was");
    // the two stage buffers as two LDS objects, so that the compiler sees that
    // reads of one need not wait for the copy into the other
    __shared__ __attribute__((aligned(16))) unsigned short Ws0[S::BUF];
    __shared__ __attribute__((aligned(16))) unsigned short Ws1[S::BUF];
    __shared__ __attribute__((aligned(16))) float Cp[(HAB ? 2 : 1) * 16 * NT];  // the projection's bias (HAB: and gate * cscale)
    __shared__ __attribute__((aligned(16))) float Cn[2 * 16 * NT];              // norm2 w, b
    __shared__ __attribute__((aligned(16))) float Cs[3 * 16 * NT];              // b2, next norm w, b (all zero past C)
    __shared__ unsigned big;                                                    // block_amax's
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform, in a scalar register
    const int lr = lane & 15, lg = lane >> 4;
    const int M = p.M;
    if ((int)blockIdx.x * TX_ROWS >= M) return;  // whole block, before any barrier
    if (tid == 0) big = 0;

    // n loads of a stage into buffer `par`
    auto issue = [&](auto nlv, auto parv, const unsigned short* src) {
        wc_issue<decltype(nlv)::value, TX_WAVES>(decltype(parv)::value ? Ws1 : Ws0, src, wave, lane);
    };
    // the loads of the step range [k0, ...) of a projection stage: at most SP
    auto issue_proj = [&](auto sv) {
        constexpr int s = decltype(sv)::value;
        constexpr int own = S::ceil_div(KS, S::SP);
        if constexpr (s < own) {
            constexpr int n = (KS - s * S::SP < S::SP ? KS - s * S::SP : S::SP) * S::STEP;
            issue(CInt<S::loads(n)>{}, CInt<(s & 1)>{}, p.w + (size_t)s * S::SP * S::STEP);
        } else if constexpr (CAB && s == own) {
            issue(CInt<S::loads(2 * S::STEP)>{}, CInt<(s & 1)>{}, p.w2gx);
        } else {
            issue(CInt<S::NL1>{}, CInt<PB>{}, p.wm);  // the MLP's first stage
        }
    };
    auto stage_begin = [&] {
        __builtin_amdgcn_s_waitcnt(0);  // this wave's loads of the stage (and its operands) have landed
        __syncthreads();                // everyone's have, and everyone is done with the stage before
    };

    issue_proj(CInt<0>{});
    for (int i = tid; i < (HAB ? 2 : 1) * 16 * NT; i += TX_WAVES * 64) {
        const int part = i / (16 * NT), c = i - part * 16 * NT;
        Cp[i] = c >= C ? 0.0f : part == 0 ? p.bias[c] : p.gate[c] * p.cscale;
    }
    for (int i = tid; i < 2 * 16 * NT; i += TX_WAVES * 64) {
        const int part = i / (16 * NT), c = i - part * 16 * NT;
        Cn[i] = c >= C ? 0.0f : part == 0 ? p.inw[c] : p.inb[c];
    }
    for (int i = tid; i < 3 * 16 * NT; i += TX_WAVES * 64) {
        const int part = i / (16 * NT), c = i - part * 16 * NT;
        Cs[i] = c >= C ? 0.0f : part == 0 ? p.b2[c] : LN ? (part == 1 ? p.nw[c] : p.nb[c]) : 0.0f;
    }
    const int mbase = blockIdx.x * TX_ROWS + wave * 32;
    // acc = the block input's rows in the projection's scale (zeros past M, C)
    f32x4 acc[2][NT];
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) {
        const int m = mbase + mt * 16 + lr;
        const float* row = p.res + (size_t)(m < M ? m : 0) * C + lg * 4;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = load_or_zero(row + nt * 16, m < M && tx_live<C>(nt, lg));
    }
    // HAB: conv2's output rows, added (times gate * cscale) to the block input
    // here, where registers are free, rather than to x' (52 registers spilled)
    f32x4 aux[HAB ? 2 : 1][HAB ? NT : 1];
    if constexpr (HAB) {
#pragma unroll
        for (int mt = 0; mt < 2; ++mt) {
            const int m = mbase + mt * 16 + lr;
            const float* row = p.aux + (size_t)(m < M ? m : 0) * C + lg * 4;
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) aux[mt][nt] = load_or_zero(row + nt * 16, m < M && tx_live<C>(nt, lg));
        }
    }

    // ---- the projection: acc = ps (x + ao . Wp^T (+ nb(t1) . W2g^T))
    {
        WcRows<C> ar;
        ar.init(p.a, mbase, M, lr);
        // ao's rows: one stage ahead
        f32x4 y[2][S::SP][2][2];
        auto load_rows = [&](auto sv) {
            constexpr int s = decltype(sv)::value;
#pragma unroll
            for (int i = 0; i < S::SP; ++i) {
                const int ks = s * S::SP + i;
                if (ks >= KS) break;
                if (S::HALF && ks == KS - 1) ar.load_half(lg, y[s & 1][i]);
                else ar.load(ks, lg, y[s & 1][i]);
            }
        };
        // conv2's B operand for its k-step s: the 3x3 neighbourhood of t1 at
        // this lane's tokens, k = 32 s + 8 lg + j = tap*6 + ci (pairs of
        // channels; taps outside the plane and k >= 54 read zeros)
        auto gather_t1 = [&](int s, f32x4 (&dst)[2][2]) {
#pragma unroll
            for (int mt = 0; mt < 2; ++mt) {
                const int m = mbase + mt * 16 + lr;
                const bool alive = m < M;
                const int yq = m / p.W, xq = m - yq * p.W;
#pragma unroll
                for (int j = 0; j < 8; j += 2) {
                    const int k = s * 32 + lg * 8 + j, tap = k / 6, ci = k - tap * 6;
                    const int yy = yq + tap / 3 - 1, xx = xq + tap % 3 - 1;
                    const bool ok = alive && tap < 9 && yy >= 0 && yy < p.H && xx >= 0 && xx < p.W;
                    const float2 v =
                        *(const float2*)(ok ? p.t1 + ((size_t)yy * p.W + xx) * CAB_CS + ci : hat_zero_row);
                    dst[mt][j / 4][j % 4] = v.x;
                    dst[mt][j / 4][j % 4 + 1] = v.y;
                }
            }
        };
        load_rows(CInt<0>{});
        auto proj_stage = [&](auto sv) {
            constexpr int s = decltype(sv)::value;
            constexpr int own = S::ceil_div(KS, S::SP);
            const unsigned short* W = s & 1 ? Ws1 : Ws0;
            stage_begin();
            issue_proj(CInt<s + 1>{});
            if constexpr (s == 0) {
#pragma unroll
                for (int mt = 0; mt < 2; ++mt)
#pragma unroll
                    for (int nt = 0; nt < NT; ++nt) {
                        if constexpr (HAB) {
                            const f32x4 g4 = *(const f32x4*)(Cp + 16 * NT + nt * 16 + lg * 4);
#pragma unroll
                            for (int j = 0; j < 4; ++j)
                                acc[mt][nt][j] = __builtin_fmaf(aux[mt][nt][j], g4[j], acc[mt][nt][j]);
                        }
                        acc[mt][nt] *= p.ps;
                    }
            }
            if constexpr (s + 1 < own) load_rows(CInt<s + 1>{});
            else if constexpr (CAB && s + 1 == own) {
#pragma unroll
                for (int i = 0; i < 2; ++i) gather_t1(i, y[(s + 1) & 1][i]);
            }
#pragma unroll
            for (int i = 0; i < S::SP; ++i) {
                const int ks = s * S::SP + i;
                if (s < own && ks >= KS) break;
                u32x4 xb[2][2];
                if (S::HALF && s < own && ks == KS - 1) {
#pragma unroll
                    for (int mt = 0; mt < 2; ++mt) xb[mt][0] = half_operand(y[s & 1][i][mt][0]);
                    ws_mma2<NT, S::ROWS, true>(W + i * S::STEP, lr, lg, xb, acc);
                } else {
                    split_pre2(y[s & 1][i], xb);
                    ws_mma2<NT, S::ROWS>(W + i * S::STEP, lr, lg, xb, acc);
                }
            }
        };
        proj_stage(CInt<0>{});
        proj_stage(CInt<1>{});
        proj_stage(CInt<2>{});
        if constexpr (NPS > 3) proj_stage(CInt<3>{});
        if constexpr (NPS > 4) {
            proj_stage(CInt<4>{});
            proj_stage(CInt<5>{});
        }
        static_assert(NPS <= 6 && NPS != 5, "the stages above");
    }
    // x' = acc / ps + bias, then norm2 of it split into fc1's operands yb, and
    // acc = ms x'
    u32x4 yb[2][KS][2];
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            const f32x4 b4 = *(const f32x4*)(Cp + nt * 16 + lg * 4);
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[mt][nt][j] = __builtin_fmaf(acc[mt][nt][j], p.pi, b4[j]);
        }
        float2 st = tx_row_stats<C>(acc[mt], lg, p.eps);
        // an opaque copy of the mean: otherwise the compiler keeps the
        // statistics' x' - mean live beside x' for the norm
        asm volatile("" : "+v"(st.x));
        auto norm_tile = [&](int nt, float* f) {
            const f32x4 w4 = *(const f32x4*)(Cn + nt * 16 + lg * 4), b4 = *(const f32x4*)(Cn + 16 * NT + nt * 16 + lg * 4);
#pragma unroll
            for (int j = 0; j < 4; ++j) f[j] = (acc[mt][nt][j] - st.x) * st.y * w4[j] + b4[j];
        };
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            float f[8];
            norm_tile(2 * ks, f);
            if (S::HALF && ks == KS - 1) {
                yb[mt][ks][0] = half_operand((f32x4){f[0], f[1], f[2], f[3]});
            } else {
                norm_tile(2 * ks + 1, f + 4);
                split2_x8(f, yb[mt][ks]);
            }
        }
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) acc[mt][nt] *= p.ms;
        __builtin_amdgcn_sched_barrier(0);
    }

    // ---- the MLP, part by part: fc1 from yb, GELU, fc2 onto acc
#pragma unroll 1
    for (int q = 0; q < S::NP; ++q) {
        const unsigned short* wq = p.wm + (size_t)q * S::PART;
        f32x4 h[2][HT];
#pragma unroll
        for (int nt = 0; nt < HT; ++nt) h[0][nt] = h[1][nt] = (f32x4){0.f, 0.f, 0.f, 0.f};
        // stage s of the part in buffer (PB + s) & 1; the one after the part's
        // last is the next part's first (after the last part: none)
        auto next = [&](auto sv) {
            constexpr int s = decltype(sv)::value;
            constexpr int par = (PB + s) & 1;
            if constexpr (s < F1) {
                constexpr int n = (KS - s * S::S1 < S::S1 ? KS - s * S::S1 : S::S1) * S::STEP1;
                issue(CInt<S::loads(n)>{}, CInt<par>{}, wq + (size_t)s * S::S1 * S::STEP1);
            } else if constexpr (s < F1 + F2) {
                constexpr int t = s - F1;
                constexpr int n = (S::K2 - t * S::S2 < S::S2 ? S::K2 - t * S::S2 : S::S2) * S::STEP;
                issue(CInt<S::loads(n)>{}, CInt<par>{}, wq + (size_t)KS * S::STEP1 + (size_t)t * S::S2 * S::STEP);
            } else if (q + 1 < S::NP) {
                issue(CInt<S::NL1>{}, CInt<par>{}, wq + S::PART);
            }
        };
        auto fc1_stage = [&](auto sv) {
            constexpr int s = decltype(sv)::value;
            const unsigned short* W = (PB + s) & 1 ? Ws1 : Ws0;
            stage_begin();
            next(CInt<s + 1>{});
#pragma unroll
            for (int i = 0; i < S::S1; ++i) {
                const int ks = s * S::S1 + i;
                if (ks >= KS) break;
                u32x4 xb[2][2];
#pragma unroll
                for (int mt = 0; mt < 2; ++mt) xb[mt][0] = yb[mt][ks][0], xb[mt][1] = yb[mt][ks][1];
                if (S::HALF && ks == KS - 1) ws_mma2<HT, S::HU, true>(W + i * S::STEP1, lr, lg, xb, h);
                else ws_mma2<HT, S::HU>(W + i * S::STEP1, lr, lg, xb, h);
            }
        };
        auto fc2_stage = [&](auto sv) {
            constexpr int s = decltype(sv)::value;
            constexpr int t = s - F1;
            const unsigned short* W = (PB + s) & 1 ? Ws1 : Ws0;
            stage_begin();
            next(CInt<s + 1>{});
            if constexpr (t == 0) {
                // the hidden units in their scale: + b1, GELU (b1x in the
                // part's packed row order)
#pragma unroll
                for (int nt = 0; nt < HT; ++nt) {
                    const f32x4 b = *(const f32x4*)(p.b1x + q * S::HU + 16 * nt + 4 * lg);
#pragma unroll
                    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
                        for (int j = 0; j < 4; ++j)
                            h[mt][nt][j] = gelu_scaled(__builtin_fmaf(h[mt][nt][j], p.h1, b[j]), p.g0, p.g1);
                }
            }
#pragma unroll
            for (int i = 0; i < S::S2; ++i) {
                const int k2 = t * S::S2 + i;
                if (k2 >= S::K2) break;
                u32x4 xb[2][2];
#pragma unroll
                for (int mt = 0; mt < 2; ++mt) {
                    const f32x4 a = h[mt][2 * k2], b = h[mt][2 * k2 + 1];
                    const float f[8] = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
                    split2_x8(f, xb[mt]);
                }
                ws_mma2<NT, S::ROWS>(W + i * S::STEP, lr, lg, xb, acc);
            }
        };
        fc1_stage(CInt<0>{});
        if constexpr (F1 > 1) fc1_stage(CInt<1>{});
        fc2_stage(CInt<F1>{});
        if constexpr (F2 > 1) fc2_stage(CInt<F1 + 1>{});
        static_assert(F1 <= 2 && F2 <= 2, "the stages above");
    }
    tx_store_rows<C>(acc, Cs, p.mi, mbase, M, lr, lg, p.eps, p.out, LN ? p.xn : nullptr, LN ? nullptr : p.amax_out, &big);
}

extern "C" __global__ __launch_bounds__(TX_WAVES * 64, 2) void hat_habx_cab_ln(TailXArgs p)
{
    habx_body<144, true, false, true>(p);
}
extern "C" __global__ __launch_bounds__(TX_WAVES * 64, 2) void hat_habx(TailXArgs p)
{
    habx_body<144, false, false, false>(p);
}
extern "C" __global__ __launch_bounds__(TX_WAVES * 64, 2) void hat_habx180_hab_ln(TailXArgs p)
{
    habx_body<180, false, true, true>(p);
}
extern "C" __global__ __launch_bounds__(TX_WAVES * 64, 2) void hat_habx180(TailXArgs p)
{
    habx_body<180, false, false, false>(p);
}
