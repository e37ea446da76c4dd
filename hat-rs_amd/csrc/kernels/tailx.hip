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
// weights and combined bias written by the gate (cab.hip); aux is
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
// A block of 4 waves takes one 128-token row tile (64 on small planes, see the
// instances below), 32 tokens a wave (each weight
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
template <int C, int MT>
__device__ __forceinline__ void tx_store_rows(const f32x4 (&acc)[MT][(C + 15) / 16], const float* Cs, float mi, int mbase,
                                              int M, int lr, int lg, float eps, float* out, float* xn,
                                              unsigned* amax_out, unsigned* lds)
{
    constexpr int NT = (C + 15) / 16;
    float big = 0.0f;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
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

// MT: 16-token tiles a wave (the block's row tile is 64 MT tokens); NB: stage
// buffers, NB - 1 stages in flight.
template <int C, bool CAB, bool HAB, bool LN, int MT, int NB>
__device__ __forceinline__ void habx_body(const TailXArgs& p)
{
    using S = TailXShape<C>;
    constexpr int NT = S::NT, KS = S::KS, HT = S::HT, D = NB - 1;
    // the projection's stages: its own steps, then (CAB) one of conv2's two;
    // then F1 + F2 a part. Stage i is in buffer i % NB.
    constexpr int OWN = S::ceil_div(KS, S::SP), NPS = OWN + (CAB ? 1 : 0);
    static_assert(!CAB || S::SP == 2, "conv2's two steps are one stage");
    constexpr int F1 = S::ceil_div(KS, S::S1), F2 = S::ceil_div(S::K2, S::S2), NF = F1 + F2;
    // the parts are walked UQ at a time, after which the buffers line up again
    constexpr int UQ = NF % NB == 0 ? 1 : NB / NF;
    static_assert(NF * UQ % NB == 0 && S::NP % UQ == 0 && D <= NPS && D <= NF * UQ, "whole rounds of the buffers");
    static_assert(NB == 2 || NB == 4, "the buffers below");
    // with more than one stage in flight nothing but the stages' copies may be
    // loaded between the waits: the projection's operands all come first
    constexpr bool UP = NB > 2;
    // the stage buffers as LDS objects of their own, so that the compiler sees
    // that reads of one need not wait for the copy into another
    __shared__ __attribute__((aligned(16))) unsigned short Ws0[S::BUF];
    __shared__ __attribute__((aligned(16))) unsigned short Ws1[S::BUF];
    __shared__ __attribute__((aligned(16))) unsigned short Ws2[NB > 2 ? S::BUF : 8];
    __shared__ __attribute__((aligned(16))) unsigned short Ws3[NB > 2 ? S::BUF : 8];
    // rows of 16 NT constants (zeros past C): the projection's bias, norm2 w, b,
    // b2, next norm w, b (LN), gate * cscale (HAB); and fc1's bias (b1x), by the
    // stages' kind of copy, so that its reads wait for no other copy
    constexpr int CROWS = 4 + (LN ? 2 : 0) + (HAB ? 1 : 0), GATE = CROWS - 1;
    __shared__ __attribute__((aligned(16))) float Cc[CROWS * 16 * NT];
    constexpr int NB1 = S::loads(2 * S::NP * S::HU);
    static_assert(NB1 * 256 <= TX_B1, "whole loads");
    __shared__ __attribute__((aligned(16))) float Cb[NB1 * 256];
    const float* const Cn = Cc + 16 * NT;
    const float* const Cs = Cc + 3 * 16 * NT;
    __shared__ unsigned big;                                                    // block_amax's
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform, in a scalar register
    const int lr = lane & 15, lg = lane >> 4;
    const int M = p.M;
    constexpr int ROWS = TX_WAVES * 16 * MT;
    if ((int)blockIdx.x * ROWS >= M) return;  // whole block, before any barrier
    if (tid == 0) big = 0;
    unsigned* const amax_out = LN ? nullptr : p.amax_out;
    const float ms = p.ms, mi = p.mi;

    auto buffer = [&](auto iv) -> unsigned short* {
        constexpr int b = decltype(iv)::value % NB;
        return b == 0 ? Ws0 : b == 1 ? Ws1 : b == 2 ? Ws2 : Ws3;
    };
    // a wave's loads of stage i; i counts the projection's stages, then the
    // stages of one part (NPS + s)
    auto stage_loads = [](int i) constexpr {
        int n = 0;
        if (i < OWN) n = (KS - i * S::SP < S::SP ? KS - i * S::SP : S::SP) * S::STEP;
        else if (i < NPS) n = 2 * S::STEP;
        else {
            const int s = (i - NPS) % NF, t = s - F1;
            n = s < F1 ? (KS - s * S::S1 < S::S1 ? KS - s * S::S1 : S::S1) * S::STEP1
                       : (S::K2 - t * S::S2 < S::S2 ? S::K2 - t * S::S2 : S::S2) * S::STEP;
        }
        return S::loads(n) / TX_WAVES;
    };
    // issue stage i: for i >= NPS stage (i - NPS) % NF of part q + (i - NPS) / NF
    auto issue = [&](auto iv, int q) {
        constexpr int i = decltype(iv)::value;
        const unsigned short* src;
        if constexpr (i < OWN) {
            src = p.w + (size_t)i * S::SP * S::STEP;
        } else if constexpr (i < NPS) {
            src = p.w2gx;
        } else {
            constexpr int s = (i - NPS) % NF, t = s - F1;
            q += (i - NPS) / NF;
            // past the last part: nothing, or (UP) the last part's again, so that
            // the counts of stage_begin hold to the end
            if constexpr (UP) q = q < S::NP ? q : S::NP - 1;
            else if (q >= S::NP) return;
            src = p.wm + (size_t)q * S::PART + (s < F1 ? (size_t)s * S::S1 * S::STEP1
                                                       : (size_t)KS * S::STEP1 + (size_t)t * S::S2 * S::STEP);
        }
        wc_issue<stage_loads(i) * TX_WAVES, TX_WAVES>(buffer(iv), src, wave, lane);
    };
    // Stage i begins: its loads have landed (everything issued before those of
    // the D - 1 stages after it), for every wave, and every wave is done with the
    // stage before, whose buffer stage i + D goes to.
    auto stage_begin = [&](auto iv) {
        constexpr int i = decltype(iv)::value;
        if constexpr (NB == 2) {
            __builtin_amdgcn_s_waitcnt(0);
            __syncthreads();
        } else {
            constexpr int n = stage_loads(i + 1) + stage_loads(i + 2);
            static_assert(D == 3 && n < 64, "the vmcnt field");
            __builtin_amdgcn_s_waitcnt(wc_vmcnt(n));
            asm volatile("s_barrier" ::: "memory");
        }
    };

    issue(CInt<0>{}, 0);
    wc_issue<NB1, TX_WAVES>((unsigned short*)Cb, (const unsigned short*)p.b1x, wave, lane);
    // all constants in flight together with the rows below; into LDS after them
    constexpr int NCV = S::ceil_div(CROWS * 16 * NT, TX_WAVES * 64);
    float cv[NCV];
#pragma unroll
    for (int k = 0; k < NCV; ++k) {
        const int i = tid + k * TX_WAVES * 64, r = i / (16 * NT), c = i - r * 16 * NT;
        const float* src = r == 0 ? p.bias : r == 1 ? p.inw : r == 2 ? p.inb : r == 3 ? p.b2 : HAB && r == GATE ? p.gate
                           : r == 4 ? p.nw : p.nb;
        cv[k] = *(c < C && r < CROWS ? src + c : hat_zero_row);
        if (HAB && r == GATE) cv[k] *= p.cscale;
    }
    auto put_constants = [&] {
#pragma unroll
        for (int k = 0; k < NCV; ++k) {
            const int i = tid + k * TX_WAVES * 64;
            if (i < CROWS * 16 * NT) Cc[i] = cv[k];
        }
    };
    const int mbase = blockIdx.x * ROWS + wave * 16 * MT;
    // acc = the block input's rows in the projection's scale (zeros past M, C)
    f32x4 acc[MT][NT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        const int m = mbase + mt * 16 + lr;
        const float* row = p.res + (size_t)(m < M ? m : 0) * C + lg * 4;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = load_or_zero(row + nt * 16, m < M && tx_live<C>(nt, lg));
    }
    // HAB: conv2's output rows, added (times gate * cscale) to the block input
    // here, where registers are free, rather than to x' (52 registers spilled)
    f32x4 aux[HAB ? MT : 1][HAB ? NT : 1];
    if constexpr (HAB) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const int m = mbase + mt * 16 + lr;
            const float* row = p.aux + (size_t)(m < M ? m : 0) * C + lg * 4;
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) aux[mt][nt] = load_or_zero(row + nt * 16, m < M && tx_live<C>(nt, lg));
        }
    }

    // ---- the projection: acc = ps (x + ao . Wp^T (+ nb(t1) . W2g^T))
    {
        WcRows<C, MT> ar;
        ar.init(p.a, mbase, M, lr);
        // ao's rows: one stage ahead, or (UP) all of them
        constexpr int NY = UP ? NPS : 2;
        f32x4 y[NY][S::SP][MT][2];
        auto load_rows = [&](auto sv) {
            constexpr int s = decltype(sv)::value;
#pragma unroll
            for (int i = 0; i < S::SP; ++i) {
                const int ks = s * S::SP + i;
                if (ks >= KS) break;
                if (S::HALF && ks == KS - 1) ar.load_half(lg, y[s % NY][i]);
                else ar.load(ks, lg, y[s % NY][i]);
            }
        };
        // conv2's B operand for its k-step s: the 3x3 neighbourhood of t1 at
        // this lane's tokens, k = 32 s + 8 lg + j = tap*6 + ci (pairs of
        // channels; taps outside the plane and k >= 54 read zeros)
        auto gather_t1 = [&](int s, f32x4 (&dst)[MT][2]) {
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
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
        if constexpr (!UP) put_constants();
        if constexpr (UP) {
            load_rows(CInt<1>{});
            load_rows(CInt<2>{});
            if constexpr (OWN > 3) {
                load_rows(CInt<3>{});
                load_rows(CInt<4>{});
                load_rows(CInt<5>{});
            }
            if constexpr (CAB) {
#pragma unroll
                for (int i = 0; i < 2; ++i) gather_t1(i, y[OWN % NY][i]);
            }
            put_constants();
            // none of those loads may sink below the copies
            __builtin_amdgcn_sched_barrier(0);
            issue(CInt<1>{}, 0);
            issue(CInt<2>{}, 0);
        }
        auto proj_stage = [&](auto sv) {
            constexpr int s = decltype(sv)::value;
            const unsigned short* W = buffer(sv);
            stage_begin(sv);
            issue(CInt<s + D>{}, 0);
            if constexpr (s == 0) {
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                    for (int nt = 0; nt < NT; ++nt) {
                        if constexpr (HAB) {
                            const f32x4 g4 = *(const f32x4*)(Cc + GATE * 16 * NT + nt * 16 + lg * 4);
#pragma unroll
                            for (int j = 0; j < 4; ++j)
                                acc[mt][nt][j] = __builtin_fmaf(aux[mt][nt][j], g4[j], acc[mt][nt][j]);
                        }
                        acc[mt][nt] *= p.ps;
                    }
            }
            if constexpr (!UP && s + 1 < OWN) load_rows(CInt<s + 1>{});
            else if constexpr (!UP && CAB && s + 1 == OWN) {
#pragma unroll
                for (int i = 0; i < 2; ++i) gather_t1(i, y[(s + 1) % NY][i]);
            }
#pragma unroll
            for (int i = 0; i < S::SP; ++i) {
                const int ks = s * S::SP + i;
                if (s < OWN && ks >= KS) break;
                u32x4 xb[MT][2];
                if (S::HALF && s < OWN && ks == KS - 1) {
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt) xb[mt][0] = half_operand(y[s % NY][i][mt][0]);
                    ws_mma2<NT, S::ROWS, true>(W + i * S::STEP, lr, lg, xb, acc);
                } else {
                    split_pre2(y[s % NY][i], xb);
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
        static_assert(NPS <= 6 && NPS != 5 && (OWN == 3 || OWN == 6), "the stages above");
    }
    // x' = acc / ps + bias, then norm2 of it split into fc1's operands yb, and
    // acc = ms x'
    u32x4 yb[MT][KS][2];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            const f32x4 b4 = *(const f32x4*)(Cc + nt * 16 + lg * 4);
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
        for (int nt = 0; nt < NT; ++nt) acc[mt][nt] *= ms;
        __builtin_amdgcn_sched_barrier(0);
    }

    // ---- the MLP, part by part: fc1 from yb, GELU, fc2 onto acc
    auto fc1_stage = [&](auto iv, int q, f32x4 (&h)[MT][HT]) {
        constexpr int s = (decltype(iv)::value - NPS) % NF;
        const unsigned short* W = buffer(iv);
        stage_begin(iv);
        issue(CInt<decltype(iv)::value + D>{}, q);
        if constexpr (s == 0) {
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int nt = 0; nt < HT; ++nt) h[mt][nt] = (f32x4){0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
        for (int i = 0; i < S::S1; ++i) {
            const int ks = s * S::S1 + i;
            if (ks >= KS) break;
            u32x4 xb[MT][2];
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) xb[mt][0] = yb[mt][ks][0], xb[mt][1] = yb[mt][ks][1];
            if (S::HALF && ks == KS - 1) ws_mma2<HT, S::HU, true>(W + i * S::STEP1, lr, lg, xb, h);
            else ws_mma2<HT, S::HU>(W + i * S::STEP1, lr, lg, xb, h);
        }
    };
    auto fc2_stage = [&](auto iv, int q, f32x4 (&h)[MT][HT]) {
        constexpr int r = decltype(iv)::value - NPS, t = r % NF - F1;
        const unsigned short* W = buffer(iv);
        stage_begin(iv);
        issue(CInt<decltype(iv)::value + D>{}, q);
        if constexpr (t == 0) {
            // the hidden units in their scale: + b1, GELU (b1x in the part's
            // packed row order)
#pragma unroll
            for (int nt = 0; nt < HT; ++nt) {
                const f32x4 b = *(const f32x4*)(Cb + (q + r / NF) * S::HU + 16 * nt + 4 * lg);
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        h[mt][nt][j] = gelu_scaled(__builtin_fmaf(h[mt][nt][j], p.h1, b[j]), p.g0, p.g1);
            }
        }
#pragma unroll
        for (int i = 0; i < S::S2; ++i) {
            const int k2 = t * S::S2 + i;
            if (k2 >= S::K2) break;
            u32x4 xb[MT][2];
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                const f32x4 a = h[mt][2 * k2], b = h[mt][2 * k2 + 1];
                const float f[8] = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
                split2_x8(f, xb[mt]);
            }
            ws_mma2<NT, S::ROWS>(W + i * S::STEP, lr, lg, xb, acc);
        }
    };
    static_assert(F1 <= 2 && F2 <= 2 && UQ <= 2, "the stages below");
#pragma unroll 1
    for (int q = 0; q < S::NP; q += UQ) {
        f32x4 h[MT][HT];
        fc1_stage(CInt<NPS>{}, q, h);
        if constexpr (F1 > 1) fc1_stage(CInt<NPS + 1>{}, q, h);
        fc2_stage(CInt<NPS + F1>{}, q, h);
        if constexpr (F2 > 1) fc2_stage(CInt<NPS + F1 + 1>{}, q, h);
        if constexpr (UQ > 1) {
            fc1_stage(CInt<NPS + NF>{}, q, h);
            if constexpr (F1 > 1) fc1_stage(CInt<NPS + NF + 1>{}, q, h);
            fc2_stage(CInt<NPS + NF + F1>{}, q, h);
            if constexpr (F2 > 1) fc2_stage(CInt<NPS + NF + F1 + 1>{}, q, h);
        }
    }
    if constexpr (UP) __builtin_amdgcn_s_waitcnt(wc_vmcnt(0));  // no copy outlives the block
    tx_store_rows<C>(acc, Cs, mi, mbase, M, lr, lg, p.eps, p.out, LN ? p.xn : nullptr, amax_out, &big);
}

// Large planes: 128-token row tiles, two blocks a CU, one stage in flight. Small
// planes (_s, at most one such block a CU: run_tailx): 64-token tiles, one block a
// CU. With one wave a SIMD nothing hides a wave's own latencies, so a wave has half
// the work, three stages are in flight and the projection's operands are all loaded
// first. The wave's issue bounds it, not the weights' latency: a second launch on
// the same, cached weights takes as long. 64 x 64 tokens: hat_habx_cab_ln 34.2 ->
// 23.3 us, hat_habx180_hab_ln 45.0 -> 30.7; 128 x 128: 37.5 -> 27.6, 49.8 -> 38.8.
extern "C" __global__ __launch_bounds__(TX_WAVES * 64, 2) void hat_habx_cab_ln(TailXArgs p) { habx_body<144, true, false, true, 2, 2>(p); }
extern "C" __global__ __launch_bounds__(TX_WAVES * 64, 1) void hat_habx_cab_ln_s(TailXArgs p) { habx_body<144, true, false, true, 1, 4>(p); }
extern "C" __global__ __launch_bounds__(TX_WAVES * 64, 2) void hat_habx(TailXArgs p) { habx_body<144, false, false, false, 2, 2>(p); }
extern "C" __global__ __launch_bounds__(TX_WAVES * 64, 1) void hat_habx_s(TailXArgs p) { habx_body<144, false, false, false, 1, 4>(p); }
extern "C" __global__ __launch_bounds__(TX_WAVES * 64, 2) void hat_habx180_hab_ln(TailXArgs p) { habx_body<180, false, true, true, 2, 2>(p); }
extern "C" __global__ __launch_bounds__(TX_WAVES * 64, 1) void hat_habx180_hab_ln_s(TailXArgs p) { habx_body<180, false, true, true, 1, 4>(p); }
extern "C" __global__ __launch_bounds__(TX_WAVES * 64, 2) void hat_habx180(TailXArgs p) { habx_body<180, false, false, false, 2, 2>(p); }
extern "C" __global__ __launch_bounds__(TX_WAVES * 64, 1) void hat_habx180_s(TailXArgs p) { habx_body<180, false, false, false, 1, 4>(p); }
