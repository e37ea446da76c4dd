#include "gpu.h"

#if defined(__x86_64__)
#include <immintrin.h>
#endif

#include <cmath>
#include <cstdio>
#include <cstring>
#include <deque>
#include <memory>
#include <atomic>
#include <thread>

#include "kargs.h"
#include "tile.h"

namespace hat {

using namespace hatk;

// ---------------------------------------------------------------------------
// Weight repacking

std::vector<float> pack_linear(const float* w, int N, int K, int* Kp)
{
    const int kp = (K + 15) / 16 * 16;
    std::vector<float> out((size_t)N * kp, 0.0f);
    for (int n = 0; n < N; ++n) memcpy(&out[(size_t)n * kp], w + (size_t)n * K, sizeof(float) * K);
    *Kp = kp;
    return out;
}


// float -> f16, round to nearest even, subnormals kept, past the range infinite
static inline unsigned short f16_rne(float x)
{
    uint32_t u;
    memcpy(&u, &x, 4);
    const uint32_t sign = (u >> 16) & 0x8000u;
    u &= 0x7fffffffu;
    if (u >= 0x477ff000u)  // rounds to 2^16 or more, infinite or NaN
        return (unsigned short)(sign | (u > 0x7f800000u ? 0x7e00u : 0x7c00u));
    if (u < 0x38800000u) {  // below 2^-14: units of 2^-24, rounded by adding 1.5 * 2^23 of them
        float a;
        memcpy(&a, &u, 4);
        const float r = a * 16777216.0f + 12582912.0f;
        uint32_t v;
        memcpy(&v, &r, 4);
        return (unsigned short)(sign | (v - 0x4b400000u));
    }
    u += 0xfffu + ((u >> 13) & 1u);
    return (unsigned short)(sign | ((u - 0x38000000u) >> 13));
}
static inline float f16_float(unsigned short h)
{
    const uint32_t e = (h >> 10) & 31u, m = h & 1023u;
    float v;
    if (e == 0) {
        v = (float)m * 5.9604644775390625e-8f;  // 2^-24
    } else {
        const uint32_t u = e == 31 ? 0x7f800000u | (m << 13) : ((e + 112u) << 23) | (m << 13);
        memcpy(&v, &u, 4);
    }
    return h & 0x8000u ? -v : v;
}

// x = h0 + h1 (+ at most 2^-22 |x|), each part the round-to-nearest f16 of what
// the one before leaves.
static inline void split2_f16(float x, unsigned short* h0, unsigned short* h1)
{
    *h0 = f16_rne(x);
    *h1 = f16_rne(x - f16_float(*h0));
}

// Eight values at once, with the conversion instructions where the host has them
// (a few million weights are split per network, and an op splits its own on every
// call). Both forms give the same bits.
#if defined(__x86_64__)
__attribute__((target("avx,f16c"))) static void split2_f16_x8_f16c(const float* x, unsigned short* h0, unsigned short* h1)
{
    const __m256 v = _mm256_loadu_ps(x);
    const __m128i a = _mm256_cvtps_ph(v, _MM_FROUND_TO_NEAREST_INT);
    const __m128i b = _mm256_cvtps_ph(_mm256_sub_ps(v, _mm256_cvtph_ps(a)), _MM_FROUND_TO_NEAREST_INT);
    _mm_storeu_si128((__m128i*)h0, a);
    _mm_storeu_si128((__m128i*)h1, b);
}
#endif
static void split2_f16_x8(const float* x, unsigned short* h0, unsigned short* h1)
{
#if defined(__x86_64__)
    static const bool f16c = __builtin_cpu_supports("avx") && __builtin_cpu_supports("f16c");
    if (f16c) return split2_f16_x8_f16c(x, h0, h1);
#endif
    for (int j = 0; j < 8; ++j) split2_f16(x[j], h0 + j, h1 + j);
}

// value(r, kk), r < rows, kk < 32: one 32-k step as two f16 planes [rows][32],
// row r's k-group g at slot ws_slot(r, g).
template <typename F>
static void split2_step(int rows, F value, unsigned short* dst)
{
    for (int r = 0; r < rows; ++r)
        for (int g = 0; g < 4; ++g) {
            float v[8];
            for (int j = 0; j < 8; ++j) v[j] = value(r, 8 * g + j);
            unsigned short* d = dst + (size_t)r * 32 + hatk::ws_slot(r, g) * 8;
            split2_f16_x8(v, d, d + (size_t)rows * 32);
        }
}

// value(r, kk), kk < 16: the packed last step of a K = 144 linear (k = 128 + kk;
// common.h half_operand): lane group g's slots j < 4 and 4 + j hold k = 128 + 4 g
// + j, the planes (a0 | a0) and (a1 | a1).
template <typename F>
static void split2_half_step(int rows, F value, unsigned short* dst)
{
    for (int r = 0; r < rows; ++r)
        for (int kk = 0; kk < 16; ++kk) {
            unsigned short* d = dst + (size_t)r * 32 + hatk::ws_slot(r, kk / 4) * 8 + kk % 4;
            split2_f16(value(r, kk), d, d + (size_t)rows * 32);
            d[4] = d[0];
            d[(size_t)rows * 32 + 4] = d[(size_t)rows * 32];
        }
}

std::vector<unsigned short> pack_linear_ws(const float* w, int N, int K, const float (&ws)[3], bool fill)
{
    // three slices, q, k and v: C = 144 of 144 rows, five k-steps; C = 180 of
    // 180 rows padded to 192, six k-steps
    if (!((K == 144 && N == 432) || (K == 180 && N == 540)))
        throw Error("pack_linear_ws: needs the qkv shapes K = 144, N = 432 or K = 180, N = 540");
    const int real = K == 144 ? 144 : 180, rows = K == 144 ? 144 : 192, ks_n = (K + 31) / 32;
    const size_t chunk = (size_t)2 * rows * 32;
    std::vector<unsigned short> out((size_t)(N / real) * ks_n * chunk, 0);
    if (!fill) return out;
    for (int sl = 0; sl < N / real; ++sl) {
        const float f = ws[sl * real / (N / 3)];
        for (int s = 0; s < ks_n; ++s) {
            auto value = [&](int r, int kk) {
                const int k = 32 * s + kk;
                return r < real && k < K ? w[((size_t)sl * real + r) * K + k] * f : 0.0f;
            };
            unsigned short* dst = &out[((size_t)sl * ks_n + s) * chunk];
            if (K == 144 && s == 4) split2_half_step(rows, value, dst);
            else split2_step(rows, value, dst);
        }
    }
    return out;
}

double abs_max(const float* w, size_t n)
{
    uint32_t m = 0;  // non-negative floats order as their bits do, a NaN above all
    for (size_t i = 0; i < n; ++i) {
        uint32_t u;
        memcpy(&u, w + i, 4);
        m = std::max(m, u & 0x7fffffffu);
    }
    float f;
    memcpy(&f, &m, 4);
    return f;
}

// fc1 output tile t, row 4g + r (lane group g, register r) -> hidden unit
// within a part (tailx.hip): fc2's 32-k step s then finds units 32 s + 8 g ..
// +7 in tiles 2 s and 2 s + 1 of lane group g.
static int tailx_unit(int row)
{
    const int t = row / 16, g = (row % 16) / 4, r = row % 4;
    return 32 * (t / 2) + 8 * g + 4 * (t % 2) + r;
}

// fc1 input position k = 32 ks + 8 g + j (ks: 32-k step, g: lane group, j < 8) ->
// channel of x': the lane's accumulator tiles 2 ks and 2 ks + 1 (channels 32 ks +
// 4 g + j and 32 ks + 16 + 4 g + j - 4); -1 past channel C - 1. (C = 144's packed
// fifth step takes channels 128 + kk in order: split2_half_step.)
int tailx_channel(int C, int k)
{
    const int ks = k >> 5, g = (k >> 3) & 3, j = k & 7;
    const int c = 32 * ks + (j < 4 ? 4 * g + j : 16 + 4 * g + (j - 4));
    return c < C ? c : -1;
}

std::vector<unsigned short> pack_tail_proj(const float* w, int C, float s, bool fill)
{
    const int rows = (C + 15) / 16 * 16, ks_n = (C + 31) / 32;
    const size_t step = (size_t)2 * rows * 32;
    std::vector<unsigned short> out(ks_n * step + TX_PAD, 0);
    if (!fill) return out;
    for (int ks = 0; ks < ks_n; ++ks) {
        auto value = [&](int n, int kk) {
            const int k = 32 * ks + kk;
            return n < C && k < C ? w[(size_t)n * C + k] * s : 0.0f;
        };
        if (C == 144 && ks == 4) split2_half_step(rows, value, &out[ks * step]);
        else split2_step(rows, value, &out[ks * step]);
    }
    return out;
}

void pack_tail_mlp(const float* w1, const float* b1, const float* w2, int C, float s1, float s2, float hs,
                   std::vector<unsigned short>* w, std::vector<float>* b1x, bool fill)
{
    const int H = 2 * C, HU = tailx_hu(C), NP = (H + HU - 1) / HU, rows = (C + 15) / 16 * 16, ks_n = (C + 31) / 32;
    const size_t step1 = (size_t)2 * HU * 32, step = (size_t)2 * rows * 32, part = ks_n * step1 + HU / 32 * step;
    w->assign(NP * part + TX_PAD, 0);
    b1x->assign(TX_B1, 0.0f);
    if (!fill) return;
    for (int q = 0; q < NP; ++q) {
        for (int r = 0; r < HU; ++r) {
            const int u = q * HU + tailx_unit(r);
            if (u < H) (*b1x)[(size_t)q * HU + r] = b1[u] * hs;
        }
        for (int ks = 0; ks < ks_n; ++ks) {
            const bool half = C == 144 && ks == 4;
            auto value = [&](int r, int kk) {
                const int u = q * HU + tailx_unit(r), c = half ? 128 + kk : tailx_channel(C, 32 * ks + kk);
                return u < H && c >= 0 ? w1[(size_t)u * C + c] * s1 : 0.0f;
            };
            unsigned short* dst = &(*w)[q * part + ks * step1];
            if (half) split2_half_step(HU, value, dst);
            else split2_step(HU, value, dst);
        }
        for (int st = 0; st < HU / 32; ++st)
            split2_step(rows, [&](int n, int kk) {
                const int u = q * HU + st * 32 + kk;
                return n < C && u < H ? w2[(size_t)n * H + u] * s2 : 0.0f;
            }, &(*w)[q * part + ks_n * step1 + st * step]);
    }
}

// [CO][CI][3][3] -> [CIp/16][9][COp][16]; with r > 0 the output channels are
// permuted so that channel o = c*r*r + i*r + j lands at o' = (i*r + j)*Cf + c
// (Cf = CO / r^2), which lets the conv store four consecutive o' as four
// consecutive channels of one pixel of the shuffled plane.
std::vector<float> pack_conv(const float* w, const float* b, int CO, int CI, int r,
                             std::vector<float>* bias_out, int* CIp, int* COp)
{
    const int cip = (CI + 15) / 16 * 16, cop = (CO + 15) / 16 * 16;
    const int Cf = r > 0 ? CO / (r * r) : 0;
    auto src_channel = [&](int o2) -> int {
        if (r <= 0) return o2;
        const int sub = o2 / Cf, c = o2 % Cf;
        const int i = sub / r, j = sub % r;
        return c * r * r + i * r + j;
    };
    std::vector<float> out((size_t)cip * 9 * cop, 0.0f);
    bias_out->assign(cop, 0.0f);
    for (int o2 = 0; o2 < CO; ++o2) {
        const int o = src_channel(o2);
        (*bias_out)[o2] = b[o];
        for (int ci = 0; ci < CI; ++ci)
            for (int tap = 0; tap < 9; ++tap) {
                const int cc = ci / 16, c16 = ci % 16;
                out[(((size_t)cc * 9 + tap) * cop + o2) * 16 + c16] = w[((size_t)o * CI + ci) * 9 + tap];
            }
    }
    *CIp = cip;
    *COp = cop;
    return out;
}

// [CO][CI][3][3] -> the Winograd F(2x2, 3x3) weights U[xi] = G g G^T of the
// hat_convwino_* kernels, G = [1 0 0; 1/2 1/2 1/2; 1/2 -1/2 1/2; 0 0 1],
// formed in double, rounded to fp32, scaled into f16's range and split into two
// f16 parts, arranged [kc][xi][nt][part][lane][8]: lane r + 16 g of (kc, xi, nt)
// holds part `part` of U[xi][16 nt + r][32 kc + 8 g .. +7]; channels past CO and CI
// are zero (CO padded to 16s, CI to 32s). With r > 0 the output channels are
// permuted as pack_conv permutes them. When the last chunk holds at most 16 real
// channels (CI = 144), it is packed as the K = 144 linears' last step
// (split2_half_step): lane r + 16 g, slots j < 4 hold channel 32 kc + 4 g + j,
// slots 4 + j the same channel and part.
std::vector<unsigned short> pack_wino(const float* w, int CO, int CI, int r, float* uinv, bool fill)
{
    if (r > 0 && CO % 16 != 0) throw Error("pack_wino: shuffled output channels must come in 16s");
    static const double G[4][3] = {{1, 0, 0}, {0.5, 0.5, 0.5}, {0.5, -0.5, 0.5}, {0, 0, 1}};
    const int NTT = (CO + 15) / 16, NKC = (CI + 31) / 32, Cf = r > 0 ? CO / (r * r) : 0;
    const bool packed = CI % 32 != 0 && CI % 32 <= 16;  // the kernels' PACK
    std::vector<unsigned short> out((size_t)NKC * 16 * NTT * 2 * 512, 0);
    *uinv = 1.0f;
    if (!fill) return out;
    std::vector<float> U((size_t)CO * CI * 16);
    for (int o2 = 0; o2 < CO; ++o2) {
        int o = o2;
        if (r > 0) {
            const int sub = o2 / Cf, c = o2 % Cf;
            o = c * r * r + (sub / r) * r + sub % r;
        }
        for (int ci = 0; ci < CI; ++ci) {
            const float* g = w + ((size_t)o * CI + ci) * 9;
            double t[4][3];  // G g
            for (int i = 0; i < 4; ++i)
                for (int b = 0; b < 3; ++b) {
                    double u = 0.0;
                    for (int a = 0; a < 3; ++a) u += G[i][a] * (double)g[a * 3 + b];
                    t[i][b] = u;
                }
            for (int i = 0; i < 4; ++i)
                for (int j = 0; j < 4; ++j) {
                    double u = 0.0;
                    for (int b = 0; b < 3; ++b) u += t[i][b] * G[j][b];
                    U[((size_t)o2 * CI + ci) * 16 + 4 * i + j] = (float)u;
                }
        }
    }
    const float su = f16_scale(abs_max(U.data(), U.size()));
    *uinv = 1.0f / su;
    for (int o2 = 0; o2 < CO; ++o2)
        for (int ci = 0; ci < CI; ++ci)
            for (int xi = 0; xi < 16; ++xi) {
                const int kc = ci / 32, c32 = ci % 32, nt = o2 / 16, rr = o2 % 16;
                const bool half = packed && kc == NKC - 1;
                const int lane = rr + 16 * (half ? c32 / 4 : c32 / 8);
                const size_t at = ((((size_t)kc * 16 + xi) * NTT + nt) * 2 * 64 + lane) * 8 + (half ? c32 % 4 : c32 % 8);
                split2_f16(U[((size_t)o2 * CI + ci) * 16 + xi] * su, &out[at], &out[at + 512]);
                if (half) out[at + 4] = out[at], out[at + 512 + 4] = out[at + 512];
            }
    return out;
}

// Which convs have a Winograd kernel (hat_convwino_*): the 144 -> 144 and
// 180 -> 180 trunk convs, conv_before_upsample 144 / 180 -> 64, the x2
// upsample convs 64 -> 256 and the unfolded CAB's 180 -> 60 and 60 -> 180.
static bool wino_conv(int CO, int CI, int r)
{
    return (r == 0 && (CI == 144 || CI == 180) && (CO == CI || CO == 64)) || (r == 2 && CI == 64 && CO == 256) ||
           (r == 0 && CI == 180 && CO == 60) || (r == 0 && CI == 60 && CO == 180);
}

// conv1 [6][144][3][3] as the split A operands of hat_cab_conv1 (CX_WPACK):
// row r = tap * 6 + co (rows 54..63 zero), each weight times sw as two f16 parts.
std::vector<unsigned short> pack_cab_conv1(const float* w, float sw)
{
    std::vector<unsigned short> out(CX_WPACK, 0);
    for (int ks = 0; ks < 9; ++ks)
        for (int nt = 0; nt < 2; ++nt)
            for (int lane = 0; lane < 64; ++lane)
                for (int j = 0; j < 8; ++j) {
                    const int r = nt * 32 + lane % 32, ci = ks * 16 + 8 * (lane / 32) + j;
                    if (r >= 9 * CAB_CC) continue;
                    const int tap = r / CAB_CC, co = r % CAB_CC;
                    unsigned short* d = &out[((size_t)((ks * 2 + nt) * 2) * 64 + lane) * 8 + j];
                    split2_f16(w[((size_t)co * CAB_C + ci) * 9 + tap] * sw, d, d + 64 * 8);
                }
    return out;
}

void cab_scales(float ts, float oscale, CabConvArgs* a)
{
    a->ts = ts;
    a->oinv = ts * oscale;
    a->g0 = 0.3275911f * 0.70710678f / ts;
    a->g1 = -0.5f * 1.4426950408889634f / (ts * ts);
}

float f16_scale(double bound)
{
    if (!(bound > 0.0) || !std::isfinite(bound)) return 1.0f;
    int e = 0;
    std::frexp(bound, &e);  // bound in [2^(e-1), 2^e)
    return std::ldexp(1.0f, std::max(-60, std::min(60, 15 - e)));
}

double ln_linear_bound(const float* w, const float* b, const float* lnw, const float* lnb, int n0, int n1, int C)
{
    double worst = 0.0;
    for (int n = n0; n < n1; ++n) {
        const float* r = w + (size_t)n * C;
        double sq[4] = {}, off[4] = {b ? b[n] : 0.0};  // four chains: an op does this on every call
        for (int c = 0; c < C; c += 4)
            for (int i = 0; i < 4 && c + i < C; ++i) {
                const double x = (double)r[c + i] * lnw[c + i];
                sq[i] += x * x;
                off[i] += (double)r[c + i] * lnb[c + i];
            }
        const double v = std::sqrt((sq[0] + sq[1] + sq[2] + sq[3]) * C) + std::fabs(off[0] + off[1] + off[2] + off[3]);
        if (std::isnan(v)) return v;
        worst = std::max(worst, v);
    }
    return worst;
}

double ln_bound(const float* lnw, const float* lnb, int C)
{
    double worst = 0.0;
    for (int c = 0; c < C; ++c) {
        const double v = std::sqrt((double)C) * std::fabs((double)lnw[c]) + std::fabs((double)lnb[c]);
        if (std::isnan(v)) return v;
        worst = std::max(worst, v);
    }
    return worst;
}

QkvScale qkv_scale(double bq, double bk, double bv, int head_dim)
{
    QkvScale s;
    s.v = f16_scale(bv);  // whichever attention runs: the split tail reads its output
    bq *= 1.4426950408889634 / std::sqrt((double)head_dim);  // the kernels split q times this
    if (!std::isfinite(bq) || !std::isfinite(bk) || !std::isfinite(bv)) return s;
    int a = 0;
    if (bq > 0.0 && bk > 0.0) a = (int)std::lround(0.5 * std::log2(bk / bq));
    if (std::abs(a) > 60 || std::ldexp(bq, a) > 32768.0 || std::ldexp(bk, -a) > 32768.0) return s;
    s.q = std::ldexp(1.0f, a);
    s.k = std::ldexp(1.0f, -a);
    s.ok = true;
    return s;
}

// TailXArgs' scales.
void tail_scales(const DevTail& t, TailXArgs* f)
{
    f->ps = t.ps;
    f->pi = 1.0f / t.ps;
    f->h1 = t.h1;
    f->g0 = 0.3275911f * 0.70710678f / t.hs;
    f->g1 = -0.5f * 1.4426950408889634f / (t.hs * t.hs);
    f->ms = t.ms;
    f->mi = 1.0f / t.ms;
}

TailPack pack_tail(const float* wp, const float* w1, const float* b1, const float* w2, const float* n2w, const float* n2b,
                   int C, float sv, float sn, const TailCab* cab, bool fill)
{
    TailPack p;
    DevTail& t = p.t;
    t.C = C;
    if (!fill) {
        p.w = pack_tail_proj(wp, C, 1.0f, false);
        pack_tail_mlp(w1, b1, w2, C, 1.0f, 1.0f, 1.0f, &p.wm, &p.b1x, false);
        return p;
    }
    // Both sums start from x, times their scale: at most 2^60, so that weights that
    // have all but vanished do not take an x of 256 past fp32 (two scales of 2^60)
    const float most = std::ldexp(1.0f, 60);
    float sp = std::min(f16_scale(abs_max(wp, (size_t)C * C)), most / sv);
    if (cab) {
        // the projection and the gated conv2 add into the same accumulators, so
        // ts gs = sv sp: each of the two as far from its limit as the other, and
        // the projection's weights scaled down where the limits leave no room
        auto limit = [](double bound) { return bound == 0.0 ? 60 : std::ilogb(f16_scale(bound)); };
        const int lt = limit(cab->t1), lg = limit(cab->w2);
        int spare = lt + lg - std::ilogb(sv) - std::ilogb(sp);
        if (spare < 0) {
            sp = std::ldexp(sp, spare);
            spare = 0;
        }
        t.ts = std::ldexp(1.0f, lt - spare / 2);
        t.gs = std::ldexp(1.0f, lg - (spare - spare / 2));
    }
    t.ps = sv * sp;
    p.w = pack_tail_proj(wp, C, sp);
    // |gelu(v)| <= |v|, and fc1 reads a norm's output
    t.hs = f16_scale(ln_linear_bound(w1, b1, n2w, n2b, 0, 2 * C, C));
    const float s1 = f16_scale(abs_max(w1, (size_t)2 * C * C)),
                s2 = std::min(f16_scale(abs_max(w2, (size_t)2 * C * C)), most / t.hs);
    t.h1 = t.hs / (sn * s1);
    t.ms = t.hs * s2;
    pack_tail_mlp(w1, b1, w2, C, s1, s2, t.hs, &p.wm, &p.b1x);
    return p;
}

// ---------------------------------------------------------------------------
// Launch helpers shared by the backend and the op entry points.

namespace {

// Column-block width of the GEMM for an output width N: 144 for the C = 144
// family, 192 for C = 180 (N = 180, 360, 540 in 1, 2, 3 blocks).
int gemm_bn(int N) { return N % 144 == 0 ? 144 : 192; }

const char* gemm_kernel(int N, int epi)
{
    const bool n9 = gemm_bn(N) == 144;
    switch (epi) {
    case EPI_STORE: return n9 ? "hat_gemm_n9_store" : "hat_gemm_n12_store";
    case EPI_GELU: return n9 ? "hat_gemm_n9_gelu" : "hat_gemm_n12_gelu";
    case EPI_QKV: return n9 ? "hat_gemm_n9_qkv" : "hat_gemm_n12_qkv";
    case EPI_RESID: return n9 ? "hat_gemm_n9_resid" : "hat_gemm_n12_resid";
    case EPI_RESID_LN: return n9 ? "hat_gemm_n9_resid_ln" : "hat_gemm_n12_resid_ln";
    case EPI_HAB_LN: return n9 ? "hat_gemm_n9_hab_ln" : "hat_gemm_n12_hab_ln";
    }
    throw Error("unknown GEMM epilogue");
}

// The weight-stationary kernels hold a block's whole weight row slice in LDS:
// K = 144 with 144-wide column blocks (N a multiple of 144), and K = 180
// (rows padded to 192) with 192-wide blocks, for the epilogues the blocks use.
// Returns the kernel and sets *bn to its column-block width.
const char* gemm_ws_kernel(const DevLinear& L, int epi, int* bn)
{
    const bool k144 = L.K == 144 && L.Kp == 144 && L.N % 144 == 0;
    const bool k180 = L.K == 180 && L.Kp == 192;
    if (!k144 && !k180) return nullptr;
    *bn = k144 ? 144 : 192;
    switch (epi) {
    case EPI_GELU: return k144 ? "hat_gemmws_gelu" : "hat_gemmws12_gelu";
    case EPI_RESID_LN: return k144 ? "hat_gemmws_resid_ln" : "hat_gemmws12_resid_ln";
    case EPI_HAB_LN: return k144 ? "hat_gemmws_hab_ln" : "hat_gemmws12_hab_ln";
    }
    return nullptr;
}

struct GemmEpilogue {
    const float* res = nullptr;   // residual
    const float* aux = nullptr;   // conv branch (HAB)
    const float* gate = nullptr;  // channel gate (HAB)
    float* xn = nullptr;          // LayerNorm output of the result rows
    const float* nw = nullptr;
    const float* nb = nullptr;
    // EPI_QKV: the CAB's conv1 in the same launch (qkv_takes_cab1): C = 144, 180
    const CabConvArgs* cab = nullptr;
    const ConvArgs* conv1 = nullptr;
};

// Does the CAB's conv1, `tiles` blocks of it (rounded up to whole rounds of the
// XCDs), ride on this qkv linear's launch? They are independent and, on a small
// plane, each a fraction of the chip for about the latency of one tile: together
// they take as long as the longer. Up to half the CUs; above, qkv's blocks (a CU
// each) become too few and the conv's run best two a CU. A forward, in two launches
// and in one: HAT-S 16 x 16 2.24 and 2.01 ms, 64 x 64 2.40 and 2.16, 128 x 128 3.24
// and 2.97, 176 x 176 (121 tiles) 4.95 and 4.80, but 192 x 192 (144) 6.18 and 6.22,
// 224 x 224 7.0 and 8.4; HAT 64 x 64 3.69 and 3.30, 112 x 112 4.79 and 4.73, 128 x 128
// (128 tiles) 5.33 and 4.91.
int qkv_conv1_blocks(int tiles) { return (tiles + 7) / 8 * 8; }
bool qkv_takes_cab1(const DevLinear& L, int heads, int hdim, int tiles)
{
    static const int cus = std::max(1, Runtime::get().cu_count());
    return L.wx && heads == 6 && qkv_conv1_blocks(tiles) <= cus / 2 &&
           ((L.K == 144 && L.N == 432 && hdim == 24) || (L.K == 180 && L.N == 540 && hdim == 30));
}

void run_gemm(hipStream_t s, const DevLinear& L, const float* a, int lda, long M, float* out,
              int ldo, int epi, const GemmEpilogue& e, int heads, int hdim, float cscale)
{
    if (L.K % 4 != 0 || lda % 4 != 0 || lda < L.K)
        throw Error("GEMM: K and lda must be multiples of 4 with lda >= K");
    if (L.N % 4 != 0 || (epi != EPI_QKV && (ldo % 4 != 0 || ldo < L.N)))
        throw Error("GEMM: N and ldo must be multiples of 4 with ldo >= N");
    if (M > 0x7fffffffL) throw Error("GEMM: too many rows");
    const int BN = gemm_bn(L.N);
    if ((epi == EPI_RESID_LN || epi == EPI_HAB_LN) && L.N > BN)
        throw Error("GEMM: a LayerNorm epilogue needs whole rows in one block");
    GemmArgs p{};
    p.a = a;
    p.w = L.w;
    p.bias = L.b;
    p.out = out;
    p.res = e.res;
    p.aux = e.aux;
    p.gate = e.gate;
    p.xn = e.xn;
    p.nw = e.nw;
    p.nb = e.nb;
    p.M = (int)M;
    p.N = L.N;
    p.K = L.K;
    p.Kp = L.Kp;
    p.lda = lda;
    p.ldo = ldo;
    p.heads = heads;
    p.hdim = hdim;
    p.cscale = cscale;
    p.eps = 1e-5f;
    if (epi == EPI_QKV && L.wx && L.K == 144 && L.N == 432 && heads == 6 && hdim == 24 && lda == 144) {
        // split-f16 qkv (gemmx.hip): weight-stationary, groups of three blocks
        static const int cus = std::max(1, Runtime::get().cu_count());
        p.w = (const float*)L.wx;
        memcpy(p.oscale, L.oscale, sizeof p.oscale);
        if (e.cab) {
            QkvCabArgs q{p, *e.cab, qkv_conv1_blocks(e.cab->H / 16 * (e.cab->W / 16))};
            launch(s, "hat_qkv_cab1", (unsigned)(q.nconv + 3 * gemmx_qkv_groups(cus - q.nconv, 3)), 1, 1, GX_THREADS, q);
            return;
        }
        launch(s, "hat_gemmx_qkv", (unsigned)(3 * gemmx_qkv_groups(cus, 3)), 1, 1, GX_THREADS, p);
        return;
    }
    if (epi == EPI_QKV && L.wx && L.K == 180 && L.N == 540 && heads == 6 && hdim == 30 && lda == 180) {
        // the same for C = 180
        static const int cus = std::max(1, Runtime::get().cu_count());
        p.w = (const float*)L.wx;
        memcpy(p.oscale, L.oscale, sizeof p.oscale);
        if (e.conv1) {
            const int tiles = e.conv1->H / 8 * (e.conv1->W / 16);
            QkvConvArgs q{p, *e.conv1, 0, tiles, 1};
            // as two column blocks a tile while those fit as well (64 x 64: 23.2 -> 18.8 us)
            if (qkv_conv1_blocks(2 * tiles) <= cus / 2) q.ntile = 2 * tiles, q.ncb = 2;
            q.nconv = qkv_conv1_blocks(q.ntile);
            launch(s, "hat_qkv_cab1_180", (unsigned)(q.nconv + 3 * gemmx_qkv_groups(cus - q.nconv, 3)), 1, 1, GX_THREADS, q);
            return;
        }
        launch(s, "hat_gemmx_qkv180", (unsigned)(3 * gemmx_qkv_groups(cus, 3)), 1, 1, GX_THREADS, p);
        return;
    }
    if (e.cab || e.conv1) throw Error("GEMM: this shape takes no CAB conv");
    if (!L.w) throw Error("GEMM: the FP32 weights were not uploaded");
    int wbn = 0;
    if (const char* ws = gemm_ws_kernel(L, epi, &wbn)) {
        // One block per CU (its 85 or 150 KB weight slice fills the LDS); the
        // (column slice, row tile) units are dealt out round-robin over the blocks.
        static const int cus = std::max(1, Runtime::get().cu_count());
        const long ntiles = (M + ws_rows(epi) - 1) / ws_rows(epi);
        const long units = ntiles * ((L.N + wbn - 1) / wbn);
        launch(s, ws, (unsigned)std::max(1L, std::min<long>(units, cus)), 1, 1, ws_waves(epi) * 64, p);
        return;
    }
    launch(s, gemm_kernel(L.N, epi), (unsigned)((M + 127) / 128), (unsigned)((L.N + BN - 1) / BN), 1,
           256, p);
}

// The MLP of one block that runs no split tail: x_out = res + fc2(gelu(fc1(a))),
// for EPI_RESID_LN also xn = LayerNorm(x_out). One fused kernel for C = 144
// (hidden 288) with the norm, else fc1 and fc2 as two GEMMs through a T x hidden
// buffer.
bool mlp_fused(const DevLinear& fc1, const DevLinear& fc2, int epi)
{
    return epi == EPI_RESID_LN && fc1.K == 144 && fc1.Kp == 144 && fc1.N == 288 && fc2.K == 288 && fc2.N == 144;
}

void run_mlp(hipStream_t s, const DevLinear& fc1, const DevLinear& fc2, const float* a, long M,
             const float* res, float* out, int epi, const GemmEpilogue& ln, float* hidden)
{
    if (epi != EPI_RESID && epi != EPI_RESID_LN) throw Error("MLP: bad epilogue");
    if (mlp_fused(fc1, fc2, epi)) {
        if (M > 0x7fffffffL) throw Error("MLP: too many rows");
        if (!fc1.w || !fc2.w) throw Error("MLP: the FP32 weights were not uploaded");
        MlpArgs p{};
        p.a = a;
        p.w1 = fc1.w;
        p.b1 = fc1.b;
        p.w2 = fc2.w;
        p.b2 = fc2.b;
        p.res = res;
        p.out = out;
        p.xn = ln.xn;
        p.nw = ln.nw;
        p.nb = ln.nb;
        p.M = (int)M;
        p.eps = 1e-5f;
        p.ldw1 = fc1.Kp;
        p.ldw2 = fc2.Kp;
        // One block per CU (113 KB of LDS), persistent over the 128-row tiles.
        static const int cus = std::max(1, Runtime::get().cu_count());
        const long ntiles = (M + MLP_ROWS - 1) / MLP_ROWS;
        const long rounds = (ntiles + cus - 1) / cus;
        const long g = std::max(1L, (ntiles + rounds - 1) / rounds);
        launch(s, "hat_mlp_resid_ln", (unsigned)g, 1, 1, MLP_WAVES * 64, p);
        return;
    }
    if (!hidden) throw Error("MLP: the unfused form needs a hidden buffer");
    GemmEpilogue e = ln;
    e.res = res;
    run_gemm(s, fc1, a, fc1.K, M, hidden, fc1.N, EPI_GELU, GemmEpilogue{}, 0, 0, 0.f);
    run_gemm(s, fc2, hidden, fc1.N, M, out, fc2.N, epi, e, 0, 0, 0.f);
}

// Folded CAB, first half: t1 = gelu(conv1(xn)) with its per-tile sums; the gate's
// arguments go to *gate, for the attention launch to run: the gate-scaled conv2
// weights (w2gx) and combined bias (bias2 = bproj + cscale * gate * b2) of the
// tail. With `conv_defer`, conv1 is not launched either (for the qkv linear's launch).
void run_cab(hipStream_t s, const DevCab& cb, const float* xn, int H, int W, const float* bproj,
             float cscale, int sq, float* t1, float* partial, float* bias2, float* gate_out,
             unsigned short* w2gx, float ts, float gs, CabGateArgs* gate, CabConvArgs* conv_defer)
{
    if (H % 16 != 0 || W % 16 != 0 || H < 16 || W < 16) throw Error("CAB: plane must be 16-aligned");
    if (sq < 1 || sq > 64) throw Error("CAB: squeeze width must be 1..64");
    static const int cus = std::max(1, Runtime::get().cu_count());
    CabConvArgs a{};
    a.xn = xn;
    a.w = cb.w1;
    a.bias = cb.b1;
    a.t1 = t1;
    a.partial = partial;
    a.H = H;
    a.W = W;
    cab_scales(ts, cb.oscale, &a);
    // Persistent over the 16 x 16 output tiles, two blocks of 4 waves per CU.
    const int tiles = (H / 16) * (W / 16);
    if (conv_defer) *conv_defer = a;
    else launch(s, "hat_cab_conv1", (unsigned)std::min(tiles, 2 * cus), 1, 1, 256, a);
    CabGateArgs& g = *gate;
    g = CabGateArgs{};
    g.partial = partial;
    g.t1 = t1;
    g.tiles = tiles;
    g.H = H;
    g.W = W;
    g.w2 = cb.w2;
    g.b2 = cb.b2;
    g.wa = cb.wa;
    g.ba = cb.ba;
    g.wb = cb.wb;
    g.bb = cb.bb;
    g.bproj = bproj;
    g.bias2 = bias2;
    g.gate = gate_out;
    g.cscale = cscale;
    g.sq = sq;
    g.w2gx = w2gx;
    g.ts = ts;
    g.gs = gs;
}

// The tail on split-f16 (tailx.hip): x' = res + a . Wp^T + bias (+ t1: the gated
// conv2 w2gx of it on the H x W plane, C = 144; + aux * gate * cscale, C = 180);
// out = x' + MLP(norm2(x')) (+ with nw: xn = norm_next(out)). The HAB's forms have
// a CAB and a next norm, the OCAB's neither. out may alias res.
struct TailCabIn {
    const float* t1 = nullptr;
    const unsigned short* w2gx = nullptr;
    const float *aux = nullptr, *gate = nullptr;
    float cscale = 0.0f;
    int H = 0, W = 0;
};
void run_tailx(hipStream_t s, const DevTail& t, const float* a, const float* res, float* out, float* xn, const float* bias,
               const float* b2, const float* n2w, const float* n2b, const float* nw, const float* nb, long M,
               const TailCabIn& cab, Amax* out_max = nullptr)
{
    const bool hab = nw != nullptr;
    if (hab != (t.C == 144 ? cab.t1 && cab.w2gx : cab.aux && cab.gate))
        throw Error("tailx: the HAB's form needs its CAB and the next norm, the OCAB's has neither");
    if (M > 0x7fffffffL) throw Error("tailx: too many rows");
    TailXArgs f{};
    f.a = a;
    f.res = res;
    f.out = out;
    f.xn = hab ? xn : nullptr;
    f.w = t.w;
    f.wm = t.wm;
    f.w2gx = cab.w2gx;
    f.t1 = cab.t1;
    f.aux = cab.aux;
    f.gate = cab.gate;
    f.bias = bias;
    f.b1x = t.b1x;
    f.b2 = b2;
    f.inw = n2w;
    f.inb = n2b;
    f.nw = nw;
    f.nb = nb;
    f.M = (int)M;
    f.H = cab.H;
    f.W = cab.W;
    f.eps = 1e-5f;
    f.cscale = cab.cscale;
    tail_scales(t, &f);
    if (out_max && !hab) {
        f.amax_out = out_max->slot;
        out_max->filled = true;
    }
    static const int cus = std::max(1, Runtime::get().cu_count());
    // One 64-token block a CU at most: there the larger blocks would leave half the
    // CUs idle, and past it two rounds of small ones take as long as one of large
    // (hat_habx_cab_ln at 4096 / 16384 / 65536 tokens: 34.2 / 37.5 / 66.1 us in
    // 128-token blocks, 23.3 / 27.6 / 98.8 in 64; C = 180: 45.0 / 49.8 / 99.1 and
    // 30.7 / 38.8 / 145.3).
    const bool small = wx_tiles((int)M, WX_ROWS_S) <= cus;
    const char* name = t.C == 144 ? (hab ? (small ? "hat_habx_cab_ln_s" : "hat_habx_cab_ln") : small ? "hat_habx_s" : "hat_habx")
                                  : hab ? (small ? "hat_habx180_hab_ln_s" : "hat_habx180_hab_ln")
                                        : small ? "hat_habx180_s" : "hat_habx180";
    launch(s, name, (unsigned)wx_tiles((int)M, small ? WX_ROWS_S : WX_ROWS), 1, 1, WX_THREADS, f);
}

// The channel-attention gate from the CAB conv's per-tile column sums:
// reduce in fixed row blocks, then squeeze-excite.
// With `defer` (C <= 192, sq <= 64), nothing is launched: *defer gets the
// arguments for the attention launch's first block, which adds the nblk
// partial rows itself.
void run_se(hipStream_t s, const float* partial, int nblk, int C, float* red, float count,
            const float* w1, const float* b1, const float* w2, const float* b2, int sq, float* gate,
            SeArgs* defer = nullptr)
{
    if (defer && C <= 192 && sq >= 1 && sq <= 64) {
        SeArgs se{};
        se.partial = partial;
        se.nblk = nblk;
        se.co_stride = C;
        se.count = count;
        se.w1 = w1;
        se.b1 = b1;
        se.w2 = w2;
        se.b2 = b2;
        se.gate = gate;
        se.C = C;
        se.sq = sq;
        *defer = se;
        return;
    }
    if (defer) defer->gate = nullptr;  // not deferred: launched here
    const int rows_per = 32;
    const int nred = (nblk + rows_per - 1) / rows_per;
    ReduceArgs r{partial, red, nblk, C, C, rows_per};
    launch(s, "hat_colsum_reduce", (unsigned)nred, 1, 1, 256, r);
    SeArgs se{};
    se.partial = red;
    se.nblk = nred;
    se.co_stride = C;
    se.count = count;
    se.w1 = w1;
    se.b1 = b1;
    se.w2 = w2;
    se.b2 = b2;
    se.gate = gate;
    se.C = C;
    se.sq = sq;
    launch(s, "hat_se_gate", 1, 1, 1, 256, se);
}

// The C = 180 CAB conv2 60 -> 180 and its column sums run on the Winograd
// kernel (hat_convwino_cab2_180, one partial row per 8x16 tile); other CO in
// (144, 192] on the wide-tile kernel (one per 16x16 tile); every other
// CEPI_COLSUM conv leaves one per 8x16 tile.
bool colsum_wide(int CO, int H, int W, int co_stride)
{
    return CO > 144 && CO <= 192 && CO != 180 && H % 16 == 0 && W % 16 == 0 && CO % 4 == 0 && co_stride % 4 == 0;
}
int colsum_rows(int CO, int H, int W, int co_stride)
{
    return colsum_wide(CO, H, W, co_stride) ? (W / 16) * (H / 16) : (W / 16) * (H / 8);
}

// The Winograd kernels' scales: V's from the host, or (in_max) of the input's
// largest magnitude, found here over its n floats where no kernel has left it.
void wino_scales(hipStream_t s, const DevConv& C, long n, Amax* in_max, Amax* out_max, ConvArgs* p)
{
    p->uinv = C.uinv;
    p->vs = C.vs;
    if (in_max) {
        if (!in_max->filled) {
            AbsMaxArgs a{p->in, in_max->slot, n};
            launch(s, "hat_absmax", (unsigned)std::min<long>((n + 4095) / 4096, 2048), 1, 1, 256, a);
            in_max->filled = true;
        }
        p->amax = in_max->slot;
    }
    if (out_max) {
        p->amax_out = out_max->slot;
        out_max->filled = true;
    }
}

// A Winograd conv, in its small planes' form while those blocks are one round of the
// CUs: the trunk convs at 64 x 64 32.9 -> 17.6 us (C = 144) and 27.1 -> 21.2 (180),
// cab2_180 14.8 -> 12.0, n4_store 18.9 -> 14.8; past one round the repeated V costs
// more than the wider spread gives (128 x 128: resid180 36.0 and 41.5 us, cab2_180 18.8
// and 21.0, the upsample conv at 128 x 128 24 and 24.9).
void launch_wino_for(hipStream_t s, const char* name, unsigned tiles, unsigned ncb, ConvArgs& p)
{
    static const unsigned cus = (unsigned)std::max(1, Runtime::get().cu_count());
    const WinoSmall k = convwino_small(name);
    if ((size_t)tiles * k.ncb <= cus) launch_wino(s, k.name.c_str(), tiles, k.ncb, p);
    else launch_wino(s, name, tiles, ncb, p);
}

// [band_r0, band_r1): with band_r1 >= 0, only that band of tile rows is
// launched (the host-memory forward's head): 8 input rows of the Winograd
// upsample conv (hat_convwino_n8_shuffle), 16 output rows of conv_last
// (hat_conv_last3), the same band indices for the two since the shuffle
// doubles the rows. Other convs are always whole planes. With `defer`, the C = 180
// CAB's conv1 is not launched: its arguments go to *defer (the qkv linear's launch).
void run_conv(hipStream_t s, const DevConv& C, const float* in, int cin_stride, int H, int W,
              float* out, int co_stride, int epi, int act, const float* res, float* partial,
              int crop_h, int crop_w, float img_range, const float* mean, int band_r0, int band_r1, Amax* in_max,
              Amax* out_max, float os, ConvArgs* defer = nullptr)
{
    if (H % 8 != 0 || W % 16 != 0) throw Error("conv: plane must be a multiple of 8x16");
    const bool band = band_r1 >= 0;
    if (band && (band_r0 < 0 || band_r0 >= band_r1)) throw Error("conv: empty band");
    if (cin_stride % 4 != 0 || cin_stride < C.CI) throw Error("conv: bad input channel stride");
    // The wide-tile kernel (16x16 pixels, a whole 64-, 96- or 128-channel
    // column block per block) for the head convs, the 60-channel CAB conv and
    // the C = 180 trunk convs.
    const char* wide = nullptr;
    int wbn = 0, wwaves = 0;
    if (H % 16 == 0 && W % 16 == 0 && C.CO % 4 == 0 && co_stride % 4 == 0) {
        if (epi == CEPI_STORE && C.CO > 16 && C.CO <= 64) {
            wide = "hat_convw_n4_store";
            wbn = 64;
            wwaves = CONVW_WAVES_N4_STORE;
        } else if (epi == CEPI_SHUFFLE) {
            wide = "hat_convw_n8_shuffle";
            wbn = 128;
            wwaves = CONVW_WAVES_N8_SHUFFLE;
        } else if (epi == CEPI_RESID && C.CO > 144 && C.CO <= 192) {
            wide = "hat_convw_n6_resid";  // C = 180 trunk convs, two 96-channel blocks
            wbn = 96;
            wwaves = CONVW_WAVES_N6_RESID;
        } else if (epi == CEPI_COLSUM && colsum_wide(C.CO, H, W, co_stride)) {
            wide = "hat_convw_n6_colsum";  // C = 180 CAB conv2
            wbn = 96;
            wwaves = CONVW_WAVES_N6_COLSUM;
        }
    }
    const char* name = nullptr;
    int BN = 16;
    switch (epi) {
    case CEPI_STORE:
        if (C.CO <= 16) { name = "hat_conv_n1_store"; BN = 16; }
        else if (C.CO <= 64) { name = "hat_conv_n4_store"; BN = 64; }
        else { name = "hat_conv_n3_store"; BN = 48; }
        break;
    case CEPI_RESID: name = "hat_conv_n3_resid"; BN = 48; break;
    case CEPI_COLSUM: name = "hat_conv_n3_colsum"; BN = 48; break;
    case CEPI_SHUFFLE:
        name = "hat_conv_n4_shuffle";
        BN = 64;
        if ((C.CO / (C.r * C.r)) % 4 != 0) throw Error("conv: shuffled width must be a multiple of 4");
        break;
    case CEPI_FINAL: name = "hat_conv_n1_final"; BN = 16; break;
    default: throw Error("conv: unknown epilogue");
    }
    ConvArgs p{};
    p.in = in;
    p.w = C.w;
    p.bias = C.b;
    p.out = out;
    p.res = res;
    p.partial = partial;
    p.H = H;
    p.W = W;
    p.CI = C.CI;
    p.CIp = C.CIp;
    p.cin_stride = cin_stride;
    p.CO = C.CO;
    p.COp = C.COp;
    p.co_stride = co_stride;
    p.act = act;
    p.r = C.r;
    p.crop_h = crop_h;
    p.crop_w = crop_w;
    p.img_range = img_range;
    if (mean) {
        p.mean0 = mean[0];
        p.mean1 = mean[1];
        p.mean2 = mean[2];
    }
    // conv_before_upsample and the x2 upsample convs by Winograd F(2x2, 3x3):
    // 8 x 16 output tiles, 32-bit element offsets into both planes
    p.wu = C.wu;
    p.os = os;
    auto wino = [&](const char* name, unsigned tiles, unsigned ncb) {
        wino_scales(s, C, (long)H * W * cin_stride, in_max, out_max, &p);
        launch_wino_for(s, name, tiles, ncb, p);
    };
    const size_t rr = C.r > 0 ? (size_t)C.r * C.r : 1;
    if (C.wu && H % 16 == 0 && W % 16 == 0 && cin_stride % 4 == 0 && cin_stride >= C.CI &&
        (size_t)H * W * cin_stride < ((size_t)1 << 31) && (size_t)H * W * rr * co_stride < ((size_t)1 << 31)) {
        const unsigned tiles = (unsigned)((W / 16) * (H / 8));
        if (epi == CEPI_STORE && act == 2 && C.CO == 64 && C.CI == 144 && co_stride >= 64) {
            wino("hat_convwino_n4_store", tiles, 1);
            return;
        }
        if (epi == CEPI_SHUFFLE && C.r == 2 && C.CO == 256 && C.CI == 64 && co_stride >= 64) {
            unsigned nt = tiles;
            if (band) {
                if (band_r1 > H / 8) throw Error("conv: band past the plane");
                p.tile0 = band_r0 * (W / 16);
                nt = (unsigned)((band_r1 - band_r0) * (W / 16));
            }
            wino("hat_convwino_n8_shuffle", nt, 2);
            return;
        }
        if (band) throw Error("conv: only the Winograd upsample conv and conv_last run in bands");
        // the C = 180 family (the residual epilogue's planes are 180 wide)
        if (epi == CEPI_STORE && act == 2 && C.CO == 64 && C.CI == 180 && co_stride >= 64) {
            wino("hat_convwino_n4_store180", tiles, 1);
            return;
        }
        if (epi == CEPI_STORE && act == 1 && C.CO == 60 && C.CI == 180 && co_stride >= 60) {
            if (defer) {
                wino_scales(s, C, (long)H * W * cin_stride, in_max, out_max, &p);
                *defer = p;
                return;
            }
            wino("hat_convwino_cab1_180", tiles, 1);
            return;
        }
        if (epi == CEPI_COLSUM && C.CO == 180 && C.CI == 60 && co_stride >= 180) {
            wino("hat_convwino_cab2_180", tiles, 2);
            return;
        }
        if (epi == CEPI_RESID && C.CO == 180 && C.CI == 180 && co_stride == 180) {
            if (in == out) throw Error("conv: the output must not overlap the input");
            wino("hat_convwino_resid180", tiles, 2);
            return;
        }
    }
    if (defer) throw Error("conv: only the C = 180 CAB's conv1 rides on another launch");
    if (band && !(epi == CEPI_FINAL && C.CO == 3 && C.CI == 64 && C.CIp == 64 && cin_stride >= 64))
        throw Error("conv: only the Winograd upsample conv and conv_last run in bands");
    if (wide) {
        launch(s, wide, (unsigned)((W / 16) * (H / 16)), (unsigned)((C.CO + wbn - 1) / wbn), 1,
               (unsigned)(wwaves * 64), p);
        return;
    }
    if (epi == CEPI_FINAL) {
        if (crop_h > H || crop_w > W || crop_h < 1 || crop_w < 1) throw Error("conv: bad crop");
        // conv_last 64 -> 3 by per-tap products, 16 x 32 output tiles
        if (C.CO == 3 && C.CI == 64 && C.CIp == 64 && cin_stride >= 64) {
            const int ntx = (W + 31) / 32, nty = (H + 15) / 16;  // 16 x 32 output tiles
            unsigned nt = (unsigned)(ntx * nty);
            if (band) {
                if (band_r1 > nty) throw Error("conv: band past the plane");
                p.tile0 = band_r0 * ntx;
                nt = (unsigned)((band_r1 - band_r0) * ntx);
            }
            launch(s, "hat_conv_last3", nt, 1, 1, 512, p);
            return;
        }
    }
    launch(s, name, (unsigned)((W / 16) * (H / 8)), (unsigned)((C.CO + BN - 1) / BN), 1, 256, p);
}

// A C -> 144 3x3 conv with every output channel in one block and a GEMM
// epilogue: EPI_STORE_LN (out, xn = LN(out)), EPI_RESID_LN (out = conv + res,
// xn = LN(out)) or EPI_RESID. out may alias res; in, out and xn must not overlap.
bool convw_fits(const DevConv& C) { return C.r == 0 && C.CO == 144 && C.COp == 144; }

void run_ln(hipStream_t s, const float* x, float* y, const float* w, const float* b, long rows, int C);

void run_convw(hipStream_t s, const DevConv& C, const float* in, int cin_stride, int H, int W,
               float* out, int epi, const float* res, float* xn, const float* nw, const float* nb, Amax* in_max,
               Amax* out_max)
{
    if (!convw_fits(C)) throw Error("convw: needs 144 output channels");
    if (H % 16 != 0 || W % 16 != 0) throw Error("convw: plane must be 16-aligned");
    if (cin_stride % 4 != 0 || cin_stride < C.CI) throw Error("convw: bad input channel stride");
    const char* name = epi == EPI_STORE_LN   ? "hat_convw_n9_store_ln"
                       : epi == EPI_RESID_LN ? "hat_convw_n9_resid_ln"
                       : epi == EPI_RESID    ? "hat_convw_n9_resid"
                                             : nullptr;
    if (!name) throw Error("convw: bad epilogue");
    const int waves = epi == EPI_STORE_LN   ? CONVW_WAVES_N9_STORE_LN
                      : epi == EPI_RESID_LN ? CONVW_WAVES_N9_RESID_LN
                                            : CONVW_WAVES_N9_RESID;
    ConvArgs p{};
    p.in = in;
    p.w = C.w;
    p.bias = C.b;
    p.out = out;
    p.res = res;
    p.H = H;
    p.W = W;
    p.CI = C.CI;
    p.CIp = C.CIp;
    p.cin_stride = cin_stride;
    p.CO = C.CO;
    p.COp = C.COp;
    p.co_stride = C.CO;
    p.xn = xn;
    p.nw = nw;
    p.nb = nb;
    p.eps = 1e-5f;
    p.wu = C.wu;
    // The 144 -> 144 residual convs by Winograd F(2x2, 3x3): 8 x 16 output
    // tiles, 32-bit element offsets into the input plane. The RHAG conv's
    // LayerNorm follows as its own HBM-bound pass over the just-written rows.
    if (C.wu && C.CI == 144 && (epi == EPI_RESID_LN || epi == EPI_RESID) && H % 8 == 0 &&
        (size_t)H * W * cin_stride < ((size_t)1 << 31)) {
        if (in == out) throw Error("convw: the output must not overlap the input");
        wino_scales(s, C, (long)H * W * cin_stride, in_max, out_max, &p);
        launch_wino_for(s, "hat_convwino_resid", (unsigned)((W / 16) * (H / 8)), 1, p);
        if (epi == EPI_RESID_LN) run_ln(s, out, xn, nw, nb, (long)H * W, C.CO);
        return;
    }
    launch(s, name, (unsigned)((W / 16) * (H / 16)), 1, 1, (unsigned)(waves * 64), p);
}

void run_attn(hipStream_t s, const float* qkv, const float* table, float* out, const Plan& pl,
              int heads, int D, bool oca, int shift, bool f16, const CabGateArgs* gate = nullptr,
              const SeArgs* se = nullptr)
{
    if (se && oca) throw Error("attention: the SE gate rides on SW launches only");
    if (gate && oca) throw Error("attention: the CAB gate rides on SW launches only");
    if (pl.win != 16 || pl.owin != 24)
        throw Error("attention: the gfx950 kernels are built for window 16 / overlap window 24");
    // The kernels wrap a rolled coordinate once, upward, and build the SW-MSA
    // mask from bit 3 of the unrolled position: only the plan's half-window
    // shift (or none) is meaningful, and the OCAB has no shift.
    if (!(shift == 0 || (!oca && shift == pl.shift)))
        throw Error("attention: shift " + std::to_string(shift) + " is not supported (0" +
                    (oca ? "" : " or " + std::to_string(pl.shift)) + ")");
    const char* name = nullptr;
    // The split-f16 kernels (attnx.hip), one (window, head) item per block,
    // where q, k and v are known to lie inside f16's range; else the FP32 ones.
    if (D != 24 && D != 30)
        throw Error("attention: head_dim " + std::to_string(D) + " has no kernel (24 and 30 do)");
    if (f16) name = oca ? (D == 24 ? "hat_attnx_oca_d24" : "hat_attnx_oca_d30")
                        : (D == 24 ? "hat_attnx_sw_d24" : "hat_attnx_sw_d30");
    else name = oca ? (D == 24 ? "hat_attn_oca_d24" : "hat_attn_oca_d30")
                    : (D == 24 ? "hat_attn_sw_d24" : "hat_attn_sw_d30");
    AttnArgs p{};
    p.qkv = qkv;
    p.table = table;
    p.out = out;
    p.hp = pl.hp;
    p.wp = pl.wp;
    p.nx = pl.nx();
    p.ny = pl.ny();
    p.heads = heads;
    p.D = D;
    p.C = heads * D;
    p.shift = shift;
    p.owin = pl.owin;
    p.opad = pl.opad();
    p.T = (int)pl.tokens();
    p.qscale = (1.0f / sqrtf((float)D)) * 1.4426950408889634f;
    if (gate) {
        p.with_gate = 1;
        p.gate = *gate;
    }
    if (se && se->gate) {
        p.with_se = 1;
        p.se = *se;
    }
    if (!f16 && attn_persistent(D, oca)) {
        static const int cus = std::max(1, Runtime::get().cu_count());
        launch(s, name, (unsigned)std::min<long>((long)pl.nw() * heads, cus), 1, 1, 512, p);
        return;
    }
    // the split-f16 SW kernels run the gate as a column of blocks of its own
    const unsigned lead = f16 && (p.with_gate || p.with_se) ? 1 : 0;
    launch(s, name, (unsigned)pl.nw() + lead, (unsigned)heads, 1, 512, p);
}

void run_ln(hipStream_t s, const float* x, float* y, const float* w, const float* b, long rows, int C)
{
    if (C > 512) throw Error("layernorm: C > 512");
    LnArgs p{x, y, w, b, (int)rows, C, 1e-5f};
    // 16 rows per block when C % 4 == 0 and C <= 192, else 4 (one per wave)
    const long per = (C % 4 == 0 && C <= 192) ? 16 : 4;
    launch(s, "hat_layernorm", (unsigned)((rows + per - 1) / per), 1, 1, 256, p);
}

}  // namespace

bool convwino_persistent(const std::string& name)
{
    // convwino.hip: the column-sum kernel (the CAB's conv2 at C = 180)
    return name == "hat_convwino_cab2_180" || name == "hat_convwino_cab2_180_s";
}

WinoSmall convwino_small(const std::string& name)
{
    const unsigned ncb = name == "hat_convwino_resid" ? 3
                         : name == "hat_convwino_resid180" || name == "hat_convwino_cab2_180" || name == "hat_convwino_n8_shuffle"
                             ? 4
                             : 2;
    return {name + "_s", ncb};
}

void launch_wino(hipStream_t s, const char* name, unsigned tiles, unsigned ncb, ConvArgs& p, unsigned max_blocks)
{
    static const unsigned cus = (unsigned)std::max(1, Runtime::get().cu_count());
    const unsigned nvb = tiles * ncb;
    if (nvb == 0 || nvb > 0x7fffffffu || ncb == 0) throw Error("convwino: bad tile count");
    const bool persist = convwino_persistent(name);
    const unsigned cap = max_blocks ? max_blocks : cus;
    const unsigned g = persist ? std::max(ncb, std::min(nvb, cap) / ncb * ncb) : nvb;
    p.nblk = persist ? (int)nvb : 0;
    launch(s, name, g, 1, 1, 512, p);
}


// ---------------------------------------------------------------------------
// GpuBackend

// Weights are allocated in whole granules, which weight_bytes_ counts. No kernel
// needs them: none reads past a tensor (tailx.hip's whole loads end inside TX_PAD and
// TX_B1), and granules of 4 KB are as fast (64 x 64 HAT-S 2.031 ms and 2.030, 512 x 512
// 30.13 and 30.15, HAT 256 x 256 14.67 and 14.66). HAT-S takes 147.5 MiB so, 54.6 in
// granules of 4 KB; the memory admission's tests are written for the former.
static constexpr size_t kWeightGranule = 128u << 10;

float* GpuBackend::upload(const float* src, size_t n) { return (float*)upload_bytes(src, n * sizeof(float)); }

void* GpuBackend::upload_bytes(const void* src, size_t bytes)
{
    const size_t room = (bytes + kWeightGranule - 1) / kWeightGranule * kWeightGranule;
    weight_bytes_ += room;
    if (count_only_) return nullptr;
    Runtime& rt = Runtime::get();
    void* d = rt.alloc(room);
    owned_.push_back(d);
    rt.h2d(d, src, bytes);
    return d;
}

void GpuBackend::upload_raw(const std::string& name)
{
    const TensorInfo& ti = wt_.info(name);
    raw_[name] = upload(wt_.t(name), ti.numel());
}

// The qkv weights for hat_gemmx_qkv*: each of q, k and v scaled into f16's range
// (w: the linear's own weights, out[3] the results' factors, in the inverse of
// the input's scale); sets oscale.
static std::vector<unsigned short> split_qkv(const float* w, int N, int K, const float* out, float in, float* oscale,
                                             bool fill = true)
{
    float ws[3] = {1.0f, 1.0f, 1.0f};
    for (int i = 0; fill && i < 3; ++i) {
        ws[i] = f16_scale(abs_max(w + (size_t)i * (N / 3) * K, (size_t)(N / 3) * K));
        oscale[i] = in * out[i] / ws[i];
    }
    return pack_linear_ws(w, N, K, ws, fill);
}

void GpuBackend::upload_linear(const std::string& name, const float* out, float in, bool bias_only)
{
    const TensorInfo& ti = wt_.info(name + ".weight");
    DevLinear L;
    L.N = (int)ti.shape[0];
    L.K = (int)ti.shape[1];
    L.Kp = (L.K + 15) / 16 * 16;
    const float *w = wt_.t(name + ".weight"), *bias = wt_.t(name + ".bias");
    std::vector<float> bs(bias, bias + L.N);
    if (out)
        for (int n = 0; n < L.N; ++n) bs[n] *= out[n / (L.N / 3)];
    L.b = upload(bs.data(), L.N);
    bool split = false;
    if (out && ((L.K == 180 && L.N == 540) || (L.K == 144 && L.N == 432))) {
        // qkv: the weight-stationary layout of hat_gemmx_qkv
        std::vector<unsigned short> x = split_qkv(w, L.N, L.K, out, in, L.oscale, !count_only_);
        L.wx = (unsigned short*)upload_bytes(x.data(), x.size() * sizeof(unsigned short));
        split = true;
    } else if (!bias_only) {
        std::vector<float> ws(w, w + (size_t)L.N * L.K);
        for (int n = 0; n < L.N; ++n) {
            const float f = (out ? out[n / (L.N / 3)] : 1.0f) * in;
            for (int k = 0; k < L.K; ++k) ws[(size_t)n * L.K + k] *= f;
        }
        std::vector<float> pk = pack_linear(ws.data(), L.N, L.K, &L.Kp);
        L.w = upload(pk.data(), pk.size());
    }
    L.rows = !split && !bias_only;
    lin_[name] = L;
}

void GpuBackend::upload_norm(const std::string& name)
{
    const int C = wt_.embed;
    const float *w = wt_.t(name + ".weight"), *b = wt_.t(name + ".bias");
    // the widths with split-f16 kernels behind their norms
    const float s = C == 144 || C == 180 ? f16_scale(ln_bound(w, b, C)) : 1.0f;
    std::vector<float> v(C);
    for (int i = 0; i < C; ++i) v[i] = w[i] * s;
    raw_[name + ".weight"] = upload(v.data(), C);
    for (int i = 0; i < C; ++i) v[i] = b[i] * s;
    raw_[name + ".bias"] = upload(v.data(), C);
    norm_scale_[name] = s;
}

void GpuBackend::upload_attn(const std::string& qkv, const std::string& proj, const std::string& ln,
                             const std::string& table)
{
    const int C = wt_.embed;
    const float *w = wt_.t(qkv + ".weight"), *b = wt_.t(qkv + ".bias"), *lw = wt_.t(ln + ".weight"),
                *lb = wt_.t(ln + ".bias");
    QkvScale s;
    if (!count_only_)
        s = qkv_scale(ln_linear_bound(w, b, lw, lb, 0, C, C), ln_linear_bound(w, b, lw, lb, C, 2 * C, C),
                      ln_linear_bound(w, b, lw, lb, 2 * C, 3 * C, C), wt_.head_dim);
    const float out[3] = {s.q, s.k, s.v};
    upload_linear(qkv, out, 1.0f / norm_scale_.at(ln));
    attn_f16_[table] = s.ok;
    v_scale_ = s.v;
}

double GpuBackend::cab_t1_bound(const std::string& cab, const std::string& norm1) const
{
    // conv1's nine taps of norm1 rows, and |gelu(v)| <= |v|
    const size_t C = (size_t)wt_.embed;
    const float *w = wt_.t(cab + "0.weight"), *b = wt_.t(cab + "0.bias"), *lw = wt_.t(norm1 + ".weight"),
                *lb = wt_.t(norm1 + ".bias");
    std::vector<float> row(C);
    double worst = 0.0;
    for (int co = 0; co < wt_.compressed; ++co) {
        double v = std::fabs((double)b[co]);
        for (int tap = 0; tap < 9; ++tap) {
            for (size_t ci = 0; ci < C; ++ci) row[ci] = w[(co * C + ci) * 9 + tap];
            v += ln_linear_bound(row.data(), nullptr, lw, lb, 0, 1, (int)C);
        }
        if (std::isnan(v)) return v;
        worst = std::max(worst, v);
    }
    return worst;
}

void GpuBackend::upload_tail(const std::string& proj, const std::string& mlp, const std::string& norm2,
                             const std::string& cab, const std::string& norm1, bool ocab)
{
    const size_t C = (size_t)wt_.embed;
    upload_norm(norm2);
    const float sn = norm_scale_.at(norm2);
    const bool tail = tail_runs(wt_, ocab);
    upload_linear(proj, nullptr, 1.0f / v_scale_, tail);
    upload_linear(mlp + ".fc1", nullptr, 1.0f / sn, tail);
    upload_linear(mlp + ".fc2", nullptr, 1.0f, tail);
    if (!tail) return;
    TailCab tc{0.0, 0.0};
    if (!cab.empty() && !count_only_) {
        tc.t1 = cab_t1_bound(cab, norm1);
        tc.w2 = std::fabs((double)wt_.conv_scale) * abs_max(wt_.t(cab + "2.weight"), C * CAB_CC * 9);
    }
    TailPack p = pack_tail(wt_.t(proj + ".weight"), wt_.t(mlp + ".fc1.weight"), wt_.t(mlp + ".fc1.bias"),
                           wt_.t(mlp + ".fc2.weight"), wt_.t(norm2 + ".weight"), wt_.t(norm2 + ".bias"), (int)C, v_scale_, sn,
                           cab.empty() ? nullptr : &tc, !count_only_);
    p.t.w = (unsigned short*)upload_bytes(p.w.data(), p.w.size() * sizeof(unsigned short));
    p.t.wm = (unsigned short*)upload_bytes(p.wm.data(), p.wm.size() * sizeof(unsigned short));
    p.t.b1x = upload(p.b1x.data(), p.b1x.size());
    tail_[mlp] = p.t;
}

void GpuBackend::upload_conv(const std::string& name, int r, float in, double bound)
{
    const TensorInfo& ti = wt_.info(name + ".weight");
    DevConv C;
    C.CO = (int)ti.shape[0];
    C.CI = (int)ti.shape[1];
    C.r = r;
    std::vector<float> bias;
    const float* w = wt_.t(name + ".weight");
    std::vector<float> ws;
    if (in != 1.0f) {
        ws.assign(w, w + ti.numel());
        for (float& x : ws) x *= in;
        w = ws.data();
    }
    std::vector<float> pk = pack_conv(w, wt_.t(name + ".bias"), C.CO, C.CI, r, &bias, &C.CIp, &C.COp);
    C.w = upload(pk.data(), pk.size());
    C.b = upload(bias.data(), bias.size());
    if (wino_conv(C.CO, C.CI, r)) {
        std::vector<unsigned short> wu = pack_wino(w, C.CO, C.CI, r, &C.uinv, !count_only_);
        C.vs = f16_scale(4.0 * bound);  // |B^T d B| <= 4 max|d|
        C.wu = (unsigned short*)upload_bytes(wu.data(), wu.size() * sizeof(unsigned short));
    }
    conv_[name] = C;
}

// Which blocks' second half runs tailx.hip: C = 180, and at C = 144 the OCAB and
// the HAB with the folded CAB (there is no 144-channel tail for conv2's output).
// The others run the projection and the MLP as FP32 linears.
bool GpuBackend::tail_runs(const Weights& wt, bool ocab)
{
    return wt.mlp_ratio == 2 && (wt.embed == 180 || (wt.embed == 144 && (ocab || cab_folded(wt))));
}

// Every linear that a block reads as FP32 rows has them (upload_all).
void GpuBackend::check_linears() const
{
    auto need = [&](const std::string& proj, const std::string& mlp, bool ocab) {
        if (tail_runs(wt_, ocab)) return;
        for (const std::string& n : {proj, mlp + ".fc1", mlp + ".fc2"})
            if (!lin_.at(n).rows) throw Error("upload: " + n + " was left out, and its block reads it");
    };
    for (size_t s = 0; s < wt_.depths.size(); ++s) {
        const std::string L = "layers." + std::to_string(s) + ".residual_group.";
        for (int b = 0; b < wt_.depths[s]; ++b) {
            const std::string p = L + "blocks." + std::to_string(b);
            need(p + ".attn.proj", p + ".mlp", false);
        }
        need(L + "overlap_attn.proj", L + "overlap_attn.mlp", true);
    }
}

// Gpu::new (gpu.rs:372-386): bring up the runtime, then upload every tensor.
GpuBackend::GpuBackend(const Weights& wt) : wt_(wt)
{
    Runtime& rt = Runtime::get();
    check_gpu_weights(wt);
    if (wt.window != 16 || wt.owin != 24)
        throw Error("the gfx950 attention kernels are built for window 16 and overlap window 24");
    if (wt.head_dim != 24 && wt.head_dim != 30)
        throw Error("head_dim " + std::to_string(wt.head_dim) + " has no attention kernel (24, 30)");
    if (wt.embed % 4 != 0 || wt.embed > 512) throw Error("embed_dim must be a multiple of 4, <= 512");
    if (wt.squeezed > 64) throw Error("squeeze width above 64 is not supported");
    if (wt.head_feat % 4 != 0) throw Error("head width must be a multiple of 4");
    for (int d : wt.depths)
        if (d < 1) throw Error("every stage needs at least one HAB");
    cab_fold_ = cab_folded(wt);
    rt.check(rt.api().StreamCreate(&stream_), "hipStreamCreate");
    upload_all();
    if (!wt.device_bytes_cache) wt.device_bytes_cache = weight_bytes_;
}

GpuBackend::GpuBackend(const Weights& wt, CountOnly) : wt_(wt), count_only_(true)
{
    cab_fold_ = cab_folded(wt);
    upload_all();
}

size_t GpuBackend::device_weight_bytes(const Weights& wt)
{
    if (!wt.device_bytes_cache) wt.device_bytes_cache = GpuBackend(wt, CountOnly{}).weight_bytes_;
    return wt.device_bytes_cache;
}

// Every tensor of the network, packed as the kernels read it (Gpu::new's upload,
// gpu.rs:372-386).
void GpuBackend::upload_all()
{
    const Weights& wt = wt_;
    upload_conv("conv_first");
    upload_raw("patch_embed.norm.weight");
    upload_raw("patch_embed.norm.bias");
    for (size_t s = 0; s < wt.depths.size(); ++s) {
        const std::string L = "layers." + std::to_string(s);
        for (int b = 0; b < wt.depths[s]; ++b) {
            const std::string p = L + ".residual_group.blocks." + std::to_string(b);
            upload_norm(p + ".norm1");
            for (const char* n : {".attn.relative_position_bias_table",
                                  ".conv_block.cab.3.attention.1.weight",
                                  ".conv_block.cab.3.attention.1.bias",
                                  ".conv_block.cab.3.attention.3.weight",
                                  ".conv_block.cab.3.attention.3.bias"})
                upload_raw(p + n);
            upload_attn(p + ".attn.qkv", p + ".attn.proj", p + ".norm1", p + ".attn.relative_position_bias_table");
            upload_tail(p + ".attn.proj", p + ".mlp", p + ".norm2", cab_fold_ ? p + ".conv_block.cab." : std::string(),
                        p + ".norm1", false);
            const float xin = 1.0f / norm_scale_.at(p + ".norm1");
            if (cab_fold_) {
                const std::string c = p + ".conv_block.cab.";
                for (const char* n : {"0.bias", "2.weight", "2.bias"}) upload_raw(c + n);
                const float* w0 = wt.t(c + "0.weight");
                const float sw = f16_scale(abs_max(w0, wt.info(c + "0.weight").numel()));
                std::vector<unsigned short> w1 = pack_cab_conv1(w0, sw);
                DevCab cb;
                cb.oscale = xin / sw;
                cb.w1 = (unsigned short*)upload_bytes(w1.data(), w1.size() * sizeof(unsigned short));
                cb.b1 = raw_.at(c + "0.bias");
                cb.w2 = raw_.at(c + "2.weight");
                cb.b2 = raw_.at(c + "2.bias");
                cb.wa = raw_.at(c + "3.attention.1.weight");
                cb.ba = raw_.at(c + "3.attention.1.bias");
                cb.wb = raw_.at(c + "3.attention.3.weight");
                cb.bb = raw_.at(c + "3.attention.3.bias");
                cab_[p] = cb;
            } else {
                // norm1's rows are below 2^15 as stored (upload_norm); conv1
                // leaves t1 scaled for conv2's transform
                const float ts = wino_conv(wt.embed, wt.compressed, 0) && !count_only_
                                     ? f16_scale(4.0 * cab_t1_bound(p + ".conv_block.cab.", p + ".norm1")) : 1.0f;
                t1_scale_[p] = ts;
                upload_conv(p + ".conv_block.cab.0", 0, xin, 32768.0);
                upload_conv(p + ".conv_block.cab.2", 0, 1.0f / ts, 8192.0);
            }
        }
        const std::string p = L + ".residual_group.overlap_attn";
        upload_norm(p + ".norm1");
        upload_raw(p + ".relative_position_bias_table");
        upload_attn(p + ".qkv", p + ".proj", p + ".norm1", p + ".relative_position_bias_table");
        upload_tail(p + ".proj", p + ".mlp", p + ".norm2", std::string(), p + ".norm1", true);
        upload_conv(L + ".conv");
    }
    upload_raw("norm.weight");
    upload_raw("norm.bias");
    upload_conv("conv_after_body", 0, 1.0f, ln_bound(wt.t("norm.weight"), wt.t("norm.bias"), wt.embed));
    upload_conv("conv_before_upsample.0");
    const auto blocks = wt.up_blocks();
    for (size_t b = 0; b < blocks.size(); ++b)
        upload_conv("upsample." + std::to_string(2 * b), blocks[b].first);
    upload_conv("conv_last");
    check_linears();
}

GpuBackend::~GpuBackend()
{
    if (count_only_) return;
    try {
        Runtime& rt = Runtime::get();
        rt.api().StreamSynchronize(stream_);
        free_batch();
        free_plan();
        for (void* p : owned_) rt.free(p);
        for (hipEvent_t e : band_ev_) rt.api().EventDestroy(e);
        for (hipEvent_t e : copy_ev_) rt.api().EventDestroy(e);
        if (copy_stream_) rt.api().StreamDestroy(copy_stream_);
        rt.api().StreamDestroy(stream_);
    } catch (...) {
    }
}

void GpuBackend::free_plan()
{
    Runtime& rt = Runtime::get();
    free_stage();
    for (void* p : acts_) rt.free(p);
    acts_.clear();
    acts_bytes_ = 0;
    a_ = Acts{};
    have_plan_ = false;
}

// The compress-to-6 CAB at C = 144 (HAT-S) runs folded (cab.hip, tailx.hip).
bool GpuBackend::cab_folded(const Weights& wt) { return wt.embed == CAB_C && wt.compressed == CAB_CC; }

size_t GpuBackend::plan_bytes(const Weights& wt, int h, int w, bool host_io)
{
    Acts a;
    size_t n = 0;
    for (auto& b : layout(wt, Plan::make(h, w, wt.window, wt.embed), a, host_io)) n += b.second * sizeof(float);
    return n;
}

// Acts::new (gpu.rs:293-334): the buffer set of one plan.
std::vector<std::pair<float**, size_t>> GpuBackend::layout(const Weights& wt_, const Plan& p, Acts& a,
                                                           bool host_io)
{
    const size_t T = (size_t)p.tokens(), C = wt_.embed;
    const size_t t1_stride = (size_t)(wt_.compressed + 3) / 4 * 4;
    const size_t nblk = (size_t)colsum_rows((int)C, p.hp, p.wp, (int)C);
    const bool cab_fold_ = cab_folded(wt_);
    // The T x hidden buffer only for MLP shapes without a fused kernel (every
    // block of a network shares one shape: fc1 C -> mlp_ratio * C).
    const bool fused_mlp = wt_.mlp_ratio == 2 && (C == 144 || C == 180);
    // Head ping-pong: the plane at each resolution goes to alternate buffers.
    size_t need[2] = {T * (size_t)wt_.head_feat, 0};
    size_t res = 1;
    int which = 0;
    for (auto& b : wt_.up_blocks()) {
        res *= (size_t)b.first * b.first;
        which ^= 1;
        need[which] = std::max(need[which], T * res * (size_t)wt_.head_feat);
    }
    const size_t s2 = (size_t)wt_.scale * wt_.scale;
    return {
        {&a.x0, T * 4},
        {&a.body, T * C},
        {&a.xa, T * C},
        {&a.xb, T * C},
        {&a.xn, T * C},
        {&a.t1, T * t1_stride},
        {&a.cab_part, cab_fold_ ? (size_t)(p.hp / 16) * (p.wp / 16) * CAB_NSUM * CAB_CS : 0},
        {&a.w2gx, cab_fold_ ? (size_t)CAB_W2GX : 0},
        {&a.bias2, cab_fold_ ? C : 0},
        // (the folded CAB's are in w2gx's buffer: magnitude_slots)
        {&a.amax, cab_fold_ ? 0 : (size_t)AMAX_SLOTS * AMAX_WORDS},
        {&a.t2, cab_fold_ ? 0 : T * C},
        {&a.partial, cab_fold_ ? 0 : nblk * C},
        {&a.red, cab_fold_ ? 0 : (nblk + 31) / 32 * C},
        {&a.gate, C},
        {&a.qkv, 3 * T * C},
        {&a.ao, T * C},
        {&a.hidden, fused_mlp ? 0 : T * C * wt_.mlp_ratio},
        {&a.head0, need[0]},
        {&a.head1, std::max<size_t>(need[1], 4)},
        {&a.din, host_io ? 3 * (size_t)p.h * p.w : 0},
        {&a.dout, host_io ? 3 * (size_t)p.h * p.w * s2 : 0},
    };
}

// One allocation set per plan, reused by every forward at that size. A new
// plan is admitted against the device's free memory first (gpu.rs:766-771).
void GpuBackend::ensure_plan(int h, int w)
{
    Plan p = Plan::make(h, w, wt_.window, wt_.embed);
    if (have_plan_ && p == plan_) return;
    check_gpu(wt_, (size_t)h, (size_t)w);
    free_plan();
    plan_ = p;
    Runtime& rt = Runtime::get();
    t1_stride_ = (wt_.compressed + 3) / 4 * 4;
    nblk_conv2_ = colsum_rows(wt_.embed, p.hp, p.wp, wt_.embed);
    a_ = Acts{};
    for (auto& b : layout(wt_, p, a_, true)) {
        if (b.second == 0) continue;
        float* d = (float*)rt.alloc(b.second * sizeof(float));
        acts_.push_back(d);
        acts_bytes_ += b.second * sizeof(float);
        *b.first = d;
    }
    have_plan_ = true;
}

void GpuBackend::layernorm(const float* x, float* y, const std::string& prefix, long rows)
{
    run_ln(stream_, x, y, raw_.at(prefix + ".weight"), raw_.at(prefix + ".bias"), rows, wt_.embed);
}

void GpuBackend::gemm(const DevLinear& L, const float* a, int lda, long M, float* out, int ldo,
                      int epi, const float* res, const float* aux, const float* gate, float* xn,
                      const std::string& norm)
{
    GemmEpilogue e;
    e.res = res;
    e.aux = aux;
    e.gate = gate;
    e.xn = xn;
    if (!norm.empty()) {
        e.nw = raw_.at(norm + ".weight");
        e.nb = raw_.at(norm + ".bias");
    }
    run_gemm(stream_, L, a, lda, M, out, ldo, epi, e, wt_.heads, wt_.head_dim, wt_.conv_scale);
}

// x = x + fc2(gelu(fc1(a_.xn))), in place; with a norm also a_.xn = norm(x).
void GpuBackend::mlp(const std::string& prefix, float* x, int epi, const std::string& norm)
{
    GemmEpilogue e;
    if (!norm.empty()) {
        e.xn = a_.xn;
        e.nw = raw_.at(norm + ".weight");
        e.nb = raw_.at(norm + ".bias");
    }
    run_mlp(stream_, lin_.at(prefix + ".fc1"), lin_.at(prefix + ".fc2"), a_.xn, plan_.tokens(), x, x, epi,
            e, a_.hidden);
}

void GpuBackend::conv(const DevConv& C, const float* in, int cin_stride, int H, int W, float* out,
                      int co_stride, int epi, int act, const float* res, float* partial,
                      int crop_h, int crop_w, int band_r0, int band_r1, Amax* in_max, Amax* out_max, float os)
{
    run_conv(stream_, C, in, cin_stride, H, W, out, co_stride, epi, act, res, partial, crop_h,
             crop_w, wt_.img_range, wt_.mean, band_r0, band_r1, in_max, out_max, os);
}

void GpuBackend::attention(const std::string& table, bool oca, int shift, const CabGateArgs* gate,
                           const SeArgs* se)
{
    run_attn(stream_, a_.qkv, raw_.at(table), a_.ao, plan_, wt_.heads, wt_.head_dim, oca, shift,
             attn_f16_.at(table), gate, se);
}

// HAB.forward (hat_arch.py:266-309; cpu.rs:1090-1166):
//   x = shortcut + attn(norm1 x) + conv_x * conv_scale;  x = x + mlp(norm2 x)
// On entry a_.xn holds norm1(x_in); on exit x_out holds the block's result and
// a_.xn holds next_norm(x_out), the input of whatever block follows.
void GpuBackend::hab(int stage, int block, float* x_in, float* x_out, const std::string& next_norm)
{
    const std::string p = "layers." + std::to_string(stage) + ".residual_group.blocks." +
                          std::to_string(block);
    const long T = plan_.tokens();
    const int C = wt_.embed, H = plan_.hp, W = plan_.wp;
    if (cab_fold_) {
        // CAB, folded: conv1 + GELU here, the gate inside the attention
        // launch (a block of its own), conv2 inside the tail's projection.
        if (!tail_runs(wt_, false)) throw Error("HAB: the folded CAB needs an MLP of twice the block's width");
        const DevTail& tail = tail_.at(p + ".mlp");
        CabGateArgs gate{};
        CabConvArgs conv1{};
        const DevLinear& qkv = lin_.at(p + ".attn.qkv");
        const bool with = qkv_takes_cab1(qkv, wt_.heads, wt_.head_dim, H / 16 * (W / 16));  // conv1 in qkv's launch
        run_cab(stream_, cab_.at(p), a_.xn, H, W, lin_.at(p + ".attn.proj").b, wt_.conv_scale, wt_.squeezed, a_.t1,
                a_.cab_part, a_.bias2, a_.gate, (unsigned short*)a_.w2gx, tail.ts, tail.gs, &gate, with ? &conv1 : nullptr);
        GemmEpilogue e;
        e.cab = with ? &conv1 : nullptr;
        run_gemm(stream_, qkv, a_.xn, C, T, a_.qkv, 0, EPI_QKV, e, wt_.heads, wt_.head_dim, wt_.conv_scale);
        attention(p + ".attn.relative_position_bias_table", false, block % 2 == 1 ? plan_.shift : 0, &gate);
        // proj + gated conv2 + shortcut, norm2, the MLP + next norm1
        TailCabIn cab;
        cab.t1 = a_.t1;
        cab.w2gx = (const unsigned short*)a_.w2gx;
        cab.H = H;
        cab.W = W;
        run_tailx(stream_, tail, a_.ao, x_in, x_out, a_.xn, a_.bias2, lin_.at(p + ".mlp.fc2").b,
                  raw_.at(p + ".norm2.weight"), raw_.at(p + ".norm2.bias"), raw_.at(next_norm + ".weight"),
                  raw_.at(next_norm + ".bias"), T, cab);
        return;
    }
    // CAB: conv3x3 -> GELU -> conv3x3 (+ per-tile channel sums) -> gate; on small
    // planes the first conv in the qkv linear's launch.
    const DevLinear& qkv = lin_.at(p + ".attn.qkv");
    const DevConv& conv1 = conv_.at(p + ".conv_block.cab.0");
    const bool with = conv1.wu && conv1.CI == 180 && conv1.CO == 60 && t1_stride_ >= 60 && (size_t)T * C < ((size_t)1 << 31) &&
                      qkv_takes_cab1(qkv, wt_.heads, wt_.head_dim, H / 8 * (W / 16));
    ConvArgs c1{};
    run_conv(stream_, conv1, a_.xn, C, H, W, a_.t1, t1_stride_, CEPI_STORE, 1, nullptr, nullptr, 0, 0, wt_.img_range,
             wt_.mean, 0, -1, nullptr, nullptr, t1_scale_.at(p), with ? &c1 : nullptr);
    if (with) {
        GemmEpilogue e;
        e.conv1 = &c1;
        run_gemm(stream_, qkv, a_.xn, C, T, a_.qkv, 0, EPI_QKV, e, wt_.heads, wt_.head_dim, wt_.conv_scale);
    }
    conv(conv_.at(p + ".conv_block.cab.2"), a_.t1, t1_stride_, H, W, a_.t2, C, CEPI_COLSUM, 0, nullptr,
         a_.partial);
    // The gate: computed by the attention launch's first block where it fits.
    SeArgs se{};
    run_se(stream_, a_.partial, nblk_conv2_, C, a_.red, (float)T,
           raw_.at(p + ".conv_block.cab.3.attention.1.weight"),
           raw_.at(p + ".conv_block.cab.3.attention.1.bias"),
           raw_.at(p + ".conv_block.cab.3.attention.3.weight"),
           raw_.at(p + ".conv_block.cab.3.attention.3.bias"), wt_.squeezed, a_.gate, &se);
    // Window attention, the roll and the partition folded into its addressing;
    // proj's epilogue adds the shortcut and the gated conv branch, then norm2.
    if (!with) gemm(qkv, a_.xn, C, T, a_.qkv, 0, EPI_QKV);
    attention(p + ".attn.relative_position_bias_table", false, block % 2 == 1 ? plan_.shift : 0, nullptr, &se);
    const DevLinear& proj = lin_.at(p + ".attn.proj");
    if (tail_runs(wt_, false)) {
        // projection + gated conv branch + shortcut, norm2, the MLP + residual + next norm
        TailCabIn cab;
        cab.aux = a_.t2;
        cab.gate = a_.gate;
        cab.cscale = wt_.conv_scale;
        run_tailx(stream_, tail_.at(p + ".mlp"), a_.ao, x_in, x_out, a_.xn, proj.b, lin_.at(p + ".mlp.fc2").b,
                  raw_.at(p + ".norm2.weight"), raw_.at(p + ".norm2.bias"), raw_.at(next_norm + ".weight"),
                  raw_.at(next_norm + ".bias"), T, cab);
        return;
    }
    gemm(proj, a_.ao, C, T, x_out, C, EPI_HAB_LN, x_in, a_.t2, a_.gate, a_.xn, p + ".norm2");
    mlp(p + ".mlp", x_out, EPI_RESID_LN, next_norm);
}

// OCAB.forward (hat_arch.py:392-438; cpu.rs:1170-1198): x = proj(attn) + x;
// x = x + mlp(norm2 x). On entry a_.xn holds norm1(x).
void GpuBackend::ocab(int stage, float* x, Amax* out_max)
{
    const std::string p = "layers." + std::to_string(stage) + ".residual_group.overlap_attn";
    const long T = plan_.tokens();
    const int C = wt_.embed;
    gemm(lin_.at(p + ".qkv"), a_.xn, C, T, a_.qkv, 0, EPI_QKV);
    attention(p + ".relative_position_bias_table", true, 0);
    const DevLinear& proj = lin_.at(p + ".proj");
    if (tail_runs(wt_, true)) {
        run_tailx(stream_, tail_.at(p + ".mlp"), a_.ao, x, x, nullptr, proj.b, lin_.at(p + ".mlp.fc2").b, raw_.at(p + ".norm2.weight"),
                  raw_.at(p + ".norm2.bias"), nullptr, nullptr, T, TailCabIn{}, out_max);
        return;
    }
    gemm(proj, a_.ao, C, T, x, C, EPI_RESID_LN, x, nullptr, nullptr, a_.xn, p + ".norm2");
    mlp(p + ".mlp", x, EPI_RESID, "");
}

// forward_planes (gpu.rs:714-748; cpu.rs:1318-1368) with Pre::adjust and finish
// (backend.rs:71-109) folded into the first and last kernels.
void GpuBackend::forward_device(int h, int w, const float* d_in, float* d_out)
{
    if (h <= 0 || w <= 0) throw Error(std::to_string(h) + "x" + std::to_string(w) + " is empty");
    ensure_plan(h, w);
    run_forward(h, w, d_in, d_out);
}

size_t GpuBackend::noalloc_bytes(int h, int w) const
{
    if (h <= 0 || w <= 0) throw Error(std::to_string(h) + "x" + std::to_string(w) + " is empty");
    Acts a;
    size_t off = 0;
    for (auto& b : layout(wt_, Plan::make(h, w, wt_.window, wt_.embed), a, false))
        if (b.second) off += (b.second * sizeof(float) + 255) / 256 * 256;
    return off;
}

// forward_device with the per-plan buffers carved, 256-byte aligned, from the
// scratch array the code object holds (hipModuleGetGlobal at start-up), in
// place of the plan's own allocations, which are left as they are.
void GpuBackend::forward_noalloc(int h, int w, const float* d_in, float* d_out)
{
    if (h <= 0 || w <= 0) throw Error(std::to_string(h) + "x" + std::to_string(w) + " is empty");
    if (!d_in || !d_out) throw Error("null argument");
    Runtime& rt = Runtime::get();
    const Plan p = Plan::make(h, w, wt_.window, wt_.embed);
    // 64 KiB of the array stay unused past the last buffer, so no buffer ends
    // at the array's end.
    const size_t need = noalloc_bytes(h, w), cap = rt.scratch_bytes() - (64u << 10);
    if (need > cap) {
        char m[192];
        snprintf(m, sizeof m, "forward_noalloc: a %dx%d forward needs %.1f MiB of scratch; the library's "
                 "fixed array holds %.1f MiB", h, w, need / 1048576.0, cap / 1048576.0);
        throw Error(m);
    }
    Acts a;
    char* base = (char*)rt.scratch();
    size_t off = 0;
    for (auto& b : layout(wt_, p, a, false)) {
        if (b.second == 0) continue;
        *b.first = (float*)(base + off);
        off += (b.second * sizeof(float) + 255) / 256 * 256;
    }
    const Acts saved = a_;
    const Plan saved_plan = plan_;
    const int saved_nblk = nblk_conv2_;
    a_ = a;
    plan_ = p;
    t1_stride_ = (wt_.compressed + 3) / 4 * 4;
    nblk_conv2_ = colsum_rows(wt_.embed, p.hp, p.wp, wt_.embed);
    try {
        run_forward(h, w, d_in, d_out);
    } catch (...) {
        a_ = saved;
        plan_ = saved_plan;
        nblk_conv2_ = saved_nblk;
        throw;
    }
    a_ = saved;
    plan_ = saved_plan;
    nblk_conv2_ = saved_nblk;
}

unsigned* GpuBackend::magnitude_slots(int i) const
{
    static_assert(CAB_W2GX >= CAB_W2GX_USED + AMAX_SLOTS * AMAX_WORDS, "the slots fit behind the gated weights");
    unsigned* base = (unsigned*)(cab_fold_ ? a_.w2gx + CAB_W2GX_USED : a_.amax);
    return base + (size_t)i * AMAX_WORDS;
}

// The forward on the current plan's buffers (a_, plan_).
void GpuBackend::run_forward(int h, int w, const float* d_in, float* d_out, std::vector<std::pair<int, int>>* bands)
{
    const long T = plan_.tokens();
    const int C = wt_.embed, H = plan_.hp, W = plan_.wp;
    const size_t S = wt_.depths.size();
    // a magnitude slot each (the loader takes 32 stages and scales of few octaves)
    if (S > AMAX_HEAD || AMAX_HEAD + 2 + wt_.up_blocks().size() > AMAX_SLOTS)
        throw Error("forward: too many stages or upsample convs");
    PreArgs pa{d_in, a_.x0, h, w, H, W, 4, wt_.mean[0], wt_.mean[1], wt_.mean[2], wt_.img_range,
               magnitude_slots(0)};
    launch(stream_, "hat_pre", (unsigned)((T + 255) / 256), 1, 1, 256, pa);
    const DevConv& cf = conv_.at("conv_first");
    // With 144 channels the trunk convs carry the LayerNorm that follows them.
    const bool fused = convw_fits(cf);
    if ((C == 144 || C == 180) && cf.CI == 3 && cf.CIp == 16 && cf.CO == C && cf.r == 0 && H % 16 == 0 &&
        W % 16 == 0) {
        // conv_first + patch_embed.norm as one K = 27 GEMM (convfirst.hip)
        ConvArgs p{};
        p.in = a_.x0;
        p.w = cf.w;
        p.bias = cf.b;
        p.out = a_.body;
        p.xn = a_.xa;
        p.nw = raw_.at("patch_embed.norm.weight");
        p.nb = raw_.at("patch_embed.norm.bias");
        p.H = H;
        p.W = W;
        p.CI = cf.CI;
        p.CIp = cf.CIp;
        p.cin_stride = 4;
        p.CO = C;
        p.COp = cf.COp;
        p.co_stride = C;
        p.eps = 1e-5f;
        launch(stream_, C == 144 ? "hat_conv_first_ln144" : "hat_conv_first_ln180", (unsigned)((W / 16) * (H / 16)), 1,
               1, 256, p);
    } else if (fused) {
        run_convw(stream_, cf, a_.x0, 4, H, W, a_.body, EPI_STORE_LN, nullptr, a_.xa,
                  raw_.at("patch_embed.norm.weight"), raw_.at("patch_embed.norm.bias"), nullptr, nullptr);
    } else {
        conv(cf, a_.x0, 4, H, W, a_.body, C, CEPI_STORE, 0);
        layernorm(a_.body, a_.xa, "patch_embed.norm", T);
    }
    for (size_t s = 0; s < S; ++s) {
        // RHAG (gpu.rs:592-610): conv3x3(blocks(x)) + x, with the stage input
        // kept in a_.xa and the blocks working in a_.xb. Each block's last GEMM
        // leaves the next block's norm1 in a_.xn; the first block's comes from
        // the previous stage's conv (or its own pass).
        const std::string L = "layers." + std::to_string(s) + ".residual_group.";
        if (!fused || s == 0) layernorm(a_.xa, a_.xn, L + "blocks.0.norm1", T);
        for (int b = 0; b < wt_.depths[s]; ++b) {
            const std::string next = b + 1 < wt_.depths[s]
                                         ? L + "blocks." + std::to_string(b + 1) + ".norm1"
                                         : L + "overlap_attn.norm1";
            hab((int)s, b, b == 0 ? a_.xa : a_.xb, a_.xb, next);
        }
        // the stage's conv needs its input's range (no norm comes between)
        Amax xmax{magnitude_slots((int)s), false};
        ocab((int)s, a_.xb, &xmax);
        const DevConv& rc = conv_.at("layers." + std::to_string(s) + ".conv");
        if (fused) {
            // x = conv(blocks) + x, then the next stage's norm1 or the final
            // norm into a_.xn (a_.xb, the conv's input, is still being read).
            const std::string nn = s + 1 < S ? "layers." + std::to_string(s + 1) + ".residual_group.blocks.0.norm1"
                                             : std::string("norm");
            run_convw(stream_, rc, a_.xb, C, H, W, a_.xa, EPI_RESID_LN, a_.xa, a_.xn, raw_.at(nn + ".weight"),
                      raw_.at(nn + ".bias"), &xmax, nullptr);
        } else {
            conv(rc, a_.xb, C, H, W, a_.xa, C, CEPI_RESID, 0, a_.xa, nullptr, 0, 0, 0, -1, &xmax);
        }
    }
    // the head's planes: conv_after_body's output, then each conv's
    Amax hmax{magnitude_slots(AMAX_HEAD), false};
    if (fused) {
        run_convw(stream_, conv_.at("conv_after_body"), a_.xn, C, H, W, a_.xa, EPI_RESID, a_.body, nullptr,
                  nullptr, nullptr, nullptr, &hmax);
    } else {
        layernorm(a_.xa, a_.xb, "norm", T);
        conv(conv_.at("conv_after_body"), a_.xb, C, H, W, a_.xa, C, CEPI_RESID, 0, a_.body, nullptr, 0, 0, 0, -1, nullptr,
             &hmax);
    }
    // Head (gpu.rs:622-653): conv + LeakyReLU, [conv + PixelShuffle] per block, conv_last.
    const int feat = wt_.head_feat;
    Amax cmax{magnitude_slots(AMAX_HEAD + 1), false};  // of cur
    conv(conv_.at("conv_before_upsample.0"), a_.xa, C, H, W, a_.head0, feat, CEPI_STORE, 2, nullptr, nullptr, 0, 0, 0, -1,
         &hmax, &cmax);
    float* cur = a_.head0;
    float* nxt = a_.head1;
    int hh = H, ww = W;
    const auto blocks = wt_.up_blocks();
    const DevConv& last = conv_.at("conv_last");
    const int oh = h * wt_.scale, ow = w * wt_.scale;
    for (size_t b = 0; b < blocks.size(); ++b) {
        const DevConv& up = conv_.at("upsample." + std::to_string(2 * b));
        if (bands && b + 1 == blocks.size() && head_bands_fit(up, last, hh, ww, feat)) {
            // The last upsample conv and conv_last over bands of tile rows
            // (eighths of the plane, the last one split in two, so that the
            // first download starts early and the last one is short),
            // conv_last's band k after the upsample's band k + 1 (its halo
            // row below), an event after each conv_last band.
            const int R = hh / 8, step = (R + 7) / 8;  // at most 8 steps + the split: 10 bands
            std::vector<int> bnd{0};
            while (bnd.back() + step < R) bnd.push_back(bnd.back() + step);
            if (R - bnd.back() >= 2) bnd.push_back(bnd.back() + (R - bnd.back()) / 2);
            bnd.push_back(R);
            const int nb = (int)bnd.size() - 1;
            if (nb > (int)band_ev_.size()) throw Error("forward: too many output bands");
            bands->clear();
            conv(up, cur, feat, hh, ww, nxt, feat, CEPI_SHUFFLE, 0, nullptr, nullptr, 0, 0, bnd[0], bnd[1], &cmax);
            for (int k = 0; k < nb; ++k) {
                if (k + 1 < nb)
                    conv(up, cur, feat, hh, ww, nxt, feat, CEPI_SHUFFLE, 0, nullptr, nullptr, 0, 0, bnd[k + 1],
                         bnd[k + 2], &cmax);
                conv(last, nxt, feat, 2 * hh, 2 * ww, d_out, 0, CEPI_FINAL, 0, nullptr, nullptr, oh, ow, bnd[k],
                     bnd[k + 1]);
                Runtime::get().check(Runtime::get().api().EventRecord(band_ev_[k], stream_), "hipEventRecord");
                bands->emplace_back(std::min(oh, 16 * bnd[k]), std::min(oh, 16 * bnd[k + 1]));
            }
            return;
        }
        Amax nmax{magnitude_slots(AMAX_HEAD + 2 + (int)b), false};
        conv(up, cur, feat, hh, ww, nxt, feat, CEPI_SHUFFLE, 0, nullptr, nullptr, 0, 0, 0, -1, &cmax,
             b + 1 < blocks.size() ? &nmax : nullptr);
        cmax = nmax;
        hh *= blocks[b].first;
        ww *= blocks[b].first;
        std::swap(cur, nxt);
    }
    conv(last, cur, feat, hh, ww, d_out, 0, CEPI_FINAL, 0, nullptr, nullptr, oh, ow);
    if (bands) {
        // one band: the whole output
        if (band_ev_.empty()) throw Error("forward: no band events");
        Runtime::get().check(Runtime::get().api().EventRecord(band_ev_[0], stream_), "hipEventRecord");
        bands->assign(1, {0, oh});
    }
}

// Whether the head's last upsample conv (input hh x ww) and conv_last run on
// the kernels that take bands of tile rows: the Winograd x2 upsample and the
// 64 -> 3 conv_last, whose 16-row tiles are the upsample's 8-row tiles doubled.
bool GpuBackend::head_bands_fit(const DevConv& up, const DevConv& last, int hh, int ww, int feat) const
{
    return up.wu && up.r == 2 && up.CO == 256 && up.CI == 64 && feat == 64 && hh % 16 == 0 && ww % 16 == 0 &&
           (size_t)hh * ww * feat < ((size_t)1 << 31) && (size_t)hh * ww * 4 * feat < ((size_t)1 << 31) &&
           last.CO == 3 && last.CI == 64 && last.CIp == 64;
}

void GpuBackend::op_hab(int stage, int block, int hp, int wp, const float* x, float* out, int iters,
                        float* ms)
{
    if (!x || !out) throw Error("hab: null argument");
    if (stage < 0 || stage >= (int)wt_.depths.size())
        throw Error("hab: stage " + std::to_string(stage) + " of " + std::to_string(wt_.depths.size()));
    if (block < 0 || block >= wt_.depths[stage])
        throw Error("hab: block " + std::to_string(block) + " of " + std::to_string(wt_.depths[stage]) +
                    " in stage " + std::to_string(stage));
    if (hp <= 0 || wp <= 0 || hp % wt_.window || wp % wt_.window)
        throw Error("hab: the plane must be a non-empty window multiple");
    ensure_plan(hp, wp);
    Runtime& rt = Runtime::get();
    const HipApi& api = rt.api();
    const long T = plan_.tokens();
    const size_t bytes = (size_t)T * wt_.embed * sizeof(float);
    const std::string p = "layers." + std::to_string(stage) + ".residual_group.blocks." + std::to_string(block);
    rt.h2d(a_.xa, x, bytes);
    // norm1 into a_.xn, then the block from a_.xa into a_.xb. The block also writes
    // the next norm's output into a_.xn; its own norm1 stands in for it.
    auto run = [&]() {
        layernorm(a_.xa, a_.xn, p + ".norm1", T);
        hab(stage, block, a_.xa, a_.xb, p + ".norm1");
    };
    run();
    rt.check(api.StreamSynchronize(stream_), "hab");
    rt.d2h(out, a_.xb, bytes);
    if (iters > 0 && ms) {
        hipEvent_t a = nullptr, b = nullptr;
        rt.check(api.EventCreate(&a), "hipEventCreate");
        rt.check(api.EventCreate(&b), "hipEventCreate");
        api.EventRecord(a, stream_);
        for (int i = 0; i < iters; ++i) run();
        api.EventRecord(b, stream_);
        rt.check(api.EventSynchronize(b), "hab timing");
        float e = 0.f;
        api.EventElapsedTime(&e, a, b);
        *ms = e / iters;
        api.EventDestroy(a);
        api.EventDestroy(b);
    }
}

void GpuBackend::free_batch()
{
    Runtime& rt = Runtime::get();
    for (BatchSlot& sl : batch_) {
        if (sl.s) {
            rt.api().StreamSynchronize(sl.s);
            rt.api().StreamDestroy(sl.s);
        }
        if (sl.hin) rt.api().HostFree(sl.hin);
        if (sl.hout) rt.api().HostFree(sl.hout);
    }
    batch_.clear();
    for (void* p : batch_dev_) rt.free(p);
    batch_dev_.clear();
}

void GpuBackend::forward_batch(int n, int h, int w, const float* in, float* out)
{
    if (n <= 0 || h <= 0 || w <= 0) throw Error("forward_batch: empty batch or image");
    if (!in || !out) throw Error("forward_batch: null argument");
    Runtime& rt = Runtime::get();
    const HipApi& api = rt.api();
    const size_t s2 = (size_t)wt_.scale * wt_.scale;
    const size_t isz = 3 * (size_t)h * w, osz = isz * s2;
    const int slots = std::min(n, kBatchSlots);
    const Plan p = Plan::make(h, w, wt_.window, wt_.embed);
    if (!(batch_plan_ == p) || (int)batch_.size() < slots) {
        free_batch();
        // admission for all the slots' buffers at once (the weights are already up)
        const MemPlan mp = gpu_plan(wt_, (size_t)h, (size_t)w);
        const uint64_t need = (uint64_t)((double)mp.activations * kSlack) * slots + mp.base;
        if (mp.have_avail && need > mp.avail)
            throw Error("not enough video memory for a batch of " + std::to_string(slots) + " concurrent " +
                        std::to_string(w) + "x" + std::to_string(h) + " passes: about " + fmt_bytes(need) +
                        " needed, " + fmt_bytes(mp.avail) + " free");
        batch_plan_ = p;
        batch_.resize(slots);
        for (BatchSlot& sl : batch_) {
            rt.check(api.StreamCreate(&sl.s), "hipStreamCreate");
            for (auto& b : layout(wt_, p, sl.a, true)) {
                if (b.second == 0) continue;
                float* d = (float*)rt.alloc(b.second * sizeof(float));
                batch_dev_.push_back(d);
                *b.first = d;
            }
            rt.check(api.HostMalloc((void**)&sl.hin, isz * sizeof(float), 0), "hipHostMalloc");
            rt.check(api.HostMalloc((void**)&sl.hout, osz * sizeof(float), 0), "hipHostMalloc");
        }
    }
    // Swap a slot's stream and buffers in for run_forward, which only enqueues.
    const hipStream_t own_stream = stream_;
    const Acts own_acts = a_;
    const Plan own_plan = plan_;
    const int own_nblk = nblk_conv2_;
    auto restore = [&]() {
        stream_ = own_stream;
        a_ = own_acts;
        plan_ = own_plan;
        nblk_conv2_ = own_nblk;
    };
    auto drain = [&](BatchSlot& sl) {
        if (sl.img < 0) return;
        rt.check(api.StreamSynchronize(sl.s), "forward_batch");
        memcpy(out + (size_t)sl.img * osz, sl.hout, osz * sizeof(float));
        sl.img = -1;
    };
    try {
        for (int i = 0; i < n; ++i) {
            BatchSlot& sl = batch_[i % slots];
            drain(sl);
            memcpy(sl.hin, in + (size_t)i * isz, isz * sizeof(float));
            rt.check(api.MemcpyAsync(sl.a.din, sl.hin, isz * sizeof(float), hipMemcpyHostToDevice, sl.s),
                     "hipMemcpyAsync H2D");
            stream_ = sl.s;
            a_ = sl.a;
            plan_ = p;
            t1_stride_ = (wt_.compressed + 3) / 4 * 4;
            nblk_conv2_ = colsum_rows(wt_.embed, p.hp, p.wp, wt_.embed);
            run_forward(h, w, sl.a.din, sl.a.dout);
            restore();
            rt.check(api.MemcpyAsync(sl.hout, sl.a.dout, osz * sizeof(float), hipMemcpyDeviceToHost, sl.s),
                     "hipMemcpyAsync D2H");
            sl.img = i;
        }
        for (BatchSlot& sl : batch_) drain(sl);
    } catch (...) {
        restore();
        for (BatchSlot& sl : batch_) {
            api.StreamSynchronize(sl.s);
            sl.img = -1;
        }
        throw;
    }
}

void GpuBackend::free_stage()
{
    Runtime& rt = Runtime::get();
    if (copy_stream_) rt.api().StreamSynchronize(copy_stream_);
    if (stage_in_) rt.api().HostFree(stage_in_);
    if (stage_out_) rt.api().HostFree(stage_out_);
    stage_in_ = stage_out_ = nullptr;
    stage_in_n_ = stage_out_n_ = 0;
}

namespace {
// Host threads of Backend::forward: each copies its share of the input into
// pinned memory, and of every output band out of it.
constexpr unsigned kStageThreads = 8;
constexpr int kMaxBands = 10;
}  // namespace

// Backend::forward (backend.rs:29-36, gpu.rs:759-803): host [3][h][w] in, host
// [3][h*s][w*s] out. Eight host threads copy the input into a pinned buffer
// (each an eighth), which goes up in one DMA. The head's last convs run in
// bands of output rows (run_forward), each band downloaded into a pinned buffer
// on a second stream as soon as its event fires, while the GPU computes the
// next bands; the threads copy each band to `out` as its download completes.
// So the 50 MB download of a 512 x 512 x4 forward overlaps the last upsample
// conv, and only the last band's download and copy (1/16 of the output) follow
// the forward. (A pageable hipMemcpy would stage through the runtime's own
// bounce buffers one piece at a time, after the whole forward.)
void GpuBackend::forward(int h, int w, const float* in, float* out)
{
    if (h <= 0 || w <= 0) throw Error(std::to_string(h) + "x" + std::to_string(w) + " is empty");
    if (!in || !out) throw Error("forward: null argument");
    ensure_plan(h, w);
    Runtime& rt = Runtime::get();
    const HipApi& api = rt.api();
    const size_t oh = (size_t)h * wt_.scale, ow = (size_t)w * wt_.scale;
    const size_t in_bytes = 3 * (size_t)h * w * sizeof(float), plane_bytes = oh * ow * sizeof(float);
    if (stage_in_n_ != in_bytes || stage_out_n_ != 3 * plane_bytes) {
        free_stage();
        rt.check(api.HostMalloc((void**)&stage_in_, in_bytes, 0), "hipHostMalloc");
        stage_in_n_ = in_bytes;
        rt.check(api.HostMalloc((void**)&stage_out_, 3 * plane_bytes, 0), "hipHostMalloc");
        stage_out_n_ = 3 * plane_bytes;
    }
    if (!copy_stream_) rt.check(api.StreamCreate(&copy_stream_), "hipStreamCreate");
    while (band_ev_.size() < (size_t)kMaxBands) {
        hipEvent_t a = nullptr, b = nullptr;
        rt.check(api.EventCreateWithFlags(&a, hipEventDisableTiming), "hipEventCreate");
        band_ev_.push_back(a);
        rt.check(api.EventCreateWithFlags(&b, hipEventDisableTiming), "hipEventCreate");
        copy_ev_.push_back(b);
    }

    constexpr unsigned T = kStageThreads;
    std::vector<std::pair<int, int>> bands;  // output rows, in the order they are written
    std::atomic<unsigned> in_done{0};
    std::atomic<int> queued{0};  // 1: every band's download is queued; -1: queueing failed
    std::vector<hipError_t> err(T, hipSuccess);
    // thread t's share [a, b) of n bytes, in 64-byte units
    auto share = [](size_t n, unsigned t) {
        const size_t u = (n + 63) / 64;
        return std::make_pair(std::min(n, u * t / T * 64), std::min(n, u * (t + 1) / T * 64));
    };
    auto copy_in = [&](unsigned t) {
        const auto r = share(in_bytes, t);
        memcpy((char*)stage_in_ + r.first, (const char*)in + r.first, r.second - r.first);
        in_done.fetch_add(1, std::memory_order_release);
    };
    auto copy_out = [&](unsigned t) {
        int q;
        while ((q = queued.load(std::memory_order_acquire)) == 0) std::this_thread::yield();
        if (q < 0) return;
        for (size_t k = 0; k < bands.size(); ++k) {
            const hipError_t e = api.EventSynchronize(copy_ev_[k]);
            if (e != hipSuccess) {
                err[t] = e;
                return;
            }
            const size_t row = ow * sizeof(float), len = (size_t)(bands[k].second - bands[k].first) * row;
            const auto r = share(len, t);
            for (int c = 0; c < 3; ++c) {
                const size_t off = c * plane_bytes + (size_t)bands[k].first * row + r.first;
                memcpy((char*)out + off, (const char*)stage_out_ + off, r.second - r.first);
            }
        }
    };
    auto worker = [&](unsigned t) {
        copy_in(t);
        copy_out(t);
    };
    std::vector<std::thread> pool;
    try {
        // inside the try: if a thread cannot be started, the ones that were are
        // released (queued = -1) and joined below, not destroyed while joinable
        for (unsigned t = 1; t < T; ++t) pool.emplace_back(worker, t);
        copy_in(0);
        while (in_done.load(std::memory_order_acquire) < T) std::this_thread::yield();
        rt.check(api.MemcpyAsync(a_.din, stage_in_, in_bytes, hipMemcpyHostToDevice, stream_), "hipMemcpyAsync H2D");
        run_forward(h, w, a_.din, a_.dout, &bands);
        for (size_t k = 0; k < bands.size(); ++k) {
            rt.check(api.StreamWaitEvent(copy_stream_, band_ev_[k], 0), "hipStreamWaitEvent");
            // the band's rows of the three planes: one 2D copy (a copy per
            // plane measured 25-45 us apart on the copy engine)
            const size_t row = ow * sizeof(float), len = (size_t)(bands[k].second - bands[k].first) * row;
            const size_t off = (size_t)bands[k].first * row;
            if (len > 0)
                rt.check(api.Memcpy2DAsync((char*)stage_out_ + off, plane_bytes, (const char*)a_.dout + off,
                                           plane_bytes, len, 3, hipMemcpyDeviceToHost, copy_stream_),
                         "hipMemcpy2DAsync D2H");
            rt.check(api.EventRecord(copy_ev_[k], copy_stream_), "hipEventRecord");
        }
    } catch (...) {
        queued.store(-1, std::memory_order_release);
        for (std::thread& th : pool) th.join();
        api.StreamSynchronize(stream_);
        api.StreamSynchronize(copy_stream_);
        throw;
    }
    queued.store(1, std::memory_order_release);
    copy_out(0);
    for (std::thread& th : pool) th.join();
    rt.check(api.StreamSynchronize(stream_), "forward");
    rt.check(api.StreamSynchronize(copy_stream_), "forward: download");
    for (hipError_t e : err) rt.check(e, "forward: download");
}

// ---------------------------------------------------------------------------
// Isolated ops.

namespace {

// An op's device buffers: one allocation, and one upload for everything small.
// The ops run once per call on buffers of their own, so a hipMalloc and hipFree
// a buffer and a blocking copy a weight were much of a call's host time (SW-MSA
// at 128 x 128, 180 channels: 2.32 -> 2.11 ms a call, most of what is left the
// two copies of the plane; OCAB at 96 x 160, 144 channels: 3.24 -> 1.88, the
// weights that only the unfused kernels read no longer packed as well). add()
// before commit(), ptr() after it.
class OpArena {
public:
    // n floats, from src if set (kept by the caller until commit)
    size_t add(size_t n, const float* src = nullptr) { return add_bytes(n * sizeof(float), src); }
    // n floats or 16-bit values the arena keeps until commit
    size_t keep(std::vector<float> v)
    {
        kept_f_.push_back(std::move(v));
        return add(kept_f_.back().size(), kept_f_.back().data());
    }
    size_t keep(std::vector<unsigned short> v)
    {
        kept_u_.push_back(std::move(v));
        return add_bytes(kept_u_.back().size() * sizeof(unsigned short), kept_u_.back().data());
    }
    void commit()
    {
        Runtime& rt = Runtime::get();
        // the small uploads first, side by side, so that one copy takes them
        size_t off = 0;
        for (int pass = 0; pass < 2; ++pass)
            for (Req& r : reqs_)
                if ((pass == 0) == (r.src && r.bytes <= kSmall)) {
                    r.off = off;
                    off += (r.bytes + 255) / 256 * 256;
                    if (pass == 0) small_ = off;
                }
        base_ = (char*)rt.alloc(off);
        std::vector<char> stage(small_);
        for (const Req& r : reqs_)
            if (r.src && r.bytes <= kSmall) memcpy(&stage[r.off], r.src, r.bytes);
        if (small_) rt.h2d(base_, stage.data(), small_);
        for (const Req& r : reqs_)
            if (r.src && r.bytes > kSmall) rt.h2d(base_ + r.off, r.src, r.bytes);
        kept_f_.clear();
        kept_u_.clear();
    }
    float* ptr(size_t i) const { return (float*)(base_ + reqs_[i].off); }
    OpArena() = default;
    ~OpArena()
    {
        if (base_) Runtime::get().free(base_);
    }
    OpArena(const OpArena&) = delete;
    OpArena& operator=(const OpArena&) = delete;

private:
    static constexpr size_t kSmall = 4u << 20;
    struct Req {
        size_t bytes, off;
        const void* src;
    };
    size_t add_bytes(size_t bytes, const void* src)
    {
        reqs_.push_back(Req{bytes, 0, src});
        return reqs_.size() - 1;
    }
    std::vector<Req> reqs_;
    std::deque<std::vector<float>> kept_f_;
    std::deque<std::vector<unsigned short>> kept_u_;
    char* base_ = nullptr;
    size_t small_ = 0;
};

// A linear of the op entry points, packed as the backend packs it
// (upload_linear, which explains out and in): a qkv of 144 or 180 channels as
// hat_gemmx_qkv takes it, so that an op runs the forward's kernels, others as
// FP32 rows; with kBias only the bias (a split tail holds the weights).
struct OpLinear {
    enum Form { kNone, kQkv, kBias };
    DevLinear L;
    size_t iw = 0, ib = 0, ix = 0;
    bool fp32 = false, split = false;
    OpLinear(OpArena& ar, const float* wt, const float* bias, int N, int K, Form form = kNone, const float* out = nullptr,
             float in = 1.0f)
    {
        L.N = N;
        L.K = K;
        L.Kp = (K + 15) / 16 * 16;
        std::vector<float> bs(bias, bias + N);
        if (out)
            for (int n = 0; n < N; ++n) bs[n] *= out[n / (N / 3)];
        ib = ar.keep(std::move(bs));
        if (form == kQkv && ((N == 432 && K == 144) || (N == 540 && K == 180))) {
            split = true;
            ix = ar.keep(split_qkv(wt, N, K, out, in, L.oscale));
        } else if (form != kBias) {
            fp32 = true;
            std::vector<float> ws(wt, wt + (size_t)N * K);
            for (int n = 0; n < N; ++n) {
                const float f = (out ? out[n / (N / 3)] : 1.0f) * in;
                for (int k = 0; k < K; ++k) ws[(size_t)n * K + k] *= f;
            }
            iw = ar.keep(pack_linear(ws.data(), N, K, &L.Kp));
        }
    }
    void bind(const OpArena& ar)
    {
        if (fp32) L.w = ar.ptr(iw);
        L.b = ar.ptr(ib);
        if (split) L.wx = (unsigned short*)ar.ptr(ix);
    }
};

// An op's projection and MLP for the split tail, as upload_tail packs them.
struct OpTail {
    DevTail t;
    size_t iw, iwm, ib1;
    OpTail(OpArena& ar, TailPack p) : t(p.t)
    {
        iw = ar.keep(std::move(p.w));
        iwm = ar.keep(std::move(p.wm));
        ib1 = ar.keep(std::move(p.b1x));
    }
    void bind(const OpArena& ar)
    {
        t.w = (unsigned short*)ar.ptr(iw);
        t.wm = (unsigned short*)ar.ptr(iwm);
        t.b1x = ar.ptr(ib1);
    }
};

// The largest |row . x + bias| for rows [n0, n1) over every x with |x_k| <= mx.
double op_linear_bound(const float* w, const float* b, int n0, int n1, int K, double mx)
{
    double worst = 0.0;
    for (int n = n0; n < n1; ++n) {
        double l1[4] = {};
        for (int k = 0; k < K; k += 4)
            for (int i = 0; i < 4 && k + i < K; ++i) l1[i] += std::fabs((double)w[(size_t)n * K + k + i]);
        const double v = (l1[0] + l1[1] + l1[2] + l1[3]) * mx + std::fabs((double)b[n]);
        if (std::isnan(v)) return v;
        worst = std::max(worst, v);
    }
    return worst;
}

struct Timer {
    hipEvent_t a = nullptr, b = nullptr;
    Timer()
    {
        const HipApi& api = Runtime::get().api();
        api.EventCreate(&a);
        api.EventCreate(&b);
    }
    ~Timer()
    {
        const HipApi& api = Runtime::get().api();
        api.EventDestroy(a);
        api.EventDestroy(b);
    }
};

}  // namespace

void op_swmsa(const float* x, float* out, int hp, int wp, int c, int heads, int shift,
              const float* qkv_w, const float* qkv_b, const float* proj_w, const float* proj_b,
              const float* table, int iters, float* ms, float* attn_ms)
{
    // Arguments are checked before the runtime is touched.
    if (!x || !out || !qkv_w || !qkv_b || !proj_w || !proj_b || !table) throw Error("swmsa: null argument");
    if (hp <= 0 || wp <= 0 || c <= 0 || heads <= 0) throw Error("swmsa: empty plane or no channels");
    if ((size_t)hp * wp > (1u << 26) || c > 4096) throw Error("swmsa: plane or channels too large");  // int token counts
    if (c % heads) throw Error("swmsa: c must be divisible by heads");
    const int D = c / heads;
    if (D != 24 && D != 30) throw Error("swmsa: head_dim " + std::to_string(D) + " has no kernel (24, 30)");
    Plan pl = Plan::make(hp, wp, 16, c);
    if (pl.hp != hp || pl.wp != wp) throw Error("swmsa: the plane must be a window multiple");
    if (shift != 0 && shift != pl.shift)
        throw Error("swmsa: shift " + std::to_string(shift) + " is not supported (0 or " +
                    std::to_string(pl.shift) + ")");
    Runtime& rt = Runtime::get();
    const HipApi& api = rt.api();
    const size_t T = (size_t)hp * wp;
    // the null stream: the op is synchronous, as are its copies, and a stream
    // of its own would be created and destroyed on each call
    hipStream_t s = nullptr;
    {
        // the planes first, and the input's largest finite |x|, which is what
        // bounds q, k and v here (no norm comes before them)
        OpArena ar;
        const std::vector<float> zero(AMAX_WORDS, 0.0f);
        const size_t ix = ar.add(T * c, x), iq = ar.add(3 * T * c), iao = ar.add(T * c), iout = ar.add(T * c),
                     imax = ar.add(AMAX_WORDS, zero.data());
        ar.commit();
        float *dx = ar.ptr(ix), *dq = ar.ptr(iq), *dao = ar.ptr(iao), *dout = ar.ptr(iout);
        AbsMaxArgs am{dx, (unsigned*)ar.ptr(imax), (long)(T * c)};
        launch(s, "hat_absmax", (unsigned)std::min<size_t>((T * c + 4095) / 4096, 512), 1, 1, 256, am);
        float lanes[AMAX_WORDS], mx = 0.0f;
        rt.d2h(lanes, ar.ptr(imax), sizeof lanes);
        for (float v : lanes) mx = std::max(mx, v);
        const QkvScale sc = qkv_scale(op_linear_bound(qkv_w, qkv_b, 0, c, c, mx),
                                      op_linear_bound(qkv_w, qkv_b, c, 2 * c, c, mx),
                                      op_linear_bound(qkv_w, qkv_b, 2 * c, 3 * c, c, mx), D);
        const float osc[3] = {sc.q, sc.k, sc.v};
        // x itself goes through the split: the largest value to the top of f16's
        // range, wherever it lies, since it says nothing about the others (one 5
        // among values of 1e-3 left unscaled: the other windows off by 1.8e-5 of their
        // size, scaled by 8e-7)
        float sx = 1.0f;
        if (c == 144 || c == 180) {
            sx = f16_scale(mx);
            ScaleArgs sa{dx, sx, (long)(T * c)};
            if (sx != 1.0f) launch(s, "hat_scale", (unsigned)std::min<size_t>((T * c + 4095) / 4096, 512), 1, 1, 256, sa);
        }
        // qkv as in the forward; the projection here has no residual, a form the
        // forward never runs, so it stays on the FP32 store epilogue
        OpArena wr;
        const size_t itab = wr.add(961 * (size_t)heads, table);
        OpLinear qkv(wr, qkv_w, qkv_b, 3 * c, c, OpLinear::kQkv, osc, 1.0f / sx),
            proj(wr, proj_w, proj_b, c, c, OpLinear::kNone, nullptr, 1.0f / sc.v);
        wr.commit();
        qkv.bind(wr);
        proj.bind(wr);
        const float* dtab = wr.ptr(itab);
        const GemmEpilogue none;
        auto run = [&]() {
            run_gemm(s, qkv.L, dx, c, (long)T, dq, 0, EPI_QKV, none, heads, D, 0.f);
            run_attn(s, dq, dtab, dao, pl, heads, D, false, shift, sc.ok);
            run_gemm(s, proj.L, dao, c, (long)T, dout, c, EPI_STORE, none, heads, D, 0.f);
        };
        run();
        rt.check(api.StreamSynchronize(s), "swmsa");
        if (iters > 0 && (ms || attn_ms)) {
            Timer t, ta;
            api.EventRecord(t.a, s);
            for (int i = 0; i < iters; ++i) run();
            api.EventRecord(t.b, s);
            api.EventRecord(ta.a, s);
            for (int i = 0; i < iters; ++i) run_attn(s, dq, dtab, dao, pl, heads, D, false, shift, sc.ok);
            api.EventRecord(ta.b, s);
            rt.check(api.EventSynchronize(ta.b), "swmsa timing");
            float e = 0.f;
            api.EventElapsedTime(&e, t.a, t.b);
            if (ms) *ms = e / iters;
            api.EventElapsedTime(&e, ta.a, ta.b);
            if (attn_ms) *attn_ms = e / iters;
        }
        rt.d2h(out, dout, T * c * sizeof(float));
    }
}

void op_ocab(const float* x, float* out, int hp, int wp, int c, int heads, int mlp_ratio,
             const float* n1w, const float* n1b, const float* qkv_w, const float* qkv_b,
             const float* proj_w, const float* proj_b, const float* table, const float* n2w,
             const float* n2b, const float* fc1_w, const float* fc1_b, const float* fc2_w,
             const float* fc2_b, int iters, float* ms, float* attn_ms)
{
    if (!x || !out || !n1w || !n1b || !qkv_w || !qkv_b || !proj_w || !proj_b || !table || !n2w || !n2b ||
        !fc1_w || !fc1_b || !fc2_w || !fc2_b)
        throw Error("ocab: null argument");
    if (hp <= 0 || wp <= 0 || c <= 0 || heads <= 0 || mlp_ratio <= 0) throw Error("ocab: empty plane or no channels");
    if ((size_t)hp * wp > (1u << 26) || c > 4096) throw Error("ocab: plane or channels too large");  // int token counts
    if (c % heads) throw Error("ocab: c must be divisible by heads");
    const int D = c / heads;
    if (D != 24 && D != 30) throw Error("ocab: head_dim " + std::to_string(D) + " has no kernel (24, 30)");
    Plan pl = Plan::make(hp, wp, 16, c);
    if (pl.hp != hp || pl.wp != wp) throw Error("ocab: the plane must be a window multiple");
    Runtime& rt = Runtime::get();
    const HipApi& api = rt.api();
    const size_t T = (size_t)hp * wp, hid = (size_t)c * mlp_ratio;
    hipStream_t s = nullptr;  // the null stream, as in op_swmsa
    {
        // the split tail's shapes; the norms into f16's range where split-f16
        // kernels read them, as GpuBackend::upload_norm
        const bool wide = c == 144 || c == 180, fits = wide && hid == 2 * (size_t)c;
        const float s1 = wide ? f16_scale(ln_bound(n1w, n1b, c)) : 1.0f,
                    s2 = fits ? f16_scale(ln_bound(n2w, n2b, c)) : 1.0f;
        std::vector<float> n1(2 * (size_t)c), n2(2 * (size_t)c);
        for (int i = 0; i < c; ++i) {
            n1[i] = n1w[i] * s1, n1[c + i] = n1b[i] * s1;
            n2[i] = n2w[i] * s2, n2[c + i] = n2b[i] * s2;
        }
        OpArena ar;
        const size_t ix = ar.add(T * c, x), iwork = ar.add(T * c), ixn = ar.add(T * c), iq = ar.add(3 * T * c),
                     iao = ar.add(T * c), itab = ar.add(1521 * (size_t)heads, table), i1w = ar.add(c, n1.data()),
                     i1b = ar.add(c, n1.data() + c), i2w = ar.add(c, n2.data()), i2b = ar.add(c, n2.data() + c);
        const QkvScale sc = qkv_scale(ln_linear_bound(qkv_w, qkv_b, n1w, n1b, 0, c, c),
                                      ln_linear_bound(qkv_w, qkv_b, n1w, n1b, c, 2 * c, c),
                                      ln_linear_bound(qkv_w, qkv_b, n1w, n1b, 2 * c, 3 * c, c), D);
        const float osc[3] = {sc.q, sc.k, sc.v};
        std::unique_ptr<OpTail> tail;
        if (fits) tail.reset(new OpTail(ar, pack_tail(proj_w, fc1_w, fc1_b, fc2_w, n2w, n2b, c, sc.v, s2, nullptr)));
        const OpLinear::Form form = fits ? OpLinear::kBias : OpLinear::kNone;
        OpLinear qkv(ar, qkv_w, qkv_b, 3 * c, c, OpLinear::kQkv, osc, 1.0f / s1),
            proj(ar, proj_w, proj_b, c, c, form, nullptr, 1.0f / sc.v), fc1(ar, fc1_w, fc1_b, (int)hid, c, form),
            fc2(ar, fc2_w, fc2_b, c, (int)hid, form);
        const size_t ih = ar.add(fits ? 1 : T * hid);
        ar.commit();
        if (tail) tail->bind(ar);
        for (OpLinear* l : {&qkv, &proj, &fc1, &fc2}) l->bind(ar);
        float *dx = ar.ptr(ix), *dwork = ar.ptr(iwork), *dxn = ar.ptr(ixn), *dq = ar.ptr(iq), *dao = ar.ptr(iao),
              *dtab = ar.ptr(itab), *d1w = ar.ptr(i1w), *d1b = ar.ptr(i1b), *d2w = ar.ptr(i2w), *d2b = ar.ptr(i2b);
        const GemmEpilogue none;
        GemmEpilogue resid_ln;
        resid_ln.res = dx;
        resid_ln.xn = dxn;
        resid_ln.nw = d2w;
        resid_ln.nb = d2b;
        // The backend's OCAB sequence (GpuBackend::ocab): norm1, qkv, attention,
        // proj + shortcut (which also writes norm2), then the MLP + residual.
        auto run = [&]() {
            run_ln(s, dx, dxn, d1w, d1b, (long)T, c);
            run_gemm(s, qkv.L, dxn, c, (long)T, dq, 0, EPI_QKV, none, heads, D, 0.f);
            run_attn(s, dq, dtab, dao, pl, heads, D, true, 0, sc.ok);
            if (tail) {
                run_tailx(s, tail->t, dao, dx, dwork, nullptr, proj.L.b, fc2.L.b, d2w, d2b, nullptr, nullptr, (long)T,
                          TailCabIn{});
            } else {
                run_gemm(s, proj.L, dao, c, (long)T, dwork, c, EPI_RESID_LN, resid_ln, heads, D, 0.f);
                run_mlp(s, fc1.L, fc2.L, dxn, (long)T, dwork, dwork, EPI_RESID, none, ar.ptr(ih));
            }
        };
        run();
        rt.check(api.StreamSynchronize(s), "ocab");
        rt.d2h(out, dwork, T * c * sizeof(float));
        if (iters > 0 && (ms || attn_ms)) {
            Timer t, ta;
            api.EventRecord(t.a, s);
            for (int i = 0; i < iters; ++i) run();
            api.EventRecord(t.b, s);
            api.EventRecord(ta.a, s);
            for (int i = 0; i < iters; ++i) run_attn(s, dq, dtab, dao, pl, heads, D, true, 0, sc.ok);
            api.EventRecord(ta.b, s);
            rt.check(api.EventSynchronize(ta.b), "ocab timing");
            float e = 0.f;
            api.EventElapsedTime(&e, t.a, t.b);
            if (ms) *ms = e / iters;
            api.EventElapsedTime(&e, ta.a, ta.b);
            if (attn_ms) *attn_ms = e / iters;
        }
    }
}

}  // namespace hat
