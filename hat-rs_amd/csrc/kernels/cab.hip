// The channel-attention block (CAB) of the compress-to-6 family (HAT-S):
//   CAB(x) = gate * conv2(gelu(conv1(x))),  gate = sigmoid(Wb relu(Wa mean_p conv2(..) + ba) + bb)
// (hat_arch.py CAB / ChannelAttention; cpu.rs cab, 1090-1120; the reference's
// GPU path runs it as lg_conv3x3 x2, a column mean and the squeeze-excite,
// src/cuda.rs:171-183, 201-214).
//
// conv2 is linear, so two of its three uses need no conv2 output at all:
//   * its pixel mean is b2 + (1/HW) sum_{tap,ci} w2[c][ci][tap] * S[tap][ci],
//     S[tap][ci] = sum of t1[.][ci] over the plane shifted by the tap (zero
//     padding): the whole-plane sum minus the row / column the shift pushes out,
//     plus the corner counted twice. hat_cab_conv1 leaves per-tile sums of t1
//     over the tile and over its pixels on the four border lines;
//   * gate[c] * conv2(t1)[p][c] * cscale is a GEMM of the 3x3 neighbourhood of
//     t1 at p (9 taps x 6 channels, k = tap*6 + ci) with weights cscale *
//     gate[c] * w2 - the gate folds them, and the block's tail (tailx.hip) runs
//     them as two more k-steps of the attention's projection.
// So conv2's T x 144 output is never written or read back.
#include "common.h"

using namespace hatk;

// ---------------------------------------------------------------------------
// conv1 (144 -> 6, 3x3, zero padding) + GELU on split-f16 MFMA, one 16 x 16
// output tile at a time: persistent over the tiles, two blocks of four waves
// per CU (on small planes in the qkv linear's launch, blocks of eight: gemmx.hip).
//
// Per-tap products: for each pixel q of the tile's 18 x 18 halo, P[q][tap*6+co]
// = sum_ci xn[q][ci] * w[co][ci][tap] is a 144-deep product with 54 outputs
// (padded to 64): v_mfma_f32_32x32x16_f16 with the 64 weight rows as A (two
// tiles of 32) and 32 halo pixels as B, nine 16-channel steps, every fp32
// operand as two f16 parts and every product as three terms (common.h; norm1
// leaves xn in f16's range, the host scales the weights, p.oinv takes both
// out). The conv output at p is then the sum over the 9 taps of P[p +
// d(tap)][tap*6 + co], read from LDS in fp32.
//
// The split weights (144 registers a lane) stay in registers for the whole
// kernel, and the rows are read CX_RING steps ahead, across halo tiles and
// output tiles: the barriers here wait for LDS only, so those loads stay in
// flight through them. That leaves two waves a SIMD (256 registers), so that
// one block's taps, GELU and stores run beside the other's MFMAs; the bf16
// split's 216 weight registers left one, in 16 x 32 tiles. HAT-S 512 x 512: 53.3
// -> 50.5 us (151 MB: 27 us at the copy kernel's rate; issue and the rows'
// latency bound it), 64 x 64, whose 16 tiles are as many blocks: 22.8 -> 12.0.
#define CX_WAVES 4
#define CX_HS 18                               // halo width and height
#define CX_HP (CX_HS * CX_HS)                  // halo pixels
#define CX_PT ((CX_HP + 31) / 32)              // 32-pixel halo tiles
#define CX_PS 60    // LDS row stride of P (56 written, 54 used): a b128 phase's 16 rows on distinct banks
#define CX_RING 3   // 16-channel steps of rows in flight

// block: of nblk; WAVES: 4 or 8, of which the first four take the taps (one pixel
// per thread). Ps: CX_HP * CX_PS floats, red: 4 * CAB_NSUM * CAB_CC.
template <int WAVES>
__device__ __forceinline__ void cab_conv1_body(const CabConvArgs& p, float* Ps, float* red, int block, int nblk)
{
    constexpr int NPW = (CX_PT + WAVES - 1) / WAVES;  // halo tiles a wave (past CX_PT: zeros, not stored)
    static_assert(WAVES % 4 == 0, "a pixel a thread of the first four waves");

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform, in a scalar register
    const int pl = lane & 31, h = lane >> 5;
    const int H = p.H, W = p.W;
    const int ntx = W / 16;
    const int ntiles = ntx * (H / 16);

    // The split weights go through LDS (the P region, free until the first
    // halo tile's stores) once per block, then into every wave's registers.
    constexpr int NWU = CX_WPACK / 8, WIT = (NWU + WAVES * 64 - 1) / (WAVES * 64);  // 16-byte units
    static_assert(NWU * 16 <= CX_HP * CX_PS * 4, "the weights fit the P region");
    u32x4 stage[WIT];
#pragma unroll
    for (int i = 0; i < WIT; ++i) {
        const int u = tid + i * WAVES * 64;
        stage[i] = ((const u32x4*)p.w)[NWU % (WAVES * 64) == 0 || u < NWU ? u : NWU - 1];
    }
    float bias[CAB_CC];
#pragma unroll
    for (int co = 0; co < CAB_CC; ++co) bias[co] = p.bias[co] * p.ts;

    // The lane's input row (channels 8h.. of each 16-channel step) for halo
    // tile i of output tile tl; hat_zero_row outside the plane, past the halo
    // and past the last tile, so that the loads are issued on every path.
    auto src_of = [&](int tl, int i) -> const float* {
        const int ty = tl / ntx, tx = tl - ty * ntx;
        const int hi = (wave + WAVES * i) * 32 + pl;
        const int hy = hi / CX_HS, hx = hi - hy * CX_HS;
        const int gy = ty * 16 - 1 + hy, gx = tx * 16 - 1 + hx;
        const bool valid = tl < ntiles && hi < CX_HP && gy >= 0 && gy < H && gx >= 0 && gx < W;
        return valid ? p.xn + (size_t)(gy * W + gx) * CAB_C + 8 * h : hat_zero_row;
    };
    // row steps in flight: step t of an output tile (halo tile t / 9, channels
    // 16 (t % 9) ..) in slot t % CX_RING
    f32x4 xr[CX_RING][2];
    const float* cur = src_of(block, 0);
#pragma unroll
    for (int t = 0; t < CX_RING; ++t) {
        xr[t][0] = *(const f32x4*)(cur + t * 16);
        xr[t][1] = *(const f32x4*)(cur + t * 16 + 4);
    }
#pragma unroll
    for (int i = 0; i < WIT; ++i) {
        const int u = tid + i * WAVES * 64;
        if (NWU % (WAVES * 64) == 0 || u < NWU) ((u32x4*)Ps)[u] = stage[i];
    }
    lds_barrier();
    u32x4 wr[9][2][2];
#pragma unroll
    for (int ks = 0; ks < 9; ++ks)
#pragma unroll
        for (int nt = 0; nt < 2; ++nt)
#pragma unroll
            for (int part = 0; part < 2; ++part)
                wr[ks][nt][part] = ((const u32x4*)Ps)[((ks * 2 + nt) * 2 + part) * 64 + lane];
    lds_barrier();  // every wave has its weights before P is written

    for (int tile = block; tile < ntiles; tile += nblk) {
        const int ty = tile / ntx, tx = tile - ty * ntx;
        const int y0 = ty * 16, x0 = tx * 16;
        // unrolled: with no back-edge here, the compiler's waits for the rows
        // read ahead are exact
#pragma unroll
        for (int i = 0; i < NPW; ++i) {
            const float* nxt = i + 1 < NPW ? src_of(tile, i + 1) : src_of(tile + nblk, 0);
            f32x16 acc[2];
#pragma unroll
            for (int j = 0; j < 16; ++j) acc[0][j] = acc[1][j] = 0.0f;
#pragma unroll
            for (int ks = 0; ks < 9; ++ks) {
                const int slot = (9 * i + ks) % CX_RING, ahead = ks + CX_RING;
                const float f[8] = {xr[slot][0][0], xr[slot][0][1], xr[slot][0][2], xr[slot][0][3],
                                    xr[slot][1][0], xr[slot][1][1], xr[slot][1][2], xr[slot][1][3]};
                u32x4 xb[2];
                split2_x8(f, xb);
                const float* src = ahead < 9 ? cur + ahead * 16 : nxt + (ahead - 9) * 16;
                xr[slot][0] = *(const f32x4*)src;
                xr[slot][1] = *(const f32x4*)(src + 4);
#pragma unroll
                for (int nt = 0; nt < 2; ++nt) acc[nt] = mfma3(wr[ks][nt], xb, acc[nt]);
                __builtin_amdgcn_sched_barrier(0);  // the loads stay in their step
            }
            cur = nxt;
            // lane (pl, h) holds P[hi][32 nt + 8 g + 4 h .. +3] in acc[nt][4g .. 4g+3];
            // columns 56.. (nt = 1, g = 3) are not stored
            const int hi = (wave + WAVES * i) * 32 + pl;
            if (hi < CX_HP) {
#pragma unroll
                for (int nt = 0; nt < 2; ++nt)
#pragma unroll
                    for (int g = 0; g < (nt == 0 ? 4 : 3); ++g)
                        *(f32x4*)(Ps + hi * CX_PS + 32 * nt + 8 * g + 4 * h) =
                            (f32x4){acc[nt][4 * g], acc[nt][4 * g + 1], acc[nt][4 * g + 2], acc[nt][4 * g + 3]};
            }
        }
        // the next output tile's first steps into slots 0 .. CX_RING - 1
        {
            f32x4 nx[CX_RING][2];
#pragma unroll
            for (int t = 0; t < CX_RING; ++t)
#pragma unroll
                for (int j = 0; j < 2; ++j) nx[t][j] = xr[(9 * NPW + t) % CX_RING][j];
#pragma unroll
            for (int t = 0; t < CX_RING; ++t)
#pragma unroll
                for (int j = 0; j < 2; ++j) xr[t][j] = nx[t][j];
        }
        lds_barrier();  // P complete

        // The 9 taps from the halo products, one output pixel per thread.
        const bool border = y0 == 0 || y0 + 16 == H || x0 == 0 || x0 + 16 == W;  // tile-uniform
        if (WAVES == 4 || wave < 4) {
            const int ox = tid & 15, oy = tid >> 4;
            float v[CAB_CC];
#pragma unroll
            for (int co = 0; co < CAB_CC; ++co) v[co] = 0.0f;
#pragma unroll
            for (int ky = 0; ky < 3; ++ky)
#pragma unroll
                for (int kx = 0; kx < 3; ++kx) {
                    const float* q = Ps + ((oy + ky) * CX_HS + ox + kx) * CX_PS + (ky * 3 + kx) * CAB_CC;
#pragma unroll
                    for (int j = 0; j < CAB_CC / 2; ++j) {
                        const float2 t = *(const float2*)(q + 2 * j);
                        v[2 * j] += t.x;
                        v[2 * j + 1] += t.y;
                    }
                }
#pragma unroll
            for (int co = 0; co < CAB_CC; ++co) v[co] = gelu_scaled(__builtin_fmaf(v[co], p.oinv, bias[co]), p.g0, p.g1);
            {
                float* dst = p.t1 + ((size_t)(y0 + oy) * W + x0 + ox) * CAB_CS;
                *(float4*)dst = make_float4(v[0], v[1], v[2], v[3]);
                *(float4*)(dst + 4) = make_float4(v[4], v[5], 0.f, 0.f);
            }

            // Per-tile sums: the tile, and its pixels on row 0, row H-1, col 0,
            // col W-1 - only tiles on the plane's border have any of the latter.
#pragma unroll
            for (int l = 0; l < CAB_NSUM; ++l) {
                if (l > 0 && !border) break;
#pragma unroll
                for (int co = 0; co < CAB_CC; ++co) {
                    const int gy = y0 + oy, gx = x0 + ox;
                    const bool on = l == 0 || (l == 1 && gy == 0) || (l == 2 && gy == H - 1) || (l == 3 && gx == 0) ||
                                    (l == 4 && gx == W - 1);
                    const float s = wave_sum_dpp(on ? v[co] : 0.0f);
                    if (lane == 0) red[wave * CAB_NSUM * CAB_CC + l * CAB_CC + co] = s;
                }
            }
        }
        lds_barrier();
        if (tid < CAB_NSUM * CAB_CS) {
            const int l = tid / CAB_CS, co = tid - l * CAB_CS;
            float s = 0.0f;
            if (co < CAB_CC && (l == 0 || border)) {
                const int k = l * CAB_CC + co;
#pragma unroll
                for (int w = 0; w < 4; ++w) s += red[w * CAB_NSUM * CAB_CC + k];  // waves in order
            }
            p.partial[(size_t)tid * ntiles + tile] = s;  // value-major: [40][tiles]
        }
        // The next tile's P stores come after this barrier; every read of Ps
        // and red above precedes it.
        lds_barrier();
    }
}

extern "C" __global__ __launch_bounds__(CX_WAVES * 64, 2) void hat_cab_conv1(CabConvArgs p)
{
    __shared__ __attribute__((aligned(16))) float Ps[CX_HP * CX_PS];
    __shared__ float red[4 * CAB_NSUM * CAB_CC];
    cab_conv1_body<CX_WAVES>(p, Ps, red, (int)blockIdx.x, (int)gridDim.x);
}

// ---------------------------------------------------------------------------
// The gate, and conv2 folded with it, for a block of WAVES waves; lds: CAB_GATE_LDS
// floats. Every reduction is a fixed-order per-lane sum followed by a fixed shuffle
// tree, so the result does not depend on timing. It rides on the attention launch as
// a block of its own (attnx.hip), so what counts is its latency, which small planes
// would wait for: conv2's weights are read once, coalesced, under the tile sums'
// loads, and the split chunks go out eight values at a time.
#define CAB_GATE_W2 (CAB_C * CAB_CC * 9)
#define CAB_GATE_LDS (CAB_GATE_W2 + CAB_NSUM * CAB_CS + 9 * CAB_CC + CAB_C + 64 + CAB_C)
template <int WAVES>
__device__ __forceinline__ void cab_gate_body(const CabGateArgs& p, float* lds)
{
    constexpr int NV = CAB_NSUM * CAB_CS;  // 40 sums per tile
    float* s_w2 = lds;
    float* s_sum = s_w2 + CAB_GATE_W2;
    float* s_S = s_sum + NV;
    float* s_mean = s_S + 9 * CAB_CC;
    float* s_z = s_mean + CAB_C;
    float* s_gate = s_z + 64;
    const int tid = threadIdx.x;
    const int wave = tid >> 6, lane = tid & 63;

    static_assert(CAB_GATE_W2 % 4 == 0, "float4 units");
    for (int i = tid; i < CAB_GATE_W2 / 4; i += WAVES * 64) ((f32x4*)s_w2)[i] = ((const f32x4*)p.w2)[i];
    // Tile sums: partial is value-major, so a wave reads 64 tiles per load.
    for (int v = wave; v < NV; v += WAVES) {
        const float* src = p.partial + (size_t)v * p.tiles;
        float acc = 0.0f;
#pragma unroll 8
        for (int t = lane; t < p.tiles; t += 64) acc += src[t];
        acc = wave_sum(acc);
        if (lane == 0) s_sum[v] = acc;
    }
    __syncthreads();
    const int H = p.H, W = p.W;
    if (tid < 9 * CAB_CC) {
        const int tap = tid / CAB_CC, ci = tid - tap * CAB_CC;
        const int dy = tap / 3 - 1, dx = tap % 3 - 1;
        float s = s_sum[0 * CAB_CS + ci];
        if (dy == 1) s -= s_sum[1 * CAB_CS + ci];   // source rows 1 .. H-1: row 0 is out
        if (dy == -1) s -= s_sum[2 * CAB_CS + ci];  // rows 0 .. H-2: row H-1 is out
        if (dx == 1) s -= s_sum[3 * CAB_CS + ci];
        if (dx == -1) s -= s_sum[4 * CAB_CS + ci];
        if (dy != 0 && dx != 0)  // the corner both lines removed
            s += p.t1[((size_t)(dy == 1 ? 0 : H - 1) * W + (dx == 1 ? 0 : W - 1)) * CAB_CS + ci];
        s_S[tid] = s;
    }
    __syncthreads();
    const float inv = 1.0f / ((float)H * (float)W * p.ts);
    for (int c = tid; c < CAB_C; c += WAVES * 64) {
        float acc = 0.0f;
#pragma unroll
        for (int ci = 0; ci < CAB_CC; ++ci)
#pragma unroll
            for (int tap = 0; tap < 9; ++tap) acc += s_w2[(c * CAB_CC + ci) * 9 + tap] * s_S[tap * CAB_CC + ci];
        s_mean[c] = p.b2[c] + acc * inv;
    }
    __syncthreads();
    for (int j = wave; j < p.sq; j += WAVES) {
        float acc = 0.0f;
        for (int c = lane; c < CAB_C; c += 64) acc += s_mean[c] * p.wa[j * CAB_C + c];
        acc = wave_sum(acc) + p.ba[j];
        if (lane == 0) s_z[j] = acc < 0.0f ? 0.0f : acc;
    }
    __syncthreads();
    for (int c = tid; c < CAB_C; c += WAVES * 64) {
        float acc = p.bb[c];
        for (int j = 0; j < p.sq; ++j) acc += s_z[j] * p.wb[c * p.sq + j];
        const float g = 1.0f / (1.0f + __expf(-acc));
        s_gate[c] = g;
        p.gate[c] = g;
        p.bias2[c] = p.bproj[c] + (p.cscale * g) * p.b2[c];
    }
    __syncthreads();
    // cscale * gate[c] * conv2 weight as the split tail's two weight steps:
    // [s][plane][c][32], row c's k-group g at slot ws_slot(c, g), k = tap*6 + ci =
    // 32 s + j, zeros from k = 54; one k-group (8 values, 16 bytes a plane) at a time
    {
        constexpr int PLANE = CAB_C * 32;
        for (int u = tid; u < 2 * CAB_C * 4; u += WAVES * 64) {
            const int s = u / (CAB_C * 4), c = (u >> 2) - s * CAB_C, g = u & 3;
            const float sc = p.cscale * s_gate[c] * p.gs;
            float f[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int k = 32 * s + 8 * g + j, tap = k / CAB_CC, ci = k - tap * CAB_CC;
                f[j] = tap < 9 ? sc * s_w2[(c * CAB_CC + ci) * 9 + tap] : 0.0f;
            }
            u32x4 parts[2];
            split2_x8(f, parts);
#pragma unroll
            for (int pl = 0; pl < 2; ++pl)
                *(u32x4*)(p.w2gx + (size_t)(2 * s + pl) * PLANE + c * 32 + ws_slot(c, g) * 8) = parts[pl];
        }
    }
}

// The unfolded CAB's gate (the C = 180 family; hat_arch.py:40-55, cpu.rs:
// 940-955) for a block of WAVES waves, straight from the conv2 partial column
// sums: thread (r, q) adds rows r, r + R, ... of the four columns of quad q,
// eight loads in flight (one row a wave and two loads in flight took 330 us for
// the 2048 rows of a 512 x 512 plane, longer than the attention launch it rides
// on), the R sums of a column are added in order through LDS, then mean,
// squeeze + ReLU, excite + sigmoid. C <= 192, a multiple of 4. lds: SE_GATE_LDS
// floats.
#define SE_GATE_ROWS 16
#define SE_GATE_LDS (SE_GATE_ROWS * 192 + 192 + 64)
template <int WAVES>
__device__ __forceinline__ void se_gate_body(const SeArgs& p, float* lds)
{
    float* s_part = lds;                          // [R][192]
    float* s_mean = s_part + SE_GATE_ROWS * 192;  // [192]
    float* s_sq = s_mean + 192;                   // [64]
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int nq = p.C / 4, R = min(WAVES * 64 / nq, SE_GATE_ROWS);
    const int r = tid / nq, q = tid - r * nq;
    if (r < R) {
        f32x4 a = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
        for (int b = r; b < p.nblk; b += R) a += *(const f32x4*)(p.partial + (size_t)b * p.co_stride + 4 * q);
        *(f32x4*)(s_part + r * 192 + 4 * q) = a;
    }
    __syncthreads();
    for (int c = tid; c < p.C; c += WAVES * 64) {
        float acc = 0.0f;
        for (int w = 0; w < R; ++w) acc += s_part[w * 192 + c];
        s_mean[c] = acc / p.count;
    }
    __syncthreads();
    for (int j = wave; j < p.sq; j += WAVES) {
        float acc = 0.0f;
        for (int c = lane; c < p.C; c += 64) acc += s_mean[c] * p.w1[(size_t)j * p.C + c];
        acc = wave_sum(acc) + p.b1[j];
        if (lane == 0) s_sq[j] = acc < 0.0f ? 0.0f : acc;
    }
    __syncthreads();
    for (int c = tid; c < p.C; c += WAVES * 64) {
        float acc = p.b2[c];
        for (int j = 0; j < p.sq; ++j) acc += s_sq[j] * p.w2[(size_t)c * p.sq + j];
        p.gate[c] = 1.0f / (1.0f + __expf(-acc));
    }
}
