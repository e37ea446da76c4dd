// Kernel argument blocks shared by the host runtime (g++) and the gfx950
// kernels (hipcc). Every kernel takes exactly one of these structs by value,
// so the host packs the kernarg segment by copying the struct: the layout is
// plain C (pointers 8 bytes, int/float 4 bytes) and identical on both sides.
#pragma once
#include <stdint.h>

namespace hatk {

// The fixed device array behind hat_backend_forward_noalloc (hat_scratch in
// misc.hip): 256 MiB, enough for the per-plan buffers of a HAT-S or HAT x4
// forward up to 128 x 128 input pixels. Every process that loads the library
// holds it on the device until it exits.
constexpr unsigned long long SCRATCH_BYTES = 256ull << 20;

// Activation layout everywhere on the device: token-major NHWC, [pixel][channel],
// pixels in image row-major order over the padded plane (hp x wp).

// out[m][n] = epilogue( A[m][:] . W[n][:] + bias[n] )
enum GemmEpi : int {
    EPI_STORE = 0,       // out[m][n] = v
    EPI_GELU = 1,        // out[m][n] = gelu(v)
    EPI_QKV = 2,         // head-major scatter: out[which][head][m][dim]
    EPI_RESID = 3,       // out[m][n] = res[m][n] + v
    EPI_HAB = 4,         // out[m][n] = (res[m][n] + v) + (aux[m][n] * gate[n]) * cscale
    EPI_RESID_LN = 5,    // EPI_RESID, and xn[m][:] = LayerNorm(out[m][:]) (full rows)
    EPI_HAB_LN = 6,      // EPI_HAB, and xn[m][:] = LayerNorm(out[m][:]) (full rows)
    EPI_STORE_LN = 7,    // EPI_STORE, and xn[m][:] = LayerNorm(out[m][:]) (full rows)
};

// Weight-stationary K = 144 GEMM launch geometry per epilogue: ws_waves waves
// per block, each owning ws_mt 16-row MFMA tiles of a ws_rows-row tile. One
// 16-row tile per wave keeps the plain epilogues at 4 waves per SIMD, so one
// wave's stores overlap the others' MFMAs; the LayerNorm epilogues need the
// registers of 2 waves per SIMD.
constexpr int ws_mt(int /*epi*/) { return 1; }
constexpr int ws_waves(int epi) { return epi == EPI_RESID_LN || epi == EPI_HAB_LN ? 8 : 16; }
constexpr int ws_rows(int epi) { return ws_waves(epi) * 16 * ws_mt(epi); }

// Waves per block of the wide-tile 3x3 conv instances (convw.hip): 8 own two
// 16-pixel tile rows each (2 waves per SIMD), 16 own one (4 per SIMD, where
// the registers allow it; measured faster for these three).
#define CONVW_WAVES_N9_STORE_LN 16
#define CONVW_WAVES_N9_RESID_LN 8
#define CONVW_WAVES_N9_RESID 8
#define CONVW_WAVES_N6_RESID 8
#define CONVW_WAVES_N6_COLSUM 8
#define CONVW_WAVES_N4_STORE 16
#define CONVW_WAVES_N8_SHUFFLE 16

struct GemmArgs {
    const float* a;      // [M][lda]
    const float* w;      // [N][Kp] row-major, K contiguous, zero-padded to Kp
    const float* bias;   // [N]
    float* out;
    const float* res;    // residual input (EPI_RESID*, EPI_HAB*)
    const float* aux;    // EPI_HAB*: conv branch [M][N]
    const float* gate;   // EPI_HAB*: channel gate [N]
    float* xn;           // EPI_*_LN: LayerNorm of the output rows [M][ldo]
    const float* nw;     // EPI_*_LN: LayerNorm weight [N]
    const float* nb;     // EPI_*_LN: LayerNorm bias [N]
    int M, N, K;         // logical sizes
    int Kp;              // K rounded up to 16 (W rows are Kp long)
    int lda, ldo;        // row strides of A and out (floats)
    int heads, hdim;     // EPI_QKV geometry (N = 3 * heads * hdim)
    float cscale;        // EPI_HAB* conv scale
    float eps;           // LayerNorm eps
    // hat_gemmx_qkv*: what takes the operands' scales out of q, k and v (the
    // bias is in the result's scale already)
    float oscale[3];
};

// CAB of the compress-to-6 family (HAT-S: 144 -> 6 -> 144), restated by the
// linearity of its second conv: conv2 becomes a K segment of the attention
// projection GEMM and its pixel mean comes from per-tile sums of conv1's output.
#define CAB_C 144
#define CAB_CC 6             // compressed channels
#define CAB_CS 8             // t1 channel stride (channels 6, 7 are zero)
// conv1's weights split for hat_cab_conv1: per 16-channel step ks (9), row
// tile nt (2 x 32 rows, row tap*6 + co, rows 54.. zero) and part (2), the
// 32x32x16 A operand of each lane (row l % 32, channels 16 ks + 8 (l / 32) .. +7)
#define CX_WPACK (9 * 2 * 2 * 64 * 8)
// floats of the gated conv2 weights' buffer: CabGateArgs::w2gx, then the forward's
// magnitude slots (AMAX_SLOTS); the rest is spare, which keeps a plan's size, and with
// it the tile that a memory budget picks, what they have been
#define CAB_W2GX 28544
#define CAB_W2GX_USED (2 * CAB_C * 32)
#define CAB_NSUM 5           // per-tile sums: whole tile, row 0, row H-1, col 0, col W-1

struct CabConvArgs {
    const float* xn;     // [H*W][144]
    const unsigned short* w;  // [9][2][2][64][8] f16: step ks, row tile nt, part, lane (CX_WPACK)
    const float* bias;   // [6]
    float* t1;           // [H*W][8]: ts * gelu(conv1(xn))
    float* partial;      // [CAB_NSUM * 8][tiles] (value-major), of t1 as stored
    int H, W;            // multiples of 16
    float ts;            // t1's scale (a power of two: the split tail's range)
    float oinv;          // ts over xn's scale and the weights'
    float g0, g1;        // gelu_scaled's constants for ts
};

struct CabGateArgs {
    const float* partial;  // [CAB_NSUM * 8][tiles] (value-major)
    const float* t1;       // corner pixels
    int tiles, H, W;
    const float* w2;     // conv2 weight [144][6][3][3]
    const float* b2;     // [144]
    const float* wa;     // channel attention squeeze [sq][144]
    const float* ba;     // [sq]
    const float* wb;     // excite [144][sq]
    const float* bb;     // [144]
    const float* bproj;  // attention projection bias [144]
    float* bias2;        // out: bproj + cscale * gate * b2, [144]
    float* gate;         // out: the gate itself [144]
    float cscale;
    int sq;
    unsigned short* w2gx;  // out: cscale * gate[c] * conv2 weight * gs as the split tail's two steps
                           // (k = tap*6 + ci), [2][144][32] each (ws_slot)
    float ts, gs;        // t1's scale; w2gx's scale (powers of two)
};

// Implicit-GEMM 3x3 convolution, stride 1, zero padding 1, NHWC.
enum ConvEpi : int {
    CEPI_STORE = 0,      // out[p][co] = v (+ act)
    CEPI_RESID = 1,      // out[p][co] = v + res[p][co]
    CEPI_SHUFFLE = 2,    // pixel shuffle by r into [H*r][W*r][co/(r*r)] (channels pre-permuted)
    CEPI_FINAL = 3,      // planar [3][ch][cw] with crop, / img_range + mean
    CEPI_COLSUM = 4,     // store + per-block column sums into partial[blk][co]
};

struct ConvArgs {
    const float* in;     // [H][W][cin_stride]
    const float* w;      // repacked: [CIp/16][9][COp][16] (chunk, tap, co, 16 ci)
    const float* bias;   // [COp]
    float* out;
    const float* res;    // CEPI_RESID
    float* partial;      // CEPI_COLSUM: [gridDim.x*gridDim.y][co_stride]
    int H, W;
    int CI, CIp, cin_stride;
    int CO, COp, co_stride;   // co_stride = channel stride of out (NHWC)
    int act;             // 0 none, 1 gelu, 2 leaky(0.01)
    int r;               // CEPI_SHUFFLE factor
    int crop_h, crop_w;  // CEPI_FINAL crop (output size)
    float img_range;     // CEPI_FINAL: out = v / img_range + mean
    float mean0, mean1, mean2;
    // hat_convw_* (all output channels per block, GEMM epilogues):
    float* xn;           // LayerNorm of the output rows [H*W][co_stride]
    const float* nw;
    const float* nb;
    float eps;
    // hat_convwino_*: Winograd F(2x2,3x3) weights U = G g G^T, scaled by 1 / uinv
    // and split into two f16 parts, arranged [kc][xi 16][nt][part 2][lane 64][8] (lane r + 16 g:
    // co 16 nt + r, ci 32 kc + 8 g .. +7; channels padded to 16s and 32s)
    const unsigned short* wu;
    // hat_convwino_* and hat_conv_last3 launched over a band of tile rows (the
    // host-memory forward's head): the band's first tile; 0 for a whole plane
    int tile0;
    // hat_convwino_*: the launch's virtual blocks (tiles x column blocks),
    // walked by a grid of at most one block per CU; 0: one per block
    int nblk;
    // hat_convwino_*: V's scale, a power of two, from the host (vs) or from the
    // input's largest magnitude (amax, its bits); where to leave the output's
    // (amax_out, null: nowhere); the scale of a GELU output (os)
    float uinv, vs, os;
    const unsigned* amax;
    unsigned* amax_out;
};

// Squeeze-excite gate: gate[c] = sigmoid(b2 + W2 relu(b1 + W1 mean)).
struct SeArgs {
    const float* partial; // [nblk][co_stride]
    int nblk, co_stride;
    float count;          // pixel count (mean = sum / count)
    const float* w1;      // [sq][C]
    const float* b1;      // [sq]
    const float* w2;      // [C][sq]
    const float* b2;      // [C]
    float* gate;          // [C]
    int C, sq;
};

// Fused window attention: one block per (window, head) (grid nw x heads), or,
// for OCA with head_dim 24, persistent blocks walking the (window, head) items
// head-major (grid: at most one block per CU, gridDim.y = 1).
constexpr bool attn_persistent(int D, bool oca) { return oca && D == 24; }
// The split-f16 kernels (attnx.hip) run one item per block, SW and OCA.
struct AttnArgs {
    const float* qkv;    // head-major [3][heads][T][D]
    const float* table;  // relative-position bias table [rows][heads]
    float* out;          // [T][C] token-major, image order
    int hp, wp, nx, ny;  // padded plane and window grid
    int heads, D, C;
    int shift;           // SW: cyclic shift (0 or win/2); mask applied iff shift > 0
    int owin, opad;      // OCA: unfold window and padding
    int T;
    float qscale;        // head_dim^-0.5 * log2(e)
    // with_gate: the launch also computes the folded CAB's gate (cab.hip), which the HAB tail after it needs: the split-f16 SW kernels in a
    // block of its own (the grid has one more column, the first), the FP32 ones
    // in block (0, 0) before its item
    int with_gate;
    CabGateArgs gate;
    // with_se: the same for the unfolded CAB's squeeze-excite gate (C = 180)
    int with_se;
    SeArgs se;
};

// Fused MLP (C = 144, hidden 288):
//   out[m][:] = res[m][:] + fc2(gelu(fc1(a[m][:]))),  xn = LayerNorm(out)
#define MLP_WAVES 8
#define MLP_ROWS (MLP_WAVES * 16)

struct MlpArgs {
    const float* a;      // [M][144]
    const float* w1;     // [288][ldw1]
    const float* b1;     // [288]
    const float* w2;     // [144][ldw2]
    const float* b2;     // [144]
    const float* res;    // [M][144] (may alias out)
    float* out;          // [M][144]
    float* xn;           // [M][144] (may alias a)
    const float* nw;
    const float* nb;
    int M;
    float eps;
    int ldw1, ldw2;      // packed weight row strides
};

// The HAB / OCAB tails on split-f16 MFMA (tailx.hip). Their weights are arrays
// of 32-k steps, each step two f16 planes [rows][32] with row r's four 16-byte
// k-groups g at slot ws_slot(r, g) (ws_mma2), copied to LDS as loads of 1 KB,
// the same number from every wave of a block; the arrays end in TX_PAD elements
// that those loads may read.
#define TX_PAD 4096
// The slot of row r's 16-byte k-group g in a 64-byte row of those planes. An
// MFMA fragment read has lane i take rows r0 + i at one k-group, 16 bytes a
// lane, and the LDS serves such reads 8 consecutive lanes at a time over its
// 32 four-byte banks; two 64-byte rows fill the banks once, so the XOR by
// (r >> 1) & 3 gives the four row pairs of every 8 lanes four distinct slots
// and the reads have no bank conflicts without padding (measured: none).
constexpr int ws_slot(int r, int g) { return g ^ ((r >> 1) & 3); }
// The MLP walks the hidden layer in parts of tailx_hu units (C = 144: 288 in
// three of 96; 180: 360 in twelve of 32, the last 24 of 384 zero): per part fc1's
// k-steps (that many rows, permuted, the columns in the order a lane holds x'),
// then fc2's (C rows in 16s, k = the part's units).
constexpr int tailx_hu(int C) { return C == 144 ? 96 : 32; }
// fc1's bias (b1x), padded to the whole loads that copy it.
#define TX_B1 1024
// Their launch geometry (tailx): blocks of 4 waves, one row tile of 128 tokens a
// block; 64 in the small planes' kernels (_s).
#define WX_THREADS 256
#define WX_ROWS 128
#define WX_ROWS_S 64
constexpr int wx_tiles(int M, int rows = WX_ROWS) { return (M + rows - 1) / rows; }

// The qkv linear (hat_gemmx_qkv, hat_gemmx_qkv180) keeps one column slice in
// LDS for the whole launch: per 32-k step two f16 planes [rows][32], unpadded,
// each row's four 16-byte k-groups stored at slot ws_slot(row, g) (so that reads
// of one k-group down the rows are free of bank conflicts), WS_CHUNK elements
// apart. Three slices, q, k and v: C = 144 of 144 rows, five k-steps; C = 180 of
// 192 rows (180 real), six k-steps (WS_CHUNK180). Groups of NS blocks (one per
// slice, on one XCD) walk the same subtiles of tokens: gemmx_qkv_groups(cus, NS)
// groups.
#define WS_CHUNK (2 * 144 * 32)
#define WS_CHUNK180 (2 * 192 * 32)
#define GX_THREADS 512
constexpr int gemmx_qkv_groups(int cus, int ns) { return cus >= 8 * ns ? cus / (8 * ns) * 8 : 1; }

// hat_qkv_cab1: blocks 0 .. nconv - 1 (a multiple of 8, at least a tile each) run
// the CAB's conv1, the others the qkv linear.
struct QkvCabArgs {
    GemmArgs g;
    CabConvArgs c;
    int nconv;
};

// hat_qkv_cab1_180: the same; conv1 is a Winograd conv of ntile tiles.
struct QkvConvArgs {
    GemmArgs g;
    ConvArgs c;
    int nconv, ntile;  // ntile: tiles times ncb
    int ncb;           // conv1's column blocks: 1, or 2 of 32 channels
};

struct TailXArgs {
    const float* a;             // [M][C] attention output, in v's scale
    const float* res;           // [M][C] block input
    float* out;                 // [M][C] (may alias res)
    float* xn;                  // [M][C] the next norm of out (LN forms)
    const unsigned short* w;    // the projection's steps
    const unsigned short* wm;   // the MLP's steps, part by part
    const unsigned short* w2gx; // CAB: the gate-scaled conv2 weights as 2 steps (k = tap*6 + ci)
    const float* t1;            // CAB: [M][CAB_CS] CAB conv1 output (scaled)
    const float* aux;           // HAB at C = 180: conv2's output [M][C]
    const float* gate;          // and its gate [C]
    const float* bias;          // projection bias (CAB: bias2)
    const float* b1x;           // fc1's bias times the hidden scale, in the parts' row order
    const float* b2;            // fc2's bias
    const float* inw;           // norm2 (scaled)
    const float* inb;
    const float* nw;            // the next norm
    const float* nb;
    int M, H, W;                // rows = the H x W plane (CAB)
    float eps, cscale;
    float ps, pi;               // the projection accumulators' scale and its inverse
    float h1, g0, g1;           // fc1's accumulators to scaled hidden units; gelu_scaled's constants
    float ms, mi;               // the output accumulators' scale and its inverse
    unsigned* amax_out;         // OCAB: out's largest finite magnitude (if set)
};

struct LnArgs {
    const float* x;
    float* y;
    const float* w;
    const float* b;
    int rows, C;
    float eps;
};

// A forward's magnitude slots: the bits of the largest finite |x| of the planes
// that no norm bounds and a Winograd conv reads (ConvArgs::amax): per stage its
// last block's output, then, from AMAX_HEAD, the head's planes. A slot is
// AMAX_LANES words AMAX_STRIDE apart (64 bytes), whose maximum it is: one a XCD, so
// that a kernel's blocks do not all meet in one word.
#define AMAX_SLOTS 64
#define AMAX_HEAD 40
#define AMAX_LANES 8
#define AMAX_STRIDE 16
#define AMAX_WORDS (AMAX_LANES * AMAX_STRIDE)

struct PreArgs {
    const float* in;     // [3][h][w]
    float* out;          // [hp][wp][cstride], channels >= 3 zeroed
    int h, w, hp, wp, cstride;
    float m0, m1, m2, range;
    unsigned* amax;      // [AMAX_SLOTS][AMAX_WORDS], zeroed (if set)
};

// dst[i] = src[i] for n4 float4 (16-byte aligned buffers).
struct CopyArgs {
    const float* src;
    float* dst;
    long n4;
};

// The largest finite |x[i]|, i < n (a multiple of 4), into a magnitude slot
// (AMAX_SLOTS) that holds zeros.
struct AbsMaxArgs {
    const float* x;
    unsigned* out;
    long n;
};

// x[i] *= s, i < n (a multiple of 4).
struct ScaleArgs {
    float* x;
    float s;
    long n;
};

// Column sums of a [nrows][stride] matrix in row blocks: out[blk][c] = sum of
// rows [blk*rows_per, blk*rows_per + rows_per) of column c.
struct ReduceArgs {
    const float* in;
    float* out;
    int nrows, C, stride, rows_per;
};

}  // namespace hatk
