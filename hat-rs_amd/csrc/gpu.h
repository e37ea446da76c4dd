// The MI355X backend behind the reference's Backend interface.
//
// Reference seam: `trait Backend { fn name(); fn forward(h, w, input) }`
// (src/backend.rs:29-36) with `Gpu::new(&Weights)` (src/gpu.rs:372-386) and
// `Gpu::forward` (src/gpu.rs:759-803). Input is [3][h][w] in [0,1] (not
// mean-adjusted); output is [3][h*s][w*s] after denormalisation.
#pragma once
#include <map>
#include <string>
#include <vector>

#include "hip_rt.h"
#include "kargs.h"
#include "plan.h"
#include "weights.h"

namespace hat {

class Backend {
public:
    virtual ~Backend() {}
    virtual const char* name() const = 0;
    virtual void forward(int h, int w, const float* in, float* out) = 0;
};

struct DevLinear {
    float* w = nullptr;  // [N][Kp], or null where the split kernels hold the weights
    bool rows = false;   // w is set (in the counting pass: would be)
    float* b = nullptr;  // [N]
    // qkv: the same weights split for hat_gemmx_qkv* (pack_linear_ws), or null
    // where the FP32 kernels run (and w is null where they do not).
    unsigned short* wx = nullptr;
    // qkv: what the split-f16 kernel multiplies q, k and v by (GemmArgs::oscale)
    float oscale[3] = {1.0f, 1.0f, 1.0f};
    int N = 0, K = 0, Kp = 0;
};

// The CAB of the compress-to-6 family, in the folded form (conv1 per-tap
// weights; conv2 and the channel attention as raw tensors for the gate kernel).
struct DevCab {
    unsigned short* w1 = nullptr;  // conv1 split for hat_cab_conv1 (CX_WPACK f16)
    float oscale = 1.0f;           // 1 over norm1's scale and the weights'
    float* b1 = nullptr;  // [6]
    float* w2 = nullptr;  // [144][6][3][3]
    float* b2 = nullptr;  // [144]
    float* wa = nullptr;  // [sq][144]
    float* ba = nullptr;
    float* wb = nullptr;  // [144][sq]
    float* bb = nullptr;
};

// conv1 weight [6][144][3][3] -> 64 rows of 144 (row tap*6 + co holds
// w[co][:][tap], rows 54..63 zero), each weight times sw and as two f16 parts in
// hat_cab_conv1's A-operand layout (CX_WPACK elements).
std::vector<unsigned short> pack_cab_conv1(const float* w, float sw);
// CabConvArgs' scales: t1's, and oscale as DevCab's.
void cab_scales(float ts, float oscale, hatk::CabConvArgs* a);

// A block's second half on split-f16 (tailx.hip): the projection's and the MLP's
// packed steps, fc1's bias in the parts' row order, and the scales (TailXArgs).
struct DevTail {
    unsigned short* w = nullptr;
    unsigned short* wm = nullptr;
    float* b1x = nullptr;
    int C = 0;  // 144 or 180
    float ps = 1.0f, h1 = 1.0f, hs = 1.0f, ms = 1.0f;  // hs: the hidden units' scale
    float ts = 1.0f, gs = 1.0f;                        // folded CAB: t1's and w2gx's scales (ps = ts gs)
};

struct DevConv {
    float* w = nullptr;  // [CIp/16][9][COp][16]
    float* b = nullptr;  // [COp]
    unsigned short* wu = nullptr;  // convs with a Winograd kernel: split U (pack_wino)
    float uinv = 1.0f;             // takes U's scale out
    float vs = 1.0f;               // V's scale where the host knows it
    int CI = 0, CIp = 0, CO = 0, COp = 0, r = 0;
};

// ---- Power-of-two scales for the split-f16 kernels (common.h), which need
// their operands inside f16's range. Every scale is exact in fp32, so the
// results do not depend on it while nothing leaves that range.

// The largest power of two s with bound * s <= 2^15 (half of f16's range: room
// for the roundings the bound leaves out); 1 for a bound that is 0 or not finite.
float f16_scale(double bound);
// A vector that a LayerNorm (w, b over C channels) can produce is n o w + b with
// |n|_2 <= sqrt(C), and |n_c| <= sqrt(C). Bounds over every such vector: of
// |row . y + bias| for rows [n0, n1) of a linear [N][C] (the largest), and of
// |y_c| over the channels.
double ln_linear_bound(const float* w, const float* b, const float* lnw, const float* lnb, int n0, int n1, int C);
double ln_bound(const float* lnw, const float* lnb, int C);
// The scales of an attention's q, k and v rows (folded into the qkv weights):
// q and k by inverse powers of two that balance their bounds, so that the scores
// do not change, v by its own (the projection's weights take it out). ok: the
// balanced bounds fit; otherwise the FP32 attention runs on q and k as they are.
// It is linear in v, which keeps its scale: the tail behind it splits its output.
struct QkvScale {
    float q = 1.0f, k = 1.0f, v = 1.0f;
    bool ok = false;
};
QkvScale qkv_scale(double bq, double bk, double bv, int head_dim);

// Host-side repacking (also used by the selftest and the op entry points). fill:
// false leaves zeros, for the counting pass that needs only the sizes.
std::vector<float> pack_linear(const float* w, int N, int K, int* Kp);
// hat_gemmx_qkv's weight-stationary slices: per slice (144 rows at K = 144, 192
// at 180) five or six chunks of two f16 planes [rows][32], each row's 16-byte
// k-groups swizzled (ws_slot), WS_CHUNK elements apart; K = 144's fifth step
// packed (split2_half_step). w = p0 + p1, each part the round-to-nearest f16 of
// what the one before leaves; q's, k's and v's rows times ws[0..2] first.
std::vector<unsigned short> pack_linear_ws(const float* w, int N, int K, const float (&ws)[3], bool fill = true);
// The largest |w[i]|, i < n (NaN if there is one).
double abs_max(const float* w, size_t n);
// The tails' steps (tailx.hip), every weight times a scale and split into two f16
// parts; both arrays end in TX_PAD zeros. The projection [C][C]: its k-steps. The
// MLP (fc1 [2C][C] + b1, fc2 [C][2C]): per part of tailx_hu(C) units fc1's k-steps
// (the unit rows in tailx_unit's order, column k the channel tailx_channel(C, k))
// and fc2's, fc1 times s1 and fc2 times s2; b1 times hs in the parts' row order.
std::vector<unsigned short> pack_tail_proj(const float* w, int C, float s, bool fill = true);
void pack_tail_mlp(const float* w1, const float* b1, const float* w2, int C, float s1, float s2, float hs,
                   std::vector<unsigned short>* w, std::vector<float>* b1x, bool fill = true);
int tailx_channel(int C, int k);
// The scales and packed weights of a tail whose attention output comes times sv
// and norm2 (n2w, n2b unscaled) times sn; cab (if set): the folded CAB's bound of
// |t1| and largest |cscale * conv2 weight|, which share the projection's scale.
struct TailPack {
    std::vector<unsigned short> w, wm;
    std::vector<float> b1x;
    DevTail t;  // the scales; no device pointers
};
struct TailCab {
    double t1, w2;
};
void tail_scales(const DevTail& t, hatk::TailXArgs* f);
TailPack pack_tail(const float* wp, const float* w1, const float* b1, const float* w2, const float* n2w, const float* n2b,
                   int C, float sv, float sn, const TailCab* cab, bool fill = true);

// Winograd U = G g G^T of a 3x3 conv [CO][CI][3][3] (formed in double), times the
// power of two 1 / *uinv and split into two f16 parts in the layout convwino.hip
// streams: [32-channel chunk][point][16-channel tile][part][lane][8].
std::vector<unsigned short> pack_wino(const float* w, int CO, int CI, int r, float* uinv, bool fill = true);
// A plane's largest magnitude on the device (ConvArgs::amax), and whether a kernel
// of this forward has left it there.
struct Amax {
    unsigned* slot = nullptr;
    bool filled = false;
};
std::vector<float> pack_conv(const float* w, const float* b, int CO, int CI, int r,
                             std::vector<float>* bias_out, int* CIp, int* COp);
// A Winograd conv kernel (convwino.hip) over `tiles` 8 x 16 tiles in `ncb`
// column blocks (p.nblk set here). The persistent ones (convwino_persistent:
// the column-sum kernel) take a grid of at most one block a CU (or
// max_blocks), a multiple of ncb so that each block keeps its column block,
// each walking the virtual blocks blockIdx.x + i gridDim.x and fetching its
// next tile's first patch chunk under the current tile's epilogue; the others
// take one block a tile.
// The kernel's form for small planes: its name and column blocks.
struct WinoSmall {
    std::string name;
    unsigned ncb;
};
WinoSmall convwino_small(const std::string& name);
bool convwino_persistent(const std::string& name);
void launch_wino(hipStream_t s, const char* name, unsigned tiles, unsigned ncb, hatk::ConvArgs& p,
                 unsigned max_blocks = 0);

class GpuBackend : public Backend {
public:
    explicit GpuBackend(const Weights& wt);
    ~GpuBackend() override;
    const char* name() const override { return "gpu"; }
    void forward(int h, int w, const float* in, float* out) override;
    // Device-resident variant: d_in [3][h][w], d_out [3][h*s][w*s].
    void forward_device(int h, int w, const float* d_in, float* d_out);
    // The same pass with every per-plan buffer carved from the library's fixed
    // scratch array: no device memory is allocated. Throws if the plan does not
    // fit. Calls that overlap on one GPU share the array and race.
    void forward_noalloc(int h, int w, const float* d_in, float* d_out);
    // n images of one size, host [n][3][h][w] in, host [n][3][h*s][w*s] out:
    // up to kBatchSlots images in flight at once, each on its own stream with
    // its own per-plan buffers and pinned staging, so the kernels of several
    // small images fill the device together. Synchronous.
    void forward_batch(int n, int h, int w, const float* in, float* out);
    static constexpr int kBatchSlots = 4;
    // Bytes forward_noalloc needs at h x w.
    size_t noalloc_bytes(int h, int w) const;
    // Device bytes of the per-plan buffers a backend over `wt` allocates for an
    // h x w forward (gpu.rs:78-290 footprint_floats), computed without a device.
    static size_t plan_bytes(const Weights& wt, int h, int w, bool host_io);
    // Device bytes the weight upload of a backend over `wt` allocates (the
    // packed FP32 tensors and their split copies), computed without a
    // device by running the upload's packers in a counting pass; cached in wt.
    static size_t device_weight_bytes(const Weights& wt);
    static bool cab_folded(const Weights& wt);
    static bool tail_runs(const Weights& wt, bool ocab);
    // HAB.forward of one block (gpu.rs:469-520 `hab`) on a window-multiple
    // hp x wp plane: host x, out token-major [hp*wp][embed]; with the block's
    // shift and mask when it is odd. iters > 0: *ms = mean device time of the
    // block (its norm1 included) over that many further runs.
    void op_hab(int stage, int block, int hp, int wp, const float* x, float* out, int iters, float* ms);
    size_t acts_bytes() const { return acts_bytes_; }
    size_t weight_bytes() const { return weight_bytes_; }
    hipStream_t stream() const { return stream_; }
    const Weights& weights() const { return wt_; }

private:
    struct CountOnly {};
    GpuBackend(const Weights& wt, CountOnly);  // the counting pass: packs, uploads nothing
    void upload_all();
    const Weights& wt_;
    bool count_only_ = false;
    hipStream_t stream_ = nullptr;
    std::map<std::string, float*> raw_;
    std::map<std::string, DevLinear> lin_;
    std::map<std::string, DevConv> conv_;
    std::map<std::string, DevCab> cab_;
    std::map<std::string, DevTail> tail_;  // by MLP name: blocks and OCABs that run tailx.hip
    std::map<std::string, bool> attn_f16_;  // by bias table name: the split-f16 attention runs
    bool cab_fold_ = false;  // the C = 144, 6-channel CAB runs folded
    std::vector<void*> owned_;
    size_t weight_bytes_ = 0;

    // The per-plan device buffers of one forward (Acts, gpu.rs:78-290). They
    // come from hipMalloc, once per input size (ensure_plan), or, for
    // forward_noalloc, from the library's fixed scratch array.
    struct Acts {
        float *x0 = nullptr, *body = nullptr, *xa = nullptr, *xb = nullptr, *xn = nullptr, *t1 = nullptr,
              *t2 = nullptr, *partial = nullptr, *red = nullptr, *gate = nullptr, *qkv = nullptr, *ao = nullptr,
              *hidden = nullptr, *head0 = nullptr, *head1 = nullptr, *din = nullptr, *dout = nullptr,
              *cab_part = nullptr, *w2gx = nullptr, *bias2 = nullptr, *amax = nullptr;
    };
    // Each buffer of plan p and its size in floats (0: not used by this
    // network); host_io adds the staging buffers of the host-memory forward.
    static std::vector<std::pair<float**, size_t>> layout(const Weights& wt, const Plan& p, Acts& a,
                                                          bool host_io);

    Plan plan_;
    bool have_plan_ = false;
    std::vector<void*> acts_;
    size_t acts_bytes_ = 0;
    Acts a_;
    int t1_stride_ = 0, nblk_conv2_ = 0;

    // forward_batch's slots: a stream, a per-plan buffer set and pinned
    // staging each, kept for the last batch size.
    struct BatchSlot {
        hipStream_t s = nullptr;
        Acts a;
        float *hin = nullptr, *hout = nullptr;
        int img = -1;
    };
    std::vector<BatchSlot> batch_;
    Plan batch_plan_;
    std::vector<void*> batch_dev_;
    void free_batch();

    // Backend::forward's host staging, kept for the plan: pinned input and
    // output buffers; the stream that downloads the output bands, an event per
    // band on each stream (computed, downloaded).
    float *stage_in_ = nullptr, *stage_out_ = nullptr;
    size_t stage_in_n_ = 0, stage_out_n_ = 0;
    hipStream_t copy_stream_ = nullptr;
    std::vector<hipEvent_t> band_ev_, copy_ev_;
    void free_stage();

    float* upload(const float* src, size_t n);
    void* upload_bytes(const void* src, size_t bytes);
    void upload_raw(const std::string& name);
    // out[3]: the factors of a qkv's q, k and v outputs (weights and bias), or
    // null; in: the factor of every weight (the inverse of its input's scale);
    // bias_only: the weights go up elsewhere (upload_tail).
    void upload_linear(const std::string& name, const float* out = nullptr, float in = 1.0f, bool bias_only = false);
    // A norm whose output feeds split-f16 kernels: its weight and bias times the
    // power of two that takes every row it can produce to f16's range.
    void upload_norm(const std::string& name);
    std::map<std::string, float> norm_scale_;
    // An attention's qkv and projection behind norm `ln`, scaled (qkv_scale);
    // attn_f16_ of its table: whether the split-f16 attention runs.
    void upload_attn(const std::string& qkv, const std::string& proj, const std::string& ln, const std::string& table);
    // in: as upload_linear's; bound: of the input's |x| as the kernel reads it, or 0
    // where only the device can know (Amax)
    void upload_conv(const std::string& name, int r = 0, float in = 1.0f, double bound = 0.0);
    // what |t1| (the CAB's conv1 output) cannot exceed behind norm1
    double cab_t1_bound(const std::string& cab, const std::string& norm1) const;
    std::map<std::string, float> t1_scale_;  // by block: the unfolded CAB's t1
    // a block's norm2, projection and MLP: the split-f16 tail where it runs
    // (tail_runs), else FP32 rows (upload_attn first; cab: the folded CAB's prefix,
    // or empty)
    void upload_tail(const std::string& proj, const std::string& mlp, const std::string& norm2, const std::string& cab,
                     const std::string& norm1, bool ocab);
    void check_linears() const;
    float v_scale_ = 1.0f;  // of the attention uploaded last
    void ensure_plan(int h, int w);
    void free_plan();
    // With bands: the output's row bands [y0, y1) in the order they are
    // written, band_ev_[k] recorded on the stream after band k (the
    // host-memory forward downloads each while later ones compute).
    void run_forward(int h, int w, const float* d_in, float* d_out,
                     std::vector<std::pair<int, int>>* bands = nullptr);
    bool head_bands_fit(const DevConv& up, const DevConv& last, int hh, int ww, int feat) const;

    void layernorm(const float* x, float* y, const std::string& prefix, long rows);
    void gemm(const DevLinear& L, const float* a, int lda, long M, float* out, int ldo, int epi,
              const float* res = nullptr, const float* aux = nullptr, const float* gate = nullptr,
              float* xn = nullptr, const std::string& norm = "");
    void conv(const DevConv& C, const float* in, int cin_stride, int H, int W, float* out,
              int co_stride, int epi, int act, const float* res = nullptr, float* partial = nullptr,
              int crop_h = 0, int crop_w = 0, int band_r0 = 0, int band_r1 = -1, Amax* in_max = nullptr,
              Amax* out_max = nullptr, float os = 1.0f);
    void attention(const std::string& table, bool oca, int shift, const hatk::CabGateArgs* gate = nullptr,
                   const hatk::SeArgs* se = nullptr);
    void mlp(const std::string& prefix, float* x, int epi, const std::string& norm);
    void hab(int stage, int block, float* x_in, float* x_out, const std::string& next_norm);
    void ocab(int stage, float* x, Amax* out_max);
    unsigned* magnitude_slots(int i) const;  // the current plan's i-th
};

// Isolated ops on host buffers (cfg2 / cfg3 of the benchmark plan). Each
// uploads, runs `warmup + iters` times, downloads, and reports the mean device
// time per run (HIP events on the op's stream) in *ms when ms is non-null.
void op_swmsa(const float* x, float* out, int hp, int wp, int c, int heads, int shift,
              const float* qkv_w, const float* qkv_b, const float* proj_w, const float* proj_b,
              const float* table, int iters, float* ms, float* attn_ms);
void op_ocab(const float* x, float* out, int hp, int wp, int c, int heads, int mlp_ratio,
             const float* n1w, const float* n1b, const float* qkv_w, const float* qkv_b,
             const float* proj_w, const float* proj_b, const float* table, const float* n2w,
             const float* n2b, const float* fc1_w, const float* fc1_b, const float* fc2_w,
             const float* fc2_b, int iters, float* ms, float* attn_ms);

// Selftest: every kernel against a host twin. Prints "  ok  <name>" per pass.
int gpu_selftest(std::string* err);

}  // namespace hat
