// Learn gradient surface: learning-signal capture during a forward run and the
// LRDS replay of dv/dw over the captured signals (the reference's LearnRuntime,
// LearnRuntime.cpp:197-2457, kernels replay_dw_dx.cu:9-731).
//
// HBM layout:
//   * captured signals It, dIt/dv, dIt/dvpre are time-major (T, N) fp32, T =
//     ksteps + 1, row 0 zero: a capture writes one contiguous row per LR tick;
//   * dense block b (bn x bn x K_len, the caller's kernel K_b[i][j][tau]) is kept
//     tau-major at [tau][i][j], rows padded with zeros to bnp = bn rounded up to 4: the
//     base term reads K_b[i][j][tau], and as K_b[j][k][tau] the same array is the
//     correction GEMM's second operand, contiguous in the reduction index k;
//   * the history is a ring of K_len + 1 slices X_tau, the correction's first operand:
//     block after block, each N rows of bnp floats (the padding zero, never written).
//     Tick tau lives in slot tau % (K_len + 1), slot 0 starts as tick 0's, and the slot a
//     tick writes is never in its own read window.  The dv/dw slices alternate between
//     two buffers (the previous one is still read for dx).
//     Each group of four columns of a slot has an fp32 scale: a power of two that keeps X
//     in range, times the Frobenius clip's rescaling of the history (instead of rewriting
//     K_len slices).
#pragma once
#include <hip/hip_runtime.h>

#include <string>
#include <vector>

namespace hx {

constexpr int kLrMaxChannels = 3;     // pure_i, didv, didvpre
// The allocation-free replay: problems of at most kNoAllocLimitBytes of signals, slices
// and vectors (16 N T + 8 R N^2 bytes and the small ones) are taken; the per-device scratch
// array holds what the kernels need for any of those (block rows padded to multiples of 4,
// the correction's split sums).
constexpr size_t kNoAllocLimitBytes = static_cast<size_t>(64) << 20;
constexpr size_t kNoAllocScratchBytes = static_cast<size_t>(256) << 20;
constexpr int kBaseTicks = 8;         // ticks whose base terms one launch makes

struct CaptureChannel {
    const int* begin = nullptr;       // N + 1: items of column c are [begin[c], begin[c+1])
    double* const* ptr = nullptr;     // item sources, grouped by column in input order
    const float* scale = nullptr;
    float* buf = nullptr;             // (T, N) time-major
};

struct CaptureArgs {
    int n_out = 0;
    double* const* out_ptr = nullptr;
    float* out_vs = nullptr;          // (nsample, n_out)
    int N = 0;
    int nch = 0;
    CaptureChannel ch[kLrMaxChannels];
};

struct ReplayBaseArgs {
    const float* kp = nullptr;
    const long long* koff = nullptr;  // per block offset into kp
    const long long* boff = nullptr;  // per block offset into base (sum of bn^2)
    const int* start = nullptr;
    const int* bn = nullptr;
    const int* bnp = nullptr;
    const float* it = nullptr;        // (T, N)
    int N = 0, T = 0, K_len = 0;
    int t0 = 0, ng = 0;               // ticks t0 .. t0 + ng - 1
    float* base = nullptr;            // tap sums, one set of base_stride floats per tick
    long long base_stride = 0;
};

// dx of one finished tick (n_in 0: none)
struct ReplayDx {
    const float* cur = nullptr;       // the tick's slice
    const int* pin = nullptr;
    int n_in = 0;
    const float* w_tick = nullptr;
    float eps = 0.f;
    int t_idx = 0, ksteps = 0;
    int clip_ran = 0;
    const float* tick_scale = nullptr;
    float* dx = nullptr;
};

// where a tick's slice goes and what is added to its correction
struct ReplayOut {
    int N = 0;
    float dt = 0.f;
    const float* gs = nullptr;        // device grad scale
    const float* base = nullptr;      // this tick's tap sums
    float* out = nullptr;
    int sanitize = 0;                 // zero non-finite entries and write norm partials
    double* norm_part = nullptr;
};

struct ReplayCorrArgs {
    const float* x = nullptr;         // the ring of X slices
    long long xslice = 0;             // floats per slice
    const long long* xoff = nullptr;  // per block offset into a slice
    const float* xscale = nullptr;    // the ring of X's scales, one per group of four columns
    const int* xgroup = nullptr;      // per block its first group
    int xgroups = 0;                  // groups per slot
    int R = 1;                        // ring slots
    int h0 = 0;                       // slot of the window's first tick
    const float* kp = nullptr;
    const long long* koff = nullptr;
    const int* start = nullptr;
    const int* bn = nullptr;
    const int* bnp = nullptr;
    const long long* boff = nullptr;
    const int2* tiles = nullptr;      // (block, first column) of each column tile
    int row_tiles = 0, nsplit = 1, ncorr = 0;   // ncorr: column tiles x row tiles x splits
    int tw = 0, k_t0 = 0;
    float* part = nullptr;            // nsplit > 1: the splits' sums, N x N each
    ReplayOut O;
    ReplayDx dx;
};

struct ReplayFinishArgs {
    const float* part = nullptr;
    int nsplit = 0;                   // 0: no correction
    int nblock = 0;                   // set by the launcher
    const int* col_block = nullptr;   // block of each column
    const int* start = nullptr;
    const int* bn = nullptr;
    const long long* boff = nullptr;
    ReplayOut O;
    ReplayDx dx;
};

// the exponents of X's groups for ticks 0 .. ticks - 1, and the ring's scales at 1
struct ReplayRangeArgs {
    int N = 0, ticks = 0, R = 1, xgroups = 0;
    const int2* group_col = nullptr;  // first column and columns of each group
    const float* dv = nullptr;        // dIt/dv and dIt/dvpre (T, N)
    const float* dp = nullptr;
    unsigned char* xdown = nullptr;   // (ticks, xgroups)
    float* xscale = nullptr;          // (R, xgroups)
};

struct ReplayTickArgs {
    int N = 0;
    const float* cur = nullptr;       // the tick's slice
    int wblocks = 0;                  // set by the launcher
    int due = 0;                      // clip tick
    const double* norm_part = nullptr;
    int npart = 0;
    float thr = 0.f;
    float* gs = nullptr;
    int R = 1, cur_slot = 0;          // ring slots, this tick's
    float* tick_scale = nullptr;
    const int* po = nullptr;
    int n_out = 0;
    const float* dl = nullptr;        // null: only X
    float* w_tick = nullptr;
    float* dw_acc = nullptr;
    float* x = nullptr;               // slot of this tick (null: no X)
    const unsigned char* xdown = nullptr;   // this tick's exponents
    float* xscale = nullptr;          // the ring of scales
    const int* col_group = nullptr;   // group of each column
    int xgroups = 0;
    const long long* xoff = nullptr;
    const int* col_block = nullptr;
    const int* start = nullptr;
    const int* bnp = nullptr;
    const int* pre = nullptr;
    const float* dv = nullptr;        // dIt/dv and dIt/dvpre at the next signal time
    const float* dp = nullptr;
};

void launch_lr_capture(const CaptureArgs& a, int sample, int lr, hipStream_t s);
void launch_rp_base(const ReplayBaseArgs& a, int nblk, int max_bn, hipStream_t s);
void launch_rp_corr(const ReplayCorrArgs& a, int tile_cols, hipStream_t s);
int rp_corr_row_tiles(int N);
int rp_corr_splits(int N, int ntiles, int max_bnp, int tw);
void launch_rp_finish(ReplayFinishArgs a, hipStream_t s);
int rp_finish_blocks(int N);
void launch_rp_range(const ReplayRangeArgs& a, hipStream_t s);
void launch_rp_tick(ReplayTickArgs a, hipStream_t s);
void launch_rp_dx(const ReplayDx& a, int N, int corr_tile_cols, hipStream_t s);   // 0: k_rp_finish's sums
void launch_rp_scale_into(const float* src, float scale, float* dst, long long n, hipStream_t s);
void launch_fill_f32(float* p, float v, long long n, hipStream_t s);
void launch_transpose_nt_tn(const float* src_nt, float* dst_tn, int N, int T, hipStream_t s);

// Host side of the learn surface, owned by a simulation handle.
class LearnRuntime {
public:
    explicit LearnRuntime(hipStream_t s) : stream_(s) {}
    ~LearnRuntime();
    LearnRuntime(const LearnRuntime&) = delete;
    LearnRuntime& operator=(const LearnRuntime&) = delete;

    std::string err;

    // LearnRuntime::set_dense_blocks_f32 / clear_dense_blocks (LearnRuntime.cpp:197-257)
    int set_dense_blocks(int nblk, const float* const* data, const int* bn, const int* k_len);
    void clear_dense_blocks();
    int k_len() const { return k_len_; }
    const std::vector<int>& block_sizes() const { return bn_; }

    // Capture session (LearnRuntime.cpp:1619-1984).  Channel c has its items'
    // sources, destination columns and scales; N = 0 captures outputs only.
    struct Channel {
        std::vector<double*> ptr;
        std::vector<int> dest;
        std::vector<float> scale;
    };
    // Where a capture's signals go: the cache that cached replays read, host
    // buffers given to end_capture (the _into variant), or a private set kept for
    // one streaming replay.  Only CACHE touches the cache.
    enum Sink { SINK_CACHE = 0, SINK_HOST, SINK_STREAM };
    // T <= 0 derives T = (nsample - 1) / k_mul + 1.
    void begin_capture(int nsample, const std::vector<double*>& out_ptr, int N, int T, int k_mul, bool percise,
                       const Channel* ch, int nch, Sink sink);
    bool capturing() const { return capturing_; }
    void sample();                                   // one record point
    void end_capture(float* out_vs_host, float* const* sig_host = nullptr);

    // Replay over the cached capture, host signals loaded by load_signals, or the
    // last streaming capture; the clip schedule follows the entry point.
    enum Source { SRC_CACHE = 0, SRC_HOST, SRC_STREAM };
    struct ReplayIn {
        const float* dl = nullptr;   // (ksteps, n_out)
        int ksteps = 0, n_out = 0, n_in = 0;
        const int* po = nullptr;
        const int* pin = nullptr;
        const int* pre = nullptr;    // N
        float* dw_out = nullptr;     // N
        float* dx_out = nullptr;     // (n_in, ksteps)
        double dt = 0, grad_scale = 1, eps = 1e-6, thr = 1e6;
        bool percise = false;
        int clip_strategy = 1, clip_every = 1;
        Source source = SRC_CACHE;
        bool cached_clip_rule = true;   // strategy 1 every tick, others every clip_every
    };
    int replay(const ReplayIn& in);
    int load_signals(const float* it_nt, const float* dv_nt, const float* dp_nt, int N, int T, bool percise);
    // The replay over host (N, T) signals with every device buffer carved from the
    // library's fixed scratch array (kNoAllocScratchBytes per device): no allocation.
    int replay_from_host_noalloc(const ReplayIn& in, const float* it_nt, const float* dv_nt, const float* dp_nt, int N,
                                 int T);
    int capture_N() const { return cap_N_; }
    int capture_T() const { return cap_T_; }
    bool capture_percise() const { return cap_percise_; }

    // kernel time of the last replay's correction GEMM launches, when timing is on
    bool timing = false;
    double corr_ms = 0;
    long long corr_launches = 0;

    struct Workspace {
        float *slices = nullptr, *x = nullptr, *part = nullptr, *base = nullptr, *xscale = nullptr, *gs = nullptr,
              *tick_scale = nullptr, *w_tick = nullptr, *dw_acc = nullptr, *dl = nullptr, *dx = nullptr,
              *dw_out = nullptr;
        unsigned char* xdown = nullptr;
        int *po = nullptr, *pre = nullptr, *pin = nullptr;
        double* norm_part = nullptr;
        int base_ticks = 0;               // ticks base holds
    };

private:
    int fail(const char* fmt, ...);
    void free_all(std::vector<void*>& v);
    int replay_on(const ReplayIn& in, const Workspace& ws, float* const* sig, int N);

    hipStream_t stream_;
    // Buffer sizes of a replay with and without the precise term, in one place for both
    // ways of providing them.
    struct Sizes {
        int R = 1;
        size_t x = 0, xscale = 0, part = 0, norm = 0;
    };
    Sizes sizes_for(int N, bool percise) const;

    // dense blocks
    int k_len_ = 0, nblk_ = 0, max_bn_ = 0, max_bnp_ = 0, tile_cols_ = 64;
    std::vector<int> bn_, start_;
    std::vector<long long> koff_, boff_, xoff_;
    long long base_len_ = 0, xcols_ = 0;    // sum of bn^2, sum of bnp
    std::vector<int2> tiles_;
    std::vector<void*> blk_mem_;
    float* d_kp_ = nullptr;
    long long *d_koff_ = nullptr, *d_boff_ = nullptr, *d_xoff_ = nullptr;
    int *d_start_ = nullptr, *d_bn_ = nullptr, *d_bnp_ = nullptr, *d_xgroup_ = nullptr, *d_col_block_ = nullptr,
        *d_col_group_ = nullptr;
    int2 *d_tiles_ = nullptr, *d_group_col_ = nullptr;
    // capture cache (T, N) per channel
    int cap_N_ = 0, cap_T_ = 0, cap_kmul_ = 0;
    bool cap_percise_ = false;
    std::vector<void*> cap_mem_;
    float* d_cap_[kLrMaxChannels] = {nullptr, nullptr, nullptr};
    // capture session
    bool capturing_ = false;
    int sample_ = 0, nsample_ = 0, kmul_ = 1, sess_T_ = 0;
    Sink sink_ = SINK_CACHE;
    std::vector<void*> sess_sig_mem_;   // HOST / STREAM signal buffers
    float* d_stream_[kLrMaxChannels] = {nullptr, nullptr, nullptr};
    int stream_N_ = 0, stream_T_ = 0;
    CaptureArgs cargs_{};
    std::vector<void*> sess_mem_;
    // host-loaded signals (T, N)
    int sig_N_ = 0, sig_T_ = 0;
    size_t sig_cap_ = 0;                // floats each signal buffer holds
    int sig_ch_ = 0;                    // signal buffers there are
    float* d_sig_stage_ = nullptr;
    std::vector<void*> sig_mem_;
    float* d_sig_[kLrMaxChannels] = {nullptr, nullptr, nullptr};
    // replay workspace, kept while the problem shape is unchanged
    std::vector<void*> ws_mem_;
    std::vector<long long> ws_key_;
    Workspace ws_;
};

}  // namespace hx
