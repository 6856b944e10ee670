// Host side of the learn gradient surface: dense blocks, the capture session
// and the per-tick LRDS replay driver (LearnRuntime.cpp:197-257, 1619-2457).
//
// The replay loop issues, per LR tick, correction GEMM [-> its splits' sum] -> tick end
// (clip decision, w_tick, X) on one stream with no host synchronisation: the Frobenius
// clip decision, the grad scale and the history rescale stay on the device
// (the reference copies the norm to the host every checked tick).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <mutex>
#include <stdexcept>
#include <string>
#include <vector>

#include "learn.h"

namespace hx {
namespace {

struct HipFail : std::runtime_error {
    using std::runtime_error::runtime_error;
};

#define LRC(x)                                                                    \
    do {                                                                          \
        hipError_t e_ = (x);                                                      \
        if (e_ != hipSuccess) throw HipFail(std::string(#x) + ": " + hipGetErrorString(e_)); \
    } while (0)

template <class T>
T* lalloc(std::vector<void*>& owned, size_t n) {
    void* p = nullptr;
    LRC(hipMalloc(&p, std::max<size_t>(n, 1) * sizeof(T)));
    owned.push_back(p);
    return static_cast<T*>(p);
}

template <class T>
T* lupload(std::vector<void*>& owned, const T* h, size_t n) {
    T* p = lalloc<T>(owned, n);
    if (n) LRC(hipMemcpy(p, h, n * sizeof(T), hipMemcpyHostToDevice));
    return p;
}

}  // namespace

LearnRuntime::~LearnRuntime() {
    free_all(blk_mem_);
    free_all(cap_mem_);
    free_all(sess_mem_);
    free_all(sig_mem_);
    free_all(ws_mem_);
}

void LearnRuntime::free_all(std::vector<void*>& v) {
    for (void* p : v) (void)hipFree(p);
    v.clear();
}

int LearnRuntime::fail(const char* fmt, ...) {
    char buf[1024];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    err = buf;
    return -1;
}

// LearnRuntime::clear_dense_blocks (LearnRuntime.cpp:246-257) also drops the
// capture cache and the replay workspace.
void LearnRuntime::clear_dense_blocks() {
    (void)hipStreamSynchronize(stream_);
    free_all(blk_mem_);
    free_all(cap_mem_);
    free_all(ws_mem_);
    free_all(sig_mem_);
    ws_key_.clear();
    k_len_ = nblk_ = max_bn_ = max_bnp_ = 0;
    bn_.clear();
    start_.clear();
    koff_.clear();
    boff_.clear();
    xoff_.clear();
    base_len_ = xcols_ = 0;
    tiles_.clear();
    cap_N_ = cap_T_ = cap_kmul_ = 0;
    cap_percise_ = false;
    sig_N_ = sig_T_ = sig_ch_ = 0;
    sig_cap_ = 0;
    d_sig_stage_ = nullptr;
    for (int c = 0; c < kLrMaxChannels; ++c) d_cap_[c] = d_sig_[c] = nullptr;
}

// LearnRuntime::set_dense_blocks_f32 (LearnRuntime.cpp:197-244): every block is
// square with one common K_len; returns K_len.
int LearnRuntime::set_dense_blocks(int nblk, const float* const* data, const int* bn, const int* k_len) {
    clear_dense_blocks();
    if (nblk <= 0) return 0;
    int kl = -1;
    for (int b = 0; b < nblk; ++b) {
        if (!data || !data[b] || bn[b] <= 0 || k_len[b] <= 0) return fail("set_dense_blocks_f32: invalid block at %d", b);
        if (kl < 0) kl = k_len[b];
        else if (k_len[b] != kl)
            return fail("set_dense_blocks_f32: K_len mismatch in block %d (%d vs %d)", b, k_len[b], kl);
    }
    try {
        int start = 0, ncol = 0;
        long long koff = 0, boff = 0;
        std::vector<int> bnp, xgroup, col_block, col_group;
        std::vector<int2> group_col;
        for (int b = 0; b < nblk; ++b) ncol += bn[b];
        for (int b = 0; b < nblk; ++b) {
            const int n = bn[b], np = (n + 3) & ~3;
            bn_.push_back(n);
            bnp.push_back(np);
            start_.push_back(start);
            koff_.push_back(koff);
            boff_.push_back(boff);
            xoff_.push_back(static_cast<long long>(ncol) * xcols_);
            xgroup.push_back(static_cast<int>(xcols_ / 4));
            for (int k = 0; k < n; k += 4) {
                col_group.insert(col_group.end(), std::min(4, n - k), static_cast<int>(group_col.size()));
                group_col.push_back(make_int2(start + k, std::min(4, n - k)));
            }
            col_block.insert(col_block.end(), n, b);
            max_bn_ = std::max(max_bn_, n);
            max_bnp_ = std::max(max_bnp_, np);
            start += n;
            koff += static_cast<long long>(n) * np * kl;
            boff += static_cast<long long>(n) * n;
            xcols_ += np;
        }
        base_len_ = boff;
        // element K[i][j][tau] goes to kp[tau][i][j], rows padded with zeros
        std::vector<float> kp(static_cast<size_t>(koff), 0.f);
        for (int b = 0; b < nblk; ++b) {
            const int n = bn[b], np = bnp[b];
            const size_t plane = static_cast<size_t>(n) * np;
            for (int i = 0; i < n; ++i)
                for (int tau = 0; tau < kl; ++tau) {
                    const float* src = data[b] + static_cast<size_t>(i) * n * kl + tau;
                    float* dst = kp.data() + koff_[b] + tau * plane + static_cast<size_t>(i) * np;
                    for (int j = 0; j < n; ++j) dst[j] = src[static_cast<size_t>(j) * kl];
                }
        }
        k_len_ = kl;
        nblk_ = nblk;
        // column tile of the correction GEMM
        tile_cols_ = max_bn_ > 64 ? 128 : max_bn_ > 32 ? 64 : 32;
        for (int b = 0; b < nblk; ++b)
            for (int j0 = 0; j0 < bn_[b]; j0 += tile_cols_) tiles_.push_back(make_int2(b, j0));
        d_kp_ = lupload(blk_mem_, kp.data(), kp.size());
        d_koff_ = lupload(blk_mem_, koff_.data(), koff_.size());
        d_boff_ = lupload(blk_mem_, boff_.data(), boff_.size());
        d_xoff_ = lupload(blk_mem_, xoff_.data(), xoff_.size());
        d_xgroup_ = lupload(blk_mem_, xgroup.data(), xgroup.size());
        d_col_group_ = lupload(blk_mem_, col_group.data(), col_group.size());
        d_group_col_ = lupload(blk_mem_, group_col.data(), group_col.size());
        d_start_ = lupload(blk_mem_, start_.data(), start_.size());
        d_bn_ = lupload(blk_mem_, bn_.data(), bn_.size());
        d_bnp_ = lupload(blk_mem_, bnp.data(), bnp.size());
        d_col_block_ = lupload(blk_mem_, col_block.data(), col_block.size());
        d_tiles_ = lupload(blk_mem_, tiles_.data(), tiles_.size());
    } catch (const std::exception& e) {
        clear_dense_blocks();
        return fail("set_dense_blocks_f32: %s", e.what());
    }
    return k_len_;
}

void LearnRuntime::begin_capture(int nsample, const std::vector<double*>& out_ptr, int N, int T, int k_mul,
                                 bool percise, const Channel* ch, int nch, Sink sink) {
    free_all(sess_mem_);
    free_all(sess_sig_mem_);
    for (int c = 0; c < kLrMaxChannels; ++c) d_stream_[c] = nullptr;
    stream_N_ = stream_T_ = 0;
    cargs_ = CaptureArgs{};
    cargs_.n_out = static_cast<int>(out_ptr.size());
    cargs_.out_ptr = lupload(sess_mem_, out_ptr.data(), out_ptr.size());
    cargs_.out_vs = lalloc<float>(sess_mem_, static_cast<size_t>(nsample) * out_ptr.size());
    cargs_.N = N;
    cargs_.nch = N > 0 ? nch : 0;
    nsample_ = nsample;
    sample_ = 0;
    kmul_ = k_mul;
    sink_ = sink;
    sess_T_ = 0;
    if (N > 0) {
        if (T <= 0) T = (nsample - 1) / k_mul + 1;
        sess_T_ = T;
        float* buf[kLrMaxChannels] = {nullptr, nullptr, nullptr};
        if (sink != SINK_CACHE) {
            for (int c = 0; c < nch; ++c) buf[c] = lalloc<float>(sess_sig_mem_, static_cast<size_t>(T) * N);
        } else {
            if (cap_N_ != N || cap_T_ != T || cap_kmul_ != k_mul || cap_percise_ != percise) {
                free_all(cap_mem_);
                for (int c = 0; c < kLrMaxChannels; ++c) d_cap_[c] = nullptr;
                for (int c = 0; c < nch; ++c) d_cap_[c] = lalloc<float>(cap_mem_, static_cast<size_t>(T) * N);
                cap_N_ = N;
                cap_T_ = T;
                cap_kmul_ = k_mul;
                cap_percise_ = percise;
            }
            for (int c = 0; c < nch; ++c) buf[c] = d_cap_[c];
        }
        for (int c = 0; c < nch; ++c) {
            // LR rows keep index 0 as zeros (LearnRuntime.cpp:1571-1574, 1938-1942)
            launch_fill_f32(buf[c], 0.f, static_cast<long long>(T) * N, stream_);
            // group the channel's items by destination column, keeping input order
            std::vector<int> begin(N + 1, 0);
            for (int d : ch[c].dest) begin[d + 1]++;
            for (int i = 0; i < N; ++i) begin[i + 1] += begin[i];
            std::vector<int> fill(begin.begin(), begin.end() - 1);
            std::vector<double*> ptr(ch[c].ptr.size());
            std::vector<float> scale(ch[c].ptr.size());
            for (size_t q = 0; q < ch[c].ptr.size(); ++q) {
                const int at = fill[ch[c].dest[q]]++;
                ptr[at] = ch[c].ptr[q];
                scale[at] = ch[c].scale[q];
            }
            cargs_.ch[c].begin = lupload(sess_mem_, begin.data(), begin.size());
            cargs_.ch[c].ptr = lupload(sess_mem_, ptr.data(), ptr.size());
            cargs_.ch[c].scale = lupload(sess_mem_, scale.data(), scale.size());
            cargs_.ch[c].buf = buf[c];
        }
    }
    capturing_ = true;
}

void LearnRuntime::sample() {
    if (!capturing_) return;
    if (sample_ >= nsample_) throw std::runtime_error("learn capture: more samples than steps");
    const int k = kmul_;
    const int lr = (cargs_.nch > 0 && sample_ > 0 && sample_ % k == 0 && sample_ / k < sess_T_) ? sample_ / k : 0;
    launch_lr_capture(cargs_, sample_, lr, stream_);
    ++sample_;
}

void LearnRuntime::end_capture(float* out_vs_host, float* const* sig_host) {
    capturing_ = false;
    LRC(hipStreamSynchronize(stream_));
    if (sample_ != nsample_) throw std::runtime_error("learn capture: sample count mismatch");
    if (out_vs_host && cargs_.n_out > 0)
        LRC(hipMemcpy(out_vs_host, cargs_.out_vs, sizeof(float) * static_cast<size_t>(nsample_) * cargs_.n_out,
                      hipMemcpyDeviceToHost));
    if (sink_ == SINK_HOST && sig_host) {
        const size_t n = static_cast<size_t>(sess_T_) * cargs_.N;
        for (int c = 0; c < kLrMaxChannels; ++c) {
            if (!sig_host[c]) continue;
            if (c < cargs_.nch)
                LRC(hipMemcpy(sig_host[c], cargs_.ch[c].buf, sizeof(float) * n, hipMemcpyDeviceToHost));
            else
                std::fill(sig_host[c], sig_host[c] + n, 0.f);
        }
    }
    if (sink_ == SINK_STREAM) {
        for (int c = 0; c < kLrMaxChannels; ++c) d_stream_[c] = c < cargs_.nch ? cargs_.ch[c].buf : nullptr;
        stream_N_ = cargs_.N;
        stream_T_ = sess_T_;
    } else {
        free_all(sess_sig_mem_);
    }
    free_all(sess_mem_);
}

// replay_compute_dw_dx_from_signals_into's signal upload (LearnRuntime.cpp:575-582):
// host (N, T) arrays are transposed on the device into the (T, N) layout.
int LearnRuntime::load_signals(const float* it_nt, const float* dv_nt, const float* dp_nt, int N, int T,
                               bool percise) {
    try {
        // the buffers of the last call serve again where they are large enough (up to four
        // times what is needed: a much smaller problem gives the memory back)
        const size_t n = static_cast<size_t>(N) * T;
        const int nch = percise ? 3 : 1;
        if (sig_cap_ < n || sig_cap_ / 4 > n || sig_ch_ < nch) {
            (void)hipStreamSynchronize(stream_);
            free_all(sig_mem_);
            sig_cap_ = 0;
            sig_ch_ = 0;
            for (int c = 0; c < kLrMaxChannels; ++c) d_sig_[c] = nullptr;
            d_sig_stage_ = lalloc<float>(sig_mem_, n * nch);
            for (int c = 0; c < nch; ++c) d_sig_[c] = lalloc<float>(sig_mem_, n);
            sig_cap_ = n;
            sig_ch_ = nch;
        }
        const float* src[3] = {it_nt, dv_nt, dp_nt};
        for (int c = 0; c < nch; ++c) {
            float* stage = d_sig_stage_ + c * n;
            LRC(hipMemcpyAsync(stage, src[c], n * sizeof(float), hipMemcpyHostToDevice, stream_));
            launch_transpose_nt_tn(stage, d_sig_[c], N, T, stream_);
        }
        LRC(hipStreamSynchronize(stream_));    // the caller's arrays are read
        sig_N_ = N;
        sig_T_ = T;
    } catch (const std::exception& e) {
        return fail("replay_compute_dw_dx_from_signals_into: %s", e.what());
    }
    return 0;
}

int LearnRuntime::replay(const ReplayIn& in) {
    const int N = in.source == SRC_CACHE ? cap_N_ : in.source == SRC_HOST ? sig_N_ : stream_N_;
    const int T = in.source == SRC_CACHE ? cap_T_ : in.source == SRC_HOST ? sig_T_ : stream_T_;
    float* const* sig = in.source == SRC_CACHE ? d_cap_ : in.source == SRC_HOST ? d_sig_ : d_stream_;
    if (N <= 0 || T != in.ksteps + 1) return fail("replay: no signals of %d ticks", in.ksteps);
    const int ks = in.ksteps;
    try {
        const Sizes z = sizes_for(N, in.percise);
        const std::vector<long long> key = {N, z.R, ks, in.n_out, in.n_in, in.percise ? 1 : 0};
        if (key != ws_key_) {
            free_all(ws_mem_);
            ws_key_.clear();
            const size_t slice = static_cast<size_t>(N) * N;
            ws_.slices = lalloc<float>(ws_mem_, 2 * slice);
            ws_.x = lalloc<float>(ws_mem_, z.x);
            ws_.part = lalloc<float>(ws_mem_, z.part);
            ws_.xscale = lalloc<float>(ws_mem_, z.xscale);
            ws_.xdown = lalloc<unsigned char>(ws_mem_, z.xscale ? static_cast<size_t>(ks) * xcols_ / 4 : 0);
            ws_.gs = lalloc<float>(ws_mem_, 1);
            ws_.tick_scale = lalloc<float>(ws_mem_, 1);
            ws_.w_tick = lalloc<float>(ws_mem_, N);
            ws_.dw_acc = lalloc<float>(ws_mem_, N);
            ws_.dl = lalloc<float>(ws_mem_, static_cast<size_t>(ks) * in.n_out);
            ws_.po = lalloc<int>(ws_mem_, in.n_out);
            ws_.pre = lalloc<int>(ws_mem_, N);
            ws_.pin = lalloc<int>(ws_mem_, std::max(in.n_in, 1));
            ws_.dx = lalloc<float>(ws_mem_, static_cast<size_t>(std::max(in.n_in, 1)) * ks);
            ws_.norm_part = lalloc<double>(ws_mem_, z.norm);
            ws_.dw_out = lalloc<float>(ws_mem_, N);
            // the base terms of as many ticks as there is memory for (one block's are N^2 floats
            // a tick; how many are made at a time changes no result)
            ws_.base = nullptr;
            for (ws_.base_ticks = kBaseTicks; !ws_.base; ws_.base_ticks /= 2) {
                void* p = nullptr;
                const size_t bytes = sizeof(float) * static_cast<size_t>(base_len_) * ws_.base_ticks;
                if (hipMalloc(&p, bytes) == hipSuccess) {
                    ws_mem_.push_back(p);
                    ws_.base = static_cast<float*>(p);
                    break;
                }
                (void)hipGetLastError();
                if (ws_.base_ticks == 1) throw HipFail("out of device memory for the base term");
            }
            // the padding of the X rows stays zero: only the columns themselves are written
            if (z.x) launch_fill_f32(ws_.x, 0.f, static_cast<long long>(z.x), stream_);
            ws_key_ = key;
        }
    } catch (const std::exception& e) {
        (void)hipGetLastError();          // not the next call's
        free_all(ws_mem_);
        ws_key_.clear();
        return fail("replay: %s", e.what());
    }
    return replay_on(in, ws_, sig, N);
}

LearnRuntime::Sizes LearnRuntime::sizes_for(int N, bool percise) const {
    Sizes z;
    const int row_tiles = rp_corr_row_tiles(N);
    const int ntiles = static_cast<int>(tiles_.size());
    z.R = percise ? k_len_ + 1 : 1;
    z.norm = static_cast<size_t>(std::max(ntiles * row_tiles, rp_finish_blocks(N)));
    if (percise) {
        const int splits = rp_corr_splits(N, ntiles, max_bnp_, k_len_);   // the most any window takes
        z.x = static_cast<size_t>(z.R) * N * xcols_;
        z.xscale = static_cast<size_t>(z.R) * xcols_ / 4;
        z.part = splits > 1 ? static_cast<size_t>(splits) * N * N : 0;
    }
    return z;
}

// The replay proper over signals sig[c] ((T, N) on the device) with the buffers of ws;
// it allocates nothing (with timing off).
int LearnRuntime::replay_on(const ReplayIn& in, const Workspace& ws, float* const* sig, int N) {
    const int K_len = k_len_;
    const int ks = in.ksteps;
    const bool need_dx = in.n_in > 0;
    try {
        const int R = in.percise ? K_len + 1 : 1;
        const size_t slice = static_cast<size_t>(N) * N;
        const long long xslice = static_cast<long long>(N) * xcols_;
        const int ntiles = static_cast<int>(tiles_.size());
        const int row_tiles = rp_corr_row_tiles(N);
        LRC(hipMemcpyAsync(ws.dl, in.dl, sizeof(float) * static_cast<size_t>(ks) * in.n_out, hipMemcpyHostToDevice,
                           stream_));
        LRC(hipMemcpyAsync(ws.po, in.po, sizeof(int) * in.n_out, hipMemcpyHostToDevice, stream_));
        LRC(hipMemcpyAsync(ws.pre, in.pre, sizeof(int) * N, hipMemcpyHostToDevice, stream_));
        if (need_dx) LRC(hipMemcpyAsync(ws.pin, in.pin, sizeof(int) * in.n_in, hipMemcpyHostToDevice, stream_));

        launch_fill_f32(ws.slices, 0.f, static_cast<long long>(slice), stream_);      // tick 0
        const int xgroups = static_cast<int>(xcols_ / 4);
        if (in.percise) {
            ReplayRangeArgs G{};
            G.N = N;
            G.ticks = ks;
            G.R = R;
            G.xgroups = xgroups;
            G.group_col = d_group_col_;
            G.dv = sig[1];
            G.dp = sig[2];
            G.xdown = ws.xdown;
            G.xscale = ws.xscale;
            launch_rp_range(G, stream_);
        }
        launch_fill_f32(ws.gs, static_cast<float>(in.grad_scale), 1, stream_);
        launch_fill_f32(ws.tick_scale, 1.f, 1, stream_);
        launch_fill_f32(ws.dw_acc, 0.f, N, stream_);
        if (need_dx) launch_fill_f32(ws.dx, 0.f, static_cast<long long>(in.n_in) * ks, stream_);

        const float dt = static_cast<float>(in.dt);
        const float eps = static_cast<float>(in.eps);
        const float thr = static_cast<float>(in.thr);
        corr_ms = 0;
        corr_launches = 0;
        std::vector<std::pair<hipEvent_t, hipEvent_t>> evs;

        ReplayTickArgs K{};
        K.N = N;
        K.norm_part = ws.norm_part;
        K.thr = thr;
        K.gs = ws.gs;
        K.xscale = ws.xscale;
        K.col_group = d_col_group_;
        K.xgroups = xgroups;
        K.R = R;
        K.tick_scale = ws.tick_scale;
        K.po = ws.po;
        K.n_out = in.n_out;
        K.w_tick = ws.w_tick;
        K.dw_acc = ws.dw_acc;
        K.xoff = d_xoff_;
        K.col_block = d_col_block_;
        K.start = d_start_;
        K.bnp = d_bnp_;
        K.pre = ws.pre;
        // X of tick t (from slice `cur` into its slot), read by the ticks after it
        auto with_x = [&](int t) {
            const bool need = in.percise && t < ks;
            K.x = need ? ws.x + static_cast<size_t>(t % R) * xslice : nullptr;
            K.xdown = need ? ws.xdown + static_cast<size_t>(t) * xgroups : nullptr;
            K.dv = need ? sig[1] + static_cast<size_t>(t + 1) * N : nullptr;
            K.dp = need ? sig[2] + static_cast<size_t>(t + 1) * N : nullptr;
        };
        K.cur = ws.slices;
        K.dl = nullptr;
        with_x(0);
        launch_rp_tick(K, stream_);

        ReplayDx X{};                     // dx of the tick before (none at the first)
        X.pin = ws.pin;
        X.w_tick = ws.w_tick;
        X.eps = eps;
        X.ksteps = ks;
        X.tick_scale = ws.tick_scale;
        X.dx = ws.dx;

        ReplayOut O{};
        O.N = N;
        O.dt = dt;
        O.gs = ws.gs;
        O.norm_part = ws.norm_part;

        for (int t_lr = 1; t_lr <= ks; ++t_lr) {
            const int tw = std::min(t_lr, K_len);
            const int cur = in.percise ? t_lr % R : 0;
            bool due = false;
            if (in.clip_strategy != 0) {
                if (in.cached_clip_rule) due = in.clip_strategy == 1 || (t_lr % in.clip_every) == 0;
                else due = in.clip_strategy == 1 && (t_lr % in.clip_every) == 0;
            }

            const int bt = (t_lr - 1) % ws.base_ticks;
            if (bt == 0) {
                ReplayBaseArgs B{};
                B.kp = d_kp_;
                B.koff = d_koff_;
                B.boff = d_boff_;
                B.start = d_start_;
                B.bn = d_bn_;
                B.bnp = d_bnp_;
                B.it = sig[0];
                B.N = N;
                B.T = ks + 1;
                B.K_len = K_len;
                B.t0 = t_lr;
                B.ng = std::min(ws.base_ticks, ks - t_lr + 1);
                B.base = ws.base;
                B.base_stride = base_len_;
                launch_rp_base(B, nblk_, max_bn_, stream_);
            }
            O.base = ws.base + static_cast<size_t>(bt) * base_len_;
            O.out = ws.slices + static_cast<size_t>(t_lr & 1) * slice;
            O.sanitize = due ? 1 : 0;

            const int nsplit = in.percise ? rp_corr_splits(N, ntiles, max_bnp_, tw) : 0;
            // timed: the GEMM and the sum of its splits, with the previous tick's dx ahead of
            // them (the same sums) instead of beside them
            hipEvent_t ev[2] = {nullptr, nullptr};
            if (timing) {
                launch_rp_dx(X, N, nsplit == 1 ? tile_cols_ : 0, stream_);
                X.n_in = 0;
                for (auto& e : ev) LRC(hipEventCreate(&e));
                evs.push_back({ev[0], ev[1]});
                LRC(hipEventRecord(ev[0], stream_));
            }
            if (in.percise) {
                ReplayCorrArgs C{};
                C.x = ws.x;
                C.xslice = xslice;
                C.xoff = d_xoff_;
                C.xscale = ws.xscale;
                C.xgroup = d_xgroup_;
                C.xgroups = xgroups;
                C.R = R;
                C.h0 = (t_lr - tw) % R;
                C.kp = d_kp_;
                C.koff = d_koff_;
                C.start = d_start_;
                C.bn = d_bn_;
                C.bnp = d_bnp_;
                C.boff = d_boff_;
                C.tiles = d_tiles_;
                C.row_tiles = row_tiles;
                C.nsplit = nsplit;
                C.ncorr = ntiles * row_tiles * nsplit;
                C.tw = tw;
                C.k_t0 = K_len - tw;
                C.part = ws.part;
                C.O = O;
                if (nsplit == 1) C.dx = X;
                launch_rp_corr(C, tile_cols_, stream_);
            }
            if (nsplit != 1) {
                ReplayFinishArgs F{};
                F.part = ws.part;
                F.nsplit = nsplit;
                F.col_block = d_col_block_;
                F.start = d_start_;
                F.bn = d_bn_;
                F.boff = d_boff_;
                F.O = O;
                F.dx = X;
                launch_rp_finish(F, stream_);
            }
            if (timing) LRC(hipEventRecord(ev[1], stream_));
            K.cur = O.out;
            K.due = due ? 1 : 0;
            K.npart = nsplit == 1 ? ntiles * row_tiles : rp_finish_blocks(N);
            K.cur_slot = cur;
            K.dl = ws.dl + static_cast<size_t>(t_lr - 1) * in.n_out;
            with_x(t_lr);
            launch_rp_tick(K, stream_);
            X.n_in = in.n_in;
            X.cur = O.out;
            X.t_idx = t_lr - 1;
            X.clip_ran = due ? 1 : 0;
        }
        launch_rp_dx(X, N, 0, stream_);
        // dw = dw_accum * (1 / ksteps) in fp32 (LearnRuntime.cpp:2281-2285)
        launch_rp_scale_into(ws.dw_acc, 1.0f / static_cast<float>(ks), ws.dw_out, N, stream_);
        LRC(hipStreamSynchronize(stream_));
        LRC(hipGetLastError());
        for (auto& pr : evs) {
            float ms = 0;
            LRC(hipEventElapsedTime(&ms, pr.first, pr.second));
            corr_ms += ms;
            corr_launches++;
            (void)hipEventDestroy(pr.first);
            (void)hipEventDestroy(pr.second);
        }
        LRC(hipMemcpy(in.dw_out, ws.dw_out, sizeof(float) * N, hipMemcpyDeviceToHost));
        if (need_dx)
            LRC(hipMemcpy(in.dx_out, ws.dx, sizeof(float) * static_cast<size_t>(in.n_in) * ks, hipMemcpyDeviceToHost));
    } catch (const std::exception& e) {
        return fail("replay: %s", e.what());
    }
    return 0;
}

// ---------------------------------------------------------------------------
// Replay without allocation: every device buffer of a host-signal replay is
// carved from one file-scope device array, `scratch`.  Each device holds its
// own copy; its address is looked up once per device with hipGetSymbolAddress
// (the array's name in host code is not a device address).  All calls on one
// device share it, so calls that overlap on one device race.
// ---------------------------------------------------------------------------
namespace {
constexpr int kScratchMaxDevices = 64;
__device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];
std::mutex scratch_mu;
unsigned char* scratch_dev[kScratchMaxDevices] = {};

// 256-byte aligned sub-allocations of the scratch array, in a fixed order; with
// base == nullptr it only measures.
struct Carver {
    unsigned char* base;
    size_t used = 0;
    template <class T>
    T* take(size_t n) {
        used = (used + 255) & ~static_cast<size_t>(255);
        T* p = base ? reinterpret_cast<T*>(base + used) : nullptr;
        used += std::max<size_t>(n, 1) * sizeof(T);
        return p;
    }
};
}  // namespace

// Address of this device's scratch array (looked up on the first call on each device).
unsigned char* noalloc_scratch() {
    int dev = 0;
    LRC(hipGetDevice(&dev));
    if (dev < 0 || dev >= kScratchMaxDevices) throw HipFail("device index out of range for the scratch table");
    std::lock_guard<std::mutex> lock(scratch_mu);
    if (!scratch_dev[dev]) {
        void* p = nullptr;
        LRC(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        scratch_dev[dev] = static_cast<unsigned char*>(p);
    }
    return scratch_dev[dev];
}

int LearnRuntime::replay_from_host_noalloc(const ReplayIn& in, const float* it_nt, const float* dv_nt,
                                           const float* dp_nt, int N, int T) {
    if (N <= 0 || T != in.ksteps + 1) return fail("replay: no signals of %d ticks", in.ksteps);
    try {
        const int nch = in.percise ? 3 : 1;
        const Sizes z = sizes_for(N, in.percise);
        const size_t slice = static_cast<size_t>(N) * N;
        const size_t sigsz = static_cast<size_t>(N) * T;
        const int ks = in.ksteps;
        // what is refused: two rings of slices (one without the precise term), the signals
        // and the vectors past the limit
        const size_t nwg = static_cast<size_t>(tiles_.size()) * rp_corr_row_tiles(N);
        Carver measure{nullptr};
        for (int ch = 0; ch <= nch; ++ch) measure.take<float>(sigsz);
        for (int ring = 0; ring < (in.percise ? 2 : 1); ++ring) measure.take<float>(slice * z.R);
        for (size_t n : {static_cast<size_t>(z.R), static_cast<size_t>(1), static_cast<size_t>(1),
                         static_cast<size_t>(N), static_cast<size_t>(N), static_cast<size_t>(ks) * in.n_out,
                         static_cast<size_t>(in.n_out), static_cast<size_t>(N),
                         static_cast<size_t>(std::max(in.n_in, 1)), static_cast<size_t>(std::max(in.n_in, 1)) * ks})
            measure.take<float>(n);
        measure.take<double>(nwg);
        measure.take<int>(nwg);
        measure.take<float>(N);
        if (measure.used > kNoAllocLimitBytes)
            return fail("replay needs %zu bytes of device scratch for N=%d, T=%d, K_len=%d%s; the allocation-free "
                        "entry point holds at most %zu bytes (use the allocating one)",
                        measure.used, N, T, k_len_, in.percise ? " (percise)" : "", kNoAllocLimitBytes);
        Workspace w;
        float* sig[kLrMaxChannels];
        float* stage = nullptr;
        // as many ticks' base terms as there is room for (they are made a few ticks at a
        // time; how many changes no result)
        auto carve = [&](Carver& c, int base_ticks) {
            stage = c.take<float>(sigsz);
            for (int ch = 0; ch < kLrMaxChannels; ++ch) sig[ch] = ch < nch ? c.take<float>(sigsz) : nullptr;
            w.slices = c.take<float>(2 * slice);
            w.x = c.take<float>(z.x);
            w.part = c.take<float>(z.part);
            w.base_ticks = base_ticks;
            w.base = c.take<float>(static_cast<size_t>(base_len_) * base_ticks);
            w.xscale = c.take<float>(z.xscale);
            w.xdown = c.take<unsigned char>(z.xscale ? static_cast<size_t>(ks) * xcols_ / 4 : 0);
            w.gs = c.take<float>(1);
            w.tick_scale = c.take<float>(1);
            w.w_tick = c.take<float>(N);
            w.dw_acc = c.take<float>(N);
            w.dl = c.take<float>(static_cast<size_t>(ks) * in.n_out);
            w.po = c.take<int>(in.n_out);
            w.pre = c.take<int>(N);
            w.pin = c.take<int>(std::max(in.n_in, 1));
            w.dx = c.take<float>(static_cast<size_t>(std::max(in.n_in, 1)) * ks);
            w.norm_part = c.take<double>(z.norm);
            w.dw_out = c.take<float>(N);
            return c.used;
        };
        int base_ticks = kBaseTicks;
        for (;; base_ticks /= 2) {
            Carver probe{nullptr};
            if (carve(probe, base_ticks) <= kNoAllocScratchBytes) break;
            if (base_ticks == 1) return fail("replay: the scratch array is too small for N=%d, T=%d", N, T);
        }
        Carver c{noalloc_scratch()};
        carve(c, base_ticks);
        if (z.x) launch_fill_f32(w.x, 0.f, static_cast<long long>(z.x), stream_);
        // (N, T) host signals -> (T, N) on the device, as load_signals does
        const float* src[kLrMaxChannels] = {it_nt, dv_nt, dp_nt};
        for (int ch = 0; ch < nch; ++ch) {
            LRC(hipMemcpyAsync(stage, src[ch], sigsz * sizeof(float), hipMemcpyHostToDevice, stream_));
            launch_transpose_nt_tn(stage, sig[ch], N, T, stream_);
        }
        const bool was_timing = timing;
        timing = false;                 // the timing path creates events
        const int rc = replay_on(in, w, sig, N);
        timing = was_timing;
        return rc;
    } catch (const std::exception& e) {
        return fail("replay: %s", e.what());
    }
}

}  // namespace hx
