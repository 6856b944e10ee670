// HIP kernels of the learn gradient surface for gfx950: learning-signal
// capture and the LRDS replay (replay_dw_dx.cu:9-731 is the reference's CUDA
// version of the same arithmetic).
//
// Per LR tick t (window tw = min(t, K_len), signal times it_t0 = t - tw + 1 ...
// t, kernel taps k_t0 = K_len - tw ... K_len - 1) the replay forms
//
//   dvtdw_t[i, s+j] = [i in block] (sum_u K_b[i-s][j][k_t0+u] It[it_t0+u][i]) dt gs
//                   + dt sum_{u,k} K_b[j][k][k_t0+u] X_{t-tw+u}[i, k]
//   X_tau[i, k] = dvtdw_tau[i, s+k] dIt/dv[tau+1][s+k]
//               + dvtdw_tau[i, pre(s+k)] dIt/dvpre[tau+1][s+k]
//
// (base term replay_dw_dx.cu:227-274, correction :282-325).  X_tau depends on its own
// tick alone, so it is formed once, when the tick's slice is done (k_rp_tick), and kept
// in a ring; the slices themselves are not kept.  The correction is a GEMM per block,
// (N x bn*tw) X times (bn*tw x bn) K on v_mfma_f32_32x32x2f32 (k_rp_corr), its reduction
// split over workgroups where the output alone does not fill the chip; k_rp_finish then
// adds the splits.  A tick is two or three launches: k_rp_corr (with the previous tick's
// dx on blocks of its own), k_rp_finish (splits, or no correction), k_rp_tick (clip
// decision, w_tick, dw, X).  The base term is made for kBaseTicks ticks at a time.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "learn.h"

namespace hx {
namespace {

typedef float f16v __attribute__((ext_vector_type(16)));

constexpr int kThreads = 256;

// ---------------------------------------------------------------- capture
// batch_gather.cu:5-10 and batch_scatter_add.cu:4-13: outputs are gathered
// every step; every k_mul steps each channel's items are rounded to fp32,
// multiplied by their scale and summed per destination column.  Items of one
// column are summed in input order (the reference's atomics leave that order
// open), so the result is reproducible.
__global__ void k_lr_capture(CaptureArgs C, int sample, int lr) {
    int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g < C.n_out) {
        C.out_vs[static_cast<size_t>(sample) * C.n_out + g] = static_cast<float>(*C.out_ptr[g]);
        return;
    }
    if (lr <= 0) return;
    g -= C.n_out;
    const int ch = g / max(C.N, 1);
    const int col = g - ch * C.N;
    if (ch >= C.nch) return;
    const CaptureChannel& Q = C.ch[ch];
    float acc = 0.f;
    for (int q = Q.begin[col]; q < Q.begin[col + 1]; ++q)
        acc = __fadd_rn(acc, __fmul_rn(static_cast<float>(*Q.ptr[q]), Q.scale[q]));
    Q.buf[static_cast<size_t>(lr) * C.N + col] = acc;
}

// ---------------------------------------------------------------- base term
// replay_base_blocks_kernel (replay_dw_dx.cu:227-274): one thread per (i, j) of a
// diagonal block and kBaseTicks ticks, taps summed in time order with fused multiply-adds.
// The taps (64 MB for 16 blocks of 128 and K_len 64) are read once for all those ticks:
// 16 us a tick when made tick by tick, 2.6 us now.
__global__ void __launch_bounds__(kThreads) k_rp_base(ReplayBaseArgs A) {
    const int b = blockIdx.y;
    const int bn = A.bn[b], bnp = A.bnp[b];
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= bn * bn) return;
    const int bi = e / bn;
    const int row = A.start[b] + bi;
    const float* K = A.kp + A.koff[b] + static_cast<size_t>(bi) * bnp + (e - bi * bn);
    const size_t plane = static_cast<size_t>(bn) * bnp;
    float sum[kBaseTicks];
#pragma unroll
    for (int g = 0; g < kBaseTicks; ++g) sum[g] = 0.f;
    // tap k0 + p of tick t0 + g meets the signal at time tau0 + p + g: a group of kBaseTicks
    // taps needs 2 kBaseTicks - 1 signals, of which the last group brought the first half.
    // Times before the first signal (and taps past the last) are skipped, so whatever is
    // loaded in their place is not used.
    const int first = A.t0 + A.ng - 1 < A.K_len ? A.K_len - (A.t0 + A.ng - 1) : 0;
    auto signal = [&](int tau) { return A.it[static_cast<size_t>(min(max(tau, 0), A.T - 1)) * A.N + row]; };
    float w[2 * kBaseTicks];
#pragma unroll
    for (int g = 0; g < kBaseTicks; ++g) w[kBaseTicks + g] = signal(A.t0 + first - A.K_len + 1 + g);
    for (int k0 = first; k0 < A.K_len; k0 += kBaseTicks) {
        const int tau0 = A.t0 + k0 - A.K_len + 1;
        float k[kBaseTicks];
#pragma unroll
        for (int p = 0; p < kBaseTicks; ++p) {
            k[p] = K[min(k0 + p, A.K_len - 1) * plane];
            w[p] = w[kBaseTicks + p];
            w[kBaseTicks + p] = signal(tau0 + kBaseTicks + p);
        }
#pragma unroll
        for (int p = 0; p < kBaseTicks; ++p)
#pragma unroll
            for (int g = 0; g < kBaseTicks; ++g)
                if (k0 + p < A.K_len && tau0 + p + g >= 1) sum[g] = fmaf(k[p], w[p + g], sum[g]);
    }
#pragma unroll
    for (int g = 0; g < kBaseTicks; ++g)
        if (g < A.ng) A.base[g * A.base_stride + A.boff[b] + e] = sum[g];
}

// Fixed-order sum over the workgroup (kT threads) of x; every thread gets it.
template <int kT, class V>
__device__ __forceinline__ V block_sum(V x, V* sh) {
    const int tid = threadIdx.x;
    sh[tid] = x;
    __syncthreads();
#pragma unroll
    for (int st = kT / 2; st > 0; st >>= 1) {
        if (tid < st) sh[tid] += sh[tid + st];
        __syncthreads();
    }
    const V r = sh[0];
    __syncthreads();
    return r;
}

// One element of a tick's slice from its correction sum c (replay_dw_dx.cu:227-325): base
// term added inside the row's own block; on clip ticks non-finite entries become 0 and the
// square goes to the norm.
template <class Base>
__device__ __forceinline__ float rp_element(const ReplayOut& O, float c, int row, int col, int s, int bn,
                                            const Base& base, float gs, double& sq) {
    float v = c * O.dt;
    if (row >= s && row < s + bn) v = base()[static_cast<size_t>(row - s) * bn + col - s] * O.dt * gs + v;
    if (O.sanitize) {
        if (!isfinite(v)) v = 0.f;
        sq += static_cast<double>(v) * v;
    }
    return v;
}

// ---------------------------------------------------------------- dx
// replay_dx_reduce_kernel / replay_dx_finalize_kernel (replay_dw_dx.cu:445-501): one
// workgroup per input column, fixed-order reduction.  A clip at that tick also rescales
// the input's earlier dx entries (LearnRuntime.cpp:2257).  A tick's dx needs the whole
// w_tick, so it rides on the next tick's first launch (a launch of its own: 3.2-5.3 us).
template <int kT>
__device__ __forceinline__ void rp_dx(const ReplayDx& X, int N, int j, float* sh) {
    const int tid = threadIdx.x;
    const int p = X.pin[j];
    const float sig = X.clip_ran ? *X.tick_scale : 1.f;
    float s = 0.f, bsum = 0.f;
    for (int i = tid; i < N; i += kT) {
        const float v = X.cur[static_cast<size_t>(i) * N + p] * sig;
        bsum += v;
        s += X.w_tick[i] / (v + X.eps);
    }
    const float st = block_sum<kT>(s, sh);
    const float bt = block_sum<kT>(bsum, sh);
    float* row = X.dx + static_cast<size_t>(j) * X.ksteps;
    if (X.clip_ran && sig != 1.f)
        for (int t = tid; t < X.t_idx; t += kT) row[t] *= sig;
    if (tid == 0) row[X.t_idx] = st * bt;
}

template <int kT>
__global__ void __launch_bounds__(kT) k_rp_dx(ReplayDx X, int N) {
    __shared__ float sh[kT];
    rp_dx<kT>(X, N, blockIdx.x, sh);
}

// ---------------------------------------------------------------- correction GEMM
// Workgroup tile: kTI rows x TJ columns of one block over a range of the reduction,
// kT threads, one 32 x (TJ/WC) sub-tile per wave.  The reduction index runs over (tap u,
// column k of the block padded to a multiple of 4), flattened, in chunks of kKC, so narrow
// blocks fill a chunk with several taps.  A chunk's X rows and taps are read as 16-byte
// groups (X ring and taps are both k-contiguous and padded with zeros, so nothing needs a
// mask but the end of the range), held in registers while the previous chunk's MFMAs run
// and staged through LDS, double-buffered; rows are kKC + 4 floats apart, which spreads a
// wave's ds_read_b128 over all banks.  Each such read feeds four MFMAs: which of the four
// k a step takes is the same for both operands.
// Bound: the fp32 matrix cores (157 TFLOP/s; a library product of 8192^3 reaches 153).
// N = 2048 in 16 blocks of 128, K_len 64, 256 ticks: 725 -> 508 us a launch, 118.7 TFLOP/s
// (before: X formed while staging from two history rings, one element per load).  Chunks of
// 32 with two workgroups per CU: 3% slower.
constexpr int kTI = 128;
constexpr int kKC = 64;
constexpr int kLd = kKC + 4;

template <int TJ>
struct CorrShape {
    static constexpr int kT = TJ == 32 ? 256 : 512;     // threads
    static constexpr int NW = kT / 64;
    static constexpr int WC = TJ == 32 ? 1 : 2;         // column groups of waves
    static constexpr int WR = NW / WC;                  // row groups: 32 rows each
    static constexpr int NC = TJ / WC / 32;             // accumulators per wave
    static constexpr int RS = kT / (kKC / 4);           // rows apart that a thread stages
    static constexpr int GA = kTI * kKC / 4 / kT;       // 16-byte groups of X per thread and chunk
    static constexpr int GB = TJ * kKC / 4 / kT;        // and of taps
    static_assert(WR * 32 == kTI && NC >= 1 && GA >= 1 && GB >= 1, "tile does not divide over the waves");
};

// kPart: write the sums of this split to the partials; otherwise the tick's slice itself.
template <int TJ, bool kPart>
__global__ void __launch_bounds__(CorrShape<TJ>::kT) k_rp_corr(ReplayCorrArgs A) {
    using S = CorrShape<TJ>;
    __shared__ __align__(16) float As[2][kTI][kLd];
    __shared__ __align__(16) float Bs[2][TJ][kLd];
    __shared__ double red_s[S::NW];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    int wg = static_cast<int>(blockIdx.x + blockIdx.y * gridDim.x);
    if (wg >= A.ncorr) {                                      // the previous tick's dx
        if (wg < A.ncorr + A.dx.n_in) rp_dx<S::kT>(A.dx, A.O.N, wg - A.ncorr, &As[0][0][0]);
        return;
    }
    // workgroups go to the eight XCDs in turn: give each XCD a run of consecutive tiles, so
    // the row tiles that share a block's taps read them from one L2
    if (A.ncorr % 8 == 0) wg = (wg & 7) * (A.ncorr >> 3) + (wg >> 3);
    const int rt = wg % A.row_tiles;
    const int q = wg / A.row_tiles;
    const int sp = q % A.nsplit;
    const int2 tl = A.tiles[q / A.nsplit];
    const int b = tl.x, j0 = tl.y;
    const int s = A.start[b], bn = A.bn[b], bnp = A.bnp[b];
    const int N = A.O.N;
    const int i0 = rt * kTI;
    const int nb4 = bnp >> 2;
    const int total = A.tw * nb4;                             // 16-byte groups of the reduction
    const int nchunk = (total + kKC / 4 - 1) / (kKC / 4);
    const int c0 = static_cast<int>(static_cast<long long>(nchunk) * sp / A.nsplit);
    const int c1 = static_cast<int>(static_cast<long long>(nchunk) * (sp + 1) / A.nsplit);

    const int kg = tid % (kKC / 4), r0 = tid / (kKC / 4);     // group within the chunk, first row
    const float* Xb = A.x + static_cast<long long>(A.xoff[b]);
    const int xgroup = A.xgroup[b];
    const float* Kb = A.kp + A.koff[b];
    typedef float f4 __attribute__((ext_vector_type(4)));
    f4 ra[S::GA], rb[S::GB];
    float sig = 0.f;
    bool in = false;
    // only loads here: the first use of what they bring is in stage(), behind the MFMAs
    auto fetch = [&](int c) {
        const int pos = c * (kKC / 4) + kg;
        const int u = pos / nb4;
        const int k4 = pos - u * nb4, k = k4 * 4;
        in = pos < total;
        int h = A.h0 + (in ? u : 0);
        if (h >= A.R) h -= A.R;
        sig = A.xscale[h * A.xgroups + xgroup + (in ? k4 : 0)];
        const float* X = Xb + h * A.xslice + (in ? k : 0);
        const float* K = Kb + static_cast<size_t>(A.k_t0 + (in ? u : 0)) * bn * bnp + (in ? k : 0);
#pragma unroll
        for (int r = 0; r < S::GA; ++r) {
            const int i = min(i0 + r0 + S::RS * r, N - 1);
            // the history streams through once per tick: keep it out of the caches, so that
            // the taps, reused by every row tile, stay in L2
            ra[r] = __builtin_nontemporal_load(reinterpret_cast<const f4*>(X + static_cast<size_t>(i) * bnp));
        }
#pragma unroll
        for (int r = 0; r < S::GB; ++r) {
            const int j = min(j0 + r0 + S::RS * r, bn - 1);
            rb[r] = *reinterpret_cast<const f4*>(K + static_cast<size_t>(j) * bnp);
        }
    };
    auto stage = [&](int buf) {
        const f4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int r = 0; r < S::GA; ++r)
            *reinterpret_cast<f4*>(&As[buf][r0 + S::RS * r][kg * 4]) = in ? ra[r] * sig : zero;
#pragma unroll
        for (int r = 0; r < S::GB; ++r)
            *reinterpret_cast<f4*>(&Bs[buf][r0 + S::RS * r][kg * 4]) = in ? rb[r] : zero;
    };

    const int wr = wave / S::WC, wc = wave % S::WC;
    f16v acc[S::NC];
#pragma unroll
    for (int n = 0; n < S::NC; ++n)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[n][r] = 0.f;
    if (c1 > c0) {
        fetch(c0);
        stage(0);
        __syncthreads();
        const int kr = (lane >> 5) * 4;
        const int ia = wr * 32 + (lane & 31);
        const int jb = wc * 32 * S::NC + (lane & 31);
        for (int c = c0; c < c1; ++c) {
            const int buf = (c - c0) & 1;
            if (c + 1 < c1) fetch(c + 1);
#pragma unroll
            for (int g = 0; g < kKC / 8; ++g) {
                const float4 av = *reinterpret_cast<const float4*>(&As[buf][ia][8 * g + kr]);
                float4 bv[S::NC];
#pragma unroll
                for (int n = 0; n < S::NC; ++n)
                    bv[n] = *reinterpret_cast<const float4*>(&Bs[buf][jb + 32 * n][8 * g + kr]);
                const float a4[4] = {av.x, av.y, av.z, av.w};
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int n = 0; n < S::NC; ++n) {
                        const float b4[4] = {bv[n].x, bv[n].y, bv[n].z, bv[n].w};
                        acc[n] = __builtin_amdgcn_mfma_f32_32x32x2f32(a4[e], b4[e], acc[n], 0, 0, 0);
                    }
            }
            if (c + 1 < c1) stage(buf ^ 1);
            __syncthreads();
        }
    }

    // accumulator n of a lane holds rows 8(r/4) + 4(lane/32) + r%4 and column 32n + lane%32
    // of its wave's sub-tile
    double sq = 0.0;
    const float gs = *A.O.gs;
    const float* base_b = A.O.base + A.boff[b];
    auto base = [&] { return base_b; };
    float* out = kPart ? A.part + static_cast<size_t>(sp) * N * N : A.O.out;
#pragma unroll
    for (int n = 0; n < S::NC; ++n) {
        const int jw = j0 + (wc * S::NC + n) * 32 + (lane & 31);
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int row = i0 + wr * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
            if (row >= N || jw >= bn) continue;
            out[static_cast<size_t>(row) * N + s + jw] =
                kPart ? acc[n][r] : rp_element(A.O, acc[n][r], row, s + jw, s, bn, base, gs, sq);
        }
    }
    if (!kPart && A.O.sanitize) {
        for (int o = 32; o > 0; o >>= 1) sq += __shfl_xor(sq, o);
        if (lane == 0) red_s[wave] = sq;
        __syncthreads();
        if (tid == 0) {
            double t = 0.0;
            for (int w = 0; w < S::NW; ++w) t += red_s[w];
            A.O.norm_part[wg] = t;
        }
    }
}

constexpr int kFinishMost = 16;     // elements a thread of k_rp_finish takes at once, at most
constexpr int kFinishBlocks = 4096; // blocks of it, at most
// Row and column of the element kThreads after the one they hold.  A division costs as much
// as the rest of an element (64 bits: more), so slices wider than kThreads step instead.
template <class I>
__device__ __forceinline__ void next_element(I N, I& row, I& col) {
    col += kThreads;
    if (col >= N) {
        col -= N;
        ++row;
    }
}

// The tick's slice from the correction's split sums, added in split order (nsplit 0: no
// correction), kE elements per thread; the previous tick's dx on blocks of its own.  The
// splits are read four at a time, so a thread has 4 kE loads in flight (5.2 us at N = 400
// with 16 splits); the block look-ups of a thread's columns are in flight together too (a
// division, a look-up and a store one element after the other: 4.2 ms at N = 32768 without
// splits, now 1.4; the 4.3 GB written take 0.85).  I indexes the N x N elements: unsigned,
// or 64 bits from about N = 65400.
template <int kE, class I>
__global__ void __launch_bounds__(kThreads) k_rp_finish(ReplayFinishArgs A) {
    __shared__ double sh[kThreads];
    if (static_cast<int>(blockIdx.x) >= A.nblock) {
        rp_dx<kThreads>(A.dx, A.O.N, blockIdx.x - A.nblock, reinterpret_cast<float*>(sh));
        return;
    }
    const I N = A.O.N, total = N * N;
    const float gs = *A.O.gs;
    double sq = 0.0;
    // one turn but for the largest slices, whose blocks are bounded (rp_finish_blocks)
    for (I e0 = static_cast<I>(blockIdx.x) * kE * kThreads + threadIdx.x; e0 < total;
         e0 += static_cast<I>(A.nblock) * kE * kThreads) {
        float c[kE];
        I at[kE];
#pragma unroll
        for (int r = 0; r < kE; ++r) {
            c[r] = 0.f;
            at[r] = min(e0 + r * kThreads, total - 1);
        }
        int sp = 0;
        for (; sp + 4 <= A.nsplit; sp += 4) {
            float x[4][kE];
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int r = 0; r < kE; ++r) x[q][r] = A.part[static_cast<size_t>(sp + q) * total + at[r]];
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int r = 0; r < kE; ++r) c[r] += x[q][r];
        }
        for (; sp < A.nsplit; ++sp)
#pragma unroll
            for (int r = 0; r < kE; ++r) c[r] += A.part[static_cast<size_t>(sp) * total + at[r]];
        I row[kE], col[kE];
        int b[kE], s[kE], bn[kE];
        row[0] = e0 / N;
        col[0] = e0 - row[0] * N;
#pragma unroll
        for (int r = 0; r < kE; ++r) {
            if (r > 0) {
                row[r] = row[r - 1];
                col[r] = col[r - 1];
                next_element<I>(N, row[r], col[r]);
            }
            b[r] = A.col_block[col[r]];
        }
#pragma unroll
        for (int r = 0; r < kE; ++r) {
            s[r] = A.start[b[r]];
            bn[r] = A.bn[b[r]];
        }
#pragma unroll
        for (int r = 0; r < kE; ++r)
            if (e0 + r * kThreads < total)
                A.O.out[at[r]] = rp_element(A.O, c[r], row[r], col[r], s[r], bn[r],
                                            [&] { return A.O.base + A.boff[b[r]]; }, gs, sq);
        if constexpr (kE < kFinishMost) break;
    }
    if (A.O.sanitize) {
        const double t = block_sum<kThreads>(sq, sh);
        if (threadIdx.x == 0) A.O.norm_part[blockIdx.x] = t;
    }
}

// ---------------------------------------------------------------- X's range
// X is formed before the clip factors of its own and of later ticks are known, so it has to
// hold products that only those factors bring back into fp32's range.  Each 16-byte group
// of columns keeps X 2^-down, down from the group's largest signal, and 2^down times the
// factors so far meets it when the correction reads X.  |X 2^-down| stays at or below |D|
// (but for signals and slices both above 2^126), and a power of two changes no bit of a
// normal number; beside a signal of 2^e, its three neighbours lose what lies below
// 2^(e - 148).  Cost at N = 2048: k_rp_corr 447.6 -> 449.4 us, k_rp_tick 16.3 -> 17.1; with
// a scale per column, 16 bytes to read beside X's 16, k_rp_corr 452 to 455.  This kernel makes down for every tick and sets the
// ring's scales to 1.
__global__ void __launch_bounds__(kThreads) k_rp_range(ReplayRangeArgs A) {
    const long long ndown = static_cast<long long>(A.ticks) * A.xgroups;
    const long long n = ndown > static_cast<long long>(A.R) * A.xgroups ? ndown : static_cast<long long>(A.R) * A.xgroups;
    for (long long i = static_cast<long long>(blockIdx.x) * kThreads + threadIdx.x; i < n;
         i += static_cast<long long>(gridDim.x) * kThreads) {
        if (i < static_cast<long long>(A.R) * A.xgroups) A.xscale[i] = 1.f;
        if (i >= ndown) continue;
        const int t = static_cast<int>(i / A.xgroups), g = static_cast<int>(i - static_cast<long long>(t) * A.xgroups);
        const size_t at = static_cast<size_t>(t + 1) * A.N + A.group_col[g].x;
        int down = 0;
        for (int c = 0; c < A.group_col[g].y; ++c) {
            const float m = fmaxf(fabsf(A.dv[at + c]), fabsf(A.dp[at + c]));
            if (m >= 0.25f && isfinite(m)) down = max(down, min(ilogbf(m) + 2, 127));
        }
        A.xdown[i] = static_cast<unsigned char>(down);
    }
}

// ---------------------------------------------------------------- a tick's end
// The Frobenius clip (replay_frobenius_*_kernel replay_dw_dx.cu:28-93, the driver's
// decision LearnRuntime.cpp:2238-2262): l2 over the finite entries; above the threshold
// the tick's slice, the history, the accumulators and the grad scale are all multiplied
// by thr / l2.  Every workgroup that needs the factor sums the norm's partials itself, in
// the same order (a launch of its own took 4 us); block 0 stores it, and all rescale their
// share of the history's scales, which only later launches read.  w_tick
// (replay_dw_dx.cu:96-114): one wave per row.  The remaining blocks form X of this tick
// from its slice.
template <int kGather, class I>
__global__ void __launch_bounds__(kThreads) k_rp_tick(ReplayTickArgs A) {
    __shared__ double sh[kThreads];
    const int tid = threadIdx.x;
    const unsigned N = A.N;
    if (static_cast<int>(blockIdx.x) >= A.wblocks) {
        const I total = static_cast<I>(N) * N;
        const I e0 = static_cast<I>(blockIdx.x - A.wblocks) * kGather * kThreads + tid;
        I row = e0 / static_cast<I>(N), c = e0 - row * N;
#pragma unroll
        for (int r = 0; r < kGather; ++r) {
            const I e = e0 + r * kThreads;
            if (e >= total) break;
            if constexpr (sizeof(I) == 8) {
                if (r > 0) next_element<I>(N, row, c);
            } else {
                row = e / N;
                c = e - row * N;
            }
            const int p = A.pre[c], b = A.col_block[c];
            const float g = p >= 0 ? A.cur[static_cast<size_t>(row) * N + p] : 0.f;
            const int down = A.xdown[A.col_group[c]];
            A.x[A.xoff[b] + static_cast<size_t>(row) * A.bnp[b] + c - A.start[b]] =
                A.cur[e] * ldexpf(A.dv[c], -down) + g * ldexpf(A.dp[c], -down);
        }
        return;
    }
    // the exponent is asked for ahead of the norm: its latency would follow the sum's
    const int g0 = blockIdx.x * kThreads + tid;
    const int down0 = A.x && g0 < A.xgroups ? A.xdown[g0] : 0;
    float sc = 1.f;
    if (A.due) {
        double acc = 0.0;
        for (int q = tid; q < A.npart; q += kThreads) acc += A.norm_part[q];
        const double l2 = sqrt(fmax(0.0, block_sum<kThreads>(acc, sh)));
        if (l2 > static_cast<double>(A.thr) && isfinite(l2)) sc = static_cast<float>(static_cast<double>(A.thr) / l2);
    }
    if (blockIdx.x == 0) {
        if (A.due && tid == 0) {
            *A.tick_scale = sc;
            if (sc != 1.f) *A.gs *= sc;
        }
    }
    if (A.x) {                                                // the scales of X's groups
        const int here = A.cur_slot * A.xgroups, stride = A.wblocks * kThreads;
        for (int g = g0; g < A.xgroups; g += stride) A.xscale[here + g] = ldexpf(sc, g == g0 ? down0 : A.xdown[g]);
        if (sc != 1.f)
            for (int q = g0; q < A.R * A.xgroups; q += stride)
                if (q < here || q >= here + A.xgroups) A.xscale[q] *= sc;
    }
    const unsigned row = blockIdx.x * (kThreads / 64) + (tid >> 6);
    const int lane = tid & 63;
    if (row >= N) return;
    const float* r = A.cur + static_cast<size_t>(row) * N;
    float acc = 0.f;
    for (int o = lane; o < A.n_out; o += 64) acc = fmaf(r[A.po[o]] * sc, A.dl[o], acc);
    for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o);
    if (lane == 0) {
        A.w_tick[row] = acc;
        A.dw_acc[row] = A.dw_acc[row] * sc + acc;
    }
}

__global__ void k_rp_scale_into(const float* src, float scale, float* dst, long long n) {
    const long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n) dst[i] = src[i] * scale;
}

__global__ void k_fill_f32(float* p, float v, long long n) {
    for (long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
         i += static_cast<long long>(gridDim.x) * blockDim.x)
        p[i] = v;
}

// (N, T) -> (T, N) through a 32 x 33 LDS tile
__global__ void k_transpose_nt_tn(const float* src, float* dst, int N, int T) {
    __shared__ float tile[32][33];
    const int t = blockIdx.x * 32 + threadIdx.x;
    const int n = blockIdx.y * 32 + threadIdx.y;
    if (n < N && t < T) tile[threadIdx.y][threadIdx.x] = src[static_cast<size_t>(n) * T + t];
    __syncthreads();
    const int n2 = blockIdx.y * 32 + threadIdx.x;
    const int t2 = blockIdx.x * 32 + threadIdx.y;
    if (n2 < N && t2 < T) dst[static_cast<size_t>(t2) * N + n2] = tile[threadIdx.x][threadIdx.y];
}

}  // namespace

void launch_lr_capture(const CaptureArgs& a, int sample, int lr, hipStream_t s) {
    const long long n = a.n_out + (lr > 0 ? static_cast<long long>(a.nch) * a.N : 0);
    if (n <= 0) return;
    hipLaunchKernelGGL(k_lr_capture, dim3(static_cast<unsigned>((n + kThreads - 1) / kThreads)), dim3(kThreads), 0,
                       s, a, sample, lr);
}

void launch_rp_base(const ReplayBaseArgs& a, int nblk, int max_bn, hipStream_t s) {
    const long long e = static_cast<long long>(max_bn) * max_bn;
    hipLaunchKernelGGL(k_rp_base, dim3(static_cast<unsigned>((e + kThreads - 1) / kThreads), nblk), dim3(kThreads),
                       0, s, a);
}

int rp_corr_row_tiles(int N) { return (N + kTI - 1) / kTI; }

// Workgroups the reduction is split over: enough for one on every CU, as long as each
// keeps a chunk.  Problem sizes alone decide, so every entry point sums in the same order.
// N = 96, K_len 8: 34 -> 6 us a launch (2 tiles, one workgroup each before); N = 701,
// K_len 24: 307 -> 32 us (36 tiles); N = 2048 has a tile per CU and is not split.
int rp_corr_splits(int N, int ntiles, int max_bnp, int tw) {
    const int wgs = ntiles * rp_corr_row_tiles(N);
    const long long chunks = (static_cast<long long>(tw) * max_bnp + kKC - 1) / kKC;
    const long long want = std::min<long long>(256 / std::max(wgs, 1), chunks);
    return static_cast<int>(std::max<long long>(want, 1));
}

template <int TJ>
void launch_corr_tile(const ReplayCorrArgs& a, hipStream_t s) {
    // a launch holds less than 2^32 threads along x: many workgroups take rows of kCorrRow
    // (a multiple of the XCD count, so the mapping to them stays)
    const int total = a.ncorr + a.dx.n_in;
    constexpr int kCorrRow = 1 << 20;
    const dim3 grid(std::min(total, kCorrRow), (total + kCorrRow - 1) / kCorrRow), block(CorrShape<TJ>::kT);
    if (a.nsplit > 1) hipLaunchKernelGGL((k_rp_corr<TJ, true>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((k_rp_corr<TJ, false>), grid, block, 0, s, a);
}

void launch_rp_corr(const ReplayCorrArgs& a, int tile_cols, hipStream_t s) {
    if (tile_cols == 128) launch_corr_tile<128>(a, s);
    else if (tile_cols == 64) launch_corr_tile<64>(a, s);
    else launch_corr_tile<32>(a, s);
}

// Elements per thread of k_rp_finish: one while that gives no more than about 1024 blocks
// (every w_tick workgroup adds up the blocks' norm partials), then as many as keep it so, up
// to kFinishMost in kFinishBlocks blocks that then take turns.
static int finish_elems(int N) {
    const long long blocks = (static_cast<long long>(N) * N + kThreads - 1) / kThreads;
    return blocks <= 1024 ? 1 : blocks <= 4096 ? 4 : blocks <= 16384 ? 8 : kFinishMost;
}

int rp_finish_blocks(int N) {
    const long long per = static_cast<long long>(finish_elems(N)) * kThreads;
    return static_cast<int>(std::min<long long>((static_cast<long long>(N) * N + per - 1) / per, kFinishBlocks));
}

// The N x N elements are indexed in 32 bits: so must be what a block's next turn starts at.
static bool narrow_slice(int N) {
    const long long turn = static_cast<long long>(kFinishBlocks) * kFinishMost * kThreads;
    return static_cast<long long>(N) * N + turn < 1LL << 32;
}

void launch_rp_finish(ReplayFinishArgs a, hipStream_t s) {
    a.nblock = rp_finish_blocks(a.O.N);
    const dim3 grid(a.nblock + a.dx.n_in);
    auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, dim3(kThreads), 0, s, a); };
    switch (finish_elems(a.O.N)) {
        case 1: go(k_rp_finish<1, unsigned>); break;
        case 4: go(k_rp_finish<4, unsigned>); break;
        case 8: go(k_rp_finish<8, unsigned>); break;
        default:
            if (narrow_slice(a.O.N)) go(k_rp_finish<kFinishMost, unsigned>);
            else go(k_rp_finish<kFinishMost, unsigned long long>);
    }
}

void launch_rp_range(const ReplayRangeArgs& a, hipStream_t s) {
    const long long n = static_cast<long long>(std::max(a.ticks, a.R)) * a.xgroups;
    const long long blocks = std::min<long long>((n + kThreads - 1) / kThreads, 4096);
    hipLaunchKernelGGL(k_rp_range, dim3(static_cast<unsigned>(blocks)), dim3(kThreads), 0, s, a);
}

void launch_rp_tick(ReplayTickArgs a, hipStream_t s) {
    a.wblocks = a.dl ? (a.N + kThreads / 64 - 1) / (kThreads / 64) : 0;
    auto go = [&](auto kernel, int elems) {
        const long long per = static_cast<long long>(elems) * kThreads;
        const long long gather = a.x ? (static_cast<long long>(a.N) * a.N + per - 1) / per : 0;
        if (a.wblocks + gather > 0)
            hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(a.wblocks + gather)), dim3(kThreads), 0, s, a);
    };
    // wide slices: enough elements a thread that the launch holds less than 2^32 of them
    if (narrow_slice(a.N)) go(k_rp_tick<4, unsigned>, 4);
    else go(k_rp_tick<16, unsigned long long>, 16);
}

// as k_rp_corr's blocks do it (their size sets the order of the sums) or as k_rp_finish's
void launch_rp_dx(const ReplayDx& a, int N, int corr_tile_cols, hipStream_t s) {
    if (a.n_in <= 0) return;
    static_assert(CorrShape<128>::kT == 512 && CorrShape<64>::kT == 512 && CorrShape<32>::kT == kThreads);
    if (corr_tile_cols >= 64) hipLaunchKernelGGL(k_rp_dx<512>, dim3(a.n_in), dim3(512), 0, s, a, N);
    else hipLaunchKernelGGL(k_rp_dx<kThreads>, dim3(a.n_in), dim3(kThreads), 0, s, a, N);
}

void launch_rp_scale_into(const float* src, float scale, float* dst, long long n, hipStream_t s) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_rp_scale_into, dim3(static_cast<unsigned>((n + kThreads - 1) / kThreads)), dim3(kThreads),
                       0, s, src, scale, dst, n);
}

void launch_fill_f32(float* p, float v, long long n, hipStream_t s) {
    if (n <= 0) return;
    const long long blocks = std::min<long long>((n + kThreads - 1) / kThreads, 4096);
    hipLaunchKernelGGL(k_fill_f32, dim3(static_cast<unsigned>(blocks)), dim3(kThreads), 0, s, p, v, n);
}

void launch_transpose_nt_tn(const float* src_nt, float* dst_tn, int N, int T, hipStream_t s) {
    if (N <= 0 || T <= 0) return;
    hipLaunchKernelGGL(k_transpose_nt_tn, dim3((T + 31) / 32, (N + 31) / 32), dim3(32, 32), 0, s, src_nt, dst_tn, N,
                       T);
}

}  // namespace hx
