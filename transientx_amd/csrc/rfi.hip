// rfi.hip -- RFI cleaning of channel x time frames on the device:
// Candidate::zdot (zero-DM matched filter) and Candidate::kadaneF
// (src/singlepulse/candidate.cpp:710-897), the formulas behind the front
// end's "zdot" and "kadaneF" items (src/singlepulse/singlepulse.cpp:305-317).
//
// A frame is nchan x nsamp floats; element (channel j, sample i) of frame f
// is x[f*fstride + j*cstride + i*tstride], so one kernel serves the
// Candidate layout [nchan][nbin] (cstride = nsamp, tstride = 1) and a
// DataBuffer block [nsamp][nchans] (cstride = 1, tstride = nchans).
//
// The arithmetic is the reference's, operation by operation: FP64
// accumulations in its sequential order (one thread per channel or per
// sample), float products where it multiplies floats, float stores where it
// assigns to float, and fused multiply-adds exactly where its build
// (g++ -O3 -mavx2 -mfma, config/ax_check_x86_features.m4:76) contracts:
// a*b + c and c - a*b fuse; in a*b - c*d the second product is rounded
// first and the first is fused; a float product added to a double is not
// fused.  Nothing else is contracted (fp contract off).  Results are
// bit-identical to the oracle's restatement.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <string>

#include "../../include/txgpu.h"
#include "device_util.h"

#pragma clang fp contract(off)

namespace txgpu {
int set_error(int code, const std::string &msg);
}
using txgpu::lds_fill;
using txgpu::lds_fill16;
using txgpu::set_error;

namespace {

struct Frames {
    float *x;
    long fstride, cstride, tstride;
    int nframes, nchan;
    long nsamp;
    __device__ float &at(long f, long j, long i) const { return x[f * fstride + j * cstride + i * tstride]; }
};

// zdot 1: per (frame, channel) mean and standard deviation over the samples
// (candidate.cpp:837-851), then the channel normalised in place (:853-859)
__global__ void k_zdot_norm(Frames F)
{
    const long g = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= (long)F.nframes * F.nchan) return;
    const long f = g / F.nchan, j = g % F.nchan;
    double m = 0., sd = 0.;
    for (long i = 0; i < F.nsamp; i++) {
        const float v = F.at(f, j, i);
        m += v;
        sd += v * v; // a float product, as data[]*data[] is
    }
    m /= F.nsamp;
    sd /= F.nsamp;
    sd = fma(-m, m, sd); // tmpstd -= tmpmean*tmpmean
    sd = sqrt(sd);
    if (sd == 0.) sd = 1.;
    for (long i = 0; i < F.nsamp; i++) {
        float v = F.at(f, j, i);
        v = (float)((double)v - m);
        v = (float)((double)v / sd);
        F.at(f, j, i) = v;
    }
}

// zdot 2: per (frame, sample) the channel mean of the normalised data,
// summed in channel order (candidate.cpp:858, 862-865)
__global__ void k_zdot_s(Frames F, double *s)
{
    const long g = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= (long)F.nframes * F.nsamp) return;
    const long f = g / F.nsamp, i = g % F.nsamp;
    double a = 0.;
    long j = 0;
    for (; j + 16 <= F.nchan; j += 16) { // 16 loads in flight, summed in channel order
        float v[16];
#pragma unroll
        for (int u = 0; u < 16; u++) v[u] = F.at(f, j + u, i);
#pragma unroll
        for (int u = 0; u < 16; u++) a += v[u];
    }
    for (; j < F.nchan; j++) a += F.at(f, j, i);
    s[g] = a / F.nchan;
}

// zdot 3: per frame sum s and sum s^2 (the same for every channel,
// candidate.cpp:879-880)
__global__ void k_zdot_ss(Frames F, const double *s, double *sess)
{
    const long f = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (f >= F.nframes) return;
    double se = 0., ss = 0.;
    const double *sf = s + f * F.nsamp;
    long i = 0;
    for (; i + 32 <= F.nsamp; i += 32) { // 32 loads in flight (one thread per frame)
        double v[32];
#pragma unroll
        for (int u = 0; u < 32; u++) v[u] = sf[i + u];
#pragma unroll
        for (int u = 0; u < 32; u++) {
            se += v[u];
            ss = fma(v[u], v[u], ss);
        }
    }
    for (; i < F.nsamp; i++) {
        se += sf[i];
        ss = fma(sf[i], sf[i], ss);
    }
    sess[2 * f] = se;
    sess[2 * f + 1] = ss;
}

// zdot 4: per (frame, channel) the least-squares fit alpha*s + beta of the
// channel, subtracted (candidate.cpp:870-896)
__global__ void k_zdot_fit(Frames F, const double *s, const double *sess)
{
    const long g = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= (long)F.nframes * F.nchan) return;
    const long f = g / F.nchan, j = g % F.nchan;
    const double *sf = s + f * F.nsamp;
    double xe = 0., xs = 0.;
    for (long i = 0; i < F.nsamp; i++) {
        const float v = F.at(f, j, i);
        xe += v;
        xs = fma((double)v, sf[i], xs);
    }
    const double se = sess[2 * f], ss = sess[2 * f + 1], nb = (double)F.nsamp;
    const double tmp = fma(se, se, -(ss * nb));
    double alpha = 0., beta = 0.;
    if (tmp != 0) {
        alpha = fma(xe, se, -(xs * nb)) / tmp;
        beta = fma(xs, se, -(xe * ss)) / tmp;
    }
    for (long i = 0; i < F.nsamp; i++) {
        const double fit = fma(alpha, sf[i], beta);
        F.at(f, j, i) = (float)((double)F.at(f, j, i) - fit);
    }
}

// ---- the same passes with memory access shaped for the two common layouts;
// every channel's sums still run sample by sample in order, so results are
// those of the kernels above.

// Channel-major frames (tstride 1): a wave takes 64 channels; 64-sample
// tiles of their rows pass through LDS (coalesced row loads, a padded
// [64][65] tile read one row per lane without bank conflicts).
constexpr int kTile = 64;

template <bool FIT>
__global__ __launch_bounds__(256) void k_zdot_rows(Frames F, const double *s, const double *sess)
{
    __shared__ float tile[4][kTile][kTile + 1];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const long g0 = ((long)blockIdx.x * 4 + w) * 64; // first (frame, channel) of the wave
    const long ntot = (long)F.nframes * F.nchan;
    const long g = g0 + lane;
    const bool live = g < ntot;
    const long f = live ? g / F.nchan : 0, j = live ? g % F.nchan : 0;
    float (*T)[kTile + 1] = tile[w];
    // rows of the wave's channels: row c is (frame, channel) g0 + c
    auto rowp = [&](int c) -> float * {
        const long gc = g0 + c;
        return F.x + (gc / F.nchan) * F.fstride + (gc % F.nchan) * F.cstride;
    };
    const int nrow = (int)min((long)64, ntot - g0);
    // 16 row loads in flight at a time (addresses clamped into the frame,
    // only rows and samples that exist are stored)
    auto load = [&](long t0) {
        const int n = (int)min((long)kTile, F.nsamp - t0);
        const long ti = t0 + min(lane, n - 1);
        for (int c0 = 0; c0 < nrow; c0 += 16) {
            float v[16];
#pragma unroll
            for (int u = 0; u < 16; u++) v[u] = rowp(min(c0 + u, nrow - 1))[ti];
#pragma unroll
            for (int u = 0; u < 16; u++)
                if (c0 + u < nrow && lane < n) T[c0 + u][lane] = v[u];
        }
        __builtin_amdgcn_wave_barrier();
        return n;
    };
    auto store = [&](long t0, int n) {
        __builtin_amdgcn_s_waitcnt(0);
        __builtin_amdgcn_wave_barrier();
        for (int c = 0; c < nrow; c++) {
            float *r = rowp(c) + t0;
            if (lane < n) r[lane] = T[c][lane];
        }
        __builtin_amdgcn_wave_barrier();
    };
    const double *sf = s + f * F.nsamp; // read only when FIT
    double a = 0., b = 0.;
    for (long t0 = 0; t0 < F.nsamp; t0 += kTile) {
        const int n = load(t0);
        if (live) {
            int i = 0;
            for (; FIT && i + 16 <= n; i += 16) {
                double sv[16]; // the channel mean's values, loaded ahead
#pragma unroll
                for (int u = 0; u < 16; u++) sv[u] = sf[t0 + i + u];
#pragma unroll
                for (int u = 0; u < 16; u++) {
                    const float v = T[lane][i + u];
                    a += v;
                    b = fma((double)v, sv[u], b);
                }
            }
            for (; i < n; i++) {
                const float v = T[lane][i];
                a += v;
                if (FIT) b = fma((double)v, sf[t0 + i], b);
                else b += v * v;
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
    double m = 0., sd = 1., alpha = 0., beta = 0.;
    if (!FIT) {
        m = a / F.nsamp;
        sd = b / F.nsamp;
        sd = fma(-m, m, sd);
        sd = sqrt(sd);
        if (sd == 0.) sd = 1.;
    } else if (live) {
        const double se = sess[2 * f], ss = sess[2 * f + 1], nb = (double)F.nsamp;
        const double tmp = fma(se, se, -(ss * nb));
        if (tmp != 0) {
            alpha = fma(a, se, -(b * nb)) / tmp;
            beta = fma(b, se, -(a * ss)) / tmp;
        }
    }
    for (long t0 = 0; t0 < F.nsamp; t0 += kTile) {
        const int n = load(t0);
        if (live) {
            int i = 0;
            for (; FIT && i + 16 <= n; i += 16) {
                double sv[16];
#pragma unroll
                for (int u = 0; u < 16; u++) sv[u] = sf[t0 + i + u];
#pragma unroll
                for (int u = 0; u < 16; u++)
                    T[lane][i + u] = (float)((double)T[lane][i + u] - fma(alpha, sv[u], beta));
            }
            for (; i < n; i++) {
                float v = T[lane][i];
                if (FIT) {
                    v = (float)((double)v - fma(alpha, sf[t0 + i], beta));
                } else {
                    v = (float)((double)v - m);
                    v = (float)((double)v / sd);
                }
                T[lane][i] = v;
            }
        }
        store(t0, n);
    }
    (void)j;
}

// n steps of a chain, 16 at a time: get(i) reads the operands of 16 steps while
// the 16 before them run (the scheduling barriers keep the reads ahead).
template <int n, class T, class Get, class Step>
__device__ __forceinline__ void chain16(Get get, Step step)
{
    T x0[16], x1[16];
    auto fetch = [&](T(&x)[16], int i) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < 16; u++) x[u] = get(i + u);
        __builtin_amdgcn_sched_barrier(0);
    };
    fetch(x0, 0);
#pragma unroll
    for (int i = 0; i < n; i += 32) {
        fetch(x1, i + 16);
#pragma unroll
        for (int u = 0; u < 16; u++) step(i + u, x0[u]);
        if (i + 32 < n) fetch(x0, i + 32);
#pragma unroll
        for (int u = 0; u < 16; u++) step(i + 16 + u, x1[u]);
    }
}

// ---- Channel-major frames whose rows fit LDS: one read of the frame for the
// statistics and the channel mean, one read and one write for the fit.  A
// workgroup keeps RB rows (32 at 512 samples, two workgroups per CU) in LDS;
// one wave runs the rows' chains, lanes r and RB + r the two sums of row r
// over the same 16-byte LDS reads (the row pitch is an odd multiple of 4
// floats, so 16 lanes' reads cover the 64 banks), and all the waves
// normalise and update along time.  Eight waves, since a tile's phases follow
// one another and only the other workgroup's fill the gaps (four waves: 1.28
// and 1.07 ms where eight take 1.10 and 0.86; 16-row tiles, four workgroups
// a CU: 1.33 and 1.32; the next tile loaded into registers ahead: no
// faster).  1024 frames of 1024 x 512 samples (2.1 GB): statistics and mean
// 0.86 ms, fit 1.10 ms (3.9 TB/s); tiles of 64 samples per pass took 3.0 and
// 2.5.
constexpr int kTileThreads = 512, kTileWaves = kTileThreads / 64;
struct RowTile {
    int RB, st; // rows per tile, row pitch in LDS (floats)
};
__host__ __device__ inline int row_pitch(long nsamp) { return (int)(((nsamp + 3) / 4) | 1) * 4; }
// LDS of a tile: the rows, 16 bytes per sample (the fit's {1, s}; the
// statistics kernel needs half of it) and 32 per row
inline size_t tile_lds(int RB, long nsamp)
{
    return (size_t)RB * row_pitch(nsamp) * 4 + (size_t)nsamp * 16 + (size_t)RB * 32;
}
constexpr size_t kTileLds = 80 * 1024; // two workgroups per CU
inline RowTile row_tile(long nsamp)
{
    for (int RB = 32; RB >= 8; RB >>= 1)
        if (nsamp <= 16384 && tile_lds(RB, nsamp) <= kTileLds) return {RB, row_pitch(nsamp)};
    return {0, 0};
}

// Few frames of many channels and short rows: k_zdot_norm_mean, whose lanes
// each walk all channels (0.115 us a channel), takes longer than the row
// kernels, whose time goes with the tiles of 64 samples (65 us each) until
// there are more rows than they keep in flight.  Row kernels and tiles, us:
// 1 frame of 1024 x 64 94 and 129, 128 frames 118 and 153, 256 frames 197 and
// 190; 1 frame of 4096 x 64 157 and 474, of 4096 x 192 301 and 486, 100 frames
// of 4096 x 128 662 and 668; 1 frame of 1024 x 128 159 and 132, 8 frames of
// 2048 x 192 262 and 229.
inline bool short_rows(int nframes, int nchan, long nsamp)
{
    const long T = (nsamp + 63) / 64;
    return T * 750 <= nchan && T * nframes <= 192;
}

// Frames from which a frame per workgroup is faster than a tile per workgroup.
// It reads the frames once less and needs two launches fewer, but a workgroup
// walks its frame's tiles one after the other while, with fewer frames than
// fill the CUs twice over, others idle: the later, the more tiles a frame has
// and the longer its rows.  Frame and tile per workgroup, us: 1024 channels,
// 128 frames of 192 samples 222 and 219, 256 of 512 560 and 609, 128 of 1012
// 1261 and 783, 512 of 1012 2543 and 2803, 256 of 1700 4242 and 3465; 256
// channels, 128 of 512 115 and 114, 400 of 1012 574 and 617; 64 channels, 200
// of 557 75 and 90, 128 of 1700 233 and 171, 256 of 1700 295 and 318.
inline long frame_per_group(int nchan, long nsamp, int RB)
{
    const long nt = (nchan + RB - 1) / RB;
    return RB == 32 ? 64 + std::min(nsamp / 3, 8 * nt) : std::min(512L, 64 + 18 * nt);
}

// Rows j0 .. j0 + nr of frame f into LDS.  Whole 16-byte lines: up to 3
// floats past a row's end are read from the rows after it; rows so near the
// frames' end that those would lie past it take 4-byte loads.
__device__ __forceinline__ void tile_load(const Frames &F, long f, int j0, int nr, const RowTile &R, float *T)
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int n = (int)F.nsamp;
    const long total = (long)F.nframes * F.nchan * n;
    for (int r = w; r < nr; r += kTileWaves) {
        const long g = f * F.nchan + j0 + r;
        const uint32_t *src = (const uint32_t *)(F.x + g * n);
        if (g * n + ((n + 3) & ~3) > total)
            lds_fill(src, (uint32_t *)(T + r * R.st), n, 0, 1, lane);
        else
            lds_fill16(src, (uint32_t *)(T + r * R.st), n, 0, 1, lane);
    }
}

// The wave that runs a tile's chains: another one for each of the workgroups
// that a CU is given in turn (every 256th), so that co-resident workgroups'
// chains sit on different SIMDs.
__device__ __forceinline__ int chain_wave() { return (int)(blockIdx.x >> 8) & 3; }

// step(i, x) over the n samples of an LDS row in order, 16-byte reads 16
// samples ahead.
template <class Step>
__device__ __forceinline__ void row_chain(const float *row, int n, Step step)
{
    const float4 *p = (const float4 *)row;
    float4 x0[4], x1[4];
    auto get = [&](float4(&x)[4], int q) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < 4; u++) x[u] = p[q + u];
        __builtin_amdgcn_sched_barrier(0);
    };
    auto run = [&](const float4(&x)[4], int i) {
#pragma unroll
        for (int u = 0; u < 4; u++) {
            step(i + 4 * u, x[u].x);
            step(i + 4 * u + 1, x[u].y);
            step(i + 4 * u + 2, x[u].z);
            step(i + 4 * u + 3, x[u].w);
        }
    };
    int i = 0;
    if (n >= 32) {
        get(x0, 0);
#pragma unroll 1
        for (; i + 32 <= n; i += 32) {
            get(x1, i / 4 + 4);
            run(x0, i);
            get(x0, i + 64 <= n ? i / 4 + 8 : 0); // the last one reads the row's start, unused
            run(x1, i + 16);
        }
    }
    for (; i < n; i++) step(i, row[i]);
}

// zdot's normalisation (candidate.cpp:853-859)
__device__ __forceinline__ float zdot_norm(float v, double m, double sd)
{
    v = (float)((double)v - m);
    return (float)((double)v / sd);
}

// The same for U values v[u] of channels with (m, sd, 1/sd) = ch(u), by one
// FP64 product each where that must give the same float, else by the
// division (an FP64 division is a dozen instructions, the product and its
// check five).  The product d*(1/sd) is within 2^-52 of d/sd, so it and the
// rounded quotient are at most 3 units of the last of 53 bits apart, and they
// round to the same float unless a boundary between floats lies within 3
// units: for normal floats that is a low part (29 bits) of 0x10000000, kept
// away from by 4 units.  Values whose magnitude is below 2^-126, infinite or
// NaN are divided, and sd outside [2^-400, 2^400] has NaN as its reciprocal.
__device__ __forceinline__ double zdot_rcp(double sd)
{
    return sd >= 0x1p-400 && sd <= 0x1p400 ? 1. / sd : (double)NAN;
}
template <int U, class Ch>
__device__ __forceinline__ void zdot_norms(float (&v)[U], Ch ch)
{
    unsigned low = ~0u, mag = 0u; // the low part above the boundary's 4 units, the magnitude above 2^-126
    float x[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
        const auto c = ch(u);
        const double q = (double)(float)((double)v[u] - c.m) * c.r;
        const unsigned long long b = (unsigned long long)__double_as_longlong(q);
        low = min(low, ((unsigned)b << 3) + (0u - (0x0FFFFFFCu << 3)));
        mag = max(mag, ((unsigned)(b >> 32) << 1) + (0u - 2u * 0x38100000u));
        x[u] = (float)q;
    }
    if (low <= 8u << 3 || mag >= 2u * (0x7FF00000u - 0x38100000u)) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            const auto c = ch(u);
            x[u] = zdot_norm(v[u], c.m, c.sd);
        }
    }
#pragma unroll
    for (int u = 0; u < U; u++) v[u] = x[u];
}
struct ChanStat {
    double m, sd, r;
};

// Mean and standard deviation of each channel (candidate.cpp:837-851) into
// stat[2*(f*nchan + j)].  MEAN: one workgroup per frame, which walks the
// channels in order and so also forms the channel mean s of the normalised
// samples (:858, 862-865) and the sums of s and s^2 (:879-880) from the same
// read; without MEAN one workgroup per tile of rows.
template <bool MEAN>
__global__ __launch_bounds__(kTileThreads) void k_zdot_tile_stats(Frames F, RowTile R, double *stat, double *s, double *sess)
{
    extern __shared__ __attribute__((aligned(16))) float T[]; // [RB][st]
    const int n = (int)F.nsamp, tid = threadIdx.x, lane = tid & 63, RB = R.RB;
    double *sacc = (double *)(T + RB * R.st); // [n]
    ChanStat *ms = (ChanStat *)(sacc + n);    // [RB]
    const int ntile = (F.nchan + RB - 1) / RB;
    const long f = MEAN ? blockIdx.x : blockIdx.x / ntile;
    for (int jt = MEAN ? 0 : (int)(blockIdx.x % ntile); jt < ntile; jt++) {
        const int j0 = jt * RB, nr = min(RB, F.nchan - j0);
        __syncthreads(); // the tile before has been used
        tile_load(F, f, j0, nr, R, T);
        txgpu::lds_fill_done();
        if (tid >> 6 == chain_wave()) {
            const bool sq = lane >= RB && lane < 2 * RB; // the lane of sum x^2
            double a = 0.;
            row_chain(T + (lane & (RB - 1)) * R.st, n, [&](int, float x) {
                a += (double)(x * (sq ? x : 1.f)); // a float product, as data[]*data[] is
            });
            const double b = __shfl(a, (lane + RB) & 63, 64);
            const double m = a / F.nsamp;
            double sd = b / F.nsamp;
            sd = fma(-m, m, sd); // tmpstd -= tmpmean*tmpmean
            sd = sqrt(sd);
            if (sd == 0.) sd = 1.;
            if (lane < nr) {
                ms[lane] = {m, sd, zdot_rcp(sd)};
                stat[2 * (f * F.nchan + j0 + lane)] = m;
                stat[2 * (f * F.nchan + j0 + lane) + 1] = sd;
            }
        }
        if (!MEAN) return;
        __syncthreads();
        for (int t = tid; t < n; t += kTileThreads) {
            double a = jt ? sacc[t] : 0.;
            int r = 0;
            for (; r + 8 <= nr; r += 8) {
                float v[8];
#pragma unroll
                for (int u = 0; u < 8; u++) v[u] = T[(r + u) * R.st + t];
                zdot_norms(v, [&](int u) { return ms[r + u]; });
#pragma unroll
                for (int u = 0; u < 8; u++) a += (double)v[u];
            }
            for (; r < nr; r++) a += (double)zdot_norm(T[r * R.st + t], ms[r].m, ms[r].sd);
            sacc[t] = a;
        }
    }
    if (!MEAN) return;
    for (int t = tid; t < n; t += kTileThreads) { // each thread its own samples
        const double a = sacc[t] / F.nchan;
        sacc[t] = a;
        s[f * F.nsamp + t] = a;
    }
    __syncthreads();
    if (tid < 2) { // sum s (lane 0: fma(s, 1, a) is a + s) and sum s^2 (lane 1)
        double a = 0.;
        int i = 0;
        for (; i + 16 <= n; i += 16) {
            double v[16];
#pragma unroll
            for (int u = 0; u < 16; u++) v[u] = sacc[i + u];
#pragma unroll
            for (int u = 0; u < 16; u++) a = fma(v[u], tid ? v[u] : 1., a);
        }
        for (; i < n; i++) a = fma(sacc[i], tid ? sacc[i] : 1., a);
        sess[2 * f + tid] = a;
    }
}

// The channel mean from the raw frame and the channels' statistics, one lane
// per sample: for batches of too few frames to give every CU one.
__global__ __launch_bounds__(64) void k_zdot_norm_mean(Frames F, const double *__restrict__ stat, double *s)
{
    const int per = (int)((F.nsamp + 63) / 64);
    const long f = blockIdx.x / per, t = (long)(blockIdx.x % per) * 64 + threadIdx.x;
    const float *x = F.x + f * F.fstride + min(t, F.nsamp - 1);
    const double *st = stat + 2 * f * F.nchan;
    double a = 0.;
    int j = 0;
    for (; j + 8 <= F.nchan; j += 8) {
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = x[(long)(j + u) * F.nsamp];
#pragma unroll
        for (int u = 0; u < 8; u++) a += (double)zdot_norm(v[u], st[2 * (j + u)], st[2 * (j + u) + 1]);
    }
    for (; j < F.nchan; j++) a += (double)zdot_norm(x[(long)j * F.nsamp], st[2 * j], st[2 * j + 1]);
    if (t < F.nsamp) s[f * F.nsamp + t] = a / F.nchan;
}

// The rows of a tile normalised in LDS, their least-squares fit to s, and
// the frame less that fit (candidate.cpp:870-896).
__global__ __launch_bounds__(kTileThreads) void k_zdot_tile_fit(Frames F, RowTile R, const double *__restrict__ stat,
                                                       const double *__restrict__ s, const double *__restrict__ sess)
{
    extern __shared__ __attribute__((aligned(16))) float T[]; // [RB][st]
    const int n = (int)F.nsamp, tid = threadIdx.x, lane = tid & 63, w = tid >> 6, RB = R.RB;
    double(*mult)[2] = (double(*)[2])(T + RB * R.st); // [n] {1, s}
    double *ms = &mult[n][0];                         // [RB][2]
    double *ab = ms + 2 * RB;                         // [RB][2]
    const int ntile = (F.nchan + RB - 1) / RB;
    const long f = blockIdx.x / ntile;
    const int j0 = (int)(blockIdx.x % ntile) * RB, nr = min(RB, F.nchan - j0);
    tile_load(F, f, j0, nr, R, T);
    for (int t = tid; t < n; t += kTileThreads) {
        mult[t][0] = 1.;
        mult[t][1] = s[f * F.nsamp + t];
    }
    if (tid < 2 * nr) ms[tid] = stat[2 * (f * F.nchan + j0) + tid];
    txgpu::lds_fill_done();
    for (int r = w; r < nr; r += kTileWaves) {
        const double m = ms[2 * r], sd = ms[2 * r + 1];
        const ChanStat c{m, sd, zdot_rcp(sd)};
        float *row = T + r * R.st;
        int t = lane;
        for (; t - lane + 256 <= n; t += 256) {
            float v[4];
#pragma unroll
            for (int u = 0; u < 4; u++) v[u] = row[t + 64 * u];
            zdot_norms(v, [&](int) { return c; });
#pragma unroll
            for (int u = 0; u < 4; u++) row[t + 64 * u] = v[u];
        }
        for (; t < n; t += 64) row[t] = zdot_norm(row[t], m, sd);
    }
    __syncthreads();
    if (w == chain_wave()) {
        const int sel = lane >= RB && lane < 2 * RB; // the lane of sum x*s
        double a = 0.;
        row_chain(T + (lane & (RB - 1)) * R.st, n, [&](int i, float x) { a = fma((double)x, mult[i][sel], a); });
        const double b = __shfl(a, (lane + RB) & 63, 64);
        const double se = sess[2 * f], ss = sess[2 * f + 1], nb = (double)F.nsamp;
        const double tmp = fma(se, se, -(ss * nb));
        double alpha = 0., beta = 0.;
        if (tmp != 0) {
            alpha = fma(a, se, -(b * nb)) / tmp;
            beta = fma(b, se, -(a * ss)) / tmp;
        }
        if (lane < nr) {
            ab[2 * lane] = alpha;
            ab[2 * lane + 1] = beta;
        }
    }
    __syncthreads();
    for (int r = w; r < nr; r += kTileWaves) {
        const double alpha = ab[2 * r], beta = ab[2 * r + 1];
        const float *row = T + r * R.st;
        float *out = F.x + (f * F.nchan + j0 + r) * F.nsamp;
#pragma unroll 4
        for (int t = lane; t < n; t += 64) out[t] = (float)((double)row[t] - fma(alpha, mult[t][1], beta));
    }
}

// ---- Time-major frames (cstride 1), the DataBuffer layout.  A channel's sums
// run over all its samples one after the other, so a search block (26,123
// samples of 4096 channels) is 4096 chains of 26,123 dependent FP64 adds and
// nothing shorter; what can be chosen is what a step of the chain costs.  On
// gfx950 a dependent FP64 add or FMA issues every 4.5 cycles and a
// conversion every 5.5 (measured), so the chains get a wave of their own
// (wave 0 of the workgroup, which only reads LDS, converts and adds) and
// four helper waves bring the samples: 32 channels (one 128-byte line of a
// sample) per workgroup, so that 4096 channels use 128 CUs, and both of a
// channel's sums in the same wave (lane l and lane l + 32).  The helpers keep
// two chunks of kColT samples in registers on their way from HBM while a
// third is written to LDS and a fourth is summed.
constexpr int kColCh = 32, kColT = 128, kColThreads = 64 + 256;
typedef float f4u __attribute__((ext_vector_type(4), aligned(4))); // 4-byte aligned 16-byte access

// The streaming part: chunks of kColT samples of 32 columns (ts floats from
// sample to sample, N samples) pass through buf; put(k, v) of a helper
// thread (h < 256) stores columns q4 .. q4 + 3 of its samples r0 + 32*u
// of chunk k, chain(k) of wave 0 works on chunk k, buf half k & 1.  NARROW:
// only nc < 32 columns exist, the last one stands in for those past it.
struct ColChunk {
    f4u v[4];
    double s;
};
template <bool NARROW, class Put, class Chain>
__device__ __forceinline__ void stream_columns(const float *__restrict__ col, const double *__restrict__ sf, long N,
                                               long ts, int nc, Put put, Chain chain)
{
    const int tid = threadIdx.x, h = tid - 64, q4 = (h & 7) * 4, r0 = h >> 3;
    const int nk = (int)((N + kColT - 1) / kColT);
    auto load = [&](int k, ColChunk &c) { // past the end: a sample that exists, unused
        const long t0 = (long)k * kColT;
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const float *row = col + min(t0 + r0 + 32 * u, N - 1) * ts;
            if (NARROW)
                c.v[u] = f4u{row[min(q4, nc - 1)], row[min(q4 + 1, nc - 1)], row[min(q4 + 2, nc - 1)],
                             row[min(q4 + 3, nc - 1)]};
            else
                c.v[u] = *(const f4u *)(row + q4);
        }
        if (sf) c.s = sf[min(t0 + (h & (kColT - 1)), N - 1)];
    };
    ColChunk A, B;
    if (tid >= 64) {
        load(0, A);
        load(1, B);
        put(0, A);
        load(2, A);
    } else {
        __builtin_amdgcn_s_setprio(3); // the chain wave goes first on its SIMD
    }
    __syncthreads();
    for (int k = 0; k < nk; k += 2) {
        if (tid < 64) {
            chain(k);
        } else {
            put(k + 1, B);
            load(k + 3, B);
        }
        __syncthreads();
        if (k + 1 >= nk) break;
        if (tid < 64) {
            chain(k + 1);
        } else {
            put(k + 2, A);
            load(k + 4, A);
        }
        __syncthreads();
    }
}

// FIT = false: mean and standard deviation of each channel (candidate.cpp:837-851)
// into stat[2*(f*nchan + j)].  FIT = true: sum x and sum x*s of each
// (already normalised) channel (:870-880) into the same place, and, in one
// extra workgroup per frame, sum s and sum s^2 into sess.  4096 channels x
// 26,123 samples (428 MB): 177 us and 214 us, 16 and 20 cycles a sample; one
// lane per channel loading for itself took 1.9 and 1.4 ms (with the update).
// NARROW: frames of fewer than 32 channels, whose chains are as long: zdot of
// 31 x 26,123 samples takes 407 us (32: 394), with one lane per channel 3.7 ms
// where it keeps 32 loads in flight and 12.6 ms where it does not.
template <bool FIT, bool NARROW>
__global__ __launch_bounds__(kColThreads) void k_zdot_chain(Frames F, const double *__restrict__ s, double *stat,
                                                            double *sess)
{
    constexpr int RS = FIT ? kColCh : 2 * kColCh; // floats per sample: x, or x then x*x
    __shared__ __attribute__((aligned(16))) float buf[2][kColT * RS];
    __shared__ double mult[FIT ? 2 : 1][FIT ? kColT : 1][2]; // {1, s} per sample
    const int tid = threadIdx.x, lane = tid & 63;
    const int per = (F.nchan + kColCh - 1) / kColCh + (FIT ? 1 : 0); // workgroups per frame
    const long f = blockIdx.x / per;
    const int g = (int)(blockIdx.x % per);
    const long N = F.nsamp;
    const double *sf = s + f * N; // read only when FIT

    struct VM {
        double v, m;
    };
    struct XM {
        float x;
        double m;
    };
    if (FIT && g == per - 1) {
        // sum s (lane 0: fma(s, 1, a) is a + s) and sum s^2 (lane 1); the
        // next 128 values are on their way while these are summed
        if (tid >= 64) return;
        double a = 0., n0 = sf[min((long)lane, N - 1)], n1 = sf[min(lane + 64L, N - 1)];
        for (long t0 = 0; t0 < N; t0 += kColT) {
            const int n = (int)min((long)kColT, N - t0);
            mult[0][lane][0] = mult[0][lane + 64][0] = 1.;
            mult[0][lane][1] = n0;
            mult[0][lane + 64][1] = n1;
            n0 = sf[min(t0 + kColT + lane, N - 1)];
            n1 = sf[min(t0 + kColT + lane + 64, N - 1)];
            __builtin_amdgcn_wave_barrier();
            if (n == kColT)
                chain16<kColT, VM>([&](int i) { return VM{mult[0][i][1], mult[0][i][lane & 1]}; },
                                   [&](int, const VM &x) { a = fma(x.v, x.m, a); });
            else
                for (int i = 0; i < n; i++) a = fma(mult[0][i][1], mult[0][i][lane & 1], a);
            __builtin_amdgcn_wave_barrier();
        }
        if (lane < 2) sess[2 * f + lane] = a;
        return;
    }

    // the last group ends at the last channel (the channels it shares with
    // the group before come out the same in both)
    const int c0 = NARROW ? 0 : min(g * kColCh, F.nchan - kColCh);
    const int nc = NARROW ? F.nchan : kColCh;
    const int h = tid - 64, q4 = (h & 7) * 4, r0 = h >> 3;
    double acc = 0.;
    const int sel = lane >> 5;
    const int ls = FIT ? (lane & 31) : lane;
    auto put = [&](int k, const ColChunk &c) {
        float *b = buf[k & 1];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            float *d = b + (r0 + 32 * u) * RS + q4;
            const f4u &v = c.v[u];
            *(float4 *)d = make_float4(v[0], v[1], v[2], v[3]);
            if (!FIT) // a float product, as data[]*data[] is
                *(float4 *)(d + kColCh) = make_float4(v[0] * v[0], v[1] * v[1], v[2] * v[2], v[3] * v[3]);
        }
        if (FIT && h < kColT) {
            mult[k & 1][h][0] = 1.;
            mult[k & 1][h][1] = c.s;
        }
    };
    auto chain = [&](int k) {
        const float *b = buf[k & 1] + ls;
        const int n = (int)min((long)kColT, N - (long)k * kColT);
        if (n == kColT) {
            if (FIT)
                chain16<kColT, XM>([&](int i) { return XM{b[i * RS], mult[k & 1][FIT ? i : 0][sel]}; },
                                   [&](int, const XM &x) { acc = fma((double)x.x, x.m, acc); });
            else
                chain16<kColT, float>([&](int i) { return b[i * RS]; }, [&](int, float x) { acc += (double)x; });
        } else {
            for (int i = 0; i < n; i++)
                acc = FIT ? fma((double)b[i * RS], mult[k & 1][i][sel], acc) : acc + (double)b[i * RS];
        }
    };
    stream_columns<NARROW>(F.x + f * F.fstride + c0, FIT ? sf : nullptr, N, F.tstride, nc, put, chain);
    if (tid >= 64) return;
    double *out = stat + 2 * (f * F.nchan + c0);
    if (FIT) {
        if (ls < nc) out[2 * ls + sel] = acc;
    } else {
        const double other = __shfl_xor(acc, 32, 64);
        const double m = acc / N;
        double sd = other / N;
        sd = fma(-m, m, sd); // tmpstd -= tmpmean*tmpmean
        sd = sqrt(sd);
        if (sd == 0.) sd = 1.;
        if (lane < nc) {
            out[2 * lane] = m;
            out[2 * lane + 1] = sd;
        }
    }
}

// The time-major frame normalised in place with the channels' (mean, sd)
// (candidate.cpp:853-859), and each sample's channel mean s, summed in
// channel order (:858, 862-865).  A workgroup takes 32 samples and walks the
// channels 128 at a time: four helper waves load, normalise, store and
// leave the values in LDS, while wave 4 (lane = sample) adds the tile before
// in channel order.  250 us for 856 MB at 4096 channels x 26,123 samples.
constexpr int kNsT = 32, kNsC = 128;
__global__ __launch_bounds__(320) void k_zdot_norm_s(Frames F, const double *__restrict__ stat, double *s)
{
    __shared__ float T[2][kNsC][kNsT + 1];
    const long per = (F.nsamp + kNsT - 1) / kNsT;
    const long f = blockIdx.x / per, t0 = (blockIdx.x % per) * kNsT;
    const int nt = (int)min((long)kNsT, F.nsamp - t0);
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    float *blk = F.x + f * F.fstride + t0 * F.tstride;
    const double *st = stat + 2 * f * F.nchan;
    const int nk = (F.nchan + kNsC - 1) / kNsC;
    double a = 0.;
    // channels c0 + lane + 64*i, samples w + 4*u, and the channels' mean and sd
    struct Tile {
        float v[2][8];
        double m[2], sd[2];
    } A, B;
    auto load = [&](int k, Tile &t) { // past the end: values that exist, unused
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const int c = min(k * kNsC + lane + 64 * i, F.nchan - 1);
            t.m[i] = st[2 * c];
            t.sd[i] = st[2 * c + 1];
#pragma unroll
            for (int u = 0; u < 8; u++) t.v[i][u] = blk[min(w + 4 * u, nt - 1) * F.tstride + c];
        }
    };
    // the next tile's loads go out before this one's stores: a wait for
    // loads then has no stores ahead of it
    auto norm = [&](int k, Tile &t, Tile &next) {
        load(k + 1, next);
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const int cc = lane + 64 * i, c = k * kNsC + cc;
            const ChanStat cs{t.m[i], t.sd[i], zdot_rcp(t.sd[i])};
            zdot_norms(t.v[i], [&](int) { return cs; });
#pragma unroll
            for (int u = 0; u < 8; u++) {
                const float x = t.v[i][u];
                T[k & 1][cc][w + 4 * u] = x;
                if (c < F.nchan && w + 4 * u < nt) blk[(w + 4 * u) * F.tstride + c] = x;
            }
        }
    };
    if (w < 4) load(0, A);
    for (int k = 0; k <= nk; k++) {
        if (w < 4) {
            if (k < nk) {
                if (k & 1)
                    norm(k, B, A);
                else
                    norm(k, A, B);
            }
        } else if (k > 0 && lane < kNsT) {
            const float(*Tk)[kNsT + 1] = T[(k - 1) & 1];
            const int n = min(kNsC, F.nchan - (k - 1) * kNsC);
            if (n == kNsC) {
                chain16<kNsC, float>([&](int j) { return Tk[j][lane]; }, [&](int, float x) { a += (double)x; });
            } else {
                for (int j = 0; j < n; j++) a += Tk[j][lane];
            }
        }
        __syncthreads();
    }
    if (w == 4 && lane < nt) s[f * F.nsamp + t0 + lane] = a / F.nchan;
}

// The time-major frame less each channel's fit alpha*s + beta
// (candidate.cpp:881-896); fit[2*(f*nchan + j)] = (sum x, sum x*s).  One
// thread per channel and 32 samples: one read and one write of the frame
// (131 us for 856 MB).
constexpr int kUpT = 32;
__global__ __launch_bounds__(256) void k_zdot_update(Frames F, const double *__restrict__ s,
                                                     const double *__restrict__ fit,
                                                     const double *__restrict__ sess)
{
    const long nct = (F.nchan + 255) / 256, per = nct * ((F.nsamp + kUpT - 1) / kUpT);
    const long f = blockIdx.x / per, r = blockIdx.x % per;
    const int j = (int)(r % nct) * 256 + threadIdx.x;
    const long t0 = r / nct * kUpT;
    if (j >= F.nchan) return;
    const int n = (int)min((long)kUpT, F.nsamp - t0);
    float *col = F.x + f * F.fstride + t0 * F.tstride + j;
    const double *sf = s + f * F.nsamp + t0;
    const double xe = fit[2 * (f * F.nchan + j)], xs = fit[2 * (f * F.nchan + j) + 1];
    const double se = sess[2 * f], ss = sess[2 * f + 1], nb = (double)F.nsamp;
    const double tmp = fma(se, se, -(ss * nb));
    double alpha = 0., beta = 0.;
    if (tmp != 0) {
        alpha = fma(xe, se, -(xs * nb)) / tmp;
        beta = fma(xs, se, -(xe * ss)) / tmp;
    }
    if (n == kUpT) {
        float v[kUpT];
#pragma unroll
        for (int u = 0; u < kUpT; u++) v[u] = col[u * F.tstride];
#pragma unroll
        for (int u = 0; u < kUpT; u++) col[u * F.tstride] = (float)((double)v[u] - fma(alpha, sf[u], beta));
    } else {
        for (int u = 0; u < n; u++) col[u * F.tstride] = (float)((double)col[u * F.tstride] - fma(alpha, sf[u], beta));
    }
}

// kadaneF 1: the td x fd downsampled frame, each output summed in float
// over k < fd (outer) and n < td (inner) (candidate.cpp:724-739); ds element
// (jd, id) of frame f is ds[f*ncd*nsd + jd*js + id*is]
__global__ void k_kad_down(Frames F, int td, int fd, int ncd, long nsd, float *ds)
{
    const long g = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= (long)F.nframes * ncd * nsd) return;
    const long f = g / ((long)ncd * nsd), r = g % ((long)ncd * nsd);
    const long jd = r / nsd, id = r % nsd;
    float a = 0.f;
    for (int k = 0; k < fd; k++)
        for (int n = 0; n < td; n++) a += F.at(f, jd * fd + k, id * td + n);
    ds[g] = a;
}

// The same for time-major frames, into ds [f][id][jd]: a thread takes one
// downsampled channel and 8 downsampled samples, so that a wavefront's reads
// and writes are consecutive channels of one sample (127 us for 428 MB at
// td 4, fd 2; 1.7 ms with a wavefront along time).
constexpr int kKdT = 8;
__global__ __launch_bounds__(256) void k_kad_down_tm(Frames F, int td, int fd, int ncd, long nsd,
                                                     float *__restrict__ ds)
{
    const long nct = (ncd + 255) / 256, per = nct * ((nsd + kKdT - 1) / kKdT);
    const long f = blockIdx.x / per, r = blockIdx.x % per;
    const int jd = (int)(r % nct) * 256 + threadIdx.x;
    const long id0 = r / nct * kKdT;
    if (jd >= ncd) return;
    const float *x = F.x + f * F.fstride + (long)jd * fd;
    float a[kKdT];
#pragma unroll
    for (int u = 0; u < kKdT; u++) a[u] = 0.f;
    for (int k = 0; k < fd; k++)
#pragma unroll 4
        for (int n = 0; n < td; n++) {
            float v[kKdT]; // samples past the end are clamped, unused
#pragma unroll
            for (int u = 0; u < kKdT; u++) v[u] = x[(min(id0 + u, nsd - 1) * td + n) * F.tstride + k];
#pragma unroll
            for (int u = 0; u < kKdT; u++) a[u] += v[u];
        }
#pragma unroll
    for (int u = 0; u < kKdT; u++)
        if (id0 + u < nsd) ds[(f * nsd + id0 + u) * ncd + jd] = a[u];
}

// The maximum-sum contiguous run of the values stepped through it (the
// XLibs kadane<float>; declared: the running sum restarts after it drops
// below zero, strict '>' keeps the earliest maximum).  sg is 1, or -1 for the
// strongest negative run (the product is exact, so the FMA is one add).
// I: the type that holds a sample's number.
template <class I> struct Kadane {
    float best = -INFINITY, cur = 0.f;
    I s = 0, bs = 0, be = 0;
    __device__ __forceinline__ void step(I i, float sg, float v)
    {
        cur = fmaf(sg, v, cur);
        const bool up = cur > best;
        best = up ? cur : best;
        bs = up ? s : bs;
        be = up ? i : be;
        const bool low = cur < 0.f;
        cur = low ? 0.f : cur;
        s = low ? i + 1 : s;
    }
    // the zapped samples [z[0], z[1]): a run longer than wl whose
    // S/N^2 = sum^2/(wn*td*fd) exceeds threshold^2, empty otherwise
    // (candidate.cpp:752-827)
    __device__ void zap(int td, int fd, int wl, float thre, long *z) const
    {
        const long wn = (long)be - bs + 1;
        float snr2 = 0.f;
        if (wn > wl) snr2 = best * best / ((float)wn * (float)(td * fd));
        const bool hit = snr2 > thre * thre;
        z[0] = hit ? (long)bs * td : 0;
        z[1] = hit ? ((long)be + 1) * td : 0;
    }
};

// kadaneF 2: per (frame, downsampled channel) the strongest positive and
// negative runs.  zap[4*g..]: positive then negative range, empty when not
// zapped.  ds as k_kad_down leaves it.
template <class I>
__global__ void k_kad_scan(int nframes, int ncd, long nsd, int td, int fd, float thre, const int *wnlimit,
                           const float *ds, long *zap)
{
    const long g = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= (long)nframes * ncd) return;
    const float *ch = ds + g * nsd;
    Kadane<I> p, m;
    long i = 0;
    for (; i + 16 <= nsd; i += 16) { // 16 loads in flight
        float v[16];
#pragma unroll
        for (int u = 0; u < 16; u++) v[u] = ch[i + u];
#pragma unroll
        for (int u = 0; u < 16; u++) {
            p.step((I)(i + u), 1.f, v[u]);
            m.step((I)(i + u), -1.f, v[u]);
        }
    }
    for (; i < nsd; i++) {
        p.step((I)i, 1.f, ch[i]);
        m.step((I)i, -1.f, ch[i]);
    }
    const int wl = wnlimit[g / ncd];
    p.zap(td, fd, wl, thre, zap + 4 * g);
    m.zap(td, fd, wl, thre, zap + 4 * g + 2);
}

// The same over ds [f][id][jd] (k_kad_down_tm): 32 consecutive downsampled
// channels per workgroup, their positive runs in the lower half of wave 0 and
// their negative ones in the upper.  A run's scan is one chain over nsd
// samples (6,530 for a search block at td = 4) of eight instructions each,
// and only ncd/32 such waves exist, so helper waves stream the samples as
// they do for the sums of zdot: 212 us for 2048 channels x 6,530 samples,
// 78 cycles a sample (one thread per channel took 1.1 ms).
__global__ __launch_bounds__(kColThreads) void k_kad_scan_tm(int ncd, long nsd, int td, int fd, float thre,
                                                             const int *wnlimit, const float *__restrict__ ds,
                                                             long *zap)
{
    __shared__ __attribute__((aligned(16))) float buf[2][kColT * kColCh];
    const int per = (ncd + kColCh - 1) / kColCh, tid = threadIdx.x, lane = tid & 63;
    const long f = blockIdx.x / per;
    const int c0 = min((int)(blockIdx.x % per) * kColCh, ncd - kColCh);
    const int h = tid - 64, q4 = (h & 7) * 4, r0 = h >> 3;
    const float sg = lane < 32 ? 1.f : -1.f;
    Kadane<int> p;
    auto put = [&](int k, const ColChunk &c) {
#pragma unroll
        for (int u = 0; u < 4; u++)
            *(float4 *)(buf[k & 1] + (r0 + 32 * u) * kColCh + q4) =
                make_float4(c.v[u][0], c.v[u][1], c.v[u][2], c.v[u][3]);
    };
    auto chain = [&](int k) {
        const float *b = buf[k & 1] + (lane & 31);
        const int i0 = k * kColT, n = (int)min((long)kColT, nsd - i0);
        if (n == kColT) {
            constexpr int U = 16;
            float x0[U], x1[U];
            auto get = [&](float(&x)[U], int i) {
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int u = 0; u < U; u++) x[u] = b[(i + u) * kColCh];
                __builtin_amdgcn_sched_barrier(0);
            };
            get(x0, 0);
#pragma unroll 1
            for (int i = 0; i < kColT; i += 2 * U) {
                get(x1, i + U);
#pragma unroll
                for (int u = 0; u < U; u++) p.step(i0 + i + u, sg, x0[u]);
                get(x0, (i + 2 * U) & (kColT - 1)); // the last one reads sample 0 again, unused
#pragma unroll
                for (int u = 0; u < U; u++) p.step(i0 + i + U + u, sg, x1[u]);
            }
        } else {
            for (int i = 0; i < n; i++) p.step(i0 + i, sg, b[i * kColCh]);
        }
    };
    stream_columns<false>(ds + f * nsd * ncd + c0, nullptr, nsd, ncd, kColCh, put, chain);
    if (tid < 64) p.zap(td, fd, wnlimit[f], thre, zap + 4 * (f * ncd + c0 + (lane & 31)) + (lane < 32 ? 0 : 2));
}

// kadaneF of channel-major frames in one pass: a workgroup takes up to 64
// downsampled channels (fd rows each), reads their samples once (lane = a
// downsampled sample), keeps the downsampled rows in LDS, scans them (wave 0
// the positive runs, wave 1 the negative ones, a lane per row) and zeroes
// what is zapped.  Reading the frames is all that is left: 0.49 ms for 2.1 GB
// (1024 frames of 1024 x 512, td 4, fd 2), 0.82 ms with the downsampled
// frames in memory and a kernel per step.
//
// A workgroup's G rows fill at most 38 KB (with the 2 KB of zap ranges four
// workgroups per CU): 64 rows to 151 downsampled samples, 32 to 303, 16 to 607
// and 8 to 1,215.  The scan keeps G lanes of two waves busy, so that longer rows
// pay for the frames read once with chains that leave the CU idle, the sooner
// the fewer samples go into a downsampled one.  k_kad_rows over the three
// kernels, 1024 channels, 64 frames and td = fd = 1: 0.70 at 128 samples, 0.89
// at 256, 1.21 at 512 (256 channels 0.71), 1.32 at 900 and 2.2 at 1800; 32
// frames and td = 4, fd = 2: 0.62 at 512, 0.83 at 900, 1.08 at 1800.  So 8 rows
// only for td*fd >= 8 and never fewer.
constexpr size_t kKrLds = 38 * 1024;
inline int kad_rows(long nsd, int td, int fd) // rows per workgroup, 0: the three kernels
{
    for (int G = 64; G >= ((long)td * fd >= 8 ? 8 : 16); G >>= 1)
        if (nsd <= 65536 && (size_t)G * (nsd | 1) * 4 <= kKrLds) return G;
    return 0;
}
__global__ __launch_bounds__(256) void k_kad_rows(Frames F, int td, int fd, int ncd, int nsd, int G, float thre,
                                                  const int *__restrict__ wnlimit)
{
    extern __shared__ float ds[]; // [G][pitch], pitch odd
    __shared__ long z[64][4];
    const int pitch = nsd | 1, tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int per = (ncd + G - 1) / G;
    const long f = blockIdx.x / per;
    const int g0 = (int)(blockIdx.x % per) * G, ng = min(G, ncd - g0);
    const float *x = F.x + f * F.fstride + (long)g0 * fd * F.nsamp;
    // each output in float over k < fd (outer) and n < td (inner) (candidate.cpp:724-739)
    auto down = [&](int r, int id) {
        const float *q = x + (long)r * fd * F.nsamp + (long)id * td;
        float a = 0.f;
        for (int k = 0; k < fd; k++)
            for (int n = 0; n < td; n++) a += q[k * F.nsamp + n];
        return a;
    };
    if (td == 4 && F.nsamp % 4 == 0 && ((uintptr_t)F.x & 15) == 0) {
        for (int r = w; r < ng; r += 4)
            for (int id = lane; id < nsd; id += 64) {
                const float4 *q = (const float4 *)(x + (long)r * fd * F.nsamp) + id;
                float a = 0.f;
#pragma unroll 4
                for (int k = 0; k < fd; k++) {
                    const float4 v = q[k * (F.nsamp / 4)];
                    a += v.x;
                    a += v.y;
                    a += v.z;
                    a += v.w;
                }
                ds[r * pitch + id] = a;
            }
    } else {
        for (int r = w; r < ng; r += 4)
            for (int id = lane; id < nsd; id += 64) ds[r * pitch + id] = down(r, id);
    }
    __syncthreads();
    if (w < 2 && lane < ng) {
        const float sg = w ? -1.f : 1.f;
        const float *row = ds + lane * pitch;
        Kadane<int> p;
#pragma unroll 8
        for (int i = 0; i < nsd; i++) p.step(i, sg, row[i]);
        p.zap(td, fd, wnlimit[f], thre, &z[lane][2 * w]);
    }
    __syncthreads();
    for (int c = w; c < ng * fd; c += 4) {
        const long *q = z[c / fd];
        float *row = F.x + f * F.fstride + ((long)g0 * fd + c) * F.nsamp;
        for (int p = 0; p < 2; p++)
            for (long i = q[2 * p] + lane; i < q[2 * p + 1]; i += 64) row[i] = 0.f;
    }
}

// kadaneF 3: zero the zapped runs of every channel of each downsampled
// channel (channels past ncd*fd are left as they are); one thread per
// channel, which writes only its zapped samples (zaps are rare)
__global__ void k_kad_zero(Frames F, int fd, int ncd, const long *zap)
{
    const long g = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const long per = (long)ncd * fd;
    if (g >= (long)F.nframes * per) return;
    const long f = g / per, j = g % per;
    const long *z = zap + 4 * (f * ncd + j / fd);
    for (int p = 0; p < 2; p++)
        for (long i = z[2 * p]; i < z[2 * p + 1]; i++) F.at(f, j, i) = 0.f;
}

// The same for time-major frames: one thread per channel and 64 samples, so
// that a long run is written by many workgroups and a wavefront's stores are
// consecutive channels.
constexpr int kKzT = 64;
__global__ __launch_bounds__(256) void k_kad_zero_tm(Frames F, int fd, int ncd, const long *zap)
{
    const int nch = ncd * fd;
    const long nct = (nch + 255) / 256, per = nct * ((F.nsamp + kKzT - 1) / kKzT);
    const long f = blockIdx.x / per, r = blockIdx.x % per;
    const int j = (int)(r % nct) * 256 + threadIdx.x;
    const long t0 = r / nct * kKzT, t1 = min(t0 + kKzT, F.nsamp);
    if (j >= nch) return;
    const long *z = zap + 4 * (f * ncd + j / fd);
    for (int p = 0; p < 2; p++)
        for (long i = max(t0, z[2 * p]); i < min(t1, z[2 * p + 1]); i++) F.at(f, j, i) = 0.f;
}

inline unsigned blocks_for(long n) { return (unsigned)((n + 255) / 256); }

// A launch holds fewer than 2^32 threads.  Frames of which each of the kernels
// here takes at most `threads` a frame go in slices of this many, one after the
// other on the stream.
inline int frames_per_launch(int nframes, long threads)
{
    return (int)std::max(1L, std::min((long)nframes, (1L << 31) / threads));
}
// Longest time-major frames of the kernels that take several threads a sample
// there (and number samples in 32 bits); longer ones take the general kernels.
constexpr long kMaxTmZdot = 1L << 28, kMaxTmKad = 1L << 26;

int check_frames(const Frames &F)
{
    if (!F.x || F.nframes < 0 || F.nchan < 1 || F.nsamp < 1 || F.cstride < 1 || F.tstride < 1 ||
        F.fstride < 0)
        return set_error(TX_EINVAL, "rfi: bad frame description");
    if ((long)F.nframes * F.nchan * F.nsamp > (1L << 40)) return set_error(TX_EINVAL, "rfi: frames too large");
    return TX_OK;
}

} // namespace

extern "C" size_t tx_rfi_work_bytes(int op, int nframes, int nchan, long nsamp, int td, int fd)
{
    if (nframes < 0 || nchan < 1 || nsamp < 1) return 0;
    if (op == TX_RFI_ZDOT) return (size_t)nframes * (nsamp + 2 + 2 * (size_t)nchan) * sizeof(double);
    if (op == TX_RFI_KADANEF) {
        if (td < 1 || fd < 1) return 0;
        const size_t ncd = nchan / fd, nsd = nsamp / td;
        const size_t ds = ((size_t)nframes * ncd * nsd * sizeof(float) + 255) / 256 * 256;
        return ds + (size_t)nframes * ncd * 4 * sizeof(long);
    }
    return 0;
}

extern "C" int tx_rfi_zdot(void *stream, float *data, int nframes, long fstride, int nchan, long nsamp,
                           long cstride, long tstride, void *work, size_t work_bytes)
{
    Frames F{data, fstride, cstride, tstride, nframes, nchan, nsamp};
    int rc = check_frames(F);
    if (rc) return rc;
    if (nframes == 0) return TX_OK;
    if (!work || work_bytes < tx_rfi_work_bytes(TX_RFI_ZDOT, nframes, nchan, nsamp, 1, 1))
        return set_error(TX_EINVAL, "rfi: work buffer smaller than tx_rfi_work_bytes");
    // at most 512 threads for 8 rows, 10 a sample, one for 32 samples of a channel
    const int most = frames_per_launch(nframes, 64L * nchan + 10 * nsamp + (nchan + 255L) * (nsamp + 31) / 32 + 1024);
    if (nframes > most) {
        for (int f = 0; f < nframes && rc == TX_OK; f += std::min(most, nframes - f))
            rc = tx_rfi_zdot(stream, data + f * fstride, std::min(most, nframes - f), fstride, nchan, nsamp, cstride,
                             tstride, work, work_bytes);
        return rc;
    }
    hipStream_t st = (hipStream_t)stream;
    double *s = (double *)work, *sess = s + (size_t)nframes * nsamp, *stat = sess + 2 * (size_t)nframes;
    const long nfc = (long)nframes * nchan, nfs = (long)nframes * nsamp;
    const double *cs = s, *css = sess;
    if (tstride == 1 && fstride == (long)nchan * nsamp && cstride == nsamp) {
        // the Candidate layout [nframes][nchan][nsamp]
        RowTile R = row_tile(nsamp);
        if (short_rows(nframes, nchan, nsamp)) R.RB = 0;
        if (R.RB) {
            const size_t shm = tile_lds(R.RB, nsamp);
            const unsigned nt = (unsigned)((nchan + R.RB - 1) / R.RB) * nframes;
            auto fit = k_zdot_tile_fit;
            (void)hipFuncSetAttribute((const void *)fit, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kTileLds);
            if (nframes >= frame_per_group(nchan, nsamp, R.RB)) {
                auto k = k_zdot_tile_stats<true>;
                (void)hipFuncSetAttribute((const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kTileLds);
                hipLaunchKernelGGL(k, dim3((unsigned)nframes), dim3(kTileThreads), shm, st, F, R, stat, s, sess);
            } else {
                auto k = k_zdot_tile_stats<false>;
                (void)hipFuncSetAttribute((const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kTileLds);
                hipLaunchKernelGGL(k, dim3(nt), dim3(kTileThreads), shm, st, F, R, stat, s, sess);
                hipLaunchKernelGGL(k_zdot_norm_mean, dim3((unsigned)((nsamp + 63) / 64 * nframes)), dim3(64), 0, st,
                                   F, (const double *)stat, s);
                hipLaunchKernelGGL(k_zdot_ss, dim3(blocks_for(nframes)), dim3(256), 0, st, F, cs, sess);
            }
            hipLaunchKernelGGL(fit, dim3(nt), dim3(kTileThreads), shm, st, F, R, (const double *)stat, cs, css);
        } else {
            const unsigned nb = (unsigned)((nfc + 255) / 256);
            hipLaunchKernelGGL(k_zdot_rows<false>, dim3(nb), dim3(256), 0, st, F, cs, css);
            hipLaunchKernelGGL(k_zdot_s, dim3(blocks_for(nfs)), dim3(256), 0, st, F, s);
            hipLaunchKernelGGL(k_zdot_ss, dim3(blocks_for(nframes)), dim3(256), 0, st, F, cs, sess);
            hipLaunchKernelGGL(k_zdot_rows<true>, dim3(nb), dim3(256), 0, st, F, cs, css);
        }
    } else if (cstride == 1 && fstride == (long)nchan * nsamp && tstride == nchan && nsamp <= kMaxTmZdot) {
        // the DataBuffer layout [nframes][nsamp][nchan]
        const unsigned ng = (unsigned)((nchan + kColCh - 1) / kColCh);
        const bool narrow = nchan < kColCh;
        const auto stats = narrow ? k_zdot_chain<false, true> : k_zdot_chain<false, false>;
        const auto fit = narrow ? k_zdot_chain<true, true> : k_zdot_chain<true, false>;
        hipLaunchKernelGGL(stats, dim3(ng * nframes), dim3(kColThreads), 0, st, F, cs, stat, sess);
        hipLaunchKernelGGL(k_zdot_norm_s, dim3((unsigned)((nsamp + kNsT - 1) / kNsT * nframes)), dim3(320), 0, st,
                           F, (const double *)stat, s);
        hipLaunchKernelGGL(fit, dim3((ng + 1) * nframes), dim3(kColThreads), 0, st, F, cs, stat, sess);
        hipLaunchKernelGGL(k_zdot_update,
                           dim3((unsigned)(((nchan + 255) / 256) * ((nsamp + kUpT - 1) / kUpT) * nframes)), dim3(256),
                           0, st, F, cs, (const double *)stat, css);
    } else {
        hipLaunchKernelGGL(k_zdot_norm, dim3(blocks_for(nfc)), dim3(256), 0, st, F);
        hipLaunchKernelGGL(k_zdot_s, dim3(blocks_for(nfs)), dim3(256), 0, st, F, s);
        hipLaunchKernelGGL(k_zdot_ss, dim3(blocks_for(nframes)), dim3(256), 0, st, F, cs, sess);
        hipLaunchKernelGGL(k_zdot_fit, dim3(blocks_for(nfc)), dim3(256), 0, st, F, cs, css);
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return set_error(TX_EHIP, std::string("rfi zdot: ") + hipGetErrorString(e));
    return TX_OK;
}

extern "C" int tx_rfi_kadanef(void *stream, float *data, int nframes, long fstride, int nchan, long nsamp,
                              long cstride, long tstride, int td, int fd, float threshold,
                              const int *wnlimit, void *work, size_t work_bytes)
{
    Frames F{data, fstride, cstride, tstride, nframes, nchan, nsamp};
    int rc = check_frames(F);
    if (rc) return rc;
    if (td < 1 || fd < 1) return set_error(TX_EINVAL, "rfi: td and fd must be >= 1");
    if (nframes == 0) return TX_OK;
    const int ncd = nchan / fd;
    const long nsd = nsamp / td;
    if (ncd == 0 || nsd == 0) return TX_OK; // nothing to downsample into
    if (!wnlimit) return set_error(TX_EINVAL, "rfi: null wnlimit");
    if (!work || work_bytes < tx_rfi_work_bytes(TX_RFI_KADANEF, nframes, nchan, nsamp, td, fd))
        return set_error(TX_EINVAL, "rfi: work buffer smaller than tx_rfi_work_bytes");
    // a thread for each downsampled sample or for 64 samples of a channel, 256 for 8 downsampled channels
    const int most = frames_per_launch(nframes, ncd * nsd + (ncd + 255L) * (nsd + 7) / 8 +
                                                    (nchan + 255L) * (nsamp + 63) / 64 + 33L * nchan + 1024);
    if (nframes > most) {
        for (int f = 0; f < nframes && rc == TX_OK; f += std::min(most, nframes - f))
            rc = tx_rfi_kadanef(stream, data + f * fstride, std::min(most, nframes - f), fstride, nchan, nsamp,
                                cstride, tstride, td, fd, threshold, wnlimit + f, work, work_bytes);
        return rc;
    }
    hipStream_t st = (hipStream_t)stream;
    float *ds = (float *)work;
    long *zap = (long *)((char *)work + ((size_t)nframes * ncd * nsd * sizeof(float) + 255) / 256 * 256);
    if (cstride == 1 && fstride == (long)nchan * nsamp && tstride == nchan && ncd >= kColCh && nsamp <= kMaxTmKad) {
        // the DataBuffer layout [nframes][nsamp][nchan]
        const long nct = (ncd + 255) / 256, nzt = ((long)ncd * fd + 255) / 256;
        hipLaunchKernelGGL(k_kad_down_tm, dim3((unsigned)(nct * ((nsd + kKdT - 1) / kKdT) * nframes)), dim3(256), 0,
                           st, F, td, fd, ncd, nsd, ds);
        hipLaunchKernelGGL(k_kad_scan_tm, dim3((unsigned)((ncd + kColCh - 1) / kColCh * nframes)), dim3(kColThreads), 0,
                           st, ncd, nsd, td, fd, threshold, wnlimit, (const float *)ds, zap);
        hipLaunchKernelGGL(k_kad_zero_tm, dim3((unsigned)(nzt * ((nsamp + kKzT - 1) / kKzT) * nframes)), dim3(256), 0,
                           st, F, fd, ncd, (const long *)zap);
    } else if (const int G = tstride == 1 && fstride == (long)nchan * nsamp && cstride == nsamp ? kad_rows(nsd, td, fd) : 0) {
        // the Candidate layout [nframes][nchan][nsamp]
        hipLaunchKernelGGL(k_kad_rows, dim3((unsigned)((ncd + G - 1) / G * nframes)), dim3(256),
                           (size_t)G * (nsd | 1) * 4, st, F, td, fd, ncd, (int)nsd, G, threshold, wnlimit);
    } else {
        hipLaunchKernelGGL(k_kad_down, dim3(blocks_for((long)nframes * ncd * nsd)), dim3(256), 0, st, F, td, fd,
                           ncd, nsd, ds);
        const auto scan = nsd < 1L << 31 ? k_kad_scan<int> : k_kad_scan<long>;
        hipLaunchKernelGGL(scan, dim3(blocks_for((long)nframes * ncd)), dim3(256), 0, st, nframes, ncd, nsd,
                           td, fd, threshold, wnlimit, (const float *)ds, zap);
        hipLaunchKernelGGL(k_kad_zero, dim3(blocks_for((long)nframes * ncd * fd)), dim3(256), 0, st, F, fd, ncd,
                           (const long *)zap);
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return set_error(TX_EHIP, std::string("rfi kadaneF: ") + hipGetErrorString(e));
    return TX_OK;
}
