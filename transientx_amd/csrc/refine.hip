// refine.hip -- the candidate refinement grid on gfx950: Candidate::dedisperse
// (incoherent), Candidate::optimize with the dedispersion tree of
// include/hough_transform.h, and Candidate::matched_filter
// (src/singlepulse/candidate.cpp:108-140,899-1087), for a batch of cutouts.
//
//   R1 k_tree_pass   a run of tree levels [a, b) in LDS.  After level l the
//                    rows form nodes of 2^(l+1) channels; row k of node j is
//                    A[k mod 2^l][i] + B[k mod 2^l][(i + s) mod ncol] with s
//                    the rounded delay between the nodes' leading channels at
//                    DM trial bitrev(k).  Row k of a node after level b-1
//                    only needs row (k mod 2^a) of each of its 2^(b-a)
//                    descendants at level a-1, so one workgroup takes such a
//                    group of rows through all levels of the pass.  The
//                    first pass loads the cutout (band order, padding and the
//                    incoherent shift fused in); the last one writes the DM
//                    rows in trial order.
//                    (k_tree_rows: rows of 32 to 2048 samples, a wave to a
//                    pair of rows.)
//   R2 k_mf_rows     rows in LDS: one lane per DM row for the sequential parts
//                    (FP64 mean/variance, the FP32 circular running sum, in the
//                    reference's order), then a wavefront per row for the width
//                    loop; per-row first maximum.  Longer rows: k_mf_scan for
//                    the sequential parts, k_mf_box for the widths.
//   R3 k_argmax      first maximum of each cutout's S/N map (row-major).
//
// All sums are elementwise FP32 adds (tree) or sequential in the reference's
// order (matched filter), so the maps are bit-identical to the restatement.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <string>
#include <vector>

#include "../../include/txgpu.h"
#include "device_util.h"

namespace txgpu {
int set_error(int code, const std::string &msg);
}
using txgpu::f4v;
using txgpu::lds_f4;
using txgpu::lds_fill;
using txgpu::lds_fill16;
using txgpu::ldc;
using txgpu::wave_max_f;
using txgpu::wave_min_i;
using txgpu::lds_fill_done;
using txgpu::set_error;

namespace {

constexpr int kTreeLdsFloats = 16384; // 64 KB of rows per tree workgroup
constexpr int kMaxItems = 16;         // pair items per thread per chunk (256 threads)
constexpr int kMaxMfBox = 64;
// Row lengths of k_tree_rows, beside k_tree_pass: the whole grid of 128 cutouts
// of 1024 channels takes 226 us against 301 at 32 samples, 253 against 359 at
// 64, 308 against 460 at 128; 64 cutouts 1256 against 1800 at 1000 samples, 32
// cutouts 2783 against 2876 at 2048.  Shorter rows would leave most of a wave
// idle, longer ones do not fit its registers.
constexpr int kTreeRowsMin = 32, kTreeRowsMax = 2048;
// Longest rows of k_mf_rows, beside k_mf_scan and k_mf_box, without and with
// maps: the same grids take 253 us against 371 at 64 samples, 308 against 458 at
// 128, 1256 against 1487 at 1000, 2783 against 3221 at 2048 without; with maps
// 629 against 742 at 512 but 1092 against 1090 at 700 and 1643 against 1515 at
// 1000 (too few rows fit LDS, and a width needs two reads a sample).
constexpr int kMfRowsMax = 2048, kMfMapsMax = 512;
// Bytes of LDS per k_mf_rows workgroup: three to a CU (512 samples, 256 cutouts:
// 824 us; four to a CU 843, two 939).
constexpr int kMfRowsLds = 52 * 1024;
// Rows of no whole 16-byte lines read LDS a word at a time; over 1536 samples
// four or three such rows fit a workgroup, and k_mf_scan, which does not
// depend on it, is the faster from about 18 x 1024 rows on: 1901 samples 1.04
// of its time at 20 x 1024 rows, 1.23 at 64, 0.82 at 8; 1601 samples 0.97, 1.18
// and 0.76; 1501 samples 0.91 at 64.  Where four rows fit and k_mf_box's rows
// leave room for two workgroups per CU, not three, only from 64 x 1024 rows on
// (1801 samples 0.89 at 24, 1.00 at 64).
inline bool mf_word_rows(int nbin, int rows, long nrows)
{
    return nbin <= 1536 || nrows <= (rows < 4 || 3 * (32 * nbin + 2048) <= 160 * 1024 ? 18 : 64) * 1024L;
}

// include/candidate.h:116-119, no contraction (the reference computes it as written)
__device__ __host__ inline double dmdelay(double dm, double fh, double fl)
{
#pragma clang fp contract(off)
    return 4.148741601e3 * dm * (1. / (fl * fl) - 1. / (fh * fh));
}

// get_shift of src/singlepulse/candidate.cpp:970-974 (dms + p*ddm contracted
// to an FMA as the reference's -mfma build does) and the modulo of
// include/hough_transform.h:88-89.
__device__ inline int tree_shift(double fh, double fl, int p, double dms, double ddm, double dm0,
                                 double tbin, int ncol)
{
#pragma clang fp contract(off)
    const double dm = fma((double)p, ddm, dms) - dm0;
    int s = (int)round(dmdelay(dm, fh, fl) / tbin);
    s %= ncol;
    if (s < 0) s += ncol;
    return s;
}

__device__ inline int bitrev(int k, int n) { return (int)(__builtin_bitreverse32((unsigned)k) >> (32 - n)); }

struct TreeArgs {
    const float *src;   // first pass: cutouts [ncand][nchan][ncol]; else rows [ncand][nrow][ncol]
    float *dst;         // rows [ncand][nrow][ncol] (node layout, or DM order in the last pass)
    const double *fP;   // [nrow] frequency of buffer row j (from the highest)
    const int *srcrow;  // [nrow] cutout channel of buffer row j, -1 for padding
    const double *fsrc; // [nchan] cutout channel frequencies
    const double *dms, *ddm, *dm0, *dmc; // per cutout
    double fmax, tbin;
    int nchan, nrow, n, ncol;
    int a, b;
    int first, last, dedisperse;
};

__global__ __launch_bounds__(256) void k_tree_pass(TreeArgs A)
{
    extern __shared__ float rows[];
    __shared__ int sh[2048]; // G <= 1024: shifts of <= 512 pairs, or G row delays
    const int tid = threadIdx.x;
    const int c = blockIdx.y;
    const int G = 1 << (A.b - A.a);
    const int g = (int)(blockIdx.x >> A.a), rho = (int)(blockIdx.x & ((1u << A.a) - 1));
    const int ncol = A.ncol;
    const double dms = A.dms[c], ddm = A.ddm[c], dm0 = A.dm0[c];

    // ---- load the group's G rows
    if (A.first) {
        // Candidate::dedisperse: cutout channel q rotated left by its delay at dmc
        for (int t = tid; t < G; t += 256) {
            const int q = A.srcrow[g * G + t];
            int d = 0;
            if (q >= 0 && A.dedisperse) {
                d = (int)round(dmdelay(A.dmc[c], A.fmax, A.fsrc[q]) / A.tbin);
                d %= ncol;
                if (d < 0) d += ncol;
            }
            sh[t] = d;
        }
        __syncthreads();
        const float *cut = A.src + (size_t)c * A.nchan * ncol;
        const int wave = tid >> 6, lane = tid & 63;
        for (int t = wave; t < G; t += 4) {
            const int q = A.srcrow[g * G + t];
            float *dst = rows + (size_t)t * ncol;
            if (q < 0) {
                for (int i = lane; i < ncol; i += 64) dst[i] = 0.f;
                continue;
            }
            // the row rotated left by d: [d, ncol) then [0, d)
            const int d = sh[t];
            const uint32_t *srow = (const uint32_t *)(cut + (size_t)q * ncol);
            lds_fill(srow + d, (uint32_t *)dst, ncol - d, 0, 1, lane);
            if (d) lds_fill(srow, (uint32_t *)dst + (ncol - d), d, 0, 1, lane);
        }
    } else {
        const float *in = A.src + (size_t)c * A.nrow * ncol;
        const int wave = tid >> 6, lane = tid & 63;
        for (int t = wave; t < G; t += 4)
            lds_fill((const uint32_t *)(in + ((size_t)(g * G + t) * (1 << A.a) + rho) * ncol),
                     (uint32_t *)(rows + (size_t)t * ncol), ncol, 0, 1, lane);
    }
    lds_fill_done();

    // ---- levels a .. b-1, in place
    const int pairs = G / 2;
    const int P = max(1, 4096 / ncol); // pairs per chunk: <= 16 items per thread
    // item -> (pair, column) and pair -> (row pair, offset) by shifts where
    // the sizes are powers of two (half always is; ncol usually)
    const bool p2 = (ncol & (ncol - 1)) == 0;
    const int lc = __builtin_ctz((unsigned)ncol);
    for (int l = A.a; l < A.b; l++) {
        const int half = 1 << (l - A.a), hs = l - A.a;
        for (int q = tid; q < pairs; q += 256) {
            const int jl = q >> hs, t = q & (half - 1);
            const int jg = (g << (A.b - l - 1)) + jl;
            const int x0 = jg << (l + 1), x1 = x0 + (1 << l);
            const int k0 = rho + (t << A.a), k1 = k0 + (1 << l);
            sh[2 * q] = tree_shift(A.fP[x0], A.fP[x1], bitrev(k0, A.n), dms, ddm, dm0, A.tbin, ncol);
            sh[2 * q + 1] = tree_shift(A.fP[x0], A.fP[x1], bitrev(k1, A.n), dms, ddm, dm0, A.tbin, ncol);
        }
        __syncthreads();
        for (int q0 = 0; q0 < pairs; q0 += P) {
            const int items = min(P, pairs - q0) * ncol;
            float o0[kMaxItems], o1[kMaxItems];
#pragma unroll
            for (int u = 0; u < kMaxItems; u++) {
                const int idx = tid + 256 * u;
                if (idx < items) {
                    const int q = q0 + (p2 ? idx >> lc : idx / ncol), i = p2 ? idx & (ncol - 1) : idx % ncol;
                    const int jl = q >> hs, t = q & (half - 1);
                    const float *Ar = rows + (size_t)(2 * jl * half + t) * ncol;
                    const float *Br = Ar + (size_t)half * ncol;
                    int i0 = i + sh[2 * q], i1 = i + sh[2 * q + 1];
                    if (i0 >= ncol) i0 -= ncol;
                    if (i1 >= ncol) i1 -= ncol;
                    const float av = Ar[i];
                    o0[u] = av + Br[i0];
                    o1[u] = av + Br[i1];
                }
            }
            __syncthreads();
#pragma unroll
            for (int u = 0; u < kMaxItems; u++) {
                const int idx = tid + 256 * u;
                if (idx < items) {
                    const int q = q0 + (p2 ? idx >> lc : idx / ncol), i = p2 ? idx & (ncol - 1) : idx % ncol;
                    const int jl = q >> hs, t = q & (half - 1);
                    float *Ar = rows + (size_t)(2 * jl * half + t) * ncol;
                    Ar[i] = o0[u];
                    Ar[(size_t)half * ncol + i] = o1[u];
                }
            }
            __syncthreads();
        }
    }

    // ---- store: node layout, or DM order after the last level
    float *out = A.dst + (size_t)c * A.nrow * ncol;
    for (int idx = tid; idx < G * ncol; idx += 256) {
        const int t = p2 ? idx >> lc : idx / ncol, i = idx - t * ncol;
        const int k = rho + (t << A.a);
        const int r = A.last ? bitrev(k, A.n) : g * (1 << A.b) + k;
        out[(size_t)r * ncol + i] = rows[idx];
    }
}

// The same pass for rows of at most 64*U samples: a wave takes whole row pairs,
// U columns a lane, all of a pair's reads in registers before its two rows
// are written, so that the levels need one barrier each; the shifts of every
// level are formed together at the start (their FP64 divisions are a long
// chain, which each level used to wait for); rows go out 16 bytes a lane where
// ncol allows.  P2: ncol is a power of two, and a wrap is a mask.
// 256 cutouts of 1024 x 512, five levels a pass: 258 us a pass, k_tree_pass 865;
// 1.07 GB read and written, 216 us at a copy's rate, bounds it.
// U steps close enough that few of a wave's steps lie past the row's end: whole
// grids with maps, 48 cutouts of 1024 x 1025, 1838 us with 20 columns a lane, 2309
// with 32, 2152 with k_tree_pass.
template <int U, bool P2>
__global__ __launch_bounds__(512) void k_tree_rows(TreeArgs A)
{
    extern __shared__ __attribute__((aligned(16))) float rows[]; // [G][ncol], then the shifts: G a level (or G row delays)
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = blockIdx.y;
    const int G = 1 << (A.b - A.a);
    int *sh = (int *)(rows + (size_t)G * A.ncol);
    const int g = (int)(blockIdx.x >> A.a), rho = (int)(blockIdx.x & ((1u << A.a) - 1));
    const int ncol = A.ncol;

    // ---- load the group's G rows, as k_tree_pass does
    if (A.first) {
        for (int t = tid; t < G; t += 512) {
            const int q = A.srcrow[g * G + t];
            int d = 0;
            if (q >= 0 && A.dedisperse) {
                d = (int)round(dmdelay(A.dmc[c], A.fmax, A.fsrc[q]) / A.tbin);
                d %= ncol;
                if (d < 0) d += ncol;
            }
            sh[t] = d;
        }
        __syncthreads();
        const float *cut = A.src + (size_t)c * A.nchan * ncol;
        for (int t = wave; t < G; t += 8) {
            const int q = A.srcrow[g * G + t];
            float *dst = rows + (size_t)t * ncol;
            if (q < 0) {
                for (int i = lane; i < ncol; i += 64) dst[i] = 0.f;
                continue;
            }
            const int d = sh[t]; // the row rotated left by d: [d, ncol) then [0, d)
            const uint32_t *srow = (const uint32_t *)(cut + (size_t)q * ncol);
            lds_fill(srow + d, (uint32_t *)dst, ncol - d, 0, 1, lane);
            if (d) lds_fill(srow, (uint32_t *)dst + (ncol - d), d, 0, 1, lane);
        }
        __syncthreads(); // sh is free again
    } else {
        const float *in = A.src + (size_t)c * A.nrow * ncol;
        for (int t = wave; t < G; t += 8)
            lds_fill((const uint32_t *)(in + ((size_t)(g * G + t) * (1 << A.a) + rho) * ncol),
                     (uint32_t *)(rows + (size_t)t * ncol), ncol, 0, 1, lane);
    }
    const int pairs = G / 2;
    const double dms = A.dms[c], ddm = A.ddm[c], dm0 = A.dm0[c];
    for (int e = tid; e < (A.b - A.a) * 2 * pairs; e += 512) {
        const int l = A.a + e / (2 * pairs), q = (e % (2 * pairs)) >> 1;
        const int hs = l - A.a, jl = q >> hs, t = q & ((1 << hs) - 1);
        const int jg = (g << (A.b - l - 1)) + jl;
        const int x0 = jg << (l + 1), x1 = x0 + (1 << l);
        const int k = rho + (t << A.a) + ((e & 1) << l);
        sh[e] = tree_shift(A.fP[x0], A.fP[x1], bitrev(k, A.n), dms, ddm, dm0, A.tbin, ncol);
    }
    lds_fill_done();

    // ---- levels a .. b-1, in place
    for (int l = A.a; l < A.b; l++) {
        const int hs = l - A.a, half = 1 << hs;
        for (int q = wave; q < pairs; q += 8) {
            const int jl = q >> hs, t = q & (half - 1);
            float *Ar = rows + (size_t)(2 * jl * half + t) * ncol;
            float *Br = Ar + (size_t)half * ncol;
            const int s0 = sh[hs * 2 * pairs + 2 * q], s1 = sh[hs * 2 * pairs + 2 * q + 1];
            float av[U], b0[U], b1[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int i = lane + 64 * u;
                int i0 = i + s0, i1 = i + s1;
                if (P2) {
                    i0 &= ncol - 1;
                    i1 &= ncol - 1;
                } else {
                    i0 -= i0 >= ncol ? ncol : 0;
                    i1 -= i1 >= ncol ? ncol : 0;
                }
                if (64 * U == ncol || i < ncol) {
                    av[u] = Ar[i];
                    b0[u] = Br[i0];
                    b1[u] = Br[i1];
                }
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int i = lane + 64 * u;
                if (64 * U == ncol || i < ncol) {
                    Ar[i] = av[u] + b0[u];
                    Br[i] = av[u] + b1[u];
                }
            }
        }
        __syncthreads();
    }

    // ---- store: node layout, or DM order after the last level
    float *out = A.dst + (size_t)c * A.nrow * ncol;
    for (int t = wave; t < G; t += 8) {
        const int k = rho + (t << A.a);
        const int r = A.last ? bitrev(k, A.n) : g * (1 << A.b) + k;
        const float *row = rows + (size_t)t * ncol;
        float *o = out + (size_t)r * ncol;
        if (ncol % 4 == 0 && ((uintptr_t)A.dst & 15) == 0) {
            for (int i = 4 * lane; i < ncol; i += 256) *(float4 *)(o + i) = *(const float4 *)(row + i);
        } else {
            for (int i = lane; i < ncol; i += 64) o[i] = row[i];
        }
    }
}

auto tree_rows_kernel(int ncol) -> void (*)(TreeArgs)
{
    const bool p2 = (ncol & (ncol - 1)) == 0;
    if (ncol <= 128) return p2 ? k_tree_rows<2, true> : k_tree_rows<2, false>;
    if (ncol <= 256) return p2 ? k_tree_rows<4, true> : k_tree_rows<4, false>;
    if (ncol <= 512) return p2 ? k_tree_rows<8, true> : k_tree_rows<8, false>;
    if (ncol <= 1024) return p2 ? k_tree_rows<16, true> : k_tree_rows<16, false>;
    if (ncol <= 1280) return k_tree_rows<20, false>;
    if (ncol <= 1536) return k_tree_rows<24, false>;
    return p2 ? k_tree_rows<32, true> : k_tree_rows<32, false>;
}

struct MfArgs {
    const float *dmt; // [rows][ncol]
    float *cs;        // [rows][2*ncol] circular running sums
    float *snr;       // [rows][ncol] or null
    int *wid;         // [rows][ncol] or null
    float *rowmax;
    int *rowarg, *rowwid;
    double *var;      // [rows] variance of each row (get_mean_var)
    const int *vwn;
    int nbox;
    long nrows;
    int ncol;
    const int *pick; // workgroup c takes row pick[c] of cutout c (nrows per cutout); else null
};

// Sequential parts of matched_filter: one 64-lane workgroup per 64 DM rows,
// one lane per row.
__global__ __launch_bounds__(64) void k_mf_scan(MfArgs M)
{
    extern __shared__ float smem[];
    float *stage = smem; // [64][65]
    const int lane = threadIdx.x;
    const long R0 = (long)blockIdx.x * 64;
    const long row = R0 + lane;
    const bool live = row < M.nrows;
    const int ncol = M.ncol;

    // get_mean_var: sequential FP64 sums (one lane per row)
    double m = 0., v = 0.;
    const int nr = (int)min((long)64, M.nrows - R0);
    for (int i0 = 0; i0 < ncol; i0 += 64) {
        for (int cc = 0; cc < nr; cc++)
            lds_fill((const uint32_t *)(M.dmt + (R0 + cc) * ncol + i0), (uint32_t *)(stage + cc * 65),
                     min(64, ncol - i0), 0, 1, lane);
        lds_fill_done();
        const int nn = min(64, ncol - i0);
        for (int ii = 0; ii < nn; ii++) {
            const double x = (double)stage[lane * 65 + ii];
            m += x;
            v = fma(x, x, v);
        }
        __syncthreads();
    }
    m /= ncol;
    v /= ncol;
    v = fma(-m, m, v);

    // csump over 2*ncol samples: (double)csum + (x - mean), rounded to float each step
    float csum = 0.f;
    for (int i0 = 0; i0 < 2 * ncol; i0 += 64) {
        const int e = i0 + lane;
        // samples e in [i0, i0 + 64) of the doubled row are x[e mod ncol]: up to two pieces
        const int end = min(i0 + 64, 2 * ncol);
        const int cut = (i0 < ncol && end > ncol) ? ncol : end;
        for (int cc = 0; cc < nr; cc++) {
            const float *xr = M.dmt + (R0 + cc) * ncol;
            const int s0 = i0 < ncol ? i0 : i0 - ncol;
            lds_fill((const uint32_t *)(xr + s0), (uint32_t *)(stage + cc * 65), cut - i0, 0, 1, lane);
            if (cut < end) lds_fill((const uint32_t *)xr, (uint32_t *)(stage + cc * 65 + (cut - i0)), end - cut, 0, 1, lane);
        }
        lds_fill_done();
        const int nn = min(64, 2 * ncol - i0);
        for (int ii = 0; ii < nn; ii++) {
            csum = (float)((double)csum + ((double)stage[lane * 65 + ii] - m));
            stage[lane * 65 + ii] = csum;
        }
        __syncthreads();
        for (int cc = 0; cc < 64; cc++) {
            const long r = R0 + cc;
            if (r < M.nrows && e < 2 * ncol) M.cs[r * 2 * ncol + e] = stage[cc * 65 + lane];
        }
        __syncthreads();
    }

    if (live) M.var[row] = v;
}

// Width loop of matched_filter: one wavefront per DM row (4 rows per
// workgroup), the row's running sums staged in LDS; U samples per lane.
template <int U>
__global__ __launch_bounds__(256) void k_mf_box(MfArgs M)
{
    extern __shared__ float smem[];
    const int ncol = M.ncol;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const long r = (long)blockIdx.x * 4 + w;
    const bool live = r < M.nrows;
    float *crow = smem + (size_t)w * 2 * ncol;
    if (live) lds_fill((const uint32_t *)(M.cs + r * 2 * ncol), (uint32_t *)crow, 2 * ncol, 0, 1, lane);
    lds_fill_done();
    if (!live) return;
    const double var = M.var[r];
    float vS[U];
    int vW[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
        vS[u] = 0.f;
        vW[u] = 0;
    }
    if (var > 0) {
        // each width's scale computed once per row, by lane k (FP64 sqrt and
        // divide, the same expression), and read back with v_readlane
        const bool lanes = M.nbox <= 64;
        const float tp = lanes && lane < M.nbox ? (float)sqrt(1. / (M.vwn[lane] * var)) : 0.f;
        for (int k = 0; k < M.nbox; k++) {
            const int wn = M.vwn[k], wl = wn / 2 + 1, wh = (wn - 1) / 2;
            const float temp = lanes ? __int_as_float(__builtin_amdgcn_readlane(__float_as_int(tp), k))
                                     : (float)sqrt(1. / (wn * var));
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int o = lane + 64 * u;
                if (o < ncol) {
                    const int i = o >= wl ? o : o + ncol;
                    const float S = (crow[i + wh] - crow[i - wl]) * temp;
                    if (S >= vS[u]) {
                        vS[u] = S;
                        vW[u] = wn;
                    }
                }
            }
        }
    }
    float best = -INFINITY;
    int bo = 0x7fffffff, bw = 0;
#pragma unroll
    for (int u = 0; u < U; u++) {
        const int o = lane + 64 * u;
        if (o < ncol) {
            if (M.snr) M.snr[r * ncol + o] = vS[u];
            if (M.wid) M.wid[r * ncol + o] = vW[u];
            if (vS[u] > best) {
                best = vS[u];
                bo = o;
                bw = vW[u];
            }
        }
    }
    // first maximum of the row: larger value, then smaller sample
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const float ob = __shfl_xor(best, off, 64);
        const int oo = __shfl_xor(bo, off, 64);
        const int ow = __shfl_xor(bw, off, 64);
        if (ob > best || (ob == best && oo < bo)) {
            best = ob;
            bo = oo;
            bw = ow;
        }
    }
    if (lane == 0) {
        M.rowmax[r] = best;
        M.rowarg[r] = bo;
        M.rowwid[r] = bw;
    }
}

// Both parts in one kernel for rows short enough that a workgroup holds a few
// of them in LDS: the running sums (2*ncol a row, written and read back between
// the two kernels) never leave the chip.  A width needs samples j and j + wn of
// the doubled row for every j < ncol, so the sums end at ncol + W, W the widest
// width (rounded up to 4 words with V4), and a row is ncol + W words: it is
// loaded with its first W samples behind the others, where the second lap finds
// them, and the sums take the samples' places.  One wave forms the rows' means
// and another their mean squares at the same time, a lane a row; the first then
// runs the sums, and the four waves take the rows' widths, 64*CU samples at a
// time.  256 cutouts of 1024 x 512 without maps: 824 us and 38 us for the 256
// best rows, k_mf_scan and k_mf_box 684 + 1031.  The chains of FP64 conversions
// and adds bound it (three a CU, as many as LDS has room for: 305 us without
// them, 585 without the widths).
struct MfRow {
    int nrows;  // rows per workgroup
    int pitch;  // words from row to row: odd, or an odd multiple of 4 with V4
    int W;
    int nchunk; // pieces of 64*CU samples
};

// f(i, the four samples from i) for i = 0, 4, ... of a run of LDS, read 16
// ahead (the compiler would put each read before its use, and the wave wait).
template <typename F> __device__ __forceinline__ void mf_walk4(const float *x, int len, F f)
{
    if (len <= 0) return;
    f4v nx[4];
#pragma unroll
    for (int q = 0; q < 4; q++) nx[q] = lds_f4(x + min(4 * q, len - 4));
    for (int i = 0; i < len; i += 16) {
        f4v cur[4];
#pragma unroll
        for (int q = 0; q < 4; q++) {
            cur[q] = nx[q];
            nx[q] = lds_f4(x + min(i + 16 + 4 * q, len - 4));
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int q = 0; q < 4; q++)
            if (i + 4 * q < len) f(i + 4 * q, cur[q]);
    }
}

// Sequential FP64 sum of the samples (SQ: of their squares).
template <bool V4, bool SQ> __device__ __forceinline__ void mf_sum(const float *x, int len, double &acc)
{
    auto step = [&](float f) {
        const double d = (double)f;
        acc = SQ ? fma(d, d, acc) : acc + d;
    };
    if (V4) {
        mf_walk4(x, len, [&](int, f4v c) {
#pragma unroll
            for (int e = 0; e < 4; e++) step(c[e]);
        });
    } else {
#pragma unroll 8
        for (int i = 0; i < len; i++) step(x[i]);
    }
}

// csump: (double)csum + (x - mean), rounded to float each step.
template <bool V4> __device__ __forceinline__ void mf_csum(const float *x, float *out, int len, double m, float &csum)
{
    auto step = [&](float f) { return csum = (float)((double)csum + ((double)f - m)); };
    if (V4) {
        mf_walk4(x, len, [&](int i, f4v c) {
            f4v o;
#pragma unroll
            for (int e = 0; e < 4; e++) o[e] = step(c[e]);
            *(f4v *)__builtin_assume_aligned(out + i, 16) = o;
        });
    } else {
        float nx[8];
#pragma unroll
        for (int q = 0; q < 8; q++) nx[q] = x[min(q, len - 1)];
        for (int i = 0; i < len; i += 8) {
            float cur[8];
#pragma unroll
            for (int q = 0; q < 8; q++) {
                cur[q] = nx[q];
                nx[q] = x[min(i + 8 + q, len - 1)];
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int q = 0; q < 8; q++)
                if (i + q < len) out[i + q] = step(cur[q]);
        }
    }
}

template <int CU, bool V4, bool MAPS>
__global__ __launch_bounds__(256) void k_mf_rows(MfArgs M, MfRow T)
{
    extern __shared__ __attribute__((aligned(16))) float smem[];
    __shared__ double smean[64], svar[64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int ncol = M.ncol, W = T.W;
    const long R0 = M.pick ? (long)blockIdx.x * M.nrows + M.pick[blockIdx.x] : (long)blockIdx.x * T.nrows;
    // the waves of a workgroup go to the four SIMDs in order: the workgroups of
    // a CU (256 apart) run their chains on different ones
    const int chain = (blockIdx.x >> 8) & 3;
    const int nr = M.pick ? 1 : (int)min((long)T.nrows, M.nrows - R0);
    for (int t = wave; t < nr; t += 4) {
        const uint32_t *x = (const uint32_t *)(M.dmt + (R0 + t) * ncol);
        uint32_t *B = (uint32_t *)(smem + t * T.pitch);
        if (V4) {
            lds_fill16(x, B + ncol, W, 0, 1, lane);
            lds_fill16(x + W, B + W, ncol - W, 0, 1, lane);
        } else {
            lds_fill(x, B + ncol, W, 0, 1, lane);
            lds_fill(x + W, B + W, ncol - W, 0, 1, lane);
        }
    }
    lds_fill_done();
    float *row = smem + lane * T.pitch;
    if (wave == chain && lane < nr) {
        double m = 0.;
        mf_sum<V4, false>(row + ncol, W, m);
        mf_sum<V4, false>(row + W, ncol - W, m);
        smean[lane] = m / ncol;
    } else if (wave == (chain ^ 1) && lane < nr) {
        double v = 0.;
        mf_sum<V4, true>(row + ncol, W, v);
        mf_sum<V4, true>(row + W, ncol - W, v);
        svar[lane] = v / ncol;
    }
    __syncthreads();
    if (wave == chain && lane < nr) {
        const double m = smean[lane];
        float csum = 0.f;
        mf_csum<V4>(row + ncol, row, W, m, csum);
        mf_csum<V4>(row + W, row + W, ncol - W, m, csum);
        mf_csum<V4>(row + ncol, row + ncol, W, m, csum);
        svar[lane] = fma(-m, m, svar[lane]);
    }
    __syncthreads();
    const int nbox = M.nbox;
    // every row's scales: row t's at scale[64*t]
    float *scale = smem + (size_t)T.nrows * T.pitch + 64 * CU * T.nchunk;
    for (int e = threadIdx.x; e < nr * nbox; e += 256) {
        const int t = e / nbox, k = e - t * nbox;
        scale[64 * t + k] = (float)sqrt(1. / (M.vwn[k] * svar[t]));
    }
    __syncthreads();
    if (MAPS) {
        for (int t = wave; t < nr; t += 4) {
            const long r = R0 + t;
            const float *B = smem + t * T.pitch;
            float best = -INFINITY;
            int bo = 0x7fffffff, bw = 0;
            for (int h = 0; h < T.nchunk; h++) {
                float vS[CU];
                int vW[CU];
#pragma unroll
                for (int u = 0; u < CU; u++) {
                    vS[u] = 0.f;
                    vW[u] = 0;
                }
                const int h0 = h * 64 * CU + lane;
                if (svar[t] > 0)
                    for (int k = 0; k < nbox; k++) {
                        const int wn = ldc(M.vwn, k), wl = wn / 2 + 1, wh = (wn - 1) / 2;
                        const float temp = scale[64 * t + k];
#pragma unroll
                        for (int u = 0; u < CU; u++) {
                            const int o = min(h0 + 64 * u, ncol - 1);
                            const int i = o >= wl ? o : o + ncol;
                            const float S = (B[i + wh] - B[i - wl]) * temp;
                            if (S >= vS[u]) {
                                vS[u] = S;
                                vW[u] = wn;
                            }
                        }
                    }
#pragma unroll
                for (int u = 0; u < CU; u++) {
                    const int o = h0 + 64 * u;
                    if (o < ncol) {
                        if (M.snr) M.snr[r * ncol + o] = vS[u];
                        if (M.wid) M.wid[r * ncol + o] = vW[u];
                        if (vS[u] > best) {
                            best = vS[u];
                            bo = o;
                            bw = vW[u];
                        }
                    }
                }
            }
            // first maximum of the row: larger value, then smaller sample
            const float rb = wave_max_f(best);
            const int first = wave_min_i(best == rb ? bo : 0x7fffffff);
            if (bo == first) {
                const long w = M.pick ? blockIdx.x : r;
                if (!M.pick) M.rowmax[r] = rb;
                M.rowarg[w] = bo;
                M.rowwid[w] = bw;
            }
        }
        return;
    }
    // Without maps only a row's largest S/N is wanted (its time and width only
    // for each cutout's best row, which is then taken once more).  A width's
    // largest S/N is its largest difference times the scale (both roundings
    // keep the order, and a NaN never counts), so the scale is applied once a
    // lane; sample j of a width belongs to time (j + wl) mod ncol, and B[j]
    // serves every width.
    for (int t = wave; t < nr; t += 4) {
        const float *B = smem + t * T.pitch;
        float best = 0.f;
        if (svar[t] > 0) {
            const float *sc = scale + 64 * t;
            for (int h = 0; h < T.nchunk; h++) {
                const int j0 = h * 64 * CU + lane;
                float c0[CU];
#pragma unroll
                for (int u = 0; u < CU; u++) c0[u] = j0 + 64 * u < ncol ? B[j0 + 64 * u] : INFINITY;
                for (int k = 0; k < nbox; k += 2) {
                    const int k2 = min(k + 1, nbox - 1);
                    const float *B1 = B + j0 + ldc(M.vwn, k), *B2 = B + j0 + ldc(M.vwn, k2);
                    const float t1 = sc[k], t2 = sc[k2];
                    float c1[CU], c2[CU], d1 = -INFINITY, d2 = -INFINITY;
#pragma unroll
                    for (int u = 0; u < CU; u++) c1[u] = B1[64 * u];
#pragma unroll
                    for (int u = 0; u < CU; u++) c2[u] = B2[64 * u];
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int u = 0; u < CU; u++) d1 = fmaxf(d1, c1[u] - c0[u]);
#pragma unroll
                    for (int u = 0; u < CU; u++) d2 = fmaxf(d2, c2[u] - c0[u]);
                    best = fmaxf(best, fmaxf(d1 * t1, d2 * t2));
                }
            }
        }
        best = wave_max_f(best);
        if (lane == 0) M.rowmax[R0 + t] = best;
    }
}

template <bool V4, bool MAPS> auto mf_rows_kernel(int cu) -> void (*)(MfArgs, MfRow)
{
    switch (cu) {
    case 1: return k_mf_rows<1, V4, MAPS>;
    case 2: return k_mf_rows<2, V4, MAPS>;
    case 3: return k_mf_rows<3, V4, MAPS>;
    case 4: return k_mf_rows<4, V4, MAPS>;
    case 5: return k_mf_rows<5, V4, MAPS>;
    case 6: return k_mf_rows<6, V4, MAPS>;
    case 7: return k_mf_rows<7, V4, MAPS>;
    default: return k_mf_rows<8, V4, MAPS>;
    }
}

__global__ __launch_bounds__(256) void k_argmax(const float *rowmax, const int *rowarg,
                                                const int *rowwid, int nrow, int *odm, int *ot,
                                                float *os, int *ow)
{
    __shared__ float sv[256];
    __shared__ int sj[256];
    const int c = blockIdx.x, tid = threadIdx.x;
    float best = -INFINITY;
    int bj = 0x7fffffff;
    for (int j = tid; j < nrow; j += 256) {
        const float v = rowmax[(size_t)c * nrow + j];
        if (v > best) {
            best = v;
            bj = j;
        }
    }
    sv[tid] = best;
    sj[tid] = bj;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (tid < s) {
            const float ov = sv[tid + s];
            const int oj = sj[tid + s];
            if (ov > sv[tid] || (ov == sv[tid] && oj < sj[tid])) {
                sv[tid] = ov;
                sj[tid] = oj;
            }
        }
        __syncthreads();
    }
    if (tid == 0) {
        const int j = sj[0];
        odm[c] = j;
        os[c] = sv[0];
        if (rowarg) {
            ot[c] = rowarg[(size_t)c * nrow + j];
            ow[c] = rowwid[(size_t)c * nrow + j];
        }
    }
}

} // namespace

// ------------------------------------------------------------------- host
struct tx_refiner {
    tx_refine_desc d{};
    int device = 0;
    int nrow = 0, n = 0, batch = 0;
    std::vector<double> freqs, fP;
    std::vector<int> srcrow, vwn;
    std::vector<std::pair<int, int>> passes;
    double fmax = 0, fmin = 0;
    hipStream_t stream = nullptr;
    double *d_fP = nullptr, *d_fsrc = nullptr, *d_par = nullptr; // par: dms, ddm, dm0, dmc [4][batch]
    int *d_srcrow = nullptr, *d_vwn = nullptr;
    float *d_t1 = nullptr, *d_t2 = nullptr, *d_cs = nullptr, *d_rowmax = nullptr, *d_res_s = nullptr;
    int *d_rowarg = nullptr, *d_rowwid = nullptr, *d_res_i = nullptr; // res_i: dm, t, w [3][batch]
    double *d_var = nullptr;
};

#define RCHK(x)                                                                                    \
    do {                                                                                           \
        hipError_t e_ = (x);                                                                       \
        if (e_ != hipSuccess) return set_error(TX_EHIP, std::string(#x) + ": " + hipGetErrorString(e_)); \
    } while (0)

static void refiner_free(tx_refiner *r)
{
    hipFree(r->d_fP);
    hipFree(r->d_fsrc);
    hipFree(r->d_par);
    hipFree(r->d_srcrow);
    hipFree(r->d_vwn);
    hipFree(r->d_t1);
    hipFree(r->d_t2);
    hipFree(r->d_cs);
    hipFree(r->d_rowmax);
    hipFree(r->d_res_s);
    hipFree(r->d_rowarg);
    hipFree(r->d_rowwid);
    hipFree(r->d_res_i);
    hipFree(r->d_var);
    if (r->stream) hipStreamDestroy(r->stream);
}

// The ladder of Candidate::matched_filter (src/singlepulse/candidate.cpp:981-993),
// held in floats as the reference holds it.
static std::vector<int> mf_ladder(long nbin, float snrloss)
{
    const float wfactor = (float)(1. / ((1. - (double)snrloss) * (1. - (double)snrloss)));
    std::vector<float> v{1.f};
    for (;;) {
        const int w1 = (int)v.back();
        int w2 = (int)((float)w1 * wfactor);
        w2 = w2 < w1 + 1 ? w1 + 1 : w2;
        if (w2 > nbin / 2) break;
        v.push_back((float)w2);
    }
    std::vector<int> out;
    for (float x : v) out.push_back((int)x);
    return out;
}

extern "C" int tx_refine_create(const tx_refine_desc *d, int max_batch, tx_refiner **out)
{
    if (!d || !out || !d->frequencies) return set_error(TX_EINVAL, "null argument");
    if (d->nchan < 2 || d->nbin < 2 || d->nbin > 4096 || d->tbin <= 0. || max_batch <= 0 || max_batch > 65535)
        return set_error(TX_EINVAL, "refine: need nchan >= 2, 2 <= nbin <= 4096, tbin > 0, 1 <= max_batch <= 65535");
    if (d->snrloss < 0.f || d->snrloss >= 1.f) return set_error(TX_EINVAL, "refine: snrloss in [0, 1)");
    RCHK(hipSetDevice(d->device));
    tx_refiner *r = new tx_refiner();
    r->d = *d;
    r->device = d->device;
    r->batch = max_batch;
    r->freqs.assign(d->frequencies, d->frequencies + d->nchan);
    r->fmax = *std::max_element(r->freqs.begin(), r->freqs.end());
    r->fmin = *std::min_element(r->freqs.begin(), r->freqs.end());
    // Candidate::optimize: 2^ceil(log2 nchan) rows from the highest frequency,
    // padding rows at f[0] + j*foff (contracted to an FMA in the reference build)
    r->nrow = (int)std::pow(2, std::ceil(std::log2((double)d->nchan)));
    r->n = 0;
    while ((1 << r->n) < r->nrow) r->n++;
    const int nchan = d->nchan, nrow = r->nrow;
    const double foff = r->freqs[1] - r->freqs[0];
    r->fP.assign(nrow, 0.);
    r->srcrow.assign(nrow, -1);
    for (int j = 0; j < nchan; j++) {
        const int q = foff < 0. ? j : nchan - 1 - j;
        r->srcrow[j] = q;
        r->fP[j] = r->freqs[q];
    }
    for (int j = nchan; j < nrow; j++)
        r->fP[j] = foff < 0. ? std::fma((double)j, foff, r->freqs[0])
                             : std::fma((double)(nchan - 1 - j), foff, r->freqs[0]);
    r->vwn = mf_ladder(d->nbin, d->snrloss);
    if ((int)r->vwn.size() > kMaxMfBox) {
        delete r;
        return set_error(TX_EINVAL, "refine: ladder too long");
    }
    // tree passes of at most Lmax levels (G rows of nbin floats in 64 KB)
    int Lmax = 0;
    while ((2 << Lmax) * d->nbin <= kTreeLdsFloats && (1 << (Lmax + 1)) <= 1024) Lmax++;
    if (Lmax < 1) {
        delete r;
        return set_error(TX_EINVAL, "refine: nbin too large for one LDS tree tile");
    }
    const int npass = (r->n + Lmax - 1) / Lmax;
    for (int p = 0, a = 0; p < npass; p++) {
        const int len = (r->n - a + (npass - p) - 1) / (npass - p);
        r->passes.push_back({a, a + len});
        a += len;
    }
    (void)hipFuncSetAttribute((const void *)k_tree_pass, hipFuncAttributeMaxDynamicSharedMemorySize,
                              kTreeLdsFloats * 4);
    if (d->nbin >= kTreeRowsMin && d->nbin <= kTreeRowsMax)
        (void)hipFuncSetAttribute((const void *)tree_rows_kernel(d->nbin), hipFuncAttributeMaxDynamicSharedMemorySize,
                                  kTreeLdsFloats * 4 + 10 * 1024 * 4);
    const size_t B = (size_t)max_batch, rowsz = (size_t)nrow * d->nbin;
    bool ok = hipStreamCreate(&r->stream) == hipSuccess &&
              hipMalloc(&r->d_fP, nrow * sizeof(double)) == hipSuccess &&
              hipMalloc(&r->d_fsrc, nchan * sizeof(double)) == hipSuccess &&
              hipMalloc(&r->d_par, 4 * B * sizeof(double)) == hipSuccess &&
              hipMalloc(&r->d_srcrow, nrow * sizeof(int)) == hipSuccess &&
              hipMalloc(&r->d_vwn, kMaxMfBox * sizeof(int)) == hipSuccess &&
              hipMalloc(&r->d_t1, B * rowsz * 4) == hipSuccess &&
              hipMalloc(&r->d_t2, B * rowsz * 4) == hipSuccess &&
              (d->nbin <= kMfMapsMax || hipMalloc(&r->d_cs, 2 * B * rowsz * 4) == hipSuccess) &&
              hipMalloc(&r->d_rowmax, B * nrow * 4) == hipSuccess &&
              hipMalloc(&r->d_rowarg, B * nrow * 4) == hipSuccess &&
              hipMalloc(&r->d_rowwid, B * nrow * 4) == hipSuccess &&
              hipMalloc(&r->d_var, B * nrow * 8) == hipSuccess &&
              hipMalloc(&r->d_res_s, B * 4) == hipSuccess &&
              hipMalloc(&r->d_res_i, 3 * B * 4) == hipSuccess;
    if (!ok) {
        refiner_free(r);
        delete r;
        return set_error(TX_ENOMEM, "refine: device allocation");
    }
    ok = hipMemcpy(r->d_fP, r->fP.data(), nrow * sizeof(double), hipMemcpyHostToDevice) == hipSuccess &&
         hipMemcpy(r->d_fsrc, r->freqs.data(), nchan * sizeof(double), hipMemcpyHostToDevice) == hipSuccess &&
         hipMemcpy(r->d_srcrow, r->srcrow.data(), nrow * sizeof(int), hipMemcpyHostToDevice) == hipSuccess &&
         hipMemcpy(r->d_vwn, r->vwn.data(), r->vwn.size() * sizeof(int), hipMemcpyHostToDevice) == hipSuccess;
    if (!ok) {
        refiner_free(r);
        delete r;
        return set_error(TX_EHIP, "refine: table upload");
    }
    *out = r;
    return TX_OK;
}

extern "C" int tx_refine_destroy(tx_refiner *r)
{
    if (!r) return TX_OK;
    hipSetDevice(r->device);
    if (r->stream) hipStreamSynchronize(r->stream);
    refiner_free(r);
    delete r;
    return TX_OK;
}

extern "C" int tx_refine_info(const tx_refiner *r, int *nrow, int *nbox, int *npass)
{
    if (!r) return set_error(TX_EINVAL, "null argument");
    if (nrow) *nrow = r->nrow;
    if (nbox) *nbox = (int)r->vwn.size();
    if (npass) *npass = (int)r->passes.size();
    return TX_OK;
}

extern "C" int tx_refine_stream(tx_refiner *r, void **stream)
{
    if (!r || !stream) return set_error(TX_EINVAL, "null argument");
    *stream = (void *)r->stream;
    return TX_OK;
}

extern "C" int tx_refine_run(tx_refiner *r, int ncand, const float *cutouts, const double *dm,
                             tx_refine_result *res, float *dmtmap, float *snrmap, int *widmap)
{
    if (!r || ncand < 0 || (ncand && (!cutouts || !dm || !res))) return set_error(TX_EINVAL, "null argument");
    RCHK(hipSetDevice(r->device));
    const int nrow = r->nrow, nbin = r->d.nbin, nchan = r->d.nchan;
    const size_t rowsz = (size_t)nrow * nbin;
    // Candidate::optimize's DM grid (src/singlepulse/candidate.cpp:901-911)
    const double tmp = 4.148741601e3 * 1. * (1. / (r->fmin * r->fmin) - 1. / (r->fmax * r->fmax));
    const double dmrange = (nbin * r->d.tbin) / tmp;
    for (int c0 = 0; c0 < ncand; c0 += r->batch) {
        const int nc = std::min(r->batch, ncand - c0);
        std::vector<double> par(4 * (size_t)r->batch, 0.);
        for (int c = 0; c < nc; c++) {
            const double dmc = dm[c0 + c];
            const double dms = std::max(0., dmc - dmrange / 2.);
            const double dme = dmc + dmrange / 2.;
            par[c] = dms;
            par[r->batch + c] = (dme - dms) / nrow;
            par[2 * r->batch + c] = r->d.isdedispersed ? dmc : 0.;
            par[3 * r->batch + c] = dmc;
        }
        RCHK(hipMemcpyAsync(r->d_par, par.data(), par.size() * sizeof(double), hipMemcpyHostToDevice,
                            r->stream));
        TreeArgs A;
        A.fP = r->d_fP;
        A.srcrow = r->d_srcrow;
        A.fsrc = r->d_fsrc;
        A.dms = r->d_par;
        A.ddm = r->d_par + r->batch;
        A.dm0 = r->d_par + 2 * r->batch;
        A.dmc = r->d_par + 3 * r->batch;
        A.fmax = r->fmax;
        A.tbin = r->d.tbin;
        A.nchan = nchan;
        A.nrow = nrow;
        A.n = r->n;
        A.ncol = nbin;
        A.dedisperse = r->d.dedisperse != 0;
        float *dmt_out = dmtmap ? dmtmap + (size_t)c0 * rowsz : r->d_t2;
        const float *src = cutouts + (size_t)c0 * nchan * nbin;
        float *bufs[2] = {r->d_t1, r->d_t2};
        const int np = (int)r->passes.size();
        for (int p = 0; p < np; p++) {
            A.a = r->passes[p].first;
            A.b = r->passes[p].second;
            A.first = p == 0;
            A.last = p == np - 1;
            A.src = src;
            // the last pass never writes the buffer it reads
            float *dst = A.last ? dmt_out : bufs[p & 1];
            if (A.last && !dmtmap && src == r->d_t2) dst = r->d_t1, dmt_out = r->d_t1;
            A.dst = dst;
            const int G = 1 << (A.b - A.a);
            dim3 grid((unsigned)((nrow >> A.b) << A.a), (unsigned)nc);
            const size_t shm = (size_t)G * nbin * 4;
            const size_t sht = (size_t)(A.b - A.a) * G * 4;
            if (nbin >= kTreeRowsMin && nbin <= kTreeRowsMax)
                hipLaunchKernelGGL(tree_rows_kernel(nbin), grid, dim3(512), shm + sht, r->stream, A);
            else
                hipLaunchKernelGGL(k_tree_pass, grid, dim3(256), shm, r->stream, A);
            RCHK(hipGetLastError());
            src = dst;
        }
        MfArgs M;
        M.dmt = dmt_out;
        M.cs = r->d_cs;
        M.snr = snrmap ? snrmap + (size_t)c0 * rowsz : nullptr;
        M.wid = widmap ? widmap + (size_t)c0 * rowsz : nullptr;
        M.rowmax = r->d_rowmax;
        M.rowarg = r->d_rowarg;
        M.rowwid = r->d_rowwid;
        M.var = r->d_var;
        M.vwn = r->d_vwn;
        M.nbox = (int)r->vwn.size();
        M.nrows = (long)nc * nrow;
        M.ncol = nbin;
        M.pick = nullptr;
        const auto argmax = [&](const int *rowarg, const int *rowwid) {
            hipLaunchKernelGGL(k_argmax, dim3((unsigned)nc), dim3(256), 0, r->stream, (const float *)r->d_rowmax, rowarg,
                               rowwid, nrow, r->d_res_i, r->d_res_i + r->batch, r->d_res_s, r->d_res_i + 2 * r->batch);
        };
        const bool maps = M.snr || M.wid;
        const bool v4 = nbin % 4 == 0 && ((uintptr_t)dmt_out & 15) == 0;
        const int nu = (nbin + 63) / 64;
        MfRow T;
        T.nchunk = (nu + 7) / 8;
        const int cu = (nu + T.nchunk - 1) / T.nchunk;
        T.W = v4 ? (r->vwn.back() + 3) / 4 * 4 : r->vwn.back();
        T.pitch = v4 ? ((nbin + T.W) / 4 | 1) * 4 : (nbin + T.W) | 1;
        T.nrows = std::max(1, std::min(64, (kMfRowsLds / 4 - 64 * cu * T.nchunk) / (T.pitch + 64)));
        if (nbin <= (maps ? kMfMapsMax : kMfRowsMax) && (v4 || mf_word_rows(nbin, T.nrows, M.nrows))) {
            // reads past a row's last sample (whose results do not count) stay in the allocation
            const auto shm = [&] { return ((size_t)T.nrows * (T.pitch + 64) + 64 * cu * T.nchunk) * 4; };
            auto kernel = [&](bool m) {
                return v4 ? (m ? mf_rows_kernel<true, true>(cu) : mf_rows_kernel<true, false>(cu))
                          : (m ? mf_rows_kernel<false, true>(cu) : mf_rows_kernel<false, false>(cu));
            };
            hipLaunchKernelGGL(kernel(maps), dim3((unsigned)((M.nrows + T.nrows - 1) / T.nrows)), dim3(256), shm(),
                               r->stream, M, T);
            RCHK(hipGetLastError());
            argmax(maps ? r->d_rowarg : nullptr, maps ? r->d_rowwid : nullptr);
            RCHK(hipGetLastError());
            if (!maps) { // the best rows once more, for their times and widths
                M.pick = r->d_res_i;
                M.nrows = nrow;
                M.rowarg = r->d_res_i + r->batch;
                M.rowwid = r->d_res_i + 2 * r->batch;
                T.nrows = 1;
                hipLaunchKernelGGL(kernel(true), dim3((unsigned)nc), dim3(256), shm(), r->stream, M, T);
                RCHK(hipGetLastError());
            }
        } else {
            hipLaunchKernelGGL(k_mf_scan, dim3((unsigned)((M.nrows + 63) / 64)), dim3(64), 64 * 65 * 4,
                               r->stream, M);
            RCHK(hipGetLastError());
            const size_t shm = 4 * 2 * (size_t)nbin * 4;
            const dim3 mg((unsigned)((M.nrows + 3) / 4));
            if (nbin <= 1024) // over kMfMapsMax: shorter rows never come here
                hipLaunchKernelGGL(k_mf_box<16>, mg, dim3(256), shm, r->stream, M);
            else if (nbin <= 2048)
                hipLaunchKernelGGL(k_mf_box<32>, mg, dim3(256), shm, r->stream, M);
            else
                hipLaunchKernelGGL(k_mf_box<64>, mg, dim3(256), shm, r->stream, M);
            RCHK(hipGetLastError());
            argmax(r->d_rowarg, r->d_rowwid);
            RCHK(hipGetLastError());
        }
        std::vector<int> ri(3 * (size_t)r->batch);
        std::vector<float> rs(r->batch);
        RCHK(hipMemcpyAsync(ri.data(), r->d_res_i, ri.size() * 4, hipMemcpyDeviceToHost, r->stream));
        RCHK(hipMemcpyAsync(rs.data(), r->d_res_s, rs.size() * 4, hipMemcpyDeviceToHost, r->stream));
        RCHK(hipStreamSynchronize(r->stream));
        for (int c = 0; c < nc; c++) {
            tx_refine_result &o = res[c0 + c];
            o.dms = par[c];
            o.ddm = par[r->batch + c];
            o.ndm = nrow;
            o.maxdmid = ri[c];
            o.maxtid = ri[r->batch + c];
            o.snr = rs[c];
            o.wn = ri[2 * r->batch + c];
            o.width = (float)(o.wn * r->d.tbin);
            o.dm_maxsnr = std::fma((double)o.maxdmid, o.ddm, o.dms); // dms + maxdmid*ddm, contracted
        }
    }
    return TX_OK;
}
