// Run records of the one-right-hand-side projections.
//
// Consecutive samples of one baseline on one cross pixel see the same map
// value and the same baseline value, so both projections
// (src/smadam_routines.f90:1038-1148, 1235-1376) need only their number and
// the sums of their weights.  A run is one 4-byte word (index in the low `sh`
// bits, number of samples above them) and, for polarised maps, the sums of w1
// and w2 in the operator's type (FP64 sums for the FP64 operator): 20 bytes in
// FP64, 12 in FP32, 4 for temperature-only maps, in place of 12 (4) bytes per
// sample.  The word and the weights are separate arrays, both read coalesced.
// Runs serve the scans whose intensity weight is 1 everywhere (w0 sums to the
// number of samples); they are built once per pointing, from the sample
// records in time order (baseline side) and from the CSR entries in pixel
// order (pixel side), and are cut at every multiple of the largest number
// that the word holds.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "madam_internal.hpp"

namespace madam {

static constexpr int RUN_TPB = 256;
static constexpr int RUN_SPAN = 512;   // items per wave of the building kernels, eight 64-bit words of start bits

// ------------------------------------------------------------ building

__global__ void k_run_marks(const int64_t *starts, int64_t n, uint32_t *mask)
{
    for (int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; k < n; k += (int64_t)gridDim.x * blockDim.x)
        atomicOr(mask + (starts[k] >> 5), 1u << (starts[k] & 31));
}

// index of item i (cross pixel of a sample, slot of an entry; < 0: takes no part)
template <int RL>
__device__ inline int32_t run_index(const void *rec, int64_t i, int dsh)
{
    int32_t p = RL == REC12 ? ((const Rec12 *)rec)[i].i : ((const int32_t *)rec)[i];
    return p >= 0 ? p >> dsh : -1;
}

// start bits of the runs, 64 items per word, and their number per RUN_SPAN
// items.  `mask` marks the items where a run may not continue the previous
// one: the baseline starts of one detector's `period` samples, or the first
// entry of every pixel (period = n).
template <int RL>
__global__ void __launch_bounds__(RUN_TPB) k_run_flags(const void *rec, int64_t n, int64_t period, int dsh,
                                                       uint32_t maxrun, const uint32_t *mask,
                                                       unsigned long long *words, int32_t *counts)
{
    int lane = threadIdx.x & 63;
    int64_t w = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) >> 6;
    int64_t i0 = w * RUN_SPAN;
    if (i0 >= n) return;   // uniform over the wave
    int cnt = 0;
#pragma unroll
    for (int u = 0; u < RUN_SPAN / 64; ++u) {
        int64_t i = i0 + u * 64 + lane;
        bool in = i < n;
        int32_t q = in ? run_index<RL>(rec, i, dsh) : -1;
        bool st = q >= 0;
        if (st && i > 0) {
            int64_t k = i % period;
            bool cut = (mask[k >> 5] >> (k & 31)) & 1u;
            st = cut || (uint32_t)i % maxrun == 0 || run_index<RL>(rec, i - 1, dsh) != q;
        }
        unsigned long long b = __ballot(st);
        cnt += __popcll(b);
        if (lane == 0) words[(i0 >> 6) + u] = b;
    }
    if (lane == 0) counts[w] = cnt;
}

// the runs: word and weight sums, added in FP64 and stored as W (double2, or
// float2 where only the FP32 operator reads them)
template <int RL, typename W>
__global__ void __launch_bounds__(RUN_TPB) k_run_write(const void *rec, int64_t n, int dsh, int sh,
                                                       const unsigned long long *words, const int64_t *offs,
                                                       uint32_t *out, W *wsum)
{
    int lane = threadIdx.x & 63;
    int64_t w = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) >> 6;
    int64_t i0 = w * RUN_SPAN;
    if (i0 >= n) return;
    int64_t at = offs[w];
    for (int u = 0; u < RUN_SPAN / 64; ++u) {
        unsigned long long b = words[(i0 >> 6) + u];
        if ((b >> lane) & 1ull) {
            int64_t i = i0 + u * 64 + lane;
            uint32_t q = (uint32_t)run_index<RL>(rec, i, dsh), m = 0;
            double2 s{0.0, 0.0};
            for (int64_t j = i;;) {
                if (RL == REC12) {
                    Rec12 r = ((const Rec12 *)rec)[j];
                    s.x += (double)r.w1;
                    s.y += (double)r.w2;
                }
                ++m;
                ++j;
                if (j >= n || ((words[j >> 6] >> (j & 63)) & 1ull) || run_index<RL>(rec, j, dsh) < 0) break;
            }
            int64_t o = at + __popcll(b & ((1ull << lane) - 1ull));
            out[o] = q | (m << sh);
            if (RL == REC12) {
                W v;
                v.x = (decltype(v.x))s.x;
                v.y = (decltype(v.y))s.y;
                wsum[o] = v;
            }
        }
        at += __popcll(b);
    }
}

// number of run starts before item i
__device__ inline int64_t run_rank(const unsigned long long *words, const int64_t *offs, int64_t i)
{
    int64_t r = offs[i / RUN_SPAN];
    int64_t w0 = i / RUN_SPAN * (RUN_SPAN / 64), w1 = i >> 6;
    for (int64_t w = w0; w < w1; ++w) r += __popcll(words[w]);
    if (i & 63) r += __popcll(words[w1] & ((1ull << (i & 63)) - 1ull));
    return r;
}

__global__ void k_run_base_starts(const int64_t *bstart, int64_t nbase, int ndet, int64_t nsamp,
                                  const unsigned long long *words, const int64_t *offs, int64_t *gst)
{
    int64_t tot = (int64_t)ndet * (nbase + 1);
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < tot; t += (int64_t)gridDim.x * blockDim.x) {
        int64_t det = t / (nbase + 1), k = t - det * (nbase + 1);
        gst[t] = run_rank(words, offs, det * nsamp + bstart[k]);
    }
}

__global__ void k_run_pixel_starts(const int64_t *segstart, int64_t nz, const unsigned long long *words,
                                   const int64_t *offs, int64_t *seg)
{
    for (int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; k <= nz; k += (int64_t)gridDim.x * blockDim.x)
        seg[k] = run_rank(words, offs, segstart[k]);
}

__global__ void k_run_cast(const double2 *in, float2 *out, int64_t n)
{
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        double2 v = in[i];
        out[i] = make_float2((float)v.x, (float)v.y);
    }
}

static unsigned run_grid(int64_t n, int64_t cap = 65535 * 8)
{
    int64_t g = (n + RUN_TPB - 1) / RUN_TPB;
    return (unsigned)(g < 1 ? 1 : (g > cap ? cap : g));
}

int64_t runs_spans(int64_t n) { return (n + RUN_SPAN - 1) / RUN_SPAN; }

// start bits (words[n / 64 + 9]) and the exclusive scan of their numbers
// (offs[runs_spans(n) + 1]); offs of the last span + 1 is the number of runs
void runs_mark(hipStream_t s, const void *rec, int rl, int64_t n, int64_t period, int dsh, uint32_t maxrun,
               const int64_t *starts, int64_t nstarts, uint32_t *mask, unsigned long long *words, int32_t *counts,
               int64_t *offs, int64_t *scan_tmp)
{
    int64_t ns = runs_spans(n);
    MADAM_CHECK(hipMemsetAsync(mask, 0, sizeof(uint32_t) * (period / 32 + 1), s));
    k_run_marks<<<run_grid(nstarts), RUN_TPB, 0, s>>>(starts, nstarts, mask);
    MADAM_CHECK(hipMemsetAsync(words + n / 64, 0, sizeof(unsigned long long) * 9, s));
    unsigned g = run_grid(ns * 64, INT32_MAX);
    if (rl == REC12)
        k_run_flags<REC12><<<g, RUN_TPB, 0, s>>>(rec, n, period, dsh, maxrun, mask, words, counts);
    else
        k_run_flags<REC4><<<g, RUN_TPB, 0, s>>>(rec, n, period, dsh, maxrun, mask, words, counts);
    launch_exclusive_scan_i32_to_i64(s, counts, ns, offs, scan_tmp, (ns + 1 + 4095) / 4096);
    MADAM_CHECK(hipGetLastError());
}

template <typename W>
void runs_write(hipStream_t s, const void *rec, int rl, int64_t n, int dsh, int sh, const unsigned long long *words,
                const int64_t *offs, uint32_t *out, W *wsum)
{
    unsigned g = run_grid(runs_spans(n) * 64, INT32_MAX);
    if (rl == REC12) k_run_write<REC12, W><<<g, RUN_TPB, 0, s>>>(rec, n, dsh, sh, words, offs, out, wsum);
    else k_run_write<REC4, W><<<g, RUN_TPB, 0, s>>>(rec, n, dsh, sh, words, offs, out, wsum);
    MADAM_CHECK(hipGetLastError());
}
template void runs_write<double2>(hipStream_t, const void *, int, int64_t, int, int, const unsigned long long *,
                                  const int64_t *, uint32_t *, double2 *);
template void runs_write<float2>(hipStream_t, const void *, int, int64_t, int, int, const unsigned long long *,
                                 const int64_t *, uint32_t *, float2 *);

void runs_base_starts(hipStream_t s, const int64_t *bstart, int64_t nbase, int ndet, int64_t nsamp,
                      const unsigned long long *words, const int64_t *offs, int64_t *gst)
{
    k_run_base_starts<<<run_grid((int64_t)ndet * (nbase + 1)), RUN_TPB, 0, s>>>(bstart, nbase, ndet, nsamp, words,
                                                                              offs, gst);
    MADAM_CHECK(hipGetLastError());
}

void runs_pixel_starts(hipStream_t s, const int64_t *segstart, int64_t nz, const unsigned long long *words,
                       const int64_t *offs, int64_t *seg)
{
    k_run_pixel_starts<<<run_grid(nz + 1), RUN_TPB, 0, s>>>(segstart, nz, words, offs, seg);
    MADAM_CHECK(hipGetLastError());
}

void runs_cast(hipStream_t s, const double2 *in, float2 *out, int64_t n)
{
    if (n <= 0) return;
    k_run_cast<<<run_grid(n), RUN_TPB, 0, s>>>(in, out, n);
    MADAM_CHECK(hipGetLastError());
}

// ------------------------------------------------------------ baseline side
// ap[b] += nna[b] p[b] - dw[b] sum_runs (n, W1, W2) . m[q].  A block owns K
// consecutive baselines of D consecutive detectors; lane t takes run t of each
// of those detectors, counted from the block's first baseline.  Detectors on
// one boresight have the same runs, so their lanes see the same pixel and
// share one map load (the address path costs per load, not per byte);
// detectors whose runs differ load their own.  One detector per block, each
// lane loading its own map rows, took 50 us where this takes 42 (FP64, 4 x
// 2^22 samples, 2.9 samples per run) and 378 us where this takes 301 (FP32, 16
// x 2^23, 1.6).  The products go through LDS,
// RG_T runs of all detectors at a time, and 256 / (K D) lanes sum each
// baseline.  Few long baselines (K = 16) leave more blocks and more lanes per
// baseline than many short ones (K = 64).
static constexpr int RG_T = 2048;   // LDS tile: RG_T / D runs per detector

template <typename T, int NMAP, int D, int K>
__global__ void __launch_bounds__(RUN_TPB) k_gather_run(int ndet, int64_t nbase, const int64_t *__restrict__ gst,
                                                        const uint32_t *__restrict__ word,
                                                        const void *__restrict__ wsum, int sh,
                                                        const T *__restrict__ m4, const T *__restrict__ dwb,
                                                        const T *__restrict__ nna, const T *__restrict__ p, T *ap,
                                                        int add)
{
    using V2 = typename VecT<T>::v2;
    constexpr int TD = RG_T / D;                                    // runs per detector and tile
    constexpr int L = K * D >= RUN_TPB ? 1 : RUN_TPB / (K * D);     // lanes per baseline
    constexpr int P = K * D > RUN_TPB ? K * D / RUN_TPB : 1;        // baselines per lane group
    __shared__ T vals[RG_T + 1];
    __shared__ int32_t bs[D][K + 1];   // first run of each baseline, relative to the detector's first in the block
    int64_t ngrp = (ndet + D - 1) / D;
    int64_t lb = xcd_block(blockIdx.x, gridDim.x);
    int64_t kb = lb / ngrp;            // time-major: neighbouring blocks share the sky
    int d0 = (int)(lb - kb * ngrp) * D;
    int nd = ndet - d0 < D ? ndet - d0 : D;
    int64_t k0 = kb * K;
    int nk = (int)(nbase - k0 < K ? nbase - k0 : K);
    int64_t c0[D];
    int nr[D], nmax = 0;
#pragma unroll
    for (int d = 0; d < D; ++d) {
        const int64_t *st = gst + (int64_t)(d0 + (d < nd ? d : 0)) * (nbase + 1) + k0;
        c0[d] = st[0];
        nr[d] = d < nd ? (int)(st[nk] - c0[d]) : 0;
        nmax = nr[d] > nmax ? nr[d] : nmax;
        for (int t = threadIdx.x; t <= nk; t += RUN_TPB) bs[d][t] = (int32_t)(st[t] - c0[d]);
    }
    const uint32_t qmask = (1u << sh) - 1u;
    const int sub = threadIdx.x % L;
    T acc[P];
#pragma unroll
    for (int i = 0; i < P; ++i) acc[i] = (T)0;
    for (int t0 = 0; t0 < nmax; t0 += TD) {
        int len = nmax - t0 < TD ? nmax - t0 : TD;
        for (int tt = threadIdx.x; tt - (int)(threadIdx.x & 63) < len; tt += RUN_TPB) {
            if (__builtin_amdgcn_readfirstlane(tt - (int)(threadIdx.x & 63)) >= len) break;   // uniform over the wave
            uint32_t wd[D];
            V2 ws[D];
#pragma unroll
            for (int d = 0; d < D; ++d) {
                int t = t0 + tt < nr[d] ? t0 + tt : (nr[d] > 0 ? nr[d] - 1 : 0);
                wd[d] = 0u;
                if (nr[d] > 0) {   // uniform over the block
                    wd[d] = __builtin_nontemporal_load(word + c0[d] + t);
                    if (NMAP == 3) ws[d] = load_wsum_nt<T>(wsum, c0[d] + t);
                }
            }
            uint32_t q[D];
            bool ld[D];
#pragma unroll
            for (int d = 0; d < D; ++d) {
                q[d] = wd[d] & qmask;
                bool seen = false;
#pragma unroll
                for (int e = 0; e < d; ++e) seen = seen || q[e] == q[d];
                ld[d] = !seen;
            }
            V2 mxy[D];   // (m.x, m.y); m.y unused for NMAP = 1
            T mz[D];
#pragma unroll
            for (int d = 0; d < D; ++d) {
                if (ld[d]) {
                    const T *mp = m4 + (int64_t)q[d] * 4;
                    if (NMAP == 1) {
                        mxy[d].x = mp[0];
                    } else {
                        mxy[d] = *(const V2 *)mp;
                        mz[d] = mp[2];
                    }
                }
            }
            // keeps the loads above from being sunk into the code below
            asm volatile("" ::: "memory");
#pragma unroll
            for (int d = 1; d < D; ++d) {
                if (!ld[d]) {
                    V2 cxy = mxy[0];
                    T cz = mz[0];
#pragma unroll
                    for (int e = 1; e < d; ++e)
                        if (q[e] == q[d] && ld[e]) {
                            cxy = mxy[e];
                            cz = mz[e];
                        }
                    mxy[d] = cxy;
                    mz[d] = cz;
                }
            }
#pragma unroll
            for (int d = 0; d < D; ++d) {
                T n = (T)(wd[d] >> sh);
                T v = NMAP == 1 ? n * mxy[d].x : n * mxy[d].x + ws[d].x * mxy[d].y + ws[d].y * mz[d];
                vals[tt < len ? d * TD + tt : RG_T] = t0 + tt < nr[d] ? v : (T)0;   // past the end: the spare slot
            }
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < P; ++i) {
            int it = threadIdx.x / L + i * (RUN_TPB / L), d = it / K, k = it % K;
            if (d < nd && k < nk) {
                int a = bs[d][k] - t0, z = bs[d][k + 1] - t0;
                a = a > 0 ? a : 0;
                z = z < TD ? z : TD;
                for (int t = a + sub; t < z; t += L) acc[i] += vals[d * TD + t];
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < P; ++i) {
        T s = acc[i];
#pragma unroll
        for (int o = L / 2; o > 0; o >>= 1) s += __shfl_xor(s, o, L);
        int it = threadIdx.x / L + i * (RUN_TPB / L), d = it / K, k = it % K;
        if (d < nd && k < nk && sub == 0) {
            int64_t b = (int64_t)(d0 + d) * nbase + k0 + k;
            ap[b] = (add ? ap[b] : (T)0) + (nna[b] * p[b] - s * dwb[b]);
        }
    }
}

template <typename T, int D, int K>
static void gather_run(hipStream_t s, int nmap, int ndet, int64_t nbase, const RunView<T> &rv, const T *m4,
                       const T *dwb, const T *nna, const T *p, T *ap, int add)
{
    unsigned grid = (unsigned)(((ndet + D - 1) / D) * ((nbase + K - 1) / K));
    if (nmap == 1)
        k_gather_run<T, 1, D, K><<<grid, RUN_TPB, 0, s>>>(ndet, nbase, rv.gst, rv.gword, rv.gw, rv.sh, m4, dwb, nna, p,
                                                          ap, add);
    else
        k_gather_run<T, 3, D, K><<<grid, RUN_TPB, 0, s>>>(ndet, nbase, rv.gst, rv.gword, rv.gw, rv.sh, m4, dwb, nna, p,
                                                          ap, add);
}

template <typename T>
void launch_gather_run(hipStream_t s, int nmap, int ndet, int64_t nbase, const RunView<T> &rv, const T *m4,
                       const T *dwb, const T *nna, const T *p, T *ap, int add)
{
    if (ndet <= 0 || nbase <= 0) return;
    // Four detectors per block where there are that many.  64 baselines per
    // block, or 16 where 64 leave less than two blocks per CU, or baselines so
    // long that an LDS tile holds few of them.  Measured, FP64, us per launch,
    // K = 64 / 16: 2,622 blocks (of 64) with 9 runs per baseline 42 / 47, 938
    // with 13 (temperature) 19 / 23, 164 with 7 10.9 / 9.4.
    const bool wide = (int64_t)((ndet + 3) / 4) * ((nbase + 63) / 64) >= 512 && rv.per_base <= 32;
    if (ndet == 1) {
        gather_run<T, 1, 64>(s, nmap, ndet, nbase, rv, m4, dwb, nna, p, ap, add);
    } else if (ndet == 2) {
        if (wide) gather_run<T, 2, 64>(s, nmap, ndet, nbase, rv, m4, dwb, nna, p, ap, add);
        else gather_run<T, 2, 16>(s, nmap, ndet, nbase, rv, m4, dwb, nna, p, ap, add);
    } else {
        if (wide) gather_run<T, 4, 64>(s, nmap, ndet, nbase, rv, m4, dwb, nna, p, ap, add);
        else gather_run<T, 4, 16>(s, nmap, ndet, nbase, rv, m4, dwb, nna, p, ap, add);
    }
}
template void launch_gather_run<double>(hipStream_t, int, int, int64_t, const RunView<double> &, const double *,
                                        const double *, const double *, const double *, double *, int);
template void launch_gather_run<float>(hipStream_t, int, int, int64_t, const RunView<float> &, const float *,
                                       const float *, const float *, const float *, float *, int);

}  // namespace madam
