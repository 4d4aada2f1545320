// Pointing expansion on the GPU: synthetic ring-scan attitude -> nested
// HEALPix pixel (int32) and (1, cos 2psi, sin 2psi) weights (float32).
//
// The reference receives pixels and weights from its caller
// (src/pointing.f90:13-14); its unused HEALPix routines
// (src/healpix_routines.f90:36-221, 407-455) are the model for the nested
// ang2pix.  Every step uses +, -, *, / and sqrt (plus the exact floor) with
// floating-point contraction disabled, so the pixels are bit-identical to the
// CPU expansion that performs the same steps in the same order.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>
#include <mutex>

#include "madam_internal.hpp"

#pragma clang fp contract(off)

namespace madam {

#define HALF_PI_D 1.5707963267948966192313216916398
#define PI_DD 3.1415926535897932384626433832795
#define SQRT3_D 1.7320508075688772935274463415059
#define TAN_PI_12_D 0.26794919243112270647255365849413

// sin and cos of 2 pi u (u in turns): exact reduction to an octant, Taylor
// polynomials to degree 19 / 20 on [0, pi/4]
__device__ void sincos_turns(double u, double *s, double *c)
{
    double f = u - floor(u);
    double q4 = f * 4.0;
    int quad = (int)q4;
    if (quad > 3) quad = 3;
    double r = q4 - (double)quad;
    int swap = 0;
    if (r > 0.5) { r = 1.0 - r; swap = 1; }
    double x = r * HALF_PI_D;
    double x2 = x * x;
    double sp = (1.0 / 121645100408832000.0);
    sp = -(1.0 / 355687428096000.0) + x2 * sp;
    sp = (1.0 / 1307674368000.0) + x2 * sp;
    sp = -(1.0 / 6227020800.0) + x2 * sp;
    sp = (1.0 / 39916800.0) + x2 * sp;
    sp = -(1.0 / 362880.0) + x2 * sp;
    sp = (1.0 / 5040.0) + x2 * sp;
    sp = -(1.0 / 120.0) + x2 * sp;
    sp = (1.0 / 6.0) + x2 * sp;
    double sn = x - x * (x2 * sp);
    double cp = (1.0 / 2432902008176640000.0);
    cp = -(1.0 / 6402373705728000.0) + x2 * cp;
    cp = (1.0 / 20922789888000.0) + x2 * cp;
    cp = -(1.0 / 87178291200.0) + x2 * cp;
    cp = (1.0 / 479001600.0) + x2 * cp;
    cp = -(1.0 / 3628800.0) + x2 * cp;
    cp = (1.0 / 40320.0) + x2 * cp;
    cp = -(1.0 / 720.0) + x2 * cp;
    cp = (1.0 / 24.0) + x2 * cp;
    cp = 0.5 - x2 * cp;
    double cs = 1.0 - x2 * cp;
    if (swap) { double t = sn; sn = cs; cs = t; }
    switch (quad) {
    case 0: *s = sn; *c = cs; break;
    case 1: *s = cs; *c = -sn; break;
    case 2: *s = -sn; *c = -cs; break;
    default: *s = -cs; *c = sn; break;
    }
}

__device__ double atan_unit(double t)
{
    double base = 0.0;
    if (t > TAN_PI_12_D) {
        t = (t * SQRT3_D - 1.0) / (t + SQRT3_D);
        base = PI_DD / 6.0;
    }
    double t2 = t * t;
    double p = (1.0 / 37.0);
    p = (1.0 / 35.0) - t2 * p;
    p = (1.0 / 33.0) - t2 * p;
    p = (1.0 / 31.0) - t2 * p;
    p = (1.0 / 29.0) - t2 * p;
    p = (1.0 / 27.0) - t2 * p;
    p = (1.0 / 25.0) - t2 * p;
    p = (1.0 / 23.0) - t2 * p;
    p = (1.0 / 21.0) - t2 * p;
    p = (1.0 / 19.0) - t2 * p;
    p = (1.0 / 17.0) - t2 * p;
    p = (1.0 / 15.0) - t2 * p;
    p = (1.0 / 13.0) - t2 * p;
    p = (1.0 / 11.0) - t2 * p;
    p = (1.0 / 9.0) - t2 * p;
    p = (1.0 / 7.0) - t2 * p;
    p = (1.0 / 5.0) - t2 * p;
    p = (1.0 / 3.0) - t2 * p;
    return base + (t - t * (t2 * p));
}

__device__ double atan2_pos(double y, double x)
{
    double ax = x < 0 ? -x : x, ay = y < 0 ? -y : y;
    if (ax == 0.0 && ay == 0.0) return 0.0;
    double a;
    if (ay <= ax) a = atan_unit(ay / ax);
    else a = HALF_PI_D - atan_unit(ax / ay);
    if (x < 0) a = PI_DD - a;
    if (y < 0) a = 2.0 * PI_DD - a;
    if (a >= 2.0 * PI_DD) a = 0.0;
    return a;
}

// bit k of v to bit 2 k (v < 2^32)
__device__ inline uint64_t spread_bits(uint64_t v)
{
    v = (v | v << 16) & 0x0000ffff0000ffffull;
    v = (v | v << 8) & 0x00ff00ff00ff00ffull;
    v = (v | v << 4) & 0x0f0f0f0f0f0f0f0full;
    v = (v | v << 2) & 0x3333333333333333ull;
    return (v | v << 1) & 0x5555555555555555ull;
}
// v < 2^16
__device__ inline uint32_t spread_bits(uint32_t v)
{
    v = (v | v << 8) & 0x00ff00ffu;
    v = (v | v << 4) & 0x0f0f0f0fu;
    v = (v | v << 2) & 0x33333333u;
    return (v | v << 1) & 0x55555555u;
}

// I, U: 32-bit integers up to Nside 8192 (every pixel number then fits them),
// 64-bit ones above.  The quotients by Nside are of non-negative numbers, so
// shifts.
template <typename I, typename U>
__device__ inline I vec2pix_nest(int64_t nside, double x, double y, double z)
{
    double rho2 = x * x + y * y;
    double za = z < 0 ? -z : z;
    double phi = atan2_pos(y, x);
    double tt = phi * (2.0 / PI_DD);
    if (tt >= 4.0) tt = 0.0;
    I face, ix, iy;
    const I ns = (I)nside;
    const int sh = __ffsll((unsigned long long)nside) - 1;
    double dn = (double)nside;
    if (za <= 2.0 / 3.0) {
        double temp1 = dn * (0.5 + tt);
        double temp2 = dn * (z * 0.75);
        I jp = (I)(temp1 - temp2);
        I jm = (I)(temp1 + temp2);
        I ifp = jp >> sh, ifm = jm >> sh;
        if (ifp == ifm) face = (ifp == 4 ? 0 : ifp) + 4;
        else if (ifp < ifm) face = ifp;
        else face = ifm + 8;
        ix = jm & (ns - 1);
        iy = ns - (jp & (ns - 1)) - 1;
    } else {
        I ntt = (I)tt;
        if (ntt > 3) ntt = 3;
        double tp = tt - (double)ntt;
        double one_minus = rho2 / (1.0 + za);
        double tmp = dn * sqrt(3.0 * one_minus);
        I jp = (I)(tp * tmp);
        I jm = (I)((1.0 - tp) * tmp);
        if (jp > ns - 1) jp = ns - 1;
        if (jm > ns - 1) jm = ns - 1;
        if (z >= 0) { face = ntt; ix = ns - jm - 1; iy = ns - jp - 1; }
        else { face = ntt + 8; ix = jp; iy = jm; }
    }
    return (I)(((U)face << (2 * sh)) + (spread_bits((U)ix) | (spread_bits((U)iy) << 1)));
}

// One sample per thread, the detectors d0 .. d0 + nd - 1 of a group in turn:
// output pix[det * ld + k], w[(det * ld + k) * 3 + j].  The precession angle is
// the sample's, the spin angle is shared by detectors of one spin offset, and
// the boresight, its pixel and the local frame by detectors of one opening too
// (the four of a horn): a detector that differs from the one before it only in
// its polarisation angle takes the values over.  The kernel is bound by FP64
// issue (about 500 operations per new boresight, 80 per further detector).
// Measured, 16 detectors in horns x 2^22 samples: 370 us, 2.9 TB/s of output (775
// GB/s before, with 64-bit divisions, bit loops and every angle per detector: 1386).
static constexpr int PT_GROUP = 8;   // most detectors per thread
template <typename I, typename U>
__global__ void __launch_bounds__(256) k_expand_pointing(ScanParams sp, const ScanDet *dets, int ndet, int group,
                                                         int64_t nside, int64_t i0, int64_t n, int64_t ld,
                                                         int32_t *pix, float *w)
{
    // the detectors' own angles, once per block
    __shared__ double trig[PT_GROUP][4];
    const int d0 = blockIdx.y * group, d1 = d0 + group < ndet ? d0 + group : ndet;
    if ((int)threadIdx.x < d1 - d0) {
        ScanDet det = dets[d0 + threadIdx.x];
        double *t = trig[threadIdx.x];
        sincos_turns(det.psi_turns, t, t + 1);
        sincos_turns(sp.opening_turns + det.open_offset_turns, t + 2, t + 3);
    }
    __syncthreads();
    int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (k >= n) return;
    const double spin_samples = sp.fsample * sp.spin_period;
    const double prec_samples = sp.fsample * sp.prec_period;
    const double di = (double)(i0 + k);
    double sl, cl;
    sincos_turns(sp.lon0_turns + di / prec_samples, &sl, &cl);
    const double spin = di / spin_samples;
    double last_open = 0, last_spin = 0;
    double dx = 0, dy = 0, dz = 0, nx = 0, ny = 0, nz = 0, ux = 0, uy = 0, uz = 0;
    double eth_x = 0, eth_y = 0, eth_z = 0, eph_x = 0, eph_y = 0, rho2 = 0;
    int32_t q = 0;
    for (int d = d0; d < d1; ++d) {
        const ScanDet det = dets[d];   // the same for the whole wave
        const bool new_spin = d == d0 || det.spin_offset_turns != last_spin;
        if (new_spin) {
            double sw, cw;
            sincos_turns(spin + det.spin_offset_turns, &sw, &cw);
            ux = -(sw * sl), uy = sw * cl, uz = cw;
            dx = -(cw * sl), dy = cw * cl, dz = -sw;
            last_spin = det.spin_offset_turns;
        }
        if (new_spin || det.open_offset_turns != last_open) {
            const double sb = trig[d - d0][2], cb = trig[d - d0][3];
            double bx = cb * cl + sb * ux;
            double by = cb * sl + sb * uy;
            double bz = sb * uz;
            nx = by * dz - bz * dy;
            ny = bz * dx - bx * dz;
            nz = bx * dy - by * dx;
            rho2 = bx * bx + by * by;
            if (rho2 > 0.0) {
                double rho = sqrt(rho2);
                eth_x = bz * bx / rho, eth_y = bz * by / rho, eth_z = -rho;
                eph_x = -by / rho, eph_y = bx / rho;
            }
            q = (int32_t)vec2pix_nest<I, U>(nside, bx, by, bz);
            last_open = det.open_offset_turns;
        }
        const double spsi = trig[d - d0][0], cpsi = trig[d - d0][1];
        double c2 = 1.0, s2 = 0.0;
        if (rho2 > 0.0) {
            double ex = cpsi * dx + spsi * nx;
            double ey = cpsi * dy + spsi * ny;
            double ez = cpsi * dz + spsi * nz;
            double u = ex * eth_x + ey * eth_y + ez * eth_z;
            double v = ex * eph_x + ey * eph_y;
            double nrm = u * u + v * v;
            c2 = (u * u - v * v) / nrm;
            s2 = -(2.0 * u * v) / nrm;
        }
        int64_t o = (int64_t)d * ld + k;
        pix[o] = q;
        w[o * 3] = 1.0f;
        w[o * 3 + 1] = (float)c2;
        w[o * 3 + 2] = (float)s2;
    }
}

void launch_expand_pointing(hipStream_t s, ScanParams sp, const ScanDet *dets, int ndet, int64_t nside, int64_t i0,
                            int64_t n, int64_t ld, int32_t *pix, float *w)
{
    if (ndet < 1 || n < 1) return;
    // detectors per thread: eight, fewer while that leaves fewer threads
    // than the GPU holds at once (2048 on each of 256 CUs)
    int group = PT_GROUP;
    while (group > 1 && n * ((ndet + group - 1) / group) < 2048 * 256) group /= 2;
    // a launch takes up to 2^31 - 1 threads in x and 65535 groups in y
    for (int dd = 0; dd < ndet; dd += 65535 * group)
        for (int64_t k0 = 0; k0 < n; k0 += 1ll << 30) {
            int64_t m = n - k0 < (1ll << 30) ? n - k0 : (1ll << 30);
            int nd = ndet - dd < 65535 * group ? ndet - dd : 65535 * group;
            dim3 g((unsigned)((m + 255) / 256), (unsigned)((nd + group - 1) / group));
            int32_t *po = pix + (int64_t)dd * ld + k0;
            float *wo = w + ((int64_t)dd * ld + k0) * 3;
            if (nside <= 8192)
                k_expand_pointing<int32_t, uint32_t><<<g, 256, 0, s>>>(sp, dets + dd, nd, group, nside, i0 + k0, m, ld,
                                                                       po, wo);
            else
                k_expand_pointing<int64_t, uint64_t><<<g, 256, 0, s>>>(sp, dets + dd, nd, group, nside, i0 + k0, m, ld,
                                                                       po, wo);
        }
}

// ---------------------------------------------------------------- the entry point that allocates nothing
//
// madam_expand_pointing stages the detector table in device memory it
// allocates per call.  The variant below stages it in `scratch`, a fixed
// array in the library's device image instead: each GPU the library runs on
// holds its own copy (NOALLOC_MAX_DETS * 24 bytes = 96 KiB) until the process
// ends.  Host code never passes `scratch` itself to a kernel (its host-side
// name is not a device address): the device address comes from
// hipGetSymbolAddress, once per device, with that device current.

static constexpr int NOALLOC_MAX_DETS = 4096;
static constexpr int NOALLOC_MAX_DEVICES = 64;
static __device__ __align__(256) ScanDet scratch[NOALLOC_MAX_DETS];

static std::mutex g_scratch_mu;
static void *g_scratch_dev[NOALLOC_MAX_DEVICES];   // scratch's device address, per device

// scratch's address on the current device (looked up on the device's first call)
static hipError_t scratch_on_current_device(void **out, int *dev_out)
{
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    *dev_out = dev;
    if (dev < 0 || dev >= NOALLOC_MAX_DEVICES) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_dev[dev]) {
        void *p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        if (!p) return hipErrorInvalidSymbol;
        g_scratch_dev[dev] = p;
    }
    *out = g_scratch_dev[dev];
    return hipSuccess;
}

}  // namespace madam

using namespace madam;

extern "C" __attribute__((visibility("default"))) int madam_expand_pointing_noalloc(
    const double *scan5, const double *dets3, int ndet, long nside, long i0, long n, int32_t *pix, float *weights,
    void *stream)
{
    char msg[256];
    if (ndet < 1 || ndet > NOALLOC_MAX_DETS) {
        snprintf(msg, sizeof msg, "madam_expand_pointing_noalloc: ndet = %d outside 1..%d (the staging array's size)",
                 ndet, NOALLOC_MAX_DETS);
        set_last_error(msg);
        return 1;
    }
    if (!scan5 || !dets3 || !pix || !weights || n < 0 || nside < 1 || (nside & (nside - 1)) || nside > (1L << 29)) {
        set_last_error("madam_expand_pointing_noalloc: null pointer, n < 0 or nside not a power of two");
        return 1;
    }
    void *sp = nullptr;
    int dev = -1;
    hipError_t e = scratch_on_current_device(&sp, &dev);
    if (e == hipSuccess) {
        hipStream_t s = (hipStream_t)stream;
        e = hipMemcpyAsync(sp, dets3, sizeof(ScanDet) * ndet, hipMemcpyHostToDevice, s);
        if (e == hipSuccess && n > 0) {
            ScanParams p{scan5[0], scan5[1], scan5[2], scan5[3], scan5[4]};
            launch_expand_pointing(s, p, (const ScanDet *)sp, ndet, nside, i0, n, n, pix, weights);
            e = hipGetLastError();
        }
    }
    if (e != hipSuccess) {
        snprintf(msg, sizeof msg, "madam_expand_pointing_noalloc: HIP error %d (%s) on device %d", (int)e,
                 hipGetErrorString(e), dev);
        set_last_error(msg);
        return 1;
    }
    return 0;
}
