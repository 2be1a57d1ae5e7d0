// Born-Wolf widefield PSF on the device: the algorithm of deconwolf's dw_bw
// (src/dw_bwpsf.c:538-775 with src/bw_gsl.c:79-157 and src/lanczos.c:102-160).
//
//   k_bw_nodes    Gauss-Legendre nodes on [0, 1], one rule for all planes
//   k_bw_profile  |A(r, z)|^2, A = int_0^1 J0(k0 NA r rho) e^{-i k0 NA^2 z rho^2/(2 ni)} rho drho,
//                 at 17 radii per pixel for each plane z <= (P-1)/2
//   k_bw_pixels   the mean over each pixel of the Lanczos-5 interpolation of
//                 that profile (8 x 8 Gauss-Legendre nodes), zero beyond
//                 radmax, for one octant of the plane
//   k_bw_mirror   the octant mirrored eight ways, and in z
//
// Double precision throughout; the pixel values are stored as float, as
// dw_bw stores them.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "dwhip.h"
#include "dwhip_internal.h"

#define BTHR 256
#define BW_OVERSAMPLING 17  // radial samples per pixel (dw_bwpsf.c:181)
#define BW_PIXEL_NODES 8

// n-point Gauss-Legendre rule on [0, 1], one thread per pair of mirrored
// nodes: Newton's iteration on P_n (three-term recurrence) from Tricomi's
// asymptotic nodes (1 - (n-1)/(8 n^3)) cos(pi (i - 1/4)/(n + 1/2)), whose
// error is O(n^-4): three steps reach double precision for every n here (64
// and more).  Stored as (rho, rho * weight).  Bound by the recurrence's serial
// chain: 33 us for the 190 nodes of a 181 x 181 x 79 PSF (9.3 ms on the host,
// with a rule for each plane).
__global__ __launch_bounds__(BTHR) void k_bw_nodes(int n, double2* __restrict__ nodes)
{
    const int i = blockIdx.x * BTHR + threadIdx.x;
    if (i >= (n + 1) / 2) return;
    const double dn = (double)n;
    double t = (1.0 - (dn - 1.0) / (8.0 * dn * dn * dn)) * cospi((i + 0.75) / (dn + 0.5));
    double dp = 0;
    for (int it = 0; it < 4; ++it) {
        double p0 = 1, p1 = t;
#pragma unroll 4
        for (int k = 2; k <= n; ++k) {
            // ((2k - 1) t p1 - (k - 1) p0) / k
            const double r = 1.0 / (double)k, tp = t * p1;
            const double p2 = fma(1.0 - r, tp - p0, tp);
            p0 = p1;
            p1 = p2;
        }
        dp = dn * (t * p1 - p0) / (t * t - 1.0);
        if (it < 3) t -= p1 / dp;  // the last pass gives the derivative at the node
    }
    const double w = 1.0 / ((1.0 - t * t) * dp * dp);  // weight 2 / (...) over [-1, 1], halved
    const double lo = 0.5 * (1.0 - t), hi = 0.5 * (1.0 + t);
    nodes[i] = make_double2(lo, lo * w);
    nodes[n - 1 - i] = make_double2(hi, hi * w);
}

// Radial profiles, [nr][nplanes].  A workgroup takes 64 radii (one per lane)
// of BW_PZ planes, its eight waves an eighth of the nodes each: J0 is
// evaluated once for BW_PZ planes, and the defocus phases of a chunk of nodes
// once per workgroup, in LDS, where all lanes of a wave read the same one.
// Bound by the chain of J0 evaluations of one wave (24 nodes): 27 us for 181 x
// 181 x 79 (202 us with one thread per plane and radius).
#define BW_PZ 8
#define BW_SEG 8
#define BW_QC 128
__global__ __launch_bounds__(64 * BW_SEG) void k_bw_profile(const double2* __restrict__ nodes, int nq, int P, int nplanes,
                                                            int nr, double k0NA, double kphase, double step_nm,
                                                            double dz_nm, double* __restrict__ prof)
{
    __shared__ double2 cs[BW_QC * BW_PZ];
    __shared__ double2 red[BW_SEG][64];
    const int lane = threadIdx.x & 63, seg = threadIdx.x >> 6;
    const int m = blockIdx.x * 64 + lane, z0 = blockIdx.y * BW_PZ;
    const double a = k0NA * (double)m * step_nm;  // J0 argument per unit rho
    double re[BW_PZ], im[BW_PZ];
#pragma unroll
    for (int z = 0; z < BW_PZ; ++z) re[z] = im[z] = 0;
    for (int q0 = 0; q0 < nq; q0 += BW_QC) {
        const int nc = min(BW_QC, nq - q0);
        __syncthreads();
        for (int i = threadIdx.x; i < nc * BW_PZ; i += 64 * BW_SEG) {
            const int q = i / BW_PZ, z = min(z0 + i % BW_PZ, nplanes - 1);
            const double rho = nodes[q0 + q].x;
            // defocus as a float (dw_bwpsf.c:549); phase per unit rho^2
            const double b = -kphase * (double)(float)(dz_nm * ((double)z - ((double)P - 1.0) / 2.0));
            sincos(b * rho * rho, &cs[i].y, &cs[i].x);
        }
        __syncthreads();
        for (int q = seg; q < nc; q += BW_SEG) {
            const double2 nd = nodes[q0 + q];
            const double f = j0(a * nd.x) * nd.y;
#pragma unroll
            for (int z = 0; z < BW_PZ; ++z) {
                const double2 c = cs[q * BW_PZ + z];
                re[z] += f * c.x;
                im[z] += f * c.y;
            }
        }
    }
#pragma unroll
    for (int z = 0; z < BW_PZ; ++z) {
        __syncthreads();
        red[seg][lane] = make_double2(re[z], im[z]);
        __syncthreads();
        if (seg == 0 && m < nr && z0 + z < nplanes) {
            double r = 0, i = 0;
            for (int k = 0; k < BW_SEG; ++k) {
                r += red[k][lane].x;
                i += red[k][lane].y;
            }
            prof[(size_t)m * nplanes + z0 + z] = r * r + i * i;
        }
    }
}

struct BwPixelNodes {
    double x[BW_PIXEL_NODES];
    double w[BW_PIXEL_NODES];
};

// Pixel means of one octant (x <= y < h), [octant pixel][plane], one wave per
// pixel.  The mean of the interpolation (lanczos5, lanczos.c:102-160: five
// samples on each side of a position, weights sinc(t) sinc(t/5)) is linear in
// the profile with weights that no plane changes: the 64 node positions span
// at most 36 samples, so the wave first adds the nodes' weights up per sample
// (lane = sample), then takes each plane as one dot product (lane = plane).
// 37 us for 181 x 181 x 79, bound by the weights' double arithmetic; 1554 us
// with one thread per pixel and plane and 20 sines per position.
// sin(pi (d + k)) and sin(pi (d + k)/5) come from d's by the addition
// theorems; positions within 1e-9 of a sample take that sample.
__global__ __launch_bounds__(BTHR) void k_bw_pixels(const double* __restrict__ prof, int nr, int N, int npix, int nplanes,
                                                    int radmax, BwPixelNodes g,
                                                    float* __restrict__ oct)
{
    struct Node {
        double d, s1, s5, c5;  // fraction, weight * sin(pi d), sin and cos(pi d / 5)
        int n;                 // sample below
        double whole;          // weight of sample n alone (0: interpolate)
    };
    __shared__ Node nodes[BTHR / 64][64];
    __shared__ double coef[BTHR / 64][64];
    __shared__ double rot[10][2];  // cos, sin(pi k / 5), k = -5 .. 4
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    if (threadIdx.x < 10) {
        const double k = (double)((int)threadIdx.x - 5);
        rot[threadIdx.x][0] = cospi(k / 5.0);
        rot[threadIdx.x][1] = sinpi(k / 5.0);
    }
    const int i = blockIdx.x * (BTHR / 64) + wid;
    // octant pixel i = y (y + 1) / 2 + x
    int y = (int)((sqrt(8.0 * (double)i + 1.0) - 1.0) * 0.5);
    while ((y + 1) * (y + 2) / 2 <= i) ++y;
    while (y * (y + 1) / 2 > i) --y;
    const int x = i - y * (y + 1) / 2;
    const double c = ((double)N - 1.0) / 2.0;
    const bool inside = i < npix && sqrt((x - c) * (x - c) + (y - c) * (y - c)) < radmax;
    int m0 = 0;
    if (inside) {
        // over [x - 1/2, x + 1/2] x [y - 1/2, y + 1/2] (dw_bwpsf.c:599-634)
        const int a = lane / BW_PIXEL_NODES, b = lane % BW_PIXEL_NODES;
        const double X = (double)x - c + (g.x[a] - 0.5), Y = (double)y - c + (g.x[b] - 0.5);
        const double r2 = X * X + Y * Y, w = g.w[a] * g.w[b];
        const double r = (fabs(r2) > 1e-10 ? sqrt(r2) : 0.0) * (double)BW_OVERSAMPLING;
        Node nd;
        nd.n = (int)floor(r);
        nd.d = r - (double)nd.n;
        nd.whole = 0;
        if (nd.d < 1e-9 || nd.d > 1 - 1e-9) {
            nd.n += nd.d < 1e-9 ? 0 : 1;
            nd.whole = w;
        }
        nd.s1 = w * sinpi(nd.d);
        nd.s5 = sinpi(nd.d / 5.0);
        nd.c5 = cospi(nd.d / 5.0);
        nodes[wid][lane] = nd;
        m0 = nd.n;
        for (int o = 32; o > 0; o >>= 1) m0 = min(m0, __shfl_xor(m0, o, 64));
        m0 -= 4;
    }
    __syncthreads();
    if (inside) {
        const int m = m0 + lane;  // below 0: the profile is symmetric
        double acc = 0;
        for (int q = 0; q < 64; ++q) {
            const Node nd = nodes[wid][q];
            const int k = nd.n - m;
            if (k < -5 || k > 4) continue;
            if (nd.whole != 0) {
                if (k == 0) acc += nd.whole;
                continue;
            }
            const double t = nd.d + (double)k;
            const double s = nd.s5 * rot[k + 5][0] + nd.c5 * rot[k + 5][1];  // sin(pi t / 5)
            const double v = nd.s1 * s * (5.0 / (M_PI * M_PI)) / (t * t);
            acc += (k & 1) ? -v : v;  // sin(pi t) = (-1)^k sin(pi d)
        }
        coef[wid][lane] = acc;
    }
    __syncthreads();
    if (i >= npix) return;
    for (int z = lane; z < nplanes; z += 64) {
        double val = 0;
        if (inside)
            for (int m = 0; m < 36; ++m)
                val += coef[wid][m] * prof[(size_t)min(abs(m0 + m), nr - 1) * nplanes + z];
        oct[(size_t)i * nplanes + z] = (float)val;
    }
}

// The whole volume from the octant means (dw_bwpsf.c:726-766, :553-558).
__global__ __launch_bounds__(BTHR) void k_bw_mirror(const float* __restrict__ oct, int N, int P, int nplanes,
                                                    float* __restrict__ V)
{
    const int n2 = N * N;
    const int z = blockIdx.y, fz = min(z, P - 1 - z);
    for (int i = blockIdx.x * BTHR + threadIdx.x; i < n2; i += gridDim.x * BTHR) {
        const int Y = i / N, X = i - Y * N;
        const int fx = min(X, N - 1 - X), fy = min(Y, N - 1 - Y);
        const int a = min(fx, fy), b = max(fx, fy);
        V[(size_t)z * n2 + i] = oct[(size_t)(b * (b + 1) / 2 + a) * nplanes + fz];
    }
}

// n-point Gauss-Legendre rule on [0, 1] on the host (the pixel rule).
static void gauss_legendre01(int n, double* xs, double* ws)
{
    for (int i = 0; i < n; ++i) {
        double t = cos(M_PI * (i + 0.75) / (n + 0.5)), dp = 0;
        for (int it = 0; it < 100; ++it) {
            double p0 = 1, p1 = t;
            for (int k = 2; k <= n; ++k) {
                const double p2 = ((2.0 * k - 1.0) * t * p1 - (k - 1.0) * p0) / k;
                p0 = p1;
                p1 = p2;
            }
            dp = n * (t * p1 - p0) / (t * t - 1.0);
            const double dt = p1 / dp;
            t -= dt;
            if (fabs(dt) < 1e-16) break;
        }
        xs[n - 1 - i] = 0.5 * (t + 1.0);
        ws[n - 1 - i] = 1.0 / ((1.0 - t * t) * dp * dp);
    }
}

extern "C" int dwhip_bw_psf_device(float* out, int64_t N, int64_t P, double lambda_nm, double NA, double ni,
                                   double dxy_nm, double dz_nm, void* stream)
{
    if (!out || N < 1 || P < 1 || N > 4095 || P > 4095 || !(lambda_nm > 0) || !(NA > 0) || !(ni > 0) ||
        !(dxy_nm > 0) || !(dz_nm > 0))
        return DWHIP_ERR_ARG;
    int rc = dwhip_init();
    if (rc != DWHIP_OK) return rc;
    hipStream_t s = (hipStream_t)stream;
    const double c = ((double)N - 1.0) / 2.0;
    const int radmax = (int)lround(sqrt(2.0 * ((double)N - c) * ((double)N - c))) + 1;
    const int nr = (radmax + 1) * BW_OVERSAMPLING + 2;
    const int nplanes = (int)((P + 1) / 2);
    const double k0 = 2.0 * M_PI / lambda_nm;
    const double step_nm = dxy_nm / BW_OVERSAMPLING;
    const double rmax_nm = (double)(nr - 1) * step_nm;
    // nodes enough for J0 up to k0 NA rmax and for the phase of the largest
    // defocus (plane 0)
    const double vmax = k0 * NA * rmax_nm;
    const double wmax = fabs(k0 * NA * NA * (double)(float)(dz_nm * ((double)P - 1.0) / 2.0) / (2.0 * ni));
    const int nq = (int)(64 + 2.0 * (vmax + wmax) / M_PI);
    BwPixelNodes g;
    gauss_legendre01(BW_PIXEL_NODES, g.x, g.w);
    const int h = (int)((N - 1) / 2 + 1), npix = h * (h + 1) / 2;
    // from the stream-ordered pool (hipMalloc and hipFree wait for the device)
    const size_t b_nodes = (size_t)nq * sizeof(double2), b_prof = (size_t)nplanes * nr * sizeof(double);
    char* mem = nullptr;
    hipError_t e = hipMallocAsync((void**)&mem, b_nodes + b_prof + (size_t)npix * nplanes * sizeof(float), s);
    if (e != hipSuccess) return e == hipErrorOutOfMemory ? DWHIP_ERR_NOMEM : DWHIP_ERR_HIP;
    double2* d_nodes = (double2*)mem;
    double* d_prof = (double*)(mem + b_nodes);
    float* d_oct = (float*)(mem + b_nodes + b_prof);
    hipLaunchKernelGGL(k_bw_nodes, dim3(((nq + 1) / 2 + BTHR - 1) / BTHR), dim3(BTHR), 0, s, nq, d_nodes);
    hipLaunchKernelGGL(k_bw_profile, dim3((nr + 63) / 64, (nplanes + BW_PZ - 1) / BW_PZ), dim3(64 * BW_SEG), 0, s,
                       d_nodes, nq, (int)P, nplanes, nr, k0 * NA, k0 * NA * NA / (2.0 * ni), step_nm, dz_nm, d_prof);
    hipLaunchKernelGGL(k_bw_pixels, dim3((npix + BTHR / 64 - 1) / (BTHR / 64)), dim3(BTHR), 0, s, d_prof, nr, (int)N,
                       npix, nplanes, radmax, g, d_oct);
    hipLaunchKernelGGL(k_bw_mirror, dim3((unsigned)((N * N + BTHR - 1) / BTHR), (unsigned)P), dim3(BTHR), 0, s, d_oct,
                       (int)N, (int)P, nplanes, out);
    e = hipGetLastError();
    {
        const hipError_t f = hipFreeAsync(mem, s);
        if (e == hipSuccess) e = f;
    }
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    return e == hipSuccess ? DWHIP_OK : dwhip_hip_fail(e, "Born-Wolf PSF", __LINE__);
}
