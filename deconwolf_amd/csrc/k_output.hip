// Output path of dw_run on the device: the statistics deconwolf takes of
// the result before writing it (largest value for the 16-bit scaling,
// scaling_for_u16 src/dw.c:98-103 over fim_max; voxels at the background
// level, get_nbg src/dw.c:2406-2418) and the float -> uint16 conversions of
// its writers:
//   DWHIP_U16_ROUND  fim_tiff_write_opt (src/fim_tiff.c:1138-1150): v*s, values
//                    above 65535 -> 65535, non-finite -> 0, round half away
//   DWHIP_U16_TRUNC  fim_imwrite_u16 to .npy (src/fim.c:5142-5147) and
//                    fim_tiff_imwrite_u16_from_raw (src/fim_tiff.c:819-822):
//                    (uint16_t)(v*s), truncation
//   DWHIP_U16_RINT   raw_to_npio (src/dw.c:187-190): nearbyintf(v*s)
// The C conversions are undefined outside [0, 65536); here they saturate to
// [0, 65535] and map NaN to 0.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>
#include <string.h>

#include <algorithm>

#include "dwhip.h"
#include "dwhip_internal.h"

#define OTHR 256

// Monotone map of floats onto unsigned ints (NaN excluded by the caller).
__device__ __forceinline__ unsigned int float_key(float f)
{
    const unsigned int b = __float_as_uint(f);
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}

__host__ __device__ __forceinline__ float key_float(unsigned int k)
{
    const unsigned int b = (k & 0x80000000u) ? (k & 0x7fffffffu) : ~k;
#ifdef __HIP_DEVICE_COMPILE__
    return __uint_as_float(b);
#else
    float f;
    memcpy(&f, &b, sizeof(f));
    return f;
#endif
}

struct OutStats {
    unsigned int maxkey;
    unsigned int pad;
    unsigned long long nbg;
};

// Both kernels stream the volume once and are bound by its bytes: four values
// per load (16-byte aligned volumes; others one by one), OUT_Q loads in flight
// per thread.  1024 x 1024 x 60: statistics 131 -> 63 us, conversion 94 -> 63.
#define OUT_Q 4
struct alignas(8) U16x4 {
    uint16_t v[4];
};

__global__ __launch_bounds__(OTHR) void k_out_stats(const float* __restrict__ v, int64_t n, int64_t n4, float bg,
                                                    OutStats* __restrict__ st)
{
    __shared__ unsigned int smax[OTHR / 64];
    __shared__ unsigned long long scnt[OTHR / 64];
    unsigned int mk = 0;
    unsigned long long cnt = 0;
    auto take = [&](float x) {
        if (x == x) mk = max(mk, float_key(x));
        cnt += (x == bg);
    };
    const int64_t S = (int64_t)gridDim.x * OTHR, i0 = (int64_t)blockIdx.x * OTHR + threadIdx.x;
    const float4* __restrict__ v4 = reinterpret_cast<const float4*>(v);
    int64_t i = i0;
    for (; i + (OUT_Q - 1) * S < n4; i += OUT_Q * S) {
        float4 x[OUT_Q];
#pragma unroll
        for (int q = 0; q < OUT_Q; ++q) x[q] = v4[i + q * S];
#pragma unroll
        for (int q = 0; q < OUT_Q; ++q) {
            take(x[q].x);
            take(x[q].y);
            take(x[q].z);
            take(x[q].w);
        }
    }
    for (; i < n4; i += S) {
        const float4 x = v4[i];
        take(x.x);
        take(x.y);
        take(x.z);
        take(x.w);
    }
    for (i = 4 * n4 + i0; i < n; i += S) take(v[i]);
    for (int o = 32; o > 0; o >>= 1) {
        mk = max(mk, __shfl_xor(mk, o));
        cnt += __shfl_xor(cnt, o);
    }
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        smax[w] = mk;
        scnt[w] = cnt;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int k = 1; k < OTHR / 64; ++k) {
            mk = max(mk, smax[k]);
            cnt += scnt[k];
        }
        atomicMax(&st->maxkey, mk);
        atomicAdd(&st->nbg, cnt);
    }
}

template <int MODE>
__device__ __forceinline__ uint16_t to_u16(float x, float scaling)
{
    float v = x * scaling;
    if (MODE == DWHIP_U16_ROUND) {
        if (v > 65535.f) v = 65535.f;
        if (!isfinite(v)) v = 0.f;
        v = roundf(v);
    } else if (MODE == DWHIP_U16_TRUNC) {
        v = truncf(v);
    } else {
        v = rintf(v);
    }
    if (!(v > 0.f)) return 0;  // also NaN
    return v >= 65535.f ? (uint16_t)65535 : (uint16_t)v;
}

template <int MODE>
__global__ __launch_bounds__(OTHR) void k_to_u16(const float* __restrict__ v, int64_t n, int64_t n4, float scaling,
                                                 uint16_t* __restrict__ out)
{
    const int64_t S = (int64_t)gridDim.x * OTHR, i0 = (int64_t)blockIdx.x * OTHR + threadIdx.x;
    const float4* __restrict__ v4 = reinterpret_cast<const float4*>(v);
    U16x4* __restrict__ o4 = reinterpret_cast<U16x4*>(out);
    auto conv = [&](float4 x) {
        return U16x4{{to_u16<MODE>(x.x, scaling), to_u16<MODE>(x.y, scaling), to_u16<MODE>(x.z, scaling),
                      to_u16<MODE>(x.w, scaling)}};
    };
    int64_t i = i0;
    for (; i + (OUT_Q - 1) * S < n4; i += OUT_Q * S) {
        float4 x[OUT_Q];
#pragma unroll
        for (int q = 0; q < OUT_Q; ++q) x[q] = v4[i + q * S];
#pragma unroll
        for (int q = 0; q < OUT_Q; ++q) o4[i + q * S] = conv(x[q]);
    }
    for (; i < n4; i += S) o4[i] = conv(v4[i]);
    for (i = 4 * n4 + i0; i < n; i += S) out[i] = to_u16<MODE>(v[i], scaling);
}

static int out_grid(int64_t n)
{
    const int64_t g = (n + 4 * OTHR - 1) / (4 * OTHR);
    return (int)(g < 4096 ? (g > 0 ? g : 1) : 4096);
}

// values taken four at a time: all but the last few of an aligned volume
static int64_t out_quads(const float* v, const uint16_t* out, int64_t n)
{
    return ((uintptr_t)v & 15) == 0 && ((uintptr_t)out & 7) == 0 ? n / 4 : 0;
}

extern "C" {

int dwhip_output_stats_device(const float* v, int64_t n, float bg, float* vmax, int64_t* n_bg, void* stream)
{
    if (!v || n < 1) return DWHIP_ERR_ARG;
    int rc = dwhip_init();
    if (rc != DWHIP_OK) return rc;
    hipStream_t s = (hipStream_t)stream;
    OutStats* d = nullptr;
    OutStats h;
    // (the stream-ordered pool gives its memory back at each synchronisation: 56 us
    // for 32768 values where this takes 31)
    hipError_t e = hipMalloc((void**)&d, sizeof(OutStats));
    if (e != hipSuccess) return e == hipErrorOutOfMemory ? DWHIP_ERR_NOMEM : DWHIP_ERR_HIP;
    e = hipMemsetAsync(d, 0, sizeof(OutStats), s);
    if (e == hipSuccess) {
        // (every workgroup ends in two atomics on one line: a thousand at most)
        hipLaunchKernelGGL(k_out_stats, dim3(std::min(out_grid(n), 1024)), dim3(OTHR), 0, s, v, n, out_quads(v, nullptr, n), bg, d);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpyAsync(&h, d, sizeof(h), hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    (void)hipFree(d);
    if (e != hipSuccess) return dwhip_hip_fail(e, "output statistics", __LINE__);
    // key 0 means every value was NaN
    if (vmax) *vmax = h.maxkey ? key_float(h.maxkey) : NAN;
    if (n_bg) *n_bg = (int64_t)h.nbg;
    return DWHIP_OK;
}

int dwhip_to_u16_device(const float* v, int64_t n, float scaling, int mode, uint16_t* out, void* stream)
{
    if (!v || !out || n < 0) return DWHIP_ERR_ARG;
    if (mode != DWHIP_U16_ROUND && mode != DWHIP_U16_TRUNC && mode != DWHIP_U16_RINT) return DWHIP_ERR_ARG;
    if (n == 0) return DWHIP_OK;
    int rc = dwhip_init();
    if (rc != DWHIP_OK) return rc;
    hipStream_t s = (hipStream_t)stream;
    const int g = out_grid(n);
    const int64_t n4 = out_quads(v, out, n);
    if (mode == DWHIP_U16_ROUND)
        hipLaunchKernelGGL(k_to_u16<DWHIP_U16_ROUND>, dim3(g), dim3(OTHR), 0, s, v, n, n4, scaling, out);
    else if (mode == DWHIP_U16_TRUNC)
        hipLaunchKernelGGL(k_to_u16<DWHIP_U16_TRUNC>, dim3(g), dim3(OTHR), 0, s, v, n, n4, scaling, out);
    else
        hipLaunchKernelGGL(k_to_u16<DWHIP_U16_RINT>, dim3(g), dim3(OTHR), 0, s, v, n, n4, scaling, out);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? DWHIP_OK : dwhip_hip_fail(e, "u16 conversion", __LINE__);
}

}  // extern "C"
