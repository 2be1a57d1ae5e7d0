// One column-pass mode (CMODE, set by the build) of the SHB loop.
#include "shb_passes.h"

#ifndef CMODE
#error "compile with -DCMODE=<mode>"
#endif
#define DWHIP_CAT2(a, b) a##b
#define DWHIP_CAT(a, b) DWHIP_CAT2(a, b)

// PASS_EXT: the mode's kernel for extended jobs; PASS_YSMALL: with the small y
// workgroups
#ifdef PASS_EXT
#define PASS_EXT_V true
#else
#define PASS_EXT_V false
#endif
#ifdef PASS_YSMALL
#define PASS_YS_V true
#else
#define PASS_YS_V false
#endif
#if defined(PASS_EXT) && defined(PASS_YSMALL)
#define PASS_LAUNCH DWHIP_CAT(dwhip_launch_cse, CMODE)
#elif defined(PASS_EXT)
#define PASS_LAUNCH DWHIP_CAT(dwhip_launch_ce, CMODE)
#elif defined(PASS_YSMALL)
#define PASS_LAUNCH DWHIP_CAT(dwhip_launch_cs, CMODE)
#else
#define PASS_LAUNCH DWHIP_CAT(dwhip_launch_c, CMODE)
#endif

extern "C" hipError_t PASS_LAUNCH(const BatchDev* bd, const JobDev* jobs, int grid, size_t lds,
                                                      hipStream_t s)
{
    static bool once = false;
    if (!once) {
        once = true;
        dwhip_allow_big_lds(reinterpret_cast<const void*>(k_colpass<CMODE, PASS_EXT_V, PASS_YS_V>));
    }
    hipLaunchKernelGGL((k_colpass<CMODE, PASS_EXT_V, PASS_YS_V>), dim3(grid), dim3((col_threads<CMODE, PASS_YS_V>())), lds, s, bd, jobs);
    return hipGetLastError();
}
