// The prefill MM's host side: which calls it takes and the launch's shape (the kernel: prefill_impl.h).
#include "prefill_args.h"

using namespace otpu;

// returns 1 when the call is not for this kernel, else a status
int otpu_prefill_try(const int8_t* q, int64_t ldq, const float* Sa, const uint8_t* da, int64_t ldda, int M, int K,
                     int ranges, const uint8_t* w, int64_t rs, const uint8_t* ws, int64_t srs, int N, int fmt, int flags,
                     int k0, const float* alpha, float* out, int64_t ors, hipStream_t s) {
    if (flags & OTPU_RMAX) return 1;
    if (((uintptr_t)da & 3) || (ldda % 4) || ldq >= (1 << 24)) return 1;
    pf::Args a = {};
    a.q = q; a.ldq = ldq; a.Sa = Sa; a.da = da; a.ldda = ldda; a.M = M; a.K = K;
    a.w = w; a.rs = rs; a.ws = ws; a.srs = srs; a.N = N; a.flags = flags;
    a.k0 = (flags & (OTPU_UNIT | OTPU_RSC)) ? 0 : k0;
    a.alpha = alpha; a.out = out; a.ors = ors; a.ranges = ranges;
    const int ms = pf::row_tiles(M, N, fmt, ranges);
    a.tiles_m = (M + 32 * ms - 1) / (32 * ms);
    a.tiles_n = (N + 127) / 128;
    a.vec4 = ((uintptr_t)out % 16 == 0) && (ors % 4 == 0);
    bool ok;
    switch (fmt) {
        case OTPU_INT8: ok = pf::launch_fmt<OTPU_INT8>(a, ms, s); break;
        case OTPU_INT4: ok = pf::launch_fmt<OTPU_INT4>(a, ms, s); break;
        case OTPU_FP4: ok = pf::launch_fmt<OTPU_FP4>(a, ms, s); break;
        default: ok = pf::launch_fmt<OTPU_NVFP4>(a, ms, s); break;
    }
    if (!ok) return otpu_fail(OTPU_EINVAL, "mm prefill: no kernel of format %d for %d rows a tile in ranges", fmt, 32 * ms);
    return otpu_launch_check("mm prefill");
}
