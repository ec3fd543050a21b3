// The batch MM's host side: which calls it takes and the launch's shape (the kernel: batch_impl.h).
#include "batch_args.h"

using namespace otpu;

// returns 1 when the call is not for this kernel, else a status
int otpu_batch_try(const int8_t* q, int64_t ldq, const float* Sa, const uint8_t* da, int64_t ldda, int M, int K,
                   int ranges, const uint8_t* w, int64_t rs, const uint8_t* ws, int64_t srs, int N, int fmt, int flags,
                   int k0, const float* alpha, float* out, int64_t ors, hipStream_t s) {
    if (flags & OTPU_RMAX) return 1;
    if (((uintptr_t)da & 3) || (ldda % 4) || ldda >= (1 << 26) || ldq >= (1 << 26)) return 1;
    bt::Args a = {};
    a.q = q; a.ldq = ldq; a.Sa = Sa; a.da = da; a.ldda = ldda; a.M = M; a.K = K;
    a.w = w; a.rs = rs; a.ws = ws; a.srs = srs; a.N = N; a.flags = flags;
    a.k0 = (flags & (OTPU_UNIT | OTPU_RSC)) ? 0 : k0;
    a.alpha = alpha; a.out = out; a.ors = ors; a.ranges = ranges;
    const int mt = M > 16 ? 2 : 1;
    const int64_t tiles_m = (M + 16 * mt - 1) / (16 * mt);
    const int parts = ranges > 1 ? ranges : K / OTPU_D;           // what the waves can split
    int kwmax = 8;
    while (kwmax > parts) kwmax >>= 1;
    const int64_t want = 8 * (int64_t)otpu_cu_count();
    // 64 weight rows a wave tile, but 32 beside 32 activation rows where those spill (int8 101 registers,
    // int4 41): us at 64 -> at 32, QACT in: int8 512 x 2048 x 1024 22.1 -> 18.3, 512 x 3072 x 1024 in ranges of 256
    // 46.0 -> 31.9, 100 x 2048 x 6000 36.3 -> 29.1; nvfp4 29.6 -> 26.0, 61.7 -> 46.7, 49.9 -> 43.2; fp4's ranges 40.2
    // -> 37.4, int4's 37.6 -> 36.4, but without ranges int4 100 x 2048 x 6000 31.7 -> 33.4, fp4 34.7 -> 34.8
    int nsub = mt == 2 && (!bt::has_wide_tile(fmt) || ranges > 1) ? 2 : 4;
    while (nsub > 1 && (int64_t)((N + 16 * nsub - 1) / (16 * nsub)) * tiles_m * kwmax < want) nsub >>= 1;
    int kw = 1;
    while (kw < kwmax && (int64_t)((N + 16 * nsub - 1) / (16 * nsub)) * tiles_m * kw < want) kw <<= 1;
    a.kw = kw;
    a.tiles_n = (N + 16 * nsub - 1) / (16 * nsub);
    a.groups_m = (int)(((M + 16 * mt - 1) / (16 * mt) + 8 / kw - 1) / (8 / kw));
    bool ok;
    switch (fmt) {
        case OTPU_INT8: ok = bt::launch_fmt<OTPU_INT8>(a, nsub, mt, s); break;
        case OTPU_INT4: ok = bt::launch_fmt<OTPU_INT4>(a, nsub, mt, s); break;
        case OTPU_FP4: ok = bt::launch_fmt<OTPU_FP4>(a, nsub, mt, s); break;
        default: ok = bt::launch_fmt<OTPU_NVFP4>(a, nsub, mt, s); break;
    }
    if (!ok) return otpu_fail(OTPU_EINVAL, "mm batch: no kernel of format %d for %d x %d rows a wave", fmt, 16 * nsub, 16 * mt);
    return otpu_launch_check("mm batch");
}
