// Shared by the batch MM's sources (batch_impl.h): the argument block of one launch and the
// per-format launchers, each in a translation unit of its own.
#pragma once
#include "otpu_common.h"

namespace otpu {
namespace bt {

struct Args {
    const int8_t* q; int64_t ldq;
    const float* Sa;                // range r's row j at Sa[r * M + j]
    const uint8_t* da; int64_t ldda;
    int M, K;
    const uint8_t* w; int64_t rs;
    const uint8_t* ws; int64_t srs;
    int N, flags, k0;
    const float* alpha;
    float* out; int64_t ors;
    int ranges;                     // equal ranges of K, their outputs added in order (ACC)
    int kw;                         // waves a workgroup splits K over (1, 2, 4 or 8)
    int tiles_n, groups_m;          // tiles of 16 NSUB weight rows; groups of 8 / kw row tiles
};

// the formats with a kernel of 64 weight rows beside 32 activation rows a wave (nsub 4, mt 2); in the others 32
// weight rows are the faster (batch.hip's rule)
constexpr bool has_wide_tile(int fmt) { return fmt == OTPU_INT4 || fmt == OTPU_FP4; }

// false: no such kernel (nothing launched)
template <int FMT>
bool launch_fmt(const Args& a, int nsub, int mt, hipStream_t s);

}  // namespace bt
}  // namespace otpu
