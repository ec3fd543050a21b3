// Shared by the prefill MM's sources (prefill_impl.h): the argument block of one launch and the
// per-format launchers, each in a translation unit of its own.
#pragma once
#include "otpu_common.h"

namespace otpu {
namespace pf {

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
    int tiles_m, tiles_n;           // tiles of 32 MS activation rows; of 128 weight rows
    int vec4;                       // out 16-byte aligned and ors a multiple of 4: float4 stores
};

template <int FMT>
void launch_fmt(const Args& a, int ms, hipStream_t s);

}  // namespace pf
}  // namespace otpu
