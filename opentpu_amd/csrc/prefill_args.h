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

// rounds of tiles of `rows` x 128 rows, one tile a CU
inline int64_t rounds(int M, int N, int rows) {
    const int64_t tiles = (int64_t)((M + rows - 1) / rows) * ((N + 127) / 128), cus = otpu_cu_count();
    return (tiles + cus - 1) / cus;
}

// row tiles of 32 a workgroup, 1 or 2.  A round of 64 rows costs ~1.7 of 32's, and a call a round's start besides
// (us at 32 -> at 64 rows a tile: int4 512 x 2048 x 8192 52.5 -> 46.1, 300 rows 40.8 -> 44.1, 64 rows 22.7 -> 30.9;
// nvfp4 2 x 1024 x 70000 in ranges 51.8 -> 82.7): this line is within 0.3% of the faster one on the mean of 818
// shapes.  int8's ranges take 32 rows (65 x 2048 x 12288 45 / 71, 512 x 2048 x 8192 80 / 79): no kernel of 64
constexpr bool has_tall_tile(int fmt, bool ranged) { return !(fmt == OTPU_INT8 && ranged); }
inline int row_tiles(int M, int N, int fmt, int ranges) {
    if (!has_tall_tile(fmt, ranges > 1)) return 1;
    return 5 * (1 + rounds(M, N, 32)) > 8 * (1 + rounds(M, N, 64)) ? 2 : 1;
}

// false: no such kernel (nothing launched)
template <int FMT>
bool launch_fmt(const Args& a, int ms, hipStream_t s);

}  // namespace pf
}  // namespace otpu
