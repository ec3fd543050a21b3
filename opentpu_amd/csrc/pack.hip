// The int4x / fp4x6 and nvfp4 weight packers on the GPU, bit-exact with opentpu/quant.py:325-367
// (_x4), :368-400 (_nv) and :403-425 (pack_scales), which the reference runs on the host in numpy
// float64.
//
// One wave per weight row; lane s takes the 32-element sub-blocks s, s+64, ...  All arithmetic
// is IEEE float64 with FMA contraction off, in the reference's order:
//   sb = max|x| / qmax (qmax 7 int4, 6 E2M1)          top = max sb over the row
//   Sw = f32(top / 63) (1 for an all-zero row)        bmax = max sb over the block
//   d  = clip(floor(log2(63 Sw / bmax)), 0, 255)      unit = Sw * 2^-d
//   for f in linspace(0.64, 1.12, 13): m = clip(rint(sb / unit * f), 1, 63), s = unit * m,
//     err = sum((grid(x / s) * s - x)^2) in numpy's pairwise order (8 running partials,
//     ((p0+p1)+(p2+p3))+((p4+p5)+(p6+p7))); the first strictly smaller err wins.
// floor(log2(v)) is taken exactly from v's exponent. numpy's rounded log2 agrees for every
// float32 input: 63 qmax Sw has at most 33 significant bits and bmax = rnd(a / qmax) for a
// float32 a, so v is a power of two or at least ~2^-34 (relative) away from every one.
#include <cmath>

#include "otpu_common.h"

namespace otpu {

struct Search { double f[13]; };

__device__ __forceinline__ double grid_value(double v, bool e2m1) {
    if (!e2m1) {
        double r = __builtin_rint(v);
        return r < -7.0 ? -7.0 : (r > 7.0 ? 7.0 : r);          // NaN passes through, as np.clip
    }
    const double a = fabs(v);
    const int code = (a > 0.25) + (a >= 0.75) + (a > 1.25) + (a >= 1.75) + (a > 2.5) + (a >= 3.5) + (a > 5.0);
    const double mag[8] = {0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0};
    const double sg = v > 0.0 ? 1.0 : (v < 0.0 ? -1.0 : (v == 0.0 ? 0.0 : v));   // np.sign
    return sg * mag[code];
}

__device__ __forceinline__ int e2m1_code(double v) {
    const double a = fabs(v);
    return (a > 0.25) + (a >= 0.75) + (a > 1.25) + (a >= 1.75) + (a > 2.5) + (a >= 3.5) + (a > 5.0);
}

// The candidates' errors without a division.  Every candidate is a float64 division, a rounding
// and a squared error an element, and those divisions were nearly all of the packers' time (int4
// 6144 x 2048: 156 us, where a copy of its bytes takes 11).  Here an element's quotient is its
// product with the scale's reciprocal, off by less than 2^-50 of itself, so
//   - the rounding goes another way only within 2^-50 |x / s| of a midpoint, where the squared
//     error of either side is the same within 2^-48 |x| s (half a step is 1 at most);
//   - e = g s - |x| is off by 2^-52 |x|, its square by 2^-51 |e| |x| + 2^-104 x^2;
// and a sum over n <= 32 elements, with its own roundings, by less than 2^-45 (E + X + 32 s^2), X
// the sum of x^2 (by Cauchy: sum |x| s <= (X + n s^2) / 2).  A winner ahead of every other
// candidate by 2^-40 of both bounds together, s the largest tried, is the exact search's;
// anything closer (equal errors among it) is searched in the reference's arithmetic, and so are
// infinities and NaN.  Measured, 6144 x 2048: int4 156 -> 42 us, fp4 320 -> 71, nvfp4 285 -> 90; one
// row of 2048: 31 -> 10, 75 -> 15, 64 -> 23; weights on half-steps, whose candidates tie in every
// wave: 157 -> 44, 322 -> 73, 286 -> 92.  Still bound by arithmetic: 5 to 8 float64 operations an
// element and candidate.
constexpr double SEARCH_TOL = 0x1p-40;

// the grid value nearest to a >= 0 (a midpoint to either side); *half: half the step there.  E2M1:
// steps of 1/2 below 2, then 1 and 2, by adding and subtracting 1.5 2^52 steps
template <bool E2M1>
__device__ __forceinline__ double near_grid(double a, double* half) {
    if (!E2M1) {
        *half = 0.5;
        return fmin(__builtin_rint(a), 7.0);
    }
    const int e = max(__double2hiint(a) & 0x7ff00000, 0x3ff00000);               // a's binade, 1 at least
    const double c = __hiloint2double(e + (0x43280000 - 0x3ff00000), 0);
    *half = __hiloint2double(e - 0x00200000, 0);
    return fmin((a + c) - c, 6.0);
}

template <bool E2M1, int NE>
__device__ __forceinline__ double near_error(const double (&xv)[NE], double s) {
    const double r = 1.0 / s;
    double p[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int i = 0; i < NE; ++i) {
        double h;
        const double g = near_grid<E2M1>(fabs(xv[i]) * r, &h), e = __builtin_fma(-g, s, fabs(xv[i]));
        p[i & 3] = __builtin_fma(e, e, p[i & 3]);
    }
    return (p[0] + p[1]) + (p[2] + p[3]);
}

template <int NE>
__device__ __forceinline__ double sum_squares(const double (&xv)[NE]) {
    double X = 0.0;
#pragma unroll
    for (int i = 0; i < NE; ++i) X = __builtin_fma(xv[i], xv[i], X);
    return X;
}

// the codes of xv / s from the same products; false if a quotient is within 2^-40 of a midpoint
// (the reference's (grid(x / s) s) / s is within 2^-52 of the grid value, and has its code)
template <bool E2M1, int NE>
__device__ __forceinline__ bool near_codes(const double (&xv)[NE], double s, uint32_t (&word)[NE / 8]) {
    const double r = 1.0 / s;
    bool clear = true;
#pragma unroll
    for (int w = 0; w < NE / 8; ++w) word[w] = 0;
#pragma unroll
    for (int i = 0; i < NE; ++i) {
        double h;
        const double a = fabs(xv[i]) * r, g = near_grid<E2M1>(a, &h);
        clear &= fabs(fabs(a - g) - h) >= 0x1p-40;        // (past the last grid value: never taken for one)
        uint32_t code;
        if (!E2M1) {
            const int k = (int)g;
            code = (uint32_t)(xv[i] < 0.0 ? -k : k) & 15;
        } else {
            const int k = (int)(2.0 * g), mag = k <= 4 ? k : (k == 6 ? 5 : (k == 8 ? 6 : 7));
            code = (uint32_t)(mag | (xv[i] < 0.0 && mag != 0 ? 8 : 0));
        }
        word[i >> 3] |= code << (4 * (i & 7));
    }
    return clear;
}

// one of a row's sub-blocks (past the row: zeros); its float64 magnitude
template <int NE>
__device__ __forceinline__ double load_block(const float* x, bool ok, double (&xv)[NE]) {
    float v[NE];
    if (ok && ((uintptr_t)x & 15) == 0) {
#pragma unroll
        for (int i = 0; i < NE / 4; ++i) *reinterpret_cast<float4*>(v + 4 * i) = *reinterpret_cast<const float4*>(x + 4 * i);
    } else {
#pragma unroll
        for (int i = 0; i < NE; ++i) v[i] = ok ? x[i] : 0.0f;
    }
    float m = 0.0f;
#pragma unroll
    for (int i = 0; i < NE; ++i) {
        m = fmaxf(m, fabsf(v[i]));
        xv[i] = (double)v[i];
    }
    return (double)m;
}

// three waves a SIMD: the 32 float64 elements a lane holds take 64 registers, the search's eight or
// so in flight the rest
template <bool E2M1>
__global__ __launch_bounds__(64, 3) void pack_x4_kernel(const float* __restrict__ W, int K, int64_t ldw,
                                                     uint8_t* __restrict__ rows, int64_t rs,
                                                     uint8_t* __restrict__ srows, int64_t srs, Search sr) {
    const int row = blockIdx.x, lane = threadIdx.x;
    const float* x = W + (int64_t)row * ldw;
    const int NS = K / 32, KB = K / 128;
    const double qmax = E2M1 ? 6.0 : 7.0;

    double xv[32], top = 0.0, amax = 0.0;
    for (int s = lane; s < (NS + 63) / 64 * 64; s += 64) {
        amax = load_block(x + 32 * s, s < NS, xv);
        top = fmax(top, amax / qmax);
    }
    for (int o = 32; o > 0; o >>= 1) top = fmax(top, __shfl_xor(top, o, 64));
    const double Sw = top == 0.0 ? 1.0 : (double)(float)(top / 63.0);
    uint8_t* srow = srows + (int64_t)row * srs;
    uint8_t* erow = rows + (int64_t)row * rs;

    for (int s0 = 0; s0 < NS; s0 += 64) {               // uniform: every lane shuffles
        const int s = s0 + lane;
        const bool ok = s < NS;
        if (NS > 64) amax = load_block(x + 32 * s, ok, xv);           // (else still held)
        const double sb = amax / qmax;
        double bmax = fmax(sb, __shfl_xor(sb, 1, 64));
        bmax = fmax(bmax, __shfl_xor(bmax, 2, 64));
        double d = 0.0;
        if (bmax > 0.0) {
            const double v = 63.0 * Sw / bmax;
            if (isinf(v)) d = 255.0;
            else if (v > 0.0) {
                int e;
                frexp(v, &e);                            // v in [2^(e-1), 2^e)
                d = (double)(e - 1);
                d = d < 0.0 ? 0.0 : (d > 255.0 ? 255.0 : d);
            }
        }
        const double unit = Sw * exp2(-d);
        const double m0 = sb / unit;
        auto mult = [&](int c) {
            const double m = __builtin_rint(m0 * sr.f[c]);
            return m < 1.0 ? 1.0 : (m > 63.0 ? 63.0 : m);
        };
        auto at = [&](int i) { return ok ? (double)x[32 * s + i] : 0.0; };    // read again: seldom used
        const double X = sum_squares(xv), inf = __builtin_inf();
        double best_m = 0.0, best_e = inf, next_e = inf, last = 0.0;
#pragma unroll 1
        for (int c = 0; c < 13; ++c) {
            const double m = mult(c);
            if (m == last) continue;                     // (multipliers never fall: an equal one is the last)
            last = m;
            const double E = near_error<E2M1>(xv, unit * m);
            if (E < best_e) { next_e = best_e; best_e = E; best_m = m; }
            else next_e = fmin(next_e, E);
        }
        // the largest scale tried bounds the errors' errors; unit 0, infinities and NaN are not plain
        const double s1 = unit * last, reach = best_e + SEARCH_TOL * (best_e + X + 64.0 * (s1 * s1));
        const bool plain = m0 < 1e6 && X < inf;
        if (!(plain && next_e > reach)) {
            bool first = true;
            last = 0.0;
#pragma unroll 1
            for (int c = 0; c < 13; ++c) {
                const double m = mult(c);
                if (m == last) continue;
                last = m;
                const double sc = unit * m;
                if (plain && near_error<E2M1>(xv, sc) > reach) continue;
                double p[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};      // (0 + e is e)
#pragma unroll 1
                for (int i0 = 0; i0 < 32; i0 += 8) {
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        const double v = at(i0 + i), q = grid_value(v / sc, E2M1) * sc;
                        p[i] = p[i] + (q - v) * (q - v);
                    }
                }
                const double err = ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
                if (first || err < best_e) { best_e = err; best_m = m; }
                first = false;
            }
        }
        // element codes of the winner: g = (grid(x/s) * s) / (unit * m)
        const double sc = unit * best_m;
        uint32_t word[4];
        if (!(near_codes<E2M1>(xv, sc, word) && plain)) {
#pragma unroll 1
            for (int w = 0; w < 4; ++w) {
                uint32_t u = 0;
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const double g = (grid_value(at(8 * w + i) / sc, E2M1) * sc) / sc;
                    uint32_t code;
                    if (!E2M1) {
                        code = (uint32_t)((long long)__builtin_rint(g) & 15);
                    } else {
                        const int mag = e2m1_code(g);
                        code = (uint32_t)(mag | ((signbit(g) && mag != 0) ? 8 : 0));
                    }
                    u |= code << (4 * i);
                }
#pragma unroll
                for (int k = 0; k < 4; ++k) word[k] = k == w ? u : word[k];
            }
        }
        if (ok) *reinterpret_cast<uint4*>(erow + 16 * s) = make_uint4(word[0], word[1], word[2], word[3]);
        // the block's scale word: dw | m_b << (8 + 6 b), assembled by the block's first lane
        const uint32_t mb = (uint32_t)best_m;
        const uint32_t m1 = __shfl_xor(mb, 1, 64), m2 = __shfl_xor(mb, 2, 64), m3 = __shfl_xor(mb, 3, 64);
        if (ok && (s & 3) == 0) {
            const uint32_t wd = (uint32_t)d | (mb << 8) | (m1 << 14) | (m2 << 20) | (m3 << 26);
            *reinterpret_cast<uint32_t*>(srow + 8 + 4 * (s >> 2)) = wd;
        }
    }
    if (lane == 0) {
        const float swf = E2M1 ? (float)(Sw * 0.5) : (float)Sw;
        *reinterpret_cast<float*>(srow) = swf;
        *reinterpret_cast<uint32_t*>(srow + 4) = 0u;
    }
    // padding: scale-row words past the last block, element bytes past K/2
    for (int t = 8 + 4 * KB + 4 * lane; t + 4 <= srs && t < 8 + 8 * ((KB + 1) / 2); t += 256)
        *reinterpret_cast<uint32_t*>(srow + t) = 0u;
    const int64_t rb = (int64_t)((K + 255) / 256) * 128;
    for (int64_t t = K / 2 + 16 * lane; t < rb; t += 1024)
        *reinterpret_cast<uint4*>(erow + t) = make_uint4(0, 0, 0, 0);
}

// E4M3 (bias 7, subnormals at E = 0, no infinities): round a non-negative float64 to nearest,
// ties to the even mantissa, saturating at 448 (code 126).  From the binade: a = f 2^e with f in
// [1, 2) -> code ((e + 7) << 3) + rint((f - 1) 8) (a mantissa carry moves into the exponent);
// below 2^-6 the subnormal step 2^-9.  Every operation is exact but the final rint.
__device__ __forceinline__ int e4m3_rne(double a) {
    if (!(a > 0.0)) return 0;
    int ex;
    frexp(a, &ex);                                               // a in [2^(ex-1), 2^ex)
    const int e = ex - 1;
    int code;
    if (e < -6) code = (int)__builtin_rint(a * 512.0);
    else code = ((e + 7) << 3) + (int)__builtin_rint((ldexp(a, -e) - 1.0) * 8.0);
    return code > 126 ? 126 : code;
}

__device__ __forceinline__ double e4m3_val(int c) {
    const int E = c >> 3, m = c & 7;
    return E == 0 ? (double)m * 0x1p-9 : (double)(8 + m) * ldexp(1.0, E - 10);
}

// nvfp4 with a per-row scale (opentpu/quant.py:368-400, _nv): one wave per row, lane t takes the
// 16-element groups t, t + 64, ...  ts = f32(row amax / 2688) (1 for a zero row); per group the
// E4M3 scale s = e4m3(amax_g / ts * f / 6) over the 13 candidates f, s = 1 where the group or s
// is 0, err = sum((sign(xb) E2M1(|xb| / s) s - xb)^2) in numpy's order for 16 terms (8 running
// partials then ((p0+p1)+(p2+p3))+((p4+p5)+(p6+p7))), the first strictly smaller err wins;
// element codes of q / s; Sw = f32(16 ts).
__global__ __launch_bounds__(64) void pack_nv_kernel(const float* __restrict__ W, int K, int64_t ldw,
                                                     uint8_t* __restrict__ rows, int64_t rs,
                                                     uint8_t* __restrict__ srows, int64_t srs, Search sr) {
    const int row = blockIdx.x, lane = threadIdx.x;
    const float* x = W + (int64_t)row * ldw;
    const int NG = K / 16, KB = K / 128;
    const double mag[8] = {0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0};

    float am = 0.0f;
    for (int i = lane; i < K; i += 64) am = fmaxf(am, fabsf(x[i]));
    for (int o = 32; o > 0; o >>= 1) am = fmaxf(am, __shfl_xor(am, o, 64));
    double ts = (double)am / 2688.0;
    ts = (double)(float)(ts == 0.0 ? 1.0 : ts);
    const double rts = 1.0 / ts;
    uint8_t* srow = srows + (int64_t)row * srs;
    uint8_t* erow = rows + (int64_t)row * rs;

    for (int g0 = 0; g0 < NG; g0 += 64) {                // uniform: every lane shuffles
        const int g = g0 + lane;
        const bool ok = g < NG;
        // the search without divisions first (see near_error), on x * (1 / ts) for x / ts
        double xq[16];
        const double amax = load_block(x + 16 * g, ok, xq) / ts;
#pragma unroll
        for (int i = 0; i < 16; ++i) xq[i] *= rts;
        auto at = [&](int i) { return ok ? (double)x[16 * g + i] : 0.0; };    // read again: seldom used
        auto scale = [&](int c) {
            const double s = e4m3_val(e4m3_rne(amax * sr.f[c] / 6.0));
            return amax == 0.0 || s == 0.0 ? 1.0 : s;
        };
        const double X = sum_squares(xq), inf = __builtin_inf();
        const bool plain = X < inf && amax < inf && ts > 0.0;         // (no NaN, no infinity)
        double best_s = 0.0, best_e = inf, next_e = inf, last = 0.0, s1 = 0.0;
#pragma unroll 1
        for (int c = 0; c < 13; ++c) {
            const double s = scale(c);
            if (s == last) continue;
            last = s;
            s1 = fmax(s1, s);
            const double E = near_error<true>(xq, s);
            if (E < best_e) { next_e = best_e; best_e = E; best_s = s; }
            else next_e = fmin(next_e, E);
        }
        const double reach = best_e + SEARCH_TOL * (best_e + X + 64.0 * (s1 * s1));
        if (!(plain && next_e > reach)) {
            bool first = true;
            last = 0.0;
#pragma unroll 1
            for (int c = 0; c < 13; ++c) {
                const double s = scale(c);
                if (s == last) continue;
                last = s;
                if (plain && near_error<true>(xq, s) > reach) continue;
                double p[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};      // (0 + e is e)
#pragma unroll 1
                for (int i0 = 0; i0 < 16; i0 += 8) {
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        const double v = at(i0 + i) / ts;
                        const double sg = v > 0.0 ? 1.0 : (v < 0.0 ? -1.0 : 0.0);
                        const double q = sg * mag[e2m1_code(v / s)] * s;
                        p[i] = p[i] + (q - v) * (q - v);
                    }
                }
                const double err = ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
                if (first || err < best_e) { best_e = err; best_s = s; }
                first = false;
            }
        }
        uint32_t word[2];
        if (!(near_codes<true>(xq, best_s, word) && plain)) {
#pragma unroll 1
            for (int w = 0; w < 2; ++w) {
                uint32_t u = 0;
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const double v = at(8 * w + i) / ts;
                    const double sg = v > 0.0 ? 1.0 : (v < 0.0 ? -1.0 : 0.0);
                    const double gq = (sg * mag[e2m1_code(v / best_s)] * best_s) / best_s;
                    const int mg = e2m1_code(gq);
                    u |= (uint32_t)(mg | ((signbit(gq) && mg != 0) ? 8 : 0)) << (4 * i);
                }
                if (w == 0) word[0] = u;
                else word[1] = u;
            }
        }
        if (ok) *reinterpret_cast<uint2*>(erow + 8 * g) = make_uint2(word[0], word[1]);
        // the block's eight E4M3 bytes, assembled by its first lane
        const uint32_t b = (uint32_t)e4m3_rne(best_s);
        uint32_t lo = 0, hi = 0;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const uint32_t v = (uint32_t)__shfl(b, (lane & ~7) + j, 64);
            if (j < 4) lo |= v << (8 * j);
            else hi |= v << (8 * (j - 4));
        }
        if (ok && (g & 7) == 0) *reinterpret_cast<uint2*>(srow + 16 + g) = make_uint2(lo, hi);
    }
    if (lane == 0) {
        *reinterpret_cast<float*>(srow) = (float)(16.0 * ts);
        *reinterpret_cast<uint32_t*>(srow + 4) = 0u;
        *reinterpret_cast<uint2*>(srow + 8) = make_uint2(0u, 0u);
        if (KB & 1) *reinterpret_cast<uint2*>(srow + 16 + 8 * KB) = make_uint2(0u, 0u);
    }
    const int64_t rb = (int64_t)((K + 255) / 256) * 128;
    for (int64_t t = K / 2 + 16 * lane; t < rb; t += 1024)
        *reinterpret_cast<uint4*>(erow + t) = make_uint4(0, 0, 0, 0);
}

}  // namespace otpu

using namespace otpu;

extern "C" int otpu_pack_x4(const float* W, int N, int K, int64_t ldw, int fmt, uint8_t* rows, int64_t rs,
                            uint8_t* srows, int64_t srs, otpu_stream_t stream) {
    if (fmt != OTPU_INT4 && fmt != OTPU_FP4 && fmt != OTPU_NVFP4)
        return otpu_fail(OTPU_EFORMAT, "pack_x4: format %d (int4, fp4 or nvfp4)", fmt);
    if (N < 1 || K < OTPU_D || K % OTPU_D || ldw < K)
        return otpu_fail(OTPU_EINVAL, "pack_x4: N %d, K %d, ldw %lld", N, K, (long long)ldw);
    const int KB = K / OTPU_D;
    const int64_t rb = (int64_t)((K + 255) / 256) * 128;
    const int64_t sb = fmt == OTPU_NVFP4 ? 16 + 16 * ((KB + 1) / 2) : 8 + 8 * ((KB + 1) / 2);
    if (rs < rb || srs < sb || rs % 16 || srs % 8)
        return otpu_fail(OTPU_EINVAL, "pack_x4: rows of %lld bytes (need %lld, a multiple of 16), scale rows of %lld (need %lld, a multiple of 8)",
                         (long long)rs, (long long)rb, (long long)srs, (long long)sb);
    if (((uintptr_t)rows & 15) || ((uintptr_t)srows & 7) || ((uintptr_t)W & 3))
        return otpu_fail(OTPU_EALIGN, "pack_x4: rows 16-byte, scale rows 8-byte aligned");
    Search sr;
    const double start = 0.64, stop = 1.12, step = (stop - start) / 12.0;   // numpy.linspace(0.64, 1.12, 13)
    for (int i = 0; i < 12; ++i) {
        volatile double t = (double)i * step;                                // no contraction
        sr.f[i] = t + start;
    }
    sr.f[12] = stop;
    hipStream_t s = (hipStream_t)stream;
    if (fmt == OTPU_NVFP4) pack_nv_kernel<<<N, 64, 0, s>>>(W, K, ldw, rows, rs, srows, srs, sr);
    else if (fmt == OTPU_FP4) pack_x4_kernel<true><<<N, 64, 0, s>>>(W, K, ldw, rows, rs, srows, srs, sr);
    else pack_x4_kernel<false><<<N, 64, 0, s>>>(W, K, ldw, rows, rs, srows, srs, sr);
    return otpu_launch_check("pack_x4");
}
