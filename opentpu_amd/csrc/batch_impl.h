// MM for a batch of activation rows (more than four, or any number in several ranges: mm_rows in
// gemv.hip) on the int8 MFMA units with the group scales applied to the products, not folded into the
// operands.  Semantics: opentpu/isasim.py:749-910
// (docs/isa.md:226-305), and the ranges' ACC chain of Builder.dot (opentpu/compiler.py:2686-2720).
//
// One v_mfma_i32_16x16x32_i8 is one 32-group of 16 activation rows x 16 weight rows: its int32 sums
// are the groups' integer dot products c, whatever offsets the operands carry, so one walk of K
// serves every activation offset and every weight multiplier (a GEMM of shifted operand planes
// walks or multiplies K once a plane).  Over a 128-block the terms m c 2^(D - da) add up in int32
// (below), and the block's sum joins an exact double: acc += t 2^(W - D - dw), one conversion and
// one fma a block and output.  Every term and sum of one MM is an integer below 2^47, which a double
// holds exactly, so neither the split of K over waves nor the order of the sums can change a bit.
//
// Work layout.  No operand goes through LDS: weights stream from memory straight into the MFMA's
// layout (lane: weight row lane & 15, 16 contiguous bytes), activations come from the caches.  A
// wave owns 16 MT activation rows x 16 NSUB weight rows and some blocks of K; kw of a workgroup's 8
// waves split K between them (their doubles meet in LDS), 8 / kw take successive row tiles of the
// same weights.  So a small grid still fills the chip: 1024 x 2048 weights at 16 rows are 64
// workgroups x 8 waves of two blocks each.
#pragma once
#include "batch_args.h"

namespace otpu {
namespace bt {

typedef int v4i __attribute__((ext_vector_type(4)));

// The windows of a block's int32 sums: activation offsets up to D and (by dw <= W - D) no dropped
// term.  Bounds of a block's |t| = sum over 4 groups of |c m| 2^D, all below 2^31:
//   int8:  |c| <= 32 128 128, D 8:               2^19 2^8 4                  = 5.4e8
//   int4:  the MFMA multiplies 16 w: 16 32 128 8 63 4, D 4:                  = 2.114e9
//   fp4:   |w| <= 12: 32 128 12 63 4, D 6:                                   = 7.9e8
//   nvfp4: two 16-groups, m 2^(E - Eb + 3) <= 15 8: 16 128 12 120 8, D 6:    = 1.51e9
// A block with an offset outside them takes the group-by-group double path (exact for any).
template <int FMT>
struct Win {
    static constexpr int W = FMT == OTPU_INT8 ? 16 : (FMT == OTPU_NVFP4 ? 13 : 11);
    static constexpr int D = FMT == OTPU_INT8 ? 8 : (FMT == OTPU_INT4 ? 4 : 6);
    static constexpr int EW = 3;                          // nvfp4: octaves below the block's largest scale
    static constexpr int PRE = FMT == OTPU_INT4 ? 4 : 0;  // the operands carry w 2^PRE
};

__device__ __forceinline__ double pow2d(int e) { return __hiloint2double((1023 + e) << 20, 0); }

// E2M1 codes (4 per dword, one per byte, 0..15) -> signed int8 values, twice the E2M1 value
__device__ __forceinline__ uint32_t e2m1x4(uint32_t nib) {
    const uint32_t sel = nib & 0x07070707u;
    const uint32_t pos = __builtin_amdgcn_perm(0x0C080604u, 0x03020100u, sel);
    const uint32_t neg = __builtin_amdgcn_perm(0xF4F8FAFCu, 0xFDFEFF00u, sel);
    return __builtin_amdgcn_perm(neg, pos, ((nib >> 1) & 0x04040404u) | 0x03020100u);
}

__device__ __forceinline__ long pair64(uint32_t lo, uint32_t hi) { return (long)(((uint64_t)hi << 32) | lo); }

// lanes 16 c + r hold the four dwords of group c: afterwards x[g] holds dword c of group g (a 4 x 4
// transpose between registers and the wave's four rows of 16 lanes)
__device__ __forceinline__ void transpose4(uint32_t (&x)[4]) {
    auto a = __builtin_amdgcn_permlane32_swap(x[0], x[2], false, false);
    auto b = __builtin_amdgcn_permlane32_swap(x[1], x[3], false, false);
    auto lo = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false);
    auto hi = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
    x[0] = lo[0];
    x[1] = lo[1];
    x[2] = hi[0];
    x[3] = hi[1];
}

// one block's operands of a wave
template <int FMT, int NSUB, int MT>
struct Stage {
    static constexpr int WL = FMT == OTPU_INT8 ? 2 : 1;   // 16-byte weight loads a row
    uint4 w[NSUB][WL];
    uint32_t sc[NSUB];                                    // the rows' scale word (int8: dw)
    uint32_t sc2[FMT == OTPU_NVFP4 ? NSUB : 1];           // nvfp4: the other four E4M3 scales
    uint4 a[MT][2];                                       // 4-bit: 4 x 8 bytes, int8: 2 x 16 bytes
    uint32_t da[MT][4];                                   // offsets of rows 4 c + t, a byte a group
};

template <int FMT, int NSUB, int MT>
__global__ __launch_bounds__(512) void batch_kernel(Args p) {
    using F = Win<FMT>;
    constexpr int W = F::W, D = F::D;
    constexpr bool I8 = FMT == OTPU_INT8, NV = FMT == OTPU_NVFP4;
    constexpr int ITEMS = 4 * NSUB * MT;                  // outputs a lane
    __shared__ __align__(16) double red[8 * ITEMS * 64];  // the K split's sums, or the ranges' fp32 rows

    const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r16 = lane & 15, c = lane >> 4;
    const int kw = p.kw, kwi = wid & (kw - 1), mi = wid / kw, mw = 8 / kw;
    // the row groups of one weight tile are neighbours on one XCD (workgroup b runs on XCD b % 8)
    int t = blockIdx.x;
    const int total = p.tiles_n * p.groups_m;
    if (total % 8 == 0) t = (t & 7) * (total >> 3) + (t >> 3);
    const int tn = t / p.groups_m, tg = t % p.groups_m;
    const int n0 = tn * 16 * NSUB, m0 = (tg * mw + mi) * 16 * MT;
    const int KB = p.K / OTPU_D;
    const bool plain = (p.flags & (OTPU_UNIT | OTPU_RSC)) != 0;

    // the wave's first rows (scalar) and this lane's byte offsets from them (past M or N: the last
    // row, whose outputs are not stored)
    const int nb = min(n0, p.N - 1), mb = min(m0, p.M - 1);
    const uint8_t* const wb = p.w + (int64_t)nb * p.rs;
    const uint8_t* const sb = p.ws + (int64_t)nb * p.srs + (I8 ? 4 + p.k0 : (NV ? 16 + 8 * p.k0 : 8 + 4 * p.k0));
    const int8_t* const qb = p.q + (int64_t)mb * p.ldq;
    const uint8_t* const db = p.da + (int64_t)mb * p.ldda;
    uint32_t wo[NSUB], so[NSUB], qo[MT], dofs[MT][4];
#pragma unroll
    for (int s = 0; s < NSUB; ++s) {
        const int dn = min(16 * s + r16, p.N - 1 - nb);
        wo[s] = (uint32_t)dn * (uint32_t)p.rs + 16u * c;
        so[s] = (uint32_t)dn * (uint32_t)p.srs;
    }
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        qo[i] = (uint32_t)min(16 * i + r16, p.M - 1 - mb) * (uint32_t)p.ldq + (I8 ? 16u : 8u) * c;
#pragma unroll
        for (int u = 0; u < 4; ++u) dofs[i][u] = (uint32_t)min(16 * i + 4 * c + u, p.M - 1 - mb) * (uint32_t)p.ldda;
    }

    using St = Stage<FMT, NSUB, MT>;
    auto load = [&](St& st, int kb) {
        const uint8_t* wk = wb + (I8 ? 128 : 64) * kb;
        const uint8_t* sk = sb + (I8 ? 1 : (NV ? 8 : 4)) * kb;
        const int8_t* qk = qb + 128 * kb;
        const uint8_t* dk = db + 4 * kb;
#pragma unroll
        for (int s = 0; s < NSUB; ++s) {
#pragma unroll
            for (int h = 0; h < St::WL; ++h)
                st.w[s][h] = *reinterpret_cast<const uint4*>(wk + wo[s] + 64 * h);
            if (plain) {
                st.sc[s] = I8 ? 0u : 0x04104100u;         // dw 0, every m 1 (nvfp4: below)
                if (NV) st.sc2[s] = 0u;
            } else if (I8) {
                st.sc[s] = sk[so[s]];
            } else if (NV) {
                st.sc[s] = *reinterpret_cast<const uint32_t*>(sk + so[s]);
                st.sc2[s] = *reinterpret_cast<const uint32_t*>(sk + so[s] + 4);
            } else {
                st.sc[s] = *reinterpret_cast<const uint32_t*>(sk + so[s]);
            }
        }
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            if (I8) {
#pragma unroll
                for (int h = 0; h < 2; ++h) st.a[i][h] = *reinterpret_cast<const uint4*>(qk + qo[i] + 64 * h);
            } else {
                uint2 v[4];
#pragma unroll
                for (int g = 0; g < 4; ++g) v[g] = *reinterpret_cast<const uint2*>(qk + qo[i] + 32 * g);
                st.a[i][0] = make_uint4(v[0].x, v[0].y, v[1].x, v[1].y);
                st.a[i][1] = make_uint4(v[2].x, v[2].y, v[3].x, v[3].y);
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) st.da[i][u] = *reinterpret_cast<const uint32_t*>(dk + dofs[i][u]);
        }
    };

    // one block into the double sums
    auto block = [&](const St& st, double (&acc)[NSUB][MT][4]) {
        // 4-bit: even and odd elements of a lane's 8 apart, as the nibbles come out; nvfp4 (16-groups)
        // and int8 (two 32-groups an MFMA): the lanes of the other group zeroed
        long a4[MT][I8 ? 1 : 4];
        uint32_t bad = 0;
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            if (!I8) {
                const uint32_t d[8] = {st.a[i][0].x, st.a[i][0].y, st.a[i][0].z, st.a[i][0].w,
                                       st.a[i][1].x, st.a[i][1].y, st.a[i][1].z, st.a[i][1].w};
#pragma unroll
                for (int g = 0; g < 4; ++g)
                    a4[i][g] = pair64(__builtin_amdgcn_perm(d[2 * g + 1], d[2 * g], 0x06040200u),
                                      __builtin_amdgcn_perm(d[2 * g + 1], d[2 * g], 0x07050301u));
            }
#pragma unroll
            for (int u = 0; u < 4; ++u)                   // an offset byte above D
                bad |= ((st.da[i][u] + (0x7Fu - D) * 0x01010101u) | st.da[i][u]) & 0x80808080u;
        }
        const uint32_t half = c < 2 ? ~0u : 0u;           // the lanes of a wave's first half
        // the products of sub-tile s, row tile i and group g (nvfp4: 16-group 2 g + h)
        auto mm = [&](const uint32_t (&b)[8], int i, int g, int h) -> v4i {
            const v4i z = {0, 0, 0, 0};
            if constexpr (I8) {
                const uint4 x = g < 2 ? st.a[i][0] : st.a[i][1];
                const uint32_t k = (g & 1) ? ~half : half;
                const v4i av = {(int)(x.x & k), (int)(x.y & k), (int)(x.z & k), (int)(x.w & k)};
                const int o = g < 2 ? 0 : 4;
                const v4i bv = {(int)b[o], (int)b[o + 1], (int)b[o + 2], (int)b[o + 3]};
                return __builtin_amdgcn_mfma_i32_16x16x64_i8(av, bv, z, 0, 0, 0);
            } else {
                long av = a4[i][g];
                if constexpr (NV) {
                    const uint32_t k = h ? ~half : half;
                    av &= pair64(k, k);
                }
                return __builtin_amdgcn_mfma_i32_16x16x32_i8(av, pair64(b[2 * g], b[2 * g + 1]), z, 0, 0, 0);
            }
        };
        auto unpack = [&](int s, uint32_t (&b)[8]) {
            if constexpr (I8) {
                const uint4 x = st.w[s][0], y = st.w[s][St::WL - 1];
                b[0] = x.x; b[1] = x.y; b[2] = x.z; b[3] = x.w;
                b[4] = y.x; b[5] = y.y; b[6] = y.z; b[7] = y.w;
            } else {
                uint32_t x[4] = {st.w[s][0].x, st.w[s][0].y, st.w[s][0].z, st.w[s][0].w};
                transpose4(x);
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    if (FMT == OTPU_INT4) {
                        b[2 * g] = (x[g] << 4) & 0xF0F0F0F0u;
                        b[2 * g + 1] = x[g] & 0xF0F0F0F0u;
                    } else {
                        b[2 * g] = e2m1x4(x[g] & 0x0F0F0F0Fu);
                        b[2 * g + 1] = e2m1x4((x[g] >> 4) & 0x0F0F0F0Fu);
                    }
                }
            }
        };
#pragma unroll
        for (int s = 0; s < NSUB; ++s) {
            uint32_t b[8];
            unpack(s, b);
            const uint32_t sc = st.sc[s], sc2 = NV ? st.sc2[s] : 0u;
            int m[NV ? 8 : 4];
            int e = W - D - F::PRE;                       // the block sum's exponent
            bool out;                                     // outside the windows
            if constexpr (NV) {
                int E[8], Eb = 0;
#pragma unroll
                for (int h = 0; h < 8; ++h) {
                    const uint32_t x = ((h < 4 ? sc : sc2) >> (8 * (h & 3))) & 0x7Fu;
                    const int ex = (int)(x >> 3);
                    m[h] = (int)(x & 7) + (ex ? 8 : 0);
                    E[h] = ex > 1 ? ex : 1;
                    Eb = max(Eb, E[h]);
                }
                bool low = false;
#pragma unroll
                for (int h = 0; h < 8; ++h) {
                    const int d = E[h] - Eb + F::EW;
                    low |= d < 0 && m[h] != 0;
                    m[h] = d < 0 ? 0 : m[h] << d;
                }
                out = low || 15 - Eb + F::EW > W - D;
                e += Eb - F::EW - 15;
                if (plain) {                              // UNIT: every m 1, dw 0
#pragma unroll
                    for (int h = 0; h < 8; ++h) m[h] = 1;
                    out = false;
                    e = W - D;
                }
            } else {
                const int dw = I8 ? (int)sc : (int)(sc & 0xFFu);
                if (!I8) {
#pragma unroll
                    for (int g = 0; g < 4; ++g) m[g] = (int)((sc >> (8 + 6 * g)) & 63u);
                }
                out = dw > W - D;
                e -= dw;
            }
            if (!__any(out || bad)) {
                const double f = pow2d(e);
#pragma unroll
                for (int i = 0; i < MT; ++i) {
                    uint32_t sh[4];
#pragma unroll
                    for (int u = 0; u < 4; ++u) sh[u] = D * 0x01010101u - st.da[i][u];
                    int tt[4] = {0, 0, 0, 0};
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
                        const v4i x = mm(b, i, g, 0);
                        v4i y = {0, 0, 0, 0};
                        if constexpr (NV) y = mm(b, i, g, 1);
#pragma unroll
                        for (int u = 0; u < 4; ++u) {
                            int v;
                            if constexpr (I8) v = x[u];
                            else if constexpr (NV) v = __mul24(x[u], m[2 * g]) + __mul24(y[u], m[2 * g + 1]);
                            else v = __mul24(x[u], m[g]);
                            tt[u] += v << ((sh[u] >> (8 * g)) & 31);
                        }
                    }
#pragma unroll
                    for (int u = 0; u < 4; ++u) acc[s][i][u] = __builtin_fma((double)tt[u], f, acc[s][i][u]);
                }
            } else {
#pragma unroll 1
                for (int h = 0; h < (NV ? 8 : 4); ++h) {
                    const int g = NV ? h >> 1 : h;
                    int mg, dw;
                    if constexpr (NV) {
                        const uint32_t x = ((h < 4 ? sc : sc2) >> (8 * (h & 3))) & 0x7Fu;
                        const int ex = (int)(x >> 3);
                        mg = plain ? 1 : (int)(x & 7) + (ex ? 8 : 0);
                        dw = plain ? 0 : 15 - (ex > 1 ? ex : 1);
                    } else {
                        dw = I8 ? (int)sc : (int)(sc & 0xFFu);
                        mg = I8 ? 1 : (int)((sc >> (8 + 6 * g)) & 63u);
                    }
#pragma unroll
                    for (int i = 0; i < MT; ++i) {
                        v4i x;
                        switch (g) {
                            case 0: x = mm(b, i, 0, h & 1); break;
                            case 1: x = mm(b, i, 1, h & 1); break;
                            case 2: x = mm(b, i, 2, h & 1); break;
                            default: x = mm(b, i, 3, h & 1); break;
                        }
#pragma unroll
                        for (int u = 0; u < 4; ++u) {
                            const int sh = W - dw - (int)((st.da[i][u] >> (8 * g)) & 0xFFu);
                            const double v = __builtin_ldexp((double)(x[u] * mg), sh - F::PRE);
                            acc[s][i][u] += sh >= 0 ? v : 0.0;
                        }
                    }
                }
            }
        }
    };

    // blocks [k, ke) of K into acc, the next block's operands in flight
    auto walk = [&](int k, int ke, double (&acc)[NSUB][MT][4]) {
#pragma unroll
        for (int s = 0; s < NSUB; ++s)
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int u = 0; u < 4; ++u) acc[s][i][u] = 0.0;
        if (k >= ke || m0 >= p.M) return;
        St cur;
        load(cur, k);
        for (; k + 1 < ke; ++k) {
            St nxt;
            load(nxt, k + 1);
            block(cur, acc);
            cur = nxt;
        }
        block(cur, acc);
    };

    // the epilogue's constants of item (s, i, u): row m = m0 + 16 i + 4 c + u, column n = n0 + 16 s + r16
    auto col = [&](int s) { return n0 + 16 * s + r16; };
    auto rowm = [&](int i, int u) { return m0 + 16 * i + 4 * c + u; };
    auto scale_n = [&](int s) {
        return (p.flags & OTPU_UNIT) ? 1.0f
                                     : ftz(*reinterpret_cast<const float*>(p.ws + (int64_t)min(col(s), p.N - 1) * p.srs));
    };
    auto scale_m = [&](int m, int r) { return fmul(p.Sa[(int64_t)r * p.M + min(m, p.M - 1)], pow2f(-W)); };
    // y joins the output's old value as the first MM of a call does (ASCALE, ACC)
    auto first = [&](float y, int m, int n) {
        if (p.flags & OTPU_ASCALE) return fadd(fmul(p.out[(int64_t)m * p.ors + n], p.alpha[m]), y);
        if (p.flags & OTPU_ACC) return fadd(p.out[(int64_t)m * p.ors + n], y);
        return y;
    };
    auto ok = [&](int m, int n) { return m < p.M && n < p.N; };

    double acc[NSUB][MT][4];
    if (p.ranges == 1) {
        walk((int)((int64_t)KB * kwi / kw), (int)((int64_t)KB * (kwi + 1) / kw), acc);
        if (kw == 1) {
#pragma unroll
            for (int s = 0; s < NSUB; ++s) {
                const float sw = scale_n(s);
#pragma unroll
                for (int i = 0; i < MT; ++i)
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        const int m = rowm(i, u), n = col(s);
                        const float y = fmul_f(fmul_f((float)acc[s][i][u], sw), scale_m(m, 0));
                        if (ok(m, n)) p.out[(int64_t)m * p.ors + n] = first(y, m, n);
                    }
            }
            return;
        }
        double* mine = red + wid * ITEMS * 64 + lane;
#pragma unroll
        for (int s = 0; s < NSUB; ++s)
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int u = 0; u < 4; ++u) mine[((s * MT + i) * 4 + u) * 64] = acc[s][i][u];
        __syncthreads();
        for (int it = kwi; it < ITEMS; it += kw) {        // this wave's share of the row tile's outputs
            const double* src = red + (mi * kw * ITEMS + it) * 64 + lane;
            double sum = 0.0;
            for (int j = 0; j < kw; ++j) sum += src[j * ITEMS * 64];
            const int s = it / (4 * MT), m = rowm(it / 4 % MT, it & 3), n = col(s);
            const float y = fmul_f(fmul_f((float)sum, scale_n(s)), scale_m(m, 0));
            if (ok(m, n)) p.out[(int64_t)m * p.ors + n] = first(y, m, n);
        }
        return;
    }
    // ranges: wave kwi takes range kwi of each round of kw; the round's fp32 rows meet in LDS and
    // are added in range order
    float* part = reinterpret_cast<float*>(red);
    float* sums = part + 8 * ITEMS * 64;                  // the fold so far
    const int KR = KB / p.ranges;
    for (int r0 = 0; r0 < p.ranges; r0 += kw) {
        const int r = r0 + kwi, rounds = min(kw, p.ranges - r0);
        walk(r * KR, r < p.ranges ? (r + 1) * KR : 0, acc);
        if (r0) __syncthreads();                          // the last round's rows read
        if (r < p.ranges) {
#pragma unroll
            for (int s = 0; s < NSUB; ++s) {
                const float sw = scale_n(s);
#pragma unroll
                for (int i = 0; i < MT; ++i)
#pragma unroll
                    for (int u = 0; u < 4; ++u)
                        part[(wid * ITEMS + (s * MT + i) * 4 + u) * 64 + lane] =
                            fmul_f(fmul_f((float)acc[s][i][u], sw), scale_m(rowm(i, u), r));
            }
        }
        __syncthreads();
        for (int it = kwi; it < ITEMS; it += kw) {
            const int m = rowm(it / 4 % MT, it & 3), n = col(it / (4 * MT));
            const float* src = part + (mi * kw * ITEMS + it) * 64 + lane;
            float* sum = sums + (mi * ITEMS + it) * 64 + lane;
            float y = src[0];
            if (r0) y = fadd(*sum, y);
            else if (ok(m, n)) y = first(y, m, n);
            for (int j = 1; j < rounds; ++j) y = fadd(y, src[j * ITEMS * 64]);
            if (r0 + kw < p.ranges) *sum = y;
            else if (ok(m, n)) p.out[(int64_t)m * p.ors + n] = y;
        }
    }
}

template <int FMT, int NSUB, int MT>
static void launch(const Args& a, hipStream_t s) {
    batch_kernel<FMT, NSUB, MT><<<(unsigned)(a.tiles_n * a.groups_m), 512, 0, s>>>(a);
}

template <int FMT>
bool launch_fmt(const Args& a, int nsub, int mt, hipStream_t s) {
    if (mt == 1) {
        if (nsub == 1) launch<FMT, 1, 1>(a, s);
        else if (nsub == 2) launch<FMT, 2, 1>(a, s);
        else launch<FMT, 4, 1>(a, s);
        return true;
    }
    if (nsub == 1) {
        launch<FMT, 1, 2>(a, s);
        return true;
    }
    if (nsub == 2) {
        launch<FMT, 2, 2>(a, s);
        return true;
    }
    if constexpr (has_wide_tile(FMT)) launch<FMT, 4, 2>(a, s);
    return has_wide_tile(FMT);
}

}  // namespace bt
}  // namespace otpu
