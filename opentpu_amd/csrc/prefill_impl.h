// MM for many activation rows (prefill) on the int8 MFMA units, every weight format.  Semantics:
// opentpu/isasim.py:749-910 (docs/isa.md:226-305), and the ranges' ACC chain of Builder.dot
// (opentpu/compiler.py:2686-2720).
//
// One v_mfma_i32_32x32x32_i8 is one 32-group of 32 weight rows x 32 activation rows (nvfp4: two of
// K 16, its 16-groups), and its int32 sums are the groups' integer dot products c whatever
// offsets the operands carry.  The terms m c 2^(W - dw - da) are added on the VALU: one walk of K
// serves every activation offset and weight multiplier.  (The same GEMM with the scales folded into
// int8 operand planes multiplies two planes of the weights once for each activation offset present,
// and expands both planes through LDS.)
//
// Exactness.  A wave keeps its sums in int32 with a running unit: acc holds the sum in units of
// 2^(W - ew - sd), ew and sd (wave-uniform) the largest weight and activation offsets met so far;
// a block that brings a larger one shifts the sums once.  Before they could pass 2^31 their upper
// part moves to a second int32 (hi: units 2^16 coarser), so the pair holds any MM's sum (|acc| <
// 2^47).  Offsets together past SMAX take the wave to units of 1 (wide), whose terms are added in 64
// bits.  Sums are exact integers throughout, and the epilogue's double holds them exactly.
//
// Work layout.  4 waves own (32 MS) activation rows x 128 weight rows; each wave 32 weight rows and
// every activation row, so a weight group is unpacked once a wave and used MS times.  K streams in
// blocks of 128 through a ring of LDS stages filled by direct-to-LDS loads (coalesced: the same
// operands loaded straight into the MFMA's layout cost an L1 access a lane, which bound it);
// 2 to 4 workgroups a CU overlap each other's barriers and epilogues.
#pragma once
#include "prefill_args.h"

#include <type_traits>

namespace otpu {
namespace pf {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef unsigned short us2 __attribute__((ext_vector_type(2)));
typedef short s2 __attribute__((ext_vector_type(2)));

// the kernel's lambdas are all inlined: a call would put its sums in memory
#define INL __attribute__((always_inline))

constexpr int TN = 128;                     // weight rows a workgroup

// |sum of one block| <= BB 2^(ew + sd) in the wave's units (4 groups of 32 terms; any int8 activation,
// -128 too, which QACT never gives):
//   int8 32 128 128 4; int4 32 128 8 63 4; fp4 32 128 12 63 4; nvfp4 16 128 12 15 8
template <int FMT>
struct Win {
    static constexpr int W = FMT == OTPU_INT8 ? 16 : (FMT == OTPU_NVFP4 ? 13 : 11);
    static constexpr int64_t BB = FMT == OTPU_INT8 ? 32 * 128 * 128 * 4
                                : FMT == OTPU_INT4 ? 32 * 128 * 8 * 63 * 4
                                : FMT == OTPU_FP4  ? 32 * 128 * 12 * 63 * 4 : 16 * 128 * 12 * 15 * 8;
    static constexpr int SMAX = FMT == OTPU_INT8 ? 9 : (FMT == OTPU_NVFP4 ? 9 : 7);
    static_assert((BB << SMAX) + 65536 < (1ll << 31), "a block's sum fits int32");
    static_assert(SMAX <= W, "no term of the windows is dropped");
    static_assert((63 << SMAX) < (1 << 15), "the multipliers fit 15 bits");
};

// a workgroup's tile: 4 MH waves, wave w owning weight rows 32 (w & 3) .. + 31 and activation rows
// 32 MS (w >> 2) .. + 32 MS - 1
template <int FMT, int MS, int MH>
struct Tile {
    static constexpr bool I8 = FMT == OTPU_INT8, NV = FMT == OTPU_NVFP4;
    static constexpr int WV = 4 * MH;
    static constexpr int TM = 32 * MS * MH;
    static constexpr int AB = TM * 128;                   // activation bytes a stage
    static constexpr int WB = TN * (I8 ? 128 : 64);       // weight bytes
    static constexpr int XD = TM + TN * (NV ? 2 : 1);     // offset and scale words
    static constexpr int XI = (XD + 63) / 64;             // ... as 64-dword loads
    static constexpr int STAGE = AB + WB + XI * 256;
    // direct loads a wave issues a stage
    static constexpr int LA = AB / 1024 / WV, LW = WB / 1024 / WV, LX = (XI + WV - 1) / WV;
    static constexpr int LOADS = LA + LW + LX;
    static constexpr int MW = NV ? 4 : 2;                 // a weight row's multipliers: words of two groups
    // stages in the ring: 4 or 3 where a CU holds two workgroups of 4 waves, or the 8 waves of one
    static constexpr int NST = MS == 1 ? (I8 ? 2 : 3) : (4 * STAGE <= (MH == 1 ? 72 : 110) * 1024 ? 4 : 3);
    static constexpr int SCALE = NST * STAGE;             // the column scales' place behind the ring
    static constexpr int MUL = SCALE + TN * 4;            // ... and the multipliers'
    static constexpr int LDS = MUL + (I8 ? 0 : WV * MW * 128);
};

__device__ __forceinline__ uint32_t lds_addr(const void* p) {
    return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)p;
}
// direct-to-LDS loads: 16 bytes a lane (lane L at M0 + 16 L) from a uniform base and a 32-bit offset
// a lane, and 4 bytes a lane (lane L at M0 + 4 L)
__device__ __forceinline__ void dma16s(const void* base, uint32_t off, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(off), "s"(base), "s"(__builtin_amdgcn_readfirstlane(lds)) : "memory");
}
__device__ __forceinline__ void dma4(const void* g, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off" : : "v"(g), "s"(__builtin_amdgcn_readfirstlane(lds)) : "memory");
}
template <int N>
__device__ __forceinline__ void wait_vm() {
    asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory");
}
// LDS accesses of this wave done, then the workgroup's barrier
__device__ __forceinline__ void bar() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" : : : "memory"); }

// 16-byte chunk c of a 128-byte row r (activations, int8 weights): XOR-swizzled, so that the rows a
// fragment read touches lie on distinct banks; of a 64-byte row (nibbles): by the row's quad
__device__ __forceinline__ int swz8(int r, int c) { return c ^ (((r >> 1) & 7) ^ ((r & 1) << 2)); }
__device__ __forceinline__ int swz4(int r, int c) { return c ^ ((r >> 2) & 3); }

// table entries of the 4-bit codes in the nibbles of x: 8 values in element order (two dwords).
// tp / tn: the values of codes 0..7 and 8..15
__device__ __forceinline__ void lookup8(uint32_t x, const uint32_t (&tp)[2], const uint32_t (&tn)[2], uint32_t& e,
                                        uint32_t& o) {
    const uint32_t y = x >> 4;
    const uint32_t se = x & 0x07070707u, so = y & 0x07070707u;
    const uint32_t pe = ((x >> 1) & 0x04040404u) | 0x03020100u, po = ((y >> 1) & 0x04040404u) | 0x03020100u;
    const uint32_t ve = __builtin_amdgcn_perm(__builtin_amdgcn_perm(tn[1], tn[0], se),
                                              __builtin_amdgcn_perm(tp[1], tp[0], se), pe);
    const uint32_t vo = __builtin_amdgcn_perm(__builtin_amdgcn_perm(tn[1], tn[0], so),
                                              __builtin_amdgcn_perm(tp[1], tp[0], so), po);
    e = __builtin_amdgcn_perm(vo, ve, 0x05010400u);       // elements 0 1 2 3
    o = __builtin_amdgcn_perm(vo, ve, 0x07030602u);       // elements 4 5 6 7
}

// the tile at rows m0, weight rows n0 (lds: Tile::LDS bytes, 16-byte aligned, no load outstanding)
template <int FMT, int MS, int MH, bool RANGED>
__device__ __forceinline__ void prefill_tile(const Args& p, int8_t* ring, int m0, int n0) {
    using F = Win<FMT>;
    using T = Tile<FMT, MS, MH>;
    constexpr bool I8 = T::I8, NV = T::NV;
    constexpr int W = F::W, NST = T::NST, MW = T::MW;
    constexpr bool NEG = FMT == OTPU_INT4 && !RANGED;     // weights and multipliers negated (dots)
    const float* const sSw = reinterpret_cast<const float*>(ring + T::SCALE);

    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wid = wave & 3, mh = wave >> 2;
    const int r32 = lane & 31, h = lane >> 5;
    // a wave's multipliers: MW words a row
    uint32_t (*const sMul)[32] = reinterpret_cast<uint32_t (*)[32]>(ring + T::MUL) + wave * MW;
    const int KB = p.K / OTPU_D;
    const bool plain = (p.flags & (OTPU_UNIT | OTPU_RSC)) != 0;

    // ---- this lane's sources of the direct loads (rows past M or N: the last one) ----
    const int mb = min(m0, p.M - 1), nb = min(n0, p.N - 1);
    const int8_t* const baseA = p.q + (int64_t)mb * p.ldq;
    const uint8_t* const baseW = p.w + (int64_t)nb * p.rs;
    uint32_t offA[T::LA], offW[T::LW];
    const uint8_t* srcX[T::LX];
    int stepX[T::LX];
#pragma unroll
    for (int u = 0; u < T::LA; ++u) {
        const int r = (wave * T::LA + u) * 8 + (lane >> 3);
        offA[u] = (uint32_t)min(r, p.M - 1 - mb) * (uint32_t)p.ldq + 16u * swz8(r, lane & 7);
    }
#pragma unroll
    for (int u = 0; u < T::LW; ++u) {
        const int r = (wave * T::LW + u) * (I8 ? 8 : 16) + (I8 ? lane >> 3 : lane >> 2);
        offW[u] = (uint32_t)min(r, p.N - 1 - nb) * (uint32_t)p.rs + 16u * (I8 ? swz8(r, lane & 7) : swz4(r, lane & 3));
    }
    // the words: TM offset words, then the scale words (int8: the aligned word that holds the block's
    // byte, nvfp4: two a row); waves past the last 64 repeat earlier ones
    auto xidx = [&](int u) INL { return (wave * T::LX + u) % T::XI; };
#pragma unroll
    for (int u = 0; u < T::LX; ++u) {
        const int d = xidx(u) * 64 + lane;
        if (d < T::TM || plain) {
            srcX[u] = p.da + (int64_t)min(m0 + min(d, T::TM - 1), p.M - 1) * p.ldda;
            stepX[u] = 4;
        } else {
            const int e = min(d - T::TM, TN * (NV ? 2 : 1) - 1), r = NV ? e >> 1 : e;
            const uint8_t* row = p.ws + (int64_t)min(n0 + r, p.N - 1) * p.srs;
            srcX[u] = I8 ? row + 4 : row + (NV ? 16 + 8 * p.k0 + 4 * (e & 1) : 8 + 4 * p.k0);
            stepX[u] = I8 ? 0 : (NV ? 8 : 4);
        }
    }
    const uint32_t ring0 = lds_addr(ring);
    auto issue = [&](int kb, int slot) INL {
        const uint32_t base = ring0 + (uint32_t)(slot * T::STAGE);
#pragma unroll
        for (int u = 0; u < T::LA; ++u) dma16s(baseA + kb * 128, offA[u], base + (uint32_t)(wave * T::LA + u) * 1024u);
#pragma unroll
        for (int u = 0; u < T::LW; ++u)
            dma16s(baseW + kb * (I8 ? 128 : 64), offW[u], base + (uint32_t)(T::AB + (wave * T::LW + u) * 1024));
#pragma unroll
        for (int u = 0; u < T::LX; ++u) {
            // (int8's scale words: four blocks' bytes a word)
            const int o = I8 && stepX[u] == 0 ? (p.k0 + kb) & ~3 : kb * stepX[u];
            dma4(srcX[u] + o, base + (uint32_t)(T::AB + T::WB + xidx(u) * 256));
        }
    };
    // the epilogue's column scales (waves 0 and 1, 64 rows each), then the first stages
    if (wave < 2 && !(p.flags & OTPU_UNIT))
        dma4(p.ws + (int64_t)min(n0 + 64 * wave + lane, p.N - 1) * p.srs, ring0 + T::SCALE + 256u * wave);
    for (int s = 0; s < NST - 1 && s < KB; ++s) issue(s, s);

    v16i acc[MS], hi[MS];
    int ew = 0, sd = 0;                                   // the unit: 2^(W - ew - sd)
    bool wide = false;                                    // the unit: 1
    uint32_t bound = 0;                                   // of |acc|
    bool low = true;                                      // every hi 0
    auto clear = [&]() INL {
#pragma unroll
        for (int i = 0; i < MS; ++i)
#pragma unroll
            for (int t = 0; t < 16; ++t) acc[i][t] = hi[i][t] = 0;
        bound = 0;
        low = true;
        if (wide) ew = sd = 0;                            // (ranges: the next one starts at this one's unit)
        wide = false;
    };
    clear();
    auto split = [&]() INL {                              // the sums' upper parts to hi
#pragma unroll
        for (int i = 0; i < MS; ++i)
#pragma unroll
            for (int t = 0; t < 16; ++t) {
                hi[i][t] += acc[i][t] >> 16;
                acc[i][t] &= 0xFFFF;
            }
        bound = 65536;
        low = false;
    };
    auto finer = [&](int up) INL {                        // to a unit 2^up finer (up <= 16)
        if (((uint64_t)bound << up) >= (1ull << 31)) {
            split();
#pragma unroll
            for (int i = 0; i < MS; ++i)
#pragma unroll
                for (int t = 0; t < 16; ++t) {
                    const uint64_t v = (uint64_t)(uint32_t)acc[i][t] << up;
                    hi[i][t] = (int)(((uint32_t)hi[i][t] << (up & 31)) + (uint32_t)(v >> 16));
                    acc[i][t] = (int)(v & 0xFFFFu);
                }
        } else {
#pragma unroll
            for (int i = 0; i < MS; ++i) {
                acc[i] <<= up;
                hi[i] <<= up;
            }
            bound <<= up;
        }
    };
    float y[RANGED ? MS : 1][16];                         // ranges: the fold so far

    const int KR = RANGED ? KB / p.ranges : KB;
    // output t of row tile i: row mrow(i), column ncol(t)
    auto mrow = [&](int i) INL { return m0 + 32 * (MS * mh + i) + r32; };
    auto ncol = [&](int t) INL { return n0 + 32 * wid + 8 * (t >> 2) + 4 * h + (t & 3); };
    // the sum's fp32 value times the scales: a sum of one int32 is rounded to fp32 as it is (then a power
    // of two >= 1), one with an upper part goes through a double
    auto value = [&](int i, int t, float sa, auto one) INL {
        float v;
        if constexpr (decltype(one)::value)
            v = (float)acc[i][t] * bitsf((uint32_t)(127 + W - ew - sd) << 23);
        else
            v = (float)(((double)hi[i][t] * 65536.0 + (double)acc[i][t]) *
                        __hiloint2double((1023 + (wide ? 0 : W - ew - sd)) << 20, 0));
        const float sw = (p.flags & OTPU_UNIT) ? 1.0f : ftz(sSw[32 * wid + 8 * (t >> 2) + 4 * h + (t & 3)]);
        return fmul_f(fmul_f(v, sw), sa);
    };
    auto scale_m = [&](int i, int r) INL { return fmul(p.Sa[(int64_t)r * p.M + min(mrow(i), p.M - 1)], pow2f(-W)); };
    auto first = [&](float v, int m, int n) INL {             // joins the old output as a call's first MM does
        const float* o = p.out + (int64_t)m * p.ors + n;
        if (p.flags & OTPU_ASCALE) return fadd(fmul(*o, p.alpha[m]), v);
        if (p.flags & OTPU_ACC) return fadd(*o, v);
        return v;
    };

    uint32_t tp[2], tn8[2];
    if (NEG) {
        tp[0] = 0xFDFEFF00u; tp[1] = 0xF9FAFBFCu; tn8[0] = 0x05060708u; tn8[1] = 0x01020304u;
    } else if (FMT == OTPU_INT4) {
        tp[0] = 0x03020100u; tp[1] = 0x07060504u; tn8[0] = 0xFBFAF9F8u; tn8[1] = 0xFFFEFDFCu;
    } else {                                              // twice the E2M1 values
        tp[0] = 0x03020100u; tp[1] = 0x0C080604u; tn8[0] = 0xFDFEFF00u; tn8[1] = 0xF4F8FAFCu;
    }

    // wait until stage s has landed, `late` later ones in flight
    auto landed = [&](int late) INL {
        if (NST > 3 && late >= 2) wait_vm<2 * T::LOADS>();
        else if (late == 1) wait_vm<T::LOADS>();
        else wait_vm<0>();
    };
    const int8_t* cur = ring;                             // block kb's stage
    const int r0 = 32 * wid + r32;                        // this lane's weight row in a stage
    auto words = [&](const int8_t* st) INL { return reinterpret_cast<const uint32_t*>(st + T::AB + T::WB); };
    // a group's weights in the MFMA's layout (row r0, elements 16 h .. 16 h + 15)
    auto weights = [&](const int8_t* st, int g) INL {
        const int8_t* B = st + T::AB;
        if constexpr (I8) {
            return *reinterpret_cast<const v4i*>(B + r0 * 128 + 16 * swz8(r0, 2 * g + h));
        } else {
            const uint2 x = *reinterpret_cast<const uint2*>(B + r0 * 64 + 16 * swz4(r0, g) + 8 * h);
            uint32_t v[4];
            lookup8(x.x, tp, tn8, v[0], v[1]);
            lookup8(x.y, tp, tn8, v[2], v[3]);
            return v4i{(int)v[0], (int)v[1], (int)v[2], (int)v[3]};
        }
    };
    auto acts = [&](const int8_t* st, int i, int g) INL {
        const int r = 32 * (MS * mh + i) + r32;
        return *reinterpret_cast<const v4i*>(st + r * 128 + 16 * swz8(r, 2 * g + h));
    };
    const v16i zero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};

    // ---- a block's words: its rows' offsets and multipliers ----
    uint32_t da[MS], own = 0;                    // own: this lane's weight row's scale word
    uint32_t dw = 0;                                      // ... and its largest weight offset
    int xsh = 0;                                          // int8: the block's byte of the word
    auto read_words = [&](const int8_t* st, int kb, uint32_t (&d)[MS]) INL {
        const uint32_t* X = words(st);
#pragma unroll
        for (int i = 0; i < MS; ++i) d[i] = X[32 * (MS * mh + i) + r32];
        own = plain ? 0u : X[T::TM + (NV ? 2 * r0 + h : r0)];     // (nvfp4: half h of its 8 scales)
        xsh = 8 * ((p.k0 + kb) & 3);
        dw = 0;
        if constexpr (I8) {
            dw = (own >> xsh) & 0xFFu;
        } else if constexpr (NV) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint32_t v = (own >> (8 * e)) & 0x7Fu;  // (a zero scale adds nothing, whatever its offset)
                dw = max(dw, v ? (uint32_t)(15 - max((int)(v >> 3), 1)) : 0u);
            }
        } else {
            dw = own & 0xFFu;
        }
    };
    // the row's multipliers m 2^(ew - dw), 16 bits a group, for the wave's lanes to read (its own LDS)
    auto write_mults = [&]() INL {
        if constexpr (NV) {
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                uint32_t word = 0;
#pragma unroll
                for (int f = 0; f < 2; ++f) {
                    const uint32_t v = (own >> (16 * e + 8 * f)) & 0x7Fu, E = v >> 3;
                    const uint32_t m = (v & 7u) | (E ? 8u : 0u);
                    word |= (m << (((uint32_t)ew - 15u + max(E, 1u)) & 31u)) << (16 * f);
                }
                sMul[2 * h + e][r32] = plain ? 0x00010001u << ew : word;
            }
        } else if constexpr (!I8) {
            const uint32_t six = plain ? 0x01041041u : own >> 8;
            const uint32_t two = h ? six >> 12 : six;     // half h of the wave: groups 2 h, 2 h + 1
            const uint32_t m2 = ((two & 63u) | ((two & (63u << 6)) << 10)) << (((uint32_t)ew - dw) & 31u);
            sMul[h][r32] = NEG ? __builtin_bit_cast(uint32_t, (us2)0 - __builtin_bit_cast(us2, m2)) : m2;
        }
    };
    // the unit made fine enough for a block of offsets d, its sums' bound counted
    auto admit = [&](const uint32_t (&d)[MS]) INL {
        if (!wide) {
            // an activation offset byte above sd (sd <= SMAX < 128: the byte sum's top bit, or its own)
            uint32_t over = 0;
#pragma unroll
            for (int i = 0; i < MS; ++i) over |= (d[i] + (uint32_t)(127 - sd) * 0x01010101u) | d[i];
            if (__any((over & 0x80808080u) || dw > (uint32_t)ew)) {
                uint32_t top = 0;
#pragma unroll
                for (int i = 0; i < MS; ++i)
                    top = max(top, max(max(d[i] & 0xFFu, (d[i] >> 8) & 0xFFu), max((d[i] >> 16) & 0xFFu, d[i] >> 24)));
                const int nsd = max(sd, (int)__builtin_amdgcn_readfirstlane(wave_max_dpp(top, 64)));
                const int new_ = max(ew, (int)__builtin_amdgcn_readfirstlane(wave_max_dpp(dw, 64)));
                if (nsd + new_ > F::SMAX) {
                    finer(W - ew - sd);
                    wide = true;
                    low = false;
                } else {
                    finer(nsd + new_ - ew - sd);
                    sd = nsd;
                    ew = new_;
                }
            }
        }
        const uint32_t add = wide ? (NV ? 8 : 4) * 65536 : (uint32_t)F::BB << (ew + sd);
        if (bound + add >= (1u << 31)) split();
        bound += add;
    };

    // ---- a block's sums: the products of pair (group g, row tile i) are issued, and the operands of
    // the pair after it read, while the sums of the pair before are added (an MFMA's result is 64
    // clocks away, an LDS read's ~130; sched_barrier: the compiler puts each MFMA next to its first
    // use otherwise).  Running the pipeline on across blocks measured slower (int8 184 -> 198 us at
    // 2000 x 2048 x 12288): the two waves a SIMD holds are bound by their own issue. ----
    constexpr int NP = 4 * MS;                            // pairs a block
    uint32_t mw[I8 ? 1 : 16];
    auto mults = [&](int k) INL {                         // the 16 rows' words k: groups 2 k, 2 k + 1 (nvfp4: 16-groups)
        if constexpr (!I8) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint4 x = *reinterpret_cast<const uint4*>(&sMul[k][8 * q + 4 * h]);
                mw[4 * q] = x.x; mw[4 * q + 1] = x.y; mw[4 * q + 2] = x.z; mw[4 * q + 3] = x.w;
            }
        }
    };
    auto pairs = [&]() INL {
        v16i c[2];
        v4i w = weights(cur, 0), a = acts(cur, 0, 0);
        mults(0);
        auto product = [&](int j) INL { c[j & 1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(w, a, zero, 0, 0, 0); };
        product(0);
        a = acts(cur, 1 % MS, 1 / MS);
        if (MS == 1) w = weights(cur, 1);
#pragma unroll
        for (int j = 0; j < NP; ++j) {
            const int g = j / MS, i = j % MS;
            __builtin_amdgcn_sched_barrier(0);
            if (j + 1 < NP) product(j + 1);
            if (j + 2 < NP) {
                a = acts(cur, (j + 2) % MS, (j + 2) / MS);
                if ((j + 2) % MS == 0) w = weights(cur, (j + 2) / MS);
            }
            __builtin_amdgcn_sched_barrier(0);
            const uint32_t sh = ((uint32_t)(I8 ? sd + ew : sd) - (da[i] >> (8 * g))) & 31u;
#pragma unroll
            for (int t = 0; t < 16; ++t) {
                int v;
                if constexpr (I8) v = c[j & 1][t];
                else v = __mul24(c[j & 1][t], (int)(g & 1 ? mw[t] >> 16 : mw[t] & 0xFFFFu));
                acc[i][t] += v << sh;
            }
            if (j + 1 < NP && (j + 1) % (NP / MW) == 0) mults((j + 1) / (NP / MW));
        }
    };
    // int4 and nvfp4: their group products fit 16 bits with any int8 activations (nvfp4: 16 128 12; int4:
    // -32 127 8 .. 32 128 8, the negated weights' -32768 .. 32512), so the terms of two groups are one
    // v_dot2: pack the products, shift the two multipliers by the activation's offsets, multiply-add
    // both.  The products of unit j + 1 run behind the sums of unit j, in the registers its packing
    // freed: 16 fewer than two sets (nvfp4's ranges at 64 rows a tile spill 5 registers, not 104).
    // Measured (us, QACT in; a multiply and a shift-add a group -> this): int4 1999 x 2048 x 12288 239 ->
    // 233; nvfp4 (its 16-groups as K 16 products, no masked lanes) 337 -> 328, 1999 x 6144 x 2048 in
    // ranges of 768 280 -> 222.  int4's ranges keep the other form (64 rows a tile: 169 against 175).
    auto dots = [&]() INL {
        constexpr int NU = MW * MS;                       // units (multiplier word k, row tile i)
        // operands: int4 two groups', nvfp4 one group's two 16-groups (8 elements a lane, K 16 products)
        using Op = std::conditional_t<NV, long, v4i>;
        Op w[2], a[2];
        auto fetch = [&](int j) INL {
            const int k = j / MS, r = 32 * (MS * mh + j % MS) + r32;
            if constexpr (NV) {
                if (j % MS == 0) {
                    const uint32_t* B = reinterpret_cast<const uint32_t*>(cur + T::AB + r0 * 64 + 16 * swz4(r0, k)) + h;
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        uint32_t lo, up;
                        lookup8(B[2 * e], tp, tn8, lo, up);
                        w[e] = (long)((uint64_t)up << 32 | lo);
                    }
                }
#pragma unroll
                for (int e = 0; e < 2; ++e) a[e] = *reinterpret_cast<const long*>(cur + r * 128 + 16 * swz8(r, 2 * k + e) + 8 * h);
            } else {
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    if (j % MS == 0) w[e] = weights(cur, 2 * k + e);
                    a[e] = acts(cur, j % MS, 2 * k + e);
                }
            }
        };
        v16i c0, c1;
        auto product = [&]() INL {
            if constexpr (NV) {
                c0 = __builtin_amdgcn_mfma_i32_32x32x16_i8(w[0], a[0], zero, 0, 0, 0);
                c1 = __builtin_amdgcn_mfma_i32_32x32x16_i8(w[1], a[1], zero, 0, 0, 0);
            } else {
                c0 = __builtin_amdgcn_mfma_i32_32x32x32_i8(w[0], a[0], zero, 0, 0, 0);
                c1 = __builtin_amdgcn_mfma_i32_32x32x32_i8(w[1], a[1], zero, 0, 0, 0);
            }
        };
        fetch(0);
        mults(0);
        product();
        fetch(1);
#pragma unroll
        for (int j = 0; j < NU; ++j) {
            const int k = j / MS, i = j % MS;
            uint32_t c[16];                               // the low halves of both products
#pragma unroll
            for (int t = 0; t < 16; ++t) c[t] = __builtin_amdgcn_perm((uint32_t)c1[t], (uint32_t)c0[t], 0x05040100u);
            __builtin_amdgcn_sched_barrier(0);
            if (j + 1 < NU) product();
            if (j + 2 < NU) fetch(j + 2);
            __builtin_amdgcn_sched_barrier(0);
            const uint32_t d0 = (da[i] >> (NV ? 8 * k : 16 * k)) & 0xFFu, d1 = NV ? d0 : (da[i] >> (16 * k + 8)) & 0xFFu;
            const us2 sh = {(unsigned short)((uint32_t)sd - d0), (unsigned short)((uint32_t)sd - d1)};
#pragma unroll
            for (int t = 0; t < 16; ++t) {
                const us2 m = __builtin_bit_cast(us2, mw[t]) << sh;
                acc[i][t] = __builtin_amdgcn_sdot2(__builtin_bit_cast(s2, c[t]), __builtin_bit_cast(s2, m), acc[i][t], false);
            }
            if (j + 1 < NU && (j + 1) % MS == 0) mults((j + 1) / MS);
        }
    };

    int slot = 0;                                         // block kb's
    for (int kb = 0; kb < KB; ++kb) {
        landed(min(NST - 2, KB - 1 - kb));                // block kb
        bar();                                            // ... everywhere; and block kb - 1 read
        if (kb + NST - 1 < KB) issue(kb + NST - 1, slot ? slot - 1 : NST - 1);
        cur = ring + slot * T::STAGE;
        slot = slot + 1 < NST ? slot + 1 : 0;
        read_words(cur, kb, da);
        admit(da);
        write_mults();

        const bool shifted = I8 && __any(dw != 0);        // (uniform)
        if (!wide && !shifted && !(I8 && sd + ew == 0)) {
            if constexpr (NV || NEG) dots();
            else pairs();
        } else {
            const uint32_t* X = words(cur);
            if (I8 && !wide && !shifted) {                // no offset so far: the MFMA's own sums
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const v4i wg = weights(cur, g);
#pragma unroll
                    for (int i = 0; i < MS; ++i)
                        acc[i] = __builtin_amdgcn_mfma_i32_32x32x32_i8(wg, acts(cur, i, g), acc[i], 0, 0, 0);
                }
            } else if (I8 && !wide) {
                uint32_t dws[16];
#pragma unroll
                for (int t = 0; t < 16; ++t)
                    dws[t] = (X[T::TM + 32 * wid + 8 * (t >> 2) + 4 * h + (t & 3)] >> xsh) & 0xFFu;
#pragma unroll 1
                for (int g = 0; g < 4; ++g) {
                    const v4i wg = weights(cur, g);
#pragma unroll
                    for (int i = 0; i < MS; ++i) {
                        const v16i x = __builtin_amdgcn_mfma_i32_32x32x32_i8(wg, acts(cur, i, g), zero, 0, 0, 0);
                        const uint32_t sh = (uint32_t)(sd + ew) - ((da[i] >> (8 * g)) & 0xFFu);
#pragma unroll
                        for (int t = 0; t < 16; ++t) acc[i][t] += x[t] << ((sh - dws[t]) & 31);
                    }
                }
            } else {
                // units of 1: each term m c 2^(W - dw - da) in 64 bits (dropped where the shift is negative)
#pragma unroll 1
                for (int g = 0; g < 4; ++g) {
                    const v4i wg = weights(cur, g);
#pragma unroll 1
                    for (int e = 0; e < (NV ? 2 : 1); ++e) {
                        const v4i we = NV ? (wg & (h == e ? -1 : 0)) : wg;
#pragma unroll
                        for (int i = 0; i < MS; ++i) {
                            const v16i x = __builtin_amdgcn_mfma_i32_32x32x32_i8(we, acts(cur, i, g), zero, 0, 0, 0);
                            const int d = (int)((da[i] >> (8 * g)) & 0xFFu);
#pragma unroll
                            for (int t = 0; t < 16; ++t) {
                                const int r = 32 * wid + 8 * (t >> 2) + 4 * h + (t & 3);
                                int m = 1, wd = 0;
                                if (!plain) {
                                    const uint32_t word = X[T::TM + (NV ? 2 * r + (g >> 1) : r)];
                                    if constexpr (I8) {
                                        wd = (int)((word >> xsh) & 0xFFu);
                                    } else if constexpr (NV) {
                                        const uint32_t v = (word >> (16 * (g & 1) + 8 * e)) & 0x7Fu;
                                        const int E = (int)(v >> 3);
                                        m = (int)(v & 7u) + (E ? 8 : 0);
                                        wd = 15 - (E > 1 ? E : 1);
                                    } else {
                                        m = (int)((word >> (8 + 6 * g)) & 63u);
                                        wd = (int)(word & 0xFFu);
                                    }
                                }
                                if (NEG) m = -m;
                                const int s = W - wd - d;
                                const int64_t v = s >= 0 ? (int64_t)(x[t] * m) << (s & 31) : 0;
                                acc[i][t] += (int)(v & 0xFFFF);
                                hi[i][t] += (int)(v >> 16);
                            }
                        }
                    }
                }
            }
        }

        if constexpr (RANGED) {
            if ((kb + 1) % KR == 0) {
                const int r = kb / KR;
                auto fold = [&](auto one) INL {
#pragma unroll
                    for (int i = 0; i < MS; ++i) {
                        const float sa = scale_m(i, r);
#pragma unroll
                        for (int t = 0; t < 16; ++t) {
                            const float v = value(i, t, sa, one);
                            if (r) y[i][t] = fadd(y[i][t], v);
                            else y[i][t] = mrow(i) < p.M && ncol(t) < p.N ? first(v, mrow(i), ncol(t)) : v;
                        }
                    }
                };
                if (low) fold(std::true_type());
                else fold(std::false_type());
                clear();
            }
        }
    }
    // ---- the outputs: 4 adjacent columns a store ----
    auto outputs = [&](auto one) INL {
#pragma unroll
        for (int i = 0; i < MS; ++i) {
            const int m = mrow(i);
            if (m >= p.M) continue;
            const float sa = RANGED ? 0.0f : scale_m(i, 0);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int n = ncol(4 * q);
                float* o = p.out + (int64_t)m * p.ors + n;
                float v[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    if constexpr (RANGED) v[u] = y[i][4 * q + u];
                    else v[u] = value(i, 4 * q + u, sa, one);
                }
                if (p.vec4 && n + 3 < p.N) {
                    if (!RANGED)
#pragma unroll
                        for (int u = 0; u < 4; ++u) v[u] = first(v[u], m, n + u);
                    *reinterpret_cast<float4*>(o) = make_float4(v[0], v[1], v[2], v[3]);
                } else {
#pragma unroll
                    for (int u = 0; u < 4; ++u)
                        if (n + u < p.N) o[u] = RANGED ? v[u] : first(v[u], m, n + u);
                }
            }
        }
    };
    if (RANGED || low) outputs(std::true_type());
    else outputs(std::false_type());
}

template <int FMT, int MS, bool RANGED>
__global__ __launch_bounds__(256, 2) void prefill_kernel(Args p) {
    using T = Tile<FMT, MS, 1>;
    __shared__ __align__(16) int8_t lds[T::LDS];
    // each XCD takes a run of tiles (workgroup b runs on XCD b % 8), the tiles in panels of 4 weight
    // tiles: the 64 it holds at once are 16 row tiles x 4, whose operands its L2 keeps
    const int b = blockIdx.x, total = p.tiles_m * p.tiles_n, x = b & 7, per = total >> 3, more = total & 7;
    const int t = x * per + min(x, more) + (b >> 3);
    const int panel = t / (4 * p.tiles_m), rest = t - panel * 4 * p.tiles_m, wide_n = min(4, p.tiles_n - 4 * panel);
    const int tm = rest / wide_n, tn = 4 * panel + rest - tm * wide_n;
    prefill_tile<FMT, MS, 1, RANGED>(p, lds, tm * T::TM, tn * TN);
}

template <int FMT>
bool launch_fmt(const Args& a, int ms, hipStream_t s) {
    const unsigned grid = (unsigned)(a.tiles_m * a.tiles_n);
    if (a.ranges == 1) {
        if (ms == 1) prefill_kernel<FMT, 1, false><<<grid, 256, 0, s>>>(a);
        else prefill_kernel<FMT, 2, false><<<grid, 256, 0, s>>>(a);
        return true;
    }
    if (ms == 1) {
        prefill_kernel<FMT, 1, true><<<grid, 256, 0, s>>>(a);
        return true;
    }
    if constexpr (has_tall_tile(FMT, true)) prefill_kernel<FMT, 2, true><<<grid, 256, 0, s>>>(a);
    return has_tall_tile(FMT, true);
}

#undef INL

}  // namespace pf
}  // namespace otpu
