// MM for many activation rows on the int8 MFMA units (prefill GEMM) with plain int8 weights (RSC or
// UNIT: no offsets of their own).  Semantics: opentpu/isasim.py:749-910 (docs/isa.md:226-305).
//
// Exactness.  MM's integer is acc = sum over 32-groups of 2^(16 - da) * c (dropped where the shift is
// negative).  A tile whose groups all carry one offset d is a plain int8 GEMM.  With two offsets the
// sum splits into two planes of masked activations, C_0 and C_1, each an int32 matrix product:
//     acc = 2^(16 - smax) * sum_p 2^(smax - d_p) * C_p,
// within int32 where K * 128^2 * 2^(smax - dmin) stays below 2^31 (checked per tile).  A tile of
// more offsets takes prefill_impl.h's walk, which adds each group's products with its own shift (the
// masked operand planes it had taken one K walk each: c3's shape with activations of three offsets
// 67 us).
//
// Work layout.  A workgroup owns a 128 x 128 output tile and streams K in 128-byte stages through a
// ring in LDS (16-byte chunks XOR-swizzled by row so the ds_read_b128 of a 16-row fragment hits
// distinct banks); each of its 4 multiplying waves computes 64 x 64 with 4 x 4
// v_mfma_i32_16x16x64_i8.  Tiles are assigned XCD-major: the workgroups of one XCD share weight
// rows, so each weight panel is fetched from HBM once into that XCD's L2.
#include "prefill_impl.h"

namespace otpu {

typedef int v4i __attribute__((ext_vector_type(4)));

constexpr int GBM = 128, GBN = 128, GBK = 128;

struct GemmArgs {
    const int8_t* q; int64_t ldq;
    const float* Sa;
    const uint8_t* da; int64_t ldda;
    int M, K;
    const int8_t* w; int64_t rs;
    const uint8_t* ws; int64_t srs;
    int N, flags, k0;
    const float* alpha;
    float* out; int64_t ors;
    int tiles_m, tiles_n;
    int vec4;                   // out 16-byte aligned and ors a multiple of 4: float4 stores
};

// byte offset of 16-byte chunk c of tile row r (rows of 128 bytes, chunks XOR-swizzled)
// The 16-byte slot of chunk c in row r is c ^ f(r), f(r) = ((r >> 1) & 7) ^ ((r & 1) << 2): the
// 8 rows a ds_read_b128 fragment's lanes 0-7 (and 8-15) read land in 8 distinct slots of a 128-byte
// bank window, and its 16 rows in 16 distinct (row parity, slot) pairs of a 256-byte one.
__device__ __forceinline__ int rowswz(int r) { return ((r >> 1) & 7) ^ ((r & 1) << 2); }
__device__ __forceinline__ int swz(int r, int c) { return r * GBK + ((c ^ rowswz(r)) << 4); }

// ---- the single-plane pipeline: a ring of NS K-stages in LDS, filled by direct-to-LDS loads ----
// A stage is the A and B tiles of 128 rows x RBK bytes; NS - 1 stages are in flight while one
// is multiplied.  global_load_lds_dwordx4 writes a wave's 64 x 16 bytes to 1 KB of LDS at M0
// (lane L at M0 + 16 L), so lane L of a wave's instruction fetches the global chunk that belongs
// at LDS slot L of its 1 KB block: with CPR = RBK / 16 chunks a row, row r = block * (64 / CPR)
// + L / CPR, stored slot L % CPR, i.e. the row's chunk (L % CPR) ^ rswz(r) (the XOR swizzle
// that puts the 16 rows a ds_read_b128 fragment reads on distinct banks).
// The loads are issued from inline assembly and their completion awaited with explicit
// s_waitcnt vmcnt(n): the compiler's own accounting would wait for every stage in flight.
#ifndef OTPU_RING_BK
#define OTPU_RING_BK 128
#endif
#ifndef OTPU_RING_NS
#define OTPU_RING_NS 4
#endif
constexpr int RBK = OTPU_RING_BK;               // K bytes a stage
constexpr int NS = OTPU_RING_NS;                // stages in the ring
constexpr int CPR = RBK / 16;                   // 16-byte chunks a row
constexpr int TILE = GBM * RBK;                 // bytes of one operand tile of a stage
constexpr int STAGE = 2 * TILE;                 // A then B
constexpr int LPS = 2 * TILE / 1024 / 4;        // direct loads a wave issues per stage
constexpr int RING = NS * STAGE > 2 * 2 * GBM * GBK ? NS * STAGE : 2 * 2 * GBM * GBK;
static_assert(RBK == 64 || RBK == 128, "ring stages of 64 or 128 bytes");
static_assert(NS >= 2 && (NS - 2) * LPS <= 63, "vmcnt holds at most 63");

__device__ __forceinline__ int rswz(int r) { return RBK == 128 ? rowswz(r) : (r >> 2) & 3; }
__device__ __forceinline__ int rof(int r, int c) { return r * RBK + ((c ^ rswz(r)) << 4); }

__device__ __forceinline__ uint32_t lds_addr(const void* p) {
    return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)p;
}

__device__ __forceinline__ void dma16(const int8_t* g, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(g), "s"(lds) : "memory");
}

// wait until at most n of this wave's direct loads are outstanding
template <int N>
__device__ __forceinline__ void wait_dma() {
    asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory");
}

// wait for stage kt when `ahead` later stages have been issued (ahead <= NS - 2)
__device__ __forceinline__ void wait_stage(int ahead) {
    switch (ahead) {
#define OTPU_WAIT_CASE(x) case x: if constexpr (x <= NS - 2) wait_dma<x * LPS>(); break;
        OTPU_WAIT_CASE(7) OTPU_WAIT_CASE(6) OTPU_WAIT_CASE(5) OTPU_WAIT_CASE(4)
        OTPU_WAIT_CASE(3) OTPU_WAIT_CASE(2) OTPU_WAIT_CASE(1)
#undef OTPU_WAIT_CASE
        default: wait_dma<0>();
    }
}

// LDS reads of the workgroup done, then the barrier (no fence: the direct loads are awaited
// by each wave before it arrives)
__device__ __forceinline__ void ring_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" : : : "memory");
}

// this lane's source rows of the ring's direct loads: instruction u of a stage reads row
// ga[u] (A, u < LPS / 2) or gb[u] (B); rows past M or N read the last valid row
struct RingSrc {
    const int8_t* ga[LPS / 2];
    const int8_t* gb[LPS / 2];
    uint32_t base;                              // the wave's LDS byte address in stage 0
};

__device__ __forceinline__ RingSrc ring_src(const GemmArgs& a, const int8_t* ring, int m0, int n0) {
    // (wave w mod 4: the loader waves 4-7 of gemm_lw_kernel issue what waves 0-3 would)
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((threadIdx.x >> 6) & 3);
    RingSrc rs;
#pragma unroll
    for (int u = 0; u < LPS / 2; ++u) {
        const int blk = w * (LPS / 2) + u;
        const int r = blk * (64 / CPR) + lane / CPR, c = (lane % CPR) ^ rswz(r);
        rs.ga[u] = a.q + (int64_t)min(m0 + r, a.M - 1) * a.ldq + 16 * c;
        rs.gb[u] = a.w + (int64_t)min(n0 + r, a.N - 1) * a.rs + 16 * c;
    }
    rs.base = lds_addr(ring) + (uint32_t)(w * (LPS / 2) * 1024);
    return rs;
}

// walk step kt into its ring slot; dk: the K stage it holds (kt, or kt rotated: see lw_rot)
__device__ __forceinline__ void ring_issue(const RingSrc& rs, int kt, int dk) {
    const uint32_t sl = rs.base + (uint32_t)((kt % NS) * STAGE);
    const int o = dk * RBK;
#pragma unroll
    for (int u = 0; u < LPS / 2; ++u) dma16(rs.ga[u] + o, sl + 1024u * u);
#pragma unroll
    for (int u = 0; u < LPS / 2; ++u) dma16(rs.gb[u] + o, sl + TILE + 1024u * u);
}

// two activation planes share one K walk: their offset words are staged in LDS by the offset scan
// (row r's word of stage kt at r * DAS + kt, four offsets a word)
constexpr int MP_MAX = 2;                       // planes one walk carries (64 registers of sums each)
constexpr int MP_KT = 32;                       // stages (K = 4096) the staged offsets cover
constexpr int DAS = MP_KT + 1;                  // their row stride in words (16 rows on 16 banks)

// The epilogue of a tile whose MM integers are acc << sh (acc the int32 sums, sh = 16 - smax >= 0):
// y = (i2f(acc << sh) * Sw[n]) * (Sa[m] * 2^-16), then ACC / ASCALE.  i2f(acc << sh) is the int32's
// RNE float times 2^sh exactly.  sa2: the tile's rows' Sa * 2^-16 in LDS (row r of the tile at r).
// A full tile leaves through LDS: each wave writes its 64 x 64 accumulators in the MFMA layout
// (rows 68 words apart: the 4 row groups of a write land on distinct banks) and reads them back
// as 4-column rows, so every store instruction writes 4 rows x 256 contiguous bytes.  The scaling
// runs after the transpose, in a loop over the 16 row groups a lane stores: the tile runs once per
// CU from a cold instruction cache, so the epilogue's code length is its latency (unrolled over
// all 64 values it was 128 rounded products of straight-line code).  `lds` is the ring's memory
// (every wave is past its last read of the ring when the epilogue starts).
constexpr int TPS = 68;                         // transpose row stride, words

// a wave's 64 x 64 accumulators into its transpose region T (rows TPS words apart)
__device__ __forceinline__ void epi_transpose(int* T, const v4i (&acc)[4][4]) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int t = 0; t < 4; ++t) T[(16 * i + 4 * (lane >> 4) + t) * TPS + 16 * j + (lane & 15)] = acc[i][j][t];
}

// this lane's 4 columns' Sw in region w's epilogue rows (1 with UNIT), as loaded: epi_rows
// flushes them where it uses them, so that no wait for these loads comes before that
__device__ __forceinline__ void epi_sw(const GemmArgs& a, int n0, int w, float (&sw)[4]) {
    const bool unit = (a.flags & OTPU_UNIT) != 0;
    const int nc = n0 + (w & 1) * 64 + 4 * (threadIdx.x & 15);
#pragma unroll
    for (int c = 0; c < 4; ++c) sw[c] = unit ? 1.0f : *reinterpret_cast<const float*>(a.ws + (int64_t)(nc + c) * a.srs);
}

// row groups s0 .. s1 - 1 of region w's 16 (region w: the 64 x 64 of wave w) from T, scaled by
// sw (epi_sw) and Sa and stored as 4-row x 256-byte float4 rows
__device__ __forceinline__ void epi_rows(const GemmArgs& a, const int* T, const float* sa2, int m0, int n0, int w,
                                         int s0, int s1, int sh, const float (&sw)[4]) {
    const int lane = threadIdx.x & 63;
    const int q = lane & 15, g = lane >> 4;
    const int rt = (w >> 1) * 64 + g;                          // the tile row of group s = 0
    const int nc = n0 + (w & 1) * 64 + 4 * q;
    const float swf[4] = {ftz(sw[0]), ftz(sw[1]), ftz(sw[2]), ftz(sw[3])};
    const bool asc = (a.flags & OTPU_ASCALE) != 0, accf = (a.flags & OTPU_ACC) != 0;
#pragma unroll 2
    for (int s = s0; s < s1; ++s) {
        const int r = rt + 4 * s;
        const int4 raw = *reinterpret_cast<const int4*>(T + (g + 4 * s) * TPS + 4 * q);
        const float sa = sa2[r];
        float y[4] = {ldexpf((float)raw.x, sh), ldexpf((float)raw.y, sh), ldexpf((float)raw.z, sh),
                      ldexpf((float)raw.w, sh)};
#pragma unroll
        for (int c = 0; c < 4; ++c) y[c] = fmul_f(fmul_f(y[c], swf[c]), sa);
        float* p = a.out + (int64_t)(m0 + r) * a.ors + nc;
        if (asc || accf) {
            const float4 old = *reinterpret_cast<const float4*>(p);
            const float o[4] = {old.x, old.y, old.z, old.w};
            const float al = asc ? a.alpha[m0 + r] : 1.0f;
#pragma unroll
            for (int c = 0; c < 4; ++c) y[c] = asc ? fadd(fmul(o[c], al), y[c]) : fadd(o[c], y[c]);
        }
#ifndef OTPU_GEMM_NT_STORE
#define OTPU_GEMM_NT_STORE 1
#endif
#if OTPU_GEMM_NT_STORE
        typedef float f32x4 __attribute__((ext_vector_type(4)));
        __builtin_nontemporal_store(f32x4{y[0], y[1], y[2], y[3]}, reinterpret_cast<f32x4*>(p));
#else
        *reinterpret_cast<float4*>(p) = make_float4(y[0], y[1], y[2], y[3]);
#endif
    }
}

__device__ __forceinline__ void tile_epilogue(const GemmArgs& a, int8_t* lds, const float* sa2, int m0, int n0,
                                              const v4i (&acc)[4][4], int sh) {
    const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const bool unit = (a.flags & OTPU_UNIT) != 0;
    const bool full = m0 + GBM <= a.M && n0 + GBN <= a.N;
    if (full && a.vec4) {
        int* T = reinterpret_cast<int*>(lds) + wid * 64 * TPS;
        float sw[4];
        epi_sw(a, n0, wid, sw);
        epi_transpose(T, acc);
        epi_rows(a, T, sa2, m0, n0, wid, 0, 16, sh, sw);
        return;
    }
    // a partial tile (or an unaligned output): each lane's own values, in the MFMA layout
    const int mb = m0 + (wid >> 1) * 64 + 4 * (lane >> 4), nb = n0 + (wid & 1) * 64 + (lane & 15);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int n = nb + j * 16;
        const float sw = (unit || n >= a.N) ? 1.0f : ftz(*reinterpret_cast<const float*>(a.ws + (int64_t)n * a.srs));
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const int m = mb + i * 16 + t;
                if (m >= a.M || n >= a.N) continue;
                float y = fmul_f(fmul_f(ldexpf((float)acc[i][j][t], sh), sw), sa2[m - m0]);
                float* o = a.out + (int64_t)m * a.ors + n;
                if (a.flags & OTPU_ASCALE) y = fadd(fmul(*o, a.alpha[m]), y);
                else if (a.flags & OTPU_ACC) y = fadd(*o, y);
                *o = y;
            }
    }
}

// The activation offsets d present in a tile (bit 17: offsets past the window) into sMask[w] for each
// wave w of threads 0-255, and the offset words into sDaAll (K <= 4096).  Packed offset rows (ldda = K / 32
// bytes, 16-byte aligned, the tile's rows all present) are one contiguous block, read with
// coalesced 16-byte loads: each line once.  Otherwise two threads a row read its words (each
// load instruction then touches 64 rows' lines, and the tile's 64 lines are requested ~32 times
// over: at the c3 shape that took the scan to 2.9 us, its requests queued among the ring's).
__device__ __forceinline__ void tile_offsets(const GemmArgs& a, int m0, int KT, uint32_t* sDaAll, uint32_t* sMask) {
    const int tid = threadIdx.x & 255, lane = tid & 63, wid = tid >> 6;
    uint32_t dm = 0;
    auto take = [&](uint32_t wd) {
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const uint32_t d = (wd >> (8 * t)) & 0xFF;
            dm |= 1u << (d <= 16 ? d : 17);
        }
    };
    const uint8_t* blk = a.da + (int64_t)m0 * a.ldda;
    const bool packed = a.ldda == 4 * KT && (KT & 3) == 0 && ((uintptr_t)blk & 15) == 0 && m0 + GBM <= a.M;
    if (packed) {
        const uint4* v = reinterpret_cast<const uint4*>(blk);
        const int NV = GBM * KT / 4;                     // 16-byte pieces of the tile's block
        for (int i = tid; i < NV; i += 256) {
            const uint4 q = v[i];
            const int r = 4 * i / KT, k = 4 * i % KT;     // row r, words k .. k + 3
            if (KT <= MP_KT) {
                sDaAll[r * DAS + k] = q.x;
                sDaAll[r * DAS + k + 1] = q.y;
                sDaAll[r * DAS + k + 2] = q.z;
                sDaAll[r * DAS + k + 3] = q.w;
            }
            take(q.x);
            take(q.y);
            take(q.z);
            take(q.w);
        }
    } else {
        const int r = tid & (GBM - 1), h = tid >> 7;
        if (m0 + r < a.M) {
            const uint32_t* drow = reinterpret_cast<const uint32_t*>(a.da + (int64_t)(m0 + r) * a.ldda);
#pragma unroll 8
            for (int k = h; k < KT; k += 2) {             // K / 128 words of four offsets
                const uint32_t wd = drow[k];
                if (KT <= MP_KT) sDaAll[r * DAS + k] = wd;
                take(wd);
            }
        }
    }
    for (int o = 32; o > 0; o >>= 1) dm |= __shfl_xor(dm, o, 64);
    if (lane == 0) sMask[wid] = dm;
}

// ---- loader waves: workgroups of 8 waves, 4 of them streaming the ring, 4 multiplying ----
// With one wave a SIMD doing both, a direct load that finds the load path full stalls the
// wave's issue and the MFMAs behind it wait: a stage's loads and MFMAs add up instead of
// overlapping.  Here waves 4-7 issue every direct load (the first NS - 1 stages before the
// tile's offset scan) and waves 0-3 only read fragments and multiply; the two groups meet at
// one barrier a stage.  A loader arrives once its part of stage kt has landed and then refills
// the slot stage kt - 1 left; a compute wave arrives with its reads of stage kt - 1 done.
// (c3 ROW x RSC: 18.5-18.7 -> 16.3-16.6 us back to back, bit-identical.)

// The K walk of a tile starts at stage rot and wraps (the int32 sums are exact in any order).
// The workgroups of one XCD run in step, so with one common order the tiles that share an A or
// a B panel ask for each line together and all wait a miss's latency for it (L2 merges the
// requests).  Staggered starts let one tile miss a line and the others hit it in L2 stages
// later: the 8 tiles of an XCD that share A rows start 2 stages apart, the 4 that share B rows
// 4 stages apart (tn & 7 and tm: the XCD-major order gives an XCD 8 consecutive column tiles).
__device__ __forceinline__ int lw_rot(int tm, int tn, int KS) { return (2 * (tn & 7) + 4 * tm) % KS; }
__device__ __forceinline__ int lw_stage(int kt, int rot, int KS) { return kt + rot < KS ? kt + rot : kt + rot - KS; }

// a loader wave's walk (its first NS - 1 stages issued): KS + 1 barriers
__device__ __forceinline__ void lw_load_walk(const RingSrc& rs, int KS, int rot) {
    for (int kt = 0; kt < KS; ++kt) {
        wait_stage(min(NS - 2, KS - 1 - kt));
        ring_barrier();                                  // stage kt landed (this wave's part)
        const int nk = kt + NS - 1;
        if (nk < KS) ring_issue(rs, nk, lw_stage(nk, rot, KS));
    }
    ring_barrier();
}

// a compute wave's walk: NP planes into acc[p]; MASK: each stage's A fragments masked to plane
// p's 32-groups (plain weights, offsets from da_lds), else the single plane.
// ALL1 (two planes covering every group): plane 1's product taken over every group instead,
// C_all, so that only plane 0 is masked (C_1 = C_all - C_0 afterwards, exactly in int32).
// KS + 1 barriers, matching lw_load_walk's.
template <int NP, bool MASK, bool ALL1 = false>
__device__ __forceinline__ void lw_mma_walk(const int8_t* ring, const uint32_t* da_lds, v4i (&acc)[NP][4][4],
                                            const int (&dv)[MP_MAX], int KS, int rot) {
    const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wid >> 1, wn = wid & 1;
    for (int kt = 0; kt < KS; ++kt) {
        ring_barrier();                                  // stage kt landed everywhere
        const int8_t* A = ring + (kt % NS) * STAGE;
        const int8_t* B = A + TILE;
        uint32_t dw4[4] = {0u, 0u, 0u, 0u};
        if constexpr (MASK) {
            const int dk = lw_stage(kt, rot, KS);
#pragma unroll
            for (int i = 0; i < 4; ++i) dw4[i] = da_lds[(wm * 64 + i * 16 + (lane & 15)) * DAS + dk];
        }
        v4i fa[2][4], fb[2][4];
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            const int c = ks * 4 + (lane >> 4);
#pragma unroll
            for (int i = 0; i < 4; ++i) fa[ks][i] = *reinterpret_cast<const v4i*>(A + rof(wm * 64 + i * 16 + (lane & 15), c));
#pragma unroll
            for (int j = 0; j < 4; ++j) fb[ks][j] = *reinterpret_cast<const v4i*>(B + rof(wn * 64 + j * 16 + (lane & 15), c));
        }
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            const int gsh = 8 * ((ks * 4 + (lane >> 4)) >> 1);   // the chunk's 32-group offset byte
#pragma unroll
            for (int p = 0; p < NP; ++p) {
                v4i fm[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const bool keep = !MASK || (ALL1 && p == 1) || ((dw4[i] >> gsh) & 0xFFu) == (uint32_t)dv[p];
                    fm[i] = keep ? fa[ks][i] : v4i{0, 0, 0, 0};
                }
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        acc[p][i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fm[i], fb[ks][j], acc[p][i][j], 0, 0, 0);
            }
        }
    }
    ring_barrier();                                      // every read of the ring done
}

// the barrier of a walk whose LDS reads the compiler tracks: its own wait for every LDS read
// (so no later wait on those reads is inserted), the barrier, and a fence that keeps the next
// stage's reads below it
__device__ __forceinline__ void ring_barrier_tracked() {
    __builtin_amdgcn_s_waitcnt(0xC07F);                  // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" : : : "memory");
}

// NP planes (as lw_mma_walk's; the kernels use it for one) with the fragment reads half a stage
// ahead (for two planes it measured no faster, its accumulators spilling a few registers).  A stage's
// fragments are two halves (K chunks 0-3 and 4-7 of its 128 bytes, 8 ds_read_b128 each);
// between barriers kt + 1 and kt + 2 a wave reads half 0 of stage kt + 1, multiplies half 1 of
// stage kt, reads half 1 of stage kt + 1 and multiplies its half 0, one read issued per 2 NP
// MFMAs, so the reads run under the MFMAs (read, then multiplied, a one-plane stage took ~1000
// cycles, twice the MFMAs' 512).  Barrier j still follows every read of stage j - 1, so the
// loaders refill its slot as lw_load_walk does.  KS + 1 barriers.
struct Half {
    v4i a[4], b[4];
};

template <bool MASK>
__device__ __forceinline__ void lw_half_read(const int8_t* ring, const uint32_t* da_lds, Half& h, uint32_t (&dw)[4],
                                             int kt, int ks, int KS, int rot) {
    const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wid >> 1, wn = wid & 1;
    const int8_t* A = ring + (kt % NS) * STAGE;
    const int8_t* B = A + TILE;
    if (MASK && ks == 0) {
        const int dk = lw_stage(kt, rot, KS);
#pragma unroll
        for (int i = 0; i < 4; ++i) dw[i] = da_lds[(wm * 64 + i * 16 + (lane & 15)) * DAS + dk];
    }
    const int c = ks * 4 + (lane >> 4);
#pragma unroll
    for (int i = 0; i < 4; ++i) h.a[i] = *reinterpret_cast<const v4i*>(A + rof(wm * 64 + i * 16 + (lane & 15), c));
#pragma unroll
    for (int j = 0; j < 4; ++j) h.b[j] = *reinterpret_cast<const v4i*>(B + rof(wn * 64 + j * 16 + (lane & 15), c));
}

template <int NP, bool MASK, bool ALL1>
__device__ __forceinline__ void lw_half_mma(const Half& h, const uint32_t (&dw)[4], v4i (&acc)[NP][4][4], int ks,
                                            const int (&dv)[MP_MAX]) {
    const int lane = threadIdx.x & 63;
    const int gsh = 8 * ((ks * 4 + (lane >> 4)) >> 1);
#pragma unroll
    for (int p = 0; p < NP; ++p) {
        v4i fm[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const bool keep = !MASK || (ALL1 && p == 1) || ((dw[i] >> gsh) & 0xFFu) == (uint32_t)dv[p];
            fm[i] = keep ? h.a[i] : v4i{0, 0, 0, 0};
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                acc[p][i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fm[i], h.b[j], acc[p][i][j], 0, 0, 0);
    }
}

// (the scheduler would move the register-only MFMAs across the barriers and sink each read next
// to its use: sched_barrier closes every region, and the group barriers interleave each half's
// reads with the MFMAs that hide them)
#define OTPU_READS_UNDER_MMA(nr, np)                                                                \
    do {                                                                                           \
        if ((nr) > 8) __builtin_amdgcn_sched_group_barrier(0x100, (nr) - 8, 0);                    \
        _Pragma("unroll") for (int g_ = 0; g_ < 8; ++g_) {                                         \
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);                                     \
            __builtin_amdgcn_sched_group_barrier(0x008, 2 * (np), 0);                              \
        }                                                                                          \
    } while (0)

template <int NP, bool MASK, bool ALL1 = false>
__device__ __forceinline__ void lw_mma_walk_h(const int8_t* ring, const uint32_t* da_lds, v4i (&acc)[NP][4][4],
                                              const int (&dv)[MP_MAX], int KS, int rot) {
    Half h0, h1;
    uint32_t dw[4] = {0u, 0u, 0u, 0u}, dwn[4] = {0u, 0u, 0u, 0u};
    ring_barrier_tracked();                              // stage 0 landed everywhere
    __builtin_amdgcn_sched_barrier(0);
    lw_half_read<MASK>(ring, da_lds, h0, dw, 0, 0, KS, rot);
    lw_half_read<MASK>(ring, da_lds, h1, dw, 0, 1, KS, rot);
    lw_half_mma<NP, MASK, ALL1>(h0, dw, acc, 0, dv);
    OTPU_READS_UNDER_MMA(MASK ? 20 : 16, NP);
    __builtin_amdgcn_sched_barrier(0);
    for (int kt = 0; kt + 1 < KS; ++kt) {
        ring_barrier_tracked();                          // stage kt + 1 landed, stage kt read
        __builtin_amdgcn_sched_barrier(0);
        lw_half_read<MASK>(ring, da_lds, h0, dwn, kt + 1, 0, KS, rot);
        lw_half_mma<NP, MASK, ALL1>(h1, dw, acc, 1, dv);
        OTPU_READS_UNDER_MMA(MASK ? 12 : 8, NP);
        lw_half_read<MASK>(ring, da_lds, h1, dwn, kt + 1, 1, KS, rot);
        lw_half_mma<NP, MASK, ALL1>(h0, dwn, acc, 0, dv);
        OTPU_READS_UNDER_MMA(8, NP);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 4; ++i) dw[i] = dwn[i];
    }
    ring_barrier_tracked();                              // the walk's end
    __builtin_amdgcn_sched_barrier(0);
    lw_half_mma<NP, MASK, ALL1>(h1, dw, acc, 1, dv);
}
#undef OTPU_READS_UNDER_MMA

// The GEMM with loader waves (workgroups of 8 waves).  DENSE: whole tiles of dense rows (RSC words, float4 stores),
// whose strides follow from the sizes: a tile runs once a round from a cold instruction cache, so the shorter
// code is its latency (512 x 2048 x 8192 ROW 14.5 -> 14.05 us).  Waves 0-3 scan the
// tile's offsets, multiply and store; waves 4-7 issue the ring's direct loads (and store half of a
// full tile).  Tiles of one or two activation offsets walk the ring with both groups; any other
// tile waits for the loaders' stages to land and takes the walk of any offsets (prefill_impl.h) on
// all 8 waves.
template <bool DENSE>
__global__ __launch_bounds__(512) void gemm_lw_kernel(GemmArgs a) {
    if constexpr (DENSE) {
        a.ldq = a.rs = a.K; a.ldda = a.K / 32; a.srs = 4; a.ors = a.N; a.vec4 = 1;
    }
    __shared__ __align__(16) int8_t sRing[RING];
    __shared__ uint32_t sMask[4];
    __shared__ uint32_t sDaAll[GBM * DAS];
    __shared__ float sSa2[GBM];

    const int tid = threadIdx.x, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const bool loader = wid >= 4;
    int b = blockIdx.x, tm, tn;
    const int ntiles = a.tiles_m * a.tiles_n;
    if (ntiles % 8 == 0 && a.tiles_n % 8 == 0) {
        const int per = ntiles / 8, x = b % 8, li = b / 8;
        const int t = x * per + li;
        tn = t / a.tiles_m;
        tm = t % a.tiles_m;
    } else {
        tn = b / a.tiles_m;
        tm = b % a.tiles_m;
    }
    const int m0 = tm * GBM, n0 = tn * GBN;
    const int KT = a.K / GBK, KS = a.K / RBK;
    const int rot = lw_rot(tm, tn, KS);

    const RingSrc rs = ring_src(a, sRing, m0, n0);
    // the epilogue's column scales, loaded early (a full tile's epilogue rows are shared by
    // wave w and loader w + 4, region w & 3): a loader's before its ring loads, which complete
    // in order after them (the stage waits' counts unchanged), a compute wave's after the
    // offset scan (whose waits would otherwise wait for them too)
    const bool split = DENSE || (m0 + GBM <= a.M && n0 + GBN <= a.N && a.vec4);
    float esw[4] = {1.0f, 1.0f, 1.0f, 1.0f};
    if (loader) {
        if (split) epi_sw(a, n0, wid & 3, esw);
#pragma unroll
        for (int s = 0; s < NS - 1; ++s)
            if (s < KS) ring_issue(rs, s, lw_stage(s, rot, KS));
    } else {
        if (tid < GBM) sSa2[tid] = m0 + tid < a.M ? fmul(a.Sa[m0 + tid], pow2f(-16)) : 0.0f;
        tile_offsets(a, m0, KT, sDaAll, sMask);       // the offsets present in this tile
        if (split) epi_sw(a, n0, wid, esw);
    }
    __syncthreads();
    const uint32_t dall = sMask[0] | sMask[1] | sMask[2] | sMask[3];
    const uint32_t dmask = dall & 0x1FFFFu;
    const bool over = (dall >> 17) & 1;
    const int np = __builtin_popcount(dmask);
    const int dmin = dmask ? __builtin_ctz(dmask) : 0, smax = dmask ? 31 - __builtin_clz(dmask) : 0;
    // the planes' sum in int32: |acc| <= K 128^2 2^(smax - dmin)
    const bool fits = (int64_t)a.K * 16384 <= (((int64_t)1 << 31) - 1) >> (smax - dmin);
    const bool single = np == 1 && !over;

    // a full tile's epilogue is shared: waves 0-3 write their transposes, then wave w and its
    // loader w + 4 store 8 row groups each (one more barrier for both groups)
    if (single || (KT <= MP_KT && (np == 1 || (np == 2 && fits)))) {
        if (loader) {
            lw_load_walk(rs, KS, rot);
            if (split) {
                __syncthreads();                         // the transposes written
                const int w = wid & 3;
                epi_rows(a, reinterpret_cast<const int*>(sRing) + w * 64 * TPS, sSa2, m0, n0, w, 8, 16, 16 - smax, esw);
            }
            return;
        }
        auto epilogue = [&](const v4i (&acc0)[4][4]) {
            if (split) {
                int* T = reinterpret_cast<int*>(sRing) + wid * 64 * TPS;
                epi_transpose(T, acc0);
                __syncthreads();
                epi_rows(a, T, sSa2, m0, n0, wid, 0, 8, 16 - smax, esw);
            } else {
                tile_epilogue(a, sRing, sSa2, m0, n0, acc0, 16 - smax);
            }
        };
        int dv[MP_MAX];
        uint32_t left = dmask;
#pragma unroll
        for (int p = 0; p < MP_MAX; ++p) {               // the planes' d in ascending order
            dv[p] = left ? __builtin_ctz(left) : 255;
            left &= left - 1;
        }
        if (single || np == 1) {                         // (one plane of plain weights: no masking
            v4i acc[1][4][4];                            // when its offset covers every group)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[0][i][j] = v4i{0, 0, 0, 0};
            if (single) lw_mma_walk_h<1, false>(sRing, sDaAll, acc, dv, KS, rot);
            else lw_mma_walk_h<1, true>(sRing, sDaAll, acc, dv, KS, rot);
            epilogue(acc[0]);
        } else {
            v4i acc[2][4][4];
#pragma unroll
            for (int p = 0; p < 2; ++p)
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int j = 0; j < 4; ++j) acc[p][i][j] = v4i{0, 0, 0, 0};
            // (no offsets past the window: the two planes cover every group, so plane 1 is C_all)
            if (!over) lw_mma_walk<2, true, true>(sRing, sDaAll, acc, dv, KS, rot);
            else lw_mma_walk<2, true>(sRing, sDaAll, acc, dv, KS, rot);
            // sum_p C_p << (smax - d_p) (the bound checked above)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const v4i c1 = over ? acc[1][i][j] : acc[1][i][j] - acc[0][i][j];
                    acc[0][i][j] = (acc[0][i][j] << (smax - dv[0])) + (c1 << (smax - dv[1]));
                }
            epilogue(acc[0]);
        }
        return;
    }
    // every other tile: the loaders' stages land, then the walk of any offsets on all 8 waves
    if (loader) wait_dma<0>();
    ring_barrier();
    pf::Args pa = {};
    pa.q = a.q; pa.ldq = a.ldq; pa.Sa = a.Sa; pa.da = a.da; pa.ldda = a.ldda; pa.M = a.M; pa.K = a.K;
    pa.w = reinterpret_cast<const uint8_t*>(a.w); pa.rs = a.rs; pa.ws = a.ws; pa.srs = a.srs; pa.N = a.N;
    pa.flags = a.flags; pa.alpha = a.alpha; pa.out = a.out; pa.ors = a.ors; pa.ranges = 1; pa.vec4 = a.vec4;
    static_assert(pf::Tile<OTPU_INT8, 2, 2>::LDS <= RING && pf::Tile<OTPU_INT8, 2, 2>::TM == GBM, "the walk's tile");
    pf::prefill_tile<OTPU_INT8, 2, 2, false>(pa, sRing, m0, n0);
}

}  // namespace otpu

using namespace otpu;

// returns 1 when the call is not for this kernel (otpu_mm then streams it), else a status
int otpu_gemm_try(const int8_t* q, int64_t ldq, const float* Sa, const uint8_t* da, int64_t ldda, int M, int K,
                  const uint8_t* w, int64_t rs, const uint8_t* ws, int64_t srs, int N, int fmt, int flags, int k0,
                  const float* alpha, float* out, int64_t ors, hipStream_t s) {
    if (fmt != OTPU_INT8 || !(flags & (OTPU_UNIT | OTPU_RSC)) || (flags & OTPU_RMAX)) return 1;
    if (((uintptr_t)da & 3) || (ldda % 4) || ((uintptr_t)q & 15) || (ldq % 16) || ((uintptr_t)w & 15) || (rs % 16))
        return 1;
    GemmArgs a = {};
    a.q = q; a.ldq = ldq; a.Sa = Sa; a.da = da; a.ldda = ldda; a.M = M; a.K = K;
    a.w = reinterpret_cast<const int8_t*>(w); a.rs = rs; a.ws = ws; a.srs = srs; a.N = N;
    a.flags = flags; a.k0 = k0; a.alpha = alpha; a.out = out; a.ors = ors;
    a.tiles_m = (M + GBM - 1) / GBM;
    a.tiles_n = (N + GBN - 1) / GBN;
    a.vec4 = ((uintptr_t)out % 16 == 0) && (ors % 4 == 0);
    const bool dense = M % GBM == 0 && N % GBN == 0 && ldq == K && rs == K && ldda == K / 32 && srs == 4 && ors == N && a.vec4;
    if (dense) gemm_lw_kernel<true><<<a.tiles_m * a.tiles_n, 512, 0, s>>>(a);
    else gemm_lw_kernel<false><<<a.tiles_m * a.tiles_n, 512, 0, s>>>(a);
    return otpu_launch_check("mm gemm");
}
