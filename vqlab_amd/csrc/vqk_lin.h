// Matrix-core VQ linear for a few rows of x: y[n, o] = sum_i x[n, i] * W[o, i],
// the decode step of a dense linear (_dense_fused, vq_switch.py:3339-3434) for
// 2..64 rows, and for one row where the block-per-lane GEMV (vqk_gemv.h) has
// no fast form (more than 64 blocks per weight row, or a ragged last block).
//
// What bounds it: the LDS lookups of the decode (one table read per code) and,
// with many rows, the x operand, so each weight is decoded ONCE for up to 64
// rows of x -- the GEMV decodes it once per row -- and goes straight into the
// A operand of v_mfma_f32_16x16x32 (lane l: weight row l % 16, 8 consecutive
// columns of lane group l / 16, each group holding one 32-code block of the
// row), W = fp16(cb * s), the bit-exact dequant.
//
// A workgroup is 8 waves = RG groups of 16 weight rows x KS slices of the
// K loop (KS * RG = 8): the waves of one row group take its supersteps (4
// blocks per row) in turn and add their partial sums through LDS, in slice
// order (no workspace, no second launch, the same bits every call). Splitting
// K inside the workgroup is what keeps all 8 waves of a CU loading weights
// when OUT / 16 alone would fill few CUs. x goes from L2 straight into the B
// operand's registers (token l % 16), in place for a few rows or from a copy
// in operand order; staged through LDS instead, with a barrier per chunk, 16
// rows ran 83 us against 56 in place (5120 -> 17408, d4 K4096): every chunk
// then waits for a load.
//
// The B operand's type (XM): fp16, x rounded as the fused kernels round it; or
// fp32 (VQK_X_KEEP, d8) through v_mfma_f32_16x16x4_f32, whose lane (row or
// token l % 16, column l / 16) takes one of the same 8 values at a time: bf16
// and fp32 x enter unrounded and so does the weight, f32(cb) * f32(s), at a
// sixteenth of the fp16 rate.
//
// Measured (MI355X, us per call, this kernel with the copy / before; bf16 x):
//   5120 -> 17408, d4 K4096:  8 rows 31 / 107, 20 rows 36 / 250, 64 rows 52 / 72
//   17408 -> 5120, d4 K4096:  1 row 25 / 1720, 20 rows 36 / 3639 (generic GEMV)
//   5120 -> 17408, d8 K65536: 8 rows 87 / 424, 20 rows 160 / 940 (fp32 products)
#pragma once

#include <type_traits>

#include "vqk_gseg.h"

namespace vqk {

// x as the B operand: fp16 as it is; bf16 / fp32 rounded to fp16; bf16 / fp32
// widened to fp32
// kXFrag: fp16 in operand order (k_lin_frag)
enum : int { kXF16 = 0, kXBF16r = 1, kXF32r = 2, kXBF16x = 3, kXF32x = 4, kXFrag = 5 };

struct LinParams {
    const uint32_t *codes;
    int64_t row_words;         // words per code row
    const uint16_t *codebook;  // fp16 [K, D], 16-byte aligned
    int32_t K;
    const uint16_t *scales;    // fp16, ngrp per code row, one per 64 columns
    int32_t ngrp;
    const int32_t *row_table;  // [OUT] or NULL
    int64_t stored_rows;       // > 0
    int32_t OUT, IN, NB;       // NB = ceil(IN / (32 D)); IN % 64 == 0
    const void *x;             // [N, IN], 16-byte aligned
    int32_t x_type;
    void *y;
    int32_t y_type;
    int32_t N;
    int32_t ks_log2;           // K slices per workgroup = 1 << ks_log2 (<= 8)
};

// Table entries in LDS: all of a table up to 128 KB; 128 KB of a larger one,
// except that of a d8 table of 65536 entries (1 MB) none are: an eighth of the
// lookups would not pay for the copy and the occupancy.
__host__ __device__ constexpr int lin_table_entries(int D, int BITS) {
    return (int64_t(1) << BITS) * D * 2 <= 128 * 1024 ? (1 << BITS)
           : (D == 8 && BITS == 16)                   ? 0
                                                      : 128 * 1024 / (2 * D);
}
constexpr int kLinWaves = 8;
__host__ __device__ constexpr size_t lin_lds(int D, int BITS, int NT) {
    const size_t tab = size_t(lin_table_entries(D, BITS) + 1) * D * 2;
    const size_t red = size_t(kLinWaves) * NT * 1024;  // the slices' sums, after the table
    return tab > red ? tab : red;
}

// Two workgroups to a CU where the registers (128 a lane) and LDS allow.
__host__ __device__ constexpr int lin_waves_per_simd(int D, int BITS, int NT) {
    return NT <= 2 && lin_lds(D, BITS, NT) <= 80 * 1024 ? 4 : 2;
}

// The raw bytes of 8 activations of one row.
template <int XM> struct LinRaw { u32x4 v; };
template <> struct LinRaw<kXF32r> { u32x4 v, w; };
template <> struct LinRaw<kXF32x> { u32x4 v, w; };

// An address past the buffer's end loads zeros: kLinNoRow is one for every
// buffer of at most 2 GB (checked on the host).
constexpr uint32_t kLinNoRow = 0x80000000u;

template <int XM>
__device__ __forceinline__ LinRaw<XM> lin_load_x(__amdgpu_buffer_rsrc_t x, uint32_t off, int base, int st) {
    LinRaw<XM> r;
    if constexpr (XM == kXF32r || XM == kXF32x) {
        r.v = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(x, off + 32 * st, base, 0));
        r.w = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(x, off + 32 * st + 16, base, 0));
    } else {
        r.v = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(x, off + 16 * st, base, 0));
    }
    return r;
}

template <int XM>
__device__ __forceinline__ void lin_floats(const LinRaw<XM> &r, float (&f)[8]) {
    if constexpr (XM == kXF32r || XM == kXF32x) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            f[i] = __uint_as_float(r.v[i]);
            f[4 + i] = __uint_as_float(r.w[i]);
        }
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            f[2 * i] = __uint_as_float(r.v[i] << 16);
            f[2 * i + 1] = __uint_as_float(r.v[i] & 0xffff0000u);
        }
    }
}

template <int XM>
__device__ __forceinline__ h8 lin_f16(const LinRaw<XM> &r) {
    if constexpr (XM == kXF16 || XM == kXFrag) {
        return __builtin_bit_cast(h8, r.v);
    } else {
        float f[8];
        lin_floats<XM>(r, f);
        h8 h;
#pragma unroll
        for (int i = 0; i < 8; ++i) h[i] = f16(f[i]);
        return h;
    }
}

template <int D, int BITS, int GPB, int NT, int XM>
__global__ void __launch_bounds__(kLinWaves * 64, lin_waves_per_simd(D, BITS, NT)) k_lin(const LinParams p) {
    constexpr int SPB = 4 * D;                  // MFMA steps per block (8 weights each)
    constexpr int CPB = 32 * D;                 // columns per block
    constexpr int CBN = lin_table_entries(D, BITS);
    constexpr bool CBL = CBN == (1 << BITS);
    constexpr bool WIDE = XM == kXBF16x || XM == kXF32x;
    // steps of x loads in flight: enough to cover an L2 latency within the
    // registers that two workgroups per CU leave
    constexpr bool F32 = XM == kXF32r || XM == kXF32x;
    constexpr int PF = F32 || WIDE || NT == 2 ? 4 : (NT == 4 ? 2 : 8);
    constexpr int GS = 2;                       // steps per scheduling group
    static_assert(SPB % PF == 0 && SPB % (2 * GS) == 0, "whole rings and group pairs per superstep");

    extern __shared__ __align__(16) uint8_t smem[];
    f16 *cbl = reinterpret_cast<f16 *>(smem);   // [CBN + 1][D]; entry CBN is zero

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));   // uniform loop bounds
    const int ln = lane & 15, lg = lane >> 4;
    const int KS = 1 << p.ks_log2, RG = kLinWaves >> p.ks_log2;
    const int rg = wave & (RG - 1), ks = wave >> (3 - p.ks_log2);
    const int o0 = (int(blockIdx.x) * RG + rg) * 16;
    const int t0 = int(blockIdx.y) * 16 * NT;

    lds_copy_async(p.codebook, cbl, min(p.K, CBN) * D * 2, (CBN + 1) * D * 2);

    // stored row of this lane's weight row (a dead or absent row reads row 0
    // and is written as +0 or not at all)
    int64_t cr = -1;
    if (o0 + ln < p.OUT) {
        cr = p.row_table ? int64_t(p.row_table[o0 + ln]) : int64_t(o0 + ln);
        if (cr >= p.stored_rows) cr = -1;
    }
    const bool dead = cr < 0;
    if (dead) cr = 0;
    constexpr int XB = XM == kXF32r || XM == kXF32x ? 4 : 2;
    constexpr bool FRAG = XM == kXFrag;
    // kXFrag: this token tile's operands, NT KB per MFMA step
    const int frag_b = FRAG ? ((p.NB + 3) >> 2) * SPB * NT * 1024 : 0;
    const uint8_t *xp = static_cast<const uint8_t *>(p.x) + int64_t(blockIdx.y) * frag_b;
    const __amdgpu_buffer_rsrc_t xbuf = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t *>(xp), 0, FRAG ? frag_b : int(uint32_t(p.N) * uint32_t(p.IN) * XB), 0x00027000);
    // byte offset of this lane's row and lane group (columns past N repeat its
    // last row, never stored)
    uint32_t xrow = FRAG ? uint32_t(lane) * 16
                         : (uint32_t(min(t0 + ln, p.N - 1)) * uint32_t(p.IN) + uint32_t(lg * CPB)) * XB;

    const int NSS = (p.NB + 3) >> 2;
    const uint32_t kmax = uint32_t(p.K - 1);
    const uint32_t kl = uint32_t(min(p.K, CBN));
    const f16 *tg = reinterpret_cast<const f16 *>(p.codebook);

    // MFMA steps of block 4 * sb + lg inside the row (SPB, fewer for a ragged
    // last block, 0 past the row's end)
    auto valid_steps = [&](int sb) { return max(0, min(SPB, (p.IN - (4 * sb + lg) * CPB) >> 3)); };
    const bool ragged = p.NB % 4 != 0 || p.IN % CPB != 0;       // the last superstep is not whole
    auto load_w = [&](int sb, uint32_t (&w)[BITS], uint16_t (&s)[GPB]) {
        const int b = min(4 * sb + lg, p.NB - 1);
        const uint32_t *src = p.codes + cr * p.row_words;
        const uint16_t *sr = p.scales + cr * p.ngrp;
        if (!ragged || sb != NSS - 1) {
#pragma unroll
            for (int i = 0; i < BITS; ++i) w[i] = src[b * BITS + i];
#pragma unroll
            for (int g = 0; g < GPB; ++g) s[g] = sr[b * GPB + g];
        } else {                                // nothing past the row's end (steps there use none of it)
#pragma unroll
            for (int i = 0; i < BITS; ++i) w[i] = src[min(b * BITS + i, int(p.row_words) - 1)];
#pragma unroll
            for (int g = 0; g < GPB; ++g) {
                const uint16_t v = sr[min(b * GPB + g, p.ngrp - 1)];
                s[g] = b * GPB + g < p.ngrp ? v : uint16_t(0);
            }
        }
    };

    f32x4 acc[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[nt] = f32x4{0.f, 0.f, 0.f, 0.f};

    LinRaw<XM> xr[PF][NT];
    auto load_x = [&](int sb, int st, LinRaw<XM> (&dst)[NT]) {
        asm volatile("" : "+v"(xrow));          // issued here, not hoisted
        if constexpr (FRAG) {
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
                dst[nt].v = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                    xbuf, xrow + 1024 * nt, (sb * SPB + st) * (NT * 1024), 0));
        } else {
            static_assert(FRAG || NT == 1, "direct loads are one row tile");
            dst[0] = lin_load_x<XM>(xbuf, 4 * sb + lg < p.NB ? xrow : kLinNoRow, sb * 4 * CPB * XB, st);
        }
    };
    // entry `c` of the table; the zero entry when !ok
    auto entry = [&](uint32_t c, bool ok) {
        typedef typename EntryT<D>::type E;
        if constexpr (CBL) {
            return reinterpret_cast<const E *>(cbl)[ok ? c : uint32_t(CBN)];
        } else if constexpr (CBN == 0) {
            E e = load_global(reinterpret_cast<const E *>(tg), min(c, kmax));
            if (!ok) e = E{};
            return e;
        } else {
            const bool inl = c < kl || !ok;
            const E el = reinterpret_cast<const E *>(cbl)[inl ? (ok ? c : uint32_t(CBN)) : 0u];
            const E eg = load_global(reinterpret_cast<const E *>(tg), inl ? 0u : min(c, kmax));
            return inl ? el : eg;
        }
    };
    // one superstep (MASK: its last block is ragged or absent for some lanes);
    // the x ring refills from superstep sb_next at its end
    auto compute = [&](auto mask_c, int sb, int vs, int sb_next,
                       uint32_t (&w)[BITS], const uint16_t (&s)[GPB]) {
        constexpr bool MASK = decltype(mask_c)::value;
        // GS steps at a time: the next group's lookups are issued before this
        // group's products, and nothing moves across a group's end (left alone
        // the compiler extracts every code of the block first and spills; the
        // pins keep extractions and conversions in their group)
        auto pin_words = [](uint32_t (&v)[BITS]) {
#pragma unroll
            for (int i = 0; i < BITS; ++i) asm volatile("" : "+v"(v[i]));
        };
        auto pin_raw = [](LinRaw<XM> &r) {
            asm volatile("" : "+v"(r.v));
            if constexpr (F32) asm volatile("" : "+v"(r.w));
        };
        h8 e0[GS], e1[GS];
        auto look = [&](int g, h8 (&e)[GS]) {
#pragma unroll
            for (int q = 0; q < GS; ++q) {
                const int st = g * GS + q;
                const bool ok = !MASK || st < vs;
                if constexpr (D == 8) {
                    e[q] = entry(block_field<BITS>(w, st), ok);
                } else if constexpr (D == 4) {
                    const h4 a = entry(block_field<BITS>(w, 2 * st), ok);
                    const h4 b = entry(block_field<BITS>(w, 2 * st + 1), ok);
                    e[q] = h8{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
                } else {
                    const h2 a = entry(block_field<BITS>(w, 4 * st), ok);
                    const h2 b = entry(block_field<BITS>(w, 4 * st + 1), ok);
                    const h2 c = entry(block_field<BITS>(w, 4 * st + 2), ok);
                    const h2 d = entry(block_field<BITS>(w, 4 * st + 3), ok);
                    e[q] = h8{a[0], a[1], b[0], b[1], c[0], c[1], d[0], d[1]};
                }
            }
        };
        auto group = [&](int g, h8 (&e)[GS], h8 (&en)[GS]) {
            pin_words(w);
            asm volatile("" : "+v"(vs));
            if (g + 1 < SPB / GS) look(g + 1, en);
#ifdef LINSB
            __builtin_amdgcn_sched_barrier(0);
#endif
#pragma unroll
            for (int q = 0; q < GS; ++q) {
                const int st = g * GS + q;
                const f16 sc = __builtin_bit_cast(f16, s[(st * GPB) / (4 * D)]);
                LinRaw<XM> (&xs)[NT] = xr[st % PF];
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) {
                    pin_raw(xs[nt]);
                    if (MASK && !FRAG && st >= vs) xs[nt] = LinRaw<XM>{};   // past the row's end
                    if constexpr (!WIDE) {
                        const h8 wv = e[q] * h8{sc, sc, sc, sc, sc, sc, sc, sc};
                        acc[nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wv, lin_f16<XM>(xs[nt]), acc[nt], 0, 0, 0);
                    } else {
                        float f[8];
                        lin_floats<XM>(xs[nt], f);
#pragma unroll
                        for (int i = 0; i < 8; ++i)
                            acc[nt] = __builtin_amdgcn_mfma_f32_16x16x4f32(float(e[q][i]) * float(sc), f[i],
                                                                           acc[nt], 0, 0, 0);
                    }
                }
                if (st + PF < SPB) load_x(sb, st + PF, xs);
                else load_x(sb_next, st + PF - SPB, xs);
            }
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) asm volatile("" : "+v"(acc[nt]));   // the products stay here too
            __builtin_amdgcn_sched_barrier(0);
        };
        look(0, e0);
#pragma unroll
        for (int g = 0; g < SPB / GS; g += 2) {
            group(g, e0, e1);
            group(g + 1, e1, e0);
        }
    };

    uint32_t w[BITS];
    uint16_t sc[GPB];
    int sb = ks;
    if (sb < NSS) {
        load_w(sb, w, sc);
#pragma unroll
        for (int st = 0; st < PF; ++st) load_x(sb, st, xr[st]);
    }
    wait_vmem();
    __syncthreads();
    // whole supersteps, the next one's weights in flight; past this wave's
    // last one the loads repeat it (never used), so every step issues the same
    const int nwhole = ragged ? NSS - 1 : NSS;
    while (sb < nwhole) {
        const int nx = sb + KS < NSS ? sb + KS : sb;
        uint32_t wn[BITS];
        uint16_t sn[GPB];
        load_w(nx, wn, sn);
        compute(std::false_type{}, sb, SPB, nx, w, sc);
#pragma unroll
        for (int i = 0; i < BITS; ++i) w[i] = wn[i];
#pragma unroll
        for (int g = 0; g < GPB; ++g) sc[g] = sn[g];
        sb += KS;
    }
    if (sb < NSS) compute(std::true_type{}, sb, valid_steps(sb), sb, w, sc);

    // ---- add the K slices in order; lane holds weight rows 4 lg + i of token
    // 16 nt + ln
    __syncthreads();                            // every wave is done with the table
    f32x4 *red = reinterpret_cast<f32x4 *>(smem);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) red[(wave * NT + nt) * 64 + lane] = acc[nt];
    const uint64_t live = __ballot(!dead);      // bit r: weight row r of this group is live
    __syncthreads();
    for (int nt = ks; nt < NT; nt += KS) {      // the group's row tiles, dealt to its slices
        f32x4 v = red[(rg * NT + nt) * 64 + lane];
        for (int q = 1; q < KS; ++q) v += red[((q * RG + rg) * NT + nt) * 64 + lane];
        const int t = t0 + 16 * nt + ln;
        if (t >= p.N) continue;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int r = 4 * lg + i;
            if (o0 + r < p.OUT)
                store_act(p.y, p.y_type, int64_t(t) * p.OUT + o0 + r, ((live >> r) & 1) ? v[i] : 0.f);
        }
    }
}

// The same through a copy of x in operand order at `frag` (lin_frag_bytes).
int launch_lin_frag_d2(const LinParams &p, int bits, void *frag, hipStream_t st);
int launch_lin_frag_d4(const LinParams &p, int bits, void *frag, hipStream_t st);
int launch_lin_frag_d8(const LinParams &p, int bits, void *frag, hipStream_t st);

// One launch over N rows with the instance for (d, bits, x mode, rows); a VQK
// status, VQK_ENOTIMPL when no instance matches.
int launch_lin_d2(const LinParams &p, int bits, int xm, hipStream_t st);
int launch_lin_d4(const LinParams &p, int bits, int xm, hipStream_t st);
int launch_lin_d8(const LinParams &p, int bits, int xm, hipStream_t st);

// x [N, IN] as the B operands of k_lin<.., NT, kXFrag>: piece (tile, superstep,
// step, nt, lane) is 8 fp16 values of token 16 (NT tile + nt) + lane % 16 at
// columns block(4 superstep + lane / 16) + 8 step, zero past N and IN. One
// operand load is then 1 KB in a row; read in place, its 64 lanes touch 64
// cache lines of 16 rows, and those lookups in the L1 took longer than the
// decode (16 rows of 5120 -> 17408, d4 K4096: 55 us against 26 for one row).
template <int D>
__global__ void __launch_bounds__(256) k_lin_frag(const void *x, int x_type, int N, int IN, int NSS, int NT,
                                                  u32x4 *out) {
    const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
    const int lane = int(i & 63);
    int64_t r = i >> 6;
    const int nt = int(r % NT);
    r /= NT;
    const int st = int(r % (4 * D));
    r /= 4 * D;
    const int sb = int(r % NSS), tile = int(r / NSS);
    const int t = 16 * (NT * tile + nt) + (lane & 15);
    const int col = (4 * sb + (lane >> 4)) * 32 * D + 8 * st;
    if (16 * NT * int64_t(tile) >= N) return;
    out[i] = t < N && col < IN ? load8_act(x, x_type, int64_t(t) * IN + col) : u32x4{0, 0, 0, 0};
}

// Rows up to which the direct loads always serve: each row of x adds its cache
// lines to every operand load (5120 -> 17408, d4 K4096: 4 rows 29 us in place,
// 8 rows 38 in place and 31 with the copy).
constexpr int kLinDirectRows = 4;

// 16-row tiles of x sharing one decode, for N rows in operand order
inline int lin_row_tiles(int64_t N) { return N <= 16 ? 1 : (N <= 32 ? 2 : 4); }

// Workgroups along OUT with 2^l K slices.
inline int lin_groups(const LinParams &p, int l) {
    const int rows = 16 * (kLinWaves >> l);
    return (p.OUT + rows - 1) / rows;
}

// log2 of the K slices of a workgroup: of 1, 2, 4, 8 (at most one per
// superstep) the one whose busiest CU walks the fewest supersteps --
// workgroups per CU, rounded up, times supersteps per wave, rounded up; the
// fewest slices of equals (each row group reads all of x). It picks the
// measured best of all four at 5120 -> 17408 (4 slices: 20 rows 36 us against
// 39 / 39 / 37), 17408 -> 5120 (4: 36 against 111 / 60 / 38) and 8192 -> 8192
// (4: 26 against 55 / 32 / 27), d4 K4096.
inline int lin_slices(const LinParams &p, int tiles) {
    const int64_t nss = (p.NB + 3) / 4;
    int best = 0;
    int64_t cost = INT64_MAX;
    for (int l = 0; l < 4 && (1 << l) <= nss; ++l) {
        const int64_t c = (int64_t(lin_groups(p, l)) * tiles + 255) / 256 * ((nss + (1 << l) - 1) >> l);
        if (c < cost) { cost = c; best = l; }
    }
    return best;
}

template <int D, int BITS, int GPB, int NT, int XM>
int go_lin_tile(LinParams p, hipStream_t st) {
    const int tiles = (p.N + 16 * NT - 1) / (16 * NT);
    p.ks_log2 = lin_slices(p, tiles);
    const dim3 grid(unsigned(lin_groups(p, p.ks_log2)), unsigned(tiles), 1);
    return launch_with_lds<k_lin<D, BITS, GPB, NT, XM>>(grid, dim3(kLinWaves * 64), lin_lds(D, BITS, NT), st, p);
}

// x in place: one 16-row tile; in operand order: tiles of 16, 32 or 64 rows.
// One 16-row weight tile per wave: two, sharing each x operand, halve the
// waves and ran 1.3-1.7x slower at every shape above (20 rows of 5120 ->
// 17408: 61 us against 36).
template <int D, int BITS, int GPB, int XM>
int go_lin(const LinParams &p, hipStream_t st) {
    if constexpr (XM != kXFrag) {
        return go_lin_tile<D, BITS, GPB, 1, XM>(p, st);
    } else {
        const int nt = lin_row_tiles(p.N);
        if (nt == 4) return go_lin_tile<D, BITS, GPB, 4, XM>(p, st);
        if (nt == 2) return go_lin_tile<D, BITS, GPB, 2, XM>(p, st);
        return go_lin_tile<D, BITS, GPB, 1, XM>(p, st);
    }
}

}  // namespace vqk
