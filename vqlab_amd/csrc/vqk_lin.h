// Matrix-core VQ linear for a few rows of x: y[n, o] = sum_i x[n, i] * W[o, i],
// the decode step of a dense linear (_dense_fused, vq_switch.py:3339-3434) for
// 2..64 rows of layers large enough for it (lin_beats_gemv, lin_beats_seg in
// vqk_lin.hip), and for every row count where the block-per-lane GEMV
// (vqk_gemv.h) has no fast form (more than 64 blocks per weight row, or a
// ragged last block).
//
// What bounds it: the LDS lookups of the decode (one table read per code) and,
// with many rows, the x operand, so each weight is decoded ONCE for up to 64
// rows of x -- the GEMV decodes it once per row -- and goes straight into an
// operand of v_mfma_f32_16x16x32: x is A (lane l: row l % 16), the codebook
// entries are B (lane l: weight row l % 16), both with 8 consecutive columns
// of lane group l / 16.
//
// The scale stays in fp32, as the GEMV has it: a product covers 32 columns of
// ONE block, so its sum has one scale per weight row, which multiplies it in
// fp32 as it is added to the row's total. Each lane group loads one block of a
// superstep's four (whole words, no shifts that depend on the lane), and the
// raw codes of 4 steps are transposed among the lane groups (v_permlane16_swap,
// v_permlane32_swap: one per step and register) so that every product gets its
// 32 columns from one block. DEQ instances multiply by the decoded weight
// fp16(cb * s) instead: vqk_dense_gemm's arithmetic.
//
// A workgroup is 8 waves = RG groups of 16 weight rows x KS slices of the
// K loop (KS * RG = 8): the waves of one row group take its supersteps (4
// blocks per row) in turn and add their partial sums through LDS, in slice
// order (no workspace, no second launch, the same bits every call). Splitting
// K inside the workgroup is what keeps all 8 waves of a CU loading weights
// when OUT / 16 alone would fill few CUs. x goes from L2 straight into the A
// operand's registers, in place for a few rows or from a copy in operand
// order; staged through LDS instead, with a barrier per chunk, 16 rows ran 83
// us against 56 in place (5120 -> 17408, d4 K4096): every chunk then waits for
// a load.
//
// The operands' type (XM): fp16, x rounded as the fused kernels round it; or
// fp32 (VQK_X_KEEP, d8) through v_mfma_f32_16x16x4_f32, whose lane (row l % 16,
// column l / 16) takes one of the same 8 values at a time: bf16 and fp32 x
// enter unrounded, at a sixteenth of the fp16 rate.
//
// Measured (MI355X, us per call, this kernel / the GEMV or, for 64 rows, the
// segment kernel; bf16 x):
//   5120 -> 17408, d4 K4096:  8 rows 28 / 102, 17 rows 35 / 204, 64 rows 51 / 68
//   17408 -> 5120, d4 K4096:  1 row 25 / 1719, 17 rows 36 / 3242 (generic GEMV)
//   5120 -> 17408, d8 K65536: 8 rows 77 / 411, 17 rows 134 / 831 (fp32 products)
#pragma once

#include <type_traits>

#include "vqk_gseg.h"

namespace vqk {

// x as an operand: fp16 as it is; bf16 / fp32 rounded to fp16; bf16 / fp32
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
    int32_t deq;               // W = fp16(cb * s), not the scale in fp32 on each group's sum
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
    const size_t tab = size_t(lin_table_entries(D, BITS)) * D * 2;
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

template <int XM>
__device__ __forceinline__ LinRaw<XM> lin_load_x(__amdgpu_buffer_rsrc_t x, uint32_t off, int base) {
    LinRaw<XM> r;
    r.v = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(x, off, base, 0));
    if constexpr (XM == kXF32r || XM == kXF32x)
        r.w = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(x, off + 16, base, 0));
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

// `width` bits from bit `bit` of a block's words on (both known after
// unrolling); the bits above them are whatever follows.
template <int BITS>
__device__ __forceinline__ uint32_t block_bits(const uint32_t (&w)[BITS], int bit, int width) {
    const int wi = bit >> 5, sh = bit & 31;
    if (sh + width <= 32) return w[wi] >> sh;
    return __builtin_amdgcn_alignbit(w[wi + 1 < BITS ? wi + 1 : BITS - 1], w[wi], sh);
}

// r[i] of lane group l becomes r[l] of lane group i (groups of 16 lanes).
__device__ __forceinline__ void transpose_groups(uint32_t (&r)[4]) {
    const auto a = __builtin_amdgcn_permlane32_swap(r[0], r[2], false, false);
    const auto b = __builtin_amdgcn_permlane32_swap(r[1], r[3], false, false);
    const auto c = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false);
    const auto d = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
    r[0] = c[0]; r[1] = c[1]; r[2] = d[0]; r[3] = d[1];
}

// r[q] = v of lane group q, in every lane group
__device__ __forceinline__ void broadcast_groups(uint32_t v, uint32_t (&r)[4]) {
    const auto a = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    const auto c = __builtin_amdgcn_permlane16_swap(a[0], a[0], false, false);
    const auto d = __builtin_amdgcn_permlane16_swap(a[1], a[1], false, false);
    r[0] = c[0]; r[1] = c[1]; r[2] = d[0]; r[3] = d[1];
}

template <int D, int BITS, int GPB, int NT, int XM, bool DEQ>
__global__ void __launch_bounds__(kLinWaves * 64, lin_waves_per_simd(D, BITS, NT)) k_lin(const LinParams p) {
    constexpr int SPB = 4 * D;                  // MFMA steps per superstep (32 columns each)
    constexpr int CPB = 32 * D;                 // columns per block
    constexpr int CBN = lin_table_entries(D, BITS);
    constexpr bool CBL = CBN == (1 << BITS);
    constexpr bool WIDE = XM == kXBF16x || XM == kXF32x;
    static_assert(!(WIDE && DEQ), "the decoded weight is fp16");
    constexpr bool F32 = XM == kXF32r || XM == kXF32x;
    // steps of x loads in flight: an L2 latency within the registers that two
    // workgroups per CU leave (8 steps instead of 4, one row tile: no faster at
    // 5120 -> 17408, 5 % slower at 4096 -> 1024)
    constexpr int PF = NT == 4 ? 2 : 4;
    // The scale after every product instead of every second, at once instead of
    // one pair of steps behind: two row tiles have no registers for the sums in
    // between (17 rows of 17408 -> 5120, d4 K4096: 37.2 us against 38.6 with
    // them and two steps of x in flight).
    constexpr bool EACH = NT == 2;
    static_assert(SPB % PF == 0 && D % 2 == 0, "whole rings and pairs of chunks per superstep");

    extern __shared__ __align__(16) uint8_t smem[];
    f16 *cbl = reinterpret_cast<f16 *>(smem);   // [CBN][D]

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));   // uniform loop bounds
    const int ln = lane & 15, lg = lane >> 4;
    const int KS = 1 << p.ks_log2, RG = kLinWaves >> p.ks_log2;
    const int rg = wave & (RG - 1), ks = wave >> (3 - p.ks_log2);
    const int o0 = (int(blockIdx.x) * RG + rg) * 16;
    const int t0 = int(blockIdx.y) * 16 * NT;

    lds_copy_async(p.codebook, cbl, min(p.K, CBN) * D * 2, CBN * D * 2);

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
    // byte offset of this lane's row and 8 columns of a step (rows past N
    // repeat the last one, never stored)
    uint32_t xrow = FRAG ? uint32_t(lane) * 16
                         : (uint32_t(min(t0 + ln, p.N - 1)) * uint32_t(p.IN) + uint32_t(lg * 8)) * XB;

    const int NSS = (p.NB + 3) >> 2;
    const uint32_t kmax = uint32_t(p.K - 1);
    const uint32_t kl = uint32_t(min(p.K, CBN));
    const f16 *tg = reinterpret_cast<const f16 *>(p.codebook);

    const bool ragged = p.NB % 4 != 0 || p.IN % CPB != 0;       // the last superstep is not whole
    // words and scales of block 4 sb + lg; in a ragged superstep those of
    // columns past the row's end are never multiplied, only kept in bounds
    auto load_w = [&](int sb, uint32_t (&w)[BITS], uint16_t (&s)[GPB]) {
        const int b = min(4 * sb + lg, p.NB - 1);
        const uint32_t *src = p.codes + cr * p.row_words;
        const uint16_t *sr = p.scales + cr * p.ngrp;
        if (!ragged || sb != NSS - 1) {
#pragma unroll
            for (int i = 0; i < BITS; ++i) w[i] = src[b * BITS + i];
#pragma unroll
            for (int g = 0; g < GPB; ++g) s[g] = sr[b * GPB + g];
        } else {
#pragma unroll
            for (int i = 0; i < BITS; ++i) w[i] = src[min(b * BITS + i, int(p.row_words) - 1)];
#pragma unroll
            for (int g = 0; g < GPB; ++g) s[g] = sr[min(b * GPB + g, p.ngrp - 1)];
        }
    };

    f32x4 acc[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[nt] = f32x4{0.f, 0.f, 0.f, 0.f};

    // x of step st = 4 j + q: columns 32 j .. 32 j + 31 of block 4 sb + q
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
            // a step past the row's end (never multiplied) reads its last columns
            const int col = min((4 * sb + (st & 3)) * CPB + 32 * (st >> 2), p.IN - 32);
            dst[0] = lin_load_x<XM>(xbuf, xrow, col * XB);
        }
    };
    auto entry = [&](uint32_t c) {
        typedef typename EntryT<D>::type E;
        if constexpr (CBL) {
            return reinterpret_cast<const E *>(cbl)[c];
        } else if constexpr (CBN == 0) {
            return load_global(reinterpret_cast<const E *>(tg), min(c, kmax));
        } else {
            const bool inl = c < kl;
            const E el = reinterpret_cast<const E *>(cbl)[inl ? c : 0u];
            const E eg = load_global(reinterpret_cast<const E *>(tg), inl ? 0u : min(c, kmax));
            return inl ? el : eg;
        }
    };
    // one superstep (MASK: columns past the row's end are left out); the x
    // ring refills from superstep sb_next at its end
    auto compute = [&](auto mask_c, int sb, int sb_next, uint32_t (&w)[BITS], const uint16_t (&s)[GPB]) {
        constexpr bool MASK = decltype(mask_c)::value;
        // Two steps at a time: the next two steps' lookups are in the same
        // scheduling group as these two's products, and nothing moves across a
        // group's end (left alone the compiler extracts every code of the block
        // first and spills; the pins keep extractions and conversions in their
        // group)
        auto pin_words = [](uint32_t (&v)[BITS]) {
#pragma unroll
            for (int i = 0; i < BITS; ++i) asm volatile("" : "+v"(v[i]));
        };
        auto pin_raw = [](LinRaw<XM> &r) {
            asm volatile("" : "+v"(r.v));
            if constexpr (F32) asm volatile("" : "+v"(r.w));
        };
        // codes of chunk j (steps 4 j .. 4 j + 3): this lane's are those of its
        // row's 8 columns from 8 lg on in each block q, which lane group q loaded
        constexpr int R = D == 2 ? 2 : 1, CPR = 8 / D / R;          // registers of a step's codes, codes of each
        constexpr uint32_t MASKB = (1u << BITS) - 1u;
        uint32_t r[R][4];
        auto codes_of = [&](int j) {
#pragma unroll
            for (int c = 0; c < R; ++c) {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    r[c][i] = block_bits<BITS>(w, ((4 * j + i) * R + c) * CPR * BITS, CPR * BITS);
                transpose_groups(r[c]);
            }
        };
        auto look = [&](int q) {
            if constexpr (D == 8) {
                return entry(r[0][q] & MASKB);
            } else if constexpr (D == 4) {
                const h4 a = entry(r[0][q] & MASKB), b = entry((r[0][q] >> BITS) & MASKB);
                return h8{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
            } else {
                const h2 a = entry(r[0][q] & MASKB), b = entry((r[0][q] >> BITS) & MASKB);
                const h2 c = entry(r[R - 1][q] & MASKB), d = entry((r[R - 1][q] >> BITS) & MASKB);
                return h8{a[0], a[1], b[0], b[1], c[0], c[1], d[0], d[1]};
            }
        };
        uint32_t sc[4];                         // scales of two groups of each block
        f32x4 sum[4][NT];                       // of one group (64 columns) of each block
        auto scales_of = [&](int g) {
            broadcast_groups(uint32_t(s[g]) | (GPB > 1 ? uint32_t(s[(g + 1) % GPB]) << 16 : 0u), sc);
        };
        auto scale = [&](int q, int g) {
            return __builtin_bit_cast(f16, uint16_t(sc[q] >> (16 * (g & 1))));
        };
        // the sums that pair h completed, scaled
        auto add_scaled = [&](int h) {
            const int j = h / 2, g = j / 2, q0 = 2 * (h & 1);
            if (!EACH && j % 2 == 0) return;
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const int q = q0 + u;
                if (MASK && (4 * sb + q) * CPB + 64 * g >= p.IN) continue;  // uniform
                const float c = float(scale(q, g));
#pragma unroll
                for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                    for (int i = 0; i < 4; ++i) acc[nt][i] = fmaf(c, sum[q][nt][i], acc[nt][i]);
            }
        };
        auto pair = [&](int h, h8 (&e)[2], h8 (&en)[2]) {
            const int j = h / 2, g = j / 2, q0 = 2 * (h & 1);
            pin_words(w);
            if (DEQ && h % 8 == 0) scales_of(g);
            if (h + 1 < 2 * D) {
                if (h & 1) codes_of(j + 1);
#pragma unroll
                for (int u = 0; u < 2; ++u) en[u] = look(2 - q0 + u);
            }
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const int q = q0 + u, st = 4 * j + q;
                LinRaw<XM> (&xs)[NT] = xr[st % PF];
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) pin_raw(xs[nt]);
                if (!MASK || (4 * sb + q) * CPB + 64 * g < p.IN) {          // uniform
                    h8 wv = e[u];
                    if constexpr (DEQ) {
                        const f16 c = scale(q, g);
                        wv = wv * h8{c, c, c, c, c, c, c, c};
                    }
#pragma unroll
                    for (int nt = 0; nt < NT; ++nt) {
                        f32x4 v = DEQ ? acc[nt] : (EACH || j % 2 == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : sum[q][nt]);
                        if constexpr (!WIDE) {
                            v = __builtin_amdgcn_mfma_f32_16x16x32_f16(lin_f16<XM>(xs[nt]), wv, v, 0, 0, 0);
                        } else {
                            float f[8];
                            lin_floats<XM>(xs[nt], f);
#pragma unroll
                            for (int i = 0; i < 8; ++i)
                                v = __builtin_amdgcn_mfma_f32_16x16x4f32(f[i], float(wv[i]), v, 0, 0, 0);
                        }
                        if constexpr (DEQ) acc[nt] = v;
                        else sum[q][nt] = v;
                    }
                }
                if (st + PF < SPB) load_x(sb, st + PF, xs);
                else load_x(sb_next, st + PF - SPB, xs);
            }
            if constexpr (!DEQ) {
                // scaled one pair behind: a product's sum is ready then
                if (!EACH && h > 0) add_scaled(h - 1);
                if (h % 8 == 0) scales_of(g);
                if (EACH) add_scaled(h);
#pragma unroll
                for (int u = 0; u < 2; ++u)
#pragma unroll
                    for (int nt = 0; nt < NT; ++nt)
                        if (!EACH) asm volatile("" : "+v"(sum[q0 + u][nt]));
            }
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) asm volatile("" : "+v"(acc[nt]));   // the products stay here too
            __builtin_amdgcn_sched_barrier(0);
        };
        h8 e0[2], e1[2];
        codes_of(0);
        e0[0] = look(0);
        e0[1] = look(1);
#pragma unroll
        for (int h = 0; h < 2 * D; h += 2) {
            pair(h, e0, e1);
            pair(h + 1, e1, e0);
        }
        if constexpr (!DEQ && !EACH) add_scaled(2 * D - 1);
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
        compute(std::false_type{}, sb, nx, w, sc);
#pragma unroll
        for (int i = 0; i < BITS; ++i) w[i] = wn[i];
#pragma unroll
        for (int g = 0; g < GPB; ++g) sc[g] = sn[g];
        sb += KS;
    }
    if (sb < NSS) compute(std::true_type{}, sb, sb, w, sc);

    // ---- add the K slices in order; lane holds tokens 4 lg + i of a row tile,
    // weight row ln
    __syncthreads();                            // every wave is done with the table
    f32x4 *red = reinterpret_cast<f32x4 *>(smem);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) red[(wave * NT + nt) * 64 + lane] = acc[nt];
    __syncthreads();
    for (int nt = ks; nt < NT; nt += KS) {      // the group's row tiles, dealt to its slices
        f32x4 v = red[(rg * NT + nt) * 64 + lane];
        for (int q = 1; q < KS; ++q) v += red[((q * RG + rg) * NT + nt) * 64 + lane];
        if (o0 + ln >= p.OUT) continue;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int t = t0 + 16 * nt + 4 * lg + i;
            if (t < p.N) store_act(p.y, p.y_type, int64_t(t) * p.OUT + o0 + ln, dead ? 0.f : v[i]);
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

// x [N, IN] as the A operands of k_lin<.., NT, kXFrag>: piece (tile, superstep,
// step 4 j + q, nt, lane) is 8 fp16 values of row 16 (NT tile + nt) + lane % 16
// at columns 32 j + 8 (lane / 16) of block 4 superstep + q, zero past N and IN.
// One operand load is then 1 KB in a row; read in place, it is 64 bytes of each
// of 16 rows.
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
    const int col = (4 * sb + (st & 3)) * 32 * D + 32 * (st >> 2) + 8 * (lane >> 4);
    if (16 * NT * int64_t(tile) >= N) return;
    out[i] = t < N && col < IN ? load8_act(x, x_type, int64_t(t) * IN + col) : u32x4{0, 0, 0, 0};
}

// Rows up to which the direct loads always serve: each row of x adds its cache
// lines to every operand load (5120 -> 17408, d4 K4096: 4 rows 28 us in place,
// 8 rows 33 in place and 26 with the copy).
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
// measured best of all four at 5120 -> 17408 (4 slices: 20 rows 35 us against
// 39 / 40 / 38), 17408 -> 5120 (4: 36 against 110 / 59 / 38) and 8192 -> 8192
// (4: 21 against 55 / 32 / 23), d4 K4096.
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

template <int D, int BITS, int GPB, int NT, int XM, bool DEQ>
int go_lin_tile(LinParams p, hipStream_t st) {
    const int tiles = (p.N + 16 * NT - 1) / (16 * NT);
    p.ks_log2 = lin_slices(p, tiles);
    const dim3 grid(unsigned(lin_groups(p, p.ks_log2)), unsigned(tiles), 1);
    return launch_with_lds<k_lin<D, BITS, GPB, NT, XM, DEQ>>(grid, dim3(kLinWaves * 64), lin_lds(D, BITS, NT), st, p);
}

// x in place: one 16-row tile; in operand order: tiles of 16, 32 or 64 rows.
// One 16-row weight tile per wave: two, sharing each x operand, halve the
// waves and, in this kernel's first form, ran 1.3-1.7x slower at every shape
// above (20 rows of 5120 -> 17408: 61 us against 36).
template <int D, int BITS, int GPB, int XM, bool DEQ>
int go_lin_mode(const LinParams &p, hipStream_t st) {
    if constexpr (XM != kXFrag) {
        return go_lin_tile<D, BITS, GPB, 1, XM, DEQ>(p, st);
    } else {
        const int nt = lin_row_tiles(p.N);
        if (nt == 4) return go_lin_tile<D, BITS, GPB, 4, XM, DEQ>(p, st);
        if (nt == 2) return go_lin_tile<D, BITS, GPB, 2, XM, DEQ>(p, st);
        return go_lin_tile<D, BITS, GPB, 1, XM, DEQ>(p, st);
    }
}

template <int D, int BITS, int GPB, int XM>
int go_lin(const LinParams &p, hipStream_t st) {
    if constexpr (XM != kXBF16x && XM != kXF32x)
        if (p.deq) return go_lin_mode<D, BITS, GPB, XM, true>(p, st);
    return go_lin_mode<D, BITS, GPB, XM, false>(p, st);
}

}  // namespace vqk
