// Matrix-core kernel for expert segments of many rows (prompts): y[t, o] =
// sum_i x[t, i] * W[o, i] for up to 96 sorted pairs t of one expert -- or, of a
// gate and an up projection at once, h = fp16(silu(g) * u).
//
// What bounds the 16-row segment kernel (vqk_gseg.h) there is that it decodes
// an expert's weights again for every 16 rows, and that one x operand feeds
// one MFMA. Here a weight is decoded once for up to 96 rows, into the A operand
// of v_mfma_f32_32x32x16 (lane l: weight row l % 32, 8 consecutive columns of
// lane group l / 32, which holds every other 32-code block of the row), and
// each 1 KB x operand read from LDS feeds a 32 x 32 tile -- two of them where
// gate and up run together. 2048 tokens x 8 of 256 experts of 2048 x 512, d4
// K4096 (MI355X, kernel trace): gate + up 135 us (69 GFLOP), down 92 us (34
// GFLOP), against 3 x ~200 us. Timing probes (of 130 us in their session) put
// ~86 us into everything but the lookups and products (the 218 MB of weights,
// x copies, stores, start-up) and ~65 us into those, half of it overlapped: two
// waves per SIMD (the sums of 96 rows take the registers of four) leave
// latencies uncovered.
//
// Workgroup = 8 waves x 32 weight rows over one tile of rows. The weights'
// words are loaded one superstep (2 blocks) ahead into registers. x is fp16
// rows in global memory and passes through LDS in chunks of 8 MFMA steps (64
// columns of each lane group), copied by global_load_lds NBUF - 1 chunks
// ahead; a row's 128 bytes of a chunk are 8 slots of 16 bytes, slot s of row r
// stored at s ^ ((r >> 1) & 7), so the 16 rows of one read phase fall on
// distinct banks. One barrier per chunk.
#pragma once

#include <type_traits>

#include "vqk_gseg.h"

namespace vqk {

typedef float f32x16w __attribute__((ext_vector_type(16)));

struct WideMod {               // one projection: E experts of OUT rows
    const uint32_t *codes;
    int64_t row_words;
    const uint16_t *codebook;  // fp16 [K, D], 16-byte aligned
    const uint16_t *scales;
    const int32_t *row_table;  // [E, OUT] or NULL
    int64_t stored_rows;       // > 0
    int32_t K, ngrp;
};

struct WideParams {
    WideMod m[2];              // m[1]: the up projection of a pair
    int32_t E, OUT, IN, NB;
    int32_t rb;                // row blocks (256 rows) per workgroup
    const uint16_t *x;         // fp16 rows of IN, 16-byte aligned
    uint32_t x_bytes;          // <= 2 GB
    int32_t xkrep;             // x row of pair n = n / xkrep; 0: row = sorted position
    void *y;
    int32_t y_type;
    int32_t ysorted;           // y row = sorted position, not pair
    int32_t N;                 // pairs; dense: rows of x
    const int32_t *tmeta;      // (expert or -1, first sorted row, rows) per tile; NULL: dense
    const int32_t *ntiles;
    const int32_t *order;      // sorted position -> pair
};

// LDS of an instance: the tables, and NBUF chunks of 32 * NT rows. A pair of
// tables of 64 KB leaves two chunks of 64 rows (160 KB to the byte).
struct WideShape { int nt, nbuf; };
__host__ __device__ constexpr WideShape wide_shape(int D, int BITS, bool pair) {
    const int tab = (1 << BITS) * D * 2 * (pair ? 2 : 1);
    return tab > 64 * 1024 ? WideShape{2, 2} : WideShape{3, 3};
}
__host__ __device__ constexpr size_t wide_lds(int D, int BITS, bool pair) {
    const WideShape s = wide_shape(D, BITS, pair);
    return size_t(1 << BITS) * D * 2 * (pair ? 2 : 1) + size_t(s.nbuf) * s.nt * 32 * 256;
}

// vector-memory loads of one block's words (16 bytes at a time) and scales
__host__ __device__ constexpr int wide_w_loads(int BITS) { return (BITS + 3) / 4 + 1; }

// the x of a lane group without a block
static __device__ const u32x4 kWideZeros[1] = {u32x4{0, 0, 0, 0}};

template <int D, int BITS, int GPB, bool PAIR, int NT>
__device__ __forceinline__ void wide_body(const WideParams &p, int expert, int row0, int nrows) {
    constexpr WideShape S = wide_shape(D, BITS, PAIR);
    constexpr int NBUF = S.nbuf, TOK = S.nt * 32;
    constexpr int NM = PAIR ? 2 : 1;
    constexpr int SPB = 4 * D, CPB = 32 * D, CPS = SPB / 8;   // steps, columns, chunks per block
    constexpr int TABE = 1 << BITS;
    extern __shared__ __align__(16) uint8_t smem[];
    f16 *tab = reinterpret_cast<f16 *>(smem);                 // [NM][TABE][D]
    uint8_t *xs = smem + size_t(NM) * TABE * D * 2;           // [NBUF][2][TOK][128 B]

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
    const int ln = lane & 31, lg = lane >> 5;

#pragma unroll
    for (int m = 0; m < NM; ++m)
        lds_copy_async(p.m[m].codebook, tab + m * TABE * D, p.m[m].K * D * 2, TABE * D * 2);

    // stored rows of this lane's weight rows in row block xb; a dead or absent
    // row reads row 0 and is written as +0 or not at all
    struct Rows {
        const uint32_t *w[NM];
        const uint16_t *s[NM];
        uint32_t live[NM];                      // bit r: row r of this wave's 32
        int o0;
    };
    auto rows_of = [&](int xb) {
        Rows r;
        r.o0 = xb * 256 + wave * 32;
#pragma unroll
        for (int m = 0; m < NM; ++m) {
            int64_t f = -1;
            if (expert >= 0 && expert < p.E && r.o0 + ln < p.OUT) {
                f = int64_t(expert) * p.OUT + r.o0 + ln;

                if (p.m[m].row_table) f = p.m[m].row_table[f];
                if (f >= p.m[m].stored_rows) f = -1;
            }
            r.live[m] = uint32_t(__ballot(f >= 0));
            if (f < 0) f = 0;
            r.w[m] = p.m[m].codes + f * p.m[m].row_words;
            r.s[m] = p.m[m].scales + f * p.m[m].ngrp;
        }
        return r;
    };
    // this lane's source of each of the wave's NT copies of a chunk: 8 rows x
    // 128 bytes of one lane group (rows past the tile repeat its last one)
    const int cg = wave & 1;
    uint32_t xsrc[NT];                          // byte offsets in x (at most 2 GB)
#pragma unroll
    for (int r = 0; r < NT; ++r) {
        const int t = ((wave >> 1) + 4 * r) * 8 + (lane >> 3);
        const int pos = row0 + min(t, nrows - 1);
        const int row = p.tmeta && p.xkrep ? p.order[pos] / p.xkrep : pos;
        xsrc[r] = (uint32_t(row) * uint32_t(p.IN) + uint32_t(cg * CPB + 8 * ((lane & 7) ^ ((t >> 1) & 7)))) * 2;
    }
    // Copied with buffer loads: the compiler takes a global_load_lds for a flat
    // access that may still return to LDS, and then waits for every LDS read
    // instead of counting them.
    const __amdgpu_buffer_rsrc_t xbuf =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(p.x), 0, int(p.x_bytes), 0x00027000);
    const __amdgpu_buffer_rsrc_t zbuf =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<u32x4 *>(kWideZeros), 0, 16, 0x00027000);
    int yrow[NT];                               // output rows of tokens 32 nt + ln, or -1
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        const int t = 32 * nt + ln;
        yrow[nt] = t < nrows ? (p.tmeta && !p.ysorted ? p.order[row0 + t] : row0 + t) : -1;
    }
    const int NSS = (p.NB + 1) >> 1, NCH = NSS * CPS;
    // x chunk c of a row block; with an odd block count the last superstep's
    // second lane group has no block: its x is zeros
    auto copy_x = [&](int c, int buf) {
        const int sb = c / CPS;
        const bool none = cg && 2 * sb + 1 >= p.NB;
        const int col = none ? 0 : (sb * 2 * CPB + (c % CPS) * 64) * 2;
        uint8_t *dst = xs + (buf * 2 + cg) * TOK * 128 + (wave >> 1) * 1024;
#pragma unroll
        for (int r = 0; r < NT; ++r)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(none ? zbuf : xbuf, (lds_void *)(dst + r * 4096), 16,
                                                     none ? 0u : xsrc[r], col, 0, 0);
    };
    auto load_w = [&](const Rows &r, int sb, uint32_t (&w)[NM][BITS], uint16_t (&s)[NM][GPB]) {
        const int b = min(2 * sb + lg, p.NB - 1);
#pragma unroll
        for (int m = 0; m < NM; ++m) {
#pragma unroll
            for (int i = 0; i < BITS; ++i) w[m][i] = r.w[m][b * BITS + i];
#pragma unroll
            for (int g = 0; g < GPB; ++g) s[m][g] = r.s[m][b * GPB + g];
        }
    };

    // a lane group without a block multiplies the zeros of its x by a weight of
    // zero: the last block's again could be infinite
    auto drop_scales = [&](int sb, uint16_t (&s)[NM][GPB]) {
#pragma unroll
        for (int m = 0; m < NM; ++m)
#pragma unroll
            for (int g = 0; g < GPB; ++g) s[m][g] = 2 * sb + lg < p.NB ? s[m][g] : uint16_t(0);
    };

    f32x16w acc[NM][NT];
    auto clear = [&]() {
#pragma unroll
        for (int m = 0; m < NM; ++m)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) acc[m][nt] = f32x16w{};
    };

    const int swz = (ln >> 1) & 7;
    // chunk C of a block: steps 8 C .. 8 C + 7 from x buffer `buf`; each step's
    // lookups and operands are read during the step before. The pins keep each
    // step's extractions, lookups and products where they are (left alone the
    // compiler extracts every code first and spills).
    auto compute = [&](auto cc, int buf, uint32_t (&w)[NM][BITS], const uint16_t (&s)[NM][GPB]) {
        constexpr int C = decltype(cc)::value;
        const uint8_t *xb = xs + (buf * 2 + lg) * TOK * 128 + ln * 128;
        struct Ops { h8 e[NM], x[NT]; };
        auto read_x = [&](int q, Ops &o) {
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
                o.x[nt] = *reinterpret_cast<const h8 *>(xb + nt * 4096 + ((q ^ swz) << 4));
        };
        auto read = [&](int q, Ops &o) {
#pragma unroll
            for (int m = 0; m < NM; ++m)
                o.e[m] = step_entries<D, BITS>(w[m], 8 * C + q, tab + m * TABE * D, 0u, false);
            read_x(q, o);
        };
        auto one = [&](int q, Ops &o, Ops &on) {
            const int st = 8 * C + q;
#pragma unroll
            for (int m = 0; m < NM; ++m)
#pragma unroll
                for (int i = 0; i < BITS; ++i) asm volatile("" : "+v"(w[m][i]));
            if (q < 7) read(q + 1, on);
            __builtin_amdgcn_sched_barrier(0);  // the reads first: they have this step's products to land in
#pragma unroll
            for (int m = 0; m < NM; ++m) {
                const f16 sc = __builtin_bit_cast(f16, s[m][(st * GPB) / SPB]);
                const h8 wv = o.e[m] * h8{sc, sc, sc, sc, sc, sc, sc, sc};
#pragma unroll
                for (int nt = 0; nt < NT; ++nt)
                    acc[m][nt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(wv, o.x[nt], acc[m][nt], 0, 0, 0);
            }
#pragma unroll
            for (int m = 0; m < NM; ++m)
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) asm volatile("" : "+v"(acc[m][nt]));
            __builtin_amdgcn_sched_barrier(0);
        };
        Ops a, b;
        read(0, a);
#pragma unroll
        for (int q = 0; q < 8; q += 2) {
            one(q, a, b);
            one(q + 1, b, a);
        }
    };
    // lane holds rows 8 j + 4 lg + i of token 32 nt + ln (register 4 j + i)
    auto store = [&](const Rows &rw) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            if (yrow[nt] < 0) continue;
            const int64_t yo = int64_t(yrow[nt]) * p.OUT;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int r = 8 * j + 4 * lg, o = rw.o0 + r;
                float v[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    v[i] = ((rw.live[0] >> (r + i)) & 1) ? acc[0][nt][4 * j + i] : 0.f;
                    if constexpr (PAIR) {
                        const float u = ((rw.live[1] >> (r + i)) & 1) ? acc[1][nt][4 * j + i] : 0.f;
                        v[i] = v[i] / (1.f + __expf(-v[i])) * u;
                    }
                }
                if (PAIR && o + 3 < p.OUT && p.OUT % 4 == 0) {
                    *reinterpret_cast<u32x2 *>(static_cast<uint16_t *>(p.y) + yo + o) =
                        u32x2{uint32_t(f32_to_h(v[0])) | (uint32_t(f32_to_h(v[1])) << 16),
                              uint32_t(f32_to_h(v[2])) | (uint32_t(f32_to_h(v[3])) << 16)};
                } else if (!PAIR && p.y_type == VQK_F32 && o + 3 < p.OUT && p.OUT % 4 == 0) {
                    *reinterpret_cast<f32x4 *>(static_cast<float *>(p.y) + yo + o) = f32x4{v[0], v[1], v[2], v[3]};
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (o + i < p.OUT) store_act(p.y, PAIR ? int32_t(VQK_F16) : p.y_type, yo + o + i, v[i]);
                }
            }
        }
    };

    const int nxb = (p.OUT + 255) / 256, xb0 = int(blockIdx.x) * p.rb;
    const int nb = min(p.rb, nxb - xb0);        // row blocks of this workgroup
    uint32_t w[NM][BITS], wn[NM][BITS];
    uint16_t sc[NM][GPB], sn[NM][GPB];
    Rows rw = rows_of(xb0);
    int next = 0;                               // x chunk that the next copy takes
    auto copy_next = [&](int buf) {
        copy_x(next, buf);
        next = next + 1 < NCH ? next + 1 : 0;   // past the last row block: a copy nobody reads
    };
#pragma unroll
    for (int c = 0; c < NBUF - 1; ++c) copy_next(c);
    load_w(rw, 0, w, sc);
    clear();
    wait_vmem();                                // the tables and the first chunks
    __syncthreads();
    int buf = 0;
    for (int k = 0; k < nb; ++k) {
        Rows rn = rw;
        for (int sb = 0; sb < NSS; ++sb) {
            const bool last = sb + 1 == NSS;
            if (last && k + 1 < nb) rn = rows_of(xb0 + k + 1);
            static_for<CPS>([&](auto cc) {
                constexpr int C = decltype(cc)::value;
                // into the buffer of the chunk before this one, which every wave has left
                copy_next(buf == 0 ? NBUF - 1 : buf - 1);
                asm volatile("" ::: "memory");
                if constexpr (C == 0) {
                    load_w(rn, last ? 0 : sb + 1, wn, sn);
                    asm volatile("" ::: "memory");
                    if (last) drop_scales(sb, sc);
                }
                compute(cc, buf, w, sc);
                // the next chunk's copies are in: of this wave's loads at most the
                // copies issued after them (NBUF - 2 chunks') are outstanding, and
                // the weights' loads when those are newer too
                constexpr int newer = (NBUF - 2) * NT;
                constexpr bool w_newer = C < NBUF - 1;
                asm volatile("" ::: "memory");
                wait_vmcnt<newer + (w_newer ? NM * wide_w_loads(BITS) : 0)>();
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
                buf = buf == NBUF - 1 ? 0 : buf + 1;
            });
#pragma unroll
            for (int m = 0; m < NM; ++m) {
#pragma unroll
                for (int i = 0; i < BITS; ++i) {
                    w[m][i] = wn[m][i];
                    asm volatile("" : "+v"(w[m][i]));   // loaded in every round: the waits count these loads
                }
#pragma unroll
                for (int g = 0; g < GPB; ++g) sc[m][g] = sn[m][g];
            }
        }
        store(rw);
        clear();
        rw = rn;
    }
    wait_vmem();                                // no copy may land after the LDS is given back
}

template <int D, int BITS, int GPB, bool PAIR>
__global__ void __launch_bounds__(512, 2) k_wide(const WideParams p) {
    constexpr int NTM = wide_shape(D, BITS, PAIR).nt;
    int expert = 0, row0, nrows;
    if (p.tmeta) {
        if (int(blockIdx.y) >= *p.ntiles) return;             // uniform, before any barrier
        const int32_t *tm = p.tmeta + 3 * blockIdx.y;
        expert = tm[0];
        row0 = tm[1];
        nrows = tm[2];
    } else {
        row0 = int(blockIdx.y) * 32 * NTM;
        nrows = min(32 * NTM, p.N - row0);
    }
    expert = __builtin_amdgcn_readfirstlane(expert);
    row0 = __builtin_amdgcn_readfirstlane(row0);
    nrows = __builtin_amdgcn_readfirstlane(nrows);
    if (nrows <= 32) wide_body<D, BITS, GPB, PAIR, 1>(p, expert, row0, nrows);
    else if (NTM == 2 || nrows <= 64) wide_body<D, BITS, GPB, PAIR, 2>(p, expert, row0, nrows);
    else if constexpr (NTM > 2) wide_body<D, BITS, GPB, PAIR, 3>(p, expert, row0, nrows);
}

// `pair`: m[0] and m[1] at once into fp16 SwiGLU rows. A VQK status,
// VQK_ENOTIMPL when no instance matches.
int launch_wide_d4(const WideParams &p, int bits, bool pair, dim3 grid, hipStream_t st);
int launch_wide_d8(const WideParams &p, int bits, bool pair, dim3 grid, hipStream_t st);

}  // namespace vqk
