// Matrix-core kernel for expert segments over d = 8 tables of 256 KB (K up to
// 16384), which do not fit LDS: y[t, o] = sum_i x[t, i] * W[o, i] for up to 32
// sorted pairs t of one expert.
//
// What bounds the segment kernels that keep part of such a table in LDS is the
// rest of it: every second code is one scattered 16-byte read of L2, one
// address at a time. Here a workgroup holds one HALF of every entry -- columns
// 0..3 or 4..7, 128 KB -- and computes the half of the sum over those columns
// of each code; the half sums (fp32) are added by the kernel that reads them.
// Every lookup is then an 8-byte LDS read. The codes are read by both halves,
// on one XCD (neighbours in its dispatch order) and while their tiles are few
// at about the same time: 0.69 GB fetched for gate and up of 64 tokens below,
// of 0.61 GB live; 1.93 GB for 509 tokens, of 1.07 GB. x comes split the same
// way ([2][rows, IN / 2]).
// 509 tokens x 10 of 512 experts of 4096 x 1024 and a shared expert, d8 K16384
// (MI355X, kernel trace, beside the shared expert): gate + up 631 us, down 267
// us; the layer, call to call, 2190 -> 976 us; 64 tokens, a fifth of the rows
// dead, 848 -> 590 us. What bounds it now, by timing probes of gate + up in one
// session on a slower box (690 us whole there): 520 without the weight loads,
// 365 without loads and lookups; leaving out the lookups or the x copies alone
// gained nothing (740, 735). The words arrive later than one superstep, and 128
// registers a wave leave no room for two.
//
// Workgroup = 16 waves x 32 weight rows; it keeps its table over several
// tiles. A superstep is two 32-code blocks, one to each lane group of
// v_mfma_f32_32x32x16 (lane l: weight row l % 32; 8 half columns = 2 codes a
// step). The next superstep's words are loaded into registers and its x (2 x 32
// rows x 256 bytes, fp16) copied straight to LDS meanwhile: 160 KB with the
// table to the byte. Slot s (16 bytes) of x row r lies at s ^ (r & 15),
// so a read phase of 16 rows falls on distinct banks.
#pragma once

#include "vqk_gseg.h"

namespace vqk {

typedef float f32x16h __attribute__((ext_vector_type(16)));

constexpr int kHalfWaves = 16, kHalfRows = 32 * kHalfWaves, kHalfTok = 32;

struct HalfMod {               // one projection: E experts of OUT rows
    const uint32_t *codes;
    int64_t row_words;
    const uint16_t *codebook;  // fp16 [K, 8], 16-byte aligned
    const uint16_t *scales;    // [stored_rows, ngrp], 8-byte aligned
    const int32_t *row_table;  // [E, OUT] or NULL
    int64_t stored_rows;       // > 0
    int32_t K, ngrp;
    float *y[2];               // half sums [N, OUT]
};

struct HalfParams {
    HalfMod m[2];
    int32_t nproj;             // projections of the launch (gate and up, or one)
    int32_t E, OUT, NB;
    int32_t rb, nxg;           // row blocks (512 rows) of an item, items of a tile
    int32_t units;             // workgroups of one half of one projection
    const uint16_t *x[2];      // half columns: fp16 rows of 128 * NB, 16-byte aligned
    uint32_t x_bytes;          // of one half, <= 2 GB
    int32_t xkrep;             // x row of pair n = n / xkrep; 0: row = sorted position
    int32_t ysorted;           // y row = sorted position, not pair
    int32_t N;                 // pairs; dense: rows of x
    const int32_t *tmeta;      // (expert or -1, first sorted row, rows) per tile; NULL: dense
    const int32_t *ntiles;
    const int32_t *order;      // sorted position -> pair
};

constexpr size_t half_lds(int BITS) { return (size_t(1) << BITS) * 8 + 2 * 2 * kHalfTok * 256; }

// the x of a lane group without a block
static __device__ const u32x4 kHalfZeros[1] = {u32x4{0, 0, 0, 0}};

template <int BITS>
__global__ void __launch_bounds__(64 * kHalfWaves) k_half(const HalfParams p) {
    constexpr int TABE = 1 << BITS, NTH = 64 * kHalfWaves;
    extern __shared__ __align__(16) uint8_t smem[];
    f16 *tab = reinterpret_cast<f16 *>(smem);                 // [TABE][4]
    uint8_t *xs = smem + size_t(TABE) * 8;                    // [2][2][32][256 B]

    const int tid = int(threadIdx.x), lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ln = lane & 31, lg = lane >> 5;

    // workgroups i and i + 8 (one XCD) are the two halves of a unit
    const int bid = int(blockIdx.x);
    const int half = (bid >> 3) & 1, unit = (bid >> 4) * 8 + (bid & 7);
    if (unit >= p.units * p.nproj) return;                    // uniform, before any barrier
    const HalfMod &m = p.m[p.nproj == 2 ? unit & 1 : 0];
    const int first = p.nproj == 2 ? unit >> 1 : unit;

    const int tiles = p.tmeta ? *p.ntiles : (p.N + kHalfTok - 1) / kHalfTok;
    const int items = tiles * p.nxg;
    if (first >= items) return;
    {
        const u32x2 *src = reinterpret_cast<const u32x2 *>(m.codebook) + half;
        u32x2 *dst = reinterpret_cast<u32x2 *>(tab);
        constexpr int PER = TABE / NTH;         // entries of a thread, 8 loads in flight
        for (int j0 = 0; j0 < PER; j0 += 8) {
            u32x2 v[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = src[2 * int64_t(min(tid + (j0 + j) * NTH, m.K - 1))];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int i = tid + (j0 + j) * NTH;
                dst[i] = i < m.K ? v[j] : u32x2{0, 0};
            }
        }
        static_assert(PER % 8 == 0, "a thread's entries come in eights");
    }
    const __amdgpu_buffer_rsrc_t xbuf =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(p.x[half]), 0, int(p.x_bytes), 0x00027000);
    const __amdgpu_buffer_rsrc_t zbuf =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<u32x4 *>(kHalfZeros), 0, 16, 0x00027000);

    const int NSS = (p.NB + 1) >> 1;
    const int nxb = (p.OUT + kHalfRows - 1) / kHalfRows;
    const int cg = wave & 1;                    // lane group and rows of this wave's x copies
    const int trow = (wave >> 1) * 4 + (lane >> 4);
    float *const y = m.y[half];

    for (int item = first; item < items; item += p.units) {
        const int tile = item / p.nxg, xb0 = (item % p.nxg) * p.rb;
        const int nb = min(p.rb, nxb - xb0);
        int expert = 0, row0 = tile * kHalfTok, nrows = min(kHalfTok, p.N - row0);
        if (p.tmeta) {
            expert = p.tmeta[3 * tile];
            row0 = p.tmeta[3 * tile + 1];
            nrows = p.tmeta[3 * tile + 2];
        }
        expert = __builtin_amdgcn_readfirstlane(expert);
        row0 = __builtin_amdgcn_readfirstlane(row0);
        nrows = __builtin_amdgcn_readfirstlane(nrows);
        if (nrows <= 0 || nb <= 0) continue;    // uniform

        // source of this lane's piece of a chunk (rows past the tile repeat its last one)
        const int pos = row0 + min(trow, nrows - 1);
        const int xrow = p.tmeta && p.xkrep ? p.order[pos] / p.xkrep : pos;
        const uint32_t xsrc =
            (uint32_t(xrow) * uint32_t(p.NB) * 128u + uint32_t(cg * 128 + 8 * ((lane & 15) ^ (trow & 15)))) * 2u;
        const int yrow = ln < nrows ? (p.tmeta && !p.ysorted ? p.order[row0 + ln] : row0 + ln) : -1;

        // with an odd block count the last superstep's second lane group has no
        // block: its x and its scales are zeros
        auto copy_x = [&](int sb, int buf) {
            const bool none = cg && 2 * sb + 1 >= p.NB;
            uint8_t *dst = xs + (buf * 2 + cg) * (kHalfTok * 256) + (wave >> 1) * 1024;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(none ? zbuf : xbuf, (lds_void *)dst, 16, none ? 0u : xsrc,
                                                     none ? 0 : sb * 512, 0, 0);
        };
        // Weight words are loaded as one stream over the item's row blocks, one
        // superstep ahead of the products. A dead or absent row reads row 0 and
        // is written as +0 or not at all.
        const uint32_t *wsrc;
        const uint16_t *ssrc;
        auto rows_of = [&](int k) -> uint32_t {
            const int o = (xb0 + k) * kHalfRows + wave * 32 + ln;
            int64_t f = -1;
            if (expert >= 0 && expert < p.E && o < p.OUT) {
                f = int64_t(expert) * p.OUT + o;
                if (m.row_table) f = m.row_table[f];
                if (f >= m.stored_rows) f = -1;
            }
            const uint32_t live = uint32_t(__ballot(f >= 0));
            if (f < 0) f = 0;
            wsrc = m.codes + f * m.row_words;
            ssrc = m.scales + f * m.ngrp;
            return live;
        };
        auto load_w = [&](int sb, uint32_t (&w)[BITS], u32x2 &s) {
            const int b = min(2 * sb + lg, p.NB - 1);
#pragma unroll
            for (int i = 0; i < BITS; ++i) w[i] = wsrc[b * BITS + i];
            s = *reinterpret_cast<const u32x2 *>(ssrc + b * 4);
        };
        f32x16h acc{};
        const int swz = ln & 15;
        // a superstep: each step's lookups and x are read during the step before;
        // the pins keep them there (left alone the compiler extracts every code
        // first and spills)
        auto compute = [&](int sb, int buf, uint32_t (&w)[BITS], u32x2 s) {
            if (2 * sb + lg >= p.NB) s = u32x2{0, 0};
            const h4 sc = __builtin_bit_cast(h4, s);
            const uint8_t *xb = xs + (buf * 2 + lg) * (kHalfTok * 256) + ln * 256;
            struct Ops { h8 e, x; };
            auto read = [&](int q, Ops &o) {
                o.e = step_entries<4, BITS>(w, q, tab, 0u, false);
                o.x = *reinterpret_cast<const h8 *>(xb + ((q ^ swz) << 4));
            };
            auto one = [&](int q, Ops &o, Ops &on) {
#pragma unroll
                for (int i = 0; i < BITS; ++i) asm volatile("" : "+v"(w[i]));
                if (q < 15) read(q + 1, on);
                __builtin_amdgcn_sched_barrier(0);
                const f16 c = sc[q / 4];
                const h8 wv = o.e * h8{c, c, c, c, c, c, c, c};
                acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(wv, o.x, acc, 0, 0, 0);
                asm volatile("" : "+v"(acc));
                __builtin_amdgcn_sched_barrier(0);
            };
            Ops a, b;
            read(0, a);
#pragma unroll
            for (int q = 0; q < 16; q += 2) {
                one(q, a, b);
                one(q + 1, b, a);
            }
        };
        // lane holds rows 8 j + 4 lg + i of token ln (register 4 j + i)
        auto store = [&](int k, uint32_t live) {
            if (yrow < 0) return;
            const int o0 = (xb0 + k) * kHalfRows + wave * 32;
            float *yr = y + int64_t(yrow) * p.OUT;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int r = 8 * j + 4 * lg, o = o0 + r;
                f32x4 v;
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] = ((live >> (r + i)) & 1) ? acc[4 * j + i] : 0.f;
                if (o + 3 < p.OUT && p.OUT % 4 == 0) {
                    *reinterpret_cast<f32x4 *>(yr + o) = v;
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (o + i < p.OUT) yr[o + i] = v[i];
                }
            }
        };

        uint32_t w[BITS], wn[BITS];
        u32x2 sc, sn;
        copy_x(0, 0);
        uint32_t live = rows_of(0), liven = live;
        load_w(0, w, sc);
        wait_vmem();
        __syncthreads();                        // the table too
        int buf = 0;
        for (int k = 0; k < nb; ++k) {
            const bool active = (xb0 + k) * kHalfRows + wave * 32 < p.OUT;
            for (int sb = 0; sb < NSS; ++sb) {
                // into the buffer of the superstep before, which every wave has
                // left; past the item's last superstep: loads nobody uses
                const int next = sb + 1 < NSS ? sb + 1 : 0;
                copy_x(next, buf ^ 1);
                asm volatile("" ::: "memory");
                if (next == 0 && k + 1 < nb) liven = rows_of(k + 1);
                load_w(next, wn, sn);
                asm volatile("" ::: "memory");
                if (active) compute(sb, buf, w, sc);    // a wave's own rows: uniform
                asm volatile("" ::: "memory");
                wait_vmem();
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
#pragma unroll
                for (int i = 0; i < BITS; ++i) w[i] = wn[i];
                sc = sn;
                buf ^= 1;
            }
            store(k, live);
            acc = f32x16h{};
            live = liven;
        }
        wait_vmem();                            // the last copy is in before its buffer is used again
        __syncthreads();
    }
}

int launch_half(const HalfParams &p, int bits, dim3 grid, hipStream_t st);

}  // namespace vqk
