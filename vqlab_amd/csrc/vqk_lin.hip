// Host side of the few-row linear kernel (vqk_lin.h): what it takes and its
// launch.
#include "vqk_internal.h"
#include "vqk_lin.h"

namespace vqk {

// The B operand form of x, or -1: fp16 enters as it is; bf16 / fp32 rounded
// to fp16, or (xf) as fp32, which only the d8 instances have.
static int lin_x_mode(int32_t D, int32_t x_type, bool xf) {
    if (x_type == VQK_F16) return kXF16;
    if (xf) return D != 8 ? -1 : (x_type == VQK_BF16 ? kXBF16x : kXF32x);
    return x_type == VQK_BF16 ? kXBF16r : kXF32r;
}

bool lin_ok(const vqk_weights *w, const Geom &g, const void *x, int32_t x_type, bool xf, int64_t N) {
    const bool bits = g.D == 2 ? (g.BITS >= 8 && g.BITS <= 12)
                               : ((g.BITS >= 8 && g.BITS <= 14) || g.BITS == 16);
    return g.E == 1 && N > 0 && g.G == 64 && bits && g.row_words > 0 && g.rows > 0 &&
           lin_x_mode(g.D, x_type, xf) >= 0 && g.OUT <= INT32_MAX && g.NB * g.BITS <= INT32_MAX &&
           (reinterpret_cast<uintptr_t>(w->codebook) & 15) == 0 &&
           (reinterpret_cast<uintptr_t>(w->codes) & 3) == 0 && (reinterpret_cast<uintptr_t>(x) & 15) == 0 &&
           N <= 16 * 65535 &&                                             // grid.y
           N <= (int64_t(1) << 31) / (g.IN * act_size(x_type));      // x as one buffer of <= 2 GB
}

// Against the GEMV, which decodes every weight once per row but has no K loop
// to start and end: the products from which the few-row kernel is ahead, by
// what bounds the GEMV there. us per call, GEMV / this kernel (MI355X, graph
// replays), the last size that stays and the first that goes:
//   d2            20e6  4096 -> 1024: 4 rows 6.0 / 7.0, 5 rows 7.0 / 7.0
//   d4            40e6  4096 -> 4096, K4096: 2 rows 7.6 / 7.6, 3 rows 10 / 7.6
//   d8 fp16 x     70e6  4096 -> 4096, K4096: 4 rows 12 / 9; 30e6 with a table
//                       beyond LDS: 4096 -> 4096, K16384: 2 rows 12 / 13
//   d8 wide x     90e6  4096 -> 4096, K4096: 4 rows 15.5 / 17, 8 rows 25 / 17,
//                       and more than two rows (5120 -> 17408: 2 rows 53 / 62);
//                       40e6 with a table beyond LDS
// Over 14 sizes from 1024 -> 512 to 5120 -> 17408 and 2..32 rows of 9 formats
// the rule is within 20 % of the better of the two, most often with it; always
// taking this kernel cost up to 3x (1024 -> 1024, d8 K4096: 5.5 against 16).
bool lin_beats_gemv(const Geom &g, bool wide, int64_t N) {
    const bool lds = cb_in_lds(g.D, g.BITS);
    if (wide && lds && N <= 2) return false;
    const int64_t from = g.D == 2 ? 20000000 : g.D == 4 ? 40000000
                       : lds ? (wide ? 90000000 : 70000000) : (wide ? 40000000 : 30000000);
    return N * g.OUT >= (from + g.IN - 1) / g.IN;
}

// Against the segment kernel, which decodes once per 16 rows with one workgroup
// to 128 weight rows and no K slices: it stays ahead over few supersteps, where
// the slices have nothing to share, and where its workgroups fill the chip in
// one round while this kernel's 64-row tile is part empty. us, segment / this:
//   d4 K4096: 1024 -> 4096 (2 supersteps) 33 rows 9.0 / 9.5; 2048 -> 2048 (4) 14 / 10;
//             5120 -> 17408 (136 workgroups to 16 rows) 33 rows 39 / 48, 49 rows 61 / 48
//   d4 K8192 (one workgroup to a CU): 3072 -> 9216 (216 workgroups) 33 rows 20 / 23
//   d8 K4096: 2048 -> 2048 (2) 33 rows 11 / 14; 5120 -> 17408 16 rows 21 / 23, 33 rows 43 / 50
//   d8 K16384, K65536: 2048 -> 2048 (2) 8 rows 19 / 14, 64 rows 18 / 22
bool lin_beats_seg(const Geom &g, int64_t N) {
    const int64_t nss = (g.NB + 3) / 4, wgs = (g.OUT + 127) / 128 * ((N + 15) / 16);
    const bool part_empty = N > 32 && N <= 48 && wgs >= 200;
    if (g.D == 2) return !(part_empty && nss <= 4);
    if (g.D == 8 && N <= 16 && wgs >= 128) return false;
    // two of the segment kernel's workgroups to a CU, or a d8 table in LDS
    if (cb_in_lds(g.D, g.BITS) && (g.D == 8 || (int64_t(1) << g.BITS) * g.D * 2 <= 32 * 1024))
        return nss > 2 && !part_empty;
    if (g.D == 4 && part_empty && wgs <= 256) return false;
    return nss > (N > 32 || g.D == 4 ? 2 : 1) || wgs >= 256;
}

// The copy pays from about 2^28 products on: below, its launch costs more (3 us
// on the GPU, 5 for a caller that waits on the host) than the direct loads
// lose (0.2 us per million weights and 16 rows: 17 us at 5120 -> 17408).
constexpr int64_t kLinFragWork = int64_t(1) << 28;

size_t lin_frag_bytes(const vqk_weights *w, const Geom &g, int64_t N) {
    if (N <= kLinDirectRows || N > kLinFragRows || !lin_ok(w, g, nullptr, VQK_F16, false, N) ||
        g.OUT * g.IN < kLinFragWork / N)
        return 0;
    const int64_t rows = 16 * lin_row_tiles(N);
    return size_t((N + rows - 1) / rows * rows) * size_t((g.NB + 3) / 4 * 4 * kBlock * g.D) * 2;
}

int launch_lin(const vqk_weights *w, const Geom &g, const void *x, int32_t x_type, bool xf, bool deq,
               int64_t N, void *y, int32_t y_type, void *ws, size_t ws_bytes, hipStream_t st) {
    LinParams p;
    memset(&p, 0, sizeof p);
    p.codes = static_cast<const uint32_t *>(w->codes);
    p.row_words = g.row_words;
    p.codebook = w->codebook;
    p.K = int32_t(g.K);
    p.scales = w->scales;
    p.ngrp = int32_t(g.NGRP);
    p.row_table = w->row_table;
    p.stored_rows = g.rows;
    p.OUT = int32_t(g.OUT);
    p.IN = int32_t(g.IN);
    p.NB = int32_t(g.NB);
    p.x = x;
    p.y = y;
    p.y_type = y_type;
    p.N = int32_t(N);
    p.x_type = x_type;
    p.deq = deq;
    const int xm = lin_x_mode(g.D, x_type, xf);
    const size_t fb = xm == kXBF16x || xm == kXF32x ? 0 : lin_frag_bytes(w, g, N);
    if (fb && ws && ws_bytes >= fb &&
        (reinterpret_cast<uintptr_t>(ws) & 15) == 0) {
        switch (g.D) {
            case 2: return launch_lin_frag_d2(p, g.BITS, ws, st);
            case 4: return launch_lin_frag_d4(p, g.BITS, ws, st);
            default: return launch_lin_frag_d8(p, g.BITS, ws, st);
        }
    }
    switch (g.D) {
        case 2: return launch_lin_d2(p, g.BITS, xm, st);
        case 4: return launch_lin_d4(p, g.BITS, xm, st);
        default: return launch_lin_d8(p, g.BITS, xm, st);
    }
}

}  // namespace vqk
