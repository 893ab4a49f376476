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

// The copy pays from about 2^28 products on: below, its launch costs more (3 us
// on the GPU, 5 for a caller that waits on the host) than the direct loads
// lose (0.3 us per million weights and 16 rows: 26 us at 5120 -> 17408).
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
