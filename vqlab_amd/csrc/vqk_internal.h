// Host-side helpers shared between libvqk translation units.
#pragma once

#include <string.h>

#include "vqk_gemv.h"

namespace vqk {

// Fills the weight-dependent fields of a GEMV parameter block.
int gemv_fill_params(const vqk_weights *w, const Geom &g, GemvParams *p);

// Dynamic LDS bytes of the fast GEMV kernel for geometry g (xf: the wide-x
// instances).
size_t gemv_fast_lds(const Geom &g, bool xf = false);

// Validates and launches the fused GEMV for N = T * xkrep pairs.
// ws: scratch for one linear's few-row kernel, or NULL (launch_lin).
int launch_gemv(const vqk_weights *w, const void *x, int32_t x_type, int64_t T,
                const uint32_t *eidx, int64_t N, int64_t xkrep, void *y, int32_t y_type,
                void *ws, size_t ws_bytes, hipStream_t st);

// The few-row linear kernel (vqk_lin.h) for N rows of one linear: whether it
// takes the module and x (xf: x unrounded, VQK_X_KEEP), and its launch.
bool lin_ok(const vqk_weights *w, const Geom &g, const void *x, int32_t x_type, bool xf, int64_t N);
// ... and whether it is the faster one for a module that the fast GEMV (wide: x
// enters as fp32) or the segment kernel takes too.
bool lin_beats_gemv(const Geom &g, bool wide, int64_t N);
bool lin_beats_seg(const Geom &g, int64_t N);
int launch_lin(const vqk_weights *w, const Geom &g, const void *x, int32_t x_type, bool xf, bool deq,
               int64_t N, void *y, int32_t y_type, void *ws, size_t ws_bytes, hipStream_t st);

// Workspace that launch_lin makes use of for N rows: the copy of x in the
// matrix cores' operand order. With less (or none) it reads x in place.
constexpr int64_t kLinFragRows = 64;
size_t lin_frag_bytes(const vqk_weights *w, const Geom &g, int64_t N);

// min(items, the current device's CU count): the grid of a kernel that
// keeps one workgroup per CU (vqk_big.hip).
int big_grid(int64_t items);

// ---- grouped expert GEMM pieces (vqk_gemm.hip): sort one routing, then run
// several projections over it with the register-decode segment kernel.
struct SegCall {
    const void *x;             // activations (x_type), or NULL with xg / xu:
    int32_t x_type;
    const float *xg, *xu;      //   row = fp16(silu(xg) * xu), fp32 rows of the module's IN
    int64_t xkrep;             // x row of pair n = n / xkrep
    void *y;                   // y[pair, OUT] in y_type
    int32_t y_type;
    int64_t N;                 // pairs (sorted) or dense rows (sort_ws == NULL)
    int32_t tok;               // sorted: the sort's tile rows (seg_tile_rows); 0 = 16
    int32_t ksplit;            // dense rows only: K slices, y holds ksplit fp32 partials
                               //   [ksplit][N][OUT] (0 or 1: no split)
    int32_t xparts;            // xg / xu hold xparts partial rows [xparts][N][IN] to add
};

// Rows per tile to sort N pairs into for module `w` over E experts:
// kSegTokNarrow when the routing puts at most ~2 pairs on an expert on
// average and w's d8 table is beyond LDS (more of it fits beside a narrow x
// chunk; the sort then picks 4- or 8-row tiles on device), else 16.
int seg_tile_rows(const vqk_weights *w, int64_t N, int64_t E);

// K slices for the segment kernel over N dense rows of `w`: enough that the
// launch fills the CUs once (at most 4 and the module's supersteps).
int seg_ksplit(const vqk_weights *w, int64_t N);

// Workspace of seg_sort for N pairs over E experts.
size_t seg_sort_bytes(int64_t N, int64_t E);

// True when the segment kernel takes module `w` for N pairs.
bool seg_ok(const vqk_weights *w, int64_t N);

// Counting sort of N pair experts (device uint32, out-of-range ids form dead
// tiles) into `ws`: pair order, records of tiles of at most `tok` rows (16
// or 4) and the tile count.
int seg_sort(const uint32_t *eidx, int64_t N, int64_t E, int tok, void *ws, hipStream_t st);

// One projection over a routing sorted into `sort_ws` (or over N dense rows
// of expert 0 when sort_ws is NULL).
int seg_run(const vqk_weights *w, const SegCall &c, const void *sort_ws, hipStream_t st);

// ---- many rows per expert (vqk_wide.h): gate and up at once into fp16 SwiGLU
// rows in sorted order, then down over those rows.
struct WideCall {
    const uint16_t *x;         // fp16 rows, 16-byte aligned
    int64_t xkrep;             // x row of pair n = n / xkrep; 0: x rows are in sorted order
    void *y;                   // pair of projections: fp16 [N, OUT] in sorted order; one: y[pair, OUT]
    int32_t y_type;
    int64_t N;                 // pairs (sorted) or dense rows (sort_ws == NULL)
    int32_t tok;               // the sort's tile rows (wide_tile_rows)
};

// Rows per tile to sort a routing of N pairs into for the projections of a layer,
// or 0 when the wide kernel does not take them.
int wide_tile_rows(const vqk_weights *gate, const vqk_weights *up, const vqk_weights *down, int64_t N);
// Whether the wide kernel is the faster one for N pairs over gate's experts (and
// a shared one).
bool wide_pays(const vqk_weights *gate, bool shared, int64_t N);
// `up`: with it, SwiGLU of (w, up). sort_ws: the sorted routing, or NULL for
// dense rows of one expert.
int wide_run(const vqk_weights *w, const vqk_weights *up, const WideCall &c, const void *sort_ws,
             hipStream_t st);
// ---- d8 tables beyond LDS, halved by entry columns (vqk_half.h): gate and up
// in one launch, or one projection, into half sums.
struct HalfCall {
    const uint16_t *x;         // fp16 half columns [2][rows, IN / 2], 16-byte aligned
    int64_t xkrep;             // x row of pair n = n / xkrep; 0: x rows are in sorted order
    float *y[2][2];            // [projection][half] fp32 [N, OUT]
    bool ysorted;              // y rows in sorted order, not by pair
    int64_t N;                 // pairs (sorted) or dense rows (sort_ws == NULL)
};
// True when the half-entry kernel takes every projection of a layer for N pairs.
bool half_ok(const vqk_weights *gate, const vqk_weights *up, const vqk_weights *down, int64_t N);
// `up`: with it, both projections. sort_ws: the routing sorted into tiles of
// kHalfTile rows, or NULL for dense rows of one expert.
constexpr int kHalfTile = 32;
int half_run(const vqk_weights *w, const vqk_weights *up, const HalfCall &c, const void *sort_ws,
             hipStream_t st);
// fp16 half columns of n (a multiple of 8) activations, 16-byte aligned, or of
// SwiGLU rows from half sums.
int launch_x_split(const void *x, int x_type, int64_t n, uint16_t *out, hipStream_t st);
int launch_swiglu_split(const float *g0, const float *g1, const float *u0, const float *u1, int64_t n,
                        uint16_t *out, hipStream_t st);
// fp16 copy of n (a multiple of 8) activations; both 16-byte aligned.
int launch_x_half(const void *x, int x_type, int64_t n, uint16_t *out, hipStream_t st);

}  // namespace vqk
