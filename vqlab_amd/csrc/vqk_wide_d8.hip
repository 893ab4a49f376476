// k_wide instances for d = 8: tables of up to 64 KB, scale groups of 64 columns.
#include "vqk_wide.h"

namespace vqk {

namespace {
template <int BITS>
int go(const WideParams &p, bool pair, dim3 grid, hipStream_t st) {
    if (pair)
        return launch_with_lds<k_wide<8, BITS, 4, true>>(grid, dim3(512), wide_lds(8, BITS, true), st, p);
    return launch_with_lds<k_wide<8, BITS, 4, false>>(grid, dim3(512), wide_lds(8, BITS, false), st, p);
}
}  // namespace

int launch_wide_d8(const WideParams &p, int bits, bool pair, dim3 grid, hipStream_t st) {
    switch (bits) {
        case 8: return go<8>(p, pair, grid, st);
        case 9: return go<9>(p, pair, grid, st);
        case 10: return go<10>(p, pair, grid, st);
        case 11: return go<11>(p, pair, grid, st);
        case 12: return go<12>(p, pair, grid, st);
        default: return set_error(VQK_ENOTIMPL, "no wide segment kernel for d=8 bits=%d", bits);
    }
}

}  // namespace vqk
