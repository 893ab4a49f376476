// k_lin instances for d = 4: the code widths that artifacts use (8 and 16 also
// serve unpacked uint8 / uint16 rows), scale groups of 64 columns.
#include "vqk_lin.h"

namespace vqk {

namespace {
template <int BITS>
int go(const LinParams &p, int xm, hipStream_t st) {
    switch (xm) {
        case kXF16: return go_lin<4, BITS, 2, kXF16>(p, st);
        case kXBF16r: return go_lin<4, BITS, 2, kXBF16r>(p, st);
        case kXF32r: return go_lin<4, BITS, 2, kXF32r>(p, st);
        default: return set_error(VQK_ENOTIMPL, "no linear kernel for d=4, x mode %d", xm);
    }
}
}  // namespace

int launch_lin_d4(const LinParams &p, int bits, int xm, hipStream_t st) {
    switch (bits) {
        case 8: return go<8>(p, xm, st);
        case 9: return go<9>(p, xm, st);
        case 10: return go<10>(p, xm, st);
        case 11: return go<11>(p, xm, st);
        case 12: return go<12>(p, xm, st);
        case 13: return go<13>(p, xm, st);
        case 14: return go<14>(p, xm, st);
        case 16: return go<16>(p, xm, st);
        default: return set_error(VQK_ENOTIMPL, "no linear kernel for d=4 bits=%d", bits);
    }
}

}  // namespace vqk
