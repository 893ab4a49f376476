// k_lin instances for d = 4 over x in operand order (the widths of
// vqk_lin_d4.hip), and the copy that makes it.
#include "vqk_lin.h"

namespace vqk {

int launch_lin_frag_d4(const LinParams &p0, int bits, void *frag, hipStream_t st) {
    LinParams p = p0;
    const int nt = lin_row_tiles(p.N), nss = (p.NB + 3) / 4;
    const int64_t pieces = int64_t((p.N + 16 * nt - 1) / (16 * nt)) * nss * (4 * 4) * nt * 64;
    hipLaunchKernelGGL(k_lin_frag<4>, dim3(unsigned((pieces + 255) / 256)), dim3(256), 0, st, p.x, p.x_type,
                       p.N, p.IN, nss, nt, static_cast<u32x4 *>(frag));
    int rc = hip_status(hipGetLastError(), "operand copy launch");
    if (rc) return rc;
    p.x = frag;
    switch (bits) {
        case 8: return go_lin<4, 8, 2, kXFrag>(p, st);
        case 9: return go_lin<4, 9, 2, kXFrag>(p, st);
        case 10: return go_lin<4, 10, 2, kXFrag>(p, st);
        case 11: return go_lin<4, 11, 2, kXFrag>(p, st);
        case 12: return go_lin<4, 12, 2, kXFrag>(p, st);
        case 13: return go_lin<4, 13, 2, kXFrag>(p, st);
        case 14: return go_lin<4, 14, 2, kXFrag>(p, st);
        case 16: return go_lin<4, 16, 2, kXFrag>(p, st);
        default: return set_error(VQK_ENOTIMPL, "no linear kernel for d=4 bits=%d", bits);
    }
}

}  // namespace vqk
