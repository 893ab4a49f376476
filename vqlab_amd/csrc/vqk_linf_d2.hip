// k_lin instances for d = 2 over x in operand order (the widths of
// vqk_lin_d2.hip), and the copy that makes it.
#include "vqk_lin.h"

namespace vqk {

int launch_lin_frag_d2(const LinParams &p0, int bits, void *frag, hipStream_t st) {
    LinParams p = p0;
    const int nt = lin_row_tiles(p.N), nss = (p.NB + 3) / 4;
    const int64_t pieces = int64_t((p.N + 16 * nt - 1) / (16 * nt)) * nss * (4 * 2) * nt * 64;
    hipLaunchKernelGGL(k_lin_frag<2>, dim3(unsigned((pieces + 255) / 256)), dim3(256), 0, st, p.x, p.x_type,
                       p.N, p.IN, nss, nt, static_cast<u32x4 *>(frag));
    int rc = hip_status(hipGetLastError(), "operand copy launch");
    if (rc) return rc;
    p.x = frag;
    switch (bits) {
        case 8: return go_lin<2, 8, 1, kXFrag>(p, st);
        case 9: return go_lin<2, 9, 1, kXFrag>(p, st);
        case 10: return go_lin<2, 10, 1, kXFrag>(p, st);
        case 11: return go_lin<2, 11, 1, kXFrag>(p, st);
        case 12: return go_lin<2, 12, 1, kXFrag>(p, st);
        default: return set_error(VQK_ENOTIMPL, "no linear kernel for d=2 bits=%d", bits);
    }
}

}  // namespace vqk
