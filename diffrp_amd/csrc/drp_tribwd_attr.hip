// Deterministic backward of interpolate: the ATTR instances of the tile passes.
#include "drp_tribwd.h"

namespace drp {

int launch_tri_bwd_attr(const TriBwdLaunch &L, int C, hipStream_t st) {
    if (L.n_diff > 0) {  // with derivative gradients: three staged rows per quad, up to 4 channels a pass
        switch (C) {
            case 1: launch_tiles<1, 1, true>(L, st); break;
            case 2: launch_tiles<1, 2, true>(L, st); break;
            case 3: launch_tiles<1, 3, true>(L, st); break;
            case 4: launch_tiles<1, 4, true>(L, st); break;
            default: return -1;
        }
        return hipGetLastError() == hipSuccess ? 0 : -2;
    }
    switch (C) {
        case 1: launch_tiles<1, 1, false>(L, st); break;
        case 2: launch_tiles<1, 2, false>(L, st); break;
        case 3: launch_tiles<1, 3, false>(L, st); break;
        case 4: launch_tiles<1, 4, false>(L, st); break;
        case 5: launch_tiles<1, 5, false>(L, st); break;
        case 6: launch_tiles<1, 6, false>(L, st); break;
        case 7: launch_tiles<1, 7, false>(L, st); break;
        case 8: launch_tiles<1, 8, false>(L, st); break;
        case 9: launch_tiles<1, 9, false>(L, st); break;
        case 10: launch_tiles<1, 10, false>(L, st); break;
        case 11: launch_tiles<1, 11, false>(L, st); break;
        case 12: launch_tiles<1, 12, false>(L, st); break;
        case 13: launch_tiles<1, 13, false>(L, st); break;
        case 14: launch_tiles<1, 14, false>(L, st); break;
        case 15: launch_tiles<1, 15, false>(L, st); break;
        case 16: launch_tiles<1, 16, false>(L, st); break;
        default: return -1;
    }
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

}  // namespace drp
