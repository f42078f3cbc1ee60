// Deterministic backward of interpolate and of the rasterize call behind it in
// one pass: the BOTH instances of the tile passes.
#include "drp_tribwd.h"

namespace drp {

int launch_tri_bwd_fused(const TriBwdLaunch &L, int C, hipStream_t st) {
    switch (C) {
        case 1: launch_tiles<2, 1, false>(L, st); break;
        case 2: launch_tiles<2, 2, false>(L, st); break;
        case 3: launch_tiles<2, 3, false>(L, st); break;
        case 4: launch_tiles<2, 4, false>(L, st); break;
        case 5: launch_tiles<2, 5, false>(L, st); break;
        case 6: launch_tiles<2, 6, false>(L, st); break;
        case 7: launch_tiles<2, 7, false>(L, st); break;
        case 8: launch_tiles<2, 8, false>(L, st); break;
        case 9: launch_tiles<2, 9, false>(L, st); break;
        case 10: launch_tiles<2, 10, false>(L, st); break;
        case 11: launch_tiles<2, 11, false>(L, st); break;
        case 12: launch_tiles<2, 12, false>(L, st); break;
        case 13: launch_tiles<2, 13, false>(L, st); break;
        case 14: launch_tiles<2, 14, false>(L, st); break;
        case 15: launch_tiles<2, 15, false>(L, st); break;
        case 16: launch_tiles<2, 16, false>(L, st); break;
        default: return -1;
    }
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

}  // namespace drp
