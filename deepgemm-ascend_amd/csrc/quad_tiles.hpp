// Instantiation of the four-wave tile kernel over the tiles of one operand kind and layout.
#pragma once

#include "gemm_tiles.hpp"
#include "quad_kernel.hpp"

namespace dg {

template <int BM, int BN, int KIND, bool AMN, bool BMN>
KernelFn pick_quad_epi(int epi) {
    switch (epi) {
        case kEpiF32: return &quad_kernel<BM, BN, KIND, kEpiF32, AMN, BMN>;
        case kEpiBf16: return &quad_kernel<BM, BN, KIND, kEpiBf16, AMN, BMN>;
        case kEpiBf16SR: return &quad_kernel<BM, BN, KIND, kEpiBf16SR, AMN, BMN>;
        case kEpiFp8:
            if constexpr (KIND == kFP8FP8 && quad_fp8_output(BM, BN)) return &quad_kernel<BM, BN, KIND, kEpiFp8, AMN, BMN>;
            else return nullptr;
        default: return nullptr;
    }
}

template <int KIND, bool AMN, bool BMN, int I = 0>
KernelFn find_quad(int bm, int bn, int epi) {
    if constexpr (I == kNumTiles) {
        return nullptr;
    } else {
        constexpr TileCfg t = kTiles[I];
        if constexpr (quad_tile(KIND, t.bm, t.bn) && (t.bm <= 256 || (!AMN && !BMN))) {
            if (bm == t.bm && bn == t.bn) return pick_quad_epi<t.bm, t.bn, KIND, AMN, BMN>(epi);
        }
        return find_quad<KIND, AMN, BMN, I + 1>(bm, bn, epi);
    }
}

}  // namespace dg
