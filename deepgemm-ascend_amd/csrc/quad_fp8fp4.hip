// Four-wave tile kernel, e4m3 x e2m1.
#include "quad_tiles.hpp"

namespace dg {
KernelFn lookup_quad_fp8fp4(int bm, int bn, int epi) { return find_quad<kFP8FP4, false, false>(bm, bn, epi); }
}  // namespace dg
