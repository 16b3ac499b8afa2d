// Four-wave tile kernel, e4m3: B MN-major.
#include "quad_tiles.hpp"

namespace dg {
KernelFn lookup_quad_fp8_mn_b(int bm, int bn, int epi) { return find_quad<kFP8FP8, false, true>(bm, bn, epi); }
}  // namespace dg
