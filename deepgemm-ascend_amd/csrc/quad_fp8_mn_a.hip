// Four-wave tile kernel, e4m3: A MN-major.
#include "quad_tiles.hpp"

namespace dg {
KernelFn lookup_quad_fp8_mn_a(int bm, int bn, int epi) { return find_quad<kFP8FP8, true, false>(bm, bn, epi); }
}  // namespace dg
