// Four-wave tile kernel, e4m3: both operands MN-major.
#include "quad_tiles.hpp"

namespace dg {
KernelFn lookup_quad_fp8_mn_ab(int bm, int bn, int epi) { return find_quad<kFP8FP8, true, true>(bm, bn, epi); }
}  // namespace dg
