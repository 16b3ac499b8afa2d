// Four-wave tile kernel, e4m3: K-major operands.
#include "quad_tiles.hpp"

namespace dg {
KernelFn lookup_quad_fp8(int bm, int bn, int epi) { return find_quad<kFP8FP8, false, false>(bm, bn, epi); }
}  // namespace dg
