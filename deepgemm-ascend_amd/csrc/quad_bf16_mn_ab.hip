// Four-wave tile kernel, bf16: both operands MN-major.
#include "quad_tiles.hpp"

namespace dg {
KernelFn lookup_quad_bf16_mn_ab(int bm, int bn, int epi) { return find_quad<kBF16, true, true>(bm, bn, epi); }
}  // namespace dg
