// Four-wave tile kernel, bf16: A MN-major.
#include "quad_tiles.hpp"

namespace dg {
KernelFn lookup_quad_bf16_mn_a(int bm, int bn, int epi) { return find_quad<kBF16, true, false>(bm, bn, epi); }
}  // namespace dg
