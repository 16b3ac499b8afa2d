// Four-wave tile kernel, bf16: B MN-major.
#include "quad_tiles.hpp"

namespace dg {
KernelFn lookup_quad_bf16_mn_b(int bm, int bn, int epi) { return find_quad<kBF16, false, true>(bm, bn, epi); }
}  // namespace dg
