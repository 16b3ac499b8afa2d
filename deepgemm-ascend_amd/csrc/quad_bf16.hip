// Four-wave tile kernel, bf16: K-major operands.
#include "quad_tiles.hpp"

namespace dg {
KernelFn lookup_quad_bf16(int bm, int bn, int epi) { return find_quad<kBF16, false, false>(bm, bn, epi); }
}  // namespace dg
