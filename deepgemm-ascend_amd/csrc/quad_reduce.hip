// Second launch of split-K plans on the four-wave tile kernel.
#include "gemm_tiles.hpp"
#include "quad_kernel.hpp"

namespace dg {
KernelFn lookup_quad_reduce(int epi) {
    switch (epi) {
        case kEpiF32: return &quad_reduce_kernel<kEpiF32>;
        case kEpiBf16: return &quad_reduce_kernel<kEpiBf16>;
        case kEpiBf16SR: return &quad_reduce_kernel<kEpiBf16SR>;
        case kEpiFp8: return &quad_reduce_kernel<kEpiFp8>;
        default: return nullptr;
    }
}
}  // namespace dg
