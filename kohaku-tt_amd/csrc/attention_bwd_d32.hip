// Attention backward gradient kernels for head dims padded to 32 (attention_bwd_tile.hpp).
#include "attention_bwd_tile.hpp"

namespace kmi {
namespace bwd {
template hipError_t launch_tile<bf16, 32>(const BwdParams&, const BwdGrid&, int, hipStream_t);
template hipError_t launch_tile<f16, 32>(const BwdParams&, const BwdGrid&, int, hipStream_t);
}  // namespace bwd
}  // namespace kmi
