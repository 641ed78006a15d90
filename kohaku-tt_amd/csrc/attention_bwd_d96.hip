// Attention backward gradient kernels for head dims padded to 96 (attention_bwd_tile.hpp).
#include "attention_bwd_tile.hpp"

namespace kmi {
namespace bwd {
template hipError_t launch_tile<bf16, 96>(const BwdParams&, const BwdGrid&, int, hipStream_t);
template hipError_t launch_tile<f16, 96>(const BwdParams&, const BwdGrid&, int, hipStream_t);
}  // namespace bwd
}  // namespace kmi
