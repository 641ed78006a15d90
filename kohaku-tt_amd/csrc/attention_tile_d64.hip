// Attention forward tile kernels for head dims padded to 64 (attention_tile.hpp).
#include "attention_tile.hpp"

namespace kmi {
namespace fwd {
template hipError_t launch_tile<bf16, 64>(const AttnParams&, int, hipStream_t);
template hipError_t launch_tile<f16, 64>(const AttnParams&, int, hipStream_t);
}  // namespace fwd
}  // namespace kmi
