// Attention forward tile kernels for head dims padded to 128 (attention_tile.hpp).
#include "attention_tile.hpp"

namespace kmi {
namespace fwd {
template hipError_t launch_tile<bf16, 128>(const AttnParams&, int, hipStream_t);
template hipError_t launch_tile<f16, 128>(const AttnParams&, int, hipStream_t);
}  // namespace fwd
}  // namespace kmi
