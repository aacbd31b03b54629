// k_move_gather from elements of 1 byte.
#include "move_gather.h"

namespace mrl {
template hipError_t launch_move_gather<1>(const MoveTile &, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t, hipStream_t);
}  // namespace mrl
