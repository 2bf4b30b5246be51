// The DMA sweep on a token tile that the host knows, with the argmax.
#include "fused_dma.hpp"

namespace tome {
template bool launch_dma<false, true>(const FusedArgs&, int, bool, bool, int, hipStream_t);
}  // namespace tome
