// The DMA sweep on a token tile chosen on the device, with the entropy.
#include "fused_dma.hpp"

namespace tome {
template void launch_dma_any<true, false>(const FusedArgs&, bool, bool, int, hipStream_t);
}  // namespace tome
