// The DMA sweep on a token tile chosen on the device, with the argmax.
#include "fused_dma.hpp"

namespace tome {
template void launch_dma_any<false, true>(const FusedArgs&, bool, bool, int, hipStream_t);
}  // namespace tome
