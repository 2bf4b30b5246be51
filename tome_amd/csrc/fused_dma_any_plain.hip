// The DMA sweep on a token tile chosen on the device, log-probs and lse only.
#include "fused_dma.hpp"

namespace tome {
template void launch_dma_any<false, false>(const FusedArgs&, bool, bool, int, hipStream_t);
}  // namespace tome
