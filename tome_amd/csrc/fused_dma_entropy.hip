// The DMA sweep on a token tile that the host knows, with the entropy.
#include "fused_dma.hpp"

namespace tome {
template bool launch_dma<true, false>(const FusedArgs&, int, bool, bool, int, hipStream_t);
}  // namespace tome
