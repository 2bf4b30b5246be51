// The DMA sweep on a token tile that the host knows, log-probs and lse only.
#include "fused_dma.hpp"

namespace tome {
template bool launch_dma<false, false>(const FusedArgs&, int, bool, bool, int, hipStream_t);
bool dma_allow_deep_lds() { return allow_big_lds(&fused_lmhead_dma_kernel<false, false, 0, true, false>, dma_lds_bytes(256, true)); }
}  // namespace tome
