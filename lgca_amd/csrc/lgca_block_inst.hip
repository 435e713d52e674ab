// lgca_block_inst.hip -- instantiates the block kernels of one model kind
// (LGCA_INST_KIND) and one number of rows per wave (LGCA_INST_M).
#include "lgca_block.hpp"

namespace lgca {

template hipError_t launch_block_km<LGCA_INST_KIND, LGCA_INST_M>(const BlockArgs&, uint32_t, uint32_t, bool, int,
                                                                 hipStream_t);

}  // namespace lgca
