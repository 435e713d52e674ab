// lgca_block_inst.hip -- instantiates the block kernels of one model kind and
// one number of rows per wave, or the batch's block kernel (all models) of one
// number of rows.  The build compiles this file once per instantiation, with
//   -DLGCA_INST_KIND=<0 HPP | 1 FHP-I | 2 FHP-II/III | -1 batch> -DLGCA_INST_M=<rows>.
#include "lgca_block.hpp"

#if !defined(LGCA_INST_KIND) || !defined(LGCA_INST_M)
#error "compile with -DLGCA_INST_KIND=<-1..2> -DLGCA_INST_M=<rows per wave>"
#endif

namespace lgca {

#if LGCA_INST_KIND >= 0
template hipError_t launch_block_km<LGCA_INST_KIND, LGCA_INST_M>(const BlockArgs&, uint32_t, uint32_t, bool, int,
                                                                 hipStream_t);
#else
template hipError_t launch_block_batch_m<LGCA_INST_M>(const BatchJob*, BatchState*, const WorkItem*, uint32_t,
                                                      uint32_t, uint32_t, bool, hipStream_t);
#endif

}  // namespace lgca
