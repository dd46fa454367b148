// One translation unit per (element type, mask source, tile hand-out) of the block-sparse forward, so that the
// variants compile in parallel: built with -DSA_FWD_DT={0,1} (bf16, fp16), -DSA_FWD_PK={0,1} (bool mask,
// bit-packed PARTIAL tiles) and -DSA_FWD_HOW={0,1,2,3,4,5} (one workgroup per Q tile, persistent workgroups, lists shared by
// several workgroups, ragged sizes (with packed tiles only), lists in two halves,
// lists with assistants).
#include "sparse_fwd_kernel.h"

#if !defined(SA_FWD_DT) || !defined(SA_FWD_PK) || !defined(SA_FWD_HOW)
#error "compile with -DSA_FWD_DT=<0|1> -DSA_FWD_PK=<0|1> -DSA_FWD_HOW=<0|1|2|3|4|5>"
#endif

namespace sa {
template hipError_t launch_fwd_variant<SA_FWD_DT, (SA_FWD_PK != 0), SA_FWD_HOW>(const FwdParams &, int, int,
                                                                                      hipStream_t);
}  // namespace sa
