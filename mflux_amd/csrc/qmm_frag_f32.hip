// The instantiations of the two-kernel path's GEMM (qmm_frag.hip) whose results are
// float32.
#define MFQ_FRAG_F32 1
#include "qmm_frag.hip"
