// The backward scan kernels for bfloat16 I/O (see ss_bwd.hip).
#define SS_BWD_TYPE bf16_t
#include "ss_bwd.hip"
