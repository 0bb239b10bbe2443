// The forward scan kernels for bfloat16 I/O (see ss_fwd.hip).
#define SS_FWD_TYPE bf16_t
#include "ss_fwd.hip"
