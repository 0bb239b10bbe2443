// The forward scan kernels for float16 I/O (see ss_fwd.hip).
#define SS_FWD_TYPE _Float16
#include "ss_fwd.hip"
