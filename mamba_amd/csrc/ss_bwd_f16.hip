// The backward scan kernels for float16 I/O (see ss_bwd.hip).
#define SS_BWD_TYPE _Float16
#include "ss_bwd.hip"
