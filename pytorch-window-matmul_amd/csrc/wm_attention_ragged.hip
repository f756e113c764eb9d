// The fused attention kernels for head widths that 16 does not divide: the sources of the plain widths with HeadWidth's
// piece arithmetic switched on, in translation units of their own so that they compile beside them.
#define RAGGED_WIDTH 1
#include "wm_attention.hip"
