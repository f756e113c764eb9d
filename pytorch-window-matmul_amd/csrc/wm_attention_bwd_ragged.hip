// Backward of the fused attention for head widths that 16 does not divide, see wm_attention_ragged.hip.
#define RAGGED_WIDTH 1
#include "wm_attention_bwd.hip"
