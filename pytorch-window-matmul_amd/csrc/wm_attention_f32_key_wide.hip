// The float32 attention key kernel for heads wider than 96, in a translation unit of its own for its compiler option.
#define F32_KEY_WIDE 1
#include "wm_attention_f32.hip"
