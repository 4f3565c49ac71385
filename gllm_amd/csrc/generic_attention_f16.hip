// generic_attention.hip for fp16 models (a unit of its own, so the model dtypes
// build in parallel).
#define GLLM_GENERIC_QT _Float16
#define GLLM_GENERIC_LAUNCH launch_generic_f16
#include "generic_attention.hip"
