// generic_attention.hip for bf16 models (a unit of its own, so the model dtypes
// build in parallel).
#define GLLM_GENERIC_QT __bf16
#define GLLM_GENERIC_LAUNCH launch_generic_bf16
#include "generic_attention.hip"
