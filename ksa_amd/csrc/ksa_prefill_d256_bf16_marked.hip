// Prefill kernel, head_dim 256, bf16, marked tile addressing: a translation unit of its own
// (see the head of ksa_prefill.hip).
#define KSA_PREFILL_UNIT 3
#include "ksa_prefill.hip"
