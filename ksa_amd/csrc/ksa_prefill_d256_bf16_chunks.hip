// Prefill kernel, head_dim 256, bf16, chunk tiles: a translation unit of its own
// (see the head of ksa_prefill.hip).
#define KSA_PREFILL_UNIT 7
#include "ksa_prefill.hip"
