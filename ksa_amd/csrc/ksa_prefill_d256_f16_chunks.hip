// Prefill kernel, head_dim 256, fp16, chunk tiles: a translation unit of its own
// (see the head of ksa_prefill.hip).
#define KSA_PREFILL_UNIT 8
#include "ksa_prefill.hip"
