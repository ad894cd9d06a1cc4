// Prefill kernel, head_dim 64 and 128, chunk tiles, with their entry point: a translation unit of its own
// (see the head of ksa_prefill.hip).
#define KSA_PREFILL_UNIT 9
#include "ksa_prefill.hip"
