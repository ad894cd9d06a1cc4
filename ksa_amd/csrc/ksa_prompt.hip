// The head of a prefill in one launch (gfx950): a prompt's token ids with the summary tokens behind every whole chunk,
// the mask of their places, and the rotary rows of all positions
//   examples/pretrain/hf_template/modeling_qwen3sa.py:1080-1177 (_expand_input_with_summary_tokens) and
//   :1018-1032 (Qwen3RotaryEmbedding.forward: angles in fp32, cos and sin rounded to the 16-bit type).
// Everything is a closed form of the slot number.  As torch operations these were some forty launches over a few
// KB each, with two host synchronisations among them that kept the host from queueing the layers; with the rows of the cache
// layout as closed forms too (ksa_copy_rows_runs: one launch a layer for six) a prefill of 4 layers of the 4B shape has
// 44 launches for 125 and none of these waits: 100 / 400 / 1500 / 2 x 3000 tokens 1323 / 1676 / 2538 / 5843 -> 830 / 1049 /
// 1882 / 5256 us.  What bounds this launch is its own latency (7 us: one trip to memory, then eight sines and
// cosines a thread); eight angles a thread fill the 16-byte stores.
// The same for a stretch of slots, with which the decode steps get their rows: left to torch, which the prefill no longer calls for
// them, the first step and the first one at a chunk's end loaded its kernels in the middle of a generation (4 layers of the 4B shape, a
// fresh process: first step 49 ms, first chunk end 30, without recordings 27 and 44; like this 25 and 1.3, 16 and 1.2).
#include <hip/hip_runtime.h>

#include "ksa_api_internal.h"
#include "ksa_cvt.h"

namespace {

struct PromptParams {
    const long long* ids;     // [batch][n], rows ids_rs apart
    long long ids_rs;
    const float* inv_freq;    // [D / 2]
    long long* out_ids;       // [batch][L], or null
    uint16_t *cos, *sin;      // [L][D], rows rope_rs apart
    uint8_t* is_summary;      // [L], or null
    long long summary_begin, rope_rs;
    int slot0, text0;         // first slot, and the place in the text of ids[0]
    int batch, C, S, L, lanes;  // lanes = D / 16: threads per slot, eight angles each
    int inner_chunk;            // text positions start again at every chunk
    int summary_kind;           // 0: position 0, 1 / 2: left / right end of the token's slice of the chunk
};

template <typename T>
__global__ __launch_bounds__(256) void ksa_expand_prompt_kernel(const PromptParams p) {
    using Cv = KsaCvt<T>;
    const unsigned t = blockIdx.x * 256u + threadIdx.x;
    const int i_slot = (int)(t / (unsigned)p.lanes), lane = (int)(t % (unsigned)p.lanes);
    if (i_slot >= p.L) return;
    const int B = p.C + p.S, slot = p.slot0 + i_slot;
    const int chunk = slot / B, off = slot - chunk * B;
    const bool summary = off >= p.C;
    int pos;
    if (summary) {
        const int k = off - p.C + (p.summary_kind == 2 ? 1 : 0);
        const int first = chunk * p.C;
        pos = p.summary_kind == 0 ? 0 : max(first + (int)((long long)k * p.C / p.S) - 1, first);
    } else {
        pos = p.inner_chunk ? off : chunk * p.C + off;
    }
    if (p.out_ids) {
        for (int b = lane; b < p.batch; b += p.lanes)
            p.out_ids[(long long)b * p.L + i_slot] =
                summary ? p.summary_begin + (off - p.C) : p.ids[b * p.ids_rs + chunk * p.C + off - p.text0];
    }
    if (p.is_summary && lane == 0) p.is_summary[i_slot] = summary ? 1 : 0;
    u32x4 c, s;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float a0 = (float)pos * p.inv_freq[8 * lane + 2 * i], a1 = (float)pos * p.inv_freq[8 * lane + 2 * i + 1];
        c[i] = Cv::down2(cosf(a0), cosf(a1));
        s[i] = Cv::down2(sinf(a0), sinf(a1));
    }
    const int D = 16 * p.lanes;
    const int64_t at = i_slot * p.rope_rs + 8 * lane;  // the two halves of a row hold the same angles
    *reinterpret_cast<u32x4*>(p.cos + at) = c;
    *reinterpret_cast<u32x4*>(p.cos + at + D / 2) = c;
    *reinterpret_cast<u32x4*>(p.sin + at) = s;
    *reinterpret_cast<u32x4*>(p.sin + at + D / 2) = s;
}

int expand_slots(PromptParams p, int slots, int inner_chunk, int summary_kind, int D, int dtype, void* stream) {
    if (!p.inv_freq || !p.cos || !p.sin || (p.out_ids && !p.ids)) return KSA_ERR_NULL;
    if (p.batch <= 0 || p.C <= 0 || p.S <= 0 || D <= 0 || summary_kind < 0 || summary_kind > 2) return KSA_ERR_INVALID;
    if (D % 16 != 0) return KSA_ERR_UNSUPPORTED;
    if (dtype != KSA_DTYPE_BF16 && dtype != KSA_DTYPE_F16) return KSA_ERR_UNSUPPORTED;
    if ((reinterpret_cast<uintptr_t>(p.cos) | reinterpret_cast<uintptr_t>(p.sin)) & 15 || p.rope_rs % 8) return KSA_ERR_ALIGN;
    const long long threads = (long long)slots * (D / 16);
    if (threads > (1ll << 31)) return KSA_ERR_INVALID;
    p.L = slots, p.lanes = D / 16;
    p.inner_chunk = inner_chunk ? 1 : 0, p.summary_kind = summary_kind;
    auto kern = dtype == KSA_DTYPE_BF16 ? ksa_expand_prompt_kernel<KsaBf16> : ksa_expand_prompt_kernel<KsaF16>;
    hipLaunchKernelGGL(kern, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, (hipStream_t)stream, p);
    return ksa_check_launch();
}

}  // namespace

extern "C" int ksa_expand_prompt(const long long* ids, long long ids_row_stride, int batch, int n, int C, int S,
                                 long long summary_begin, int inner_chunk, int summary_kind, const float* inv_freq, int D,
                                 long long* out_ids, void* cos, void* sin, void* is_summary, int dtype, void* stream) {
    if (!ids || !out_ids || !is_summary) return KSA_ERR_NULL;
    if (n <= 0 || C <= 0 || S <= 0) return KSA_ERR_INVALID;
    const long long L = (long long)(n / C) * S + n;
    if (L > INT32_MAX) return KSA_ERR_INVALID;
    PromptParams p{};
    p.ids = ids, p.ids_rs = ids_row_stride;
    p.inv_freq = inv_freq;
    p.out_ids = out_ids;
    p.cos = (uint16_t*)cos, p.sin = (uint16_t*)sin, p.rope_rs = D;
    p.is_summary = (uint8_t*)is_summary;
    p.summary_begin = summary_begin;
    p.batch = batch, p.C = C, p.S = S;
    return expand_slots(p, (int)L, inner_chunk, summary_kind, D, dtype, stream);
}

// Slots [slot0, slot0 + slots) of the same: ids[b][0] is the text token of the first of them that is one.
extern "C" int ksa_expand_slots(const long long* ids, long long ids_row_stride, int batch, int slot0, int slots, int C, int S,
                                long long summary_begin, int inner_chunk, int summary_kind, const float* inv_freq, int D,
                                long long* out_ids, void* cos, void* sin, long long rope_row_stride, int dtype, void* stream) {
    if (slot0 < 0 || slots <= 0 || C <= 0 || S <= 0 || (long long)slot0 + slots > INT32_MAX || (long long)C + S > INT32_MAX)
        return KSA_ERR_INVALID;
    const int chunk = slot0 / (C + S), off = slot0 % (C + S);
    PromptParams p{};
    p.ids = ids, p.ids_rs = ids_row_stride;
    p.inv_freq = inv_freq;
    p.out_ids = out_ids;
    p.cos = (uint16_t*)cos, p.sin = (uint16_t*)sin, p.rope_rs = rope_row_stride;
    p.summary_begin = summary_begin;
    p.slot0 = slot0, p.text0 = chunk * C + (off < C ? off : C);
    p.batch = batch, p.C = C, p.S = S;
    return expand_slots(p, slots, inner_chunk, summary_kind, D, dtype, stream);
}
