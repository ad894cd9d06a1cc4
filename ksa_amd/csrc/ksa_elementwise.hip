// Two element-wise steps of a decoder layer around the attention path, one pass over HBM each
// (gfx950), with the rounding points of the reference's 16-bit tensor ops:
//   * residual add + RMSNorm over the hidden size
//       examples/pretrain/hf_template/modeling_qwen3sa.py:64-79 (Qwen3RMSNorm.forward: fp32
//       normalisation, result rounded to the 16-bit type, times the 16-bit weight) and the
//       residual adds of Qwen3DecoderLayer.forward :946, :952
//   * SiLU(gate) * up of the MLP (:507-514)
// Both replace chains of 3-8 library element-wise launches; at decode batch sizes a layer step
// is bound by the number of launches.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "ksa_api_internal.h"
#include "ksa_cvt.h"

namespace {

struct NormParams {
    const uint16_t* x;
    const float* part;     // partial-sum variant: x = rounded sum of `ksplit` fp32 slices [ksplit][ksa_partial_rows(rows)][H]
    int ksplit;
    const uint16_t* res;   // may be null
    const uint16_t* w;
    uint16_t* out_norm;
    uint16_t* out_sum;     // x + res (null if res is null)
    int64_t rows;
    int64_t xs, rs, ns, ss;  // row strides (elements)
    int H;
    float eps;
};
// kEmbed: row r of x is row ids[r] of a table of x_rows rows; the row behind the last one copies row *rope_row of a
// second table.  (Parameters of their own: the other launches would carry them along, 1 % of a few-rows norm.)
struct EmbedParams : NormParams {
    const long long* ids;
    int64_t x_rows;
    const uint16_t* rope;  // [rope_rows][rope_width]
    const int32_t* rope_row;
    int rope_rows, rope_width;
    uint16_t* rope_out;
};

// One wave per row; the row (after the residual add) stays in registers between the
// sum-of-squares pass and the scaling pass.  NI = 16-byte items per lane.  Inputs are read once:
// non-temporal loads.
// What bounds it is HBM for many rows, the one trip to memory for few; all items of a row and its residual are on their way
// before the first is used.  (One item after the other, each under its own condition, made a chain of NI trips of it: 2560 x
// 100 / 740 / 6368 / 34816 rows behind one another in a graph 7.3 / 10.0 / 30.0 / 140 -> 4.7 / 6.8 / 26.7 / 136 us, 5.3 TB/s; 5120 x 100 /
// 6368 16.2 / 59.3 -> 7.1 / 48.2, 8192 24.6 / 91.5 -> 9.9 / 74.7.)
// kEmbed: the head of a decode step - embedding rows, their norm for the first layer, the step's rotary row - whose
// cost is its launches (4.5 us each behind one another, for some 10 KB): as one, and with the ids read where the
// caller has them, a decode step of 8 layers went from 649 to 643 us (batch 1) and from 759 to 754 (batch 8).
template <typename T, int NI, bool kEmbed = false>
__global__ __launch_bounds__(256) void ksa_add_rmsnorm_kernel(const std::conditional_t<kEmbed, EmbedParams, NormParams> p) {
    using C = KsaCvt<T>;
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int items = p.H / 8;
    if constexpr (kEmbed) {
        if ((int64_t)blockIdx.x * 4 + wave == p.rows) {
            const int64_t from = min(max(*p.rope_row, 0), p.rope_rows - 1);
            for (int i = 8 * lane; i < p.rope_width; i += 512)
                *reinterpret_cast<u32x4*>(p.rope_out + i) = *reinterpret_cast<const u32x4*>(p.rope + from * p.rope_width + i);
        }
    }
    for (int64_t row = (int64_t)blockIdx.x * 4 + wave; row < p.rows; row += (int64_t)gridDim.x * 4) {
        u32x4 r[NI], q[kEmbed ? 1 : NI];
        float ss = 0.f;
        int64_t src = row;
        bool inside = true;
        if constexpr (kEmbed) {  // (a negative id counts from the end; one outside the table gives a row of NaN)
            src = p.ids[row];
            if (src < 0) src += p.x_rows;
            inside = src >= 0 && src < p.x_rows;
            if (!inside) src = 0;
        }
#pragma unroll
        for (int j = 0; j < NI; ++j) {  // (lanes past the row's end repeat its last item)
            const int idx = min(lane + 64 * j, items - 1);
            r[j] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p.x + src * p.xs + 8 * idx));
        }
        if constexpr (!kEmbed) {
            if (p.res) {
#pragma unroll
                for (int j = 0; j < NI; ++j)
                    q[j] = __builtin_nontemporal_load(
                        reinterpret_cast<const u32x4*>(p.res + row * p.rs + 8 * min(lane + 64 * j, items - 1)));
            }
        }
#pragma unroll
        for (int j = 0; j < NI; ++j) {
            const int idx = lane + 64 * j;
            if (idx < items) {
                if constexpr (kEmbed) {
                    if (!inside) r[j] = u32x4{0x7fff7fffu, 0x7fff7fffu, 0x7fff7fffu, 0x7fff7fffu};
                    *reinterpret_cast<u32x4*>(p.out_sum + row * p.ss + 8 * idx) = r[j];
                } else if (p.res) {
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        r[j][i] = C::down2(C::lo(r[j][i]) + C::lo(q[j][i]), C::hi(r[j][i]) + C::hi(q[j][i]));
                    *reinterpret_cast<u32x4*>(p.out_sum + row * p.ss + 8 * idx) = r[j];
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float a = C::lo(r[j][i]), b = C::hi(r[j][i]);
                    ss = fmaf(a, a, ss);
                    ss = fmaf(b, b, ss);
                }
            }
        }
#pragma unroll
        for (int m = 32; m >= 1; m >>= 1) ss += __shfl_xor(ss, m);
        const float inv = rsqrtf(ss / (float)p.H + p.eps);
#pragma unroll
        for (int j = 0; j < NI; ++j) {
            const int idx = lane + 64 * j;
            if (idx < items) {
                const u32x4 wv = *reinterpret_cast<const u32x4*>(p.w + 8 * idx);
                u32x4 o;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const uint32_t y = C::down2(C::lo(r[j][i]) * inv, C::hi(r[j][i]) * inv);
                    o[i] = C::down2(C::lo(wv[i]) * C::lo(y), C::hi(wv[i]) * C::hi(y));
                }
                *reinterpret_cast<u32x4*>(p.out_norm + row * p.ns + 8 * idx) = o;
            }
        }
    }
}

// The same step for the few rows of a decode step when x is still the K-split partial sums of
// the GEMM that produced it (fp32 [ksplit][rows in whole 16-row blocks][H], as ksa_gemm_rows leaves them): one workgroup
// per row, as many threads as the row has 16-byte items (up to 512, then NJ = 2 items per thread),
// adds the slices in split order, rounds (which is what the GEMM's own reduction does), adds the
// residual and normalises.  Everything that does not depend on the sums is requested first.
// kBatch: slices requested together; every further batch is another trip to memory, which is what this kernel's time
// is.  Twenty take the 19 slices of the 4B shape's down projection in one trip (184 registers, no matter with
// one workgroup per row) where eight take three: decode step of 8 layers 643.1 -> 640.0 us (batch 1), 752.6 -> 750.1
// (batch 8).  That pays where three trips become one and a workgroup is small: 17 to 20 slices of up to 2560 elements
// (1 row of 1024 / 2560, 19 slices 3.92 / 5.40 -> 3.77 / 5.30 us; 3584 6.08 -> 6.33, so not there).  Elsewhere the
// requests past the last slice cost more than the trips (9 / 16 / 24 slices of 2560 4.0 / 4.3 / 5.7 -> 4.7 / 4.9 / 7.3
// us, of 4096 4.3 / 5.2 / 6.3 -> 5.4 / 6.3 / 9.3): eight.
template <typename T, int NJ, int kBatch>
__global__ __launch_bounds__(512) void ksa_add_rmsnorm_partials_kernel(const NormParams p) {
    using C = KsaCvt<T>;
    __shared__ float s_ss[8];
    const int tid = threadIdx.x, nthr = blockDim.x;
    const int row = blockIdx.x;
    const int items = p.H / 8;
    u32x4 r[NJ], wv[NJ], q[NJ];
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {  // the weights and the residual do not wait for the sums
        const int idx = tid + nthr * j;
        if (idx < items) {
            wv[j] = *reinterpret_cast<const u32x4*>(p.w + 8 * idx);
            q[j] = *reinterpret_cast<const u32x4*>(p.res + (int64_t)row * p.rs + 8 * idx);
        }
    }
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        const int idx = tid + nthr * j;
        if (idx < items) {
            const u32x4 x = ksa_sum_partials8<T, kBatch>(p.part, p.ksplit, ksa_partial_rows(p.rows), p.H, row, 8 * idx);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                r[j][i] = C::down2(C::lo(x[i]) + C::lo(q[j][i]), C::hi(x[i]) + C::hi(q[j][i]));
                const float a = C::lo(r[j][i]), b = C::hi(r[j][i]);
                ss = fmaf(a, a, ss);
                ss = fmaf(b, b, ss);
            }
            *reinterpret_cast<u32x4*>(p.out_sum + (int64_t)row * p.ss + 8 * idx) = r[j];
        }
    }
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) ss += __shfl_xor(ss, m);
    if ((tid & 63) == 0) s_ss[tid >> 6] = ss;
    __syncthreads();
    ss = 0.f;
    for (int w = 0; w < nthr / 64; ++w) ss += s_ss[w];
    const float inv = rsqrtf(ss / (float)p.H + p.eps);
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        const int idx = tid + nthr * j;
        if (idx < items) {
            u32x4 o;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t y = C::down2(C::lo(r[j][i]) * inv, C::hi(r[j][i]) * inv);
                o[i] = C::down2(C::lo(wv[j][i]) * C::lo(y), C::hi(wv[j][i]) * C::hi(y));
            }
            *reinterpret_cast<u32x4*>(p.out_norm + (int64_t)row * p.ns + 8 * idx) = o;
        }
    }
}

template <typename T>
int dispatch_norm_partials(const NormParams& p, hipStream_t st) {
    const int items = p.H / 8;
    const int threads = items >= 512 ? 512 : (items + 63) / 64 * 64;
    const int need = (items + threads - 1) / threads;
    const dim3 grid((unsigned)p.rows), block(threads);
    if (items <= 320 && p.ksplit > 16 && p.ksplit <= 20) hipLaunchKernelGGL((ksa_add_rmsnorm_partials_kernel<T, 1, 20>), grid, block, 0, st, p);
    else if (need <= 1) hipLaunchKernelGGL((ksa_add_rmsnorm_partials_kernel<T, 1, 8>), grid, block, 0, st, p);
    else if (need <= 2) hipLaunchKernelGGL((ksa_add_rmsnorm_partials_kernel<T, 2, 8>), grid, block, 0, st, p);
    else return KSA_ERR_UNSUPPORTED;
    return ksa_check_launch();
}

template <typename T, int NI>
int launch_norm(const NormParams& p, hipStream_t st) {
    const int64_t blocks = (p.rows + 3) / 4;
    // one short-lived workgroup per four rows (measured 5 % faster than a capped grid with a
    // grid-stride loop); the loop only serves row counts beyond the grid limit
    const int64_t cap = 0x7fffffff;
    hipLaunchKernelGGL((ksa_add_rmsnorm_kernel<T, NI>), dim3((unsigned)(blocks < cap ? blocks : cap)), dim3(256), 0,
                       st, p);
    return ksa_check_launch();
}
template <typename T, int NI>
int launch_norm(const EmbedParams& p, hipStream_t st) {
    hipLaunchKernelGGL((ksa_add_rmsnorm_kernel<T, NI, true>), dim3((unsigned)((p.rows + 1 + 3) / 4)), dim3(256), 0, st, p);
    return ksa_check_launch();
}

template <typename T, typename P>
int dispatch_norm(const P& p, hipStream_t st) {
    const int need = (p.H / 8 + 63) / 64;
    if (need <= 1) return launch_norm<T, 1>(p, st);
    if (need <= 2) return launch_norm<T, 2>(p, st);
    if (need <= 4) return launch_norm<T, 4>(p, st);
    if (need <= 5) return launch_norm<T, 5>(p, st);
    if (need <= 8) return launch_norm<T, 8>(p, st);
    if (need <= 16) return launch_norm<T, 16>(p, st);
    return KSA_ERR_UNSUPPORTED;
}

struct ActParams {
    const uint16_t* gate;
    const uint16_t* up;
    uint16_t* out;
    int64_t gs, us, os;  // row strides (elements)
    int I;
    const float* part;   // if set: gate | up as K-split partial sums, see the kernel
    int ksplit;
};

// blockIdx.x = row, blockIdx.y = block of 256 16-byte items inside the row
// kPartials: a variant of its own, so that the streaming variant does not carry its registers
template <typename T, bool kPartials>
__global__ __launch_bounds__(256) void ksa_silu_mul_kernel(const ActParams p) {
    using C = KsaCvt<T>;
    const int64_t row = blockIdx.x;
    const int idx = blockIdx.y * 256 + threadIdx.x;
    if (idx >= p.I / 8) return;
    u32x4 g, u;
    if constexpr (kPartials) {  // gate | up still as the partial sums of the fused projection [ksplit][ksa_partial_rows(rows)][2 I]
        g = ksa_sum_partials8<T>(p.part, p.ksplit, ksa_partial_rows((int)gridDim.x), 2 * p.I, (int)row, 8 * idx);
        u = ksa_sum_partials8<T>(p.part, p.ksplit, ksa_partial_rows((int)gridDim.x), 2 * p.I, (int)row, p.I + 8 * idx);
    } else {
        g = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p.gate + row * p.gs + 8 * idx));
        u = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p.up + row * p.us + 8 * idx));
    }
    u32x4 o;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float a = C::lo(g[i]), b = C::hi(g[i]);
        const uint32_t s = C::down2(a / (1.f + expf(-a)), b / (1.f + expf(-b)));
        o[i] = C::down2(C::lo(s) * C::lo(u[i]), C::hi(s) * C::hi(u[i]));
    }
    *reinterpret_cast<u32x4*>(p.out + row * p.os + 8 * idx) = o;
}

bool al16(const void* q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; }

// ---- greedy token choice: index of the largest value of every row ----
// Among equal values the lowest index wins and a NaN counts as the largest value, as torch.argmax has it.
struct ArgmaxParams {
    const uint16_t* x;
    long long* out;
    int64_t xs;
    int N;
};

// the larger of the two values in a word, NaNs aside, and the word's magnitudes (for the NaN test)
template <typename T>
__device__ __forceinline__ float argmax_pair(uint32_t w) {
    return fmaxf(KsaCvt<T>::lo(w), KsaCvt<T>::hi(w));
}
__device__ __forceinline__ uint32_t max_u16x2(uint32_t a, uint32_t b) {
    typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(u16x2, a), __builtin_bit_cast(u16x2, b)));
}

// One workgroup per row.  What bounds a row of the 4B shape's vocabulary (151936 values, 300 KB through one CU) is
// vector issue: looking at value, NaN and index of every element took 24 us.  Here the walk only
// keeps each thread's largest value and the request batch it came from (about 2.5 instructions an element);
// the threads that hold the row's maximum look into that one batch again for its place.  A row with a NaN
// (its magnitudes exceed infinity's) is searched once more for the first one.  1 / 8 / 64 rows
// 25.0 / 25.5 / 26.9 -> 8.4 / 9.0 / 11.3 us; of 32000 values 8.3 / 8.5 / 9.1 -> 5.2 / 5.6 / 5.9, of 1000 4.0 / 4.3 / 4.5 ->
// 3.1 / 3.4 / 3.6.
template <typename T>
__global__ __launch_bounds__(1024) void ksa_argmax_rows_kernel(const ArgmaxParams p) {
    using C = KsaCvt<T>;
    constexpr int kBatch = 10;
    constexpr uint32_t kInf = C::kInfBits;
    const uint16_t* row = p.x + (int64_t)blockIdx.x * p.xs;
    const int tid = threadIdx.x;
    const int items = p.N / 8;                     // whole 16-byte items; item j belongs to thread j % 1024
    const int last = max(items - 1, 0);
    float best = -INFINITY;
    int from = tid;                                // first item of the batch that holds `best`
    uint32_t mag = 0;
    for (int j0 = tid; j0 < items; j0 += kBatch * 1024) {
        u32x4 v[kBatch];                           // (items past the end repeat the last one: no new values)
#pragma unroll
        for (int u = 0; u < kBatch; ++u) v[u] = *reinterpret_cast<const u32x4*>(row + 8 * (int64_t)min(j0 + 1024 * u, last));
        float m = -INFINITY;
#pragma unroll
        for (int u = 0; u < kBatch; ++u)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                m = fmaxf(m, argmax_pair<T>(v[u][i]));
                mag = max_u16x2(mag, v[u][i] & 0x7fff7fffu);
            }
        if (m > best) best = m, from = j0;
    }
    const int t = 8 * items + tid;                 // the values behind the last whole item: one per thread
    const bool has_t = t < p.N;
    const uint16_t tail = has_t ? row[t] : 0;
    const float tail_v = has_t ? C::up(tail) : -INFINITY;
    mag = max_u16x2(mag, tail & 0x7fffu);
    bool nan = (mag & 0xffffu) > kInf || (mag >> 16) > kInf;

    __shared__ float sv[16];
    __shared__ int si[16];
    float mx = fmaxf(best, tail_v);
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) mx = fmaxf(mx, __shfl_xor(mx, m));
    if ((tid & 63) == 0) sv[tid >> 6] = mx;
    nan = __syncthreads_or(nan);
#pragma unroll
    for (int w = 0; w < 16; ++w) mx = fmaxf(mx, sv[w]);
    int idx = 0x7fffffff;
    auto look = [&](int j) {                       // item j: first NaN, or first value equal to the maximum
        const u32x4 v = *reinterpret_cast<const u32x4*>(row + 8 * (int64_t)j);
#pragma unroll
        for (int i = 3; i >= 0; --i) {
            const uint32_t lo = v[i] & 0xffffu, hi = v[i] >> 16;
            if (nan ? (hi & 0x7fffu) > kInf : C::hi(v[i]) == mx) idx = min(idx, 8 * j + 2 * i + 1);
            if (nan ? (lo & 0x7fffu) > kInf : C::lo(v[i]) == mx) idx = min(idx, 8 * j + 2 * i);
        }
    };
    if (nan) {
        for (int j = tid; j < items; j += 1024) look(j);
        if (has_t && (tail & 0x7fffu) > kInf) idx = min(idx, t);
    } else {
        if (best == mx) {
#pragma unroll
            for (int u = 0; u < kBatch; ++u)
                if (from + 1024 * u < items) look(from + 1024 * u);
        }
        if (has_t && tail_v == mx) idx = min(idx, t);
    }
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) idx = min(idx, __shfl_xor(idx, m));
    if ((tid & 63) == 0) si[tid >> 6] = idx;
    __syncthreads();
    if (tid == 0) {
        for (int w = 1; w < 16; ++w) idx = min(idx, si[w]);
        p.out[blockIdx.x] = idx;
    }
}

}  // namespace

extern "C" int ksa_add_rmsnorm(const void* x, const void* residual, const void* weight, void* out_norm,
                               void* out_sum, long long rows, int H, long long x_row_stride,
                               long long residual_row_stride, long long norm_row_stride,
                               long long sum_row_stride, int dtype, float eps, void* stream) {
    if (!x || !weight || !out_norm) return KSA_ERR_NULL;
    if (residual && !out_sum) return KSA_ERR_NULL;
    if (rows <= 0 || H <= 0 || H % 8 != 0 || !(eps >= 0.f)) return KSA_ERR_INVALID;
    if (dtype != KSA_DTYPE_BF16 && dtype != KSA_DTYPE_F16) return KSA_ERR_UNSUPPORTED;
    if (!al16(x) || !al16(weight) || !al16(out_norm) || (residual && (!al16(residual) || !al16(out_sum))))
        return KSA_ERR_ALIGN;
    if (x_row_stride % 8 || norm_row_stride % 8 || (residual && (residual_row_stride % 8 || sum_row_stride % 8)))
        return KSA_ERR_ALIGN;
    NormParams p{};
    p.x = (const uint16_t*)x;
    p.res = (const uint16_t*)residual;
    p.w = (const uint16_t*)weight;
    p.out_norm = (uint16_t*)out_norm;
    p.out_sum = residual ? (uint16_t*)out_sum : nullptr;
    p.rows = rows;
    p.xs = x_row_stride, p.rs = residual_row_stride, p.ns = norm_row_stride, p.ss = sum_row_stride;
    p.H = H;
    p.eps = eps;
    return dtype == KSA_DTYPE_BF16 ? dispatch_norm<KsaBf16>(p, (hipStream_t)stream)
                                   : dispatch_norm<KsaF16>(p, (hipStream_t)stream);
}

extern "C" int ksa_embed_rmsnorm(const void* table, long long table_rows, long long table_row_stride, const long long* ids,
                                 const void* weight, void* out, void* out_norm, int rows, int H, const void* rope_table,
                                 int rope_rows, int rope_width, const int32_t* rope_row, void* rope_out, int dtype,
                                 float eps, void* stream) {
    if (!table || !ids || !weight || !out || !out_norm || !rope_table || !rope_row || !rope_out) return KSA_ERR_NULL;
    if (rows <= 0 || rows > (1 << 20) || H <= 0 || H % 8 != 0 || table_rows <= 0 || rope_rows <= 0 || rope_width <= 0 ||
        rope_width % 8 != 0 || !(eps >= 0.f))
        return KSA_ERR_INVALID;
    if (dtype != KSA_DTYPE_BF16 && dtype != KSA_DTYPE_F16) return KSA_ERR_UNSUPPORTED;
    if (!al16(table) || !al16(weight) || !al16(out) || !al16(out_norm) || !al16(rope_table) || !al16(rope_out) ||
        table_row_stride % 8)
        return KSA_ERR_ALIGN;
    EmbedParams p{};
    p.x = (const uint16_t*)table, p.x_rows = table_rows, p.xs = table_row_stride;
    p.ids = ids;
    p.w = (const uint16_t*)weight;
    p.out_norm = (uint16_t*)out_norm, p.out_sum = (uint16_t*)out;
    p.rows = rows, p.ns = p.ss = H, p.H = H;
    p.eps = eps;
    p.rope = (const uint16_t*)rope_table, p.rope_rows = rope_rows, p.rope_width = rope_width;
    p.rope_row = rope_row, p.rope_out = (uint16_t*)rope_out;
    return dtype == KSA_DTYPE_BF16 ? dispatch_norm<KsaBf16>(p, (hipStream_t)stream)
                                   : dispatch_norm<KsaF16>(p, (hipStream_t)stream);
}

extern "C" int ksa_add_rmsnorm_partials(const float* partials, int ksplit, const void* residual,
                                        const void* weight, void* out_norm, void* out_sum, int rows, int H,
                                        long long residual_row_stride, long long norm_row_stride,
                                        long long sum_row_stride, int dtype, float eps, void* stream) {
    if (!partials || !residual || !weight || !out_norm || !out_sum) return KSA_ERR_NULL;
    if (rows <= 0 || rows > kMaxPartialRows || ksplit < 1 || ksplit > 64 || H <= 0 || H % 8 != 0 || !(eps >= 0.f))
        return KSA_ERR_INVALID;
    if (dtype != KSA_DTYPE_BF16 && dtype != KSA_DTYPE_F16) return KSA_ERR_UNSUPPORTED;
    if (!al16(partials) || !al16(residual) || !al16(weight) || !al16(out_norm) || !al16(out_sum)) return KSA_ERR_ALIGN;
    if (residual_row_stride % 8 || norm_row_stride % 8 || sum_row_stride % 8) return KSA_ERR_ALIGN;
    NormParams p{};
    p.part = partials;
    p.ksplit = ksplit;
    p.res = (const uint16_t*)residual;
    p.w = (const uint16_t*)weight;
    p.out_norm = (uint16_t*)out_norm;
    p.out_sum = (uint16_t*)out_sum;
    p.rows = rows;
    p.rs = residual_row_stride, p.ns = norm_row_stride, p.ss = sum_row_stride;
    p.H = H;
    p.eps = eps;
    return dtype == KSA_DTYPE_BF16 ? dispatch_norm_partials<KsaBf16>(p, (hipStream_t)stream)
                                   : dispatch_norm_partials<KsaF16>(p, (hipStream_t)stream);
}

extern "C" int ksa_silu_mul(const void* gate, const void* up, void* out, long long rows, int I,
                            long long gate_row_stride, long long up_row_stride, long long out_row_stride,
                            int dtype, void* stream) {
    if (!gate || !up || !out) return KSA_ERR_NULL;
    if (rows <= 0 || rows >= (1ll << 31) || I <= 0 || I % 8 != 0) return KSA_ERR_INVALID;
    if (dtype != KSA_DTYPE_BF16 && dtype != KSA_DTYPE_F16) return KSA_ERR_UNSUPPORTED;
    if (!al16(gate) || !al16(up) || !al16(out) || gate_row_stride % 8 || up_row_stride % 8 || out_row_stride % 8)
        return KSA_ERR_ALIGN;
    const int yblocks = (I / 8 + 255) / 256;
    if (yblocks > 65535) return KSA_ERR_INVALID;
    ActParams p{(const uint16_t*)gate, (const uint16_t*)up, (uint16_t*)out, gate_row_stride, up_row_stride,
                out_row_stride, I, nullptr, 0};
    if (dtype == KSA_DTYPE_BF16)
        hipLaunchKernelGGL((ksa_silu_mul_kernel<KsaBf16, false>), dim3((unsigned)rows, yblocks), dim3(256), 0,
                           (hipStream_t)stream, p);
    else
        hipLaunchKernelGGL((ksa_silu_mul_kernel<KsaF16, false>), dim3((unsigned)rows, yblocks), dim3(256), 0,
                           (hipStream_t)stream, p);
    return ksa_check_launch();
}

extern "C" int ksa_silu_mul_partials(const float* partials, int ksplit, void* out, int rows, int I,
                                     long long out_row_stride, int dtype, void* stream) {
    if (!partials || !out) return KSA_ERR_NULL;
    if (rows <= 0 || rows > kMaxPartialRows || ksplit < 1 || ksplit > 64 || I <= 0 || I % 8 != 0) return KSA_ERR_INVALID;
    if (dtype != KSA_DTYPE_BF16 && dtype != KSA_DTYPE_F16) return KSA_ERR_UNSUPPORTED;
    if (!al16(partials) || !al16(out) || out_row_stride % 8) return KSA_ERR_ALIGN;
    const int yblocks = (I / 8 + 255) / 256;
    if (yblocks > 65535) return KSA_ERR_INVALID;
    ActParams p{nullptr, nullptr, (uint16_t*)out, 0, 0, out_row_stride, I, partials, ksplit};
    if (dtype == KSA_DTYPE_BF16)
        hipLaunchKernelGGL((ksa_silu_mul_kernel<KsaBf16, true>), dim3((unsigned)rows, yblocks), dim3(256), 0,
                           (hipStream_t)stream, p);
    else
        hipLaunchKernelGGL((ksa_silu_mul_kernel<KsaF16, true>), dim3((unsigned)rows, yblocks), dim3(256), 0,
                           (hipStream_t)stream, p);
    return ksa_check_launch();
}

extern "C" int ksa_argmax_rows(const void* x, long long* out, int rows, int N, long long x_row_stride,
                               int dtype, void* stream) {
    if (!x || !out) return KSA_ERR_NULL;
    if (rows <= 0 || rows > 65535 || N <= 0) return KSA_ERR_INVALID;
    if (dtype != KSA_DTYPE_BF16 && dtype != KSA_DTYPE_F16) return KSA_ERR_UNSUPPORTED;
    if (!al16(x) || x_row_stride % 8) return KSA_ERR_ALIGN;
    ArgmaxParams p{(const uint16_t*)x, out, x_row_stride, N};
    if (dtype == KSA_DTYPE_BF16)
        hipLaunchKernelGGL(ksa_argmax_rows_kernel<KsaBf16>, dim3(rows), dim3(1024), 0, (hipStream_t)stream, p);
    else
        hipLaunchKernelGGL(ksa_argmax_rows_kernel<KsaF16>, dim3(rows), dim3(1024), 0, (hipStream_t)stream, p);
    return ksa_check_launch();
}
