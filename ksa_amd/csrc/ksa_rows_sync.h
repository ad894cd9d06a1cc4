// What the one-launch kernels of a decode step share: data and counts handed from workgroup to workgroup inside a
// launch, and the residual add + RMSNorm of one row at the head of a launch.
//
// Data that one workgroup writes and another one of the same launch reads goes through agent-scope stores and
// loads that are not served from an XCD's L2 (the L2 caches of the eight XCDs are not coherent with each other for plain
// accesses).  A writer waits until its stores have left, then counts itself off on a word in device memory; a reader
// polls that word.  Workgroups are started in the order of their numbers and readers have higher numbers than the
// writers they depend on, so no wait needs the grid to be resident as a whole; every wait is bounded all the same.
#pragma once
#include <hip/hip_runtime.h>

#include "ksa_cvt.h"

constexpr int kWordStride = 64;  // 64-bit words are 512 bytes apart

__device__ __forceinline__ unsigned long long ld_agent(const unsigned long long* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_agent(unsigned long long* p, unsigned long long v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_agent(float* p, float v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned long long add_agent(unsigned long long* p, unsigned long long v) {
    return __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// 16 / 8 bytes written by another workgroup of this launch, `off` bytes behind the base: buffer loads with the
// cache-control bit that the compiler sets for agent-scope atomic loads (those stop at 8 bytes), which it tracks like any
// other load, so that several are in flight.
struct KsaAgentBuffer {
    __amdgpu_buffer_rsrc_t rsrc;
    __device__ __forceinline__ KsaAgentBuffer(const void* base, uint32_t bytes)
        : rsrc(__builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)bytes, 0x00020000)) {}
    static constexpr int kSc1 = 16;
    __device__ __forceinline__ u32x4 ld4(uint32_t off, uint32_t uniform_off = 0) const {
        return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)off, (int)uniform_off, kSc1));
    }
    __device__ __forceinline__ u32x2 ld2(uint32_t off, uint32_t uniform_off = 0) const {
        return __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(rsrc, (int)off, (int)uniform_off, kSc1));
    }
};

// Called by a whole wave: waits until the word of every lane that is `live` has reached `want`.  False: another workgroup
// has set the status word, or the wait was given up here (and the word set).
__device__ __forceinline__ bool ksa_wave_wait(const unsigned long long* word, bool live, long long want,
                                              unsigned long long* status, unsigned spin_limit) {
    for (unsigned spins = 1;; ++spins) {
        const bool there = !live || (long long)ld_agent(word) >= want;
        if (__all(there)) return true;
        __builtin_amdgcn_s_sleep(2);
        if (spins > spin_limit) {
            st_agent(status, 1ull);
            return false;
        }
        if ((spins & 63) == 0 && ld_agent(status) != 0) return false;
    }
}

// Words of the workspace of ksa_decode_qkv_o_fwd and ksa_add_rmsnorm_gemm_rows, the latter's rows behind them.  The words
// are zero between launches: the last workgroup of a launch to have seen them clears them.
enum {
    kStepStatus = 0,
    kStepAttnDone = 1,       // workgroups of the o projection that are through with their wait
    kStepHead0 = 4,          // attention workgroups of kv head h that have left their sums
    kStepMaxHeads = 128,
    kStepNormCopies = 8,     // (hundreds of workgroups would queue at one word)
    kStepNormDone0 = kStepHead0 + kStepMaxHeads,       // workgroups that have read a copy of the norm's sums
    kStepNorm0 = kStepNormDone0 + kStepNormCopies,     // a copy: 2^32 | sum of squares, [chunk of 512 columns][row]
    kStepWords = kStepNorm0 + kStepNormCopies,
    kStepNormRows = 8,
    kStepMaxHidden = kWordStride / kStepNormRows * 512,
};
constexpr size_t kStepBytes = (size_t)kStepWords * kWordStride * 8 + (size_t)kStepNormRows * kStepMaxHidden * 2;

// ---- residual add + RMSNorm of one row by the 512 threads of a workgroup ----
// x' = residual + rounded sum of the K-split partial sums (plain store, for later launches), h = norm(x') w (for the
// workgroups of this launch that wait for it).  Arithmetic and summation order of ksa_add_rmsnorm_partials.
struct KsaNormStage {
    const float* part;        // [ksplit][16][H] partial sums
    const uint16_t* res;      // residual rows [M][H]
    const uint16_t* w;        // norm weight [H]
    uint16_t* out_sum;        // x' [M][H]
    unsigned long long* hbuf; // h [M][H / 4], four values per word
    int64_t res_rs, sum_rs;
    int ksplit;
    float eps;
};
// kBatch: slices requested at a time (eight registers each); s_ss: eight floats of LDS.  H up to 4096, a multiple of 8.
// On return every store of this thread has left; a barrier of the workgroup then says so of the row.
template <typename T, int kBatch>
__device__ __forceinline__ void ksa_norm_row(const KsaNormStage& p, int H, int row, int tid, float* s_ss) {
    using C = KsaCvt<T>;
    const int lane = tid & 63, wave = tid >> 6;
    const int items = H / 8;  // at most 512: one per thread
    float ss = 0.f;
    u32x4 rsum = {0u, 0u, 0u, 0u}, wv = {0u, 0u, 0u, 0u};
    if (tid < items) {
        wv = *reinterpret_cast<const u32x4*>(p.w + 8 * tid);
        const u32x4 q = *reinterpret_cast<const u32x4*>(p.res + (int64_t)row * p.res_rs + 8 * tid);
        float ac[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        for (int sp0 = 0; sp0 < p.ksplit; sp0 += kBatch) {
            f32x4 lo[kBatch], hi[kBatch];
#pragma unroll
            for (int k = 0; k < kBatch; ++k) {
                const float* src = p.part + ((int64_t)min(sp0 + k, p.ksplit - 1) * 16 + row) * H + 8 * tid;
                lo[k] = *reinterpret_cast<const f32x4*>(src);
                hi[k] = *reinterpret_cast<const f32x4*>(src + 4);
            }
#pragma unroll
            for (int k = 0; k < kBatch; ++k) {
                if (sp0 + k < p.ksplit) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) ac[i] += lo[k][i], ac[4 + i] += hi[k][i];
                }
            }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t x = C::down2(ac[2 * i], ac[2 * i + 1]);
            rsum[i] = C::down2(C::lo(x) + C::lo(q[i]), C::hi(x) + C::hi(q[i]));
            const float a_ = C::lo(rsum[i]), b_ = C::hi(rsum[i]);
            ss = fmaf(a_, a_, ss);
            ss = fmaf(b_, b_, ss);
        }
        *reinterpret_cast<u32x4*>(p.out_sum + (int64_t)row * p.sum_rs + 8 * tid) = rsum;
    }
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) ss += __shfl_xor(ss, m);
    if (lane == 0) s_ss[wave] = ss;
    __syncthreads();
    ss = 0.f;
    for (int w = 0; w < (items + 63) / 64; ++w) ss += s_ss[w];
    const float inv = rsqrtf(ss / (float)H + p.eps);
    if (tid < items) {
        uint32_t o[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t y = C::down2(C::lo(rsum[i]) * inv, C::hi(rsum[i]) * inv);
            o[i] = C::down2(C::lo(wv[i]) * C::lo(y), C::hi(wv[i]) * C::hi(y));
        }
        unsigned long long* hp = p.hbuf + (int64_t)row * (H / 4) + 2 * tid;
        st_agent(hp, (unsigned long long)o[0] | ((unsigned long long)o[1] << 32));
        st_agent(hp + 1, (unsigned long long)o[2] | ((unsigned long long)o[3] << 32));
    }
    // Every thread waits until its own stores have left (they write through to memory), and only then joins the
    // caller's barrier: the barrier itself does not wait for the stores of the other waves.
    __builtin_amdgcn_s_waitcnt(0);
}
