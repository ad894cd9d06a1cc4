// Residual add + RMSNorm and the product behind them at a decode step as ONE launch (gfx950):
//
//   x' = residual + sum of the K-split partial sums of the product in front    (modeling_qwen3sa.py:950-952)
//   y  = (norm(x') w) W^T, left as K-split partial sums                        (:938, :660-662, the next layer's q | k | v)
//
// for the few rows of a small batch.  The norm is a chain of memory trips of one workgroup per row that leaves the other CUs
// idle, and the product's weights (31 MB at 6144 x 2560) could only start to move behind it.  Here a workgroup owns eight
// column tiles of 16 (one per wave) times one chunk of 512 elements of K; one wave per row adds up that chunk of the
// row itself (39 KB of 19 slices, out of the L2 for all but the first workgroup of an XCD) with the weights requested right
// behind, and the workgroups only hand each other the sums of squares of their chunks, one word per row.  What bounds it is
// that chain - sums, hand-over, product - and, row by row, the repeated sums: 0.75 us per row, which is why more rows take the
// two launches (ksa_amd/gemm.py, add_rmsnorm_linear_rows_pays, with the figures).  With the rows made by one workgroup each at
// the head of the grid and handed over whole it took 13.3 us where the two launches take 12.0.
#include <hip/hip_runtime.h>

#include "ksa_api_internal.h"
#include "ksa_cvt.h"
#include "ksa_rows_mfma.h"
#include "ksa_rows_sync.h"

namespace {

constexpr int kThreads = 512;
constexpr int kWaves = kThreads / 64;
constexpr int kSlices = 20;     // slices requested at once (the 19 of a 9728-wide down projection are one trip to memory)

struct NormGemmParams {
    const float* in;           // [ksplit][16][H] partial sums
    const uint16_t* res;       // residual rows [M][H]
    const uint16_t* nw;        // norm weight [H]
    uint16_t* out_sum;         // x' [M][H]
    int64_t res_rs, sum_rs;
    const uint16_t* w;         // streaming layout [N / 16][H / 32][1 KB]
    float* part;               // [chunks][16][N]
    unsigned long long* sync;  // words of the step's workspace
    int M, H, N, ksplit, chunks, groups;
    float eps;
    unsigned spin_limit;
};

template <typename T>
__global__ __launch_bounds__(kThreads) void ksa_norm_gemm_rows_kernel(const NormGemmParams p) {
    using C = KsaCvt<T>;
    __shared__ __attribute__((aligned(16))) unsigned char xs[kStepNormRows * kRowB];
    __shared__ int s_there[kWaves];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int grp = blockIdx.x / p.chunks, chunk = blockIdx.x - grp * p.chunks;
    const int r = lane & 15, kq = lane >> 4;
    const int tiles = p.N / 16, steps = p.H / 32;
    const int tile = grp * kWaves + wave;
    const int nst = min(kChunkSteps, steps - chunk * kChunkSteps);

    // this wave's row: eight columns per lane (lanes past a short chunk repeat its last piece and add nothing)
    const bool norm = wave < p.M, mine = lane < nst * 4;
    const int col = chunk * kChunkK + 8 * min(lane, nst * 4 - 1);
    const float* src = p.in + (int64_t)wave * p.H + col;
    const int64_t pitch = (int64_t)16 * p.H;
    f32x4 lo[kSlices], hi[kSlices];
    u32x4 wv, q;
    if (norm) {
#pragma unroll
        for (int k = 0; k < kSlices; ++k) {
            const float* sp = src + pitch * min(k, p.ksplit - 1);
            lo[k] = *reinterpret_cast<const f32x4*>(sp);
            hi[k] = *reinterpret_cast<const f32x4*>(sp + 4);
        }
        q = *reinterpret_cast<const u32x4*>(p.res + wave * p.res_rs + col);
        wv = *reinterpret_cast<const u32x4*>(p.nw + col);
    }
    __builtin_amdgcn_sched_barrier(0);
    // The other waves hold their requests back for a trip to memory (1.6 us), so that the slices do not queue behind them:
    // 2560 x 6144, 19 slices, 1 / 2 / 3 rows 9.5 / 10.6 / 11.3 us without, 8.6 / 10.2 / 11.4 with; held back by 2.4 us
    // 9.0 / 9.7 / 11.3, behind a barrier instead 9.9 / 10.8 / 11.4.
    if (!norm) __builtin_amdgcn_s_sleep(60);
    // (a wave past the last tile repeats it, steps past the end of a short chunk its last one; nothing of them is used)
    const KsaWeightLane wl = ksa_weight_lane(p.w, kWTiled, p.H, 16 * (int64_t)min(tile, tiles - 1), r, kq, p.N);
    u32x4 a[kChunkSteps];
#pragma unroll
    for (int u = 0; u < kChunkSteps; ++u)
        a[u] = ksa_load_weights<true>(wl.p + (int64_t)wl.step * (chunk * kChunkSteps + min(u, nst - 1)));
    __builtin_amdgcn_sched_barrier(0);

    if (norm) {  // (arithmetic and order of ksa_add_rmsnorm_partials: a chunk is one of its waves)
        float ac[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < kSlices; ++k) {
            if (k < p.ksplit) {
#pragma unroll
                for (int i = 0; i < 4; ++i) ac[i] += lo[k][i], ac[4 + i] += hi[k][i];
            }
        }
        for (int k = kSlices; k < p.ksplit; ++k) {
            const f32x4 l4 = *reinterpret_cast<const f32x4*>(src + pitch * k);
            const f32x4 h4 = *reinterpret_cast<const f32x4*>(src + pitch * k + 4);
#pragma unroll
            for (int i = 0; i < 4; ++i) ac[i] += l4[i], ac[4 + i] += h4[i];
        }
        u32x4 sum;
        float ss = 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t x = C::down2(ac[2 * i], ac[2 * i + 1]);
            sum[i] = C::down2(C::lo(x) + C::lo(q[i]), C::hi(x) + C::hi(q[i]));
            const float a_ = C::lo(sum[i]), b_ = C::hi(sum[i]);
            ss = fmaf(a_, a_, ss);
            ss = fmaf(b_, b_, ss);
        }
        if (!mine) ss = 0.f;
#pragma unroll
        for (int m = 32; m >= 1; m >>= 1) ss += __shfl_xor(ss, m);
        // Every group of column tiles has the same sums; the first eight leave them, one copy each, for the groups that are
        // a multiple of eight behind them.  A word says by itself that it is there, and is zero between launches.
        const int copy = grp % kStepNormCopies;
        unsigned long long* words = p.sync + kWordStride * (kStepNorm0 + copy) + wave;
        if (grp < kStepNormCopies && lane == 0) st_agent(words + kStepNormRows * chunk, 1ull << 32 | __float_as_uint(ss));
        if (grp == 0 && mine) *reinterpret_cast<u32x4*>(p.out_sum + wave * p.sum_rs + col) = sum;
        unsigned long long got = 0;
        bool there = true;
        for (unsigned spins = 1;; ++spins) {
            if (lane < p.chunks) got = ld_agent(words + kStepNormRows * lane);
            if (__all(lane >= p.chunks || got != 0)) break;
            __builtin_amdgcn_s_sleep(1);
            if (spins > p.spin_limit) st_agent(p.sync + kWordStride * kStepStatus, 1ull);
            if ((spins & 63) == 0 && ld_agent(p.sync + kWordStride * kStepStatus) != 0) {
                there = false;
                break;
            }
        }
        if (lane == 0) s_there[wave] = there;
        if (there) {
            float all = 0.f;
            for (int c = 0; c < p.chunks; ++c) all += __uint_as_float((unsigned)__builtin_amdgcn_readlane((int)(unsigned)got, c));
            const float inv = rsqrtf(all / (float)p.H + p.eps);
            u32x4 o;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t y = C::down2(C::lo(sum[i]) * inv, C::hi(sum[i]) * inv);
                o[i] = C::down2(C::lo(wv[i]) * C::lo(y), C::hi(wv[i]) * C::hi(y));
            }
            if (mine) *reinterpret_cast<u32x4*>(xs + wave * kRowB + 16 * lane) = o;
        }
    }
    __syncthreads();
    for (int m = 0; m < p.M; ++m)
        if (!s_there[m]) return;
    f32x4 c = {0.f, 0.f, 0.f, 0.f};
    const unsigned char* xb = xs + min(r, p.M - 1) * kRowB + 16 * kq;  // (rows past the last repeat it, nothing of them is stored)
#pragma unroll
    for (int u = 0; u < kChunkSteps; ++u)
        if (u < nst) c = mfma16<T>(a[u], *reinterpret_cast<const u32x4*>(xb + 64 * u), c);
    if (r < p.M && tile < tiles)
        *reinterpret_cast<f32x4*>(p.part + ((int64_t)chunk * 16 + r) * p.N + 16 * tile + 4 * kq) = c;
    // the last reader of a copy clears it
    if (wave == 0) {
        const int copy = grp % kStepNormCopies;
        const int readers = (p.groups - copy + kStepNormCopies - 1) / kStepNormCopies * p.chunks;
        unsigned long long* done = p.sync + kWordStride * (kStepNormDone0 + copy);
        int last = 0;
        if (lane == 0) last = add_agent(done, 1ull) == (unsigned long long)readers - 1;
        if (__builtin_amdgcn_readfirstlane(last)) {
            st_agent(p.sync + kWordStride * (kStepNorm0 + copy) + lane, 0ull);
            if (lane == 0) st_agent(done, 0ull);
        }
    }
}

int chunks_of(int H) { return (H + kChunkK - 1) / kChunkK; }
int groups_of(int N) { return (N / 16 + kWaves - 1) / kWaves; }

}  // namespace

extern "C" int ksa_add_rmsnorm_gemm_rows_splits(int M, int N, int H) {
    if (M <= 0 || M > kStepNormRows || N <= 0 || N % 16 != 0 || H <= 0 || H % 32 != 0 || H > kStepMaxHidden) return 0;
    return groups_of(N) * chunks_of(H) <= ksa_cu_count_or(256) ? chunks_of(H) : 0;
}

extern "C" int ksa_add_rmsnorm_gemm_rows(const float* partials, int ksplit, const void* residual, const void* norm_weight,
                                         void* out_sum, const void* weight, float* out_partials, int M, int N, int H,
                                         long long residual_row_stride, long long sum_row_stride, int dtype, float eps,
                                         void* step_workspace, size_t step_workspace_bytes, void* stream) {
    if (!partials || !residual || !norm_weight || !out_sum || !weight || !out_partials || !step_workspace) return KSA_ERR_NULL;
    if (M <= 0 || N <= 0 || H <= 0 || ksplit < 1 || ksplit > 64 || !(eps >= 0.f)) return KSA_ERR_INVALID;
    if (dtype != KSA_DTYPE_BF16 && dtype != KSA_DTYPE_F16) return KSA_ERR_UNSUPPORTED;
    if (M > kStepNormRows || N % 16 != 0 || H % 32 != 0 || H > kStepMaxHidden) return KSA_ERR_UNSUPPORTED;
    for (const void* ptr : {(const void*)partials, residual, norm_weight, (const void*)out_sum, weight,
                            (const void*)out_partials, (const void*)step_workspace})
        if (reinterpret_cast<uintptr_t>(ptr) & 15) return KSA_ERR_ALIGN;
    if (residual_row_stride % 8 || sum_row_stride % 8) return KSA_ERR_ALIGN;
    if (step_workspace_bytes < kStepBytes) return KSA_ERR_WORKSPACE;
    NormGemmParams p{};
    p.sync = (unsigned long long*)step_workspace;
    p.in = partials, p.ksplit = ksplit;
    p.res = (const uint16_t*)residual, p.nw = (const uint16_t*)norm_weight;
    p.out_sum = (uint16_t*)out_sum;
    p.res_rs = residual_row_stride, p.sum_rs = sum_row_stride;
    p.eps = eps;
    p.w = (const uint16_t*)weight;
    p.part = out_partials;
    p.M = M, p.H = H, p.N = N;
    p.chunks = chunks_of(H), p.groups = groups_of(N);
    p.spin_limit = 1u << 19;  // polls of a microsecond or two: about a second
    const dim3 grid(p.groups * p.chunks), block(kThreads);
    if (dtype == KSA_DTYPE_BF16)
        hipLaunchKernelGGL(ksa_norm_gemm_rows_kernel<KsaBf16>, grid, block, 0, (hipStream_t)stream, p);
    else
        hipLaunchKernelGGL(ksa_norm_gemm_rows_kernel<KsaF16>, grid, block, 0, (hipStream_t)stream, p);
    return ksa_check_launch();
}
