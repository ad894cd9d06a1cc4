// Residual add + RMSNorm and the product behind them at a decode step as ONE launch (gfx950):
//
//   x' = residual + sum of the K-split partial sums of the product in front    (modeling_qwen3sa.py:950-952)
//   y  = (norm(x') w) W^T, left as K-split partial sums                        (:938, :660-662, the next layer's q | k | v)
//
// for at most 8 rows.  The norm is a chain of memory trips of one workgroup per row that leaves the other CUs idle, and the
// product's weights (31 MB at 6144 x 2560) could only start to move behind it.  Here the first workgroups of the grid add
// up the rows, 512 columns each, and hand over x' and the sum of squares of their columns; those of the product, behind
// them, own eight column tiles of 16 (one per wave) times one chunk of 512 elements of K, request all their weights at once,
// wait for the sums of all chunks of the rows and scale their own.  What bounds it is that chain - slices, hand-over, x',
// product; the weights travel next to it.  us, the two launches / this one, by rows (19 slices to add, 2560 x 6144): 1 11.7 /
// 8.7, 2 12.0 / 9.0, 4 12.2 / 9.7, 8 12.6 / 11.3.  Other forms: a whole row per workgroup at the head of the grid 13.3 at one
// row (the row alone is 194 KB through one CU, behind the others' weights); every workgroup adding up its chunk of the
// rows for itself, with only the squares handed over, 8.6 / 10.2 / 12.1 at 1 / 2 / 4 rows; the weights held back by 1 us
// 9.5 / 9.7 / 10.3.
#include <hip/hip_runtime.h>

#include "ksa_api_internal.h"
#include "ksa_cvt.h"
#include "ksa_rows_mfma.h"
#include "ksa_rows_sync.h"

namespace {

constexpr int kThreads = 512;
constexpr int kWaves = kThreads / 64;
constexpr int kMaxRows = kStepNormRows;
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
    unsigned long long* xbuf;  // x' for this launch [M][H / 4], four values per word
    int M, H, N, ksplit, chunks, wgs;  // wgs: workgroups of the product
    int heads, head_rows;              // workgroups of the sums, rows of each (1 .. 4)
    float eps;
    unsigned spin_limit;
};

__device__ __forceinline__ unsigned long long* norm_words(unsigned long long* sync, int copy) {
    return sync + kWordStride * (kStepNorm0 + copy);
}

// one chunk of the rows row0 .. (up to four, two waves each): their sums, four columns per thread
template <typename T>
__device__ __forceinline__ void norm_chunk(const NormGemmParams& p, int row0, int chunk, int nst, unsigned char* lds) {
    using C = KsaCvt<T>;
    const int tid = threadIdx.x, end = min(row0 + p.head_rows, p.M);
    const int piece = tid & 127;
    int row = row0 + (tid >> 7);
    if (row < end && piece < 8 * nst) {
        const int col = chunk * kChunkK + 4 * piece;
        const float* src = p.in + (int64_t)row * p.H + col;
        const int64_t pitch = (int64_t)16 * p.H;
        f32x4 v[kSlices];
#pragma unroll
        for (int k = 0; k < kSlices; ++k) v[k] = *reinterpret_cast<const f32x4*>(src + pitch * min(k, p.ksplit - 1));
        const u32x2 q = *reinterpret_cast<const u32x2*>(p.res + row * p.res_rs + col);
        f32x4 ac = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < kSlices; ++k)
            if (k < p.ksplit) ac += v[k];
        for (int k = kSlices; k < p.ksplit; ++k) ac += *reinterpret_cast<const f32x4*>(src + pitch * k);
        u32x2 sum;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint32_t x = C::down2(ac[2 * i], ac[2 * i + 1]);
            sum[i] = C::down2(C::lo(x) + C::lo(q[i]), C::hi(x) + C::hi(q[i]));
        }
        st_agent(p.xbuf + ((int64_t)row * p.H + col) / 4, (unsigned long long)sum[0] | (unsigned long long)sum[1] << 32);
        *reinterpret_cast<u32x2*>(p.out_sum + row * p.sum_rs + col) = sum;
        *reinterpret_cast<u32x2*>(lds + 8 * tid) = sum;
    }
    __builtin_amdgcn_s_waitcnt(0);  // this thread's piece has left; the barrier says so of all
    __syncthreads();
    const int lane = tid & 63;
    row = row0 + (tid >> 6);
    if (row < end) {  // one wave per row (in the order of ksa_add_rmsnorm_partials, one of whose waves has these columns)
        float ss = 0.f;
        if (lane < 4 * nst) {
            const u32x4 x = *reinterpret_cast<const u32x4*>(lds + 1024 * (tid >> 6) + 16 * lane);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float a_ = C::lo(x[i]), b_ = C::hi(x[i]);
                ss = fmaf(a_, a_, ss);
                ss = fmaf(b_, b_, ss);
            }
        }
#pragma unroll
        for (int m = 32; m >= 1; m >>= 1) ss += __shfl_xor(ss, m);
        // (a word says by itself that it is there, and is zero between launches)
        if (lane < min(kStepNormCopies, p.wgs))  // (a copy without readers would not be cleared)
            st_agent(norm_words(p.sync, lane) + kMaxRows * chunk + row, 1ull << 32 | __float_as_uint(ss));
    }
}

template <typename T>
__global__ __launch_bounds__(kThreads, 4) void ksa_norm_gemm_rows_kernel(const NormGemmParams p) {
    using C = KsaCvt<T>;
    __shared__ __attribute__((aligned(16))) unsigned char xs[kMaxRows * kRowB];
    __shared__ int s_there[kWaves];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int tiles = p.N / 16, steps = p.H / 32;
    if ((int)blockIdx.x < p.heads) {
        const int rb = blockIdx.x / p.chunks, chunk = blockIdx.x - rb * p.chunks;
        norm_chunk<T>(p, rb * p.head_rows, chunk, min(kChunkSteps, steps - chunk * kChunkSteps), xs);
        return;
    }
    const int idx = blockIdx.x - p.heads;
    const int grp = idx / p.chunks, chunk = idx - grp * p.chunks;
    const int r = lane & 15, kq = lane >> 4;
    const int tile = grp * kWaves + wave;
    const int nst = min(kChunkSteps, steps - chunk * kChunkSteps);
    const bool mine = lane < nst * 4;
    const int col = chunk * kChunkK + 8 * min(lane, nst * 4 - 1);
    const u32x4 wv = *reinterpret_cast<const u32x4*>(p.nw + col);
    // (a wave past the last tile repeats it, steps past the end of a short chunk its last one; nothing of them is used)
    const KsaWeightLane wl = ksa_weight_lane(p.w, kWTiled, p.H, 16 * (int64_t)min(tile, tiles - 1), r, kq, p.N);
    u32x4 a[kChunkSteps];
#pragma unroll
    for (int u = 0; u < kChunkSteps; ++u)
        a[u] = ksa_load_weights<true>(wl.p + (int64_t)wl.step * (chunk * kChunkSteps + min(u, nst - 1)));

    // this wave's row: lane c watches chunk c
    const int copy = idx % kStepNormCopies;
    bool there = true;
    if (wave < p.M) {
        const bool live = lane < p.chunks;
        const unsigned long long* word = norm_words(p.sync, copy) + kMaxRows * (lane % kWaves) + wave;
        unsigned long long got = 0;
        for (unsigned spins = 1;; ++spins) {
            if (live) got = ld_agent(word);
            if (__all(!live || got != 0)) break;
            __builtin_amdgcn_s_sleep(1);
            if (spins > p.spin_limit) st_agent(p.sync + kWordStride * kStepStatus, 1ull);
            if ((spins & 63) == 0 && ld_agent(p.sync + kWordStride * kStepStatus) != 0) {
                there = false;
                break;
            }
        }
        if (there) {
            const KsaAgentBuffer xb(p.xbuf, (uint32_t)(p.M * p.H) * 2u);  // past this XCD's L2
            const u32x4 sum = xb.ld4((uint32_t)(wave * p.H + col) * 2u);
            float all = 0.f;
            for (int k = 0; k < p.chunks; ++k) all += __uint_as_float((unsigned)__builtin_amdgcn_readlane((int)(unsigned)got, k));
            const float inv = rsqrtf(all / (float)p.H + p.eps);
            u32x4 o;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint32_t y = C::down2(C::lo(sum[e]) * inv, C::hi(sum[e]) * inv);
                o[e] = C::down2(C::lo(wv[e]) * C::lo(y), C::hi(wv[e]) * C::hi(y));
            }
            if (mine) *reinterpret_cast<u32x4*>(xs + wave * kRowB + 16 * lane) = o;
        }
    }
    if (lane == 0) s_there[wave] = there;
    __syncthreads();
    for (int w = 0; w < kWaves; ++w)
        if (!s_there[w]) return;
    f32x4 c = {0.f, 0.f, 0.f, 0.f};
    const unsigned char* xb = xs + min(r, p.M - 1) * kRowB + 16 * kq;  // (rows past the last repeat it, nothing of them is stored)
#pragma unroll
    for (int u = 0; u < kChunkSteps; ++u)
        if (u < nst) c = mfma16<T>(a[u], *reinterpret_cast<const u32x4*>(xb + 64 * u), c);
    if (r < p.M && tile < tiles)
        *reinterpret_cast<f32x4*>(p.part + ((int64_t)chunk * 16 + r) * p.N + 16 * tile + 4 * kq) = c;
    // the last reader of a copy clears it
    if (wave == 0) {
        unsigned long long* done = p.sync + kWordStride * (kStepNormDone0 + copy);
        const int readers = (p.wgs - copy + kStepNormCopies - 1) / kStepNormCopies;
        int last = 0;
        if (lane == 0) last = add_agent(done, 1ull) == (unsigned long long)readers - 1;
        if (__builtin_amdgcn_readfirstlane(last)) {
            st_agent(norm_words(p.sync, copy) + lane, 0ull);
            if (lane == 0) st_agent(done, 0ull);
        }
    }
}

int chunks_of(int H) { return (H + kChunkK - 1) / kChunkK; }
int groups_of(int N) { return (N / 16 + kWaves - 1) / kWaves; }

}  // namespace

extern "C" int ksa_add_rmsnorm_gemm_rows_splits(int M, int N, int H) {
    if (M <= 0 || M > kStepNormRows || N <= 0 || N % 16 != 0 || H <= 0 || H % 32 != 0 || H > kStepMaxHidden) return 0;
    return chunks_of(H);
}

// Whether the one launch is the faster way.  It saves the norm's launch, which takes longer with long rows and many slices, and
// pays with the hand-over, which takes longer with many rows.  Timed against add_rmsnorm + ksa_gemm_rows at 23 shapes (H 544 to
// 4096, N 16 to 16384), 4 to 37 slices, 1 to 8 rows, 1610 in all: 1018 are taken, at 0.87 of the two launches on average, 1.04 at
// the worst (8 rows of 3072 x 5120, 12 slices).  Outside, by line: short rows of few slices (1024 x 4096, 8 slices, 1 / 8 rows 1.00 / 1.07); more slices than are requested at once, which then come one behind the other (37 slices of 2560 x
// 6144, 4 / 8 rows 1.00 / 1.07; 24 of 3072 x 5120, 8 rows 1.09, but of 4096 x 6144 0.91); a product wide against its rows (2560 x 16384
// 1.03 to 1.15, 2048 x 16384, 24 slices 0.98 to 1.10); more than 4 rows of few slices (2560 x 12288, 8 rows, 4 slices 1.04), or up to 16
// where a few workgroups of the product come in a second round (3840 x 4352, 272 of them, 9 slices 1.03 to 1.09).
extern "C" int ksa_add_rmsnorm_gemm_rows_pays(int M, int N, int H, int ksplit) {
    const int cus = ksa_cu_count_or(256);
    if (ksa_add_rmsnorm_gemm_rows_splits(M, N, H) == 0) return 0;
    const int wgs = groups_of(N) * chunks_of(H);
    if (wgs > 3 * cus || N > 6 * H || ksplit > (M <= 6 || H > 3584 ? 28 : 20)) return 0;
    if (M <= 4) return ksplit > (H >= 2048 ? 0 : 16);
    const bool few_more = wgs > cus && 4 * wgs <= 5 * cus;
    return ksplit > (H >= 2048 && !few_more ? 8 : 16);
}

namespace {
// `spin_limit` polls of a microsecond or two at the most; without `sums` nobody leaves what the product waits for
int norm_gemm_rows(const float* partials, int ksplit, const void* residual, const void* norm_weight, void* out_sum,
                   const void* weight, float* out_partials, int M, int N, int H, long long residual_row_stride,
                   long long sum_row_stride, int dtype, float eps, void* step_workspace, size_t step_workspace_bytes,
                   bool sums, unsigned spin_limit, void* stream) {
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
    p.xbuf = p.sync + kStepWords * kWordStride;
    p.w = (const uint16_t*)weight;
    p.part = out_partials;
    p.M = M, p.H = H, p.N = N;
    p.chunks = chunks_of(H), p.wgs = groups_of(N) * p.chunks;
    // as few rows to a workgroup of the sums as leave every workgroup a CU of its own (4 / 8 rows of 2560 x 6144: 20 / 40
    // workgroups next to the 240 of the product 10.7 / 11.7 us, 10 / 15 of them 9.7 / 11.3); one where no number does (3584 x 4608, 252 of
    // the product, 24 slices: 4 rows in one workgroup 14.8 us, one each 12.8)
    const int cus = ksa_cu_count_or(256);
    auto heads = [&](int rows) { return (M + rows - 1) / rows * p.chunks; };
    p.head_rows = 1;
    while (p.head_rows < 4 && heads(p.head_rows) + p.wgs > cus && heads(4) + p.wgs <= cus) ++p.head_rows;
    p.heads = heads(p.head_rows);
    if (!sums) p.heads = 0;
    p.spin_limit = spin_limit;
    const dim3 grid(p.heads + p.wgs), block(kThreads);
    if (dtype == KSA_DTYPE_BF16)
        hipLaunchKernelGGL(ksa_norm_gemm_rows_kernel<KsaBf16>, grid, block, 0, (hipStream_t)stream, p);
    else
        hipLaunchKernelGGL(ksa_norm_gemm_rows_kernel<KsaF16>, grid, block, 0, (hipStream_t)stream, p);
    return ksa_check_launch();
}
}  // namespace

extern "C" int ksa_add_rmsnorm_gemm_rows(const float* partials, int ksplit, const void* residual, const void* norm_weight,
                                         void* out_sum, const void* weight, float* out_partials, int M, int N, int H,
                                         long long residual_row_stride, long long sum_row_stride, int dtype, float eps,
                                         void* step_workspace, size_t step_workspace_bytes, void* stream) {
    return norm_gemm_rows(partials, ksplit, residual, norm_weight, out_sum, weight, out_partials, M, N, H,
                          residual_row_stride, sum_row_stride, dtype, eps, step_workspace, step_workspace_bytes, true,
                          1u << 19, stream);  // (about a second)
}

extern "C" int ksa_debug_norm_gemm_rows_give_up(const float* partials, int ksplit, const void* residual,
                                                const void* norm_weight, void* out_sum, const void* weight,
                                                float* out_partials, int M, int N, int H, int dtype, float eps,
                                                void* step_workspace, size_t step_workspace_bytes, void* stream) {
    return norm_gemm_rows(partials, ksplit, residual, norm_weight, out_sum, weight, out_partials, M, N, H, H, H, dtype, eps,
                          step_workspace, step_workspace_bytes, false, 200, stream);
}
