// Block-sparsity index for Summary Attention on gfx950.
//
// Produces the four int32 tensors of the reference's BlockSparsityKernel
//   flash_attn_cute wheel, flash_attn/cute/compute_block_sparsity.py:189-274
// (mask_block_cnt[M], mask_block_idx[M,N], full_block_cnt[M], full_block_idx[M,N];
//  zero padded, ascending n; classification over in-bounds elements only),
// but from the closed-form row counts in ksa_mask.h.  Two facts keep the work far below one count
// per (row, tile):
//   * Only two runs of n-tiles can hold anything for the rows of an m-tile: those that start below
//     the last row's old-summary bound, and those from the start of the first row's window to the
//     diagonal (`candidates`).  At 139264 rows that is 80 of 2304 tiles on average.
//   * Inside one chunk the visible sets of the text rows are nested (same window, growing causal
//     bound), and so are those of its summary rows.  "Some row sees something of the tile" is
//     decided by the last row of such a group, "some row misses something" by its first one: four
//     counts per chunk of the m-tile instead of one per row.
// One workgroup per m-tile compacts the classes of the candidates with wave ballots, which keeps
// the lists ascending without atomics, and zero-fills the tails with 16-byte stores: what is left is
// bound by the two index rows it writes.  Calls of 139264 x 147456 positions (20 MB of index) behind one another in a graph:
// 8.5 us with the compiler's divisions in the counts and the zeros behind them, 6.8 with one multiplication for a division, the
// zeros in front and past the caches: 3.3 us (6.2 TB/s, the rate of a large copy) above the 3.5 us of a call at 2000
// tokens.  256 threads a workgroup; 512 / 128 / 64 3.0 / 0.7 / 1.3 us slower.
#include <hip/hip_runtime.h>

#include "ksa_api_internal.h"
#include "ksa_mask.h"

namespace {

constexpr int kIdxThreads = 256;
typedef int32_t i32x4 __attribute__((ext_vector_type(4)));

// row[from, N) = 0 by the whole workgroup
__device__ __forceinline__ void zero_range(int32_t* row, int from, int N, int tid) {
    if (from >= N) return;
    const int lead = (int)((16 - (reinterpret_cast<uintptr_t>(row + from) & 15)) & 15) / 4;  // to the next 16-byte border
    const int body = from + min(lead, N - from);
    if (from + tid < body) row[from + tid] = 0;
    const int quads = (N - body) / 4;
    i32x4* q = reinterpret_cast<i32x4*>(row + body);
    for (int i = tid; i < quads; i += kIdxThreads) __builtin_nontemporal_store(i32x4{0, 0, 0, 0}, q + i);
    const int rest = body + 4 * quads;
    if (rest + tid < N) row[rest + tid] = 0;
}

__global__ __launch_bounds__(kIdxThreads) void ksa_block_index_kernel(
    KsaMask mk, FastDiv by_block, int tile_m, int tile_n, int N, int32_t* __restrict__ mask_cnt,
    int32_t* __restrict__ mask_idx, int32_t* __restrict__ full_cnt,
    int32_t* __restrict__ full_idx) {
    const int m = blockIdx.x;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    constexpr int kWaves = kIdxThreads / 64;
    __shared__ int s_part[kWaves], s_full[kWaves];

    const int q0 = m * tile_m;
    const int q1 = min(mk.Sq, q0 + tile_m);
    const int B = mk.C + mk.S;
    const int c_first = by_block.div(q0), c_last = by_block.div(q1 - 1);
    int32_t* mrow = mask_idx + (size_t)m * N;
    int32_t* frow = full_idx + (size_t)m * N;
    int run_part = 0, run_full = 0;

    // candidates: n in [0, n_a) (old summaries of the last chunk's text rows; in-line mode has none there)
    // and in [n_b, n_e) (window or own chunk of the first row up to the diagonal; in-line mode without
    // skip_old sees old summaries anywhere in front of the window)
    const int w_first = c_first > mk.W ? c_first - mk.W : 0;
    const int w_last = c_last > mk.W ? c_last - mk.W : 0;
    const int n_e = min(N, (mk.P + q1 - 1) / tile_n + 1);
    const int n_a = (mk.P > 0 && !mk.skip_old) ? min(n_e, (w_last * mk.S + tile_n - 1) / tile_n) : 0;
    const int n_b = max(n_a, (mk.P > 0 || mk.skip_old) ? (mk.P + w_first * B) / tile_n : 0);
    const int ncand = n_a + max(n_e - n_b, 0);
    // the unused tails are zero, so that callers may hand in uninitialised buffers: what no candidate can reach, nearly
    // all of it, is on its way before the first count
    const int most = min(ncand, N);
    zero_range(mrow, most, N, tid);
    zero_range(frow, most, N, tid);

    for (int base = 0; base < ncand; base += kIdxThreads) {
        const int i = base + tid;
        const int n = i < n_a ? i : n_b + (i - n_a);
        int cls = 0;  // 0 empty, 1 partial, 2 full
        if (i < ncand) {
            const int32_t a = n * tile_n;
            const int32_t b = ksa_imin(mk.Sk, a + tile_n);
            const int32_t width = b - a;
            bool any_vis = false, any_hid = false;
            for (int c = c_first; c <= c_last && !(any_vis && any_hid); ++c) {
                const int32_t r0 = ksa_imax(q0, c * B), rs = c * B + mk.C, r1 = ksa_imin(q1, (c + 1) * B);
                const int32_t t1 = ksa_imin(r1, rs), u0 = ksa_imax(r0, rs);  // text rows [r0, t1), summary rows [u0, r1)
                if (r0 < t1) {
                    any_vis |= ksa_count_visible(mk, t1 - 1, a, b, by_block) > 0;
                    any_hid |= ksa_count_visible(mk, r0, a, b, by_block) < width;
                }
                if (u0 < r1) {
                    any_vis |= ksa_count_visible(mk, r1 - 1, a, b, by_block) > 0;
                    any_hid |= ksa_count_visible(mk, u0, a, b, by_block) < width;
                }
            }
            cls = any_vis ? (any_hid ? 1 : 2) : 0;
        }
        const uint64_t bp = __ballot(cls == 1);
        const uint64_t bf = __ballot(cls == 2);
        if (lane == 0) {
            s_part[wave] = __popcll(bp);
            s_full[wave] = __popcll(bf);
        }
        __syncthreads();
        int off_p = run_part, off_f = run_full, tot_p = 0, tot_f = 0;
        for (int w = 0; w < kWaves; ++w) {
            if (w < wave) {
                off_p += s_part[w];
                off_f += s_full[w];
            }
            tot_p += s_part[w];
            tot_f += s_full[w];
        }
        const uint64_t below = (1ull << lane) - 1ull;
        if (cls == 1) mrow[off_p + __popcll(bp & below)] = n;
        if (cls == 2) frow[off_f + __popcll(bf & below)] = n;
        run_part += tot_p;
        run_full += tot_f;
        __syncthreads();
    }
    zero_range(mrow, run_part, most, tid);
    zero_range(frow, run_full, most, tid);
    if (tid == 0) {
        mask_cnt[m] = run_part;
        full_cnt[m] = run_full;
    }
}

}  // namespace

extern "C" int ksa_block_index(int Sq, int Sk, int C, int S, int W, int P, int skip_old, int tile_m,
                               int tile_n, int32_t* mask_cnt, int32_t* mask_idx, int32_t* full_cnt,
                               int32_t* full_idx, void* stream) {
    if (Sq <= 0 || Sk < Sq || C <= 0 || S <= 0 || W < 0 || tile_m <= 0 || tile_n <= 0)
        return KSA_ERR_INVALID;
    if (P != Sk - Sq) return KSA_ERR_INVALID;
    if (!mask_cnt || !mask_idx || !full_cnt || !full_idx) return KSA_ERR_NULL;
    const int M = (Sq + tile_m - 1) / tile_m;
    const int N = (Sk + tile_n - 1) / tile_n;
    const KsaMask mk = ksa_make_mask(C, S, W, P, skip_old, Sq, Sk);
    hipLaunchKernelGGL(ksa_block_index_kernel, dim3(M), dim3(kIdxThreads), 0, (hipStream_t)stream,
                       mk, FastDiv((uint32_t)(mk.C + mk.S)), tile_m, tile_n, N, mask_cnt, mask_idx, full_cnt, full_idx);
    return ksa_check_launch();
}

extern "C" long long ksa_debug_count_visible(long long q, long long a, long long b, int C, int S,
                                             int W, int P, int skip_old, int Sq, int Sk) {
    KsaMask mk{C, S, W, P, skip_old ? 1 : 0, Sq, Sk};
    if (a < 0) a = 0;
    if (b > Sk) b = Sk;
    if (b <= a) return 0;
    return ksa_count_visible(mk, (int)q, (int)a, (int)b, KsaPlainDiv{C + S});
}
