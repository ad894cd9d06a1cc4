// Decode attention over the contiguous ring-buffer KV slice for gfx950.
//
// Replaces the reference's decode attention function
//   examples/pretrain/hf_template/modeling_qwen3sa.py:591-612 (_sdpa_attention_forward)
//   examples/pretrain/hf_template/modeling_qwen3sa.py:557-566 (repeat_kv)
// i.e. softmax(q K^T * scale) V without any mask over rows [start_b, end_b) of the
// cache slice returned by Qwen3RingBufferCache.get_attention_kv (:402-434).  The
// reference materialises g copies of K and V per step; here every K/V row is read
// from HBM exactly once per kv head and shared by the g query heads (and by all
// query tokens of a chunk-boundary step) as columns of one MFMA tile.
//
// Split-K: a workgroup owns (sequence, kv head, split); its 4 waves stream disjoint
// 32-row tiles with private LDS staging (no workgroup barrier in the loop) and keep
// private (max, sum, O^T) state that is merged across the waves through LDS at the
// end; with more than one split the un-normalised partials go to a workspace and a
// second kernel merges them.
//
// A one-token step of the decoder can hand over the K-split partial sums of its fused q | k | v projection instead
// of q (kPre): the kernel then does the pre-attention step itself - sums, norm and rotary embedding of the query
// rows of its group in every workgroup, of the new key and value rows in the one workgroup whose
// slice holds their cache row - one launch, and one round trip of the rows through memory, less.
//
// With kO the launch also holds the o projection behind the attention: see ksa_decode_o_stage.
#include <hip/hip_runtime.h>
#include <math.h>

#include <mutex>
#include <type_traits>

#include "ksa_api_internal.h"
#include "ksa_pre_row.h"
#include "ksa_rows_mfma.h"
#include "ksa_rows_sync.h"
#include "ksa_tile.h"

namespace {

struct DecodeParams {
    const uint16_t* q;
    const uint16_t* k;
    const uint16_t* v;
    uint16_t* out;
    const int32_t* start;  // per sequence or null
    const int32_t* end;
    int start0, end0;
    int Hq, Hkv, g, Q;
    int ncols;   // Q * g columns per kv head
    int nsplit;
    int64_t q_bs, q_hs, q_qs;   // element strides of q [B,Hq,Q,D]
    int64_t k_bs, k_hs, k_rs;   // cache [B,Hkv,rows,D]
    int64_t v_bs, v_hs, v_rs;
    int64_t o_bs, o_qs, o_hs;   // out [B,Q,Hq,D]
    float* ws_o;   // [B,Hkv,nsplit,ncols_pad,D] un-normalised partial outputs
    float* ws_ml;  // [B,Hkv,nsplit,ncols_pad,2]  (max in log2 units, sum)
    int ncols_pad;
    float scale_log2;
    int wide;      // workgroups of eight waves (ksa_decode_wide_kernel)
    // Chunk-boundary form (split_q != 0): query token 0 (the chunk's last text token) attends the rows
    // [start, end) and has column block 0 to itself (g columns); the other Q - 1 query tokens (the
    // chunk's summary tokens) attend [start2, end2) and fill the column blocks behind it.
    int split_q;
    const int32_t* start2;
    const int32_t* end2;
    int start20, end20;
    // kPre: one new token per sequence, from the projection's partial sums (q and q_bs .. are then unused)
    const float* qkv;           // [qkv_ksplit][qkv_prows][(Hq + 2 Hkv) D]
    int qkv_ksplit, qkv_prows;
    const uint16_t* wq;         // norm weights [D]
    const uint16_t* wk;
    const uint16_t* cos;        // rotary row of the token [D], batch stride c_bs
    const uint16_t* sin;
    int64_t c_bs;
    float eps;
    uint16_t* kw;               // the caches, to be written at the new row
    uint16_t* vw;
    const int32_t* row_seq;     // cache row of the new token per sequence, or null: row0
    int row0;
};
// kO: the o projection in the same launch
struct DecodeOParams : DecodeParams {
    const uint16_t* o_w;        // streaming layout [o_n / 16][Hq D / 32][1 KB]
    float* o_part;              // [o_chunks][16][o_n]
    unsigned long long* sync;
    int batch, n_attn;          // n_attn: workgroups of the attention
    int o_n, o_chunks, o_wgs;
    unsigned spin_limit;
};

// column lq of column block colblk -> (query token, head in the group); false: no such column
__device__ __forceinline__ bool ksa_decode_column(const DecodeParams& p, int colblk, int lq, int& qi, int& gi) {
    if (!p.split_q) {
        const int col = colblk * 32 + lq;
        qi = col / p.g, gi = col % p.g;
        return col < p.ncols;
    }
    if (colblk == 0) {
        qi = 0, gi = lq;
        return lq < p.g;
    }
    const int c = (colblk - 1) * 32 + lq;
    qi = 1 + c / p.g, gi = c % p.g;
    return c < (p.Q - 1) * p.g;
}
// slot of the logical column (query token qi, head gi) in the workspace's column axis
__device__ __forceinline__ int ksa_decode_slot(const DecodeParams& p, int qi, int gi) {
    if (!p.split_q) return qi * p.g + gi;
    return qi == 0 ? gi : 32 + (qi - 1) * p.g + gi;
}

typedef float floatx4 __attribute__((ext_vector_type(4)));
// the same as the caller's workspace holds them: on any 4-byte border (still one wide load each)
typedef float floatx4_ws __attribute__((ext_vector_type(4), aligned(4)));
typedef float floatx2_ws __attribute__((ext_vector_type(2), aligned(4)));

constexpr int kThreads = 256;
constexpr int kWaves = 4;
constexpr int kRows = 32;  // key rows per wave tile

// The o projection (modeling_qwen3sa.py:879) behind the attention of a one-token step, at most 16 rows: a workgroup owns
// 128 columns (two tiles of 16 per wave) times one chunk of 512 elements of K, i.e. 512 / D heads.  It requests all its
// weights at once, waits until the attention workgroups of those heads have left their sums, merges the splits of its
// heads into the rows of x and multiplies.  Against the three launches it stands for the weights (21 MB at 4096 x 2560) move
// while the attention runs, and two ramps and a trip of the rows through memory are gone; what bounds it is the chain
// projection sums - scores - sums - merge - product (figures at ksa_decode_qkv_o_splits).  Every workgroup merges for
// itself, rows x splits x 2 KB of sums, 131 KB at the most (kMaxOSums), which is why it has 128 columns and not fewer.
// In a launch of workgroups of NW = 8 waves, of which a CU holds one, a workgroup owns 256 columns: half as many of them hold
// a CU back from the attention.
constexpr int kMaxOSums = 64;  // rows x splits
template <typename T, int D, int NW>
__device__ __forceinline__ void ksa_decode_o_stage(const DecodeOParams& p, int idx, unsigned char* smem) {
    using Ops = KsaOps<T>;
    constexpr int HPC = kChunkK / D;   // heads of a chunk
    constexpr int kCols = 2;           // column tiles of a wave
    constexpr int kBatch = 16;         // splits requested at a time
    constexpr int kParts = NW / 2;     // groups of 128 threads, a piece of four elements of x each
    constexpr int kMl = (kMaxOSums * HPC + 64 * NW - 1) / (64 * NW);  // maxima and sums of a thread
    __shared__ int s_there;
    unsigned char* xs = smem;                                                    // [16][kRowB]
    float* s_m = reinterpret_cast<float*>(smem + 16 * kRowB);                    // [rows][HPC][splits]
    floatx2_ws* s_f = reinterpret_cast<floatx2_ws*>(s_m + kMaxOSums * HPC);      // factor and factor x sum
    floatx4* s_part = reinterpret_cast<floatx4*>(s_f + kMaxOSums * HPC);         // [kParts - 1][128] sums of the other parts, their l
    float* s_part_l = reinterpret_cast<float*>(s_part + (kParts - 1) * 128);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, kq = lane >> 4;
    const int grp = idx / p.o_chunks, chunk = idx - grp * p.o_chunks;
    const int tiles = p.o_n / 16, steps = p.Hq * D / 32;
    u32x4 a[kCols][kChunkSteps];
#pragma unroll
    for (int t = 0; t < kCols; ++t) {
        const int tile = min(grp * (NW * kCols) + wave * kCols + t, tiles - 1);
        const char* wt = reinterpret_cast<const char*>(p.o_w) + ((int64_t)tile * steps + chunk * kChunkSteps) * 1024;
#pragma unroll
        for (int u = 0; u < kChunkSteps; ++u)
            a[t][u] = ksa_load_weights<true>(reinterpret_cast<const uint16_t*>(wt + u * 1024 + (uint32_t)(64 * r + 16 * kq)));
    }
    const int ns = p.nsplit, M = p.batch;
    // this thread's maxima and sums (row, head, split) and its piece of four elements of x
    const uint32_t slot_step = (uint32_t)p.ncols_pad, row_step = (uint32_t)(p.Hkv * ns) * slot_step;
    const int count = M * HPC * ns;
    uint32_t ml_off[kMl];
#pragma unroll
    for (int i = 0; i < kMl; ++i) {
        const int e = min(tid + 64 * NW * i, count - 1);
        const int rh = e / ns, sp = e - rh * ns, hh = rh % HPC, head = chunk * HPC + hh;
        const int kvh = head / p.g;
        ml_off[i] = ((uint32_t)(rh / HPC) * row_step + (uint32_t)(kvh * ns + sp) * slot_step + (uint32_t)(head - kvh * p.g)) * 8u;
    }
    const int piece = tid & 127, part = wave >> 1;
    const int hh = 4 * piece / D, head = chunk * HPC + hh, kvh = head / p.g;
    const uint32_t o_off = (((uint32_t)(kvh * ns) * slot_step + (uint32_t)(head - kvh * p.g)) * D + (uint32_t)(4 * piece % D)) * 4u;

    // The entries of a thread: rows part, part + kParts, .. with all their splits one after the other; of a single row the parts take
    // every kParts-th split.  Lane j holds entry j: the offset of its sums; the place of its factor and, in
    // the upper half behind the last split of a row, the row + 1.
    const bool one = M == 1;
    const int n = one ? (ns - part + kParts - 1) / kParts : (M - part + kParts - 1) / kParts * ns;  // at most 64
    const int erow = one ? 0 : part + kParts * (lane / ns), esp = one ? kParts * lane + part : lane % ns;
    const uint32_t ent_off = ((uint32_t)erow * row_step + (uint32_t)esp * slot_step) * (uint32_t)(D * 4);
    const int ent = (erow * HPC * ns + esp) | (!one && esp == ns - 1 ? (erow + 1) << 16 : 0);

    if (wave == 0) {
        const int kv0 = chunk * HPC / p.g, kv1 = (chunk * HPC + HPC - 1) / p.g;
        const bool there = ksa_wave_wait(p.sync + kWordStride * (kStepHead0 + min(kv0 + lane, kv1)), lane <= kv1 - kv0,
                                         (long long)M * ns, p.sync + kWordStride * kStepStatus, p.spin_limit);
        if (lane == 0) s_there = there;
    }
    __syncthreads();
    if (!s_there) return;

    const uint32_t slots = (uint32_t)M * row_step;
    const KsaAgentBuffer so(p.ws_o, slots * D * 4u), sml(p.ws_ml, slots * 8u);
    floatx2_ws ml[kMl];
#pragma unroll
    for (int i = 0; i < kMl; ++i) ml[i] = __builtin_bit_cast(floatx2_ws, sml.ld2(ml_off[i]));
    floatx4 o[kBatch];
    auto request = [&](int j0) {
#pragma unroll
        for (int u = 0; u < kBatch; ++u)
            if (j0 + u < n) o[u] = __builtin_bit_cast(floatx4, so.ld4(o_off, (uint32_t)__builtin_amdgcn_readlane((int)ent_off, j0 + u)));
    };
    request(0);
#pragma unroll
    for (int i = 0; i < kMl; ++i)
        if (tid + 64 * NW * i < count) s_m[tid + 64 * NW * i] = ml[i][0];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kMl; ++i) {
        const int e = tid + 64 * NW * i;
        if (e < count) {
            const int e0 = e / ns * ns;
            float mx = -INFINITY;
            for (int j = 0; j < ns; ++j) mx = fmaxf(mx, s_m[e0 + j]);
            const float m = ml[i][0];
            // (an empty slice leaves its sums unwritten: nothing of it may enter, not even times zero)
            const float f = m == -INFINITY ? -1.f : ksa_exp2(m - mx);
            s_f[e] = floatx2_ws{f, m == -INFINITY ? 0.f : f * ml[i][1]};
        }
    }
    __syncthreads();
    floatx4 acc = {0.f, 0.f, 0.f, 0.f};
    float l = 0.f;
    auto x_store = [&](int row) {
        const float inv = l > 0.f ? 1.f / l : 0.f;
        u32x2 w;
        w[0] = Ops::pack2(acc[0] * inv, acc[1] * inv), w[1] = Ops::pack2(acc[2] * inv, acc[3] * inv);
        *reinterpret_cast<u32x2*>(xs + row * kRowB + 8 * piece) = w;
    };
    for (int j0 = 0; j0 < n; j0 += kBatch) {
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {
            if (j0 + u < n) {
                const int e = __builtin_amdgcn_readlane(ent, j0 + u);
                const floatx2_ws f = s_f[(e & 0xffff) + hh * ns];
                const bool live = f[0] >= 0.f;
                l += f[1];
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[i] = fmaf(live ? o[u][i] : 0.f, f[0], acc[i]);
                if (e >> 16) {
                    x_store((e >> 16) - 1);
                    acc = floatx4{0.f, 0.f, 0.f, 0.f}, l = 0.f;
                }
            }
        }
        if (j0 + kBatch < n) request(j0 + kBatch);
    }
    if (one) {
        if (part) s_part[(part - 1) * 128 + piece] = acc, s_part_l[(part - 1) * 128 + piece] = l;
        __syncthreads();
        if (!part) {
#pragma unroll
            for (int i = 0; i < kParts - 1; ++i) acc += s_part[i * 128 + piece], l += s_part_l[i * 128 + piece];
            x_store(0);
        }
    }
    __syncthreads();
    f32x4 c[kCols];
#pragma unroll
    for (int t = 0; t < kCols; ++t) c[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    const unsigned char* xb = xs + min(r, M - 1) * kRowB + 16 * kq;  // (rows past the last repeat it, nothing of them is stored)
#pragma unroll
    for (int u = 0; u < kChunkSteps; ++u) {
        const u32x4 b = *reinterpret_cast<const u32x4*>(xb + 64 * u);
#pragma unroll
        for (int t = 0; t < kCols; ++t) c[t] = mfma16<T>(a[t][u], b, c[t]);
    }
#pragma unroll
    for (int t = 0; t < kCols; ++t) {
        const int tile = grp * (NW * kCols) + wave * kCols + t;
        if (r < M && tile < tiles)
            *reinterpret_cast<f32x4*>(p.o_part + ((int64_t)chunk * 16 + r) * p.o_n + 16 * tile + 4 * kq) = c[t];
    }
    // (everybody who counts here has seen the sums)
    if (tid == 0 && add_agent(p.sync + kWordStride * kStepAttnDone, 1ull) == (unsigned long long)p.o_wgs - 1) {
        for (int h = 0; h < p.Hkv; ++h) add_agent(p.sync + kWordStride * (kStepHead0 + h), -(unsigned long long)(M * ns));
        st_agent(p.sync + kWordStride * kStepAttnDone, 0ull);
    }
}

// (kPre) Row `it` of a workgroup's new rows - the query heads of its group, then the key and the value row, which also go to the
// cache - from the projection's partial sums: eight elements (lane t of D / 8).  Requested in this order: the partial sums (first
// eight slices), the rotary row and the weight, what `then` requests - the sums are worked on while that is on its way.
template <typename T, int D, typename Then>
__device__ __forceinline__ u32x4 ksa_decode_new_row(const DecodeParams& p, int bz, int kvh, int it, int new_row, int t, Then then) {
    using C = KsaCvt<T>;
    constexpr int LPR = D / 8;
    const int width = (p.Hq + 2 * p.Hkv) * D;
    const int hrow = it < p.g ? kvh * p.g + it : p.Hq + (it - p.g) * p.Hkv + kvh;
    const float* src = p.qkv + (int64_t)bz * width + (int64_t)hrow * D + 8 * t;
    const int64_t pitch = (int64_t)p.qkv_prows * width;
    f32x4 lo[8], hi[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
        const float* sp = src + pitch * min(u, p.qkv_ksplit - 1);
        lo[u] = *reinterpret_cast<const f32x4*>(sp);
        hi[u] = *reinterpret_cast<const f32x4*>(sp + 4);
    }
    const u32x4 w = *reinterpret_cast<const u32x4*>((it < p.g ? p.wq : p.wk) + 8 * t);
    const u32x4 cr = *reinterpret_cast<const u32x4*>(p.cos + bz * p.c_bs + 8 * t);
    const u32x4 sr = *reinterpret_cast<const u32x4*>(p.sin + bz * p.c_bs + 8 * t);
    then();
    float ac[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};  // summed and rounded as ksa_sum_partials8
#pragma unroll
    for (int u = 0; u < 8; ++u) {
        if (u < p.qkv_ksplit) {
#pragma unroll
            for (int i = 0; i < 4; ++i) ac[i] += lo[u][i], ac[4 + i] += hi[u][i];
        }
    }
    for (int u = 8; u < p.qkv_ksplit; ++u) {
        const f32x4 l4 = *reinterpret_cast<const f32x4*>(src + pitch * u);
        const f32x4 h4 = *reinterpret_cast<const f32x4*>(src + pitch * u + 4);
#pragma unroll
        for (int i = 0; i < 4; ++i) ac[i] += l4[i], ac[4 + i] += h4[i];
    }
    u32x4 raw;
#pragma unroll
    for (int i = 0; i < 4; ++i) raw[i] = C::down2(ac[2 * i], ac[2 * i + 1]);
    const uint32_t sgn = t < LPR / 2 ? 0x80008000u : 0u;
    uint32_t wl[4], wh[4], cl[4], ch[4], sl[4], sh[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        wl[i] = w[i] & 0xffffu, wh[i] = w[i] & 0xffff0000u;
        cl[i] = cr[i] & 0xffffu, ch[i] = cr[i] & 0xffff0000u;
        sl[i] = (sr[i] ^ sgn) & 0xffffu, sh[i] = (sr[i] ^ sgn) & 0xffff0000u;
    }
    const u32x4 z = ksa_row_scale<T>(raw, ksa_row_inv_rms<T, LPR>(raw, p.eps), wl, wh);
    const u32x4 rot = ksa_row_rope<T, LPR>(z, cl, ch, sl, sh);
    const u32x4 val = it == p.g + 1 ? raw : rot;  // (the value row changes its place only)
    if (it >= p.g) {
        uint16_t* dst = it == p.g ? p.kw + bz * p.k_bs + kvh * p.k_hs + (int64_t)new_row * p.k_rs
                                  : p.vw + bz * p.v_bs + kvh * p.v_hs + (int64_t)new_row * p.v_rs;
        __builtin_nontemporal_store(val, reinterpret_cast<u32x4*>(dst + 8 * t));
    }
    return val;
}

// kPre against the pre-attention launch in front, a decode step of 8 layers of the 4B shape: batch 1 665 -> 652 us,
// batch 8 772 -> 759.  The chain of trips that it puts in front of the first scores (row and range, partial sums, LDS)
// runs next to the loads of the first K / V tile; what it costs is that every split repeats it, and a
// workgroup that is not among the first on its CU runs it behind full memory queues (who calls it keeps to launches whose
// workgroups all fit at once).
template <typename T, int D, bool kPre, bool kO = false>
__global__ __launch_bounds__(kThreads, (D <= 128 ? 2 : 1)) void ksa_decode_kernel(
    const std::conditional_t<kO, DecodeOParams, DecodeParams> p) {
    using Ops = KsaOps<T>;
    constexpr int KS = D / 16;
    constexpr int DB = D / 32;
    constexpr int KROW = D + 8;
    constexpr int VROW = D + 16;
    constexpr int CPR = D / 8;
    constexpr int KLD = (kRows * CPR) / 64;          // K (and V) loads per lane
    constexpr int kStage = kRows * (KROW + VROW);    // elements of one wave's staging area
    constexpr int kMergeFloats = kWaves * 32 * (D + 2);
    constexpr int kSmemBytes = (kWaves * kStage * 2 > kMergeFloats * 4) ? kWaves * kStage * 2
                                                                        : kMergeFloats * 4;
    __shared__ __attribute__((aligned(16))) unsigned char smem[kSmemBytes];
    // (kPre) the query rows of the group, then the new key and value row
    __shared__ __attribute__((aligned(16))) uint16_t s_new[kPre ? (32 + 2) * D : 8];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int lq = lane & 31;
    const int lh = lane >> 5;

    int split = blockIdx.x, unit = blockIdx.y, bz = blockIdx.z;
    if constexpr (kO) {  // the same order in one dimension, the o projection behind it
        if ((int)blockIdx.x >= p.n_attn) {
            ksa_decode_o_stage<T, D, kWaves>(p, blockIdx.x - p.n_attn, smem);
            return;
        }
        unit = blockIdx.x / p.nsplit;
        split = blockIdx.x - unit * p.nsplit;
        bz = unit / p.Hkv;
        unit -= bz * p.Hkv;
    }
    const int kvh = unit % p.Hkv;
    // (kO) the sums of this workgroup have left and are counted off
    auto arrive = [&]() {
        if constexpr (kO) {
            __builtin_amdgcn_s_waitcnt(0);
            __syncthreads();
            if (tid == 0) add_agent(p.sync + kWordStride * (kStepHead0 + kvh), 1ull);
        }
    };
    auto put = [&](float* dst, float v) {
        if constexpr (kO) st_agent(dst, v);
        else *dst = v;
    };

    uint16_t* Kw = reinterpret_cast<uint16_t*>(smem) + wave * kStage;
    uint16_t* Vw = Kw + kRows * KROW;

    // One column block per workgroup - except in the chunk-boundary form, where the workgroup of the text
    // token's block takes the summary tokens' blocks behind it (their row range is one chunk: a tile or two
    // for two of the splits, nothing for the others).  As workgroups of their own, scattered between the long
    // ones, those short blocks held places of a CU for a chain of memory round trips under full load, and the
    // long workgroups that had to wait for the places ended late: +8 us per small-window layer and +27 us
    // per large-window layer of a boundary step.
    const int colblk_first = p.split_q ? 0 : unit / p.Hkv;
    const int colblk_last = p.split_q ? p.ncols_pad / 32 - 1 : colblk_first;
    for (int colblk = colblk_first; colblk <= colblk_last; ++colblk) {
    if (colblk != colblk_first) __syncthreads();  // the previous block's merge area becomes staging again
    const bool second = p.split_q && colblk > 0;  // the summary tokens' columns and their own row range
    const int r_begin = second ? (p.start2 ? p.start2[bz] : p.start20) : (p.start ? p.start[bz] : p.start0);
    const int r_end = second ? (p.end2 ? p.end2[bz] : p.end20) : (p.end ? p.end[bz] : p.end0);
    const int L = max(r_end - r_begin, 0);
    // rows per split: a multiple of the 128 rows the four waves cover per round
    const int per = ((L + p.nsplit - 1) / p.nsplit + kWaves * kRows - 1) / (kWaves * kRows) *
                    (kWaves * kRows);
    const int s0 = r_begin + split * per;
    const int s1 = min(r_end, s0 + per);

    if (p.nsplit > 1 && s0 >= s1) {
        // an empty slice (a short range: the summary tokens' chunk at a boundary step, a sequence with few
        // rows): the merge only needs to know that there is nothing here (it does not read the sums then)
        const int ncol = !p.split_q ? min(32, p.ncols - colblk * 32)
                                    : (colblk == 0 ? p.g : min(32, (p.Q - 1) * p.g - (colblk - 1) * 32));
        if (tid < ncol) {
            const int64_t slot = (((int64_t)bz * p.Hkv + kvh) * p.nsplit + split) * p.ncols_pad + colblk * 32 + tid;
            put(p.ws_ml + slot * 2, -INFINITY);
            put(p.ws_ml + slot * 2 + 1, 0.f);
        }
        arrive();
        continue;
    }

    // column (query token qi, head gi of the group) owned by this lane
    int qi, gi;
    const bool col_ok = ksa_decode_column(p, colblk, lq, qi, gi);
    if (!col_ok) qi = 0, gi = 0;
    const int head = kvh * p.g + gi;

    const uint16_t* kbase = p.k + bz * p.k_bs + kvh * p.k_hs;
    const uint16_t* vbase = p.v + bz * p.v_bs + kvh * p.v_hs;
    const int last_row = max(r_end - 1, r_begin);

    u32x4 kreg[KLD];
    u32x4 vreg[KLD];

    // K/V rows are read once and never again: non-temporal loads
    auto load_piece = [&](int row0, int i) {
        const int u = lane + 64 * i;
        const int row = min(row0 + u / CPR, last_row);
        kreg[i] = __builtin_nontemporal_load(
            reinterpret_cast<const u32x4*>(kbase + (int64_t)row * p.k_rs + 8 * (u % CPR)));
        vreg[i] = __builtin_nontemporal_load(
            reinterpret_cast<const u32x4*>(vbase + (int64_t)row * p.v_rs + 8 * (u % CPR)));
    };
    auto load_tile = [&](int row0) {
#pragma unroll
        for (int i = 0; i < KLD; ++i) load_piece(row0, i);
    };

    floatx16 oacc[DB];
#pragma unroll
    for (int b = 0; b < DB; ++b)
#pragma unroll
        for (int i = 0; i < 16; ++i) oacc[b][i] = 0.f;
    float m_run = -INFINITY;  // in raw score units
    float l_run = 0.f;
    const float c2 = p.scale_log2;

    int row0 = s0 + wave * kRows;
    u32x4 qf[KS];
    int new_row = -1;  // (kPre) the new token's cache row, if it lies in this workgroup's slice
    if constexpr (!kPre) {
        const uint16_t* qp = p.q + bz * p.q_bs + head * p.q_hs + qi * p.q_qs + 8 * lh;
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            u32x4 z = {0u, 0u, 0u, 0u};
            qf[s] = col_ok ? *reinterpret_cast<const u32x4*>(qp + 16 * s) : z;
        }
        if (row0 < s1) load_tile(row0);
    } else {
        // (ksa_decode_new_row written out: called here, the compiler keeps 66 scalar registers more and spills 16 others to memory; the
        // tests hold both, bit for bit, against ksa_pre_attention_partials)
        using C = KsaCvt<T>;
        constexpr int LPR = D / 8;      // lanes per head row
        constexpr int RPW = 64 / LPR;   // head rows per wave
        const int t = lane % LPR;
        new_row = p.row_seq ? p.row_seq[bz] : p.row0;
        if (new_row < s0 || new_row >= s1) new_row = -1;
        const int rows_here = p.g + (new_row >= 0 ? 2 : 0);  // query rows, then the key and the value row
        const int width = (p.Hq + 2 * p.Hkv) * D;
        bool loaded = false;
        for (int i0 = wave * RPW; i0 < rows_here; i0 += kWaves * RPW) {  // (at most once for up to 14 query rows of 128)
            const int it = min(i0 + lane / LPR, rows_here - 1);          // (lanes past the last row repeat it)
            const int hrow = it < p.g ? kvh * p.g + it : p.Hq + (it - p.g) * p.Hkv + kvh;
            // requested in this order: the partial sums (first eight slices), the rotary row and the weight, the
            // first K / V tile - the sums are then worked on while the tile is on its way
            const float* src = p.qkv + (int64_t)bz * width + (int64_t)hrow * D + 8 * t;
            const int64_t pitch = (int64_t)p.qkv_prows * width;
            f32x4 lo[8], hi[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const float* sp = src + pitch * min(u, p.qkv_ksplit - 1);
                lo[u] = *reinterpret_cast<const f32x4*>(sp);
                hi[u] = *reinterpret_cast<const f32x4*>(sp + 4);
            }
            const u32x4 w = *reinterpret_cast<const u32x4*>((it < p.g ? p.wq : p.wk) + 8 * t);
            const u32x4 cr = *reinterpret_cast<const u32x4*>(p.cos + bz * p.c_bs + 8 * t);
            const u32x4 sr = *reinterpret_cast<const u32x4*>(p.sin + bz * p.c_bs + 8 * t);
            if (!loaded && row0 < s1) load_tile(row0);
            loaded = true;
            float ac[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};  // summed and rounded as ksa_sum_partials8
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                if (u < p.qkv_ksplit) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) ac[i] += lo[u][i], ac[4 + i] += hi[u][i];
                }
            }
            for (int u = 8; u < p.qkv_ksplit; ++u) {
                const f32x4 l4 = *reinterpret_cast<const f32x4*>(src + pitch * u);
                const f32x4 h4 = *reinterpret_cast<const f32x4*>(src + pitch * u + 4);
#pragma unroll
                for (int i = 0; i < 4; ++i) ac[i] += l4[i], ac[4 + i] += h4[i];
            }
            u32x4 raw;
#pragma unroll
            for (int i = 0; i < 4; ++i) raw[i] = C::down2(ac[2 * i], ac[2 * i + 1]);
            const uint32_t sgn = t < LPR / 2 ? 0x80008000u : 0u;
            uint32_t wl[4], wh[4], cl[4], ch[4], sl[4], sh[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                wl[i] = w[i] & 0xffffu, wh[i] = w[i] & 0xffff0000u;
                cl[i] = cr[i] & 0xffffu, ch[i] = cr[i] & 0xffff0000u;
                sl[i] = (sr[i] ^ sgn) & 0xffffu, sh[i] = (sr[i] ^ sgn) & 0xffff0000u;
            }
            const u32x4 z = ksa_row_scale<T>(raw, ksa_row_inv_rms<T, LPR>(raw, p.eps), wl, wh);
            const u32x4 rot = ksa_row_rope<T, LPR>(z, cl, ch, sl, sh);
            const u32x4 val = it == p.g + 1 ? raw : rot;  // (the value row changes its place only)
            *reinterpret_cast<u32x4*>(s_new + (it < p.g ? it : 32 + it - p.g) * D + 8 * t) = val;
            if (it >= p.g) {
                uint16_t* dst = it == p.g ? p.kw + bz * p.k_bs + kvh * p.k_hs + (int64_t)new_row * p.k_rs
                                          : p.vw + bz * p.v_bs + kvh * p.v_hs + (int64_t)new_row * p.v_rs;
                __builtin_nontemporal_store(val, reinterpret_cast<u32x4*>(dst + 8 * t));
            }
        }
        if (!loaded && row0 < s1) load_tile(row0);
        __syncthreads();
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            u32x4 z = {0u, 0u, 0u, 0u};
            qf[s] = col_ok ? *reinterpret_cast<const u32x4*>(s_new + gi * D + 16 * s + 8 * lh) : z;
        }
    }

    for (; row0 < s1; row0 += kWaves * kRows) {
        ksa_wave_lds_fence();
        // registers -> LDS, and each register pair is refilled with the next tile right behind
        // its store, so the loads of the next tile are in flight for the whole step
        const int next = row0 + kWaves * kRows;
        const bool has_next = next < s1;
#pragma unroll
        for (int i = 0; i < KLD; ++i) {
            const int u = lane + 64 * i;
            *reinterpret_cast<u32x4*>(Kw + (u / CPR) * KROW + 8 * (u % CPR)) = kreg[i];
            *reinterpret_cast<u32x4*>(Vw + (u / CPR) * VROW + 8 * (u % CPR)) = vreg[i];
            if (has_next) load_piece(next, i);
        }
        if constexpr (kPre) {
            // the new row, over what the cache held in its place - and, where it is the last one, over its
            // repetitions in the rows past the end (their probabilities are 0, so they have to be finite)
            if (new_row >= row0 && new_row < row0 + kRows) {
                const bool is_v = lane >= CPR;
                const u32x4 v = *reinterpret_cast<const u32x4*>(s_new + (is_v ? 33 : 32) * D + 8 * (lane % CPR));
                const int first = new_row - row0, last = new_row == last_row ? kRows - 1 : first;
                for (int j = first; j <= last; ++j)
                    if (lane < 2 * CPR)
                        *reinterpret_cast<u32x4*>((is_v ? Vw + j * VROW : Kw + j * KROW) + 8 * (lane % CPR)) = v;
            }
        }
        ksa_wave_lds_fence();

        floatx16 sacc;
#pragma unroll
        for (int i = 0; i < 16; ++i) sacc[i] = 0.f;
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            const u32x4 a = *reinterpret_cast<const u32x4*>(Kw + lq * KROW + 16 * s + 8 * lh);
            sacc = Ops::mfma(a, qf[s], sacc);
        }
        if (row0 + kRows > s1) {  // tail tile: rows past the slice end do not exist
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int r = row0 + 8 * (i / 4) + 4 * lh + (i % 4);
                if (r >= s1) sacc[i] = -INFINITY;
            }
        }
        float mloc = -INFINITY;
#pragma unroll
        for (int i = 0; i < 16; ++i) mloc = fmaxf(mloc, sacc[i]);
        mloc = fmaxf(mloc, ksa_xor32(mloc));
        const float m_new = fmaxf(m_run, mloc);  // finite: every tile has >= 1 real row
        const float alpha = ksa_exp2((m_run - m_new) * c2);
        const float mc = m_new * c2;
        m_run = m_new;
        float rowsum = 0.f;
        u32x4 pf[2];
#pragma unroll
        for (int i = 0; i < 16; i += 2) {
            const float p0 = ksa_exp2(fmaf(sacc[i], c2, -mc));
            const float p1 = ksa_exp2(fmaf(sacc[i + 1], c2, -mc));
            rowsum += p0 + p1;
            pf[i / 8][(i % 8) / 2] = Ops::pack2(p0, p1);
        }
        l_run = l_run * alpha + rowsum;
        if (__any(alpha != 1.f)) {
#pragma unroll
            for (int b = 0; b < DB; ++b)
#pragma unroll
                for (int i = 0; i < 16; ++i) oacc[b][i] *= alpha;
        }
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
            for (int b = 0; b < DB; ++b) {
                const u32x4 a = ksa_read_vt_frag<VROW>(Vw, ks, b, lq, lh);
                oacc[b] = Ops::mfma(a, pf[ks], oacc[b]);
            }
    }

    // ---- merge the four waves through LDS ----
    l_run += ksa_xor32(l_run);
    __syncthreads();  // staging areas are dead from here on
    float* mg = reinterpret_cast<float*>(smem);  // [wave][col 32][D + 2]
    {
        float* row = mg + (wave * 32 + lq) * (D + 2);
#pragma unroll
        for (int b = 0; b < DB; ++b)
#pragma unroll
            for (int i = 0; i < 16; ++i) row[32 * b + 8 * (i / 4) + 4 * lh + (i % 4)] = oacc[b][i];
        if (lh == 0) {
            row[D] = m_run * c2;  // log2 units; -inf if this wave saw no row
            row[D + 1] = l_run;
        }
    }
    __syncthreads();
    const int ncol_here = !p.split_q ? min(32, p.ncols - colblk * 32)
                                     : (colblk == 0 ? p.g : min(32, (p.Q - 1) * p.g - (colblk - 1) * 32));
    for (int e = tid; e < ncol_here * D; e += kThreads) {
        const int c = e / D, d = e % D;
        float mx = -INFINITY;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) mx = fmaxf(mx, mg[(w * 32 + c) * (D + 2) + D]);
        float acc = 0.f, l = 0.f;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
            const float* row = mg + (w * 32 + c) * (D + 2);
            const float f = (row[D] == -INFINITY) ? 0.f : ksa_exp2(row[D] - mx);
            acc += row[d] * f;
            l += row[D + 1] * f;
        }
        const int cg = colblk * 32 + c;
        if (!kO && p.nsplit == 1) {
            int oq, og;
            ksa_decode_column(p, colblk, c, oq, og);
            const float val = l > 0.f ? acc / l : 0.f;
            uint16_t* op = p.out + bz * p.o_bs + oq * p.o_qs + (kvh * p.g + og) * p.o_hs + d;
            const uint32_t pk = Ops::pack2(val, 0.f);
            *op = (uint16_t)(pk & 0xffffu);
        } else {
            const int64_t slot = (((int64_t)bz * p.Hkv + kvh) * p.nsplit + split) * p.ncols_pad + cg;
            put(p.ws_o + slot * D + d, acc);
            if (d == 0) {
                put(p.ws_ml + slot * 2, mx);
                put(p.ws_ml + slot * 2 + 1, l);
            }
        }
    }
    arrive();
    }  // column blocks of this workgroup
}

// Second stage: merge the splits of one (sequence, kv head, column).  A chain of memory trips, nothing else, so
// there are few: D / 4 threads take four elements each, the G such groups of a workgroup every G-th split, and a
// group requests up to eight splits with their maxima and sums at once; the groups meet in LDS.  One trip takes 32
// splits with a thread per element (G = 4), which is the workgroup up to there, and 128 / 64 / 32 at head_dim
// 64 / 128 / 256 with 256 threads, which is the one above; another trip takes as many more.  (256 threads for few
// splits too cost a launch of thousands of columns more than it saved: 9 query tokens of 32 heads, 8 x 1500 rows in 5
// splits at head_dim 64 16.7 -> 19.0 us, with a thread per element 16.4; 3 x 4096 rows in 16 18.9 -> 18.5, and 16.8.)  (A thread per element that walked the splits eight at a time, maxima first, took 2 to 16 trips:
// decode + merge of one sequence of 16384 rows in
// 64 splits 29.8 -> 19.4 us, 4096 rows in 16 13.4 -> 12.0.)
template <typename T, int D, int kThreads>
__global__ __launch_bounds__(kThreads) void ksa_decode_merge_kernel(const DecodeParams p) {
    using Ops = KsaOps<T>;
    constexpr int TPG = D / 4;                 // threads of a group
    constexpr int G = kThreads / TPG;
    constexpr int kBatch = 8;
    __shared__ float s_m[G], s_l[G];
    __shared__ __attribute__((aligned(16))) float s_o[G][D];
    const int oq = blockIdx.x / p.g, og = blockIdx.x % p.g;  // logical column: query token, head in the group
    const int cg = ksa_decode_slot(p, oq, og);
    const int kvh = blockIdx.y;
    const int bz = blockIdx.z;
    const int grp = threadIdx.x / TPG, d4 = 4 * (threadIdx.x % TPG);
    const int64_t base = (((int64_t)bz * p.Hkv + kvh) * p.nsplit) * p.ncols_pad + cg;
    floatx4 acc = {0.f, 0.f, 0.f, 0.f};
    float mx = -INFINITY, l = 0.f;
    for (int s0 = grp; s0 < p.nsplit; s0 += kBatch * G) {
        floatx4 o[kBatch];
        floatx2_ws ml[kBatch];
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {
            const int64_t slot = base + (int64_t)min(s0 + u * G, p.nsplit - 1) * p.ncols_pad;
            ml[u] = *reinterpret_cast<const floatx2_ws*>(p.ws_ml + slot * 2);
            o[u] = *reinterpret_cast<const floatx4_ws*>(p.ws_o + slot * D + d4);
        }
        float m_new = mx;
#pragma unroll
        for (int u = 0; u < kBatch; ++u) m_new = fmaxf(m_new, ml[u][0]);
        const float f0 = mx == -INFINITY ? 0.f : ksa_exp2(mx - m_new);
        l *= f0;
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] *= f0;
        mx = m_new;
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {
            // (an empty slice leaves its sums unwritten: nothing of it may enter, not even times zero)
            if (s0 + u * G < p.nsplit && ml[u][0] != -INFINITY) {
                const float f = ksa_exp2(ml[u][0] - mx);
                l = fmaf(ml[u][1], f, l);
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[i] = fmaf(o[u][i], f, acc[i]);
            }
        }
    }
    *reinterpret_cast<floatx4*>(&s_o[grp][d4]) = acc;
    if (d4 == 0) s_m[grp] = mx, s_l[grp] = l;
    __syncthreads();
    const int d = threadIdx.x;
    if (d < D) {
        const int ng = min(G, p.nsplit);
        float top = -INFINITY, sum = 0.f, val = 0.f;
        for (int w = 0; w < ng; ++w) top = fmaxf(top, s_m[w]);
        for (int w = 0; w < ng; ++w) {
            const float f = s_m[w] == -INFINITY ? 0.f : ksa_exp2(s_m[w] - top);
            sum = fmaf(s_l[w], f, sum);
            val = fmaf(s_o[w][d], f, val);
        }
        val = sum > 0.f ? val / sum : 0.f;
        uint16_t* op = p.out + bz * p.o_bs + oq * p.o_qs + (kvh * p.g + og) * p.o_hs + d;
        *op = (uint16_t)(Ops::pack2(val, 0.f) & 0xffffu);
    }
}

// The same in workgroups of eight waves, one to a CU, for up to 16 columns (query tokens x heads of a group) at head_dim 64 and
// 128: what a call takes that does not name a split count (ksa_decode_wide_splits).  A round of the kernel above is a chain of
// trips - a tile's loads, LDS, scores, sums - with 64 KB on its way, and a launch of few sequences is some of them and a merge.
// Here a wave takes 64 rows at once on 16x16x32 products: with 16 columns instead of 32 the sums take half the registers, K goes
// from memory straight to the operand registers (64 bytes of 16 rows an instruction), V through LDS, and a round's 256 KB are
// requested before the round in front is worked on.  What bounds it: with many sequences the memory (64 of 9000 rows 6.8 TB/s, its waves 61 % of
// the time waiting to issue the next loads, every byte read once), with few the chain of trips, once per launch (1 of 1500 rows: 71 % in
// waits for what is requested), and what one CU fetches, 50 GB/s of its own and 27 when all do; the split counts follow that
// (ksa_decode_wide_splits).
// Attention and merge of calls behind one another in a graph, 32 / 8 heads of 128, in the kernel above -> here, us: 1 sequence of 150 / 300 /
// 1500 / 9000 rows 6.2 / 8.1 / 8.7 / 15.4 -> 5.7 / 7.1 / 8.4 / 13.5; 4 of 300 / 3000 9.8 / 16.7 -> 7.8 / 14.9; 8 of 1500 18.1 ->
// 15.0; 16 of 737 / 3000 16.0 / 38.7 -> 13.6 / 37.7; 24 of 737 / 1500 / 9000 20.6 / 37.3 / 172 -> 15.4 / 27.3 / 139; 32 of 737 / 9000
// 23.4 / 180 -> 19.0 / 175; 48 of 1100 / 9000 45.1 / 286 -> 43.3 / 264; 64 of 9000 340 -> 341.
// The probabilities enter the second product as two 16-bit parts, value and remainder: a wave's first tile of 64 rows fixes its
// reference, where the kernel above has more of them, and a row at its reference has no rounding; with one part the output lay 1.3 %
// further from 64 bits than the kernel above (60 shapes, up to 5 %), with two 12 % nearer (0.76 to 1.0 times), for 0.2 us a launch.
// An infinite value has no product with a remainder of 0 or below, nor with the probability 0 of its repetitions past the end: an
// element that comes out as NaN is made once more by the thread that has it, behind everything else.  (Looked for in the sums of each
// wave, with a second walk of its tiles, it cost every launch 0.17 us.)
// kPre as above; the new key goes to the operand registers, the new value to the tile.  kO as above; a decode step's attention and o
// projection, 32 / 8 heads of 128, N 2560, in the kernel above -> here: 1 sequence of 737 / 4097 rows 15.8 / 18.2 -> 11.7 / 14.6 us, 8
// of 737 / 4097 21.3 / 38.6 -> 16.2 / 34.9, 16 of 737 / 4097 26.4 / 61.7 -> 22.2 / 54.6.
constexpr int kWideWaves = 8, kWideRows = 64, kWideColumns = 16;
// (as an integer: the compiler takes floats for numbers)
__device__ __forceinline__ bool ksa_is_nan(float x) { return __builtin_bit_cast(uint32_t, x) << 1 > 0xff000000u; }
template <typename T, int D, bool kPre, bool kO = false>
__global__ __launch_bounds__(64 * kWideWaves) void ksa_decode_wide_kernel(const std::conditional_t<kO, DecodeOParams, DecodeParams> p) {
    using Ops = KsaOps<T>;
    using C = KsaCvt<T>;
    constexpr int KS = D / 32, DB = D / 16, NB = kWideRows / 16, NT = kWideRows / 32, CPR = D / 8;
    constexpr int VLD = kWideRows * CPR / 64;  // V loads per lane and round
    constexpr int VROW = D + 16;
    constexpr int kStage = kWideRows * VROW;   // elements of one wave's V tile
    __shared__ __attribute__((aligned(16))) uint16_t smem[kWideWaves * kStage];
    // (kPre) the query rows of the group, then the new key and value row
    __shared__ __attribute__((aligned(16))) uint16_t s_new[kPre ? (16 + 2) * D : 8];
    static_assert(kWideWaves * 16 * (D + 2) * 4 <= sizeof(smem), "the merge reuses the tiles");
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, kq = lane >> 4;
    int split = blockIdx.x, kvh = blockIdx.y, bz = blockIdx.z;
    if constexpr (kO) {
        if ((int)blockIdx.x >= p.n_attn) {
            ksa_decode_o_stage<T, D, kWideWaves>(p, blockIdx.x - p.n_attn, reinterpret_cast<unsigned char*>(smem));
            return;
        }
        kvh = blockIdx.x / p.nsplit;
        split = blockIdx.x - kvh * p.nsplit;
        bz = kvh / p.Hkv;
        kvh -= bz * p.Hkv;
    }
    // (kO) the sums of this workgroup have left and are counted off
    auto arrive = [&]() {
        if constexpr (kO) {
            __builtin_amdgcn_s_waitcnt(0);
            __syncthreads();
            if (tid == 0) add_agent(p.sync + kWordStride * (kStepHead0 + kvh), 1ull);
        }
    };
    auto put = [&](float* dst, float v) {
        if constexpr (kO) st_agent(dst, v);
        else *dst = v;
    };
    const int r_first = p.start ? p.start[bz] : p.start0;
    const int r_last = p.end ? p.end[bz] : p.end0;
    // rows per split: whole tiles of a wave
    const int per = ((max(r_last - r_first, 0) + p.nsplit - 1) / p.nsplit + kWideRows - 1) / kWideRows * kWideRows;
    const int r_begin = r_first + split * per, r_end = min(r_last, r_begin + per);
    const int last_row = max(r_end - 1, r_first);
    const int64_t slot0 = (((int64_t)bz * p.Hkv + kvh) * p.nsplit + split) * p.ncols_pad;
    if (p.nsplit > 1 && r_begin >= r_end) {  // an empty slice: the merge does not read its sums
        if (tid < p.ncols) put(p.ws_ml + (slot0 + tid) * 2, -INFINITY), put(p.ws_ml + (slot0 + tid) * 2 + 1, 0.f);
        arrive();
        return;
    }
    const uint16_t* kbase = p.k + bz * p.k_bs + kvh * p.k_hs + 8 * kq;
    const uint16_t* vbase = p.v + bz * p.v_bs + kvh * p.v_hs + 8 * (lane % CPR);
    uint16_t* Vw = smem + wave * kStage;

    u32x4 kreg[NB][KS], vreg[VLD];
    auto load_k = [&](int row0) {
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            // (plain loads: the other half of the line is the next instruction's)
            const uint16_t* kp = kbase + (int64_t)min(row0 + 16 * b + r, last_row) * p.k_rs;
#pragma unroll
            for (int s = 0; s < KS; ++s) kreg[b][s] = *reinterpret_cast<const u32x4*>(kp + 32 * s);
        }
    };
    auto load_v = [&](int row0, int i) {
        const int row = min(row0 + (lane + 64 * i) / CPR, last_row);
        vreg[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(vbase + (int64_t)row * p.v_rs));
    };
    int row0 = r_begin + wave * kWideRows;
    auto load_first = [&]() {
        if (row0 < r_end) {
            load_k(row0);
#pragma unroll
            for (int i = 0; i < VLD; ++i) load_v(row0, i);
        }
    };
    int qi, gi;
    const bool col_ok = ksa_decode_column(p, 0, r, qi, gi);
    if (!col_ok) qi = 0, gi = 0;
    u32x4 qf[KS];
    int new_row = -1;  // (kPre) the new token's cache row, if it lies in this slice
    if constexpr (!kPre) {
        load_first();
        const uint16_t* qp = p.q + bz * p.q_bs + (kvh * p.g + gi) * p.q_hs + qi * p.q_qs + 8 * kq;
#pragma unroll
        for (int s = 0; s < KS; ++s) qf[s] = col_ok ? *reinterpret_cast<const u32x4*>(qp + 32 * s) : u32x4{0u, 0u, 0u, 0u};
    } else {
        new_row = p.row_seq ? p.row_seq[bz] : p.row0;
        if (new_row < r_begin || new_row >= r_end) new_row = -1;
        const int rows_here = p.g + (new_row >= 0 ? 2 : 0);
        constexpr int LPR = D / 8, RPW = 64 / LPR;
        static_assert(kWideWaves * RPW >= 18, "one pass over the rows");
        if (wave * RPW < rows_here) {
            const int it = min(wave * RPW + lane / LPR, rows_here - 1);
            const u32x4 val = ksa_decode_new_row<T, D>(p, bz, kvh, it, new_row, lane % LPR, load_first);
            *reinterpret_cast<u32x4*>(s_new + (it < p.g ? it : 16 + it - p.g) * D + 8 * (lane % LPR)) = val;
        } else {
            load_first();
        }
        __syncthreads();
#pragma unroll
        for (int s = 0; s < KS; ++s)
            qf[s] = col_ok ? *reinterpret_cast<const u32x4*>(s_new + gi * D + 32 * s + 8 * kq) : u32x4{0u, 0u, 0u, 0u};
    }

    f32x4 oacc[DB];
#pragma unroll
    for (int b = 0; b < DB; ++b) oacc[b] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m_run = -INFINITY, l_run = 0.f;
    const float c2 = p.scale_log2;
    for (; row0 < r_end; row0 += kWideWaves * kWideRows) {
        const int next = row0 + kWideWaves * kWideRows;
        const bool has_next = next < r_end;
        const int at = new_row - row0;  // (kPre) place of the new row in the tile
        if constexpr (kPre) {
            if (at >= 0 && at < kWideRows) {
#pragma unroll
                for (int b = 0; b < NB; ++b)
#pragma unroll
                    for (int s = 0; s < KS; ++s)
                        if (16 * b + r == at) kreg[b][s] = *reinterpret_cast<const u32x4*>(s_new + 16 * D + 32 * s + 8 * kq);
            }
        }
        f32x4 sacc[NB];
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            sacc[b] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < KS; ++s) sacc[b] = mfma16<T>(kreg[b][s], qf[s], sacc[b]);
        }
        if (has_next) load_k(next);
        ksa_wave_lds_fence();  // the reads of the round before are done
#pragma unroll
        for (int i = 0; i < VLD; ++i) {
            const int u = lane + 64 * i;
            *reinterpret_cast<u32x4*>(Vw + (u / CPR) * VROW + 8 * (u % CPR)) = vreg[i];
            if (has_next) load_v(next, i);
        }
        if constexpr (kPre) {
            // over what the cache held in its place - and, where it is the last one, over its repetitions in the rows
            // past the end (their probabilities are 0, so they have to be finite)
            if (at >= 0 && at < kWideRows) {
                const u32x4 v = *reinterpret_cast<const u32x4*>(s_new + 17 * D + 8 * (lane % CPR));
                const int end = new_row == last_row ? kWideRows : at + 1;
                for (int j = at + lane / CPR; j < end; j += 64 / CPR) *reinterpret_cast<u32x4*>(Vw + j * VROW + 8 * (lane % CPR)) = v;
            }
        }
        ksa_wave_lds_fence();
        // lane: column r, rows 16 b + 4 kq + i of the tile
        if (row0 + kWideRows > r_end) {
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (row0 + 16 * b + 4 * kq + i >= r_end) sacc[b][i] = -INFINITY;
        }
        float mloc = -INFINITY;
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int i = 0; i < 4; ++i) mloc = fmaxf(mloc, sacc[b][i]);
        mloc = fmaxf(mloc, __shfl_xor(mloc, 16));
        mloc = fmaxf(mloc, __shfl_xor(mloc, 32));
        const float m_new = fmaxf(m_run, mloc);  // finite: every tile has at least one row
        const float alpha = ksa_exp2((m_run - m_new) * c2), mc = m_new * c2;
        m_run = m_new;
        float rowsum = 0.f;
        u32x4 pf[NT], pl[NT];  // the probabilities in 16 bits, and what that leaves of them
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int i = 0; i < 4; i += 2) {
                const float p0 = ksa_exp2(fmaf(sacc[b][i], c2, -mc)), p1 = ksa_exp2(fmaf(sacc[b][i + 1], c2, -mc));
                rowsum += p0 + p1;
                const uint32_t pk = Ops::pack2(p0, p1);
                pf[b / 2][2 * (b % 2) + i / 2] = pk;
                pl[b / 2][2 * (b % 2) + i / 2] = Ops::pack2(p0 - C::lo(pk), p1 - C::hi(pk));
            }
        l_run = l_run * alpha + rowsum;
        if (__any(alpha != 1.f)) {
#pragma unroll
            for (int b = 0; b < DB; ++b)
#pragma unroll
                for (int i = 0; i < 4; ++i) oacc[b][i] *= alpha;
        }
        // contraction element 8 kq + 4 a + j of step t is row 32 t + 16 a + 4 kq + j: what this lane holds of the probabilities
        typedef __attribute__((address_space(3))) ksa_short4* lds_ptr;
        const uint16_t* vp = Vw + (4 * kq + (r >> 2)) * VROW + 4 * (r & 3);
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int b = 0; b < DB; ++b) {
                const u32x2 lo = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(vp + 32 * t * VROW + 16 * b)));
                const u32x2 hi =
                    __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(vp + (32 * t + 16) * VROW + 16 * b)));
                const u32x4 a = {lo[0], lo[1], hi[0], hi[1]};
                oacc[b] = mfma16<T>(a, pf[t], oacc[b]);
                oacc[b] = mfma16<T>(a, pl[t], oacc[b]);
            }
    }

    l_run += __shfl_xor(l_run, 16);
    l_run += __shfl_xor(l_run, 32);
    __syncthreads();  // the tiles are dead from here on
    float* mg = reinterpret_cast<float*>(smem);  // [wave][column 16][D + 2]
    if (col_ok) {
        float* row = mg + (wave * 16 + r) * (D + 2);
#pragma unroll
        for (int b = 0; b < DB; ++b)
#pragma unroll
            for (int i = 0; i < 4; ++i) row[16 * b + 4 * kq + i] = oacc[b][i];
        if (kq == 0) row[D] = m_run * c2, row[D + 1] = l_run;  // (log2 units; -inf of a wave without rows)
    }
    __syncthreads();
    auto merged = [&](int c, int d, float& mx, float& l) {
        const float* row = mg + c * (D + 2);
        float acc = 0.f;
        mx = -INFINITY, l = 0.f;
#pragma unroll
        for (int w = 0; w < kWideWaves; ++w) mx = fmaxf(mx, row[w * 16 * (D + 2) + D]);
#pragma unroll
        for (int w = 0; w < kWideWaves; ++w) {
            const float m = row[w * 16 * (D + 2) + D];
            const float f = m == -INFINITY ? 0.f : ksa_exp2(m - mx);
            acc += row[w * 16 * (D + 2) + d] * f;
            l += row[w * 16 * (D + 2) + D + 1] * f;
        }
        return acc;
    };
    auto leave = [&](int c, int d, float mx, float acc, float l) {
        if (kO || p.nsplit > 1) {
            put(p.ws_o + (slot0 + c) * D + d, acc);
            if (d == 0) put(p.ws_ml + (slot0 + c) * 2, mx), put(p.ws_ml + (slot0 + c) * 2 + 1, l);
            return;
        }
        int oq, og;
        ksa_decode_column(p, 0, c, oq, og);
        p.out[bz * p.o_bs + oq * p.o_qs + (kvh * p.g + og) * p.o_hs + d] = (uint16_t)(Ops::pack2(l > 0.f ? acc / l : 0.f, 0.f) & 0xffffu);
    };
    bool nan = false;
    for (int e = tid; e < p.ncols * D; e += 64 * kWideWaves) {
        float mx, l;
        const float acc = merged(e / D, e % D, mx, l);
        nan |= ksa_is_nan(acc);
        leave(e / D, e % D, mx, acc, l);
    }
    if (__builtin_expect(__any(nan), 0)) {
        // the sum of column c and element d from its definition, at reference mx
        auto element = [&](int c, int d, float mx) {
            int oq, og;
            ksa_decode_column(p, 0, c, oq, og);
            const uint16_t* qp = kPre ? s_new + og * D : p.q + bz * p.q_bs + (kvh * p.g + og) * p.q_hs + oq * p.q_qs;
            float acc = 0.f;
#pragma unroll 1
            for (int row = r_begin; row < r_end; ++row) {
                const bool fresh = kPre && row == new_row;
                const uint16_t* kp = fresh ? s_new + 16 * D : p.k + bz * p.k_bs + kvh * p.k_hs + (int64_t)row * p.k_rs;
                const uint16_t v = fresh ? s_new[17 * D + d] : p.v[bz * p.v_bs + kvh * p.v_hs + (int64_t)row * p.v_rs + d];
                float score = 0.f;
#pragma unroll 1
                for (int i = 0; i < D; i += 8) {
                    const u32x4 a = *reinterpret_cast<const u32x4*>(kp + i), b = *reinterpret_cast<const u32x4*>(qp + i);
#pragma unroll
                    for (int j = 0; j < 4; ++j) score = C::dot2(a[j], b[j], score);
                }
                acc = fmaf(ksa_exp2(fmaf(score, c2, -mx)), C::up(v), acc);
            }
            return acc;
        };
        for (int e = tid; e < p.ncols * D; e += 64 * kWideWaves) {
            float mx, l;
            const float acc = merged(e / D, e % D, mx, l);
            if (ksa_is_nan(acc) && !ksa_is_nan(l)) leave(e / D, e % D, mx, element(e / D, e % D, mx), l);
        }
    }
    arrive();
}

template <typename T, int D>
int launch(const DecodeParams& p, int batch, hipStream_t stream) {
    const int colblks = p.split_q ? 1 : p.ncols_pad / 32;  // (boundary form: a workgroup walks its column blocks)
    dim3 grid(p.nsplit, p.Hkv * colblks, batch);
    if (p.wide) {
        if constexpr (D <= 128) {
            auto kern = p.qkv ? ksa_decode_wide_kernel<T, D, true> : ksa_decode_wide_kernel<T, D, false>;
            hipLaunchKernelGGL(kern, grid, dim3(64 * kWideWaves), 0, stream, p);
        } else {
            return KSA_ERR_UNSUPPORTED;
        }
    } else if (p.qkv) {
        if constexpr (D <= 128)
            hipLaunchKernelGGL((ksa_decode_kernel<T, D, true>), grid, dim3(kThreads), 0, stream, p);
        else
            return KSA_ERR_UNSUPPORTED;
    } else {
        hipLaunchKernelGGL((ksa_decode_kernel<T, D, false>), grid, dim3(kThreads), 0, stream, p);
    }
    if (p.nsplit > 1) {
        dim3 g2(p.ncols, p.Hkv, batch);
        if (p.nsplit <= 32)
            hipLaunchKernelGGL((ksa_decode_merge_kernel<T, D, D>), g2, dim3(D), 0, stream, p);
        else
            hipLaunchKernelGGL((ksa_decode_merge_kernel<T, D, 256>), g2, dim3(256), 0, stream, p);
    }
    return ksa_check_launch();
}

int pad_cols(int ncols) { return (ncols + 31) / 32 * 32; }
// column slots of the chunk-boundary form: a block of 32 for the text token, the summary tokens behind it
int pad_cols_boundary(int Q, int g) { return 32 + pad_cols((Q - 1) * g); }

}  // namespace

extern "C" size_t ksa_decode_workspace_bytes(int batch, int Hq, int Hkv, int Q, int D, int nsplit) {
    if (nsplit <= 1 || batch <= 0 || Hkv <= 0 || Hq % Hkv != 0) return 0;
    const size_t cols = (size_t)pad_cols(Q * (Hq / Hkv));
    return (size_t)batch * Hkv * nsplit * cols * (D + 2) * sizeof(float);
}

// Number of splits by sequences, kv heads and rows alone: at least two workgroups per CU of the current device
// (256 CUs assumed when no device can be asked), but never splits shorter than 256 rows.  Kept for callers of
// ksa_decode_fwd_noalloc, whose scratch is of a fixed size; ksa_decode_splits below is faster on few rows.
extern "C" int ksa_decode_auto_splits(int batch, int Hkv, int max_rows) {
    if (batch <= 0 || Hkv <= 0 || max_rows <= 0) return 1;
    const int units = batch * Hkv;
    const int want = 2 * ksa_cu_count_or(256);
    int n = (want + units - 1) / units;
    const int cap = max_rows / 256 > 1 ? max_rows / 256 : 1;
    if (n > cap) n = cap;
    if (n > 64) n = 64;
    return n < 1 ? 1 : n;
}

// Several blocks of 32 columns (query tokens x heads of a group) up to head_dim 128: each block is a workgroup of its
// own that reads the slice's K / V again.  The blocks of a slice are nsplit x kv heads workgroups apart: a multiple of 8
// puts them on one XCD, where the K / V of the first one is in the L2 for the others, worth more than the last
// workgroups' round alone.  From half a workgroup per CU on the count goes up to such a multiple if the one by the
// slices alone allows it (from one split on long ranges only; at head_dim 64 it is the one by the slices if not), below
// that down to a multiple, or to the least count with as many rounds of 128 rows.  head_dim 128, 9 query tokens, count by
// the slices / by the workgroups / this one: 64 sequences of 4096 rows, 1 kv head of 8 72 / 97 / 72 us, 2 of 4 82 / 97 / 82;
// 20 of 4096, 4 of 8 103 / 98 / 82; 64 of 600 and 4096, 4 of 8 71 / 54 / 54 and 202 / 235 / 196; 40 of 1650, 8 of 8 139 /
// 99 / 99; 8 of 760, 4 of 8 19.3 / 22.4 / 18.4; 8 of 4096, 1 of 8 21.6 / 22.8 / 19.7; 3 of 1500, 8 of 4 18.6 / 18.9 / 17.1;
// 1 of 1500, 8 of 4 16.4 / 12.6 / 12.6.  At head_dim 64 100 of 4096, 2 of 4 84 / 100 / 84.
static int splits_of_column_blocks(int64_t slices, int64_t blocks, int Hkv, int D, int64_t max_rows, int64_t cus) {
    const int64_t units = slices * blocks, rounds = (max_rows + 127) / 128;
    int64_t a = 8;  // 8 / gcd(8, kv heads)
    for (int h = Hkv; a > 1 && h % 2 == 0; h /= 2) a /= 2;
    int64_t cap = max_rows / 256;
    if (2 * units > cus) {
        int64_t n = (2 * cus + units - 1) / units;
        const int64_t by_slices = (2 * cus + slices - 1) / slices, aligned = (n + a - 1) / a * a;
        if (aligned <= by_slices && (n > 1 || max_rows >= 2048)) n = aligned;
        else if (n > 1 && n % a && D <= 64) n = by_slices;
        n = n < cap ? n : cap;
        return (int)(n < 1 ? 1 : n < 64 ? n : 64);
    }
    if (3 * units <= cus && blocks <= 4) cap = max_rows <= (D <= 64 ? 512 : 384) ? 1 : rounds;
    int64_t n = 2 * cus / units;
    n = n < cap ? n : cap;
    n = n < 64 ? n : 64;
    if (n <= 1) return 1;
    if (a > 1 && n >= a) return (int)(n - n % a);
    const int64_t per = (rounds + n - 1) / n;
    return (int)((rounds + per - 1) / per);
}

// One block of columns, less than half a workgroup per CU (a third at head_dim 64): a round of 128 rows per split where
// that is at most two workgroups per CU (eight workgroups more do no harm at head_dim 128, sixteen at 64 with few
// columns), otherwise two per CU; but where those would walk several rounds and splits of 256 rows put one workgroup
// on a CU, these.  Rounded up past two per CU the last workgroups run alone: 9 / 11 sequences of 8 kv heads, 4096 rows,
// 8 -> 7 / 6 -> 5 splits 38.1 -> 33.2 / 48.7 -> 39.0 us, 1100 rows of 9 in 4 / 8 / 7 18.8 / 20.8 / 16.3; 3 of 2700 rows in 10 /
// 22 / 21 14.7 / 15.1 / 15.3, with 20 columns 17.6 / 20.8 / 19.1; at head_dim 64 40 slices of 4096 rows in 13 -> 12 17.1
// -> 16.0, at 128 25.5 -> 26.1.  Above 32 splits of more than 16 columns, the least count with as many rounds: 6 slices of
// 10000 rows, 32 columns, 39 / 64 / 40 splits 18.8 / 20.4 / 18.0.
static int splits_of_few_slices(int64_t units, int64_t columns, int D, int64_t max_rows, int64_t cus) {
    if (max_rows <= (D <= 64 ? 512 : 384)) return 1;
    const int64_t rounds = (max_rows + 127) / 128;
    int64_t n = 2 * cus / units;
    if (D <= 64 && columns <= 16 && rounds == n + 1 && n * units < 2 * cus) n = rounds;
    if (rounds <= n) {
        n = rounds;
    } else {
        if (D > 64) n = (2 * cus + cus / 32) / units;
        const int64_t long_ones = max_rows / 256;
        if (long_ones < n && long_ones * units <= cus && n * units > cus) n = long_ones;
    }
    if (n > 64) n = 64;
    if (n > 32 && columns > 16) {
        const int64_t per = (rounds + n - 1) / n;
        n = (rounds + per - 1) / per;
    }
    return (int)n;
}

// Number of splits for Q query tokens of Hq heads: two workgroups per CU, but splits of no fewer rows than a
// workgroup's waves cover in one round (128) - a launch over few rows is a chain of memory trips per
// round, 2.1 us each, and a split more costs the merge next to nothing.  From half a workgroup per CU on
// (128 of them) a split must save two rounds (256 rows) to be worth the partial sums.  Decode + merge at
// head_dim 128, 8 kv heads, former count -> this one: 1 sequence of 760 / 1500 / 4096 / 16384 rows
// 13.2 / 13.4 / 13.4 / 29.8 -> 9.0 / 9.2 / 10.4 / 19.4 us (the last by the merge kernel alone), 8 sequences of
// 760 / 1500 rows 14.5 / 19.9 -> 12.8 / 18.6; 16 and 32 sequences the same counts as before.
// Up to three rounds (four of half the bytes at head_dim 64) one workgroup walks them faster than the merge's launch:
// 1 split against several, 1 sequence of 200 / 300 / 500 rows 6.2 / 7.5 / 10.2 against 7.5 / 7.7 / 8.2 us, at head_dim
// 64 4.9 / 5.7 / 6.5 against 6.8 / 6.9 / 6.9; there 120 units of 1000 rows also want the 3 splits (12.7 us) and not 5 (13.3).
// At head_dim 256 a CU holds one workgroup, so two per CU run one behind the other, with a second start: there the
// count is the one with the least rounds x (steps of 128 rows + 2 for the start) + 1.5 for the merge, in units of a
// step.  8 kv heads, count by the rule above -> this one: 1 sequence of 4430 / 16384 rows 24.3 / 39.3 -> 18.8 / 33.6 us,
// 2 of 4430 32.3 -> 25.5 (before either rule 24.9), 4 of 3000 35.1 -> 27.9, 8 of 1500 37.4 -> 28.1, 16 of 3000 80.3 -> 74.8,
// 20 of 6000 191 -> 173; few rows the same counts.
extern "C" int ksa_decode_splits(int batch, int Hq, int Hkv, int Q, int D, int max_rows) {
    if (batch <= 0 || Hkv <= 0 || Hq <= 0 || Hq % Hkv != 0 || Q <= 0 || D <= 0 || max_rows <= 0) return 1;
    const int64_t blocks = (Q * (int64_t)(Hq / Hkv) + 31) / 32, units = (int64_t)batch * Hkv * blocks;
    const int cus = ksa_cu_count_or(256);
    if (D > 128) {
        const int64_t steps = ((int64_t)max_rows + 127) / 128;
        int best = 1;
        int64_t least = INT64_MAX;  // (in half steps)
        for (int i = 1; i <= 64 && i <= steps; ++i) {
            const int64_t per = (steps + i - 1) / i, used = (steps + per - 1) / per;  // splits that have rows
            const int64_t cost = (units * used + cus - 1) / cus * (2 * per + 4) + (used > 1 ? 3 : 0);
            if (cost < least) least = cost, best = (int)used;
        }
        return best;
    }
    if (blocks > 1) return splits_of_column_blocks((int64_t)batch * Hkv, blocks, Hkv, D, max_rows, cus);
    if ((D <= 64 ? 3 : 2) * units < cus) return splits_of_few_slices(units, (int64_t)Q * (Hq / Hkv), D, max_rows, cus);
    int64_t n = (2 * (int64_t)cus + units - 1) / units;
    const int64_t cap = max_rows / 256;
    if (n > cap) n = cap;
    if (n > 64) n = 64;
    return n < 1 ? 1 : (int)n;
}

// Split count of the wide kernel, at most `most`: the one with the least time by what was measured of one workgroup to a CU, 5 us for the
// start of a round of workgroups (the first one takes 3, for every count alike), 10.2 ns a row of head_dim 128 and CU when the other CUs are
// idle and 9.4 more when all are at work (half of that at head_dim 64), 2.2 to 3.8 us for the merge.  Against the best of nine counts around
// it (2081 calls): within 5 % but for 18.
static int wide_count(int64_t units, int D, int64_t max_rows, int64_t cus, int64_t most) {
    const unsigned tiles = (unsigned)((max_rows + kWideRows - 1) / kWideRows);
    most = most < tiles ? most : tiles;
    most = most < 1 ? 1 : most < 64 ? most : 64;
    const double row = D / 128.0 * 0.0102, load = D / 128.0 * 0.0094;
    int best = 1, before = 0;
    double least = 1e30;
    for (unsigned n = 1; n <= (unsigned)most; ++n) {  // (every call walks this: no 64-bit divisions but for more than a round)
        const unsigned per_tiles = (tiles + n - 1) / n;
        const int used = (int)((tiles + per_tiles - 1) / per_tiles);  // slices that have rows
        if (used == before) continue;
        before = used;
        const int64_t per = per_tiles, wgs = units * used, full = wgs < cus ? 0 : wgs / cus, rest = wgs - full * cus;
        double us = full * (5.0 + per * kWideRows * (row + load));
        if (rest) us += 5.0 + per * kWideRows * (row + load * rest / cus);
        if (used > 1) us += 2.2 + (full ? 1.6 : 1.6 * rest / cus);
        if (us < least) least = us, best = used;
    }
    return best;
}

// Number of splits for ksa_decode_wide_fwd, or 0 where ksa_decode_fwd is the one to call: more than 16 columns, head_dim 256, and
// where it measured faster.  Both were timed in graphs over 1 to 64 sequences, eight forms of heads, 150 to 131000 rows: of 3848 calls
// 3636 taken, 0.91 times the time of the other on average, more than 1.04 times in 33 (profiles/decode_wide_vs_four_waves.md).
//  - More pairs of sequence and kv head than CUs (units) over few rows: two of its workgroups share a CU.  Up to 600 rows: 48 / 64
//    sequences of 8 kv heads, 150 / 300 / 500 rows 11.3 / 16.6 / 21.5 against 12.3 / 17.0 / 24.0 us, 12.3 / 19.0 / 25.3 against
//    13.2 / 19.2 / 25.8.  Up to 2500 rows from one and a half rounds of units on, and below that from 1200 rows on: 512 units of 737 /
//    2000 rows 1.04 to 1.07 (head_dim 64: 1.03 to 1.10) times its time, 1536 and 2048 of 737 1.08 (1.13), 384 of 2000 1.02 to 1.05; but 384
//    of 1100 rows 0.89 to 0.97.
//  - head_dim 128, its workgroups are one to a CU at the most and walk their rows in one round (128 rows), and slices here are longer than
//    a wave's 64 rows: 2 to 4 of the eight waves then have rows, 64 of them each where its four have 32.  8 units of 2000 rows 1.04 to
//    1.08 times its time, 24 of 737 1.04 to 1.09, 32 of 900 1.05 to 1.07; in slices of 64 rows 0.93 to 1.03.  (Head_dim 64: 0.93 to 1.10,
//    as fast on average.)
extern "C" int ksa_decode_wide_splits(int batch, int Hq, int Hkv, int Q, int D, int max_rows) {
    if (batch <= 0 || Hkv <= 0 || Hq <= 0 || Hq % Hkv != 0 || Q <= 0 || max_rows <= 0 || (D != 64 && D != 128)) return 0;
    const int64_t units = (int64_t)batch * Hkv, cus = ksa_cu_count_or(256);
    if ((int64_t)Q * (Hq / Hkv) > kWideColumns) return 0;
    if (units > cus && max_rows <= 2500 && (max_rows <= 600 || max_rows > 1200 || 2 * units > 3 * cus)) return 0;
    const int best = wide_count(units, D, max_rows, cus, 4 * cus / units);
    if (D == 128 && (int64_t)best * kWideRows < max_rows && units <= cus && units * max_rows <= 128 * cus) {  // (may be one round)
        const int four = ksa_decode_splits(batch, Hq, Hkv, Q, D, max_rows);
        if (four > 1 && units * four <= cus && four * 128 >= max_rows) return 0;
    }
    return best;
}

// The same for ksa_decode_qkv_wide_fwd, where all workgroups run at once: so the outputs are bit for bit those of ksa_decode_wide_fwd behind
// the pre-attention step wherever that runs in one round.  Of 32 / 8 heads, 1 to 32 sequences of 737 to 24000 rows 0.64 to 1.03 times the
// time of what took its place before.  Not taken for long ranges where one round of slices leaves CUs idle, and their share of the memory's
// rate: 11 / 12 sequences of 8 kv heads, 176 / 192 workgroups, 6000 to 24000 rows 1.04 to 1.10; at head_dim 64 17 to 21 sequences of
// 12000 and 24000 rows 1.02 to 1.16.
extern "C" int ksa_decode_qkv_wide_splits(int batch, int Hq, int Hkv, int D, int max_rows) {
    const int n = ksa_decode_wide_splits(batch, Hq, Hkv, 1, D, max_rows);
    const int64_t units = (int64_t)batch * Hkv, cus = ksa_cu_count_or(256);
    if (n == 0 || units > cus) return 0;
    const int64_t most = cus / units, round = most * units;
    if (D == 128 ? 5 * round < 4 * cus && max_rows > 5000 : 3 * round < 2 * cus && max_rows > 10000) return 0;
    return n < most ? n : (int)most;
}

namespace {

template <typename T>
int launch_head_dim(const DecodeParams& p, int D, int batch, hipStream_t st) {
    if (D == 128) return launch<T, 128>(p, batch, st);
    if (D == 64) return launch<T, 64>(p, batch, st);
    if (D == 256) return launch<T, 256>(p, batch, st);
    return KSA_ERR_UNSUPPORTED;
}

int decode_fwd_impl(const void* q, const void* kcache, const void* vcache, void* out,
                    const int32_t* start, const int32_t* end, int start0, int end0, int batch, int Hq,
                    int Hkv, int Q, int D, int dtype, const int64_t* q_strides,
                    const int64_t* k_strides, const int64_t* v_strides, const int64_t* out_strides,
                    float scale, int nsplit, void* workspace, size_t workspace_bytes, void* stream,
                    bool boundary = false, const int32_t* start2 = nullptr, const int32_t* end2 = nullptr,
                    int start20 = 0, int end20 = 0, bool wide = false) {
    if (!q || !kcache || !vcache || !out || !q_strides || !k_strides || !v_strides || !out_strides)
        return KSA_ERR_NULL;
    if ((start == nullptr) != (end == nullptr)) return KSA_ERR_NULL;
    if (boundary) {
        if ((start2 == nullptr) != (end2 == nullptr)) return KSA_ERR_NULL;
        if (Q < 2 || Hkv <= 0 || Hq % Hkv != 0 || Hq / Hkv > 32) return KSA_ERR_INVALID;
        if (!start2 && (start20 < 0 || end20 <= start20)) return KSA_ERR_INVALID;
    }
    if (batch <= 0 || Hq <= 0 || Hkv <= 0 || Hq % Hkv != 0 || Q <= 0 || nsplit < 1) return KSA_ERR_INVALID;
    if (!start && (start0 < 0 || end0 <= start0)) return KSA_ERR_INVALID;
    if (dtype != KSA_DTYPE_BF16 && dtype != KSA_DTYPE_F16) return KSA_ERR_UNSUPPORTED;
    if ((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(kcache) |
         reinterpret_cast<uintptr_t>(vcache)) & 15)
        return KSA_ERR_ALIGN;
    for (int i = 0; i < 3; ++i)
        if ((q_strides[i] % 8) || (k_strides[i] % 8) || (v_strides[i] % 8)) return KSA_ERR_ALIGN;

    DecodeParams p{};
    p.q = (const uint16_t*)q;
    p.k = (const uint16_t*)kcache;
    p.v = (const uint16_t*)vcache;
    p.out = (uint16_t*)out;
    p.start = start;
    p.end = end;
    p.start0 = start0;
    p.end0 = end0;
    p.Hq = Hq;
    p.Hkv = Hkv;
    p.g = Hq / Hkv;
    p.Q = Q;
    p.ncols = Q * p.g;
    p.ncols_pad = boundary ? pad_cols_boundary(Q, p.g) : pad_cols(p.ncols);
    p.split_q = boundary ? 1 : 0;
    p.wide = wide;
    if (wide && p.ncols > kWideColumns) return KSA_ERR_UNSUPPORTED;
    p.start2 = start2, p.end2 = end2, p.start20 = start20, p.end20 = end20;
    p.nsplit = nsplit;
    p.q_bs = q_strides[0], p.q_hs = q_strides[1], p.q_qs = q_strides[2];
    p.k_bs = k_strides[0], p.k_hs = k_strides[1], p.k_rs = k_strides[2];
    p.v_bs = v_strides[0], p.v_hs = v_strides[1], p.v_rs = v_strides[2];
    p.o_bs = out_strides[0], p.o_qs = out_strides[1], p.o_hs = out_strides[2];
    p.scale_log2 = scale * 1.4426950408889634f;
    if (nsplit > 1) {
        const size_t need = (size_t)batch * Hkv * nsplit * p.ncols_pad * (D + 2) * sizeof(float);
        if (!workspace || workspace_bytes < need) return KSA_ERR_WORKSPACE;
        p.ws_o = (float*)workspace;
        p.ws_ml = p.ws_o + (size_t)batch * Hkv * nsplit * p.ncols_pad * D;
    }
    hipStream_t st = (hipStream_t)stream;
    return dtype == KSA_DTYPE_BF16 ? launch_head_dim<KsaBf16>(p, D, batch, st) : launch_head_dim<KsaF16>(p, D, batch, st);
}

// ---- scratch of the entry point that allocates nothing ----
// Split-K partials of ksa_decode_fwd_noalloc live in this array instead of a caller-provided
// workspace.  Every GPU the library is loaded on holds its own copy at its own address; the
// array's name is only a host-side handle, so the device address is asked for once per device
// (hipGetSymbolAddress) and kept.
constexpr size_t kNoAllocScratchBytes = KSA_DECODE_NOALLOC_SCRATCH_BYTES;
constexpr int kMaxDevices = 64;
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];
std::mutex g_scratch_mutex;
void* g_scratch_ptr[kMaxDevices] = {};

// device address of `scratch` on the current device, or null
void* noalloc_scratch() {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return nullptr;
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[dev]) {
        void* ptr = nullptr;
        if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess || !ptr) {
            (void)hipGetLastError();
            return nullptr;
        }
        g_scratch_ptr[dev] = ptr;
    }
    return g_scratch_ptr[dev];
}

}  // namespace

extern "C" int ksa_decode_fwd(const void* q, const void* kcache, const void* vcache, void* out,
                              const int32_t* start, const int32_t* end, int start0, int end0,
                              int batch, int Hq, int Hkv, int Q, int D, int dtype,
                              const int64_t* q_strides, const int64_t* k_strides,
                              const int64_t* v_strides, const int64_t* out_strides, float scale,
                              int nsplit, void* workspace, size_t workspace_bytes, void* stream) {
    return decode_fwd_impl(q, kcache, vcache, out, start, end, start0, end0, batch, Hq, Hkv, Q, D, dtype,
                           q_strides, k_strides, v_strides, out_strides, scale, nsplit, workspace,
                           workspace_bytes, stream);
}

// ksa_decode_fwd in workgroups of eight waves, see ksa_decode_wide_kernel: Q Hq / Hkv <= 16, head_dim 64 or 128.
extern "C" int ksa_decode_wide_fwd(const void* q, const void* kcache, const void* vcache, void* out, const int32_t* start,
                                   const int32_t* end, int start0, int end0, int batch, int Hq, int Hkv, int Q, int D, int dtype,
                                   const int64_t* q_strides, const int64_t* k_strides, const int64_t* v_strides,
                                   const int64_t* out_strides, float scale, int nsplit, void* workspace, size_t workspace_bytes,
                                   void* stream) {
    if (D != 64 && D != 128) return KSA_ERR_UNSUPPORTED;
    return decode_fwd_impl(q, kcache, vcache, out, start, end, start0, end0, batch, Hq, Hkv, Q, D, dtype, q_strides, k_strides,
                           v_strides, out_strides, scale, nsplit, workspace, workspace_bytes, stream, false, nullptr, nullptr, 0, 0,
                           true);
}

// Chunk-boundary step (HF:831-876): the chunk's last text token and its summary tokens in one launch.
// Query token 0 attends rows [text_start, text_end) (the slice of get_attention_kv after update_text,
// HF:844-856), query tokens 1 .. Q - 1 attend [sum_start, sum_end) (the [own summaries | chunk] rows of
// get_summary_attention_kv, HF:858-870), un-masked both, as the reference's two calls of its decode
// attention function do; out [batch, Q, Hq, D] is their torch.cat (HF:875).
extern "C" size_t ksa_decode_boundary_workspace_bytes(int batch, int Hq, int Hkv, int Q, int D, int nsplit) {
    if (nsplit <= 1 || batch <= 0 || Hkv <= 0 || Hq % Hkv != 0 || Q < 2) return 0;
    return (size_t)batch * Hkv * nsplit * (size_t)pad_cols_boundary(Q, Hq / Hkv) * (D + 2) * sizeof(float);
}

extern "C" int ksa_decode_boundary_fwd(const void* q, const void* kcache, const void* vcache, void* out,
                                       const int32_t* text_start, const int32_t* text_end, int text_start0,
                                       int text_end0, const int32_t* sum_start, const int32_t* sum_end,
                                       int sum_start0, int sum_end0, int batch, int Hq, int Hkv, int Q, int D,
                                       int dtype, const int64_t* q_strides, const int64_t* k_strides,
                                       const int64_t* v_strides, const int64_t* out_strides, float scale,
                                       int nsplit, void* workspace, size_t workspace_bytes, void* stream) {
    return decode_fwd_impl(q, kcache, vcache, out, text_start, text_end, text_start0, text_end0, batch, Hq, Hkv, Q, D,
                           dtype, q_strides, k_strides, v_strides, out_strides, scale, nsplit, workspace,
                           workspace_bytes, stream, true, sum_start, sum_end, sum_start0, sum_end0);
}

// A decode step's attention from the K-split partial sums of its fused q | k | v projection: the pre-attention step
// (HF:660-666) and the attention over the cache (HF:591-612) in one launch.  Arithmetic and results are those of
// ksa_pre_attention_partials followed by ksa_decode_fwd.
namespace {
// `p` filled from the arguments that the two forms share
int decode_qkv_params(DecodeParams& p, const float* qkv_partials, int qkv_ksplit, const void* q_weight, const void* k_weight,
                      const void* cos, const void* sin, long long cos_batch_stride, float eps, void* kcache, void* vcache,
                      const int32_t* row, int row0, const int32_t* start, const int32_t* end, int start0, int end0,
                      int batch, int Hq, int Hkv, int D, int dtype, const int64_t* k_strides, const int64_t* v_strides,
                      float scale, int nsplit, void* workspace) {
    if (!qkv_partials || !q_weight || !k_weight || !cos || !sin || !kcache || !vcache || !k_strides || !v_strides)
        return KSA_ERR_NULL;
    if ((start == nullptr) != (end == nullptr)) return KSA_ERR_NULL;
    if (batch <= 0 || batch > kMaxPartialRows || Hq <= 0 || Hkv <= 0 || Hq % Hkv != 0 || Hq / Hkv > 32 || qkv_ksplit < 1 ||
        qkv_ksplit > 64 || nsplit < 1 || nsplit > 64 || !(eps >= 0.f))
        return KSA_ERR_INVALID;
    if (!start && (start0 < 0 || end0 <= start0)) return KSA_ERR_INVALID;
    if (!row && (row0 < 0 || (!start && (row0 < start0 || row0 >= end0)))) return KSA_ERR_INVALID;
    if (dtype != KSA_DTYPE_BF16 && dtype != KSA_DTYPE_F16) return KSA_ERR_UNSUPPORTED;
    if (D != 64 && D != 128) return KSA_ERR_UNSUPPORTED;
    for (const void* ptr : {(const void*)qkv_partials, q_weight, k_weight, cos, sin, (const void*)kcache, (const void*)vcache,
                            (const void*)workspace})
        if (reinterpret_cast<uintptr_t>(ptr) & 15) return KSA_ERR_ALIGN;
    for (int i = 0; i < 3; ++i)
        if ((k_strides[i] % 8) || (v_strides[i] % 8)) return KSA_ERR_ALIGN;
    if (cos_batch_stride % 8) return KSA_ERR_ALIGN;
    p.qkv = qkv_partials, p.qkv_ksplit = qkv_ksplit, p.qkv_prows = ksa_partial_rows(batch);
    p.wq = (const uint16_t*)q_weight, p.wk = (const uint16_t*)k_weight;
    p.cos = (const uint16_t*)cos, p.sin = (const uint16_t*)sin, p.c_bs = cos_batch_stride;
    p.eps = eps;
    p.k = p.kw = (uint16_t*)kcache;
    p.v = p.vw = (uint16_t*)vcache;
    p.row_seq = row, p.row0 = row0;
    p.start = start, p.end = end, p.start0 = start0, p.end0 = end0;
    p.Hq = Hq, p.Hkv = Hkv, p.g = Hq / Hkv, p.Q = 1;
    p.ncols = p.g;
    p.ncols_pad = pad_cols(p.ncols);
    p.nsplit = nsplit;
    p.k_bs = k_strides[0], p.k_hs = k_strides[1], p.k_rs = k_strides[2];
    p.v_bs = v_strides[0], p.v_hs = v_strides[1], p.v_rs = v_strides[2];
    p.scale_log2 = scale * 1.4426950408889634f;
    return KSA_OK;
}
}  // namespace

namespace {
int decode_qkv_impl(bool wide, const float* qkv_partials, int qkv_ksplit, const void* q_weight, const void* k_weight,
                    const void* cos, const void* sin, long long cos_batch_stride, float eps, void* kcache,
                    void* vcache, void* out, const int32_t* row, int row0, const int32_t* start,
                    const int32_t* end, int start0, int end0, int batch, int Hq, int Hkv, int D, int dtype,
                    const int64_t* k_strides, const int64_t* v_strides, const int64_t* out_strides,
                    float scale, int nsplit, void* workspace, size_t workspace_bytes, void* stream) {
    if (!out || !out_strides) return KSA_ERR_NULL;
    DecodeParams p{};
    const int rc = decode_qkv_params(p, qkv_partials, qkv_ksplit, q_weight, k_weight, cos, sin, cos_batch_stride, eps, kcache,
                                     vcache, row, row0, start, end, start0, end0, batch, Hq, Hkv, D, dtype, k_strides,
                                     v_strides, scale, nsplit, workspace);
    if (rc != KSA_OK) return rc;
    p.wide = wide;
    if (wide && p.ncols > kWideColumns) return KSA_ERR_UNSUPPORTED;
    p.out = (uint16_t*)out;
    p.o_bs = out_strides[0], p.o_qs = out_strides[1], p.o_hs = out_strides[2];
    if (nsplit > 1) {
        if (!workspace || workspace_bytes < ksa_decode_workspace_bytes(batch, Hq, Hkv, 1, D, nsplit)) return KSA_ERR_WORKSPACE;
        p.ws_o = (float*)workspace;
        p.ws_ml = p.ws_o + (size_t)batch * Hkv * nsplit * p.ncols_pad * D;
    }
    hipStream_t st = (hipStream_t)stream;
    return dtype == KSA_DTYPE_BF16 ? launch_head_dim<KsaBf16>(p, D, batch, st) : launch_head_dim<KsaF16>(p, D, batch, st);
}
}  // namespace

extern "C" int ksa_decode_qkv_fwd(const float* qkv_partials, int qkv_ksplit, const void* q_weight, const void* k_weight,
                                  const void* cos, const void* sin, long long cos_batch_stride, float eps, void* kcache,
                                  void* vcache, void* out, const int32_t* row, int row0, const int32_t* start,
                                  const int32_t* end, int start0, int end0, int batch, int Hq, int Hkv, int D, int dtype,
                                  const int64_t* k_strides, const int64_t* v_strides, const int64_t* out_strides,
                                  float scale, int nsplit, void* workspace, size_t workspace_bytes, void* stream) {
    return decode_qkv_impl(false, qkv_partials, qkv_ksplit, q_weight, k_weight, cos, sin, cos_batch_stride, eps, kcache, vcache, out, row,
                           row0, start, end, start0, end0, batch, Hq, Hkv, D, dtype, k_strides, v_strides, out_strides, scale,
                           nsplit, workspace, workspace_bytes, stream);
}

// ... in workgroups of eight waves
extern "C" int ksa_decode_qkv_wide_fwd(const float* qkv_partials, int qkv_ksplit, const void* q_weight, const void* k_weight,
                                       const void* cos, const void* sin, long long cos_batch_stride, float eps, void* kcache,
                                       void* vcache, void* out, const int32_t* row, int row0, const int32_t* start,
                                       const int32_t* end, int start0, int end0, int batch, int Hq, int Hkv, int D, int dtype,
                                       const int64_t* k_strides, const int64_t* v_strides, const int64_t* out_strides,
                                       float scale, int nsplit, void* workspace, size_t workspace_bytes, void* stream) {
    return decode_qkv_impl(true, qkv_partials, qkv_ksplit, q_weight, k_weight, cos, sin, cos_batch_stride, eps, kcache, vcache, out, row,
                           row0, start, end, start0, end0, batch, Hq, Hkv, D, dtype, k_strides, v_strides, out_strides, scale,
                           nsplit, workspace, workspace_bytes, stream);
}

// ksa_decode_qkv_fwd and the o projection behind it (modeling_qwen3sa.py:879) in one launch: see ksa_decode_o_stage.
extern "C" size_t ksa_decode_qkv_o_workspace_bytes(int batch, int Hq, int Hkv, int D, int nsplit) {
    if (batch <= 0 || Hkv <= 0 || Hq % Hkv != 0 || D <= 0 || nsplit < 1) return 0;
    return (size_t)batch * Hkv * nsplit * (size_t)pad_cols(Hq / Hkv) * (D + 2) * sizeof(float);
}

extern "C" size_t ksa_step_workspace_bytes(void) { return kStepBytes; }
extern "C" size_t ksa_step_status_offset(void) { return (size_t)kWordStride * kStepStatus * 8; }

// Splits for the one launch.  The count for the attention alone as long as its workgroups leave every CU room for one of the
// product (units * n <= CUs) and the sums to merge stay few; otherwise five attention workgroups to eight CUs, so that those of the
// product find places next to them.  One sequence of 32768 rows and more takes every split that a workgroup of the product
// merges, 64: there the attention is all of the time.  Attention + product at 32 / 8 heads of 128, N 2560, us, separate launches /
// five to eight CUs / this rule where it differs: 1 sequence of 4096 / 32768 / 131072 rows 19.5 / 18.1 / 17.9, 38.3 / 36.6 / 36.5,
// 101.3 / 101.3 / 99.0; N 4096, 65536 rows 60.3 / 61.5 / 58.5; 4 of 700 18.7 / 18.8 / 17.6; N 4096, 8 of 400 21.4 / 22.2 / 21.3.
// The rule kept at five to eight, separate / it / the count alone: 8 of 4096 / 32768 39.0 / 35.6 / 37.1, 180.5 / 168.2 / 176.3; 16 of
// 4096 60.0 / 55.2 / 57.6; 1 of 16384 28.2 / 27.0 / 27.3.
extern "C" int ksa_decode_qkv_o_splits(int batch, int Hq, int Hkv, int D, int max_rows) {
    if (batch <= 0 || batch > 16 || Hkv <= 0) return 1;
    const int units = batch * Hkv, cus = ksa_cu_count_or(256);
    int n = min(ksa_decode_splits(batch, Hq, Hkv, 1, D, max_rows), kMaxOSums / batch);
    if (!(batch == 1 && max_rows >= 32768) && (units * n > cus || batch * n > 32)) n = min(n, (cus * 5 / 8 + units - 1) / units);
    return n < 1 ? 1 : n;
}

// Whether the one launch is the faster way.  Its gain is two ramps and a trip of the rows, 1 to 3 us, and the time of o's
// weights where they are many; its price the merge of batch * n sums in every workgroup of the product, fewer splits, and the
// attention's places on the CUs that the product holds.  By a sweep over 1675 shapes (1 to 16 sequences of 400 to 131072 rows, 8 to
// 64 heads of 128 and 64, 1 to 32 kv heads, N 1024 to 5120) three kinds are taken, 461 of
// them, at 0.94 of the separate launches on average and 1.02 at the worst; one launch / separate ones at the lines' other sides:
//   as many splits as the attention alone takes, but few sums: 16 / 4 heads, 2 x 1400 rows (22 sums) 0.94, 4 x 1400 (40) 1.06, 8 x 700 (40)
//     1.13; one split, where there is no merge to save, at head_dim 64 1.00 to 1.07
//   32 heads of 128 and more: 32 / 2 heads, 8 sequences (64 sums) 1.01 to 1.12, 32 / 1, 16 (64 sums, 4 splits instead of 32) 1.05 to 1.92;
//     16 / 8 heads, 1 or 2 x 8192 1.04; head_dim 64 from 4096 rows on 1.05 to 1.65 (a split is half the work and as many trips)
//   many workgroups of the attention: 24 / 8 heads, 8 x 400 rows 1.02, 4 x 4096 1.03; 16 / 8, 8 x 5000 1.03 to 1.05
// and none with far more workgroups of the product than CUs (64 heads, N 5120, 640 of them, 1.00 to 1.14) or more than 8 kv heads
// (32 / 32 0.89 to 1.12).
extern "C" int ksa_decode_qkv_o_pays(int batch, int Hq, int Hkv, int D, int N, int max_rows) {
    if (batch <= 0 || batch > 16 || Hkv <= 0 || Hkv > 8 || Hq % Hkv != 0 || N <= 0 || max_rows <= 0) return 0;
    const int64_t product = (N + 127) / 128 * (int64_t)(Hq * D / kChunkK), cus = ksa_cu_count_or(256);
    const int n = ksa_decode_qkv_o_splits(batch, Hq, Hkv, D, max_rows), sums = batch * n;
    if (product <= cus && n > 1 && sums <= 20 && n == ksa_decode_splits(batch, Hq, Hkv, 1, D, max_rows)) return 1;
    if (D != 128) return 0;
    if (product <= cus && Hq * D >= 4096 && (sums <= 32 || (batch == 1 && max_rows >= 32768))) return 1;
    return product <= 2 * cus && batch * Hkv >= (Hq >= 24 ? 64 : 96) && max_rows >= 1400 && sums <= 32;
}

namespace {
// workgroups of the o projection in a launch of workgroups of so many waves
int o_workgroups(int N, int chunks, int waves) { return (N / 16 + 2 * waves - 1) / (2 * waves) * chunks; }

int decode_qkv_o_impl(bool wide, const float* qkv_partials, int qkv_ksplit, const void* q_weight, const void* k_weight,
                      const void* cos, const void* sin, long long cos_batch_stride, float eps, void* kcache,
                      void* vcache, const int32_t* row, int row0, const int32_t* start, const int32_t* end,
                      int start0, int end0, int batch, int Hq, int Hkv, int D, int dtype,
                      const int64_t* k_strides, const int64_t* v_strides, float scale, int nsplit,
                      const void* o_weight, float* o_partials, int N, void* workspace, size_t workspace_bytes,
                      void* step_workspace, size_t step_workspace_bytes, void* stream) {
    if (!o_weight || !o_partials || !workspace || !step_workspace) return KSA_ERR_NULL;
    if (N <= 0) return KSA_ERR_INVALID;
    DecodeOParams p{};
    p.wide = wide;
    const int rc = decode_qkv_params(p, qkv_partials, qkv_ksplit, q_weight, k_weight, cos, sin, cos_batch_stride, eps, kcache,
                                     vcache, row, row0, start, end, start0, end0, batch, Hq, Hkv, D, dtype, k_strides,
                                     v_strides, scale, nsplit, workspace);
    if (rc != KSA_OK) return rc;
    if (batch > 16 || batch * nsplit > kMaxOSums || Hkv > kStepMaxHeads || Hq * D % kChunkK != 0 || Hq * D > 64 * kChunkK ||
        N % 16 != 0 || (wide && p.ncols > kWideColumns))
        return KSA_ERR_UNSUPPORTED;
    for (const void* ptr : {o_weight, (const void*)o_partials, (const void*)step_workspace})
        if (reinterpret_cast<uintptr_t>(ptr) & 15) return KSA_ERR_ALIGN;
    if (workspace_bytes < ksa_decode_qkv_o_workspace_bytes(batch, Hq, Hkv, D, nsplit)) return KSA_ERR_WORKSPACE;
    if (step_workspace_bytes < ksa_step_workspace_bytes()) return KSA_ERR_WORKSPACE;
    p.ws_o = (float*)workspace;
    p.ws_ml = p.ws_o + (size_t)batch * Hkv * nsplit * p.ncols_pad * D;
    p.o_w = (const uint16_t*)o_weight, p.o_part = o_partials;
    p.sync = (unsigned long long*)step_workspace;
    p.batch = batch, p.n_attn = batch * Hkv * nsplit;
    p.o_n = N, p.o_chunks = Hq * D / kChunkK;
    const int waves = wide ? kWideWaves : kWaves;
    p.o_wgs = o_workgroups(N, p.o_chunks, waves);
    p.spin_limit = 1u << 19;  // polls of a microsecond or two: about a second
    const dim3 grid(p.n_attn + p.o_wgs), block(64 * waves);
    auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, grid, block, 0, (hipStream_t)stream, p);
        return ksa_check_launch();
    };
    if (wide) {
        if (dtype == KSA_DTYPE_BF16)
            return D == 128 ? go(ksa_decode_wide_kernel<KsaBf16, 128, true, true>) : go(ksa_decode_wide_kernel<KsaBf16, 64, true, true>);
        return D == 128 ? go(ksa_decode_wide_kernel<KsaF16, 128, true, true>) : go(ksa_decode_wide_kernel<KsaF16, 64, true, true>);
    }
    if (dtype == KSA_DTYPE_BF16)
        return D == 128 ? go(ksa_decode_kernel<KsaBf16, 128, true, true>) : go(ksa_decode_kernel<KsaBf16, 64, true, true>);
    return D == 128 ? go(ksa_decode_kernel<KsaF16, 128, true, true>) : go(ksa_decode_kernel<KsaF16, 64, true, true>);
}
}  // namespace

extern "C" int ksa_decode_qkv_o_fwd(const float* qkv_partials, int qkv_ksplit, const void* q_weight, const void* k_weight,
                                    const void* cos, const void* sin, long long cos_batch_stride, float eps, void* kcache,
                                    void* vcache, const int32_t* row, int row0, const int32_t* start, const int32_t* end,
                                    int start0, int end0, int batch, int Hq, int Hkv, int D, int dtype,
                                    const int64_t* k_strides, const int64_t* v_strides, float scale, int nsplit,
                                    const void* o_weight, float* o_partials, int N, void* workspace, size_t workspace_bytes,
                                    void* step_workspace, size_t step_workspace_bytes, void* stream) {
    return decode_qkv_o_impl(false, qkv_partials, qkv_ksplit, q_weight, k_weight, cos, sin, cos_batch_stride, eps, kcache, vcache, row, row0,
                             start, end, start0, end0, batch, Hq, Hkv, D, dtype, k_strides, v_strides, scale, nsplit, o_weight,
                             o_partials, N, workspace, workspace_bytes, step_workspace, step_workspace_bytes, stream);
}

// ... in workgroups of eight waves
extern "C" int ksa_decode_qkv_o_wide_fwd(const float* qkv_partials, int qkv_ksplit, const void* q_weight, const void* k_weight,
                                         const void* cos, const void* sin, long long cos_batch_stride, float eps, void* kcache,
                                         void* vcache, const int32_t* row, int row0, const int32_t* start, const int32_t* end,
                                         int start0, int end0, int batch, int Hq, int Hkv, int D, int dtype,
                                         const int64_t* k_strides, const int64_t* v_strides, float scale, int nsplit,
                                         const void* o_weight, float* o_partials, int N, void* workspace, size_t workspace_bytes,
                                         void* step_workspace, size_t step_workspace_bytes, void* stream) {
    return decode_qkv_o_impl(true, qkv_partials, qkv_ksplit, q_weight, k_weight, cos, sin, cos_batch_stride, eps, kcache, vcache, row, row0,
                             start, end, start0, end0, batch, Hq, Hkv, D, dtype, k_strides, v_strides, scale, nsplit, o_weight,
                             o_partials, N, workspace, workspace_bytes, step_workspace, step_workspace_bytes, stream);
}

// Splits of ksa_decode_qkv_o_wide_fwd, or 0 where it does not take the call.  The terms of ksa_decode_wide_splits without rounds (one
// workgroup to a CU), 30 ns for every row and split that a workgroup of the product merges, and 4 us more where the product's
// workgroups have to wait for a CU: 32 / 8 heads of 128, N 2560, 8 sequences of 737 / 1100 / 4097 rows in 2 / 4 splits 16.2 / 19.2 / 38.7
// and 19.2 / 20.5 / 34.9 us (176 CUs are left to the attention, 64 slices a split).  Not taken either where the four-wave form is faster:
// long ranges at head_dim 128 where a round of slices leaves more than a fifth of the CUs idle, 11 / 12 sequences of 8 kv heads, 9000 to
// 34816 rows 1.02 to 1.08 times its time.
extern "C" int ksa_decode_qkv_o_wide_splits(int batch, int Hq, int Hkv, int D, int N, int max_rows) {
    if (batch <= 0 || batch > 16 || Hkv <= 0 || Hkv > kStepMaxHeads || Hq <= 0 || Hq % Hkv != 0 || Hq / Hkv > kWideColumns || N <= 0 ||
        N % 16 != 0 || max_rows <= 0 || (D != 64 && D != 128) || Hq * D % kChunkK != 0 || Hq * D > 64 * kChunkK)
        return 0;
    const int64_t units = (int64_t)batch * Hkv, cus = ksa_cu_count_or(256);
    if (units > cus || (D == 128 && 5 * (cus / units * units) < 4 * cus && max_rows > 5000)) return 0;
    const int64_t room = cus - o_workgroups(N, Hq * D / kChunkK, kWideWaves);
    const int64_t tiles = ((int64_t)max_rows + kWideRows - 1) / kWideRows;
    int64_t most = cus / units;
    most = most < kMaxOSums / batch ? most : kMaxOSums / batch;
    most = most < tiles ? most : tiles;
    const double row = D / 128.0 * 0.0102, load = D / 128.0 * 0.0094;
    int best = 0, before = 0;
    double least = 1e30;
    for (int64_t n = 1; n <= most; ++n) {
        const int64_t per = (tiles + n - 1) / n;
        const int used = (int)((tiles + per - 1) / per);
        if (used == before) continue;
        before = used;
        const double us = per * kWideRows * (row + load * (double)(units * used) / cus) + 0.03 * batch * used +
                          (units * used > room ? 4.0 : 0.0);
        if (us < least) least = us, best = used;
    }
    return best;
}

// Whether ksa_decode_qkv_o_wide_fwd is faster than ksa_decode_qkv_fwd in its faster form and ksa_gemm_rows behind it
// (1630 shapes timed - 17 of heads, head_dim and N, 1 to 16 sequences of 300 to 34816 rows; graphs -, 1024 taken, 0.91 of the two on average,
// more than 1.03 in 15; profiles/decode_wide_vs_four_waves.md).
// Left to the two: a product of more workgroups than CUs (64 heads, N 5120 up to 1.20); few kv heads over long ranges (16 / 2
// heads, 4352 rows and more up to 1.26 times the two), whose count the sums limit; half a CU's worth of slices and more of few heads (16 / 8,
// 16 x 300 rows 1.06) or of any (32 / 32, 8 x 300 1.15); at head_dim 64 few rows (1.05 to 1.15), many slices (1.1 to 1.46) and
// long ranges (1.01 to 1.09).
extern "C" int ksa_decode_qkv_o_wide_pays(int batch, int Hq, int Hkv, int D, int N, int max_rows) {
    if (ksa_decode_qkv_o_wide_splits(batch, Hq, Hkv, D, N, max_rows) == 0) return 0;
    const int64_t units = (int64_t)batch * Hkv, cus = ksa_cu_count_or(256);
    if (o_workgroups(N, Hq * D / kChunkK, kWideWaves) > cus) return 0;
    if (Hkv < 4 && max_rows > (Hq * D < 4096 ? 1100 : 2048)) return 0;
    if (D == 128) return 2 * units < cus || (2 * units == cus && Hq * D >= 4096);
    return 8 * units <= 3 * cus && max_rows >= 600 && max_rows <= 8192;
}

extern "C" size_t ksa_decode_noalloc_max_workspace_bytes(void) { return kNoAllocScratchBytes; }

// ksa_decode_fwd without the workspace arguments: the split-K partials go to the library's own
// fixed device array.  Nothing is allocated, freed or synchronised here; the kernels are the
// ones ksa_decode_fwd launches and receive the array's device address as their workspace.
// Every (sequence, kv head, split, column) slot the merge kernel reads is written by the
// decode kernel of the same call, so nothing has to be cleared between calls.
extern "C" int ksa_decode_fwd_noalloc(const void* q, const void* kcache, const void* vcache, void* out,
                                      const int32_t* start, const int32_t* end, int start0, int end0,
                                      int batch, int Hq, int Hkv, int Q, int D, int dtype,
                                      const int64_t* q_strides, const int64_t* k_strides,
                                      const int64_t* v_strides, const int64_t* out_strides,
                                      float scale, int nsplit, void* stream) {
    if (nsplit <= 1)
        return decode_fwd_impl(q, kcache, vcache, out, start, end, start0, end0, batch, Hq, Hkv, Q, D,
                               dtype, q_strides, k_strides, v_strides, out_strides, scale, nsplit,
                               nullptr, 0, stream);
    if (batch <= 0 || Hq <= 0 || Hkv <= 0 || Hq % Hkv != 0 || Q <= 0) return KSA_ERR_INVALID;
    const size_t need = ksa_decode_workspace_bytes(batch, Hq, Hkv, Q, D, nsplit);
    if (need > kNoAllocScratchBytes) return KSA_ERR_WORKSPACE;
    void* ws = noalloc_scratch();
    if (!ws) return KSA_ERR_LAUNCH;
    return decode_fwd_impl(q, kcache, vcache, out, start, end, start0, end0, batch, Hq, Hkv, Q, D, dtype,
                           q_strides, k_strides, v_strides, out_strides, scale, nsplit, ws,
                           kNoAllocScratchBytes, stream);
}
