// A whole mixture-of-experts block: (token, expert) pairs sorted by expert, the grouped products, and the weighted sum
// over each token's experts.
//
// The reference loops over the experts in Python (python/llm/src/ipex_llm/transformers/models/qwen2_moe.py:375-430: a
// `where`, two index selects and an index_add per expert); its closed decode kernel takes one token
// (models/deepseek.py:290-315).  Two small kernels stand around the products of gemm_grouped.hip:
//   sort     the stable counting sort of the pairs and the rows of x in that order (more than 4096 pairs: two launches, the
//            sort in one workgroup)
//   combine  out[t] = sum_j weight[t, j] * y[position of pair (t, j)], in fp32, rounded once
// They are latency, not bandwidth: 1024 pairs over 8 experts with rows of 4096 take 5.4 us to combine, and took 6.1 + 6.3 to sort and
// gather in two launches.  (The same steps
// as torch operators - argsort, bincount, cumsum, index, mul, index_add - were 17 launches and 105 us, with bincount
// waiting for the GPU in the middle of them.)
//
// Few pairs go through the streaming kernel instead (use_streaming): every pair reads its expert's weights, two
// launches in all.
#include "lowbit_mfma.h"

namespace lowbit {

int launch_moe_gemv(const void *x, const void *ids, bool ids64, const void *route_w, int route_dtype, int tokens, int top_k,
                    int n_exp, const void *gates, const void *ups, const void *downs, void *h, void *y, int qtype, int act_dtype,
                    int hidden, int inter, int act, hipStream_t st);
int launch_grouped_gemm(const void *x, const void *const *w, const void *const *w_up, void *y, const int32_t *offsets,
                        int n_groups, int total_rows, int qtype, int act_dtype, int N, int K, int act, void *workspace,
                        size_t workspace_bytes, hipStream_t st);
size_t grouped_workspace_bytes(int total_rows, int n_groups, int N, int K);

constexpr int MOE_MAX_EXPERTS = 4096;                    // the sort's counters live in LDS

// offsets[e] = first position of expert e's pairs (offsets[n_exp] = their number), order[position] = pair,
// pos[pair] = position, or -1 for an id outside [0, n_exp).  Pairs of one expert keep their order.
// One workgroup: a pass over the ids counts, a second one places 64 pairs per wave at a time - the lanes of one expert
// find each other by ballot, the waves' counts meet in LDS.
__global__ __launch_bounds__(1024) void moe_route_kernel(const int64_t *__restrict__ ids, int pairs, int n_exp,
                                                         int32_t *__restrict__ offsets, int32_t *__restrict__ order,
                                                         int32_t *__restrict__ pos) {
    extern __shared__ int32_t counters[];
    int32_t *const base = counters;                      // [n_exp] pairs counted, then the next free position
    int32_t *const mine = counters + n_exp;              // [waves][n_exp] pairs of this round
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
    for (int e = threadIdx.x; e < n_exp * (waves + 1); e += blockDim.x) counters[e] = 0;
    __syncthreads();
    auto expert_of = [&](int p) {
        const int64_t e = p < pairs ? ids[p] : -1;
        return e >= 0 && e < n_exp ? (int)e : -1;
    };
    for (int p = threadIdx.x; p < pairs; p += blockDim.x) {
        const int e = expert_of(p);
        if (e >= 0) atomicAdd(&base[e], 1);
        else pos[p] = -1;
    }
    __syncthreads();
    if (wave == 0) {
        int before = 0;
        for (int e0 = 0; e0 < n_exp; e0 += 64) {
            const int e = e0 + lane, n = e < n_exp ? base[e] : 0;
            int incl = n;
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const int up = __shfl_up(incl, d);
                if (lane >= d) incl += up;
            }
            if (e < n_exp) base[e] = offsets[e] = before + incl - n;
            before += __shfl(incl, 63);
        }
        if (lane == 0) offsets[n_exp] = before;
    }
    __syncthreads();
    for (int p0 = 0; p0 < pairs; p0 += blockDim.x) {
        const int p = p0 + threadIdx.x, e = expert_of(p);
        int rank = 0;
        for (uint64_t left = __ballot(e >= 0); left;) {
            const int leader = __ffsll((unsigned long long)left) - 1;
            const int el = __builtin_amdgcn_readlane(e, leader);
            const uint64_t same = __ballot(e == el);
            if (e == el) rank = __popcll(same & ((1ull << lane) - 1ull));
            if (lane == leader) mine[wave * n_exp + el] = __popcll(same);
            left &= ~same;
        }
        __syncthreads();
        if (e >= 0) {
            int at = base[e] + rank;
            for (int v = 0; v < wave; v++) at += mine[v * n_exp + e];
            pos[p] = at;
            order[at] = p;
        }
        __syncthreads();
        for (int x = threadIdx.x; x < n_exp; x += blockDim.x)
            for (int v = 0; v < waves; v++) {
                base[x] += mine[v * n_exp + x];
                mine[v * n_exp + x] = 0;
            }
        __syncthreads();
    }
}

// Row i of xs = row order[i] / top_k of x; one workgroup per row, 16 bytes per lane (rows are whole 16-byte chunks: K is
// a multiple of 128).
__global__ __launch_bounds__(256) void moe_gather_kernel(const u32x4 *__restrict__ x, const int32_t *__restrict__ order,
                                                         const int32_t *__restrict__ n_rows, u32x4 *__restrict__ xs, int top_k,
                                                         int chunks) {
    const int i = blockIdx.x;
    if (i >= *n_rows) return;                            // pairs without an expert have no row
    const u32x4 *from = x + (int64_t)(order[i] / top_k) * chunks;
    u32x4 *to = xs + (int64_t)i * chunks;
    for (int c = threadIdx.x; c < chunks; c += 256) to[c] = from[c];
}

// Both at once for up to MOE_SORT_PAIRS pairs: workgroup p counts the pairs that come before pair p - those of lower experts, and the
// earlier ones of its own - and copies its row of x there; workgroup pairs + e writes offsets[e].  pairs^2 ids come out of L2, which
// costs less than a second launch that waits for a single workgroup's sort (39 pairs over 5 experts 3.3 + 3.4 us in a kernel
// trace, 472 over 10 4.4 + 3.9, 1024 over 8 6.4 + 6.1).  At the limit of 4096 pairs it is still the shorter way: over 8 experts with rows
// of 4096 18.2 us against 13.1 + 10.8 and the gap between two launches, of 1024 15.4 / 13.1 + 4.8, over 16 of 3072 16.8 / 15.8 +
// 8.6, over 60 of 2048 15.7 / 23.1 + 6.7; at 2048 pairs 8.6 / 7.5 + 6.4, 8.2 / 7.3 + 4.2, 7.9 / 8.6 + 5.2, 7.3 / 12.6 + 4.7.  Whole experts: 118 tokens, four of 10 of [1408 x 1664], 46.2 -> 40.5 us, 600,
// four of 60 of [768 x 1024], 81.2 -> 69.4.
constexpr int MOE_SORT_PAIRS = 4096;
__global__ __launch_bounds__(256) void moe_sort_gather_kernel(const int64_t *__restrict__ ids, const u32x4 *__restrict__ x, int pairs,
                                                              int n_exp, int32_t *__restrict__ offsets, int32_t *__restrict__ pos,
                                                              u32x4 *__restrict__ xs, int top_k, int chunks) {
    __shared__ int32_t part[4];
    const int b = blockIdx.x, t = threadIdx.x;
    const bool is_pair = b < pairs;
    constexpr int HELD = 2;                              // 16-byte pieces of the row on their way while the pairs are counted
    const u32x4 *const from = x + (int64_t)(is_pair ? b / top_k : 0) * chunks;
    u32x4 held[HELD] = {};
#pragma unroll
    for (int i = 0; i < HELD; i++)
        if (is_pair && t + i * 256 < chunks) held[i] = from[t + i * 256];
    const int64_t own = is_pair ? ids[b] : b - pairs;
    int before = 0;
    for (int j0 = t; j0 - t < pairs; j0 += 2048) {
        int64_t e[8];
#pragma unroll
        for (int i = 0; i < 8; i++) e[i] = j0 + i * 256 < pairs ? ids[j0 + i * 256] : -1;
#pragma unroll
        for (int i = 0; i < 8; i++)
            before += __popcll(__ballot(e[i] >= 0 && e[i] < n_exp && (e[i] < own || (is_pair && e[i] == own && j0 + i * 256 < b))));
    }
    if ((t & 63) == 0) part[t >> 6] = before;
    __syncthreads();
    before = part[0] + part[1] + part[2] + part[3];
    if (!is_pair) {
        if (t == 0) offsets[own] = before;
        return;
    }
    const bool valid = own >= 0 && own < n_exp;
    if (t == 0) pos[b] = valid ? before : -1;
    if (!valid) return;                                  // pairs without an expert have no row
    u32x4 *const to = xs + (int64_t)before * chunks;
#pragma unroll
    for (int i = 0; i < HELD; i++)
        if (t + i * 256 < chunks) to[t + i * 256] = held[i];
    for (int c = t + HELD * 256; c < chunks; c += 256) to[c] = from[c];
}

// U pairs of one token: their places and weights on their way together, then their rows; added in order.
template <int U, typename AT, typename WT>
__device__ inline void combine_pairs(float (&sum)[8], const AT *__restrict__ y, const int32_t *__restrict__ pos, const WT *__restrict__ weight,
                                     int N) {
    using V8 = typename Vec8<AT>::type;
    int p[U];
    float w[U];
    V8 v[U];
#pragma unroll
    for (int j = 0; j < U; j++) {
        p[j] = pos[j];
        w[j] = (float)weight[j];
    }
#pragma unroll
    for (int j = 0; j < U; j++) v[j] = *(const V8 *)(y + (int64_t)(p[j] < 0 ? 0 : p[j]) * N);    // (a pair without an expert: any row, not added)
#pragma unroll
    for (int j = 0; j < U; j++) {
        if (p[j] < 0) continue;
#pragma unroll
        for (int i = 0; i < 8; i++) sum[i] = fmaf(w[j], (float)v[j][i], sum[i]);
    }
}

// Eight columns of one token per lane.  Bound by latency (3.8 us in a trace at 472 pairs of 1664 columns, 1.6 MB): a pair's place, its weight and
// its row one after the other, pair by pair, were three waits per pair; four pairs at a time are two (118 tokens, four of 10 experts
// of [1024 x 1664] in asym_int4, the whole call 34.9 -> 33.6 us, 32 tokens, two of 13, 30.2 -> 29.0, 512 of [14336 x 4096] 498 -> 496).
template <typename AT, typename WT>
__global__ __launch_bounds__(256) void moe_combine_kernel(const AT *__restrict__ y, const int32_t *__restrict__ pos,
                                                          const WT *__restrict__ weight, AT *__restrict__ out, int top_k, int N) {
    using V8 = typename Vec8<AT>::type;
    const int t = blockIdx.y, n = (blockIdx.x * 256 + threadIdx.x) * 8;
    if (n >= N) return;
    float sum[8] = {};
    y += n;
    pos += t * top_k;
    weight += t * top_k;
    int left = top_k;
    for (; left >= 4; left -= 4, pos += 4, weight += 4) combine_pairs<4>(sum, y, pos, weight, N);
    if (left == 3) combine_pairs<3>(sum, y, pos, weight, N);
    else if (left == 2) combine_pairs<2>(sum, y, pos, weight, N);
    else if (left == 1) combine_pairs<1>(sum, y, pos, weight, N);
    V8 o;
#pragma unroll
    for (int i = 0; i < 8; i++) o[i] = to_at<AT>(sum[i]);
    *(V8 *)(out + (int64_t)t * N + n) = o;
}

template <typename AT>
static void launch_combine(const void *y, const int32_t *pos, const void *weight, int w_dtype, void *out, int tokens, int top_k,
                           int N, hipStream_t st) {
    const dim3 grid((N / 8 + 255) / 256, tokens);
    if (w_dtype == DT_F32)
        hipLaunchKernelGGL((moe_combine_kernel<AT, float>), grid, dim3(256), 0, st, (const AT *)y, pos, (const float *)weight, (AT *)out, top_k, N);
    else if (w_dtype == DT_F16)
        hipLaunchKernelGGL((moe_combine_kernel<AT, _Float16>), grid, dim3(256), 0, st, (const AT *)y, pos, (const _Float16 *)weight, (AT *)out, top_k, N);
    else
        hipLaunchKernelGGL((moe_combine_kernel<AT, __bf16>), grid, dim3(256), 0, st, (const AT *)y, pos, (const __bf16 *)weight, (AT *)out, top_k, N);
}

// Whether the pairs go through the streaming kernel, which reads an expert's weights once per pair: while there are no
// more pairs than experts, so that few experts are read twice.  Measured (streaming / grouped, us): 60 experts of
// [1408 x 2048] sym_int4 at 8 / 32 / 64 pairs 17 / 41, 40 / 71, 74 / 78; 8 experts of [14336 x 4096] fp8_e4m3 at 4 / 8 /
// 12 pairs 146 / 213, 272 / 269, 396 / 319; 16 experts of [4096 x 2048] nf4 at 8 / 16 / 32 pairs 40 / 78, 72 / 80,
// 132 / 108.
static bool use_streaming(int pairs, int n_exp, int tokens) { return tokens == 1 || pairs <= n_exp; }

struct ExpertsWorkspace {
    size_t offsets, order, pos, xs, h, y, split, bytes;
};
static ExpertsWorkspace experts_workspace(int tokens, int top_k, int n_exp, int hidden, int inter) {
    const int64_t pairs = (int64_t)tokens * top_k;
    size_t at = 0;
    auto take = [&](size_t bytes) {
        const size_t here = at;
        at += (bytes + 255) & ~(size_t)255;
        return here;
    };
    ExpertsWorkspace w{};
    w.h = take(pairs * inter * 2);
    if (!use_streaming((int)pairs, n_exp, tokens)) {
        w.offsets = take((n_exp + 1) * sizeof(int32_t));
        w.order = take(pairs * sizeof(int32_t));
        w.pos = take(pairs * sizeof(int32_t));
        w.xs = take(pairs * hidden * 2);
        w.y = take(pairs * hidden * 2);
        w.split = take(grouped_workspace_bytes((int)pairs, n_exp, hidden, inter));
    }
    w.bytes = at;
    return w;
}

size_t experts_workspace_bytes(int tokens, int top_k, int n_exp, int hidden, int inter) {
    return experts_workspace(tokens, top_k, n_exp, hidden, inter).bytes;
}

// The caller has checked the arguments (shapes tileable, workspace of experts_workspace_bytes, n_exp <= MOE_MAX_EXPERTS,
// tokens * top_k < 2^24).
int launch_experts(const void *x, const int64_t *ids, const void *weight, int w_dtype, int tokens, int top_k, int n_exp,
                   const void *const *gates, const void *const *ups, const void *const *downs, void *workspace, void *out,
                   int qtype, int act_dtype, int hidden, int inter, int act, hipStream_t st) {
    if (n_exp > MOE_MAX_EXPERTS) return -3;
    const int pairs = tokens * top_k;
    const ExpertsWorkspace at = experts_workspace(tokens, top_k, n_exp, hidden, inter);
    uint8_t *const ws = (uint8_t *)workspace;
    void *const h = ws + at.h;
    if (use_streaming(pairs, n_exp, tokens))
        return launch_moe_gemv(x, ids, true, weight, w_dtype, tokens, top_k, n_exp, gates, ups, downs, h, out, qtype,
                               act_dtype, hidden, inter, act, st);
    int32_t *const offsets = (int32_t *)(ws + at.offsets), *const order = (int32_t *)(ws + at.order), *const pos = (int32_t *)(ws + at.pos);
    void *const xs = ws + at.xs, *const y = ws + at.y;
    const int waves = n_exp <= 512 ? 16 : 2;          // at most 48 KiB of counters
    if (pairs <= MOE_SORT_PAIRS && n_exp <= 512) {
        hipLaunchKernelGGL(moe_sort_gather_kernel, dim3(pairs + n_exp + 1), dim3(256), 0, st, ids, (const u32x4 *)x, pairs, n_exp, offsets,
                           pos, (u32x4 *)xs, top_k, hidden / 8);
    } else {
        hipLaunchKernelGGL(moe_route_kernel, dim3(1), dim3(64 * waves), (size_t)n_exp * (waves + 1) * sizeof(int32_t), st, ids, pairs, n_exp,
                           offsets, order, pos);
        hipLaunchKernelGGL(moe_gather_kernel, dim3(pairs), dim3(256), 0, st, (const u32x4 *)x, order, offsets + n_exp, (u32x4 *)xs, top_k,
                           hidden / 8);
    }
    if (int rc = launch_grouped_gemm(xs, gates, ups, h, offsets, n_exp, pairs, qtype, act_dtype, inter, hidden, act, nullptr, 0, st))
        return rc;
    if (int rc = launch_grouped_gemm(h, downs, nullptr, y, offsets, n_exp, pairs, qtype, act_dtype, hidden, inter, 0, ws + at.split,
                                     at.bytes - at.split, st)) return rc;
    if (act_dtype == DT_F16) launch_combine<_Float16>(y, pos, weight, w_dtype, out, tokens, top_k, hidden, st);
    else launch_combine<__bf16>(y, pos, weight, w_dtype, out, tokens, top_k, hidden, st);
    return 0;
}

}  // namespace lowbit
