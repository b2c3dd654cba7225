// Fused packed log_softmax + gather + entropy over bf16 logits, and its
// backward, for gfx950.
//
// Forward (replaces the chunk loop of TitanTrainer._forward_logprobs,
// meshy/backend/titan/trainer.py:451-527, i.e. -cross_entropy(z.float(), y)
// at trainer.py:414-428 and logsumexp(z) - sum(softmax(z) * z) at
// trainer.py:430-449, and the chunked gather of gather_logprobs,
// meshy/backend/titan/topk_loss.py:35-57): one workgroup streams one row of
// V logits from HBM exactly once with 16-byte loads, whatever the row's
// alignment, and keeps, per lane, the online (m, s, t) state of rowstream.h,
// updated once per register tile.
// Lanes and waves merge their triples; then
//     lse = m + ln s,  logp_k = z_{y_k} - lse,  H = ln 2 * (log2 s - t / s)
// for the row's n_ids gather ids y_k.  No fp32 copy of the logits is made.
//
// Backward: grad[r, v] = sum_k g[r,k] onehot(y_k)[v] - G_r exp(z[r, v] - lse[r]),
// G_r = sum_k g[r,k], written as bf16 in three launches: a per-row prep
// (-G_r and -lse_r log2 e into the workspace), the streaming pass of the
// softmax term, and a fixup of the n_ids one-hot positions.  The streaming
// pass walks the flattened [rows * V] grid with a grid-stride loop when the
// logits are contiguous: on MI355X that order writes 8 % faster than one
// workgroup per row.
#include <algorithm>
#include <atomic>
#include <mutex>

#include "rowstream.h"

namespace meshy {
namespace {

// thread 0: lse, entropy, and (with one id) the log-prob.
__device__ __forceinline__ float id_logp(int64_t y, float zy, float lse, int64_t V) {
    if (y == kIgnoreIndex) return 0.f;
    if (y < 0 || y >= V) return __builtin_nanf("");
    return zy - lse;
}

// Loads the row's gather id for thread `tid` (< n_ids) and its logit.
__device__ __forceinline__ void load_id(const uint16_t* row, const int64_t* ids, int64_t r, int n_ids,
                                        int64_t V, int64_t& y, float& zy) {
    y = 0;
    zy = 0.f;
    const int tid = threadIdx.x;
    if (ids && tid < n_ids) {
        y = ids[r * n_ids + tid];
        if (y >= 0 && y < V) zy = bf16_to_f32(row[y]);
    }
}

// Writes the row's outputs once block_merge has left (m, s, t) in thread 0.
template <int NT>
__device__ __forceinline__ void finish_row(int64_t r, float m, float s, float t, int64_t y, float zy,
                                           int64_t V, int n_ids, float* logp, float* ent, float* lse_out) {
    __shared__ float s_lse;
    if (threadIdx.x == 0) {
        const float l2s = __log2f(s);
        const float lse = fmaf(l2s, kLn2, m);
        if (lse_out) lse_out[r] = lse;
        if (ent) ent[r] = kLn2 * (l2s - t / s);
        if (n_ids == 1 && logp) logp[r] = id_logp(y, zy, lse, V);
        s_lse = lse;
    }
    if (n_ids > 1 && logp) {
        __syncthreads();
        if (static_cast<int>(threadIdx.x) < n_ids) logp[r * n_ids + threadIdx.x] = id_logp(y, zy, s_lse, V);
    }
}

// The row's last rem (< NT * GMAX) 16-byte chunks as one tile of
// G = ceil(rem / NT) loads per thread, all in flight together.
template <int NT, int G, int GMAX>
__device__ __forceinline__ void lpe_tail(const v4u* base, int64_t rem, int tid, float& m, float& s, float& t) {
    if constexpr (G <= GMAX) {
        if (rem > static_cast<int64_t>(G) * NT) {
            lpe_tail<NT, G + 1, GMAX>(base, rem, tid, m, s, t);
            return;
        }
        v4u v[G];
        bool ok[G];
        load_tail<NT, G>(base, rem, tid, v, ok);
        float z[G * 8];
        unpack(v, z);
        accumulate_masked<true>(z, ok, m, s, t);
    }
}

// The exact tile update (tile max, rescale, accumulate) out of line: the rare
// fallback of accumulate_at, kept from sharing registers with the common path.
template <int U>
__device__ __forceinline__ void accumulate_exact(v4u (&v)[U], float& m, float& s, float& t) {
    float z[U * 8];
    unpack(v, z);
    accumulate(z, m, s, t);
}

// Bound by the read of the logits.  NT threads per row (fwd_threads), U 16-byte
// loads in flight per thread per tile.  A lane's first tile sets its running max; later tiles are accumulated against it
// (accumulate_at) and take the tile max only when an element lies more than 44
// above it.  The chunks left after the full tiles form one predicated tile.
// The elements outside the row's 16-byte chunks (row_span) are loaded before
// the first tile and added after the last, one per thread: 4096 rows of 50257
// logits take 65.6 us (6.28 TB/s) against 81.3 with 2-byte loads throughout.
template <int NT, int U>
__global__ __launch_bounds__(NT) void k_lpe_fwd_vec(const uint16_t* __restrict__ logits, int64_t T,
                                                    int64_t V, int64_t stride_b, int64_t stride_t,
                                                    const int64_t* __restrict__ ids, int n_ids,
                                                    float* __restrict__ logp, float* __restrict__ ent,
                                                    float* __restrict__ lse_out) {
    const int64_t r = blockIdx.x;
    const uint16_t* row = row_ptr(logits, r, T, stride_b, stride_t);
    const RowSpan sp = row_span(row, V);
    const int tid = threadIdx.x;
    int64_t y;
    float zy;
    load_id(row, ids, r, n_ids, V, y, zy);
    bool edge;
    const int64_t e = edge_element(sp, V, tid, edge);
    const float z_edge = edge ? bf16_to_f32(row[e]) : 0.f;

    float m = kInit, s = 0.f, t = 0.f;
    constexpr int64_t kTile = static_cast<int64_t>(NT) * U;
    const int64_t n_full = sp.n8 / kTile;
    const v4u* p = sp.body + tid;
    for (int64_t it = 0; it < n_full; ++it, p += kTile) {
        v4u v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = __builtin_nontemporal_load(p + u * NT);
        if (it == 0) {
            float z[U * 8];
            unpack(v, z);
            accumulate(z, m, s, t);
        } else if (!accumulate_at<true>(v, m, s, t)) {
            accumulate_exact(v, m, s, t);
        }
    }
    const int64_t rem = sp.n8 - n_full * kTile;
    if (rem > 0) lpe_tail<NT, 1, U>(sp.body + n_full * kTile, rem, tid, m, s, t);
    accumulate_one(z_edge, edge, m, s, t);

    block_merge<NT>(m, s, t);
    finish_row<NT>(r, m, s, t, y, zy, V, n_ids, logp, ent, lse_out);
}

// ---------------------------------------------------------------- backward

// Per row: ng = -G (NaN when an id is neither -100 nor in [0, V)) and
// nl = -lse * log2 e.
__global__ __launch_bounds__(256) void k_lp_bwd_prep(const int64_t* __restrict__ ids, int n_ids,
                                                     const float* __restrict__ lse,
                                                     const float* __restrict__ grad, int64_t n_rows,
                                                     int64_t V, float* __restrict__ ng,
                                                     float* __restrict__ nl) {
    const int64_t r = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (r >= n_rows) return;
    float G = 0.f;
    bool bad = false;
    for (int k = 0; k < n_ids; ++k) {
        const int64_t y = ids[r * n_ids + k];
        if (y == kIgnoreIndex) continue;
        if (y < 0 || y >= V) bad = true;
        G += grad[r * n_ids + k];
    }
    ng[r] = bad ? __builtin_nanf("") : -G;
    nl[r] = -lse[r] * kLog2e;
}

__device__ __forceinline__ v4u softmax_term8(v4u v, float ng, float nl) {
    float z[8];
    const v4u vv[1] = {v};
    unpack(vv, z);
    float q[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) q[k] = ng * fast_exp2(fmaf(z[k], kLog2e, nl));
    v4u o;
    o.x = pack_bf16x2(q[0], q[1]);
    o.y = pack_bf16x2(q[2], q[3]);
    o.z = pack_bf16x2(q[4], q[5]);
    o.w = pack_bf16x2(q[6], q[7]);
    return o;
}

// Row index of 16-byte chunk c of a contiguous [rows, V] grid (n8 chunks per
// row): a double-precision estimate corrected by one step.
__device__ __forceinline__ uint32_t row_of_chunk(uint32_t c, uint32_t n8, double inv_n8) {
    uint32_t r = static_cast<uint32_t>(static_cast<double>(c) * inv_n8);
    if (r * n8 > c) --r;
    else if ((r + 1) * n8 <= c) ++r;
    return r;
}

// Streaming pass over contiguous logits [rows, V], V % 8 == 0: grid-stride
// over the n_chunks 16-byte chunks, U loads in flight per thread.
template <int NT, int U>
__global__ __launch_bounds__(NT) void k_lp_bwd_flat(const v4u* __restrict__ z4, uint32_t n8,
                                                    uint32_t n_chunks, double inv_n8,
                                                    const float* __restrict__ ng,
                                                    const float* __restrict__ nl,
                                                    v4u* __restrict__ g4) {
    uint32_t i = blockIdx.x * (NT * U) + threadIdx.x;
    const uint32_t stride = gridDim.x * (NT * U);
    for (; i + (U - 1) * NT < n_chunks; i += stride) {
        v4u v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = __builtin_nontemporal_load(z4 + i + u * NT);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t c = i + u * NT;
            const uint32_t r = row_of_chunk(c, n8, inv_n8);
            __builtin_nontemporal_store(softmax_term8(v[u], ng[r], nl[r]), g4 + c);
        }
    }
    for (; i < n_chunks; i += NT) {
        const uint32_t r = row_of_chunk(i, n8, inv_n8);
        __builtin_nontemporal_store(softmax_term8(__builtin_nontemporal_load(z4 + i), ng[r], nl[r]), g4 + i);
    }
}

// Streaming pass, one workgroup per row: strided logits with 16-byte aligned
// rows and V % 8 == 0.
template <int NT, int U>
__global__ __launch_bounds__(NT) void k_lp_bwd_rows(const uint16_t* __restrict__ logits, int64_t T,
                                                    int64_t V, int64_t stride_b, int64_t stride_t,
                                                    const float* __restrict__ ng,
                                                    const float* __restrict__ nl,
                                                    uint16_t* __restrict__ grad) {
    const int64_t r = blockIdx.x;
    const v4u* row4 = reinterpret_cast<const v4u*>(row_ptr(logits, r, T, stride_b, stride_t));
    v4u* grow4 = reinterpret_cast<v4u*>(grad + r * V);
    const float g = ng[r], l = nl[r];
    const int64_t n8 = V >> 3;
    int64_t c = threadIdx.x;
    for (; c + (U - 1) * NT < n8; c += NT * U) {
        v4u v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = __builtin_nontemporal_load(row4 + c + u * NT);
#pragma unroll
        for (int u = 0; u < U; ++u) __builtin_nontemporal_store(softmax_term8(v[u], g, l), grow4 + c + u * NT);
    }
    for (; c < n8; c += NT) __builtin_nontemporal_store(softmax_term8(__builtin_nontemporal_load(row4 + c), g, l), grow4 + c);
}

// Streaming pass, generic: any alignment, stride and V.
template <int NT>
__global__ __launch_bounds__(NT) void k_lp_bwd_any(const uint16_t* __restrict__ logits, int64_t T,
                                                   int64_t V, int64_t stride_b, int64_t stride_t,
                                                   const float* __restrict__ ng,
                                                   const float* __restrict__ nl,
                                                   uint16_t* __restrict__ grad) {
    const int64_t r = blockIdx.x;
    const uint16_t* row = row_ptr(logits, r, T, stride_b, stride_t);
    uint16_t* grow = grad + r * V;
    const float g = ng[r], l = nl[r];
    for (int64_t e = threadIdx.x; e < V; e += NT)
        grow[e] = __bfloat16_as_ushort(__float2bfloat16(g * fast_exp2(fmaf(bf16_to_f32(row[e]), kLog2e, l))));
}

// One thread per (row, id): the final value at the id's position, i.e. the
// softmax term recomputed exactly as the streaming pass computed it, plus the
// gradients of every id of the row equal to this one.  Threads of duplicate
// ids store the same value.
__global__ __launch_bounds__(256) void k_lp_bwd_fix(const uint16_t* __restrict__ logits, int64_t T, int64_t V,
                                                    int64_t stride_b, int64_t stride_t,
                                                    const int64_t* __restrict__ ids, int n_ids,
                                                    const float* __restrict__ grad,
                                                    const float* __restrict__ ng,
                                                    const float* __restrict__ nl, int64_t n_rows,
                                                    uint16_t* __restrict__ out) {
    const int64_t j = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (j >= n_rows * n_ids) return;
    const int64_t r = j / n_ids;
    const int64_t y = ids[j];
    if (y < 0 || y >= V) return;  // ignored id, or a NaN row already written
    const float g = ng[r];
    if (isnan(g)) return;
    const uint16_t* row = row_ptr(logits, r, T, stride_b, stride_t);
    float q = g * fast_exp2(fmaf(bf16_to_f32(row[y]), kLog2e, nl[r]));
    for (int k = 0; k < n_ids; ++k)
        if (ids[r * n_ids + k] == y) q += grad[r * n_ids + k];
    out[r * V + y] = __bfloat16_as_ushort(__float2bfloat16(q));
}

// 8 16-byte loads in flight per thread per tile (4 are slower at every size).
// The flat backward: 256 threads x 4 loads, 65536 workgroups (sweep over
// 16384..65536 workgroups, 2..8 loads).
constexpr int kFwdUnroll = 8;
constexpr int kBwdThreads = 256;
constexpr int kBwdUnroll = 4;
constexpr uint32_t kBwdFlatBlocks = 65536;
constexpr int kMaxIds = 256;  // gather ids per row (one thread each)

// Shape checks; an empty call (rows * T == 0) accepts NULL arrays, as an
// empty tensor has no storage.
int check_common(const void* logits, int64_t rows, int64_t T, int64_t V, int64_t stride_b,
                 int64_t stride_t, const char* who) {
    if (rows < 0 || T < 0 || V <= 0)
        return set_error(MESHY_EINVAL, "%s: bad shape rows=%lld T=%lld V=%lld", who,
                         static_cast<long long>(rows), static_cast<long long>(T),
                         static_cast<long long>(V));
    if (stride_b < 0 || stride_t < 0) return set_error(MESHY_EINVAL, "%s: negative stride", who);
    if (T > 0 && rows > INT32_MAX / T) return set_error(MESHY_EINVAL, "%s: too many rows", who);
    if (!logits && rows * T > 0) return set_error(MESHY_ENULL, "%s: logits is NULL", who);
    return MESHY_OK;
}

bool vector_ok(const void* logits, int64_t stride_b, int64_t stride_t) {
    return (reinterpret_cast<uintptr_t>(logits) % 16 == 0) && (stride_b % 8 == 0) && (stride_t % 8 == 0);
}

// Threads of a row's workgroup.  Up to 256 rows there is one workgroup per CU
// at most, and a CU streams in proportion to its loads in flight: 512 threads
// take 13.0 us for 37 rows of 151936 logits and 16.0 for 256, against 19.1 and
// 21.1 with 256 threads (1024 threads: 12.4 and 16.3).  From 257 rows on, 256
// threads spread the rows more evenly (512 rows: 27.4 against 28.1 us; 4096
// rows of 50257: 65.6 against 72.2, where most of a row is the predicated last
// tile of 4096 chunks).  Many rows of at least 3 full tiles of 512 threads
// stream faster with those (4096 rows of 131072: 158.0 against 162.4 us; 16384
// of 151936: 703 against 714; 4096 of 81920, 2.5 tiles: 102.2 against 103.5).
int fwd_threads(int64_t n, int64_t V) {
    return n <= 256 || (n >= 2048 && V >= 3 * 512 * kFwdUnroll * 8) ? 512 : 256;
}

int launch_fwd(const uint16_t* logits, int64_t rows, int64_t T, int64_t V, int64_t stride_b,
               int64_t stride_t, const int64_t* ids, int n_ids, float* out, float* entropy, float* lse,
               hipStream_t stream, const char* who) {
    const int64_t n = rows * T;
    if (n == 0) return MESHY_OK;
    const dim3 grid(static_cast<unsigned>(n));
    auto go = [&](auto kernel, int threads) {
        hipLaunchKernelGGL(kernel, grid, dim3(threads), 0, stream, logits, T, V, stride_b, stride_t, ids, n_ids, out,
                           entropy, lse);
    };
    if (fwd_threads(n, V) == 512)
        go(k_lpe_fwd_vec<512, kFwdUnroll>, 512);
    else
        go(k_lpe_fwd_vec<256, kFwdUnroll>, 256);
    return check_launch(who);
}

size_t bwd_ws_bytes(int64_t n_rows) { return 2 * align_up(sizeof(float) * static_cast<size_t>(n_rows), 256); }

int launch_bwd(const uint16_t* logits, int64_t rows, int64_t T, int64_t V, int64_t stride_b,
               int64_t stride_t, const int64_t* ids, int n_ids, const float* lse, const float* grad_out,
               uint16_t* grad_logits, void* workspace, size_t workspace_bytes, hipStream_t stream,
               const char* who) {
    const int64_t n = rows * T;
    if (n == 0) return MESHY_OK;
    if (!workspace || workspace_bytes < bwd_ws_bytes(n))
        return set_error(MESHY_ESPACE, "%s: workspace needs %zu bytes", who, bwd_ws_bytes(n));
    float* ng = static_cast<float*>(workspace);
    float* nl = reinterpret_cast<float*>(static_cast<char*>(workspace) + bwd_ws_bytes(n) / 2);
    const unsigned row_blocks = static_cast<unsigned>(ceil_div(n, 256));
    hipLaunchKernelGGL(k_lp_bwd_prep, dim3(row_blocks), dim3(256), 0, stream, ids, n_ids, lse, grad_out, n, V, ng,
                       nl);
    int rc = check_launch(who);
    if (rc) return rc;
    const bool vec = vector_ok(logits, stride_b, stride_t) && reinterpret_cast<uintptr_t>(grad_logits) % 16 == 0 &&
                     V % 8 == 0;
    const bool contiguous = stride_t == V && (rows == 1 || stride_b == T * V);
    const int64_t n_chunks = n * (V / 8);
    // The grid-stride index stays below 2^32: n_chunks plus one grid stride.
    if (vec && contiguous && n_chunks <= (int64_t{1} << 32) - (int64_t{1} << 28)) {
        const int64_t need = ceil_div(n_chunks, kBwdThreads * kBwdUnroll);
        const unsigned blocks = static_cast<unsigned>(std::min<int64_t>(need, kBwdFlatBlocks));
        hipLaunchKernelGGL((k_lp_bwd_flat<kBwdThreads, kBwdUnroll>), dim3(blocks), dim3(kBwdThreads), 0, stream,
                           reinterpret_cast<const v4u*>(logits), static_cast<uint32_t>(V / 8),
                           static_cast<uint32_t>(n_chunks), 1.0 / static_cast<double>(V / 8), ng, nl,
                           reinterpret_cast<v4u*>(grad_logits));
    } else if (vec) {
        hipLaunchKernelGGL((k_lp_bwd_rows<kBwdThreads, kBwdUnroll>), dim3(static_cast<unsigned>(n)),
                           dim3(kBwdThreads), 0, stream, logits, T, V, stride_b, stride_t, ng, nl, grad_logits);
    } else {
        hipLaunchKernelGGL((k_lp_bwd_any<kBwdThreads>), dim3(static_cast<unsigned>(n)), dim3(kBwdThreads), 0,
                           stream, logits, T, V, stride_b, stride_t, ng, nl, grad_logits);
    }
    rc = check_launch(who);
    if (rc) return rc;
    const unsigned fix_blocks = static_cast<unsigned>(ceil_div(n * n_ids, 256));
    hipLaunchKernelGGL(k_lp_bwd_fix, dim3(fix_blocks), dim3(256), 0, stream, logits, T, V, stride_b, stride_t, ids,
                       n_ids, grad_out, ng, nl, n, grad_logits);
    return check_launch(who);
}

}  // namespace
}  // namespace meshy

extern "C" int meshy_logprob_entropy_fwd(const uint16_t* logits, int64_t rows, int64_t T, int64_t V,
                                         int64_t stride_b, int64_t stride_t, const int64_t* labels,
                                         float* logp, float* entropy, float* lse,
                                         hipStream_t stream) {
    using namespace meshy;
    clear_error();
    const char* who = "meshy_logprob_entropy_fwd";
    int rc = check_common(logits, rows, T, V, stride_b, stride_t, who);
    if (rc) return rc;
    if (rows * T == 0) return MESHY_OK;
    if (logp && !labels) return set_error(MESHY_ENULL, "%s: logp needs labels", who);
    return launch_fwd(logits, rows, T, V, stride_b, stride_t, logp ? labels : nullptr, logp ? 1 : 0, logp,
                      entropy, lse, stream, who);
}

extern "C" int meshy_gather_logprobs_fwd(const uint16_t* logits, int64_t rows, int64_t T, int64_t V,
                                         int64_t stride_b, int64_t stride_t, const int64_t* ids,
                                         int64_t n_ids, float* out, float* lse, hipStream_t stream) {
    using namespace meshy;
    clear_error();
    const char* who = "meshy_gather_logprobs_fwd";
    int rc = check_common(logits, rows, T, V, stride_b, stride_t, who);
    if (rc) return rc;
    if (n_ids < 1 || n_ids > kMaxIds)
        return set_error(MESHY_EINVAL, "%s: n_ids must be in [1, %d], got %lld", who, kMaxIds,
                         static_cast<long long>(n_ids));
    if (rows * T == 0) return MESHY_OK;
    if (!ids || !out) return set_error(MESHY_ENULL, "%s: ids and out are required", who);
    return launch_fwd(logits, rows, T, V, stride_b, stride_t, ids, static_cast<int>(n_ids), out, nullptr, lse,
                      stream, who);
}

extern "C" size_t meshy_logprob_bwd_workspace_size(int64_t n_rows) {
    return n_rows < 0 ? 0 : meshy::bwd_ws_bytes(n_rows);
}

extern "C" int meshy_logprob_bwd(const uint16_t* logits, int64_t rows, int64_t T, int64_t V,
                                 int64_t stride_b, int64_t stride_t, const int64_t* labels,
                                 const float* lse, const float* grad_logp, uint16_t* grad_logits,
                                 void* workspace, size_t workspace_bytes, hipStream_t stream) {
    using namespace meshy;
    clear_error();
    const char* who = "meshy_logprob_bwd";
    int rc = check_common(logits, rows, T, V, stride_b, stride_t, who);
    if (rc) return rc;
    if (rows * T == 0) return MESHY_OK;
    if (!labels || !lse || !grad_logp || !grad_logits)
        return set_error(MESHY_ENULL, "%s: labels, lse, grad_logp and grad_logits are required", who);
    return launch_bwd(logits, rows, T, V, stride_b, stride_t, labels, 1, lse, grad_logp, grad_logits, workspace,
                      workspace_bytes, stream, who);
}

// ------------------------------------------------ allocation-free backward
//
// meshy_logprob_bwd_noalloc runs the kernels of meshy_logprob_bwd with their
// two floats per row (-G and -lse log2 e) in this file-scope device array
// instead of a caller workspace.  Each GPU holds its own copy; host code
// reaches it only through the address hipGetSymbolAddress reports for the
// current device, looked up once per device and cached below.  Nothing in it
// must start at zero: the prep kernel writes every row's pair before the
// streaming pass and the fixup read it.  Calls that overlap on one GPU (on
// different streams) share the array and race.
static __device__ __align__(256) float scratch[2 * MESHY_NOALLOC_MAX_ROWS];

namespace meshy {
namespace {

constexpr int kMaxDevices = 64;
std::atomic<float*> g_scratch[kMaxDevices];
std::mutex g_scratch_mu;

// The current device's copy of `scratch` (looked up on its first use).
int scratch_of_current_device(float** out, const char* who) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return set_error(static_cast<int>(e), "%s: hipGetDevice: %s", who, hipGetErrorString(e));
    if (dev < 0 || dev >= kMaxDevices) return set_error(MESHY_EINVAL, "%s: device %d out of range", who, dev);
    float* p = g_scratch[dev].load(std::memory_order_acquire);
    if (!p) {
        std::lock_guard<std::mutex> lock(g_scratch_mu);
        p = g_scratch[dev].load(std::memory_order_relaxed);
        if (!p) {
            void* addr = nullptr;
            e = hipGetSymbolAddress(&addr, HIP_SYMBOL(scratch));
            if (e != hipSuccess || !addr)
                return set_error(e != hipSuccess ? static_cast<int>(e) : MESHY_EINVAL,
                                 "%s: hipGetSymbolAddress(scratch) on device %d: %s", who, dev,
                                 hipGetErrorString(e));
            p = static_cast<float*>(addr);
            g_scratch[dev].store(p, std::memory_order_release);
        }
    }
    *out = p;
    return MESHY_OK;
}

}  // namespace
}  // namespace meshy

extern "C" int meshy_logprob_bwd_noalloc(const uint16_t* logits, int64_t rows, int64_t T, int64_t V,
                                         int64_t stride_b, int64_t stride_t, const int64_t* labels,
                                         const float* lse, const float* grad_logp, uint16_t* grad_logits,
                                         hipStream_t stream) {
    using namespace meshy;
    clear_error();
    const char* who = "meshy_logprob_bwd_noalloc";
    int rc = check_common(logits, rows, T, V, stride_b, stride_t, who);
    if (rc) return rc;
    const int64_t n = rows * T;
    if (n == 0) return MESHY_OK;
    if (!labels || !lse || !grad_logp || !grad_logits)
        return set_error(MESHY_ENULL, "%s: labels, lse, grad_logp and grad_logits are required", who);
    if (n > MESHY_NOALLOC_MAX_ROWS)
        return set_error(MESHY_ESPACE, "%s: %lld rows exceed the static scratch of %d rows", who,
                         static_cast<long long>(n), MESHY_NOALLOC_MAX_ROWS);
    float* ws = nullptr;
    rc = scratch_of_current_device(&ws, who);
    if (rc) return rc;
    return launch_bwd(logits, rows, T, V, stride_b, stride_t, labels, 1, lse, grad_logp, grad_logits, ws,
                      bwd_ws_bytes(n), stream, who);
}

extern "C" int meshy_gather_logprobs_bwd(const uint16_t* logits, int64_t rows, int64_t T, int64_t V,
                                         int64_t stride_b, int64_t stride_t, const int64_t* ids,
                                         int64_t n_ids, const float* lse, const float* grad_out,
                                         uint16_t* grad_logits, void* workspace, size_t workspace_bytes,
                                         hipStream_t stream) {
    using namespace meshy;
    clear_error();
    const char* who = "meshy_gather_logprobs_bwd";
    int rc = check_common(logits, rows, T, V, stride_b, stride_t, who);
    if (rc) return rc;
    if (n_ids < 1 || n_ids > kMaxIds)
        return set_error(MESHY_EINVAL, "%s: n_ids must be in [1, %d], got %lld", who, kMaxIds,
                         static_cast<long long>(n_ids));
    if (rows * T == 0) return MESHY_OK;
    if (!ids || !lse || !grad_out || !grad_logits)
        return set_error(MESHY_ENULL, "%s: ids, lse, grad_out and grad_logits are required", who);
    return launch_bwd(logits, rows, T, V, stride_b, stride_t, ids, static_cast<int>(n_ids), lse, grad_out,
                      grad_logits, workspace, workspace_bytes, stream, who);
}

namespace meshy {
namespace {

// Bandwidth probe with K1's access pattern and no arithmetic.
template <int NT, int U>
__global__ __launch_bounds__(NT) void k_stream_read(const v4u* __restrict__ src, int64_t n16_per_row,
                                                    uint32_t* __restrict__ out) {
    const v4u* row = src + static_cast<int64_t>(blockIdx.x) * n16_per_row;
    uint32_t acc = 0;
    constexpr int64_t kTile = static_cast<int64_t>(NT) * U;
    int64_t c = threadIdx.x;
    for (; c + (U - 1) * NT < n16_per_row; c += kTile) {
        v4u v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = __builtin_nontemporal_load(row + c + u * NT);
#pragma unroll
        for (int u = 0; u < U; ++u) acc ^= v[u].x ^ v[u].y ^ v[u].z ^ v[u].w;
    }
    for (; c < n16_per_row; c += NT) {
        const v4u v = __builtin_nontemporal_load(row + c);
        acc ^= v.x ^ v.y ^ v.z ^ v.w;
    }
    acc = wave_sum(acc);
    if (threadIdx.x == 0 && acc == 0x9e3779b9u) out[0] = acc;  // keeps the loads live
}

}  // namespace
}  // namespace meshy

extern "C" int meshy_stream_read(const void* src, int64_t rows, int64_t row_bytes, uint32_t* out,
                                 hipStream_t stream) {
    using namespace meshy;
    clear_error();
    if (!src || !out) return set_error(MESHY_ENULL, "meshy_stream_read: NULL pointer");
    if (rows < 0 || row_bytes < 0 || row_bytes % 16 != 0 || rows > INT32_MAX)
        return set_error(MESHY_EINVAL, "meshy_stream_read: bad shape");
    if (reinterpret_cast<uintptr_t>(src) % 16 != 0) return set_error(MESHY_EALIGN, "meshy_stream_read: src misaligned");
    if (rows == 0) return MESHY_OK;
    hipLaunchKernelGGL((k_stream_read<256, 8>), dim3(static_cast<unsigned>(rows)), dim3(256), 0, stream,
                       static_cast<const v4u*>(src), row_bytes / 16, out);
    return check_launch("meshy_stream_read");
}
