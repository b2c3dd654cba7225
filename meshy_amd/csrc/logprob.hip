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
// G_r = sum_k g[r,k], written as bf16 in one pass over the 16-byte chunks of the
// flattened [rows * V] gradient, each taken once by a grid that covers them
// (k_lp_bwd_flat); short rows go whole to waves or workgroups.
#include <algorithm>
#include <atomic>
#include <type_traits>

#include "rowstream.h"

namespace meshy {
namespace {

constexpr int kMaxIds = 256;  // gather ids per row

// The log-prob of an id with logit zy.
__device__ __forceinline__ float id_logp(int64_t y, float zy, const Lse& lse, int64_t V) {
    if (y == kIgnoreIndex) return 0.f;
    if (y < 0 || y >= V) return __builtin_nanf("");
    return minus_lse(zy, lse);
}

// The row's gather ids that a thread of NT takes (id tid + NT j in y[j]) and
// their logits.
template <int NT>
struct RowIds {
    static constexpr int kPer = (kMaxIds + NT - 1) / NT;
    int64_t y[kPer];
    float z[kPer];
};

template <int NT>
__device__ __forceinline__ RowIds<NT> load_ids(const uint16_t* row, const int64_t* ids, int64_t r, int n_ids,
                                               int64_t V) {
    RowIds<NT> w;
#pragma unroll
    for (int j = 0; j < RowIds<NT>::kPer; ++j) {
        const int k = threadIdx.x + j * NT;
        w.y[j] = 0;
        w.z[j] = 0.f;
        if (ids && k < n_ids) {
            w.y[j] = ids[r * n_ids + k];
            if (w.y[j] >= 0 && w.y[j] < V) w.z[j] = bf16_to_f32(row[w.y[j]]);
        }
    }
    return w;
}

// ln s - ln 2 (t / s), rounded once: the quotient with its remainder, its
// product with ln 2 as two parts, and the errors of the large terms' sum.
__device__ __forceinline__ float entropy_of(float s, float t, const Lse& ln_s) {
    const float q = t / s;
    const float rest = fmaf(-q, s, t) * __builtin_amdgcn_rcpf(s);
    const float p = -q * kLn2High;
    float err;
    const float h = add_with_error(ln_s.hi, p, err);
    return h + (err + fmaf(-q, kLn2High, -p) + fmaf(-q, kLn2Low, ln_s.lo) - rest * kLn2);
}

// Writes the row's outputs once block_merge has left (m, s, t) in thread 0,
// which finishes them in two fp32 parts (in double it took 1.1 us longer where
// a CU has one row: 256 rows of 151936 logits 17.6 us, 16.5 so).
template <int NT>
__device__ __forceinline__ void finish_row(int64_t r, float m, float s, float t, const RowIds<NT>& w,
                                           int64_t V, int n_ids, float* logp, float* ent, float* lse_out) {
    __shared__ Lse s_lse;
    if (threadIdx.x == 0) {
        const Lse ln_s = ln_of(s);
        const Lse lse = lse_of(m, ln_s);
        if (lse_out) lse_out[r] = lse.hi + lse.lo;
        if (ent) ent[r] = entropy_of(s, t, ln_s);
        if (n_ids == 1 && logp) logp[r] = id_logp(w.y[0], w.z[0], lse, V);
        s_lse = lse;
    }
    if (n_ids > 1 && logp) {
        __syncthreads();
#pragma unroll
        for (int j = 0; j < RowIds<NT>::kPer; ++j) {
            const int k = threadIdx.x + j * NT;
            if (k < n_ids) logp[r * n_ids + k] = id_logp(w.y[j], w.z[j], s_lse, V);
        }
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

// A row's parts meet in slots: the triple of one part, each float in the low
// half of a 64-bit word whose high half is a tag drawn from the call, the slot
// and the word.  A word is one single-copy atomic, so a reader takes it exactly
// when its tag is the call's; whatever else the slot held carries another tag,
// and nothing is cleared.  Call e uses entry e % kSplitRing: a call overlapped
// by a later one of the same entry (kSplitRing calls on, on another stream) can
// lose a word, and then streams the row's other parts itself.
constexpr int kMaxParts = 16;     // merged in one row of 16 lanes
constexpr int kSplitSlots = 256;  // at least a launch's rows * parts
constexpr int kSplitRing = 64;
constexpr int kSplitPolls = 4000;  // of a waiting wave, some ms in all

struct SplitSlot {
    unsigned long long w[4];
};
__device__ SplitSlot g_split[kSplitRing][kSplitSlots];

__device__ __forceinline__ uint32_t split_tag(unsigned long long call, int slot, int w) {
    unsigned long long x = call * 0x9E3779B97F4A7C15ull + static_cast<unsigned>(slot * 4 + w) * 0xBF58476D1CE4E5B9ull;
    x ^= x >> 31;
    x *= 0x94D049BB133111EBull;
    x ^= x >> 29;
    return static_cast<uint32_t>(x >> 32);
}

// Merges the triples of a row's parts, part p in lane p, in a fixed order; the
// result in lane 0.
__device__ __forceinline__ void merge_parts(int parts, float& m, float& s, float& t) {
    const bool in = static_cast<int>(threadIdx.x) < parts;
    m = in ? m : kInit, s = in ? s : 0.f, t = in ? t : 0.f;
    merge_rows16<true>(m, s, t);
}

// Wave 0 polls, max_polls times at most, for the triples of parts 0 ..
// parts - 2 of row r, part p's in lane p.  Returns whether the polls ran out.
__device__ __forceinline__ bool poll_parts(const SplitSlot* slots, int r, int n_rows, int parts,
                                           unsigned long long call, int max_polls, float& m, float& s, float& t) {
    const int lane = threadIdx.x;
    const int slot = lane * n_rows + r;
    bool ready = lane + 1 >= parts;
    for (int poll = 0; poll < max_polls; ++poll) {
        if (!ready) {
            unsigned long long x[3];
#pragma unroll
            for (int w = 0; w < 3; ++w)
                x[w] = __hip_atomic_load(&slots[slot].w[w], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            ready = static_cast<uint32_t>(x[0] >> 32) == split_tag(call, slot, 0) &&
                    static_cast<uint32_t>(x[1] >> 32) == split_tag(call, slot, 1) &&
                    static_cast<uint32_t>(x[2] >> 32) == split_tag(call, slot, 2);
            if (ready) {
                m = __uint_as_float(static_cast<uint32_t>(x[0]));
                s = __uint_as_float(static_cast<uint32_t>(x[1]));
                t = __uint_as_float(static_cast<uint32_t>(x[2]));
            }
        }
        if (__ballot(!ready) == 0) return false;
        __builtin_amdgcn_s_sleep(1);
    }
    return true;
}

struct Split {
    int n_rows, parts;
    unsigned long long call;
    int max_polls;
};

// Bound by the read of the logits.  NT threads per workgroup and U 16-byte loads
// in flight per thread per tile (fwd_shape).  The wave's first tile
// sets the reference; later tiles are accumulated against it (accumulate_at) and
// take the tile max only when an element lies 8 above it.  The chunks left
// after the full tiles form one predicated tile.
// The elements outside the row's 16-byte chunks (row_span) are loaded before
// the first tile and added after the last, one per thread: 4096 rows of 50257
// logits take 65.6 us (6.28 TB/s) against 81.3 with 2-byte loads throughout.
//
// One workgroup takes a row, or with kSplit a part of one, where there are too
// few rows to fill the chip (fwd_parts): part p of row r is workgroup
// p * n_rows + r.  All but the last part publish their triple and end; the last
// one, dispatched after them, polls for theirs, merges and writes the row's
// outputs.  If its polls run out it streams the other parts itself, part by
// part, so that the result has the same bits whoever took them.
template <int NT, int U, bool kSplit>
__global__ __launch_bounds__(NT) void k_lpe_fwd_vec(const uint16_t* __restrict__ logits, int64_t T,
                                                    int64_t V, int64_t stride_b, int64_t stride_t,
                                                    const int64_t* __restrict__ ids, int n_ids,
                                                    float* __restrict__ logp, float* __restrict__ ent,
                                                    float* __restrict__ lse_out, Split sx) {
    static_assert(NT >= kLineElems + 8, "a thread per element outside the chunks");
    const int part = kSplit ? static_cast<int>(blockIdx.x) / sx.n_rows : 0;
    const int64_t r = kSplit ? static_cast<int>(blockIdx.x) % sx.n_rows : static_cast<int64_t>(blockIdx.x);
    const bool last = !kSplit || part + 1 == sx.parts;
    const uint16_t* row = row_ptr(logits, r, T, stride_b, stride_t);
    const RowSpan sp = row_span(row, V);
    const int tid = threadIdx.x;
    const RowIds<NT> w = load_ids<NT>(row, ids, r, n_ids, V);
    bool edge;
    const int64_t e = edge_element(sp, V, tid, edge);
    edge = edge && last;
    const float z_edge = edge ? bf16_to_f32(row[e]) : 0.f;

    float m, s, t;
    for (int p = part;;) {
        const v4u* body = sp.body;
        int64_t n8 = sp.n8;
        if constexpr (kSplit) {
            // Parts of whole 128-byte lines; the last ones may be short or empty.
            const int64_t per = ((sp.n8 + sx.parts - 1) / sx.parts + 7) / 8 * 8;
            const int64_t lo = min(p * per, sp.n8);
            body += lo;
            n8 = min(per, sp.n8 - lo);
        }
        m = kInit, s = 0.f, t = 0.f;
        constexpr int64_t kTile = static_cast<int64_t>(NT) * U;
        const int64_t n_full = n8 / kTile;
        const v4u* c = body + tid;
        for (int64_t it = 0; it < n_full; ++it, c += kTile) {
            v4u v[U];
#pragma unroll
            for (int u = 0; u < U; ++u) v[u] = __builtin_nontemporal_load(c + u * NT);
            if (it == 0) {
                float z[U * 8];
                unpack(v, z);
                accumulate_first<true>(z, m, s, t);
            } else if (!accumulate_at<true>(v, m, s, t)) {
                accumulate_exact(v, m, s, t);
            }
        }
        const int64_t rem = n8 - n_full * kTile;
        if (rem > 0) lpe_tail<NT, 1, U>(body + n_full * kTile, rem, tid, m, s, t);
        accumulate_one(z_edge, edge && p == part, m, s, t);

        block_merge<NT>(m, s, t);
        if constexpr (!kSplit) {
            break;
        } else {
            SplitSlot* slots = g_split[sx.call % kSplitRing];
            if (!last) {
                if (tid == 0) {
                    const int slot = part * sx.n_rows + static_cast<int>(r);
                    const float v[3] = {m, s, t};
#pragma unroll
                    for (int i = 0; i < 3; ++i)
                        __hip_atomic_store(&slots[slot].w[i],
                                           (static_cast<unsigned long long>(split_tag(sx.call, slot, i)) << 32) |
                                               __float_as_uint(v[i]),
                                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
                return;
            }
            __shared__ float s_part[kMaxParts][3];
            __shared__ int s_gave_up;
            if (tid < kWave) {
                if (tid == 0) s_part[p][0] = m, s_part[p][1] = s, s_part[p][2] = t;
                if (p == part) {  // the workgroup's own
                    const float own[3] = {lane_f32(m, 0), lane_f32(s, 0), lane_f32(t, 0)};
                    const bool gave_up = poll_parts(slots, static_cast<int>(r), sx.n_rows, sx.parts, sx.call,
                                                    sx.max_polls, m, s, t);
                    if (tid == part) m = own[0], s = own[1], t = own[2];
                    if (tid == 0) s_gave_up = gave_up;
                }
            }
            __syncthreads();  // also keeps block_merge's scratch for the next part
            if (p == part ? !s_gave_up : p + 2 == sx.parts) {
                if (tid < kWave) {
                    if (p != part) {
                        const float* q = s_part[min(tid, part)];
                        m = q[0], s = q[1], t = q[2];
                    }
                    merge_parts(sx.parts, m, s, t);
                }
                break;
            }
            p = p == part ? 0 : p + 1;
        }
    }
    finish_row<NT>(r, m, s, t, w, V, n_ids, logp, ent, lse_out);
}

// ---------------------------------------------------------------- backward

struct BwdArgs {
    const uint16_t* logits;
    int64_t V, stride_b, stride_t;
    uint32_t T;         // 0: every row lies stride_t after the one before
    int64_t row0;       // the launch's first row (a multiple of 8); the arrays below start at it
    int64_t n_elems;    // of the launch's gradient
    uint32_t n_chunks;  // ceil(n_elems / 8)
    double inv_v;
    int n_ids;
    const int64_t* ids;
    const float* lse;
    const float* grad_logp;
    uint16_t* out;
};

__device__ __forceinline__ uint16_t bf16_bits(float x) { return __bfloat16_as_ushort(__float2bfloat16(x)); }

// The k-th id of a row (-1 where it adds nothing) and its gradient; returns
// whether it is neither -100 nor in [0, V).
__device__ __forceinline__ bool row_id(const BwdArgs& a, int64_t r, int k, int64_t& y, float& g) {
    y = a.ids[r * a.n_ids + k];
    g = a.grad_logp[r * a.n_ids + k];
    const bool ignored = y == kIgnoreIndex;
    const bool bad = !ignored && (y < 0 || y >= a.V);
    if (ignored) g = 0.f;
    if (ignored || bad) y = -1;
    return bad;
}

__device__ __forceinline__ const uint16_t* row_at(const BwdArgs& a, uint32_t r) {
    if (a.T == 0) return a.logits + r * a.stride_t;
    const uint32_t b = r / a.T;
    return a.logits + b * a.stride_b + (r - b * a.T) * a.stride_t;
}

// What the pass needs of a row: ng = -G (NaN when an id is out of range),
// nl = -lse log2 e, and its ids with their gradients, NB 64-id blocks with one
// id per lane.  NB = 0: one id, the same in every lane.
template <int NB>
struct BwdRow {
    float ng, nl;
    int64_t y[NB ? NB : 1];
    float g[NB ? NB : 1];
};

// Row r, wave-uniform; all 64 lanes active.
template <int NB>
__device__ __forceinline__ BwdRow<NB> bwd_row(const BwdArgs& a, int64_t r) {
    BwdRow<NB> w;
    w.nl = -a.lse[r] * kLog2e;
    if constexpr (NB == 0) {
        const bool bad = row_id(a, r, 0, w.y[0], w.g[0]);
        w.ng = bad ? __builtin_nanf("") : -w.g[0];
    } else {
        bool bad = false;
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const int k = b * kWave + threadIdx.x % kWave;
            const bool over = row_id(a, r, min(k, a.n_ids - 1), w.y[b], w.g[b]);
            bad |= over && k < a.n_ids;
            if (k >= a.n_ids) w.y[b] = -1, w.g[b] = 0.f;
        }
        float G = 0.f;
#pragma unroll
        for (int b = 0; b < NB; ++b) G += wave_sum(w.g[b]);
        w.ng = __ballot(bad) ? __builtin_nanf("") : -G;
    }
    return w;
}

// q[0 .. 7] += the row's one-hot terms among the 512 elements of the wave whose
// first is the row's column lo: lane l holds columns lo + 8 l .. lo + 8 l + 7.
// Duplicate ids add in order of k.
template <int NB>
__device__ __forceinline__ void add_onehot(const BwdRow<NB>& w, int64_t lo, float (&q)[8]) {
    const int lane = threadIdx.x % kWave;
    auto add = [&](int off, float g) {  // wave-uniform offset from lo
        const float gl = lane == off >> 3 ? g : 0.f;
#pragma unroll
        for (int k = 0; k < 8; ++k)
            if ((off & 7) == k) q[k] += gl;
    };
#pragma unroll
    for (int b = 0; b < (NB ? NB : 1); ++b) {
        const int64_t off = w.y[b] - lo;
        const bool in = w.y[b] >= 0 && static_cast<uint64_t>(off) < 8 * kWave;
        if constexpr (NB == 0) {
            if (in) add(static_cast<int>(off), w.g[0]);
        } else {
            uint64_t hit = __ballot(in);
            while (hit) {
                const int l = __builtin_ctzll(hit);
                hit &= hit - 1;
                add(__builtin_amdgcn_readlane(static_cast<int>(off), l), lane_f32(w.g[b], l));
            }
        }
    }
}

// Row and column of element e of the launch's [rows, V] gradient: a
// double-precision estimate (e is exact in it) corrected by one step.
__device__ __forceinline__ void locate(const BwdArgs& a, int64_t e, uint32_t& r, int64_t& pos) {
    r = static_cast<uint32_t>(static_cast<double>(e) * a.inv_v);
    pos = e - r * a.V;
    if (pos < 0) {
        --r;
        pos += a.V;
    } else if (pos >= a.V) {
        ++r;
        pos -= a.V;
    }
}

// 16 bytes at any element (the hardware's global loads need no alignment).
typedef v4u v4u_any __attribute__((aligned(2)));

__device__ __forceinline__ v4u load_any(const uint16_t* p) {
    return __builtin_nontemporal_load(reinterpret_cast<const v4u_any*>(p));
}

// The last n (1 .. 7) of a's 8 elements, then b's first ones.
__device__ __forceinline__ v4u join(const v4u& a, const v4u& b, int n) {
    const uint64_t a0 = a.x | static_cast<uint64_t>(a.y) << 32, a1 = a.z | static_cast<uint64_t>(a.w) << 32;
    const uint64_t b0 = b.x | static_cast<uint64_t>(b.y) << 32, b1 = b.z | static_cast<uint64_t>(b.w) << 32;
    const int up = 16 * (n & 3), down = 64 - up;
    uint64_t lo, hi;
    if (n > 4) {
        lo = up ? a0 >> down | a1 << up : a0;
        hi = up ? a1 >> down | b0 << up : a1;
    } else {
        lo = up ? a1 >> down | b0 << up : a1;
        hi = up ? b0 >> down | b1 << up : b0;
    }
    return v4u{static_cast<uint32_t>(lo), static_cast<uint32_t>(lo >> 32), static_cast<uint32_t>(hi),
               static_cast<uint32_t>(hi >> 32)};
}

// A wave-uniform value moved to scalar registers.
__device__ __forceinline__ int64_t uniform_i64(int64_t x) {
    return (static_cast<int64_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(x >> 32))) << 32) |
           static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(x)));
}

// The whole backward in one pass over the 16-byte chunks of the contiguous
// gradient, bound by its read and write: 5.95 TB/s on [8192, 151936] (837 us
// with the forward's 358 in one loop; 861 in three launches), 5.99 on
// [8192, 50257] (275 us; 610 with 2-byte accesses).  Each wave takes U groups
// of 64 consecutive chunks, its U loads per lane in flight together, and the
// grid covers the chunks once: U = 2 takes 1160 us forward and backward on
// [8192, 151936], U = 4 and 8 1205 and 1243, a grid-stride loop of 65536
// workgroups 1200; going from the last chunk to the first (towards what the
// forward read last) changes nothing.  kContig: the logits are contiguous too,
// so a chunk is 8 consecutive elements of both whatever V is; other logits are
// read at their row's address, and where a chunk holds a row's end, the row's
// last 8 and the next row's first 8 are joined (16384 strided rows of 1000 logits
// 14 us, 38 with such chunks read one by one).  Most waves' U groups lie in one row, whose
// factors and ids are then wave-uniform: the wave reads them itself while its
// logits are in flight, which costs less than the two passes over the rows
// (factors before, one-hot terms after) that it replaces.  Waves that hold a
// row's end take each of their rows in turn.
template <int NT, int U, int NB, bool kContig>
__global__ __launch_bounds__(NT) void k_lp_bwd_flat(BwdArgs a) {
    const int lane = threadIdx.x % kWave;
    const uint32_t c0 = blockIdx.x * (NT * U) + __builtin_amdgcn_readfirstlane(threadIdx.x / kWave) * (kWave * U);
    if (c0 >= a.n_chunks) return;
    const int64_t last = a.n_chunks - 1;
    const int64_t e0 = static_cast<int64_t>(c0) * 8;
    uint32_t r;
    int64_t lo;
    locate(a, e0, r, lo);
    r = __builtin_amdgcn_readfirstlane(r);
    lo = uniform_i64(lo);
    const uint16_t* row = row_at(a, static_cast<uint32_t>(a.row0) + r);
    // Lanes past the end repeat the last chunk.  A chunk whose 8 logits do not
    // lie together (`part` of them end a row, or the tensor) is read below.
    v4u v[U];
    const uint16_t* src[U];
    int part[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int64_t e = min<int64_t>(c0 + u * kWave + lane, last) * 8;
        part[u] = 0;
        if constexpr (kContig) {
            src[u] = a.logits + a.row0 * a.V + e;
            if (e + 8 > a.n_elems) part[u] = static_cast<int>(a.n_elems - e);
        } else {
            uint32_t er = r;
            int64_t pos = lo + (e - e0);
            src[u] = row + pos;
            if (pos + 8 > a.V) {
                locate(a, e, er, pos);
                src[u] = row_at(a, static_cast<uint32_t>(a.row0) + er) + pos;
                if (pos + 8 > a.V) part[u] = static_cast<int>(a.V - pos);
            }
        }
        if (part[u]) src[u] -= 8 - part[u];
        v[u] = load_any(src[u]);
    }
    const BwdRow<NB> w0 = bwd_row<NB>(a, r);
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int64_t c = static_cast<int64_t>(c0) + u * kWave + lane;
        const int64_t e = c * 8;
        if (part[u]) {
            v4u next{0, 0, 0, 0};
            if constexpr (!kContig) {  // the next row's first logits
                uint32_t er;
                int64_t pos;
                locate(a, min(c, last) * 8, er, pos);
                if ((er + 1) * a.V < a.n_elems) next = load_any(row_at(a, static_cast<uint32_t>(a.row0) + er + 1));
            }
            v[u] = join(v[u], next, part[u]);
        }
        float z[8], q[8];
        const v4u vv[1] = {v[u]};
        unpack(vv, z);
#pragma unroll
        for (int k = 0; k < 8; ++k) q[k] = w0.ng * fast_exp2(fmaf(z[k], kLog2e, w0.nl));
        add_onehot(w0, lo + u * 8 * kWave, q);
        // Elements of the rows that start inside this group.
        const int64_t end = min<int64_t>(e0 + (u + 1) * 8 * kWave, a.n_elems);
        for (uint32_t rr = r + 1; rr * a.V < end; ++rr) {
            const int64_t at = e - rr * a.V;  // the lane's column in row rr
            const BwdRow<NB> w = bwd_row<NB>(a, rr);
            float x[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) x[k] = w.ng * fast_exp2(fmaf(z[k], kLog2e, w.nl));
            add_onehot(w, e0 + u * 8 * kWave - rr * a.V, x);
#pragma unroll
            for (int k = 0; k < 8; ++k) q[k] = at + k >= 0 ? x[k] : q[k];
        }
        if (c <= last) {
            v4u o;
            o.x = pack_bf16x2(q[0], q[1]);
            o.y = pack_bf16x2(q[2], q[3]);
            o.z = pack_bf16x2(q[4], q[5]);
            o.w = pack_bf16x2(q[6], q[7]);
            if (e + 8 <= a.n_elems) {
                __builtin_nontemporal_store(o, reinterpret_cast<v4u*>(a.out) + c);
            } else {
                for (int k = 0; e + k < a.n_elems; ++k) a.out[e + k] = bf16_bits(q[k]);
            }
        }
    }
}

// Orders the wave's memory operations before and after it across its lanes.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

// Short rows: each wave takes R rows (a power of two, 8 to 64), whose gradient is
// a whole number of 16-byte chunks of its own.  The lanes first read the rows'
// factors (64 / R of them to a row's ids) into LDS, then take the chunks, each
// with the factors of its row or rows.  One id per row is added in registers;
// several are written again after the chunks, each with the gradients of every
// id equal to its own.  inv = floor(2^32 / V) + 1: the rows' R V elements are few
// enough for the row of one to be the high half of its product with inv.
template <int NT, bool kOneId, bool kContig>
__global__ __launch_bounds__(NT) void k_lp_bwd_short(BwdArgs a, uint32_t n_rows, int R, uint32_t inv) {
    __shared__ float s_ng[NT / kWave][kWave], s_nl[NT / kWave][kWave], s_g[NT / kWave][kWave];
    __shared__ int s_y[NT / kWave][kWave];
    const int lane = threadIdx.x % kWave;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int64_t first = (static_cast<int64_t>(blockIdx.x) * (NT / kWave) + wid) * R;
    if (first >= n_rows) return;
    const uint32_t r0 = static_cast<uint32_t>(first);
    const int rows = min(R, static_cast<int>(n_rows - r0));
    const int V = static_cast<int>(a.V);
    float *ng = s_ng[wid], *nl = s_nl[wid], *sg = s_g[wid];
    int* sy = s_y[wid];
    {
        const int rl = lane & (R - 1);
        const bool in = rl < rows;
        float G = 0.f, g = 0.f;
        int64_t y = -1;
#pragma unroll 4
        for (int k = lane / R; in && k < a.n_ids; k += kWave / R) {
            const bool bad = row_id(a, r0 + rl, k, y, g);
            G += bad ? __builtin_nanf("") : g;
        }
        for (int off = R; off < kWave; off <<= 1) G += __shfl_xor(G, off, kWave);
        if (lane < R) {
            ng[rl] = -G;
            nl[rl] = in ? -a.lse[r0 + rl] * kLog2e : 0.f;
            if (kOneId) {
                sy[rl] = static_cast<int>(y);
                sg[rl] = g;
            }
        }
    }
    wave_sync();
    const int64_t base = r0 * a.V;  // the wave's first element (a multiple of 8)
    const int n_el = rows * V;
    for (int e = 8 * lane; e < n_el; e += 8 * kWave) {
        int rl = static_cast<int>(__umulhi(static_cast<uint32_t>(e), inv));
        int col = e - rl * V;
        const bool whole = e + 8 <= n_el;  // else the tensor's end
        float z[8];
        if (kContig || col + 8 <= V) {
            const uint16_t* src = kContig ? a.logits + base + e : row_at(a, r0 + rl) + col;
            const v4u v[1] = {whole ? load_any(src) : join(load_any(src - (8 - (n_el - e))), v4u{0, 0, 0, 0}, n_el - e)};
            unpack(v, z);
        } else {
            uint32_t h[8];
            int er = rl, ec = col;
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                if (ec == V) ec = 0, er = min(er + 1, rows - 1);
                h[k] = row_at(a, r0 + er)[ec++];
            }
#pragma unroll
            for (int k = 0; k < 8; ++k) z[k] = bf16_to_f32(static_cast<uint16_t>(h[k]));
        }
        float q[8];
        if (col + 8 <= V) {
            const float n = ng[rl], l = nl[rl];
            const int d = kOneId ? sy[rl] - col : 0;  // below 0 without an id
            const float g = kOneId ? sg[rl] : 0.f;
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                q[k] = n * fast_exp2(fmaf(z[k], kLog2e, l));
                if (kOneId) q[k] += d == k ? g : 0.f;
            }
        } else {
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                if (col == V) col = 0, rl = min(rl + 1, rows - 1);
                q[k] = ng[rl] * fast_exp2(fmaf(z[k], kLog2e, nl[rl]));
                if (kOneId) q[k] += sy[rl] == col ? sg[rl] : 0.f;
                ++col;
            }
        }
        uint16_t* out = a.out + base + e;
        if (whole) {
            const v4u o{pack_bf16x2(q[0], q[1]), pack_bf16x2(q[2], q[3]), pack_bf16x2(q[4], q[5]),
                        pack_bf16x2(q[6], q[7])};
            *reinterpret_cast<v4u*>(out) = o;
        } else {
            for (int k = 0; e + k < n_el; ++k) out[k] = bf16_bits(q[k]);
        }
    }
    if constexpr (!kOneId) {
        wave_sync();  // the chunks are written
        for (int i = lane; i < rows * a.n_ids; i += kWave) {
            const int rl = i / a.n_ids;
            const int64_t id0 = static_cast<int64_t>(r0 + rl) * a.n_ids;
            const int64_t y = a.ids[id0 + i - rl * a.n_ids];
            const float n = ng[rl];
            if (y < 0 || y >= V || isnan(n)) continue;  // ignored, or a row of NaN
            float q = n * fast_exp2(fmaf(bf16_to_f32(row_at(a, r0 + rl)[y]), kLog2e, nl[rl]));
            for (int k = 0; k < a.n_ids; ++k) q += a.ids[id0 + k] == y ? a.grad_logp[id0 + k] : 0.f;
            a.out[base + rl * V + y] = bf16_bits(q);
        }
    }
}

// One workgroup per row, an element per thread at a time: short rows with many
// ids (kBwdShortV), gradients that are not 16-byte aligned, and tensors of one
// logit per row or fewer than 8 in all.  The one-hot positions are written
// again after the row, each with the gradients of every id equal to its own.
template <int NT, int NB>
__global__ __launch_bounds__(NT) void k_lp_bwd_any(BwdArgs a) {
    const int64_t r = blockIdx.x;
    const uint16_t* row = row_at(a, static_cast<uint32_t>(r));
    uint16_t* grow = a.out + r * a.V;
    const BwdRow<NB> w = bwd_row<NB>(a, r);
    auto term = [&](int64_t e) { return w.ng * fast_exp2(fmaf(bf16_to_f32(row[e]), kLog2e, w.nl)); };
    for (int64_t e = threadIdx.x; e < a.V; e += NT) {
        const float q = term(e);
        grow[e] = bf16_bits(NB == 0 && w.y[0] == e ? q + w.g[0] : q);
    }
    if constexpr (NB > 0) {
        static_assert(NT >= kMaxIds, "one thread per id");
        __shared__ int64_t s_y[kMaxIds];
        __shared__ float s_g[kMaxIds];
        const int j = threadIdx.x;
        int64_t y = -1;
        float g = 0.f;
        if (j < a.n_ids) {
            row_id(a, r, j, y, g);
            s_y[j] = y;
            s_g[j] = g;
        }
        __syncthreads();
        if (y < 0) return;
        float q = term(y);
        for (int k = 0; k < a.n_ids; ++k) q += s_y[k] == y ? s_g[k] : 0.f;
        grow[y] = bf16_bits(q);
    }
}

// 16-byte loads in flight per thread per tile, for the rows that fill several
// tiles, for middle ones and for the others (the last tile is predicated and
// rounds up).
constexpr int kFwdUnroll = 8, kFwdMidUnroll = 3, kFwdShortUnroll = 2;
constexpr int kBwdThreads = 256;
constexpr int kBwdUnroll = 2;
// Below this a wave of the flat pass holds several rows and waits for the
// factors of one after the other: with more than one id, rows go whole to waves
// if they are many and their ids few, else to workgroups, whose threads add up
// a row's ids from LDS.  In us (before: three launches through a workspace):
//   rows x logits, ids     flat    waves   workgroups   before
//   131072 x 64, 1                 8.3     43           17
//   65536 x 264, 1         20      15                   20
//   65536 x 264, 9         41      31                   39
//   65536 x 200, 16                31      61           44
//   65536 x 200, 64                216     88           256
//   8192 x 256, 9          10.8    8.3     7.3          12.4
//   1000 x 256, 64         41      77      5.7          34
//   65536 x 512, 9         38      45      70           55
// One id: the flat pass takes rows from half this length on.
constexpr int64_t kBwdShortV = 512;
constexpr int64_t kBwdMaxElems = int64_t{1} << 33;  // of one launch: 32-bit chunk indices

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

// Threads and loads per thread of a workgroup that takes a whole row.
// Up to 256 rows there is one workgroup per CU at most, and a CU streams in
// proportion to its loads in flight: 512 threads of 8 loads take 13.0 us for 37
// undivided rows of 151936 logits, 256 threads 19.1.  From 2048 rows on, long
// rows (3 full tiles and more) stream fastest with those too (16384 rows of
// 151936: 703 us against 714 with 256 threads; 4096: 181 against 184 with 2
// loads).  All others take the registers of 2 or 3 loads and 8 waves per SIMD, in
// fewer threads where a short row would leave them idle, as long as the rows
// still fill the CUs (128 threads: 16 workgroups per CU, 4096 in all):
//   4206 rows of 50257 logits    512 x 3: 67 us   512 x 2: 68   256 x 8: 67
//   2048 rows of 50257           512 x 3: 33      512 x 2: 35   256 x 8: 35
//   4096 rows of 65537           512 x 3: 80      512 x 2: 80   256 x 8: 83
//   4096 rows of 32768           512 x 2: 42      256 x 2: 43   256 x 8: 43
//   4096 rows of 16384           256 x 2: 23      512 x 2: 24   256 x 8: 25
//   1024 rows of 24576           512 x 2: 9.9     256 x 2: 10.3 256 x 8: 11.2
//   16384 rows of 8192           128 x 2: 42      256 x 2: 44   256 x 8: 58
//   2048 rows of 8192            256 x 2: 8.2     128 x 2: 9.2  256 x 8: 10.2
//   131072 rows of 64            128 x 2: 84      256 x 2: 150  256 x 8: 190
// Many gather ids of a row that is not the shortest want more threads (16384
// rows of 4096, 200 ids: 38 us with 256, 42 with 128).
struct FwdShape {
    int threads, unroll;
};

FwdShape fwd_shape(int64_t n, int64_t V, int n_ids) {
    if (n <= 256 || (n >= 2048 && V >= 3 * 512 * kFwdUnroll * 8)) return {512, kFwdUnroll};
    if (V <= 1024 || (n_ids <= 128 && (V <= 4096 || (V <= 8192 && n >= 4096)))) return {128, kFwdShortUnroll};
    const bool mid = V >= 3 * 512 * kFwdMidUnroll * 8 && V < 3 * 512 * kFwdUnroll * 8;
    return {V < 32768 && n > 1024 ? 256 : 512, mid ? kFwdMidUnroll : kFwdShortUnroll};
}

// Workgroups per row.  One workgroup to a row is bound by its CU's exponentials
// (8 of its 11 us for 151936 logits), so rows that leave CUs idle are divided:
// the kernel alone takes 4.9 us for one row of 151936 logits instead of 10.1,
// 7.3 for 37 instead of 13.1 and 11.5 for 128 instead of 13.7; 37 rows of 50257
// 6.0 instead of 7.1.  Two workgroups to a CU are slower (37 rows: 7.9 us, 128:
// 12.1), as are parts of fewer than 8192 logits, and at 32000 logits the meeting
// costs what the split gains (37 rows: 5.9 us in 3 parts, 5.5 whole).
constexpr int64_t kSplitRows = 128;
constexpr int64_t kSplitWorkgroups = 256;
constexpr int64_t kSplitMinV = 49152;
constexpr int64_t kSplitPartV = 8192;
static_assert(kSplitWorkgroups <= kSplitSlots, "a slot per workgroup");

int fwd_parts(int64_t n, int64_t V) {
    if (n > kSplitRows || V < kSplitMinV) return 1;
    return static_cast<int>(std::min<int64_t>({kMaxParts, kSplitWorkgroups / n, V / kSplitPartV}));
}

int launch_fwd(const uint16_t* logits, int64_t rows, int64_t T, int64_t V, int64_t stride_b,
               int64_t stride_t, const int64_t* ids, int n_ids, float* out, float* entropy, float* lse,
               hipStream_t stream, const char* who, int max_polls) {
    const int64_t n = rows * T;
    if (n == 0) return MESHY_OK;
    const int parts = fwd_parts(n, V);
    // A replay would take the slots of the one before: a captured call is not
    // divided (its last bits may then differ; the last part's workgroups taking
    // every part in turn gives the same ones in 19 us for 37 rows of 151936
    // logits and 32 for one, where whole rows take 10.6 and 10.2).
    if (parts > 1 && !capturing(stream)) {
        static std::atomic<unsigned long long> calls{0};  // the slots' tags tell calls apart
        const unsigned long long call = calls.fetch_add(1, std::memory_order_relaxed) + 1;
        hipLaunchKernelGGL((k_lpe_fwd_vec<512, kFwdUnroll, true>), dim3(static_cast<unsigned>(n * parts)), dim3(512), 0,
                           stream, logits, T, V, stride_b, stride_t, ids, n_ids, out, entropy, lse,
                           Split{static_cast<int>(n), parts, call, max_polls});
        return check_launch(who);
    }
    const dim3 grid(static_cast<unsigned>(n));
    const FwdShape shape = fwd_shape(n, V, n_ids);
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, dim3(shape.threads), 0, stream, logits, T, V, stride_b, stride_t, ids, n_ids,
                           out, entropy, lse, Split{});
    };
    if (shape.unroll == kFwdUnroll) go(k_lpe_fwd_vec<512, kFwdUnroll, false>);
    else if (shape.unroll == kFwdMidUnroll) go(k_lpe_fwd_vec<512, kFwdMidUnroll, false>);
    else if (shape.threads == 512) go(k_lpe_fwd_vec<512, kFwdShortUnroll, false>);
    else if (shape.threads == 256) go(k_lpe_fwd_vec<256, kFwdShortUnroll, false>);
    else go(k_lpe_fwd_vec<128, kFwdShortUnroll, false>);
    return check_launch(who);
}

// The workspace that the backward's entry points have always asked for.  The
// single pass needs none; they go on refusing a call without it.
size_t bwd_ws_bytes(int64_t n_rows) { return 2 * align_up(sizeof(float) * static_cast<size_t>(n_rows), 256); }

int check_bwd_ws(int64_t n, const void* workspace, size_t workspace_bytes, const char* who) {
    if (!workspace || workspace_bytes < bwd_ws_bytes(n))
        return set_error(MESHY_ESPACE, "%s: workspace needs %zu bytes", who, bwd_ws_bytes(n));
    return MESHY_OK;
}

int launch_bwd(const uint16_t* logits, int64_t rows, int64_t T, int64_t V, int64_t stride_b,
               int64_t stride_t, const int64_t* ids, int n_ids, const float* lse, const float* grad_out,
               uint16_t* grad_logits, hipStream_t stream, const char* who) {
    const int64_t n = rows * T;
    BwdArgs a{};
    a.logits = logits;
    a.T = rows == 1 || stride_b == T * stride_t ? 0 : static_cast<uint32_t>(T);
    a.V = V, a.stride_b = stride_b, a.stride_t = stride_t;
    a.inv_v = 1.0 / static_cast<double>(V);
    a.ids = ids, a.lse = lse, a.grad_logp = grad_out;
    a.out = grad_logits;
    a.n_ids = n_ids;
    // The ids that a lane holds, in blocks of 64.
    auto by_ids = [&](auto go) {
        if (n_ids == 1) go(std::integral_constant<int, 0>());
        else if (n_ids <= kWave) go(std::integral_constant<int, 1>());
        else if (n_ids <= 2 * kWave) go(std::integral_constant<int, 2>());
        else go(std::integral_constant<int, kMaxIds / kWave>());
    };
    int rc;
    const bool contiguous = stride_t == V && a.T == 0;
    const bool aligned = reinterpret_cast<uintptr_t>(grad_logits) % 16 == 0;
    const bool flat = V >= kBwdShortV || (V >= kBwdShortV / 2 && n_ids == 1);
    const bool by_waves = V >= 2 && n * V >= 8 && (n_ids == 1 || (n_ids <= 16 && n > 8192));
    if (aligned && !flat && by_waves) {
        int R = 8;  // rows of a wave: about 1024 elements, if there are rows for 8 waves per CU
        while (R < kWave && R * V < 1024 && n >= 2 * R * 2048) R *= 2;
        const dim3 blocks(static_cast<unsigned>(ceil_div(n, R * (kBwdThreads / kWave))));
        const uint32_t inv = static_cast<uint32_t>((int64_t{1} << 32) / V + 1);
        auto go = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, blocks, dim3(kBwdThreads), 0, stream, a, static_cast<uint32_t>(n), R, inv);
        };
        if (n_ids == 1) {
            if (contiguous) go(k_lp_bwd_short<kBwdThreads, true, true>);
            else go(k_lp_bwd_short<kBwdThreads, true, false>);
        } else {
            if (contiguous) go(k_lp_bwd_short<kBwdThreads, false, true>);
            else go(k_lp_bwd_short<kBwdThreads, false, false>);
        }
        return check_launch(who);
    }
    if (aligned && flat) {
        const int64_t step = std::max<int64_t>(8, kBwdMaxElems / V / 8 * 8);
        for (int64_t r0 = 0; r0 < n; r0 += step) {
            a.row0 = r0;
            a.n_elems = std::min(step, n - r0) * V;
            a.n_chunks = static_cast<uint32_t>(ceil_div(a.n_elems, 8));
            const dim3 blocks(static_cast<unsigned>(ceil_div(a.n_chunks, kBwdThreads * kBwdUnroll)));
            by_ids([&](auto nb) {
                constexpr int NB = decltype(nb)::value;
                if (contiguous)
                    hipLaunchKernelGGL((k_lp_bwd_flat<kBwdThreads, kBwdUnroll, NB, true>), blocks, dim3(kBwdThreads),
                                       0, stream, a);
                else
                    hipLaunchKernelGGL((k_lp_bwd_flat<kBwdThreads, kBwdUnroll, NB, false>), blocks, dim3(kBwdThreads),
                                       0, stream, a);
            });
            if ((rc = check_launch(who))) return rc;
            a.ids += step * n_ids, a.lse += step, a.grad_logp += step * n_ids, a.out += step * V;
        }
    } else {
        const dim3 blocks(static_cast<unsigned>(n));
        by_ids([&](auto nb) {
            hipLaunchKernelGGL((k_lp_bwd_any<kBwdThreads, decltype(nb)::value>), blocks, dim3(kBwdThreads), 0, stream,
                               a);
        });
        return check_launch(who);
    }
    return MESHY_OK;
}

}  // namespace
}  // namespace meshy

namespace meshy {
namespace {

int entropy_fwd(const uint16_t* logits, int64_t rows, int64_t T, int64_t V, int64_t stride_b, int64_t stride_t,
                const int64_t* labels, float* logp, float* entropy, float* lse, int32_t max_polls,
                hipStream_t stream, const char* who) {
    clear_error();
    int rc = check_common(logits, rows, T, V, stride_b, stride_t, who);
    if (rc) return rc;
    if (max_polls < 0) return set_error(MESHY_EINVAL, "%s: negative max_polls", who);
    if (rows * T == 0) return MESHY_OK;
    if (logp && !labels) return set_error(MESHY_ENULL, "%s: logp needs labels", who);
    return launch_fwd(logits, rows, T, V, stride_b, stride_t, logp ? labels : nullptr, logp ? 1 : 0, logp,
                      entropy, lse, stream, who, std::min(max_polls, kSplitPolls));
}

int gather_fwd(const uint16_t* logits, int64_t rows, int64_t T, int64_t V, int64_t stride_b, int64_t stride_t,
               const int64_t* ids, int64_t n_ids, float* out, float* lse, int32_t max_polls, hipStream_t stream,
               const char* who) {
    clear_error();
    int rc = check_common(logits, rows, T, V, stride_b, stride_t, who);
    if (rc) return rc;
    if (n_ids < 1 || n_ids > kMaxIds)
        return set_error(MESHY_EINVAL, "%s: n_ids must be in [1, %d], got %lld", who, kMaxIds,
                         static_cast<long long>(n_ids));
    if (max_polls < 0) return set_error(MESHY_EINVAL, "%s: negative max_polls", who);
    if (rows * T == 0) return MESHY_OK;
    if (!ids || !out) return set_error(MESHY_ENULL, "%s: ids and out are required", who);
    return launch_fwd(logits, rows, T, V, stride_b, stride_t, ids, static_cast<int>(n_ids), out, nullptr, lse,
                      stream, who, std::min(max_polls, kSplitPolls));
}

}  // namespace
}  // namespace meshy

extern "C" int meshy_logprob_entropy_fwd(const uint16_t* logits, int64_t rows, int64_t T, int64_t V,
                                         int64_t stride_b, int64_t stride_t, const int64_t* labels,
                                         float* logp, float* entropy, float* lse,
                                         hipStream_t stream) {
    return meshy::entropy_fwd(logits, rows, T, V, stride_b, stride_t, labels, logp, entropy, lse,
                              meshy::kSplitPolls, stream, "meshy_logprob_entropy_fwd");
}

extern "C" int meshy_logprob_entropy_fwd_polls(const uint16_t* logits, int64_t rows, int64_t T, int64_t V,
                                               int64_t stride_b, int64_t stride_t, const int64_t* labels,
                                               float* logp, float* entropy, float* lse, int32_t max_polls,
                                               hipStream_t stream) {
    return meshy::entropy_fwd(logits, rows, T, V, stride_b, stride_t, labels, logp, entropy, lse, max_polls, stream,
                              "meshy_logprob_entropy_fwd_polls");
}

extern "C" int meshy_gather_logprobs_fwd(const uint16_t* logits, int64_t rows, int64_t T, int64_t V,
                                         int64_t stride_b, int64_t stride_t, const int64_t* ids,
                                         int64_t n_ids, float* out, float* lse, hipStream_t stream) {
    return meshy::gather_fwd(logits, rows, T, V, stride_b, stride_t, ids, n_ids, out, lse, meshy::kSplitPolls, stream,
                             "meshy_gather_logprobs_fwd");
}

extern "C" int meshy_gather_logprobs_fwd_polls(const uint16_t* logits, int64_t rows, int64_t T, int64_t V,
                                               int64_t stride_b, int64_t stride_t, const int64_t* ids,
                                               int64_t n_ids, float* out, float* lse, int32_t max_polls,
                                               hipStream_t stream) {
    return meshy::gather_fwd(logits, rows, T, V, stride_b, stride_t, ids, n_ids, out, lse, max_polls, stream,
                             "meshy_gather_logprobs_fwd_polls");
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
    if ((rc = check_bwd_ws(rows * T, workspace, workspace_bytes, who))) return rc;
    return launch_bwd(logits, rows, T, V, stride_b, stride_t, labels, 1, lse, grad_logp, grad_logits, stream, who);
}

// meshy_logprob_bwd without the workspace argument, for callers that cannot
// allocate; it keeps the row limit that it is declared with.
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
        return set_error(MESHY_ESPACE, "%s: %lld rows exceed the static scratch limit of %d rows", who,
                         static_cast<long long>(n), MESHY_NOALLOC_MAX_ROWS);
    return launch_bwd(logits, rows, T, V, stride_b, stride_t, labels, 1, lse, grad_logp, grad_logits, stream, who);
}

namespace meshy {
namespace {

int check_gather_bwd(const uint16_t* logits, int64_t rows, int64_t T, int64_t V, int64_t stride_b, int64_t stride_t,
                     const int64_t* ids, int64_t n_ids, const float* lse, const float* grad_out,
                     const uint16_t* grad_logits, const char* who) {
    int rc = check_common(logits, rows, T, V, stride_b, stride_t, who);
    if (rc) return rc;
    if (n_ids < 1 || n_ids > kMaxIds)
        return set_error(MESHY_EINVAL, "%s: n_ids must be in [1, %d], got %lld", who, kMaxIds,
                         static_cast<long long>(n_ids));
    if (rows * T > 0 && (!ids || !lse || !grad_out || !grad_logits))
        return set_error(MESHY_ENULL, "%s: ids, lse, grad_out and grad_logits are required", who);
    return MESHY_OK;
}

}  // namespace
}  // namespace meshy

extern "C" int meshy_gather_logprobs_bwd(const uint16_t* logits, int64_t rows, int64_t T, int64_t V,
                                         int64_t stride_b, int64_t stride_t, const int64_t* ids,
                                         int64_t n_ids, const float* lse, const float* grad_out,
                                         uint16_t* grad_logits, void* workspace, size_t workspace_bytes,
                                         hipStream_t stream) {
    using namespace meshy;
    clear_error();
    const char* who = "meshy_gather_logprobs_bwd";
    int rc = check_gather_bwd(logits, rows, T, V, stride_b, stride_t, ids, n_ids, lse, grad_out, grad_logits, who);
    if (rc || rows * T == 0) return rc;
    if ((rc = check_bwd_ws(rows * T, workspace, workspace_bytes, who))) return rc;
    return launch_bwd(logits, rows, T, V, stride_b, stride_t, ids, static_cast<int>(n_ids), lse, grad_out,
                      grad_logits, stream, who);
}

extern "C" int meshy_gather_logprobs_bwd_noalloc(const uint16_t* logits, int64_t rows, int64_t T, int64_t V,
                                                 int64_t stride_b, int64_t stride_t, const int64_t* ids,
                                                 int64_t n_ids, const float* lse, const float* grad_out,
                                                 uint16_t* grad_logits, hipStream_t stream) {
    using namespace meshy;
    clear_error();
    const char* who = "meshy_gather_logprobs_bwd_noalloc";
    const int rc =
        check_gather_bwd(logits, rows, T, V, stride_b, stride_t, ids, n_ids, lse, grad_out, grad_logits, who);
    if (rc || rows * T == 0) return rc;
    return launch_bwd(logits, rows, T, V, stride_b, stride_t, ids, static_cast<int>(n_ids), lse, grad_out,
                      grad_logits, stream, who);
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
