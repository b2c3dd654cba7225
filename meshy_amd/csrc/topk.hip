// Teacher Top-K of bf16 logits with their log-probabilities, for gfx950.
//
// Replaces teacher_topk (meshy/backend/titan/topk_loss.py:20-32): per row,
// the K largest logits (indices and values - logsumexp) of the fp32-upcast
// logits, sorted by value, in one streaming pass over the row instead of an
// fp32 copy, a topk and a logsumexp per chunk.
//
// One workgroup per row, streamed as the log-prob kernel streams it
// (rowstream.h), with the online log-sum-exp.  The list work is kept off the
// stream:
//   * the first tile sets a floor, the K-th largest of the workgroup's lane
//     maxima: K lanes hold an element that reaches it, so nothing below it can
//     be among the row's K best;
//   * from then on a 16-byte chunk whose maximum reaches the wave's threshold
//     is appended, as loaded, to the wave's buffer in LDS (a ballot, a prefix
//     count and one store), the others cost one compare;
//   * a buffer that would overflow keeps the K chunks with the largest maxima
//     (equal ones by column), and the K-th of them becomes the threshold that
//     later chunks of the wave must exceed;
//   * at the end the K-th largest maximum over all buffered chunks bounds the
//     elements that can be among the row's K best: these (K and a few) are
//     listed and each takes its rank by counting the listed elements before it.
// The K-th largest of a wave's values is found by building its 16-bit key from
// the top bits down, one ballot per value and candidate: no sort and no lane
// traffic.
//
// [4096, 151936]: 193 us at K = 8 and 209 at K = 64, where per-wave sorted
// lists with serial insertion took 199 and 527 (the read alone 176); [4096,
// 50257] 75 and 88 us, against 307 and 600 with 2-byte loads as well; [16,
// 151936] 16 and 19 us, against 28 and 137.  Rows of equal values: 1024 of
// 151936 take 62 us, against 5.4 ms.
//
// Order: torch.sort(descending=True, stable=True)'s, which torch.topk
// follows: NaN ranks above every number (+inf included), larger values before
// smaller, and equal values (NaNs among themselves, -0 and +0 alike) by
// smaller index.  16-bit integer keys carry it.  The stream compares floats,
// whose chunk maxima skip NaN: a wave that has met NaN or +inf (its running
// sum turns NaN) collects its chunks again by their keys.  Every wave operation
// runs with all 64 lanes active: loops are wave-uniform and absent elements
// are masked by a flag.
#include <algorithm>
#include <type_traits>

#include "rowstream.h"

namespace meshy {
namespace {

constexpr int kMaxTopK = kWave;
constexpr int64_t kTopkLongRow = 65536, kTopkManyRows = 2048;
// Chunks of a wave's buffer.  About 9 tiles of 1.1 K chunks (k <= kGroupK) or
// 1.4 K pass the floor on an unsorted row of 151936 logits, over 4 waves.
constexpr int kGroupK = 32;
constexpr int kBufSmallK = 192, kBufLargeK = 256;
// Elements listed at the end: with the exact bound, those of k + 32 chunks.
constexpr int kMaxReach = kMaxTopK + 32;
constexpr int kMaxListed = 8 * kMaxReach;

// 16-bit keys in rank order: NaN first, then by value, -0 as +0; every bf16
// value's key is above kAbsentKey.
constexpr uint32_t kAbsentKey = 0, kNanKey = 0xffff, kMinusInfKey = 0x007f;

__device__ __forceinline__ uint32_t key_of(uint32_t h) {
    if ((h & 0x7fff) > 0x7f80) return kNanKey;
    if (h == 0x8000) h = 0;
    return (h & 0x8000) ? ~h & 0xffff : h | 0x8000;
}

__device__ __forceinline__ float value_of(uint32_t key) {
    return __uint_as_float(((key & 0x8000) ? key & 0x7fff : ~key & 0xffff) << 16);
}

// The smallest float a chunk maximum must reach for its key to reach `key`
// (NaN, which no number reaches, above +inf).
__device__ __forceinline__ float threshold_of(uint32_t key) {
    return key <= kMinusInfKey ? -__builtin_inff() : value_of(key);
}

__device__ __forceinline__ uint32_t half_of(const v4u& v, int j) {
    const uint32_t w = j < 2 ? v.x : j < 4 ? v.y : j < 6 ? v.z : v.w;
    return (j & 1) ? w >> 16 : w & 0xffff;
}

typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

// The largest key of the chunk's elements.
__device__ __forceinline__ uint32_t chunk_key(const v4u& v) {
    auto magnitude = [](uint32_t w) { return __builtin_bit_cast(u16x2, w & 0x7fff7fffu); };
    const u16x2 most = __builtin_elementwise_max(__builtin_elementwise_max(magnitude(v.x), magnitude(v.y)),
                                                 __builtin_elementwise_max(magnitude(v.z), magnitude(v.w)));
    float z[8];
    const v4u one[1] = {v};
    unpack(one, z);
    return max(most.x, most.y) > 0x7f80 ? kNanKey : key_of(__float_as_uint(tile_max(z)) >> 16);
}

// The k-th largest of the wave's keys (R per lane), kAbsentKey if there are
// fewer; the same in every lane.  Two bits a step: the three candidates' ballots
// are independent, and a step's latency is that of its chain to the next.
template <int R>
__device__ __forceinline__ uint32_t kth_key(const uint32_t (&key)[R], int k) {
    uint32_t t = 0;
#pragma unroll
    for (int bit = 14; bit >= 0; bit -= 2) {
        int n[3] = {0, 0, 0};
#pragma unroll
        for (int i = 0; i < R; ++i) {
#pragma unroll
            for (int q = 0; q < 3; ++q) n[q] += __popcll(__ballot(key[i] >= (t | ((q + 1u) << bit))));
        }
        t |= static_cast<uint32_t>((n[0] >= k) + (n[1] >= k) + (n[2] >= k)) << bit;
    }
    return t;
}

// Lanes below this one among the set bits of a ballot.
__device__ __forceinline__ int rank_in(uint64_t ballot) {
    return __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(ballot >> 32),
                                     __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(ballot), 0));
}

// A wave's buffer, in column order: cnt chunks as loaded with their first
// columns.  A chunk enters when its key reaches `key` (its maximum reaches tv).
template <int CAP>
struct WaveBuf {
    v4u* data;
    int32_t* col;
    int cnt;
    uint32_t key;
    float tv;
};

template <int CAP>
__device__ __forceinline__ void set_threshold(WaveBuf<CAP>& w, uint32_t key) {
    w.key = key;
    w.tv = threshold_of(key);
}

// The keys of the buffer's entries, entry lane + 64 j in key[j].
template <int CAP>
__device__ __forceinline__ void entry_keys(const WaveBuf<CAP>& w, uint32_t (&key)[CAP / kWave]) {
#pragma unroll
    for (int j = 0; j < CAP / kWave; ++j) {
        const int i = threadIdx.x % kWave + j * kWave;
        key[j] = kAbsentKey;
        if (j * kWave < w.cnt) key[j] = i < w.cnt ? chunk_key(w.data[i]) : kAbsentKey;
    }
}

// Keeps the k chunks with the largest keys, equal ones by column; later
// chunks must exceed the k-th: an element equal to it would rank after one
// element of each chunk kept.  cnt >= k.
template <int CAP>
__device__ __forceinline__ void compact(WaveBuf<CAP>& w, int k) {
    constexpr int R = CAP / kWave;
    const int lane = threadIdx.x % kWave;
    uint32_t key[R];
    entry_keys(w, key);
    const uint32_t t = kth_key(key, k);
    int above = 0;
#pragma unroll
    for (int j = 0; j < R; ++j) above += __popcll(__ballot(key[j] > t));
    int ties_left = k - above, n = 0;
#pragma unroll
    for (int j = 0; j < R; ++j) {
        // Entries move to places before their own: block j is read before any
        // of it is written over.
        const int i = lane + j * kWave;
        const v4u d = w.data[i];
        const int32_t col = w.col[i];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        const bool is_tie = key[j] == t && i < w.cnt;
        const uint64_t tie = __ballot(is_tie);
        const bool keep = key[j] > t || (is_tie && rank_in(tie) < ties_left);
        const uint64_t kept = __ballot(keep);
        if (keep) {
            w.data[n + rank_in(kept)] = d;
            w.col[n + rank_in(kept)] = col;
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        ties_left -= min(ties_left, static_cast<int>(__popcll(tie)));
        n += __popcll(kept);
    }
    w.cnt = n;
    set_threshold(w, t + 1);
}

// Appends the chunk of each lane with hit set (their ballot is b); the buffer
// has room.
template <int CAP>
__device__ __forceinline__ void append(WaveBuf<CAP>& w, const v4u& v, int32_t col, bool hit, uint64_t b) {
    if (hit) {
        const int at = w.cnt + rank_in(b);
        w.data[at] = v;
        w.col[at] = col;
    }
    w.cnt += __popcll(b);
}

// Appends the chunks of the wave from c (of lane 0) on, every `step` chunks
// below `end`, that reach the threshold by their keys, compacting the buffer
// when it is full.  Taken for a tile with more hits than there is room for, and
// for rows that hold NaN or +inf.
template <int CAP>
__device__ __forceinline__ void collect(WaveBuf<CAP>& w, const RowSpan& sp, int64_t c, int64_t end, int step,
                                        int k) {
    const int lane = threadIdx.x % kWave;
#pragma unroll 1
    for (; c < end; c += step) {
        const bool ok = c + lane < end;
        const v4u v = sp.body[ok ? c + lane : 0];
        const int32_t col = sp.head + static_cast<int32_t>(8 * (c + lane));
        const uint32_t key = ok ? chunk_key(v) : kAbsentKey;
        bool hit = ok && key >= w.key;
        uint64_t b = __ballot(hit);
        if (w.cnt + __popcll(b) > CAP) {
            compact(w, k);
            hit = ok && key >= w.key;
            b = __ballot(hit);
        }
        append(w, v, col, hit, b);
    }
}

// Makes the compiler take the chunks as new values here: what was unpacked
// from them before is unpacked again rather than kept in registers (135
// VGPRs, 3 waves per SIMD, without).
template <int G>
__device__ __forceinline__ void forget(v4u (&v)[G]) {
#pragma unroll
    for (int g = 0; g < G; ++g) asm("" : "+v"(v[g].x), "+v"(v[g].y), "+v"(v[g].z), "+v"(v[g].w));
}

// The maximum of each of the thread's chunks and sum exp(z - m) over those with
// ok set.
template <int G, class OkF>
__device__ __forceinline__ float maxima_and_sum(const v4u (&v)[G], float m, OkF ok, float (&cm)[G]) {
    const float nm = ref(m);
    float s0 = 0.f, s1 = 0.f;
#pragma unroll
    for (int g = 0; g < G; ++g) {
        float z[8];
        const v4u one[1] = {v[g]};
        unpack(one, z);
        cm[g] = tile_max(z);
        float c0 = 0.f, c1 = 0.f;
#pragma unroll
        for (int j = 0; j < 8; j += 2) {
            c0 += fast_exp2(fmaf(z[j], kLog2e, nm));
            c1 += fast_exp2(fmaf(z[j + 1], kLog2e, nm));
        }
        s0 += ok(g) ? c0 : 0.f;
        s1 += ok(g) ? c1 : 0.f;
    }
    return s0 + s1;
}

template <int G, class OkF>
__device__ __forceinline__ float max_of(const v4u (&v)[G], OkF ok) {
    float tm = -__builtin_inff();
#pragma unroll
    for (int g = 0; g < G; ++g) {
        float z[8];
        const v4u one[1] = {v[g]};
        unpack(one, z);
        tm = ok(g) ? fmaxf(tm, tile_max(z)) : tm;
    }
    return tm;
}

// The floor for the row: the k-th largest of the maxima of 64 groups of lanes
// (of 128 for k > kGroupK), lane l of every wave (of every second wave) one
// group.  k groups hold an element that reaches it.
template <int NT, int CAP>
__device__ __forceinline__ void set_floor(WaveBuf<CAP>& w, float lane_max, bool present, int k) {
    constexpr int kRows = NT / kWave;
    static_assert(kRows % 4 == 0, "four keys per 8-byte read");
    __shared__ __align__(8) uint16_t s_max[kWave][kRows];
    const int lane = threadIdx.x % kWave;
    s_max[lane][threadIdx.x / kWave] =
        present ? static_cast<uint16_t>(key_of(__float_as_uint(lane_max) >> 16)) : kAbsentKey;
    __syncthreads();
    uint32_t even = 0, odd = 0;
#pragma unroll
    for (int i = 0; i < kRows; i += 4) {
        const uint2 q = *reinterpret_cast<const uint2*>(&s_max[lane][i]);
        even = max(even, max(q.x & 0xffff, q.y & 0xffff));
        odd = max(odd, max(q.x >> 16, q.y >> 16));
    }
    if (k <= kGroupK) {
        const uint32_t key[1] = {max(even, odd)};
        set_threshold(w, kth_key(key, k));
    } else {
        const uint32_t key[2] = {even, odd};
        set_threshold(w, kth_key(key, k));
    }
}

// Of a tile, against a reference that stays: an element 14 above it has its
// exponent rounded at the size of 20, 1e-6 of the sum.
constexpr float kMaxSum = 0x1p20f;

// One tile of G chunks per thread, those with ok set; the thread's first
// starts at column col and the others NT chunks apart.  Its part of the
// log-sum-exp, the row's floor if it is the first, and the chunks that reach
// the threshold.  The sum is taken against the wave's maximum of the first tile
// as it stands (rowstream.h, accumulate_at); where an element lies 14 above it,
// the lane's reference is raised first.
// Returns false, with no chunk appended, when the buffer has no room for them
// all; collect() then takes the tile.
template <int NT, int CAP, int G, class OkF>
__device__ __forceinline__ bool topk_tile(v4u (&v)[G], OkF ok, int32_t col, bool first, int k, WaveBuf<CAP>& w,
                                          float& m, float& s) {
    float t = 0.f;
    if (first) {
        const float tm = max_of(v, ok);
        raise_max(m, s, t, wave_max(tm));
        set_floor<NT>(w, tm, ok(0), k);
        forget(v);
    }
    float cm[G];
    float st = maxima_and_sum(v, m, ok, cm);
    if (!(st <= kMaxSum)) {
        forget(v);
        raise_max(m, s, t, max_of(v, ok));
        forget(v);
        st = maxima_and_sum(v, m, ok, cm);
    }
    s += st;
    int hits = 0;
#pragma unroll
    for (int g = 0; g < G; ++g) hits += __popcll(__ballot(ok(g) && cm[g] >= w.tv));
    if (w.cnt + hits > CAP) return false;
#pragma unroll
    for (int g = 0; g < G; ++g) {
        const bool hit = ok(g) && cm[g] >= w.tv;
        const uint64_t b = __ballot(hit);
        if (b) append(w, v[g], col + 8 * g * NT, hit, b);
    }
    return true;
}

// Bound by the read of the logits; NT threads per row as in the log-prob
// forward.
template <int NT, int U, int CAP>
__global__ __launch_bounds__(NT) void k_topk_vec(const uint16_t* __restrict__ logits, int64_t T, int64_t V,
                                                 int64_t stride_b, int64_t stride_t, int k,
                                                 int64_t* __restrict__ ids, float* __restrict__ lps,
                                                 float* __restrict__ lse_out) {
    constexpr int kWaves = NT / kWave;
    constexpr int kKeyRows = kWaves + 2;
    __shared__ v4u s_data[kWaves][CAP];
    __shared__ int32_t s_col[kWaves][CAP];
    __shared__ uint16_t s_key[kKeyRows][kWave];  // the waves' chunks, then the row's head and tail elements
    __shared__ uint64_t s_list[kMaxListed];
    __shared__ int s_listed;
    __shared__ Lse s_lse;
    const int64_t r = blockIdx.x;
    const uint16_t* row = row_ptr(logits, r, T, stride_b, stride_t);
    const RowSpan sp = row_span(row, V);
    const int tid = threadIdx.x;
    const int lane = tid % kWave;
    const int wid = __builtin_amdgcn_readfirstlane(tid / kWave);
    if (tid == 0) s_listed = 0;

    // One element of the row's head (wave 0) or tail (wave 1) per thread.
    bool edge;
    const int64_t edge_col = edge_element(sp, V, tid, edge);
    const uint32_t edge_h = edge ? row[edge_col] : 0u;

    float m = kInit, s = 0.f, t = 0.f;
    WaveBuf<CAP> w{s_data[wid], s_col[wid], 0, kAbsentKey, -__builtin_inff()};
    constexpr int64_t kTile = static_cast<int64_t>(NT) * U;
    const int64_t n_full = sp.n8 / kTile;
    for (int64_t it = 0; it < n_full; ++it) {
        const int64_t c0 = it * kTile + tid;
        v4u v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = __builtin_nontemporal_load(sp.body + c0 + u * NT);
        if (!topk_tile<NT>(v, [](int) { return true; }, sp.head + static_cast<int32_t>(8 * c0), it == 0, k, w, m, s))
            collect(w, sp, it * kTile + wid * kWave, (it + 1) * kTile, NT, k);
    }
    // The chunks left, U / 2 per thread at a time (one copy of the tile's code,
    // not one for each number of chunks: the kernel stays in the instruction
    // cache).
    for (int64_t c0 = n_full * kTile; c0 < sp.n8; c0 += kTile / 2) {
        v4u v[U / 2];
        bool ok[U / 2];
        load_tail<NT, U / 2>(sp.body + c0, sp.n8 - c0, tid, v, ok);
        if (!topk_tile<NT>(v, [&](int g) { return ok[g]; }, sp.head + static_cast<int32_t>(8 * (c0 + tid)),
                                  c0 == 0, k, w, m, s))
            collect(w, sp, c0 + wid * kWave, min(c0 + kTile / 2, sp.n8), NT, k);
    }
    // A lane's running sum is NaN once it has met NaN or +inf: such a wave
    // collects its chunks again, by key (rows of ordinary logits never do).
    if (__ballot(isnan(s))) {
        w.cnt = 0;
        set_threshold(w, kAbsentKey);
        collect(w, sp, wid * kWave, sp.n8, NT, k);
    }
    accumulate_one(bf16_to_f32(static_cast<uint16_t>(edge_h)), edge, m, s, t);

    // Each lane's best entry, and the edges.  A wave's entries fill its lanes
    // from 0 on: its row of keys starts at a lane of its own, so that maxima
    // over the rows are over groups of entries.
    constexpr int kShift = kWave / kWaves;
    constexpr int R = CAP / kWave;
    uint32_t mine[R];
    entry_keys(w, mine);
    uint32_t best = mine[0];
#pragma unroll
    for (int j = 1; j < R; ++j) best = max(best, mine[j]);
    const uint32_t edge_key = edge ? key_of(edge_h) : kAbsentKey;
    s_key[wid][(lane + wid * kShift) % kWave] = static_cast<uint16_t>(best);
    if (wid < 2) s_key[kWaves + wid][lane] = static_cast<uint16_t>(edge_key);
    block_merge<NT, false>(m, s, t);  // its barrier publishes the keys

    // A bound that k groups reach: k elements of the row do, and the elements
    // that do not are not among its k best.
    uint32_t even = kAbsentKey, odd = kAbsentKey;
#pragma unroll
    for (int i = 0; i < kKeyRows; ++i) {
        const uint32_t key = s_key[i][lane];
        if (i & 1) odd = max(odd, key);
        else even = max(even, key);
    }
    const bool nan = max(even, odd) == kNanKey;
    uint32_t bound;
    if (k <= kGroupK) {
        const uint32_t key[1] = {max(even, odd)};
        bound = kth_key(key, k);
    } else {
        const uint32_t key[2] = {even, odd};
        bound = kth_key(key, k);
    }
    bound = max(bound, kAbsentKey + 1);

    // Lists the elements of entry i that reach the bound, as far as there is room.
    auto listed_at = [&](uint32_t ekey, int32_t col) {
        return (static_cast<uint64_t>(ekey) << 32) | static_cast<uint32_t>(~col);
    };
    auto list_entry = [&](int i) {
        const v4u d = w.data[i];
        const int32_t col = w.col[i];
        uint32_t ek[8];
        int n = 0;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            ek[j] = key_of(half_of(d, j));
            n += ek[j] >= bound;
        }
        int at = atomicAdd(&s_listed, n);
        if (at + n > kMaxListed) return;
#pragma unroll
        for (int j = 0; j < 8; ++j)
            if (ek[j] >= bound) s_list[at++] = listed_at(ek[j], col + j);
    };
    auto list_edge = [&] {
        const int at = atomicAdd(&s_listed, 1);
        if (at < kMaxListed) s_list[at] = listed_at(edge_key, static_cast<int32_t>(edge_col));
    };
#pragma unroll 1
    for (int j = 0; j * kWave < w.cnt; ++j) {
        uint32_t key = mine[0];
#pragma unroll
        for (int q = 1; q < R; ++q) key = j == q ? mine[q] : key;
        if (key >= bound) list_entry(lane + j * kWave);
    }
    if (edge_key >= bound) list_edge();
    if (tid < kWave) {
        // torch.logsumexp: NaN for a row holding NaN; otherwise +inf for a row
        // whose max is +inf (its candidates' log-probs are then NaN for the
        // +inf logit and -inf for finite ones), where s is NaN.
        const Lse lse = __ballot(nan) ? Lse{__builtin_nanf(""), 0.f}
                        : m == __builtin_inff() ? Lse{m, 0.f}
                                                : lse_of(m, ln_of(s));
        if (tid == 0) {
            s_lse = lse;
            if (lse_out) lse_out[r] = lse.hi + lse.lo;
        }
    }
    __syncthreads();
    if (s_listed > kMaxListed) {
        // Too many elements reach that bound (many equal logits): each wave
        // keeps its k best chunks, the bound is the k-th largest of all
        // entries' keys, and of more entries tied at it only the first can hold
        // one of the k best; the last of those starts at column last_tie.
        __syncthreads();
        if (tid == 0) s_listed = 0;
        if (w.cnt > kWave) compact(w, k);
        const uint32_t my_key = lane < w.cnt ? chunk_key(w.data[lane]) : kAbsentKey;
        s_key[wid][lane] = static_cast<uint16_t>(my_key);
        __syncthreads();
        uint32_t key[kKeyRows];
#pragma unroll
        for (int i = 0; i < kKeyRows; ++i) key[i] = s_key[i][lane];
        auto count = [&](uint32_t from) {
            int n = 0;
#pragma unroll
            for (int i = 0; i < kKeyRows; ++i) n += __popcll(__ballot(key[i] >= from));
            return n;
        };
        bound = max(kth_key(key, k), kAbsentKey + 1);
        int32_t last_tie = INT32_MAX;
        if (count(bound) > kMaxReach) {
            const int ties = k - count(bound + 1);
            int32_t col[kKeyRows];
#pragma unroll
            for (int i = 0; i < kWaves; ++i) col[i] = s_col[i][lane];
            col[kWaves] = lane;
            col[kWaves + 1] = static_cast<int32_t>(V) - sp.tail + lane;
            last_tie = 0;
#pragma unroll 1
            for (int bit = 30; bit >= 0; --bit) {
                const int32_t cand = last_tie | (1 << bit);
                int n = 0;
#pragma unroll
                for (int i = 0; i < kKeyRows; ++i) n += __popcll(__ballot(key[i] == bound && col[i] < cand));
                if (n < ties) last_tie = cand;
            }
        }
        if (my_key > bound || (my_key == bound && w.col[lane] <= last_tie)) list_entry(lane);
        if (edge_key > bound || (edge_key == bound && edge_col <= last_tie)) list_edge();
        __syncthreads();
    }
    const int listed = s_listed;
    const Lse lse = s_lse;
    for (int i = tid; i < listed; i += NT) {
        const uint64_t own = s_list[i];
        int rank = 0;
#pragma unroll 8
        for (int j = 0; j < listed; ++j) rank += s_list[j] > own;
        if (rank < k) {
            ids[r * k + rank] = static_cast<int32_t>(~static_cast<uint32_t>(own));
            lps[r * k + rank] = minus_lse(value_of(static_cast<uint32_t>(own >> 32)), lse);
        }
    }
}

}  // namespace
}  // namespace meshy

extern "C" int meshy_topk_logprobs(const uint16_t* logits, int64_t rows, int64_t T, int64_t V, int64_t stride_b,
                                   int64_t stride_t, int64_t k, int64_t* ids, float* logprobs, float* lse,
                                   hipStream_t stream) {
    using namespace meshy;
    clear_error();
    const char* who = "meshy_topk_logprobs";
    if (rows < 0 || T < 0 || V <= 0 || stride_b < 0 || stride_t < 0)
        return set_error(MESHY_EINVAL, "%s: bad shape rows=%lld T=%lld V=%lld", who, static_cast<long long>(rows),
                         static_cast<long long>(T), static_cast<long long>(V));
    if (V > INT32_MAX) return set_error(MESHY_EINVAL, "%s: V must fit in int32", who);
    if (k < 1 || k > kMaxTopK || k > V)
        return set_error(MESHY_EINVAL, "%s: k must be in [1, min(%d, V)], got %lld", who, kMaxTopK,
                         static_cast<long long>(k));
    if (T > 0 && rows > INT32_MAX / T) return set_error(MESHY_EINVAL, "%s: too many rows", who);
    const int64_t n = rows * T;
    if (n == 0) return MESHY_OK;  // an empty call: NULL arrays are accepted
    if (!logits || !ids || !logprobs) return set_error(MESHY_ENULL, "%s: logits, ids and logprobs are required", who);
    const dim3 grid(static_cast<unsigned>(n));
    auto go = [&](auto kernel, int threads) {
        hipLaunchKernelGGL(kernel, grid, dim3(threads), 0, stream, logits, T, V, stride_b, stride_t,
                           static_cast<int>(k), ids, logprobs, lse);
    };
    // 16-byte loads in flight per thread: 8 for many long rows (4096 rows of
    // 151936, K = 8: 188 us against 194 with 4; of 100000: 128 against 131), else
    // 4, with 8 waves per SIMD, where the work around a row weighs more (1024
    // rows of 151936: 55.1 us against 56.2; 4096 of 50257: 71 against 76; of
    // 20000: 38 against 45).  512 threads up to 256 rows, as in the log-prob
    // forward (37 rows of 151936: 20.4 us against 22.2 with 256).
    auto by_unroll = [&](auto cap) {
        constexpr int CAP = decltype(cap)::value;
        const bool long_rows = V > kTopkLongRow;
        if (n <= 256 && long_rows) go(k_topk_vec<512, 8, CAP>, 512);
        else if (n <= 256) go(k_topk_vec<512, 4, CAP>, 512);
        else if (n >= kTopkManyRows && long_rows) go(k_topk_vec<256, 8, CAP>, 256);
        else go(k_topk_vec<256, 4, CAP>, 256);
    };
    if (k <= kGroupK) by_unroll(std::integral_constant<int, kBufSmallK>());
    else by_unroll(std::integral_constant<int, kBufLargeK>());
    return check_launch(who);
}
