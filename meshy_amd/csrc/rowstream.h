// Building blocks of the kernels that stream one row of bf16 logits per
// workgroup: 16-byte register tiles, the online log-sum-exp state and its
// merges, and the block-wide merge for 64-wide wavefronts.
//
// The online state of a row is a triple over the elements seen so far:
//     m = running max of z,
//     s = sum exp(z - m),
//     t = sum exp(z - m) * (z - m) * log2(e)   (only for the entropy)
// updated once per register tile: the tile max first, then one exp2 per
// element.  lse = m + ln s and H = ln 2 * (log2 s - t / s).
// The exponent of an element is one fma, z log2(e) + ref(m), whose ref(m) is
// -m log2(e) rounded: every term of s is off by the same 2^(m log2(e) + ref(m)),
// which moves from one reference to the next by the difference of the two ref's
// and is taken out at the end (ref_error).
#pragma once

#include <hip/hip_bf16.h>

#include "common.h"

namespace meshy {

// Native 4 x u32 vector: what the nontemporal load/store builtins accept.
typedef unsigned int v4u __attribute__((ext_vector_type(4)));

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.69314718055994531f;
constexpr float kInit = -1e30f;  // finite "minus infinity": keeps 0 * d finite
constexpr int64_t kIgnoreIndex = -100;

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// (Its product must not be fused with what it is added to: the same ref(m) has
// to come out everywhere.)
__device__ __forceinline__ float ref(float m) {
#pragma clang fp contract(off)
    return -m * kLog2e;
}

// log2 of the factor that every term of s carries.
__device__ __forceinline__ float ref_error(float m) { return fmaf(m, kLog2e, ref(m)); }

__device__ __forceinline__ float row16_max(float v) {
    v = fmaxf(v, dpp_f32<kDppRowRor8>(v));
    v = fmaxf(v, dpp_f32<kDppRowRor4>(v));
    v = fmaxf(v, dpp_f32<kDppRowRor2>(v));
    return fmaxf(v, dpp_f32<kDppRowRor1>(v));
}

__device__ __forceinline__ float wave_max(float v) {
    v = row16_max(v);
    return fmaxf(fmaxf(lane_f32(v, 0), lane_f32(v, 16)), fmaxf(lane_f32(v, 32), lane_f32(v, 48)));
}

// Moves the running max to at least `tm`, rescaling s and t.
__device__ __forceinline__ void raise_max(float& m, float& s, float& t, float tm) {
    const float mn = fmaxf(m, tm);
    const float d = ref(mn) - ref(m);
    const float a = fast_exp2(d);
    t = a * fmaf(d, s, t);
    s = a * s;
    m = mn;
}

template <int N>
__device__ __forceinline__ void unpack(const v4u (&v)[N], float (&z)[N * 8]) {
#pragma unroll
    for (int u = 0; u < N; ++u) {
        z[8 * u + 0] = bf16_lo(v[u].x);
        z[8 * u + 1] = bf16_hi(v[u].x);
        z[8 * u + 2] = bf16_lo(v[u].y);
        z[8 * u + 3] = bf16_hi(v[u].y);
        z[8 * u + 4] = bf16_lo(v[u].z);
        z[8 * u + 5] = bf16_hi(v[u].z);
        z[8 * u + 6] = bf16_lo(v[u].w);
        z[8 * u + 7] = bf16_hi(v[u].w);
    }
}

template <int K>
__device__ __forceinline__ float tile_max(const float (&z)[K]) {
    float tm = z[0];
#pragma unroll
    for (int i = 1; i < K; ++i) tm = fmaxf(tm, z[i]);
    return tm;
}

// Accumulates a full register tile (every element valid) whose max is tm.
// kEntropy = false leaves t untouched (log-sum-exp only).
template <bool kEntropy, int K>
__device__ __forceinline__ void accumulate(const float (&z)[K], float tm, float& m, float& s, float& t) {
    raise_max(m, s, t, tm);
    const float nm = ref(m);
    float s0 = 0.f, s1 = 0.f, t0 = 0.f, t1 = 0.f;
#pragma unroll
    for (int i = 0; i < K; i += 2) {
        const float x0 = fmaf(z[i], kLog2e, nm);
        const float x1 = fmaf(z[i + 1], kLog2e, nm);
        const float e0 = fast_exp2(x0);
        const float e1 = fast_exp2(x1);
        s0 += e0;
        s1 += e1;
        if (kEntropy) {
            t0 = fmaf(e0, x0, t0);
            t1 = fmaf(e1, x1, t1);
        }
    }
    s += s0 + s1;
    if (kEntropy) t += t0 + t1;
}

template <bool kEntropy = true, int K>
__device__ __forceinline__ void accumulate(const float (&z)[K], float& m, float& s, float& t) {
    accumulate<kEntropy>(z, tile_max(z), m, s, t);
}

// A lane's first tile: its reference is the wave's maximum, which later tiles
// rarely exceed by much.
template <bool kEntropy, int K>
__device__ __forceinline__ void accumulate_first(const float (&z)[K], float& m, float& s, float& t) {
    accumulate<kEntropy>(z, wave_max(tile_max(z)), m, s, t);
}

// Accumulates a full tile against the running reference m as it stands, without
// a tile max.  Any reference gives the same lse and entropy (s and t are both
// relative to m), but the exponent of an element d above it, and t, are rounded
// at the size of d log2(e): this is taken only when the tile's sum is at most
// 2^12, i.e. no element exceeds m by more than 12 / log2(e) = 8.3.  Otherwise
// (and for NaN or infinite inputs) it returns false with (s, t) untouched, and
// the caller accumulates the tile with its max.  (With 2^64, a logit of 16 to 40
// among N(0, 1/4) left errors of 4e-6 in its log-prob and 1.3e-5 in the entropy;
// now below 7e-7.)  Saves the tile max and the rescale of every tile after a
// lane's first.
constexpr float kMaxTileSum = 0x1p12f;

template <bool kEntropy, int U>
__device__ __forceinline__ bool accumulate_at(const v4u (&v)[U], float m, float& s, float& t) {
    const float nm = ref(m);
    float s0 = 0.f, s1 = 0.f, t0 = 0.f, t1 = 0.f;
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const uint32_t w[4] = {v[u].x, v[u].y, v[u].z, v[u].w};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const float x0 = fmaf(bf16_lo(w[k]), kLog2e, nm);
            const float x1 = fmaf(bf16_hi(w[k]), kLog2e, nm);
            const float e0 = fast_exp2(x0);
            const float e1 = fast_exp2(x1);
            s0 += e0;
            s1 += e1;
            if (kEntropy) {
                t0 = fmaf(e0, x0, t0);
                t1 = fmaf(e1, x1, t1);
            }
        }
    }
    // Both sums are formed before the test and kept or dropped by a select:
    // a branch around the t update would keep every exp of the tile live.
    const float st = s0 + s1;
    const bool ok = st <= kMaxTileSum;
    s = ok ? s + st : s;
    if (kEntropy) t = ok ? t + (t0 + t1) : t;
    return ok;
}

// Accumulates a tile in which only the 8-element groups with ok[g] hold
// data; the others are ignored whatever their contents.
template <bool kEntropy, int G>
__device__ __forceinline__ void accumulate_masked(float (&z)[G * 8], const bool (&ok)[G], float& m, float& s,
                                                  float& t) {
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
        for (int k = 0; k < 8; ++k) z[8 * g + k] = ok[g] ? z[8 * g + k] : kInit;
    raise_max(m, s, t, tile_max(z));
    const float nm = ref(m);
    float s0 = 0.f, t0 = 0.f;
#pragma unroll
    for (int g = 0; g < G; ++g) {
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const float x = fmaf(z[8 * g + k], kLog2e, nm);
            const float e = ok[g] ? fast_exp2(x) : 0.f;
            s0 += e;
            if (kEntropy) t0 = fmaf(e, x, t0);
        }
    }
    s += s0;
    if (kEntropy) t += t0;
}

// Loads the last rem (<= NT * G) 16-byte chunks of a row, starting at base,
// G per thread, all issued before any is used: thread tid's chunk g is
// tid + g * NT; past rem it reads chunk 0 instead and its ok flag is false.
template <int NT, int G>
__device__ __forceinline__ void load_tail(const v4u* base, int64_t rem, int tid, v4u (&v)[G], bool (&ok)[G]) {
#pragma unroll
    for (int g = 0; g < G; ++g) {
        const int64_t c = tid + static_cast<int64_t>(g) * NT;
        ok[g] = c < rem;
        v[g] = __builtin_nontemporal_load(base + (ok[g] ? c : 0));
    }
}

// Accumulates one element that may be absent.
__device__ __forceinline__ void accumulate_one(float z, bool ok, float& m, float& s, float& t) {
    if (!ok) return;
    raise_max(m, s, t, z);
    const float x = fmaf(z, kLog2e, ref(m));
    const float e = fast_exp2(x);
    s += e;
    t = fmaf(e, x, t);
}

// Moves the triple to the reference point top (>= m); kEntropy = false leaves
// t untouched.
template <bool kEntropy>
__device__ __forceinline__ void rebase(float& m, float& s, float& t, float top) {
    const float d = ref(top) - ref(m);
    const float a = fast_exp2(d);
    if (kEntropy) t = a * fmaf(d, s, t);
    s = a * s;
    m = top;
}

// The merge over each 16-lane row, valid in every lane of the row.
template <bool kEntropy>
__device__ __forceinline__ void merge_rows16(float& m, float& s, float& t) {
    rebase<kEntropy>(m, s, t, row16_max(m));
    s = row16_sum(s);
    if (kEntropy) t = row16_sum(t);
}

// Block-wide merge of the per-lane triples; the result lands in wave 0.  The
// maximum first, then every triple is moved to it and the sums add up, all
// through DPP rotations: one exponential per wave.  (A tree of pairwise merges,
// two exponentials each, is bound by the SIMDs' arithmetic for short rows:
// 131072 rows of 64 logits took 262 us with one.)
template <int NT, bool kEntropy = true>
__device__ __forceinline__ void block_merge(float& m, float& s, float& t) {
    rebase<kEntropy>(m, s, t, wave_max(m));
    s = wave_sum(s);
    if (kEntropy) t = wave_sum(t);
    if constexpr (NT > kWave) {
        constexpr int kWaves = NT / kWave;
        static_assert(kWaves <= 16, "the waves' triples are merged in one row of 16 lanes");
        __shared__ float sm[kWaves], ss[kWaves], st[kWaves];
        const int lane = threadIdx.x % kWave;
        const int wid = threadIdx.x / kWave;
        if (lane == 0) {
            sm[wid] = m;
            ss[wid] = s;
            if (kEntropy) st[wid] = t;
        }
        __syncthreads();
        if (wid == 0) {
            const bool in = lane < kWaves;
            m = in ? sm[lane] : kInit;
            s = in ? ss[lane] : 0.f;
            t = kEntropy && in ? st[lane] : 0.f;
            merge_rows16<kEntropy>(m, s, t);
        }
    }
}

// m + ln s as hi + lo in fp32, |lo| < 1, good to a few 2^-24: s = f 2^e with f in
// [1, 2), so that a sum of 1 (one logit has all the weight) gives m itself, and
// e ln 2 is split so that its high part is exact.  Rounded to one fp32, the
// log-sum-exp of a row of 150 thousand logits lies 3e-7 off, as much as
// everything else together.
struct Lse {
    float hi, lo;
};

constexpr float kLn2High = 2839.f / 4096.f;
constexpr float kLn2Low = static_cast<float>(0.6931471805599453 - 2839.0 / 4096.0);

// a + b = sum + err exactly, as long as sum is finite.
__device__ __forceinline__ float add_with_error(float a, float b, float& err) {
    const float sum = a + b;
    const float bb = sum - a;
    err = (a - (sum - bb)) + (b - bb);
    return sum;
}

// ln s as high + low, the high part exact.
__device__ __forceinline__ Lse ln_of(float s) {
    int e;
    const float f = 2.f * frexpf(s, &e);
    const float ef = static_cast<float>(e - 1);
    return Lse{ef * kLn2High, fmaf(__log2f(f), kLn2, ef * kLn2Low)};
}

__device__ __forceinline__ Lse lse_of(float m, const Lse& ln_s) {
    float err;
    const float hi = add_with_error(m, ln_s.hi, err);
    return Lse{hi, ln_s.lo + fmaf(-ref_error(m), kLn2, err)};
}

// z - lse, rounded once where it is finite; not above 0, by which the sum's own
// rounding can pass it where one logit has all the weight.
__device__ __forceinline__ float minus_lse(float z, const Lse& lse) {
    float err;
    const float d = add_with_error(z, -lse.hi, err);
    const float lp = d + ((isfinite(d) ? err : 0.f) - lse.lo);
    return lp > 0.f ? 0.f : lp;
}

// How a row of V logits is streamed: `head` elements up to the first 128-byte
// boundary, n8 16-byte chunks from there, and `tail` elements after them.
// Rows start at any element (V odd, strided or offset views), and a wave's
// 1 KB load instruction then still covers whole 128-byte lines.
constexpr int kLineElems = 64;  // elements of a 128-byte line

struct RowSpan {
    const v4u* body;
    int64_t n8;
    int line;  // elements from the row's start to the boundary (< kLineElems)
    int head;  // line, or V if the row ends before it
    int tail;  // < 8
};

__device__ __forceinline__ RowSpan row_span(const uint16_t* row, int64_t V) {
    RowSpan sp;
    const uintptr_t past = reinterpret_cast<uintptr_t>(row) % (2 * kLineElems);
    sp.line = past ? static_cast<int>((2 * kLineElems - past) / 2) : 0;
    sp.head = static_cast<int>(min(static_cast<int64_t>(sp.line), V));
    sp.body = reinterpret_cast<const v4u*>(row + sp.head);
    sp.n8 = (V - sp.head) >> 3;
    sp.tail = static_cast<int>((V - sp.head) & 7);
    return sp;
}

// The element of the row's head or tail that thread tid holds (head elements
// in threads 0 .., tail elements from thread kLineElems on), and whether it
// holds one.
__device__ __forceinline__ int64_t edge_element(const RowSpan& sp, int64_t V, int tid, bool& ok) {
    const bool in_head = tid < sp.head;
    const bool in_tail = tid >= kLineElems && tid < kLineElems + sp.tail;
    ok = in_head || in_tail;
    return in_tail ? V - sp.tail + (tid - kLineElems) : (in_head ? tid : 0);
}

__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
    const __hip_bfloat16 a = __float2bfloat16(lo);
    const __hip_bfloat16 b = __float2bfloat16(hi);
    return static_cast<uint32_t>(__bfloat16_as_ushort(a)) |
           (static_cast<uint32_t>(__bfloat16_as_ushort(b)) << 16);
}

// Row r of a [rows, T, V] tensor with element strides (stride_b, stride_t).
__device__ __forceinline__ const uint16_t* row_ptr(const uint16_t* logits, int64_t r, int64_t T,
                                                   int64_t stride_b, int64_t stride_t) {
    const int64_t b = r / T;
    return logits + b * stride_b + (r - b * T) * stride_t;
}

}  // namespace meshy
