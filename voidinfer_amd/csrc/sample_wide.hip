// sample_wide.hip — full-vocabulary rows of the batched sampler for fp32
// logits (temperature > 0 and top_k = 0 or > 64): penalties, temperature,
// top-k / min-p / top-p over the whole vocabulary and the Philox inverse-CDF
// draw.  Semantics as the 16-bit route's: order (z desc, id asc), weights
// exp(z - z_max), the cap, the min-p and top-p cuts, the draw.
//
// A 16-bit logit takes one of 65,536 patterns, so a count per pattern
// describes its row exactly; a 32-bit one does not.  Here a row is described
// in two levels, both keyed by z = x' * (1/T) itself:
//   * bins of z: bin j holds floor(64 z) = anchor - j, counted down from the
//     largest z (anchor = floor(64 z_max)).  4,096 bins of width 1/64 cover the
//     64 below the top; one deep bin holds the rest, whose weights (below
//     e^-63 of the largest) are counted but carry no mass.  A logit's weight
//     inside its bin, exp(z - bin floor) in [1, e^(1/64)), is kept as 2^-31
//     fixed point: bin masses are integer sums, exact in any order, and every
//     later sum over the same logits gives the same integers;
//   * the logits of the one bin a decision lands in, narrowed by 8-bit digits
//     of the 32-bit order key until one key remains; the rank among equal keys
//     follows from their common weight, the owner from their ids.
//
// Launches: (history route with penalties) the rows' presence bitmaps and
// count hashes;
//   1. one workgroup per (row, slice of 16,384 logits) counts and weighs the
//      slice's bins: one LDS atomic per logit;
//   2. one workgroup per row adds the slices' bins and finds, from the bins'
//      running counts and masses alone, the bins that the cap, the cuts and the
//      draw can fall into (a few: the exact cap and cut lie inside their bins,
//      so what depends on them is bounded by the bins' ends);
//   3. one workgroup per (row, slice) reads the logits again (from the Infinity
//      Cache) and lists the (key, offset) pairs of those bins;
//   4. one workgroup per row narrows the decisions inside the bins and names
//      the token;
//   5. optionally the filtered distribution.
// What a row's bins look like does not matter to the cost: the passes of 1 and
// 3 are the same for flat and for peaked rows, and 4 handles a few bins' pairs.
// (Listing pairs in the first pass and reading a slice's logits again in the
// per-row pass when a decision fell past the listed ones cost a near-flat row of
// 117,056 logits 320 us a call.)
//
// Roofline: HBM; V x 4 bytes of logits per row read once (and once more from
// cache); per slice the occupied bins' sums written and read back.
#include <math.h>

#include "keys16.h"
#include "penalty_state.h"
#include "vi_device.h"
#include "vi_internal.h"

namespace vi {
namespace {

constexpr int kT = 1024;
constexpr int kW = kT / kWave;
constexpr int kSL = 16384;                 // logits per slice (slice offsets fit 16 bits)
constexpr int kVPT = kSL / (4 * kT);       // 16-byte vectors per thread and slice
constexpr int kMaxSlices = 32;
constexpr int kNB = 4096;                  // bins of width 1/64 below the top
constexpr int kDeep = kNB;                 // everything further down
constexpr double kPerUnit = 64.0;
constexpr double kFixScale = 1.0 / 2147483648.0;
constexpr int kCap = 12288;                // pairs staged in LDS (more are read from memory)
constexpr int kDig = 256;
constexpr int kRanges = 4;                 // bin ranges a row's decisions can need: cap, min-p, top-p, draw
constexpr uint32_t kTakeAll = 0xffffffffu;
static_assert(kVPT * 4 * kT == kSL && kNB == 4 * kT, "slice and bin geometry");

struct WideHead {
    double anchor;                 // floor(64 z_top) of the slice
    uint32_t top_key, n_valid, flags;
    uint32_t nbins;                // bins 0 .. nbins - 1 may hold logits (the rest only the deep bin)
};
static_assert(sizeof(WideHead) == 24, "slice head");

// A bin's sums in one word: logits << 32 | sum of (weight - 1) in 2^-23 units.
// A weight exp(z - bin floor) in [1, e^(1/64)) is a float whose mantissa is that
// excess; 16,384 of them stay below 2^32, so the two halves never mix.
__host__ __device__ __forceinline__ uint32_t bin_count(unsigned long long w) { return uint32_t(w >> 32); }
__host__ __device__ __forceinline__ unsigned long long bin_fix(unsigned long long w) {   // 2^-31 units
    return ((w >> 32) << 31) + ((w & 0xffffffffull) << 8);
}

// What the per-row launches hand on: the row's anchor and top, the bins in use
// and the bin ranges whose pairs the gather lists (empty: lo > hi).
struct WidePlan {
    double A;                      // floor(64 z_max)
    uint32_t top, n_valid, flags, ok;   // ok: the row is served (0: written already)
    uint32_t bins;                 // running sums written for bins 0 .. bins
    int nranges;                   // ranges in use (the first ones; the rest are empty)
    int lo[kRanges], hi[kRanges];
};

using WideBound = FullBound;   // what the probs kernel and verification need to rebuild the support

struct WideArgs {
    const void* logits;
    int rows, vocabulary, slices;
    int64_t stride;
    const vi_row_params* params;
    unsigned char* pstate;         // per-lane penalty states (or null: histories)
    PenaltyLayout pl;
    const int32_t* histories;
    const int64_t* offsets;
    int64_t max_history;
    uint32_t* hbits;               // [rows][words] presence bitmaps (history route)
    int words;
    uint2* hash;                   // [rows][hash_slots] (token + 1, count) (history route)
    int hash_shift, hash_slots;
    uint32_t* row_flags;           // [rows] history flags (history route)
    int record;
    int32_t* tokens;
    double* uniforms;
    float* probs;
    int64_t probs_stride;
    vi_sample_stats* stats;
    // workspace
    WideHead* heads;               // [rows][slices]
    unsigned long long* hist;      // [rows][slices][kNB]: bin sums, bins 0 .. nbins - 1
    WidePlan* plans;               // [rows]
    uint32_t* exc;                 // [rows][kNB + 2]: logits in the bins before J; [bins in use ..] all but deep
    double* exm;                   // [rows][kNB + 1]: mass of the bins before J
    uint32_t* npairs;              // [rows][slices]
    uint2* pairs;                  // [rows][slices][kSL]: (key, slice << 16 | offset), in any order
    int want_bounds;               // bounds wanted (probs, or verification)
    int draw_every;                // rows whose token is drawn: every n-th (row % n == n - 1), or none (0)
    WideBound* bounds;             // [rows]
};

__device__ __forceinline__ bool full_row(const vi_row_params& p) { return !topk_route(p); }

// Order key of a finite z (+0 and -0 share +0's), and back.  Finite z have
// keys in [0x00800000, 0xff7fffff]; key 0 marks "no valid logit".
__device__ __forceinline__ uint32_t key32(float z) {
    uint32_t u = __builtin_bit_cast(uint32_t, z);
    if (z == 0.0f) u = 0u;
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float unkey32(uint32_t k) {
    return __builtin_bit_cast(float, (k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

// Bin of a finite z below `anchor` (kDeep past the 4,096th) and its weight's
// excess, exp(z - bin floor) - 1 in 2^-23 units (0 in the deep bin).  In single
// precision and still exact: 64 z is a scaling by a power of two, its floor and
// fraction are representable, and anchor - floor is exact where it is below
// 4,096 (both below 2^24, or within a factor of two of one another) and rounds to
// no less than 4,096 elsewhere.  |64 z| past the float range is -inf, deep;
// anchors there (kWideBig) take the double form.  A NaN counts as deep.
struct BinW {
    int bin;
    uint32_t ex;
};
constexpr float kWideBig = 0x1p120f;
template <bool BIG>
__device__ __forceinline__ BinW bin_of_z(float z, float anchor_f, double anchor_d) {
    float frac;
    int j;
    if constexpr (BIG) {
        const double zz = double(z) * kPerUnit, f = floor(zz), dj = anchor_d - f;
        if (!(dj < double(kNB))) return {kDeep, 0u};
        j = int(dj);
        frac = float(zz - f);
    } else {
        const float zz = z * float(kPerUnit), f = floorf(zz), dj = anchor_f - f;
        if (!(dj < float(kNB))) return {kDeep, 0u};
        j = int(dj);
        frac = zz - f;
    }
    const float w = __builtin_amdgcn_exp2f(frac * (1.44269504088896340736f / 64.0f));   // in [1, 2)
    return {j, __builtin_elementwise_sub_sat(__builtin_bit_cast(uint32_t, w), 0x3f800000u)};
}
__device__ __forceinline__ int bin_of_key(uint32_t k, double anchor) {
    const double dj = anchor - floor(double(unkey32(k)) * kPerUnit);
    return dj < double(kNB) ? int(dj) : kDeep;
}
// A key's weight in its bin, 2^-31 units.
__device__ __forceinline__ uint32_t weight_fix(uint32_t k) {
    const double zz = double(unkey32(k)) * kPerUnit;
    const float w = __builtin_amdgcn_exp2f(float(zz - floor(zz)) * (1.44269504088896340736f / 64.0f));
    return 0x80000000u + (__builtin_elementwise_sub_sat(__builtin_bit_cast(uint32_t, w), 0x3f800000u) << 8);
}

// ------------------------------------------------------------------ penalties
struct WPen {
    bool on;
    const uint32_t* bits;   // presence bitmap (token t: bit t & 31 of word t >> 5)
    const uint2* table;     // (token + 1, count), linear probing
    int shift, slots;
};
__device__ __forceinline__ WPen wpen(const WideArgs& a, int row, const vi_row_params& p) {
    WPen w{};
    if (!penalties_active(p)) return w;
    if (a.pstate) {
        const unsigned char* st = a.pstate + size_t(row) * a.pl.lane_bytes;
        w.on = true;
        w.bits = reinterpret_cast<const uint32_t*>(st + a.pl.off_b1);
        w.table = reinterpret_cast<const uint2*>(st + a.pl.off_hash);
        w.shift = a.pl.shift;
        w.slots = a.pl.slots;
    } else if (a.histories && a.offsets && a.hash && a.offsets[row + 1] > a.offsets[row]) {
        w.on = true;
        w.bits = a.hbits + size_t(row) * size_t(a.words);
        w.table = a.hash + size_t(row) * size_t(a.hash_slots);
        w.shift = a.hash_shift;
        w.slots = a.hash_slots;
    }
    return w;
}

// z of a logit (raw bits b) seen c times; NaN when x, the penalized x' or z is
// not finite (*bad set).  -0 comes out as +0.  logit_z: of token t, its count
// looked up where the presence word `word` holds its bit; `unrecord`: a token
// whose count is one too high (the sampler recorded it already).
__device__ __forceinline__ float counted_z(const vi_row_params& p, float inv_t, uint32_t b, uint32_t c, bool* bad) {
    float x = __builtin_bit_cast(float, b);
    if (c && isfinite(x)) x = __builtin_bit_cast(float, penalize_bits<VI_F32>(b, c, p));
    const float z = x * inv_t + 0.0f;
    const bool ok = isfinite(z);   // (not for an infinite or NaN x)
    *bad |= !ok;
    return ok ? z : __builtin_nanf("");
}
__device__ __forceinline__ float logit_z(const WPen& w, const vi_row_params& p, float inv_t, int t, uint32_t b,
                                         uint32_t word, bool* bad, int unrecord = -1) {
    uint32_t c = 0u;
    if (w.on && ((word >> (t & 31)) & 1u)) {
        c = hash_count(w.table, w.shift, w.slots, t);
        if (t == unrecord && c) --c;
    }
    return counted_z(p, inv_t, b, c, bad);
}

// The history route's presence bitmap and count hash of each full-route row
// with penalties (the top-k route builds its own rows' hashes), both in LDS and
// copied out; a table past kHistLdsSlots is built in place.  Bound by the chain of
// compare-and-swap round trips: 23 rows of 739 tokens over 151,936 take 12.6 us with
// 256 threads and every atomic in global memory.
constexpr int kHistLdsSlots = 8192;
constexpr int kHistWords = kMaxSlices * kSL / 32;
__global__ __launch_bounds__(kT) void wide_history_kernel(WideArgs a) {
    __shared__ uint2 s_table[kHistLdsSlots];
    __shared__ uint32_t s_bits[kHistWords];
    __shared__ uint32_t s_flags;
    const int r = blockIdx.x, tid = threadIdx.x;
    const vi_row_params p = a.params[r];
    if (!full_row(p) || !penalties_active(p)) return;
    const int64_t b = a.offsets[r], n = a.offsets[r + 1] - b;
    if (n <= 0) return;
    uint32_t* bits = a.hbits + size_t(r) * size_t(a.words);
    uint2* out = a.hash + size_t(r) * size_t(a.hash_slots);
    const bool in_lds = a.hash_slots <= kHistLdsSlots;
    auto build = [&](uint2* table) {
        for (int i = tid; i < a.hash_slots; i += kT) table[i] = make_uint2(0u, 0u);
        __syncthreads();
        if (n > a.max_history) {
            if (tid == 0) s_flags = VI_FLAG_ERROR;
            return;
        }
        constexpr int kU = 4;   // (the history loads of a round issued together)
        for (int64_t i0 = 0; i0 < n; i0 += int64_t(kU) * kT) {
            int32_t tk[kU];
#pragma unroll
            for (int u = 0; u < kU; ++u) tk[u] = a.histories[b + min(i0 + int64_t(u) * kT + tid, n - 1)];
#pragma unroll
            for (int u = 0; u < kU; ++u) {
                if (i0 + int64_t(u) * kT + tid >= n) continue;
                const int32_t t = tk[u];
                if (t < 0 || t >= a.vocabulary) { atomicOr(&s_flags, uint32_t(VI_FLAG_BAD_HISTORY)); continue; }
                atomicOr(&s_bits[t >> 5], 1u << (t & 31));
                uint32_t s = (uint32_t(t) * 0x9E3779B1u) >> a.hash_shift;
                for (int probe = 0; probe < a.hash_slots; ++probe) {
                    const uint32_t old = atomicCAS(&table[s].x, 0u, uint32_t(t) + 1u);
                    if (old == 0u || old == uint32_t(t) + 1u) { atomicAdd(&table[s].y, 1u); break; }
                    s = (s + 1u) & uint32_t(a.hash_slots - 1);
                }
            }
        }
    };
    if (tid == 0) s_flags = 0u;
    for (int i = tid; i < a.words; i += kT) s_bits[i] = 0u;
    if (in_lds) build(s_table);
    else build(out);
    __syncthreads();
    for (int i = tid; i < a.words; i += kT) bits[i] = s_bits[i];
    if (in_lds)
        for (int i = tid; i < a.hash_slots; i += kT) out[i] = s_table[i];
    if (tid == 0) a.row_flags[r] = s_flags;
}

struct WGeo {
    int s0, n, nvec;        // first token, tokens, whole 16-byte vectors (at the row's alignment)
    const uint32_t* base;
};
__device__ __forceinline__ WGeo wgeo(const WideArgs& a, int row, int s) {
    WGeo g;
    g.s0 = s * kSL;
    g.n = min(kSL, a.vocabulary - g.s0);
    g.nvec = g.n / 4;
    g.base = static_cast<const uint32_t*>(a.logits) + int64_t(row) * a.stride + g.s0;
    return g;
}

__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) {
#pragma unroll
    for (int o = 32; o; o >>= 1) v = max(v, uint32_t(__shfl_xor(int(v), o, kWave)));
    return v;
}

// A slice's z held by the workgroup: thread t's vectors i kT + t (i < kVPT) and
// one of the up to three logits past the last vector; NaN where there is no
// valid logit.
struct SliceZ {
    float z[kVPT][4], tail;
    bool bad;
};
// PEN: the call has penalty inputs (lane states or histories).
template <bool PEN>
__device__ __forceinline__ SliceZ slice_z(const WideArgs& a, const WGeo& g, int row, const vi_row_params& p) {
    const int tid = threadIdx.x;
    uint4 v[kVPT];
    if (g.nvec > 0) {   // (uniform; clamped addresses: no load under a divergent branch)
#pragma unroll
        for (int i = 0; i < kVPT; ++i) v[i] = load16_cached(g.base + 4 * size_t(min(i * kT + tid, g.nvec - 1)));
    } else {
#pragma unroll
        for (int i = 0; i < kVPT; ++i) v[i] = make_uint4(0u, 0u, 0u, 0u);
    }
    const int tt = 4 * g.nvec + tid;
    const uint32_t tb = tt < g.n ? g.base[tt] : 0u;
    const WPen w = PEN ? wpen(a, row, p) : WPen{};
    const float inv_t = 1.0f / p.temperature;
    SliceZ r;
    r.bad = false;
    if (w.on) {   // (uniform)
        // History tokens take their counts from the hash: a vector's four tokens
        // share a bitmap word; the first probes of two vectors are requested
        // together (absent tokens read slot 0), and only a probe that meets
        // another token goes on by itself.  (The first four slots of each chain
        // requested together, for one vector at a time, was slower: 89 rows x 69,440
        // with 4,318-token histories 26.5 us against 21.)
        uint32_t word[kVPT];
#pragma unroll
        for (int i = 0; i < kVPT; ++i) word[i] = w.bits[(g.s0 + 4 * min(i * kT + tid, max(g.nvec - 1, 0))) >> 5];
#pragma unroll
        for (int i0 = 0; i0 < kVPT; i0 += 2) {
            uint2 first[2][4];
            uint32_t here[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int x = (i0 + h) * kT + tid, t0 = g.s0 + 4 * x;
                here[h] = x < g.nvec ? (word[i0 + h] >> (t0 & 31)) & 0xfu : 0u;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const uint32_t slot = (uint32_t(t0 + e) * 0x9E3779B1u) >> w.shift;
                    first[h][e] = w.table[((here[h] >> e) & 1u) ? slot : 0u];
                }
            }
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int x = (i0 + h) * kT + tid, t0 = g.s0 + 4 * x;
                bool bad = false;   // (not of a lane past the last vector: its logits lack their counts)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const uint32_t b = vec_bits<VI_F32>(v[i0 + h], e);
                    uint32_t c = 0u;
                    if ((here[h] >> e) & 1u) {
                        c = first[h][e].x == uint32_t(t0 + e) + 1u ? first[h][e].y
                            : first[h][e].x == 0u                  ? 0u
                                                  : hash_count(w.table, w.shift, w.slots, t0 + e);
                    }
                    r.z[i0 + h][e] = counted_z(p, inv_t, b, c, &bad);
                }
                r.bad |= bad && x < g.nvec;
            }
        }
    } else {
#pragma unroll
        for (int i = 0; i < kVPT; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) r.z[i][e] = counted_z(p, inv_t, vec_bits<VI_F32>(v[i], e), 0u, &r.bad);
    }
    // (lanes past the last vector hold its logits again)
    const float none = __builtin_nanf("");
#pragma unroll
    for (int i = 0; i < kVPT; ++i)
        if ((i + 1) * kT > g.nvec) {   // (uniform)
#pragma unroll
            for (int e = 0; e < 4; ++e) r.z[i][e] = i * kT + tid < g.nvec ? r.z[i][e] : none;
        }
    r.tail = none;
    if (tt < g.n) r.tail = logit_z(w, p, inv_t, g.s0 + tt, tb, w.on ? w.bits[(g.s0 + tt) >> 5] : 0u, &r.bad);
    return r;
}

// ------------------------------------------------------------------ 1. the slices' bins
// Bound by the LDS atomics (one u64 per logit, at data-dependent banks) and the
// VALU work per logit (128 x 248,320: 35.6 us, 92 with a count and a mass atomic per
// logit, 64-bit floating bin arithmetic and the pairs placed here).
template <bool PEN>
__global__ __launch_bounds__(kT, 8) void wide_hist_kernel(WideArgs a) {
    __shared__ __attribute__((aligned(16))) unsigned long long H[kNB];
    __shared__ uint32_t s_top, s_flags, s_nb, s_invalid;
    const int s = blockIdx.x, row = blockIdx.y, tid = threadIdx.x;
    const vi_row_params p = a.params[row];
    if (!full_row(p)) return;
#pragma unroll
    for (int i = 0; i < kNB / 2 / kT; ++i) reinterpret_cast<uint4*>(H)[i * kT + tid] = make_uint4(0u, 0u, 0u, 0u);
    if (tid == 0) { s_top = 0u; s_flags = 0u; s_nb = 0u; s_invalid = 0u; }
    const WGeo g = wgeo(a, row, s);
    const SliceZ r = slice_z<PEN>(a, g, row, p);
    float mz = r.tail;   // (fmaxf passes NaN over)
#pragma unroll
    for (int i = 0; i < kVPT; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) mz = fmaxf(mz, r.z[i][e]);
    const uint32_t mk = wave_max_u32(isnan(mz) ? 0u : key32(mz));
    __syncthreads();   // (LDS cleared)
    if (lane_id() == 0 && mk) atomicMax(&s_top, mk);
    if (ballot(r.bad)) {   // (wave-uniform, rare) the invalid logits, taken from the slice's
        uint32_t ni = tid < g.n - 4 * g.nvec && isnan(r.tail) ? 1u : 0u;
#pragma unroll
        for (int i = 0; i < kVPT; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) ni += i * kT + tid < g.nvec && isnan(r.z[i][e]) ? 1u : 0u;
        ni = wave_sum_u32(ni);
        if (lane_id() == 0) {
            atomicOr(&s_flags, uint32_t(VI_FLAG_NONFINITE));
            atomicAdd(&s_invalid, ni);
        }
    }
    __syncthreads();
    const uint32_t top = s_top;
    WideHead* hd = a.heads + size_t(row) * a.slices + s;
    if (top == 0u) {
        if (tid == 0) *hd = WideHead{0.0, 0u, 0u, s_flags, 0u};
        return;
    }
    const float zt = unkey32(top);
    const double anchor = floor(double(zt) * kPerUnit);
    const float anchor_f = float(anchor);
    uint32_t nbl = 0u;   // one past the last non-deep bin holding logits
    auto count_all = [&](auto big) {
        auto count = [&](float z) {
            const BinW b = bin_of_z<decltype(big)::value>(z, anchor_f, anchor);
            if (b.bin >= kNB) return;
            atomicAdd(&H[b.bin], (1ull << 32) | b.ex);
            nbl = max(nbl, uint32_t(b.bin) + 1u);
        };
#pragma unroll
        for (int i = 0; i < kVPT; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) count(r.z[i][e]);
        count(r.tail);
    };
    if (fabsf(zt) < kWideBig) count_all(std::false_type{});
    else count_all(std::true_type{});
    nbl = wave_max_u32(nbl);
    if (lane_id() == 0 && nbl) atomicMax(&s_nb, nbl);
    __syncthreads();
    const uint32_t nb = s_nb;
    unsigned long long* out = a.hist + (size_t(row) * a.slices + s) * kNB;
    for (uint32_t i = tid; i < nb; i += kT) out[i] = H[i];
    if (tid == 0) *hd = WideHead{anchor, top, uint32_t(g.n) - s_invalid, s_flags, nb};
}

// ------------------------------------------------------------------ the bins' running sums
// EXC[J] logits and EXM[J] mass in the bins before J (J <= kNB; EXC[kNB + 1] the
// row's logits).  The first bin in order that holds logits and whose inclusive
// count (mode 0: >= target; the deep bin included) or mass (1: >=, 2: >) reaches
// the target, or -1; every wave alike.
struct BinSums {
    const uint32_t* EXC;
    const double* EXM;
};
__device__ __forceinline__ int find_bin(const BinSums& B, int mode, double target) {
    const int last = mode == 0 ? kNB : kNB - 1;
    int J = wave_search(0, last + 1, [&](int j) {
        if (mode == 0) return double(B.EXC[j + 1]) >= target;
        return mode == 1 ? B.EXM[j + 1] >= target : B.EXM[j + 1] > target;
    });
    while (J <= last && B.EXC[J + 1] == B.EXC[J]) ++J;   // (rounding of the running masses)
    return J <= last ? J : -1;
}
__device__ __forceinline__ double unit_of(double A, double z0, int J) {   // 2^-31 x exp(bin floor - z0)
    return kFixScale * exp((A - double(J)) / kPerUnit - z0);
}

// Smallest key in [lo, hi) with pred(key) (monotone false -> true), or hi;
// one wave, 64 probes per round.
template <class P>
__device__ __forceinline__ uint32_t wave_search_u32(uint32_t lo, uint32_t hi, P pred) {
    const int lane = lane_id();
    uint64_t l = lo, h = hi;
    while (h > l) {
        const uint64_t n = h - l;
        if (n <= uint64_t(kWave)) {
            const uint64_t m = ballot(uint64_t(lane) < n && pred(uint32_t(l + lane)));
            return m ? uint32_t(l + __builtin_ctzll(m)) : uint32_t(h);
        }
        const uint64_t step = (n + kWave - 1) / kWave;
        const uint64_t p = l + uint64_t(lane) * step;
        const uint64_t valid = ballot(p < h);
        const uint64_t m = ballot(p < h && pred(uint32_t(p)));
        if (!m) {
            l = l + uint64_t(63 - __builtin_clzll(valid)) * step + 1;
            continue;
        }
        const int f = __builtin_ctzll(m);
        if (f == 0) return uint32_t(l);
        const uint64_t nl = l + uint64_t(f - 1) * step + 1;
        h = l + uint64_t(f) * step;
        l = nl;
    }
    return uint32_t(l);
}
// The min-p cut: the smallest key whose weight reaches min_p; one wave.
__device__ __forceinline__ uint32_t minp_cut(const vi_row_params& p, uint32_t top, double z0) {
    const double mp = double(p.min_p);
    return wave_search_u32(0x00800000u, top + 1u, [&](uint32_t key) { return exp(double(unkey32(key)) - z0) >= mp; });
}

__device__ __forceinline__ void write_row(const WideArgs& a, int row, int32_t token, double u, uint32_t flags,
                                          uint32_t support, uint32_t finite, double s_n) {
    a.tokens[row] = token;
    if (a.uniforms) a.uniforms[row] = u;
    if (a.stats) {
        vi_sample_stats st{};
        st.flags = flags;
        st.support = support;
        st.finite = finite;
        st.support_mass = s_n;
        st.uniform = u;
        a.stats[row] = st;
    }
}

// ------------------------------------------------------------------ 2. the row's bins and ranges
__global__ __launch_bounds__(kT) void wide_plan_kernel(WideArgs a) {
    __shared__ uint32_t EXC[kNB + 2];
    __shared__ double EXM[kNB + 1];
    __shared__ unsigned long long PX[3 * (kT / 4) * 4];   // partial sums of the other thread groups
    __shared__ uint32_t PC[3 * (kT / 4) * 4];
    __shared__ double dscan[kW + 1], s_anchor;
    __shared__ uint32_t uscan[kW + 1], s_top, s_valid, s_flags, s_rb;
    __shared__ int s_delta[kMaxSlices], s_nbin[kMaxSlices];
    const int row = blockIdx.x, tid = threadIdx.x, lane = lane_id(), wave = tid / kWave;
    const vi_row_params p = a.params[row];
    if (!full_row(p)) return;
    const int S = a.slices, V = a.vocabulary;
    const size_t rs0 = size_t(row) * S;

    // ---- slice heads: the row's anchor, top key, valid logits and flags
    if (tid == 0) { s_top = 0u; s_valid = 0u; s_flags = 0u; s_anchor = 0.0; s_rb = 0u; }
    __syncthreads();
    WideHead hd{};
    if (tid < S) {
        hd = a.heads[rs0 + tid];
        atomicAdd(&s_valid, hd.n_valid);
        atomicOr(&s_flags, hd.flags);
        if (hd.n_valid) atomicMax(&s_top, hd.top_key);
    }
    if (tid == 0) {
        uint32_t pf = 0u;
        if (a.pstate) {
            if (penalties_active(p))
                pf = reinterpret_cast<const PenaltyHeader*>(a.pstate + size_t(row) * a.pl.lane_bytes)->flags;
        } else if (a.row_flags && a.histories && a.offsets && a.hash && penalties_active(p) &&
                   a.offsets[row + 1] > a.offsets[row]) {
            pf = a.row_flags[row];
        }
        atomicOr(&s_flags, pf & uint32_t(VI_FLAG_BAD_HISTORY | VI_FLAG_ERROR));
    }
    __syncthreads();
    const uint32_t top = s_top, N = s_valid;
    if (tid < S && hd.n_valid && hd.top_key == top) s_anchor = hd.anchor;   // (equal tops: equal anchors)
    __syncthreads();
    const double A = s_anchor, z0 = double(unkey32(top));
    const uint32_t out_flags = s_flags & uint32_t(VI_FLAG_NONFINITE | VI_FLAG_BAD_HISTORY);
    const bool fail = (s_flags & VI_FLAG_ERROR) != 0u;
    if (fail || N == 0u) {
        if (tid == 0) {
            write_row(a, row, fail ? -1 : V, 0.0, out_flags | (fail ? VI_FLAG_ERROR : VI_FLAG_EMPTY), 0u, 0u, 0.0);
            if (a.want_bounds) a.bounds[row] = WideBound{0.0, 0.0, 0.0f, 0u, 0, 0u};
            a.plans[row].ok = 0u;
        }
        return;
    }
    if (tid < kMaxSlices) {
        int d = -1;
        if (tid < S && hd.n_valid) {
            const double dd = A - hd.anchor;
            d = dd < double(kNB + 1) ? int(dd) : kNB + 1;
        }
        s_delta[tid] = d;
        s_nbin[tid] = int(hd.nbins);
        if (d >= 0 && d < kNB) atomicMax(&s_rb, uint32_t(min(kNB, d + int(hd.nbins))));   // (row bins in use)
    }
    __syncthreads();

    // ---- counts and masses summed over the slices (thread t: bins 4t .. 4t + 3),
    // then their exclusive prefixes in bin order (four slices' loads issued
    // together, unconditional at clamped places and dropped afterwards: a load
    // under a branch waits for the ones before).  When the row's bins in use fit
    // in a half or a quarter of the 4,096, the slices are shared out between two
    // or four groups of threads (fewer dependent load rounds each), whose sums
    // meet in LDS.
    const int rb = int(s_rb);
    const int ways = rb <= kNB / 4 ? 4 : rb <= kNB / 2 ? 2 : 1;
    const int per = kT / ways, way = tid / per, quad = tid - way * per;
    const int sp = (S + ways - 1) / ways, sb = min(S, way * sp), se = min(S, sb + sp);
    uint32_t bc[4] = {0u, 0u, 0u, 0u};
    unsigned long long bx[4] = {0ull, 0ull, 0ull, 0ull};   // (excesses: 2^-23 units)
    for (int s0 = sb; s0 < se; s0 += 4) {
        unsigned long long w[4][4];
        bool on[4][4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int sc = min(s0 + u, se - 1), d = s_delta[sc], nb = s_nbin[sc];
            const bool live = s0 + u < se && d >= 0 && d < kNB;
            const unsigned long long* h = a.hist + (rs0 + sc) * kNB;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int j = 4 * quad + q - d;
                on[u][q] = live && j >= 0 && j < nb;
                w[u][q] = h[on[u][q] ? j : 0];
            }
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (on[u][q]) { bc[q] += bin_count(w[u][q]); bx[q] += w[u][q] & 0xffffffffull; }
    }
    if (ways > 1) {
        if (way > 0) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                PC[((way - 1) * per + quad) * 4 + q] = bc[q];
                PX[((way - 1) * per + quad) * 4 + q] = bx[q];
            }
        }
        __syncthreads();
        if (way == 0) {
            for (int v = 1; v < ways; ++v)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    bc[q] += PC[((v - 1) * per + quad) * 4 + q];
                    bx[q] += PX[((v - 1) * per + quad) * 4 + q];
                }
        } else {   // (their bins 4 tid .. 4 tid + 3 lie past the bins in use)
#pragma unroll
            for (int q = 0; q < 4; ++q) { bc[q] = 0u; bx[q] = 0ull; }
        }
    }
    double bm[4];
    uint32_t csum = 0u;
    double msum = 0.0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const unsigned long long fix = ((unsigned long long)bc[q] << 31) + (bx[q] << 8);
        bm[q] = bc[q] ? double(fix) * unit_of(A, z0, 4 * tid + q) : 0.0;
        csum += bc[q];
        msum += bm[q];
    }
    uint32_t ctot = 0u;
    const uint32_t cex = block_exclusive_scan_u32<kT>(csum, uscan, &ctot);
    {   // exclusive prefix of the per-thread masses, wave by wave in a fixed order
        const double incl = wave_incl_scan_f64(msum);
        const int src = max(lane - 1, 0);
        const uint64_t bits = __builtin_bit_cast(uint64_t, incl);
        const uint32_t lo = uint32_t(__builtin_amdgcn_ds_bpermute(src << 2, int(uint32_t(bits))));
        const uint32_t hi = uint32_t(__builtin_amdgcn_ds_bpermute(src << 2, int(uint32_t(bits >> 32))));
        const double wex = lane ? __builtin_bit_cast(double, (uint64_t(hi) << 32) | lo) : 0.0;
        if (lane == kWave - 1) dscan[wave] = incl;
        __syncthreads();
        if (wave == 0) {
            const double t = lane < kW ? dscan[lane] : 0.0;
            const double it = wave_incl_scan_f64(t);
            if (lane < kW) dscan[lane] = it - t;
        }
        __syncthreads();
        double m = dscan[wave] + wex;
        uint32_t cc = cex;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            EXC[4 * tid + q] = cc;
            EXM[4 * tid + q] = m;
            cc += bc[q];
            m += bm[q];
        }
        if (tid == kT - 1) {
            EXC[kNB] = cc;
            EXC[kNB + 1] = N;
            EXM[kNB] = m;
        }
    }
    __syncthreads();
    // the running sums, for the last launch (bins past the ones in use repeat the
    // last value)
    uint32_t* exc = a.exc + size_t(row) * (kNB + 2);
    double* exm = a.exm + size_t(row) * (kNB + 1);
    for (int i = tid; i <= rb; i += kT) { exc[i] = EXC[i]; exm[i] = EXM[i]; }
    if (wave != 0) return;

    // ---- the ranges: the bin of the cap; the bin of the min-p cut; the bins the
    // top-p cut can fall in while the cap's mass is known to its bin's ends; the
    // bins the draw can fall in while the support's mass is known to the ends of
    // the bins before
    const BinSums B{EXC, EXM};
    const double s_all = EXM[kNB];
    WidePlan pl{};
#pragma unroll
    for (int i = 0; i < kRanges; ++i) { pl.lo[i] = 1; pl.hi[i] = 0; }
    double cap_lo = s_all, cap_hi = s_all, n_lo = s_all, n_hi = s_all;
    auto ends = [&](int lo, int hi, double* ml, double* mh) {   // (bins lo .. hi)
        *ml = lo < kNB ? EXM[lo] : s_all;
        *mh = hi < kNB ? EXM[hi + 1] : s_all;
    };
    auto shrink = [&](double ml, double mh) { n_lo = fmin(n_lo, ml); n_hi = fmin(n_hi, mh); };
    if (p.top_k > 0 && uint32_t(p.top_k) < N) {
        const int J = find_bin(B, 0, double(p.top_k));
        pl.lo[0] = pl.hi[0] = J;
        ends(J, J, &cap_lo, &cap_hi);
        shrink(cap_lo, cap_hi);
    }
    if (p.min_p > 0.0f) {
        const uint32_t kf = minp_cut(p, top, z0);
        const int J = kf <= top ? bin_of_key(kf, A) : 0;
        pl.lo[1] = pl.hi[1] = J;
        double ml, mh;
        ends(J, J, &ml, &mh);
        shrink(kf <= top ? ml : 1.0, kf <= top ? mh : 1.0);   // (no logit passes: the support is the first)
    }
    const int last = max(rb - 1, 0);
    // (the exact masses are sums of the same terms in another order: widened by
    // more than their rounding)
    constexpr double kSlack = 1e-9;
    if (p.top_p < 1.0f) {
        const int j0 = find_bin(B, 1, double(p.top_p) * cap_lo * (1.0 - kSlack));
        const int j1 = find_bin(B, 1, double(p.top_p) * cap_hi * (1.0 + kSlack));
        if (j0 >= 0) {
            pl.lo[2] = j0;
            pl.hi[2] = j1 >= 0 ? j1 : last;
            double ml, mh;
            ends(j0, pl.hi[2], &ml, &mh);
            shrink(ml, mh);
        }
    }
    const double u = philox_uniform(p.seed, p.lane, p.position, 0u);
    const int d0 = find_bin(B, 2, u * n_lo * (1.0 - kSlack)), d1 = find_bin(B, 2, u * n_hi * (1.0 + kSlack));
    if (d0 >= 0) {
        pl.lo[3] = d0;
        pl.hi[3] = d1 >= 0 ? d1 : last;
    }
    pl.A = A;
    pl.top = top;
    pl.n_valid = N;
    pl.flags = out_flags;
    pl.ok = 1u;
    pl.bins = uint32_t(rb);
    // the ranges in use to the front; the rest empty
    WidePlan out = pl;
    int nr = 0;
#pragma unroll
    for (int i = 0; i < kRanges; ++i) { out.lo[i] = 1; out.hi[i] = 0; }
#pragma unroll
    for (int i = 0; i < kRanges; ++i) {
        if (pl.lo[i] > pl.hi[i]) continue;
#pragma unroll
        for (int q = 0; q < kRanges; ++q)
            if (q == nr) { out.lo[q] = pl.lo[i]; out.hi[q] = pl.hi[i]; }
        ++nr;
    }
    out.nranges = nr;
    if (lane == 0) a.plans[row] = out;
}

// ------------------------------------------------------------------ 3. the ranges' pairs
template <bool PEN>
__global__ __launch_bounds__(kT, 8) void wide_gather_kernel(WideArgs a) {
    __shared__ uint32_t s_n;
    const int s = blockIdx.x, row = blockIdx.y, tid = threadIdx.x, lane = lane_id();
    const vi_row_params p = a.params[row];
    if (!full_row(p)) return;
    const WidePlan pl = a.plans[row];
    if (!pl.ok) return;
    if (tid == 0) s_n = 0u;
    const WGeo g = wgeo(a, row, s);
    const SliceZ r = slice_z<PEN>(a, g, row, p);
    const float A_f = float(pl.A);
    uint32_t hit = 0u;   // bit 4i + e: vector i's element e; bit 31: the tail
    // (the bin as a float, anchor - floor(64 z): the deep ones at or past 4,096;
    // NaN is in no range)
    auto mark_all = [&](auto big, auto ranges) {
        constexpr int R = decltype(ranges)::value;
        float lo[R], hi[R];
#pragma unroll
        for (int i = 0; i < R; ++i) {
            lo[i] = float(pl.lo[i]);
            hi[i] = pl.hi[i] == kDeep ? kInfF : float(pl.hi[i]);
        }
        auto mark = [&](float z, uint32_t bit) {
            float j;
            if constexpr (decltype(big)::value) j = float(fmin(pl.A - floor(double(z) * kPerUnit), double(kNB)));
            else j = A_f - floorf(z * float(kPerUnit));
            if constexpr (decltype(big)::value) j = isnan(z) ? z : j;   // (fmin passes NaN over)
            bool in = false;
#pragma unroll
            for (int i = 0; i < R; ++i) in |= (j >= lo[i]) & (j <= hi[i]);
            hit |= in ? bit : 0u;
        };
#pragma unroll
        for (int i = 0; i < kVPT; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) mark(r.z[i][e], 1u << (4 * i + e));
        mark(r.tail, 0x80000000u);
    };
    if (!(fabsf(unkey32(pl.top)) < kWideBig)) mark_all(std::true_type{}, std::integral_constant<int, kRanges>{});
    else if (pl.nranges <= 2) mark_all(std::false_type{}, std::integral_constant<int, 2>{});
    else mark_all(std::false_type{}, std::integral_constant<int, kRanges>{});
    __syncthreads();
    const uint32_t n = uint32_t(__builtin_popcount(hit)), incl = wave_incl_scan_u32(n);
    uint32_t at = 0u;
    if (lane == kWave - 1 && incl) at = atomicAdd(&s_n, incl);
    at = uint32_t(readlane_i(int(at), kWave - 1)) + incl - n;
    uint2* out = a.pairs + (size_t(row) * a.slices + s) * kSL;
    auto put = [&](float z, uint32_t bit, int off) {
        if (hit & bit) out[at++] = make_uint2(key32(z), (uint32_t(s) << 16) | uint32_t(off));
    };
    if (n) {
#pragma unroll
        for (int i = 0; i < kVPT; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) put(r.z[i][e], 1u << (4 * i + e), 4 * (i * kT + tid) + e);
        put(r.tail, 0x80000000u, 4 * g.nvec + tid);
    }
    __syncthreads();
    if (tid == 0) a.npairs[size_t(row) * a.slices + s] = s_n;
}

// ------------------------------------------------------------------ 4. the decisions
struct FinishLds {
    uint32_t EXC[kNB + 2];
    double EXM[kNB + 1];
    uint32_t CK[kCap];              // the row's listed pairs: keys
    uint32_t CI[kCap];              // and slice << 16 | offset
    uint32_t BC[kDig];
    unsigned long long BF[kDig];
    uint32_t OB[kSL / 32];          // owner bitmap
    uint32_t uscan[kW + 1];
    uint32_t pre[kMaxSlices + 1], pcnt[kMaxSlices];   // pairs before each slice's; a key's per slice
    int lo[kRanges], hi[kRanges];   // bins listed
    // scratch for block decisions
    uint32_t u0, u1, u2, u3, kmin, kmax, nbin;
    unsigned long long f0;
    double d0;
    uint32_t staged, n;             // pairs listed, and whether they are in LDS
};

// Result of narrowing one bin: the key the target falls on, the rank there,
// and what the bin's higher keys hold.
struct RHit {
    bool found;
    uint32_t key, rank, cnt_key, cnt_before;
    unsigned long long fix_before, fix_key;
};

struct RowCtx {
    const WideArgs* a;
    int row, S;
    size_t rs0;       // row * slices
    double A, z0;
    uint32_t top;     // the row's largest key
    const vi_row_params* p;
};

// Pair i of the listed ones.
__device__ __forceinline__ uint2 cand(const RowCtx& c, const FinishLds& L, uint32_t i) {
    if (L.staged) return make_uint2(L.CK[i], L.CI[i]);
    int s = 0;
    while (s + 1 < c.S && L.pre[s + 1] <= i) ++s;
    return c.a->pairs[(c.rs0 + s) * kSL + (i - L.pre[s])];
}
__device__ __forceinline__ uint32_t cand_key(const RowCtx& c, const FinishLds& L, uint32_t i) {
    return L.staged ? L.CK[i] : cand(c, L, i).x;
}

// The pairs of bin J alone, listed again from the row's logits (a bin outside
// the planned ranges: a decision that rounding moved).  All threads.
__device__ __forceinline__ void relist(const RowCtx& c, FinishLds& L, int J) {
    const WideArgs& a = *c.a;
    const int tid = threadIdx.x;
    const WPen w = wpen(a, c.row, *c.p);
    const float inv_t = 1.0f / c.p->temperature;
    const uint32_t* base = static_cast<const uint32_t*>(a.logits) + int64_t(c.row) * a.stride;
    __syncthreads();
    if (tid == 0) L.n = 0u;
    __syncthreads();
    bool bad = false;
    for (int t = tid; t < a.vocabulary; t += kT) {
        const float z = logit_z(w, *c.p, inv_t, t, base[t], w.on ? w.bits[t >> 5] : 0u, &bad);
        if (isnan(z) || bin_of_key(key32(z), c.A) != J) continue;
        const uint32_t at = atomicAdd(&L.n, 1u);   // (at most V pairs: the row's slices' room together)
        a.pairs[c.rs0 * kSL + at] = make_uint2(key32(z), (uint32_t(t / kSL) << 16) | uint32_t(t % kSL));
    }
    __threadfence();   // (the stores, then the reads of this workgroup)
    __syncthreads();
    if (tid <= kMaxSlices) L.pre[tid] = tid == 0 ? 0u : L.n;   // (one list, from the row's first place)
    if (tid < kRanges) { L.lo[tid] = tid == 0 ? J : 1; L.hi[tid] = tid == 0 ? J : 0; }
    if (tid == 0) L.staged = 0u;
    __syncthreads();
}

// Smallest key of bin J (J < kNB): that of the smallest float z with 64 z >=
// anchor - J.  (|anchor| below 2^52, so anchor - J is exact.)
__device__ __forceinline__ uint32_t bin_low_key(double A, int J) {
    const double zl = (A - double(J)) / kPerUnit;
    const float zf = float(zl);
    return key32(zf) + (double(zf) < zl ? 1u : 0u);
}

// Bin J's pairs are the listed ones with keys in [kmin, kmax]; n of them.
struct BinSel {
    uint32_t kmin, kmax, n;
};
// Lists bin J's pairs if they are not.  All threads.
__device__ __forceinline__ BinSel select_bin(const RowCtx& c, FinishLds& L, int J) {
    bool have = false;
#pragma unroll
    for (int i = 0; i < kRanges; ++i) have = have || (L.lo[i] <= J && J <= L.hi[i]);
    if (!have) relist(c, L, J);   // (uniform)
    if (fabs(c.A) < 0x1p52) {
        BinSel b;
        b.kmin = J < kNB ? bin_low_key(c.A, J) : 0x00800000u;
        b.kmax = J > 0 ? bin_low_key(c.A, J - 1) - 1u : c.top;
        b.n = L.EXC[J + 1] - L.EXC[J];
        return b;
    }
    // (the bins' ends are not exact so far out: taken from the pairs)
    const int tid = threadIdx.x;
    __syncthreads();
    if (tid == 0) { L.kmin = 0xffffffffu; L.kmax = 0u; L.nbin = 0u; }
    __syncthreads();
    uint32_t mn = 0xffffffffu, mx = 0u, n = 0u;
    for (uint32_t i = tid; i < L.n; i += kT) {
        const uint32_t k = cand_key(c, L, i);
        if (bin_of_key(k, c.A) != J) continue;
        mn = min(mn, k);
        mx = max(mx, k);
        ++n;
    }
    mn = ~wave_max_u32(~mn);
    mx = wave_max_u32(mx);
    n = wave_sum_u32(n);
    if (lane_id() == 0 && n) { atomicMin(&L.kmin, mn); atomicMax(&L.kmax, mx); atomicAdd(&L.nbin, n); }
    __syncthreads();
    const BinSel b{L.kmin, L.kmax, L.nbin};
    __syncthreads();
    return b;
}

// Narrows the selected bin J (b) to the logit at which the cumulative count
// (mode 0: >= target) or mass (mode 1: >= target, mode 2: > target) over the
// bin's logits in order is reached; target counts from the bin's start.  The
// running sums said that it is reached in this bin: where rounding of the
// differences says otherwise, the bin's last logit.  All threads; the result in
// every thread.
__device__ __forceinline__ RHit narrow(const RowCtx& c, FinishLds& L, int J, const BinSel& b0, int mode, double target) {
    const int tid = threadIdx.x, lane = lane_id(), wave = tid / kWave;
    const bool massy = J < kNB;   // (the deep bin's logits carry no mass)
    const double unit = massy ? unit_of(c.A, c.z0, J) : 0.0;
    const uint32_t n = L.n;
    uint32_t klo = b0.kmin, khi = b0.kmax;
    RHit h{};
    if (b0.n == 0u) return h;
    h.cnt_key = b0.n;
    double tgt = target;
    while (klo < khi) {
        if (h.cnt_key <= uint32_t(kWave)) {
            // few enough for a wave: one key per lane, what lies above it counted
            // against all the others
            if (tid == 0) L.u0 = 0u;
            __syncthreads();
            for (uint32_t i = tid; i < n; i += kT) {
                const uint32_t k = cand_key(c, L, i);
                if (k >= klo && k <= khi) L.BC[atomicAdd(&L.u0, 1u)] = k;
            }
            __syncthreads();
            if (wave == 0) {
                const uint32_t m = min(L.u0, uint32_t(kWave)), k = lane < int(m) ? L.BC[lane] : 0u;
                const uint32_t wk = massy && k ? weight_fix(k) : 0u;
                uint32_t above = 0u, eq = 0u;
                unsigned long long fa = 0ull;
                for (uint32_t q = 0; q < m; ++q) {
                    const uint32_t kq = uint32_t(readlane_i(int(k), int(q))), wq = uint32_t(readlane_i(int(wk), int(q)));
                    above += kq > k ? 1u : 0u;
                    eq += kq == k ? 1u : 0u;
                    fa += kq > k ? wq : 0u;
                }
                const double incl = double(fa + (unsigned long long)eq * wk) * unit;
                const bool hit = k && (mode == 0 ? double(above + eq) >= tgt : mode == 1 ? incl >= tgt : incl > tgt);
                const uint32_t best = ballot(hit) ? wave_max_u32(hit ? k : 0u) : ~wave_max_u32(k ? ~k : 0u);
                if (k == best && lane == __builtin_ctzll(ballot(k == best))) {
                    L.u0 = best;
                    L.u1 = above;
                    L.u2 = eq;
                    L.f0 = fa;
                }
            }
            __syncthreads();
            const uint32_t best = L.u0, ca = L.u1, ce = L.u2;
            const unsigned long long f = L.f0;
            __syncthreads();
            if (!best) return h;   // (no pair in the range)
            h.cnt_before += ca;
            h.fix_before += f;
            h.cnt_key = ce;
            tgt -= mode == 0 ? double(ca) : double(f) * unit;
            klo = khi = best;
            break;
        }
        const uint32_t span = khi - klo;
        const int shift = max(0, 32 - __builtin_clz(span) - 8);
        if (tid < kDig) { L.BC[tid] = 0u; L.BF[tid] = 0ull; }
        __syncthreads();
        for (uint32_t i = tid; i < n; i += kT) {
            const uint32_t k = cand_key(c, L, i);
            if (k < klo || k > khi) continue;
            const uint32_t d = (k - klo) >> shift;
            atomicAdd(&L.BC[d], 1u);
            if (massy) atomicAdd(&L.BF[d], (unsigned long long)weight_fix(k));
        }
        __syncthreads();
        if (wave == 0) {
            // lane l: buckets 255 - 4l - q, highest keys first
            uint32_t bc[4];
            double bf[4];
            uint32_t tc = 0u;
            double tf = 0.0;   // (integers below 2^53: exact)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int b = kDig - 1 - 4 * lane - q;
                bc[q] = L.BC[b];
                bf[q] = double(L.BF[b]);
                tc += bc[q];
                tf += bf[q];
            }
            uint32_t cc = wave_incl_scan_u32(tc) - tc;
            double cf = wave_incl_scan_f64(tf) - tf;
            int fq = -1, lq = -1;   // the lane's first bucket that reaches the target, its last with logits
            uint32_t fc = 0u, lc = 0u;
            double ff = 0.0, lf = 0.0;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint32_t nc = cc + bc[q];
                const double nf = cf + bf[q];
                bool hit;
                if (mode == 0) hit = double(nc) >= tgt;
                else if (mode == 1) hit = nf * unit >= tgt;
                else hit = nf * unit > tgt;
                if (fq < 0 && bc[q] && hit) { fq = q; fc = cc; ff = cf; }
                if (bc[q]) { lq = q; lc = cc; lf = cf; }
                cc = nc;
                cf = nf;
            }
            const uint64_t m = ballot(fq >= 0), o = ballot(lq >= 0);
            if (lane == 0) L.u0 = o ? 1u : 0u;
            if (!m) { fq = lq; fc = lc; ff = lf; }
            if (o && lane == (m ? __builtin_ctzll(m) : 63 - __builtin_clzll(o))) {
                const uint32_t b = uint32_t(kDig - 1 - 4 * lane - fq);
                L.u1 = b;
                L.u2 = fc;
                L.u3 = bc[0] * (fq == 0) + bc[1] * (fq == 1) + bc[2] * (fq == 2) + bc[3] * (fq == 3);
                L.d0 = ff;
            }
        }
        __syncthreads();
        if (!L.u0) { __syncthreads(); return h; }   // (no pair in the range)
        const uint32_t b = L.u1;
        h.cnt_before += L.u2;
        h.fix_before += (unsigned long long)(L.d0);
        h.cnt_key = L.u3;
        tgt -= mode == 0 ? double(L.u2) : L.d0 * unit;
        const uint32_t nlo = klo + (b << shift);
        const uint32_t nhi = uint32_t(min(uint64_t(khi), uint64_t(nlo) + ((1ull << shift) - 1ull)));
        klo = nlo;
        khi = nhi;
        __syncthreads();
    }
    h.key = klo;
    h.found = true;
    if (massy) h.fix_key = weight_fix(klo);
    if (mode == 0) {
        h.rank = uint32_t(max(0.0, tgt - 1.0));
    } else {
        const double wk = double(h.fix_key) * unit;
        const uint32_t cnt = max(h.cnt_key, 1u);
        const double x = tgt / wk;
        double rr = mode == 1 ? ceil(x) - 1.0 : floor(x);
        rr = fmin(fmax(rr, 0.0), double(cnt - 1u));
        uint32_t r = uint32_t(rr);
        for (int it = 0; it < 4; ++it) {   // settle the rounding of the estimate
            const double at = double(r) * wk, up = double(r + 1u) * wk;
            if (r > 0u && (mode == 1 ? at >= tgt : at > tgt)) --r;
            else if (r + 1u < cnt && (mode == 1 ? up < tgt : up <= tgt)) ++r;
            else break;
        }
        h.rank = r;
    }
    return h;
}

// Count and fixed mass of the selected bin's logits with key >= kmin.
__device__ __forceinline__ void bin_above(const RowCtx& c, FinishLds& L, const BinSel& b, uint32_t kmin, uint32_t* cnt,
                          unsigned long long* fix, bool with_mass) {
    const int tid = threadIdx.x;
    if (tid == 0) { L.u0 = 0u; L.f0 = 0ull; }
    __syncthreads();
    uint32_t cn = 0u;
    unsigned long long fx = 0ull;
    for (uint32_t i = tid; i < L.n; i += kT) {
        const uint32_t k = cand_key(c, L, i);
        if (k >= kmin && k <= b.kmax) { ++cn; if (with_mass) fx += weight_fix(k); }
    }
    if (cn) { atomicAdd(&L.u0, cn); atomicAdd(&L.f0, fx); }
    __syncthreads();
    *cnt = L.u0;
    *fix = L.f0;
    __syncthreads();
}

// Logits of key k per slice (L.pcnt), its bin listed.
__device__ __forceinline__ void key_per_slice(const RowCtx& c, FinishLds& L, uint32_t key) {
    const int tid = threadIdx.x;
    if (tid < kMaxSlices) L.pcnt[tid] = 0u;
    __syncthreads();
    for (uint32_t i = tid; i < L.n; i += kT) {
        const uint2 e = cand(c, L, i);
        if (e.x == key) atomicAdd(&L.pcnt[e.y >> 16], 1u);
    }
    __syncthreads();
}

// The rank-th logit of key `key` in id order, its bin listed: its token.
__device__ __forceinline__ int32_t owner(const RowCtx& c, FinishLds& L, uint32_t key, uint32_t rank) {
    const int tid = threadIdx.x;
    key_per_slice(c, L, key);
    if (tid < kWave) {
        const uint32_t cnt = tid < kMaxSlices ? L.pcnt[tid] : 0u;
        const uint32_t incl = wave_incl_scan_u32(cnt);
        const uint64_t m = ballot(tid < c.S && incl > rank);
        if (tid == 0) L.u0 = m ? uint32_t(__builtin_ctzll(m)) : 0xffffffffu;
        if (m && tid == __builtin_ctzll(m)) L.u1 = rank - (incl - cnt);
    }
    if (tid < kSL / 32) L.OB[tid] = 0u;
    __syncthreads();
    const uint32_t os = L.u0;
    if (os == 0xffffffffu) { __syncthreads(); return -1; }
    for (uint32_t i = tid; i < L.n; i += kT) {
        const uint2 e = cand(c, L, i);
        if (e.x == key && (e.y >> 16) == os) atomicOr(&L.OB[(e.y & 0xffffu) >> 5], 1u << (e.y & 31u));
    }
    __syncthreads();
    const uint32_t word = tid < kSL / 32 ? L.OB[tid] : 0u;
    uint32_t tot = 0u;
    const uint32_t before = block_exclusive_scan_u32<kT>(uint32_t(__builtin_popcount(word)), L.uscan, &tot);
    const uint32_t want = L.u1;
    if (tid == 0) L.u2 = 0xffffffffu;
    __syncthreads();
    if (want >= before && want < before + uint32_t(__builtin_popcount(word))) {
        uint32_t m = word;
        for (uint32_t r = want - before; r > 0u; --r) m &= m - 1u;
        L.u2 = uint32_t(tid) * 32u + uint32_t(__builtin_ctz(m));
    }
    __syncthreads();
    const uint32_t off = L.u2;
    __syncthreads();
    return off == 0xffffffffu ? -1 : int32_t(os * kSL + off);
}

// Position order: (key desc, rank asc).  True when (k1, r1) comes after (k2, r2).
__device__ __forceinline__ bool after(uint32_t k1, uint32_t r1, uint32_t k2, uint32_t r2) {
    return k1 < k2 || (k1 == k2 && r1 > r2);
}

__global__ __launch_bounds__(kT) void wide_finish_kernel(WideArgs a) {
    __shared__ FinishLds L;
    const int row = blockIdx.x, tid = threadIdx.x, lane = lane_id(), wave = tid / kWave;
    const vi_row_params p = a.params[row];
    if (!full_row(p)) return;
    const WidePlan pl = a.plans[row];
    if (!pl.ok) return;   // (written by the plan launch)
    const int S = a.slices, V = a.vocabulary;
    const size_t rs0 = size_t(row) * S;
    const uint32_t top = pl.top, N = pl.n_valid;
    const double z0 = double(unkey32(top));
    const RowCtx c{&a, row, S, rs0, pl.A, z0, top, &p};

    // ---- the running sums and the listed pairs into LDS
    if (wave == 0) {
        const uint32_t n = lane < S ? a.npairs[rs0 + lane] : 0u;
        const uint32_t incl = wave_incl_scan_u32(n);
        if (lane < kMaxSlices) L.pre[lane] = incl - n;
        if (lane == kWave - 1) { L.pre[kMaxSlices] = incl; L.n = incl; L.staged = incl <= uint32_t(kCap) ? 1u : 0u; }
    }
    if (tid < kRanges) { L.lo[tid] = a.plans[row].lo[tid]; L.hi[tid] = a.plans[row].hi[tid]; }
    // (of the running sums only the planned ranges', a wave each, unless a range is
    // long; the rest when a decision falls outside them)
    const uint32_t* exc = a.exc + size_t(row) * (kNB + 2);
    const double* exm = a.exm + size_t(row) * (kNB + 1);
    bool whole = false;   // (uniform) every running sum is in LDS
#pragma unroll
    for (int i = 0; i < kRanges; ++i) whole = whole || pl.hi[i] - pl.lo[i] > kWave - 3;
    auto load_sum = [&](int J) {
        const int j = min(J, int(pl.bins));
        L.EXC[J] = J == kNB + 1 ? N : exc[j];
        if (J <= kNB) L.EXM[J] = exm[j];
    };
    auto load_whole = [&]() {
        for (int J = tid; J <= kNB + 1; J += kT) load_sum(J);
    };
    if (whole) {
        load_whole();
    } else {
#pragma unroll
        for (int i = 0; i < kRanges; ++i)
            if (wave == i + 1 && pl.lo[i] + lane <= min(pl.hi[i] + 1, kNB + 1) && pl.lo[i] <= pl.hi[i]) load_sum(pl.lo[i] + lane);
        if (tid == 0) load_sum(kNB);
    }
    __syncthreads();
    if (L.staged) {   // (a wave per slice at a time)
        for (int s = wave; s < S; s += kW) {
            const uint32_t b = L.pre[s], n = (s + 1 < S ? L.pre[s + 1] : L.n) - b;
            const uint2* src = a.pairs + (rs0 + s) * kSL;
            for (uint32_t i = lane; i < n; i += kWave) {
                const uint2 e = src[i];
                L.CK[b + i] = e.x;
                L.CI[b + i] = e.y;
            }
        }
        __syncthreads();
    }
    const BinSums B{L.EXC, L.EXM};
    const double s_all = L.EXM[kNB];
    auto fill = [&]() {   // (uniform)
        __syncthreads();
        load_whole();
        whole = true;
        __syncthreads();
    };
    auto need = [&](int J) {   // bin J's running sums in LDS
        bool in = whole;
#pragma unroll
        for (int i = 0; i < kRanges; ++i) in = in || (pl.lo[i] <= J && J <= pl.hi[i]);
        if (!in) fill();
    };
    // find_bin, looked for in the planned ranges first: the bin is inside a range
    // whose ends enclose the target
    auto find = [&](int mode, double t) -> int {
        if (!whole) {
#pragma unroll
            for (int i = 0; i < kRanges; ++i) {
                const int lo = pl.lo[i], hi = pl.hi[i];
                if (lo > hi || (mode != 0 && hi >= kNB)) continue;
                const double b = mode == 0 ? double(L.EXC[lo]) : L.EXM[lo], e = mode == 0 ? double(L.EXC[hi + 1]) : L.EXM[hi + 1];
                if (!(mode == 2 ? b <= t && e > t : b < t && e >= t)) continue;
                for (int J = lo; J <= hi; ++J) {
                    if (L.EXC[J + 1] == L.EXC[J]) continue;
                    if (mode == 0 ? double(L.EXC[J + 1]) >= t : mode == 1 ? L.EXM[J + 1] >= t : L.EXM[J + 1] > t) return J;
                }
            }
            fill();
        }
        return find_bin(B, mode, t);
    };
    auto unit = [&](int J) { return unit_of(pl.A, z0, J); };

    // ---- the top-k cap
    bool cap_on = false;
    uint32_t cap_key = 0u, cap_take = kTakeAll;
    double cap_mass = s_all;
    if (p.top_k > 0 && uint32_t(p.top_k) < N) {
        const int J = find(0, double(p.top_k));
        const RHit h = narrow(c, L, J, select_bin(c, L, J), 0, double(p.top_k) - double(L.EXC[J]));
        cap_on = true;
        cap_key = h.key;
        cap_take = h.rank + 1u;
        cap_mass = J < kNB ? L.EXM[J] + double(h.fix_before + (unsigned long long)cap_take * h.fix_key) * unit(J)
                           : s_all;
    }

    // ---- the min-p cut: the smallest key whose weight reaches min_p
    uint32_t minp_key = 0u;
    const bool minp_on = p.min_p > 0.0f;
    if (minp_on) minp_key = minp_cut(p, top, z0);   // (every wave alike)

    // ---- the top-p cut over the cap's mass
    bool topp_on = false;
    uint32_t topp_key = 0u, topp_take = kTakeAll;
    int topp_bin = -1;
    RHit topp_h{};
    if (p.top_p < 1.0f) {
        const double target = double(p.top_p) * cap_mass;
        const int J = find(1, target);
        if (J >= 0) {
            topp_h = narrow(c, L, J, select_bin(c, L, J), 1, target - L.EXM[J]);
            if (topp_h.found) { topp_on = true; topp_key = topp_h.key; topp_take = topp_h.rank + 1u; topp_bin = J; }
        }
    }

    // ---- the support's end: the earliest of the cap, the min-p cut and the
    // top-p cut (at least the first logit); its size and mass
    bool all = true;
    int src = 0;   // 1 cap, 2 min-p, 3 top-p, 4 forced first logit
    uint32_t ek = 0u, et = kTakeAll;
    auto consider = [&](uint32_t k, uint32_t t, int from) {
        if (all || k > ek || (k == ek && t < et)) { ek = k; et = t; all = false; src = from; }
    };
    if (cap_on) consider(cap_key, cap_take, 1);
    if (minp_on) consider(minp_key, kTakeAll, 2);
    if (topp_on) consider(topp_key, topp_take, 3);
    if (!all && ek > top) { ek = top; et = 1u; src = 4; }   // no logit passes min-p: the first one
    uint32_t n_sup = N;
    double s_n = s_all;
    if (src == 1) {
        n_sup = uint32_t(p.top_k);
        s_n = cap_mass;
    } else if (src == 3) {
        n_sup = L.EXC[topp_bin] + topp_h.cnt_before + topp_take;
        s_n = L.EXM[topp_bin] +
              double(topp_h.fix_before + (unsigned long long)topp_take * topp_h.fix_key) * unit(topp_bin);
    } else if (src == 2) {
        const int b = bin_of_key(ek, pl.A);
        need(b);
        uint32_t cn = 0u;
        unsigned long long fx = 0ull;
        bin_above(c, L, select_bin(c, L, b), ek, &cn, &fx, b < kNB);
        n_sup = L.EXC[b] + cn;
        s_n = L.EXM[b] + (b < kNB ? double(fx) * unit(b) : 0.0);
    } else if (src == 4) {
        n_sup = 1u;
        s_n = 1.0;
    }

    // ---- the draw: the first support logit whose inclusive cumulative mass
    // exceeds u x S_n (the last support logit when rounding passes them all)
    const double u = philox_uniform(p.seed, p.lane, p.position, 0u);
    const double target = u * s_n;
    const bool draw = a.draw_every > 0 && row % a.draw_every == a.draw_every - 1;   // (uniform)
    int dbin = draw ? find(2, target) : -1;
    uint32_t dkey = 0u, drank = 0u;
    bool dfound = !draw;
    if (dbin >= 0) {
        const RHit h = narrow(c, L, dbin, select_bin(c, L, dbin), 2, target - L.EXM[dbin]);
        if (h.found && (all || !after(h.key, h.rank, ek, et == kTakeAll ? 0xffffffffu : et - 1u))) {
            dfound = true;
            dkey = h.key;
            drank = h.rank;
        }
    }
    if (!dfound) {   // (the support's last logit)
        dbin = find(0, double(n_sup));
        if (dbin >= 0) {
            const RHit h = narrow(c, L, dbin, select_bin(c, L, dbin), 0, double(n_sup) - double(L.EXC[dbin]));
            dkey = h.key;
            drank = h.rank;
        }
    }
    const int32_t tok = !draw ? 0 : dbin >= 0 ? owner(c, L, dkey, drank) : -1;

    // ---- results; where the support cuts its last key's logits, the id of the
    // last one inside
    int32_t end_id = 0x7fffffff;
    if (a.want_bounds && !all && et != kTakeAll) {
        const int eb = bin_of_key(ek, pl.A);
        need(eb);
        (void)select_bin(c, L, eb);
        end_id = owner(c, L, ek, et - 1u);
    }
    if (tid == 0) {
        if (!draw) {   // (no token of this row is wanted)
            if (a.stats) {
                vi_sample_stats st{};
                st.flags = pl.flags;
                a.stats[row] = st;
            }
        } else if (tok < 0) {   // the bins disagree with the lists: cannot happen for consistent inputs
            write_row(a, row, -1, u, pl.flags | VI_FLAG_ERROR, 0u, 0u, 0.0);
        } else {
            write_row(a, row, tok, u, pl.flags, n_sup, N, s_n);
            if (a.record && a.pstate && tok < V) {   // (the passes over the logits, earlier launches, have read the state)
                const LaneState ls = lane_state(a.pstate + size_t(row) * a.pl.lane_bytes, a.pl);
                state_record_one(ls, a.pl, V, tok);
            }
        }
        if (a.want_bounds)
            a.bounds[row] = WideBound{z0, s_n, 1.0f / p.temperature, all ? 0u : ek, end_id,
                                      tok >= 0 && end_id >= 0 ? 1u : 0u};
    }
}

// Filtered distribution of the full-route rows: exp(z - z0) / S_n on the support,
// 0 elsewhere.  Bound by the memory (4 bytes read and 4 written per logit) and, for
// few rows, by one pass' latency: four consecutive logits per lane and one round
// per thread (23 x 151,936, 739-token histories: 13.4 us; with a cheaper exponential
// 11.4, and 18.7 with four rounds; 128 rows 45.4 and 51.0).
constexpr int kPT = 256;              // threads
constexpr int kPChunk = 4 * kPT;      // logits per workgroup
__global__ __launch_bounds__(kPT) void wide_probs_kernel(WideArgs a) {
    typedef float f32x4_t __attribute__((ext_vector_type(4)));
    typedef f32x4_t f32x4_any_t __attribute__((aligned(4)));
    const int row = blockIdx.y, V = a.vocabulary, i = int(blockIdx.x) * kPChunk + 4 * int(threadIdx.x);
    const vi_row_params p = a.params[row];
    if (!full_row(p) || i >= V) return;
    const WideBound bd = a.bounds[row];
    const WPen w = wpen(a, row, p);
    const int unrec = a.record && a.pstate ? a.tokens[row] : -1;
    const uint32_t* base = static_cast<const uint32_t*>(a.logits) + int64_t(row) * a.stride;
    float* out = a.probs + size_t(row) * size_t(a.probs_stride);
    const bool whole = i + 4 <= V;
    const uint4 v = whole ? load16(base + i) : make_uint4(0u, 0u, 0u, 0u);
    const uint32_t word = w.on ? w.bits[i >> 5] : 0u;   // (four logits share a presence word)
    const double inv_s = bd.valid ? 1.0 / bd.s_n : 0.0;
    auto prob = [&](uint32_t bits, int id) {
        bool bad = false;
        const float z = logit_z(w, p, bd.inv_t, id, bits, word, &bad, unrec);
        const uint32_t k = isnan(z) ? 0u : key32(z);
        const bool in = bd.valid && k && (k > bd.end_key || (k == bd.end_key && id <= bd.end_id));
        return in ? float(exp(double(z) - bd.z0) * inv_s) : 0.0f;
    };
    if (whole) {
        f32x4_t q;
        q[0] = prob(v.x, i);
        q[1] = prob(v.y, i + 1);
        q[2] = prob(v.z, i + 2);
        q[3] = prob(v.w, i + 3);
        *reinterpret_cast<f32x4_any_t*>(out + i) = q;
    } else {   // (up to three logits past the row's last four)
        for (int j = i; j < V; ++j) out[j] = prob(base[j], j);
    }
}

inline int wide_slices(int vocabulary) { return (vocabulary + kSL - 1) / kSL; }
inline int bitmap_words(int vocabulary) { return int(align_up((size_t(vocabulary) + 31) / 32, 4)); }

}  // namespace

bool wide_supported(int vocabulary, int64_t stride) {
    return vocabulary > 0 && vocabulary <= kMaxSlices * kSL && stride >= vocabulary;
}

size_t wide_workspace(int rows, int vocabulary) {
    if (rows <= 0 || vocabulary <= 0) return 0;
    const size_t rs = size_t(rows) * size_t(wide_slices(vocabulary));
    return align_up(rs * sizeof(WideHead), 256) + align_up(rs * kNB * 8, 256) +
           align_up(size_t(rows) * sizeof(WidePlan), 256) + align_up(size_t(rows) * (kNB + 2) * 4, 256) +
           align_up(size_t(rows) * (kNB + 1) * 8, 256) + align_up(rs * 4, 256) + align_up(rs * kSL * 8, 256) +
           align_up(size_t(rows) * size_t(bitmap_words(vocabulary)) * 4, 256) +
           align_up(size_t(rows) * sizeof(WideBound), 256) + 256;
}

vi_status launch_wide(const SampleArgs& s, unsigned char* ws, size_t ws_bytes, uint2* hash, int hash_shift,
                      int hash_slots, uint32_t* row_flags, hipStream_t stream) {
    if (!wide_supported(s.vocabulary, s.stride) || reinterpret_cast<uintptr_t>(s.logits) % 4) return VI_ERR_UNSUPPORTED;
    WideArgs a{};
    a.slices = wide_slices(s.vocabulary);
    const size_t rs = size_t(s.rows) * size_t(a.slices);
    Carver c(ws, ws_bytes);
    a.heads = c.take<WideHead>(rs);
    a.hist = c.take<unsigned long long>(rs * kNB);
    a.plans = c.take<WidePlan>(size_t(s.rows));
    a.exc = c.take<uint32_t>(size_t(s.rows) * (kNB + 2));
    a.exm = c.take<double>(size_t(s.rows) * (kNB + 1));
    a.npairs = c.take<uint32_t>(rs);
    a.pairs = c.take<uint2>(rs * kSL);
    a.words = bitmap_words(s.vocabulary);
    a.hbits = c.take<uint32_t>(size_t(s.rows) * size_t(a.words));
    a.bounds = c.take<WideBound>(size_t(s.rows));
    if (!c.ok) return VI_ERR_WORKSPACE;
    a.logits = s.logits; a.rows = s.rows; a.vocabulary = s.vocabulary; a.stride = s.stride;
    a.params = s.params;
    if (s.pstate) {
        a.pstate = s.pstate; a.pl = s.playout; a.record = s.record;
    } else if (hash && s.histories && s.offsets) {
        a.histories = s.histories; a.offsets = s.offsets; a.max_history = s.max_history;
        a.hash = hash; a.hash_shift = hash_shift; a.hash_slots = hash_slots; a.row_flags = row_flags;
    }
    a.tokens = s.tokens; a.uniforms = s.uniforms; a.probs = s.probs; a.probs_stride = s.probs_stride;
    a.stats = s.stats;
    if (s.full_out) a.bounds = s.full_out->bounds;
    a.draw_every = s.full_out ? s.full_out->draw_every : 1;
    a.want_bounds = (s.probs || s.full_out) ? 1 : 0;
    if (a.hash) hipLaunchKernelGGL(wide_history_kernel, dim3(s.rows), dim3(kT), 0, stream, a);
    const bool pen = a.pstate || a.hash;
    const dim3 slices(a.slices, s.rows);
    if (pen) hipLaunchKernelGGL(wide_hist_kernel<true>, slices, dim3(kT), 0, stream, a);
    else hipLaunchKernelGGL(wide_hist_kernel<false>, slices, dim3(kT), 0, stream, a);
    hipLaunchKernelGGL(wide_plan_kernel, dim3(s.rows), dim3(kT), 0, stream, a);
    if (pen) hipLaunchKernelGGL(wide_gather_kernel<true>, slices, dim3(kT), 0, stream, a);
    else hipLaunchKernelGGL(wide_gather_kernel<false>, slices, dim3(kT), 0, stream, a);
    hipLaunchKernelGGL(wide_finish_kernel, dim3(s.rows), dim3(kT), 0, stream, a);
    vi_status st = launch_status();
    if (st != VI_OK || !s.probs) return st;
    hipLaunchKernelGGL(wide_probs_kernel, dim3((s.vocabulary + kPChunk - 1) / kPChunk, s.rows), dim3(kPT), 0, stream, a);
    return launch_status();
}

}  // namespace vi
