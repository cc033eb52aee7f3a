// sample_stream.hip — full-vocabulary rows of the batched sampler, 16-bit
// logits (temperature > 0, top_k = 0 or > 64): penalties, temperature, top-k /
// min-p / top-p over the whole vocabulary and the Philox inverse-CDF draw.
// Every 16-bit full-vocabulary row comes here, at any row alignment: the sampler's
// (tokens, uniforms, stats, recording into penalty states, on request the
// filtered distribution) and verification's (the distributions' bounds).
// (Rows with an odd vocabulary, probabilities or bounds had kernels of their own,
// which named the support's end by ranks.  This way / that way, us per call:
// verification of 8 lanes x 16 drafts over 248,320 tokens, bf16 and fp16, 127 / 229;
// 24 x 65,537 fp16 with probabilities 68 / 93; 56 x 66,181 bf16, odd, no penalties
// 29.7 / 28.3; 2 x 248,319 bf16, odd, 500-token histories 37.6 / 33.3: few odd rows
// pay for the history view's launch.)
//
// Key fact: bf16 / fp16 logits, and penalized logits stored back in the same
// dtype, take one of 65,536 bit patterns, and z = x' * (1/T) is a strictly
// monotone function of the pattern's order key (for T <= 65,536; +0 and -0
// share z = 0).  The multiset of z over a row is a count histogram over
// patterns; every truncation and the draw are prefix sums over the occupied
// patterns in key order, with one exp per occupied pattern, not per token.
//
// Stream launch (stream_kernel).  A row is cut into P parts of at most 65,504
// tokens, so a part's count of one pattern fits 16 bits.  Persistent
// workgroups of 1024 threads (one per CU: the histogram takes 128 KB of LDS)
// take the parts of their XCD's rows in a fixed order, with the next part's
// first logits in flight while the current part finishes.  Each wave owns one
// 16-byte vector per lane and round (512 consecutive tokens), four rounds in
// flight per thread; no workgroup barrier runs inside the stream.  Every token
// adds one to its raw pattern's u16 count (histogram word = pattern & 0x7fff,
// half = sign).  Where the row has penalties, the wave stages its vectors in
// LDS, lists its history tokens (the presence bitmap's byte of each vector)
// and handles them 64 at a time, one per lane: the count moves from the raw
// pattern to the penalized one (occurrence count 1).  Tokens seen more than
// once (the repeat list) are corrected at the end of the part: one count moves
// from the count-1 pattern to the count-c one.  Each thread then owns 32
// histogram words (a group: 32 positive and 32 negative keys); the non-empty
// groups are stored at their place in the part's table, with occupancy bitmaps
// of the groups holding positive and negative patterns, and the words are cleared.
//
// Merge launch (merge_kernel, one workgroup per row, on the XCD whose L2 holds
// the row's tables).  The row's occupied groups are summed over its parts per
// key; each occupied key is weighed exp(z - z0) once; prefix sums over 32-key
// blocks in descending key order (2^-40 fixed point: exact, independent of
// order) locate the top-k cap, the min-p and top-p cuts and the draw, each
// resolved inside its block; the part holding the drawn key's rank is read
// again to name the token (id order among equal keys), a history token's
// penalized key recognised from its raw key through the preimage of the drawn
// key under the (monotone) penalty.  A caller that wants the filtered distribution
// gets the support's end as a key and the last id of that key inside, named the
// same way (a support is then a comparison per logit, with no ranks to count).
//
// Probabilities (probs_kernel, then repeat_probs_kernel for the tokens seen more
// than once): every logit's penalized key compared with the support's end.
//
// Roofline: HBM; V x 2 bytes of logits per row, plus the presence bitmap
// (V / 8 bytes) and the repeat list where the row has penalties.
#include <math.h>

#include <algorithm>

#include "keys16.h"
#include "penalty_state.h"
#include "vi_device.h"
#include "vi_internal.h"

namespace vi {
namespace {

constexpr int kT = 1024;                 // threads per workgroup
constexpr int kW = kT / kWave;           // waves per workgroup
constexpr int kHW = 32768;               // histogram words
constexpr int kGroups = 1024;            // 32-word groups (one per thread when published)
constexpr int kGW = 32;
constexpr int kDepth = 4;                // rounds of logits in flight per thread
constexpr int kXcds = 8;
constexpr int kRepPF = 2;                // repeat-list entries prefetched per thread
constexpr int kMaxParts = 16;            // parts per row
constexpr int kMaxVocabulary = 524288;   // (every full-vocabulary route's limit)
constexpr int kMaxPartLen = 65504;       // tokens per part (a multiple of 32 below 65,536)
constexpr int kPub = 64;                 // words per part header: the occupancy bitmaps, by sign
// Place of group g in an occupancy bitmap of 32 words: byte g & 127, bit g >> 7
// (the order in which a publishing thread meets its groups).
struct GroupBit {
    uint32_t word, shift;
};
__device__ __forceinline__ GroupBit group_bit(uint32_t g) { return GroupBit{(g & 127u) >> 2, ((g & 3u) << 3) | (g >> 7)}; }
constexpr uint32_t kTakeAll = 0xffffffffu;
constexpr double kFix = 0x1p40;          // fixed-point scale of the masses (w <= 1, counts <= 2^20)

// Stream LDS (bytes): H, the histogram (u16 counts in pairs: word p & 0x7fff,
// low half sign 0, high half sign 1); the waves' staged vectors; their lists
// of history tokens (u8 offsets inside the wave's 512 tokens; the lists of
// lanes 32..63 continue those of lanes 0..31, their offsets 256 higher).
constexpr int kOffH = 0;
constexpr int kOffStage = kOffH + 4 * kHW;
constexpr int kOffList = kOffStage + 16 * kT;
constexpr int kLds = kOffList + 8 * kT;
static_assert(kLds == 155648, "LDS map");

// Merge LDS (bytes).  The per-key counts of the row's occupied groups take
// what the fixed arrays leave (more groups than that are summed again from the
// parts' tables when needed).
constexpr int kOffMBits = 0;                          // u32[kMaxParts][32]: each part's occupied groups
constexpr int kOffMOcc = kOffMBits + 4 * 32 * kMaxParts;   // u32[3][32]: occupied in any part, by sign too
constexpr int kOffMSlot = kOffMOcc + 384;             // u16[1024]: slot of group g
constexpr int kOffMGroupOf = kOffMSlot + 2048;        // u16[1024]: group of slot s
constexpr int kOffMBcnt = kOffMGroupOf + 2048;        // u32[2048]: logits per 32-key block
constexpr int kOffMBmass = kOffMBcnt + 8192;          // u64[2048]: block masses, fixed point
constexpr int kOffMCab = kOffMBmass + 16384;          // u32[2048]: logits in the blocks above
constexpr int kOffMMab = kOffMCab + 8192;             // u64[2048]: mass of the blocks above
constexpr int kOffMFlip = kOffMMab + 16384;           // u32[2048]: rescan flips (65,536 bits)
constexpr int kOffMKeys = kOffMFlip + 8192;           // uint4[slot][16]: (lo, hi) counts of word pairs; then (the
                                                      // rescan) uint2[2048]: the owner part's repeat entries
constexpr int kMLds = 155648;
constexpr uint32_t kSlotCap = (kMLds - kOffMKeys) / (16 * 16);
constexpr uint32_t kNoSlot = 0xffffu;    // slot of a group no part holds
static_assert(kOffMKeys % 16 == 0 && kSlotCap >= 256, "merge map");

struct StreamArgs {
    const void* logits;
    int rows, vocabulary, parts, part_len, grid, xcd;
    int64_t stride;
    const vi_row_params* params;
    // penalty views: lane states, or the history prepass's bitmaps and lists
    const unsigned char* pstate;
    PenaltyLayout pl;
    const uint32_t* hb1;       // [rows][hwords] presence bitmaps (history route)
    const uint2* hlist;        // [rows][hcap] (token, count >= 2)
    const uint32_t* hhead;     // [rows][2]: repeat entries, flags
    int hwords, hcap;
    int record;
    int32_t* tokens;
    double* uniforms;
    float* probs;
    int64_t probs_stride;
    vi_sample_stats* stats;
    FullBound* bounds;         // [rows] (or null): the rows' filtered distributions
    int draw_every;            // rows whose token is drawn: every one (1), every n-th (row % n == n - 1), none (0)
    int row0;                  // row 0's number in the call (a call of very many rows takes several launches)
    // the parts' tables: header (the occupied groups' bitmaps, by sign) and
    // the occupied groups' 32 words at their place
    uint32_t* ppub;            // [rows * parts][kPub]
    uint4* pwords;             // [rows * parts][kGroups][8]
};

// threadIdx.x behind an empty asm: address arithmetic on it stays in the loop
// that uses it instead of being hoisted and held across the persistent loop
__device__ __forceinline__ int opaque_tid() {
    int t = int(threadIdx.x);
    asm volatile("" : "+v"(t));
    return t;
}

// A workgroup barrier that orders LDS only (the stream's loads stay in flight).
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}
// Exclusive prefix sum of v over the workgroup (total in *total), its barriers
// LDS-only: loads in flight stay in flight.
__device__ __forceinline__ uint32_t block_scan_lds(uint32_t v, uint32_t* tmp, uint32_t* total) {
    const int lane = lane_id(), wave = threadIdx.x / kWave;
    const uint32_t x = wave_incl_scan_u32(v);
    if (lane == kWave - 1) tmp[wave] = x;
    lds_barrier();
    if (wave == 0) {
        const uint32_t t = lane < kW ? tmp[lane] : 0u;
        const uint32_t it = wave_incl_scan_u32(t);
        if (lane < kW) tmp[lane] = it - t;
        if (lane == kW - 1) tmp[kW] = it;
    }
    lds_barrier();
    const uint32_t r = tmp[wave] + x - v;
    *total = tmp[kW];
    lds_barrier();
    return r;
}
// s_waitcnt vmcnt(0): every vector memory access of the wave complete.
__device__ __forceinline__ void vm_drain() { __builtin_amdgcn_s_waitcnt(0x0f70); }
__device__ __forceinline__ void wave_lds_fence() { __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront", "local"); }

__device__ __forceinline__ void lds_add(uint32_t* p, uint32_t v) {
    __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
// +1 / -1 at a 16-bit pattern's histogram half
__device__ __forceinline__ void hist_inc(uint32_t* H, uint32_t pat) {
    lds_add(&H[pat & 0x7fffu], (pat & 0x8000u) ? 0x10000u : 1u);
}
__device__ __forceinline__ void hist_dec(uint32_t* H, uint32_t pat) {
    lds_add(&H[pat & 0x7fffu], (pat & 0x8000u) ? 0xffff0000u : 0xffffffffu);
}

__device__ __forceinline__ uint32_t readlane_u(uint32_t v, int l) { return uint32_t(__builtin_amdgcn_readlane(int(v), l)); }
__device__ __forceinline__ uint64_t readlane_u64(uint64_t v, int l) {
    return uint64_t(readlane_u(uint32_t(v), l)) | (uint64_t(readlane_u(uint32_t(v >> 32), l)) << 32);
}
// Inclusive prefix sums of u64 values over the wave (DPP, carries by hand).
__device__ __forceinline__ uint64_t wave_incl_scan_u64(uint64_t x) {
    auto step = [](uint64_t v, auto dpp) {
        const uint64_t o = uint64_t(dpp(uint32_t(v))) | (uint64_t(dpp(uint32_t(v >> 32))) << 32);
        return v + o;
    };
    x = step(x, [](uint32_t u) { return dpp_u32<0x111, 0xf, true>(u); });
    x = step(x, [](uint32_t u) { return dpp_u32<0x112, 0xf, true>(u); });
    x = step(x, [](uint32_t u) { return dpp_u32<0x114, 0xf, true>(u); });
    x = step(x, [](uint32_t u) { return dpp_u32<0x118, 0xf, true>(u); });
    x = step(x, [](uint32_t u) { return dpp_u32<0x142, 0xa, false>(u); });
    x = step(x, [](uint32_t u) { return dpp_u32<0x143, 0xc, false>(u); });
    return x;
}

// ------------------------------------------------------------------ items
struct Item {
    int row, part, s0, n, nvec, rounds;
};
__device__ __forceinline__ Item part_geo(const StreamArgs& a, int row, int part) {
    Item it;
    it.row = row;
    it.part = part;
    it.s0 = part * a.part_len;
    it.n = min(a.part_len, a.vocabulary - it.s0);
    it.nvec = it.n >> 3;   // (up to seven logits past the last vector)
    it.rounds = max(1, (it.nvec + kT - 1) / kT);
    return it;
}
// Parts of XCD x (the rows x, x + 8, ... when the launch is XCD-aware, else
// every row), in row-major order; the workgroups of the XCD take every nx-th.
__device__ __forceinline__ int xcd_rows(const StreamArgs& a, int x) { return a.xcd ? (a.rows - x + kXcds - 1) / kXcds : a.rows; }
__device__ __forceinline__ int xcd_wgs(const StreamArgs& a, int x) { return a.xcd ? (a.grid - x + kXcds - 1) / kXcds : a.grid; }
__device__ __forceinline__ Item item_at(const StreamArgs& a, int x, int q) {
    const int r = q / a.parts;
    return part_geo(a, a.xcd ? x + kXcds * r : r, q % a.parts);
}
__device__ __forceinline__ bool stream_row(const vi_row_params& p) { return !topk_route(p); }

// A row's penalty inputs.  flags: the failures of the lane's state or history,
// which concern only the rows that take penalties from it (none without `pen`).
struct PenView {
    const unsigned char* b1;
    const uint2* list;
    uint32_t nrep, flags;
    bool pen;
};
__device__ __forceinline__ PenView pen_view(const StreamArgs& a, int row, const vi_row_params& p) {
    PenView v{};
    if (a.pstate) {
        const unsigned char* st = a.pstate + size_t(row) * a.pl.lane_bytes;
        const PenaltyHeader* h = reinterpret_cast<const PenaltyHeader*>(st);
        v.b1 = st + a.pl.off_b1;
        v.list = reinterpret_cast<const uint2*>(st + a.pl.off_list);
        v.nrep = min(h->nrep, uint32_t(a.pl.slots));
        v.pen = penalties_active(p);
        v.flags = v.pen ? h->flags & (VI_FLAG_BAD_HISTORY | VI_FLAG_ERROR) : 0u;
    } else if (a.hb1) {
        v.b1 = reinterpret_cast<const unsigned char*>(a.hb1 + size_t(row) * a.hwords);
        v.list = a.hlist + size_t(row) * a.hcap;
        v.nrep = a.hhead[2 * row];
        v.pen = penalties_active(p);
        v.flags = v.pen ? a.hhead[2 * row + 1] : 0u;
    }
    return v;
}

// Penalized pattern of a 16-bit pattern seen `count` times; non-finite
// patterns stay as they are (they never reach the distribution).
template <int DT>
__device__ __forceinline__ uint32_t pen_pattern(uint32_t raw, uint32_t count, const vi_row_params& p, float inv_r,
                                                bool rep_fast) {
    if (!Elem<DT>::finite_bits(raw)) return raw;
    return penalize_fast<DT>(raw, count, p, inv_r, rep_fast) & 0xffffu;
}

// ------------------------------------------------------------------ weights
// exp(z(key) - z0): z in fp32 as the oracle forms it, the difference in fp64
// (exact), then 2^(d log2 e) as the hardware exp2 of the exponent rounded to
// fp32, corrected to first order by the rounding's remainder (relative error
// about one fp32 ulp).
template <int DT>
__device__ __forceinline__ double key_weight(uint32_t key, float inv_t, double z0) {
    const double d = double(key_z<DT>(key, inv_t)) - z0;
    const double a = d * 1.4426950408889634;
    const float ah = float(a);
    const float al = float(a - double(ah));
    const float e = __builtin_amdgcn_exp2f(ah);
    return ah < -125.0f ? 0.0 : double(e) * (1.0 + double(al) * 0.6931471805599453);
}
__device__ __forceinline__ uint64_t fixed_mass(uint32_t count, double w) {
    return uint64_t(llrint(double(count) * w * kFix));
}

// Keys of histogram word w: low half (sign 0) -> 0x8000 + w, high half (sign 1)
// -> 0x7fff - w.  Valid: a finite pattern whose z is finite (kmin..kmax).
template <int DT>
__device__ __forceinline__ bool key_valid(uint32_t key, uint32_t kmin, uint32_t kmax) {
    return key >= kmin && key <= kmax;
}

// ------------------------------------------------------------------ stream
constexpr int kMaxItems = 1024;          // parts one workgroup can take

struct StreamShared {
    int items[kMaxItems];                // the workgroup's parts (indices among its XCD's), in order
    uint32_t scan[kW + 1];
    // the part's groups holding positive and negative patterns (GroupBit's order)
    unsigned char occb[2][kGroups / 8];
};

// The presence bytes (one per vector) of a row from token s0: the lane
// state's or the history prepass's bitmap; without either, any readable byte
// per vector (the logits; the byte is then ignored).
__device__ __forceinline__ const unsigned char* presence_at(const StreamArgs& a, int row, int s0,
                                                            const unsigned char* vb) {
    if (a.pstate) return a.pstate + size_t(row) * a.pl.lane_bytes + a.pl.off_b1 + (s0 >> 3);
    if (a.hb1) return reinterpret_cast<const unsigned char*>(a.hb1 + size_t(row) * a.hwords) + (s0 >> 3);
    return vb;
}

// One part as the stream sees it: geometry, logits, presence bytes, repeat
// list, penalty parameters.
struct PartView {
    Item it;
    const unsigned char* vb;
    const unsigned char* pb;
    const uint2* list;
    uint32_t nrep;
    bool pen;
    float rep, pres, freq;
};

// PB: the call has presence bytes (lane states or the history prepass).
template <int DT, bool PB>
__global__ __launch_bounds__(kT) void stream_kernel(StreamArgs a) {
    __shared__ __attribute__((aligned(16))) unsigned char lds[kLds];
    __shared__ StreamShared sh;
    uint32_t* H = reinterpret_cast<uint32_t*>(lds + kOffH);
    const int tid = threadIdx.x, lane = lane_id(), wave = tid / kWave;
    const int w = blockIdx.x;
    const int x = a.xcd ? w % kXcds : 0;
    const int wx = a.xcd ? w / kXcds : w;   // index among the XCD's workgroups
    const int nx = xcd_wgs(a, x), items = xcd_rows(a, x) * a.parts;

    // the histogram starts empty (every part leaves it so)
#pragma unroll
    for (int q = 0; q < kHW / 4 / kT; ++q)
        reinterpret_cast<uint4*>(H)[q * kT + tid] = make_uint4(0u, 0u, 0u, 0u);
    // the workgroup's parts: wx, wx + nx, ... of its XCD's (at most kMaxItems:
    // the launch checks), rows the kernel does not serve passed over
    int nitems;
    {
        const int ncand = wx < items ? (items - 1 - wx) / nx + 1 : 0;
        const int q = wx + tid * nx;
        const uint32_t ok = (tid < ncand && stream_row(a.params[item_at(a, x, q).row])) ? 1u : 0u;
        uint32_t tot;
        const uint32_t pos = block_scan_lds(ok, sh.scan, &tot);
        if (ok) sh.items[pos] = q;
        nitems = int(tot);
        lds_barrier();
    }
    if (nitems == 0) return;

    // A part's description.  The penalty parameters, the repeat list's length
    // and (a part ahead) its first entries come in through vector loads (the
    // address laundered into a VGPR): an outstanding scalar load would hold up
    // every LDS wait of the stream in between.
    auto view = [&](int k) -> PartView {
        PartView c;
        const int q = __builtin_amdgcn_readfirstlane(sh.items[k]);
        c.it = item_at(a, x, q);
        c.vb = static_cast<const unsigned char*>(a.logits) + 2 * (size_t(c.it.row) * size_t(a.stride) + size_t(c.it.s0));
        if (c.it.nvec == 0) c.vb = reinterpret_cast<const unsigned char*>(a.params);   // (no whole vector: read, never used)
        c.pb = presence_at(a, c.it.row, c.it.s0, c.vb);
        int z = 0;
        asm volatile("" : "+v"(z));
        const vi_row_params* pp = a.params + c.it.row + z;
        c.rep = pp->repetition_penalty;
        c.pres = pp->presence_penalty;
        c.freq = pp->frequency_penalty;
        c.pen = false;   // (settle)
        const uint32_t* nr;
        if (a.pstate) {
            const unsigned char* st = a.pstate + size_t(c.it.row) * a.pl.lane_bytes;
            c.list = reinterpret_cast<const uint2*>(st + a.pl.off_list);
            nr = &reinterpret_cast<const PenaltyHeader*>(st)->nrep;
        } else if (a.hb1) {
            c.list = a.hlist + size_t(c.it.row) * a.hcap;
            nr = a.hhead + 2 * c.it.row;
        } else {
            c.list = nullptr;
            nr = reinterpret_cast<const uint32_t*>(a.params);
        }
        c.nrep = nr[z];
        return c;
    };
    // the loaded fields made uniform (after their loads have landed)
    auto settle = [&](PartView& c) {
        auto rf = [](float f) { return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, f))); };
        c.rep = rf(c.rep);
        c.pres = rf(c.pres);
        c.freq = rf(c.freq);
        c.pen = PB && (c.rep != 1.0f || c.pres != 0.0f || c.freq != 0.0f);
        c.nrep = uint32_t(__builtin_amdgcn_readfirstlane(int(c.nrep)));
        if (a.pstate) c.nrep = min(c.nrep, uint32_t(a.pl.slots));
    };
    // The lane's repeat-list entries of a part (kRepPF of them), requested a
    // part ahead, whatever the list's length (read within the list's
    // capacity; entries past the length are dropped when used).
    const uint32_t list_cap = a.pstate ? uint32_t(a.pl.slots) : uint32_t(max(a.hcap, 1));
    auto load_re = [&](const PartView& c, uint2* e) {
#pragma unroll
        for (int j = 0; j < kRepPF; ++j) {
            e[j] = make_uint2(0u, 0u);
            if (PB) e[j] = c.list[min(uint32_t(j * kT + tid), list_cap - 1u)];
        }
    };

    PartView cur = view(0);
    bool has_next = nitems > 1;
    PartView nxt = has_next ? view(1) : cur;
    uint2 re[kRepPF];   // the current part's entries (those of the next once its corrections are made)
    load_re(cur, re);

    // Rounds in flight: a part's rounds are padded to whole turns of the ring
    // (the padding rounds count nothing), so round rho of every part sits in
    // slot rho % kDepth.  The round kDepth ahead is requested once the current
    // one is used: the current part's, the next part's, or (past the last
    // part) the last vector again, never used.  Every round issues exactly one
    // vector load (and one presence load), straight-line, so the waits count
    // on the loads' order.
    uint4 rv[kDepth];
    uint32_t rb[kDepth] = {};
    auto padded = [](int r) { return (r + kDepth - 1) & ~(kDepth - 1); };
    auto issue = [&](uint4& dv, uint32_t& db, int rel) {   // rel: rounds after the current part's first
        const int Rp = padded(cur.it.rounds);
        const bool in_nxt = rel >= Rp && has_next;
        const unsigned char* vb = in_nxt ? nxt.vb : cur.vb;
        const unsigned char* pb = in_nxt ? nxt.pb : cur.pb;
        const int nv = in_nxt ? nxt.it.nvec : cur.it.nvec;
        const int rr = in_nxt ? rel - Rp : rel;
        const int v = max(min(rr * kT + opaque_tid(), nv - 1), 0);
        dv = load16(vb + size_t(v) * 16);
        // the dword holding the vector's presence byte (a 32-bit load result
        // stays in its register across the loop; a byte would be re-extended)
        if (PB) db = *reinterpret_cast<const uint32_t*>(pb + (v & ~3));
    };
#pragma unroll
    for (int s = 0; s < kDepth; ++s) issue(rv[s], rb[s], s);
    settle(cur);

    for (int k = 0;;) {
        vi_row_params p{};   // the fields the penalties read
        p.repetition_penalty = cur.rep;
        p.presence_penalty = cur.pres;
        p.frequency_penalty = cur.freq;
        const float inv_r = rep_inverse(p);
        const bool rep_fast = rep_fast_ok(p);
        const bool pen = cur.pen;
        const Item it = cur.it;
        const uint16_t* row16 = reinterpret_cast<const uint16_t*>(static_cast<const unsigned char*>(a.logits) +
                                                                  2 * size_t(it.row) * size_t(a.stride));
        auto in_part = [&](uint2 e) { return e.y >= 2u && int(e.x) >= it.s0 && int(e.x) < it.s0 + it.n; };
        // one count of a repeated token from its count-1 pattern to its count-c one
        auto correct = [&](uint2 e, uint32_t raw) {
            const uint32_t p1 = pen_pattern<DT>(raw, 1u, p, inv_r, rep_fast);
            const uint32_t pc = pen_pattern<DT>(raw, e.y, p, inv_r, rep_fast);
            if (p1 != pc) { hist_dec(H, p1); hist_inc(H, pc); }
        };
        uint32_t rraw[kRepPF] = {};

        // ---- the stream.  The repeat entries' logits are gathered at the
        // start of the last turn but one and their corrections made at the
        // start of the last turn (counts are added and taken in any order: the
        // 32-bit word holds their sum).
        const int Rp = padded(it.rounds);
        const int gather_turn = max(0, Rp - 2 * kDepth), corr_turn = Rp - kDepth;
        uint4* stage = reinterpret_cast<uint4*>(lds + kOffStage) + wave * kWave;
        const uint16_t* stage16 = reinterpret_cast<const uint16_t*>(stage);
        unsigned char* list = lds + kOffList + wave * 512;
        for (int gb = 0; gb < Rp; gb += kDepth) {
            if (pen && gb == gather_turn) {
#pragma unroll
                for (int j = 0; j < kRepPF; ++j) {
                    if (uint32_t(j * kT + tid) >= cur.nrep) re[j].y = 0u;
                    rraw[j] = in_part(re[j]) ? uint32_t(row16[re[j].x]) : 0u;
                }
            }
            if (pen && gb == corr_turn) {
#pragma unroll
                for (int j = 0; j < kRepPF; ++j)
                    if (in_part(re[j])) correct(re[j], rraw[j]);
            }
            if (gb == corr_turn && has_next) load_re(nxt, re);   // (in place: no copy waits for it)
#pragma unroll
            for (int s = 0; s < kDepth; ++s) {
                const int rho = gb + s;
                const uint4 v = rv[s];
                const bool valid = rho * kT + tid < it.nvec;   // (none on a padding round)
                const uint32_t b = (PB && valid) ? (rb[s] >> (8 * (tid & 3))) & 0xffu : 0u;
                if (valid) {
                    hist_inc(H, v.x & 0xffffu); hist_inc(H, v.x >> 16);
                    hist_inc(H, v.y & 0xffffu); hist_inc(H, v.y >> 16);
                    hist_inc(H, v.z & 0xffffu); hist_inc(H, v.z >> 16);
                    hist_inc(H, v.w & 0xffffu); hist_inc(H, v.w >> 16);
                }
                if (pen) {   // (uniform) the history tokens of the wave's 512 tokens
                    stage[lane] = v;
                    const uint32_t n = uint32_t(__builtin_popcount(b));
                    const uint32_t incl = wave_incl_scan_u32(n);
                    const uint32_t N = readlane_u(incl, kWave - 1), NA = readlane_u(incl, 31);
                    if (N) {
                        uint32_t pos = incl - n;
                        const uint32_t base = uint32_t(lane) * 8u;
#pragma unroll
                        for (int j = 0; j < 8; ++j) {
                            if ((b >> j) & 1u) {
                                list[pos] = uint8_t(base + uint32_t(j));
                                ++pos;
                            }
                        }
                        wave_lds_fence();
                        for (uint32_t q0 = 0; q0 < N; q0 += kWave) {
                            const uint32_t q = q0 + uint32_t(lane);
                            if (q < N) {
                                const uint32_t off = uint32_t(list[q]) + (q >= NA ? 256u : 0u);
                                const uint32_t raw = stage16[off];
                                const uint32_t pb = pen_pattern<DT>(raw, 1u, p, inv_r, rep_fast);
                                if (pb != raw) { hist_dec(H, raw); hist_inc(H, pb); }
                            }
                        }
                        wave_lds_fence();
                    }
                }
                issue(rv[s], rb[s], rho + kDepth);
            }
        }

        if (it.n & 7) {   // (uniform: the last part of an odd vocabulary) the logits past the last vector
            if (tid < (it.n & 7)) {
                const int off = 8 * it.nvec + tid;
                const uint32_t raw = uint32_t(row16[it.s0 + off]);
                const bool present = pen && ((uint32_t(cur.pb[it.nvec]) >> tid) & 1u);
                hist_inc(H, present ? pen_pattern<DT>(raw, 1u, p, inv_r, rep_fast) : raw);
            }
        }
        lds_barrier();
        if (pen && cur.nrep > uint32_t(kRepPF * kT)) {   // (long repeat lists: the rest of the entries)
            for (uint32_t i = uint32_t(kRepPF * kT + tid); i < cur.nrep; i += kT) {
                const uint2 e = cur.list[i];
                if (in_part(e)) correct(e, row16[e.x]);
            }
            lds_barrier();
        }

        // ---- publication: the non-empty groups at their place in the part's
        // table and the occupancy bitmap; the histogram cleared.  Eight lanes
        // hold a group (lane 8i + j: its words 4j .. 4j + 3), so the LDS reads
        // are conflict-free and the stores coalesce.  Plain stores: the merge
        // launch reads them.
        {
            const size_t pi = size_t(it.row) * a.parts + it.part;
            uint4* dst = a.pwords + pi * (kGroups * kGW / 4);
            const int t = opaque_tid();
            uint4* H4 = reinterpret_cast<uint4*>(H);
            uint32_t occ_p = 0u, occ_n = 0u;   // bit q: the thread's group of round q
#pragma unroll
            for (int q = 0; q < kHW / 4 / kT; ++q) {
                const int c = q * kT + t;            // 16-byte chunk c: words 4c .. 4c + 3 of group c / 8
                const uint4 d = H4[c];
                H4[c] = make_uint4(0u, 0u, 0u, 0u);
                // the halves any word of the group holds: over its eight lanes, lane
                // ^ 1, ^ 2, then the mirrored half row (uniform quads by then)
                uint32_t any = (d.x | d.y) | (d.z | d.w);
                any |= dpp_u32<0xb1, 0xf, false>(any);
                any |= dpp_u32<0x4e, 0xf, false>(any);
                any |= dpp_u32<0x141, 0xf, false>(any);
                if (any) dst[c] = d;
                occ_p |= min(any & 0xffffu, 1u) << q;
                occ_n |= min(any >> 16, 1u) << q;
            }
            if ((lane & 7) == 0) {   // groups q * 128 + wave * 8 + lane / 8
                sh.occb[0][tid >> 3] = uint8_t(occ_p);
                sh.occb[1][tid >> 3] = uint8_t(occ_n);
            }
            lds_barrier();
            if (tid < kPub) a.ppub[pi * kPub + tid] = reinterpret_cast<const uint32_t*>(sh.occb)[tid];
            // Stores and loads share one counter and may complete out of order:
            // with a store outstanding every wait on a load would have to drain
            // the counter.  Drain it once here instead.
            vm_drain();
        }

        // ---- the next part (its first turn already in flight)
        if (++k >= nitems) break;
        cur = nxt;
        settle(cur);
        has_next = k + 1 < nitems;
        if (has_next) nxt = view(k + 1);
    }
}

// ------------------------------------------------------------------ merge
struct MergeShared {
    uint32_t scan[kW + 1];
    uint32_t wtot[8][kW];
    uint64_t wmass[kW];
    uint32_t wci[kW];   // the running sums through each wave's 128 blocks
    uint64_t wmi[kW];
    uint32_t nslots, total_cnt, z0key, owner, orank, flags, kmin, kmax;
    uint64_t total_mass;
    // the ranks to name: [0] the last end-key logit inside the support (when the
    // support cuts its key's logits), [1] the draw
    uint32_t want[2], key[2], rank[2];
    int32_t id[2];
    uint32_t end_key;
    uint32_t n_support, ok, lo1, hi1, nflip, nown;
    double s_n, u;
};

// Key k's histogram location: group, word inside the group, half (0: low).
struct KeyLoc {
    uint32_t group, word, hi;
};
__device__ __forceinline__ KeyLoc key_loc(uint32_t k) {
    const uint32_t wd = k >= 0x8000u ? k - 0x8000u : 0x7fffu - k;
    return KeyLoc{wd >> 5, wd & 31u, k >= 0x8000u ? 0u : 1u};
}
// Order key of each 16-bit half of a word, -0 kept apart just below +0
// (0x7fff): the key is pattern ^ 0x8000 for a clear sign bit, ~pattern for a
// set one.
__device__ __forceinline__ uint32_t halves_key(uint32_t d) {
    typedef short s2 __attribute__((ext_vector_type(2)));
    const s2 sg = __builtin_bit_cast(s2, d) >> 15;   // 0 or -1 per half
    return d ^ (__builtin_bit_cast(uint32_t, sg) | 0x80008000u);
}
// Per 16-bit half: a - b (wrapping), max(a - b, 0), and min(a, 1).  The last
// two are written as the packed instructions (the compiler otherwise turns the
// pair into a compare and a select per half).
__device__ __forceinline__ uint32_t pk_sub_u16(uint32_t a, uint32_t b) {
    typedef unsigned short u2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(u2, a) - __builtin_bit_cast(u2, b));
}
__device__ __forceinline__ uint32_t pk_sub_sat_u16(uint32_t a, uint32_t b) {
    uint32_t r;
    asm("v_pk_sub_u16 %0, %1, %2 clamp" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ uint32_t pk_nonzero_u16(uint32_t a) {
    uint32_t r;
    asm("v_pk_min_u16 %0, %1, %2" : "=v"(r) : "v"(a), "s"(0x00010001u));
    return r;
}

template <int DT>
__global__ __launch_bounds__(kT) void merge_kernel(StreamArgs a) {
    __shared__ __attribute__((aligned(16))) unsigned char lds[kMLds];
    __shared__ MergeShared sh;
    const int row = blockIdx.x;
    const vi_row_params p = a.params[row];
    if (!stream_row(p)) return;
    const int tid = threadIdx.x, lane = lane_id(), wave = tid / kWave;
    const int P = a.parts, V = a.vocabulary;
    uint32_t* pbits = reinterpret_cast<uint32_t*>(lds + kOffMBits);
    uint32_t* occ = reinterpret_cast<uint32_t*>(lds + kOffMOcc);
    uint16_t* slot_of = reinterpret_cast<uint16_t*>(lds + kOffMSlot);
    uint16_t* group_of = reinterpret_cast<uint16_t*>(lds + kOffMGroupOf);
    uint32_t* bcnt = reinterpret_cast<uint32_t*>(lds + kOffMBcnt);
    uint64_t* bmass = reinterpret_cast<uint64_t*>(lds + kOffMBmass);
    uint32_t* cab = reinterpret_cast<uint32_t*>(lds + kOffMCab);
    uint64_t* mab = reinterpret_cast<uint64_t*>(lds + kOffMMab);
    uint32_t* flip = reinterpret_cast<uint32_t*>(lds + kOffMFlip);
    uint4* keys = reinterpret_cast<uint4*>(lds + kOffMKeys);
    const size_t pi0 = size_t(row) * P;
    const PenView pv = pen_view(a, row, p);
    const float inv_t = 1.0f / p.temperature;

    // ---- 0. the parts' occupancy bitmaps; the valid key range
    if (tid < 96) occ[tid] = 0u;
    uint32_t pub[2] = {0u, 0u};   // (thread i: word i % 32 of part i / 32; at most 512 words)
    static_assert(kMaxParts * 32 <= kT, "one bitmap word per thread");
    if (tid < P * 32) {
        pub[0] = a.ppub[(pi0 + tid / 32) * kPub + tid % 32];
        pub[1] = a.ppub[(pi0 + tid / 32) * kPub + 32 + tid % 32];
        pbits[tid] = pub[0] | pub[1];
    }
    // The first repeat entries (two per thread), requested now (reads within
    // the list whatever it holds); their logits are gathered once the owner
    // part is known, for the entries inside it only.
    const uint16_t* row16 = reinterpret_cast<const uint16_t*>(static_cast<const unsigned char*>(a.logits) +
                                                              2 * size_t(row) * size_t(a.stride));
    uint2 rep[2];
    {
        const uint2* rl = pv.pen ? pv.list : reinterpret_cast<const uint2*>(a.params);
        const uint32_t rn = pv.pen ? max(pv.nrep, 1u) : 1u;
#pragma unroll
        for (int j = 0; j < 2; ++j) rep[j] = rl[min(uint32_t(j * kT + tid), rn - 1u)];
    }
    if (wave == 1) {
        const uint32_t km = valid_key_range<DT>(p.temperature);
        if (lane == 0) { sh.kmin = km & 0xffffu; sh.kmax = km >> 16; }
    }
    for (int i = tid; i < 2048; i += kT) { bcnt[i] = 0u; bmass[i] = 0ull; }
    if (tid == 2 * kWave) sh.u = philox_uniform(p.seed, p.lane, p.position, 0u);
    if (tid == 0) { sh.flags = pv.flags; sh.ok = 1u; sh.z0key = 0u; }
    lds_barrier();
    if (tid < P * 32) {
        atomicOr(&occ[tid % 32], pub[0] | pub[1]);
        atomicOr(&occ[32 + tid % 32], pub[0]);
        atomicOr(&occ[64 + tid % 32], pub[1]);
    }
    lds_barrier();
    // a slot per occupied group
    {
        const GroupBit gb = group_bit(uint32_t(tid));
        const uint32_t o = (occ[gb.word] >> gb.shift) & 1u;
        uint32_t n = 0u;
        const uint32_t e = block_scan_lds(o, sh.scan, &n);
        slot_of[tid] = uint16_t(o ? e : kNoSlot);
        if (o) group_of[e] = uint16_t(tid);
        if (tid == 0) sh.nslots = n;
    }
    lds_barrier();
    const uint32_t nslots = sh.nslots;
    const bool store_keys = nslots <= kSlotCap;
    const uint32_t kmin = sh.kmin, kmax = sh.kmax;
    const bool fail = (sh.flags & VI_FLAG_ERROR) != 0u || !(p.temperature <= kMaxTemperature);

    // Counts of words 2q, 2q + 1 of group g summed over the parts: (lo0, hi0,
    // lo1, hi1); the parts' loads four at a time.
    auto sum_pair = [&](uint32_t g, uint32_t q) -> uint4 {
        uint4 c = make_uint4(0u, 0u, 0u, 0u);
        const GroupBit gb = group_bit(g);
        const uint64_t* src = reinterpret_cast<const uint64_t*>(a.pwords);
        for (int p0 = 0; p0 < P; p0 += 4) {
            uint64_t w2[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int pp = p0 + k;
                w2[k] = 0ull;
                if (pp < P && ((pbits[pp * 32 + gb.word] >> gb.shift) & 1u))
                    w2[k] = src[((pi0 + pp) * kGroups + g) * 16 + q];
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const uint32_t w0 = uint32_t(w2[k]), w1 = uint32_t(w2[k] >> 32);
                c.x += w0 & 0xffffu; c.y += w0 >> 16; c.z += w1 & 0xffffu; c.w += w1 >> 16;
            }
        }
        if (g == 0u && q == 0u) { c.x += c.y; c.y = 0u; }   // -0 is +0
        return c;
    };
    // ---- 1. the highest valid key present, z0's, by the last wave: the highest
    // group holding a positive pattern (the lowest holding a negative one) is
    // known from the bitmaps, so one read of its 32 words finds the key
    auto word_or = [&](uint32_t g) -> uint32_t {   // (lanes 0..31: word `lane` of group g, any part's halves)
        uint32_t w = 0u;
        const GroupBit gb = group_bit(g);
        const uint32_t* src = reinterpret_cast<const uint32_t*>(a.pwords);
        for (int p0 = 0; p0 < P; p0 += 4) {
            uint32_t w4[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int pp = min(p0 + k, P - 1);
                w4[k] = src[((pi0 + pp) * kGroups + g) * kGW + uint32_t(lane & 31)];
                if (!((pbits[pp * 32 + gb.word] >> gb.shift) & 1u)) w4[k] = 0u;
            }
            w |= (w4[0] | w4[1]) | (w4[2] | w4[3]);
        }
        return lane < 32 ? w : 0u;
    };
    auto find_top = [&]() -> uint32_t {
        if (kmin > kmax) return 0u;
        // (byte j of word `lane`: bit q is group q * 128 + 4 * lane + j)
        uint32_t m = lane < 32 ? occ[32 + lane] : 0u;   // groups of positive patterns, highest first
        while (ballot(m != 0u)) {
            uint32_t g = 0u;
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j) {
                const uint32_t b = (m >> (8u * j)) & 0xffu;
                if (b) g = max(g, ((31u - uint32_t(__builtin_clz(b))) << 7) | (4u * uint32_t(lane) + j));
            }
#pragma unroll
            for (int o = 32; o; o >>= 1) g = max(g, uint32_t(__shfl_xor(int(g), o, kWave)));
            const GroupBit gb = group_bit(g);
            if (uint32_t(lane) == gb.word) m &= ~(1u << gb.shift);
            if (0x8000u + 32u * g > kmax) continue;
            const uint64_t h = ballot((word_or(g) & 0xffffu) && 0x8000u + 32u * g + uint32_t(lane) <= kmax);
            if (h) return 0x8000u + 32u * g + 63u - uint32_t(__builtin_clzll(h));
        }
        m = lane < 32 ? occ[64 + lane] : 0u;            // negative patterns, lowest first (-0 is +0)
        while (ballot(m != 0u)) {
            uint32_t g = kGroups;
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j) {
                const uint32_t b = (m >> (8u * j)) & 0xffu;
                if (b) g = min(g, (uint32_t(__builtin_ctz(b)) << 7) | (4u * uint32_t(lane) + j));
            }
#pragma unroll
            for (int o = 32; o; o >>= 1) g = min(g, uint32_t(__shfl_xor(int(g), o, kWave)));
            const GroupBit gb = group_bit(g);
            if (uint32_t(lane) == gb.word) m &= ~(1u << gb.shift);
            const uint32_t wd = 32u * g + uint32_t(lane & 31);
            const uint64_t h = ballot((word_or(g) >> 16) && (wd == 0u || 0x7fffu - wd >= kmin));
            if (h) {
                const uint32_t w0 = 32u * g + uint32_t(__builtin_ctzll(h));
                return w0 == 0u ? 0x8000u : 0x7fffu - w0;
            }
        }
        return 0u;
    };
    // ---- 2. per-key counts summed over the parts and the block sums in one
    // pass (a task: four words of a group, 16 bytes per part; two tasks per
    // thread, their loads issued together, the first pair's while the last wave
    // finds z0).  A 32-key block's sums are the eight lanes' of its group and
    // sign.  Counts of the first kSlotCap occupied groups are kept for the
    // decisions (past it they are summed again there).  (With z0 found from the
    // counts, rows of more groups than the LDS keeps took two passes and an
    // atomic per key: fp16 N(0, 1.4), 81 x 168,896, merge
    // 48.6 us then, 31.8 now.)
    const uint32_t ntask = nslots * 8u;
    auto sum_quad = [&](uint32_t t, uint32_t (&lo)[4], uint32_t (&hi)[4]) {
#pragma unroll
        for (int i = 0; i < 4; ++i) lo[i] = hi[i] = 0u;
        if (t >= ntask) return;
        const uint32_t g = group_of[t >> 3], q = t & 7u;
        const GroupBit gb = group_bit(g);
        for (int p0 = 0; p0 < P; p0 += 4) {
            uint4 w4[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int pp = p0 + k;
                w4[k] = make_uint4(0u, 0u, 0u, 0u);
                if (pp < P && ((pbits[pp * 32 + gb.word] >> gb.shift) & 1u))
                    w4[k] = a.pwords[((pi0 + pp) * kGroups + g) * (kGW / 4) + q];
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                lo[0] += w4[k].x & 0xffffu; hi[0] += w4[k].x >> 16;
                lo[1] += w4[k].y & 0xffffu; hi[1] += w4[k].y >> 16;
                lo[2] += w4[k].z & 0xffffu; hi[2] += w4[k].z >> 16;
                lo[3] += w4[k].w & 0xffffu; hi[3] += w4[k].w >> 16;
            }
        }
        if (g == 0u && q == 0u) { lo[0] += hi[0]; hi[0] = 0u; }   // -0 is +0
    };
    double z0 = 0.0;
    uint32_t z0key = 0u;
    bool invalid = false;
    auto add_quad = [&](uint32_t t, const uint32_t (&lo)[4], const uint32_t (&hi)[4]) {
        const uint32_t s = min(t, ntask - 1u) >> 3, g = group_of[s], q = t & 7u, w0 = g * kGW + 4u * q;
        if (store_keys && t < ntask) {
            keys[s * 16u + 2u * q] = make_uint4(lo[0], hi[0], lo[1], hi[1]);
            keys[s * 16u + 2u * q + 1u] = make_uint4(lo[2], hi[2], lo[3], hi[3]);
        }
        uint32_t cp = 0u, cn = 0u;
        uint64_t mp = 0ull, mn = 0ull;
        auto add = [&](uint32_t k, uint32_t c, uint32_t& cs, uint64_t& ms) {
            if (!c) return;
            if (!key_valid<DT>(k, kmin, kmax)) { invalid = true; return; }
            cs += c;
            ms += fixed_mass(c, key_weight<DT>(k, inv_t, z0));
        };
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            add(0x8000u + w0 + uint32_t(i), lo[i], cp, mp);
            add(0x7fffu - w0 - uint32_t(i), hi[i], cn, mn);
        }
        // over the group's eight lanes: lane ^ 1, ^ 2, then the mirrored half row
        // (uniform quads by then)
        auto dpp64 = [](uint64_t v, auto dpp) {
            return uint64_t(dpp(uint32_t(v))) | (uint64_t(dpp(uint32_t(v >> 32))) << 32);
        };
        auto step = [&](auto dpp) {
            cp += dpp(cp);
            cn += dpp(cn);
            mp += dpp64(mp, dpp);
            mn += dpp64(mn, dpp);
        };
        step([](uint32_t u) { return dpp_u32<0xb1, 0xf, false>(u); });
        step([](uint32_t u) { return dpp_u32<0x4e, 0xf, false>(u); });
        step([](uint32_t u) { return dpp_u32<0x141, 0xf, false>(u); });
        if (t < ntask && q == 0u) {
            bcnt[1024u + g] = cp;
            bmass[1024u + g] = mp;
            bcnt[1023u - g] = cn;
            bmass[1023u - g] = mn;
        }
    };
    for (uint32_t t0 = 0; t0 < ntask || t0 == 0u; t0 += 2 * kT) {   // (uniform; the first turn always: z0)
        uint32_t la[4], ha[4], lb[4], hb[4];
        const uint32_t ta = t0 + uint32_t(tid), tb = ta + kT;
        if (t0 == 0u && wave == kW - 1) {
            const uint32_t top = find_top();
            if (lane == 0) sh.z0key = top;
        }
        sum_quad(ta, la, ha);
        sum_quad(tb, lb, hb);
        if (t0 == 0u) {
            lds_barrier();
            z0key = sh.z0key;
            z0 = double(key_z<DT>(z0key, inv_t));
            if (ntask == 0u) break;
        }
        add_quad(ta, la, ha);
        if (t0 + kT < ntask) add_quad(tb, lb, hb);   // (uniform)
    }
    if (ballot(invalid) && lane == 0) atomicOr(&sh.flags, uint32_t(VI_FLAG_NONFINITE));
    lds_barrier();
    // ---- 3. descending prefix sums over the 2048 blocks (thread t: blocks
    // 2047 - 2t and 2046 - 2t)
    {
        const int b0 = 2047 - 2 * tid, b1 = b0 - 1;
        const uint32_t c0 = bcnt[b0], c1 = bcnt[b1];
        const uint64_t m0 = bmass[b0], m1 = bmass[b1];
        const uint32_t ci = wave_incl_scan_u32(c0 + c1);
        const uint64_t mi = wave_incl_scan_u64(m0 + m1);
        if (lane == kWave - 1) { sh.scan[wave] = ci; sh.wmass[wave] = mi; }
        lds_barrier();
        uint32_t cb = 0u;
        uint64_t mb = 0ull;
        {   // the earlier waves' totals, one per lane, summed across the wave (exact integers)
            const bool e = lane < wave;
            cb = readlane_u(wave_incl_scan_u32(e ? sh.scan[lane] : 0u), kWave - 1);
            mb = readlane_u64(wave_incl_scan_u64(e ? sh.wmass[lane] : 0ull), kWave - 1);
        }
        if (lane == kWave - 1) { sh.wci[wave] = cb + ci; sh.wmi[wave] = mb + mi; }
        if (tid == kT - 1) { sh.total_cnt = cb + ci; sh.total_mass = mb + mi; }
        const uint32_t ce = cb + ci - (c0 + c1);
        const uint64_t me = mb + mi - (m0 + m1);
        cab[b0] = ce; mab[b0] = me;
        cab[b1] = ce + c0; mab[b1] = me + m0;
    }
    lds_barrier();
    const uint32_t N = sh.total_cnt;
    const uint64_t Mtot = sh.total_mass;
    const uint32_t out_flags = sh.flags & (VI_FLAG_NONFINITE | VI_FLAG_BAD_HISTORY);
    if (fail || N == 0u) {
        if (tid == 0) {
            a.tokens[row] = fail ? -1 : V;
            if (a.uniforms) a.uniforms[row] = 0.0;
            if (a.stats) {
                vi_sample_stats st{};
                st.flags = out_flags | (fail ? VI_FLAG_ERROR : VI_FLAG_EMPTY);
                a.stats[row] = st;
            }
            if (a.bounds) a.bounds[row] = FullBound{0.0, 0.0, 0.0f, 0u, 0, 0u};
        }
        return;
    }

    // Count of key 32 b + 31 - lane (lanes < 32: the block's keys in descending
    // order; 0 for lanes >= 32 and invalid keys).  Wave-uniform b.
    auto block_key_count = [&](uint32_t b) -> uint32_t {
        const uint32_t k = 32u * b + 31u - uint32_t(lane & 31);
        if (lane >= 32 || !key_valid<DT>(k, kmin, kmax)) return 0u;
        const KeyLoc kl = key_loc(k);
        const uint32_t slot = slot_of[kl.group];
        if (slot == kNoSlot) return 0u;
        const uint4 c = store_keys ? keys[slot * 16u + (kl.word >> 1)] : sum_pair(kl.group, kl.word >> 1);
        const uint32_t lo = (kl.word & 1u) ? c.z : c.x, hi = (kl.word & 1u) ? c.w : c.y;
        return kl.hi ? hi : lo;
    };
    // Wave 0: the first block (descending) at which the cumulative count
    // (mode 0: >= target) or fixed-point mass (mode 1: >= target, mode 2: >
    // target) is reached; -1 if none.  First the wave of the running sums that
    // holds it, then its 128 blocks, two to a lane.  (A search over the 2048
    // sums themselves probes every 32nd first, all in one LDS bank: 1,700 cycles.)
    auto block_search = [&](int mode, uint64_t target) -> int {
        auto reached = [&](uint64_t x) { return mode == 2 ? x > target : x >= target; };
        const int wl = lane & (kW - 1);
        const uint64_t wm = ballot(lane < kW && reached(mode == 0 ? uint64_t(sh.wci[wl]) : sh.wmi[wl]));
        if (!wm) return -1;
        const int b0 = 2047 - 128 * __builtin_ctzll(wm) - 2 * lane, b1 = b0 - 1;
        const uint64_t s0 = mode == 0 ? uint64_t(cab[b1]) : mab[b1];   // (through b0)
        const uint64_t s1 = s0 + (mode == 0 ? uint64_t(bcnt[b1]) : bmass[b1]);
        const uint64_t m0 = ballot(reached(s0)), m1 = ballot(reached(s1));
        if (!m1) return -1;
        const int L = __builtin_ctzll(m1);
        return 2047 - 128 * __builtin_ctzll(wm) - 2 * L - (((m0 >> L) & 1ull) ? 0 : 1);
    };
    struct Fine {
        bool found;
        uint32_t key, take;   // position: the first `take` logits of `key` in id order
        uint32_t of, cnt;     // logits of the key, and up to the position
        uint64_t mass;        // mass up to the position
    };
    // Wave 0, inside block b: the first key at which the cumulative count
    // (mode 0: >= target) or mass (1: >= target, 2: > target) is reached, with
    // the counts limited to the position (lim_key, lim_take); target relative
    // to the block's start.
    auto fine_find = [&](uint32_t b, int mode, uint64_t target, uint32_t lim_key, uint32_t lim_take) -> Fine {
        const uint32_t k = 32u * b + 31u - uint32_t(lane & 31);
        const uint32_t of = block_key_count(b);
        const uint64_t ma = mab[b];
        const uint32_t ca = cab[b];
        uint32_t c = of;
        if (k < lim_key) c = 0u;
        else if (k == lim_key) c = min(c, lim_take);
        const double w = c ? key_weight<DT>(k, inv_t, z0) : 0.0;
        const uint64_t m = c ? fixed_mass(c, w) : 0ull;
        const uint64_t mi = wave_incl_scan_u64(m);
        const uint32_t ci = wave_incl_scan_u32(c);
        const uint64_t me = mi - m;
        const uint32_t cexcl = ci - c;
        bool hit = false;
        uint32_t take = 0u;
        if (c) {
            if (mode == 0) {
                hit = uint64_t(ci) >= target;
                if (hit) take = uint32_t(target - cexcl);
            } else {
                // (m / c: one logit's mass)
                hit = mode == 1 ? mi >= target : mi > target;
                if (hit) {
                    const double x = double(target - me) * double(c) / double(m);
                    take = mode == 1 ? uint32_t(ceil(x)) : uint32_t(floor(x)) + 1u;
                }
            }
            take = min(max(take, 1u), c);
        }
        const uint64_t hm = ballot(hit);
        Fine f{};
        if (hm) {
            const int L = __builtin_ctzll(hm);
            f.found = true;
            f.key = 32u * b + 31u - uint32_t(L);
            f.take = readlane_u(take, L);
            f.of = readlane_u(of, L);
            f.cnt = ca + readlane_u(cexcl + take, L);
            f.mass = ma + readlane_u64(me + (take ? fixed_mass(take, w) : 0ull), L);
        }
        return f;
    };
    // Wave 0: mass and count of the support through position (key, take).
    // (of: logits of the key)
    auto mass_through = [&](uint32_t key, uint32_t take, uint64_t* mass, uint32_t* cnt, uint32_t* of) {
        const uint32_t b = key >> 5;
        const uint32_t k = 32u * b + 31u - uint32_t(lane & 31);
        uint32_t c = block_key_count(b);
        *of = readlane_u(c, 31 - int(key & 31u));
        if (k < key) c = 0u;
        else if (k == key) c = min(c, take);
        const uint64_t m = c ? fixed_mass(c, key_weight<DT>(k, inv_t, z0)) : 0ull;
        *mass = mab[b] + readlane_u64(wave_incl_scan_u64(m), kWave - 1);
        *cnt = cab[b] + readlane_u(wave_incl_scan_u32(c), kWave - 1);
    };

    // ---- 4. the decisions, in wave 0: the top-k cap, the min-p cut, the top-p
    // cut, the support's end (the earliest of them) and the draw
    if (wave == 0) {
        const bool has_cap = p.top_k > 0 && uint32_t(p.top_k) < N;
        uint32_t cap_key = 0u, cap_take = kTakeAll;
        Fine cap{}, topp{};
        double s_cap = double(Mtot);
        if (has_cap) {
            const int b = block_search(0, uint64_t(p.top_k));
            cap = fine_find(uint32_t(b), 0, uint64_t(p.top_k) - cab[b], 0u, kTakeAll);
            cap_key = cap.key;
            cap_take = cap.take;
            s_cap = double(cap.mass);
        }
        // min-p: the lowest key whose weight reaches min_p (in double precision: the
        // masses' weights are good to an fp32 ulp, which a key near the cut may miss)
        uint32_t minp_key = 0u;
        if (p.min_p > 0.0f) {
            const double mp = double(p.min_p);
            minp_key = uint32_t(wave_search(int(kmin), int(z0key) + 1, [&](int k) {
                return exp(double(key_z<DT>(uint32_t(k), inv_t)) - z0) >= mp;
            }));
        }
        // top-p: the first position whose cumulative mass reaches top_p of the cap's
        if (p.top_p < 1.0f) {
            // (a target of less than one unit, of any top_p <= 0 too: the first logit)
            const uint64_t target = uint64_t(std::max(llrint(double(p.top_p) * s_cap), 1ll));
            const int b = block_search(1, target);
            const int lowest = has_cap ? int(cap_key >> 5) : 0;
            if (b >= lowest) {
                const bool in_cap = has_cap && uint32_t(b) == (cap_key >> 5);
                topp = fine_find(uint32_t(b), 1, target - mab[b], in_cap ? cap_key : 0u, in_cap ? cap_take : kTakeAll);
            }
        }
        // the support's end, its mass, the uniform and the draw's target
        bool all = true, known = false, cuts = false;   // (known: its mass and count; cuts: it cuts its last key's logits)
        uint32_t ek = 0u, et = kTakeAll;
        uint64_t sm = Mtot;
        uint32_t sc = N;
        auto consider = [&](uint32_t k, uint32_t t, const Fine& f) {
            if (!(all || k > ek || (k == ek && t < et))) return;
            ek = k; et = t; all = false;
            known = f.found; cuts = f.found && t < f.of; sm = f.mass; sc = f.cnt;
        };
        if (has_cap) consider(cap_key, cap_take, cap);
        if (p.min_p > 0.0f) consider(minp_key, kTakeAll, Fine{});
        if (topp.found) consider(topp.key, topp.take, topp);
        if (!all && ek > z0key) { ek = z0key; et = 1u; known = false; }   // no logit passes min-p: the best one
        if (!all && !known) {
            uint32_t of;
            mass_through(ek, et, &sm, &sc, &of);
            cuts = et < of;
        }
        const bool draw = a.draw_every > 0 && (a.row0 + row) % a.draw_every == a.draw_every - 1;
        const double u = sh.u;
        const double target_d = u * double(sm);
        // the draw: the first support logit whose inclusive mass exceeds u * S_n
        const uint64_t t = uint64_t(target_d);
        int b = draw ? block_search(2, t) : -1;
        const int lowest = all ? 0 : int(ek >> 5);
        if (b < lowest) b = -1;
        uint32_t dk = 0u, dr = 0u;
        bool ok = !draw;
        if (b >= 0) {
            const bool in_end = !all && uint32_t(b) == (ek >> 5);
            const Fine f = fine_find(uint32_t(b), 2, t - mab[b], in_end ? ek : 0u, in_end ? et : kTakeAll);
            if (f.found) { dk = f.key; dr = f.take - 1u; ok = true; }
        }
        if (!ok) {   // rounding past the support's last logit: that logit
            for (int bb = lowest; bb < 2048 && !ok; ++bb) {
                if (!bcnt[bb]) continue;
                const uint32_t k = 32u * uint32_t(bb) + 31u - uint32_t(lane & 31);
                uint32_t c = block_key_count(uint32_t(bb));
                if (!all) {
                    if (k < ek) c = 0u;
                    else if (k == ek) c = min(c, et);
                }
                const uint64_t hm = ballot(c > 0u);
                if (hm) {
                    const int L = 63 - __builtin_clzll(hm);
                    dk = 32u * uint32_t(bb) + 31u - uint32_t(L);
                    dr = readlane_u(c, L) - 1u;
                    ok = true;
                }
            }
        }
        if (lane == 0) {
            sh.s_n = double(sm);
            sh.n_support = sc;
            sh.end_key = all ? 0u : ek;
            sh.want[0] = a.bounds && cuts ? 1u : 0u;
            sh.key[0] = ek;
            sh.rank[0] = et - 1u;
            sh.id[0] = 0x7fffffff;
            sh.want[1] = draw ? 1u : 0u;
            sh.key[1] = dk;
            sh.rank[1] = dr;
            sh.id[1] = -1;
            sh.ok = ok ? 1u : 0u;
        }
    }
    lds_barrier();

    // ---- 5. the part holding the rank to name (parts in id order) and, for the
    // rescan, the key's preimage under the count-1 penalty: a history token
    // counted once has the key exactly when its raw key lies in [lo1, hi1) (the
    // penalty is monotone in the logit)
    const float inv_r = rep_inverse(p);
    const bool rep_fast = rep_fast_ok(p);
#pragma unroll 1
    for (int which = 0; which < 2; ++which) {
        if (!sh.want[which]) continue;   // (uniform)
        lds_barrier();   // (the rank named before: its scratch is free)
        const uint32_t dk = sh.key[which];
        if (wave == 0 && sh.ok) {
            const KeyLoc kl = key_loc(dk);
            const GroupBit gb = group_bit(kl.group);
            uint32_t c = 0u;
            if (lane < P && ((pbits[lane * 32 + gb.word] >> gb.shift) & 1u)) {
                const uint64_t* src = reinterpret_cast<const uint64_t*>(a.pwords) + ((pi0 + lane) * kGroups + kl.group) * 16;
                const uint64_t w2 = src[kl.word >> 1];
                const uint32_t wd = (kl.word & 1u) ? uint32_t(w2 >> 32) : uint32_t(w2);
                c = kl.hi ? (wd >> 16) : (wd & 0xffffu);
                if (dk == 0x8000u) c = (wd & 0xffffu) + (wd >> 16);   // +0 and -0
            }
            const uint32_t incl = wave_incl_scan_u32(c);
            const uint32_t rank = sh.rank[which];
            const uint64_t hm = ballot(lane < P && incl > rank);
            if (hm) {
                const int L = __builtin_ctzll(hm);
                if (lane == L) { sh.owner = uint32_t(L); sh.orank = rank - (incl - c); }
            } else if (lane == 0) {
                sh.ok = 0u;
            }
        }
        if (wave == 1 && pv.pen && sh.ok) {
            constexpr int kNegMin = DT == VI_BF16 ? 0x0080 : 0x0400;
            constexpr int kPosMax = DT == VI_BF16 ? 0xff7f : 0xfbff;
            auto fk = [&](int k) { return key16(pen_pattern<DT>(unkey16(uint32_t(k)), 1u, p, inv_r, rep_fast)); };
            const uint32_t lo = uint32_t(wave_search(kNegMin, kPosMax + 1, [&](int k) { return fk(k) >= dk; }));
            const uint32_t hi = uint32_t(wave_search(kNegMin, kPosMax + 1, [&](int k) { return fk(k) > dk; }));
            if (lane == 0) { sh.lo1 = lo; sh.hi1 = hi; }
        }
        for (int i = tid; i < 2048; i += kT) flip[i] = 0u;
        if (tid == 0) { sh.nflip = 0u; sh.nown = 0u; }
        // presence masks by byte for the rescan, in the decisions' running-sum
        // table (free now): entry b, word q: the halves of tokens 2q and 2q + 1 all
        // ones where that token is in the history
        {
            const uint32_t b = uint32_t(tid) >> 2, q = uint32_t(tid) & 3u;
            reinterpret_cast<uint32_t*>(lds + kOffMCab)[tid] = (((b >> (2u * q)) & 1u) ? 0x0000ffffu : 0u) |
                                                              (((b >> (2u * q + 1u)) & 1u) ? 0xffff0000u : 0u);
        }
        static_assert(256 * 16 <= kOffMMab - kOffMCab && kT == 1024, "presence masks");
        lds_barrier();

        // ---- 6. the owner part read again: its orank-th logit (id order) whose
        // penalized key is the drawn key.  Repeated tokens whose count changes the
        // answer are flipped.
        if (sh.ok) {
            const Item it = part_geo(a, row, int(sh.owner));
            const bool pen = pv.pen;
            const unsigned char* vb = static_cast<const unsigned char*>(a.logits) +
                                      2 * (size_t(row) * size_t(a.stride) + size_t(it.s0));
            const unsigned char* pb = pen ? pv.b1 + (it.s0 >> 3) : nullptr;
            static_assert(kMaxPartLen / 8 <= 8 * kT, "a part is at most 8 rounds");
            // the part's logits and presence bytes, eight rounds of 1024 vectors,
            // all requested before the flips are worked out
            auto load_vec = [&](int v, uint4* d, uint32_t* b) {
                const int vc = max(min(v, it.nvec - 1), 0);
                *d = load16_cached((it.nvec > 0 ? vb : reinterpret_cast<const unsigned char*>(a.params)) + size_t(vc) * 16);
                *b = pb ? uint32_t(pb[vc]) : 0u;
            };
            uint4 vv[8];
            uint32_t bb[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) load_vec(k * kT + tid, &vv[k], &bb[k]);
            // The owner part's repeat entries gathered into a list (the other parts'
            // would leave most lanes idle below), their logits requested behind the
            // part (their flips are worked out after the count, which they correct)
            auto in_owner = [&](uint2 e) { return e.y >= 2u && int(e.x) >= it.s0 && int(e.x) < it.s0 + it.n; };
            uint2* own = reinterpret_cast<uint2*>(lds + kOffMKeys);
            static_assert(16 * 16 * kSlotCap >= 2 * kT * sizeof(uint2), "repeat entries");
            uint2 oe[2] = {make_uint2(0u, 0u), make_uint2(0u, 0u)};
            uint32_t raw[2] = {0u, 0u}, nown = 0u;
            if (pen && pv.nrep) {   // (uniform)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const bool mine = uint32_t(j * kT + tid) < pv.nrep && in_owner(rep[j]);
                    const uint64_t m = ballot(mine);
                    uint32_t at = 0u;
                    if (lane == 0 && m) at = atomicAdd(&sh.nown, uint32_t(__builtin_popcountll(m)));
                    at = readlane_u(at, 0) + uint32_t(__builtin_popcountll(m & ((1ull << lane) - 1ull)));
                    if (mine) own[at] = rep[j];
                }
                lds_barrier();
                nown = readlane_u(sh.nown, 0);
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    if (uint32_t(j * kT + tid) >= nown) continue;
                    oe[j] = own[j * kT + tid];
                    raw[j] = uint32_t(row16[oe[j].x]);
                }
            }
            const uint4* pmask = reinterpret_cast<const uint4*>(lds + kOffMCab);
            // In the halves' key space (-0 just below +0): an absent token matches
            // when its key lies in [a0, a0 + w0] (the drawn key, with -0 for +0), a
            // history token when it lies in [a1, a1 + w1] (the preimage; none when
            // empty).
            const uint32_t a0 = dk == 0x8000u ? 0x7fffu : dk, w0 = dk == 0x8000u ? 1u : 0u;
            uint32_t a1 = 0u, w1 = 0u;
            bool empty1 = true;
            if (pen && sh.hi1 > sh.lo1) {
                uint32_t lo = sh.lo1, hi = sh.hi1 - 1u;
                if (lo <= 0x8000u && hi >= 0x8000u) lo = min(lo, 0x7fffu);
                a1 = lo; w1 = hi - lo; empty1 = false;
            }
            const uint32_t A0 = a0 | (a0 << 16), W0 = w0 | (w0 << 16), A1 = a1 | (a1 << 16), W1 = w1 | (w1 << 16);
            const uint32_t force = empty1 ? 0xffffffffu : 0u;   // history halves never match
            // Matches per round before the flips, three rounds to a word in 10-bit
            // fields (a wave's sums stay below 1024): per half, the range of the
            // token's kind is selected by the presence mask and tested as
            // max(key - base - width, 0) == 0.
            uint32_t pc[3] = {0u, 0u, 0u};
#pragma unroll
            for (int r = 0; r < 8; ++r) {
                const int v = r * kT + tid;
                uint32_t c = 0u;
                if (v < it.nvec) {
                    const uint4 M = pmask[bb[r]];
                    const uint32_t w4[4] = {vv[r].x, vv[r].y, vv[r].z, vv[r].w};
                    const uint32_t m4[4] = {M.x, M.y, M.z, M.w};
                    uint32_t miss = 0u;
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const uint32_t base = (m4[q] & A1) | (~m4[q] & A0), width = (m4[q] & W1) | (~m4[q] & W0);
                        const uint32_t t = pk_sub_u16(halves_key(w4[q]), base);
                        miss += pk_nonzero_u16(pk_sub_sat_u16(t, width) | (m4[q] & force));
                    }
                    c = 8u - (miss & 0xffffu) - (miss >> 16);
                }
                pc[r / 3] += c << (10 * (r % 3));
            }
            auto field = [](uint32_t w, int r) { return (w >> (10 * (r % 3))) & 0x3ffu; };
            // exact match of a 16-bit pattern (the scalar form of the count)
            auto match_one = [&](uint32_t pat, uint32_t present) -> uint32_t {
                const uint32_t k = (pat & 0x8000u) ? (~pat & 0xffffu) : (pat | 0x8000u);
                return (present ? !empty1 && k - a1 <= w1 : k - a0 <= w0) ? 1u : 0u;
            };
            // Repeated tokens whose count changes the answer are flipped
            if (pen) {
                auto flip_if = [&](uint2 e, uint32_t rw) {
                    if (!in_owner(e) || !Elem<DT>::finite_bits(rw)) return;
                    const uint32_t mc = key16(pen_pattern<DT>(rw, e.y, p, inv_r, rep_fast)) == dk ? 1u : 0u;
                    if (match_one(rw, 1u) != mc) {
                        const uint32_t off = e.x - uint32_t(it.s0);
                        atomicOr(&flip[off >> 5], 1u << (off & 31u));
                        atomicAdd(&sh.nflip, 1u);
                    }
                };
#pragma unroll 1
                for (uint32_t j = 0; j < 2u && j * kT < nown; ++j) flip_if(j ? oe[1] : oe[0], j ? raw[1] : raw[0]);   // (uniform)
                for (uint32_t i = uint32_t(2 * kT + tid); i < pv.nrep; i += kT) {   // (long repeat lists)
                    const uint2 e = pv.list[i];
                    if (in_owner(e)) flip_if(e, uint32_t(row16[e.x]));
                }
            }
            lds_barrier();
            const bool flips = sh.nflip != 0u;
            auto match_bits = [&](uint4 d, uint32_t b, int v) -> uint32_t {   // (of a vector, flips applied)
                const uint32_t w4[4] = {d.x, d.y, d.z, d.w};
                uint32_t m = 0u;
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    m |= match_one((j & 1) ? w4[j >> 1] >> 16 : w4[j >> 1] & 0xffffu, (b >> j) & 1u) << j;
                if (flips) m ^= (flip[v >> 2] >> ((v & 3) * 8)) & 0xffu;
                return m;
            };
            if (flips) {   // (uniform) the flipped vectors counted again
#pragma unroll
                for (int r = 0; r < 8; ++r) {
                    const int v = r * kT + tid;
                    if (v < it.nvec && ((flip[v >> 2] >> ((v & 3) * 8)) & 0xffu)) {
                        const uint32_t c = uint32_t(__builtin_popcount(match_bits(vv[r], bb[r], v)));
                        pc[r / 3] += (c - field(pc[r / 3], r)) << (10 * (r % 3));
                    }
                }
            }
            uint32_t pin[3];
#pragma unroll
            for (int i = 0; i < 3; ++i) pin[i] = wave_incl_scan_u32(pc[i]);
            if (lane == kWave - 1) {
#pragma unroll
                for (int r = 0; r < 8; ++r) sh.wtot[r][wave] = field(pin[r / 3], r);
            }
            lds_barrier();
            // exclusive offsets of the (round, wave) blocks in id order (wave 0:
            // lane l holds blocks 2l and 2l + 1 of the 128)
            if (wave == 0) {
                const uint32_t b0 = sh.wtot[(2 * lane) >> 4][(2 * lane) & 15], b1 = sh.wtot[(2 * lane + 1) >> 4][(2 * lane + 1) & 15];
                const uint32_t incl = wave_incl_scan_u32(b0 + b1);
                sh.wtot[(2 * lane) >> 4][(2 * lane) & 15] = incl - b0 - b1;
                sh.wtot[(2 * lane + 1) >> 4][(2 * lane + 1) & 15] = incl - b1;
            }
            lds_barrier();
            const uint32_t want = sh.orank;
            // the vector holding the rank, then its logit
            uint4 hv = make_uint4(0u, 0u, 0u, 0u);
            uint32_t hb = 0u, he = 0u;
            int at = -1;
#pragma unroll
            for (int r = 0; r < 8; ++r) {
                const uint32_t c = field(pc[r / 3], r);
                const uint32_t e = sh.wtot[r][wave] + field(pin[r / 3], r) - c;
                if (c && want >= e && want < e + c) { at = r * kT + tid; hv = vv[r]; hb = bb[r]; he = e; }
            }
            if (at >= 0) {
                uint32_t m = match_bits(hv, hb, at);
                for (uint32_t k = want - he; k > 0u; --k) m &= m - 1u;
                sh.id[which] = it.s0 + 8 * at + __builtin_ctz(m);
            }
            if ((it.n & 7) && wave == kW - 1) {   // (uniform) the logits past the last vector: behind every vector
                const uint32_t body = sh.wtot[7][kW - 1] + uint32_t(__builtin_amdgcn_readlane(int(field(pin[2], 7)), kWave - 1));
                const bool in = lane < (it.n & 7);
                const int off = 8 * it.nvec + min(lane, (it.n & 7) - 1);
                const uint32_t tb = pb ? uint32_t(pb[it.nvec]) : 0u, raw = uint32_t(row16[it.s0 + off]);
                const uint32_t one = match_one(raw, (tb >> (off & 7)) & 1u);
                const bool hit = in && (one ^ (flips ? (flip[off >> 5] >> (off & 31)) & 1u : 0u));
                const uint64_t m = ballot(hit);
                const uint32_t before = uint32_t(__builtin_popcountll(m & ((1ull << lane) - 1ull)));
                if (hit && want == body + before) sh.id[which] = it.s0 + off;
            }
            lds_barrier();
        }
    }

    // ---- 7. outputs
    if (tid == 0) {
        const int32_t tok = sh.want[1] ? sh.id[1] : 0;
        if (a.bounds)
            a.bounds[row] = FullBound{z0, sh.s_n / kFix, inv_t, sh.end_key, sh.id[0], tok >= 0 ? 1u : 0u};
        if (!sh.want[1]) {   // (no token of this row is wanted)
            if (a.stats) {
                vi_sample_stats st{};
                st.flags = out_flags;
                a.stats[row] = st;
            }
        } else if (tok < 0) {   // the tables disagree with the logits: cannot happen for consistent inputs
            a.tokens[row] = -1;
            if (a.uniforms) a.uniforms[row] = sh.u;
            if (a.stats) {
                vi_sample_stats st{};
                st.flags = out_flags | VI_FLAG_ERROR;
                a.stats[row] = st;
            }
        } else {
            a.tokens[row] = tok;
            if (a.uniforms) a.uniforms[row] = sh.u;
            if (a.stats) {
                vi_sample_stats st{};
                st.flags = out_flags;
                st.support = sh.n_support;
                st.finite = N;
                st.support_mass = sh.s_n / kFix;
                st.uniform = sh.u;
                a.stats[row] = st;
            }
            if (a.record && a.pstate && !a.probs && tok < V) {   // (with probabilities: repeat_probs_kernel)
                const LaneState ls = lane_state(const_cast<unsigned char*>(a.pstate) + size_t(row) * a.pl.lane_bytes,
                                                a.pl);
                state_record_one(ls, a.pl, V, tok);
            }
        }
    }
}

// ------------------------------------------------------------ history view
// Presence bitmap and repeat list of each row's history, in the layout the
// stream reads from a penalty state: one workgroup per row; bitmaps of the
// tokens seen once (B1) and more than once (B2) built with LDS atomics, then
// each B2 token's rank (population count of B2 before it) indexes its count.
// The bitmaps of the largest vocabulary fit the LDS; counts that no longer do
// beside them are kept in the workspace (every access to them at agent scope):
// 2 rows x 500,001 tokens with histories of 30,000, 60 us per call, 190 with the
// bitmaps there too.
struct HistArgs {
    const int32_t* histories;
    const int64_t* offsets;
    int vocabulary, words, cap;
    uint32_t* hb1;     // [rows][words]
    uint2* hlist;      // [rows][cap]
    uint32_t* hhead;   // [rows][2]
    uint32_t* tmp;     // [rows][cap]: the counts, where they are not in LDS
};
// History tokens per thread held in registers: the first of 4, 8, 16 and 32 that
// covers the longest history, else 32.  (A batch's steps are issued whatever part of
// it holds tokens.  16 rows x 131,071, us per call with histories of 4,096 / 6,000 /
// 12,000 / 16,384 / 20,000 tokens: 36 / 37 / 40 / 41 / 46; with 4 and 32 alone
// 36 / 44 / 44 / 45 / 46.)
constexpr int kHistLong = 32;

constexpr int kHistLdsWords = 40896;       // B1 + B2 + counts (160 KB less the scalars): one workgroup per CU
constexpr int kHistLdsHalf = 20352;        // the same where two fit a CU (4,096 rows x 1,001: 398 us per call, 414)
constexpr int kHistLdsBits = 2 * kMaxVocabulary / 32;   // B1 + B2

// WORDS: the LDS (kHistLdsBits: the counts are in the workspace).
template <int WORDS, int kHistBatch>
__global__ __launch_bounds__(kT) void history_view_kernel(HistArgs h) {
    constexpr bool LDS = WORDS != kHistLdsBits;
    __shared__ __attribute__((aligned(16))) uint32_t hl[WORDS];
    const int row = blockIdx.x, tid = threadIdx.x;
    const int W = h.words;
    uint32_t* B1 = hl;              // then the prefix of B2 per word
    uint32_t* B2 = hl + W;
    uint32_t* cnt = LDS ? hl + 2 * W : h.tmp + size_t(row) * size_t(h.cap);     // [cap]
    auto sync = []() {              // (the counts' stores and atomics with it)
        if (!LDS) __threadfence();
        __syncthreads();
    };
    __shared__ uint32_t flags, nrep, scan[kW + 1];
    const int64_t b = h.offsets[row], e = h.offsets[row + 1];
    const int V = h.vocabulary;
    // The history in batches of kHistBatch tokens per thread (one batch: kept in
    // registers for the second pass; the first is requested before the LDS is
    // cleared).  Each pass issues a batch's LDS operations back to back and uses
    // their results after, so their latencies overlap.
    const bool one_batch = e - b <= int64_t(kHistBatch) * kT;
    int32_t t[kHistBatch];
    auto load = [&](int64_t base) {
#pragma unroll
        for (int j = 0; j < kHistBatch; ++j) {
            const int64_t i = base + int64_t(j) * kT + tid;
            t[j] = i < e ? h.histories[i] : -1;
        }
    };
    load(b);
    for (int i = tid; i < (2 * W + 3) / 4; i += kT) reinterpret_cast<uint4*>(hl)[i] = make_uint4(0u, 0u, 0u, 0u);
    if (tid == 0) flags = 0u;
    __syncthreads();
    for (int64_t base = b; base < e; base += int64_t(kHistBatch) * kT) {
        if (base != b) load(base);
#pragma unroll
        for (int j0 = 0; j0 < kHistBatch; j0 += kHistBatch / 2) {
            uint32_t old[kHistBatch / 2];
#pragma unroll
            for (int j = 0; j < kHistBatch / 2; ++j) {
                const int32_t tj = t[j0 + j];
                old[j] = 0u;
                if (tj >= 0 && tj < V) old[j] = atomicOr(&B1[tj >> 5], 1u << (tj & 31));
                else if (base + int64_t(j0 + j) * kT + tid < e) flags = VI_FLAG_BAD_HISTORY;   // (not past the end)
            }
#pragma unroll
            for (int j = 0; j < kHistBatch / 2; ++j) {
                const int32_t tj = t[j0 + j];
                const uint32_t bit = 1u << (tj & 31);
                if (tj >= 0 && tj < V && (old[j] & bit)) atomicOr(&B2[tj >> 5], bit);
            }
        }
    }
    __syncthreads();
    // B1 out; its LDS then holds the B2 rank of each word's first bit
    uint32_t* out = h.hb1 + size_t(row) * W;
    for (int i = tid; i < W; i += kT) out[i] = B1[i];
    // (ranks in the order of the threads' words tid, tid + kT, ...: the list's order is
    // free, and the words a thread would hold in a run lie in few LDS banks)
    uint32_t own = 0u;
    for (int i = tid; i < W; i += kT) own += uint32_t(__builtin_popcount(B2[i]));
    uint32_t total = 0u;
    const uint32_t ex = block_exclusive_scan_u32<kT>(own, scan, &total);   // (barriers: B1 read before)
    if (total > uint32_t(h.cap)) {   // cannot happen: the launcher sizes cap for the longest history
        if (tid == 0) { h.hhead[2 * row] = 0u; h.hhead[2 * row + 1] = flags | VI_FLAG_ERROR; }
        return;
    }
    {
        uint32_t r = ex;
        for (int i = tid; i < W; i += kT) { B1[i] = r; r += uint32_t(__builtin_popcount(B2[i])); }
    }
    for (uint32_t i = tid; i < total; i += kT) {
        if (LDS) cnt[i] = 0u;
        else __hip_atomic_store(&cnt[i], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    sync();
    for (int64_t base = b; base < e; base += int64_t(kHistBatch) * kT) {
        if (!one_batch) load(base);
#pragma unroll
        for (int j0 = 0; j0 < kHistBatch; j0 += kHistBatch / 2) {   // (half a batch at a time: registers)
            uint32_t wd[kHistBatch / 2], r0[kHistBatch / 2];
#pragma unroll
            for (int j = 0; j < kHistBatch / 2; ++j) {
                const int32_t tj = t[j0 + j];
                const bool ok = tj >= 0 && tj < V;
                wd[j] = ok ? B2[tj >> 5] : 0u;
                r0[j] = ok ? B1[tj >> 5] : 0u;
            }
#pragma unroll
            for (int j = 0; j < kHistBatch / 2; ++j) {
                const uint32_t bit = 1u << (t[j0 + j] & 31);
                if (wd[j] & bit) atomicAdd(&cnt[r0[j] + uint32_t(__builtin_popcount(wd[j] & (bit - 1u)))], 1u);
            }
        }
    }
    sync();
    uint2* lst = h.hlist + size_t(row) * h.cap;
    for (int i = tid; i < W; i += kT) {
        uint32_t wd = B2[i], r = B1[i];
        while (wd) {
            const int j = __builtin_ctz(wd);
            wd &= wd - 1u;
            lst[r] = make_uint2(uint32_t(32 * i + j), LDS ? cnt[r] : load_agent(&cnt[r]));
            ++r;
        }
    }
    if (tid == 0) { h.hhead[2 * row] = total; h.hhead[2 * row + 1] = flags; }
}

// ------------------------------------------------------------ probabilities
// The filtered distribution of each row: exp(z - z0) / S_n on the support, 0
// elsewhere.  Bound by the memory: 2 bytes read and 4 written per logit.  Four
// consecutive logits per lane and round (8-byte loads and 16-byte stores, whole
// lines per wave), every round's loads requested first.  A wave's history tokens
// are listed over all its rounds and penalized one per lane with count 1 (where
// they lie, nearly every wave would run the penalty for nearly every logit of a
// lane); the tokens seen more than once are written again by repeat_probs_kernel.
// (24 x 151,936 bf16, 2,048-token histories: 12.4 us, and 4.6 for the repeats; 48.6 with
// eight logits per thread, each slice's penalties rebuilt in LDS and end-key ranks
// counted.  Two rounds: with a cheaper exponential, 24 / 128 rows took 11.7 / 38.3 us,
// 11.0 / 40.5 with one round, 14.0 / 40.4 with four.)
constexpr int kPT = 256;                          // threads
constexpr int kPRounds = 2;
constexpr int kPChunk = kPT * kPRounds * 4;       // logits per workgroup

// p of a logit with (penalized) pattern pat
template <int DT>
__device__ __forceinline__ float pattern_prob(uint32_t pat, int id, const FullBound& B, double inv_s) {
    const uint32_t k = key16(pat);
    const float z = Elem<DT>::decode(unkey16(k)) * B.inv_t;
    const bool in = Elem<DT>::finite_bits(pat) && isfinite(z) && (k > B.end_key || (k == B.end_key && id <= B.end_id));
    return in ? float(exp(double(z) - B.z0) * inv_s) : 0.0f;
}

template <int DT>
__global__ __launch_bounds__(kPT) void probs_kernel(StreamArgs a) {
    typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
    typedef u32x2_t u32x2_any_t __attribute__((aligned(2)));
    typedef float f32x4_t __attribute__((ext_vector_type(4)));
    typedef f32x4_t f32x4_any_t __attribute__((aligned(4)));
    __shared__ __attribute__((aligned(16))) u32x2_t stage_all[kPT / kWave][kPRounds * kWave];
    __shared__ uint16_t list_all[kPT / kWave][kPRounds * kWave * 4];
    const int row = blockIdx.y, V = a.vocabulary, lane = lane_id(), wave = int(threadIdx.x) / kWave;
    const vi_row_params p = a.params[row];
    if (!stream_row(p)) return;
    const FullBound B = a.bounds[row];
    const PenView pv = pen_view(a, row, p);
    const uint16_t* row16 = reinterpret_cast<const uint16_t*>(static_cast<const unsigned char*>(a.logits) +
                                                              2 * size_t(row) * size_t(a.stride));
    float* out = a.probs + size_t(row) * size_t(a.probs_stride);
    const int i0 = int(blockIdx.x) * kPChunk + 4 * int(threadIdx.x);
    u32x2_t v[kPRounds];
    uint32_t b[kPRounds];
#pragma unroll
    for (int r = 0; r < kPRounds; ++r) {
        const int i = i0 + r * 4 * kPT;
        v[r] = u32x2_t{0u, 0u};
        b[r] = 0u;
        if (i + 4 <= V) v[r] = *reinterpret_cast<const u32x2_any_t*>(row16 + i);
        if (pv.pen && i < V) b[r] = (uint32_t(pv.b1[i >> 3]) >> (i & 4)) & 0xfu;
    }
    const float inv_r = rep_inverse(p);
    const bool rep_fast = rep_fast_ok(p);
    const double inv_s = B.valid ? 1.0 / B.s_n : 0.0;
    if (pv.pen && B.valid) {   // (uniform)
        u32x2_t* stage = stage_all[wave];
        uint16_t* stage16 = reinterpret_cast<uint16_t*>(stage);
        uint16_t* list = list_all[wave];
        uint32_t m = 0u;   // bit 4 r + j: logit j of round r
#pragma unroll
        for (int r = 0; r < kPRounds; ++r) {
            if (i0 + r * 4 * kPT + 4 <= V) m |= b[r] << (4 * r);
            stage[r * kWave + lane] = v[r];
        }
        const uint32_t n = uint32_t(__builtin_popcount(m)), incl = wave_incl_scan_u32(n), N = readlane_u(incl, kWave - 1);
        uint32_t pos = incl - n;
        while (m) {
            const uint32_t t = uint32_t(__builtin_ctz(m));
            list[pos++] = uint16_t((t >> 2) * (4 * kWave) + 4u * uint32_t(lane) + (t & 3u));
            m &= m - 1u;
        }
        wave_lds_fence();
        for (uint32_t q = uint32_t(lane); q < N; q += kWave) {
            const uint32_t off = list[q];
            stage16[off] = uint16_t(pen_pattern<DT>(stage16[off], 1u, p, inv_r, rep_fast));
        }
        wave_lds_fence();
#pragma unroll
        for (int r = 0; r < kPRounds; ++r) v[r] = stage[r * kWave + lane];
    }
#pragma unroll
    for (int r = 0; r < kPRounds; ++r) {
        const int i = i0 + r * 4 * kPT;
        if (i + 4 <= V) {
            f32x4_t q = {0.0f, 0.0f, 0.0f, 0.0f};
            if (B.valid) {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    q[j] = pattern_prob<DT>((j & 1) ? v[r][j >> 1] >> 16 : v[r][j >> 1] & 0xffffu, i + j, B, inv_s);
            }
            *reinterpret_cast<f32x4_any_t*>(out + i) = q;
        } else {   // (up to three logits past the row's last four)
            for (int j = i; j < V; ++j) {
                uint32_t raw = uint32_t(row16[j]);
                if ((b[r] >> (j - i)) & 1u) raw = pen_pattern<DT>(raw, 1u, p, inv_r, rep_fast);
                out[j] = B.valid ? pattern_prob<DT>(raw, j, B, inv_s) : 0.0f;
            }
        }
    }
}

// The tokens seen more than once, with their counts (one workgroup per row,
// after probs_kernel); then, with `record`, the row's token into its lane's
// state: the distribution is the one before that occurrence.
template <int DT>
__global__ __launch_bounds__(kPT) void repeat_probs_kernel(StreamArgs a) {
    const int row = blockIdx.x, tid = threadIdx.x;
    const vi_row_params p = a.params[row];
    if (!stream_row(p)) return;
    const FullBound B = a.bounds[row];
    const PenView pv = pen_view(a, row, p);
    const uint16_t* row16 = reinterpret_cast<const uint16_t*>(static_cast<const unsigned char*>(a.logits) +
                                                              2 * size_t(row) * size_t(a.stride));
    float* out = a.probs + size_t(row) * size_t(a.probs_stride);
    if (pv.pen && B.valid) {   // (uniform)
        const float inv_r = rep_inverse(p);
        const bool rep_fast = rep_fast_ok(p);
        const double inv_s = 1.0 / B.s_n;
        for (uint32_t i = uint32_t(tid); i < pv.nrep; i += kPT) {
            const uint2 e = pv.list[i];
            if (e.y < 2u || e.x >= uint32_t(a.vocabulary)) continue;
            out[e.x] = pattern_prob<DT>(pen_pattern<DT>(uint32_t(row16[e.x]), e.y, p, inv_r, rep_fast), int(e.x), B, inv_s);
        }
    }
    if (a.record && a.pstate) {
        __syncthreads();   // (the list has been read)
        const int32_t tok = a.tokens[row];
        if (tid == 0 && tok >= 0 && tok < a.vocabulary) {
            const LaneState ls = lane_state(const_cast<unsigned char*>(a.pstate) + size_t(row) * a.pl.lane_bytes, a.pl);
            state_record_one(ls, a.pl, a.vocabulary, tok);
        }
    }
}

}  // namespace

// ------------------------------------------------------------------ host
constexpr int kShortestPart = 12288;   // tokens of a bf16 part, unless the row has fewer (fp16: twice that)

struct StreamPlan {
    int parts, part_len;
};
static StreamPlan stream_plan(int rows, int vocabulary, int dtype) {
    const int cus = device_cus();
    int parts = (vocabulary + kMaxPartLen - 1) / kMaxPartLen;
    const int fill = (cus + std::max(rows, 1) - 1) / std::max(rows, 1);   // parts that give every CU one
    // Few rows: as many parts as the CUs take, but none so short that the merge,
    // one workgroup per row that reads every part's table, loses more than the
    // stream wins.  fp16 rows spread over some hundred groups a part, bf16 rows
    // over a few dozen.  Stream + merge, us, with 16 / 8 / 4 parts: fp16 2 x
    // 162,880 8.8 + 43.2 / 10.5 + 34.1 / 12.8 + 30.6; bf16 8 x 248,320 9.5 + 19.8 /
    // 11.0 + 19.8 / 15.0 + 20.1; bf16 3 x 45,568 6.4 + 16.9 / 6.3 + 15.8 / 6.4 + 14.7.
    const int shortest = dtype == VI_F16 ? 2 * kShortestPart : kShortestPart;
    parts = std::max(parts, std::min({kMaxParts, fill, vocabulary / shortest}));
    // a multiple of 32 tokens: every part's presence bytes start 4-byte aligned
    const int len = ((vocabulary + parts - 1) / parts + 31) / 32 * 32;
    return {(vocabulary + len - 1) / len, len};
}
// Most parts of a launch of up to `rows` rows (stream_plan's, whatever the count
// of rows up to that: a workspace for more rows serves fewer).
static size_t stream_parts_most(int rows, int vocabulary) {
    const size_t r = size_t(rows), least = size_t(vocabulary + kMaxPartLen - 1) / kMaxPartLen;
    const size_t split = std::min<size_t>(kMaxParts, size_t(vocabulary / kShortestPart));
    return std::max(r * least, std::min(r * split, size_t(device_cus()) + r));
}

// The stream launch: workgroups and XCD-aware mapping.
struct StreamGrid {
    int grid, xcd;
};
static StreamGrid stream_grid(int rows, int parts) {
    StreamGrid g;
    g.grid = std::min(device_cus(), rows * parts);
    g.xcd = (rows >= kXcds && g.grid % kXcds == 0) ? 1 : 0;
    return g;
}

static int hist_words(int vocabulary) { return (vocabulary + 31) / 32; }
// tokens of a history that can be seen more than once
static int hist_cap(int vocabulary, int64_t max_history) {
    return int(std::max<int64_t>(std::min<int64_t>(max_history / 2, vocabulary), 1));
}
// words of LDS that the bitmaps and counts take
static int hist_lds(int vocabulary, int64_t max_history) {
    return 2 * hist_words(vocabulary) + hist_cap(vocabulary, max_history);
}
template <int WORDS>
static void launch_history_view(const HistArgs& h, int rows, int64_t max_history, hipStream_t stream) {
    auto* kernel = max_history <= 4 * kT    ? &history_view_kernel<WORDS, 4>
                   : max_history <= 8 * kT  ? &history_view_kernel<WORDS, 8>
                   : max_history <= 16 * kT ? &history_view_kernel<WORDS, 16>
                                            : &history_view_kernel<WORDS, kHistLong>;
    hipLaunchKernelGGL(kernel, dim3(rows), dim3(kT), 0, stream, h);
}

// Rows per launch: as many as keep a workgroup's parts within kMaxItems and the
// probabilities' grid within its limit (a multiple of 8: each XCD's rows the
// same); more rows than that take several launches, over the same tables.
static int stream_chunk(int rows, int parts) {
    const int most = std::min((kMaxItems - 1) * device_cus() / parts, 32768) / kXcds * kXcds;
    return std::min(rows, most);
}

bool stream_supported(int dtype, int vocabulary, int64_t stride) {
    return (dtype == VI_BF16 || dtype == VI_F16) && vocabulary > 0 && vocabulary <= kMaxVocabulary && stride >= vocabulary;
}

size_t stream_workspace(int rows, int vocabulary, int64_t max_history) {
    if (rows <= 0 || vocabulary <= 0 || vocabulary > kMaxVocabulary) return 0;
    const size_t np = stream_parts_most(std::min(rows, stream_chunk(rows, 1)), vocabulary), r = size_t(rows);
    size_t b = align_up(np * kPub * 4, 256) + align_up(np * kGroups * kGW * 4, 256) + align_up(r * sizeof(FullBound), 256);
    if (max_history > 0) {
        const size_t words = size_t(hist_words(vocabulary)), cap = size_t(hist_cap(vocabulary, max_history));
        b += align_up(r * words * 4, 256) + align_up(r * cap * 8, 256) + align_up(r * 8, 256);
        if (hist_lds(vocabulary, max_history) > kHistLdsWords) b += align_up(r * cap * 4, 256);
    }
    return b + 256;
}

template <int DT>
static void launch_rows(const StreamArgs& a, hipStream_t stream) {
    const bool pen = a.pstate || a.hb1;
    if (pen) hipLaunchKernelGGL((stream_kernel<DT, true>), dim3(a.grid), dim3(kT), 0, stream, a);
    else hipLaunchKernelGGL((stream_kernel<DT, false>), dim3(a.grid), dim3(kT), 0, stream, a);
    // the merge's workgroup of row r runs on the XCD whose workgroups streamed
    // the row (workgroup r goes to XCD r % 8, as the stream's rows do)
    hipLaunchKernelGGL(merge_kernel<DT>, dim3(a.rows), dim3(kT), 0, stream, a);
    if (!a.probs) return;
    hipLaunchKernelGGL(probs_kernel<DT>, dim3((a.vocabulary + kPChunk - 1) / kPChunk, a.rows), dim3(kPT), 0, stream, a);
    if (pen) hipLaunchKernelGGL(repeat_probs_kernel<DT>, dim3(a.rows), dim3(kPT), 0, stream, a);
}

vi_status launch_stream(const SampleArgs& s, unsigned char* ws, size_t ws_bytes, hipStream_t stream) {
    if (!stream_supported(s.dtype, s.vocabulary, s.stride)) return VI_ERR_UNSUPPORTED;
    if (reinterpret_cast<uintptr_t>(s.logits) % 16) return VI_ERR_UNSUPPORTED;
    if (s.rows <= 0) return VI_OK;
    const StreamPlan pl = stream_plan(s.rows, s.vocabulary, s.dtype);
    const int chunk = stream_chunk(s.rows, pl.parts);
    StreamArgs a{};
    a.vocabulary = s.vocabulary; a.stride = s.stride;
    a.parts = pl.parts; a.part_len = pl.part_len;
    const size_t np = size_t(chunk) * pl.parts;
    Carver c(ws, ws_bytes);
    a.ppub = c.take<uint32_t>(np * kPub);
    a.pwords = c.take<uint4>(np * kGroups * (kGW / 4));
    FullBound* bounds = c.take<FullBound>(size_t(s.rows));
    if (s.full_out) bounds = s.full_out->bounds;
    else if (!s.probs) bounds = nullptr;
    a.draw_every = s.full_out ? s.full_out->draw_every : 1;
    const bool hist = !s.pstate && s.histories && s.offsets && s.max_history > 0;
    HistArgs h{};
    if (hist) {
        h.histories = s.histories; h.offsets = s.offsets; h.vocabulary = s.vocabulary;
        h.words = hist_words(s.vocabulary);
        h.cap = hist_cap(s.vocabulary, s.max_history);
        h.hb1 = c.take<uint32_t>(size_t(s.rows) * h.words);
        h.hlist = c.take<uint2>(size_t(s.rows) * h.cap);
        h.hhead = c.take<uint32_t>(size_t(s.rows) * 2);
        if (hist_lds(s.vocabulary, s.max_history) > kHistLdsWords)
            h.tmp = c.take<uint32_t>(size_t(s.rows) * size_t(h.cap));
        a.hwords = h.words; a.hcap = h.cap;
    }
    if (!c.ok) return VI_ERR_WORKSPACE;
    if (hist) {
        if (h.tmp) hipLaunchKernelGGL((history_view_kernel<kHistLdsBits, kHistLong>), dim3(s.rows), dim3(kT), 0, stream, h);
        else if (hist_lds(s.vocabulary, s.max_history) <= kHistLdsHalf) launch_history_view<kHistLdsHalf>(h, s.rows, s.max_history, stream);
        else launch_history_view<kHistLdsWords>(h, s.rows, s.max_history, stream);
        if (launch_status() != VI_OK) return VI_ERR_LAUNCH;
    }
    for (int r0 = 0; r0 < s.rows; r0 += chunk) {
        const size_t at = size_t(r0);
        a.row0 = r0;
        a.rows = std::min(chunk, s.rows - r0);
        a.logits = static_cast<const unsigned char*>(s.logits) + 2 * at * size_t(s.stride);
        a.params = s.params + at;
        a.tokens = s.tokens + at;
        if (s.uniforms) a.uniforms = s.uniforms + at;
        if (s.stats) a.stats = s.stats + at;
        if (bounds) a.bounds = bounds + at;
        if (s.probs) { a.probs = s.probs + at * size_t(s.probs_stride); a.probs_stride = s.probs_stride; }
        if (s.pstate) {
            a.pl = s.playout;
            a.pstate = s.pstate + at * s.playout.lane_bytes;
            a.record = s.record;
        } else if (hist) {
            a.hb1 = h.hb1 + at * size_t(h.words);
            a.hlist = h.hlist + at * size_t(h.cap);
            a.hhead = h.hhead + 2 * at;
        }
        const StreamGrid sg = stream_grid(a.rows, pl.parts);
        a.grid = sg.grid;
        a.xcd = sg.xcd;
        if (s.dtype == VI_BF16) launch_rows<VI_BF16>(a, stream);
        else launch_rows<VI_F16>(a, stream);
        if (launch_status() != VI_OK) return VI_ERR_LAUNCH;
    }
    return VI_OK;
}

}  // namespace vi
