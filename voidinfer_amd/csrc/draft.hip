// draft.hip — the DFlash2 draft's proposals: the coupled sampled choice
// (DraftSelectSampling / dflash_sampled_choice, src/exl3/dflash2_draft.cu:2554-2610)
// over given scores, and the fused selector chain that computes the scores
// (dflash_selector_fused_chain_kernel, :2615-2678).
//
// Each lane proposes one token per draft position from that position's 16
// candidates, in position order (an earlier proposal is part of the presence
// history of the later ones).  With inv_temperature > 0 the proposal is the
// token the target's coupled sampler most likely picks: the candidates'
// presence-penalized scores are ordered (stable, score descending), truncated
// like the target sampler (top_k, then min_p / top_p of exp(score/T - max))
// and the argmax of score/T + Gumbel(seed, key_base + position, token) over the
// support wins.  Otherwise the raw scores' first maximum wins.  One thread per
// lane; the per-thread candidate arrays live in LDS.
#include <math.h>

#include <algorithm>

#include "vi_device.h"
#include "vi_internal.h"

namespace vi {
namespace {

constexpr int kDraftK = 16;       // candidates per draft position
constexpr int kDraftLanes = 64;   // lanes per workgroup

// The coupled sampled choice at one draft position (dflash_sampled_choice,
// src/exl3/dflash2_draft.cu:2570-2610): index of the chosen candidate.  `chain`
// holds the `pos` earlier proposals; val / prob / order are per-thread LDS rows.
__device__ __forceinline__ int sampled_pick(const vi_draft_sampling& s, int pos, int vocabulary, const float* sc,
                                            const int64_t* cd, int64_t seed_token, const int64_t* chain, float* val,
                                            float* prob, int* order) {
    const int key = s.key_base + pos;
    for (int c = 0; c < kDraftK; ++c) {
        float v = sc[c];
        if (s.presence_penalty != 0.0f) {
            const int64_t token = cd[c];
            bool seen = token == seed_token ||
                        (s.first_occurrence && token >= 0 && token < vocabulary && s.first_occurrence[token] < key);
            for (int i = 0; i < pos && !seen; ++i) seen = chain[i] == token;
            if (seen) v -= s.presence_penalty;
        }
        val[c] = v;
        order[c] = c;
    }
    for (int i = 1; i < kDraftK; ++i) {   // stable insertion sort, score descending
        const int o = order[i];
        int j = i;
        while (j > 0 && val[o] > val[order[j - 1]]) { order[j] = order[j - 1]; --j; }
        order[j] = o;
    }
    int cap = kDraftK;
    if (s.top_k > 0 && s.top_k < cap) cap = s.top_k;
    const float m = val[order[0]] * s.inv_temperature;
    float sum = 0.0f;
    for (int j = 0; j < cap; ++j) { prob[j] = expf(fmaf(val[order[j]], s.inv_temperature, -m)); sum += prob[j]; }
    const float min_p_thresh = s.min_p > 0.0f ? s.min_p * prob[0] : -1.0f;
    float cum = 0.0f;
    int support = 0;
    for (int j = 0; j < cap; ++j) {
        if (min_p_thresh >= 0.0f && prob[j] < min_p_thresh) break;
        cum += prob[j];
        support = j + 1;
        if (s.top_p < 1.0f && cum >= s.top_p * sum) break;
    }
    if (support < 1) support = 1;
    int best = order[0];
    float best_value = -kInfF;
    for (int j = 0; j < support; ++j) {
        const int c = order[j];
        const float v = fmaf(val[c], s.inv_temperature, gumbel(s.seed, key, int(cd[c])));
        if (v > best_value) { best_value = v; best = c; }
    }
    return best;
}

// First maximum of 16 scores (NaN never replaces the incumbent).
__device__ __forceinline__ int first_max16(const float* sc) {
    int best = 0;
    float bs = sc[0];
    for (int c = 1; c < kDraftK; ++c)
        if (sc[c] > bs) { bs = sc[c]; best = c; }
    return best;
}

__global__ __launch_bounds__(kDraftLanes) void draft_choice_kernel(int lanes, int positions, int vocabulary,
                                                                  const float* scores, const int64_t* candidates,
                                                                  const int64_t* seed_tokens,
                                                                  const vi_draft_sampling* sampling,
                                                                  int64_t* proposals) {
    __shared__ float s_val[kDraftLanes][kDraftK + 1];
    __shared__ float s_prob[kDraftLanes][kDraftK + 1];
    __shared__ int s_ord[kDraftLanes][kDraftK + 1];
    const int t = threadIdx.x, l = blockIdx.x * kDraftLanes + t;
    if (l >= lanes) return;
    const vi_draft_sampling s = sampling[l];
    const int64_t seed_token = seed_tokens ? seed_tokens[l] : -1;
    int64_t* out = proposals + size_t(l) * positions;
    for (int pos = 0; pos < positions; ++pos) {
        const size_t at = (size_t(l) * positions + pos) * kDraftK;
        const float* sc = scores + at;
        const int64_t* cd = candidates + at;
        const int best = s.inv_temperature > 0.0f
                             ? sampled_pick(s, pos, vocabulary, sc, cd, seed_token, out, s_val[t], s_prob[t], s_ord[t])
                             : first_max16(sc);
        out[pos] = cd[best];
    }
}

// The fused selector chain (dflash_selector_fused_chain_kernel,
// src/exl3/dflash2_draft.cu:2615-2678): per draft position, candidate c's
// score is unary[c] + sum_r pred[anchor][r] * hidden[pos][r] * succ[cand_c][r]
// (rank 256, fp16 codebooks, fp32 arithmetic, each product rounded as
// (pred * hidden) * succ), and the first maximum becomes the proposal and the
// next position's anchor.  With inv_temperature > 0 the coupled sampled choice
// over the unary scores decides instead (the selector's terms are not
// calibrated as logits).
//
// Bound: latency.  The chain is serial (a position's anchor is the one before's
// choice), but everything it reads is known beforehand: position p's possible
// anchors are position p - 1's candidates.  So one workgroup takes a lane and
// requests a whole chunk of positions at once: the candidates' succ rows and the
// hidden rows into registers, their pred rows on to LDS.  The serial part is then
// one LDS read of the anchor's row, the dots, one barrier and a 16-lane maximum
// per position.
// Four waves, each four candidates (a CU has four SIMDs: more waves would repeat
// the maximum on the same issue slots).  Lane k of a wave holds ranks
// 4k .. 4k + 3; the candidate sums are reduced across the wave with DPP in a
// fixed order.  That order is this kernel's own; near ties may therefore resolve
// differently from another order, within the sums' rounding.  Measured, 8 lanes x
// 16 positions over a 248,320-token codebook: 14.9 us per call, 47.4 with one wave per
// lane loading each position after the one before.
constexpr int kRank = 256;
constexpr int kChainWaves = 4;
constexpr int kChainThreads = kChainWaves * kWave;
constexpr int kRanksPerLane = kRank / kWave;       // 4
constexpr int kChainMax = 16;                      // positions per chunk (the largest)
static_assert(kRanksPerLane == 4, "four fp16 ranks = one 8-byte load");
static_assert(kDraftK == 4 * kChainWaves, "four candidates per wave");

__device__ __forceinline__ float4 decode4(uint2 v) {
    return make_float4(Elem<VI_F16>::decode(v.x & 0xffffu), Elem<VI_F16>::decode(v.x >> 16),
                       Elem<VI_F16>::decode(v.y & 0xffffu), Elem<VI_F16>::decode(v.y >> 16));
}
// ranks 4k .. 4k + 3 of an fp16 row
__device__ __forceinline__ uint2 rank4(const uint16_t* row, int k) {
    return *reinterpret_cast<const uint2*>(row + kRanksPerLane * k);
}
// Index of the first maximum of 16 scores held one per lane in every 16-lane
// row (score[0] wins if it is NaN; another NaN never wins): the serial rule
// "replace when greater" as a maximum over order keys.
__device__ __forceinline__ int first_max16_lanes(float score, int c) {
    const uint32_t b = __builtin_bit_cast(uint32_t, score + 0.0f);   // -0 and +0 compare equal
    const bool nan = (b & 0x7fffffffu) > 0x7f800000u;
    const uint32_t key = nan ? (c == 0 ? 0xffffffffu : 0u) : ((b & 0x80000000u) ? ~b : (b | 0x80000000u));
    uint32_t m = key;
    m = max(m, lanes_xor_dpp<1>(m));
    m = max(m, lanes_xor_dpp<2>(m));
    m = max(m, lanes_xor_dpp<4>(m));
    m = max(m, lanes_xor_dpp<8>(m));
    return __builtin_ctzll(ballot(key == m));
}

// CH: positions per chunk.  GROUPS: the first groups of the grid take the sampled
// lanes, one per wave, and a workgroup per lane the others; else every lane has a
// workgroup.
template <int CH, bool GROUPS>
__global__ __launch_bounds__(kChainThreads) void selector_chain_kernel(
    int lanes, int positions, int vocabulary, const int64_t* anchors, const int64_t* candidates, const float* unary,
    const uint16_t* hidden, const uint16_t* pred_cb, const uint16_t* succ_cb, const vi_draft_sampling* sampling,
    int64_t* proposals) {
    __shared__ __attribute__((aligned(16))) uint16_t s_pred[CH][kDraftK][kRank];
    __shared__ int s_cand[CH][kDraftK];
    __shared__ float s_unary[CH][kDraftK];
    __shared__ __attribute__((aligned(16))) float s_score[2][kDraftK];
    __shared__ int s_valid[kChainWaves];
    constexpr int kSerial = GROUPS ? kChainWaves : 1;   // sampled lanes of a workgroup
    __shared__ float s_val[kSerial][kDraftK + 1], s_prob[kSerial][kDraftK + 1];
    __shared__ int s_ord[kSerial][kDraftK + 1];
    const int t = threadIdx.x, w = t / kWave, k = lane_id();
    int l = blockIdx.x;
    if constexpr (GROUPS) {
        const int groups = (lanes + kChainWaves - 1) / kChainWaves;
        const bool group = l < groups;
        l = group ? l * kChainWaves + w : l - groups;
        if (l >= lanes || (sampling[l].inv_temperature > 0.0f) != group) return;   // (whole waves; a group has no barrier)
    }
    const int64_t seed_token = anchors[l];
    int64_t* out = proposals + size_t(l) * positions;
    const int64_t* lane_cand = candidates + size_t(l) * positions * kDraftK;
    const float* lane_unary = unary + size_t(l) * positions * kDraftK;
    bool bad = seed_token < 0 || seed_token >= vocabulary;   // ends the chain (workgroup-uniform)
    if (sampling && sampling[l].inv_temperature > 0.0f) {
        // the coupled choice over the unary scores: serial, one wave
        if (!GROUPS && w != 0) return;
        const int own = GROUPS ? w : 0;
        const vi_draft_sampling smp = sampling[l];
        for (int pos = 0; pos < positions; ++pos) {
            const int64_t* cd = lane_cand + size_t(pos) * kDraftK;
            const int64_t mine = cd[k & (kDraftK - 1)];
            bad = bad || ballot(mine < 0 || mine >= vocabulary) != 0;
            if (k != 0) continue;
            if (bad) { out[pos] = -1; continue; }
            const int best = sampled_pick(smp, pos, vocabulary, lane_unary + size_t(pos) * kDraftK, cd, seed_token, out,
                                          s_val[own], s_prob[own], s_ord[own]);
            out[pos] = cd[best];
        }
        return;
    }
    // pred[anchor] of the current position (ranks 4k .. 4k + 3)
    uint2 pa = rank4(pred_cb + size_t(bad ? 0 : seed_token) * kRank, k);
    for (int p0 = 0; p0 < positions; p0 += CH) {
        // the chunk's candidates and unary scores, and the positions up to the
        // first invalid candidate
        const int n = min(CH, positions - p0);
        int firstbad = CH;
        for (int i = t; i < CH * kDraftK; i += kChainThreads) {
            const int p = i / kDraftK, c = i % kDraftK;
            const bool in = p < n;
            const size_t at = size_t(p0 + (in ? p : n - 1)) * kDraftK + c;
            const int64_t id = lane_cand[at];
            const bool ok = id >= 0 && id < vocabulary;
            if (in && !ok) firstbad = min(firstbad, p);
            s_cand[p][c] = ok ? int(id) : 0;
            s_unary[p][c] = lane_unary[at];
        }
#pragma unroll
        for (int m = 1; m < kWave; m <<= 1) firstbad = min(firstbad, __shfl_xor(firstbad, m, kWave));
        if (k == 0) s_valid[w] = firstbad;
        __syncthreads();   // (and the previous chunk's LDS rows are free)
        int valid = bad ? 0 : n;
#pragma unroll
        for (int i = 0; i < kChainWaves; ++i) valid = min(valid, s_valid[i]);
        valid = __builtin_amdgcn_readfirstlane(valid);
        bad = bad || valid < n;
        if (t >= valid && t < n) out[p0 + t] = -1;   // n <= the workgroup's threads
        if (valid == 0) { __syncthreads(); continue; }
        // every row of the chunk in flight (positions past the end repeat the last
        // one's; never used)
        uint2 h[CH], sv[CH][4], pv[CH][4];
#pragma unroll
        for (int p = 0; p < CH; ++p) {
            const int q = min(p, valid - 1);
            h[p] = rank4(hidden + (size_t(l) * positions + size_t(p0 + q)) * kRank, k);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const size_t id = size_t(s_cand[q][4 * w + j]);
                sv[p][j] = rank4(succ_cb + id * kRank, k);
                pv[p][j] = rank4(pred_cb + id * kRank, k);
            }
        }
#pragma unroll
        for (int p = 0; p < CH; ++p)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                *reinterpret_cast<uint2*>(&s_pred[p][4 * w + j][kRanksPerLane * k]) = pv[p][j];
        __syncthreads();
#pragma unroll
        for (int p = 0; p < CH; ++p) {
            if (p >= valid) continue;   // (workgroup-uniform)
            const float4 a = decode4(pa), hh = decode4(h[p]);
            const float4 ah = make_float4(a.x * hh.x, a.y * hh.y, a.z * hh.z, a.w * hh.w);
            float sc[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float4 s = decode4(sv[p][j]);
                sc[j] = wave_sum_f32((ah.x * s.x + ah.y * s.y) + (ah.z * s.z + ah.w * s.w));
            }
            if (k == 0) *reinterpret_cast<float4*>(&s_score[p & 1][4 * w]) = make_float4(sc[0], sc[1], sc[2], sc[3]);
            __syncthreads();
            const int c = k & (kDraftK - 1);
            const int best = first_max16_lanes(s_unary[p][c] + s_score[p & 1][c], c);
            pa = *reinterpret_cast<const uint2*>(&s_pred[p][best][kRanksPerLane * k]);   // the next anchor's row
            if (t == 0) out[p0 + p] = s_cand[p][best];
        }
        __syncthreads();   // the chunk's rows are read
    }
}
}  // namespace

vi_status launch_draft_choice(int lanes, int positions, int vocabulary, const float* scores,
                              const int64_t* candidates, const int64_t* seed_tokens,
                              const vi_draft_sampling* sampling, int64_t* proposals, hipStream_t stream) {
    hipLaunchKernelGGL(draft_choice_kernel, dim3((lanes + kDraftLanes - 1) / kDraftLanes), dim3(kDraftLanes), 0,
                       stream, lanes, positions, vocabulary, scores, candidates, seed_tokens, sampling, proposals);
    return launch_status();
}

vi_status launch_selector_chain(int lanes, int positions, int vocabulary, const int64_t* anchors,
                                const int64_t* candidates, const float* unary, const void* hidden,
                                const void* pred_codebook, const void* succ_codebook,
                                const vi_draft_sampling* sampling, int64_t* proposals, hipStream_t stream) {
    // The smallest chunk that holds the chain (its rows are all requested at once),
    // unless its LDS leaves lanes waiting for a CU: one workgroup fits a CU with 16
    // positions, two with 8, four with 4.  (16 positions, us, chunks of 16 / by this
    // rule: 512 lanes 39 / 28, 1,024 lanes 74 / 42, 4,096 lanes 277 / 153.)
    // A sampled lane works with one thread: past what the CUs hold at once, four of
    // them share a workgroup.  (All sampled, a workgroup each with chunks of 16 / by
    // this rule: 512 lanes 314 / 172, 1,024 lanes 624 / 181, 4,096 lanes 2,458 / 213.)
    const int cus = device_cus(), most = lanes <= cus ? kChainMax : lanes <= 2 * cus ? 8 : 4;
    const int chunk = std::min(positions <= 4 ? 4 : positions <= 8 ? 8 : kChainMax, most);
    const bool groups = sampling && lanes > 4 * cus;
    auto* kernel = groups       ? &selector_chain_kernel<4, true>
                   : chunk == 4 ? &selector_chain_kernel<4, false>
                   : chunk == 8 ? &selector_chain_kernel<8, false>
                                : &selector_chain_kernel<kChainMax, false>;
    const int extra = groups ? (lanes + kChainWaves - 1) / kChainWaves : 0;
    hipLaunchKernelGGL(kernel, dim3(extra + lanes), dim3(kChainThreads), 0, stream, lanes, positions, vocabulary,
                       anchors, candidates, unary, static_cast<const uint16_t*>(hidden),
                       static_cast<const uint16_t*>(pred_codebook), static_cast<const uint16_t*>(succ_codebook),
                       sampling, proposals);
    return launch_status();
}

}  // namespace vi
