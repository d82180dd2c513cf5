// Wave-level donor selection (one 64-lane wavefront per row).
//
// Restates the reference's two selectors, which agree by construction:
// codec.py:137-178 (_reuse_map, torch) and triton_selection.py:11-43 (_select).
//   1. sources = the `count` channels of largest saliency, ties to the lower
//      channel (stable descending argsort), listed in ascending order;
//   2. min_error: only the `count` non-source channels of smallest donor
//      error (ties to the lower channel) may donate; otherwise every
//      non-source channel may;
//   3. for each source s in ascending order: candidates are the available
//      immediate neighbours s-1, s+1; if none, the available channels at the
//      smallest distance from either boundary of s's contiguous salient run;
//      the donor is the candidate of least saliency, lowest channel on ties.
// Saliency and error are non-negative, so their IEEE bit patterns order them.
#pragma once

#include "iq_common.h"

#include <type_traits>

#define IQ_MAXD 1024
#define IQ_MAXCHUNK (IQ_MAXD / 64)

// Total order used by torch's stable sorts on non-NaN floats, as integers.
__device__ __forceinline__ uint32_t iq_nonneg_bits(float f) { return __float_as_uint(f); }

// Marks in out[] the `count` eligible lanes of largest key, ties to the lower
// channel (channel = 64 k + lane), which is the stable descending sort's
// top `count`.  The count-th largest key is found by a bitwise radix search
// over ballots, then ties at that key are taken in channel order.
template <int NC>
__device__ __forceinline__ void iq_wave_top(const uint32_t (&key)[NC], const uint64_t (&elig)[NC], int count,
                                            uint64_t (&out)[NC])
{
    const int lane = threadIdx.x & 63;
    if (count <= 0) {
#pragma unroll
        for (int k = 0; k < NC; ++k) out[k] = 0;
        return;
    }
    uint32_t thr = 0;
    for (int bit = 31; bit >= 0; --bit) {
        const uint32_t cand = thr | (1u << bit);
        int n = 0;
#pragma unroll
        for (int k = 0; k < NC; ++k)
            n += __popcll(__ballot(((elig[k] >> lane) & 1ull) && key[k] >= cand));
        if (n >= count) thr = cand;
    }
    int need = count;
#pragma unroll
    for (int k = 0; k < NC; ++k) {
        out[k] = __ballot(((elig[k] >> lane) & 1ull) && key[k] > thr);
        need -= __popcll(out[k]);
    }
#pragma unroll
    for (int k = 0; k < NC; ++k) {
        uint64_t eq = __ballot(((elig[k] >> lane) & 1ull) && key[k] == thr);
        while (eq && need > 0) {
            const uint64_t low = eq & (~eq + 1);
            out[k] |= low;
            eq ^= low;
            --need;
        }
    }
}

// key[c >> 6] of lane c & 63 (c wave-uniform), read without a cross-lane exchange.
template <int NC>
__device__ __forceinline__ uint32_t lane_key(const uint32_t (&key)[NC], int c)
{
    uint32_t v = 0;
#pragma unroll
    for (int k = 0; k < NC; ++k)
        if ((c >> 6) == k) v = __builtin_amdgcn_readlane(key[k], c & 63);
    return v;
}

// Highest set bit of the NC-word mask strictly below pos, or -1.
template <int NC>
__device__ __forceinline__ int iq_bit_below(const uint64_t (&m)[NC], int pos)
{
    int r = -1;
#pragma unroll
    for (int k = 0; k < NC; ++k) {
        const int base = 64 * k;
        uint64_t w = pos <= base ? 0ull : pos >= base + 64 ? m[k] : m[k] & ((1ull << (pos - base)) - 1);
        if (w) r = base + 63 - __builtin_clzll(w);
    }
    return r;
}

// Lowest set bit of the NC-word mask strictly above pos, or `none`.
template <int NC>
__device__ __forceinline__ int iq_bit_above(const uint64_t (&m)[NC], int pos, int none)
{
    int r = none;
#pragma unroll
    for (int k = NC - 1; k >= 0; --k) {
        const int base = 64 * k;
        uint64_t w = pos >= base + 63 ? 0ull : pos < base ? m[k] : m[k] & ~((2ull << (pos - base)) - 1);
        if (w) r = base + __builtin_ctzll(w);
    }
    return r;
}

__device__ __forceinline__ uint32_t iq_row_min(uint32_t v)      // least of each 16 lanes, in all of them
{
    auto ror = [](uint32_t x, auto n) {
        return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x120 + decltype(n)::value, 0xf, 0xf, false);
    };
    v = min(v, ror(v, std::integral_constant<int, 8>{}));
    v = min(v, ror(v, std::integral_constant<int, 4>{}));
    v = min(v, ror(v, std::integral_constant<int, 2>{}));
    return min(v, ror(v, std::integral_constant<int, 1>{}));
}

// The sequential donor picks of a row whose pool holds exactly `count` <= 16
// channels (the min_error policy), any head size.  src_out lists the sources
// and don_out the pool, both ascending; is_src is 0 and src_of -1 everywhere.
// One wavefront calls it.
//
// A source prefers its free immediate neighbours, then the free channels
// nearest either boundary of its run of sources, on a tie the one of less
// saliency and then the lower channel: an order of the pool that does not
// depend on what is free, so each pick is the least key among the free pool
// members.  Lane m of each row of 16 holds pool member m; a pick is four
// rotations and minima, two compares, and nothing scalar waits for it (the
// source's place is read ahead of the chain).  With the picks by bit scans of
// the free mask below, each a chain of scalar operations and branches, a lone
// wavefront took 7.0 us for the whole selection of 16 sources from 128
// channels; with these 4.4, and the 16-token page encoder 41.7 us instead of
// 51.8 for 32768 tokens of four heads.
__device__ __forceinline__ void iq_pick_pool16(const float *sal, int count, int16_t *src_out, int16_t *don_out,
                                               uint8_t *is_src, int16_t *src_of)
{
    const int lane = threadIdx.x & 63, m = lane & 15;
    const bool has = m < count;
    const int c = has ? don_out[m] : 0, s = has ? src_out[m] : 0;
    const int before = has && m > 0 ? src_out[m - 1] : -2;
    const uint32_t sk = has ? iq_nonneg_bits(sal[c]) : ~0u;
    // rank of the member's saliency in the pool, ties to the lower channel
    uint32_t rank = 0;
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        const uint32_t other = __builtin_amdgcn_readlane(sk, j);
        rank += (other < sk || (other == sk && j < m)) ? 1u : 0u;
    }
    // the run [lb, rb] of neighbouring sources around source m, from the places where runs begin
    const uint32_t begins = (uint32_t)__ballot(has && s != before + 1) & 0xffffu;
    const int first = 31 - __builtin_clz((begins & ((2u << m) - 1)) | 1u);
    const uint32_t later = begins >> (m + 1);
    const int last = later ? m + __builtin_ctz(later) : count - 1;
    const int lb = s - (m - first), rb = s + (last - m);
    const uint32_t place = (uint32_t)s | ((uint32_t)lb << 10) | ((uint32_t)rb << 20);   // channels < 1024
    uint32_t taken = has ? 0u : 1u << 31;
    int to = 0;
    for (int i = 0; i < count; ++i) {
        const uint32_t w = __builtin_amdgcn_readlane(place, i);
        const int si = (int)(w & 1023u), lbi = (int)((w >> 10) & 1023u), rbi = (int)(w >> 20);
        const bool next = c == si - 1 || c == si + 1;
        const uint32_t dist = next ? 0u : (uint32_t)max(lbi - c, c - rbi);
        const uint32_t key = (dist << 4) | rank | taken;
        if (key == iq_row_min(key)) {         // one lane of each row
            taken = 1u << 31;
            to = i;
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    if (lane < count) {
        don_out[to] = (int16_t)c;
        src_of[c] = src_out[to];
        is_src[s] = 1;
    }
}

// sal/err: LDS arrays of D floats (err may be null), D <= 64 * NC.  Outputs
// src/don (count entries each, LDS) and is_src / src_of (LDS, D entries)
// describing roles for the quantizer.  Must be called by exactly one full
// wavefront.  Saliencies and errors stay in registers as their bit patterns.
template <int NC>
__device__ __forceinline__ void iq_select_wave_t(const float *sal, const float *err, int D, int count,
                                 int16_t *src_out, int16_t *don_out, uint8_t *is_src, int16_t *src_of)
{
    const int lane = threadIdx.x & 63;
    uint32_t skey[NC], ekey[NC];
    uint64_t valid[NC], sel_mask[NC], avail_mask[NC];
#pragma unroll
    for (int k = 0; k < NC; ++k) {
        const int c = k * 64 + lane;
        const bool ok = c < D;
        skey[k] = ok ? iq_nonneg_bits(sal[c]) : 0u;
        // ascending error == descending complement of its bit pattern
        ekey[k] = ok && err ? ~iq_nonneg_bits(err[c]) : 0u;
        valid[k] = __ballot(ok);
    }
    // 1. stable top-`count` by saliency
    iq_wave_top<NC>(skey, valid, count, sel_mask);
    // 2. donor pool: every other channel, or the `count` of least error
    uint64_t rest[NC];
#pragma unroll
    for (int k = 0; k < NC; ++k) rest[k] = valid[k] & ~sel_mask[k];
    if (err) iq_wave_top<NC>(ekey, rest, count, avail_mask);
    else
#pragma unroll
        for (int k = 0; k < NC; ++k) avail_mask[k] = rest[k];
    uint64_t nonsel[NC];
#pragma unroll
    for (int k = 0; k < NC; ++k) nonsel[k] = valid[k] & ~sel_mask[k];
    // role tables for the quantizer (filled in as sources are assigned)
    for (int c = lane; c < D; c += 64) {
        is_src[c] = 0;
        src_of[c] = -1;
    }

    // 3. sequential donor picks; sources visited in ascending channel order
    if (err && count <= 16) {
        int ns = 0, np = 0;
#pragma unroll
        for (int k = 0; k < NC; ++k) {
            const uint64_t below = (1ull << lane) - 1;
            if ((sel_mask[k] >> lane) & 1ull) src_out[ns + __popcll(sel_mask[k] & below)] = (int16_t)(64 * k + lane);
            if ((avail_mask[k] >> lane) & 1ull) don_out[np + __popcll(avail_mask[k] & below)] = (int16_t)(64 * k + lane);
            ns += __popcll(sel_mask[k]);
            np += __popcll(avail_mask[k]);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        iq_pick_pool16(sal, count, src_out, don_out, is_src, src_of);
        return;
    }
    int i = 0;
#pragma unroll
    for (int k = 0; k < NC; ++k) {
        uint64_t m = sel_mask[k];
        while (m && i < count) {
            const int bit = __builtin_ctzll(m);
            m &= m - 1;
            const int s = k * 64 + bit;
            const bool left_ok = s - 1 >= 0 && ((avail_mask[(s - 1) >> 6] >> ((s - 1) & 63)) & 1ull);
            const bool right_ok = s + 1 < D && ((avail_mask[(s + 1) >> 6] >> ((s + 1) & 63)) & 1ull);
            int donor = 0;            // an empty pool only arises from non-finite statistics
            if (left_ok || right_ok) {
                // at most two candidates: read their saliencies from their lanes
                // (lower saliency wins, the lower channel on ties)
                const uint32_t kl = left_ok ? lane_key<NC>(skey, s - 1) : ~0u;
                const uint32_t kr = right_ok ? lane_key<NC>(skey, s + 1) : ~0u;
                donor = (!right_ok || (left_ok && kl <= kr)) ? s - 1 : s + 1;
            } else {
                // The run of selected channels around s is [lb, rb]; every
                // available channel lies outside it, so the nearest available
                // channel to either boundary is the highest one below lb or the
                // lowest one above rb (less saliency, then lower channel, on a
                // distance tie).  Bit scans of the uniform masks find both.
                const int lb = iq_bit_below<NC>(nonsel, s) + 1;
                const int rb = iq_bit_above<NC>(nonsel, s, D) - 1;
                const int pl = iq_bit_below<NC>(avail_mask, lb);
                const int pr = iq_bit_above<NC>(avail_mask, rb, D);
                const int dl = pl >= 0 ? lb - pl : 0x7fffffff;
                const int dr = pr < D ? pr - rb : 0x7fffffff;
                if (dl < dr) donor = pl;
                else if (dr < dl) donor = pr;
                else if (dl != 0x7fffffff)
                    donor = lane_key<NC>(skey, pl) <= lane_key<NC>(skey, pr) ? pl : pr;
            }
            avail_mask[donor >> 6] &= ~(1ull << (donor & 63));
            if (lane == 0) {
                is_src[s] = 1;
                src_out[i] = (int16_t)s;
                don_out[i] = (int16_t)donor;
                src_of[donor] = (int16_t)s;
            }
            ++i;
        }
    }
}

// Lanes' versions of iq_bit_below / iq_bit_above for D = 128 (two mask words,
// per-lane position).
__device__ __forceinline__ int iq_lane_bit_below(uint64_t m0, uint64_t m1, int pos)
{
    const uint64_t w1 = pos <= 64 ? 0ull : pos >= 128 ? m1 : m1 & ((1ull << (pos - 64)) - 1);
    const uint64_t w0 = pos <= 0 ? 0ull : pos >= 64 ? m0 : m0 & ((1ull << pos) - 1);
    return w1 ? 127 - __builtin_clzll(w1) : w0 ? 63 - __builtin_clzll(w0) : -1;
}

__device__ __forceinline__ int iq_lane_bit_above(uint64_t m0, uint64_t m1, int pos)
{
    const uint64_t w0 = pos >= 63 ? 0ull : pos < 0 ? m0 : m0 & ~((2ull << pos) - 1);
    const uint64_t w1 = pos >= 127 ? 0ull : pos < 64 ? m1 : m1 & ~((2ull << (pos - 64)) - 1);
    return w0 ? __builtin_ctzll(w0) : w1 ? 64 + __builtin_ctzll(w1) : 128;
}

// The sequential donor picks of iq_select_wave_t<2> for one D = 128 row, run
// by one wavefront: sel0 / sel1 mark the sources (channels lane and
// 64 + lane), av0 / av1 the channels that may donate.  The neighbour order
// and run boundaries are precomputed one source per lane, so a pick with a
// free neighbour is a handful of scalar operations.  pool: av0 / av1 hold
// exactly `count` channels (min_error).  LDS scratch: list[64].
__device__ __forceinline__ void iq_pick_donors128(const float *sal, uint64_t sel0, uint64_t sel1, uint64_t av0,
                                                  uint64_t av1, bool pool, int count, int16_t *src_out,
                                                  int16_t *don_out, uint8_t *is_src, int16_t *src_of, int16_t *list)
{
    const int lane = threadIdx.x & 63;
    const uint64_t below = (1ull << lane) - 1;
    if (pool && count <= 16) {
        if ((sel0 >> lane) & 1ull) src_out[__popcll(sel0 & below)] = (int16_t)lane;
        if ((sel1 >> lane) & 1ull) src_out[__popcll(sel0) + __popcll(sel1 & below)] = (int16_t)(64 + lane);
        if ((av0 >> lane) & 1ull) don_out[__popcll(av0 & below)] = (int16_t)lane;
        if ((av1 >> lane) & 1ull) don_out[__popcll(av0) + __popcll(av1 & below)] = (int16_t)(64 + lane);
        is_src[lane] = is_src[64 + lane] = 0;
        src_of[lane] = src_of[64 + lane] = -1;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        iq_pick_pool16(sal, count, src_out, don_out, is_src, src_of);
        return;
    }
    if ((sel0 >> lane) & 1ull) list[__popcll(sel0 & below)] = (int16_t)lane;
    if ((sel1 >> lane) & 1ull) list[__popcll(sel0) + __popcll(sel1 & below)] = (int16_t)(64 + lane);
    // lanes read list entries other lanes of this wavefront wrote: LDS
    // operations of a wavefront complete in order, so this fence emits
    // nothing; it keeps the compiler from moving the reads above the writes
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    is_src[lane] = (uint8_t)((sel0 >> lane) & 1ull);
    is_src[64 + lane] = (uint8_t)((sel1 >> lane) & 1ull);
    src_of[lane] = -1;
    src_of[64 + lane] = -1;
    const uint32_t sk0 = iq_nonneg_bits(sal[lane]), sk1 = iq_nonneg_bits(sal[64 + lane]);
    // lane i: the i-th source s, whether its left neighbour wins a saliency
    // comparison with the right one, and its selected run [lb, rb], packed
    // into one word so that a pick reads them with a single readlane
    const int s = lane < count ? list[lane] : 0;
    const uint32_t kl = s >= 1 ? iq_nonneg_bits(sal[s - 1]) : ~0u;
    const uint32_t kr = s + 1 < 128 ? iq_nonneg_bits(sal[s + 1]) : ~0u;
    const int lb = iq_lane_bit_below(~sel0, ~sel1, s) + 1;
    const int rb = iq_lane_bit_above(~sel0, ~sel1, s) - 1;
    const uint32_t wv = (uint32_t)s | ((kl <= kr ? 1u : 0u) << 8) | ((uint32_t)lb << 9) | ((uint32_t)(rb + 1) << 17);
    int don_v = 0;
    for (int i = 0; i < count; ++i) {
        const uint32_t w = __builtin_amdgcn_readlane(wv, i);
        const int si = (int)(w & 255u), l1 = si - 1, r1 = si + 1;
        const bool lo = l1 >= 0 && (((l1 < 64 ? av0 : av1) >> (l1 & 63)) & 1ull);
        const bool ro = r1 < 128 && (((r1 < 64 ? av0 : av1) >> (r1 & 63)) & 1ull);
        int donor;
        if (lo || ro) {
            donor = (lo && (!ro || ((w >> 8) & 1u))) ? l1 : r1;
        } else {
            // the nearest available channel below the run or above it; less
            // saliency, then the lower channel, on a distance tie
            const int lbi = (int)((w >> 9) & 255u), rbi = (int)((w >> 17) & 255u) - 1;
            const uint64_t m[2] = {av0, av1};
            const int pl = iq_bit_below<2>(m, lbi);
            const int pr = iq_bit_above<2>(m, rbi, 128);
            const int dl = pl >= 0 ? lbi - pl : 0x7fffffff;
            const int dr = pr < 128 ? pr - rbi : 0x7fffffff;
            donor = 0;            // an empty pool only arises from non-finite statistics
            if (dl < dr) donor = pl;
            else if (dr < dl) donor = pr;
            else if (dl != 0x7fffffff) {
                const uint32_t ka = __builtin_amdgcn_readlane(pl < 64 ? sk0 : sk1, pl & 63);
                const uint32_t kb = __builtin_amdgcn_readlane(pr < 64 ? sk0 : sk1, pr & 63);
                donor = ka <= kb ? pl : pr;
            }
        }
        if (donor < 64) av0 &= ~(1ull << donor);
        else av1 &= ~(1ull << (donor - 64));
        don_v = lane == i ? donor : don_v;
    }
    if (lane < count) {
        src_out[lane] = (int16_t)s;
        don_out[lane] = (int16_t)don_v;
        src_of[don_v] = (int16_t)s;
    }
}

// The selection of iq_select_wave_t<2> for one D = 128 row, computed by a
// whole 256-thread workgroup (every thread calls it: it holds barriers).
// Sources and the min_error pool come from ranks over all channel pairs:
// each channel gets a 64-bit key that orders it exactly as the stable sort
// does (the value's bits, then the channel as tie-break), and its rank is the
// number of keys ordered before it, each thread comparing against 64 of
// them.  The sequential donor picks then run on one wavefront (threads 0-63 of the order the caller passes) from the neighbour
// order and run boundaries precomputed one source per lane, so a pick with a
// free neighbour is a handful of scalar operations.  LDS scratch: key[128],
// part[256], flag[128], list[64].
__device__ __forceinline__ void iq_select_tile128(const float *sal, const float *err, int count,
                                                  int16_t *src_out, int16_t *don_out, uint8_t *is_src,
                                                  int16_t *src_of, uint64_t *key, int *part, uint8_t *flag,
                                                  int16_t *list, int tid)
{
    typedef __attribute__((ext_vector_type(2))) uint64_t v2u64;
    const int c = tid & 127, half = tid >> 7, lane = tid & 63;
    // 1. sources: the `count` channels first in descending saliency, ties to
    //    the lower channel; as one ascending key: ~bits, then the channel
    if (tid < 128) key[c] = ((uint64_t)~iq_nonneg_bits(sal[c]) << 7) | (uint64_t)c;
    __syncthreads();
    {
        const uint64_t mine = key[c];
        int r = 0;
#pragma unroll 8
        for (int k = 0; k < 64; k += 2) {
            const v2u64 kk = *(const v2u64 *)(key + 64 * half + k);
            r += kk[0] < mine;
            r += kk[1] < mine;
        }
        part[tid] = r;
    }
    __syncthreads();
    const bool sel = part[c] + part[c + 128] < count;
    bool avail = !sel;
    if (err) {  // 2. pool: the `count` non-sources first in ascending error, ties to the lower channel
        if (tid < 128) key[c] = sel ? ~0ull : ((uint64_t)iq_nonneg_bits(err[c]) << 7) | (uint64_t)c;
        __syncthreads();
        const uint64_t mine = key[c];
        int r = 0;
#pragma unroll 8
        for (int k = 0; k < 64; k += 2) {
            const v2u64 kk = *(const v2u64 *)(key + 64 * half + k);
            r += kk[0] < mine;
            r += kk[1] < mine;
        }
        __syncthreads();            // every thread has read part[] for sel
        part[tid] = r;
        __syncthreads();
        avail = !sel && part[c] + part[c + 128] < count;
    }
    if (tid < 128) flag[c] = (sel ? 1 : 0) | (avail ? 2 : 0);
    __syncthreads();
    if (tid >= 64) return;

    // 3. sequential donor picks on the wavefront of tid 0-63; sources in ascending channel order
    const uint32_t f0 = flag[lane], f1 = flag[64 + lane];
    iq_pick_donors128(sal, __ballot(f0 & 1u), __ballot(f1 & 1u), __ballot(f0 & 2u), __ballot(f1 & 2u), err != nullptr,
                      count, src_out, don_out, is_src, src_of, list);
}

// Top `count` of the 128 keys k0 (channel lane) and k1 (channel 64 + lane)
// among the eligible channels (masks e0, e1), ties to the lower channel: the
// selection of iq_wave_top<2>, with the comparisons made straight into lane
// masks.  Ineligible keys are zeroed first, so that the radix search, whose
// candidates are never 0, needs no mask; only the ties at the threshold do.
__device__ __forceinline__ void iq_top128(uint32_t k0, uint32_t k1, uint64_t e0, uint64_t e1, int count, uint64_t &o0,
                                          uint64_t &o1)
{
    constexpr int UGT = 34, UGE = 35, EQ = 32;    // integer predicates of the lane-mask compares
    const int lane = threadIdx.x & 63;
    k0 = ((e0 >> lane) & 1ull) ? k0 : 0u;
    k1 = ((e1 >> lane) & 1ull) ? k1 : 0u;
    if (count <= 0) {
        o0 = o1 = 0;
        return;
    }
    uint32_t thr = 0;
#pragma unroll
    for (int bit = 31; bit >= 0; --bit) {
        const uint32_t cand = thr | (1u << bit);
        const int n = __popcll(__builtin_amdgcn_uicmp(k0, cand, UGE)) + __popcll(__builtin_amdgcn_uicmp(k1, cand, UGE));
        if (n >= count) thr = cand;
    }
    o0 = __builtin_amdgcn_uicmp(k0, thr, UGT) & e0;
    o1 = __builtin_amdgcn_uicmp(k1, thr, UGT) & e1;
    int need = count - __popcll(o0) - __popcll(o1);
    uint64_t eq0 = __builtin_amdgcn_uicmp(k0, thr, EQ) & e0, eq1 = __builtin_amdgcn_uicmp(k1, thr, EQ) & e1;
    for (; eq0 && need > 0; --need) {
        const uint64_t low = eq0 & (~eq0 + 1);
        o0 |= low;
        eq0 ^= low;
    }
    for (; eq1 && need > 0; --need) {
        const uint64_t low = eq1 & (~eq1 + 1);
        o1 |= low;
        eq1 ^= low;
    }
}

// The selection of iq_select_wave_t<2> for one D = 128 row by one wavefront
// (sal / err in LDS, err null for the plain policy): radix top-k for the
// sources and the min_error pool, then iq_pick_donors128.  LDS scratch:
// list[64].
__device__ __forceinline__ void iq_select_wave128(const float *sal, const float *err, int count, int16_t *src_out,
                                                  int16_t *don_out, uint8_t *is_src, int16_t *src_of, int16_t *list)
{
    const int lane = threadIdx.x & 63;
    uint64_t sel0, sel1;
    iq_top128(iq_nonneg_bits(sal[lane]), iq_nonneg_bits(sal[64 + lane]), ~0ull, ~0ull, count, sel0, sel1);
    uint64_t av0 = ~sel0, av1 = ~sel1;
    if (err)  // ascending error == descending complement of its bit pattern
        iq_top128(~iq_nonneg_bits(err[lane]), ~iq_nonneg_bits(err[64 + lane]), ~sel0, ~sel1, count, av0, av1);
    iq_pick_donors128(sal, sel0, sel1, av0, av1, err != nullptr, count, src_out, don_out, is_src, src_of, list);
}

// WIDE: D > 256.
template <bool WIDE>
__device__ __forceinline__ void iq_select_wave(const float *sal, const float *err, int D, int count,
                                               int16_t *src_out, int16_t *don_out, uint8_t *is_src,
                                               int16_t *src_of)
{
    if constexpr (WIDE) {
        if (D <= 512) iq_select_wave_t<8>(sal, err, D, count, src_out, don_out, is_src, src_of);
        else iq_select_wave_t<16>(sal, err, D, count, src_out, don_out, is_src, src_of);
    } else {
        if (D <= 64) iq_select_wave_t<1>(sal, err, D, count, src_out, don_out, is_src, src_of);
        else if (D <= 128) iq_select_wave_t<2>(sal, err, D, count, src_out, don_out, is_src, src_of);
        else iq_select_wave_t<4>(sal, err, D, count, src_out, don_out, is_src, src_of);
    }
}
