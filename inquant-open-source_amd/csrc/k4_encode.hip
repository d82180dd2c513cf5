// K4 neighbor-slot encoder and standalone donor selector (gfx950).
//
// A (batch, head) row of x[B, H, T, D] goes through
//   1  per-channel statistics: sampled saliency and mean in torch's CPU
//      summation order, full-row amax, and for min_error the donor error
//      (codec.py:200-210);
//   2  donor selection (select_dev.h);
//   3  scales, 4-bit slots, 8-bit salient codes split across the source and
//      donor slots, nibble packing, padding (codec.py:218-233).
// Results are bit-identical to the reference CPU implementation.
#include "k4_stats_dev.h"
#include "select_dev.h"
#include "v_rows_dev.h"

#include <cstdarg>
#include <cstdio>

namespace {

constexpr int K4_THREADS = 256;

// Rows whose donor pool the order-free sums left uncertain (k4_stats.h), so
// that they took the sequential pass: iq_k4_uncertain_rows.
__device__ uint32_t uncertain_rows;

struct K4Args {
    const void *x;
    int dt;
    int64_t sb, sh, st, sc;   // element strides
    int64_t H, T, D, count, stride;
    int min_error;
    uint8_t *payload;
    float *scales;
    void *src, *don;
    int desc_bytes;
    float *padding;
    int *bad;
    // page mode (k4_encode_tile<..., true>): row (b, h) is written into the
    // physical page ids[b] of `pool` (byte offsets of the page fields), with
    // an int16 role map instead of descriptors, and the value rows of v
    // (element strides vsb, vsh, vst) are V2-encoded into the same page
    uint8_t *pool;
    int64_t pool_pages, page_bytes;
    const void *ids;
    int id_bytes;
    int64_t off_kpay, off_kscale, off_kmap, off_kpad, off_vpay, off_vscale, off_voff;
    const uint16_t *v;
    int64_t vsb, vsh, vst;
    int *vbad, *badid, *clear;  // value flag; out-of-range page id flag; flag triple the next page launch uses, zeroed here
    // page mode, optional: page b starts at token row page_rows[b] of x / v
    // (offsets page_rows[b] * st, page_rows[b] * vst) instead of b * sb, b * vsb
    const int64_t *page_rows;
    // fused key/value mode (k4_encode_tile<..., VB = 2 or 4>): the value rows
    // of v are encoded group-wise into the outputs of iq_v_quantize
    uint8_t *vpayload;
    uint16_t *vscales, *voffsets;
};

__device__ __forceinline__ void store_desc(void *p, int64_t i, int v, int bytes)
{
    if (bytes == 1) ((uint8_t *)p)[i] = (uint8_t)v;
    else if (bytes == 4) ((int32_t *)p)[i] = v;
    else ((int64_t *)p)[i] = v;
}

// Calls f(v, i) for i = 0 .. n - 1 in order with v the element at
// base + (i * mul + add) * step, loading SEQ_PF elements ahead of their use
// (one memory round trip per SEQ_PF elements of a sequential reduction).
constexpr int SEQ_PF = 16;

template <int DT, typename F>
__device__ __forceinline__ void for_each_seq_t(const void *x, int64_t base, int64_t step, int64_t n, int64_t mul,
                                               int64_t add, F &f)
{
    // whole groups without a bound check per element, the next group's loads
    // issued before the current group is reduced (its round trip overlaps
    // SEQ_PF steps of the reduction), then the ragged end
    const int64_t nfull = n - n % SEQ_PF;
    float cur[SEQ_PF];
    if (nfull > 0) {
#pragma unroll
        for (int u = 0; u < SEQ_PF; ++u)
            cur[u] = iq_load_f32(x, base + (u * mul + add) * step, DT);   // DT constant: no branch per load
    }
    for (int64_t i0 = 0; i0 < nfull; i0 += SEQ_PF) {
        float nxt[SEQ_PF];
        const int64_t i1 = i0 + SEQ_PF < nfull ? i0 + SEQ_PF : i0;   // the last group reloads itself
#pragma unroll
        for (int u = 0; u < SEQ_PF; ++u)
            nxt[u] = iq_load_f32(x, base + ((i1 + u) * mul + add) * step, DT);
#pragma unroll
        for (int u = 0; u < SEQ_PF; ++u) f(cur[u], i0 + u);
#pragma unroll
        for (int u = 0; u < SEQ_PF; ++u) cur[u] = nxt[u];
    }
    if (nfull < n) {
        float v[SEQ_PF];
#pragma unroll
        for (int u = 0; u < SEQ_PF; ++u) {
            const int64_t i = nfull + u < n ? nfull + u : n - 1;
            v[u] = iq_load_f32(x, base + (i * mul + add) * step, DT);
        }
#pragma unroll
        for (int u = 0; u < SEQ_PF; ++u)
            if (nfull + u < n) f(v[u], nfull + u);
    }
}

// RN(1 / n) for an integer 1 <= n <= 2^24: the float reciprocal (exact
// input, within a few ulp) and two Newton steps with fma.  After them the
// relative error before the last rounding is ~2^-84, while 1 / n lies at
// least 2^-78 (relative) from a rounding midpoint of the doubles for
// n <= 2^24, so the result is the correctly rounded reciprocal
// (tests/test_welford_division.py checks every such n with the float start
// off by up to 4 ulp either way).
__device__ __forceinline__ double iq_rcp_small_int(uint32_t n)
{
    const double d = (double)n;
    double y = (double)__builtin_amdgcn_rcpf((float)n);
    y = __builtin_fma(y, __builtin_fma(-d, y, 1.0), y);
    return __builtin_fma(y, __builtin_fma(-d, y, 1.0), y);
}

// lane l's double, read by the whole wave (l uniform)
__device__ __forceinline__ double iq_read_lane_f64(double v, int l)
{
    const uint64_t b = (uint64_t)__double_as_longlong(v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, l);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), l);
    return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}

// Sampled sums of one channel in torch's order (cascade, or interleaved row_sum).
template <int DT>
__device__ __forceinline__ void sampled_sums(const void *x, int64_t base, int64_t step, int64_t ns, bool cascade_col,
                                             float &sum_abs, float &sum)
{
    if (cascade_col) {
        IqCascade a, s;
        a.init(ns);
        s.init(ns);
        auto f = [&](float v, int64_t) {
            a.add(fabsf(v));
            s.add(v);
        };
        for_each_seq_t<DT>(x, base, step, ns, 1, 0, f);
        sum_abs = a.finish();
        sum = s.finish();
    } else {
        const int64_t g = ns / 4;
        float pa[4], ps[4];
        for (int k = 0; k < 4; ++k) {
            IqCascade a, s;
            a.init(g);
            s.init(g);
            auto f = [&](float v, int64_t) {
                a.add(fabsf(v));
                s.add(v);
            };
            for_each_seq_t<DT>(x, base, step, g, 4, k, f);
            pa[k] = a.finish();
            ps[k] = s.finish();
        }
        for (int64_t r = 4 * g; r < ns; ++r) {
            const float v = iq_load_f32(x, base + r * step, DT);
            pa[0] = __fadd_rn(pa[0], fabsf(v));
            ps[0] = __fadd_rn(ps[0], v);
        }
        sum_abs = __fadd_rn(__fadd_rn(__fadd_rn(pa[0], pa[1]), pa[2]), pa[3]);
        sum = __fadd_rn(__fadd_rn(__fadd_rn(ps[0], ps[1]), ps[2]), ps[3]);
    }
}

template <bool F16IN>
__device__ __forceinline__ float tile_f32(uint32_t bits16)
{
    if constexpr (F16IN) return iq_f16_to_f32((uint16_t)bits16);
    else return __uint_as_float(bits16 << 16);
}

// ---------------------------------------------------------------------------
// General rows: any dtype, stride, length and (even) head size.  A row of up
// to LONG_ROW tokens is one workgroup's (k4_encode_kernel); a longer one is
// spread over the chip in three launches (k4_row_stats, k4_row_select,
// k4_quantize_rows).  Both take the donor errors from order-free sums with a
// certificate (k4_stats.h), so nothing but the saliency sums has an order
// to keep, and torch's cascade leaves those in independent pieces.  Eight rows
// of 32768 bf16 tokens x 128 channels: 22.7 + 16.4 + 21.8 us (3.0, then 3.8
// TB/s of rows read and words written; 3390 + 89 us with a sequential fp64
// chain per channel); four of 4096: 6.3 + 12.3 + 6.4 us (342 + 23).  The
// second launch is latency: a few workgroups, one after the other the partial
// results' round trips, the radix selections and the picks.
constexpr int ROW_THREADS = 512;
constexpr int ROW_WAVES = ROW_THREADS / 64;
constexpr int ROW_GROUPS = ROW_WAVES / 2;
// Two rows of 64 fp16 channels take 17.4 us in one workgroup each and 18.3
// spread at 256 tokens, 19.9 and 18.5 at 384, 51 and 19 at 2048; 512 rows 35
// and 37 at 256 tokens, 46 and 44 at 512.
constexpr int64_t LONG_ROW = 256;

struct RowLds {
    float sal[IQ_MAXD], smean[IQ_MAXD], err[IQ_MAXD], ehi[IQ_MAXD], scale[IQ_MAXD];
    int16_t src_of[IQ_MAXD], src[IQ_MAXD / 2], don[IQ_MAXD / 2], list[64];
    uint8_t is_src[IQ_MAXD];
    int bad, again;
};

// Partial sums of 64 channels by one wavefront.
struct RowPart {
    double s1[64], s2[64];
    float amax[64];
};

// Sums, largest magnitude and finiteness of one channel's tokens t0, t0 +
// step, ... < t1, sixteen loads in flight.
template <int DT>
__device__ __forceinline__ void stats_slice(const void *x, int64_t cb, int64_t st, int64_t t0, int64_t t1, int64_t step,
                                            double &s1, double &s2, float &amax, bool &bad)
{
    s1 = s2 = 0.0;
    amax = 0.0f;
    bad = false;
    constexpr int U = 16;
    for (int64_t t = t0; t < t1; t += U * step) {
        float v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t tt = t + u * step;
            v[u] = iq_load_f32(x, cb + (tt < t1 ? tt : t0) * st, DT);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (t + u * step >= t1) v[u] = 0.0f;
            bad |= !iq_isfinite(v[u]);
            amax = fmaxf(amax, fabsf(v[u]));
            const double d = (double)v[u];
            s1 = __dadd_rn(s1, d);
            s2 = __builtin_fma(d, d, s2);
        }
    }
}

// The reference's donor error of one channel by its sequential fp64 Welford
// chain (rows whose pool the order-free sums leave uncertain).  Every lane of
// the wavefront runs it (lanes past the last channel repeat it), G tokens at a
// time, the next ones in flight.  While every channel of the wavefront still
// holds its first value the chain's mean is that value and its sum zero, so it
// starts where a channel first differs: rows of equal tokens, which are
// uncertain as a rule (relative to a variance of zero the sums' bound is not
// small), need no chain.  Eight rows of 32768 tokens x 128 channels, all three
// launches: equal tokens 1.17 ms, near ties 1.64, certain rows 58 us (bf16; 3.47
// ms each with the chain in place of the sums).  SHORT: T <= 2^24.
template <int DT, int G, bool SHORT>
__device__ __forceinline__ float welford_error(const void *x, int64_t cb, int64_t st, int64_t T, float smean)
{
    const int lane = threadIdx.x & 63;
    // a global pointer in a called function too (a generic one's loads count as LDS operations as well)
    typedef typename std::conditional<DT == IQ_F32, float, typename std::conditional<DT == IQ_F64, double, uint16_t>::type>::type E;
    const auto *xc = (const __attribute__((address_space(1))) E *)(uintptr_t)x + cb;
    float cur[G], nxt[G];
    auto load = [&](int64_t t0, float (&v)[G]) {
        const auto *p = xc + min(t0, T - 1) * st;
        int64_t left = T - 1 - t0;               // past the last token: the last one again
#pragma unroll
        for (int u = 0; u < G; ++u, --left) {
            const E e = *p;
            p += left > 0 ? st : 0;
            if constexpr (DT == IQ_BF16) v[u] = iq_bf16_to_f32(e);
            else if constexpr (DT == IQ_F16) v[u] = iq_f16_to_f32(e);
            else v[u] = (float)e;
        }
    };
    load(0, cur);
    const float first = cur[0];
    double mean = 0.0, m2 = 0.0;
    auto step = [&](float v, double n, double y) {
        // delta / n as RN(1 / n) (off the dependent chain) and one remainder
        // correction: the correctly rounded quotient
        // (tests/test_welford_division.py, n up to 2^24)
        const double dv = (double)v;
        const double delta = __dsub_rn(dv, mean);
        const double q0 = __dmul_rn(delta, y);
        const double r = __builtin_fma(-q0, n, delta);
        mean = __dadd_rn(mean, __builtin_fma(r, y, q0));
        m2 = __dadd_rn(m2, __dmul_rn(delta, __dsub_rn(dv, mean)));
    };
    bool flat = true;
#pragma unroll 1
    for (int64_t t0 = 0; t0 < T; t0 += G) {
        load(t0 + G, nxt);
        if (flat) {
            uint32_t diff = 0;
#pragma unroll
            for (int u = 0; u < G; ++u) diff |= __float_as_uint(cur[u]) ^ __float_as_uint(first);
            flat = __ballot(diff != 0) == 0;
            if (flat || t0 > 0) mean = (double)first;
        }
        if (!flat) {
            // lane l computes the reciprocal of step l % G, and each step reads its own
            const int64_t mine = t0 + 1 + (lane & (G - 1));
            const double ys = SHORT || T <= (int64_t(1) << 24) ? iq_rcp_small_int((uint32_t)mine) : 1.0 / (double)mine;
            const double n0 = (double)t0;
            if (t0 + G <= T) {
#pragma unroll
                for (int u = 0; u < G; ++u) step(cur[u], n0 + (u + 1), iq_read_lane_f64(ys, u));
            } else {
#pragma unroll
                for (int u = 0; u < G - 1; ++u)
                    if (t0 + u < T) step(cur[u], n0 + (u + 1), iq_read_lane_f64(ys, u));
            }
        }
#pragma unroll
        for (int u = 0; u < G; ++u) cur[u] = nxt[u];
    }
    const float var = (float)(m2 / (double)T);
    const float diff = __fsub_rn((float)mean, smean);
    return __fadd_rn(var, __fmul_rn(diff, diff));
}

// v, the same in every lane, in scalar registers (a called function's arguments are not)
__device__ __forceinline__ int64_t uniform64(int64_t v)
{
    return (int64_t)(((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(v >> 32)) << 32) |
                     (uint32_t)__builtin_amdgcn_readfirstlane((int)v));
}

// The selection on the sequential errors, for rows whose pool is uncertain.
// A call of its own: inlined, its registers and hoisted address arithmetic cost
// the rows that never need it 6 us of 18 (one 256-token row a workgroup).
template <int DT, bool WIDE>
__device__ __attribute__((noinline)) void select_sequential(const void *x, int64_t base, int64_t sc, int64_t st, int64_t T,
                                                            int D, int count, RowLds *s)
{
    const int tid = threadIdx.x, lane = tid & 63;
    st = uniform64(st);
    T = uniform64(T);
    for (int c0 = tid - lane; c0 < D; c0 += ROW_THREADS) {
        const int c = min(c0 + lane, D - 1);
        const float e = welford_error<DT, 32, false>(x, base + c * sc, st, T, s->smean[c]);
        if (c0 + lane < D) s->err[c] = e;
    }
    __syncthreads();
    if (tid < 64) iq_select_wave<WIDE>(s->sal, s->err, D, count, s->src, s->don, s->is_src, s->src_of);
}

// Selection, scales, descriptors and padding of a row whose statistics are in
// LDS (s.scale holds the largest magnitudes; a barrier behind them).  Every
// thread of the workgroup calls it; it ends with a barrier.  WIDE: D > 256
// (the selection's lane masks of 512 and 1024 channels spill registers, which
// the narrower rows' kernels should not carry).
template <int DT, bool WIDE>
__device__ __forceinline__ void row_select(const K4Args &a, RowLds &s, int64_t row, int64_t base)
{
    const int tid = threadIdx.x, lane = tid & 63;
    const int64_t D = a.D;
    if (tid < 64) {
        const float *err = a.min_error ? s.err : nullptr;
        if (!WIDE && D == 128) iq_select_wave128(s.sal, err, (int)a.count, s.src, s.don, s.is_src, s.src_of, s.list);
        else iq_select_wave<WIDE>(s.sal, err, (int)D, (int)a.count, s.src, s.don, s.is_src, s.src_of);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        const bool again = a.min_error && !s.bad && !iq_pool_certain(s.err, s.ehi, (int)D, s.is_src, s.src_of);
        if (lane == 0) s.again = again;
    }
    __syncthreads();
    if (s.again) {
        if (tid == 0) atomicAdd(&uncertain_rows, 1u);
        select_sequential<DT, WIDE>(a.x, base, a.sc, a.st, a.T, (int)D, (int)a.count, &s);
        __syncthreads();
    }
    const float flt_min = 1.17549435e-38f;
    for (int64_t c = tid; c < D; c += ROW_THREADS) {
        const float q = s.scale[c] / (s.is_src[c] ? 127.0f : 7.0f);
        const float sc = q < flt_min ? flt_min : q;
        s.scale[c] = sc;
        a.scales[row * D + c] = sc;
    }
    for (int64_t i = tid; i < a.count; i += ROW_THREADS) {
        store_desc(a.src, row * a.count + i, s.src[i], a.desc_bytes);
        store_desc(a.don, row * a.count + i, s.don[i], a.desc_bytes);
        a.padding[row * a.count + i] = s.smean[s.don[i]];
    }
    if (tid == 0 && s.bad) atomicOr(a.bad, 1);
    __syncthreads();
}

// The 4-bit slots of a row's tokens [t0, t1), one payload byte per step, the
// inputs of P3_UNROLL steps loaded before any is used: any layout.
template <int DT, int NT>
__device__ __forceinline__ void quantize_bytes(const K4Args &a, const float *scale, const uint8_t *is_src,
                                               const int16_t *src_of, int64_t row, int64_t base, int64_t t0, int64_t t1)
{
    const int64_t half = a.D / 2;
    uint8_t *out = a.payload + row * a.T * half;
    constexpr int P3_UNROLL = 8;
    for (int64_t idx0 = t0 * half + threadIdx.x; idx0 < t1 * half; idx0 += (int64_t)NT * P3_UNROLL) {
        float xv[P3_UNROLL][2];
#pragma unroll
        for (int u = 0; u < P3_UNROLL; ++u) {
            const int64_t idx = idx0 + (int64_t)u * NT;
            const int64_t ic = idx < t1 * half ? idx : t1 * half - 1;
            const int64_t t = ic / half, j = ic - t * half;
            const int64_t tb = base + t * a.st;
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const int64_t c = 2 * j + e;
                const int16_t owner = src_of[c];
                const int64_t sc = (is_src[c] || owner < 0) ? c : owner;    // the channel slot c encodes
                xv[u][e] = iq_load_f32(a.x, tb + sc * a.sc, DT);
            }
        }
#pragma unroll
        for (int u = 0; u < P3_UNROLL; ++u) {
            const int64_t idx = idx0 + (int64_t)u * NT;
            if (idx >= t1 * half) break;
            const int64_t j = idx % half;
            uint32_t slots[2];
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const int64_t c = 2 * j + e;
                const int16_t owner = src_of[c];
                float q;
                if (is_src[c] || owner >= 0) {
                    const int64_t sc = is_src[c] ? c : owner;
                    q = rintf(xv[u][e] / scale[sc]);
                    q = fminf(fmaxf(q, -127.0f), 127.0f);
                    const uint32_t code = (uint32_t)(q + 128.0f);
                    slots[e] = is_src[c] ? (code >> 4) : (code & 15u);
                } else {
                    q = rintf(xv[u][e] / scale[c]);
                    q = fminf(fmaxf(q, -7.0f), 7.0f);
                    slots[e] = (uint32_t)(q + 8.0f);
                }
            }
            out[idx] = (uint8_t)(slots[0] | (slots[1] << 4));
        }
    }
}

// The eight 4-bit slots of channels 8 j .. 8 j + 7 (one packed word per
// token): per-slot constants, computed once from the role tables and pinned
// in registers (opaque to the compiler, which would otherwise rebuild them
// from the role masks at every token: four extra instructions per element).
// srcc[e] is the channel whose value slot e encodes: its own, or for a donor
// slot its source's.
struct K4Slots {
    float scl[8], rscl[8], top[8], bias[8];
    uint32_t shift[8];
    int srcc[8];

    __device__ __forceinline__ void init(int j, const uint8_t *is_src, const int16_t *src_of, const float *scale)
    {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int c = 8 * j + e;
            const bool hi = is_src[c];
            const int owner = src_of[c];
            const bool lo = !hi && owner >= 0;
            srcc[e] = lo ? owner : c;
            scl[e] = scale[srcc[e]];
            rscl[e] = __builtin_amdgcn_rcpf(scl[e]);
            const float lim = (hi || lo) ? 127.0f : 7.0f;
            // q + lim + 1 lands in the low mantissa bits of 1.5 * 2^23 + (lim + 1);
            // the clamp to [-lim, lim] is then [1.5 * 2^23 + 1, top]
            bias[e] = 12582912.0f + lim + 1.0f;
            top[e] = bias[e] + lim;
            shift[e] = hi ? 4u : 0u;
            asm volatile("" : "+v"(scl[e]), "+v"(rscl[e]), "+v"(top[e]), "+v"(bias[e]), "+v"(shift[e]));
        }
    }

    // The packed word of one token, v[e] the value of channel srcc[e].  The
    // reciprocal quotient p = v * rscl decides the rounding unless it is
    // within 2^-13 of a half-integer, where the IEEE quotient decides.  Below
    // |p| = 256, p is within 2^-14 of the IEEE quotient (v_rcp_f32 is within
    // 1 ulp, plus the quotient's own half ulp), so no rounding can differ
    // outside that band; beyond it every code clamps to +-lim either way.
    // One fma rounds p onto the integer grid of bias = 1.5 * 2^23 + lim + 1
    // (spacing 1 there): y = bias + rint(p) exactly, whose low mantissa bits
    // are the code plus lim + 1 once y is clamped to bias +- lim.  A second
    // fma gives p - rint(p) with one rounding for the band test, one max
    // over the lane's eight distances; the rare lanes inside it redo only
    // the slots that are.
    __device__ __forceinline__ uint32_t word(const float (&v)[8]) const
    {
        float y[8], q[8];
        float dmax = 0.0f;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            y[e] = __builtin_fmaf(v[e], rscl[e], bias[e]);
            q[e] = __fsub_rn(y[e], bias[e]);                 // rint(p), exact
            dmax = fmaxf(dmax, fabsf(__builtin_fmaf(v[e], rscl[e], -q[e])));
        }
        constexpr float band = 0.5f - 0x1p-13f;
        if (__builtin_expect(dmax >= band, 0)) {
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (fabsf(__builtin_fmaf(v[e], rscl[e], -q[e])) >= band)
                    y[e] = __fadd_rn(rintf(v[e] / scl[e]), bias[e]);
        }
        uint32_t w = 0;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float yc = __builtin_amdgcn_fmed3f(y[e], 12582913.0f, top[e]);
            w |= __builtin_amdgcn_ubfe(__float_as_uint(yc), shift[e], 4) << (4 * e);
        }
        return w;
    }
};

// quantize_bytes for channel-contiguous rows on 16-byte boundaries, D a
// multiple of 8: a thread loads 8 channels of one token (two steps ahead of
// their use), the step's tokens meet in LDS, where a donor slot finds its
// source's value, and each thread packs one word.  The tile holds two steps,
// so one barrier a step suffices.
template <int DT, int NT>
struct RowTile {
    static constexpr int EB = DT == IQ_F32 ? 4 : 2;      // element bytes
    uint8_t x[2][NT * 8 * EB];
};

template <int DT, int NT>
__device__ __forceinline__ void quantize_words(const K4Args &a, const float *scale, const uint8_t *is_src,
                                               const int16_t *src_of, RowTile<DT, NT> &tile, int64_t row, int64_t base,
                                               int64_t t0, int64_t t1)
{
    constexpr int EB = RowTile<DT, NT>::EB, NV = EB / 2;
    const int L = (int)a.D / 8, tps = NT / L;             // lanes per token, tokens per step
    const int tid = threadIdx.x, tt = tid / L, j = tid - tt * L;
    const bool live = tt < tps;
    K4Slots slots;
    slots.init(j, is_src, src_of, scale);
    // 64 / L whole tokens a wavefront: it reads only what it wrote, so its
    // own in-order LDS operations are all the synchronization
    const bool local = 64 % L == 0;
    const int64_t pitch = a.st * EB, step = tps * pitch;
    const char *src = (const char *)a.x + (base + 8 * j) * EB + (t0 + tt) * pitch;
    const char *const last = (const char *)a.x + (base + 8 * j) * EB + (t1 - 1) * pitch;
    uint32_t *out = (uint32_t *)a.payload + (row * a.T + t0 + tt) * L + j;
    u32x4_t cur[NV], nxt[NV], far[NV];
    auto load = [&](const char *p, int64_t t, u32x4_t (&r)[NV]) {     // t: the token p stands on
        const u32x4_t *q = (const u32x4_t *)(t < t1 ? p : last);
#pragma unroll
        for (int k = 0; k < NV; ++k) r[k] = q[k];
    };
    load(src, t0 + tt, cur);
    load(src + step, t0 + tt + tps, nxt);
    int buf = 0;
    for (int64_t t = t0 + tt; t - tt < t1; t += tps, buf ^= 1) {
        src += step;
        load(src + step, t + 2 * tps, far);
        uint8_t *xs = tile.x[buf] + tt * (int)a.D * EB;
        if (live) {
#pragma unroll
            for (int k = 0; k < NV; ++k) ((u32x4_t *)(xs + 8 * j * EB))[k] = cur[k];
        }
        if (local) __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        else __syncthreads();
        if (live && t < t1) {
            float v[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = iq_load_f32(xs, slots.srcc[e], DT);
            __builtin_nontemporal_store(slots.word(v), out);
        }
        out += tps * L;
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            cur[k] = nxt[k];
            nxt[k] = far[k];
        }
    }
}

// WORDS: the rows take quantize_words.
template <int DT, bool WORDS, bool WIDE>
__global__ __launch_bounds__(ROW_THREADS) void k4_encode_kernel(K4Args a)
{
    __shared__ RowLds s;
    // the statistics' partial sums, then the quantizer's tile
    constexpr size_t PART = ROW_WAVES * sizeof(RowPart), TILE = sizeof(RowTile<DT, ROW_THREADS>);
    __shared__ __attribute__((aligned(16))) uint8_t scratch[WORDS && TILE > PART ? TILE : PART];
    RowPart *const part = (RowPart *)scratch;

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t row = blockIdx.x;
    const int64_t b = row / a.H, h = row % a.H;
    const int64_t base = b * a.sb + h * a.sh;
    const int64_t T = a.T, D = a.D;
    const int64_t ns = (T + a.stride - 1) / a.stride;
    const int64_t ncasc = iq_cascade_columns(D);

    if (tid == 0) s.bad = 0;
    __syncthreads();

    // ---- statistics, up to 4 groups of 64 channels at a time: a wavefront
    // of each group takes the sampled sums, the others every slices-th token
    for (int64_t g0 = 0; 64 * g0 < D; g0 += ROW_GROUPS) {
        const int ng = (int)min((D + 63) / 64 - g0, (int64_t)ROW_GROUPS), slices = ROW_WAVES / ng - 1;
        const int g = wave % ng, slice = wave / ng;
        const int64_t c = min(64 * (g0 + g) + lane, D - 1);
        if (slice == slices) {
            float sum_abs, sum;
            sampled_sums<DT>(a.x, base + c * a.sc, a.st * a.stride, ns, c < ncasc, sum_abs, sum);
            s.sal[c] = sum_abs / (float)ns;
            s.smean[c] = sum / (float)ns;
        } else if (slice < slices) {
            bool bad;
            stats_slice<DT>(a.x, base + c * a.sc, a.st, slice, T, slices, part[wave].s1[lane], part[wave].s2[lane],
                            part[wave].amax[lane], bad);
            if (bad) s.bad = 1;
        }
        __syncthreads();
        // one thread per channel of these groups
        const int64_t co = 64 * g0 + tid;
        if (wave < ng && co < D) {
            double s1 = 0.0, s2 = 0.0;
            float amax = 0.0f;
            for (int k = 0; k < slices; ++k) {
                const RowPart &p = part[wave + k * ng];
                s1 = __dadd_rn(s1, p.s1[lane]);
                s2 = __dadd_rn(s2, p.s2[lane]);
                amax = fmaxf(amax, p.amax[lane]);
            }
            s.scale[co] = amax;
            const IqErrRange r = iq_err_range(s1, s2, amax, s.smean[co], T, false);
            s.err[co] = r.lo;
            s.ehi[co] = r.hi;
        }
        __syncthreads();
    }
    row_select<DT, WIDE>(a, s, row, base);
    if constexpr (WORDS)
        quantize_words<DT, ROW_THREADS>(a, s.scale, s.is_src, s.src_of, *(RowTile<DT, ROW_THREADS> *)scratch, row, base, 0, T);
    else
        quantize_bytes<DT, ROW_THREADS>(a, s.scale, s.is_src, s.src_of, row, base, 0, T);
}

// ---- rows of more than LONG_ROW tokens
//
// Launch 1 leaves every partial result in the row's own payload bytes, which
// nothing else holds until launch 3 writes them: per chunk of `chunk` tokens
// the sums and largest magnitude of each channel, and the pieces of torch's
// cascade sums of the sampled tokens.  A cascade adds 2^lp values from zero
// into a level-0 sum, 2^lp of those into a level-1 sum and so on, so each
// level-1 sum is its own piece (a workgroup's), and only the sums of pieces
// are left for launch 2.  The columns past iq_cascade_columns(D) are four
// interleaved cascades of a quarter of the samples each: a sequence is a
// column, or one of those quarters.
struct RowPlan {
    int64_t chunk, nchunk;      // tokens per chunk, chunks
    int64_t pieces;             // level-1 sums of the longest sequence, the unfinished one included
    int64_t nseq;               // sequences
    int64_t off_s2, off_amax, off_piece, bytes;
};

__host__ __device__ inline RowPlan row_plan(int64_t T, int64_t D, int64_t stride, int64_t chunk)
{
    RowPlan p;
    const int64_t ns = (T + stride - 1) / stride, ncasc = iq_cascade_columns(D);
    p.chunk = chunk;
    p.nchunk = (T + chunk - 1) / chunk;
    p.nseq = ncasc + 4 * (D - ncasc);
    auto pieces = [](int64_t n) {
        int lp = 0;
        for (int64_t x = n > 1 ? n - 1 : 0; x; x >>= 1) ++lp;
        lp = lp / 4 < 4 ? 4 : lp / 4;
        return (n >> (2 * lp)) + 1;
    };
    const int64_t pc = ncasc > 0 ? pieces(ns) : 0, pr = ncasc < D ? pieces(ns / 4) : 0;
    p.pieces = pc > pr ? pc : pr;
    p.off_s2 = p.nchunk * D * 8;
    p.off_amax = 2 * p.off_s2;
    p.off_piece = p.off_amax + (p.nchunk * D * 4 + 7) / 8 * 8;
    // piece k of sequence q: (sum of |x|, sum); slot `pieces`: the samples past the last whole level-0 sum
    p.bytes = p.off_piece + (p.pieces + 1) * p.nseq * 8;
    return p;
}

// The row's scratch: its payload bytes from the first 16-byte boundary on.
__device__ __forceinline__ uint8_t *row_scratch(const K4Args &a, int64_t row)
{
    return (uint8_t *)(((uintptr_t)(a.payload + row * a.T * (a.D / 2)) + 15) & ~(uintptr_t)15);
}

struct RowSeq {
    int64_t c, mul, add, n;     // channel, sample j * mul + add for j < n
    int lp;
    bool row_sum;
};

__device__ __forceinline__ RowSeq row_seq(int64_t q, int64_t ncasc, int64_t ns)
{
    RowSeq r;
    r.row_sum = q >= ncasc;
    r.c = r.row_sum ? ncasc + (q - ncasc) / 4 : q;
    r.mul = r.row_sum ? 4 : 1;
    r.add = r.row_sum ? (q - ncasc) % 4 : 0;
    r.n = r.row_sum ? ns / 4 : ns;
    r.lp = max(iq_ceil_log2(r.n) / 4, 4);
    return r;
}

// Launch 1: grid (pieces, then chunks, rows).  WORDS: 16-byte loads.
template <int DT, bool WORDS>
__global__ __launch_bounds__(K4_THREADS) void k4_row_stats(K4Args a, RowPlan p)
{
    constexpr int WAVES = K4_THREADS / 64;
    constexpr int MAXSUMS = 64;     // level-0 sums per level-1 sum: 2^lp, lp <= 6 for up to 2^27 samples
    constexpr int WS = WORDS ? K4_THREADS * 4 : 1;
    __shared__ union {
        RowPart part[WAVES];
        float2 sums[MAXSUMS][64];
        struct {
            double s1[WS], s2[WS];
            float amax[WS];
        } words;
    } s;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t row = blockIdx.y, b = row / a.H, h = row % a.H;
    const int64_t base = b * a.sb + h * a.sh, D = a.D;
    uint8_t *const scratch = row_scratch(a, row);
    // the pieces' workgroups first: they wait longest for their loads
    const int64_t groups = (p.nseq + 63) / 64, npiece = p.pieces * groups;
    if ((int64_t)blockIdx.x >= npiece) {
        const int64_t k = blockIdx.x - npiece, t0 = k * p.chunk, t1 = min(t0 + p.chunk, a.T);
        double *const out1 = (double *)scratch + k * D, *const out2 = (double *)(scratch + p.off_s2) + k * D;
        float *const outm = (float *)(scratch + p.off_amax) + k * D;
        if constexpr (WORDS) {
            // lane (tt, j) = (tid / L, tid % L): channels 8 j .. of the tokens tt, tt + tps, ...
            constexpr int EB = DT == IQ_F32 ? 4 : 2, NV = EB / 2, U = 8 / NV;
            const int L = (int)D / 8, tps = K4_THREADS / L, tt = tid / L, j = tid - tt * L;
            double s1[8], s2[8];
            float amax[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                s1[e] = s2[e] = 0.0;
                amax[e] = 0.0f;
            }
            bool bad = false;
            if (tt < tps) {
                const char *xb = (const char *)a.x + (base + 8 * j) * EB;
                for (int64_t t = t0 + tt; t < t1; t += U * tps) {
                    u32x4_t raw[U][NV];
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        const int64_t tc = t + u * tps < t1 ? t + u * tps : t;
#pragma unroll
                        for (int n = 0; n < NV; ++n) raw[u][n] = ((const u32x4_t *)(xb + tc * a.st * EB))[n];
                    }
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        if (t + u * tps >= t1) break;
#pragma unroll
                        for (int e = 0; e < 8; ++e) {
                            float v;
                            if constexpr (EB == 4) v = __uint_as_float(raw[u][e / 4][e % 4]);
                            else v = tile_f32<DT == IQ_F16>(e & 1 ? raw[u][0][e / 2] >> 16 : raw[u][0][e / 2] & 0xffffu);
                            amax[e] = fmaxf(amax[e], fabsf(v));
                            const double d = (double)v;
                            s1[e] = __dadd_rn(s1[e], d);
                            s2[e] = __builtin_fma(d, d, s2[e]);
                        }
                    }
                }
                // squares of finite floats sum to a finite double, any other value does not
#pragma unroll
                for (int e = 0; e < 8; ++e) bad |= !(s2[e] < (double)INFINITY);
            }
            if (bad) atomicOr(a.bad, 1);
            // the tokens' sums meet in LDS, four channels of each lane at a time
#pragma unroll
            for (int half = 0; half < 2; ++half) {
                const int W = (int)D / 2;            // channels of a half
                if (tt < tps) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        // channel 8 j + 4 half + e at e L + j: neighbouring lanes on neighbouring banks
                        s.words.s1[tt * W + e * L + j] = s1[4 * half + e];
                        s.words.s2[tt * W + e * L + j] = s2[4 * half + e];
                        s.words.amax[tt * W + e * L + j] = amax[4 * half + e];
                    }
                }
                __syncthreads();
                for (int c = tid; c < W; c += K4_THREADS) {
                    double r1 = 0.0, r2 = 0.0;
                    float rm = 0.0f;
                    for (int i = 0; i < tps; ++i) {
                        r1 = __dadd_rn(r1, s.words.s1[i * W + c]);
                        r2 = __dadd_rn(r2, s.words.s2[i * W + c]);
                        rm = fmaxf(rm, s.words.amax[i * W + c]);
                    }
                    const int e = c / L, ch = 8 * (c - e * L) + 4 * half + e;
                    out1[ch] = r1;
                    out2[ch] = r2;
                    outm[ch] = rm;
                }
                __syncthreads();
            }
            return;
        }
        for (int64_t g0 = 0; 64 * g0 < D; g0 += WAVES) {
            const int ng = (int)min((D + 63) / 64 - g0, (int64_t)WAVES), slices = WAVES / ng;
            const int g = wave % ng, slice = wave / ng;
            const int64_t c = min(64 * (g0 + g) + lane, D - 1);
            if (slice < slices) {
                bool bad;
                stats_slice<DT>(a.x, base + c * a.sc, a.st, t0 + slice, t1, slices, s.part[wave].s1[lane],
                                s.part[wave].s2[lane], s.part[wave].amax[lane], bad);
                if (bad) atomicOr(a.bad, 1);
            }
            __syncthreads();
            const int64_t co = 64 * g0 + tid;
            if (wave < ng && co < D) {
                double s1 = 0.0, s2 = 0.0;
                float amax = 0.0f;
                for (int i = 0; i < slices; ++i) {
                    const RowPart &q = s.part[wave + i * ng];
                    s1 = __dadd_rn(s1, q.s1[lane]);
                    s2 = __dadd_rn(s2, q.s2[lane]);
                    amax = fmaxf(amax, q.amax[lane]);
                }
                out1[co] = s1;
                out2[co] = s2;
                outm[co] = amax;
            }
            __syncthreads();
        }
        return;
    }
    // piece k of 64 sequences; the wavefronts share its level-0 sums
    const int64_t k = blockIdx.x / groups, q0 = (blockIdx.x - k * groups) * 64;
    const int64_t ns = (a.T + a.stride - 1) / a.stride, ncasc = iq_cascade_columns(D);
    float2 *const piece = (float2 *)(scratch + p.off_piece);
    const bool own = q0 + lane < p.nseq;
    const int64_t q = own ? q0 + lane : p.nseq - 1;
    const RowSeq r = row_seq(q, ncasc, ns);
    const int64_t per = int64_t(1) << (2 * r.lp), first = k * per;
    const int64_t left = r.n - first;                       // samples of this piece and the later ones
    const int64_t nsum = left <= 0 ? 0 : min(left, per) >> r.lp;      // whole level-0 sums
    const int64_t xb = base + r.c * a.sc, xs = a.st * a.stride;
    auto level0 = [&](int64_t j0, int64_t j1) {              // samples j0 .. j1 - 1 added from zero
        float2 acc = {0.0f, 0.0f};
        for (int64_t jb = j0; jb < j1; jb += 16) {
            float v[16];
#pragma unroll
            for (int u = 0; u < 16; ++u) {
                const int64_t jj = jb + u < j1 ? jb + u : j0;
                v[u] = iq_load_f32(a.x, xb + (jj * r.mul + r.add) * xs, DT);
            }
#pragma unroll
            for (int u = 0; u < 16; ++u) {
                if (jb + u < j1) {
                    acc.x = __fadd_rn(acc.x, fabsf(v[u]));
                    acc.y = __fadd_rn(acc.y, v[u]);
                }
            }
        }
        return acc;
    };
    // the unfinished piece's samples past its last whole level-0 sum go to the last wavefront's lanes
    const bool tail = left >= 0 && left < per;
    if (r.lp == 4) {
        // the usual length: the 16 samples of all four of a wavefront's sums in flight together
        float v[4][16];
        const int64_t sample = nsum > 0 ? r.mul * xs : 0;     // elements between a sequence's samples
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            const int64_t i = wave + WAVES * m, j0 = i < nsum ? first + 16 * i : 0;
            int64_t at = xb + r.add * xs * (nsum > 0) + j0 * sample;
#pragma unroll
            for (int u = 0; u < 16; ++u, at += sample) v[m][u] = iq_load_f32(a.x, at, DT);
        }
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            float2 acc = {0.0f, 0.0f};
#pragma unroll
            for (int u = 0; u < 16; ++u) {
                acc.x = __fadd_rn(acc.x, fabsf(v[m][u]));
                acc.y = __fadd_rn(acc.y, v[m][u]);
            }
            if (wave + WAVES * m < nsum) s.sums[wave + WAVES * m][lane] = acc;
        }
    } else {
        for (int64_t i = wave; i < nsum; i += WAVES) s.sums[i][lane] = level0(first + (i << r.lp), first + ((i + 1) << r.lp));
    }
    if (wave == WAVES - 1 && own && tail) piece[p.pieces * p.nseq + q] = level0(first + (nsum << r.lp), r.n);
    __syncthreads();
    if (wave == 0 && own && left >= 0) {
        float2 acc = {0.0f, 0.0f};
        for (int64_t i = 0; i < nsum; ++i) {
            acc.x = __fadd_rn(acc.x, s.sums[i][lane].x);
            acc.y = __fadd_rn(acc.y, s.sums[i][lane].y);
        }
        piece[k * p.nseq + q] = acc;
    }
}

// Launch 2: one workgroup per row adds the partial results and selects.
template <int DT, bool WIDE>
__global__ __launch_bounds__(ROW_THREADS) void k4_row_select(K4Args a, RowPlan p)
{
    __shared__ RowLds s;
    __shared__ RowPart part[ROW_WAVES];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t row = blockIdx.x, b = row / a.H, h = row % a.H;
    const int64_t base = b * a.sb + h * a.sh, D = a.D;
    const uint8_t *const scratch = row_scratch(a, row);
    const int64_t ns = (a.T + a.stride - 1) / a.stride, ncasc = iq_cascade_columns(D);
    const float2 *const piece = (const float2 *)(scratch + p.off_piece);
    if (tid == 0) s.bad = 0;
    __syncthreads();
    // the sampled sums of column c: one sequence, or four and their leftovers
    auto cascade = [&](int64_t q) {
        const RowSeq r = row_seq(q, ncasc, ns);
        const int64_t whole = r.n >> (2 * r.lp);
        float2 a2 = {0.0f, 0.0f}, a3 = {0.0f, 0.0f};
        const float2 *pq = piece + q;
        for (int64_t k0 = 0; k0 < whole; k0 += 8) {
            float2 v[8];
            const float2 *pk = pq;
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                v[u] = *pk;
                pk += k0 + u + 1 < whole ? p.nseq : 0;
            }
            pq = pk;
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                if (k0 + u < whole) {
                    a2.x = __fadd_rn(a2.x, v[u].x);
                    a2.y = __fadd_rn(a2.y, v[u].y);
                    if (((k0 + u + 1) & ((int64_t(1) << r.lp) - 1)) == 0) {
                        a3.x = __fadd_rn(a3.x, a2.x);
                        a3.y = __fadd_rn(a3.y, a2.y);
                        a2 = {0.0f, 0.0f};
                    }
                }
            }
        }
        const float2 a1 = piece[whole * p.nseq + q], a0 = piece[p.pieces * p.nseq + q];
        return float2{__fadd_rn(__fadd_rn(__fadd_rn(a0.x, a1.x), a2.x), a3.x),
                      __fadd_rn(__fadd_rn(__fadd_rn(a0.y, a1.y), a2.y), a3.y)};
    };
    // as in k4_encode_kernel: one wavefront of a channel group adds the
    // sampled sums, the others the chunks
    for (int64_t g0 = 0; 64 * g0 < D; g0 += ROW_GROUPS) {
        const int ng = (int)min((D + 63) / 64 - g0, (int64_t)ROW_GROUPS), slices = ROW_WAVES / ng - 1;
        const int g = wave % ng, slice = wave / ng;
        const int64_t c = min(64 * (g0 + g) + lane, D - 1);
        if (slice == slices) {
            float2 sums;
            if (c < ncasc) {
                sums = cascade(c);
            } else {
                float2 quarter[4];
                for (int k = 0; k < 4; ++k) quarter[k] = cascade(ncasc + 4 * (c - ncasc) + k);
                for (int64_t r = ns / 4 * 4; r < ns; ++r) {
                    const float v = iq_load_f32(a.x, base + c * a.sc + r * a.st * a.stride, DT);
                    quarter[0].x = __fadd_rn(quarter[0].x, fabsf(v));
                    quarter[0].y = __fadd_rn(quarter[0].y, v);
                }
                sums.x = __fadd_rn(__fadd_rn(__fadd_rn(quarter[0].x, quarter[1].x), quarter[2].x), quarter[3].x);
                sums.y = __fadd_rn(__fadd_rn(__fadd_rn(quarter[0].y, quarter[1].y), quarter[2].y), quarter[3].y);
            }
            s.sal[c] = sums.x / (float)ns;
            s.smean[c] = sums.y / (float)ns;
        } else if (slice < slices) {
            double s1 = 0.0, s2 = 0.0;
            float amax = 0.0f;
            // 32-bit indices: a uniform base and one add per load (few
            // instructions: the launch's code is fetched by a handful of
            // workgroups, once)
            const double *p1 = (const double *)scratch, *p2 = (const double *)(scratch + p.off_s2);
            const float *pm = (const float *)(scratch + p.off_amax);
            const uint32_t n = (uint32_t)p.nchunk, step = (uint32_t)(slices * D), end = n * (uint32_t)D;
            constexpr int U = 8;
            for (uint32_t at = (uint32_t)(slice * D + c); at < end; at += U * step) {
                double v1[U], v2[U];
                float vm[U];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const uint32_t x = at + u * step < end ? at + u * step : at;
                    v1[u] = p1[x];
                    v2[u] = p2[x];
                    vm[u] = pm[x];
                }
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const bool in = at + u * step < end;
                    s1 = __dadd_rn(s1, in ? v1[u] : 0.0);
                    s2 = __dadd_rn(s2, in ? v2[u] : 0.0);
                    amax = fmaxf(amax, vm[u]);
                }
            }
            part[wave].s1[lane] = s1;
            part[wave].s2[lane] = s2;
            part[wave].amax[lane] = amax;
        }
        __syncthreads();
        const int64_t co = 64 * g0 + tid;
        if (wave < ng && co < D) {
            double s1 = 0.0, s2 = 0.0;
            float amax = 0.0f;
            for (int k = 0; k < slices; ++k) {
                const RowPart &q = part[wave + k * ng];
                s1 = __dadd_rn(s1, q.s1[lane]);
                s2 = __dadd_rn(s2, q.s2[lane]);
                amax = fmaxf(amax, q.amax[lane]);
            }
            s.scale[co] = amax;
            const IqErrRange r = iq_err_range(s1, s2, amax, s.smean[co], a.T, false);
            s.err[co] = r.lo;
            s.ehi[co] = r.hi;
            if (!iq_isfinite(amax) || s2 != s2) s.bad = 1;
        }
        __syncthreads();
    }
    row_select<DT, WIDE>(a, s, row, base);
}

// Launch 3: grid (tiles of q_tokens tokens, rows); a workgroup takes the row's
// scales and descriptors from global memory.
template <int DT, bool WORDS>
__global__ __launch_bounds__(K4_THREADS) void k4_quantize_rows(K4Args a, int64_t q_tokens)
{
    __shared__ float s_scale[IQ_MAXD];
    __shared__ int16_t s_src_of[IQ_MAXD];
    __shared__ uint8_t s_is_src[IQ_MAXD];
    __shared__ __attribute__((aligned(16))) RowTile<DT, WORDS ? K4_THREADS : 1> tile;
    const int tid = threadIdx.x;
    const int64_t row = blockIdx.y, b = row / a.H, h = row % a.H;
    const int64_t base = b * a.sb + h * a.sh, D = a.D;
    auto desc = [&](const void *p, int64_t i) -> int {
        return a.desc_bytes == 1 ? ((const uint8_t *)p)[i]
               : a.desc_bytes == 4 ? ((const int32_t *)p)[i] : (int)((const int64_t *)p)[i];
    };
    for (int64_t c = tid; c < D; c += K4_THREADS) {
        s_scale[c] = a.scales[row * D + c];
        s_is_src[c] = 0;
        s_src_of[c] = -1;
    }
    __syncthreads();
    for (int64_t i = tid; i < a.count; i += K4_THREADS) {
        const int sc = desc(a.src, row * a.count + i), dn = desc(a.don, row * a.count + i);
        s_is_src[sc] = 1;
        s_src_of[dn] = (int16_t)sc;
    }
    __syncthreads();
    const int64_t t0 = (int64_t)blockIdx.x * q_tokens, t1 = min(t0 + q_tokens, a.T);
    if constexpr (WORDS) quantize_words<DT, K4_THREADS>(a, s_scale, s_is_src, s_src_of, tile, row, base, t0, t1);
    else quantize_bytes<DT, K4_THREADS>(a, s_scale, s_is_src, s_src_of, row, base, t0, t1);
}

// ---------------------------------------------------------------------------
// Tile encoder for the cache shapes: D = 128, 16-bit input, T <= 256 tokens,
// channel-contiguous rows.  The block streams through LDS in 32-token chunks
// (16-byte loads; sealed blocks by direct loads with three chunks in flight
// while one is consumed, others double-buffered through registers), twice:
//   pass 1  thread (half, channel) sums x and x^2 of every other token in
//           fp64 (min_error only) and takes amax and finiteness as an integer
//           max of the 16-bit magnitudes; one half also adds the sampled
//           sums (torch cascade order).  The donor errors come from the sums
//           with a certificate (k4_stats.h);
//   then    donor selection by the whole workgroup (iq_select_tile128);
//           the sequential donor picks run on one wavefront alone, and with a
//           value row to encode (page mode, or VB = 2 / 4) the other three
//           group-encode the values meanwhile (v_encode16, the same bits as
//           v_encode_rows), reading them from HBM while it is otherwise idle;
//   pass 2  every thread quantizes 8 channels of a token per step, writing
//           4 payload bytes.
// With a sequential fp64 Welford chain per channel on two of the wavefronts
// (they waited for each other at every chunk) a layer of 32768 tokens x 8
// heads took 82 us with K4 keys and values and 58-62 with 2-bit values; with
// the sums on all four 76-78 and 57-58, and 32768 tokens x 4 heads in
// 256-token pages 38.9 instead of 42.3.
// LDS stays under 40 KiB, so four blocks share a compute unit and their
// latency-bound phases (the chunk waits, the donor picks) overlap.
// Bit-identical to k4_encode_kernel.
constexpr int TILE_D = 128;
constexpr int TILE_T = 256;
constexpr int CH = 32;                   // tokens per staged chunk
constexpr int KPF = 1;                   // chunks in flight
constexpr int XROW = TILE_D + 8;         // u16 per staged row: 68 dwords (16-byte aligned rows, distinct banks)
// sealed blocks stream by direct global -> LDS loads into NBUF chunk buffers
// (unpadded rows), NBUF - 1 chunks in flight while one is processed
constexpr int NBUF_DMA = 4;

// s_waitcnt vmcnt(2 * ahead) lgkmcnt(0), then s_barrier: this wave's loads
// of every chunk but the `ahead` newest have landed in LDS and its LDS reads
// are done; after the barrier the same holds for every wave.  Vector memory
// operations retire in issue order, so at most 2 * ahead outstanding means
// every older load is done; stores issued after a chunk's loads only make
// the wait longer.  (A plain __syncthreads would wait for all loads in
// flight.)
__device__ __forceinline__ void wait_chunk_barrier(int ahead)
{
    switch (ahead) {
    case 0: asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory"); break;
    case 1: asm volatile("s_waitcnt vmcnt(2) lgkmcnt(0)\n\ts_barrier" ::: "memory"); break;
    case 2: asm volatile("s_waitcnt vmcnt(4) lgkmcnt(0)\n\ts_barrier" ::: "memory"); break;
    default: asm volatile("s_waitcnt vmcnt(6) lgkmcnt(0)\n\ts_barrier" ::: "memory"); break;
    }
}

// The V2 codes and group parameters of token t of head h in a page (value
// lanes of 16 channels, vj = 0 .. 7, four lanes per 64-channel group).
__device__ __forceinline__ void store_page_values(const K4Args &a, uint8_t *page, int64_t h, int T, int t, int vj,
                                                  uint32_t code, uint16_t off_h, uint16_t sc_h)
{
    const int64_t r = h * T + t;
    __builtin_nontemporal_store(code, (uint32_t *)(page + a.off_vpay + r * 32) + vj);
    if ((vj & 3) == 0) ((uint16_t *)(page + a.off_voff))[r * 2 + (vj >> 2)] = off_h;
    if ((vj & 3) == 3) ((uint16_t *)(page + a.off_vscale))[r * 2 + (vj >> 2)] = sc_h;
}

// NCH > 0: the block length is NCH chunks (a sealed cache block), known at
// compile time, so the chunk loops unroll without branches and each load is
// waited for exactly when its chunk is stored (a branch around loads makes
// the compiler wait for all of them).  NCH = 0: any T <= 256.
// PAGES: the row goes into a physical page, values V2 with 64-channel groups.
// VB = 2 / 4 (not PAGES): the row's values are encoded too, VB bits with
// 16 * VGL-channel groups, into the outputs of iq_v_quantize.
// The body of one workgroup: row (b, h) of the encode `a`; `lin` is the
// workgroup's linear index (neighbouring blocks alternate their wave roles).
template <bool F16IN, int NCH, bool PAGES = false, int VB = 0, int VGL = 4>
__device__ __forceinline__ void k4_tile_body(const K4Args &a, int64_t b, int64_t h, int lin)
{
    constexpr int VBITS = PAGES ? 2 : VB;
    constexpr int GLV = PAGES ? 4 : VGL;
    static_assert(VBITS == 0 || VBITS == 2 || VBITS == 4, "value bits");
    static_assert(GLV == 2 || GLV == 4 || GLV == 8, "value group");
    constexpr bool DMA = NCH > 0;
    constexpr int NBUF = DMA ? NBUF_DMA : 2;
    constexpr int ROWLEN = DMA ? TILE_D : XROW;       // u16 per staged row
    static_assert(!DMA || (NBUF >= 2 && NBUF <= 4), "chunk buffers");
    __shared__ __attribute__((aligned(16))) uint16_t s_x[NBUF][CH * ROWLEN];
    __shared__ __attribute__((aligned(16))) float s_sal[TILE_D], s_smean[TILE_D], s_err[TILE_D], s_ehi[TILE_D], s_amax[TILE_D],
        s_scale[TILE_D];
    __shared__ int16_t s_src_of[TILE_D];
    __shared__ uint8_t s_is_src[TILE_D];
    __shared__ int16_t s_src[TILE_D / 2], s_don[TILE_D / 2];
    __shared__ __attribute__((aligned(16))) uint64_t s_key[TILE_D];
    __shared__ __attribute__((aligned(16))) int s_part[K4_THREADS];
    __shared__ __attribute__((aligned(16))) uint8_t s_flag[TILE_D];
    __shared__ int16_t s_list[TILE_D / 2];
    __shared__ int s_bad, s_again;

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t row = b * a.H + h;
    uint8_t *page = nullptr;
    __shared__ int16_t s_role[TILE_D];
    if constexpr (PAGES) {
        if (b == 0 && h == 0 && threadIdx.x < 3) a.clear[threadIdx.x] = 0;
        const int64_t id = a.id_bytes == 8 ? ((const int64_t *)a.ids)[b] : (int64_t)((const int32_t *)a.ids)[b];
        if (id < 0 || id >= a.pool_pages) {             // uniform: before any barrier or load
            if (threadIdx.x == 0) *a.badid = 1;
            return;
        }
        page = a.pool + id * a.page_bytes;
        if (threadIdx.x < TILE_D) s_role[threadIdx.x] = -1;
    }
    const int64_t prow = PAGES && a.page_rows ? a.page_rows[b] : -1;
    const int64_t xoff = prow >= 0 ? prow * a.st : b * a.sb, voff = prow >= 0 ? prow * a.vst : b * a.vsb;
    const uint16_t *xr = (const uint16_t *)a.x + xoff + h * a.sh;
    const int T = NCH > 0 ? NCH * CH : (int)a.T;
    const int stride = (int)min(a.stride, (int64_t)TILE_T);   // a larger stride samples token 0 only
    const int ns = (T + stride - 1) / stride;
    const int nch = (T + CH - 1) / CH;

    // chunk staging: thread tid moves segments tid and tid + 256 (row i / 16,
    // 8 channels at 8 (i % 16)); rows past T are clamped copies, never read.
    // The next chunk is in flight in registers while one is processed.
    u32x4_t seg[KPF][2];
    auto load_chunk = [&](int ch, u32x4_t (&sg)[2]) {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const int i = tid + K4_THREADS * k;
            const int t = min(ch * CH + (i >> 4), T - 1);
            sg[k] = *(const u32x4_t *)(xr + (int64_t)t * a.st + 8 * (i & 15));
        }
    };
    auto store_chunk = [&](const u32x4_t (&sg)[2], int buf) {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const int i = tid + K4_THREADS * k;
            *(u32x4_t *)(s_x[buf] + (i >> 4) * ROWLEN + 8 * (i & 15)) = sg[k];
        }
    };
    // direct loads of chunk ch into buffer ch % NBUF: each wave fills its two
    // 1 KiB quarters (64 lanes x 16 bytes, 4 rows each); every row is a whole
    // block row, so no clamping
    // LDS byte address of the staging buffers
    const uint32_t s_x_lds = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint16_t *)&s_x[0][0];
    // lane byte offset of segment 128 wave + lane within a chunk (rows 4 on
    // for the second load); the chunk base is wave-uniform
    const uint32_t dma_off = (uint32_t)(((8 * wave + (lane >> 4)) * (int)a.st + 8 * (lane & 15)) * 2);
    auto dma_chunk = [&](int ch) {
        const char *cb = (const char *)xr + (int64_t)ch * CH * a.st * 2;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const uint32_t dst = s_x_lds + (uint32_t)((ch % NBUF) * CH * ROWLEN * 2 + 16 * (128 * wave + 64 * k));
            lds_load16(cb, dma_off + (uint32_t)(k * 4 * (int)a.st * 2), dst);
        }
    };
    auto buf_of = [&](int ch) -> const uint16_t * { return s_x[DMA ? ch % NBUF : ch & 1]; };
    // registers: chunks 0..KPF-1 are loaded and chunk 0 is in LDS buffer 0;
    // direct loads: chunks 0..NBUF-2 are requested
    auto start_stream = [&]() {
        if constexpr (DMA) {
#pragma unroll
            for (int r = 0; r < NBUF - 1; ++r)
                if (r < NCH) dma_chunk(r);
        } else {
#pragma unroll
            for (int r = 0; r < KPF; ++r)
                if (r < nch) load_chunk(r, seg[r]);
        }
    };
    // visits chunks in order, chunk ch in buf_of(ch) during body(ch)
    auto stream = [&](auto &&body) {
        if constexpr (DMA) {
            // rolled: unrolled, the statistics spill 38 registers
#pragma unroll 1
            for (int ch = 0; ch < NCH; ++ch) {
                // requested so far: chunks 0 .. ch + NBUF - 2
                wait_chunk_barrier(min(NBUF - 2, NCH - 1 - ch));
                // every wave is past body(ch - 1): its buffer takes chunk ch + NBUF - 1
                if (ch + NBUF - 1 < NCH) dma_chunk(ch + NBUF - 1);
                body(ch);
            }
        } else {
            for (int c0 = 0; c0 < nch; c0 += KPF) {
#pragma unroll
                for (int r = 0; r < KPF; ++r) {
                    const int ch = c0 + r;
                    if (ch < nch) {
                        if (ch + KPF < nch) load_chunk(ch + KPF, seg[r]);   // seg[r] already sits in LDS
                        body(ch);
                        if (ch + 1 < nch) store_chunk(seg[(r + 1) % KPF], (ch + 1) & 1);
                        __syncthreads();
                    }
                }
            }
        }
    };

    start_stream();
    if (tid == 0) s_bad = 0;
    if constexpr (!DMA) store_chunk(seg[0], 0);
    __syncthreads();

    // ---- pass 1: statistics.  Thread (half, channel c1) takes the tokens of
    // one parity; which wavefronts are half 1, and add the samples as well,
    // alternates between the blocks that share a compute unit.
    const int half = (tid >> 7) ^ ((lin >> 8) & 1);
    double *const s_sum1 = (double *)s_key, *const s_sum2 = (double *)s_part;     // half 1's sums, until the selection
    double sum1 = 0.0, sum2 = 0.0;
    IqCascade sa, sm;                             // half 1
    sa.init(ns);
    sm.init(ns);
    uint32_t amax_bits = 0;
    int next_sample = 0;
    const int c1 = tid & (TILE_D - 1);
    auto pass1 = [&](auto sums, int ch) {
        const uint16_t *xs = buf_of(ch) + c1;
        const int t0 = ch * CH, nt = min(CH, T - t0);
        // |x| as 16-bit integers: for finite values their order is the
        // order of the magnitudes, and inf / NaN sort above every finite one
        auto take = [&](uint32_t u) {
            amax_bits = max(amax_bits, u & 0x7fffu);
            if constexpr (decltype(sums)::value) {
                const double d = (double)tile_f32<F16IN>(u);
                sum1 = __dadd_rn(sum1, d);
                sum2 = __builtin_fma(d, d, sum2);
            }
        };
        if (nt == CH) {
            uint32_t u[CH / 2];
#pragma unroll
            for (int k = 0; k < CH / 2; ++k) u[k] = xs[(2 * k + half) * ROWLEN];
#pragma unroll
            for (int k = 0; k < CH / 2; ++k) take(u[k]);
        } else {
            for (int k = half; k < nt; k += 2) take(xs[k * ROWLEN]);
        }
        if (half) {
            // the samples r * stride that fall in this chunk, in order
            for (; next_sample < t0 + nt; next_sample += stride) {
                const float v = tile_f32<F16IN>(xs[(next_sample - t0) * ROWLEN]);
                sa.add(fabsf(v));
                sm.add(v);
            }
        }
    };
    // the policy decided once: with a branch per element 127 x 8 blocks, K4 keys and values, bf16, took 66.6 us with
    // neighbors and 70.4 with min_error, now 60.1 and 67.7 (61.5 and 79.1 with a chain on two wavefronts)
    if (a.min_error) stream([&](int ch) { pass1(std::true_type{}, ch); });
    else stream([&](int ch) { pass1(std::false_type{}, ch); });
    if (half) {
        s_sum1[c1] = sum1;
        s_sum2[c1] = sum2;
        s_amax[c1] = __uint_as_float(amax_bits);
        s_sal[c1] = sa.finish() / (float)ns;
        s_smean[c1] = sm.finish() / (float)ns;
    }
    // A sealed block's last NBUF chunks are still in the buffers after pass 1
    // and pass 2 quantizes them first (RESIDENT), reloading the others into
    // the buffers they free; otherwise the first chunks of pass 2 load during
    // the selection (once every wave is done with pass 1's buffers).
    constexpr bool RESIDENT = DMA && NCH == 2 * NBUF;
    __syncthreads();
    if constexpr (!RESIDENT) start_stream();

    // ---- values (VBITS > 0), encoded by three wavefronts while the fourth
    // makes the sequential donor picks, with the row's HBM reads in that otherwise
    // idle stretch.  Thread vt of the three value wavefronts takes channels 16 vj .. 16 vj + 15
    // of token vtok0 + 24 it in iteration it (192 threads = 24 tokens), so a
    // group's GLV lanes are adjacent lanes of one wavefront.  A sealed block
    // (11 iterations) issues its first VPF iterations' loads here, before
    // the ranks; the rest run VPF iterations ahead.
    constexpr int VT = K4_THREADS - 64;
    constexpr int VIT = NCH > 0 ? (NCH * CH * 8 + VT - 1) / VT : 1;
    constexpr int VPF = 4;
    // The picking wavefront rotates between the workgroups that share a
    // compute unit (linear indices 256 apart): each SIMD then holds one
    // picking wavefront and three encoding values, instead of one SIMD
    // holding every picker while its VALU idles.  vtid is the thread's index
    // in that rotated order (virtual wave 0 picks).
    const int vtid = (tid + 64 * ((lin >> 8) & 3)) & (K4_THREADS - 1), vwave = vtid >> 6;
    const int vt = vtid - 64, vj = vt & 7, vtok0 = vt >> 3;
    u32x4_t vraw[NCH > 0 ? VIT : 1][2];
    auto vload = [&](int it, u32x4_t(&r)[2]) {
        const int t = min(vtok0 + 24 * it, T - 1);
        const u32x4_t *p = (const u32x4_t *)(a.v + voff + h * a.vsh + (int64_t)t * a.vst + 16 * vj);
        r[0] = __builtin_nontemporal_load(p);
        r[1] = __builtin_nontemporal_load(p + 1);
    };
    auto vencode = [&](int it, const u32x4_t(&r)[2], bool &vbad) {
        const int t = vtok0 + 24 * it;
        const bool live = t < T;
        uint32_t code[VBITS > 0 ? VBITS / 2 : 1];
        uint16_t off_h, sc_h;
        if constexpr (VBITS > 0) v_encode16<F16IN, VBITS, GLV>(r, live, code, off_h, sc_h, vbad);
        if (VBITS > 0 && live) {
            if constexpr (PAGES) {
                store_page_values(a, page, h, T, t, vj, code[0], off_h, sc_h);
            } else {
                constexpr int PB = TILE_D * (VBITS > 0 ? VBITS : 2) / 8;   // payload bytes per token
                constexpr int GROUPS = 8 / GLV;
                const int64_t vr = row * T + t;
                if constexpr (VBITS == 2) {
                    __builtin_nontemporal_store(code[0], (uint32_t *)(a.vpayload + vr * PB) + vj);
                } else {
                    typedef __attribute__((ext_vector_type(2))) uint32_t u32x2_t;
                    ((u32x2_t *)(a.vpayload + vr * PB))[vj] = u32x2_t{code[0], code[VBITS / 2 - 1]};
                }
                if (vj % GLV == 0) a.voffsets[vr * GROUPS + vj / GLV] = off_h;
                if (vj % GLV == GLV - 1) a.vscales[vr * GROUPS + vj / GLV] = sc_h;
            }
        }
    };
    if constexpr (VBITS > 0 && NCH > 0) {
        if (vwave > 0) {
#pragma unroll
            for (int it = 0; it < VPF; ++it) vload(it, vraw[it]);
        }
    }

    if (!half) {
        amax_bits = max(amax_bits, __float_as_uint(s_amax[c1]));
        const float amax = tile_f32<F16IN>(amax_bits);
        s_amax[c1] = amax;
        if (amax_bits >= (F16IN ? 0x7c00u : 0x7f80u)) s_bad = 1;     // an inf or NaN in the channel
        if (a.min_error) {
            const double s1 = __dadd_rn(sum1, s_sum1[c1]), s2 = __dadd_rn(sum2, s_sum2[c1]);
            const IqErrRange r = iq_err_range(s1, s2, amax, s_smean[c1], T, iq_same16(s1, s2, amax, T));
            s_err[c1] = r.lo;
            s_ehi[c1] = r.hi;
        }
    }
    __syncthreads();

    // the sequential donor picks on the picking wavefront hold up the whole block: top priority
    if (vwave == 0) __builtin_amdgcn_s_setprio(3);
    else __builtin_amdgcn_s_setprio(0);
    iq_select_tile128(s_sal, a.min_error ? s_err : nullptr, (int)a.count, s_src, s_don, s_is_src, s_src_of,
                      s_key, s_part, s_flag, s_list, vtid);
    if (vwave == 0) {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        const bool again = a.min_error && !s_bad && !iq_pool_certain(s_err, s_ehi, TILE_D, s_is_src, s_src_of);
        if (lane == 0) s_again = again;
    }
    if constexpr (VBITS > 0) {
        if (vwave > 0) {
            bool vbad = false;
            if constexpr (NCH > 0) {
#pragma unroll
                for (int it = 0; it < VIT; ++it) {
                    if (it + VPF < VIT) vload(it + VPF, vraw[it + VPF]);
                    vencode(it, vraw[it], vbad);
                }
            } else {
                const int nit = (T * 8 + VT - 1) / VT;
                for (int it = 0; it < nit; ++it) {
                    vload(it, vraw[0]);
                    vencode(it, vraw[0], vbad);
                }
            }
            if (__ballot(vbad) != 0 && lane == 0) atomicOr(a.vbad, 1);
        }
    }
    __builtin_amdgcn_s_setprio(1);
    __syncthreads();
    if (__builtin_expect(s_again, 0)) {
        // the pool is uncertain (errors that tie in real arithmetic and differ in their roundings; channels of one
        // value are exact, iq_same16): the reference's sequential errors, and the selection on them.  1024 rows of 256
        // bf16 tokens: 60 us where all take it, 37 where none does and 32 where all tokens are equal; with the chain in
        // place of the sums 38, 43 and 36
        if (tid == 0) atomicAdd(&uncertain_rows, 1u);
        if (tid < TILE_D)
            s_err[tid] = welford_error<F16IN ? IQ_F16 : IQ_BF16, 16, true>(xr, tid, a.st, T, s_smean[tid]);
        __syncthreads();
        if (tid < 64) iq_select_wave128(s_sal, s_err, (int)a.count, s_src, s_don, s_is_src, s_src_of, s_list);
        __syncthreads();
    }

    const float flt_min = 1.17549435e-38f;
    if (tid < TILE_D) {
        const float s = s_amax[tid] / (s_is_src[tid] ? 127.0f : 7.0f);
        const float sc = s < flt_min ? flt_min : s;
        s_scale[tid] = sc;
        if constexpr (PAGES) ((float *)(page + a.off_kscale))[h * TILE_D + tid] = sc;
        else a.scales[row * TILE_D + tid] = sc;
    }
    if (tid < a.count) {
        if constexpr (PAGES) {
            // page role map: the donor channel for a source, -2 - k for donor k
            s_role[s_src[tid]] = (int16_t)s_don[tid];
            s_role[s_don[tid]] = (int16_t)(-2 - tid);
            ((float *)(page + a.off_kpad))[h * a.count + tid] = s_smean[s_don[tid]];
        } else {
            store_desc(a.src, row * a.count + tid, s_src[tid], a.desc_bytes);
            store_desc(a.don, row * a.count + tid, s_don[tid], a.desc_bytes);
            a.padding[row * a.count + tid] = s_smean[s_don[tid]];
        }
    }
    if (tid == 0 && s_bad) atomicOr(a.bad, 1);
    if constexpr (!DMA) store_chunk(seg[0], 0);
    __syncthreads();

    // ---- pass 2: quantize; thread owns channels 8 j .. 8 j + 7 of tokens
    // t0 + 8 wave + tq and t0 + 8 wave + tq + 4 of every chunk
    const int j = lane & 15, tq = lane >> 4;
    K4Slots slots;
    slots.init(j, s_is_src, s_src_of, s_scale);
    // xe[e]: LDS address of slot e's value in row 8 wave + tq of buffer 0;
    // every other row and buffer is a constant offset from it
    const uint16_t *xe[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) xe[e] = &s_x[0][0] + (8 * wave + tq) * ROWLEN + slots.srcc[e];
    if constexpr (PAGES) {
        if (tid < TILE_D) ((int16_t *)(page + a.off_kmap))[h * TILE_D + tid] = s_role[tid];
    }
    uint32_t *out = PAGES ? (uint32_t *)(page + a.off_kpay + h * (int64_t)T * (TILE_D / 2))
                          : (uint32_t *)(a.payload + row * (int64_t)T * (TILE_D / 2));
    // chunks NCH - NBUF .. NCH - 1 from the buffers pass 1 left them in, then
    // chunk c < NCH - NBUF, loaded into buffer c % NBUF once every wave is
    // done with the resident chunk c + NBUF there (issued NBUF - 1 chunks
    // ahead of its use; waits as in stream(): vector memory operations retire
    // in order, and the stores issued in between only lengthen them)
    auto stream2 = [&](auto &&body) {
#pragma unroll
        for (int k = 0; k < NCH; ++k) {
            const int ch = k < NBUF ? NCH - NBUF + k : k - NBUF;
            if (k >= NBUF) wait_chunk_barrier(min(NBUF - 2, NCH - 1 - k));
            else if (k > 0) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            if (k > 0 && k <= NBUF) dma_chunk(k - 1);
            body(ch);
        }
    };
    auto pass2 = [&](int ch) {
        const int t0 = ch * CH;
#pragma unroll
        for (int it = 0; it < 2; ++it) {
            const int tl = 8 * wave + 4 * it + tq, t = t0 + tl;
            if (t < T) {
                const int off = (DMA ? ch % NBUF : ch & 1) * CH * ROWLEN + 4 * it * ROWLEN;
                float v[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] = tile_f32<F16IN>(xe[e][off]);
                __builtin_nontemporal_store(slots.word(v), &out[t * (TILE_D / 8) + j]);
            }
        }
    };
    if constexpr (RESIDENT) stream2(pass2);
    else stream(pass2);
}

// grid (blocks, heads): no 64-bit division for the row's coordinates
template <bool F16IN, int NCH, bool PAGES = false, int VB = 0, int VGL = 4>
__global__ __launch_bounds__(K4_THREADS, 4) void k4_encode_tile(K4Args a)
{
    k4_tile_body<F16IN, NCH, PAGES, VB, VGL>(a, blockIdx.x, blockIdx.y, (int)(blockIdx.x + gridDim.x * blockIdx.y));
}

// Keys and values of the same blocks, both K4, in one launch: grid (blocks,
// 2 H), rows h < H of the keys `ak`, the others of the values `av`.
template <bool F16IN, int NCH>
__global__ __launch_bounds__(K4_THREADS, 4) void k4_encode_pair(K4Args ak, K4Args av)
{
    const bool val = (int64_t)blockIdx.y >= ak.H;
    const K4Args a = val ? av : ak;
    k4_tile_body<F16IN, NCH>(a, blockIdx.x, val ? blockIdx.y - ak.H : blockIdx.y,
                             (int)(blockIdx.x + gridDim.x * blockIdx.y));
}

// Pages of T = 16 or 32 tokens: one wavefront encodes one (page, head) row,
// keys and values, and a workgroup holds four rows (pages 4 blockIdx.x + wave
// of head blockIdx.y) that share nothing, so there is no workgroup barrier.
// A short row keeps the serial phases of the 256-thread tile encoder (the
// donor selection is the same 16 picks for 16 tokens as for 256) while its
// other waves idle; here each wavefront runs its own row from start to end
// and a compute unit interleaves twenty rows.  The arithmetic and its order
// are the tile encoder's, so the page bytes are the same:
//   lane l owns channels 2 l and 2 l + 1 for the statistics (fp64 Welford
//   with the exact reciprocals 1 / n, amax as 16-bit magnitudes, sampled sums
//   in torch's cascade order), iq_select_wave128 makes the selection, lane
//   (j, tq) = (l % 16, l / 16) packs channels 8 j .. 8 j + 7 of tokens
//   tq + 4 i, and lane (vj, vt) = (l % 8, l / 8) encodes channels
//   16 vj .. 16 vj + 15 of value tokens vt + 8 i.
// Lanes read LDS words other lanes of the same wavefront wrote: a
// wavefront's LDS operations complete in order, so the wavefront-scope
// fences emit nothing and only keep the compiler from reordering.
template <bool F16IN, int T>
__global__ __launch_bounds__(K4_THREADS) void k4_encode_page_rows(K4Args a, int64_t n_pages)
{
    static_assert(T == 16 || T == 32, "short pages");
    constexpr int ROW = TILE_D + 8;            // u16 per staged token row
    constexpr int KSEG = T * (TILE_D / 8) / 64; // 16-byte key segments per lane
    constexpr int VIT = T / 8;                 // value tokens per lane
    __shared__ __attribute__((aligned(16))) uint16_t s_x[4][T * ROW];
    __shared__ __attribute__((aligned(8))) float s_sal[4][TILE_D], s_err[4][TILE_D], s_mean[4][TILE_D];
    __shared__ int16_t s_src[4][TILE_D / 2], s_don[4][TILE_D / 2], s_src_of[4][TILE_D], s_role[4][TILE_D];
    __shared__ int16_t s_list[4][TILE_D / 2];
    __shared__ uint8_t s_is_src[4][TILE_D];

    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int64_t b = (int64_t)blockIdx.x * 4 + wave, h = blockIdx.y;
    if (blockIdx.x == 0 && h == 0 && threadIdx.x < 3) a.clear[threadIdx.x] = 0;
    if (b >= n_pages) return;                  // wave-uniform, as the page check below
    const int64_t id = a.id_bytes == 8 ? ((const int64_t *)a.ids)[b] : (int64_t)((const int32_t *)a.ids)[b];
    if (id < 0 || id >= a.pool_pages) {
        if (lane == 0) *a.badid = 1;
        return;
    }
    uint8_t *const page = a.pool + id * a.page_bytes;
    const int64_t prow = a.page_rows ? a.page_rows[b] : -1;
    const uint16_t *const xr = (const uint16_t *)a.x + (prow >= 0 ? prow * a.st : b * a.sb) + h * a.sh;
    const uint16_t *const vr = a.v + (prow >= 0 ? prow * a.vst : b * a.vsb) + h * a.vsh;

    // every load of the row first: key segment i = lane + 64 k is token i / 16,
    // channels 8 (i % 16) ..; value lane (vj, vt) reads 16 channels of token vt + 8 it
    const int vj = lane & 7, vt = lane >> 3;
    u32x4_t kseg[KSEG], vraw[VIT][2];
#pragma unroll
    for (int k = 0; k < KSEG; ++k) {
        const int i = lane + 64 * k;
        kseg[k] = *(const u32x4_t *)(xr + (int64_t)(i >> 4) * a.st + 8 * (i & 15));
    }
#pragma unroll
    for (int it = 0; it < VIT; ++it) {
        const u32x4_t *p = (const u32x4_t *)(vr + (int64_t)(vt + 8 * it) * a.vst + 16 * vj);
        vraw[it][0] = __builtin_nontemporal_load(p);
        vraw[it][1] = __builtin_nontemporal_load(p + 1);
    }
    uint16_t *const xs = s_x[wave];
#pragma unroll
    for (int k = 0; k < KSEG; ++k) {
        const int i = lane + 64 * k;
        *(u32x4_t *)(xs + (i >> 4) * ROW + 8 * (i & 15)) = kseg[k];
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");

    // ---- statistics of channels 2 lane and 2 lane + 1
    double mean[2] = {0.0, 0.0}, m2[2] = {0.0, 0.0};
    uint32_t amax_bits[2] = {0u, 0u};
#pragma unroll
    for (int t = 0; t < T; ++t) {
        const uint32_t w = *(const uint32_t *)(xs + t * ROW + 2 * lane);
        // delta / n with y_hi = RN(1/n) and y_lo = RN((1 - y_hi n) / n) (the
        // residual 1 - y_hi n is exact) is one fma: RN(delta y_hi +
        // RN(delta y_lo)).  A quotient by an integer n <= 256 is never a
        // midpoint between doubles and lies at least ulp / 512 from one, while
        // the fma's exact argument is within 2^-52 ulp of it
        // (tests/test_welford_division.py)
        const double n = (double)(t + 1);
        const double yh = 1.0 / n;
        const double yl = __builtin_fma(-yh, n, 1.0) / n;
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const uint32_t u = e ? w >> 16 : w & 0xffffu;
            amax_bits[e] = max(amax_bits[e], u & 0x7fffu);
            const double dv = (double)tile_f32<F16IN>(u);
            const double delta = __dsub_rn(dv, mean[e]);
            mean[e] = __dadd_rn(mean[e], __builtin_fma(delta, yh, __dmul_rn(delta, yl)));
            m2[e] = __dadd_rn(m2[e], __dmul_rn(delta, __dsub_rn(dv, mean[e])));
        }
    }
    const int stride = (int)min(a.stride, (int64_t)TILE_T);   // a larger stride samples token 0 only
    const int ns = (T + stride - 1) / stride;
    IqCascade sa[2], sm[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        sa[e].init(ns);
        sm[e].init(ns);
    }
    for (int t = 0; t < T; t += stride) {
        const uint32_t w = *(const uint32_t *)(xs + t * ROW + 2 * lane);
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const float v = tile_f32<F16IN>(e ? w >> 16 : w & 0xffffu);
            sa[e].add(fabsf(v));
            sm[e].add(v);
        }
    }
    float amax[2];
    bool kbad = false;
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        const int c = 2 * lane + e;
        const float smean = sm[e].finish() / (float)ns;
        const float diff = __fsub_rn((float)mean[e], smean);
        s_err[wave][c] = __fadd_rn((float)(m2[e] / (double)T), __fmul_rn(diff, diff));
        s_sal[wave][c] = sa[e].finish() / (float)ns;
        s_mean[wave][c] = smean;
        amax[e] = tile_f32<F16IN>(amax_bits[e]);
        kbad |= amax_bits[e] >= (F16IN ? 0x7c00u : 0x7f80u);   // an inf or NaN in the channel
    }
    if (__ballot(kbad) != 0 && lane == 0) atomicOr(a.bad, 1);

    // ---- values, while the selection's inputs settle
    bool vbad = false;
#pragma unroll
    for (int it = 0; it < VIT; ++it) {
        uint32_t code[1];
        uint16_t off_h, sc_h;
        v_encode16<F16IN, 2, 4>(vraw[it], true, code, off_h, sc_h, vbad);
        store_page_values(a, page, h, T, vt + 8 * it, vj, code[0], off_h, sc_h);
    }
    if (__ballot(vbad) != 0 && lane == 0) atomicOr(a.vbad, 1);

    // ---- selection, scales, role map and padding
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    const int count = (int)a.count;
    iq_select_wave128(s_sal[wave], s_err[wave], count, s_src[wave], s_don[wave], s_is_src[wave], s_src_of[wave],
                      s_list[wave]);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    const float flt_min = 1.17549435e-38f;
    float *const kscale = (float *)(page + a.off_kscale) + h * TILE_D;
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        const int c = 2 * lane + e;
        const float s = amax[e] / (s_is_src[wave][c] ? 127.0f : 7.0f);
        const float sc = s < flt_min ? flt_min : s;
        s_sal[wave][c] = sc;                   // the saliencies are spent: scales from here on
        kscale[c] = sc;
        s_role[wave][c] = -1;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    if (lane < count) {
        // page role map: the donor channel for a source, -2 - k for donor k
        const int s = s_src[wave][lane], d = s_don[wave][lane];
        s_role[wave][s] = (int16_t)d;
        s_role[wave][d] = (int16_t)(-2 - lane);
        ((float *)(page + a.off_kpad))[h * count + lane] = s_mean[wave][d];
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    int16_t *const kmap = (int16_t *)(page + a.off_kmap) + h * TILE_D;
    kmap[2 * lane] = s_role[wave][2 * lane];
    kmap[2 * lane + 1] = s_role[wave][2 * lane + 1];

    // ---- 4-bit slots
    const int j = lane & 15, tq = lane >> 4;
    K4Slots slots;
    slots.init(j, s_is_src[wave], s_src_of[wave], s_sal[wave]);
    uint32_t *const out = (uint32_t *)(page + a.off_kpay + h * (int64_t)T * (TILE_D / 2));
#pragma unroll
    for (int it = 0; it < T / 4; ++it) {
        const int t = tq + 4 * it;
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = tile_f32<F16IN>(xs[t * ROW + slots.srcc[e]]);
        __builtin_nontemporal_store(slots.word(v), &out[t * (TILE_D / 8) + j]);
    }
}

struct SelectArgs {
    const float *sal, *err;
    int64_t D, count;
    int64_t *src, *don;
};

// NC: 4 for D <= 256, else the 64-channel groups of 512 or 1024 channels, each
// in a kernel of its own (together their lane masks spill twice as many scalar
// registers: 1024 rows of 512 channels, 256 picks, 197 us instead of 177).
template <int NC>
__global__ __launch_bounds__(64) void reuse_map_kernel(SelectArgs a)
{
    __shared__ float s_sal[IQ_MAXD];
    __shared__ float s_err[IQ_MAXD];
    __shared__ int16_t s_src_of[IQ_MAXD];
    __shared__ uint8_t s_is_src[IQ_MAXD];
    __shared__ int16_t s_src[IQ_MAXD / 2];
    __shared__ int16_t s_don[IQ_MAXD / 2];
    const int64_t row = blockIdx.x;
    for (int64_t c = threadIdx.x; c < a.D; c += 64) {
        s_sal[c] = a.sal[row * a.D + c];
        if (a.err) s_err[c] = a.err[row * a.D + c];
    }
    __syncthreads();
    const float *const err = a.err ? s_err : nullptr;
    if constexpr (NC > 4) iq_select_wave_t<NC>(s_sal, err, (int)a.D, (int)a.count, s_src, s_don, s_is_src, s_src_of);
    else iq_select_wave<false>(s_sal, err, (int)a.D, (int)a.count, s_src, s_don, s_is_src, s_src_of);
    __syncthreads();
    for (int64_t i = threadIdx.x; i < a.count; i += 64) {
        a.src[row * a.count + i] = s_src[i];
        a.don[row * a.count + i] = s_don[i];
    }
}

// D = 128: one wavefront per row with the radix top-k selection of the page
// row encoder (iq_select_wave128), the same picks as iq_select_wave.
__global__ __launch_bounds__(64) void reuse_map128_kernel(SelectArgs a)
{
    __shared__ float s_sal[128], s_err[128];
    __shared__ int16_t s_src_of[128], s_src[64], s_don[64], s_list[64];
    __shared__ uint8_t s_is_src[128];
    const int64_t row = blockIdx.x;
    const int lane = threadIdx.x;
    s_sal[lane] = a.sal[row * 128 + lane];
    s_sal[64 + lane] = a.sal[row * 128 + 64 + lane];
    if (a.err) {
        s_err[lane] = a.err[row * 128 + lane];
        s_err[64 + lane] = a.err[row * 128 + 64 + lane];
    }
    __syncthreads();
    iq_select_wave128(s_sal, a.err ? s_err : nullptr, (int)a.count, s_src, s_don, s_is_src, s_src_of, s_list);
    __syncthreads();
    if (lane < a.count) {
        a.src[row * a.count + lane] = s_src[lane];
        a.don[row * a.count + lane] = s_don[lane];
    }
}

}  // namespace

namespace {

// the tile encoder's layout: 16-bit channel-contiguous rows of 128 channels,
// 16-byte aligned, at most 256 tokens, 32-bit lane offsets within a chunk
bool tile_ok(const void *x, int dtype, const int64_t *s, int64_t T, int64_t D)
{
    return (dtype == IQ_BF16 || dtype == IQ_F16) && D == TILE_D && T <= TILE_T && s[3] == 1 && s[2] % 8 == 0 &&
           s[1] % 8 == 0 && s[0] % 8 == 0 && ((uintptr_t)x & 15) == 0 && s[2] >= 0 && s[2] <= (1 << 24);
}

}  // namespace

namespace {

// General rows: B * H rows of `a`.
template <int DT>
int launch_rows(const K4Args &a, int64_t B, hipStream_t st)
{
    const int64_t rows = B * a.H, T = a.T, D = a.D;
    // quantize_words: 16-byte pieces of channel-contiguous rows, whole words out
    constexpr int64_t EB = DT == IQ_F64 ? 8 : DT == IQ_F32 ? 4 : 2, VE = 16 / EB;
    const bool words = DT != IQ_F64 && D % 8 == 0 && a.sc == 1 && a.st % VE == 0 && a.sh % VE == 0 && a.sb % VE == 0 &&
                       ((uintptr_t)a.x & 15) == 0 && ((uintptr_t)a.payload & 3) == 0;
    // long rows (up to 2^24 tokens: the level-0 sums of a piece fit its LDS):
    // chunks for about 1024 workgroups (eight rows of 32768 tokens: 63 us for
    // the three launches, 68 with 512 and 83 with 2048), and the partial
    // results in the row's payload bytes
    constexpr int64_t MAXCH = 1024;
    int64_t chunk = 64;
    while (chunk < 1024 && rows * ((T + chunk - 1) / chunk) > MAXCH) chunk *= 2;
    const RowPlan p = row_plan(T, D, a.stride, chunk);
    if (T > LONG_ROW && T <= (int64_t(1) << 24) && rows <= 65535 && p.bytes + 15 <= T * (D / 2)) {
        const dim3 parts((unsigned)(p.nchunk + p.pieces * ((p.nseq + 63) / 64)), (unsigned)rows);
        const dim3 tiles((unsigned)p.nchunk, (unsigned)rows);
        if constexpr (DT != IQ_F64) {
            if (words) hipLaunchKernelGGL((k4_row_stats<DT, true>), parts, dim3(K4_THREADS), 0, st, a, p);
        }
        if (!words) hipLaunchKernelGGL((k4_row_stats<DT, false>), parts, dim3(K4_THREADS), 0, st, a, p);
        if (D > 256) hipLaunchKernelGGL((k4_row_select<DT, true>), dim3((unsigned)rows), dim3(ROW_THREADS), 0, st, a, p);
        else hipLaunchKernelGGL((k4_row_select<DT, false>), dim3((unsigned)rows), dim3(ROW_THREADS), 0, st, a, p);
        if constexpr (DT != IQ_F64) {
            if (words) hipLaunchKernelGGL((k4_quantize_rows<DT, true>), tiles, dim3(K4_THREADS), 0, st, a, p.chunk);
        }
        if (!words) hipLaunchKernelGGL((k4_quantize_rows<DT, false>), tiles, dim3(K4_THREADS), 0, st, a, p.chunk);
        IQ_CHECK_LAUNCH("k4_row_stats, k4_row_select, k4_quantize_rows");
        return IQ_OK;
    }
    const dim3 grid((unsigned)rows), block(ROW_THREADS);
    if constexpr (DT != IQ_F64) {
        if (words && D > 256) hipLaunchKernelGGL((k4_encode_kernel<DT, true, true>), grid, block, 0, st, a);
        else if (words) hipLaunchKernelGGL((k4_encode_kernel<DT, true, false>), grid, block, 0, st, a);
    }
    if (!words && D > 256) hipLaunchKernelGGL((k4_encode_kernel<DT, false, true>), grid, block, 0, st, a);
    else if (!words) hipLaunchKernelGGL((k4_encode_kernel<DT, false, false>), grid, block, 0, st, a);
    IQ_CHECK_LAUNCH("k4_encode_kernel");
    return IQ_OK;
}

}  // namespace

extern "C" int iq_k4_uncertain_rows(uint32_t *rows)
{
    IQ_CHECK_ARG(rows, "iq_k4_uncertain_rows: null pointer");
    const hipError_t e = hipMemcpyFromSymbol(rows, HIP_SYMBOL(uncertain_rows), sizeof *rows);
    if (e != hipSuccess) return iq_fail(IQ_ERR_DEVICE, "iq_k4_uncertain_rows: %s", hipGetErrorString(e));
    return IQ_OK;
}

extern "C" int iq_k4_quantize(const void *x, int x_dtype, const int64_t *x_strides, int64_t B, int64_t H,
                              int64_t T, int64_t D, int64_t count, int64_t sample_stride, int min_error,
                              uint8_t *payload, float *scales, void *src, void *don, int desc_bytes,
                              float *padding, int *bad_flag, void *stream)
{
    IQ_CHECK_ARG(x && x_strides && payload && scales && bad_flag, "iq_k4_quantize: null pointer");
    IQ_CHECK_ARG(x_dtype >= IQ_F32 && x_dtype <= IQ_F64, "iq_k4_quantize: bad dtype %d", x_dtype);
    IQ_CHECK_ARG(B >= 1 && H >= 1 && T >= 1, "iq_k4_quantize: empty shape");
    IQ_CHECK_ARG(D >= 2 && D % 2 == 0 && D <= IQ_MAXD, "iq_k4_quantize: D=%lld must be even and <= %d",
                 (long long)D, IQ_MAXD);
    IQ_CHECK_ARG(count >= 0 && 2 * count <= D, "iq_k4_quantize: count=%lld out of range", (long long)count);
    IQ_CHECK_ARG(count == 0 || (src && don && padding), "iq_k4_quantize: null descriptor output");
    IQ_CHECK_ARG(sample_stride >= 1, "iq_k4_quantize: sample_stride must be positive");
    IQ_CHECK_ARG(desc_bytes == 1 || desc_bytes == 4 || desc_bytes == 8, "iq_k4_quantize: desc_bytes");
    IQ_CHECK_ARG(B * H <= 0x7fffffffLL, "iq_k4_quantize: too many rows");
    K4Args a{x, x_dtype, x_strides[0], x_strides[1], x_strides[2], x_strides[3], H, T, D, count, sample_stride,
             min_error ? 1 : 0, payload, scales, src, don, desc_bytes, padding, bad_flag};
    if (tile_ok(x, x_dtype, x_strides, T, D) && H <= 65535) {
        const dim3 grid((unsigned)B, (unsigned)H), block(K4_THREADS);
        const hipStream_t st = (hipStream_t)stream;
        if (x_dtype == IQ_F16) {
            if (T == TILE_T) hipLaunchKernelGGL((k4_encode_tile<true, TILE_T / CH>), grid, block, 0, st, a);
            else hipLaunchKernelGGL((k4_encode_tile<true, 0>), grid, block, 0, st, a);
        } else {
            if (T == TILE_T) hipLaunchKernelGGL((k4_encode_tile<false, TILE_T / CH>), grid, block, 0, st, a);
            else hipLaunchKernelGGL((k4_encode_tile<false, 0>), grid, block, 0, st, a);
        }
        IQ_CHECK_LAUNCH("k4_encode_tile");
        return IQ_OK;
    }
    const hipStream_t st = (hipStream_t)stream;
    switch (x_dtype) {
    case IQ_BF16: return launch_rows<IQ_BF16>(a, B, st);
    case IQ_F16: return launch_rows<IQ_F16>(a, B, st);
    case IQ_F64: return launch_rows<IQ_F64>(a, B, st);
    default: return launch_rows<IQ_F32>(a, B, st);
    }
}

namespace {

template <bool F16IN, int VB>
void launch_kv_tile(int VGL, dim3 grid, hipStream_t st, const K4Args &a)
{
    constexpr int N = TILE_T / CH;
    switch (VGL) {
    case 2: hipLaunchKernelGGL((k4_encode_tile<F16IN, N, false, VB, 2>), grid, dim3(K4_THREADS), 0, st, a); break;
    case 4: hipLaunchKernelGGL((k4_encode_tile<F16IN, N, false, VB, 4>), grid, dim3(K4_THREADS), 0, st, a); break;
    default: hipLaunchKernelGGL((k4_encode_tile<F16IN, N, false, VB, 8>), grid, dim3(K4_THREADS), 0, st, a); break;
    }
}

}  // namespace

extern "C" int iq_kv_quantize(const void *keys, const void *values, int dtype, const int64_t *k_strides,
                              const int64_t *v_strides, int64_t B, int64_t H, int64_t T, int64_t D,
                              int64_t count, int64_t sample_stride, int min_error, uint8_t *k_payload,
                              float *k_scales, void *src, void *don, int desc_bytes, float *padding,
                              int value_bits, int value_group, uint8_t *v_payload, uint16_t *v_scales,
                              uint16_t *v_offsets, int *key_bad, int *value_bad, void *stream)
{
    IQ_CHECK_ARG(keys && values && k_strides && v_strides && k_payload && k_scales && v_payload && v_scales &&
                     v_offsets && key_bad && value_bad,
                 "iq_kv_quantize: null pointer");
    IQ_CHECK_ARG(value_bits == 2 || value_bits == 4, "iq_kv_quantize: value_bits must be 2 or 4");
    IQ_CHECK_ARG(value_group == 32 || value_group == 64 || value_group == 128,
                 "iq_kv_quantize: value_group must be 32, 64 or 128");
    auto rows16 = [](const void *p, const int64_t *s) {
        return ((uintptr_t)p & 15) == 0 && s[3] == 1 && s[0] % 8 == 0 && s[1] % 8 == 0 && s[2] % 8 == 0 &&
               s[2] >= 0 && s[2] <= (1 << 23);
    };
    const bool fused = (dtype == IQ_BF16 || dtype == IQ_F16) && D == TILE_D && T == TILE_T && B >= 1 &&
                       B <= 0x7fffffffLL && H >= 1 && H <= 65535 && B * H <= 0x7fffffffLL && count >= 0 &&
                       2 * count <= D && (count == 0 || (src && don && padding)) && sample_stride >= 1 &&
                       (desc_bytes == 1 || desc_bytes == 4 || desc_bytes == 8) && rows16(keys, k_strides) &&
                       rows16(values, v_strides);
    if (!fused) {
        // any other shape: the two encoders back to back on the stream
        const int rk = iq_k4_quantize(keys, dtype, k_strides, B, H, T, D, count, sample_stride, min_error,
                                      k_payload, k_scales, src, don, desc_bytes, padding, key_bad, stream);
        if (rk != IQ_OK) return rk;
        return iq_v_quantize(values, dtype, v_strides, B, H, T, D, value_bits, value_group, v_payload, v_scales,
                             v_offsets, value_bad, stream);
    }
    K4Args a{};
    a.x = keys;
    a.dt = dtype;
    a.sb = k_strides[0];
    a.sh = k_strides[1];
    a.st = k_strides[2];
    a.sc = 1;
    a.H = H;
    a.T = T;
    a.D = D;
    a.count = count;
    a.stride = sample_stride;
    a.min_error = min_error ? 1 : 0;
    a.payload = k_payload;
    a.scales = k_scales;
    a.src = src;
    a.don = don;
    a.desc_bytes = desc_bytes;
    a.padding = padding;
    a.bad = key_bad;
    a.v = (const uint16_t *)values;
    a.vsb = v_strides[0];
    a.vsh = v_strides[1];
    a.vst = v_strides[2];
    a.vbad = value_bad;
    a.vpayload = v_payload;
    a.vscales = v_scales;
    a.voffsets = v_offsets;
    const dim3 grid((unsigned)B, (unsigned)H);
    const hipStream_t st = (hipStream_t)stream;
    const int VGL = value_group / 16;
    if (dtype == IQ_F16) {
        if (value_bits == 2) launch_kv_tile<true, 2>(VGL, grid, st, a);
        else launch_kv_tile<true, 4>(VGL, grid, st, a);
    } else {
        if (value_bits == 2) launch_kv_tile<false, 2>(VGL, grid, st, a);
        else launch_kv_tile<false, 4>(VGL, grid, st, a);
    }
    IQ_CHECK_LAUNCH("k4_encode_tile (keys and values)");
    return IQ_OK;
}

extern "C" int iq_k4_quantize_kv(const void *keys, const void *values, int dtype, const int64_t *k_strides,
                                 const int64_t *v_strides, int64_t B, int64_t H, int64_t T, int64_t D, int64_t count,
                                 int64_t sample_stride, int min_error, uint8_t *k_payload, float *k_scales,
                                 void *k_src, void *k_don, float *k_padding, uint8_t *v_payload, float *v_scales,
                                 void *v_src, void *v_don, float *v_padding, int desc_bytes, int *key_bad,
                                 int *value_bad, void *stream)
{
    IQ_CHECK_ARG(keys && values && k_strides && v_strides && key_bad && value_bad, "iq_k4_quantize_kv: null pointer");
    const bool fused = tile_ok(keys, dtype, k_strides, T, D) && tile_ok(values, dtype, v_strides, T, D) && B >= 1 &&
                       B <= 0x7fffffffLL && H >= 1 && 2 * H <= 65535 && T >= 1 && count >= 0 && 2 * count <= D &&
                       sample_stride >= 1 && (desc_bytes == 1 || desc_bytes == 4 || desc_bytes == 8) &&
                       k_payload && k_scales && v_payload && v_scales &&
                       (count == 0 || (k_src && k_don && k_padding && v_src && v_don && v_padding));
    if (!fused) {
        // any other shape: the two encodes back to back on the stream
        const int rk = iq_k4_quantize(keys, dtype, k_strides, B, H, T, D, count, sample_stride, min_error, k_payload,
                                      k_scales, k_src, k_don, desc_bytes, k_padding, key_bad, stream);
        if (rk != IQ_OK) return rk;
        return iq_k4_quantize(values, dtype, v_strides, B, H, T, D, count, sample_stride, min_error, v_payload,
                              v_scales, v_src, v_don, desc_bytes, v_padding, value_bad, stream);
    }
    const K4Args ak{keys, dtype, k_strides[0], k_strides[1], k_strides[2], k_strides[3], H, T, D, count,
                    sample_stride, min_error ? 1 : 0, k_payload, k_scales, k_src, k_don, desc_bytes, k_padding,
                    key_bad};
    const K4Args av{values, dtype, v_strides[0], v_strides[1], v_strides[2], v_strides[3], H, T, D, count,
                    sample_stride, min_error ? 1 : 0, v_payload, v_scales, v_src, v_don, desc_bytes, v_padding,
                    value_bad};
    const dim3 grid((unsigned)B, (unsigned)(2 * H)), block(K4_THREADS);
    const hipStream_t st = (hipStream_t)stream;
    if (dtype == IQ_F16) {
        if (T == TILE_T) hipLaunchKernelGGL((k4_encode_pair<true, TILE_T / CH>), grid, block, 0, st, ak, av);
        else hipLaunchKernelGGL((k4_encode_pair<true, 0>), grid, block, 0, st, ak, av);
    } else {
        if (T == TILE_T) hipLaunchKernelGGL((k4_encode_pair<false, TILE_T / CH>), grid, block, 0, st, ak, av);
        else hipLaunchKernelGGL((k4_encode_pair<false, 0>), grid, block, 0, st, ak, av);
    }
    IQ_CHECK_LAUNCH("k4_encode_pair");
    return IQ_OK;
}

extern "C" int iq_reuse_map(const float *saliency, const float *donor_error, int64_t rows, int64_t D,
                            int64_t count, int64_t *src, int64_t *don, void *stream)
{
    IQ_CHECK_ARG(rows >= 0 && D >= 1 && D <= IQ_MAXD, "iq_reuse_map: D=%lld unsupported", (long long)D);
    IQ_CHECK_ARG(count >= 0 && 2 * count <= D, "iq_reuse_map: count=%lld out of range", (long long)count);
    IQ_CHECK_ARG(rows <= 0x7fffffffLL, "iq_reuse_map: too many rows");
    if (rows == 0 || count == 0) return IQ_OK;
    IQ_CHECK_ARG(saliency && src && don, "iq_reuse_map: null pointer");
    SelectArgs a{saliency, donor_error, D, count, src, don};
    if (D == 128) hipLaunchKernelGGL(reuse_map128_kernel, dim3((unsigned)rows), dim3(64), 0, (hipStream_t)stream, a);
    else if (D > 512) hipLaunchKernelGGL(reuse_map_kernel<16>, dim3((unsigned)rows), dim3(64), 0, (hipStream_t)stream, a);
    else if (D > 256) hipLaunchKernelGGL(reuse_map_kernel<8>, dim3((unsigned)rows), dim3(64), 0, (hipStream_t)stream, a);
    else hipLaunchKernelGGL(reuse_map_kernel<4>, dim3((unsigned)rows), dim3(64), 0, (hipStream_t)stream, a);
    IQ_CHECK_LAUNCH("reuse_map_kernel");
    return IQ_OK;
}

extern "C" int iq_encode_pages(const void *keys, const void *values, int dtype, const int64_t *k_strides,
                               const int64_t *v_strides, int64_t n_pages, int64_t H, int64_t block_tokens,
                               uint8_t *pool, int64_t pool_pages, const void *page_ids, int id_bytes, int *flags,
                               int *next_flags, void *stream)
{
    return iq_encode_pages_at(keys, values, dtype, k_strides, v_strides, nullptr, n_pages, H, block_tokens, pool,
                              pool_pages, page_ids, id_bytes, flags, next_flags, stream);
}

extern "C" int iq_encode_pages_at(const void *keys, const void *values, int dtype, const int64_t *k_strides,
                                  const int64_t *v_strides, const int64_t *page_rows, int64_t n_pages, int64_t H,
                                  int64_t block_tokens, uint8_t *pool, int64_t pool_pages, const void *page_ids,
                                  int id_bytes, int *flags, int *next_flags, void *stream)
{
    IQ_CHECK_ARG(keys && values && k_strides && v_strides && pool && page_ids && flags && next_flags,
                 "iq_encode_pages: null pointer");
    IQ_CHECK_ARG(dtype == IQ_BF16 || dtype == IQ_F16, "iq_encode_pages: keys/values must be bf16 or f16");
    IQ_CHECK_ARG(id_bytes == 4 || id_bytes == 8, "iq_encode_pages: id_bytes");
    const int64_t B = block_tokens;
    IQ_CHECK_ARG(B == 16 || B == 32 || B == 64 || B == 128 || B == 256, "iq_encode_pages: %lld-token pages",
                 (long long)B);
    IQ_CHECK_ARG(n_pages >= 0 && n_pages <= 0x7fffffffLL && H >= 1 && H <= 65535, "iq_encode_pages: shape");
    // rows read as 16-byte vectors (keys through direct-to-LDS chunk loads)
    auto rows_ok = [](const void *p, const int64_t *st) {
        return ((uintptr_t)p & 15) == 0 && st[3] == 1 && st[0] % 8 == 0 && st[1] % 8 == 0 && st[2] % 8 == 0 &&
               st[2] >= 0 && st[2] <= (1 << 24);
    };
    IQ_CHECK_ARG(rows_ok(keys, k_strides) && rows_ok(values, v_strides),
                 "iq_encode_pages: key/value rows must be contiguous and 16-byte aligned");
    const int64_t page_bytes = H * (104 * B + 832);
    K4Args a{};
    a.x = keys;
    a.dt = dtype;
    a.sb = k_strides[0];
    a.sh = k_strides[1];
    a.st = k_strides[2];
    a.sc = 1;
    a.H = H;
    a.T = B;
    a.D = TILE_D;
    a.count = 16;
    a.stride = 8;
    a.min_error = 1;
    a.bad = flags;
    a.pool = pool;
    a.pool_pages = pool_pages;
    a.page_bytes = page_bytes;
    a.ids = page_ids;
    a.id_bytes = id_bytes;
    a.off_kpay = 0;
    a.off_kscale = H * B * 64;
    a.off_kmap = a.off_kscale + H * 128 * 4;
    a.off_kpad = a.off_kmap + H * 128 * 2;
    a.off_vpay = a.off_kpad + H * 16 * 4;
    a.off_vscale = a.off_vpay + H * B * 32;
    a.off_voff = a.off_vscale + H * B * 2 * 2;
    a.v = (const uint16_t *)values;
    a.vsb = v_strides[0];
    a.vsh = v_strides[1];
    a.vst = v_strides[2];
    a.vbad = flags + 1;
    a.badid = flags + 2;
    a.clear = next_flags;
    a.page_rows = page_rows;
    if (n_pages == 0) return IQ_OK;
    const hipStream_t st = (hipStream_t)stream;
    if (B <= 32) {
        // one wavefront per (page, head) row, four pages of one head per workgroup
        const dim3 rows_grid((unsigned)((n_pages + 3) / 4), (unsigned)H);
        if (dtype == IQ_F16) {
            if (B == 16) hipLaunchKernelGGL((k4_encode_page_rows<true, 16>), rows_grid, dim3(K4_THREADS), 0, st, a, n_pages);
            else hipLaunchKernelGGL((k4_encode_page_rows<true, 32>), rows_grid, dim3(K4_THREADS), 0, st, a, n_pages);
        } else {
            if (B == 16) hipLaunchKernelGGL((k4_encode_page_rows<false, 16>), rows_grid, dim3(K4_THREADS), 0, st, a, n_pages);
            else hipLaunchKernelGGL((k4_encode_page_rows<false, 32>), rows_grid, dim3(K4_THREADS), 0, st, a, n_pages);
        }
        IQ_CHECK_LAUNCH("k4_encode_page_rows");
        return IQ_OK;
    }
    const dim3 grid((unsigned)n_pages, (unsigned)H), block(K4_THREADS);
    if (dtype == IQ_F16) {
        if (B == TILE_T) hipLaunchKernelGGL((k4_encode_tile<true, TILE_T / CH, true>), grid, block, 0, st, a);
        else hipLaunchKernelGGL((k4_encode_tile<true, 0, true>), grid, block, 0, st, a);
    } else {
        if (B == TILE_T) hipLaunchKernelGGL((k4_encode_tile<false, TILE_T / CH, true>), grid, block, 0, st, a);
        else hipLaunchKernelGGL((k4_encode_tile<false, 0, true>), grid, block, 0, st, a);
    }
    IQ_CHECK_LAUNCH("k4_encode_tile (pages)");
    return IQ_OK;
}
