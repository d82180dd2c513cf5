// Causal prefill attention over exact K/V on matrix cores (gfx950).
//
// Replaces the vLLM plugin's prefill call
//   flash_attn_varlen_func(q, k, v, out, cu_seqlens_q=cu, cu_seqlens_k=cu,
//                          max_seqlen_q=n, max_seqlen_k=n, causal=True, softmax_scale)
// (extensions/vllm/src/inquant_vllm/backend.py:139-144): every query attends to
// the keys at or before its position in its own sequence, in the K/V dtype
// with fp32 logits, softmax and accumulation.  Layout is vLLM's token-major
// [tokens, heads, 128] with runtime (token, head) strides; sequences are
// delimited by cu_seqlens.
//
// One workgroup = 128 queries of one query head: four wavefronts of 32
// queries, one per SIMD, so the two wavefronts that share a SIMD belong to
// different workgroups and overlap each other's matrix products with their
// softmax.  Keys are the rows of S^T = K Q^T on v_mfma_f32_32x32x16 (queries
// as columns): lane (query l % 32, half l / 32) holds 16 keys of its query per
// 32-key block, so the row maximum is an in-lane maximum and one permlane32
// swap, and the softmax weights land in the lanes and k-slots of the B
// operand of O^T = V^T P^T (k-slot 8 h + i of a 16-key chunk c is key
// 16 c + 4 h + i % 4 + 8 (i / 4)), so P needs no transpose.  Per 32 queries a
// key byte read from LDS feeds twice the products of 16-query wavefronts on
// 16x16x32 (0.92 -> 0.75 ms for the 8K causal Qwen2.5-7B prefill; earlier
// forms: 2.16 ms with four wavefronts of 16, 1.13 ms with eight and register
// double buffering, two 16-query subtiles per wavefront 1.33 ms).  Key tiles
// of 64 stream global -> LDS by direct loads (no registers) into two LDS
// stages of row-major K and V with XOR-swizzled 16-byte chunks; the V
// operand of O^T = V^T P^T comes out of LDS already transposed
// (ds_read_b64_tr_b16); one barrier per tile.  Masks only on the diagonal
// and last tiles; query tiles longest-first, spread evenly over the XCDs.
// 184 VGPRs: two wavefronts per SIMD.
#include "decode_common.h"

namespace {

constexpr int D = 128;
constexpr int NW = 4;               // wavefronts per workgroup
constexpr int NT = 64 * NW;         // threads per workgroup
constexpr int QW = 32;              // queries per wavefront
constexpr int QT = QW * NW;         // queries per workgroup
constexpr int KT = 64;              // keys per tile

typedef __attribute__((ext_vector_type(16))) float f32x16;

struct PrefillArgs {
    const uint16_t *q, *k, *v;
    void *out;
    int64_t q_st, q_sh, k_st, k_sh, v_st, v_sh, o_st, o_sh;   // element strides (token, head)
    const int32_t *cu;                                        // [n_seq + 1] token offsets
    int tiles, span, share, n_seq, Hq;                        // query tiles per sequence, places per group, an XCD's items of one, sequences, query heads
    int G;
    float c_log2;                                             // softmax scale * log2(e)
    int odt;
    int vec_out;                                              // output rows aligned for 4-channel stores
};

// two stages: one is computed while the next tile lands in the other.  Rows
// of 128 channels (256 bytes); the 16-byte chunk c of K row r sits at chunk
// slot c ^ (r % 16) and that of V row r at slot c ^ 4 (r % 4), so that the
// operand reads below hit 64 distinct banks per 16 (K) or 32 (V) lanes.
struct __attribute__((aligned(16))) PrefillSmem {
    uint16_t k[2][KT * D];
    uint16_t v[2][KT * D];
};
static_assert(2 * sizeof(PrefillSmem) <= 160 * 1024, "two workgroups per compute unit");

// ds_read_b64_tr_b16: within each group of 16 lanes, lane i receives element
// i % 4 of the 4 halves that lanes i / 4, i / 4 + 4, i / 4 + 8 and i / 4 + 12
// address (in that order).  When lane s reads key K0 + s / 4, channels
// c0 + 4 (s % 4) .. + 3, lane i receives channel c0 + i of keys K0 .. K0 + 3.
typedef short gv16x4 __attribute__((__vector_size__(4 * sizeof(short))));
__device__ __forceinline__ u32x2 tr_read(const uint16_t *p)
{
    const gv16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (__attribute__((address_space(3))) gv16x4 *)(__attribute__((address_space(3))) uint16_t *)p);
    return __builtin_bit_cast(u32x2, v);
}

// 32x32x16 product: lane l holds A[l % 32][8 (l / 32) .. + 7], B[8 (l / 32) .. + 7][l % 32]
// and C[8 (i / 4) + 4 (l / 32) + i % 4][l % 32] in register i
template <bool F16>
__device__ __forceinline__ f32x16 mma3232(u32x4 a, u32x4 b, f32x16 c)
{
    if constexpr (F16)
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c,
                                                      0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b),
                                                       c, 0, 0, 0);
}

// reductions over the lane pair l, l ^ 32 (one query's two halves)
__device__ __forceinline__ float pair_max(float v)
{
    const auto h = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(h[0]), __uint_as_float(h[1]));
}

__device__ __forceinline__ float pair_sum(float v)
{
    const auto h = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(h[0]) + __uint_as_float(h[1]);
}

template <bool F16>
__global__ __launch_bounds__(NT, 2) void prefill_attn(PrefillArgs a)
{
    __shared__ PrefillSmem sm;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int c32 = lane & 31, h32 = lane >> 5;
    // Workgroup i runs on XCD i % 8 (the dispatcher deals workgroups
    // round-robin over the eight XCDs).  An item is a (query tile, sequence,
    // query head); its cost grows with the tile's place in its sequence alone.
    // Tiles go from the last places to the first, over all sequences, so the
    // longest items start first and the last to run are short; of each group
    // of `span` places an XCD takes the same share of neighbouring heads in
    // every sequence (span Hq / 8 items), so the work of the XCDs is even and
    // an XCD's resident workgroups read the K/V of a KV head at about the same
    // time, out of its own L2.  8K causal, 28 query heads, eager: 519 us (927
    // TFLOP/s) with a contiguous range of (head, tile) items per XCD, where
    // four of the XCDs had 15% more work than the others and ended on long
    // tiles, 463 (1039) with these; seven prompts of up to 4.1K tokens, 32
    // heads: 293 and 281.  span = 0 is that contiguous range, a sequence after
    // the other (blockIdx.y).
    const int xcd = (int)(blockIdx.x & 7), j = (int)(blockIdx.x >> 3);
    int seq, hq, place;
    if (a.span == 0) {
        const int item = xcd * a.share + j;
        if (item >= a.tiles * a.Hq) return;      // the slice's padding
        seq = blockIdx.y;
        hq = item / a.tiles;
        place = a.tiles - 1 - (item - hq * a.tiles);
    } else {
        const int per = a.n_seq * a.share, group = j / per, rest = j - group * per;
        seq = rest / a.share;
        const int at = xcd * a.share + rest - seq * a.share;
        hq = at / a.span;
        place = a.tiles - 1 - (group * a.span + at - hq * a.span);
        if (place < 0) return;                   // the last group's padding
    }
    const int h = hq / a.G;
    const int start = a.cu[seq], len = a.cu[seq + 1] - start;
    const int q0 = place * QT;
    if (q0 >= len) return;                       // uniform: no barrier is skipped by part of the group
    const int qw = q0 + QW * wave;               // this wavefront's first query
    const int my_q = qw + c32;                   // the query of this lane's column
    u32x4 qb[8];                                 // B operand: Q[my_q][16 d + 8 h32 .. + 7]
    {
        const int qq = my_q < len ? my_q : len - 1;
        const uint16_t *qp = a.q + (int64_t)(start + qq) * a.q_st + (int64_t)hq * a.q_sh + 8 * h32;
#pragma unroll
        for (int d = 0; d < 8; ++d) qb[d] = ld16(qp + 16 * d);
    }
    const uint16_t *kbase = a.k + (int64_t)start * a.k_st + (int64_t)h * a.k_sh;
    const uint16_t *vbase = a.v + (int64_t)start * a.v_st + (int64_t)h * a.v_sh;
    float m_run = NEG_INF, l_run = 0.0f;         // l_run: this lane's share of the column sum
    f32x16 acc[4];                               // O^T rows 32 db .. 32 db + 31 (output channels)
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[db][i] = 0.0f;
    const int kend = q0 + QT < len ? q0 + QT : len;
    // Key tiles stream global -> LDS directly (no registers).  Each wavefront
    // moves 16 of the tile's 64 rows of K and of V, four rows (1 KB) per
    // direct load: lane l fills chunk slot l % 16 of row l / 16 with the
    // chunk that belongs there under the swizzle.  Rows past the sequence's
    // end repeat its last row (masked).  Offsets are 32-bit from the tile's
    // first row (token strides below 2^25 elements).
    const uint32_t lds_k = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint16_t *)&sm.k[0][0];
    const uint32_t lds_v = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint16_t *)&sm.v[0][0];
    auto dma_tile = [&](int k0, int st) {
        const int last = len - 1 - k0;
        const uint16_t *kt = kbase + (int64_t)k0 * a.k_st, *vt = vbase + (int64_t)k0 * a.v_st;
#pragma unroll
        for (int it = 0; it < 4; ++it) {
            const int r0 = 16 * wave + 4 * it;            // first row of this load (wave-uniform)
            const int r = r0 + (lane >> 4), p = lane & 15;
            const int rr = r < last ? r : last;
            const uint32_t ko = (uint32_t)((rr * a.k_st + 8 * (p ^ (r & 15))) * 2);
            const uint32_t vo = (uint32_t)((rr * a.v_st + 8 * (p ^ (4 * (r & 3)))) * 2);
            lds_load16(kt, ko, lds_k + (uint32_t)((st * KT + r0) * D * 2));
            lds_load16(vt, vo, lds_v + (uint32_t)((st * KT + r0) * D * 2));
        }
    };
    dma_tile(0, 0);
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
    int s = 0;
    for (int k0 = 0; k0 < kend; k0 += KT, s ^= 1) {
        // stage s ^ 1 was last read before the previous barrier
        if (k0 + KT < kend) dma_tile(k0 + KT, s ^ 1);
        if (k0 <= qw + QW - 1) {                 // some key of this tile is visible to this wavefront (uniform)
            const uint16_t *sk = sm.k[s];
            const uint16_t *sv = sm.v[s];
            // S^T blocks kb: lane holds keys k0 + 32 kb + 8 (i / 4) + 4 h32 + i % 4 of column my_q;
            // the two blocks' products alternate, so neither waits for its own previous one
            f32x16 sc[2];
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                for (int i = 0; i < 16; ++i) sc[kb][i] = 0.0f;
#pragma unroll
            for (int d = 0; d < 8; ++d)
#pragma unroll
                for (int kb = 0; kb < 2; ++kb)
                    sc[kb] = mma3232<F16>(*(const u32x4 *)(sk + (32 * kb + c32) * D + 8 * ((2 * d + h32) ^ (c32 & 15))),
                                          qb[d], sc[kb]);
            // raw logits: the scale is positive, so the maximum commutes with it
            // and p = 2^(s c - m) takes one fma per logit.  Only a tile that
            // reaches past this wavefront's first query or the sequence's end
            // has keys to mask (wave-uniform).
            if (k0 + KT - 1 > qw || k0 + KT > len) {
#pragma unroll
                for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                    for (int i = 0; i < 16; ++i) {
                        const int key = k0 + 32 * kb + 8 * (i >> 2) + 4 * h32 + (i & 3);
                        if (!(key <= my_q && key < len)) sc[kb][i] = NEG_INF;
                    }
            }
            float cmax = NEG_INF;
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                for (int i = 0; i < 16; ++i) cmax = fmaxf(cmax, sc[kb][i]);
            cmax = pair_max(cmax) * a.c_log2;
            // The reference maximum moves only when the tile's exceeds it by
            // more than 2^8 (or on the first tile): the weights 2^(s c - m) then
            // stay below 256, exact in range for the 16-bit P operand and the
            // fp32 sums, and the output rescale is skipped on most tiles.
            const float m_new = cmax > m_run + 8.0f ? cmax : m_run;   // finite: key 0 is visible to every query
            const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
            float lsum = 0.0f;
            u32x4 pb[2][2];                          // B operand of the 16-key chunk (kb, c): registers 8 c .. 8 c + 7
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                for (int c = 0; c < 2; ++c)
#pragma unroll
                    for (int w = 0; w < 4; ++w) {
                        const float p0 = __builtin_amdgcn_exp2f(fmaf(sc[kb][8 * c + 2 * w], a.c_log2, -m_new));
                        const float p1 = __builtin_amdgcn_exp2f(fmaf(sc[kb][8 * c + 2 * w + 1], a.c_log2, -m_new));
                        lsum += p0;
                        lsum += p1;
                        pb[kb][c][w] = pack2<F16>(p0, p1);
                    }
            // the two lanes of a column share m, so their partial sums take
            // the same rescale and are added once, after the last tile
            l_run = fmaf(l_run, alpha, lsum);
            m_run = m_new;
            // alpha is exactly 1 wherever the maximum did not grow: when that
            // holds in every lane the rescale is the identity and is skipped
            if (__builtin_amdgcn_ballot_w64(alpha != 1.0f)) {
#pragma unroll
                for (int db = 0; db < 4; ++db) acc[db] *= alpha;
            }
            // A operand of chunk (kb, c): V^T row 32 db + c32, keys 32 kb + 16 c + 4 h32 + 0..3 and
            // + 8..11, as two transposed reads: lane s of a 16-lane group (g = the group's
            // half of the 32 rows) reads key K0 + s / 4, channels 32 db + 16 g + 4 (s % 4) .. + 3
            const int s16 = lane & 15, g = (lane >> 4) & 1;
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                for (int c = 0; c < 2; ++c)
#pragma unroll
                    for (int db = 0; db < 4; ++db) {
                        const int K0 = 32 * kb + 16 * c + 4 * h32 + (s16 >> 2);      // K0 % 4 == s16 / 4
                        const int cl = 4 * db + 2 * g + ((s16 & 3) >> 1);
                        const int sw = 4 * (s16 >> 2), half = 4 * (s16 & 1);
                        const u32x2 lo = tr_read(sv + K0 * D + 8 * (cl ^ sw) + half);
                        const u32x2 hi = tr_read(sv + (K0 + 8) * D + 8 * (cl ^ sw) + half);
                        acc[db] = mma3232<F16>(u32x4{lo[0], lo[1], hi[0], hi[1]}, pb[kb][c], acc[db]);
                    }
        }
        // this wavefront's direct loads of stage s ^ 1 have landed and its LDS
        // reads of stage s are done; after the barrier that holds for every
        // wavefront
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    }
    l_run = pair_sum(l_run);
    if (my_q < len) {
        const float inv = 1.0f / l_run;
        const int64_t o = (int64_t)(start + my_q) * a.o_st + (int64_t)hq * a.o_sh + 4 * h32;
        // four consecutive channels per register group: one 16- or 8-byte store
        // when the rows are aligned for it (vec_out), else element by element
        if (a.vec_out && a.odt == IQ_F32) {
#pragma unroll
            for (int db = 0; db < 4; ++db)
#pragma unroll
                for (int g = 0; g < 4; ++g)
                    *(f32x4 *)((float *)a.out + o + 32 * db + 8 * g) =
                        f32x4{acc[db][4 * g] * inv, acc[db][4 * g + 1] * inv, acc[db][4 * g + 2] * inv,
                              acc[db][4 * g + 3] * inv};
        } else if (a.vec_out && a.odt != IQ_F32) {
#pragma unroll
            for (int db = 0; db < 4; ++db)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const bool f16 = a.odt == IQ_F16;
                    const float v0 = acc[db][4 * g] * inv, v1 = acc[db][4 * g + 1] * inv;
                    const float v2 = acc[db][4 * g + 2] * inv, v3 = acc[db][4 * g + 3] * inv;
                    *(u32x2 *)((uint16_t *)a.out + o + 32 * db + 8 * g) =
                        f16 ? u32x2{pack2<true>(v0, v1), pack2<true>(v2, v3)}
                            : u32x2{pack2<false>(v0, v1), pack2<false>(v2, v3)};
                }
        } else {
#pragma unroll
            for (int db = 0; db < 4; ++db)
#pragma unroll
                for (int i = 0; i < 16; ++i)
                    iq_store_as(a.out, o + 32 * db + 8 * (i >> 2) + (i & 3), acc[db][i] * inv, a.odt);
        }
    }
}

}  // namespace

extern "C" int iq_prefill_attention_tokens(const void *q, const void *k, const void *v, int dtype, int64_t q_st,
                                    int64_t q_sh, int64_t k_st, int64_t k_sh, int64_t v_st, int64_t v_sh,
                                    const int32_t *cu_seqlens, int64_t n_seq, int64_t max_seqlen, int64_t tokens, int64_t Hq,
                                    int64_t H, int64_t head_dim, float scale, void *out, int64_t o_st,
                                    int64_t o_sh, int out_dtype, void *stream)
{
    IQ_CHECK_ARG(q && k && v && out && cu_seqlens, "iq_prefill_attention: null pointer");
    IQ_CHECK_ARG(dtype == IQ_BF16 || dtype == IQ_F16, "iq_prefill_attention: q/k/v must be bf16 or f16");
    IQ_CHECK_ARG(out_dtype >= IQ_F32 && out_dtype <= IQ_F16, "iq_prefill_attention: bad output dtype");
    IQ_CHECK_ARG(head_dim == D, "iq_prefill_attention: head_dim %lld (128 required)", (long long)head_dim);
    IQ_CHECK_ARG(H >= 1 && Hq >= 1 && Hq % H == 0 && Hq <= 65535, "iq_prefill_attention: heads %lld / %lld",
                 (long long)Hq, (long long)H);
    IQ_CHECK_ARG(n_seq >= 1 && n_seq <= 65535 && max_seqlen >= 1 && max_seqlen <= 0x7fffffffLL - QT,
                 "iq_prefill_attention: bad sequence count or length");
    IQ_CHECK_ARG(tokens >= 0 && tokens <= (int64_t(1) << 60), "iq_prefill_attention: bad token count");
    // a key tile's rows are addressed by 32-bit byte offsets from its first row
    IQ_CHECK_ARG(k_st >= 0 && v_st >= 0 && k_st < (1LL << 25) && v_st < (1LL << 25),
                 "iq_prefill_attention: token stride too large");
    // rows are read as 16-byte vectors
    const uintptr_t bases = (uintptr_t)q | (uintptr_t)k | (uintptr_t)v;
    IQ_CHECK_ARG(bases % 16 == 0 && (q_st | q_sh | k_st | k_sh | v_st | v_sh) % 8 == 0,
                 "iq_prefill_attention: q/k/v rows must be 16-byte aligned");
    // 4-channel output stores need every row start aligned to 4 elements' bytes
    const int64_t obytes = out_dtype == IQ_F32 ? 4 : 2;
    const int vec_out = (uintptr_t)out % (4 * obytes) == 0 && o_st % 4 == 0 && o_sh % 4 == 0;
    const int64_t tiles = (max_seqlen + QT - 1) / QT;
    // places per group: the least number for which the XCDs' shares are whole;
    // with several sequences a share is at least 4 items, so the 64 workgroups
    // resident on an XCD read the K/V of at most 16 of them (eight prompts of
    // up to 4.1K tokens, 8 heads over 8: 183 us with a contiguous range per
    // XCD, 210 with shares of one item, 162 with four; seven of 37-4100 tokens,
    // 32 heads over 8: 291, and 280 with four, 290 with eight).  Where a head's
    // K/V exceed the XCD's 4 MB L2 (8192 tokens) a sequence's items follow
    // each other: all its places at once if the heads divide among the XCDs,
    // else shares of 224 (sixteen prompts of 2K-30K tokens, 28 heads over 4:
    // 34.5 ms with a contiguous range, 36.5 with shares of 7, 34.4 with 224;
    // six of up to 12K: 3.07, 3.16 and 3.00)
    int64_t span = 1;
    while (span * Hq % 8) span *= 2;
    // Workgroups past their sequence's end leave at once, and as an XCD deals
    // its workgroups round-robin over its CUs, the others meet on a part of
    // them where they stand at a fixed stride.  So the groups are for batches
    // whose tokens are at least two fifths of what the bound allows (under
    // that: 8 heads over 8, 200 prompts of 129 tokens bound by 516, 66 us in
    // contiguous ranges and 209 in groups; eight prompts, one of 4096 tokens,
    // 81 and 105; above: 28 heads over 4, prompts of 300 to 4000 tokens, 203
    // and 174) and that have more places than a group (64 prompts of 1 token,
    // 14 heads: 12.4 us, and 15.8 padded to groups of 4).
    const int64_t least = n_seq == 1 ? 1 : max_seqlen <= 8192 ? 4 : 224;
    if (least == 224 && Hq % 8 == 0) span = tiles;
    while (span * Hq / 8 < least && span < tiles) span *= 2;
    const bool groups = span < tiles && 5 * tokens >= 2 * n_seq * max_seqlen;
    if (!groups) span = 0;
    const int64_t share = groups ? span * Hq / 8 : (tiles * Hq + 7) / 8;
    const int64_t per_seq = groups ? (tiles + span - 1) / span * share * 8 : share * 8;
    constexpr int64_t MOST = 0xffffffffLL / NT;          // workgroups of a launch (2^32 threads)
    IQ_CHECK_ARG(per_seq <= MOST, "iq_prefill_attention: too many query tiles");
    const int64_t most = groups ? MOST / per_seq : n_seq;
    for (int64_t s0 = 0; s0 < n_seq; s0 += most) {
        const int64_t n = n_seq - s0 < most ? n_seq - s0 : most;
        PrefillArgs a{(const uint16_t *)q, (const uint16_t *)k, (const uint16_t *)v, out, q_st, q_sh, k_st, k_sh,
                      v_st, v_sh, o_st, o_sh, cu_seqlens + s0, (int)tiles, (int)span, (int)share, (int)n, (int)Hq, (int)(Hq / H),
                      scale * 1.44269504088896341f, out_dtype, vec_out};
        const dim3 grid((unsigned)(groups ? per_seq * n : per_seq), groups ? 1u : (unsigned)n), block(NT);
        if (dtype == IQ_F16) hipLaunchKernelGGL(prefill_attn<true>, grid, block, 0, (hipStream_t)stream, a);
        else hipLaunchKernelGGL(prefill_attn<false>, grid, block, 0, (hipStream_t)stream, a);
    }
    IQ_CHECK_LAUNCH("prefill_attn");
    return IQ_OK;
}

extern "C" int iq_prefill_attention(const void *q, const void *k, const void *v, int dtype, int64_t q_st, int64_t q_sh,
                                    int64_t k_st, int64_t k_sh, int64_t v_st, int64_t v_sh, const int32_t *cu_seqlens,
                                    int64_t n_seq, int64_t max_seqlen, int64_t Hq, int64_t H, int64_t head_dim,
                                    float scale, void *out, int64_t o_st, int64_t o_sh, int out_dtype, void *stream)
{
    // one sequence is as long as its bound; of several nothing is known
    return iq_prefill_attention_tokens(q, k, v, dtype, q_st, q_sh, k_st, k_sh, v_st, v_sh, cu_seqlens, n_seq, max_seqlen,
                                       n_seq == 1 && max_seqlen > 0 ? max_seqlen : 0, Hq, H, head_dim, scale, out, o_st,
                                       o_sh, out_dtype, stream);
}
