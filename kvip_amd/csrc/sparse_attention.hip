// Sparse attention over the 2048 selected KV rows of each query row: the consumer of the
// LIFetch outputs (the sparse flash attention the reference's service runs on the hot
// cache, tests/operators/lifetch/support/correctness.py:261-339; row format
// workloads.py:493-515).
//
// A 656-byte row holds 512 fp8 e4m3 "nope" features, 64 bf16 rope features and four fp32
// scales (one per 128 nope features). key = [nope * scale, rope] (576 features), value =
// nope * scale (512). For query row r and head h:
//   out[r, h] = sum_j p_j value_j / sum_j p_j,  p_j = exp(s_j - max_j s_j),
//   s_j = scale * <q[r, h], key_j>  over the row's indices j >= 0.
//
// A workgroup takes (query row, set of one or two groups of 16 heads, split of the 2048 indices).
// It resolves its indices to cache rows once (block table), then streams them as four token
// streams of 32-token tiles, one wave per stream and head group. A wave keeps its group's query
// and the whole [16 heads, 512] accumulator in registers and exchanges nothing until the four
// streams' softmaxes are merged through LDS at the end; the waves of the two groups share the
// tiles of a stream (one barrier per tile and one per rope buffer; a single group has none).
//   - A tile stays as it is in the cache: direct-to-LDS loads put its 512 fp8 bytes per token into a
//     two-slot ring, tile k + 4 landing while tile k is computed. No dequantised copy is made.
//   - Logits: fp8 MFMA (16x16x128, one scale group per instruction) of the raw key bytes with the
//     query as two fp8 terms, which hold bf16's eight significant bits over 2^14, so no key byte is
//     converted; each scale group's dot products are summed on their own and added as
//     fma(group, scale, s) in fp32. A query whose features lie further apart (sa_wide) stays bf16 and
//     the key bytes are converted (exactly) for bf16 MFMA. The rope features are bf16 MFMA.
//   - Values: bf16 MFMA of the value bytes, converted as they are read (two features per
//     v_cvt_scalef32_pk_bf16_fp8 with scale 1, exact), with the probabilities times the group's
//     scale (fp32, then rounded to bf16). One rounding per product instead of one on either side.
//   - The logits are computed transposed (tokens as M, heads as N), so a lane holds one head's logits
//     of 8 tokens: the softmax takes two lane swaps per tile, and the probabilities are the value
//     product's B operand (features as M, heads as N) without leaving their registers, because
//     the token order along K is free as long as both operands share it. The value operand (8
//     tokens of one feature per lane) comes from the token-major tile by ds_read_b64_tr_b8, whose
//     lanes address the tokens in that order.
//   - The running maximum is rescaled lazily: only when a tile's maximum exceeds it by kSaMargin (the
//     probabilities are then at most e^8, well inside bf16 and fp32), which after a row's first
//     tiles is rare.
//
// What bounds it: 16 heads read each row once, ~5 TB/s of 128-byte lines, between ~6 us of start
// (indices, table, first tile) and ~7 us of merges; more heads are bound by issue and LDS reads
// (about 620 instructions per wave and tile). LDS (ring 128 KB, rope 16 KB, cache rows 8 KB,
// scales 4 KB) allows one workgroup per CU. Measured, 64 rows, against the version that
// dequantised tiles to bf16 in LDS and exchanged probabilities between waves: 16 heads of 16384
// hot slots 37.4 -> 30.7 us per call, 128 heads of 2048 slots 98.7 -> 72.3; 32 heads 47.1 -> 34.4,
// 64 heads 58.2 -> 45.4; one row of 16 heads 21.8 -> 12.8. Error against 64 bits on N(0, 1) rows:
// 1.1e-3 (1.9e-3 with both sides rounded). Looking the query over for far smaller features takes 0.3 us
// of a call; one that has them takes 14.9 us for one row, 30.5 for 64 rows of 16 heads and
// 78.6 of 128 (that version: 21.8, 35.5, 96.9; two terms alone: 12.5, 27.5, 68.1).
// A variant with groups of 32 heads per wave (32x32x16 MFMA, 256 accumulators) spilled (356 us at 128
// heads); scratch reloads wait for every load in flight, so the tile loop must not spill.
#include <type_traits>

#include "lds_async.h"

namespace kvip {
namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
typedef __attribute__((ext_vector_type(2))) float f32x2;
typedef int i32x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((ext_vector_type(2))) uint16_t u16x2;
// Output and workspace are float arrays of any alignment (the card takes 16-byte accesses at
// 4-byte addresses).
typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));
typedef float f32x2_any __attribute__((ext_vector_type(2), aligned(4)));

constexpr int kSaHeads = 16;                // heads per wave (MFMA N)
constexpr int kSaStreams = 4;               // token streams per workgroup
constexpr int kSaTile = 32;                 // tokens per tile (value MFMA K)
constexpr int kKeyDim = 576;                // 512 nope + 64 rope
constexpr int kValueDim = 512;
constexpr int kScaleGroups = 4;
constexpr int kGroupDim = kValueDim / kScaleGroups;  // nope features that share a scale
constexpr int kMaxSplits = 16;
constexpr int kWideMark = 256;              // in place of a query exponent: the query stays bf16
constexpr int kPartial = kValueDim + 2;     // floats per (row, head, split): output, max, sum
constexpr float kLog2e = 1.44269504088896341f;
constexpr float kSaMargin = 8.0f * kLog2e;  // lazy rescale: 8 in natural-log units

// LDS map (bytes): per stream two tile slots of nope bytes, one tile of rope, two tiles of
// scales [group][token]; the cache rows of the split's indices; per stream a tile's row addresses;
// the query's block exponents and second rope fragments (two waves per SIMD leave 256 registers,
// 128 of them accumulators).
constexpr int kNopeSlot = kSaTile * kValueDim;
constexpr int kRopeSlot = kSaTile * 128;
constexpr int kScaleSlot = kScaleGroups * kSaTile * 4;
constexpr int kLdsRope = kSaStreams * 2 * kNopeSlot;
constexpr int kLdsScale = kLdsRope + kSaStreams * kRopeSlot;
constexpr int kLdsRows = kLdsScale + kSaStreams * 2 * kScaleSlot;
constexpr int kLdsBase = kLdsRows + kTopK * 4;
constexpr int kLdsQuery = kLdsBase + kSaStreams * kSaTile * 8;  // query exponents, then a rope fragment per group
constexpr int kLdsBytes = kLdsQuery + 2 * kSaHeads * kScaleGroups * 4 + 2 * 1024;
static_assert(kLdsBytes <= 160 * 1024, "LDS of a CU");

// Head groups of 16 per workgroup, and workgroups per row before index splits.
__host__ __device__ inline int sa_group_set(int heads) { return heads > kSaHeads ? 2 : 1; }
__host__ __device__ inline int sa_sets(int heads) {
    const int per = kSaHeads * sa_group_set(heads);
    return (heads + per - 1) / per;
}

// Index splits per (row, head set): the count with the shortest estimated launch, in units of
// one tile per stream (about 1 us): rounds of 256 workgroups (one per CU), each of its tiles per
// stream plus about 3 for resolving the indices, the first tile's latency and the merge of the
// streams; 5 more for the merge launch when there are splits. Every split count timed at 24 shapes
// of 1 to 256 rows and 16 to 128 heads: the choice was the fastest at 23 and 3 % slower at the other
// (4 rows of 128 heads, 8 splits 21.2 us, 16 21.9). us with 1 / 2 / 4 / 8 / 16 splits: 1 row of 16
// heads 40.3 26.5 18.2 14.1 12.6, 64 rows 43.1 31.2 27.5 36.4 52.0, 128 rows 45.2 41.2 49.3 67.8 98.7,
// 192 rows 53.8 70.1 74.6 103 148; 32 rows of 128 heads 59.3 43.4 52.1 74.5 113, 64 rows 63.9 79.5 99.3
// 154 259.
__host__ __device__ inline int sa_splits(int rows, int heads) {
    const int64_t units = static_cast<int64_t>(rows) * sa_sets(heads);
    int best = 1;
    int64_t best_cost = 0;
    for (int s = 1; s <= kMaxSplits; s *= 2) {
        const int64_t cost = (units * s + 255) / 256 * (kTopK / (kSaTile * kSaStreams) / s + 3) + (s > 1 ? 5 : 0);
        if (s == 1 || cost < best_cost) {
            best = s;
            best_cost = cost;
        }
    }
    return best;
}

typedef __attribute__((address_space(3))) const f32x4* LdsF32x4;
typedef __attribute__((address_space(3))) i32x2* LdsI32x2;

// x, recomputed from here on: keeps the compiler from hoisting the dozens of addresses derived
// from a loop constant out of the tile loop, where they would not fit the registers.
KVIP_DEVICE int fresh(int x) {
    asm volatile("" : "+v"(x));
    return x;
}

KVIP_DEVICE uint32_t pack_bf16(float a, float b) {  // hardware round to nearest even
    const bf16x2 v = {static_cast<__bf16>(a), static_cast<__bf16>(b)};
    return __builtin_bit_cast(uint32_t, v);
}

// Eight fp8 e4m3 features as bf16 (exact).
KVIP_DEVICE bf16x8 fp8x8_to_bf16(int lo, int hi) {
    const v4i r = {
        __builtin_bit_cast(int, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 1.0f, false)),
        __builtin_bit_cast(int, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 1.0f, true)),
        __builtin_bit_cast(int, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 1.0f, false)),
        __builtin_bit_cast(int, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 1.0f, true))};
    return __builtin_bit_cast(bf16x8, r);
}

// Max / sum over lanes l, l ^ 16, l ^ 32, l ^ 48.
KVIP_DEVICE float rows4_max(float x) {
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
    const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
KVIP_DEVICE float rows4_sum(float x) {
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = __uint_as_float(a[0]) + __uint_as_float(a[1]);
    const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// Places of a token's 16-byte pieces in its 512-byte LDS row: piece j sits at place j ^ swz(token).
// Linear over XOR, and such that both a key read (16 consecutive lanes: one piece of 16 consecutive
// tokens) and a value read (two 16-lane blocks of a transpose load: one piece of the 8 tokens
// 4 kg .. + 3 and 16 + 4 kg .. + 3 for kg and kg + 1) touch every bank once.
KVIP_DEVICE constexpr int sa_swz(int t) { return (t & 7) | ((((t >> 3) ^ (t >> 4)) & 1) << 3); }

// Whether a query must stay bf16, by one head's scale group: `held` of its features lie within 2^13 of
// the largest one's power of two (2^14 where that is even), where the two fp8 terms are exact, and
// `tiny` nonzero ones lie below, where the terms are off by up to 2^-22 of the largest. With 32 held
// features beside each tiny one (so at most three of the 128 are) that error is lost. With fewer, a
// key that is zero at the large features would show it. An infinity or NaN (`top`, the largest biased
// exponent, is 255) has no terms. N(0, 1) queries have one tiny feature in about 60 groups and hardly
// ever four in one.
KVIP_DEVICE bool sa_wide(int top, int held, int tiny) { return top == 255 || 32 * tiny > held; }

// 16 tokens x 16 heads over 128 features: fp8 keys (scale 1) by fp8 query terms with block scale
// byte g of `scales`.
KVIP_DEVICE f32x4 sa_mma8(v8i a, v8i b, f32x4 c, int g, int scales) {
    switch (g) {  // a constant after unrolling: the byte select is an immediate
        case 0: return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, c, 0, 0, 0, 127, 0, scales);
        case 1: return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, c, 0, 0, 0, 127, 1, scales);
        case 2: return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, c, 0, 0, 0, 127, 2, scales);
        default: return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, c, 0, 0, 0, 127, 3, scales);
    }
}

// Barrier for LDS data: unlike __syncthreads it leaves the direct-to-LDS loads in flight.
KVIP_DEVICE void lds_sync() {
    asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" : : : "memory");
}

template <int G>
__global__ __launch_bounds__(kSaStreams * G * 64, 1) void sparse_attention_kernel(const KvipSparseAttnArgs p,
                                                                                  int splits) {
    constexpr int kWaves = kSaStreams * G;
    constexpr int kThreads = kWaves * 64;
    constexpr int kBlocks = kValueDim / 16;            // accumulator blocks of 16 features
    __shared__ __align__(16) uint8_t s_mem[kLdsBytes];
    int32_t* s_row = reinterpret_cast<int32_t*>(s_mem + kLdsRows);

    // XCD-aware order: the head sets of one (query row, split), which read the same KV rows, share
    // blockIdx % 8, so they run on one XCD, whose L2 then serves the rows to every set after the first
    // read; rows and splits are dealt over all XCDs.
    const int sets = sa_sets(p.heads);
    const int chunk = blockIdx.x / (8 * sets), within = blockIdx.x % (8 * sets);
    const int job = chunk * 8 + within % 8, hs = within / 8;
    const int r = job / splits, sp = job % splits;
    if (r >= p.rows) return;
    const int b = r / p.rows_per_request;
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int st = w & (kSaStreams - 1), gi = w / kSaStreams;  // stream, head group of the set
    const int n = lane & 15, kg = lane >> 4;
    const int h0 = (hs * G + gi) * kSaHeads;
    const bool live = h0 < p.heads;                    // uniform: a set's last group may hold no heads

    // Cache rows of the split's indices, resolved once through the block table (-1: none): all
    // index loads, then the query's, then all table loads, so that the latencies overlap.
    const int span = kTopK / splits;
    constexpr int kIt = kTopK / kThreads;
    const int* idx_row = p.indices + static_cast<size_t>(r) * kTopK + sp * span;
    const int* table = p.block_table + static_cast<size_t>(b) * p.max_blocks;
    const int capacity = p.max_blocks * kBlockTokens;
    int idx[kIt];
#pragma unroll
    for (int i = 0; i < kIt; ++i) idx[i] = idx_row[min(i * kThreads + tid, span - 1)];
    // Query of head h0 + n (heads past p.heads read another one's; their outputs are not written). The
    // streams share the work: wave st takes scale group st, the 32 features that the lane's key bytes of
    // that group are (pieces 8 st + kg and 8 st + 4 + kg), and rope piece 4 (st & 1) + kg.
    v4i qraw[4], qrope;
    {
        const uint16_t* q = p.query + (static_cast<size_t>(r) * p.heads + min(h0 + n, p.heads - 1)) * kKeyDim;
#pragma unroll
        for (int x = 0; x < 4; ++x) {
            qraw[x] = *reinterpret_cast<const v4i*>(q + st * 128 + (x >> 1) * 64 + kg * 16 + (x & 1) * 8);
        }
        qrope = *reinterpret_cast<const v4i*>(q + kValueDim + (st & 1) * 32 + kg * 8);
    }
    uint32_t err = 0;
    {
        int blk[kIt];
#pragma unroll
        for (int i = 0; i < kIt; ++i) blk[i] = table[min(max(idx[i], 0), capacity - 1) >> 7];
#pragma unroll
        for (int i = 0; i < kIt; ++i) {
            const bool ok = static_cast<unsigned>(blk[i]) < static_cast<unsigned>(p.num_blocks);
            const bool in = idx[i] >= 0 && idx[i] < capacity;
            err |= idx[i] >= capacity ? KVIP_STATUS_BAD_TOKEN : (in && !ok ? KVIP_STATUS_BAD_BLOCK : 0u);
            if (i * kThreads + tid < span) {
                s_row[i * kThreads + tid] = in && ok ? blk[i] * kBlockTokens + (idx[i] & 127) : -1;
            }
        }
    }
    f32x4 o[kBlocks];
#pragma unroll
    for (int t = 0; t < kBlocks; ++t) o[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m_run = -INFINITY;  // reference maximum of head n, log2 units
    float l_sum = 0.f;        // this lane's share of its probability sum
    const float scale2 = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(p.scale * kLog2e)));
    __syncthreads();

    uint8_t* ring = s_mem + st * 2 * kNopeSlot;
    uint8_t* rope = s_mem + kLdsRope + st * kRopeSlot;
    uint8_t* scales = s_mem + kLdsScale + st * 2 * kScaleSlot;
    int64_t* s_base = reinterpret_cast<int64_t*>(s_mem + kLdsBase) + st * kSaTile;
    const uint32_t ring_lds = lds_addr(ring), rope_lds = lds_addr(rope), scales_lds = lds_addr(scales);

    // Tokens of tile k that have a row (bit t: token t), and their row addresses to s_base (0: none; the
    // waves of a stream write the same values).
    auto describe = [&](int k) -> uint32_t {
        const int ln = fresh(lane);
        const int row = s_row[k * kSaTile + (ln & 31)];
        if (ln < kSaTile) {
            s_base[ln] = row < 0 ? 0
                                   : reinterpret_cast<int64_t>(p.kv_cache) +
                                         static_cast<int64_t>(row >> 7) * p.kv_block_stride +
                                         static_cast<int64_t>(row & 127) * p.row_stride;
        }
        return static_cast<uint32_t>(__ballot(row >= 0));
    };
    // This wave's share (1 / G) of the loads of the described tile's nope bytes and scales into
    // slot `slot`. LDS row t holds piece s ^ swz(t) at place s; scales sit as [group][token]. Tokens
    // without a row get zero bytes and zero scales (their probabilities are zero, and zero times a
    // stray NaN would not be).
    constexpr uint32_t kAll = 0xFFFFFFFFu;
    auto load_nope = [&](int slot, uint32_t have) {
        const int ln = fresh(lane);
        constexpr int kLoads = kSaTile / 2 / G;  // of tokens 2 v and 2 v + 1 each
        const int from = ((ln & 31) ^ sa_swz(ln >> 5) ^ (G == 2 ? sa_swz(16) * gi : 0)) * 16;
        const int v0 = gi * kLoads, g0 = gi * (2 / G);
        const int64_t base = s_base[ln & 31];  // scales: groups 2 v and 2 v + 1 per load
        const uint8_t* sc_src = reinterpret_cast<const uint8_t*>(base) + 640 + 8 * g0 + 4 * (ln >> 5);
        const uint32_t sc_dst = scales_lds + slot * kScaleSlot + g0 * 256, dst = ring_lds + slot * kNopeSlot + v0 * 1024;
        if (have == kAll) {
            int64_t row[kLoads];  // every address first: one LDS latency, not one per load
#pragma unroll
            for (int x = 0; x < kLoads; ++x) row[x] = s_base[2 * (v0 + x) + (ln >> 5)];
#pragma unroll
            for (int x = 0; x < kLoads; ++x) {
                dma16(reinterpret_cast<const uint8_t*>(row[x]) + (from ^ (sa_swz(2 * x) * 16)), dst + x * 1024);
            }
#pragma unroll
            for (int x = 0; x < 2 / G; ++x) dma4(sc_src + 8 * x, sc_dst + x * 256);
        } else {
#pragma unroll 1
            for (int x = 0; x < kLoads; ++x) {
                const int64_t row = s_base[2 * (v0 + x) + (ln >> 5)];
                if (row != 0) {
                    dma16(reinterpret_cast<const uint8_t*>(row) + (from ^ (sa_swz(2 * x) * 16)), dst + x * 1024);
                } else {
                    *(__attribute__((address_space(3))) v4i*)(dst + x * 1024 + ln * 16) = v4i{0, 0, 0, 0};
                }
            }
#pragma unroll 1
            for (int x = 0; x < 2 / G; ++x) {
                if (base != 0) dma4(sc_src + 8 * x, sc_dst + x * 256);
                else *(__attribute__((address_space(3))) float*)(sc_dst + x * 256 + ln * 4) = 0.f;
            }
        }
    };
    // And of its rope features: LDS row t (128 bytes) holds piece s ^ (t / 2 % 8) at place s. A token
    // without a row keeps stale bytes: its logits are replaced.
    auto load_rope = [&] {
        const int ln = fresh(lane);
        constexpr int kLoads = kSaTile / 8 / G;  // of tokens 8 v .. 8 v + 7 each
        int64_t row[kLoads];
#pragma unroll
        for (int x = 0; x < kLoads; ++x) row[x] = s_base[8 * (gi * kLoads + x) + (ln >> 3)];
#pragma unroll
        for (int x = 0; x < kLoads; ++x) {
            const int piece = (ln & 7) ^ (((4 * x) & 7) ^ (ln >> 4));
            if (row[x] != 0) {
                dma16(reinterpret_cast<const uint8_t*>(row[x]) + kValueDim + piece * 16,
                      rope_lds + (gi * kLoads + x) * 1024);
            }
        }
    };
    // Every load and LDS access of this wave is done, and (waves sharing a stream) of all waves.
    auto settle = [&](bool loads) {
        if (loads) asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" : : : "memory");
        else asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
        if constexpr (G > 1) {
            __builtin_amdgcn_s_barrier();
            asm volatile("" : : : "memory");
        }
    };

    const int tiles = span / kSaTile;  // a multiple of the streams
    uint32_t mask = describe(st);
    load_nope(0, mask);
    load_rope();
    report(p.status, err);

    // The query as two fp8 e4m3 terms, q = (hi + lo 2^-5) 2^e with one e per head and 128 features (the
    // block scales of the MFMA): hi takes the upper four of bf16's eight significant bits, lo the rest
    // (at most 2^3 where the largest feature is below 2^8, so 2^8 after its scale). That is exact
    // down to 2^-14 of the largest feature; with more features below it than sa_wide allows, the
    // whole workgroup's query stays bf16. Wave st converts group st; the terms go through LDS (the ring's second
    // slots, free until the first tile has landed) to the waves of the other streams.
    v4i* s_qf = reinterpret_cast<v4i*>(s_mem + kNopeSlot) + gi * 256;  // + stream * 2 slots: its group's terms
    int* s_qe = reinterpret_cast<int*>(s_mem + kLdsQuery);             // [group of heads][head][scale group]
    {
        // Two features to a register, sign bits set: their largest by magnitude.
        auto features = [&](int x) { return static_cast<uint32_t>(qraw[x >> 2][x & 3]) | 0x80008000u; };
        u16x2 largest = __builtin_bit_cast(u16x2, features(0));
#pragma unroll
        for (int x = 1; x < 16; ++x) largest = __builtin_elementwise_max(largest, __builtin_bit_cast(u16x2, features(x)));
        const int top = static_cast<int>(rows4_max(static_cast<float>((max(largest[0], largest[1]) & 0x7FFF) >> 7)));
        const int e = max(top, 13);                         // biased exponent of the largest
        const float mul = __int_as_float((261 - e) << 23);  // 2^(134 - e): the largest below 2^8
        // How many of the group's features are at least 2^(2 k) (pairs of exponents, so that four features'
        // high bytes share a register): with the sign bits set, a subtraction leaves the bit where the byte
        // is not below what is taken away, and borrows nothing across.
        auto at_least = [&](int k) {
            int count = 0;
#pragma unroll
            for (int x = 0; x < 16; x += 2) {
                const uint32_t high = __builtin_amdgcn_perm(features(x), features(x + 1), 0x07050301u);
                count += __popc((high - static_cast<uint32_t>(k) * 0x01010101u) & 0x80808080u);
            }
            return static_cast<int>(rows4_sum(static_cast<float>(count)));
        };
        const int held = at_least((max(e - 14, 1) + 1) >> 1);
        bool wide = sa_wide(top, held, kGroupDim - held);    // zeros taken for tiny ones
        if (__ballot(wide) != 0ull) wide = sa_wide(top, held, at_least(1) - held);
        v4i* dst = s_qf + st * (2 * kNopeSlot / 16) + lane;
#pragma unroll
        for (int half = 0; half < 2; ++half) {  // features of the lane's first, second piece
            v4i hi, lo;
#pragma unroll
            for (int x = 0; x < 4; ++x) {
                int h = 0, l = 0;
#pragma unroll
                for (int y = 0; y < 2; ++y) {
                    const uint32_t v = static_cast<uint32_t>(qraw[2 * half + (x >> 1)][(x & 1) * 2 + y]);
                    const float a = __uint_as_float(v << 16) * mul, c = __uint_as_float(v & 0xFFFF0000u) * mul;
                    h = y ? __builtin_amdgcn_cvt_pk_fp8_f32(a, c, h, true) : __builtin_amdgcn_cvt_pk_fp8_f32(a, c, h, false);
                    const f32x2 back = y ? __builtin_amdgcn_cvt_pk_f32_fp8(h, true) : __builtin_amdgcn_cvt_pk_f32_fp8(h, false);
                    const float ra = (a - back[0]) * 32.0f, rc = (c - back[1]) * 32.0f;
                    l = y ? __builtin_amdgcn_cvt_pk_fp8_f32(ra, rc, l, true) : __builtin_amdgcn_cvt_pk_fp8_f32(ra, rc, l, false);
                }
                hi[x] = h;
                lo[x] = l;
            }
            dst[half * 64] = hi;
            dst[(2 + half) * 64] = lo;
        }
        if (kg == 0) s_qe[(gi * kSaHeads + n) * kScaleGroups + st] = wide ? kWideMark : e - 7;
    }
    v4i* s_rope = reinterpret_cast<v4i*>(s_mem + kLdsQuery + 2 * kSaHeads * kScaleGroups * 4) + gi * 64;
    if (st == 0) s_qf[512 + lane] = qrope;  // past the terms of both head groups
    if (st == 1) s_rope[lane] = qrope;
    lds_sync();
    v8i qh[kScaleGroups], ql[kScaleGroups];
    int qscale = 0;  // byte g: E8M0 scale of group g's hi terms (lo: 5 less)
    const v4i* s_qe4 = reinterpret_cast<const v4i*>(s_qe);
    const v4i qe = s_qe4[gi * kSaHeads + n], qe_other = s_qe4[(G - 1 - gi) * kSaHeads + n];
    bool wide = false;
#pragma unroll
    for (int g = 0; g < kScaleGroups; ++g) {
        const v4i* src = s_qf + g * (2 * kNopeSlot / 16) + lane;
        const v4i a = src[0], c = src[64], d = src[128], f = src[192];
        qh[g] = v8i{a[0], a[1], a[2], a[3], c[0], c[1], c[2], c[3]};
        ql[g] = v8i{d[0], d[1], d[2], d[3], f[0], f[1], f[2], f[3]};
        wide |= qe[g] == kWideMark || qe_other[g] == kWideMark;
        qscale |= (qe[g] & 255) << (8 * g);
    }
    wide = __ballot(wide) != 0ull;  // the same in every wave: the copies of the tile loop hold barriers
    const int qscale_lo = qscale - 0x05050505;  // every byte is at least 6 (unless wide)
    if (wide) {  // the bf16 features of each group: the lane's first piece in qh, its second in ql
        const uint16_t* q = p.query + (static_cast<size_t>(r) * p.heads + min(h0 + n, p.heads - 1)) * kKeyDim + kg * 16;
#pragma unroll
        for (int g = 0; g < kScaleGroups; ++g) {
            const v4i* src = reinterpret_cast<const v4i*>(q + g * 128);
            const v4i a = src[0], c = src[1], d = src[8], f = src[9];
            qh[g] = v8i{a[0], a[1], a[2], a[3], c[0], c[1], c[2], c[3]};
            ql[g] = v8i{d[0], d[1], d[2], d[3], f[0], f[1], f[2], f[3]};
        }
        // Waited for here: the tile loop would wait for them each time round, and so for its own loads.
#pragma unroll
        for (int g = 0; g < kScaleGroups; ++g) asm volatile("" : "+v"(qh[g]), "+v"(ql[g]));
    }
    const bf16x8 q_rope = __builtin_bit_cast(bf16x8, s_qf[512 + lane]);
    lds_sync();  // the ring's second slots are free
    // The tiles of this wave's stream, in two copies: a branch within the loop spilled 76 registers.
    auto stream = [&](auto wide_query) {
        constexpr bool kWide = decltype(wide_query)::value;
        int slot = 0;
        for (int k = st; k < tiles; k += kSaStreams, slot ^= 1) {
            const bool more = k + kSaStreams < tiles;
            settle(true);  // the tile has landed; the other slot is free
            uint32_t next = 0;
            if (more) {
                next = describe(k + kSaStreams);
                load_nope(slot ^ 1, next);
            }
            // LDS addresses of this lane's reads, derived anew for each tile (held over the loop they
            // would cost registers that the accumulators need). Keys: piece 4 j + kg of token 16 u + n; the
            // XOR with 64 j moves between pieces. Values: block kg of a transpose load covers 16 features
            // (one piece) of the 8 tokens that lane group kg holds probabilities of: 4 kg + 0 .. 3 and
            // 16 + 4 kg + 0 .. 3.
            const int ln = fresh(lane), tn = ln & 15, tk = ln >> 4;
            const uint32_t ro = rope_lds + tn * 128 + ((tk ^ ((tn >> 1) & 7)) << 4);
            const uint32_t ko = ring_lds + slot * kNopeSlot + tn * kValueDim + ((tk ^ sa_swz(tn)) << 4);
            const int vt = 4 * tk + ((tn >> 1) & 3) + 16 * (tn >> 3);
            const uint32_t vo = ring_lds + slot * kNopeSlot + vt * kValueDim + (sa_swz(vt) << 4) + 8 * (ln & 1);
            const uint32_t sl = scales_lds + slot * kScaleSlot + 16 * tk;  // scales of tokens 4 kg .. + 3

            // Logits [tokens, heads], lane: tokens 16 u + 4 kg + i of head n. Rope first, whose buffer
            // then takes the next tile's rope.
            f32x4 sv[2];
            {
                const v4i q1 = *(LdsV4i)lds_addr(s_rope + ln);
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const v4i k0 = *(LdsV4i)(ro + u * 16 * 128), k1 = *(LdsV4i)((ro ^ 64) + u * 16 * 128);
                    sv[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, k0), q_rope,
                                                                    f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
                    sv[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, k1),
                                                                    __builtin_bit_cast(bf16x8, q1), sv[u], 0, 0, 0);
                }
            }
            settle(false);
            if (more) load_rope();
            if (live) {
                // One scale group of 16 tokens per step (i: token half i / 4, group i % 4), its key bytes read
                // one step ahead; the raw fp8 bytes are the A operand.
                auto key = [&](int i) {
                    const uint32_t at = ko ^ ((i & 3) * 128) ^ (sa_swz(16 * (i >> 2)) * 16);
                    const v4i x = *(LdsV4i)(at + (i >> 2) * 16 * kValueDim);
                    const v4i y = *(LdsV4i)((at ^ 64) + (i >> 2) * 16 * kValueDim);
                    return v8i{x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
                };
                auto logits = [&](auto&& dot) {
                    v8i kv[2] = {key(0), v8i{}};
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        const int u = i >> 2, g = i & 3;
                        const f32x4 s4 = *(LdsF32x4)(sl + (g * kSaTile + 16 * u) * 4);
                        if (i + 1 < 8) kv[(i + 1) & 1] = key(i + 1);
                        __builtin_amdgcn_sched_barrier(0);
                        const f32x4 part = dot(kv[i & 1], g);
#pragma unroll
                        for (int e = 0; e < 4; ++e) sv[u][e] = fmaf(part[e], s4[e], sv[u][e]);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                };
                if constexpr (!kWide) {
                    logits([&](v8i k, int g) {
                        const f32x4 part = sa_mma8(k, qh[g], f32x4{0.f, 0.f, 0.f, 0.f}, g, qscale);
                        return sa_mma8(k, ql[g], part, g, qscale_lo);
                    });
                } else {
                    logits([&](v8i k, int g) {
                        f32x4 part = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                        for (int x = 0; x < 4; ++x) {
                            const v8i& q = x < 2 ? qh[g] : ql[g];
                            const v4i qx = {q[4 * (x & 1)], q[4 * (x & 1) + 1], q[4 * (x & 1) + 2], q[4 * (x & 1) + 3]};
                            part = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fp8x8_to_bf16(k[2 * x], k[2 * x + 1]),
                                                                           __builtin_bit_cast(bf16x8, qx), part, 0, 0, 0);
                        }
                        return part;
                    });
                }
                // Softmax: pr = 2^(logit - m), the logits of tokens without a row at -inf.
                float pr[8];
                float mx = -INFINITY;
#pragma unroll
                for (int i = 0; i < 8; ++i) pr[i] = sv[i >> 2][i & 3] * scale2;
                if (mask != kAll) {
                    const uint32_t mine = mask >> (4 * tk);
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        if (!((mine >> (16 * (i >> 2) + (i & 3))) & 1u)) pr[i] = -INFINITY;
                    }
                }
#pragma unroll
                for (int i = 0; i < 8; ++i) mx = fmaxf(mx, pr[i]);
                mx = rows4_max(mx);
                const bool raise = mx > m_run + kSaMargin;  // also the first finite maximum
                if (__ballot(raise) != 0ull) {
                    const float m_new = raise ? mx : m_run;
                    const float alpha = m_run == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_run - m_new);
                    const float a = raise ? alpha : 1.f;
                    l_sum *= a;
#pragma unroll
                    for (int t = 0; t < kBlocks; ++t) o[t] *= a;
                    m_run = m_new;
                }
                const float bias = m_run == -INFINITY ? 0.f : -m_run;
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    pr[i] = __builtin_amdgcn_exp2f(pr[i] + bias);
                    l_sum += pr[i];
                }
                // Value product [features, heads]: the transpose loads of kAhead blocks ahead of the MFMAs
                // of the kAhead before them; each scale group's probabilities as its first block comes up.
                constexpr int kAhead = G == 1 ? 4 : 2;  // two waves per SIMD have no registers for more
                auto value = [&](int t) {
                    return __builtin_amdgcn_ds_read_tr8_b64_v2i32((LdsI32x2)((vo ^ ((t & 15) * 16)) + (t & 16) * 16));
                };
                i32x2 raw[2][kAhead];
#pragma unroll
                for (int i = 0; i < kAhead; ++i) raw[0][i] = value(i);
                bf16x8 pb;
#pragma unroll
                for (int t = 0; t < kBlocks; t += kAhead) {
                    const int now = t / kAhead & 1;
                    if (t + kAhead < kBlocks) {
#pragma unroll
                        for (int i = 0; i < kAhead; ++i) raw[now ^ 1][i] = value(t + kAhead + i);
                    }
                    if (t % 8 == 0) {
                        v4i packed;
#pragma unroll
                        for (int u = 0; u < 2; ++u) {
                            const f32x4 s4 = *(LdsF32x4)(sl + (t / 8 * kSaTile + 16 * u) * 4);
                            packed[2 * u] = static_cast<int>(pack_bf16(pr[4 * u] * s4[0], pr[4 * u + 1] * s4[1]));
                            packed[2 * u + 1] = static_cast<int>(pack_bf16(pr[4 * u + 2] * s4[2], pr[4 * u + 3] * s4[3]));
                        }
                        pb = __builtin_bit_cast(bf16x8, packed);
                    }
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int i = 0; i < kAhead; ++i) {
                        const i32x2 x = raw[now][i];
                        o[t + i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fp8x8_to_bf16(x[0], x[1]), pb, o[t + i], 0, 0, 0);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            mask = next;
        }
    };
    if (!wide) stream(std::false_type{});
    else stream(std::true_type{});

    // Merge of the streams: with the maximum M over them, out = sum_w 2^(m_w - M) o_w / l and
    // l = sum_w 2^(m_w - M) l_w, 512 / G features at a time through LDS.
    const int le = fresh(lane), mn = le & 15, mk = le >> 4;  // n and kg, not held over the tiles
    const float l_all = rows4_sum(l_sum);
    float* s_m = reinterpret_cast<float*>(s_mem + kLdsScale);  // [wave][head], then the sums
    float* s_f = s_m + 2 * kWaves * kSaHeads;                  // [wave][head]: factor of the wave's output
    float* buf = reinterpret_cast<float*>(s_mem);              // [wave][head][features]
    constexpr int kPitch = kValueDim / G + 4;
    static_assert(kWaves * kSaHeads * kPitch * 4 <= kLdsScale, "merge buffer inside ring and rope");
    __syncthreads();  // every wave is done with its ring, rope and scales
    if (mk == 0) {
        s_m[w * kSaHeads + mn] = m_run;
        s_m[(kWaves + w) * kSaHeads + mn] = l_all;
    }
#pragma unroll
    for (int g = 0; g < G; ++g) {
        if (g > 0) __syncthreads();  // the features before have been read
#pragma unroll
        for (int t = 0; t < kBlocks / G; ++t) {
            *reinterpret_cast<f32x4*>(buf + (w * kSaHeads + mn) * kPitch + t * 16 + 4 * mk) = o[g * (kBlocks / G) + t];
        }
        __syncthreads();
        if (g == 0) {
            if (tid < kSaHeads * G) {
                const int w0 = tid / kSaHeads * kSaStreams, hn = tid % kSaHeads;  // the head's waves
                float m = -INFINITY;
#pragma unroll
                for (int v = 0; v < kSaStreams; ++v) m = fmaxf(m, s_m[(w0 + v) * kSaHeads + hn]);
                float l = 0.f, f[kSaStreams];
#pragma unroll
                for (int v = 0; v < kSaStreams; ++v) {
                    f[v] = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(s_m[(w0 + v) * kSaHeads + hn] - m);
                    l += f[v] * s_m[(kWaves + w0 + v) * kSaHeads + hn];
                }
                const int h = hs * G * kSaHeads + tid;
                float inv = 1.f;
                if (splits == 1) {
                    inv = l > 0.f ? 1.f / l : 0.f;
                } else if (h < p.heads) {
                    float* ml = p.workspace + static_cast<size_t>(p.rows) * p.heads * splits * kValueDim +
                                ((static_cast<size_t>(r) * p.heads + h) * splits + sp) * 2;
                    ml[0] = m;
                    ml[1] = l;
                }
#pragma unroll
                for (int v = 0; v < kSaStreams; ++v) s_f[(w0 + v) * kSaHeads + hn] = f[v] * inv;
            }
            __syncthreads();
        }
        // Thread: features f .. + 4 of every kStep-th head; consecutive threads on consecutive features.
        constexpr int kPerHead = kValueDim / G / 4;
        constexpr int kStep = kThreads / kPerHead;
        const int f = tid % kPerHead * 4;
#pragma unroll
        for (int hl = tid / kPerHead; hl < kSaHeads * G; hl += kStep) {
            const int w0 = hl / kSaHeads * kSaStreams;
            f32x4 v = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int x = 0; x < kSaStreams; ++x) {
                const int at = (w0 + x) * kSaHeads + hl % kSaHeads;
                v += s_f[at] * *reinterpret_cast<const f32x4*>(buf + at * kPitch + f);
            }
            const int h = hs * G * kSaHeads + hl;
            if (h < p.heads) {
                const size_t rh = static_cast<size_t>(r) * p.heads + h;
                float* out = splits == 1 ? p.output + rh * kValueDim : p.workspace + (rh * splits + sp) * kValueDim;
                *reinterpret_cast<f32x4_any*>(out + g * (kValueDim / G) + f) = v;
            }
        }
    }
}

// Merge of the splits: 128 threads per (row, head), four features each; every load is issued before the
// first is used (one memory latency, whatever the split count).
template <int SPLITS>
__global__ __launch_bounds__(256) void sparse_attention_merge_kernel(const KvipSparseAttnArgs p) {
    const int64_t rh = static_cast<int64_t>(blockIdx.x) * 2 + (threadIdx.x >> 7);
    if (rh >= static_cast<int64_t>(p.rows) * p.heads) return;
    const int f = (threadIdx.x & 127) * 4;
    const float* ws = p.workspace + rh * SPLITS * kValueDim + f;
    const float* ml = p.workspace + static_cast<size_t>(p.rows) * p.heads * SPLITS * kValueDim + rh * SPLITS * 2;
    f32x4 part[SPLITS];
    f32x2 sums[SPLITS];
#pragma unroll
    for (int s = 0; s < SPLITS; ++s) sums[s] = *reinterpret_cast<const f32x2_any*>(ml + 2 * s);
#pragma unroll
    for (int s = 0; s < SPLITS; ++s) part[s] = *reinterpret_cast<const f32x4_any*>(ws + s * kValueDim);
    float m = -INFINITY;
#pragma unroll
    for (int s = 0; s < SPLITS; ++s) m = fmaxf(m, sums[s][0]);
    float l = 0.f;
    f32x4 v = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < SPLITS; ++s) {
        const float wgt = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(sums[s][0] - m);
        l += wgt * sums[s][1];
        v += wgt * part[s];
    }
    *reinterpret_cast<f32x4_any*>(p.output + rh * kValueDim + f) = v * (l > 0.f ? 1.f / l : 0.f);
}

template <int SPLITS>
void launch_merge(const KvipSparseAttnArgs& a, hipStream_t stream) {
    const int64_t pairs = (static_cast<int64_t>(a.rows) * a.heads + 1) / 2;
    hipLaunchKernelGGL(sparse_attention_merge_kernel<SPLITS>, dim3(static_cast<unsigned>(pairs)), dim3(256), 0, stream, a);
}

}  // namespace

uint64_t sparse_attention_workspace_bytes(int rows, int heads) {
    if (rows < 1 || heads < 1) return 0;
    const int splits = sa_splits(rows, heads);
    return splits > 1 ? static_cast<uint64_t>(rows) * heads * splits * kPartial * sizeof(float) : 0;
}

uint32_t validate_sparse_attention(const KvipSparseAttnArgs* a) {
    if (a == nullptr) return KVIP_ERR_INVALID;
    const bool ok = a->query && a->kv_cache && a->block_table && a->indices && a->output && a->rows >= 1 &&
                    a->rows_per_request >= 1 && a->rows % a->rows_per_request == 0 && a->heads >= 1 &&
                    a->heads <= 128 && a->max_blocks >= 1 && a->max_blocks <= (1 << 24) / kBlockTokens &&
                    a->num_blocks >= 1 && a->num_blocks < (1 << 24) && a->row_stride >= KVIP_KV_ROW_BYTES &&
                    a->row_stride % 16 == 0 &&
                    a->kv_block_stride % 16 == 0 &&
                    a->kv_block_stride >= static_cast<int64_t>(kBlockTokens) * a->row_stride &&
                    (reinterpret_cast<uintptr_t>(a->kv_cache) & 15u) == 0 &&
                    (reinterpret_cast<uintptr_t>(a->query) & 15u) == 0 && a->rows <= 65535 * 64 &&
                    (a->workspace != nullptr || sparse_attention_workspace_bytes(a->rows, a->heads) == 0);
    return ok ? KVIP_OK : KVIP_ERR_INVALID;
}

}  // namespace kvip

extern "C" uint32_t kvip_hip_sparse_attention(const KvipSparseAttnArgs* args, void* stream) {
    const uint32_t rc = kvip::validate_sparse_attention(args);
    if (rc != KVIP_OK) return rc;
    const int sets = kvip::sa_sets(args->heads);
    const int splits = kvip::sa_splits(args->rows, args->heads);
    const hipStream_t s = static_cast<hipStream_t>(stream);
    const dim3 grid((args->rows * splits + 7) / 8 * 8 * sets);
    if (args->heads > 16) {
        hipLaunchKernelGGL(kvip::sparse_attention_kernel<2>, grid, dim3(512), 0, s, *args, splits);
    } else {
        hipLaunchKernelGGL(kvip::sparse_attention_kernel<1>, grid, dim3(256), 0, s, *args, splits);
    }
    switch (splits) {
        case 2: kvip::launch_merge<2>(*args, s); break;
        case 4: kvip::launch_merge<4>(*args, s); break;
        case 8: kvip::launch_merge<8>(*args, s); break;
        case 16: kvip::launch_merge<16>(*args, s); break;
        default: break;
    }
    return static_cast<uint32_t>(hipGetLastError());
}

extern "C" uint64_t kvip_hip_sparse_attention_workspace_bytes(int32_t rows, int32_t heads) {
    return kvip::sparse_attention_workspace_bytes(rows, heads);
}
