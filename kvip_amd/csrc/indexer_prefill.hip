// Prefill (and mixed-batch) lightning-indexer scoring on gfx950 MFMA: packed query rows of
// several sequences against their paged index-K under a right-down causal mask, fp8 e4m3
// or bf16 Q/K.
//
// Work unit = (query block, context segment): 8 consecutive query rows of one sequence
// against up to 4096 key positions (one unit per workgroup, or a bounded grid whose workgroups
// stride over the units, kvip_hip_indexer_prefill_grid). fp8: 4 waves own 2 query rows
// each; bf16 (Q fragments twice as large): 8 waves own one row each. A wave keeps its rows'
// Q fragments and per-lane head weights (w'_h = w_h * qscale_h for the 32 heads a lane
// reduces) in registers. The segment streams through LDS in chunks of 256 tokens (fp8 32 KiB,
// bf16 64 KiB), double buffered: every wave issues direct-to-LDS 16-byte loads
// (global_load_lds_dwordx4) for its share of the next chunk, with the XOR swizzle applied
// on the global side so that the fragment reads (lane n of a 32-token tile reads row n)
// hit distinct bank groups. Each chunk tile (32 tokens) is one B fragment set read once
// from LDS and reused by the wave's rows x 2 head tiles: 2 K slices each of
// v_mfma_scale_f32_32x32x64_f8f6f4 (fp8) or 8 of v_mfma_f32_32x32x16_bf16 (bf16). The
// epilogue is the decode kernel's: ReLU, head weights, head reduction, key scale, bf16
// half-away rounding, sortable key; keys go through a per-wave LDS strip to coalesced
// stores, and a per-workgroup 256-bin histogram of the key high byte (two 16-bit counters
// per word: bins b and b + 128; bf16, whose 64 lanes add to one row, keeps four copies per
// row) is added to the row histograms at the end. fp8 runs two workgroups per CU, bf16 one
// (two waves per SIMD either way).
//
// Bound: matrix cores and VALU together, under the card's power limit. A 32-token tile of one fp8
// row with 64 heads is 256 cycles of MFMA and 64 VALU operations (ReLU and weight FMA). A loop of
// just these takes 190-197 ns per tile with two waves per SIMD and 186 ns with three or four; its
// MFMAs alone take 149 ns, at the 1.7 GHz that they leave on random data. This kernel takes about
// 235 ns, with its staging, LDS reads, the finish of each tile and the histogram. The order of MFMA
// and VALU operations within a tile moves it by less than 3%; one fp8 row per wave at four waves
// per SIMD spills and is twice as slow. What could be trimmed is around the loop: both rows (bf16:
// both tiles) are joined by one lane swap, the key comes straight from the rounded 32-bit pattern,
// the next tile's fragments are requested under the epilogue, and bf16 chunks are as long as fp8
// ones, with half the barriers they had at 128 tokens. With 4096 keys per item on either side, scoring
// 4096 rows causally against 65536 keys went from 1917 to 1881 us in fp8 and 3640 to 3485 in bf16, 2048
// rows against 16384 keys from 251 to 246 and 458 to 440.
//
// Reference: the native prefill LI (torch_npu.npu_quant_lightning_indexer, TND layout,
// sparse_mode 3) that the vLLM selector runs for prefill rows (python/kvip/adapters/vllm/
// selector.py:126-154); the score formula is the decode one (op_kernel/indexer/
// indexer_cube.h:161-322, indexer_score.h:384-426, score_common.h:66-97).
#include <algorithm>

#include "indexer_tile.h"
#include "lds_async.h"

namespace kvip {
namespace {

constexpr int kPfBlockRows = 8;                             // query rows per workgroup
// Waves per workgroup and query rows per wave: fp8 runs 4 waves of 2 rows (one row per lane
// half at the finish) and two workgroups per CU; bf16 Q fragments are twice as large, so it
// runs 8 waves of 1 row, which keeps a wave under 256 registers and gives two waves per SIMD
// in the one workgroup per CU.
template <int ELEM>
struct PfShape {
    static constexpr int kWaves = ELEM == 1 ? 4 : 8;
    static constexpr int kRows = kPfBlockRows / kWaves;
    static constexpr int kThreads = kWaves * 64;
};
constexpr int kPfChunk = 256;                               // key positions staged at a time
constexpr int kPfSegment = 4096;                            // most key positions per work item
constexpr int kPfPages = kPfSegment / kBlockTokens;         // 32
constexpr int kPfMaxSeq = KVIP_PREFILL_MAX_SEQUENCES;
// LDS piece swizzle of a staged K row of 8 (fp8) or 16 (bf16) 16-byte pieces: piece j of
// row r sits at slot j ^ (r & 15) (j ^ (r & 7) for 8 pieces). A fragment read (lane n
// reads piece j of row n) then touches distinct 16-byte slots in every group of 8 (16)
// consecutive lanes, i.e. every bank once per phase.
template <int ELEM>
KVIP_DEVICE int pf_swizzle(int row) { return row & (8 * ELEM - 1); }

template <bool W_BF16>
KVIP_DEVICE float pf_weight(const KvipPrefillArgs& p, size_t idx) {
    float w;
    if constexpr (W_BF16) {
        w = bf16_to_float(static_cast<const uint16_t*>(p.weights)[idx]);
    } else {
        w = static_cast<const float*>(p.weights)[idx];
    }
    return w * (p.query_scale != nullptr ? p.query_scale[idx] : 1.0f);
}

// Counts a key's high byte in a row histogram of two 16-bit counters per word: bins b and
// b ^ 128 share a word (the populated bins of a row are adjacent and would otherwise serialise
// on one word's atomics).
KVIP_DEVICE void pf_count(uint32_t hist, uint32_t key) {
    __hip_atomic_fetch_add((LdsU32)(hist + ((key >> 6) & 0x1FCu)), key & 0x8000u ? 0x10000u : 1u, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_WORKGROUP);
}

template <int ELEM, int HEADS, bool W_BF16>
__global__ __launch_bounds__(PfShape<ELEM>::kThreads, 3 - ELEM) void indexer_prefill_kernel(const KvipPrefillArgs p, const int segment) {
    constexpr int kPfWaves = PfShape<ELEM>::kWaves;
    constexpr int kPfRowsPerWave = PfShape<ELEM>::kRows;
    constexpr int kPfThreads = PfShape<ELEM>::kThreads;
    constexpr int kPfChunkBytes = kPfChunk * kIndexDim * ELEM;
    constexpr int MT = HEADS / 32;
    constexpr int NV = Mma<ELEM>::NV;              // 16-byte pieces of a half row per lane
    constexpr int STEPS = Mma<ELEM>::STEPS;        // MFMAs per 128-dim contraction
    constexpr int kRowBytes = kIndexDim * ELEM;
    constexpr int kPieces = kRowBytes / 16;        // 16-byte pieces per K row
    constexpr int kPfTiles = kPfChunk / 32;
    constexpr int kChunkPages = kPfChunk / kBlockTokens;  // pages per chunk (2)
    constexpr int kRowsPerLoad = 64 / kPieces;     // K rows one 64-lane 16-byte load fills
    static_assert(kPfRowsPerWave == 1 || kPfRowsPerWave == 2, "the finish maps row q to lane half q");
    constexpr int kStageLoads = (kPfChunk / kPfWaves) / kRowsPerLoad;  // staging loads per wave and chunk
    static_assert(kStageLoads * kRowsPerLoad * kPfWaves == kPfChunk, "whole staging loads");
    __shared__ __align__(16) uint8_t s_k[2][kPfChunkBytes];
    __shared__ __align__(16) float s_ks[2][kPfChunk];
    __shared__ __align__(16) uint16_t s_keys[kPfWaves][kPfRowsPerWave][kPfChunk];
    // Row histograms: bins b (low half) and b + 128 (high half) of a word. bf16 (one row per
    // wave, all 64 lanes adding to one row) keeps kHistCopies copies per row, lane l adding to
    // copy l % kHistCopies, so that lanes whose keys share a bin do not serialise on one word;
    // the copies sit 144 words apart, i.e. 16 banks apart.
    constexpr int kHistCopies = kPfRowsPerWave == 1 ? 4 : 1;
    constexpr int kHistStride = kHistCopies > 1 ? 144 : 128;
    constexpr int kHistWords = kHistCopies * kHistStride;
    __shared__ uint32_t s_hist[kPfBlockRows][kHistWords];
    __shared__ int s_prefix[kPfMaxSeq + 1];
    __shared__ uint32_t s_scan[kPfWaves];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform: row data stays scalar
    const int n = lane & 31;
    const int g = lane >> 5;

    // Work items (query block, segment), block-fastest: the launch holds one workgroup per
    // item, or fewer that stride over them (a bounded grid, for callers that run other
    // kernels beside the prefill: workgroups that run out of items free their CU instead
    // of queueing more items behind the other kernels).
    const int nb_items = p.rows / kPfBlockRows + p.sequences;
    // Block tables are often far wider than the sequences: a workgroup whose first segment starts past
    // every sequence (its later ones do too) has nothing to do, and leaves before it clears and scans.
    // The segment is chosen by the table's width: 2 x 1000 rows against 750-1500 keys in tables of 65536
    // took 34 us with 4096 keys per item, 45 with the shorter one chosen and every workgroup scanning,
    // 32 as it is (bf16 58, 58 and 37).
    const int begin = static_cast<int>(blockIdx.x) / nb_items * segment;
    auto blocks_of = [&](int s) {
        return s < p.sequences ? max((p.cu_seqlens_q[s + 1] - p.cu_seqlens_q[s] + kPfBlockRows - 1) / kPfBlockRows, 0) : 0;
    };
    int longest = lane < p.sequences ? p.seq_lens_k[lane] : 0;
    int mine = blocks_of(tid);
    asm volatile("" : "+v"(longest), "+v"(mine));  // one memory latency for both
    for (int s = lane + 64; s - lane < p.sequences; s += 64) longest = max(longest, s < p.sequences ? p.seq_lens_k[s] : 0);
    if (begin > 0 && __ballot(longest > begin) == 0ull) return;  // uniform

    // Query blocks per sequence -> prefix sums; this workgroup's sequence and rows.
    int running = 0;
    for (int base = 0; base < p.sequences; base += kPfThreads) {
        const int s = base + tid;
        uint32_t total;
        const uint32_t excl = block_exclusive_scan(static_cast<uint32_t>(base == 0 ? mine : blocks_of(s)), s_scan, &total);
        if (s < p.sequences) s_prefix[s] = running + static_cast<int>(excl);
        running += static_cast<int>(total);
    }
    if (tid == 0) s_prefix[p.sequences] = running;
    for (int i = tid; i < kPfBlockRows * kHistWords; i += kPfThreads) (&s_hist[0][0])[i] = 0u;
    __syncthreads();
    const int64_t n_items =
        static_cast<int64_t>(nb_items) * ((p.max_blocks * kBlockTokens + segment - 1) / segment);
    uint32_t err = 0;
    for (int64_t item = blockIdx.x; item < n_items; item += gridDim.x) {
    const int block = static_cast<int>(item) % nb_items;  // n_items <= 2^31 - 1 (validated)
    const int segi = static_cast<int>(item) / nb_items;
    if (block >= s_prefix[p.sequences]) continue;  // uniform
    int lo = 0, hi = p.sequences - 1;            // largest s with s_prefix[s] <= block
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (s_prefix[mid] <= block) lo = mid; else hi = mid - 1;
    }
    const int seq = lo;
    const int q0 = p.cu_seqlens_q[seq];
    const int q_len = p.cu_seqlens_q[seq + 1] - q0;
    const int k_len = min(max(p.seq_lens_k[seq], 0), p.max_blocks * kBlockTokens);
    const int j0 = (block - s_prefix[seq]) * kPfBlockRows;

    // The wave's two rows: visibility (right-down causal) and row_valid.
    int vis[kPfRowsPerWave];
    int rowi[kPfRowsPerWave];
#pragma unroll
    for (int q = 0; q < kPfRowsPerWave; ++q) {
        const int j = j0 + wave * kPfRowsPerWave + q;
        const bool live = j < q_len;
        rowi[q] = q0 + min(j, q_len - 1);
        vis[q] = live ? min(max(k_len - q_len + j + 1, 0), k_len) : 0;
        if (live && segi == 0 && lane == 0) p.row_valid[q0 + j] = vis[q];
    }
    const int last = min(j0 + kPfBlockRows, q_len) - 1;
    const int vis_max = min(max(k_len - q_len + last + 1, 0), k_len);
    const int seg0 = segi * segment;
    const int seg_end = min(seg0 + segment, vis_max);
    if (seg0 >= seg_end) continue;  // uniform: nothing visible in this segment
    const int nchunks = (seg_end - seg0 + kPfChunk - 1) / kPfChunk;

    // Q fragments and head weights of the wave's rows.
    v4i qa[kPfRowsPerWave][MT][NV];
    float wr[kPfRowsPerWave][MT * 16];
#pragma unroll
    for (int q = 0; q < kPfRowsPerWave; ++q) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const v4i* src = reinterpret_cast<const v4i*>(static_cast<const uint8_t*>(p.query) +
                                                          (static_cast<size_t>(rowi[q]) * HEADS + mt * 32 + n) * kRowBytes +
                                                          g * (kRowBytes / 2));
#pragma unroll
            for (int v = 0; v < NV; ++v) qa[q][mt][v] = src[v];
#pragma unroll
            for (int r4 = 0; r4 < 4; ++r4) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    wr[q][mt * 16 + r4 * 4 + j] =
                        pf_weight<W_BF16>(p, static_cast<size_t>(rowi[q]) * HEADS + mt * 32 + r4 * 8 + g * 4 + j);
                }
            }
        }
    }

    // Page ids of the segment (lane i < 32 holds page seg0/128 + i, clamped to the
    // sequence's last page; out-of-range ids read block 0 with zero key scale).
    const int pages_k = (k_len + kBlockTokens - 1) / kBlockTokens;
    int my_page = 0;
    float my_ok = 0.0f;
    if (lane < kPfPages) {
        const int pi = min(seg0 / kBlockTokens + lane, max(pages_k - 1, 0));
        const int id = p.block_table[static_cast<size_t>(seq) * p.max_blocks + pi];
        const bool ok = static_cast<unsigned>(id) < static_cast<unsigned>(p.num_blocks);
        my_page = ok ? id : 0;
        my_ok = ok ? 1.0f : 0.0f;
        if (!ok) err |= KVIP_STATUS_BAD_BLOCK;
    }
    const bool pages_ok = __ballot(lane < kPfPages && my_ok == 0.0f) == 0ull;  // uniform
    const uint8_t* kbase = static_cast<const uint8_t*>(p.keys);

    // Wave w stages rows [w * chunk/4, (w + 1) * chunk/4) of a chunk (one page's rows):
    // 8 direct-to-LDS loads of kRowsPerLoad rows each.
    constexpr int kWaveRows = kPfChunk / kPfWaves;
    const uint32_t k_lds = lds_addr(&s_k[0][0]), ks_lds = lds_addr(&s_ks[0][0]);
    auto stage = [&](int c, int buf) {
        const int pg = __builtin_amdgcn_readlane(my_page, c * kChunkPages + (wave * kWaveRows) / kBlockTokens);
#pragma unroll
        for (int v = 0; v < kStageLoads; ++v) {
            const int row = wave * kWaveRows + v * kRowsPerLoad + lane / kPieces;
            const int piece = (lane % kPieces) ^ pf_swizzle<ELEM>(row);
            const uint8_t* src = kbase + static_cast<size_t>(pg) * p.key_block_stride +
                                 (row & (kBlockTokens - 1)) * kRowBytes + piece * 16;
            dma16(src, k_lds + buf * kPfChunkBytes + (wave * kWaveRows + v * kRowsPerLoad) * kRowBytes);
        }
        if (wave == 0 && p.key_scale != nullptr && lane < kPfChunk / 4) {
            const int row = lane * 4;  // 4 consecutive scales of one page
            // readlane takes a wave-uniform lane index: read both pages, pick per half-wave.
            const int pg0 = __builtin_amdgcn_readlane(my_page, c * kChunkPages);
            const int pg1 = __builtin_amdgcn_readlane(my_page, c * kChunkPages + kChunkPages - 1);
            const int pg = lane < 32 ? pg0 : pg1;
            const float* src = p.key_scale + static_cast<size_t>(pg) * p.scale_block_stride + (row & 127);
            dma16(reinterpret_cast<const uint8_t*>(src), ks_lds + buf * kPfChunk * 4);
        }
    };
    if (p.key_scale == nullptr) {  // unit key scales, written once before the loop
        for (int i = tid; i < 2 * kPfChunk; i += kPfThreads) (&s_ks[0][0])[i] = 1.0f;
        __syncthreads();
    }

    // This lane half's row (one row per wave: the row of both halves).
    int vis_mine, vis_max_wave;
    if constexpr (kPfRowsPerWave == 2) {
        vis_mine = g == 0 ? vis[0] : vis[1];
        vis_max_wave = max(vis[0], vis[1]);
    } else {
        vis_mine = vis[0] - 32 * g;  // lane half g finishes tile k + g
        vis_max_wave = vis[0];
    }
    const int hist_row = wave * kPfRowsPerWave + (kPfRowsPerWave == 2 ? g : 0);
    // Per-lane LDS addresses: the tile row's first swizzled K piece (the swizzle of row k*32 + n
    // does not depend on k; piece u sits at the address XOR 16 u), its key scale, and the key strip
    // slots.
    const uint32_t ka = k_lds + n * kRowBytes + (((g * NV) ^ pf_swizzle<ELEM>(n)) * 16);
    const uint32_t ksa = ks_lds + n * 4;
    const uint32_t keya = lds_addr(&s_keys[wave][kPfRowsPerWave == 2 ? g : 0][n]);
    const uint32_t hista = lds_addr(&s_hist[hist_row][(lane % kHistCopies) * kHistStride]);
    constexpr uint32_t kKBuf = kPfChunkBytes;          // bytes between the two K buffers
    constexpr uint32_t kSBuf = kPfChunk * 4;           // bytes between the two scale buffers

    stage(0, 0);
    int stores = 0;  // key stores this wave issued after the latest staging loads
    for (int c = 0; c < nchunks; ++c) {
        const int buf = c & 1;
        lds_barrier(stores);  // chunk c landed and is visible; buffer c+1 is free again
        if (c + 1 < nchunks) stage(c + 1, buf ^ 1);
        const int cstart = seg0 + c * kPfChunk;
        // A lane's key of tile k is visible while 32 k is below this.
        const int left = vis_mine - cstart - n;
        const float page_ok0 =
            __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, my_ok), c * kChunkPages));
        const float page_ok1 = __builtin_bit_cast(
            float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, my_ok), c * kChunkPages + kChunkPages - 1));
        // Tile k's fragments and key scale. They are requested as soon as the MFMAs of the tile before
        // are issued, so that the reads pass under that tile's epilogue; the chunk's last tile repeats
        // its own.
        auto load_tile = [&](int k, v4i (&kb)[NV], float& ks) {
            const uint32_t a = ka + buf * kKBuf + k * 32 * kRowBytes;
#pragma unroll
            for (int u = 0; u < NV; ++u) kb[u] = *(LdsV4i)(a ^ (u * 16));
            ks = *(LdsF32)(ksa + buf * kSBuf + k * 128);
        };
        if constexpr (kPfRowsPerWave == 1) {
            // One row per wave (bf16): two tiles per step, finished together. Lane half g
            // finishes tile k + g: one lane-half swap joins both tiles' head halves, so every
            // lane stores a key and counts it (the same sums, in the same order, as one tile
            // at a time).
            v4i kb[NV];
            float ks_raw[2];
            load_tile(0, kb, ks_raw[0]);
#pragma unroll 1
            for (int k = 0; k < kPfTiles; k += 2) {
                const int t0 = cstart + k * 32;
                if (t0 >= vis_max_wave) break;  // uniform per wave: later tiles are masked too
                float pj[2][4], ks;
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    pj[h][0] = pj[h][1] = pj[h][2] = pj[h][3] = 0.f;
                    if (h == 0 || g == 1) ks = ks_raw[h];
                    // As below, with head tiles of STEPS MFMAs each: head tile u + 1's MFMAs are issued
                    // between the 32 VALU ops of head tile u.
                    v16f acc[2];
#pragma unroll
                    for (int u = -1; u < MT; ++u) {  // step -1: head tile 0's MFMAs
                        v16f& nxt = acc[(u + 1) & 1];
                        if (u + 1 < MT) {
                            nxt = v16f{0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
                            for (int st = 0; st < STEPS; ++st) Mma<ELEM>::step(st, qa[0][u + 1], kb, nxt);
                        }
                        if (u >= 0) {
                            const v16f& cur = acc[u & 1];
#pragma unroll
                            for (int r4 = 0; r4 < 4; ++r4) {
#pragma unroll
                                for (int j = 0; j < 4; ++j) {
                                    const float relu = __int_as_float(max(__float_as_int(cur[r4 * 4 + j]), 0));
                                    pj[h][j] = fmaf(relu, wr[0][u * 16 + r4 * 4 + j], pj[h][j]);
                                }
                            }
                        }
                        if (u >= 0 && u + 1 < MT) {
#pragma unroll
                            for (int st = 0; st < STEPS; ++st) {
                                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                                __builtin_amdgcn_sched_group_barrier(0x002, 32 / STEPS, 0);
                            }
                        }
                        if (u + 1 < MT) __builtin_amdgcn_sched_barrier(0);
                        if (u + 2 == MT) {  // the tile's last MFMAs are issued
                            load_tile(min(k + h + 1, kPfTiles - 1), kb, ks_raw[1 - h]);
                            __builtin_amdgcn_sched_barrier(0);
                        }
                    }
                }
                if (!pages_ok) ks *= k + g < kPfTiles / 2 ? page_ok0 : page_ok1;
                const float part0 = (pj[0][0] + pj[0][1]) + (pj[0][2] + pj[0][3]);
                const float part1 = (pj[1][0] + pj[1][1]) + (pj[1][2] + pj[1][3]);
                // [tile k lanes 0-31, tile k + 1 lanes 0-31] + [tile k lanes 32-63, tile k + 1 lanes 32-63].
                const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_int(part0), __float_as_int(part1), false, false);
                const float total = __int_as_float(sw[0]) + __int_as_float(sw[1]);
                const uint32_t key = score_key(total * ks);
                *(LdsU16)(keya + (k + g) * 64) = static_cast<uint16_t>(key);
                if (k * 32 < left) pf_count(hista, key);
            }
        } else {
            v4i kb[NV];
            float ks_raw;
            load_tile(0, kb, ks_raw);
#pragma unroll 1
            for (int k = 0; k < kPfTiles; ++k) {
                const int t0 = cstart + k * 32;
                if (t0 >= vis_max_wave) break;  // uniform per wave: later tiles are masked too
                const float ks = pages_ok ? ks_raw : ks_raw * (k < kPfTiles / 2 ? page_ok0 : page_ok1);
                // Units u = (row q = u / MT, head tile mt = u % MT), two dependent K-slice MFMAs
                // each. Unit u+1's MFMAs are issued between the 32 VALU ops (ReLU, weight FMA) of
                // unit u's epilogue so that the matrix core and the VALU work side by side.
                constexpr int U = kPfRowsPerWave * MT;
                float pj[kPfRowsPerWave][4];
#pragma unroll
                for (int q = 0; q < kPfRowsPerWave; ++q) pj[q][0] = pj[q][1] = pj[q][2] = pj[q][3] = 0.f;
                v16f acc[2];
#pragma unroll
                for (int u = -1; u < U; ++u) {  // step -1: unit 0's MFMAs
                    v16f& nxt = acc[(u + 1) & 1];
                    if (u + 1 < U) {
                        nxt = v16f{0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
                        for (int st = 0; st < STEPS; ++st) Mma<ELEM>::step(st, qa[(u + 1) / MT][(u + 1) % MT], kb, nxt);
                    }
                    if (u >= 0) {
                        const int q = u / MT, mt = u % MT;
                        const v16f& cur = acc[u & 1];
#pragma unroll
                        for (int r4 = 0; r4 < 4; ++r4) {
#pragma unroll
                            for (int j = 0; j < 4; ++j) {
                                const float relu = __int_as_float(max(__float_as_int(cur[r4 * 4 + j]), 0));
                                pj[q][j] = fmaf(relu, wr[q][mt * 16 + r4 * 4 + j], pj[q][j]);
                            }
                        }
                    }
                    if (u >= 0 && u + 1 < U) {
                        // The next unit's STEPS MFMAs spread over this unit's 32 VALU ops (1 MFMA, 16
                        // VALU, 1 MFMA, 16 VALU); nothing crosses into the next unit.
#pragma unroll
                        for (int st = 0; st < STEPS; ++st) {
                            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                            __builtin_amdgcn_sched_group_barrier(0x002, 32 / STEPS, 0);
                        }
                    }
                    if (u + 1 < U) __builtin_amdgcn_sched_barrier(0);
                    if (u + 2 == U) {  // the tile's last MFMAs are issued
                        load_tile(min(k + 1, kPfTiles - 1), kb, ks_raw);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
                // The two rows finish together: after the swap [row 0 lanes 0-31, row 1 lanes 0-31] +
                // [row 0 lanes 32-63, row 1 lanes 32-63], i.e. lanes 0-31 hold row 0's total for token n
                // and lanes 32-63 row 1's.
                const float part0 = (pj[0][0] + pj[0][1]) + (pj[0][2] + pj[0][3]);
                const float part1 = (pj[1][0] + pj[1][1]) + (pj[1][2] + pj[1][3]);
                const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_int(part0), __float_as_int(part1), false, false);
                const float total = __int_as_float(sw[0]) + __int_as_float(sw[1]);
                const uint32_t key = score_key(total * ks);
                *(LdsU16)(keya + k * 64) = static_cast<uint16_t>(key);
                if (k * 32 < left) pf_count(hista, key);
            }
        }
        // Flush the chunk's keys of the wave's rows (8-byte stores, inside the row stride).
        // Lane 0's store is always in range (cstart < key_stride, both multiples of 8), so
        // each live row issues exactly one store instruction.
        stores = 0;
#pragma unroll
        for (int q = 0; q < kPfRowsPerWave; ++q) {
            if (cstart >= vis[q]) continue;  // uniform
            const int o = min(lane * 4, kPfChunk - 4);
            const v2i v = *reinterpret_cast<const v2i*>(&s_keys[wave][q][o]);
            if (lane * 4 < kPfChunk && cstart + o + 4 <= p.key_stride) {
                *reinterpret_cast<v2i*>(p.score_keys + static_cast<size_t>(rowi[q]) * p.key_stride + cstart + o) = v;
            }
            ++stores;
        }
    }
    lds_barrier(0);
    // Histogram of the workgroup's rows.
    for (int i = tid; i < kPfBlockRows * 256; i += kPfThreads) {
        const int rq = i >> 8;
        const int bin = i & 255;
        const int j = j0 + rq;
        uint32_t c = 0u;
#pragma unroll
        for (int cp = 0; cp < kHistCopies; ++cp) c += (s_hist[rq][cp * kHistStride + (bin & 127)] >> (16 * (bin >> 7))) & 0xFFFFu;
        if (j < q_len && c != 0u) atomicAdd(&p.histogram[static_cast<size_t>(q0 + j) * 256 + bin], c);
    }
    if (item + gridDim.x < n_items) {  // uniform: clear the row histograms for the next item
        __syncthreads();
        for (int i = tid; i < kPfBlockRows * kHistWords; i += kPfThreads) (&s_hist[0][0])[i] = 0u;
        __syncthreads();
    }
    }
    report(p.status, err);
}

// Work items: (query blocks bound) x (segments of the bound context).
int64_t prefill_items(const KvipPrefillArgs& a, int segment) {
    const int64_t blocks = a.rows / kPfBlockRows + a.sequences;  // bound on the per-sequence blocks
    return blocks * ((static_cast<int64_t>(a.max_blocks) * kBlockTokens + segment - 1) / segment);
}

// Key positions per work item. With few items a long segment leaves CUs idle (one chunk of 256
// keys takes about 5 us, 16 of them 80 us) or ends in a last round that few of them share; a short
// one pays an item's Q fragments, staging latency and histogram flush more often. The launch is
// priced as (all items, or one per CU, + a tail from uneven items) x (lead + chunks) in chunk times
// and the cheapest segment taken. Lead and tail are fitted to every segment measured at 16
// shapes of 16 to 8192 rows against 1024 to 65536 keys: lead 0.5 and tail 1 for fp8, 1.25 and
// 0.25 for bf16 (twice the Q, one workgroup per CU); the choice is within 1% (fp8) and 3% (bf16) of
// the best segment on average, 19% at worst. Against 4096 keys throughout, scoring alone, us fp8 /
// bf16: 16 rows x 4096 keys 79.2 -> 12.3 / 90.0 -> 14.5, 64 x 16384 79.8 -> 24.5 / 92.3 -> 41.5, 512 x
// 8192 80.9 -> 45.9 / 97.2 -> 63.7, six sequences of 33-900 rows against 900-9000 keys 140 -> 120 / 206
// (the same), 4096 x 16384 477 -> 450 / 817 (the same). Long segments stay where items are many:
// 2048 x 65536 takes 974 us with 4096 keys and 1447 with 256. A bounded grid keeps 4096 keys: its
// launch runs beside other kernels, which take the CUs of the workgroups that run out of items, and
// items of equal size would hold all of them to the end (a round of 32 decode requests beside
// chunks of 2048 x 8192 and 1536 x 1536: 307-310 us with short segments, 276-279 with these).
int prefill_segment(const KvipPrefillArgs& a, int workgroups) {
    if (workgroups > 0) return kPfSegment;
    constexpr int64_t cus = 256;
    const bool fp8 = a.qk_dtype == KVIP_DTYPE_FP8_E4M3;
    const int64_t lead = fp8 ? 2 : 5, tail = fp8 ? 4 : 1;  // quarters of a chunk, of an item per CU
    const int64_t context_chunks = (static_cast<int64_t>(a.max_blocks) * kBlockTokens + kPfChunk - 1) / kPfChunk;
    // Likely blocks (prefill_items has the bound): a further sequence ends in half a block on average.
    const int64_t blocks = (a.rows + kPfBlockRows / 2 * (a.sequences - 1) + kPfBlockRows - 1) / kPfBlockRows;
    int best = kPfSegment;
    int64_t best_cost = INT64_MAX;
    for (int segment = kPfSegment; segment >= kPfChunk; segment /= 2) {
        if (prefill_items(a, segment) > INT32_MAX) break;  // the kernel's item index
        const int64_t items = blocks * ((static_cast<int64_t>(a.max_blocks) * kBlockTokens + segment - 1) / segment);
        const int64_t item = lead + 4 * std::min<int64_t>(segment / kPfChunk, context_chunks);
        const int64_t cost = 4 * std::max(items * lead + blocks * 4 * context_chunks, cus * item) + tail * cus * item;
        if (cost < best_cost) best = segment, best_cost = cost;
    }
    return best;
}

template <int ELEM, int HEADS>
hipError_t launch_heads(const KvipPrefillArgs& a, int workgroups, hipStream_t stream) {
    const int segment = prefill_segment(a, workgroups);
    const int64_t items = prefill_items(a, segment);
    const dim3 grid(static_cast<unsigned>(workgroups > 0 ? std::min<int64_t>(items, workgroups) : items));
    if (a.weight_dtype == KVIP_DTYPE_BF16) {
        hipLaunchKernelGGL((indexer_prefill_kernel<ELEM, HEADS, true>), grid, dim3(PfShape<ELEM>::kThreads), 0, stream,
                           a, segment);
    } else {
        hipLaunchKernelGGL((indexer_prefill_kernel<ELEM, HEADS, false>), grid, dim3(PfShape<ELEM>::kThreads), 0, stream,
                           a, segment);
    }
    return hipGetLastError();
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

}  // namespace

uint32_t validate_prefill(const KvipPrefillArgs* a) {
    if (a == nullptr) return KVIP_ERR_INVALID;
    const bool ok =
        a->query != nullptr && a->weights != nullptr && a->keys != nullptr && a->block_table != nullptr &&
        a->cu_seqlens_q != nullptr && a->seq_lens_k != nullptr && a->score_keys != nullptr &&
        a->histogram != nullptr && a->row_valid != nullptr &&
        (a->qk_dtype == KVIP_DTYPE_FP8_E4M3 || a->qk_dtype == KVIP_DTYPE_BF16) &&
        (a->weight_dtype == KVIP_DTYPE_FP32 || a->weight_dtype == KVIP_DTYPE_BF16) &&
        (a->heads == 32 || a->heads == 64) && a->sequences >= 1 && a->sequences <= kPfMaxSeq && a->rows >= 1 &&
        a->rows <= (1 << 24) && a->max_blocks >= 1 && a->num_blocks >= 1 &&
        a->max_blocks <= (1 << 24) / kBlockTokens &&
        static_cast<int64_t>(a->key_stride) >= static_cast<int64_t>(a->max_blocks) * kBlockTokens &&
        a->key_stride % 8 == 0 && a->key_block_stride % 16 == 0 &&
        a->key_block_stride >=
            static_cast<int64_t>(kBlockTokens) * kIndexDim * (a->qk_dtype == KVIP_DTYPE_BF16 ? 2 : 1) &&
        (a->key_scale == nullptr || (a->scale_block_stride >= kBlockTokens && a->scale_block_stride % 4 == 0 &&
                                     (reinterpret_cast<uintptr_t>(a->key_scale) & 15u) == 0)) &&
        aligned16(a->query) && aligned16(a->keys) && aligned16(a->score_keys) &&
        prefill_items(*a, kPfSegment) <= 0x7FFFFFFF;
    return ok ? KVIP_OK : KVIP_ERR_INVALID;
}

hipError_t launch_prefill(const KvipPrefillArgs& a, hipStream_t stream, int workgroups) {
    if (a.qk_dtype == KVIP_DTYPE_BF16) {
        return a.heads == 64 ? launch_heads<2, 64>(a, workgroups, stream) : launch_heads<2, 32>(a, workgroups, stream);
    }
    return a.heads == 64 ? launch_heads<1, 64>(a, workgroups, stream) : launch_heads<1, 32>(a, workgroups, stream);
}

}  // namespace kvip

extern "C" uint32_t kvip_hip_indexer_prefill(const KvipPrefillArgs* args, void* stream) {
    const uint32_t rc = kvip::validate_prefill(args);
    if (rc != KVIP_OK) return rc;
    return static_cast<uint32_t>(kvip::launch_prefill(*args, static_cast<hipStream_t>(stream), 0));
}

extern "C" uint32_t kvip_hip_indexer_prefill_grid(const KvipPrefillArgs* args, int32_t workgroups, void* stream) {
    const uint32_t rc = kvip::validate_prefill(args);
    if (rc != KVIP_OK) return rc;
    if (workgroups < 0) return KVIP_ERR_INVALID;
    return static_cast<uint32_t>(kvip::launch_prefill(*args, static_cast<hipStream_t>(stream), workgroups));
}
