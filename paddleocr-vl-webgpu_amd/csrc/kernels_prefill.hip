// Causal prefill for gfx950: rotary + range append into the paged cache, then
// MFMA flash attention over the cache; both in one kernel for short prompts
// (prefill_short_kernel).
//
// Kernel 1 (one 16-token cache block per workgroup): rotates the 2 key heads
// and writes them with the values into the blocked cache (the same rounding as the decode
// append, so prefill and decode leave bit-identical rows), and, when the
// caller passes a query scratch, writes the rotated queries there.  Replaces
// decoder_prefill_mrope_f32 and decoder_kv_append_range_f32
// (crates/pvlc-wgsl/src/lib.rs:1334-1416).
//
// Kernel 2 (attention) has two forms, chosen in launch_prefill:
//
//  * prefill_wave_attention_kernel (prompts beyond kPrefillShortTokens or with
//    a query scratch, up to kPrefillWaveTokens, and any
//    length without a workspace): one workgroup per (16-token query block, 1
//    or 2 heads), its waves taking the key steps in turn, each streaming its
//    keys and values from L2 into registers with no barrier in the loop, and
//    merging through LDS at the end.  Short prompts have few query blocks, so
//    the heads and the keys of a block are spread over workgroups and waves.
//  * prefill_attention_kernel (longer prompts, with a workspace): one
//    workgroup per (query block or part of one, kv head) serves the 8 query
//    heads of the group, 2 per wave, over keys and values that stream through
//    double-buffered LDS in steps of 64 keys, laid out so every operand read
//    is conflict-free; long blocks split over two workgroups (pair schedule).
//
// Both compute
//   S^T[key][row] = K . Q^T           v_mfma_f32_16x16x32_f16
//   O[row][dim]  += P[row][key] V      v_mfma_f32_16x16x32_f16
//   l[row]       += P[row][key] 1      (same MFMA, ones operand)
// The key slot order of the cache (key_slot) makes the score MFMA leave each
// lane 8 consecutive keys of one tile, which is the P operand of the P.V MFMA.
// Online softmax in log2 units (scale folded into one FMA per score), the
// causal mask only on steps that reach the diagonal, and the rescale skipped
// while the running max stays near its reference.  Replaces
// decoder_prefill_gqa_f32 (crates/pvlc-wgsl/src/lib.rs:1262-1332); arithmetic
// reference causal_gqa_f32 (crates/pvlc-cpu-ref/src/lib.rs:782-853).

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "pvlc_device.hpp"
#include "pvlc_internal.hpp"

namespace pvlc {
namespace {

constexpr float kLog2e = 1.4426950408889634f;
constexpr int kQueryBlock = 16;  // query tokens per workgroup
constexpr int kKeyStep = 64;     // keys per softmax step (4 cache blocks)
constexpr int kStepTiles = kKeyStep / 16;
constexpr int kWaves = 4;        // each wave: 2 of the 8 heads of the group
constexpr float kLazyRescaleLog2 = 8.0f;  // softmax reference moves only past 2^8
// Longest prompt of the one-head form of prefill_wave_attention_kernel.
constexpr uint32_t kPrefillOneHeadTokens = 768;

struct PrefillParams {
    uint32_t tokens;
    uint32_t num_blocks;
    const int32_t *block_table;
    uint16_t *key_cache;
    uint16_t *value_cache;
    const uint16_t *query;
    const uint16_t *key;
    const uint16_t *value;
    uint16_t *out;
    const float *rope_cos;
    const float *rope_sin;
    uint32_t rope_rows;
    const int32_t *positions;
    uint16_t *qrot;
    uint32_t *error_word;
    float scale_log2;
    // split-K pair schedule (prefill_attention_kernel)
    uint32_t *counters;  // [pair][kv head], cleared by the append kernel (null: no pair schedule)
    float *partials;     // [pair][kv head][2 parts][kPrefillPartialFloats]
    // f32 operands (pvlc_hip_paged_prefill_f32io): query, key, value, output;
    // null for the fp16 entry point.
    const float *query32;
    const float *key32;
    const float *value32;
    float *out32;
};

__device__ inline uint32_t cache_block(const PrefillParams &p, uint32_t tile, bool *ok) {
    if (p.block_table == nullptr) {
        *ok = tile < p.num_blocks;
        return *ok ? tile : 0u;
    }
    const int32_t b = load_const(p.block_table, tile);
    *ok = b >= 0 && static_cast<uint32_t>(b) < p.num_blocks;
    return *ok ? static_cast<uint32_t>(b) : 0u;
}

// Mask of the values of keys key .. key + 7 that belong to a prompt of n tokens.
// A partly filled last block keeps what the planes held in its other tokens:
// their weights are 0, but 0 times a NaN or an infinity there is NaN.
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
__device__ inline u32x4_t value_keep(int key, int n) {
    u32x4_t keep;
#pragma unroll
    for (int d = 0; d < 4; ++d) keep[d] = key + 2 * d + 1 < n ? ~0u : key + 2 * d < n ? 0xffffu : 0u;
    return keep;
}

// Kernel 1: one workgroup per 16-token cache block, both key heads.  Every
// thread rotates one pair of 8-dim key chunks, c and c + 8, which are each
// other's rotary partners (item = head, chunk pair, token; 16 consecutive
// threads fill one 256-byte run of the key slab), and writes one 32-byte value
// row of the slab (head, dim: 16 tokens) after a transpose of the block's
// value rows through LDS, so every cache store is a full 16-byte vector and
// each 32-byte sector is written once.  It is bound by its chain of dependent
// memory rounds, so there are three: positions, block id, keys and values;
// cos and sin; the stores (the optional arrays are read through a stand-in
// when not given, so no load waits behind a branch).  One chunk at a time,
// positions read behind a branch for each, it took five: whole prefill calls
// 25.7 -> 24.0 us at 1157 tokens, 84.6 -> 83.8 at 4096.  With a query scratch the
// workgroup also writes the rotated queries of its tokens (the attention
// kernel rotates its own query fragments, so the scratch is only an output for
// callers that want it).
constexpr int kAppendThreads = 256;

// Rotary position of token t and whether its tables hold it (bit 4 of the
// error word otherwise, reported once per token by the caller's choice).
__device__ inline int rope_position(const PrefillParams &p, uint32_t t, bool *rope) {
    const int pos = p.positions ? p.positions[t] : static_cast<int>(t);
    *rope = p.rope_cos != nullptr && pos >= 0 && static_cast<uint32_t>(pos) < p.rope_rows;
    return pos;
}

template <bool F32IO>
__global__ __launch_bounds__(kAppendThreads) void prefill_rope_append_kernel(PrefillParams p) {
    const int i = threadIdx.x;
    const uint32_t b = blockIdx.x;  // cache block (16 tokens) of the sequence
    const uint32_t t0 = b * kBlockTokens;
    const uint32_t ntok = min(p.tokens - t0, kBlockTokens);
    __shared__ uint16_t sv[kBlockTokens][kRowElems + 8];  // value rows, padded against bank conflicts

    const float *stand_in = F32IO ? p.value32 : reinterpret_cast<const float *>(p.value);
    // item: head hh, chunk pair (c, c + 8), token t (the last one again past
    // the end of the sequence, not stored)
    const int tt = i & 15, c = (i >> 4) & 7, hh = i >> 7;
    const uint32_t t = t0 + min(static_cast<uint32_t>(tt), ntok - 1);
    const int32_t pos_raw = (p.positions ? p.positions : reinterpret_cast<const int32_t *>(stand_in))[t];
    const int32_t id_raw = load_const(p.block_table ? p.block_table : reinterpret_cast<const int32_t *>(stand_in), b);
    typedef std::conditional_t<F32IO, float4_t, half8_t> Raw;
    constexpr int kRawLoads = F32IO ? 2 : 1, kRawElems = F32IO ? 4 : 8;
    Raw key[2][kRawLoads], val[2][kRawLoads];
    const size_t koff = (static_cast<size_t>(t) * kKvHeads + hh) * kHeadDim + c * 8;
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        // value rows of the block: 16 tokens x 256, two 8-element pieces per thread
        const int k = i + r * kAppendThreads;
        const size_t voff = static_cast<size_t>(t0 + min(static_cast<uint32_t>(k >> 5), ntok - 1)) * kRowElems + (k & 31) * 8;
#pragma unroll
        for (int f = 0; f < kRawLoads; ++f) {
            if constexpr (F32IO) {
                key[r][f] = *reinterpret_cast<const Raw *>(p.key32 + koff + r * 64 + f * kRawElems);
                val[r][f] = *reinterpret_cast<const Raw *>(p.value32 + voff + f * kRawElems);
            } else {
                key[r][f] = *reinterpret_cast<const Raw *>(p.key + koff + r * 64);
                val[r][f] = *reinterpret_cast<const Raw *>(p.value + voff);
            }
        }
    }
    const int pos = p.positions ? pos_raw : static_cast<int>(t);
    const bool rope = p.rope_cos != nullptr && pos >= 0 && static_cast<uint32_t>(pos) < p.rope_rows;
    float4_t cs[2], sn[2];
    {
        const float *cr = rope ? p.rope_cos + static_cast<size_t>(pos) * 64 + c * 8 : stand_in;
        const float *sr = rope ? p.rope_sin + static_cast<size_t>(pos) * 64 + c * 8 : stand_in;
#pragma unroll
        for (int f = 0; f < 2; ++f) {
            cs[f] = *reinterpret_cast<const float4_t *>(cr + f * 4);
            sn[f] = *reinterpret_cast<const float4_t *>(sr + f * 4);
        }
    }
    __builtin_amdgcn_sched_barrier(0);  // every load ahead of the arithmetic
    const int32_t id = p.block_table ? id_raw : static_cast<int32_t>(b);
    const bool ok = id >= 0 && static_cast<uint32_t>(id) < p.num_blocks;
    const uint32_t blk = ok ? static_cast<uint32_t>(id) : 0u;
    // keys, exactly as rotate_chunk rotates them
    half8_t lo, hi;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const float x = static_cast<float>(key[0][j / kRawElems][j % kRawElems]);
        const float y = static_cast<float>(key[1][j / kRawElems][j % kRawElems]);
        const float co = cs[j >> 2][j & 3], si = sn[j >> 2][j & 3];
        lo[j] = to_h(rope ? x * co + (-y) * si : x);
        hi[j] = to_h(rope ? y * co + x * si : y);
    }
    if constexpr (!F32IO) {
        if (!rope) {  // as given, bit for bit
            lo = key[0][0];
            hi = key[1][0];
        }
    }
    if (ok && static_cast<uint32_t>(tt) < ntok) {
        uint16_t *dst = p.key_cache + (static_cast<size_t>(blk) * kKvHeads + hh) * kBlockHeadElems + c * 128 + key_slot(tt) * 8;
        *reinterpret_cast<half8_t *>(dst) = lo;
        *reinterpret_cast<half8_t *>(dst + 8 * 128) = hi;
    }
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        const int k = i + r * kAppendThreads;
        half8_t v;
        if constexpr (F32IO) {
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = to_h(val[r][j / kRawElems][j % kRawElems]);
        } else {
            v = val[r][0];
        }
        *reinterpret_cast<half8_t *>(&sv[k >> 5][(k & 31) * 8]) = v;
    }
    if (p.error_word) {
        if (!ok && i == 0) atomicOr(p.error_word, 2u);
        if (!rope && p.rope_cos != nullptr && c == 0 && hh == 0 && static_cast<uint32_t>(tt) < ntok) atomicOr(p.error_word, 4u);
    }
    __syncthreads();
    if (ok) {
        // value slab row (head, dim): the block's 16 tokens; a partial last
        // block keeps the slab's other tokens as they were
        const int hh = i >> 7, d = i & 127;
        const size_t slab = (static_cast<size_t>(blk) * kKvHeads + hh) * kBlockHeadElems;
        uint16_t *dst = p.value_cache + slab + d * kBlockTokens;
        if (ntok == kBlockTokens) {
            u16x8_t lo, hi;
#pragma unroll
            for (int tt = 0; tt < 8; ++tt) {
                lo[tt] = sv[tt][hh * kHeadDim + d];
                hi[tt] = sv[tt + 8][hh * kHeadDim + d];
            }
            *reinterpret_cast<u16x8_t *>(dst) = lo;
            *reinterpret_cast<u16x8_t *>(dst + 8) = hi;
        } else {
            for (uint32_t tt = 0; tt < ntok; ++tt) dst[tt] = sv[tt][hh * kHeadDim + d];
        }
    }
    if (p.counters && i == 0) {
        // The pair schedule's arrival counters (one per block, and one more
        // for an odd number) start at zero whatever lay there: a workspace may
        // have served a shorter prompt, whose partials begin where a longer
        // one's counters are.
        p.counters[b] = 0;
        if (b + 1 == gridDim.x && (gridDim.x & 1u) != 0) p.counters[b + 1] = 0;
    }
    if (p.qrot) {
        // (token, head, 8-dim chunk) items of the block's tokens
        for (int k = i; k < static_cast<int>(kBlockTokens * kQueryHeads * 16); k += kAppendThreads) {
            const int tt = k / (kQueryHeads * 16);
            if (static_cast<uint32_t>(tt) >= ntok) break;
            const uint32_t tq = t0 + tt;
            const int h = (k >> 4) % kQueryHeads, d0 = (k & 15) * 8;
            bool rope;
            const int pos = rope_position(p, tq, &rope);
            const size_t qoff = (static_cast<size_t>(tq) * kQueryHeads + h) * kHeadDim;
            half8_t q;
            if constexpr (F32IO) {
                q = rope ? rotate_chunk(p.query32 + qoff, d0, p.rope_cos + static_cast<size_t>(pos) * 64,
                                        p.rope_sin + static_cast<size_t>(pos) * 64)
                         : round_chunk(p.query32 + qoff + d0);
            } else {
                const uint16_t *qrow = p.query + qoff;
                q = rope ? rotate_chunk(qrow, d0, p.rope_cos + static_cast<size_t>(pos) * 64,
                                        p.rope_sin + static_cast<size_t>(pos) * 64)
                         : *reinterpret_cast<const half8_t *>(qrow + d0);
            }
            *reinterpret_cast<half8_t *>(p.qrot + (static_cast<size_t>(tq) * kQueryHeads + h) * kHeadDim + d0) = q;
        }
    }
}

// LDS layouts of one 64-key step (2 pairs of 16-token tiles), chosen so every
// 16-lane group of an MFMA operand read is one contiguous 256-byte run (no
// bank conflicts):
//   keys   [pair][16 dim-chunks][score MFMA h][tile of pair][8 slots][8 dims]
//   values [pair][tile of pair][token half][128 dims][8 tokens]
constexpr int kStepElems = kStepTiles * kBlockHeadElems;  // fp16 elements per plane and step

__device__ inline int lds_key_offset(int j, int chunk, int h, int tile, int slot8) {
    return ((((j * 16 + chunk) * 2 + h) * 2 + tile) * 8 + slot8) * 8;
}
__device__ inline int lds_value_offset(int j, int tile, int half, int dim) {
    return (((j * 2 + tile) * 2 + half) * kHeadDim + dim) * 8;
}

template <bool F32IO>
__global__ __launch_bounds__(kWaves * 64, 2) void prefill_attention_kernel(PrefillParams p) {
    const int n = static_cast<int>(p.tokens);
    const int qblocks = (n + kQueryBlock - 1) / kQueryBlock;
    uint32_t g, pair = 0;
    PrefillSegment seg0{}, seg1{};
    const int nseg = static_cast<int>(prefill_pair_segments(blockIdx.x, static_cast<uint32_t>(qblocks), &g, &pair, &seg0, &seg1));
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int row = lane & 15, kg = lane >> 4;
    // Four distinct arrays (not one indexed by parity): the main loop picks
    // them at compile time, so the compiler sees that a step's loads into LDS
    // and its LDS reads touch different buffers and does not wait for the
    // loads before the reads.
    __shared__ __align__(16) uint16_t sk0[kStepElems], sk1[kStepElems];
    __shared__ __align__(16) uint16_t sv0[kStepElems], sv1[kStepElems];
    __shared__ bool sm_last;

  // One segment: a whole query block, or one part of a split one.
  auto run_segment = [&](const PrefillSegment sg) {
    const int qb = static_cast<int>(sg.qb);
    const uint32_t part = sg.part, nparts = sg.nparts;
    const int s_begin = static_cast<int>(sg.step_begin), steps = static_cast<int>(sg.steps);
    const int t0 = qb * kQueryBlock;
    const int my_token = t0 + row;  // query token of this lane's column

    // Query fragments (B operand): column = token t0 + row of head h, dims
    // kb*32 + kg*8 .. +8, rotated here (rotate-half: the partner of chunk kb
    // is chunk kb^2 of the same lane) exactly as rotate_chunk does.
    const int tq = min(my_token, n - 1);
    const int qpos = p.positions ? p.positions[tq] : tq;
    const bool qrope = p.rope_cos != nullptr && qpos >= 0 && static_cast<uint32_t>(qpos) < p.rope_rows;
    float4_t qc[2][2], qs[2][2];  // cos/sin of pairs hk*32 + kg*8 .. +8 (hk = kb & 1)
    {
        // Without rotary the loads read the query as a stand-in, in the
        // operand width that was given (the other pointer is null).
        const float *stand_in = F32IO ? p.query32 : reinterpret_cast<const float *>(p.query);
        const float *cr = qrope ? p.rope_cos + static_cast<size_t>(qpos) * 64 : stand_in;
        const float *sr = qrope ? p.rope_sin + static_cast<size_t>(qpos) * 64 : stand_in;
#pragma unroll
        for (int hk = 0; hk < 2; ++hk)
#pragma unroll
            for (int f = 0; f < 2; ++f) {
                qc[hk][f] = *reinterpret_cast<const float4_t *>(cr + hk * 32 + kg * 8 + f * 4);
                qs[hk][f] = *reinterpret_cast<const float4_t *>(sr + hk * 32 + kg * 8 + f * 4);
            }
    }
    half8_t qf[2][4];
#pragma unroll
    for (int ct = 0; ct < 2; ++ct) {
        const int h = static_cast<int>(g) * kGroup + wave * 2 + ct;
        const size_t qoff = (static_cast<size_t>(tq) * kQueryHeads + h) * kHeadDim;
        if constexpr (F32IO) {
            // f32 query: rotated from its f32 values and rounded once.
            float raw[4][8];
#pragma unroll
            for (int kb = 0; kb < 4; ++kb) {
                const float4_t lo = *reinterpret_cast<const float4_t *>(p.query32 + qoff + kb * 32 + kg * 8);
                const float4_t hi = *reinterpret_cast<const float4_t *>(p.query32 + qoff + kb * 32 + kg * 8 + 4);
#pragma unroll
                for (int jj = 0; jj < 4; ++jj) {
                    raw[kb][jj] = lo[jj];
                    raw[kb][jj + 4] = hi[jj];
                }
            }
#pragma unroll
            for (int kb = 0; kb < 4; ++kb) {
                half8_t q;
#pragma unroll
                for (int jj = 0; jj < 8; ++jj) {
                    if (qrope) {
                        const float c = qc[kb & 1][jj >> 2][jj & 3];
                        const float sn = qs[kb & 1][jj >> 2][jj & 3];
                        const float x = raw[kb][jj];
                        const float y = raw[kb ^ 2][jj];
                        q[jj] = kb < 2 ? to_h(x * c + (-y) * sn) : to_h(x * c + y * sn);
                    } else {
                        q[jj] = to_h(raw[kb][jj]);
                    }
                }
                qf[ct][kb] = my_token < n ? q : half8_t{};
            }
        } else {
            const uint16_t *qrow = p.query + qoff;
            half8_t raw[4];
#pragma unroll
            for (int kb = 0; kb < 4; ++kb) raw[kb] = *reinterpret_cast<const half8_t *>(qrow + kb * 32 + kg * 8);
#pragma unroll
            for (int kb = 0; kb < 4; ++kb) {
                half8_t q = raw[kb];
                if (qrope) {
#pragma unroll
                    for (int jj = 0; jj < 8; ++jj) {
                        const float c = qc[kb & 1][jj >> 2][jj & 3];
                        const float sn = qs[kb & 1][jj >> 2][jj & 3];
                        const float x = static_cast<float>(raw[kb][jj]);
                        const float y = static_cast<float>(raw[kb ^ 2][jj]);
                        q[jj] = kb < 2 ? to_h(x * c + (-y) * sn) : to_h(x * c + y * sn);
                    }
                }
                qf[ct][kb] = my_token < n ? q : half8_t{};
            }
        }
    }

    const int nkeys = min(t0 + kQueryBlock, n);
    const int last_tile = (nkeys - 1) >> 4;
    const bool last_part = part + 1 == nparts;

    // Double-buffered LDS, filled by direct global-to-LDS loads (16 bytes a
    // lane: lane l of a wave's load lands at the wave's LDS base + 16 l).
    // Each wave issues 4 key and 4 value loads per step; lane and load index
    // pick the global chunk that belongs at that LDS position of the layouts
    // above.  Steps past the end re-read the last tile (never used).
    typedef __attribute__((address_space(3))) void *lds_ptr;
    // ln: the lane id (passed in, so the last steps can use a separately
    // computed copy; see the tail loop below).
    auto dma_k = [&](int step, uint16_t *dst, int ln) {
        // LDS chunk q = 64 k + ln (k = 4 wave + r): slot8 = ln & 7,
        // tile = ln bit 3, h = ln bit 4, dim-chunk = 2 (k & 7) + ln bit 5, pair j = k >> 3
        const int j = wave >> 1;
        bool ok;
        const uint32_t b0 = cache_block(p, static_cast<uint32_t>(min(step * kStepTiles + 2 * j, last_tile)), &ok);
        const uint32_t b1 = cache_block(p, static_cast<uint32_t>(min(step * kStepTiles + 2 * j + 1, last_tile)), &ok);
        const uint32_t blk = (ln & 8) ? b1 : b0;
        const uint16_t *src = p.key_cache + (static_cast<size_t>(blk) * kKvHeads + g) * kBlockHeadElems +
                              (((ln >> 4) & 1) * 8 + (ln & 7)) * 8 + (ln >> 5) * 128;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int k = 4 * wave + r;
            __builtin_amdgcn_global_load_lds(src + (2 * (k & 7)) * 128, (lds_ptr)(dst + 64 * k * 8), 16, 0, 0);
        }
    };
    auto dma_v = [&](int step, uint16_t *dst, int ln) {
        // LDS chunk q = 64 k + ln: dim = (k & 1) 64 + ln, half = (k >> 1) & 1,
        // tile = (k >> 2) & 1 = wave & 1, pair j = k >> 3 = wave >> 1
        bool ok;
        const uint32_t blk = cache_block(p, static_cast<uint32_t>(min(step * kStepTiles + wave, last_tile)), &ok);
        const uint16_t *src = p.value_cache + (static_cast<size_t>(blk) * kKvHeads + g) * kBlockHeadElems + ln * 16;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int k = 4 * wave + r;
            __builtin_amdgcn_global_load_lds(src + (r & 1) * 64 * 16 + (r >> 1) * 8, (lds_ptr)(dst + 64 * k * 8), 16,
                                             0, 0);
        }
    };

    float4_t o[2][9];  // 8 column tiles of the output, then the row sums
#pragma unroll
    for (int ct = 0; ct < 2; ++ct)
#pragma unroll
        for (int c = 0; c < 9; ++c) o[ct][c] = float4_t{0.f, 0.f, 0.f, 0.f};
    half8_t ones;
#pragma unroll
    for (int e = 0; e < 8; ++e) ones[e] = static_cast<_Float16>(1.0f);
    const float scale = p.scale_log2;

    // Scores of one step: MFMA h of pair j leaves lane (column = query token,
    // kg) the keys (kg & 1)*8 + h*4 + r of the pair's tile kg >> 1.
    typedef float Scores[2][2][8];
    auto scores = [&](const uint16_t *kl, Scores &x) {
        // 8 independent accumulator chains (pair j, slot half h, head ct), the
        // 32-dim chunk kb outermost, so no MFMA waits on the previous one
        float4_t acc[2][2][2];
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int ct = 0; ct < 2; ++ct) acc[j][h][ct] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) {
            half8_t kf[2][2];
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    kf[j][h] = *reinterpret_cast<const half8_t *>(kl + lds_key_offset(j, kb * 4 + kg, h, row >> 3, row & 7));
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int ct = 0; ct < 2; ++ct)
                        acc[j][h][ct] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[j][h], qf[ct][kb], acc[j][h][ct], 0, 0, 0);
        }
#pragma unroll
        for (int ct = 0; ct < 2; ++ct)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int r = 0; r < 4; ++r) x[ct][j][h * 4 + r] = acc[j][h][ct][r];
    };
    // The causal mask and the end of the sequence only touch steps that
    // reach past the first query token of the block.
    auto needs_mask = [&](int step) { return step * kKeyStep + kKeyStep - 1 > t0 || step * kKeyStep + kKeyStep > n; };
    auto apply_mask = [&](int step, Scores &x) {
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int key = step * kKeyStep + (2 * j + (kg >> 1)) * 16 + (kg & 1) * 8 + e;
                const bool keep = key <= my_token && key < n;
#pragma unroll
                for (int ct = 0; ct < 2; ++ct) x[ct][j][e] = keep ? x[ct][j][e] : -INFINITY;
            }
    };
    // Running max of the column (the 4 lanes of a column hold its 64 keys).
    auto column_max = [&](const Scores &x, const float (&m)[2], float (&m_new)[2]) {
#pragma unroll
        for (int ct = 0; ct < 2; ++ct) {
            float c = m[ct];
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int e = 0; e < 8; ++e) c = fmaxf(c, x[ct][j][e]);
            c = fmaxf(c, __shfl_xor(c, 16));
            m_new[ct] = fmaxf(c, __shfl_xor(c, 32));
        }
    };
    // P of pair j in fp16 (the A operand of P.V), log2 units, scale folded in.
    auto probs = [&](const Scores &x, const float (&ms)[2], int j, half8_t (&pa)[2][2]) {
#pragma unroll
        for (int ct = 0; ct < 2; ++ct)
#pragma unroll
            for (int e = 0; e < 8; ++e) pa[ct][j][e] = to_h(__builtin_amdgcn_exp2f(__builtin_fmaf(x[ct][j][e], scale, -ms[ct])));
    };
    // O += P.V over pair j, and the row sums += P.1 (exactly the rounded weights).
    // The pair's 8 value fragments are read from LDS before its MFMAs.
    auto pv_mfma = [&](const uint16_t *vl, int j, const half8_t (&pa)[2][2]) {
        half8_t vf[8];
#pragma unroll
        for (int c = 0; c < 8; ++c)
            vf[c] = *reinterpret_cast<const half8_t *>(vl + lds_value_offset(j, kg >> 1, kg & 1, c * 16 + row));
#pragma unroll
        for (int c = 0; c < 8; ++c) {
#pragma unroll
            for (int ct = 0; ct < 2; ++ct) o[ct][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(pa[ct][j], vf[c], o[ct][c], 0, 0, 0);
        }
#pragma unroll
        for (int ct = 0; ct < 2; ++ct) o[ct][8] = __builtin_amdgcn_mfma_f32_16x16x32_f16(pa[ct][j], ones, o[ct][8], 0, 0, 0);
    };

    // The f32 entry point's weights and P.V for pair j: each weight p as the
    // pair hi = fp16(p), lo = fp16(p - hi) (p - hi is exact in f32), so the
    // weights keep ~22 bits instead of 11; P.V and the row sums take hi, then
    // lo, over one read of the value fragments.
    auto pv_mfma_hi_lo = [&](const uint16_t *vl, int j, const Scores &x, const float (&ms)[2]) {
        half8_t hi[2], lo[2];
#pragma unroll
        for (int ct = 0; ct < 2; ++ct)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float pf = __builtin_amdgcn_exp2f(__builtin_fmaf(x[ct][j][e], scale, -ms[ct]));
                hi[ct][e] = to_h(pf);
                lo[ct][e] = to_h(pf - static_cast<float>(hi[ct][e]));
            }
        half8_t vf[8];
#pragma unroll
        for (int c = 0; c < 8; ++c)
            vf[c] = *reinterpret_cast<const half8_t *>(vl + lds_value_offset(j, kg >> 1, kg & 1, c * 16 + row));
#pragma unroll
        for (int pass = 0; pass < 2; ++pass) {
#pragma unroll
            for (int c = 0; c < 8; ++c) {
#pragma unroll
                for (int ct = 0; ct < 2; ++ct)
                    o[ct][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(pass ? lo[ct] : hi[ct], vf[c], o[ct][c], 0, 0, 0);
            }
#pragma unroll
            for (int ct = 0; ct < 2; ++ct)
                o[ct][8] = __builtin_amdgcn_mfma_f32_16x16x32_f16(pass ? lo[ct] : hi[ct], ones, o[ct][8], 0, 0, 0);
        }
    };

    // Software pipeline: while the score MFMAs of step i+1 run, the VALU
    // exponentiates step i (and rescales O when the reference moved); while
    // P.V of step i runs, it masks step i+1 and takes its max.
    // K stays one step ahead of V through LDS: step i (parity i & 1) reads
    // K(i+1) from sk[(i+1)&1] and V(i) from sv[i&1], and at its start loads
    // K(i+2) into sk[i&1] and V(i+1) into sv[(i+1)&1] (both freed by step
    // i-1), waited for at its closing barrier.
    dma_k(s_begin, sk0, lane);
    dma_v(s_begin, sv0, lane);
    dma_k(s_begin + 1, sk1, lane);
    __syncthreads();
    Scores xa, xb;
    float m_run[2], ms[2], alpha[2] = {1.f, 1.f};
    bool rescale = false;
    {
        scores(sk0, xa);
        if (needs_mask(s_begin)) apply_mask(s_begin, xa);  // uniform: only the block's last step
        const float minus_inf[2] = {-INFINITY, -INFINITY};
        column_max(xa, minus_inf, m_run);  // finite: key 0 <= every query token
    }
    __syncthreads();  // every wave has read sk[0] before step 0 stores K(2) there

    // Step i of the unit (block step s_begin + i).  more: a step i+1 exists
    // (its scores are computed here); mask_next: step i+1 is the block's last
    // step, the only one that reaches the diagonal or the end of the sequence
    // (query blocks are 16-aligned inside 64-key steps), so the mask stays out
    // of the main loop.  K(i+2) is loaded when more && !mask_next (a unit that
    // is not the block's last part loads one step past its end, never read).  The main loop passes compile-time
    // flags (one straight-line region, buffers known at compile time); the
    // last steps pass runtime flags.
    auto step_body = [&](auto more, auto mask_next, auto odd, int i, Scores &xc, Scores &xn, int ln) {
        uint16_t *k_read = odd ? sk0 : sk1;  // K(i+1)
        uint16_t *k_load = odd ? sk1 : sk0;  // K(i+2)
        uint16_t *v_read = odd ? sv1 : sv0;  // V(i)
        uint16_t *v_load = odd ? sv0 : sv1;  // V(i+1)
        if (rescale) {  // uniform: some column's max moved in step i
#pragma unroll
            for (int ct = 0; ct < 2; ++ct)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float a = __shfl(alpha[ct], kg * 4 + r);
#pragma unroll
                    for (int c = 0; c < 9; ++c) o[ct][c][r] *= a;
                }
        }
        if (more && !mask_next) dma_k(s_begin + i + 2, k_load, ln);
        if (more) dma_v(s_begin + i + 1, v_load, ln);
#pragma unroll
        for (int ct = 0; ct < 2; ++ct) ms[ct] = m_run[ct] * scale;
        half8_t pa[2][2];
        if constexpr (F32IO) {
            // The f32 entry point: weights as hi + lo fp16 pairs, one tile
            // pair at a time (pv_mfma_hi_lo), before the scores of step i+1
            // (with both steps' scores live the registers run out).
            __builtin_amdgcn_s_setprio(1);
            pv_mfma_hi_lo(v_read, 0, xc, ms);
            pv_mfma_hi_lo(v_read, 1, xc, ms);
            __builtin_amdgcn_s_setprio(0);
            if (more) scores(k_read, xn);
        } else {
            // scores of step i+1 | P of step i, pair 0
            if (more) scores(k_read, xn);
            probs(xc, ms, 0, pa);
            probs(xc, ms, 1, pa);
            // P.V of both pairs | mask and max of step i+1.  The P.V MFMAs run at
            // raised wave priority, so the SIMD's other wave fills the gaps with
            // its VALU work.
            __builtin_amdgcn_s_setprio(1);
            pv_mfma(v_read, 0, pa);
            pv_mfma(v_read, 1, pa);
            __builtin_amdgcn_s_setprio(0);
        }
        if (more) {
            if (mask_next) apply_mask(s_begin + i + 1, xn);
            // Lazy rescale: m_run is the exponent reference of the column,
            // and it moves (with O and the row sums rescaled) only when the
            // column's maximum exceeds it by more than kLazyRescaleLog2;
            // until then every weight 2^(s - m_run) stays below 2^8, exact
            // in fp16 and far from f32 overflow in the sums.  O / l is the
            // same quotient whatever the reference, and the split merge
            // takes m_run as the reference its part used.
            float m_new[2];
            column_max(xn, m_run, m_new);
            bool far = false;
#pragma unroll
            for (int ct = 0; ct < 2; ++ct) far |= (m_new[ct] - m_run[ct]) * scale > kLazyRescaleLog2;
            rescale = __any(far);
            if (rescale) {  // uniform
#pragma unroll
                for (int ct = 0; ct < 2; ++ct) {
                    alpha[ct] = __builtin_amdgcn_exp2f((m_run[ct] - m_new[ct]) * scale);
                    m_run[ct] = m_new[ct];
                }
            }
        }
        __syncthreads();  // waits for this wave's loads into LDS, then for every wave
    };
    const std::integral_constant<bool, true> yes;
    const std::integral_constant<bool, false> no;
    int i = 0;
    for (; i + 3 < steps; i += 2) {
        step_body(yes, no, no, i, xa, xb, lane);
        step_body(yes, no, yes, i + 1, xb, xa, lane);
    }
    // The last steps and the epilogue take their lane coordinates from a lane
    // id computed here (mbcnt), a value the compiler cannot merge with the one
    // computed before the main loop.  Otherwise it computes their per-lane
    // addresses before the main loop, where they share the loop's registers
    // and are spilled around it.
    const int tail_lane = static_cast<int>(__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)));
    for (; i < steps; ++i) {  // the last one to three steps
        if (i + 1 == steps && last_part && t0 + kQueryBlock > n) {  // uniform: the block's tokens end inside a cache block
            // V(i) has landed; its tokens past the prompt are zeroed in LDS
            // (value_keep): one tile a round, half and dim by thread.
            uint16_t *vl = (i & 1) != 0 ? sv1 : sv0;
            const int half = wave >> 1, dim = (wave & 1) * 64 + tail_lane;
#pragma unroll
            for (int tile = 0; tile < kStepTiles; ++tile) {
                const int key = (s_begin + i) * kKeyStep + tile * 16 + half * 8;
                u32x4_t *v = reinterpret_cast<u32x4_t *>(vl + lds_value_offset(tile >> 1, tile & 1, half, dim));
                if (key + 8 > n) *v &= value_keep(key, n);
            }
            __syncthreads();
        }
        step_body(i + 1 < steps, i + 2 == steps && last_part, (i & 1) != 0, i, xa, xb, tail_lane);
#pragma unroll
        for (int ct = 0; ct < 2; ++ct)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int e = 0; e < 8; ++e) xa[ct][j][e] = xb[ct][j][e];
    }

    const int lane_e = tail_lane, row_e = tail_lane & 15, kg_e = tail_lane >> 4;
    if (nparts > 1) {
        // Split block: store this part's (m, O, l), count it, and let the part
        // that arrives last merge the other one.  Partials move as 8-byte
        // relaxed agent-scope atomics (coherent across the XCDs' L2s); every
        // store of the workgroup completes before thread 0 counts the arrival.
        // The second part first reads the count: when the first part has
        // arrived (its workgroup runs it before its light block, so it
        // usually has), its stores are complete, and the second part merges
        // it without storing its own (the first part's count is then the
        // last it touches).  Slab of a part: O/l tiles [wave][ct][tile][half]
        // [lane] as float pairs, then m [wave][ct][lane].
        const uint32_t item = pair * kKvHeads + g;  // the heavy block of the pair
        auto slab = [&](uint32_t q) {
            return reinterpret_cast<uint64_t *>(p.partials + (static_cast<size_t>(item) * 2 + q) * kPrefillPartialFloats);
        };
        auto pair_idx = [&](int ct, int c, int hf) { return (((wave * 2 + ct) * 9 + c) * 2 + hf) * 64 + lane_e; };
        auto m_ptr = [&](uint32_t q, int ct) {
            return p.partials + (static_cast<size_t>(item) * 2 + q) * kPrefillPartialFloats + 4 * 2 * 9 * 4 * 64 +
                   (wave * 2 + ct) * 64 + lane_e;
        };
        bool merge_now = false;
        if (part == 1) {
            if (wave == 0 && lane_e == 0)
                sm_last = __hip_atomic_load(p.counters + item, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 1u;
            __syncthreads();
            merge_now = sm_last;  // uniform
            __syncthreads();      // every wave has read it before it is written again below
        }
        if (!merge_now) {
            uint64_t *own = slab(part);
#pragma unroll
            for (int ct = 0; ct < 2; ++ct) {
#pragma unroll
                for (int c = 0; c < 9; ++c)
#pragma unroll
                    for (int hf = 0; hf < 2; ++hf) {
                        const uint64_t bits = static_cast<uint64_t>(__float_as_uint(o[ct][c][2 * hf])) |
                                              (static_cast<uint64_t>(__float_as_uint(o[ct][c][2 * hf + 1])) << 32);
                        __hip_atomic_store(own + pair_idx(ct, c, hf), bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    }
                __hip_atomic_store(m_ptr(part, ct), m_run[ct], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
            if (wave == 0 && lane_e == 0) {
                const uint32_t prev =
                    __hip_atomic_fetch_add(p.counters + item, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                sm_last = prev == nparts - 1;
            }
            __syncthreads();
            if (!sm_last) return;  // uniform: the other part merges and writes the block
        }
        const uint32_t q = part ^ 1u;  // two parts
        const uint64_t *other = slab(q);
#pragma unroll
        for (int ct = 0; ct < 2; ++ct) {
            const float mo = __hip_atomic_load(m_ptr(q, ct), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            float4_t ov[9];
#pragma unroll
            for (int c = 0; c < 9; ++c)
#pragma unroll
                for (int hf = 0; hf < 2; ++hf) {
                    const uint64_t bits = __hip_atomic_load(other + pair_idx(ct, c, hf), __ATOMIC_RELAXED,
                                                            __HIP_MEMORY_SCOPE_AGENT);
                    ov[c][2 * hf] = __uint_as_float(static_cast<uint32_t>(bits));
                    ov[c][2 * hf + 1] = __uint_as_float(static_cast<uint32_t>(bits >> 32));
                }
            const float m_new = fmaxf(m_run[ct], mo);
            const float a_self = __builtin_amdgcn_exp2f((m_run[ct] - m_new) * scale);
            const float a_other = __builtin_amdgcn_exp2f((mo - m_new) * scale);
            m_run[ct] = m_new;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float as = __shfl(a_self, kg_e * 4 + r);
                const float ao = __shfl(a_other, kg_e * 4 + r);
#pragma unroll
                for (int c = 0; c < 9; ++c) o[ct][c][r] = o[ct][c][r] * as + ov[c][r] * ao;
            }
        }
        if (wave == 0 && lane_e == 0)
            __hip_atomic_store(p.counters + item, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }

    // Normalise: output row kg*4 + r of tile ct is query token t0 + kg*4 + r;
    // its row sum is element r of the sums tile in the same lane.  Each wave
    // stages its two heads' 16 x 128 outputs in its own K/V buffer (free after
    // the last step: no load into LDS is in flight) as [head][token][dim],
    // then stores whole 16-byte chunks (8 fp16 or 4 f32 outputs) instead of
    // one 2- or 4-byte element per lane and store.
    using OutT = std::conditional_t<F32IO, float, uint16_t>;
    constexpr int kChunk = 16 / static_cast<int>(sizeof(OutT));  // outputs per 16-byte chunk
    static_assert(2 * kQueryBlock * kHeadDim * sizeof(OutT) <= sizeof(sk0),
                  "a wave's two staged 16 x 128 output tiles fit its own K/V buffer");
    OutT *stage =reinterpret_cast<OutT *>(wave == 0 ? sk0 : wave == 1 ? sk1 : wave == 2 ? sv0 : sv1);
#pragma unroll
    for (int ct = 0; ct < 2; ++ct) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float inv = 1.0f / o[ct][8][r];
            OutT *srow = stage + (ct * kQueryBlock + kg_e * 4 + r) * kHeadDim + row_e;
#pragma unroll
            for (int c = 0; c < 8; ++c) {
                if constexpr (F32IO) srow[c * 16] = o[ct][c][r] * inv;
                else srow[c * 16] = __builtin_bit_cast(uint16_t, to_h(o[ct][c][r] * inv));
            }
        }
    }
    __builtin_amdgcn_wave_barrier();  // the wave reads what its other lanes wrote (LDS is in order per wave)
    constexpr int kChunks = 2 * kQueryBlock * kHeadDim / kChunk;  // of the wave: 512 (fp16) or 1024 (f32)
#pragma unroll
    for (int j = 0; j < kChunks / 64; ++j) {
        const int q = j * 64 + lane_e;                   // chunk: [head][token][chunk of the row]
        const int ct = q / (kQueryBlock * kHeadDim / kChunk);
        const int tt = (q / (kHeadDim / kChunk)) % kQueryBlock, d0 = (q % (kHeadDim / kChunk)) * kChunk;
        const int t = t0 + tt, h = static_cast<int>(g) * kGroup + wave * 2 + ct;
        if (t < n) {
            const float4_t v = *reinterpret_cast<const float4_t *>(stage + (ct * kQueryBlock + tt) * kHeadDim + d0);
            OutT *dst = (F32IO ? reinterpret_cast<OutT *>(p.out32) : reinterpret_cast<OutT *>(p.out)) +
                        (static_cast<size_t>(t) * kQueryHeads + h) * kHeadDim + d0;
            *reinterpret_cast<float4_t *>(dst) = v;
        }
    }
    // Every wave has read its staged outputs before the next segment loads
    // its first stages into these buffers.
    __syncthreads();
  };
  // the first part of a heavy block, then a light block (two inlined
  // copies: each is register-allocated like a single segment)
  if (nseg > 0) run_segment(seg0);
  if (nseg > 1) run_segment(seg1);
}

// CT query heads x 16 query tokens per workgroup, KG waves: wave w takes the
// 32-key steps w, w + KG, .. of the block.  Per step a lane loads its key
// fragments (2 score MFMAs x 4 dim slices, 16 bytes each, in runs of 128
// bytes) and value fragments (8 x 16 bytes) of one pair of cache tiles
// straight into registers, in the operand order of the cache layout; the next
// step's keys are issued behind this step's score MFMAs and its values behind
// P.V, so each has most of a step to arrive, and nothing in the loop waits for
// another wave.  Every wave keeps its own softmax reference; the waves merge
// in LDS.
//
// What bounds it: short prompts by latency (launch, the first loads, the
// merge; 2 to 4 steps a wave), longer ones by the compute unit's load path:
// every wave loads all its keys and values, 16 KiB for 34 MFMAs (544 clocks)
// at 64 bytes per clock.  That is why prompts beyond kPrefillWaveTokens share
// them through LDS when they have the workspace to split their long blocks.
// One workgroup per (query block, kv head), as before, kept at most 2 ceil(N /
// 16) compute units busy, each for the block's whole length: N=211 f16 16.4 ->
// 9.2 us, 1157 37.5 -> 22.2 (f32 46.8 -> 26.2), 2048 60.2 -> 39.1 (74.7 ->
// 46.5); without a workspace 4096 109 -> 100 (141 -> 124), 8192 385 -> 347
// (both kernels' launches included).
//
// Workgroup b: kv head b % 2, then the head set, then the query blocks from
// the last (longest) to the first.  The 16 / CT workgroups of a query block
// are a multiple of the 8 XCDs, so each XCD reads the keys and values of one
// kv head only.
template <bool F32IO, int CT, int KG>
__global__ __launch_bounds__(KG * 64, 2) void prefill_wave_attention_kernel(PrefillParams p) {
    constexpr int kHeadSets = kGroup / CT;
    constexpr int kWaveStep = 32;  // keys per step: one pair of cache tiles
    const int n = static_cast<int>(p.tokens);
    const int qblocks = (n + kQueryBlock - 1) / kQueryBlock;
    const uint32_t g = blockIdx.x & 1u;
    const int hs = static_cast<int>((blockIdx.x >> 1) % kHeadSets);
    const int qb = qblocks - 1 - static_cast<int>((blockIdx.x >> 1) / kHeadSets);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int row = lane & 15, kg = lane >> 4;
    const int t0 = qb * kQueryBlock, my_token = t0 + row;
    const int nkeys = min(t0 + kQueryBlock, n), last_tile = (nkeys - 1) >> 4;
    const int steps = (nkeys + kWaveStep - 1) / kWaveStep;
    const int h0 = static_cast<int>(g) * kGroup + hs * CT;  // first query head

    // Block ids of the wave's tiles, one per lane: lane 2 i + j holds tile j
    // of the wave's step i0 + i (32 steps a load; a clamped tile past the
    // end).  Optional arrays are read through the query pointer when they are
    // not given (at least as long), so no load sits behind a branch.
    const int32_t *stand_in = F32IO ? reinterpret_cast<const int32_t *>(p.query32) : reinterpret_cast<const int32_t *>(p.query);
    const int32_t *table = p.block_table ? p.block_table : stand_in;
    auto tile_of = [&](int i0) { return min(2 * (wave + (i0 + (lane >> 1)) * KG) + (lane & 1), last_tile); };
    auto tile_id = [&](int t, int32_t b) -> uint32_t {  // an id outside the planes reads block 0
        if (p.block_table == nullptr) b = t;
        return b >= 0 && static_cast<uint32_t>(b) < p.num_blocks ? static_cast<uint32_t>(b) : 0u;
    };
    const int tq = min(my_token, n - 1);
    const int32_t id_raw = table[tile_of(0)], pos_raw = (p.positions ? p.positions : stand_in)[tq];
    __builtin_amdgcn_sched_barrier(0);

    // Raw query: the CT x 2 pairs of 32-dim slices (kb, kb + 2) of a head,
    // which rotate together, are shared out over the waves.
    constexpr int kItems = CT * 2, kMine = (kItems + KG - 1) / KG;
    typedef std::conditional_t<F32IO, float4_t, half8_t> Raw;
    constexpr int kRawLoads = F32IO ? 2 : 1, kRawElems = F32IO ? 4 : 8;
    Raw raw[kMine][2][kRawLoads];
#pragma unroll
    for (int it = 0; it < kMine; ++it) {
        const int item = min(wave + it * KG, kItems - 1);
        const size_t qoff = (static_cast<size_t>(tq) * kQueryHeads + h0 + (item >> 1)) * kHeadDim + (item & 1) * 32 + kg * 8;
#pragma unroll
        for (int k2 = 0; k2 < 2; ++k2)
#pragma unroll
            for (int f = 0; f < kRawLoads; ++f) {
                const size_t at = qoff + k2 * 64 + f * kRawElems;
                if constexpr (F32IO) raw[it][k2][f] = *reinterpret_cast<const Raw *>(p.query32 + at);
                else raw[it][k2][f] = *reinterpret_cast<const Raw *>(p.query + at);
            }
    }
    __builtin_amdgcn_sched_barrier(0);
    uint32_t ids = tile_id(tile_of(0), id_raw);
    const int qpos = p.positions ? pos_raw : tq;
    const bool qrope = p.rope_cos != nullptr && qpos >= 0 && static_cast<uint32_t>(qpos) < p.rope_rows;
    float4_t qc[kMine][2], qs[kMine][2];
    {
        const float *cr = qrope ? p.rope_cos + static_cast<size_t>(qpos) * 64 : reinterpret_cast<const float *>(stand_in);
        const float *sr = qrope ? p.rope_sin + static_cast<size_t>(qpos) * 64 : reinterpret_cast<const float *>(stand_in);
#pragma unroll
        for (int it = 0; it < kMine; ++it) {
            const int d0 = (min(wave + it * KG, kItems - 1) & 1) * 32 + kg * 8;
#pragma unroll
            for (int f = 0; f < 2; ++f) {
                qc[it][f] = *reinterpret_cast<const float4_t *>(cr + d0 + f * 4);
                qs[it][f] = *reinterpret_cast<const float4_t *>(sr + d0 + f * 4);
            }
        }
    }
    half8_t kf[2][4], vf[8];
    auto id_of = [&](int i, int j) {
        return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(ids), 2 * (i & 31) + j));
    };
    auto load_k = [&](int i) {
        const uint32_t b0 = id_of(i, 0), b1 = id_of(i, 1);
        const uint16_t *src = p.key_cache + (static_cast<size_t>(row < 8 ? b0 : b1) * kKvHeads + g) * kBlockHeadElems;
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int kb = 0; kb < 4; ++kb)
                kf[h][kb] = *reinterpret_cast<const half8_t *>(src + (kb * 4 + kg) * 128 + (h * 8 + (row & 7)) * 8);
    };
    auto load_v = [&](int i) {
        const uint32_t b0 = id_of(i, 0), b1 = id_of(i, 1);
        const uint16_t *src = p.value_cache + (static_cast<size_t>(kg < 2 ? b0 : b1) * kKvHeads + g) * kBlockHeadElems;
#pragma unroll
        for (int c = 0; c < 8; ++c)
            vf[c] = *reinterpret_cast<const half8_t *>(src + (c * 16 + row) * 16 + (kg & 1) * 8);
    };
    load_k(0);
    __builtin_amdgcn_sched_barrier(0);
    load_v(0);
    __builtin_amdgcn_sched_barrier(0);

    // Rotate (exactly as rotate_chunk does) while the keys and values are in
    // flight, and share the query fragments (B operand: column = token t0 +
    // row, dims kb*32 + kg*8 .. +8) through LDS.
    constexpr int kRow = kHeadDim + 4;  // padded against bank conflicts
    __shared__ float sm_m[KG][CT * 16], sm_l[KG][CT * 16];
    __shared__ __align__(16) float sm_o[KG][CT * 16][kRow];
    half8_t *sm_q = reinterpret_cast<half8_t *>(&sm_o[0][0][0]);  // [head][kb][lane], before the merge
    static_assert(CT * 4 * 64 * sizeof(half8_t) <= sizeof(sm_o), "the query fragments fit the merge buffer");
#pragma unroll
    for (int it = 0; it < kMine; ++it) {
        const int item = wave + it * KG;
        if (item < kItems) {
            half8_t q[2];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const float c = qc[it][j >> 2][j & 3], sn = qs[it][j >> 2][j & 3];
                const float x = static_cast<float>(raw[it][0][j / kRawElems][j % kRawElems]);
                const float y = static_cast<float>(raw[it][1][j / kRawElems][j % kRawElems]);
                q[0][j] = to_h(qrope ? x * c + (-y) * sn : x);
                q[1][j] = to_h(qrope ? y * c + x * sn : y);
            }
            sm_q[((item >> 1) * 4 + (item & 1)) * 64 + lane] = q[0];
            sm_q[((item >> 1) * 4 + (item & 1) + 2) * 64 + lane] = q[1];
        }
    }
    // (fences limited to LDS: the key and value loads stay in flight)
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    half8_t qf[CT][4];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) qf[ct][kb] = sm_q[(ct * 4 + kb) * 64 + lane];

    float4_t o[CT][9];  // 8 column tiles of the output, then the row sums
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int c = 0; c < 9; ++c) o[ct][c] = float4_t{0.f, 0.f, 0.f, 0.f};
    half8_t ones;
#pragma unroll
    for (int e = 0; e < 8; ++e) ones[e] = static_cast<_Float16>(1.0f);
    const float scale = p.scale_log2;
    float m_run[CT];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) m_run[ct] = -INFINITY;
    // Maximum over the 4 lanes of a column (l, l ^ 16, l ^ 32, l ^ 48).
    auto column_max = [](float c) {
        typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
        u32x2 v = __builtin_amdgcn_permlane16_swap(__float_as_uint(c), __float_as_uint(c), false, false);
        c = fmaxf(__uint_as_float(v[0]), __uint_as_float(v[1]));
        v = __builtin_amdgcn_permlane32_swap(__float_as_uint(c), __float_as_uint(c), false, false);
        return fmaxf(__uint_as_float(v[0]), __uint_as_float(v[1]));
    };

    // Step s, the wave's i-th.  The block's last step is the only one that
    // reaches the diagonal or the end of the sequence; it has code of its own
    // (last, compile time), since the compiler made its masks unconditional in a
    // common loop: 500 tokens f16 10.46 us a call there, 10.18 here (10.36 with
    // the masks of the scores only), 2900 tokens 56.9, 55.9 (56.5).
    auto step = [&](auto last, int s, int i) __attribute__((always_inline)) {
        // The last step of a 32-step block of ids loads the next 32.
        if (!last && ((i + 1) & 31) == 0 && s + KG < steps) ids = tile_id(tile_of(i + 1), table[tile_of(i + 1)]);
        // Scores: MFMA h leaves lane (column = query token, kg) the keys
        // (kg & 1)*8 + h*4 + r of the pair's tile kg >> 1.
        float x[CT][8];
        {
            float4_t acc[CT][2];
#pragma unroll
            for (int ct = 0; ct < CT; ++ct)
#pragma unroll
                for (int h = 0; h < 2; ++h) acc[ct][h] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int kb = 0; kb < 4; ++kb)
#pragma unroll
                for (int ct = 0; ct < CT; ++ct)
#pragma unroll
                    for (int h = 0; h < 2; ++h)
                        acc[ct][h] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[h][kb], qf[ct][kb], acc[ct][h], 0, 0, 0);
#pragma unroll
            for (int ct = 0; ct < CT; ++ct)
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int r = 0; r < 4; ++r) x[ct][h * 4 + r] = acc[ct][h][r];
        }
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (!last) load_k(i + 1);  // past the wave's last step: a clamped tile, never used
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (last) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int key = s * kWaveStep + (kg >> 1) * 16 + (kg & 1) * 8 + e;
                const bool keep = key <= my_token && key < n;
#pragma unroll
                for (int ct = 0; ct < CT; ++ct) x[ct][e] = keep ? x[ct][e] : -INFINITY;
            }
            if (t0 + kQueryBlock > n) {  // uniform: the last cache block is partly filled
                const u32x4_t keep = value_keep(s * kWaveStep + kg * 8, n);
#pragma unroll
                for (int c = 0; c < 8; ++c) vf[c] = __builtin_bit_cast(half8_t, __builtin_bit_cast(u32x4_t, vf[c]) & keep);
            }
        }
        // Lazy rescale, as in prefill_attention_kernel: the reference moves
        // when a column's maximum passes it by more than kLazyRescaleLog2
        // (the first step sets it).
        bool far = false;
        float m_new[CT];
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
            float c = m_run[ct];
#pragma unroll
            for (int e = 0; e < 8; ++e) c = fmaxf(c, x[ct][e]);
            m_new[ct] = column_max(c);
            far |= (m_new[ct] - m_run[ct]) * scale > kLazyRescaleLog2;
        }
        if (__any(far)) {  // uniform
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) {
                const float alpha = __builtin_amdgcn_exp2f((m_run[ct] - m_new[ct]) * scale);
                m_run[ct] = m_new[ct];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float a = __shfl(alpha, kg * 4 + r);
#pragma unroll
                    for (int c = 0; c < 9; ++c) o[ct][c][r] *= a;
                }
            }
        }
        // P in fp16; the f32 entry point's weights as the pair hi = fp16(p),
        // lo = fp16(p - hi) (exact in f32).  A column whose scores are all
        // -infinity so far has weights 0.
        half8_t hi[CT], lo[CT];
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
            const float ms = m_run[ct] == -INFINITY ? 0.f : m_run[ct] * scale;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float pf = __builtin_amdgcn_exp2f(__builtin_fmaf(x[ct][e], scale, -ms));
                hi[ct][e] = to_h(pf);
                if constexpr (F32IO) lo[ct][e] = to_h(pf - static_cast<float>(hi[ct][e]));
            }
        }
#pragma unroll
        for (int pass = 0; pass < (F32IO ? 2 : 1); ++pass) {
#pragma unroll
            for (int c = 0; c < 8; ++c)
#pragma unroll
                for (int ct = 0; ct < CT; ++ct)
                    o[ct][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(pass ? lo[ct] : hi[ct], vf[c], o[ct][c], 0, 0, 0);
#pragma unroll
            for (int ct = 0; ct < CT; ++ct)
                o[ct][8] = __builtin_amdgcn_mfma_f32_16x16x32_f16(pass ? lo[ct] : hi[ct], ones, o[ct][8], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (!last) load_v(i + 1);
        __builtin_amdgcn_sched_barrier(0);
    };
    const std::integral_constant<bool, true> yes;
    const std::integral_constant<bool, false> no;
    int s = wave, i = 0;
    for (; s + 1 < steps; s += KG, ++i) step(no, s, i);
    if (s + 1 == steps) step(yes, s, i);  // uniform: the wave that the last step falls to

    // Merge: every wave scales its O and row sums to the common maximum (a
    // wave without steps holds zeros at -infinity) and stores them; then the
    // workgroup adds the waves in order, normalises and stores 16-byte chunks.
    if (kg == 0) {
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) sm_m[wave][ct * 16 + row] = m_run[ct];
    }
    __syncthreads();  // and every wave has read the query fragments
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
        float m = sm_m[0][ct * 16 + row];
#pragma unroll
        for (int w = 1; w < KG; ++w) m = fmaxf(m, sm_m[w][ct * 16 + row]);
        const float alpha = __builtin_amdgcn_exp2f((m_run[ct] - m) * scale);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float a = __shfl(alpha, kg * 4 + r);
            float *dst = sm_o[wave][ct * 16 + kg * 4 + r] + row;
#pragma unroll
            for (int c = 0; c < 8; ++c) dst[c * 16] = o[ct][c][r] * a;
            if (row == 0) sm_l[wave][ct * 16 + kg * 4 + r] = o[ct][8][r] * a;
        }
    }
    __syncthreads();
    constexpr int kPer = F32IO ? 4 : 8;  // outputs per 16-byte chunk
    constexpr int kRowChunks = kHeadDim / kPer, kChunks = CT * 16 * kRowChunks;
    static_assert(kChunks % (KG * 64) == 0, "every thread stores the same number of chunks");
#pragma unroll
    for (int j = 0; j < kChunks / (KG * 64); ++j) {
        const int q = j * (KG * 64) + static_cast<int>(threadIdx.x);  // chunk: [token][head][chunk of the row]
        const int d0 = q % kRowChunks * kPer, tt = q / kRowChunks / CT, ct = q / kRowChunks % CT;
        const int r = ct * 16 + tt, t = t0 + tt;
        float l = 0.f;
        float4_t v[kPer / 4];
#pragma unroll
        for (int e = 0; e < kPer / 4; ++e) v[e] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < KG; ++w) {
            l += sm_l[w][r];
#pragma unroll
            for (int e = 0; e < kPer / 4; ++e) v[e] += *reinterpret_cast<const float4_t *>(&sm_o[w][r][d0 + e * 4]);
        }
        const float inv = 1.0f / l;
        if (t < n) {
            const size_t off = (static_cast<size_t>(t) * kQueryHeads + h0 + ct) * kHeadDim + d0;
            if constexpr (F32IO) {
                *reinterpret_cast<float4_t *>(p.out32 + off) = v[0] * inv;
            } else {
                half8_t h;
#pragma unroll
                for (int e = 0; e < 8; ++e) h[e] = to_h(v[e >> 2][e & 3] * inv);
                *reinterpret_cast<half8_t *>(p.out + off) = h;
            }
        }
    }
}

// Prompts of at most kPrefillShortTokens in one launch: append and attention
// together.  A workgroup takes one head of a 16-token query block, and wave w
// its 32-key step w, so there is no loop.  Keys and values come from the
// call's own rows, not from the cache that another workgroup is writing: each
// wave rotates and rounds its keys in registers (the same arithmetic, hence
// the same bits, as the append kernel), its values pass through LDS into P.V
// operand order, and the first head of each group stores the query block's
// own rows into the cache.
//
// What bounds it: latency (the launch; positions and rows; cos and sin; the
// merge), and from three steps on the compute unit's load path: rows and angles
// of a step are 32 KiB, in lines half used, for every head and later query
// block again.  Two launches pay that once, and a launch gap.  us a call, one
// launch / two (f16, then f32): 16 tokens 5.1 / 7.7, 5.4 / 7.8; 64 tokens 5.7 /
// 7.5, 6.3 / 7.7; 96 tokens 6.5 / 7.6, 7.4 / 7.9; 128 tokens 7.3 / 7.6, 8.4 /
// 8.0; 211 tokens 11.1 / 8.1, 13.0 / 9.0.
constexpr uint32_t kPrefillShortTokens = 96;
constexpr int kShortWaves = 4;  // the last one has no keys: with the one before it, it rotates the query
static_assert(kPrefillShortTokens <= kShortWaves * 32, "a wave for each step");

template <bool F32IO>
__global__ __launch_bounds__(kShortWaves * 64, 2) void prefill_short_kernel(PrefillParams p) {
    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    constexpr int KG = kShortWaves;
    const int n = static_cast<int>(p.tokens);
    const int qblocks = (n + kQueryBlock - 1) / kQueryBlock;
    const uint32_t g = blockIdx.x & 1u;
    const int hs = static_cast<int>((blockIdx.x >> 1) % kGroup);
    const int qb = qblocks - 1 - static_cast<int>((blockIdx.x >> 1) / kGroup);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int row = lane & 15, kg = lane >> 4;
    const int t0 = qb * kQueryBlock, my_token = t0 + row;
    const int steps = (qb + 2) >> 1, k0 = wave * 32;  // 32-key steps of the block; first key of this wave's
    const bool live = wave < steps;                   // uniform
    const int h0 = static_cast<int>(g) * kGroup + hs;

    constexpr int kRow = kHeadDim + 4;  // padded against bank conflicts
    __shared__ float sm_m[KG][16], sm_l[KG][16];
    __shared__ __align__(16) half8_t sm_q[4 * 64];  // [kb][lane]
    // a wave's values [32 tokens][kRow fp16], then (behind a barrier) its O [16][kRow f32]
    __shared__ __align__(16) float sm_o[KG][16][kRow];
    uint32_t *sm_v = reinterpret_cast<uint32_t *>(&sm_o[wave][0][0]);

    typedef std::conditional_t<F32IO, float4_t, half8_t> Raw;
    constexpr int kRawLoads = F32IO ? 2 : 1, kRawElems = F32IO ? 4 : 8;
    auto raw_load = [&](const float *src32, const uint16_t *src, size_t at, Raw (&dst)[kRawLoads]) {
#pragma unroll
        for (int f = 0; f < kRawLoads; ++f) {
            if constexpr (F32IO) dst[f] = *reinterpret_cast<const Raw *>(src32 + at + f * kRawElems);
            else dst[f] = *reinterpret_cast<const Raw *>(src + at);
        }
    };
    // Lane (row, kg) holds, for score MFMA h, the key in slot h * 8 + row % 8
    // of tile row / 8 of the step, dims kb * 32 + kg * 8 .. +8 (as load_k of
    // prefill_wave_attention_kernel); tokens past the end repeat the last one.
    // Optional arrays are read through the query when not given, so that no
    // load waits behind a branch.
    const int32_t *stand_in = F32IO ? reinterpret_cast<const int32_t *>(p.query32) : reinterpret_cast<const int32_t *>(p.query);
    const int key_tile = 2 * wave + (row >> 3);
    int kt[2], kpos_raw[2];
    const int tq = min(my_token, n - 1);
    const int qpos_raw = (p.positions ? p.positions : stand_in)[tq];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        kt[h] = min(key_tile * 16 + key_slot(h * 8 + (row & 7)), n - 1);
        kpos_raw[h] = (p.positions ? p.positions : stand_in)[kt[h]];
    }
    const int32_t id_raw = load_const(p.block_table ? p.block_table : stand_in, static_cast<uint32_t>(qb));
    const float *stand_in32 = reinterpret_cast<const float *>(stand_in);
    auto rope_at = [&](int raw, int t, bool *rope) {
        const int pos = p.positions ? raw : t;
        *rope = p.rope_cos != nullptr && pos >= 0 && static_cast<uint32_t>(pos) < p.rope_rows;
        return static_cast<size_t>(pos) * 64;
    };
    auto rotate_pair = [&](const Raw (&a)[kRawLoads], const Raw (&b)[kRawLoads], const float4_t *cs, const float4_t *sn,
                           bool rope, half8_t *lo, half8_t *hi) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float x = static_cast<float>(a[j / kRawElems][j % kRawElems]);
            const float y = static_cast<float>(b[j / kRawElems][j % kRawElems]);
            const float co = cs[j >> 2][j & 3], si = sn[j >> 2][j & 3];
            (*lo)[j] = to_h(rope ? x * co + (-y) * si : x);
            (*hi)[j] = to_h(rope ? y * co + x * si : y);
        }
        if constexpr (!F32IO) {
            if (!rope) {  // as given, bit for bit
                *lo = a[0];
                *hi = b[0];
            }
        }
    };
    half8_t kf[2][4];
    bool krope[2] = {true, true};
    if (live) {
        Raw kr[2][4][kRawLoads], vr[8][kRawLoads];
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int kb = 0; kb < 4; ++kb)
                raw_load(p.key32, p.key, (static_cast<size_t>(kt[h]) * kKvHeads + g) * kHeadDim + kb * 32 + kg * 8, kr[h][kb]);
#pragma unroll
        for (int j = 0; j < 8; ++j)  // value pieces: token j * 4 + kg of the step, 16 bytes `row` of its fp16 row
            raw_load(p.value32, p.value, (static_cast<size_t>(min(k0 + j * 4 + kg, n - 1)) * kKvHeads + g) * kHeadDim + row * 8, vr[j]);
        float4_t kc[2][2][2], ks[2][2][2];  // [h][dims hk * 32 + kg * 8 .. +8]
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const size_t at = rope_at(kpos_raw[h], kt[h], &krope[h]);
            const float *cr = krope[h] ? p.rope_cos + at : stand_in32, *sr = krope[h] ? p.rope_sin + at : stand_in32;
#pragma unroll
            for (int hk = 0; hk < 2; ++hk)
#pragma unroll
                for (int f = 0; f < 2; ++f) {
                    kc[h][hk][f] = *reinterpret_cast<const float4_t *>(cr + hk * 32 + kg * 8 + f * 4);
                    ks[h][hk][f] = *reinterpret_cast<const float4_t *>(sr + hk * 32 + kg * 8 + f * 4);
                }
        }
        __builtin_amdgcn_sched_barrier(0);  // every load ahead of the arithmetic
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            half8_t v;
            if constexpr (F32IO) {
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] = to_h(vr[j][e / kRawElems][e % kRawElems]);
            } else {
                v = vr[j][0];
            }
            const u32x4 w = __builtin_bit_cast(u32x4, v);
            u32x2 *dst = reinterpret_cast<u32x2 *>(sm_v + (j * 4 + kg) * (kRow / 2) + row * 4);  // 8-byte aligned
            dst[0] = u32x2{w[0], w[1]};
            dst[1] = u32x2{w[2], w[3]};
        }
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
                rotate_pair(kr[h][kb], kr[h][kb + 2], kc[h][kb], ks[h][kb], krope[h], &kf[h][kb], &kf[h][kb + 2]);
    }
    // Query fragments (B operand: column = token t0 + row, dims kb * 32 + kg *
    // 8 .. +8): the last two waves, most often without keys, take one rotary
    // pair (kb, kb + 2) each.
    if (wave >= KG - 2) {  // uniform
        const int kb = wave - (KG - 2);
        const size_t at = (static_cast<size_t>(tq) * kQueryHeads + h0) * kHeadDim + kb * 32 + kg * 8;
        Raw a[kRawLoads], b[kRawLoads];
        raw_load(p.query32, p.query, at, a);
        raw_load(p.query32, p.query, at + 64, b);
        bool rope;
        const size_t tab = rope_at(qpos_raw, tq, &rope);
        const float *cr = rope ? p.rope_cos + tab : stand_in32, *sr = rope ? p.rope_sin + tab : stand_in32;
        float4_t cs[2], sn[2];
#pragma unroll
        for (int f = 0; f < 2; ++f) {
            cs[f] = *reinterpret_cast<const float4_t *>(cr + kb * 32 + kg * 8 + f * 4);
            sn[f] = *reinterpret_cast<const float4_t *>(sr + kb * 32 + kg * 8 + f * 4);
        }
        half8_t lo, hi;
        rotate_pair(a, b, cs, sn, rope, &lo, &hi);
        sm_q[kb * 64 + lane] = lo;
        sm_q[(kb + 2) * 64 + lane] = hi;
    }
    __syncthreads();

    float4_t o[9];  // dims (c / 2) * 32 + 2 * row + c % 2 of 8 column tiles, then the row sums
#pragma unroll
    for (int c = 0; c < 9; ++c) o[c] = float4_t{0.f, 0.f, 0.f, 0.f};
    const float scale = p.scale_log2;
    float m_run = -INFINITY;
    if (live) {
        float4_t acc[2] = {float4_t{0.f, 0.f, 0.f, 0.f}, float4_t{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) {
            const half8_t qf = sm_q[kb * 64 + lane];
#pragma unroll
            for (int h = 0; h < 2; ++h) acc[h] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[h][kb], qf, acc[h], 0, 0, 0);
        }
        float x[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int key = k0 + kg * 8 + e;
            x[e] = key <= my_token && key < n ? acc[e >> 2][e & 3] : -INFINITY;
            m_run = fmaxf(m_run, x[e]);
        }
        {  // over the 4 lanes of a column
            u32x2 v = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane16_swap(__float_as_uint(m_run), __float_as_uint(m_run), false, false));
            m_run = fmaxf(__uint_as_float(v[0]), __uint_as_float(v[1]));
            v = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane32_swap(__float_as_uint(m_run), __float_as_uint(m_run), false, false));
            m_run = fmaxf(__uint_as_float(v[0]), __uint_as_float(v[1]));
        }
        const float ms = m_run == -INFINITY ? 0.f : m_run * scale;
        half8_t hi, lo, ones;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float pf = __builtin_amdgcn_exp2f(__builtin_fmaf(x[e], scale, -ms));
            hi[e] = to_h(pf);
            lo[e] = F32IO ? to_h(pf - static_cast<float>(hi[e])) : static_cast<_Float16>(0.0f);
            ones[e] = static_cast<_Float16>(1.0f);
        }
        // The query block's own rows into the cache, from the workgroup of the
        // group's first head: keys as they lie in kf, values as in vf below.
        const bool writer = hs == 0 && wave == steps - 1;  // uniform
        const int32_t id = p.block_table ? id_raw : static_cast<int32_t>(qb);
        const bool ok = id >= 0 && static_cast<uint32_t>(id) < p.num_blocks;
        const size_t slab = (static_cast<size_t>(ok ? id : 0) * kKvHeads + g) * kBlockHeadElems;
        if (writer && key_tile == qb) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int slot = h * 8 + (row & 7);
                if (qb * 16 + key_slot(slot) >= n) continue;
                if (p.error_word && kg == 0 && !krope[h] && p.rope_cos != nullptr) atomicOr(p.error_word, 4u);
                if (!ok) continue;
#pragma unroll
                for (int kb = 0; kb < 4; ++kb)
                    *reinterpret_cast<half8_t *>(p.key_cache + slab + (kb * 4 + kg) * 128 + slot * 8) = kf[h][kb];
            }
        }
        if (writer && !ok && lane == 0 && p.error_word) atomicOr(p.error_word, 2u);
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            // keys kg * 8 .. +8 of dims c * 32 + 2 * row and the next: 32 banks
            // apart over kg, one dword each over row
            uint32_t d[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) d[e] = sm_v[(kg * 8 + e) * (kRow / 2) + c * 16 + row];
            u32x4 even, odd;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                even[e] = (d[2 * e] & 0xffffu) | (d[2 * e + 1] << 16);
                odd[e] = (d[2 * e] >> 16) | (d[2 * e + 1] & 0xffff0000u);
            }
            const half8_t vf[2] = {__builtin_bit_cast(half8_t, even), __builtin_bit_cast(half8_t, odd)};
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                o[2 * c + i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(hi, vf[i], o[2 * c + i], 0, 0, 0);
                if constexpr (F32IO) o[2 * c + i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(lo, vf[i], o[2 * c + i], 0, 0, 0);
            }
            if (writer && ok && 2 * wave + (kg >> 1) == qb) {
                const int left = n - (qb * 16 + (kg & 1) * 8);  // tokens of this half
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    uint16_t *dst = p.value_cache + slab + (c * 32 + 2 * row + i) * 16 + (kg & 1) * 8;
                    if (left >= 8) {
                        *reinterpret_cast<half8_t *>(dst) = vf[i];
                    } else {
#pragma unroll
                        for (int e = 0; e < 8; ++e)
                            if (e < left) dst[e] = __builtin_bit_cast(uint16_t, static_cast<_Float16>(vf[i][e]));
                    }
                }
            }
        }
        o[8] = __builtin_amdgcn_mfma_f32_16x16x32_f16(hi, ones, o[8], 0, 0, 0);
        if constexpr (F32IO) o[8] = __builtin_amdgcn_mfma_f32_16x16x32_f16(lo, ones, o[8], 0, 0, 0);
    }

    // Merge, as in prefill_wave_attention_kernel (waves without a step are left out).
    if (kg == 0) sm_m[wave][row] = m_run;
    __syncthreads();  // and every wave has read its values
    if (live) {
        float m = sm_m[0][row];
        for (int w = 1; w < steps; ++w) m = fmaxf(m, sm_m[w][row]);
        const float alpha = __builtin_amdgcn_exp2f((m_run - m) * scale);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float a = __shfl(alpha, kg * 4 + r);
            float *dst = sm_o[wave][kg * 4 + r] + 2 * row;
#pragma unroll
            for (int c = 0; c < 8; ++c) dst[(c >> 1) * 32 + (c & 1)] = o[c][r] * a;
            if (row == 0) sm_l[wave][kg * 4 + r] = o[8][r] * a;
        }
    }
    __syncthreads();
    constexpr int kChunks = kQueryBlock * kHeadDim / 4;  // of 4 outputs
    static_assert(kChunks % (KG * 64) == 0, "every thread stores the same number of chunks");
#pragma unroll
    for (int j = 0; j < kChunks / (KG * 64); ++j) {
        const int q = j * (KG * 64) + static_cast<int>(threadIdx.x), r = q / (kHeadDim / 4), d0 = q % (kHeadDim / 4) * 4, t = t0 + r;
        float l = 0.f;
        float4_t v = float4_t{0.f, 0.f, 0.f, 0.f};
        for (int w = 0; w < steps; ++w) {
            l += sm_l[w][r];
            v += *reinterpret_cast<const float4_t *>(&sm_o[w][r][d0]);
        }
        if (t < n) {
            const float inv = 1.0f / l;
            const size_t off = (static_cast<size_t>(t) * kQueryHeads + h0) * kHeadDim + d0;
            if constexpr (F32IO) {
                *reinterpret_cast<float4_t *>(p.out32 + off) = v * inv;
            } else {
                typedef _Float16 half4 __attribute__((ext_vector_type(4)));
                half4 h;
#pragma unroll
                for (int e = 0; e < 4; ++e) h[e] = to_h(v[e] * inv);
                *reinterpret_cast<half4 *>(p.out + off) = h;
            }
        }
    }
}

// Whether the call's key and value rows lie apart from everything the
// one-launch form writes while other workgroups still read them.
bool rows_apart(const PrefillParams &p, bool f32) {
    const size_t bytes = f32 ? 4 : 2, rows = p.tokens * size_t{kRowElems} * bytes;
    const size_t plane = static_cast<size_t>(p.num_blocks) * kKvHeads * kBlockHeadElems * 2;
    auto apart = [](const void *a, size_t an, const void *b, size_t bn) {
        const uintptr_t x = reinterpret_cast<uintptr_t>(a), y = reinterpret_cast<uintptr_t>(b);
        return x + an <= y || y + bn <= x;
    };
    const void *out = f32 ? static_cast<const void *>(p.out32) : p.out;
    for (const void *in : {f32 ? static_cast<const void *>(p.key32) : p.key, f32 ? static_cast<const void *>(p.value32) : p.value})
        if (!apart(in, rows, out, rows / kKvHeads * kQueryHeads) || !apart(in, rows, p.key_cache, plane) ||
            !apart(in, rows, p.value_cache, plane))
            return false;
    return true;
}

}  // namespace

int launch_prefill(const pvlc_hip_paged_prefill_args *a, void *stream, const PrefillOperands32 *f32) {
    PrefillParams p{};
    p.tokens = a->tokens;
    p.num_blocks = a->num_blocks;
    p.block_table = a->block_table;
    p.key_cache = a->key_cache;
    p.value_cache = a->value_cache;
    p.query = a->query;
    p.key = a->key;
    p.value = a->value;
    p.out = a->out;
    p.rope_cos = a->rope_cos;
    p.rope_sin = a->rope_sin;
    p.rope_rows = a->rope_rows;
    p.positions = a->positions;
    p.qrot = a->query_scratch;
    p.error_word = a->error_word;
    p.scale_log2 = kLog2e / sqrtf(static_cast<float>(kHeadDim));
    if (f32) {
        p.query32 = f32->query;
        p.key32 = f32->key;
        p.value32 = f32->value;
        p.out32 = f32->out;
    }
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (a->tokens <= kPrefillShortTokens && a->query_scratch == nullptr && rows_apart(p, f32 != nullptr)) {
        const dim3 grid((a->tokens + kQueryBlock - 1) / kQueryBlock * kQueryHeads), threads(kShortWaves * 64);
        if (f32) hipLaunchKernelGGL(prefill_short_kernel<true>, grid, threads, 0, st, p);
        else hipLaunchKernelGGL(prefill_short_kernel<false>, grid, threads, 0, st, p);
        return static_cast<int>(hipGetLastError());
    }
    const bool paired = a->workspace != nullptr && a->tokens > kPrefillWaveTokens;
    if (paired) {
        const PrefillWorkspace ws = prefill_workspace_layout(a->tokens);
        p.counters = static_cast<uint32_t *>(a->workspace);
        p.partials = reinterpret_cast<float *>(static_cast<unsigned char *>(a->workspace) + ws.partial_offset);
    }
    const dim3 append_grid((a->tokens + kBlockTokens - 1) / kBlockTokens);
    if (f32) hipLaunchKernelGGL(prefill_rope_append_kernel<true>, append_grid, dim3(kAppendThreads), 0, st, p);
    else hipLaunchKernelGGL(prefill_rope_append_kernel<false>, append_grid, dim3(kAppendThreads), 0, st, p);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return static_cast<int>(e);
    const unsigned qblocks = (a->tokens + kQueryBlock - 1) / kQueryBlock;
    if (!paired) {
        // 1 head and 2 waves a workgroup while the prompt is short (16
        // workgroups a query block), 2 heads and 4 waves beyond.  N=211 f16:
        // 9.2 us against 10.5, 700: 14.5 against 14.8, 1157: 24.5 against
        // 22.2 (f32: 10.4 / 12.0, 16.7 / 17.7, 27.8 / 26.2).
        const bool one = a->tokens <= kPrefillOneHeadTokens;
        const dim3 grid(qblocks * kKvHeads * kGroup / (one ? 1 : 2)), threads(one ? 128 : 256);
        if (one) {
            if (f32) hipLaunchKernelGGL((prefill_wave_attention_kernel<true, 1, 2>), grid, threads, 0, st, p);
            else hipLaunchKernelGGL((prefill_wave_attention_kernel<false, 1, 2>), grid, threads, 0, st, p);
        } else {
            if (f32) hipLaunchKernelGGL((prefill_wave_attention_kernel<true, 2, 4>), grid, threads, 0, st, p);
            else hipLaunchKernelGGL((prefill_wave_attention_kernel<false, 2, 4>), grid, threads, 0, st, p);
        }
        return static_cast<int>(hipGetLastError());
    }
    const unsigned grid = prefill_pair_workgroups(qblocks);
    if (f32) hipLaunchKernelGGL(prefill_attention_kernel<true>, dim3(grid), dim3(kWaves * 64), 0, st, p);
    else hipLaunchKernelGGL(prefill_attention_kernel<false>, dim3(grid), dim3(kWaves * 64), 0, st, p);
    return static_cast<int>(hipGetLastError());
}

}  // namespace pvlc
