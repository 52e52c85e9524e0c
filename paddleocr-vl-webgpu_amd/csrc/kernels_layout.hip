// Bit-exact moves between the compact reference rows [tokens][2][128] (the
// cache planes of DecoderKvSessionDescriptor, runtime-core lib.rs:833-843) and
// the blocked device layout (see pvlc_hip.h), through a block table.

#include <hip/hip_runtime.h>

#include <cstdint>

#include "pvlc_internal.hpp"

namespace pvlc {
namespace {

typedef uint16_t u16x8_t __attribute__((ext_vector_type(8)));
// The same in global memory: rows and planes need only their elements'
// alignment, so the 16-byte accesses must not assume more (the instructions are
// those of aligned ones: the target allows unaligned global accesses).
typedef u16x8_t u16x8_any __attribute__((aligned(2)));

// Both kernels: one workgroup per 16-token cache block, both heads, with the
// block transposed through LDS, so that the rows (32 lanes on the 512 bytes of
// a token) and the slabs (a wave on 1 KiB) move in 16-byte vectors on
// contiguous runs on either side.  A thread per (token, head, chunk) without
// LDS scattered the values 2 bytes at a time on the cache side.  They are
// bound by latency for a few thousand tokens (loads, LDS, stores) and by memory
// beyond: 5003 tokens 13.1 -> 8.6 us for the pair of calls (two launches from
// the host are 8.2 of it), 65536 tokens, four prefixes in turn, 100.6 -> 47.2.
// There a pack takes 27.2 us (4.9 TB/s, what a large copy reaches) and the pair
// less than twice that, since the unpack finds part of the planes in the
// Infinity Cache; one prefix over and over, which fits there, 84.9 -> 40.9.
constexpr int kMoveThreads = 256;
constexpr int kValuePad = 8;  // elements after each 256-dim LDS row, against bank conflicts

// Block of tile b through the table (false: an id outside the planes).
__device__ inline bool table_block(const int32_t *table, uint32_t b, uint32_t num_blocks, uint32_t *blk) {
    const int32_t id = table ? table[b] : static_cast<int32_t>(b);
    *blk = static_cast<uint32_t>(id);
    return id >= 0 && static_cast<uint32_t>(id) < num_blocks;
}

// Key piece k (0..511) of a block's slabs, 16 bytes: head k / 256, chunk (k /
// 16) % 16, slot k % 16.  Row piece k: token k / 32, head (k / 16) % 2, chunk
// k % 16.
__device__ inline int key_piece(int token, int head, int chunk) { return head * 256 + chunk * 16 + key_slot(token); }

__global__ __launch_bounds__(kMoveThreads) void kv_pack_kernel(
    const uint16_t *__restrict__ key_rows, const uint16_t *__restrict__ value_rows, uint32_t tokens,
    const int32_t *__restrict__ table, uint32_t num_blocks, uint16_t *__restrict__ key_cache,
    uint16_t *__restrict__ value_cache, uint32_t *__restrict__ error_word) {
    __shared__ __align__(16) u16x8_t sk[2 * kMoveThreads];
    __shared__ __align__(16) uint16_t sv[kBlockTokens][kRowElems + kValuePad];
    const int i = threadIdx.x;
    const uint32_t t0 = blockIdx.x * kBlockTokens, ntok = min(tokens - t0, kBlockTokens);
    uint32_t blk;
    const bool ok = table_block(table, blockIdx.x, num_blocks, &blk);
    u16x8_t kr[2], vr[2];
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        const int k = i + r * kMoveThreads;  // row piece; tokens past the end repeat the last one
        const size_t src = static_cast<size_t>(t0 + min(static_cast<uint32_t>(k >> 5), ntok - 1)) * kRowElems + (k & 31) * 8;
        kr[r] = *reinterpret_cast<const u16x8_any *>(key_rows + src);
        vr[r] = *reinterpret_cast<const u16x8_any *>(value_rows + src);
    }
    if (!ok) {  // uniform
        if (i == 0 && error_word) atomicOr(error_word, 2u);
        return;
    }
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        const int k = i + r * kMoveThreads;
        sk[key_piece(k >> 5, (k >> 4) & 1, k & 15)] = kr[r];
        *reinterpret_cast<u16x8_t *>(&sv[k >> 5][(k & 31) * 8]) = vr[r];
    }
    __syncthreads();
    const size_t block = static_cast<size_t>(blk) * kKvHeads * kBlockHeadElems;
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        const int k = i + r * kMoveThreads;  // slab piece; the other tokens of a partial block stay as they are
        if (static_cast<uint32_t>(key_slot(k & 15)) < ntok)  // (the slot map is its own inverse)
            *reinterpret_cast<u16x8_any *>(key_cache + block + static_cast<size_t>(k) * 8) = sk[k];
    }
    // value slab row i = (head, dim): 16 tokens
    uint16_t *dst = value_cache + block + static_cast<size_t>(i) * kBlockTokens;
    if (ntok == kBlockTokens) {
        u16x8_t lo, hi;
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            lo[t] = sv[t][i];
            hi[t] = sv[t + 8][i];
        }
        *reinterpret_cast<u16x8_any *>(dst) = lo;
        *reinterpret_cast<u16x8_any *>(dst + 8) = hi;
    } else {
        for (uint32_t t = 0; t < ntok; ++t) dst[t] = sv[t][i];
    }
}

// The values of a block in LDS, as dwords of two tokens: token pair p (0..7)
// of row d = (head, dim) (0..255).  16-byte pieces of a 128-byte line and the
// dwords of a piece are exchanged by the row's chunk c = d / 8, so that the 32
// lanes that read one (d % 8, p) of 32 chunks fall on 32 banks.
__device__ inline int value_piece(int d, int half) { return (d * 2 + half) ^ ((d >> 3) & 7); }
__device__ inline int value_dword(int d, int p) { return value_piece(d, p >> 2) * 4 + ((p & 3) ^ ((d >> 6) & 3)); }

__global__ __launch_bounds__(kMoveThreads) void kv_unpack_kernel(
    const uint16_t *__restrict__ key_cache, const uint16_t *__restrict__ value_cache, uint32_t tokens,
    const int32_t *__restrict__ table, uint32_t num_blocks, uint16_t *__restrict__ key_rows,
    uint16_t *__restrict__ value_rows) {
    typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
    __shared__ __align__(16) u16x8_t sk[2 * kMoveThreads];
    __shared__ __align__(16) uint32_t sv[kRowElems * kBlockTokens / 2];
    const int i = threadIdx.x;
    const uint32_t t0 = blockIdx.x * kBlockTokens, ntok = min(tokens - t0, kBlockTokens);
    uint32_t blk;
    const bool ok = table_block(table, blockIdx.x, num_blocks, &blk);
    if (ok) {  // uniform
        const size_t block = static_cast<size_t>(blk) * kKvHeads * kBlockHeadElems;
        u16x8_t kr[2];
        u32x4_t vr[2];
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            const size_t k = i + r * kMoveThreads;
            kr[r] = *reinterpret_cast<const u16x8_any *>(key_cache + block + k * 8);
            vr[r] = __builtin_bit_cast(u32x4_t, static_cast<u16x8_t>(*reinterpret_cast<const u16x8_any *>(value_cache + block + k * 8)));
        }
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            const int k = i + r * kMoveThreads, d = k >> 1;  // value piece: row d, token half k % 2
            sk[k] = kr[r];
            u32x4_t v = vr[r];
            if (d & 64) v = __builtin_shufflevector(v, v, 1, 0, 3, 2);
            if (d & 128) v = __builtin_shufflevector(v, v, 2, 3, 0, 1);
            *reinterpret_cast<u32x4_t *>(&sv[value_piece(d, k & 1) * 4]) = v;
        }
    }
    __syncthreads();
    // Key row pieces: token k / 32, 16 bytes k % 32 of its row.
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        const int k = i + r * kMoveThreads, t = k >> 5;
        if (static_cast<uint32_t>(t) >= ntok) continue;
        u16x8_t kv{};
        if (ok) kv = sk[key_piece(t, (k >> 4) & 1, k & 15)];
        *reinterpret_cast<u16x8_any *>(key_rows + static_cast<size_t>(t0 + t) * kRowElems + (k & 31) * 8) = kv;
    }
    // Value row pieces, two tokens a thread: pair i / 32, 16 bytes i % 32.
    const int p = i >> 5, c = i & 31;
    u16x8_t even{}, odd{};
    if (ok) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const uint32_t two = sv[value_dword(c * 8 + j, p)];
            even[j] = static_cast<uint16_t>(two);
            odd[j] = static_cast<uint16_t>(two >> 16);
        }
    }
    uint16_t *dst = value_rows + static_cast<size_t>(t0 + 2 * p) * kRowElems + c * 8;
    if (static_cast<uint32_t>(2 * p) < ntok) *reinterpret_cast<u16x8_any *>(dst) = even;
    if (static_cast<uint32_t>(2 * p + 1) < ntok) *reinterpret_cast<u16x8_any *>(dst + kRowElems) = odd;
}

}  // namespace

int launch_kv_pack(const uint16_t *key_rows, const uint16_t *value_rows, uint32_t tokens, const int32_t *table,
                   uint32_t num_blocks, uint16_t *key_cache, uint16_t *value_cache, uint32_t *error_word,
                   void *stream) {
    if (tokens == 0) return 0;
    hipLaunchKernelGGL(kv_pack_kernel, dim3(tokens / kBlockTokens + (tokens % kBlockTokens != 0)), dim3(kMoveThreads), 0,
                       static_cast<hipStream_t>(stream), key_rows, value_rows, tokens, table, num_blocks, key_cache, value_cache, error_word);
    return static_cast<int>(hipGetLastError());
}

int launch_kv_unpack(const uint16_t *key_cache, const uint16_t *value_cache, uint32_t tokens, const int32_t *table,
                     uint32_t num_blocks, uint16_t *key_rows, uint16_t *value_rows, void *stream) {
    if (tokens == 0) return 0;
    hipLaunchKernelGGL(kv_unpack_kernel, dim3(tokens / kBlockTokens + (tokens % kBlockTokens != 0)), dim3(kMoveThreads), 0,
                       static_cast<hipStream_t>(stream), key_cache, value_cache, tokens, table, num_blocks, key_rows, value_rows);
    return static_cast<int>(hipGetLastError());
}

}  // namespace pvlc
