// Prefill projection with fp16 weights for gfx950: out[r][n] = sum_k in[r][k]
// * W[n][k] + bias[n], f32 activations, fp16 weights output-major, f32 bias
// and output.  Replaces linear_projection_f16_weights (crates/pvlc-wgsl/src/
// lib.rs:1836-1964), which widens the weights and accumulates in f32
// (arithmetic reference: linear_f32, crates/pvlc-cpu-ref/src/lib.rs:88-140).
//
// The products run on MFMA without giving up f32 activations: each input row
// is scaled by a power of two 2^-e (so its largest element lies in
// [2^13, 2^14)) and split exactly into fp16 hi + fp16 lo (lo = the f32
// remainder, rounded), so hi + lo carries about 22 bits of every element.
// Two fp16 MFMAs per product (W.hi + W.lo, exact products, f32 accumulation)
// then give f32-grade sums at half the fp16 MFMA rate; the epilogue multiplies
// by 2^e (exact) and adds the bias.
//
// Kernel 1 (split): one workgroup per 8 rows: the row maxima, the exponents,
// and the hi/lo planes written in the GEMM's tile order (per 128-row tile and
// 32-wide k step one 16 KiB block [plane][k-chunk (4)][row (128)][8]), so a
// GEMM stage of the activations is one contiguous 16 KiB run.
// Kernel 2 (GEMM): one template from 128 x 192 down to 16 x 16 output tiles;
// the host picks the tile by the measured times of a compute unit's first tile
// and its further ones (choose_projection_tile).  The waves of
// a workgroup own rows of the tile (activation fragments straight from the
// planes into registers, no byte read twice) and share its weight columns,
// which move by direct global-to-LDS loads in whole 128-byte lines; small
// tiles split the depth over groups of waves.

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "pvlc_device.hpp"
#include "pvlc_internal.hpp"

namespace pvlc {
namespace {

constexpr int kSplitThreads = 256;
constexpr int kSplitRows = 8;  // rows per split workgroup: 8 x 16 bytes = one 128-byte line per chunk
constexpr int kTileM = kProjectionTileRows, kTileK = kProjectionStepK;
constexpr int kTileElems = kTileM * kTileK;  // fp16 elements of one 128 x 32 operand tile
constexpr int kBlockElems = 2 * kTileElems;  // one activation block: hi and lo planes
// s_waitcnt immediate (gfx9 encoding: vmcnt bits 3:0 and 15:14, expcnt 6:4,
// lgkmcnt 11:8) -- as builtins, so the compiler's own wait insertion knows
// which loads they retire.
constexpr int wait_vm(int n) { return 0x0F70 | (n & 15) | ((n >> 4) << 14); }  // vmcnt(n), lgkmcnt left at its maximum
constexpr int kLgkm0 = ~0x0F00;                                                 // mask: lgkmcnt(0) as well

// Exponent e of a row whose largest magnitude is m: m * 2^-e in [2^13, 2^14)
// (0 for an all-zero row).
__device__ inline int split_exponent(float m) {
    if (!(m > 0.f)) return 0;
    int x;
    (void)__builtin_frexpf(m, &x);  // m = f * 2^x, f in [0.5, 1)
    return x - 14;
}

// Offset (fp16 elements) of row r, k-chunk c (8 elements) in the tile-ordered
// planes: block (r / 128, c / 4), plane hi; lo is kTileElems further.
__device__ inline size_t plane_offset(uint32_t r, uint32_t c, uint32_t steps) {
    const size_t block = static_cast<size_t>(r / kTileM) * steps + c / 4;
    return block * kBlockElems + ((c % 4) * kTileM + r % kTileM) * 8;
}

// Thread t of the workgroup serves row 8 g + t % 8 and the k-chunks t / 8 +
// 32 i; the 8 threads of one chunk write one whole 128-byte line of each
// plane.  Rows past the end (padding of the last tile) are written as zeros.
// CPT > 0: K = 256 CPT, the thread's CPT chunks stay in registers between the
// row maximum and the split (one pass over the input); CPT = 0: any K that is
// a multiple of 32, the chunks are read again for the split.
template <int CPT>
__global__ __launch_bounds__(kSplitThreads) void projection_split_kernel(const float *__restrict__ input,
                                                                        uint32_t rows, uint32_t k_width,
                                                                        uint16_t *__restrict__ tiles,
                                                                        int32_t *__restrict__ exponents) {
    const uint32_t rr = threadIdx.x % kSplitRows, c0 = threadIdx.x / kSplitRows;
    constexpr uint32_t kChunkStride = kSplitThreads / kSplitRows;
    const uint32_t row = blockIdx.x * kSplitRows + rr, chunks = k_width / 8, steps = k_width / kTileK;
    const bool live = row < rows;
    const float *in = input + static_cast<size_t>(live ? row : 0) * k_width;
    auto load = [&](uint32_t c, float4_t &a, float4_t &b) {
        a = *reinterpret_cast<const float4_t *>(in + c * 8);
        b = *reinterpret_cast<const float4_t *>(in + c * 8 + 4);
    };
    auto chunk_max = [](float m, const float4_t &a, const float4_t &b) {
#pragma unroll
        for (int j = 0; j < 4; ++j) m = fmaxf(m, fmaxf(fabsf(a[j]), fabsf(b[j])));
        return m;
    };
    float m = 0.f;
    float4_t va[CPT > 0 ? CPT : 1], vb[CPT > 0 ? CPT : 1];
    if constexpr (CPT > 0) {
        // Padding rows read row 0 (every load unconditional) and are zeroed below.
#pragma unroll
        for (int i = 0; i < CPT; ++i) load(c0 + i * kChunkStride, va[i], vb[i]);
#pragma unroll
        for (int i = 0; i < CPT; ++i) m = chunk_max(m, va[i], vb[i]);
        if (!live) m = 0.f;
    } else if (live) {
        for (uint32_t c = c0; c < chunks; c += kChunkStride) {
            float4_t a, b;
            load(c, a, b);
            m = chunk_max(m, a, b);
        }
    }
    // Lanes of one row differ in lane bits 3..5; then the 4 waves.
#pragma unroll
    for (int o = 8; o < 64; o <<= 1) m = fmaxf(m, __shfl_xor(m, o));
    __shared__ float sm_max[kSplitThreads / 64][kSplitRows];
    if ((threadIdx.x & 63) < kSplitRows) sm_max[threadIdx.x >> 6][rr] = m;
    __syncthreads();
    m = fmaxf(fmaxf(sm_max[0][rr], sm_max[1][rr]), fmaxf(sm_max[2][rr], sm_max[3][rr]));
    const int e = split_exponent(m);
    if (threadIdx.x < kSplitRows) exponents[row] = e;
    auto split_store = [&](uint32_t c, const float4_t &a, const float4_t &b) {
        half8_t h, l;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float s = live ? __builtin_ldexpf(j < 4 ? a[j] : b[j - 4], -e) : 0.f;  // exact: a power of two
            h[j] = to_h(s);
            l[j] = to_h(s - static_cast<float>(h[j]));  // the remainder is exact in f32
        }
        const size_t off = plane_offset(row, c, steps);
        *reinterpret_cast<half8_t *>(tiles + off) = h;
        *reinterpret_cast<half8_t *>(tiles + off + kTileElems) = l;
    };
    if constexpr (CPT > 0) {
#pragma unroll
        for (int i = 0; i < CPT; ++i) split_store(c0 + i * kChunkStride, va[i], vb[i]);
    } else {
        for (uint32_t c = c0; c < chunks; c += kChunkStride) {
            float4_t a = {0.f, 0.f, 0.f, 0.f}, b = a;
            if (live) load(c, a, b);
            split_store(c, a, b);
        }
    }
}

// Calls f(integral_constant<U>) for U = B .. E-1 (compile-time ring indices).
template <int B, int E> struct StageUnroll {
    template <class F> __device__ __forceinline__ static void run(F &&f) {
        f(std::integral_constant<int, B>{});
        StageUnroll<B + 1, E>::run(f);
    }
};
template <int E> struct StageUnroll<E, E> {
    template <class F> __device__ __forceinline__ static void run(F &&) {}
};

// Slot U of the weight ring: distinct LDS arrays (one function-scope array
// per instantiation), so the compiler sees that loads into one slot and
// fragment reads of another do not alias and adds no wait of its own.
template <int U, int ELEMS> __device__ __forceinline__ uint16_t *weight_ring() {
    __shared__ __align__(16) uint16_t buf[ELEMS];
    return buf;
}

// Tile order.  Workgroup b runs on XCD b % 8, so XCD x takes the workgroups
// b = 8 i + x and, with them, one block of the output: the row tiles split
// into 8 / col_groups bands and the column tiles into col_groups bands.
// Inside the block, generations of `gen` columns: all row tiles of the block
// for columns [g gen, g gen + gen), row-major, so the workgroups resident at
// once share both operands in the XCD's L2.
__device__ inline bool ordered_tile(const ProjectionOrder &o, uint32_t b, uint32_t *mt, uint32_t *nt) {
    const uint32_t x = b % kXcds, idx = b / kXcds;
    const uint32_t row_groups = kXcds / o.col_groups;
    const uint32_t xr = x / o.col_groups, xc = x % o.col_groups;
    const uint32_t r0 = xr * o.row_tiles / row_groups, r1 = (xr + 1) * o.row_tiles / row_groups;
    const uint32_t c0 = xc * o.col_tiles / o.col_groups, c1 = (xc + 1) * o.col_tiles / o.col_groups;
    const uint32_t rb = r1 - r0, cb = c1 - c0;
    if (idx >= rb * cb) return false;
    const uint32_t gen = o.gen < cb ? o.gen : cb;
    const uint32_t span = rb * gen, full = cb / gen;
    uint32_t g, rem, w;
    if (idx < full * span) {
        g = idx / span;
        rem = idx % span;
        w = gen;
    } else {
        g = full;
        rem = idx - full * span;
        w = cb - full * gen;
    }
    *mt = r0 + rem / w;
    *nt = c0 + g * gen + rem % w;
    return true;
}

// (16 RB RW) x (16 CB) output tiles, RW x KG waves.
//
// K group g of KG walks its share of the depth in stages of 64; wave rw of
// the group owns rows rw 16 RB .. of the tile and every column: per 32-deep
// half stage it multiplies RB (hi, lo) activation fragments with CB weight
// fragments.  The activation fragments come straight from the planes (16 rows
// x 8 k are one 256-byte run) into a ring of AD register sets; no other wave
// reads them.  The weights of a stage (16 CB rows x 128 bytes) are shared by
// the group's RW waves through a ring of S LDS slots.
//
// Why 64-deep weight stages: a weight row is then read in whole 128-byte
// lines.  With 32-deep stages every load took half a line, and the compute
// unit's load path moves lines: L2-resident reads of 16 rows x 64 bytes
// measured 17 TB/s device-wide against 33 for 8 rows x 128 bytes (direct to
// LDS or to registers alike), which bound the 128 x 256 and 128 x 160 tile
// kernels this one replaced.  N=4096, one projection repeated back to back
// with its split kernel, before -> now: q|k|v 55-58 -> 48-50 us, o 50-51 -> 44-45,
// gate|up 115-118 -> 93-94 (1.1 PFLOP/s of MFMAs, 1.2 without the split; a large
// bf16 library product reaches 1.4), down 68-69 -> 62-63; the four in order,
// whose activations come from further away, 318-322 -> 270-277.
//
// Small launches are bound by latency and by idle compute units, so their
// tiles are small and the depth is split over KG groups, whose sums are added
// through LDS in a fixed order (the result does not depend on timing).  211
// rows: q|k|v 25.8 -> 13.5 us, o 36.2 -> 13.3, gate|up 26.9 -> 16.1, down
// 47.3 -> 16.7; 16 rows: 18.5 -> 8.0, 29.0 -> 9.3, 18.4 -> 8.4, 40.4 -> 11.5.
//
// LDS slot layout [row][8 chunks of 8 k], chunk c of row r in place c ^ (r %
// 8): a load's 8 lanes still read one line, and the 8 rows of a fragment read
// fall on distinct 16-byte bank groups.  The last column tile is shifted to
// end at the last column (n_width >= 16 CB; columns of the overlap are
// computed twice, bit-identically); CB = 1 serves narrower outputs with
// clamped weight rows.
template <int RB, int RW, int CB, int KG, int S, int AD, int MIN_WAVES>
__global__ __launch_bounds__(RW *KG * 64, MIN_WAVES) void projection_gemm_kernel(
    const uint16_t *__restrict__ tiles, const int32_t *__restrict__ exponents, const uint16_t *__restrict__ weight,
    const float *__restrict__ bias, float *__restrict__ out, uint32_t rows, uint32_t k_width, uint32_t n_width,
    ProjectionOrder order) {
    typedef int int4_t __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) void *lds_ptr;
    constexpr int kTM = RB * RW * 16, kTN = CB * 16;
    constexpr int kStageElems = CB * 1024;           // one K group's weight stage: 16 CB rows x 64 k
    constexpr int kSlotElems = KG * kStageElems;
    constexpr int kWLoads = 2 * CB / RW;             // weight loads per wave and stage: 8 rows x 128 bytes each
    constexpr int kW0 = (kWLoads + 1) / 2;           // of them, issued in the stage's first half
    constexpr int kALoads = 2 * RB;                  // activation loads per half stage
    static_assert(kTileM % kTM == 0, "a row tile lies in one 128-row block of the planes");
    static_assert((2 * CB) % RW == 0, "every wave of a K group loads as much of a stage");
    static_assert(KG == 1 || (KG - 1) * RW <= 2 * KG, "one ring slot holds the partial sums of a reduction phase");
    uint32_t mt, nt;
    if (!ordered_tile(order, blockIdx.x, &mt, &nt)) return;  // uniform: a smaller block of this XCD
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int rw = wave % RW, group = wave / RW;
    const int row16 = lane & 15, kg = lane >> 4;
    const uint32_t m0 = mt * kTM + rw * (RB * 16);
    const uint32_t n0 = CB == 1 ? nt * kTN : min(nt * kTN, n_width - kTN);
    const uint32_t steps = k_width / kTileK, stages = (steps + 1) / 2;
    const uint32_t per_group = (stages + KG - 1) / KG, first = group * per_group;
    const bool odd = (steps & 1) != 0;  // the last stage has one half

    const uint16_t *a_base = tiles + static_cast<size_t>(m0 / kTileM) * steps * kBlockElems;
    const uint32_t a_lane = (kg * kTileM + m0 % kTileM + row16) * 8;
    // Lane l of a weight load fills LDS place l % 8 of row l / 8 (byte
    // offsets, which choose_projection_tile keeps within 32 bits; 8-element
    // chunks for CB = 1, within 32 bits up to a depth of 2^31, whose planes of
    // 128 rows or more would take a terabyte; w_tail for an odd last stage,
    // whose second half re-reads the first and is not used).
    const uint32_t chunk = (lane & 7) ^ (lane >> 3), unit = CB == 1 ? 1 : 16;
    uint32_t w_lane[2], w_tail[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const uint32_t r = CB == 1 ? min(j * 8 + static_cast<uint32_t>(lane >> 3), n_width - 1 - n0) : lane >> 3;
        w_lane[j] = (r * (k_width / 8) + chunk) * unit;
        w_tail[j] = (r * (k_width / 8) + (chunk & 3)) * unit;
    }
    const uint16_t *w_base = weight + static_cast<size_t>(n0) * k_width;

    struct Act {
        half8_t h[RB], l[RB];
    };
    // Loads past the end re-read the last step or stage (never used), so
    // every wave has the same loads in flight.
    auto load_a = [&](uint32_t step, Act &f) {
        const uint16_t *a = a_base + static_cast<size_t>(min(step, steps - 1)) * kBlockElems;
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
            f.h[rb] = *reinterpret_cast<const half8_t *>(a + a_lane + rb * 128);
            f.l[rb] = *reinterpret_cast<const half8_t *>(a + kTileElems + a_lane + rb * 128);
        }
    };
    auto load_w = [&](uint32_t stage, uint16_t *slot, int begin, int end) {
        const uint32_t st = min(stage, stages - 1);
        const bool tail = odd && st == stages - 1;
        const uint16_t *w = w_base + static_cast<size_t>(st) * 64;
#pragma unroll
        for (int i = begin; i < end; ++i) {
            const int j = rw * kWLoads + i, q = CB == 1 ? i : 0;
            const uint32_t lo = tail ? w_tail[q] : w_lane[q];
            const void *src;
            if constexpr (CB == 1) src = reinterpret_cast<const half8_t *>(w) + lo;
            else src = reinterpret_cast<const char *>(w + static_cast<size_t>(j) * 8 * k_width) + lo;
            __builtin_amdgcn_global_load_lds(src, (lds_ptr)(slot + group * kStageElems + j * 512), 16, 0, 0);
        }
    };

    float4_t acc[RB][CB];
#pragma unroll
    for (int a = 0; a < RB; ++a)
#pragma unroll
        for (int b = 0; b < CB; ++b) acc[a][b] = float4_t{0.f, 0.f, 0.f, 0.f};

    // Half stage H (compile time, counted from stage `t` of the group): waits
    // for its operands (the weights of a stage by vmcnt and, with several
    // waves in the group, the barrier that also frees the slot of the stage
    // before; the fragments by the compiler's own wait), reads the weight
    // fragments, issues its half of the weight loads of stage +S-1 and the
    // activation loads of half stage +AD-1, then its 2 RB CB MFMAs (16 x 16 x
    // 32: A = activations, lane row l % 16, k (l / 16) * 8 ..; B = W^T, lane
    // column l % 16, same k).  The scheduling barriers keep the loads ahead of
    // the MFMAs: left alone the compiler sinks them to the end of the stage,
    // right before the next wait.
    // Outstanding loads allowed: at a stage's start everything issued after
    // its last weight load, 2 S - 4 half stages and one half's activations.
    constexpr int kHalfLoads = kALoads + kWLoads / 2;  // (at least)
    constexpr int kWaitWeights = (2 * S - 4) * kHalfLoads + kALoads, kWaitActs = (AD - 2) * kHalfLoads;
    constexpr int kWaitStage = kWaitActs < kWaitWeights ? kWaitActs : kWaitWeights;
    static_assert(S >= 2 && AD >= 2 && kWaitActs <= 63, "vmcnt holds at most 63 outstanding loads");
    Act f[AD];
    uint32_t t = 0;
    auto half = [&](auto hc) {
        constexpr int H = decltype(hc)::value, kSlot = (H / 2) % S, kNext = (H / 2 + S - 1) % S;
        const uint32_t st = first + t + H / 2;
        if constexpr (H % 2 == 0) {
            __builtin_amdgcn_s_waitcnt(wait_vm(kWaitStage) & kLgkm0);
            if constexpr (RW > 1) __builtin_amdgcn_s_barrier();
        } else {
            __builtin_amdgcn_s_waitcnt(wait_vm(kWaitActs));
        }
        const uint16_t *sw = weight_ring<kSlot, kSlotElems>() + group * kStageElems;
        half8_t b[12];  // the first CB (a fixed size: an array whose size depends on the template arguments,
                        // captured in a generic lambda, makes hipcc's host pass drop the launch stub)
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) {
            const int r = cb * 16 + row16, c = (H % 2) * 4 + kg;
            b[cb] = *reinterpret_cast<const half8_t *>(sw + (r * 8 + (c ^ (r & 7))) * 8);
        }
        load_w(st + S - 1, weight_ring<kNext, kSlotElems>(), H % 2 ? kW0 : 0, H % 2 ? kWLoads : kW0);
        // Where the wait for a stage's weights allows no more than the activation
        // loads behind them (S = 2), the two keep this order.
        if constexpr (H % 2 == 1 && kWaitStage > (2 * S - 4) * kHalfLoads) __builtin_amdgcn_sched_barrier(0);
        load_a(2 * st + H % 2 + AD - 1, f[(H + AD - 1) % AD]);
        __builtin_amdgcn_sched_barrier(0);
        if (2 * st + H % 2 < steps) {  // uniform
#pragma unroll
            for (int rb = 0; rb < RB; ++rb) {
#pragma unroll
                for (int cb = 0; cb < CB; ++cb)
                    acc[rb][cb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(f[H % AD].h[rb], b[cb], acc[rb][cb], 0, 0, 0);
#pragma unroll
                for (int cb = 0; cb < CB; ++cb)
                    acc[rb][cb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(f[H % AD].l[rb], b[cb], acc[rb][cb], 0, 0, 0);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    StageUnroll<0, S - 1>::run([&](auto uc) {
        constexpr int U = decltype(uc)::value;
        load_w(first + U, weight_ring<U, kSlotElems>(), 0, kWLoads);
    });
    StageUnroll<0, AD - 1>::run([&](auto uc) { load_a(2 * first + decltype(uc)::value, f[decltype(uc)::value]); });
    __builtin_amdgcn_sched_barrier(0);
    // The prologue's loads are not in the loop's order: waited for here, so
    // that the compiler's counts in the loop stay those of the loop.
    __builtin_amdgcn_s_waitcnt(wait_vm(0));
    // Unrolled over the period of both rings, so slots and register sets are
    // compile-time.
    constexpr int kHalves = 2 * S % AD == 0 ? 2 * S : 2 * S * AD;
    constexpr uint32_t kPeriod = kHalves / 2;
    for (; t + kPeriod <= per_group; t += kPeriod) StageUnroll<0, kHalves>::run(half);
    StageUnroll<0, static_cast<int>(kPeriod) - 1>::run([&](auto uc) {
        constexpr int U = decltype(uc)::value;
        if (t + U < per_group) {
            half(std::integral_constant<int, 2 * U>{});
            half(std::integral_constant<int, 2 * U + 1>{});
        }
    });
    int4_t ex[RB];
    float bn[CB];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) ex[rb] = *reinterpret_cast<const int4_t *>(exponents + m0 + rb * 16 + kg * 4);
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) bn[cb] = bias[min(n0 + cb * 16 + row16, n_width - 1)];
    __builtin_amdgcn_s_waitcnt(wait_vm(0));  // no load into LDS outlives the loop
    if constexpr (KG > 1) __syncthreads();   // every wave has read its last stages: the ring is free

    // Row block rb: the groups other than its owner (rb % KG) hand their sums
    // over through ring slot rb % 2; the owner adds them in the groups' order,
    // scales by the row's 2^e (exact), adds the bias and stores.  (A slot is
    // written again two phases later, behind the barrier that its reader
    // reaches after reading.)
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
        if constexpr (KG > 1) {
            const int owner = rb % KG;
            float4_t *sums = reinterpret_cast<float4_t *>(rb & 1 ? weight_ring<1, kSlotElems>() : weight_ring<0, kSlotElems>());
            if (group != owner) {
                float4_t *mine = sums + ((group < owner ? group : group - 1) * RW + rw) * CB * 64 + lane;
#pragma unroll
                for (int cb = 0; cb < CB; ++cb) mine[cb * 64] = acc[rb][cb];
            }
            __syncthreads();
            if (group != owner) continue;  // uniform per wave; every wave reaches every barrier
#pragma unroll
            for (int g = 0; g < KG - 1; ++g)
#pragma unroll
                for (int cb = 0; cb < CB; ++cb) acc[rb][cb] += sums[((g * RW + rw) * CB + cb) * 64 + lane];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t r = m0 + rb * 16 + kg * 4 + i;
            if (r >= rows) continue;
#pragma unroll
            for (int cb = 0; cb < CB; ++cb) {
                const uint32_t n = n0 + cb * 16 + row16;
                if (n < n_width) out[static_cast<size_t>(r) * n_width + n] = __builtin_ldexpf(acc[rb][cb][i], ex[rb][i]) + bn[cb];
            }
        }
    }
}

}  // namespace

int launch_linear_projection_f16(const float *input, const uint16_t *weight, const float *bias, float *out,
                                 uint32_t rows, uint32_t k_width, uint32_t n_width, const ProjectionWorkspace &ws,
                                 void *stream) {
    hipStream_t st = static_cast<hipStream_t>(stream);
    ProjectionOrder order{};
    uint64_t block = 0;
    const int shape = choose_projection_tile(rows, k_width, n_width, &order, &block);
    if (shape < 0) return static_cast<int>(hipErrorInvalidConfiguration);  // (operands beyond any device's memory)
    const uint32_t m_tiles = (rows + kTileM - 1) / kTileM;
    const dim3 split_grid(m_tiles * (kTileM / kSplitRows));
    switch (k_width) {
    case 1024: hipLaunchKernelGGL(projection_split_kernel<4>, split_grid, dim3(kSplitThreads), 0, st, input, rows, k_width, ws.tiles, ws.exponents); break;
    case 2048: hipLaunchKernelGGL(projection_split_kernel<8>, split_grid, dim3(kSplitThreads), 0, st, input, rows, k_width, ws.tiles, ws.exponents); break;
    case 3072: hipLaunchKernelGGL(projection_split_kernel<12>, split_grid, dim3(kSplitThreads), 0, st, input, rows, k_width, ws.tiles, ws.exponents); break;
    case 4096: hipLaunchKernelGGL(projection_split_kernel<16>, split_grid, dim3(kSplitThreads), 0, st, input, rows, k_width, ws.tiles, ws.exponents); break;
    default: hipLaunchKernelGGL(projection_split_kernel<0>, split_grid, dim3(kSplitThreads), 0, st, input, rows, k_width, ws.tiles, ws.exponents); break;
    }
    if (hipError_t e = hipGetLastError()) return static_cast<int>(e);
    const dim3 grid(static_cast<uint32_t>(kXcds * block));
#define PVLC_PROJECTION_LAUNCH(I, RB, RW, CB, KG, S, AD, MW)                                                       \
    do {                                                                                                           \
        static_assert(kProjectionTiles[I].rows == (RB) * (RW) * 16 && kProjectionTiles[I].cols == (CB) * 16 &&     \
                      kProjectionTiles[I].threads == (RW) * (KG) * 64, "the tile that choose_projection_tile weighed"); \
        hipLaunchKernelGGL((projection_gemm_kernel<RB, RW, CB, KG, S, AD, MW>), grid, dim3((RW) * (KG) * 64), 0, st, \
                           ws.tiles, ws.exponents, weight, bias, out, rows, k_width, n_width, order);              \
    } while (0)
    switch (shape) {  // kProjectionTiles
    case 0: PVLC_PROJECTION_LAUNCH(0, 2, 4, 12, 1, 3, 3, 2); break;
    case 1: PVLC_PROJECTION_LAUNCH(1, 2, 4, 10, 1, 3, 3, 2); break;
    case 2: PVLC_PROJECTION_LAUNCH(2, 2, 4, 8, 1, 3, 3, 2); break;
    case 3: PVLC_PROJECTION_LAUNCH(3, 2, 4, 4, 2, 3, 3, 2); break;
    case 4: PVLC_PROJECTION_LAUNCH(4, 2, 2, 4, 2, 3, 3, 2); break;
    case 5: PVLC_PROJECTION_LAUNCH(5, 2, 4, 6, 2, 3, 3, 2); break;
    case 6: PVLC_PROJECTION_LAUNCH(6, 2, 2, 6, 2, 3, 3, 2); break;
    case 7: PVLC_PROJECTION_LAUNCH(7, 2, 1, 4, 4, 2, 4, 2); break;
    case 8: PVLC_PROJECTION_LAUNCH(8, 1, 1, 4, 4, 2, 4, 2); break;
    case 9: PVLC_PROJECTION_LAUNCH(9, 1, 1, 2, 8, 2, 4, 4); break;
    default: PVLC_PROJECTION_LAUNCH(10, 1, 1, 1, 8, 2, 4, 4); break;
    }
#undef PVLC_PROJECTION_LAUNCH
    return static_cast<int>(hipGetLastError());
}

}  // namespace pvlc
