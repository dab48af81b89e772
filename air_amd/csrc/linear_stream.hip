// linear_stream.hip -- the decode linear for M = 2..64 rows over split
// activations, in the tile formats and over dense F16 and Q6_K rows: weights
// streamed through registers, activations shared through LDS by waves that do
// nothing else.
//
// The arithmetic of skinny_kernel / skinny_lds_kernel (linear_skinny.hip);
// what differs is how the operands travel:
//
//   * a workgroup is W consumer waves that own W * TN 16-row weight tiles and
//     every activation row, and kProducers waves; one workgroup per CU;
//   * a consumer's codes and scales go straight to its registers, a ring of
//     kRing records ahead of their use, with no barrier on their way; past
//     the end of the range the loads repeat the last record (a cache hit)
//     instead of branching, so the compiler's load counting stays exact and a
//     wave waits for its oldest record only;
//   * the producers move the activation fragments global -> LDS directly,
//     chunks of kChunk steps, three ahead of the consumers.  Loads return in
//     order: in one wave, every wait for a chunk of activations (L2) would
//     also wait for the weights (HBM) asked for before it, and a pending
//     direct load makes the compiler wait for every load before any register
//     of one is read.  Staging by the consumers cost 9 us of gate|up at 32
//     rows and 28 at 64 (7B, Q8_0, timed with the staging left out);
//   * one bare barrier per chunk; a chunk's fragments are read from LDS one
//     stage ahead of the MFMAs that use them;
//   * the activations come split under one power-of-two scale per row, or per
//     (row, 32-block) where the kernel this one is taken instead of scaled
//     blocks or steps (BLOCKS);
//   * the K sum is formed in levels where registers allow (kLevels says where,
//     with the errors): pairs of steps, trips of the ring, then the total.
//
// What bounds it (counters of 7B gate|up in profiles/decode_stream_sq_counters.md):
// at one activation tile HBM (Q8_0 at 8 rows 144 MB in 32.5 us, 4.4 TB/s).  At more no
// unit is full: at 64 rows VALU issue is at 33..47 % of its ceiling, the matrix
// cores are busy 22..29 % of the time, LDS 28..35 % without a bank conflict,
// and half of the wave time is waiting with three waves on a SIMD; time grows with
// the instructions per weight tile, which grow with M.  Row tiles per workgroup
// are chosen so that the grid is one round of the 256 CUs: a CU with two
// workgroups of eight tiles finishes last (7B gate|up at 32 rows: 296 workgroups
// of eight tiles 48 us, 237 of ten 36).
//
// Measured per linear (Qwen2-7B shapes, graph replay over copies of 320 MB or
// more, the split launch included; kernels replaced -> this, both in one run;
// - where the other kernel stays):
//
//                 M = 8           16            32            64
//   gate|up Q8_0  38.2 -> 33.1    40.4 -> 33.4  -             64.4 -> 57.2 us
//           Q4_0  34.9 -> 26.2    35.6 -> 26.7  45.6 -> 34.8  64.5 -> 51.7
//           Q4_K  39.1 -> 30.7    39.0 -> 30.6  51.9 -> 40.9  79.4 -> 60.5
//   down    Q8_0  -               -             36.5 -> 34.9  45.8 -> 43.7
//           Q4_0  -               -             33.8 -> 31.8  43.1 -> 40.8
//           Q4_K  31.4 -> 23.8    31.8 -> 24.5  39.4 -> 34.9  49.3 -> 45.6
//   q|k|v   Q8_0  -               -             17.5 -> 17.2  23.6 -> 22.0
//           Q4_0  -               -             16.5 -> 16.1  21.2 -> 21.5
//           Q4_K  -               -             18.1 -> 17.8  24.5 -> 23.6
//   lm_head Q8_0  123 -> 108      123 -> 111    138 -> 129    196 -> 184
//           Q4_0  96 -> 78        97 -> 80      125 -> 111    194 -> 165
//           Q4_K  124 -> 99       123 -> 98     156 -> 129    253 -> 202
//
// Dense rows (dense_mfma_kernel before, which asks for a Q6_K step in eight
// 4-byte loads a lane; here a super-block is three 16-byte loads and its
// scales): Q6_K down at 13 rows 63.6 -> 30.4, at 64 200 -> 60.9; gate|up 91.7
// -> 39.6 and 254 -> 97.6; lm_head 331 -> 139 and 949 -> 369; F16 gate|up at 24
// rows 102 -> 79.1, at 64 287 -> 86.3; down 78.2 -> 50.9 and 154 -> 55.7.
//
// Replaces specialized_matmul_kernel / specialized_matmul_batch_reuse_kernel
// (src/cuda/cuda_backend.cu:501-583) for batched decode.
#include "air_hip_device.hpp"
#include "air_hip_kernels.hpp"
#include "air_hip_steps.hpp"

#include <algorithm>
#include <type_traits>
#include <utility>

namespace air_hip {
namespace {

typedef _Float16 half4v __attribute__((ext_vector_type(4)));

struct StreamArgs {
    const void* codes;           // tile codes, or dense rows (F16) / records (Q6_K)
    const void* scales;          // tile scales, or the records' f16 d plane (Q6_K)
    std::uint32_t nt, kt;
    std::uint64_t n, k;
    const u32x4* xs;             // split activations [block][MT][2][64] x 16 B
    std::uint32_t blocks;        // 32-element blocks of the workspace
    const float* inv_scale;      // [mp] inverse power-of-two scale of each row; BLOCKS: [block][mp]
    const float* block_sums;     // [block][mp] sums of the scaled values (Q4_K)
    const float* bias;           // fused when not split over workgroups
    float* out;                  // y, or partials [splits][m][n]
    std::uint32_t m;
    std::uint32_t groups;
    std::uint32_t steps;
    std::uint32_t steps_per_split;
    std::uint32_t partial;
    // K split combined in the kernel (chain_combine): slots [splits-1][m][n],
    // y and the bias the last arrival adds; null: partials for a reduction.
    std::uint64_t* chain;
    float* y;
    const float* chain_bias;
    std::uint32_t splits;
    // SWIGLU: the matrix is a fused gate|up of 2 * ffn_tiles row tiles and out
    // is [m][n / 2].  serial: K splits one workgroup sums itself, in order.
    std::uint32_t ffn_tiles;
    std::uint32_t serial;
};

// silu(g) * u in silu_mul_kernel's arithmetic (no fused products).
__device__ __forceinline__ float swiglu(float g, float u) {
#pragma clang fp contract(off)
    const float s = g / (1.0f + expf(-g));
    return s * u;
}

typedef __attribute__((address_space(3))) void lds_void_t;
typedef __attribute__((address_space(1))) void global_void_t;

// Lane l's 16 (or 4) bytes land at lds_wave_base + l * 16 (l * 4).
__device__ __forceinline__ void lds_load16(const void* src, void* lds_wave_base) {
    __builtin_amdgcn_global_load_lds((global_void_t*)(const_cast<void*>(src)), (lds_void_t*)(lds_wave_base), 16, 0, 0);
}
__device__ __forceinline__ void lds_load4(const void* src, void* lds_wave_base) {
    __builtin_amdgcn_global_load_lds((global_void_t*)(const_cast<void*>(src)), (lds_void_t*)(lds_wave_base), 4, 0, 0);
}

// s_waitcnt for vmcnt <= n only (expcnt and lgkmcnt at their maxima).
template <unsigned n>
__device__ __forceinline__ void wait_vm() {
    static_assert(n < 64u, "vmcnt is six bits");
    __builtin_amdgcn_s_waitcnt((n & 0xfu) | ((n >> 4) << 14) | (0x7u << 4) | (0xfu << 8));
}

// Workgroup barrier ordering LDS accesses only: loads in flight stay so.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

template <unsigned N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    [&]<std::size_t... I>(std::index_sequence<I...>) {
        (f(std::integral_constant<unsigned, static_cast<unsigned>(I)>{}), ...);
    }(std::make_index_sequence<N>{});
}

// A lane's share of one resident record of a row tile: kUnit steps of codes
// and scales.
template <int FMT>
struct Record;
template <>
struct Record<kQ8_0> {
    u32x4 c;
    std::uint32_t d;
};
template <>
struct Record<kQ4_0> {
    u32x4 c;
    u32x2 d;
};
template <>
struct Record<kQ4_K> {
    u32x4 c[2];
    u32x4 h;
};

// Dense storage: F16 rows as they are (both blocks of a step), Q6_K
// super-blocks as linear_dense.hip records (a lane group's 48 code bytes, the
// row's sixteen sub-block scales, d).
template <>
struct Record<kF16> {
    u32x4 v[2];
};
template <>
struct Record<kQ6_K> {
    u32x4 c[3];
    u32x4 s;
    std::uint32_t d;
};

template <int FMT>
constexpr unsigned kUnit = FMT == kQ8_0 || FMT == kF16 ? 1u : FMT == kQ4_0 ? 2u : 4u;   // 64-k steps per record

constexpr unsigned kQ6kRecord = 208u;

// Record `unit` of the lane's row of a dense matrix.
template <int FMT>
__device__ __forceinline__ void load_dense_record(const StreamArgs& a, std::uint64_t row, std::uint32_t unit,
                                                  std::uint32_t lane, Record<FMT>& out) {
    const unsigned char* base = static_cast<const unsigned char*>(a.codes);
    const std::uint32_t g = lane >> 4;
    if constexpr (FMT == kQ6_K) {
        const std::uint64_t blk = row * (a.k / 256u) + unit;
        const unsigned char* rec = base + blk * kQ6kRecord;
#pragma unroll
        for (unsigned i = 0; i < 3u; ++i) {
            out.c[i] = *reinterpret_cast<const u32x4*>(rec + q6k_code_offset(g, 16u * i));
        }
        out.s = *reinterpret_cast<const u32x4*>(rec + 192u);
        out.d = static_cast<const std::uint16_t*>(a.scales)[blk];
    } else {
        // A row that ends on the first block of a step has no second one: the
        // first again, not used (half_step).  Nothing here may touch what is
        // loaded, or the wave waits for this record instead of its oldest.
        const std::uint64_t col = static_cast<std::uint64_t>(unit) * kStepK + 8u * g;
        const unsigned char* at = base + (row * a.k + col) * 2u;
        out.v[0] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(at));
        out.v[1] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(at + (col + 32u < a.k ? 64u : 0u)));
    }
}

// Four 6-bit codes (low nibbles `nibble` of ql's bytes, high pairs at bits
// `pair` of qh's) as exact f16 values q - 32.
template <unsigned nibble, unsigned pair>
__device__ __forceinline__ half4v q6_codes(std::uint32_t ql, std::uint32_t qh) {
    const std::uint32_t low = (ql >> (4u * nibble)) & 0x0f0f0f0fu;
    const std::uint32_t high = (pair < 4u ? qh << (4u - pair) : qh >> (pair - 4u)) & 0x30303030u;
    const std::uint32_t q = low | high;
    const half2v bias = {(_Float16)1056.0f, (_Float16)1056.0f};
    const half2v p0 = bits_as_half2(__builtin_amdgcn_perm(0x64646464u, q, 0x04010400u)) - bias;
    const half2v p1 = bits_as_half2(__builtin_amdgcn_perm(0x64646464u, q, 0x04030402u)) - bias;
    return half4v{p0[0], p0[1], p1[0], p1[1]};
}

template <int FMT>
__device__ __forceinline__ void load_record(const void* codes, const void* scales, std::uint64_t tile,
                                            std::uint32_t lane, Record<FMT>& out) {
    const u32x4* c = static_cast<const u32x4*>(codes);
    if constexpr (FMT == kQ8_0) {
        out.c = __builtin_nontemporal_load(c + tile * 64u + lane);
        out.d = static_cast<const std::uint32_t*>(scales)[tile * 16u + (lane & 15u)];
    } else if constexpr (FMT == kQ4_0) {
        out.c = __builtin_nontemporal_load(c + tile * 64u + lane);
        out.d = static_cast<const u32x2*>(scales)[tile * 16u + (lane & 15u)];
    } else {
        out.c[0] = __builtin_nontemporal_load(c + tile * 128u + lane);
        out.c[1] = __builtin_nontemporal_load(c + tile * 128u + 64u + lane);
        out.h = static_cast<const u32x4*>(scales)[tile * 16u + (lane & 15u)];
    }
}

// Step `sub` (0 .. kUnit - 1) of a record as the step the shared decode reads.
template <int FMT, unsigned sub>
__device__ __forceinline__ StepCodes<FMT> record_step(const Record<FMT>& r) {
    StepCodes<FMT> s;
    if constexpr (FMT == kQ8_0) {
        s.c = r.c;
        s.d = r.d;
    } else if constexpr (FMT == kQ4_0) {
        s.c = sub == 0u ? u32x2{r.c.x, r.c.y} : u32x2{r.c.z, r.c.w};
        s.d = sub == 0u ? r.d.x : r.d.y;
    } else {
        const u32x4 c = r.c[sub >> 1];
        s.c = (sub & 1u) == 0u ? u32x2{c.x, c.y} : u32x2{c.z, c.w};
        s.h = r.h;
    }
    return s;
}

// Steps per LDS chunk: kBuffers chunks of 4 C MT KiB are 128 KiB (96 with
// three activation tiles), one workgroup per CU.
template <int MT>
constexpr unsigned kChunk = MT == 1 ? 8u : MT == 2 ? 4u : 2u;
constexpr unsigned kBuffers = 4u;
// Weight records in flight per wave: 8 KiB of codes (Q8_0), less where three
// or four activation tiles need the registers.
template <int FMT, int MT, int TN>
constexpr unsigned kRing = FMT == kQ8_0 || FMT == kF16 ? (MT <= 2 ? 8u : 4u) / TN
                           : FMT == kQ4_0 ? (MT <= 2 && TN == 1 ? 4u : 2u)
                                          : (TN == 1 && (FMT == kQ4_K || MT <= 2) ? 2u : 1u);   // Q4_K, Q6_K
constexpr int kProducers = 2;
// Levels of the K sum: three at one and two activation tiles and for Q6_K, else
// two (one where two would spill), one in the serial SwiGLU, whose plan has no
// more.  Relative L2 from 64 bits at K = 3584 unsplit, the kernels replaced ->
// this:
//   three  Q8_0 at 8 rows 1.60e-7 -> 1.54e-7, Q4_0 1.58e-7 -> 1.54e-7, Q6_K at 64
//          1.56e-7 -> 1.51e-7;
//   two    Q8_0 lm_head at 40 rows 2.32e-7 -> 1.70e-7, F16 gate|up at 64 1.69e-7 ->
//          1.66e-7;
//   one    Q4_K from 33 rows (gate|up 4.40e-7 -> 4.27e-7, most of it from codes
//          that start at 0), Q8_0 and Q4_0 at 49..64 with two row tiles a wave
//          (lm_head 2.32e-7 either way: the kernel replaced has one too).
// Q4_K at four activation and two row tiles and Q6_K at four activation tiles
// keep one register in scratch.
template <int FMT, int MT, int TN>
constexpr unsigned kLevels = FMT == kF16 && MT == 2 && TN == 2      ? 2u
                             : MT <= 2 || FMT == kQ6_K              ? 3u
                             : FMT == kQ4_K || (MT == 4 && TN == 2) ? 1u
                                                                    : 2u;

// SWIGLU: the workgroup's tiles are W * TN / 2 gate tiles and the up tiles
// that belong to them (TN = 2: both in one wave; else waves w and w + W / 2,
// which meet in LDS), and it stores silu(gate) * up: the SwiGLU launch and
// its round trip through the fused rows go away.  7B gate|up with its SwiGLU,
// graph replay: at 32 rows Q8_0 46.0 -> 38.7 us (eight-wave kernel and its
// reduction before), Q4_0 44.4 -> 33.3, Q4_K 50.9 -> 39.7; at 64 67.2 -> 57.1,
// 67.0 -> 50.9, 81.2 -> 60.1 (the streaming kernel's share included).
// SERIAL: the K splits of a plan that sums them in a reduction, one after the
// other in one workgroup: each in one running sum, scaled, then added from
// zero in split order -- that plan's bits.
// BLOCKS: the activations were split under one scale per (row, 32-block), which
// travels with the fragments and is undone on each block's products; else under
// one per row, undone on the total.  Where the kernel that would otherwise run
// scales steps or blocks, the rows' small blocks beside a large one keep their
// bits only so.
template <int FMT, int MT, int TN, int W, bool SWIGLU, bool SERIAL, bool BLOCKS>
__global__ __launch_bounds__(64 * (W + kProducers), (W + kProducers + 3) / 4) void stream_kernel(StreamArgs a) {
    static_assert(!(SERIAL && BLOCKS), "the serial plan scales rows");
    static_assert(BLOCKS || !dense_storage(FMT), "dense rows take block scales");
    constexpr unsigned P = kProducers;
    constexpr unsigned U = kUnit<FMT>;
    constexpr unsigned D = kRing<FMT, MT, TN>;
    constexpr unsigned C = kChunk<MT>;
    constexpr unsigned L = SERIAL ? 1u : kLevels<FMT, MT, TN>;
    // Steps per trip: the ring comes full circle.  At three levels, and at two
    // where the ring is two steps (F16, three activation and two row tiles), the second one covers
    // eight steps (two trips of four with four activation tiles, which would
    // spill in a trip of eight).
    constexpr bool kEight = (L > 2u && MT <= (FMT == kQ6_K ? 2 : 3)) || (L == 2u && FMT == kF16 && MT == 3 && TN == 2);
    constexpr unsigned kBody = D * U > C && D * U > (kEight ? 8u : 0u) ? D * U : kEight && C < 8u ? 8u : C;
    constexpr bool kHold = L > 2u && kBody < 8u;
    constexpr bool kSums = FMT == kQ4_K;
    constexpr bool kDense = dense_storage(FMT);
    constexpr bool kLateInv = FMT == kQ6_K && MT == 4;   // no registers to hold them through the MFMAs
    constexpr unsigned kMp = 16u * MT;
    constexpr unsigned kParts = MT <= 2 ? 2u : 1u;
    constexpr unsigned kFrags = 2u * C * 2u * MT;           // 1 KiB activation fragments per chunk
    constexpr unsigned kXBytes = kFrags * 1024u;
    constexpr unsigned kSumLoads = kSums ? 2u * C * kMp / 64u : 0u;   // 64-float loads of a chunk's block sums
    constexpr unsigned kInvLoads = BLOCKS ? 2u * C * kMp / 64u : 0u;  // and of its inverse scales
    constexpr unsigned kInvAt = kXBytes + kSumLoads * 256u;
    constexpr unsigned kChunkBytes = kInvAt + kInvLoads * 256u;
    constexpr unsigned kXLoads =                            // per producer and chunk
        (kFrags + P - 1u) / P + (kSumLoads + P - 1u) / P + (kInvLoads + P - 1u) / P;
    static_assert(kBody % C == 0u && kBody % (D * U) == 0u, "a trip is whole chunks and ring turns");
    static_assert((kBuffers - 2u) * kXLoads < 64u, "vmcnt is six bits");
    __shared__ __attribute__((aligned(1024))) unsigned char chunks[kBuffers * kChunkBytes];

    const std::uint32_t lane = threadIdx.x & 63u;
    const std::uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const std::uint32_t group = blockIdx.x % a.groups;
    const std::uint32_t split = blockIdx.x / a.groups;
    const std::uint32_t range = a.steps_per_split * (SERIAL ? a.serial : 1u);
    const std::uint32_t s_begin = split * range;
    const std::uint32_t s_end = min(a.steps, s_begin + range);
    // Row tile j of the wave.
    const auto row_tile = [&](int j) __attribute__((always_inline)) -> std::uint32_t {
        if constexpr (!SWIGLU) return (group * W + wave) * TN + static_cast<std::uint32_t>(j);
        else if constexpr (TN == 2) return group * W + wave + (j != 0 ? a.ffn_tiles : 0u);
        else return wave < W / 2 ? group * (W / 2) + wave : a.ffn_tiles + group * (W / 2) + wave - W / 2;
    };
    const std::uint32_t chunk_count = (s_end - s_begin + C - 1u) / C;   // ranges are never empty

    if (wave >= W) {
        // Producer: fragment f of a chunk is block f / (2 MT) from its first,
        // tile (f / 2) % MT, part f % 2; blocks past the workspace repeat the
        // last one (not used), and so do loads past the chunk.
        const std::uint32_t producer = wave - W;
        const auto fill = [&](std::uint32_t c) __attribute__((always_inline)) {
            unsigned char* base = chunks + (c % kBuffers) * kChunkBytes;
            const std::uint32_t b0 = 2u * (s_begin + c * C);
#pragma unroll
            for (unsigned j = 0; j < (kFrags + P - 1u) / P; ++j) {
                const unsigned f = min(producer + P * j, kFrags - 1u);
                const std::uint32_t b = min(b0 + f / (2u * MT), a.blocks - 1u);
                lds_load16(a.xs + (static_cast<std::uint64_t>(b) * (2u * MT) + f % (2u * MT)) * 64u + lane, base + f * 1024u);
            }
            const auto per_block = [&](const float* from, unsigned loads, unsigned at) __attribute__((always_inline)) {
#pragma unroll
                for (unsigned j = 0; j < (loads + P - 1u) / P; ++j) {
                    const unsigned q = min(producer + P * j, loads - 1u);
                    const unsigned e = q * 64u + lane;
                    const std::uint32_t b = min(b0 + e / kMp, a.blocks - 1u);
                    lds_load4(from + static_cast<std::uint64_t>(b) * kMp + e % kMp, base + at + q * 256u);
                }
            };
            per_block(a.block_sums, kSumLoads, kXBytes);
            per_block(a.inv_scale, kInvLoads, kInvAt);
        };
#pragma unroll
        for (unsigned c = 0; c + 1u < kBuffers; ++c) fill(c);
        for (std::uint32_t c = 0; c < chunk_count; ++c) {
            wait_vm<(kBuffers - 2u) * kXLoads>();   // chunk c has landed
            lds_barrier();                          // ... and chunk c - 1 is read
            fill(c + kBuffers - 1u);
        }
        wait_vm<0u>();                              // nothing lands after the workgroup ends
        return;
    }

    const std::uint32_t u_last = (s_end - 1u) / U;
    float4v acc[TN][MT];
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[j][t] = float4v{0.0f, 0.0f, 0.0f, 0.0f};

    float4v pair[L > 2u ? TN : 1][L > 2u ? MT : 1];   // the running pair of steps
    float4v part[L > 1u ? TN : 1][L > 1u ? MT : 1];   // the running trip
    // Tiles past the last row tile read the last one; they are not stored.
    std::uint64_t wtile[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        if constexpr (kDense) {   // the lane's row
            wtile[j] = min(static_cast<std::uint64_t>(row_tile(j)) * 16u + (lane & 15u), a.n - 1u);
        } else {
            wtile[j] = static_cast<std::uint64_t>(min(row_tile(j), a.nt - 1u)) * a.kt;
        }
    }
    Record<FMT> ring[D][TN];
    const auto load_w = [&](Record<FMT>(&dst)[TN], std::uint32_t unit) __attribute__((always_inline)) {
        const std::uint32_t u = min(unit, u_last);
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            if constexpr (kDense) load_dense_record<FMT>(a, wtile[j], u, lane, dst[j]);
            else load_record<FMT>(a.codes, a.scales, wtile[j] + u, lane, dst[j]);
        }
    };
    // Stage q of a chunk (compile time): its fragments from LDS, read one
    // stage ahead of the arithmetic so that no MFMA waits for an LDS read.  A
    // stage is a block's two parts, or one of them (hi, then lo) with three
    // or four activation tiles, whose registers hold no more.
    half8v frag[2][MT][kParts];
    float4v sums[kSums ? MT : 1];
    float4v invs[BLOCKS ? MT : 1];
    const auto read_stage = [&]<unsigned q>(const unsigned char* base) __attribute__((always_inline)) {
        constexpr unsigned blk = q * kParts / 2u;
#pragma unroll
        for (int t = 0; t < MT; ++t) {
#pragma unroll
            for (unsigned i = 0; i < kParts; ++i) {
                const unsigned f = (blk * MT + static_cast<unsigned>(t)) * 2u + (kParts == 2u ? i : q % 2u);
                if constexpr (FMT == kQ6_K) {
                    // Elements 4 (l / 16)..+3 of both 16-element halves, as
                    // its 16-weight sub-blocks take them.
                    const unsigned char* at = base + f * 1024u + ((lane & 15u) + 16u * (lane >> 5)) * 16u + 8u * ((lane >> 4) & 1u);
                    const u32x2 h0 = *reinterpret_cast<const u32x2*>(at), h1 = *reinterpret_cast<const u32x2*>(at + 512u);
                    frag[q & 1u][t][i] = __builtin_bit_cast(half8v, u32x4{h0.x, h0.y, h1.x, h1.y});
                } else {
                    frag[q & 1u][t][i] = *reinterpret_cast<const half8v*>(base + f * 1024u + lane * 16u);
                }
            }
        }
    };
    // The products of block `blk` of a chunk, block b of step `sub` of a
    // record: every tile's high parts, then the low parts on top, so that
    // neighbouring MFMAs do not depend on each other.  LAST: the chunk's last.
    // absent: the block lies past the row.
    const auto compute = [&]<unsigned blk, unsigned sub, unsigned b, bool LAST>(
                             const unsigned char* base, const Record<FMT>(&w_in)[TN], bool absent)
                             __attribute__((always_inline)) {
        constexpr unsigned q = blk * 2u / kParts;       // the block's first stage
        half8v w[TN];
        float ws[TN], wo[TN];
        float ws2[FMT == kQ6_K ? TN : 1];               // the block's second sub-block
        float4v p[TN][MT];
        float4v p2[FMT == kQ6_K ? TN : 1][FMT == kQ6_K ? MT : 1];
        if constexpr (!LAST || kParts == 1u) read_stage.template operator()<q + 1u>(base);
        const auto read_sums = [&]() __attribute__((always_inline)) {
#pragma unroll
            for (int t = 0; t < MT; ++t) {
                const unsigned at = (blk * kMp + static_cast<unsigned>(t) * 16u + 4u * (lane >> 4)) * 4u;
                if constexpr (kSums) sums[t] = *reinterpret_cast<const float4v*>(base + kXBytes + at);
                if constexpr (BLOCKS && !kLateInv) invs[t] = *reinterpret_cast<const float4v*>(base + kInvAt + at);
            }
        };
        if constexpr (kParts == 2u) read_sums();
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            if constexpr (FMT == kF16) {
                const u32x4 none{0u, 0u, 0u, 0u};
                w[j] = __builtin_bit_cast(half8v, absent ? none : w_in[j].v[b]);
            } else if constexpr (FMT == kQ6_K) {
                // Half `sub / 2`, quadrant 2 (sub % 2) + b: dwords {low
                // nibbles of even, odd quadrants, high pairs} per
                // half-quadrant (linear_dense.hip).
                constexpr unsigned d0 = 6u * (sub >> 1), d1 = d0 + 3u, pair = 4u * (sub & 1u) + 2u * b;
                const auto word = [&](unsigned i) { return w_in[j].c[i / 4u][i % 4u]; };
                const half4v c0 = q6_codes<sub & 1u, pair>(word(d0 + b), word(d0 + 2u));
                const half4v c1 = q6_codes<sub & 1u, pair>(word(d1 + b), word(d1 + 2u));
                w[j] = __builtin_shufflevector(c0, c1, 0, 1, 2, 3, 4, 5, 6, 7);
                const float d = f16_bits_value(w_in[j].d);
                const int sc = static_cast<int>(w_in[j].s[sub]);
                ws[j] = d * static_cast<float>((sc << (24u - 16u * b)) >> 24);
                ws2[j] = d * static_cast<float>((sc << (16u - 16u * b)) >> 24);
            } else {
                const StepCodes<FMT> w_step = record_step<FMT, sub>(w_in[j]);
                w[j] = step_codes<FMT>(w_step, b);
                step_scale<FMT>(w_step, sub, b, ws[j], wo[j]);
            }
        }
        const auto lower = [](const half8v& v) { return __builtin_shufflevector(v, v, 0, 1, 2, 3); };
        const auto upper = [](const half8v& v) { return __builtin_shufflevector(v, v, 4, 5, 6, 7); };
        // First products of a block, then the low parts on top of them.
        const auto first = [&](int j, int t, const half8v& f) __attribute__((always_inline)) {
            const float4v zero{0.0f, 0.0f, 0.0f, 0.0f};
            if constexpr (FMT == kQ6_K) {
                p[j][t] = __builtin_amdgcn_mfma_f32_16x16x16f16(lower(f), lower(w[j]), zero, 0, 0, 0);
                p2[j][t] = __builtin_amdgcn_mfma_f32_16x16x16f16(upper(f), upper(w[j]), zero, 0, 0, 0);
            } else {
                p[j][t] = mfma16x16x32(f, w[j], zero);
            }
        };
        const auto second = [&](int j, int t, const half8v& f) __attribute__((always_inline)) {
            if constexpr (FMT == kQ6_K) {
                p[j][t] = __builtin_amdgcn_mfma_f32_16x16x16f16(lower(f), lower(w[j]), p[j][t], 0, 0, 0);
                p2[j][t] = __builtin_amdgcn_mfma_f32_16x16x16f16(upper(f), upper(w[j]), p2[j][t], 0, 0, 0);
            } else {
                p[j][t] = mfma16x16x32(f, w[j], p[j][t]);
            }
        };
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int t = 0; t < MT; ++t) first(j, t, frag[q & 1u][t][0]);
        if constexpr (kParts == 1u) {
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (!LAST) read_stage.template operator()<q + 2u>(base);
            read_sums();
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int t = 0; t < MT; ++t) {
                second(j, t, kParts == 2u ? frag[q & 1u][t][kParts - 1u] : frag[(q + 1u) & 1u][t][0]);
            }
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int t = 0; t < MT; ++t) {
                float4v& sum = L > 2u ? pair[j][t] : L > 1u ? part[j][t] : acc[j][t];
                constexpr bool kFirst = L > 2u && blk % 4u == 0u;
                if constexpr (kLateInv) {
                    invs[t] = *reinterpret_cast<const float4v*>(
                        base + kInvAt + (blk * kMp + static_cast<unsigned>(t) * 16u + 4u * (lane >> 4)) * 4u);
                }
                const auto add = [&](const float4v& by, const float4v& v) __attribute__((always_inline)) {
                    if constexpr (kFirst) sum = by * v;
                    else sum += by * v;
                };
                const float4v w4{ws[j], ws[j], ws[j], ws[j]};
                if constexpr (FMT == kF16) {
                    add(invs[t], p[j][t]);
                } else if constexpr (!BLOCKS) {
                    add(w4, p[j][t]);
                    if constexpr (kSums) sum -= wo[j] * sums[t];
                } else if constexpr (FMT == kQ6_K) {
                    float4v v = ws[j] * p[j][t];
                    v += ws2[j] * p2[j][t];
                    add(invs[t], v);
                } else if constexpr (kSums) {
                    add(invs[t], ws[j] * p[j][t] - wo[j] * sums[t]);
                } else {
                    // A power of two scales without rounding, so this product
                    // rounds once, as under a row's scale.
                    add(w4, invs[t] * p[j][t]);
                }
                if constexpr (L > 2u && blk % 4u == 3u) part[j][t] += sum;
            }
    };

    // The weights' first records.
    static_for<D>([&](auto d) __attribute__((always_inline)) {
        load_w(ring[d.value], s_begin / U + d.value);
        __builtin_amdgcn_sched_barrier(0);   // the loop's load counting needs this order too
    });
    float4v inv[MT];
    const auto load_inv = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < MT; ++t) inv[t] = reinterpret_cast<const float4v*>(a.inv_scale)[t * 4 + (lane >> 4)];
    };
    float4v total[SERIAL ? TN : 1][SERIAL ? MT : 1];
    std::uint32_t flush = s_begin + a.steps_per_split;
    const auto flush_split = [&]() __attribute__((always_inline)) {
#pragma clang fp contract(off)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int t = 0; t < MT; ++t) {
                total[SERIAL ? j : 0][SERIAL ? t : 0] += acc[j][t] * inv[t];
                acc[j][t] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
            }
        flush += a.steps_per_split;
    };
    if constexpr (SERIAL) {
        load_inv();
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int t = 0; t < MT; ++t) total[j][t] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
    }
    // F16 rows of an odd number of blocks: the last step is half a one.
    const bool half_step = FMT == kF16 && s_end == a.steps && a.k % kStepK != 0u;
    // One trip: kBody steps from s.  WHOLE: all of them, in full, lie in the range.
    std::uint32_t buffer = 0u;
    bool first_half = true;   // kHold: of the second level's eight steps
    const auto trip = [&](std::uint32_t s, auto whole_tag) __attribute__((always_inline)) {
        constexpr bool WHOLE = decltype(whole_tag)::value;
        bool done = false;
        if (L > 1u && (!kHold || first_half)) {
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int t = 0; t < MT; ++t) part[j][t] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
        }
        const unsigned char* cur = chunks;
        static_for<kBody>([&](auto i_tag) __attribute__((always_inline)) {
            constexpr unsigned i = i_tag.value;
            constexpr unsigned cs = i % C;                  // step of its chunk
            if (!WHOLE && done) return;
            if constexpr (cs == 0u) {
                if (!WHOLE && i != 0u && s + i >= s_end) {
                    done = true;
                    return;
                }
                lds_barrier();
                cur = chunks + buffer * kChunkBytes;
                buffer = (buffer + 1u) % kBuffers;
                read_stage.template operator()<0>(cur);
            }
            if (WHOLE || s + i < s_end) {
                if constexpr (SERIAL) {
                    if (s + i == flush) flush_split();
                }
                compute.template operator()<2u * cs, i % U, 0, false>(cur, ring[(i / U) % D], false);
                compute.template operator()<2u * cs + 1u, i % U, 1, cs + 1u == C>(
                    cur, ring[(i / U) % D], FMT == kF16 && !WHOLE && half_step && s + i + 1u == s_end);
            }
            if constexpr (i % U == U - 1u) load_w(ring[(i / U) % D], (s + i) / U + D);
            __builtin_amdgcn_sched_barrier(0);
        });
        // A range that ends on the first step of a pair.
        const bool open = L > 2u && !WHOLE && ((s_end - s_begin) & 1u) != 0u;
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int t = 0; t < MT; ++t) {
                if constexpr (L > 2u) {
                    if (open) part[j][t] += pair[j][t];
                }
                if (L > 1u && (!kHold || !first_half || !WHOLE)) acc[j][t] += part[j][t];
            }
        if constexpr (kHold) first_half = !first_half;
    };
    std::uint32_t s = s_begin;
    for (; s + kBody <= s_end - (half_step ? 1u : 0u); s += kBody) trip(s, std::true_type{});
    if (s < s_end) {
        trip(s, std::false_type{});
    } else if (kHold && !first_half) {
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int t = 0; t < MT; ++t) acc[j][t] += part[L > 1u ? j : 0][L > 1u ? t : 0];
    }

    // D[row = activation row][col = weight row], as skinny_kernel.
    if constexpr (SERIAL) flush_split();
    else if constexpr (!BLOCKS) load_inv();
    const auto value = [&](int j, int t, int i, float bn) __attribute__((always_inline)) {
        if constexpr (SERIAL) return total[j][t][i] + bn;
        else if constexpr (BLOCKS) return acc[j][t][i] + bn;
        else return acc[j][t][i] * inv[t][i] + bn;
    };
    if constexpr (SWIGLU) {
        __shared__ float4v up_rows[TN == 2 ? 1 : W / 2][MT][64];
        const std::uint64_t ffn = a.n / 2u;
        const std::uint64_t n = static_cast<std::uint64_t>(row_tile(0)) * 16u + (lane & 15u);   // gate (or up) row
        const bool is_up = TN == 1 && wave >= W / 2;
        const bool live = n < (is_up ? a.n : ffn);
        const float b0 = a.bias && live ? a.bias[n] : 0.0f;
        if constexpr (TN == 1) {
            if (is_up) {
#pragma unroll
                for (int t = 0; t < MT; ++t)
#pragma unroll
                    for (int i = 0; i < 4; ++i) up_rows[wave - W / 2][t][lane][i] = value(0, t, i, b0);
            }
            lds_barrier();
            if (is_up) return;
        }
        if (!live) return;
        const float b1 = TN == 2 && a.bias ? a.bias[ffn + n] : 0.0f;
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            float4v u;
            if constexpr (TN == 2) {
#pragma unroll
                for (int i = 0; i < 4; ++i) u[i] = value(TN - 1, t, i, b1);
            } else {
                u = up_rows[wave][t][lane];
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const std::uint32_t m = static_cast<std::uint32_t>(t) * 16u + 4u * (lane >> 4) + static_cast<std::uint32_t>(i);
                if (m < a.m) a.out[static_cast<std::uint64_t>(m) * ffn + n] = swiglu(value(0, t, i, b0), u[i]);
            }
        }
        return;
    }
    float* out = a.out + (a.partial ? static_cast<std::uint64_t>(split) * a.m * a.n : 0u);
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        const std::uint64_t n = static_cast<std::uint64_t>(row_tile(j)) * 16u + (lane & 15u);
        if (row_tile(j) >= a.nt || n >= a.n) continue;
        const float bn = a.bias ? a.bias[n] : 0.0f;
#pragma unroll
        for (int t = 0; t < MT; ++t) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const std::uint32_t m = static_cast<std::uint32_t>(t) * 16u + 4u * (lane >> 4) + static_cast<std::uint32_t>(i);
                if (m >= a.m) continue;
                const std::uint64_t e = static_cast<std::uint64_t>(m) * a.n + n;
                float v = value(j, t, i, bn);
                if (a.chain) {
                    if (chain_combine(a.chain, static_cast<std::uint64_t>(a.m) * a.n, e, split, a.splits, v)) {
                        a.y[e] = a.chain_bias ? v + a.chain_bias[n] : v;
                    }
                } else {
                    out[e] = v;
                }
            }
        }
    }
}

// What the rules reach.  Scales: blocks always over dense rows, else only at one
// activation tile (Q4_K on eight waves) and, Q8_0 on eight waves, two; rows of
// the tile formats at any width.  F16 from two activation tiles.  Ten waves of
// one row tile over Q8_0 at two activation tiles only for the serial SwiGLU
// (2049..2560 row tiles); no SwiGLU over matrices narrow enough for Q8_0's
// blocks at two.
template <int FMT, int MT, int TN, int W, bool SWIGLU, bool BLOCKS>
constexpr bool kReached = dense_storage(FMT)           ? BLOCKS && !SWIGLU && (FMT != kF16 || MT >= 2)
                          : FMT == kQ8_0 && MT == 2    ? (BLOCKS ? W == 8 && !SWIGLU : W == 8 || TN == 2)
                          : BLOCKS                     ? MT == 1 && (FMT != kQ4_K || W == 8)
                                                       : true;

template <int FMT, int MT, int TN, int W, bool BLOCKS>
hipError_t launch_scaled(const StreamArgs& a, std::uint32_t blocks, hipStream_t stream) {
    const dim3 threads(64 * (W + kProducers));
    const dim3 grid(blocks);
    if (a.ffn_tiles == 0u) {
        if constexpr (kReached<FMT, MT, TN, W, false, BLOCKS>) {
            hipLaunchKernelGGL((stream_kernel<FMT, MT, TN, W, false, false, BLOCKS>), grid, threads, 0, stream, a);
            return hipGetLastError();
        }
    } else if (a.serial > 1u) {
        if constexpr (FMT == kQ8_0 && MT == 2 && W == 10 && !BLOCKS) {
            hipLaunchKernelGGL((stream_kernel<FMT, MT, TN, W, true, true, false>), grid, threads, 0, stream, a);
            return hipGetLastError();
        }
    } else if constexpr (kReached<FMT, MT, TN, W, true, BLOCKS>) {
        hipLaunchKernelGGL((stream_kernel<FMT, MT, TN, W, true, false, BLOCKS>), grid, threads, 0, stream, a);
        return hipGetLastError();
    }
    return hipErrorInvalidConfiguration;
}

template <int FMT, int MT, int TN, int W>
hipError_t launch_w(const StreamArgs& a, const SkinnyShape& s, std::uint32_t blocks, hipStream_t stream) {
    return s.block_scaled ? launch_scaled<FMT, MT, TN, W, true>(a, blocks, stream)
                          : launch_scaled<FMT, MT, TN, W, false>(a, blocks, stream);
}

// One wave per 32-element block and 16-row tile: lane l holds row l % 16,
// elements 8 (l / 16)..+7, the fragment's own order, so loads are whole 128-byte
// runs and stores 1 KiB.  Rows past m and blocks past k are zeros.
__global__ __launch_bounds__(256) void split_blocks_kernel(const float* __restrict__ x, std::uint32_t m, std::uint64_t k,
                                                           std::uint32_t blocks, std::uint32_t mtiles,
                                                           u32x4* __restrict__ xs, float* __restrict__ block_sums,
                                                           float* __restrict__ inv_scale) {
#pragma clang fp contract(off)
    const std::uint32_t lane = threadIdx.x & 63u;
    const std::uint32_t w = blockIdx.x * 4u + (threadIdx.x >> 6);
    if (w >= blocks * mtiles) return;
    const std::uint32_t b = w / mtiles, t = w % mtiles;
    const std::uint32_t row = t * 16u + (lane & 15u);
    float v[8];
    const std::uint64_t col = static_cast<std::uint64_t>(b) * 32u + 8u * (lane >> 4);
    if (row < m && col < k) {
        const float4v* src = reinterpret_cast<const float4v*>(x + static_cast<std::uint64_t>(row) * k + col);
        const float4v lo = src[0], hi = src[1];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            v[e] = lo[e];
            v[4 + e] = hi[e];
        }
    } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = 0.0f;
    }
    float amax = 0.0f;
#pragma unroll
    for (int e = 0; e < 8; ++e) amax = fmaxf(amax, fabsf(v[e]));
    amax = fmaxf(amax, __shfl_xor(amax, 16));
    amax = fmaxf(amax, __shfl_xor(amax, 32));
    float s, inv;
    block_scale(amax, s, inv);
    half8v hi, lo;
    split8(v, s, hi, lo);
    const float sum01 = v[0] * s + v[1] * s, sum23 = v[2] * s + v[3] * s;
    const float sum45 = v[4] * s + v[5] * s, sum67 = v[6] * s + v[7] * s;
    float sum = (sum01 + sum23) + (sum45 + sum67);
    sum += __shfl_xor(sum, 16);
    sum += __shfl_xor(sum, 32);
    xs[static_cast<std::uint64_t>(w) * 128u + lane] = __builtin_bit_cast(u32x4, hi);
    xs[static_cast<std::uint64_t>(w) * 128u + 64u + lane] = __builtin_bit_cast(u32x4, lo);
    if (lane < 16u) {
        block_sums[static_cast<std::uint64_t>(b) * mtiles * 16u + row] = sum;
        inv_scale[static_cast<std::uint64_t>(b) * mtiles * 16u + row] = inv;
    }
}

template <int FMT, int MT>
hipError_t launch_mt(const StreamArgs& a, const SkinnyShape& s, std::uint32_t blocks, hipStream_t stream) {
    if constexpr (!(FMT == kQ6_K && MT >= 2) && !(FMT == kF16 && MT >= 4)) {   // stream_tile_n
        if (s.waves == 10u && s.tile_n == 2u) return launch_w<FMT, MT, 2, 10>(a, s, blocks, stream);
    }
    if (s.waves == 10u && s.tile_n == 1u) return launch_w<FMT, MT, 1, 10>(a, s, blocks, stream);
    if (s.waves == 8u && s.tile_n == 1u) return launch_w<FMT, MT, 1, 8>(a, s, blocks, stream);
    return hipErrorInvalidConfiguration;
}

template <int FMT>
hipError_t launch_fmt(const StreamArgs& a, const SkinnyShape& s, std::uint32_t blocks, hipStream_t stream) {
    switch (s.mt) {
    case 1: return launch_mt<FMT, 1>(a, s, blocks, stream);
    case 2: return launch_mt<FMT, 2>(a, s, blocks, stream);
    case 3: return launch_mt<FMT, 3>(a, s, blocks, stream);
    default: return launch_mt<FMT, 4>(a, s, blocks, stream);
    }
}

} // namespace

hipError_t launch_split_activations_blocks(const float* x, std::uint32_t m, std::uint64_t k, std::uint64_t kp,
                                           const SplitWorkspace& ws, hipStream_t stream) {
    const std::uint64_t mtiles = ceil_div(m, 16u), waves = kp / 32u * mtiles;
    if (m == 0u || m > 64u || k % 32u != 0u || waves > 0x7fffffffu) return hipErrorInvalidValue;
    hipLaunchKernelGGL(split_blocks_kernel, dim3(static_cast<unsigned>(ceil_div(waves, 4u))), dim3(256), 0, stream, x, m,
                       k, static_cast<std::uint32_t>(kp / 32u), static_cast<std::uint32_t>(mtiles),
                       static_cast<u32x4*>(ws.xs), ws.block_sums, ws.inv_scale);
    return hipGetLastError();
}

namespace {

// Row tiles a wave takes (plan_stream's comment says why).  Not two where the
// registers then hold fewer levels of the K sum than the kernel replaced had
// (from 64 bits at K = 2048, before / two tiles / one: F16 at four activation
// tiles 1.6e-7 / 2.0e-7 / 1.6e-7, Q6_K at two 1.49e-7 / 1.52e-7 / 1.48e-7).
std::uint32_t stream_tile_n(const TilePlanes& p, std::uint32_t m) {
    return p.nt > 2560u && !(p.type == kQ6_K && m > 16u) && !(p.type == kF16 && m > 48u) ? 2u : 1u;
}
std::uint32_t stream_waves(const TilePlanes& p) { return p.nt > 2048u ? 10u : 8u; }

// Whether a wide matrix's workgroups fill their rounds of the CUs.  Twenty
// tiles a workgroup (from 2561 row tiles) leave half of the CUs idle at first:
// one round needs 160 workgroups (Q8_0, K = 3584 at 8 rows, time of the kernels
// before over this: 3000 row tiles 0.85, 3200 1.02; at 33..48 rows 176, 3200
// 0.95..0.98), several need the last to bring their slots to 78 % (5130 row
// tiles, 50 %: 0.69..1.0; 7600, 74 %: 0.90..1.12; 8200, 80 %: 1.07..1.15;
// 11500, 75 %: 0.86..1.15; 12800, 83 %: 1.0..1.16), Q8_0 at up to four rows to 88
// % (8200 and 12800 0.95..0.97, 9504 1.04).
bool stream_fills(const TilePlanes& p, std::uint32_t m) {
    const std::uint64_t groups = ceil_div(p.nt, stream_waves(p) * stream_tile_n(p, m));
    const bool q8 = p.type == kQ8_0;
    if (groups <= 256u) return p.nt <= 2560u || groups >= (q8 && m > 32u && m <= 48u ? 176u : 160u);
    return groups * 100u >= ceil_div(groups, 256u) * 256u * (q8 && m <= 4u ? 88u : 78u);
}

} // namespace

bool stream_preferred(const TilePlanes& p, std::uint32_t m) {
    // Measured against the kernels it replaces (graph replay over 400 MB of
    // copies, split launch included) in every format at 3, 8, 16, 20, 26, 32,
    // 40, 56 and 64 rows: 30 counts of row tiles from 1032 to 12800 at K = 2048
    // and 3584, 15 from 96 to 1000 at K = 2048, 3584, 4352, 8192 and 18944.
    // Taken where it is faster or even; figures are old time over new.
    //  * wide matrices (over 1024 row tiles) whose workgroups fill their
    //    rounds (stream_fills): 1.0..1.4, but for Q8_0 ones of 2000..4096 row
    //    tiles at 17..32 rows, whose eight-wave plan and its two splits stay,
    //    and short K at up to four rows (0.96 at 1900 row tiles of 2048) or, in
    //    several rounds, from 49 (0.92..0.98);
    //  * 257..1024 row tiles at two or more activation tiles: 1.0..1.4 from K =
    //    3584 on.  At K = 2048 the K splits that fill the GPU cost more than
    //    they stream: Q8_0 0.77..1.0, Q4_0 0.75..0.95 up to 640 row tiles;
    //  * up to 256 row tiles with long K at two or more (the wave-split kernel
    //    keeps short K): 1.0..1.4; Q8_0 at two only from 25 rows, 128 row tiles
    //    and K = 8192 (K = 4352 0.94..0.98, 96 row tiles of 18944 0.94);
    //  * at four activation tiles the K splits of the skinny kernel can fill
    //    its two workgroups a CU; then it is as fast up to K = 8192 (Q8_0 512
    //    row tiles of 3584 0.92, 256 of 8192 0.96, Q4_0 0.95..1.0);
    //  * at one activation tile only Q4_K with long K (1.1..2.2);
    //  * fewer than 128 row tiles only with K over 8192 (96 of 8192: Q8_0 0.84,
    //    Q4_0 0.95, Q4_K 0.92 at 8 rows, 1.2 at 3).
    // Short K (under 32 steps) leaves the ring and the chunks nothing to run
    // ahead of, and so do fewer than 96 row tiles.
    if (m < 2u || m > 64u || p.kp / kStepK < 32u || p.nt < 96u) return false;
    const bool one = m <= 16u, two = !one && m <= 32u;
    const bool wide = p.nt > 1024u, long_k = p.k > 4096u;
    if (p.type == kQ6_K) {
        // Against dense_mfma_kernel: 1.1 to 5.6 times faster but for narrow
        // short-K matrices below 16 rows (o at 13 rows 14.7 against 15.2 us),
        // or below 33 of K = 2048 (0.81..0.97).
        return p.nt > 256u || long_k || m > 32u || (m >= 16u && p.k >= 3072u);
    }
    if (p.type == kF16) {
        // Against dense_mfma_kernel, which reads the weights once for 64 rows
        // too but from half the waves: from 33 rows 1.5..4.8 times faster but
        // for narrow short-K matrices below 49; at 17..32 1.0..2.9 where the
        // rounds are filled (3000 row tiles 0.9) and K is not short (1400 row
        // tiles of 2048 0.94).
        if (one) return false;
        if (two) return stream_fills(p, m) && (p.nt > 1700u || (p.nt > 256u && p.k >= 3072u) || p.k > 8192u);
        return p.nt > 256u || long_k || m > 48u;
    }
    if (p.type == kQ4_K && m > 32u &&
        plan_stream(p, m).steps_per_split * 16u > plan_skinny(p, m, 0u, 0u).steps_per_split * 17u) {
        // A longer running sum than it replaces; a sixteenth longer measures
        // even (K = 3584..18944: -6..+1.3 % of the error), a twelfth 2 % more.
        return false;
    }
    if (wide) {
        if (p.type == kQ8_0 && two && p.nt >= 2000u && p.nt <= 4096u) return false;
        if (p.type == kQ8_0 && p.k < 3072u && ((m <= 4u && p.nt <= 2048u) || (m > 48u && p.nt > 5120u))) return false;
        return stream_fills(p, m);
    }
    if (p.nt < 128u && p.k <= 8192u && !(one && m <= 4u)) return false;
    if (one) return p.type == kQ4_K && long_k;
    if (m > 48u && p.type != kQ4_K && p.k <= 8192u) {
        const SkinnyShape s = plan_skinny(p, m, 0u, 0u);
        if (s.groups * s.splits >= 384u) return false;
    }
    if (p.nt > 256u) {
        const std::uint32_t least = p.type == kQ8_0 ? 1025u : p.type == kQ4_0 ? 800u : 0u;   // row tiles at short K
        return p.k >= 3072u || p.nt >= least;
    }
    if (p.type == kQ4_K && !two && p.k < 8192u) return false;   // even or slower at 33..64 rows (27.7, 28.2 us)
    if (p.type == kQ8_0 && two) return m > 24u && p.k >= 8192u && p.nt >= 128u;
    return long_k;
}

SkinnyShape plan_stream(const TilePlanes& p, std::uint32_t m) {
    SkinnyShape s;
    s.stream = true;
    s.mt = static_cast<std::uint32_t>(ceil_div(m, 16u));
    s.steps = static_cast<std::uint32_t>(p.kp / kStepK);
    // One round of 256 workgroups where the row tiles allow it: eight tiles a
    // workgroup, ten from 2049 row tiles, twenty (two per wave, which also
    // halves the activations read per tile: lm_head 141 -> 121 us at 32 rows)
    // from 2561, where ten would start a second round.
    s.tile_n = stream_tile_n(p, m);
    s.waves = stream_waves(p);
    s.groups = static_cast<std::uint32_t>(ceil_div(p.nt, s.waves * s.tile_n));
    // Otherwise K is split over workgroups up to that round, at least twelve
    // steps each (the partials' round trip: Q8_0 q|k|v at 32 rows 16.9 us with
    // four splits, 17.6 with seven; ten with three or four activation tiles
    // and eight for Q4_K, whose steps take longer: 18.4 and 17.3 us with four
    // and six), and no further than plan_skinny would.
    const std::uint32_t least = p.type == kQ4_K || p.type == kQ6_K ? 8u : s.mt >= 3u ? 10u : 12u;
    std::uint32_t splits = std::min(256u / std::min(s.groups, 256u), s.steps / least);
    if (!dense_storage(p.type)) splits = std::min(splits, plan_skinny(p, m, 0u, 0u).splits);
    splits = std::max(splits, 1u);
    const std::uint32_t unit = p.type == kQ8_0 || p.type == kF16 ? 1u : p.type == kQ4_0 ? 2u : 4u;   // kUnit
    s.steps_per_split = static_cast<std::uint32_t>(ceil_div(ceil_div(s.steps, splits), unit) * unit);
    // Q4_K at three and four activation tiles keeps one running sum a split
    // (kLevels), so no split may be longer than the skinny kernel's: whole
    // records go down, not up, where the extra split has its workgroups (down
    // at 64 rows, 40 steps 4.04e-7 from 64 bits, 36 3.96e-7, the skinny
    // kernel's 37 3.97e-7).
    const std::uint32_t down = static_cast<std::uint32_t>(ceil_div(s.steps, splits) / unit * unit);
    if (p.type == kQ4_K && s.mt >= 3u && splits > 1u && down > 0u && down < s.steps_per_split &&
        s.groups * ceil_div(s.steps, down) <= 256u) {
        s.steps_per_split = down;
    }
    s.splits = static_cast<std::uint32_t>(ceil_div(s.steps, s.steps_per_split));
    return s;
}

namespace {

hipError_t launch_stream(const TilePlanes& p, const SplitWorkspace& ws, StreamArgs a, std::uint32_t m,
                         const SkinnyShape& s, hipStream_t stream) {
    if (m == 0u || m > 64u || s.mt != ceil_div(m, 16u) || s.steps == 0u || s.steps_per_split == 0u) {
        return hipErrorInvalidValue;
    }
    a.codes = p.codes;
    a.scales = p.scales;
    a.nt = p.nt;
    a.kt = p.kt;
    a.n = p.n;
    a.k = p.k;
    a.xs = static_cast<const u32x4*>(ws.xs);
    a.blocks = static_cast<std::uint32_t>(p.kp / 32u);
    a.inv_scale = ws.inv_scale;
    a.block_sums = ws.block_sums;
    a.m = m;
    a.groups = s.groups;
    a.steps = s.steps;
    a.steps_per_split = s.steps_per_split;
    const std::uint32_t blocks = s.groups * (a.serial > 1u ? 1u : s.splits);
    switch (p.type) {
    case kQ8_0: return launch_fmt<kQ8_0>(a, s, blocks, stream);
    case kQ4_0: return launch_fmt<kQ4_0>(a, s, blocks, stream);
    case kQ4_K: return launch_fmt<kQ4_K>(a, s, blocks, stream);
    case kF16: return launch_fmt<kF16>(a, s, blocks, stream);
    case kQ6_K:
        a.scales = static_cast<const unsigned char*>(p.codes) + p.n * (p.k / 256u) * kQ6kRecord;
        return launch_fmt<kQ6_K>(a, s, blocks, stream);
    default: return hipErrorInvalidValue;
    }
}

} // namespace

hipError_t launch_stream_linear(const TilePlanes& p, const SplitWorkspace& ws, const float* bias, float* y,
                                std::uint32_t m, const SkinnyShape& shape, float* partials, hipStream_t stream,
                                const SplitEpilogue* epilogue, std::uint64_t* chain) {
    StreamArgs a{};
    a.serial = 1u;
    const bool split = shape.splits > 1u;
    const bool chained = split && chain && !epilogue;
    a.partial = split ? 1u : 0u;
    a.bias = split ? nullptr : bias;
    a.out = split ? partials : y;
    if (chained) {
        a.chain = chain;
        a.y = y;
        a.chain_bias = bias;
        a.splits = shape.splits;
    }
    const hipError_t err = launch_stream(p, ws, a, m, shape, stream);
    if (err != hipSuccess || !split || chained) return err;
    if (epilogue) return launch_split_epilogue(partials, shape.splits, m, p.n, bias, *epilogue, stream);
    return launch_split_reduce(partials, shape.splits, m, p.n, bias, y, stream);
}

bool plan_stream_swiglu(const TilePlanes& p, std::uint32_t m, const SkinnyShape& linear, SkinnyShape& s) {
    if (dense_storage(p.type) || p.n % 32u != 0u || m < 2u || m > 64u) return false;
    const std::uint32_t ffn_tiles = p.nt / 2u;
    if (linear.stream) {
        // The linear's own workgroups, with half gate and half up tiles; a K
        // split goes through the reduction, which carries the SwiGLU.
        if (linear.splits != 1u) return false;
        s = linear;
    } else {
        // Q8_0 at 17..32 rows, 2000..4096 row tiles: the plain linear keeps
        // the eight-wave kernel (37.8 us; its two splits reduce in another
        // 5 with the SwiGLU); here its splits are summed in the workgroup,
        // where the workgroups fill the GPU (2800 row tiles 0.84..0.99 times
        // the reduction's speed).
        if (p.type != kQ8_0 || m <= 16u || m > 32u || p.nt < 2000u || p.nt > 4096u || p.kp / kStepK < 32u ||
            !stream_fills(p, m)) {
            return false;
        }
        s = linear;
        s.stream = true;
        s.waves = 10u;
        s.tile_n = p.nt > 2560u ? 2u : 1u;
    }
    s.groups = static_cast<std::uint32_t>(ceil_div(ffn_tiles, s.waves * s.tile_n / 2u));
    return true;
}

hipError_t launch_stream_swiglu(const TilePlanes& p, const SplitWorkspace& ws, const float* bias, float* out,
                                std::uint32_t m, const SkinnyShape& s, hipStream_t stream) {
    StreamArgs a{};
    a.serial = s.splits;
    a.ffn_tiles = p.nt / 2u;
    a.bias = bias;
    a.out = out;
    return launch_stream(p, ws, a, m, s, stream);
}

} // namespace air_hip
