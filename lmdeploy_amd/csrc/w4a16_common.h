// Shared device helpers of the gfx950 W4A16 library: vector types, the int4 -> fp16
// conversion and the tiled weight layout.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "w4a16_internal.h"

namespace w4a16 {

typedef _Float16 half_t;
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float    float4_t __attribute__((ext_vector_type(4)));
typedef float    float16_t __attribute__((ext_vector_type(16)));

constexpr int kGroup = 128;  // quantisation group size == rows of one weight tile
constexpr int kTileN = 16;   // columns of one weight tile
constexpr int kWave  = 64;

// Layout of the repacked weights.  One tile = 16 columns x 128 rows = 1024 bytes, stored as
// 64 lanes x uint4.  Tile index = kt * (N/16) + nt: the column tiles of one group are
// contiguous, so waves on neighbouring columns stream neighbouring DRAM pages (measured: about
// 10 % more bandwidth on a 240 MB matrix than with the tiles of a column contiguous).
// Lane l = 16*b + c holds column
// 16*nt + c; its word j holds rows 128*kt + 32*j + 8*b + e (e = 0..7), row offset e in
// nibble kNibbleOfRow[e].  One word is therefore one B operand of v_mfma_f32_16x16x32_f16.
// Pack order along the rows is the AWQ order [0,2,4,6,1,3,5,7], which lets the unpack
// below produce rows (0,1), (2,3), (4,5), (6,7) as fp16 pairs with a single shift.
__device__ __host__ constexpr int row_of_nibble(int p)
{
    return (p & 3) * 2 + (p >> 2);  // [0,2,4,6,1,3,5,7]
}
__device__ __host__ constexpr int nibble_of_row(int e)
{
    return (e & 1) * 4 + (e >> 1);  // [0,4,1,5,2,6,3,7]
}

__device__ __forceinline__ half2_t as_half2(uint32_t u)
{
    return __builtin_bit_cast(half2_t, u);
}
__device__ __forceinline__ uint32_t as_u32(half2_t h)
{
    return __builtin_bit_cast(uint32_t, h);
}

// Mask and magic constants of the unpack, held in registers.  gfx9-family VOP3 encodings take
// no 32-bit literals, so (w & mask) | magic only becomes one v_and_or_b32 when both constants
// already live in registers; the empty asm statements keep the optimiser from folding them
// back into literals (which would cost a separate v_and_b32 and v_or_b32 per pair).
struct UnpackConsts {
    uint32_t mask_lo, mask_hi;    // SGPRs
    uint32_t magic_lo, magic_hi;  // VGPRs
    __device__ __forceinline__ UnpackConsts()
    {
        mask_lo  = 0x000f000fu;
        mask_hi  = 0x00f000f0u;
        magic_lo = 0x64006400u;
        magic_hi = 0x54005400u;
        asm volatile("" : "+s"(mask_lo), "+s"(mask_hi));
        asm volatile("" : "+v"(magic_lo), "+v"(magic_hi));
    }
};

// The four fp16 pairs of one weight word, still carrying their offsets:
//   v[0] = 1024 + rows (0,1), v[1] = 64 + rows (2,3), v[2] = 1024 + rows (4,5), v[3] = 64 + rows (6,7)
// 0x6400 is 1024.0 (ulp 1) so OR-ing a nibble into bits 0..3 adds it; 0x5400 is 64.0
// (ulp 1/16) so OR-ing a nibble into bits 4..7 adds it too.
__device__ __forceinline__ void unpack_offset(uint32_t w, uint32_t (&v)[4])
{
    const uint32_t w8 = w >> 8;
    v[0] = (w & 0x000f000fu) | 0x64006400u;
    v[1] = (w & 0x00f000f0u) | 0x54005400u;
    v[2] = (w8 & 0x000f000fu) | 0x64006400u;
    v[3] = (w8 & 0x00f000f0u) | 0x54005400u;
}
__device__ __forceinline__ void unpack_offset(uint32_t w, uint32_t (&v)[4], const UnpackConsts& k)
{
    const uint32_t w8 = w >> 8;
    v[0] = (w & k.mask_lo) | k.magic_lo;
    v[1] = (w & k.mask_hi) | k.magic_hi;
    v[2] = (w8 & k.mask_lo) | k.magic_lo;
    v[3] = (w8 & k.mask_hi) | k.magic_hi;
}

// One weight word -> eight fp16 weights, rows 0..7 in order: fp16_rn((q - z) * s), the reference's
// weight.  z1024 = (1024 + z) x2 and z64 = (64 + z) x2; both subtractions are exact.
__device__ __forceinline__ half8_t dequant_full(uint32_t w, half2_t z1024, half2_t z64, half2_t s,
                                                const UnpackConsts& k)
{
    uint32_t v[4];
    unpack_offset(w, v, k);
    const half2_t a = (as_half2(v[0]) - z1024) * s;
    const half2_t b = (as_half2(v[1]) - z64) * s;
    const half2_t c = (as_half2(v[2]) - z1024) * s;
    const half2_t d = (as_half2(v[3]) - z64) * s;
    half8_t r;
    r[0] = a[0]; r[1] = a[1]; r[2] = b[0]; r[3] = b[1];
    r[4] = c[0]; r[5] = c[1]; r[6] = d[0]; r[7] = d[1];
    return r;
}

// The same without the scale: the exact integers q - z.
__device__ __forceinline__ half8_t unpack_full(uint32_t w, half2_t z1024, half2_t z64, const UnpackConsts& k)
{
    uint32_t v[4];
    unpack_offset(w, v, k);
    const half2_t a = as_half2(v[0]) - z1024, b = as_half2(v[1]) - z64, c = as_half2(v[2]) - z1024, d = as_half2(v[3]) - z64;
    return half8_t{a[0], a[1], b[0], b[1], c[0], c[1], d[0], d[1]};
}

// The reference multiplies (q - z) by the scale with flush-to-zero (mul.ftz.f16x2, common.h:229-230):
// a subnormal scale counts as zero, and that is the only case in which the flush acts, because a
// normal scale times a non-zero integer is never subnormal.  True if the scale of Q word `q` is normal.
__device__ __forceinline__ bool scale_is_normal(uint32_t q)
{
    return (q & 0x7c000000u) != 0;
}

// A Q entry is half2(64 + z, s) with bits 0x5400 | z << 4 in the low half.
__device__ __forceinline__ void split_q(uint32_t q, half2_t& z1024, half2_t& z64, half_t& s)
{
    const half2_t h = as_half2(q);
    z64             = half2_t{h[0], h[0]};
    const uint32_t zb = ((q >> 4) & 0xfu) | 0x6400u;
    z1024           = as_half2(zb | (zb << 16));
    s               = scale_is_normal(q) ? h[1] : (half_t)0.f;
}

// The (zero, scale) words of a weight tile with NQ quantisation groups come in one load, a row of sixteen lanes per group
// (row b brings group b % NQ of the tile's sixteen columns).  Here every row gets all of them: the swaps exchange rows
// between two copies of the register.  (Against a load per group: 4096 x 12288 with group size 32 at one token 11.2 -> 10.4 us.)
template<int NQ>
__device__ __forceinline__ void spread_q(uint32_t x, uint32_t* q)
{
    static_assert(NQ == 1 || NQ == 2 || NQ == 4, "group sizes 128, 64 and 32");
    if constexpr (NQ == 1) {
        q[0] = x;
    }
    else {
        const auto even_odd = __builtin_amdgcn_permlane16_swap(x, x, false, false);  // rows (0, 0, 2, 2) and (1, 1, 3, 3)
        if constexpr (NQ == 2) {
            q[0] = even_odd[0];
            q[1] = even_odd[1];
        }
        else {
            const auto e = __builtin_amdgcn_permlane32_swap(even_odd[0], even_odd[0], false, false);
            const auto o = __builtin_amdgcn_permlane32_swap(even_odd[1], even_odd[1], false, false);
            q[0] = e[0];
            q[1] = o[0];
            q[2] = e[1];
            q[3] = o[1];
        }
    }
}

// Between what the lanes of a wave write to LDS and what other lanes of the same wave read of it.  LDS serves a wave in order, so it
// is no instruction; it keeps the compiler, which sees one thread's accesses to different places, from swapping them.
__device__ __forceinline__ void wave_exchange()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// n / d for n below some bound: d == 1 has the reciprocal 0, the others floor(2^32 / d) + 1 (exact while n d < 2^32, Granlund
// and Montgomery), or 1 where the bound does not allow that and n is divided by d.
inline uint32_t reciprocal(uint64_t bound, uint32_t d)
{
    return d == 1 ? 0 : bound * d < (1ull << 32) ? (uint32_t)((1ull << 32) / d) + 1 : 1;
}
__host__ __device__ __forceinline__ uint32_t divide_by(uint32_t n, uint32_t d, uint32_t reciprocal)
{
    if (reciprocal == 0) return n;
    if (reciprocal == 1) return n / d;
    return (uint32_t)((uint64_t)n * reciprocal >> 32);
}

// The place of a workgroup of the MFMA tile kernels: which tile, and which quantisation groups of K.  Workgroups are dealt
// round-robin to the 8 XCDs; each XCD gets a contiguous run of tiles, so that its private L2 sees the reuse.  Inside a run, tiles
// go four token tiles at a time across the feature tiles: the ~64 workgroups an XCD runs concurrently then cover 4 token tiles x 16
// feature tiles, which minimises what they fetch together (a token tile of activations is four times larger than a feature tile
// of int4 weights).  split K: the groups are dealt in pairs, so that only the last split can have an odd number of them.
inline int log2_of(int splits) { return splits >= 8 ? 3 : splits >= 4 ? 2 : splits >= 2 ? 1 : 0; }
struct TilePlace {
    int tile_t, tile_n, gbeg, gend;
};
// what the tiles are divided by on the way, for `reciprocal`
inline uint32_t tile_divisor(int tiles_t, int tiles_n) { return (uint32_t)(tiles_t % 4 == 0 ? tiles_n : tiles_t); }
__host__ __device__ __forceinline__ TilePlace tile_place(int id, int tiles_t, int tiles_n, uint32_t by_divisor, int G, int split, int log_splits)
{
    TilePlace p;
    if (tiles_t % 4 == 0) {
        const int r = id >> 2, q = (int)divide_by((uint32_t)r, (uint32_t)tiles_n, by_divisor);
        p.tile_n = r - q * tiles_n;
        p.tile_t = q * 4 + (id & 3);
    }
    else {
        p.tile_n = (int)divide_by((uint32_t)id, (uint32_t)tiles_t, by_divisor);
        p.tile_t = id - p.tile_n * tiles_t;
    }
    const uint32_t pairs = ((uint32_t)G + 1) / 2;  // (K below 2^31: times eight splits in 32 bits)
    const int      from = 2 * (int)(pairs * (uint32_t)split >> log_splits), to = 2 * (int)(pairs * (uint32_t)(split + 1) >> log_splits);
    p.gbeg = G < from ? G : from;
    p.gend = G < to ? G : to;
    return p;
}

// The place of workgroup `id` of a batch kernel, of `strips` of columns times `tiles_t` blocks of tokens times K splits.  Again each
// XCD gets a contiguous run, the token tiles of a strip next to each other (they share its weights), the splits of K outermost
// (each touches its own part of the activations).
struct BatchPlace {
    int      tile_t, strip;
    uint32_t split;
};
// their reciprocals: what is divided by `tiles_t` is below all workgroups, what by `strips` below the strips of all splits
inline uint32_t by_batch_strips(uint32_t strips, uint32_t log_splits) { return reciprocal((uint64_t)strips << log_splits, strips); }
inline uint32_t by_batch_tiles(uint32_t strips, uint32_t tiles_t, uint32_t log_splits)
{
    return reciprocal(((uint64_t)strips << log_splits) * tiles_t, tiles_t);
}
__host__ __device__ __forceinline__ BatchPlace batch_place(uint32_t id, uint32_t strips, uint32_t tiles_t, uint32_t by_strips, uint32_t by_tiles_t,
                                                           uint32_t log_splits)
{
    const uint32_t total = (strips * tiles_t) << log_splits;
    if (total % 8 == 0) id = (id & 7) * (total >> 3) + (id >> 3);
    BatchPlace     p;
    const uint32_t row = divide_by(id, tiles_t, by_tiles_t);  // of strips, split by split
    p.tile_t = (int)(id - row * tiles_t);
    p.split  = log_splits ? divide_by(row, strips, by_strips) : 0;
    p.strip  = (int)(row - p.split * strips);
    return p;
}

// Split K: a workgroup announces that its partial tile is complete; true for the last of `splits`, which leaves the counter
// at zero for the next launch.  Counters are eight bytes each (`counters`: in ints).  epoch 0: they belong to a handle, which nobody else
// touches, or were cleared right before this launch.  Otherwise they are shared by every caller on the GPU, and launches that overlapped
// against the rules may have left anything in them.  Every arrival adds one, and the launch's epoch in the upper half of the word: what d arrivals of other
// launches left is taken for this launch's own only if their epochs add up to d times its own.  Those of one launch do so when
// the epochs have come round (2^19 - 1 launches), those of several also if one of them has a higher epoch than this launch and their mean is
// its own.  The sum is exact: d below the splits, at most 4095, and 19 bits of epoch.  Where the count did not start from zero, no
// arrival of the launch finds what it should, and they count again on a second counter, whose words say by their tag whose
// counts they hold; the last one clears both, so that one misuse does not spoil the launches after it and none of them has to be
// preceded by one that clears the counters.  (us a call, 8192 x 1024 at 16 tokens, split in four: tagged words and their exchange loop alone,
// a load and up to `splits` contended exchanges, 7.7; raising a tagged word and then adding to it 6.3; one addition to a word of four
// bytes, with 20 bits for the sum of the epochs, 5.1; this 4.6, half as many counters to a cache line.  All kinds of counters go
// one way, for every instruction here comes with each kernel: with a way of their own for handles the 14 KB of a batch kernel had 140 bytes more, and
// a chain of eight launches at 48 tokens took 0.9 % longer.)
__host__ __device__ __forceinline__ bool arrive_last(int* counters, int tile, int splits, int epoch)
{
    uint64_t* const counter = reinterpret_cast<uint64_t*>(counters) + tile;
    const uint64_t  one     = (uint64_t)(uint32_t)epoch << 32 | 1;
    const uint64_t  found   = __hip_atomic_fetch_add(counter, one, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const uint32_t  j       = (uint32_t)found;
    if (__builtin_expect(epoch == 0 || (j < (uint32_t)splits && (uint32_t)(found >> 32) == j * (uint32_t)epoch), 1)) {
        const bool last = j == (uint32_t)splits - 1;
        if (last) __hip_atomic_store(counter, (uint64_t)0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return last;
    }
    int* const tagged = counters + kStaticTagged + tile;
    int        seen   = __hip_atomic_load(tagged, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    for (;;) {  // (a failed exchange means that another workgroup has arrived: at most `splits` rounds)
        const int n    = (seen >> kEpochShift) == epoch ? seen & ((1 << kEpochShift) - 1) : 0;
        const int next = n == splits - 1 ? 0 : (epoch << kEpochShift) | (n + 1);
        if (__hip_atomic_compare_exchange_strong(tagged, &seen, next, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
            if (n == splits - 1) __hip_atomic_store(counter, (uint64_t)0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            return n == splits - 1;
        }
    }
}

// Measurement aid: the engine clock a kernel ran at.  One thread of a launch subtracts the core-clock counter and the
// constant-rate counter from clk[0] and clk[1] when it starts and adds them when it ends (clk[2] counts launches), so
// that nothing stays in a register in between; summed over launches, clk[0] / clk[1] x the constant rate is the
// clock.  clk == nullptr (every ordinary launch) records nothing.
__device__ __forceinline__ void clock_record_start(unsigned long long* clk, bool this_thread)
{
    if (clk != nullptr && this_thread) {
        atomicAdd(clk, 0ull - (unsigned long long)clock64());
        atomicAdd(clk + 1, 0ull - (unsigned long long)wall_clock64());
        // (the kernels that follow wait for their loads by count: nothing else may be in flight)
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
}
__device__ __forceinline__ void clock_record_stop(unsigned long long* clk, bool this_thread)
{
    if (clk != nullptr && this_thread) {
        atomicAdd(clk, (unsigned long long)clock64());
        atomicAdd(clk + 1, (unsigned long long)wall_clock64());
        atomicAdd(clk + 2, 1ull);
    }
}

}  // namespace w4a16
