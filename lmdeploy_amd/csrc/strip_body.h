// The strip decomposition of the decode (skinny) W4A16 GEMM for gfx950, shared by the one-GEMM
// kernel (gemm_strip.hip) and the persistent kernel that runs a sequence of GEMMs in one launch
// (gemm_sequence.hip).
//
// The weight matrix is a grid of 1 KiB tiles (16 columns x one 128-row quantisation group).  The
// column tiles are dealt out as evenly as possible to B workgroups: workgroup b owns a strip of R or
// R-1 adjacent column tiles over the whole of K.  Its eight waves deal the groups of K out
// round-robin; a wave walks its groups and, per group, loads the strip's R tiles (R KiB contiguous
// in the group-major tile layout) and its own activations of that group straight into registers -
// no cooperative staging, no barrier and no other wave involved until the end, when the eight
// partial strips are added in LDS in slice order.
#pragma once

#include <stddef.h>

#include "pipeline.h"

namespace w4a16 {

namespace strip {

constexpr int kWaves   = 8;  // = K slices per workgroup
constexpr int kWavesNarrow = 16;  // ... of one-tile strips at up to eight tokens
constexpr int kMaxR    = 8;  // column tiles per strip
constexpr int kMaxR32  = 8;  // ... with 32 tokens per workgroup
constexpr int kDmaTokens = 32;  // token block from which the activations go straight to LDS

struct StripParams {
    uint16_t*       C;
    const u32x4_t*  A;
    const uint16_t* X;
    const uint32_t* Q;
    const uint16_t* Rsd;
    int             N, T, K;
    int             base;  // column tiles of a narrow strip
    int             rem;   // the first `rem` strips have base + 1
    int             epilogue;  // read by kernels whose epilogue is chosen at run time (EPI == kEpiRuntime)
    int             passes;    // strips per workgroup, one after the other (strip number = pass * workgroups + workgroup)
    int             grid = 0;  // workgroups side by side
    unsigned long long* clk = nullptr;  // measurement aid (clock_record_start / _stop); null in every ordinary launch (host side)
};

// The kernels take these one by one: the first fourteen words of a kernel's arguments are put into scalar registers by the
// command processor (kernarg preloading, which does not look into a struct), so that the first loads go out at once instead of
// behind two trips to memory for the pointers.  What only the epilogue needs comes last.  A narrow matrix is done a few
// microseconds after its launch, and everything in front of the first load counts in full: with this, addresses that advance
// instead of being multiplied out for every group, and one change of the mask for up to four loads, 4096 x 4096 at one token
// went from 4.43 to 4.10 us, 4096 x 12288 7.33 -> 6.95, 4096 x 22016 11.42 -> 10.95, 11008 x 4096 7.05 -> 6.62 (cold weights).
// One list, from which their parameters, the parameters' names and their places in memory come.
#define STRIP_LIST(EACH, LAST)                                                                                         \
    EACH(const u32x4_t*, A) EACH(const uint16_t*, X) EACH(const uint32_t*, Q) EACH(int, N) EACH(int, T) EACH(int, K)   \
    EACH(int, rem) EACH(int, passes) EACH(uint32_t, how) EACH(uint16_t*, C) EACH(const uint16_t*, Rsd)                 \
    LAST(unsigned long long*, clk)
#define STRIP_PARAM(type, name) type name,
#define STRIP_LAST_PARAM(type, name) type name
#define STRIP_NAME(type, name) name,
#define STRIP_LAST_NAME(type, name) name
#define STRIP_FIELD(type, name) type name;
#define STRIP_ARGS STRIP_LIST(STRIP_PARAM, STRIP_LAST_PARAM)
#define STRIP_ARG_NAMES STRIP_LIST(STRIP_NAME, STRIP_LAST_NAME)
struct StripMemory {  // (kernel arguments lie in memory as the members of a struct do)
    STRIP_LIST(STRIP_FIELD, STRIP_FIELD)
};
// `how`: workgroups side by side (16 bits, read where they take several strips: one for each CU then), width of a narrow strip (8), epilogue (2), and whether the clock is recorded
constexpr uint32_t kHowClock = 1u << 31;
__device__ __forceinline__ StripParams strip_params(STRIP_ARGS)
{
    return StripParams{C, A, X, Q, Rsd, N, T, K, (int)(how >> 16 & 0xff), rem, (int)(how >> 28 & 3), passes, (int)(how & 0xffff)};
}
template<typename F>
hipError_t launch_strip(F* kernel, dim3 grid, dim3 block, size_t lds, hipStream_t st, const StripParams& p)
{
    const uint32_t how = ((uint32_t)p.grid & 0xffff) | (uint32_t)p.base << 16 | (uint32_t)p.epilogue << 28 | (p.clk ? kHowClock : 0);
    return launch_kernel(kernel, grid, block, lds, st, p.A, p.X, p.Q, p.N, p.T, p.K, p.rem, p.passes, how, p.C, p.Rsd, p.clk);
}
// The measurement aid's pointer is read where it is used, and not, as the compiler would have it, up front with a wait for it.
__device__ __forceinline__ unsigned long long* strip_clock()
{
    typedef __attribute__((address_space(1))) unsigned long long* counters;
    auto args = (__attribute__((address_space(4))) const char*)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(args));
    return (unsigned long long*)*(__attribute__((address_space(4))) const counters*)(args + offsetof(StripMemory, clk));
}

constexpr int kEpiRuntime = 3;  // template value: take the epilogue from StripParams

// Loads of the software pipeline: issued from inline assembly, in place ("+v"), with a scalar
// base, a per-lane 32-bit offset and an immediate, and waited for by count (the compiler would
// drain every load in flight at the loop header).  They run under an EXEC mask of all lanes or none
// (every lane is active around them, which asm_lint.py checks): with none the instructions still issue and still count in vmcnt, but touch
// neither memory nor their destination, which lets the last trips of a loop skip their refills without
// a branch - the number of loads in flight stays a compile-time constant.  Up to four loads share one change of the mask:
// the scalar instructions between the loads of all waves of a SIMD add up.
#define W4A16_MASKED(body) "s_mov_b64 exec, %[mk]\n\t" body "s_mov_b64 exec, -1"
#define W4A16_LOAD(INS, i, CACHE) INS " %[d" #i "], %[vo], %[sb] offset:%[i" #i "]" CACHE "\n\t"
#define W4A16_LOADS(INS, CACHE, N, OFF)                                                                                \
    if constexpr (N == 1)                                                                                              \
        asm volatile(W4A16_MASKED(W4A16_LOAD(INS, 0, CACHE))                                                           \
                     : [d0] "+v"(dst[0])                                                                               \
                     : [vo] "v"(voff), [sb] "s"(sbase), [mk] "s"(mask), [i0] "n"(OFF(0)));                             \
    if constexpr (N == 2)                                                                                              \
        asm volatile(W4A16_MASKED(W4A16_LOAD(INS, 0, CACHE) W4A16_LOAD(INS, 1, CACHE))                                 \
                     : [d0] "+v"(dst[0]), [d1] "+v"(dst[1])                                                            \
                     : [vo] "v"(voff), [sb] "s"(sbase), [mk] "s"(mask), [i0] "n"(OFF(0)), [i1] "n"(OFF(1)));           \
    if constexpr (N == 3)                                                                                              \
        asm volatile(W4A16_MASKED(W4A16_LOAD(INS, 0, CACHE) W4A16_LOAD(INS, 1, CACHE) W4A16_LOAD(INS, 2, CACHE))       \
                     : [d0] "+v"(dst[0]), [d1] "+v"(dst[1]), [d2] "+v"(dst[2])                                         \
                     : [vo] "v"(voff), [sb] "s"(sbase), [mk] "s"(mask), [i0] "n"(OFF(0)), [i1] "n"(OFF(1)),            \
                       [i2] "n"(OFF(2)));                                                                              \
    if constexpr (N == 4)                                                                                              \
        asm volatile(W4A16_MASKED(W4A16_LOAD(INS, 0, CACHE) W4A16_LOAD(INS, 1, CACHE) W4A16_LOAD(INS, 2, CACHE)        \
                                      W4A16_LOAD(INS, 3, CACHE))                                                       \
                     : [d0] "+v"(dst[0]), [d1] "+v"(dst[1]), [d2] "+v"(dst[2]), [d3] "+v"(dst[3])                      \
                     : [vo] "v"(voff), [sb] "s"(sbase), [mk] "s"(mask), [i0] "n"(OFF(0)), [i1] "n"(OFF(1)),            \
                       [i2] "n"(OFF(2)), [i3] "n"(OFF(3)));

// N (zero, scale) words, of tiles FIRST, FIRST + 1, ... of a strip
template<int N, int FIRST>
__device__ __forceinline__ void mload_q(uint32_t* dst, uint32_t voff, const void* sbase, uint64_t mask)
{
#define W4A16_OFF(i) (FIRST + (i)) * 64
    W4A16_LOADS("global_load_dword", "", N, W4A16_OFF)
#undef W4A16_OFF
}
// N adjacent weight tiles
template<int N>
__device__ __forceinline__ void mload_w(u32x4_t* dst, uint32_t voff, const void* sbase, uint64_t mask)
{
#define W4A16_OFF(i) (i) * 1024
    W4A16_LOADS("global_load_dwordx4", " nt", N, W4A16_OFF)
#undef W4A16_OFF
}
__device__ __forceinline__ void mload128(u32x4_t& dst, uint32_t voff, const void* sbase, uint64_t mask)
{
    asm volatile(W4A16_MASKED("global_load_dwordx4 %[d], %[vo], %[sb]\n\t") : [d] "+v"(dst) : [vo] "v"(voff), [sb] "s"(sbase), [mk] "s"(mask));
}
// the same at agent scope: for data that another workgroup of the same launch, possibly on another
// XCD (each XCD has its own L2), has written with agent-scope stores
__device__ __forceinline__ void mload128_agent(u32x4_t& dst, uint32_t voff, const void* sbase, uint64_t mask)
{
    asm volatile(W4A16_MASKED("global_load_dwordx4 %[d], %[vo], %[sb] sc1\n\t") : [d] "+v"(dst) : [vo] "v"(voff), [sb] "s"(sbase), [mk] "s"(mask));
}

__device__ __forceinline__ void mload128_lds(uint32_t lds_base, uint32_t voff, const void* sbase, uint64_t mask)
{
    asm volatile("s_mov_b32 m0, %[lb]\n\t" W4A16_MASKED("global_load_lds_dwordx4 %[vo], %[sb]\n\t")
                 :
                 : [vo] "v"(voff), [sb] "s"(sbase), [mk] "s"(mask), [lb] "s"(lds_base)
                 : "m0", "memory");
}
// Everything one wave holds for one group: R weight tiles, their Q words, and the activations of
// the group (NX loads of four token rows x 256 bytes each, one 16-byte chunk per lane).
// (With 2 or 4 quantisation groups per weight tile, tile r's words are spread over the lanes of q[r]: spread_q.)
template<int R, int NX>
struct Stage {
    u32x4_t  w[R];
    uint32_t q[R];
    u32x4_t  x[NX > 0 ? NX : 1];  // (NX = 0: the activations go straight to LDS)
};

// The whole kernel for a strip of exactly R column tiles starting at tile `col0`.
// SEQ: the GEMM is one of a sequence inside a persistent launch.  Its activations and residual may
// have been written by other workgroups of the same launch, so they are read at agent scope, and its
// output is written at agent scope (write-through) for the same reason; the token block is 0.  The
// weights and (scale, zero) words of the first groups are requested at once; `inputs_ready()` is then
// called by every wave (it returns, workgroup-wide, when activations and residual may be read and LDS
// may be overwritten) before anything else is touched.
struct NoWait {
    __device__ __forceinline__ void operator()() const {}
};
// NW = waves of the workgroup = slices of K.
// NQ: quantisation groups per 128-row weight tile (group sizes 128, 64, 32 = NQ 1, 2, 4).  The weight layout does
// not depend on it; Q then has NQ rows per tile row, and every 128 / NQ rows of a tile have their own scale and
// zero point: NQ shorter MFMA chains per tile, each scaled into the accumulator by itself.
// DD: groups in flight per wave.  Two, unless the strip is so wide that two groups of it from every wave of the CU
// are more than the memory system takes at once (the launcher decides); then one.
template<int R, int TP, int EPI, bool SEQ = false, int NW = kWaves, typename Ready = NoWait, int NQ = 1, int DD = 2>
__device__ __forceinline__ void strip_body(const StripParams& p, int col0, u32x4_t* smem, Ready&& inputs_ready = Ready{})
{
    const int tid  = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c    = lane & 15;
    const int b    = lane >> 4;
    const int N = p.N, T = p.T, K = p.K;
    const int G  = (int)((uint32_t)K / kGroup);
    const int NT = (int)((uint32_t)N / kTileN);
    // H row blocks of 16 tokens share every unpacked weight (H = 2 for the 32-token variant)
    constexpr int H  = TP > 16 ? TP / 16 : 1;
    const int     t0 = SEQ ? 0 : blockIdx.y * (16 * H);
    const int     Tl = min(16 * H, T - t0);

    // this wave's groups: wave, wave + 8, wave + 16, ...  Interleaved rather than blocked, so that
    // at any moment the whole chip reads one contiguous run of a few dozen group rows of the
    // group-major weight array instead of eight distant ones (measured: DRAM prefers that).
    const int cnt = (int)((uint32_t)(G - wave + NW - 1) / NW);  // 0 if wave >= G
    // per-lane byte offsets; everything that depends on the group is scalar
    const uint32_t w_off = (uint32_t)(lane * 16);                    // + (g * NT + col0 + r) * 1024
    const uint32_t q_off = (uint32_t)((b % NQ * N + c) * 4);         // + (g * NQ * N + (col0 + r) * 16) * 4
    // Activations: load i of a group fetches token rows 4i .. 4i+3, lane l the 16-byte chunk l % 16
    // of row 4i + l / 16 - a quarter wave reads one contiguous 256-byte row, two cache lines.
    // (Fetching straight in MFMA operand order, lane (c, b) = row c, makes every quarter wave
    // touch 16 rows; the cache looks up one line per row and request, and at 16 tokens that cost
    // more than the weight stream.)  The wave turns the rows into operand order through a private
    // patch of LDS; chunk p of row r sits at position p ^ r so that both the row-wise writes and
    // the column-wise reads are free of bank conflicts.
    // With 32 tokens the rows go from global memory straight into the patch instead (no registers, no
    // LDS write), one patch per group in flight; the swizzle is then applied on the way in: the lane
    // that lands at position p of row r fetches chunk p ^ r.
    constexpr int  D    = DD;  // groups in flight per wave
    static_assert(D == 2 || (D == 1 && !SEQ), "one or two groups in flight");
    constexpr bool XDMA = TP >= kDmaTokens && !SEQ;
    constexpr int  NX   = TP / 4;
    constexpr int  NXR  = XDMA ? 0 : NX;  // activation loads that land in registers
    uint32_t       x_off[NX];
#pragma unroll
    for (int i = 0; i < NX; ++i) {
        const int r     = 4 * i + (lane >> 4);
        const int chunk = XDMA ? ((lane & 15) ^ (r & 15)) : (lane & 15);
        x_off[i]        = (uint32_t)min(t0 + r, T - 1) * (uint32_t)(K * 2) + (uint32_t)(chunk * 16);
    }
    u32x4_t* const xw = smem + wave * (TP * 16) * (XDMA ? D : 1);  // this wave's patch(es): [TP rows][16 chunks]
    const uint32_t xw_lds = __builtin_amdgcn_readfirstlane(lds_addr(xw));
    int            xw_at[NX], xr_at[H][4];
#pragma unroll
    for (int i = 0; i < NX; ++i) {
        const int r = 4 * i + (lane >> 4);
        xw_at[i]    = r * 16 + ((lane & 15) ^ (r & 15));
    }
#pragma unroll
    for (int h = 0; h < H; ++h)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int r = 16 * h + (c & (TP - 1));  // MFMA rows >= TP repeat a lower row: they only feed outputs that are never stored
            xr_at[h][j] = r * 16 + ((4 * j + b) ^ (r & 15));
        }

    // Where the next requests go.  The first stages are requested unmasked, by waves that have no group for them too: those
    // ask for their last group again, or for the last group there is.
    const uint32_t gw = (uint32_t)min(wave, G - 1);
    const char*    wp = reinterpret_cast<const char*>(p.A) + (uint64_t)(gw * (uint32_t)NT + (uint32_t)col0) * 1024;
    const char*    qp = reinterpret_cast<const char*>(p.Q) + ((uint64_t)(gw * NQ) * (uint32_t)N + (uint64_t)(uint32_t)col0 * kTileN) * 4;
    const char*    xp = reinterpret_cast<const char*>(p.X) + (uint64_t)gw * 256;
    const uint64_t w_step = (uint64_t)(uint32_t)NT * (NW * 1024), q_step = (uint64_t)(uint32_t)N * (NQ * NW * 4);

    // All loads of the next group into stage s (number d); a mask of 0 turns them into no-ops that still count.
    using StageT = Stage<R, NXR>;
    static_assert(NQ == 1 || ((NQ == 2 || NQ == 4) && H == 1), "group sizes 128, 64 and 32");
    auto issue_x = [&](StageT& s, int d, uint64_t mask) {
        static_for<0, NX>([&](auto i) {
            if constexpr (XDMA) mload128_lds(xw_lds + (uint32_t)(d * TP * 256 + i * 1024), x_off[i], xp, mask);
            else if constexpr (SEQ) mload128_agent(s.x[i], x_off[i], xp, mask);
            else mload128(s.x[i], x_off[i], xp, mask);
        });
    };
    auto issue_wq = [&](StageT& s, uint64_t mask) {
        static_for<0, (R + 3) / 4>([&](auto r4) { mload_q<(R - r4 * 4 < 4 ? R - r4 * 4 : 4), r4 * 4>(s.q + r4 * 4, q_off, qp, mask); });
        // (the tiles of a group are contiguous; immediates reach 4 KiB, so every fourth tile gets a new base)
        static_for<0, (R + 3) / 4>([&](auto r4) { mload_w<(R - r4 * 4 < 4 ? R - r4 * 4 : 4)>(s.w + r4 * 4, w_off, wp + r4 * 4096, mask); });
    };
    auto issue = [&](StageT& s, int d, uint64_t mask) {
        issue_x(s, d, mask);
        issue_wq(s, mask);
    };
    constexpr uint64_t kAll = ~0ull;
    constexpr int kLoads = 2 * R + NX;  // loads per stage

    const UnpackConsts uc;
    // B operand of the chain that sums the activations: -(unpack offset) in columns 0-7, -1 in columns 8-15
    half8_t bsum;
    {
        const half_t lo = c < 8 || NQ > 1 ? (half_t)-1024.f : (half_t)-1.f, hi = c < 8 || NQ > 1 ? (half_t)-64.f : (half_t)-1.f;
        bsum = half8_t{lo, lo, hi, hi, lo, lo, hi, hi};
    }
    // (more than one group per tile: -(unpack offset) in all columns there, and A operands with -1 in the rows of one lane row)
    half8_t asum[NQ];
#pragma unroll
    for (int sub = 0; sub < NQ; ++sub) {
        const half_t v = c / 4 == sub ? (half_t)-1.f : (half_t)0.f;
        asum[sub]      = half8_t{v, v, v, v, v, v, v, v};
    }
    float4_t           acc[H][R];
#pragma unroll
    for (int h = 0; h < H; ++h)
#pragma unroll
        for (int r = 0; r < R; ++r) acc[h][r] = float4_t{0.f, 0.f, 0.f, 0.f};

    // One tile of one group.  U tiles are worked on at a time with their MFMA chains interleaved:
    // a chain is four or eight dependent MFMAs, and a dependent MFMA cannot issue before its predecessor
    // has left the pipe.
    auto compute = [&](StageT& s, auto dc) {
        half8_t xf[H][4];
        if constexpr (XDMA) {
            // the group's rows are in patch d: row block h is 4 KiB further on
            constexpr int d = decltype(dc)::value;
            static_for<0, H * 4>([&](auto hj) {
                constexpr int h = decltype(hj)::value / 4, j = decltype(hj)::value % 4;
                lds_read128<d * TP * 256 + h * 4096>(xf[h][j], xw_lds + (uint32_t)(xr_at[0][j] * 16));
            });
            // (every fragment exactly once: a register named twice would be copied before the wait)
            static_assert(H <= 2, "the wait below names the fragments of at most two row blocks");
            if constexpr (H == 1)
                asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(xf[0][0]), "+v"(xf[0][1]), "+v"(xf[0][2]), "+v"(xf[0][3]));
            else
                asm volatile("s_waitcnt lgkmcnt(0)"
                             : "+v"(xf[0][0]), "+v"(xf[0][1]), "+v"(xf[0][2]), "+v"(xf[0][3]), "+v"(xf[H - 1][0]),
                               "+v"(xf[H - 1][1]), "+v"(xf[H - 1][2]), "+v"(xf[H - 1][3]));
        }
        else {
#pragma unroll
            for (int i = 0; i < NXR; ++i) xw[xw_at[i]] = s.x[i];
            wave_exchange();
#pragma unroll
            for (int h = 0; h < H; ++h)
#pragma unroll
                for (int j = 0; j < 4; ++j) xf[h][j] = __builtin_bit_cast(half8_t, xw[xr_at[h][j]]);
        }
        constexpr int U  = 2;
        constexpr int JN = 4 / NQ;  // k32 chunks per quantisation group
        auto unpacked = [&](uint32_t word) {
            uint32_t v[4];
            unpack_offset(word, v, uc);
            half8_t wf;
            wf[0] = as_half2(v[0])[0]; wf[1] = as_half2(v[0])[1]; wf[2] = as_half2(v[1])[0]; wf[3] = as_half2(v[1])[1];
            wf[4] = as_half2(v[2])[0]; wf[5] = as_half2(v[2])[1]; wf[6] = as_half2(v[3])[0]; wf[7] = as_half2(v[3])[1];
            return wf;
        };
        if constexpr (NQ > 1 && R == 1) {
            // one tile: as for one group below, a second chain per group with -(o + z) as its B operand
            const uint32_t qw = s.q[0];  // half2(64 + z, scale) of group b % NQ
            float          sb = scale_is_normal(qw) ? (float)as_half2(qw)[1] : 0.f;
            asm volatile("" : "+v"(sb));  // (nothing of the word may stay live past the refill)
            uint32_t q[NQ], sf[NQ];
            spread_q<NQ>(qw, q);
            spread_q<NQ>(__builtin_bit_cast(uint32_t, sb), sf);
            float4_t g4[NQ];
#pragma unroll
            for (int sub = 0; sub < NQ; ++sub) {
                const half2_t  h2 = as_half2(q[sub]), n64 = half2_t{h2[0], h2[0]} * half2_t{(half_t)-1.f, (half_t)-1.f};
                const half2_t  z2 = as_half2(((q[sub] >> 4) & 0xfu) * 0x10001u + 0xE400E400u);  // -(1024 + z) twice
                const half8_t  bz = {z2[0], z2[1], n64[0], n64[1], z2[0], z2[1], n64[0], n64[1]};
                g4[sub] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int j = sub * JN; j < (sub + 1) * JN; ++j) g4[sub] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xf[0][j], bz, g4[sub], 0, 0, 0);
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) g4[j / JN] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xf[0][j], unpacked(s.w[0][j]), g4[j / JN], 0, 0, 0);
#pragma unroll
            for (int sub = 0; sub < NQ; ++sub) acc[0][0] += __builtin_bit_cast(float, sf[sub]) * g4[sub];
            return;
        }
        if constexpr (NQ > 1) {
            // sum x (q + o) - P - z S = sum x (q - z), as below, with NQ sums, scales and zero points per tile: what bounds
            // these strips is the arithmetic around the MFMAs, so as little of it as possible is done per quantisation
            // group.  -P starts every chain (an MFMA whose B operand is -o in all columns has it where the chain wants it).
            // The zero points' share, sum over the groups of (s z) x (-S), is a matrix product of depth NQ: -S comes out of
            // its MFMAs with group b in lane row b, s z is computed in the layout that the words are loaded in - all groups
            // of a tile at once - and one fp32 MFMA of depth four adds it.  Only s is spread over the rows.
            // (group size 32, us at one token, before and after: 4096 x 12288 10.4 -> 9.0, 4096 x 22016 15.6 -> 13.6, 8192 x 57344
            // 59.0 -> 49.7; group size 64: 9.2 -> 8.5, 12.6 -> 12.3, 46.4 -> 45.2)
            float4_t nP[NQ], nS = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int sub = 0; sub < NQ; ++sub) {
                nP[sub] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int j = sub * JN; j < (sub + 1) * JN; ++j) {
                    nP[sub] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xf[0][j], bsum, nP[sub], 0, 0, 0);
                    nS      = __builtin_amdgcn_mfma_f32_16x16x32_f16(asum[sub], xf[0][j], nS, 0, 0, 0);
                }
            }
#pragma unroll
            for (int r0 = 0; r0 < R; r0 += U) {
                float4_t g4[U][NQ];
                uint32_t sf[U][NQ];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    if (r0 + u < R) {
                        const uint32_t qw = s.q[r0 + u];  // half2(64 + z, scale) of group b % NQ
                        float          sb = scale_is_normal(qw) ? (float)as_half2(qw)[1] : 0.f;
                        float          zb = (float)((qw >> 4) & 0xfu) * sb;
                        asm volatile("" : "+v"(sb), "+v"(zb));  // (nothing of the word may stay live past the refill)
                        spread_q<NQ>(__builtin_bit_cast(uint32_t, sb), sf[u]);
                        acc[0][r0 + u] = __builtin_amdgcn_mfma_f32_16x16x4f32(nS[0], zb, acc[0][r0 + u], 0, 0, 0);
                    }
                }
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int u = 0; u < U; ++u)
                        if (r0 + u < R)
                            g4[u][j / JN] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xf[0][j], unpacked(s.w[r0 + u][j]), j % JN ? g4[u][j / JN] : nP[j / JN], 0, 0, 0);
#pragma unroll
                for (int sub = 0; sub < NQ; ++sub)
#pragma unroll
                    for (int u = 0; u < U; ++u)
                        if (r0 + u < R) acc[0][r0 + u] += __builtin_bit_cast(float, sf[u][sub]) * g4[u][sub];
            }
            return;
        }
        // What the unpack offsets and the zero points add to every dot product depends on the weights only
        // through z: sum x (q + o) - P - z S = sum x (q - z) with P = sum o x (o = 1024 under the low-nibble
        // pairs, 64 under the high ones) and S = sum x.  A strip of two or more tiles takes P and S from one
        // MFMA chain (columns 0-7 of its B operand hold -o, columns 8-15 hold -1) and
        // every tile starts its own chain from -P: four MFMAs per tile instead of eight.  A strip of one tile
        // runs the second chain per tile, with -(o + z) as its B operand; that costs it no more MFMAs and
        // saves the exchange between the two halves of the columns.
        constexpr bool kSums = R >= 2;
        float4_t nP[H], nS[H];
        if constexpr (kSums) {
#pragma unroll
            for (int h = 0; h < H; ++h) {
                float4_t ps = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    ps = __builtin_amdgcn_mfma_f32_16x16x32_f16(xf[h][j], bsum, ps, 0, 0, 0);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    // the lane eight columns away, row_ror:8 (source given as the old value too: with a constant
                    // there the compiler merges the four moves into one)
                    const int   mine  = __builtin_bit_cast(int, (float)ps[i]);
                    const float other = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(mine, mine, 0x128, 0xf, 0xf, false));
                    nP[h][i] = c < 8 ? ps[i] : other;
                    nS[h][i] = c < 8 ? other : ps[i];
                }
            }
        }
#pragma unroll
        for (int r0 = 0; r0 < R; r0 += U) {
            float4_t g4[H][U];
            float    sf[U], zf[U];
            half8_t  bz[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int      r  = r0 + u < R ? r0 + u : R - 1;
                const uint32_t qw = s.q[r];  // half2(64 + z, scale): z is bits 4-7
                const half2_t  h2 = as_half2(qw);
                if constexpr (kSums) {
                    zf[u] = (float)((qw >> 4) & 0xfu);
                    asm volatile("" : "+v"(zf[u]));
                }
                else {
                    // -(1024 + z) under the low-nibble pairs, -(64 + z) under the high-nibble pairs
                    const half2_t  n64 = half2_t{h2[0], h2[0]} * half2_t{(half_t)-1.f, (half_t)-1.f};
                    const uint32_t zb  = ((qw >> 4) & 0xfu) * 0x10001u + 0xE400E400u;  // -(1024 + z) twice
                    bz[u][0] = as_half2(zb)[0]; bz[u][1] = as_half2(zb)[1]; bz[u][2] = n64[0]; bz[u][3] = n64[1];
                    bz[u][4] = bz[u][0]; bz[u][5] = bz[u][1]; bz[u][6] = bz[u][2]; bz[u][7] = bz[u][3];
                }
                // Convert the scale now and hide it from the optimiser: otherwise the conversion is
                // folded into the final multiply-add, the Q word stays live past the refill of this
                // stage, and the refill lands in a copy that is moved back while still in flight.
                sf[u] = scale_is_normal(qw) ? (float)h2[1] : 0.f;
                asm volatile("" : "+v"(sf[u]));
#pragma unroll
                for (int h = 0; h < H; ++h) {
                    if constexpr (kSums) g4[h][u] = nP[h];
                    else g4[h][u] = float4_t{0.f, 0.f, 0.f, 0.f};
                }
            }
            if constexpr (!kSums) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
#pragma unroll
                    for (int u = 0; u < U; ++u)
#pragma unroll
                        for (int h = 0; h < H; ++h)
                            if (r0 + u < R) g4[h][u] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xf[h][j], bz[u], g4[h][u], 0, 0, 0);
                }
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    if (r0 + u < R) {
                        const half8_t wf = unpacked(s.w[r0 + u][j]);
#pragma unroll
                        for (int h = 0; h < H; ++h)
                            g4[h][u] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xf[h][j], wf, g4[h][u], 0, 0, 0);
                    }
                }
            }
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int h = 0; h < H; ++h)
                    if (r0 + u < R) {
                        if constexpr (kSums) acc[h][r0 + u] += sf[u] * (g4[h][u] + zf[u] * nS[h]);
                        else acc[h][r0 + u] += sf[u] * g4[h][u];
                    }
        }
    };
    // Wait until the stage's loads are complete (loads return in order: at most `kLoads` younger
    // ones may still be in flight, or none after the last issue), then pin its registers below
    // the wait.
    auto pin = [&](StageT& s) {
#pragma unroll
        for (int r = 0; r < R; ++r) asm volatile("" : "+v"(s.w[r]));
#pragma unroll
        for (int r = 0; r < R; ++r) asm volatile("" : "+v"(s.q[r]));
#pragma unroll
        for (int i = 0; i < NXR; ++i) asm volatile("" : "+v"(s.x[i]));
    };
    // Two groups in flight per wave.  (Three or four fit the register file for narrow strips but
    // measured slower: the unrolled loop body grows with D and is executed only once or twice.)
    static_assert((D - 1) * kLoads <= 63, "vmcnt is a 6-bit counter");
    StageT st[D];

    // One group: wait for the stage (exactly D - 1 younger stages are in flight behind it), use
    // it, refill it.  Nothing of a stage may be live when it is refilled (the refill is in place
    // and asynchronous), so the scheduler must not move the stage's arithmetic below its refill.
    auto step = [&](auto dc, bool use, int left) {  // (a group to refill with: left < 0)
        constexpr int d = decltype(dc)::value;
        StageT&       s = st[d];
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((D - 1) * kLoads) : "memory");
        pin(s);
        if (use) compute(s, dc);
        __builtin_amdgcn_sched_barrier(0);
        wp += w_step;
        qp += q_step;
        xp += NW * 256;
        issue(s, d, (uint64_t)(int64_t)__builtin_amdgcn_readfirstlane(left >> 31));
    };

    const bool second = D == 2 && cnt > 1;  // a second group to advance to
    if constexpr (SEQ) {
        // weights first (they depend on nothing), then wait for the producers of the activations, then the
        // activations; all of it complete before the loop, whose counted waits assume whole stages in order
        issue_wq(st[0], kAll);
        if constexpr (D == 2) {
            wp += second ? w_step : 0;
            qp += second ? q_step : 0;
            issue_wq(st[1], kAll);
        }
        inputs_ready();
        issue_x(st[0], 0, kAll);
        if constexpr (D == 2) {
            xp += second ? NW * 256 : 0;
            issue_x(st[1], 1, kAll);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    else {
        issue(st[0], 0, kAll);
        if constexpr (D == 2) {
            wp += second ? w_step : 0;
            qp += second ? q_step : 0;
            xp += second ? NW * 256 : 0;
            issue(st[1], 1, kAll);
        }
    }
    // D groups per trip, so that each stage keeps its registers; all conditions are wave-uniform
    // and none of them surrounds a load.
    for (int i = 0; i < cnt; i += D) {
        static_for<0, D>([&](auto dc) {
            constexpr int d = decltype(dc)::value;
            step(dc, i + d < cnt, i + d + D - cnt);
        });
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the masked refills of the last trip
    static_for<0, D>([&](auto d) { pin(st[d]); });  // (whose registers are nobody else's until then)

    // ---- add the slices in LDS, in slice order: a unit is four tokens of a tile, lane (i, c) of a wave takes column c of token i ----
    // (One wave per tile, four tokens to a lane, was the first way: the last wave of a workgroup then ran sixteen 128-bit reads and
    // four masked stores by itself, and for a residual a trip to memory in front of them, 1200 of a narrow kernel's 4700 cycles.
    // us, 11008 x 4096 with a residual at 4 / 8 tokens 7.31 -> 6.75 / 8.13 -> 7.60, 4096 x 4096 at one 4.06 -> 3.88; group size 64
    // at 4 tokens, four Llama-2-7B matrices 32.6 -> 31.2, group size 32 35.8 -> 34.0.)
    constexpr int kQuads = TP < 16 ? TP / 4 : 4, kUnits = R * H * kQuads, kMine = (kUnits + NW - 1) / NW;
    const int     epi = EPI == kEpiRuntime ? p.epilogue : EPI;
    int           row[kMine], col[kMine];
    uint16_t      res[kMine];  // (requested before the waves wait for each other)
#pragma unroll
    for (int m = 0; m < kMine; ++m) {
        const int u = wave + m * NW;
        row[m]      = u / kQuads % H * 16 + u % kQuads * 4 + b;
        col[m]      = (col0 + u / (kQuads * H)) * kTileN + c;
        res[m]      = 0;
        if (epi == kEpiAdd && u < kUnits && row[m] < Tl) {
            const uint16_t* at = p.Rsd + (int64_t)(t0 + row[m]) * N + col[m];
            if constexpr (SEQ) res[m] = __hip_atomic_load(at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            else res[m] = *at;
        }
    }
    // red[slice][r][h][lane] as float4, over the activation patches: every wave must be done with its own
    __syncthreads();
    if (4 * b < TP) {
        float4_t* red4 = reinterpret_cast<float4_t*>(smem);
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int h = 0; h < H; ++h) red4[((wave * R + r) * H + h) * 64 + lane] = acc[h][r];
    }
    __syncthreads();
    const float* red = reinterpret_cast<const float*>(smem);
#pragma unroll
    for (int m = 0; m < kMine; ++m) {
        const int u = wave + m * NW;
        if (u >= kUnits) break;
        // (unit u of a slice: quad u % kQuads of the 64 lanes' float4 of tile and row block u / kQuads)
        const float* from = red + (u / kQuads * 64 + u % kQuads * 16 + c) * 4 + b;
        float        v    = 0.f;
#pragma unroll
        for (int s = 0; s < NW; ++s) v += from[s * (R * H * 256)];

        // ---- epilogue ----
        const half_t hv    = (half_t)v;
        const int    token = t0 + row[m], n = col[m];
        const bool   in    = row[m] < Tl;
        auto put = [&](int64_t at, half_t o) {
            const uint16_t bits = __builtin_bit_cast(uint16_t, o);
            if constexpr (SEQ) __hip_atomic_store(p.C + at, bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            else p.C[at] = bits;
        };
        if (epi == kEpiSilu) {
            // gate = even column, up = odd column: fetch the neighbour lane's value
            const float mine  = (float)hv;
            const float other = __shfl_xor(mine, 1);
            if (in && (c & 1) == 0) put((int64_t)token * (N / 2) + (n >> 1), (half_t)(mine / (1.f + __expf(-mine)) * other));
        }
        else if (in) {
            const int64_t at = (int64_t)token * N + n;
            if (epi == kEpiGemm) put(at, hv);
            else put(at, (half_t)((float)__builtin_bit_cast(half_t, res[m]) + (float)hv));
        }
    }
}

}  // namespace strip

}  // namespace w4a16
