// W4A16 GEMM for gfx950 for some dozens to a few hundred tokens (batched decode, short prompts): too many for the
// weight stream alone to set the time, too few to give 256 CUs large tiles.
//
// What bounds this range is the activations' way to the matrix pipes: through the CU's vector memory path (64 B per
// clock) and through LDS, where a tile kernel's waves each read the whole activation tile.  Here a workgroup owns R
// column tiles x 16 H tokens, and its eight waves share out K, not the features: a wave fetches the activation rows of
// its own quantisation groups straight from memory into a private LDS patch, reads every fragment exactly once and
// uses it for R weight tiles (the tile kernels' waves, side by side along the features, read it for one or two).  No
// wave waits for another before the end, when the eight partial tiles are added in LDS in wave order.
//
// A patch holds half a group (64 rows of K): two per wave, one being multiplied while the other is in flight, are
// 32 H KiB per workgroup, which leaves room for eight waves at up to five token blocks; a whole group per patch would
// leave room for four waves, and four waves per CU stream weights at half the rate of eight.
//
// The weights are unpacked chunk by chunk (32 rows) to the exact integers q - z in fp16, the B operand of 16 x 16 x 32
// MFMAs; the sums of half a group (of a chunk where the scale changes that often: NQ = 1, 2, 4 groups per 128-row tile,
// group sizes 128, 64, 32) are multiplied by the scale in fp32.  Nothing is rounded before the result, as in the strip
// kernels, at no more vector instructions than scaling the weights themselves takes while H is small: 9 per fragment
// instead of 13, and 4 H per half group.  A column's scale is in the lanes that hold its sums, for the price of
// sums that lie along the tokens: the reduction in LDS turns them.
//
// A grid that leaves CUs idle splits K across workgroups as well: partial tiles through the workspace, the last
// workgroup to arrive adds them in split order.
#include "pipeline.h"

namespace w4a16 {

namespace {

constexpr int kWaves = 8;

// The kernel takes its arguments one by one: the first fourteen words are preloaded into scalar registers (see
// strip_body.h), and they are what it takes to issue the first loads.  The place of a workgroup comes out of them without a
// division: three of those, one of them 64 bits wide, took longer than a K step (16 tokens, us: 8192 x 1024 split in four 6.6 -> 6.1,
// 4096 x 4096 5.7 -> 5.1, 4096 x 12288 8.7 -> 8.2; at 48 tokens 12.0 -> 11.3).
struct BatchArgs {
    const u32x4_t*  A;
    const uint16_t* X;
    const uint32_t* Q;
    int             N, T, K;
    uint32_t        strips, tiles_t;
    uint32_t        by_strips, by_tiles_t;  // their reciprocals (divide_by)
    uint32_t        how;                    // log2 of the K splits (8 bits), epilogue
    uint16_t*       C;
    const uint16_t* Rsd;
    float*          ws;
    int*            cnt;
    int             epoch;
};

// Loads of the software pipeline, waited for by count.  Their outputs are not tied to the value they replace: nothing
// reads a stage between its refill and its wait, and the register allocator then has no reason to move a value whose
// load is in flight (the build checks that it does not).
template<int IM>
__device__ __forceinline__ void load32(uint32_t& dst, uint32_t voff, const char* sbase)
{
    asm volatile("global_load_dword %0, %1, %2 offset:%3" : "=v"(dst) : "v"(voff), "s"(sbase), "n"(IM));
}
template<int IM>
__device__ __forceinline__ void load128(u32x4_t& dst, uint32_t voff, const char* sbase)
{
    asm volatile("global_load_dwordx4 %0, %1, %2 offset:%3" : "=v"(dst) : "v"(voff), "s"(sbase), "n"(IM));
}
// Memory straight into LDS, `M` KiB at lds, lds + 1024, ...: the instruction's offset moves both addresses, so one M0 value
// serves four loads (the caller's lane offsets take it out of the memory address again).
template<int M>
__device__ __forceinline__ void load_lds(uint32_t lds, const uint32_t* voff, const char* sbase)
{
    static_assert(M == 2 || M == 4, "");
    if constexpr (M == 4)
        asm volatile("s_mov_b32 m0, %5\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %4\n\tglobal_load_lds_dwordx4 %1, %4 offset:1024\n\t"
                     "global_load_lds_dwordx4 %2, %4 offset:2048\n\tglobal_load_lds_dwordx4 %3, %4 offset:3072"
                     :
                     : "v"(voff[0]), "v"(voff[1]), "v"(voff[2]), "v"(voff[3]), "s"(sbase), "s"(lds)
                     : "memory", "m0");
    else
        asm volatile("s_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %2\n\tglobal_load_lds_dwordx4 %1, %2 offset:1024"
                     :
                     : "v"(voff[0]), "v"(voff[1]), "s"(sbase), "s"(lds)
                     : "memory", "m0");
}

// wait until at most N LDS reads are in flight; the fragments named are complete then
template<int N, int H>
__device__ __forceinline__ void wait_frags(half8_t (&x)[H])
{
    static_assert(H >= 1 && H <= 5, "");
    if constexpr (H == 1) asm volatile("s_waitcnt lgkmcnt(%1)" : "+v"(x[0]) : "n"(N));
    if constexpr (H == 2) asm volatile("s_waitcnt lgkmcnt(%2)" : "+v"(x[0]), "+v"(x[1]) : "n"(N));
    if constexpr (H == 3) asm volatile("s_waitcnt lgkmcnt(%3)" : "+v"(x[0]), "+v"(x[1]), "+v"(x[2]) : "n"(N));
    if constexpr (H == 4) asm volatile("s_waitcnt lgkmcnt(%4)" : "+v"(x[0]), "+v"(x[1]), "+v"(x[2]), "+v"(x[3]) : "n"(N));
    if constexpr (H == 5)
        asm volatile("s_waitcnt lgkmcnt(%5)" : "+v"(x[0]), "+v"(x[1]), "+v"(x[2]), "+v"(x[3]), "+v"(x[4]) : "n"(N));
}

template<int R, int H, int NQ>
__global__ void __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(2, 2))) 
batch_kernel(const u32x4_t* A, const uint16_t* X, const uint32_t* Q, int N, int T, int K, uint32_t strips, uint32_t tiles_t,
             uint32_t by_strips, uint32_t by_tiles_t, uint32_t how, uint16_t* C, const uint16_t* Rsd, float* ws, int* counters, int epoch)
{
    extern __shared__ __attribute__((aligned(16))) u32x4_t smem[];  // patches [8 waves][2][16 H rows][8 chunks], then sums
    constexpr int TP     = 16 * H;
    constexpr int kPatch = TP * 128;  // bytes of half a group
    constexpr int NX     = 2 * H;     // loads per patch: 8 rows x 128 bytes each
    constexpr int NW     = 2 * R;

    const int tid  = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c    = lane & 15;
    const int b    = lane >> 4;
    const int G  = (int)((uint32_t)K / kGroup);
    const int NT = (int)((uint32_t)N / kTileN);

    const uint32_t   log_splits = how & 0xff, splits = 1u << log_splits;
    const BatchPlace at = batch_place(blockIdx.x, strips, tiles_t, by_strips, by_tiles_t, log_splits);
    const int        tile_t = at.tile_t, strip = at.strip;
    const uint32_t   split = at.split;
    // the last strip may overlap its neighbour: it then leaves the tiles below `first` to it
    const int first = strip * R;
    const int col0  = min(first, NT - R);
    const int t0    = tile_t * TP;
    const int gb    = (int)((uint32_t)G * split >> log_splits);  // (K below 2^31: G splits in 32 bits)
    const int ge    = (int)((uint32_t)G * (split + 1) >> log_splits);
    const int g0    = gb + wave;  // this wave's groups: every eighth
    const int cnt   = (int)((uint32_t)(ge - g0 + kWaves - 1) / kWaves);  // (never negative: at least one group per split)
    // The loop takes them in pairs, without a branch around anything: an odd number is padded in front with a group
    // whose activations are zeros in LDS (and whose weights are those of the first real group).
    const int pad   = cnt & 1;
    const int steps = cnt + pad;

    const uint32_t w_off = (uint32_t)(lane * 16);
    const uint32_t q_off = (uint32_t)((b % NQ * N + c) * 4);
    // Patch: row r is 128 bytes, its 16-byte chunk k at position k ^ f(r), f(r) = (r & 7) ^ (r >> 3 & 1): the 16 lanes that
    // read one chunk of 16 rows then touch every bank group equally, whether LDS serves 8 or 16 lanes per clock.
    // Load i brings rows 8i .. 8i + 7; the swizzle is applied by which chunk each lane fetches.
    // (Lane offsets are biased by 3 KiB - the load's position in its group of four, which load_lds adds to both addresses.
    // They count from the block's first token: at most 16 H - 1 rows of X and the bias, which 32 bits hold wherever they
    // hold X; from the first row of X the bias would carry the last rows of a 4 GiB X past them.)
    uint32_t x_off[NX];
#pragma unroll
    for (int i = 0; i < NX; ++i) {
        const int r = 8 * i + (lane >> 3);
        x_off[i]    = (uint32_t)min(r, T - 1 - t0) * (uint32_t)(K * 2) + (uint32_t)(((lane & 7) ^ (r & 7) ^ (r >> 3 & 1)) * 16 + (3 - i % 4) * 1024);
    }
    const uint32_t patch = __builtin_amdgcn_readfirstlane(lds_addr(smem) + (uint32_t)(wave * 2 * kPatch));
    uint32_t       xr[2];  // fragment of chunk j of a patch: row c, chunk 4j + b
#pragma unroll
    for (int j = 0; j < 2; ++j) xr[j] = patch + (uint32_t)(c * 128 + (((4 * j + b) ^ (c & 7) ^ (c >> 3)) & 7) * 16);

    // where the next requests go: weights, (zero, scale) words and activations advance by eight groups at a time
    const uint64_t w_step = (uint64_t)(uint32_t)NT * (kWaves * 1024), q_step = (uint64_t)(uint32_t)N * (NQ * kWaves * 4);
    const char*    wp = reinterpret_cast<const char*>(A) + (uint64_t)((uint32_t)g0 * (uint32_t)NT + (uint32_t)col0) * 1024;
    const char*    qp = reinterpret_cast<const char*>(Q) + ((uint64_t)((uint32_t)g0 * NQ) * (uint32_t)N + (uint64_t)(uint32_t)col0 * kTileN) * 4;
    const char*    xp = reinterpret_cast<const char*>(X) + ((uint32_t)t0 * ((uint32_t)K * 2) + (uint64_t)((uint32_t)g0 * 256)) - 3072;

    struct Stage {
        u32x4_t  w[R];
        uint32_t q[R];
    };
    auto issue_x = [&](int hf) {
        static_for<0, (NX + 3) / 4>([&](auto m) {
            constexpr int at = decltype(m)::value * 4;
            load_lds<(NX - at < 4 ? NX - at : 4)>(patch + (uint32_t)(hf * kPatch + at * 1024), x_off + at, xp + hf * 128);
        });
    };
    auto issue_w = [&](Stage& s) {
        static_for<0, R>([&](auto r) { load32<r * 64>(s.q[r], q_off, qp); });
        static_for<0, R>([&](auto r) { load128<(r % 4) * 1024>(s.w[r], w_off, wp + (r / 4) * 4096); });
    };
    auto pin = [&](Stage& s) {
#pragma unroll
        for (int r = 0; r < R; ++r) asm volatile("" : "+v"(s.w[r]));
#pragma unroll
        for (int r = 0; r < R; ++r) asm volatile("" : "+v"(s.q[r]));
    };

    const UnpackConsts uc;
    float4_t           acc[R][H];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int h = 0; h < H; ++h) acc[r][h] = float4_t{0.f, 0.f, 0.f, 0.f};

    // Four quantisation groups per tile: its words, a lane row for each group, are spread over the rows once, in the first half, a scale that
    // reads as zero being cleared before that for all of them.  (Beside two waves' MFMAs there is little room for vector instructions: 22
    // a tile and half went into its words, now 10.  Group size 32, cold weights, spread and taken apart in either half -> once, us:
    // 11008 x 4096 at 32 / 100 tokens 14.0 -> 13.3 / 26.1 -> 25.2, 4096 x 4096 at 24 / 100 6.64 -> 6.42 / 11.7 -> 11.4, 4096 x 22016 at 48 22.6
    // -> 22.2, 4096 x 12288 at 48 13.4 -> 13.2.  Blocks of 4 x 5 and 6 x 4, whose registers are all in use, gain nothing (300 tokens of a 7B layer 173.5
    // and 174.4) and keep the other way, and so do two groups or one, where there is less to save and 6 x 4 spills.)
    constexpr bool kOnce = NQ == 4 && R * H < 20;
    uint32_t       late[R][2];  // of the second half's groups
    constexpr int kSubs = NQ == 4 ? 2 : 1;  // quantisation groups in half a tile
    // Half a group: two chunks of 32 rows of K.  All fragments are read first: the patch is then free, and its next rows
    // are requested before the arithmetic, so that both patches of a wave are in flight nearly all the time (what the
    // vector memory path of a CU needs to stay busy is about 130 KiB in flight).
    auto multiply = [&](Stage& s, auto hc, auto more) {
        constexpr int hf = decltype(hc)::value;
        half8_t       xf[2][H];
        static_for<0, 2>([&](auto j) { static_for<0, H>([&](auto h) { lds_read128<hf * kPatch + h * 2048>(xf[j][h], xr[j]); }); });
        // the scales of a tile, as fp32, and what the unpacked nibbles carry beside q - z: of every quantisation group in
        // this half
        float         sf[kSubs];
        half2_t       z1024[kSubs], z64[kSubs];
        auto          words = [&](int r) {
            if constexpr (!kOnce) {
                uint32_t q[NQ];
                spread_q<NQ>(s.q[r], q);
#pragma unroll
                for (int u = 0; u < kSubs; ++u) {
                    half_t sc;
                    split_q(q[NQ == 1 ? 0 : NQ == 2 ? hf : 2 * hf + u], z1024[u], z64[u], sc);
                    sf[u] = (float)sc;
                }
            }
            else {
                uint32_t q[2];
                if constexpr (hf == 0) {
                    uint32_t all[4];
                    spread_q<4>(scale_is_normal(s.q[r]) ? s.q[r] : s.q[r] & 0xffffu, all);
                    q[0] = all[0], q[1] = all[1];
                    late[r][0] = all[2], late[r][1] = all[3];
                }
                else {
#pragma unroll
                    for (int u = 0; u < 2; ++u) {
                        q[u] = late[r][u];
                        asm volatile("" : "+v"(q[u]));  // (what is made of it is made here: the first half has no registers for it)
                    }
                }
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const half2_t h = as_half2(q[u]), z = as_half2(((q[u] >> 4) & 0xfu) | 0x6400u);
                    z64[u]   = half2_t{h[0], h[0]};
                    z1024[u] = half2_t{z[0], z[0]};
                    sf[u]    = (float)h[1];
                }
            }
        };
        auto integers = [&](int r, auto j) {
            constexpr int u = decltype(j)::value * (kSubs - 1);
            return unpack_full(s.w[r][2 * hf + decltype(j)::value], z1024[u], z64[u], uc);
        };
        words(0);
        half8_t wf = integers(0, std::integral_constant<int, 0>{});
        wait_frags<0, H>(xf[0]);
        wait_frags<0, H>(xf[1]);
        if constexpr (decltype(more)::value) issue_x(hf);
        const float4_t zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int r = 0; r < R; ++r) {
            if (r > 0) words(r);
            float4_t g[H];
            static_for<0, 2>([&](auto j) {
                if (r > 0 || decltype(j)::value > 0) wf = integers(r, j);
#pragma unroll
                for (int h = 0; h < H; ++h)
                    g[h] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xf[decltype(j)::value][h], wf, decltype(j)::value == 0 || kSubs == 2 ? zero : g[h], 0, 0, 0);
                if constexpr (decltype(j)::value == 1 || kSubs == 2) {
#pragma unroll
                    for (int h = 0; h < H; ++h)
#pragma unroll
                        for (int i = 0; i < 4; ++i) acc[r][h][i] = __builtin_fmaf(sf[decltype(j)::value * (kSubs - 1)], g[h][i], acc[r][h][i]);
                }
            });
        }
    };

    // Order of the requests: W(0) XA(0) XB(0) W(1) | XA(1) XB(1) W(2) | XA(2) XB(2) W(3) | ... - so the loads that may still
    // be in flight when a half's operands are complete are one patch and one stage of weights, until the last two steps,
    // which request less.
    Stage st[2];
    static_assert(NX + NW <= 63, "vmcnt is a 6-bit counter");
    using yes = std::true_type;
    using no  = std::false_type;
    auto step = [&](auto dc, auto more_x, auto more_w) {
        Stage& s = st[decltype(dc)::value];
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NX + (decltype(more_x)::value ? NW : 0)) : "memory");
        pin(s);
        if constexpr (decltype(more_x)::value) xp += kWaves * 256;
        multiply(s, std::integral_constant<int, 0>{}, more_x);
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(decltype(more_x)::value ? NX + NW : 0) : "memory");
        multiply(s, std::integral_constant<int, 1>{}, more_x);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (decltype(more_w)::value) {
            wp += w_step;
            qp += q_step;
            issue_w(s);
        }
    };
    using S0 = std::integral_constant<int, 0>;
    using S1 = std::integral_constant<int, 1>;
    if (steps > 0) {
        issue_w(st[0]);
        if (pad) {
            u32x4_t* const z = smem + wave * (2 * kPatch / 16) + lane;
#pragma unroll
            for (int i = 0; i < 2 * kPatch / 1024; ++i) z[i * 64] = u32x4_t{0, 0, 0, 0};
            xp -= kWaves * 256;
        }
        else {
            issue_x(0);
            issue_x(1);
            wp += w_step;
            qp += q_step;
        }
        issue_w(st[1]);
        // (a padded wave has no activation loads behind its first weights: the first step waits for all but W(1))
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NW) : "memory");
        for (int i = 2; i < steps; i += 2) {
            step(S0{}, yes{}, yes{});
            step(S1{}, yes{}, yes{});
        }
        step(S0{}, yes{}, no{});
        step(S1{}, no{}, no{});
    }

    const int    epi  = (int)(how >> 8);
    const int    tile = (int)(strip * tiles_t + tile_t);
    float4_t*    red4 = reinterpret_cast<float4_t*>(smem);
    const float* red  = reinterpret_cast<const float*>(smem);
    // split K, as in the tile kernels: stores through to memory, an arrival counter, the last one adds
    auto last_to_arrive = [&]() {
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        int* const last_flag = reinterpret_cast<int*>(smem);
        if (tid == 0) {
            const bool last = arrive_last(counters, tile, (int)splits, epoch);
            *last_flag = last;
        }
        __syncthreads();
        return *last_flag != 0;
    };
    // One or two tiles of sums are shared out by units of four tokens, more of them by tiles: a wave that adds up a whole tile
    // stores eight bytes to a lane, where units store two, but with fewer tiles than waves it is what everything waits for (us,
    // tiles and units, 16 tokens: 8192 x 1024 split in four 6.20 and 5.77; 48 tokens: 4096 x 12288 11.65 and 11.85).
    if constexpr (R * H <= 2) {
        // lane (i, c) of a unit takes column c of token i
        auto      emit = [&](int u, float v, uint16_t res) {
            const int    token = t0 + u / 4 % H * 16 + u % 4 * 4 + b, r = u / (4 * H), n = (col0 + r) * kTileN + c;
            const half_t hv = (half_t)v;
            const bool   in = token < T && col0 + r >= first;
            if (epi == kEpiSilu) {  // gate = even column, up = odd column
                const float mine = (float)hv, other = __shfl_xor(mine, 1);
                float        y = mine / (1.f + __expf(-mine)) * other;
                asm volatile("" : "+v"(y));  // (rounded to fp32 and then to fp16, as everywhere: one instruction could do both)
                const half_t o = (half_t)y;
                if (in && (c & 1) == 0) C[(int64_t)token * (N / 2) + (n >> 1)] = __builtin_bit_cast(uint16_t, o);
            }
            else if (in) {
                const half_t o = epi == kEpiAdd ? (half_t)((float)__builtin_bit_cast(half_t, res) + (float)hv) : hv;
                C[(int64_t)token * N + n] = __builtin_bit_cast(uint16_t, o);
            }
        };
        auto residual = [&](int u) -> uint16_t {
            const int token = t0 + u / 4 % H * 16 + u % 4 * 4 + b, r = u / (4 * H);
            return token < T ? Rsd[(int64_t)token * N + (col0 + r) * kTileN + c] : (uint16_t)0;
        };
        constexpr int kUnits = R * H * 4, kMine = (kUnits + kWaves - 1) / kWaves;
        float* const  mine = ws + ((int64_t)tile * (int)splits) * (kUnits * 64) + lane;
        uint16_t      res[kMine];  // (requested before the waves wait for each other)
#pragma unroll
        for (int m = 0; m < kMine; ++m) res[m] = epi == kEpiAdd && splits == 1 && wave + m * kWaves < kUnits ? residual(wave + m * kWaves) : (uint16_t)0;
        __syncthreads();
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int h = 0; h < H; ++h) red4[((wave * R + r) * H + h) * 64 + lane] = acc[r][h];
        __syncthreads();
#pragma unroll
        for (int m = 0; m < kMine; ++m) {
            const int u = wave + m * kWaves;
            if (u >= kUnits) break;
            const float* from = red + (u / 4 * 64 + u % 4 * 16 + c) * 4 + b;
            float        v    = 0.f;
#pragma unroll
            for (int s = 0; s < kWaves; ++s) v += from[s * (R * H * 256)];
            if (splits == 1) emit(u, v, res[m]);
            else __hip_atomic_store(mine + ((int64_t)(int)split * kUnits + u) * 64, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        if (splits == 1 || !last_to_arrive()) return;
#pragma unroll
        for (int m = 0; m < kMine; ++m) {
            const int u = wave + m * kWaves;
            if (u >= kUnits) break;
            float part[4];  // of up to four splits
#pragma unroll
            for (int z = 0; z < 4; ++z)
                part[z] = __hip_atomic_load(mine + ((int64_t)min(z, (int)splits - 1) * kUnits + u) * 64, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const uint16_t rs  = epi == kEpiAdd ? residual(u) : (uint16_t)0;
            float          sum = 0.f;
#pragma unroll
            for (int z = 0; z < 4; ++z)
                if (z < (int)splits) sum += part[z];
            emit(u, sum, rs);
        }
        return;
    }
    auto      emit = [&](int r, int h, const float4_t v) {  // lane (c, b): token t0 + 16h + c, features n .. n + 3
        const int token = t0 + 16 * h + c;
        if (token >= T || col0 + r < first) return;
        const int    n  = (col0 + r) * kTileN + 4 * b;
        const half_t h0 = (half_t)v[0], h1 = (half_t)v[1], h2 = (half_t)v[2], h3 = (half_t)v[3];
        if (epi == kEpiSilu) {
            const float  ga = (float)h0, ua = (float)h1, gc = (float)h2, uc2 = (float)h3;
            const half_t o0 = (half_t)(ga / (1.f + __expf(-ga)) * ua);
            const half_t o1 = (half_t)(gc / (1.f + __expf(-gc)) * uc2);
            const uint32_t o = as_u32(half2_t{o0, o1});
            __builtin_memcpy(C + (int64_t)token * (N / 2) + (n >> 1), &o, 4);
            return;
        }
        uint2 o{as_u32(half2_t{h0, h1}), as_u32(half2_t{h2, h3})};
        if (epi == kEpiAdd) {
            uint2 rr;
            __builtin_memcpy(&rr, Rsd + (int64_t)token * N + n, 8);  // (four bytes of alignment are all that is asked for)
            const half2_t r0 = as_half2(rr.x), r1 = as_half2(rr.y);
            o.x = as_u32(half2_t{(half_t)((float)r0[0] + (float)h0), (half_t)((float)r0[1] + (float)h1)});
            o.y = as_u32(half2_t{(half_t)((float)r1[0] + (float)h2), (half_t)((float)r1[1] + (float)h3)});
        }
        __builtin_memcpy(C + (int64_t)token * N + n, &o, 8);
    };

    // ---- add the eight slices in LDS, in wave order, four columns of tiles at a time (they fill the patches) ----
    // Lane (c, b) has feature c of tokens 4b .. 4b + 3 and takes over token c, features 4b .. 4b + 3: the 16 bytes of (c, b)
    // are at position 16b + (c ^ b), and the 64 lanes that read one word each then touch 64 banks.
    const int put_at = 16 * b + (c ^ b);
    int       get_at[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) get_at[i] = (16 * (c >> 2) + ((4 * b + i) ^ (c >> 2))) * 4 + (c & 3);
    constexpr int RC   = R < 4 ? R : 4;
    float* const  mine = ws + ((int64_t)tile * (int)splits) * (R * H) * 256 + lane * 4;
#pragma unroll
    for (int r0 = 0; r0 < R; r0 += RC) {
        __syncthreads();
#pragma unroll
        for (int r = r0; r < r0 + RC && r < R; ++r)
#pragma unroll
            for (int h = 0; h < H; ++h) red4[((wave * RC + r - r0) * H + h) * 64 + put_at] = acc[r][h];
        __syncthreads();
        const int n = (R - r0 < RC ? R - r0 : RC) * H;
        for (int t = wave; t < n; t += kWaves) {
            float4_t v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < kWaves; ++s)
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] += red[(s * RC * H + t) * 256 + get_at[i]];
            if ((int)splits == 1) {
                emit(r0 + t / H, t % H, v);
            }
            else {
                uint64_t* o = reinterpret_cast<uint64_t*>(mine + ((int64_t)(int)split * (R * H) + r0 * H + t) * 256);
                __hip_atomic_store(o, pack2(v[0], v[1]), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                __hip_atomic_store(o + 1, pack2(v[2], v[3]), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
    }
    if (splits == 1 || !last_to_arrive()) return;
    for (int t = wave; t < R * H; t += kWaves) {
        float4_t sum = {0.f, 0.f, 0.f, 0.f};
        for (int s0 = 0; s0 < (int)splits; s0 += 4) {
            uint64_t v[4][2];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const uint64_t* ip = reinterpret_cast<const uint64_t*>(mine + ((int64_t)min(s0 + u, (int)splits - 1) * (R * H) + t) * 256);
                v[u][0] = __hip_atomic_load(ip, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                v[u][1] = __hip_atomic_load(ip + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (s0 + u < (int)splits) {
                    sum[0] += lo_float(v[u][0]);
                    sum[1] += hi_float(v[u][0]);
                    sum[2] += lo_float(v[u][1]);
                    sum[3] += hi_float(v[u][1]);
                }
        }
        emit(t / H, t % H, sum);
    }
}

template<int R, int H, int NQ>
hipError_t launch_one(const BatchArgs& p, hipStream_t st)
{
    auto                         kfn = batch_kernel<R, H, NQ>;
    constexpr int                lds = H * 32 * 1024;
    static std::atomic<uint64_t> raised{0};
    if (lds > 64 * 1024) {
        const hipError_t e = raise_lds_limit(reinterpret_cast<const void*>(kfn), lds, raised);
        if (e != hipSuccess) return e;
    }
    return launch_kernel(kfn, dim3((p.strips * p.tiles_t) << (p.how & 0xff)), dim3(64 * kWaves), (size_t)lds, st, p.A, p.X, p.Q, p.N, p.T, p.K, p.strips,
                         p.tiles_t, p.by_strips, p.by_tiles_t, p.how, p.C, p.Rsd, p.ws, p.cnt, p.epoch);
}

// the widths that exist: up to four column tiles, and six or eight while the accumulators leave room (a workgroup costs about as
// much beside its K steps as one of them, and its activations are shared among more features: 4096 x 12288 at 128 tokens 21.4
// -> 18.8 us with 6 x 4, 8192 x 10240 35.5 -> 30.1, 8192 x 57344 at 24 tokens 65.5 -> 53.6 with 8 x 2)
constexpr bool width_exists(int r, int h)
{
    return r >= 1 && h >= 1 && h <= 5 && (r <= 4 || (r == 6 && h >= 2 && h <= 4) || (r == 8 && h == 2)) && !(r == 1 && h > 3);
}

template<int H, int NQ>
hipError_t launch_r(int r, const BatchArgs& p, hipStream_t st)
{
    switch (r) {
        case 1:
            if constexpr (width_exists(1, H)) return launch_one<1, H, NQ>(p, st);
            break;
        case 2: return launch_one<2, H, NQ>(p, st);
        case 3: return launch_one<3, H, NQ>(p, st);
        case 4: return launch_one<4, H, NQ>(p, st);
        case 6:
            if constexpr (width_exists(6, H)) return launch_one<6, H, NQ>(p, st);
            break;
        case 8:
            if constexpr (width_exists(8, H)) return launch_one<8, H, NQ>(p, st);
            break;
        default: break;
    }
    return hipErrorInvalidValue;
}

template<int NQ>
hipError_t launch_h(int r, int h, const BatchArgs& p, hipStream_t st)
{
    switch (h) {
        case 1: return launch_r<1, NQ>(r, p, st);
        case 2: return launch_r<2, NQ>(r, p, st);
        case 3: return launch_r<3, NQ>(r, p, st);
        case 4: return launch_r<4, NQ>(r, p, st);
        case 5: return launch_r<5, NQ>(r, p, st);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace

bool batch_feasible(const BatchConfig& cf, int N, int T, int K, size_t ws_bytes, int cnt_len)
{
    if (N <= 0 || T <= 0 || K <= 0 || N % kTileN != 0 || K % kGroup != 0) return false;
    if (!width_exists(cf.r, cf.h) || N / kTileN < cf.r) return false;
    // the bound of the strips, which run on this kernel up to kWidestBatchStrip tiles wide (its own offsets reach one block)
    if ((int64_t)T * K * 2 >= (1ll << 32)) return false;
    const int64_t tiles = (int64_t)((N / kTileN + cf.r - 1) / cf.r) * ((T + 16 * cf.h - 1) / (16 * cf.h));
    if (cf.splits > 1 && (K / kGroup < cf.splits || tiles > cnt_len || (int64_t)batch_scratch_bytes(cf, N, T) > (int64_t)ws_bytes)) return false;
    return (cf.splits == 1 || cf.splits == 2 || cf.splits == 4) && tiles * cf.splits < (1ll << 31);
}

size_t batch_scratch_bytes(const BatchConfig& cf, int N, int T)
{
    if (cf.splits <= 1) return 0;
    return (size_t)((N / kTileN + cf.r - 1) / cf.r) * ((T + 16 * cf.h - 1) / (16 * cf.h)) * cf.splits * cf.r * cf.h * 1024;
}

int batch_grid(const BatchConfig& cf, int N, int T)
{
    return (N / kTileN + cf.r - 1) / cf.r * ((T + 16 * cf.h - 1) / (16 * cf.h)) * cf.splits;
}

hipError_t batch_launch(const BatchConfig& cf, int nq, const GemmArgs& a, const Scratch& sc, hipStream_t st)
{
    if (cf.splits > 1 && (sc.ws == nullptr || sc.cnt == nullptr)) return hipErrorInvalidValue;
    const uint32_t strips = (uint32_t)((a.N / kTileN + cf.r - 1) / cf.r), tiles_t = (uint32_t)((a.T + 16 * cf.h - 1) / (16 * cf.h));
    const uint32_t log_splits = (uint32_t)log2_of(cf.splits);
    BatchArgs      p{reinterpret_cast<const u32x4_t*>(a.A), a.X, a.Q, a.N, a.T, a.K, strips, tiles_t, by_batch_strips(strips, log_splits),
                by_batch_tiles(strips, tiles_t, log_splits), log_splits | (uint32_t)a.epilogue << 8, a.C, a.R, sc.ws, sc.cnt, sc.epoch};
    switch (nq) {
        case 1: return launch_h<1>(cf.r, cf.h, p, st);
        case 2: return launch_h<2>(cf.r, cf.h, p, st);
        default: return launch_h<4>(cf.r, cf.h, p, st);
    }
}

}  // namespace w4a16
