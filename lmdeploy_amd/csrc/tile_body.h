// W4A16 GEMM for gfx950 for a hundred tokens and more: bound by the fp16 MFMA rate (and, from a few hundred tokens on, by
// the power it takes).  Included by one translation unit per quantisation group size.
//
// A workgroup of four waves, one per SIMD, computes a (16*TTILES tokens) x (64*NTW features) output tile; the waves split
// the features.  Each loads its weight tiles straight from global memory into registers (one 128-bit load per lane and
// tile), dequantises them to the reference's exact fp16 weight fp16_rn((q - z) * s) and uses them as the A operand.
// The activations of the tile go from global memory directly into LDS (no registers, no ds_write), one 128-wide K step
// per stage, and are read as the B operand by all waves.
//
// What a tile has to be: the waves of a CU read TTILES fragments of 1 KiB per 32 rows of K each, for TTILES x NTW MFMAs
// (counted in 16 x 16 x 32).  With NTW = 1 or 2 that is up to what LDS delivers, and with eight narrow waves per CU (the
// kernels of gemm_prefill.hip) the matrix pipes cannot be fed any faster; NTW = 4 halves it.  A wave of 16 x 4 tiles
// needs 256 accumulators and so a SIMD to itself, which in turn asks for 32 x 32 MFMAs (see below).
// Llama-2-70B gate_up at 2048 tokens: 1.53 -> 1.43 ms (1.35 PFLOP/s at 1.6 GHz, the power limit; matrix pipes 77 % busy).
//
// The K loop is one hand-scheduled instruction stream per wave: every MFMA is followed by its share of the NEXT chunk's
// dequantisation, LDS fragment reads and global loads.  The MFMAs are inline assembly with the accumulators tied in place
// in AGPRs; loads are inline assembly waited for by count.
#pragma once

#include "pipeline.h"

namespace w4a16 {

namespace {

// Direct-to-LDS loads whose address in LDS (M0) serves several requests, each a statement of its own: the build's assembly
// check verifies that nothing else writes M0 in a kernel that relies on this.
__device__ __forceinline__ void set_m0(uint32_t v)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0" : : "s"(v) : "memory", "m0");
}
template<int OFF>
__device__ __forceinline__ void gload_lds128_m0(uint32_t voff, const void* sbase)
{
    asm volatile("global_load_lds_dwordx4 %0, %1 offset:%2" : : "v"(voff), "s"(sbase), "n"(OFF) : "memory");
}
// g / (1 + exp(-g)) with the quotient rounded as a division rounds it: the approximate quotient and one correction by its exact
// remainder (Markstein), special cases by the instruction that ends the compiler's division too.  Without the scaling that
// a division of any two numbers needs: the denominator is at least one, and where its reciprocal is no longer a normal
// number the result is zero in fp16.  The scaling goes through VCC, one quotient after the other, and a wave of this kernel
// has its SIMD to itself: a 7B layer at 2048 tokens takes 714 us with `/`, 711 with this and 707 with the reciprocal alone, which
// rounds one half in thirty thousand differently from the other kernels.
__device__ __forceinline__ float silu_quotient(float g)
{
    const float d = 1.f + __expf(-g), r = __builtin_amdgcn_rcpf(d), q = g * r;
    return __builtin_amdgcn_div_fixupf(__builtin_fmaf(__builtin_fmaf(-d, q, g), r, q), d, g);
}

// A wave computes 16 TTILES tokens x 16 NTW features in blocks of 32 x 32 (v_mfma_f32_32x32x16_f16); the four waves of a
// workgroup are side by side along the features.  D = groups in flight per wave (2 or 4): the loads of group g + D are issued while group g is being
// multiplied.  NQ = quantisation groups per 128-row weight tile: 1 (group size 128), 2 (64) or 4 (32); with NQ > 1 every
// k32 chunk (or pair of chunks) has its own scale and zero point, taken from the tile's NQ Q words right before the
// chunk is dequantised instead of once per K step.
//
// Register budget: one wave per SIMD, 512 registers, the accumulators in AGPRs.  Stating it keeps the allocator from
// squeezing the kernel into fewer VGPRs and parking values in AGPRs, which is fatal here: a register parked while an
// inline-assembly load into it is still in flight is handed to another value, and the load then lands on that value
// (the build rejects kernels that use AGPRs beyond their accumulators).
// Why 32 x 32: a wave that has a SIMD to itself issues one vector instruction per eight cycles; behind a 16 x 16 x 32 MFMA (16
// cycles) there is room for one other instruction, a second one costs four and a third eight more.  The kernel needs
// 0.8 vector instructions, a quarter of an LDS read and half a request or wait per 16 cycles.  Behind a 32 x 32 x 16 MFMA
// (32 cycles, half as many of them) they fit.  Two 16-column weight tiles make one operand: a lane exchange between
// the two packed words (v_permlane16_swap) gives one word with rows 0..7 and 16..23 of both tiles' chunk and one with rows
// 8..15 and 24..31; which rows of K a fragment covers does not matter as long as the activation fragment has the same.
template<int TTILES, int NTW, int D, int NQ>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1)))
tile_kernel(const u32x4_t* __restrict__ A, const uint16_t* __restrict__ X, const uint32_t* __restrict__ Q, int N, int T, int K, int tiles_t,
            int tiles_n, uint32_t by_divisor, uint32_t how /* log2 of the K splits (8 bits), epilogue */, uint16_t* __restrict__ C,
            const uint16_t* R_, float* ws, int* cnt, int epoch)
{
    extern __shared__ __attribute__((aligned(16))) uint8_t xs[];  // [D][4 TTILES][kBlock]
    constexpr int WAVES = 4;
    constexpr int TT    = 16 * TTILES;
    constexpr int kBlock = 1024 + 16, kStage = 4 * TTILES * kBlock;  // bytes of LDS
    constexpr int TB    = TTILES / 2, NB = NTW / 2;  // 32 x 32 blocks
    static_assert(TTILES % 2 == 0 && NTW % 2 == 0, "blocks of 32");
    constexpr int XB    = TTILES;  // 1 KiB activation blocks (4 token rows) that each wave fetches per group
    static_assert(D == 2 || D == 4, "stages alternate in parity, so their number is even");
    static_assert(NQ == 1 || NQ == 2 || NQ == 4, "group sizes 128, 64 and 32");

    const int tid  = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c    = lane & 31;
    const int hi   = lane >> 5;
    const int G    = (int)((uint32_t)K / kGroup);
    const int NT   = (int)((uint32_t)N / kTileN);
    const int total = tiles_t * tiles_n;
    int       id    = blockIdx.x;
    if (total % 8 == 0) id = (id & 7) * (total >> 3) + (id >> 3);
    const int       log_splits = (int)(how & 0xff), splits = 1 << log_splits, epi = (int)(how >> 8);
    const TilePlace at = tile_place(id, tiles_t, tiles_n, by_divisor, G, (int)blockIdx.y, log_splits);
    const int       tile_n = at.tile_n, gbeg = at.gbeg, gend = at.gend;
    const int       T0 = at.tile_t * TT;
    // this wave's weight tiles; at the right edge they overlap the neighbour's, which then owns those below `first`
    const int first = (tile_n * WAVES + wave) * NTW;
    const int nt0   = min(first, NT - NTW);

    // per-thread byte offsets; the group-dependent part of every address is scalar
    const uint32_t w_off = (uint32_t)(nt0 * 1024 + lane * 16);  // + g * NT * 1024 (+ nt * 1024)
    const uint32_t q_off = (uint32_t)((nt0 * kTileN + c) * 4);  // + g * N * 4    (+ nb * 128)
    // X staging, direct global -> LDS: wave w, request i brings the block m = w*XB + i, token rows 4m .. 4m+3 of the tile,
    // a quarter wave one contiguous row of 256 bytes (lanes that jump between rows keep the address unit busy four times
    // as long).  Row r of a block holds K-chunks 4j .. 4j+3 at position j ^ r, and 16 bytes of padding follow a block:
    // the 16 lanes that read a chunk of 16 rows then touch every bank once, and a fragment's address is a lane register
    // per j and stage plus an immediate.
    // Rows past the last token re-read the last valid row; their outputs are never stored.  (The instruction's offset
    // moves the LDS and the memory address, so four requests share one M0 value; the bias of three blocks less the
    // request's offset takes it out of the memory address.)
    uint32_t x_off[XB];
#pragma unroll
    for (int i = 0; i < XB; ++i) {
        const int r = lane >> 4, row = 4 * (wave * XB + i) + r;
        x_off[i]    = (uint32_t)min(T0 + row, T - 1) * (uint32_t)(K * 2) + (uint32_t)(((lane & 15) ^ (4 * r)) * 16 + (3 - i % 4) * kBlock);
    }
    // fragment reads: sub-step s of chunk j: lane reads row 32*tb + c, K-chunk 4j + s + 2 hi
    uint32_t xr[D][4];
#pragma unroll
    for (int d = 0; d < D; ++d)
#pragma unroll
        for (int j = 0; j < 4; ++j)
            xr[d][j] = lds_addr(xs) + (uint32_t)(d * kStage + (c >> 2) * kBlock + (c & 3) * 256 + (j ^ (c & 3)) * 64 + 2 * hi * 16);

    const UnpackConsts uc;

    // (zeroed by the matrix pipe: a vector of constants would be built in VGPRs first, sixteen for every block)
    float16_t acc[TB][NB];
    {
        half8_t zero = {0, 0, 0, 0, 0, 0, 0, 0};
        asm volatile("" : "+v"(zero));
#pragma unroll
        for (int tb = 0; tb < TB; ++tb)
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, %1, 0" : "=a"(acc[tb][nb]) : "v"(zero));
    }

    constexpr int NQW = NB * NQ;  // Q words per K step: the 32 columns of block nb are qv[nb * NQ ..]
    u32x4_t  w[D][NTW];  // weights and (scale, zero) words of the D groups in flight; stage = group index mod D
    uint32_t q[D][NQW];
#pragma unroll
    for (int d = 0; d < D; ++d) {
#pragma unroll
        for (int nt = 0; nt < NTW; ++nt) w[d][nt] = u32x4_t{0, 0, 0, 0};
#pragma unroll
        for (int i = 0; i < NQW; ++i) q[d][i] = 0;
    }
    constexpr int kLoads = NTW + NQW + XB;             // requests per group
    constexpr int kVmOps = kLoads + (XB + 3) / 4;      // ... and M0 settings
    constexpr int kWqOps = NTW + NQW;
    auto vm_op = [&](auto M, u32x4_t (&ws_)[NTW], uint32_t (&qv)[NQW], uint32_t xo, const char* wbase, const char* qbase,
                     const char* xbase) {
        constexpr int m = decltype(M)::value;
        if constexpr (m < NTW) {
            gload128<(m % 4) * 1024>(ws_[m], w_off, wbase + (m / 4) * 4096);
        }
        else if constexpr (m < kWqOps) {
            constexpr int nb = (m - NTW) / NQ, sub = (m - NTW) % NQ;
            gload32<nb * 128>(qv[m - NTW], q_off, qbase + (int64_t)sub * N * 4);
        }
        else {
            constexpr int i = (m - kWqOps) / 5 * 4 + (m - kWqOps) % 5 - 1;  // M0, four requests, M0, ...
            if constexpr ((m - kWqOps) % 5 == 0) set_m0(xo + (uint32_t)((wave * XB + i + 1) * kBlock));
            else gload_lds128_m0<(i % 4) * kBlock>(x_off[i], xbase);
        }
    };
    auto wbase_of = [&](int g) { return reinterpret_cast<const char*>(A) + (int64_t)g * NT * 1024; };
    auto qbase_of = [&](int g) { return reinterpret_cast<const char*>(Q) + (int64_t)g * NQ * N * 4; };
    auto xbase_of = [&](int g) { return reinterpret_cast<const char*>(X) + (int64_t)g * 256 - 3 * kBlock; };
    const uint32_t xs_lds = __builtin_amdgcn_readfirstlane(lds_addr(xs));
    // wait until at most `Pending` loads are in flight, then release the stage's registers
    auto wait_loads = [&](auto Pending, u32x4_t (&ws_)[NTW], uint32_t (&qv)[NQW]) {
        constexpr int n = decltype(Pending)::value;
        static_assert(n <= 63, "vmcnt is a 6-bit counter");
#pragma unroll
        for (int nt = 0; nt < NTW; ++nt) wait_vm<n>(ws_[nt]);
#pragma unroll
        for (int i = 0; i < NQW; ++i) wait_vm<n>(qv[i]);
    };
    using I0 = std::integral_constant<int, 0>;

    // State carried from one chunk to the next (and across K steps): dequantised weights of the current / next chunk,
    // zero points and scale of the current / next group, and the ring of activation fragments.
    //
    // The ring holds the fragments of one chunk (two, for up to eight token tiles); fragment f sits in slot f mod kRing,
    // is requested right after the MFMAs of fragment f + 1 - kRing and so has kRing - 1 fragments' MFMAs to arrive.  A
    // second full set of fragments, which the registers of a wide tile have no room for, would not hide more.
    constexpr int kRing = TTILES <= 8 ? 2 * TTILES : TTILES;
    static_assert(kRing - 2 <= 15, "lgkmcnt is a 4-bit counter");
    half8_t wf[2][2][NB];  // [chunk parity][sub-step][block]
    half8_t xf[kRing];
    half2_t z1024[2][NB], z64[2][NB], sc[2][NB];

    auto split = [&](auto P_, uint32_t (&qv)[NQW]) {
        constexpr int P = decltype(P_)::value;
        if constexpr (NQ > 1) return;  // (taken chunk by chunk inside dequant_op)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            half_t s;
            split_q(qv[nb], z1024[P][nb], z64[P][nb], s);
            sc[P][nb] = half2_t{s, s};
        }
    };
    // The dequantisation of word J of every pair of tiles of `w`, as 27 * NB single vector instructions
    // (op = NB * k + nb) so that they can be dealt out between the MFMAs of a chunk:
    // k = 0: the lane exchange; then for either sub-step's word
    // 0: w >> 8;  1..4: (w & mask) | magic;  5..8: - (offset + zero);  9..12: * scale.
    uint32_t dw[NB][2], dq[NB][5];
    auto dequant_op = [&](auto P, auto J, auto OP, u32x4_t (&ws_)[NTW], uint32_t (&qv)[NQW]) {
        // (NQ > 1: the zero points and the scale of word j's quantisation group replace parity p's for this word)
        constexpr int p = NQ > 1 ? 0 : decltype(P)::value, j = decltype(J)::value;
        constexpr int nb = decltype(OP)::value % NB, op = decltype(OP)::value / NB;
        if constexpr (op == 0) {
            if constexpr (NQ > 1) {
                half_t s;
                split_q(qv[nb * NQ + j * NQ / 4], z1024[0][nb], z64[0][nb], s);
                sc[0][nb] = half2_t{s, s};
            }
            const auto both = __builtin_amdgcn_permlane16_swap(ws_[2 * nb][j], ws_[2 * nb + 1][j], false, false);
            dw[nb][0] = both[0], dw[nb][1] = both[1];
            return;
        }
        constexpr int s = (op - 1) / 13 & 1, k = (op + 12) % 13;
        if constexpr (k == 0) dq[nb][4] = dw[nb][s] >> 8;
        else if constexpr (k <= 4) {
            constexpr int i  = k - 1;
            const uint32_t src = i < 2 ? dw[nb][s] : dq[nb][4];
            dq[nb][i] = (src & (i & 1 ? uc.mask_hi : uc.mask_lo)) | (i & 1 ? uc.magic_hi : uc.magic_lo);
        }
        else if constexpr (k <= 8) {
            constexpr int i = k - 5;
            dq[nb][i]       = as_u32(as_half2(dq[nb][i]) - (i & 1 ? z64[p][nb] : z1024[p][nb]));
        }
        else {
            constexpr int i = k - 9;
            const half2_t r = as_half2(dq[nb][i]) * sc[p][nb];
            wf[j & 1][s][nb][2 * i]     = r[0];
            wf[j & 1][s][nb][2 * i + 1] = r[1];
        }
    };
    constexpr int kOps = 27 * NB;
    // fragment F of the K step on stage S (F >= 4 TTILES: of the next stage): chunk, sub-step, token block
    auto read_frag = [&](auto S_, auto F_) {
        constexpr int f = decltype(F_)::value, stage = (decltype(S_)::value + f / (4 * TTILES)) % D;
        constexpr int j = f / TTILES % 4, s = f % TTILES / TB, tb = f % TB;
        lds_read128<tb * 8 * kBlock + s * 16>(xf[f % kRing], xr[stage][j]);
    };

    // The schedule of a K step (see `step`): where it synchronises, and how the requests of a group are dealt out.
    constexpr int kSyncChunk = 4 - kRing / TTILES;
    constexpr int kSyncAt    = TTILES - 1 < (5 + NB) / NB ? TTILES - 1 : (5 + NB) / NB;
    constexpr int kSlots     = TTILES * NB;                                          // MFMAs per chunk
    constexpr int kVmFrom    = kSyncChunk == 3 ? (kSyncAt + 1) * NB : 0;             // first slot of chunk 3 with requests
    constexpr int kVmSlots   = (kSlots - kVmFrom) + (kSyncChunk == 3 ? 2 : 1) * kSlots;  // in three (two) chunks
    constexpr int kFirst = (kSlots - kVmFrom) * kVmOps / kVmSlots;  // operations dealt to chunk 3, and the requests among them
    constexpr int kFirstLoads = kFirst <= kWqOps ? kFirst : kFirst - (kFirst - kWqOps + 4) / 5;

    // ---- prologue: the first D groups in flight, first operands of the first one prepared ----
    // The K loop works through the groups D at a time (the D parts of its body differ in which
    // registers and which LDS buffer hold the current group).  A group count that is not a
    // multiple of D is padded with phantom groups in front: their activation tile is overwritten with zeros
    // and their weights are those of the first real group, so they add exactly zero.
    const int pad    = (D - (gend - gbeg) % D) % D;
    const int gstart = gbeg - pad;
    static_for<0, D>([&](auto dc) {
        constexpr int d = decltype(dc)::value;
        const int     g = max(gstart + d, gbeg);
        // (of the last stage only what precedes the first step: the rest is dealt out there)
        static_for<0, d == D - 1 ? kFirst : kVmOps>([&](auto m) { vm_op(m, w[d], q[d], xs_lds + (uint32_t)(d * kStage), wbase_of(g), qbase_of(g), xbase_of(g)); });
    });
    wait_loads(std::integral_constant<int, (D - 2) * kLoads + kFirstLoads>{}, w[0], q[0]);  // only the first stage has to be there
    if (pad) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        for (int i = tid; i < pad * kStage / 16; i += 64 * WAVES) reinterpret_cast<u32x4_t*>(xs)[i] = u32x4_t{0, 0, 0, 0};
    }
    __syncthreads();
    split(I0{}, q[0]);
    static_for<0, kOps>([&](auto op) { dequant_op(I0{}, I0{}, op, w[0], q[0]); });
    static_for<0, kRing - 1>([&](auto f) { read_frag(I0{}, f); });

    // One K step (a quantisation group, four k32 chunks) on stage S: weights w[S], LDS buffer S, group parity S & 1.
    // Every chunk runs its MFMAs interleaved with the dequantisation of the NEXT chunk's weights and the requests for
    // the fragments a ring ahead.  Fragment requests reach the next stage's buffer in chunk kSyncChunk: the workgroup
    // synchronises there, kSyncAt fragments into the chunk, when the last reads of buffer S - issued right at its
    // beginning - have returned without a wait; the requests due up to then follow the barrier.  The last chunk starts
    // on the next group's weights (stage S + 1, requested D - 1 K steps ago).  Stage S, whose registers and LDS buffer
    // nobody reads any more, is requested anew for group g + D from there to the second chunk of the next step: spread
    // that thinly, because every instruction beyond those that fit behind an MFMA holds the matrix pipe up.
    auto step = [&](auto S_, int g) {
        constexpr int S = decltype(S_)::value, SN = (S + 1) % D, SP = (S + D - 1) % D;
        constexpr int p = S & 1;
        using P         = std::integral_constant<int, p>;
        using PN        = std::integral_constant<int, p ^ 1>;
        const int   g2 = min(g + D, gend - 1), g1 = min(g - 1 + D, gend - 1);  // (the last steps re-read the last group: no branch)
        const char *wb2 = wbase_of(g2), *qb2 = qbase_of(g2), *xb2 = xbase_of(g2);
        const char *wb1 = wbase_of(g1), *qb1 = qbase_of(g1), *xb1 = xbase_of(g1);
        static_for<0, 4>([&](auto jc) {
            constexpr int  j    = decltype(jc)::value;
            constexpr bool last = j == 3;
            if constexpr (j == kSyncChunk) {
                // stages S + 2 .. S + D - 1 may still be in flight behind stage S + 1
                wait_loads(std::integral_constant<int, (D - 2) * kLoads>{}, w[SN], q[SN]);
            }
            if constexpr (last) split(PN{}, q[SN]);
            static_for<0, TTILES>([&](auto tc) {
                constexpr int t = decltype(tc)::value, f = j * TTILES + t, s = t / TB, tb = t % TB;
                // requests younger than fragment f at this point (two fragments per wait)
                constexpr int kYoung = j == kSyncChunk && t >= 1 && t <= kSyncAt ? kRing - 1 - t : kRing - 2;
                if constexpr (t % 2 == 0) {
                    constexpr int kYoung1 = j == kSyncChunk && t + 1 <= kSyncAt ? kRing - 2 - t : kRing - 2;
                    constexpr int kBoth   = kYoung1 - 1 < kYoung - 1 ? kYoung1 : kYoung - 1;
                    asm volatile("s_waitcnt lgkmcnt(%2)" : "+v"(xf[f % kRing]), "+v"(xf[(f + 1) % kRing]) : "n"(kBoth < 0 ? 0 : kBoth));
                }
                static_for<0, NB>([&](auto nc) {
                    constexpr int nb = decltype(nc)::value, i = t * NB + nb;
                    __builtin_amdgcn_sched_barrier(0);
                    asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, %2, %0"
                                 : "+a"(acc[tb][nb])
                                 : "v"(wf[j & 1][s][nb]), "v"(xf[f % kRing]));
                    __builtin_amdgcn_sched_barrier(0);
                    static_for<i * kOps / kSlots, (i + 1) * kOps / kSlots>([&](auto op) {
                        if constexpr (!last) dequant_op(P{}, std::integral_constant<int, j + 1>{}, op, w[S], q[S]);
                        else dequant_op(PN{}, I0{}, op, w[SN], q[SN]);
                    });
                    if constexpr (last && i >= kVmFrom) {
                        constexpr int at = i - kVmFrom;
                        static_for<at * kVmOps / kVmSlots, (at + 1) * kVmOps / kVmSlots>(
                            [&](auto m) { vm_op(m, w[S], q[S], xs_lds + (uint32_t)(S * kStage), wb2, qb2, xb2); });
                    }
                    if constexpr (j < (kSyncChunk == 3 ? 2 : 1)) {
                        constexpr int at = (kSlots - kVmFrom) + j * kSlots + i;
                        static_for<at * kVmOps / kVmSlots, (at + 1) * kVmOps / kVmSlots>(
                            [&](auto m) { vm_op(m, w[SP], q[SP], xs_lds + (uint32_t)(SP * kStage), wb1, qb1, xb1); });
                    }
                });
                // the fragment a ring ahead of the previous one
                if constexpr (j == kSyncChunk && t == kSyncAt) {
                    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                    __builtin_amdgcn_s_barrier();
                    static_for<1, kSyncAt + 1>([&](auto u) { read_frag(S_, std::integral_constant<int, j * TTILES + decltype(u)::value - 1 + kRing>{}); });
                }
                else if constexpr (!(j == kSyncChunk && t >= 1 && t < kSyncAt)) {
                    read_frag(S_, std::integral_constant<int, f - 1 + kRing>{});
                }
                __builtin_amdgcn_sched_barrier(0);
            });
        });
    };

    // Whole multiples of D only (see `pad` above): no K step outside the loop, so the compiler never
    // has a reason to move an accumulator while the loop's MFMAs may still be writing it.
    for (int g = gstart; g + D - 1 < gend; g += D) {  // no branch inside: the 4*TTILES*NTW accumulators stay in place
        static_for<0, D>([&](auto dc) { step(dc, g + decltype(dc)::value); });
    }
    // no load may still be writing LDS or registers when the wave ends
    static_for<0, D>([&](auto dc) { wait_loads(I0{}, w[decltype(dc)::value], q[decltype(dc)::value]); });
    // The last steps requested activation fragments for a step that does not exist.  Nothing
    // reads them, so the compiler may hand their registers out again at once while the LDS reads
    // are still on their way and would land on the new owner: wait for them first.  (Tying the
    // registers to the wait would keep the whole ring alive and cost registers in the loop;
    // the build's assembly check verifies instead that nothing touches them before this wait.)
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    // the MFMAs are inline assembly, so the compiler does not know that the accumulators are
    // still being written: cover the longest MFMA-result-to-VALU-read distance by hand (the
    // build's assembly check verifies that no accumulator is read before this)
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
    // (every block is taken out of its AGPRs where it is used: left alone, the compiler copies all of them to VGPRs here)
    auto finished = [&](int tb, int nb) {
        asm volatile("" : "+a"(acc[tb][nb]));
        return acc[tb][nb];
    };

    // The epilogue of a 32 x 32 block: register 4m + i of a lane holds token T0 + 32 tb + c, feature 8m + 4 hi + i.  Two
    // registers' exchange between the halves of the wave gives every lane eight features in a row.
    auto emit = [&](int tb, int nb, const float16_t v) {
        const int token = T0 + tb * 32 + c;
        if (token >= T) return;
#pragma unroll
        for (int m = 0; m < 4; m += 2) {
            uint32_t g[2][2];  // [4-feature group m, m + 1][pair]
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int i = 0; i < 2; ++i) g[u][i] = as_u32(half2_t{(half_t)v[4 * (m + u) + 2 * i], (half_t)v[4 * (m + u) + 2 * i + 1]});
            uint32_t o[4];  // features n .. n + 7
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const auto both = __builtin_amdgcn_permlane32_swap(g[0][i], g[1][i], false, false);
                o[i] = both[0], o[2 + i] = both[1];
            }
            const int tile = nt0 + 2 * nb + m / 2;  // the 16-column tile these features belong to
            if (tile < first) continue;
            const int n = tile * kTileN + 8 * hi;
            if (epi == kEpiSilu) {
                uint32_t r[2];
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    half_t h[2];
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        const half2_t gu = as_half2(o[2 * i + e]);
                        const float   ga = (float)gu[0], up = (float)gu[1];
                        h[e] = (half_t)(silu_quotient(ga) * up);
                    }
                    r[i] = as_u32(half2_t{h[0], h[1]});
                }
                __builtin_memcpy(C + (int64_t)token * (N / 2) + (n >> 1), r, 8);
                continue;
            }
            if (epi == kEpiAdd) {
                uint32_t rr[4];
                __builtin_memcpy(rr, R_ + (int64_t)token * N + n, 16);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const half2_t a = as_half2(rr[i]), y = as_half2(o[i]);
                    o[i] = as_u32(half2_t{(half_t)((float)a[0] + (float)y[0]), (half_t)((float)a[1] + (float)y[1])});
                }
            }
            __builtin_memcpy(C + (int64_t)token * N + n, o, 16);
        }
        __builtin_amdgcn_sched_barrier(0);  // (one block at a time: the epilogue must not cost the loop registers)
    };

    // ---- split K: exchange partial tiles through the workspace ----
    // Each wave writes its accumulators as it holds them, with agent-scope atomic stores and loads: the L2 caches of the
    // XCDs are not coherent with each other, and these go through to memory without a full cache write-back.
    // A store is complete when the wave's store counter drains, so draining it before the arrival
    // counter is incremented orders the two.  The last workgroup to arrive adds the partial tiles
    // in split order, its own included, so the sum does not depend on which one is last.
    if (splits > 1) {
        constexpr int kBlocks = TB * NB;
        const int64_t per_split = (int64_t)total * WAVES * kBlocks * 1024;  // floats
        // (the lane index is hidden from the optimiser here so that none of these addresses is
        // computed before the K loop and carried through it in registers)
        int lane_now = lane;
        asm volatile("" : "+v"(lane_now));
        float* const mine_base = ws + ((int64_t)id * WAVES + wave) * kBlocks * 1024 + lane_now * 2;
        {
            float* wp = mine_base + blockIdx.y * per_split;
#pragma unroll
            for (int tb = 0; tb < TB; ++tb)
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) {
                    const float16_t v = finished(tb, nb);
                    uint64_t*       o = reinterpret_cast<uint64_t*>(wp + (tb * NB + nb) * 1024);
#pragma unroll
                    for (int i = 0; i < 8; ++i) __hip_atomic_store(o + 64 * i, pack2(v[2 * i], v[2 * i + 1]), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
        }
        __builtin_amdgcn_s_waitcnt(0);  // all of this wave's stores are complete
        __syncthreads();                // ... and every wave is done with the activation tiles in LDS
        int* const last_flag = reinterpret_cast<int*>(xs);
        if (tid == 0) {
            const bool last = arrive_last(cnt, id, splits, epoch);
            *last_flag = last;
        }
        __syncthreads();
        if (!*last_flag) return;
        // Partial tiles are a trip to memory away, so eight blocks of them - four of either split, two of each of four - are requested
        // together: 64 loads a lane, what the load counter holds.  (Block by block and split by split, eight loads at a time, us, cold weights, ->
        // this way: 4096 x 4096 at 300 tokens, 256 x 128 in two 34.2 -> 32.3, 128 x 256 in four 30.9 -> 29.0; 4096 x 12288 at 200, 224 x 128 in two
        // 35.5 -> 34.3; 11008 x 4096 at 300, 160 x 128 in four 44.7 -> 43.3.  The rest of the exchange is the way of the stores to memory.)
        auto add_up = [&](auto S_) {
            constexpr int S = decltype(S_)::value, kTogether = 8 / S;
#pragma unroll 1
            for (int k0 = 0; k0 < kBlocks; k0 += kTogether) {
                uint64_t v[kTogether][S][8];
#pragma unroll
                for (int k = 0; k < kTogether; ++k)
#pragma unroll
                    for (int z = 0; z < S; ++z) {
                        const uint64_t* ip = reinterpret_cast<const uint64_t*>(mine_base + z * per_split + min(k0 + k, kBlocks - 1) * 1024);
#pragma unroll
                        for (int i = 0; i < 8; ++i) v[k][z][i] = __hip_atomic_load(ip + 64 * i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    }
#pragma unroll
                for (int k = 0; k < kTogether; ++k) {
                    if (k0 + k >= kBlocks) break;
                    float16_t sum;
#pragma unroll
                    for (int i = 0; i < 16; ++i) sum[i] = 0.f;
#pragma unroll
                    for (int z = 0; z < S; ++z)
#pragma unroll
                        for (int i = 0; i < 8; ++i) sum[2 * i] += lo_float(v[k][z][i]), sum[2 * i + 1] += hi_float(v[k][z][i]);
                    emit((k0 + k) / NB, (k0 + k) % NB, sum);
                }
            }
        };
        if (splits == 2) add_up(std::integral_constant<int, 2>{});
        else if (splits == 4) add_up(std::integral_constant<int, 4>{});
        else add_up(std::integral_constant<int, 8>{});
        return;
    }

#pragma unroll
    for (int tb = 0; tb < TB; ++tb)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) emit(tb, nb, finished(tb, nb));
}

template<int TTILES, int NTW, int D, int NQ>
hipError_t launch_tile_one(int splits, const GemmArgs& a, const Scratch& sc, hipStream_t st)
{
    constexpr int TT = 16 * TTILES, TN = 64 * NTW;
    const int     tiles_t = (a.T + TT - 1) / TT, tiles_n = (a.N + TN - 1) / TN;
    const size_t  lds     = (size_t)D * 4 * TTILES * (1024 + 16);
    auto          kfn     = tile_kernel<TTILES, NTW, D, NQ>;
    static std::atomic<uint64_t> raised{0};  // per instantiation, one bit per device
    const hipError_t             e = raise_lds_limit(reinterpret_cast<const void*>(kfn), (int)lds, raised);
    if (e != hipSuccess) return e;
    const uint32_t how = (uint32_t)log2_of(splits) | (uint32_t)a.epilogue << 8;
    return launch_kernel(kfn, dim3(tiles_t * tiles_n, splits), dim3(256), lds, st, reinterpret_cast<const u32x4_t*>(a.A), a.X, a.Q, a.N, a.T, a.K,
                         tiles_t, tiles_n, reciprocal((uint64_t)tiles_t * tiles_n, tile_divisor(tiles_t, tiles_n)), how, a.C, a.R, sc.ws, sc.cnt,
                         sc.epoch);
}

// The tiles that exist (api.cpp has their prices), stages by what LDS holds.
template<int NQ>
hipError_t launch_tile(const TileConfig& cf, const GemmArgs& a, const Scratch& sc, hipStream_t st)
{
    switch (cf.ttiles * 8 + cf.ntw) {
        case 16 * 8 + 4: return launch_tile_one<16, 4, 2, NQ>(cf.splits, a, sc, st);
        case 14 * 8 + 4: return launch_tile_one<14, 4, 2, NQ>(cf.splits, a, sc, st);
        case 12 * 8 + 4: return launch_tile_one<12, 4, 2, NQ>(cf.splits, a, sc, st);
        case 10 * 8 + 4: return launch_tile_one<10, 4, 2, NQ>(cf.splits, a, sc, st);
        case 8 * 8 + 4: return launch_tile_one<8, 4, 2, NQ>(cf.splits, a, sc, st);
        case 4 * 8 + 4: return launch_tile_one<4, 4, 4, NQ>(cf.splits, a, sc, st);
        case 16 * 8 + 2: return launch_tile_one<16, 2, 2, NQ>(cf.splits, a, sc, st);
        case 14 * 8 + 2: return launch_tile_one<14, 2, 2, NQ>(cf.splits, a, sc, st);
        case 12 * 8 + 2: return launch_tile_one<12, 2, 2, NQ>(cf.splits, a, sc, st);
        case 10 * 8 + 2: return launch_tile_one<10, 2, 2, NQ>(cf.splits, a, sc, st);
        case 8 * 8 + 2: return launch_tile_one<8, 2, 4, NQ>(cf.splits, a, sc, st);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace

}  // namespace w4a16
