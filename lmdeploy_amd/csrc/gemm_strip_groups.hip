// The strip kernels for group sizes 64 and 32 (NQ = 2, 4 quantisation groups per 128-row weight tile): the deal, the widths,
// the groups in flight and the narrow variant are those of group size 128 (gemm_strip.hip); the epilogue is chosen at run
// time, which costs nothing measurable and leaves a third of the instantiations.
#include "strip_body.h"

#include <algorithm>

namespace w4a16 {

namespace {

using namespace strip;

template<int RMAX, int TP, int D, int NQ>
__global__ void __launch_bounds__(64 * kWaves) strip_kernel_q(STRIP_ARGS)
{
    extern __shared__ __attribute__((aligned(16))) u32x4_t smem[];
    const StripParams p = strip_params(STRIP_ARG_NAMES);
    for (int pass = 0; pass < p.passes; ++pass) {
        const int  bx   = pass * p.grid + blockIdx.x;
        const bool wide = bx < p.rem;
        const int  col0 = bx * p.base + min(bx, p.rem);
        if (pass) __syncthreads();  // the sums of the previous strip have been read out of LDS
        bool done = false;
        if constexpr (RMAX > 1) {
            if (!wide && p.base == RMAX - 1) {
                strip_body<RMAX - 1, TP, kEpiRuntime, false, kWaves, NoWait, NQ, D>(p, col0, smem);
                done = true;
            }
        }
        if (!done) strip_body<RMAX, TP, kEpiRuntime, false, kWaves, NoWait, NQ, D>(p, col0, smem);
    }
}

template<int TP, int D, int NQ>
__global__ void __launch_bounds__(64 * kWavesNarrow) strip_kernel_q_narrow(STRIP_ARGS)
{
    extern __shared__ __attribute__((aligned(16))) u32x4_t smem[];
    const StripParams p = strip_params(STRIP_ARG_NAMES);
    strip_body<1, TP, kEpiRuntime, false, kWavesNarrow, NoWait, NQ, D>(p, (int)blockIdx.x, smem);
}

template<int RMAX, int D, int NQ>
hipError_t launch_tp(int tp, const StripParams& p, dim3 grid, size_t lds, hipStream_t st)
{
    const dim3 block(64 * kWaves);
    if (tp == 4) return launch_strip(strip_kernel_q<RMAX, 4, D, NQ>, grid, block, lds, st, p);
    if (tp == 8) return launch_strip(strip_kernel_q<RMAX, 8, D, NQ>, grid, block, lds, st, p);
    return launch_strip(strip_kernel_q<RMAX, 16, D, NQ>, grid, block, lds, st, p);
}

template<int NQ>
hipError_t launch_q(const StripPlan& pl, int tp, const StripParams& p, dim3 grid, hipStream_t st)
{
    if (pl.narrow) {
        const dim3   block(64 * kWavesNarrow);
        const size_t lds = (size_t)kWavesNarrow * std::max(1024, tp * 256);
        if (tp == 4) return launch_strip(strip_kernel_q_narrow<4, 2, NQ>, grid, block, lds, st, p);
        return launch_strip(strip_kernel_q_narrow<8, 1, NQ>, grid, block, lds, st, p);
    }
    const size_t lds = (size_t)kWaves * std::max(pl.rmax * 1024, tp * 256);
    switch (pl.rmax) {
        case 1: return launch_tp<1, 2, NQ>(tp, p, grid, lds, st);
        case 2: return launch_tp<2, 2, NQ>(tp, p, grid, lds, st);
        case 3: return pl.depth == 1 ? launch_tp<3, 1, NQ>(tp, p, grid, lds, st) : launch_tp<3, 2, NQ>(tp, p, grid, lds, st);
        case 4: return pl.depth == 1 ? launch_tp<4, 1, NQ>(tp, p, grid, lds, st) : launch_tp<4, 2, NQ>(tp, p, grid, lds, st);
        case 5: return launch_tp<5, 1, NQ>(tp, p, grid, lds, st);
        case 6: return launch_tp<6, 1, NQ>(tp, p, grid, lds, st);
        case 7: return launch_tp<7, 1, NQ>(tp, p, grid, lds, st);
        default: return launch_tp<8, 1, NQ>(tp, p, grid, lds, st);
    }
}

}  // namespace

hipError_t strip_groups_launch(int nq, int cus, int per_cu, const GemmArgs& a, hipStream_t st)
{
    const StripPlan pl = strip_plan(cus, per_cu, 16, a.N, a.T, a.K);
    if (!pl.ok || (nq != 2 && nq != 4)) return hipErrorInvalidValue;
    const int   tp = a.T <= 4 ? 4 : (a.T <= 8 ? 8 : 16);
    StripParams p{a.C, reinterpret_cast<const u32x4_t*>(a.A), a.X, a.Q, a.R, a.N, a.T, a.K, pl.base, pl.rem,
                  a.epilogue, pl.passes, pl.strips};
    const dim3  grid(pl.strips, (a.T + 15) / 16);
    return nq == 2 ? launch_q<2>(pl, tp, p, grid, st) : launch_q<4>(pl, tp, p, grid, st);
}

}  // namespace w4a16
