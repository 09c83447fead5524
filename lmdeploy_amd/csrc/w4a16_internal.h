// Internal C++ interface between the C ABI (api.cpp) and the kernel launchers.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>
#include <tuple>

namespace w4a16 {

typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

enum Epilogue { kEpiGemm = 0, kEpiSilu = 1, kEpiAdd = 2 };

struct GemmArgs {
    uint16_t*       C;   // fp16 out [T, N] or [T, N/2]
    const uint32_t* A;   // tiled int4 weights
    const uint16_t* X;   // fp16 [T, K]
    const uint32_t* Q;   // half2 [K/128, N]
    const uint16_t* R;   // fp16 residual [T, N] or null
    int             N, T, K;
    int             epilogue;
    unsigned long long* clk = nullptr;  // measurement aid: where a strip kernel adds its cycle and tick counts (3 words)
};

// One dispatchable kernel configuration.
// A decode kernel configuration: r column tiles per wave, wn waves per slice, sk slices per
// workgroup, `depth` groups of weights in flight per wave; fill > 0 additionally splits K
// across workgroups until about `fill` workgroups per CU exist.
struct DecodeConfig {
    int r, wn, sk, depth, fill;
};

// A batch kernel configuration: r column tiles and h blocks of 16 tokens per workgroup, K split over `splits` workgroups.
struct BatchConfig {
    int r, h, splits;
};

// A tile kernel configuration: 16 * ttiles tokens x 64 * ntw features per workgroup, K split over `splits` workgroups.
struct TileConfig {
    int ttiles, ntw, splits;
};

enum Family { kDecode, kStrip, kPrefill, kTile, kBatch };

// What a launch of a configuration costs, in microseconds (algo_cost): fitted to measurements of every configuration on 17
// matrices (1024 x 3072 to 8192 x 57344, with cold weights) at 17 token counts from 20 to 2048, batch kernels and 64-token
// tiles on 11 of them at 24 to 256 tokens.  On 90 sizes that were not fitted (33 to 2048 tokens, cold weights, launches in a
// graph) the choices take 2.0 % longer than the best configuration that the rounding rule allows: seven in ten are the best one,
// and the worst are 40 % (1280 x 1536 at 68 tokens, 6.6 against 4.7), above 128 tokens 14 % (4096 x 12288 at 512, 58.8 against 51.7).
struct Cost {
    float launch, tile;   // per launch, and per workgroup beside its K steps
    float step, step2;    // per K step with one workgroup per CU, and with two side by side (where two fit)
    float idle;           // share of a step's cost that a CU pays for its neighbours: less on a chip that is not full
    float split, megabyte;  // split K: the exchange, and per million partial sums
};

struct Algo {
    int          kind;     // as w4a16_metric reports it: 0 decode (column blocks), 1 MFMA tiles, 2 decode (strips), 3 batch
    Family       family;
    int          tile_n;   // output features per workgroup
    int          tile_t;   // tokens per workgroup
    int          slices;   // as w4a16_metric reports them
    int          param;    // prefill: variant index; strips: strips per CU aimed for
    DecodeConfig dc;       // decode only
    BatchConfig  bc;       // batch only
    TileConfig   tc;       // tile only
    int          depth;    // K steps come in multiples of this
    int          resident; // workgroups that fit a CU
    Cost         cost, few;  // few: of batch kernels at up to 128 tokens, 32 with group sizes 64 and 32 (pick_by_cost)
};

// Scratch of the split-K kernels: fp32 partial tiles and arrival counters.  A handle's scratch has
// exactly this size (the partial tiles are allocated on first need, the counters with the handle),
// so feasibility of a split-K launch does not depend on the handle.  `ws_bytes` / `cnt_len` say
// how much a launch may use; `ws` may still be null while they are non-zero (not yet allocated).
constexpr size_t kWorkspaceBytes = 64u << 20;
constexpr int    kCounters       = 1 << 16;
struct Scratch {
    float* ws;
    size_t ws_bytes;
    int*   cnt;      // eight bytes each
    int    cnt_len;  // counters
    int    epoch;  // tag of this launch's counts where the counters are shared, else 0 (arrive_last)
    int    cus;    // compute units of the device that all this is on, which the strips are dealt to and the prices counted in
};
constexpr int kEpochShift = 12;  // a tagged counter word: the epoch above, up to 4095 arrivals below

// Launches `kernel` and returns this launch's own status.  (The triple-chevron form reports through
// hipGetLastError, which also returns - and clears - an error some earlier call of the caller left behind.)
template<typename... P, typename... A>
inline hipError_t launch_kernel(void (*kernel)(P...), dim3 grid, dim3 block, size_t lds, hipStream_t st, A... args)
{
    std::tuple<P...> held{static_cast<P>(args)...};
    void*            ptrs[sizeof...(P) > 0 ? sizeof...(P) : 1];
    int              i = 0;
    std::apply([&](auto&... v) { ((ptrs[i++] = (void*)&v), ...); }, held);
    return hipLaunchKernel(reinterpret_cast<const void*>(kernel), grid, block, ptrs, lds, st);
}

// Raises a kernel's dynamic LDS limit once per kernel instantiation (`done`: one bit per device) and
// device; kernels that ask for more than 64 KiB need it before their first launch on a device.
inline hipError_t raise_lds_limit(const void* kernel, int bytes, std::atomic<uint64_t>& done)
{
    int        dev = 0;
    hipError_t e   = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    const uint64_t bit = 1ull << (dev & 63);
    if (done.load(std::memory_order_acquire) & bit) return hipSuccess;
    e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e == hipSuccess) done.fetch_or(bit, std::memory_order_release);
    return e;
}

int         algo_count();
const Algo& algo_at(int id);
// true if algo `id` can run the shape with the scratch `lim` allows
bool algo_feasible(int id, int N, int T, int K, const Scratch& lim);
// bytes of partial-tile scratch the launch would use (0: the kernel needs neither workspace nor counters)
size_t algo_scratch_bytes(int id, int N, int T, int K, const Scratch& lim);
// heuristic choice (the counterpart of Estimate) for nq quantisation groups per weight tile, among the kernels that do not round
// weights if so asked; -1 if nothing is feasible
int algo_pick(int nq, int N, int T, int K, const Scratch& lim, bool unrounded = false);
// whether a size's scales multiply sums in fp32, and not the weights, which rounds them (rounding_domain.cpp); `lim` as in algo_pick
bool scales_in_fp32(int nq, int N, int T, int K, const Scratch& lim);
// workgroups the launch would use
int algo_grid(int id, int N, int T, int K, const Scratch& sc);
hipError_t algo_launch(int id, int nq, const GemmArgs& a, const Scratch& sc, hipStream_t st);

// The scratch that lives in a file-scope device array (static_scratch.hip), for callers that cannot
// allocate: its address on the current device, looked up once per device.
constexpr size_t kStaticCounters       = 4096;
// In front of the partial tiles, so many of each (arrive_last): counters of launches made at once, eight bytes each; from int kStaticTagged
// on, the second ones, four bytes, for counts that did not start from zero; from int kStaticRecorded on, eight bytes, those of launches
// recorded into a graph.
constexpr size_t kStaticTagged         = 2 * kStaticCounters;
constexpr size_t kStaticRecorded       = 3 * kStaticCounters;
constexpr size_t kStaticCounterInts    = 5 * kStaticCounters;
constexpr size_t kStaticWorkspaceBytes = 8u << 20;
hipError_t static_scratch(Scratch* out);
// before a launch that uses `n` of its counters: sets the tag, and clears them where the launch is being recorded into a graph
hipError_t prepare_static_counters(Scratch* sc, int n, hipStream_t st);

hipError_t launch_convert(uint32_t* A_dst, uint32_t* Q_dst, const uint32_t* A_src, const uint16_t* scales,
                          const uint32_t* qzeros, int m, int k, int group, hipStream_t st);
// up to three AWQ tensors -> one deployable (A, Q): side by side, or (interleave) gate/up column pairs
hipError_t launch_deploy(uint32_t* A_dst, uint32_t* Q_dst, const uint32_t* const qw[3], const uint32_t* const qz[3],
                         const uint16_t* const s[3], const int width[3], const int rotary[3], int interleave, int k,
                         int group, hipStream_t st);
// q, k, v, o, gate, up, down in; q|k|v, o, gate|up, down out
hipError_t launch_deploy_layer(uint32_t* const A[4], uint32_t* const Q[4], const uint32_t* const qw[7], const uint32_t* const qz[7],
                               const uint16_t* const s[7], const int n[7], const int k[4], int size_per_head, int group, hipStream_t st);
hipError_t launch_unpack(uint32_t* qweight, uint32_t* qzeros, uint16_t* scales, const uint32_t* A,
                         const uint32_t* Q, int m, int k, int group, hipStream_t st);
hipError_t launch_dequantize_repacked(uint16_t* W, const uint32_t* A, const uint32_t* Q, int m, int k, int group,
                                      hipStream_t st);
hipError_t launch_dequantize_s4(void* dst, const uint32_t* src, size_t count, hipStream_t st);
hipError_t launch_fuse_w1_w3(uint32_t* dst, const uint32_t* src, int m, int k, hipStream_t st);
hipError_t launch_transpose_qk(uint32_t* dst, const uint32_t* src, int m, int k, int size_per_head, hipStream_t st);
hipError_t launch_from_reference(uint32_t* dst, const uint32_t* ref, int m, int k, hipStream_t st);

// measurement aid (probe.hip): a plain streaming read of `bytes`; sink = at least 8 * cus words
hipError_t launch_probe_read(const void* src, size_t bytes, void* sink, int cus, hipStream_t st);
// the same with the GEMM kernels' load pipeline: `in_flight` (2, 4, 8, 16) loads of 16 bytes per lane kept in
// flight by count, `wg_per_cu` (1, 2, 4) workgroups of eight waves per CU, hint 0 none / 1 nt / 2 sc0 sc1
bool       probe_stream_config_ok(int wg_per_cu, int in_flight, int hint);
// (clk: optional counters of clock_record_start / _stop)
hipError_t launch_probe_mfma(void* sink, int cus, int waves_per_cu, int iters, unsigned long long* clk, hipStream_t st);
hipError_t launch_probe_stream(const void* src, size_t bytes, void* sink, int cus, int wg_per_cu, int in_flight, int hint,
                               hipStream_t st, unsigned long long* clk = nullptr);

// decode (skinny) kernels
bool       decode_feasible(const DecodeConfig& cf, int N, int T, int K);
size_t     decode_scratch_bytes(const DecodeConfig& cf, int N, int T, int K, size_t ws_bytes, int cnt_len);
int        decode_grid(const DecodeConfig& cf, int N, int T, int K, size_t ws_bytes, int cnt_len);
hipError_t decode_launch(const DecodeConfig& cf, const GemmArgs& a, const Scratch& sc, hipStream_t st);

// decode kernels, strip decomposition (gemm_strip.hip); block_t = tokens per workgroup, 16 or 32, dealt to `cus` CUs
bool       strip_feasible(int cus, int per_cu, int block_t, int N, int T, int K);
int        strip_grid(int cus, int per_cu, int block_t, int N, int T, int K);
int        strip_width(int cus, int per_cu, int block_t, int N, int T, int K);  // column tiles of the widest strip
hipError_t strip_launch(int cus, int per_cu, int block_t, const GemmArgs& a, hipStream_t st);
// the same for group sizes 64 and 32 (nq = 2, 4 quantisation groups per 128-row weight tile; gemm_strip_groups.hip), 16 tokens
// per workgroup
hipError_t strip_groups_launch(int nq, int cus, int per_cu, const GemmArgs& a, hipStream_t st);
// How the column tiles are dealt out: `strips` workgroups, strips of base tiles (the first rem: one more), rmax wide at most.
struct StripPlan {
    int  strips, base, rem, rmax;
    int  passes;  // strips that each workgroup takes in turn
    int  depth;   // groups in flight per wave
    bool narrow;  // sixteen waves per workgroup
    bool ok;
};
StripPlan strip_plan(int cus, int per_cu, int block_t, int N, int T, int K);

// The 32-token strips: up to this many column tiles wide, the batch kernel's way of feeding the activations is ahead of
// the strip kernel's (7B qkv, strips of three, at 20 tokens 14.6 -> 9.6 us, o 6.3 -> 5.6); wider ones stream weights most
// of the time and stay with the strip kernel (7B gate_up 15.4 against 16.0, 70B gate_up 57 against 66).
constexpr int kWidestBatchStrip = 4;

// A sequence of decode GEMMs (up to 16 tokens) in one persistent launch (gemm_sequence.hip)
struct SeqGemm {
    uint16_t*       C;
    const u32x4_t*  A;
    const uint16_t* X;
    const uint32_t* Q;
    const uint16_t* R;
    int             N, K;
    int             epilogue;
    int             flags;  // bit 0: reads what an earlier GEMM of the sequence writes - wait for all of them
};
constexpr int kSeqMax   = 32;    // GEMMs per launch (the descriptors travel as kernel arguments)
constexpr int kSyncInts = 64 * 80;  // arrival counters, flag, error word of the device-wide barrier
bool       sequence_feasible(const SeqGemm* g, int count, int T);
int        sequence_error_index();  // index of the error word in the sync area
// `cus` workgroups (one per CU: they must all be resident at once); `spin_ticks` bounds each barrier wait
hipError_t sequence_launch(const SeqGemm* g, int count, int T, int* sync, int cus, long long spin_ticks, hipStream_t st);

// measurement aid: `iters` device-wide barriers of `cus` workgroups (tree = 0: all arrivals on one counter)
hipError_t launch_probe_barrier(int* sync, int iters, int tree, int cus, long long spin_ticks, hipStream_t st);

// batch kernels (gemm_batch.hip); nq = quantisation groups per 128-row weight tile (1, 2, 4)
bool       batch_feasible(const BatchConfig& cf, int N, int T, int K, size_t ws_bytes, int cnt_len);
size_t     batch_scratch_bytes(const BatchConfig& cf, int N, int T);
int        batch_grid(const BatchConfig& cf, int N, int T);
hipError_t batch_launch(const BatchConfig& cf, int nq, const GemmArgs& a, const Scratch& sc, hipStream_t st);

// MFMA kernels, tiles of two waves per SIMD (gemm_prefill.hip)
int        prefill_variants();
void       prefill_tile(int variant, int& tile_n, int& tile_t);
// `splits` > 1 divides the quantisation groups among that many workgroups per output tile; the
// last one to arrive adds the partial tiles (in split order) and runs the epilogue.
bool       prefill_feasible(int variant, int splits, int N, int T, int K, size_t ws_bytes, int cnt_len);
size_t     prefill_scratch_bytes(int variant, int splits, int N, int T, int K);
int        prefill_grid(int variant, int splits, int N, int T, int K);
hipError_t prefill_launch(int variant, int splits, const GemmArgs& a, const Scratch& sc, hipStream_t st);

// MFMA kernels, tiles of one wave per SIMD (tile_body.h), per group size
hipError_t tile_launch_g128(const TileConfig& cf, const GemmArgs& a, const Scratch& sc, hipStream_t st);
hipError_t tile_launch_g64(const TileConfig& cf, const GemmArgs& a, const Scratch& sc, hipStream_t st);
hipError_t tile_launch_g32(const TileConfig& cf, const GemmArgs& a, const Scratch& sc, hipStream_t st);

}  // namespace w4a16
