// Integer repack kernels: AWQ int4 tensors <-> the gfx950 tiled layout, and the other
// nibble permutations of the reference's format.cu.  Every destination word is built whole
// by one thread, so no atomics and no pre-zeroed destination are needed.
#include "w4a16_common.h"
#include "w4a16_internal.h"

namespace w4a16 {

namespace {

constexpr int kThreads = 256;

__device__ __forceinline__ uint32_t nib(uint32_t w, int p)
{
    return (w >> (4 * p)) & 0xfu;
}

// logical column c (0..7) of an AWQ word sits in nibble nibble_of_row(c): the AWQ order and
// its inverse are the same pair of tables that the tiled layout uses along its rows.
__device__ __forceinline__ uint32_t awq_col(uint32_t w, int c)
{
    return nib(w, nibble_of_row(c));
}

__device__ __forceinline__ int64_t global_id()
{
    return (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
}

// The columns of a deployable matrix, gathered from up to three AWQ tensors of the checkpoint:
// side by side (q | k | v, deploy.py:251-260 `merge_qkv`), optionally with the columns of every
// head re-ordered for rotary embedding (dst column 2i + r of a head <- column r * D/2 + i:
// deploy.py:371-383 `permute`, format.cu:115-121), or interleaved in pairs (gate, up:
// deploy.py:641-658 `fuse_w1_w3_s4`, format.cu:123-130).
struct ColumnSource {
    const uint32_t* qw[3];
    const uint32_t* qz[3];
    const uint16_t* s[3];
    int             width[3];   // columns of each source
    int             rotary[3];  // head size if the block's columns are re-ordered, else 0
    int             interleave; // 1: column n comes from source n & 1, column n >> 1
};
struct Located {
    int src, col;
};
__device__ __forceinline__ Located locate(const ColumnSource& cs, int n)
{
    if (cs.interleave) return Located{n & 1, n >> 1};
    int b = 0;
    while (b < 2 && n >= cs.width[b]) n -= cs.width[b++];
    if (const int D = cs.rotary[b]) {
        const int j = n % D;
        n           = n - j + (j & 1) * (D / 2) + (j >> 1);
    }
    return Located{b, n};
}

// A_dst word `w` <- 8 rows of one column, taken from wherever the column lives: any head size and any alignment,
// one gather of eight words per destination word
__global__ void __launch_bounds__(kThreads)
deploy_weights_kernel(uint32_t* __restrict__ dst, const ColumnSource cs, int N, int K)
{
    const int64_t w     = global_id();
    const int64_t words = (int64_t)N * K / 8;
    if (w >= words) return;
    const int     NT   = N / kTileN;
    const int     j    = (int)(w & 3);
    const int     lane = (int)((w >> 2) & 63);
    const int64_t tile = w >> 8;
    const int     kt   = (int)(tile / NT);
    const int     nt   = (int)(tile % NT);
    const Located at   = locate(cs, nt * kTileN + (lane & 15));
    const int     k0   = kt * kGroup + 32 * j + 8 * (lane >> 4);
    const int     ld   = cs.width[at.src] / 8;
    const uint32_t* src = cs.qw[at.src];
    uint32_t      out  = 0;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const uint32_t v = src[(int64_t)(k0 + e) * ld + (at.col >> 3)];
        out |= awq_col(v, at.col & 7) << (4 * nibble_of_row(e));
    }
    dst[w] = out;
}

__global__ void __launch_bounds__(kThreads) deploy_q_kernel(uint32_t* __restrict__ Q, const ColumnSource cs, int N, int G)
{
    const int64_t i = global_id();
    if (i >= (int64_t)N * G) return;
    const int      g  = (int)(i / N);
    const Located  at = locate(cs, (int)(i % N));
    const int64_t  e  = (int64_t)g * cs.width[at.src] + at.col;
    const uint32_t z  = awq_col(cs.qz[at.src][e >> 3], (int)(e & 7));
    Q[i]              = (0x5400u | (z << 4)) | ((uint32_t)cs.s[at.src][e] << 16);
}

// ---- weights and (zero, scale) words of whole tiles: the path every conversion takes whose columns come in runs of 8 ----
//
// A tile's 16 columns are two source words per row (8 columns each): side by side, or - rotary re-ordering, gate/up
// interleave - the columns of the two words taken in turn.  Between a source word (one row, 8 columns) and a tiled
// word (one column, 8 rows) lies a transposition of 8 x 8 nibbles, and because the tiled layout orders rows inside a
// word as AWQ orders columns, it is a plain one: nibble p of output q = nibble q of input p, inputs and outputs taken
// in AWQ order.  One thread reads the 32 words that one source word column holds for its quarter (b) of the tile's
// rows - coalesced over the lanes, all in flight together -, transposes them in registers and holds eight 16-byte
// vectors, which lanes exchange through LDS so that a store covers 256 contiguous bytes of four tiles; the (zero, scale) words
// ride in the same launch.  Bound by HBM: every byte is read and written once.  Stored as the threads held them, sixteen bytes
// in each of 64 cache lines at a time, the weights kept the L2s busy with requests: Llama-2-70B's four matrices (899 MB moved)
// 222.6 us, 4.0 TB/s, exchanged first 178, and with non-temporal stores 168.8, 5.3 TB/s (a device copy reaches 5.15), in one launch
// 158.2.
struct TilePair {
    const uint32_t* qw[2];  // the two word columns of the tile
    const uint32_t* qz[2];
    const uint16_t* s[2];
    int             ld[2];  // words per row of their tensors
    int             turn;   // 1: output column 2i + h = column i of word h; 0: 8h + i
};

// where tile nt's two word columns are
__device__ __forceinline__ TilePair locate_tile(const ColumnSource& cs, int nt)
{
    TilePair t;
    if (cs.interleave) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            t.qw[h] = cs.qw[h] + nt, t.qz[h] = cs.qz[h] + nt, t.s[h] = cs.s[h] + 8 * nt, t.ld[h] = cs.width[h] / 8;
        }
        t.turn = 1;
        return t;
    }
    int b = 0, n = nt * kTileN;
    while (b < 2 && n >= cs.width[b]) n -= cs.width[b++];
    const int D  = cs.rotary[b];
    const int w0 = D ? (n - n % D + (n % D) / 2) / 8 : n / 8;
    const int w1 = D ? w0 + D / 16 : w0 + 1;
    t.qw[0] = cs.qw[b] + w0, t.qw[1] = cs.qw[b] + w1;
    t.qz[0] = cs.qz[b] + w0, t.qz[1] = cs.qz[b] + w1;
    t.s[0] = cs.s[b] + 8 * w0, t.s[1] = cs.s[b] + 8 * w1;
    t.ld[0] = t.ld[1] = cs.width[b] / 8;
    t.turn  = D ? 1 : 0;
    return t;
}

// b[q] nibble p = a[p] nibble q: halves of words at distance 4, bytes at distance 2, nibbles at distance 1
__device__ __forceinline__ void transpose_nibbles(uint32_t (&a)[8])
{
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t x = a[i], y = a[i + 4];
        a[i]     = __builtin_amdgcn_perm(y, x, 0x05040100);
        a[i + 4] = __builtin_amdgcn_perm(y, x, 0x07060302);
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int      i = (k & 1) + (k & 2) * 2;
        const uint32_t x = a[i], y = a[i + 2];
        a[i]     = __builtin_amdgcn_perm(y, x, 0x06020400);
        a[i + 2] = __builtin_amdgcn_perm(y, x, 0x07030501);
    }
#pragma unroll
    for (int i = 0; i < 8; i += 2) {
        const uint32_t x = a[i], y = a[i + 1];
        a[i]     = (x & 0x0f0f0f0fu) | ((y << 4) & 0xf0f0f0f0u);
        a[i + 1] = ((x >> 4) & 0x0f0f0f0fu) | (y & 0xf0f0f0f0u);
    }
}

// One launch converts several matrices, each by a run of blocks of its own: those of a decoder layer one by one paid for
// three more kernel boundaries and ramps (Llama-2-7B's 213 MB: four launches 46.9 us, one 37.5; Llama-2-70B's 899 MB 168.8 and 158.2).
struct Conversion {
    ColumnSource cs;
    uint32_t*    dst;
    uint32_t*    Q;
    int          NT;
    int          w_across, w_blocks, q_across;
    int          end;  // the first block of the next matrix
};
template<int M>
struct Conversions {
    Conversion of[M];
};

// A matrix's first w_blocks blocks convert weights: 64 word columns (32 tiles) of one row of tiles, wave b the rows 32j + 8b ..
// Those beyond build the Q words of 256 tiles' columns of one quantisation group row each.
template<int M>
__global__ void __launch_bounds__(kThreads) convert_tiles_kernel(const Conversions<M> all)
{
    __shared__ u32x4_t exchange[4][512];  // one part for each wave, which waits for nobody else
    const int          tid = threadIdx.x;
    int                which = 0, block = blockIdx.x;
#pragma unroll
    for (int i = 0; i + 1 < M; ++i)
        if ((int)blockIdx.x >= all.of[i].end) which = i + 1, block = (int)blockIdx.x - all.of[i].end;
    const Conversion&   of = all.of[which];
    const ColumnSource& cs = of.cs;
    uint32_t* const     dst = of.dst;
    uint32_t* const     Q   = of.Q;
    const int           NT  = of.NT;
    if (block < of.w_blocks) {
        const int kt   = block / of.w_across;
        const int base = (block % of.w_across) * 64;  // first word column: tile base / 2
        const int lane = tid & 63, b = tid >> 6;
        const int at   = min(base + lane, 2 * NT - 1);  // word column: tile at / 2, word at % 2
        const int nt = at >> 1, h = at & 1;
        const TilePair  t  = locate_tile(cs, nt);
        const uint32_t* p  = (h ? t.qw[1] : t.qw[0]) + (int64_t)(kt * kGroup + 8 * b) * (h ? t.ld[1] : t.ld[0]);
        const int       ld = h ? t.ld[1] : t.ld[0];
        uint32_t        in[4][8];
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int e = 0; e < 8; ++e) in[j][e] = __builtin_nontemporal_load(p + (int64_t)(32 * j + row_of_nibble(e)) * ld);
#pragma unroll
        for (int j = 0; j < 4; ++j) transpose_nibbles(in[j]);
        // A thread has eight 16-byte vectors of one tile, a store instruction should have 256 contiguous bytes (this wave's quarter)
        // of four: they change places in the wave's part of LDS.  Vector v of tile t is at position v ^ g(t): the sixteen lanes
        // that LDS serves together, two of eight tiles each or all of one, then touch every bank once, whichever way columns run.
        const auto  g   = [](int tile) { return (tile & 7) | (tile & 1) << 3; };
        u32x4_t* const mine = exchange[b];
        const int   tl = lane >> 1;
        if (base + lane < 2 * NT)
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const int col = row_of_nibble(q);
                mine[tl * 16 + ((t.turn ? 2 * col + h : 8 * h + col) ^ g(tl))] = u32x4_t{in[0][q], in[1][q], in[2][q], in[3][q]};
            }
        wave_exchange();
        u32x4_t* const out = reinterpret_cast<u32x4_t*>(dst) + ((int64_t)kt * NT + (base >> 1)) * 64 + b * 16 + (lane & 15);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int tile = 4 * i + (lane >> 4);
            if ((base >> 1) + tile < NT) __builtin_nontemporal_store(mine[tile * 16 + ((lane & 15) ^ g(tile))], out + tile * 64);
        }
        return;
    }
    const int blk = block - of.w_blocks;
    const int g   = blk / of.q_across;
    const int nt  = (blk % of.q_across) * kThreads + tid;
    if (nt >= NT) return;
    const TilePair t = locate_tile(cs, nt);
    uint32_t       z[2], out[16];
    u32x4_t        s[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        z[h] = t.qz[h][(int64_t)g * t.ld[h]];
        s[h] = *reinterpret_cast<const u32x4_t*>(t.s[h] + (int64_t)g * t.ld[h] * 8);
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const uint32_t v = (0x5400u | (awq_col(z[h], i) << 4)) | ((i & 1 ? s[h][i / 2] >> 16 : s[h][i / 2] & 0xffffu) << 16);
            out[8 * h + i] = v;
        }
    u32x4_t* const qd = reinterpret_cast<u32x4_t*>(Q + ((int64_t)g * NT + nt) * kTileN);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int a = 2 * i;  // in turn: columns 2i, 2i + 1 of both words
        qd[i] = t.turn ? u32x4_t{out[a], out[8 + a], out[a + 1], out[8 + a + 1]} :
                         u32x4_t{out[4 * i], out[4 * i + 1], out[4 * i + 2], out[4 * i + 3]};
    }
}

// inverse of repack_weights_kernel: one thread per AWQ word [k, n/8]
__global__ void __launch_bounds__(kThreads)
unrepack_weights_kernel(uint32_t* __restrict__ dst, const uint32_t* __restrict__ A, int N, int K)
{
    const int64_t w     = global_id();
    const int64_t words = (int64_t)N * K / 8;
    if (w >= words) return;
    const int ld = N / 8;
    const int k  = (int)(w / ld);
    const int n0 = (int)(w % ld) * 8;
    const int NT = N / kTileN;
    const int kt = k / kGroup, r = k % kGroup;
    const int j = r >> 5, b = (r >> 3) & 3, e = r & 7;
    uint32_t  out = 0;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        const int     n  = n0 + c;
        const int64_t sw = (((int64_t)kt * NT + n / kTileN) * 64 + b * 16 + (n % kTileN)) * 4 + j;
        out |= nib(A[sw], nibble_of_row(e)) << (4 * nibble_of_row(c));
    }
    dst[w] = out;
}

__global__ void __launch_bounds__(kThreads)
split_q_kernel(uint32_t* __restrict__ qzeros, uint16_t* __restrict__ scales, const uint32_t* __restrict__ Q,
               int64_t words)
{
    const int64_t w = global_id();
    if (w >= words) return;
    uint32_t out = 0;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        const uint32_t q = Q[w * 8 + c];
        out |= ((q >> 4) & 0xfu) << (4 * nibble_of_row(c));
        if (scales) scales[w * 8 + c] = (uint16_t)(q >> 16);
    }
    if (qzeros) qzeros[w] = out;
}

// W[k, n] = mul.ftz(sub(64 + q, 64 + z), s): one thread per repacked word (8 rows of a column)
__global__ void __launch_bounds__(kThreads)
dequantize_repacked_kernel(uint16_t* __restrict__ W, const uint32_t* __restrict__ A,
                           const uint32_t* __restrict__ Q, int N, int K, int group)
{
    const int64_t w     = global_id();
    const int64_t words = (int64_t)N * K / 8;
    if (w >= words) return;
    const int     NT   = N / kTileN;
    const int     j    = (int)(w & 3);
    const int     lane = (int)((w >> 2) & 63);
    const int64_t tile = w >> 8;
    const int     kt   = (int)(tile / NT);
    const int     nt   = (int)(tile % NT);
    const int     n    = nt * kTileN + (lane & 15);
    const int     k0   = kt * kGroup + 32 * j + 8 * (lane >> 4);
    half2_t       z1024, z64;
    half_t        s;
    split_q(Q[(int64_t)(k0 / group) * N + n], z1024, z64, s);  // (a word's 8 rows never straddle two groups: group >= 32)
    // flush a subnormal scale first, as the .ftz multiply of the reference reads it
    uint16_t sb = __builtin_bit_cast(uint16_t, s);
    if ((sb & 0x7c00u) == 0) sb &= 0x8000u;
    s = __builtin_bit_cast(half_t, sb);
    const half8_t v = dequant_full(A[w], z1024, z64, half2_t{s, s}, UnpackConsts());
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        uint16_t bits = __builtin_bit_cast(uint16_t, (half_t)v[e]);
        if ((bits & 0x7c00u) == 0) bits &= 0x8000u;  // flush a subnormal product
        W[(int64_t)(k0 + e) * N + n] = bits;
    }
}

// raw nibble values of AWQ words as fp16, logical column order
__global__ void __launch_bounds__(kThreads)
dequantize_s4_kernel(uint4* __restrict__ dst, const uint32_t* __restrict__ src, int64_t count)
{
    const int64_t i = global_id();
    if (i >= count) return;
    const uint32_t w = src[i];
    uint32_t       v[4];
    unpack_offset(w, v);  // applied to an AWQ word this yields columns (0,1), (2,3), (4,5), (6,7)
    const half2_t k1024 = as_half2(0x64006400u), k64 = as_half2(0x54005400u);
    uint4         o;
    o.x = as_u32(as_half2(v[0]) - k1024);
    o.y = as_u32(as_half2(v[1]) - k64);
    o.z = as_u32(as_half2(v[2]) - k1024);
    o.w = as_u32(as_half2(v[3]) - k64);
    dst[i] = o;
}

// dst AWQ [k, 2m/8] <- interleave of AWQ w1, w3 [2, k, m/8]
__global__ void __launch_bounds__(kThreads)
fuse_w1_w3_kernel(uint32_t* __restrict__ dst, const uint32_t* __restrict__ src, int m, int k)
{
    const int64_t w     = global_id();
    const int     ldd   = 2 * m / 8;
    const int64_t words = (int64_t)k * ldd;
    if (w >= words) return;
    const int     row = (int)(w / ldd);
    const int     c0  = (int)(w % ldd) * 8;
    const int     lds = m / 8;
    uint32_t      out = 0;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        const int      col = c0 + c, sel = col & 1, js = col >> 1;
        const uint32_t s   = src[((int64_t)sel * k + row) * lds + (js >> 3)];
        out |= awq_col(s, js & 7) << (4 * nibble_of_row(c));
    }
    dst[w] = out;
}

// within each head of D columns: dst[2i + r] = src[r * D/2 + i]
__global__ void __launch_bounds__(kThreads)
transpose_qk_kernel(uint32_t* __restrict__ dst, const uint32_t* __restrict__ src, int m, int k, int D)
{
    const int64_t w     = global_id();
    const int     ld    = m / 8;
    const int64_t words = (int64_t)k * ld;
    if (w >= words) return;
    const int row = (int)(w / ld);
    const int c0  = (int)(w % ld) * 8;
    uint32_t  out = 0;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        const int      col = c0 + c, h = col / D, ci = col % D;
        const int      sc  = h * D + (ci & 1) * (D / 2) + (ci >> 1);
        const uint32_t s   = src[(int64_t)row * ld + (sc >> 3)];
        out |= awq_col(s, sc & 7) << (4 * nibble_of_row(c));
    }
    dst[w] = out;
}

// ours <- the reference's tiled layout: word ((kt*(N/32)+nt)*32 + lane)*4 + (k16*2 + n16),
// nibble 4*klo + 2*k8 + n8 holds k = 32kt + 16k16 + 8k8 + 2*(lane%4) + klo,
// n = 32nt + 16n16 + 8n8 + lane/4.
__global__ void __launch_bounds__(kThreads)
from_reference_kernel(uint32_t* __restrict__ dst, const uint32_t* __restrict__ ref, int N, int K)
{
    const int64_t w     = global_id();
    const int64_t words = (int64_t)N * K / 8;
    if (w >= words) return;
    const int     NT   = N / kTileN;
    const int     j    = (int)(w & 3);
    const int     lane = (int)((w >> 2) & 63);
    const int64_t tile = w >> 8;
    const int     kt   = (int)(tile / NT);
    const int     nt   = (int)(tile % NT);
    const int     n    = nt * kTileN + (lane & 15);
    const int     k0   = kt * kGroup + 32 * j + 8 * (lane >> 4);
    uint32_t      out  = 0;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const int     kk = k0 + e;
        const int     rl = (n & 7) * 4 + ((kk >> 1) & 3);
        const int64_t rw = (((int64_t)(kk >> 5) * (N / 32) + (n >> 5)) * 32 + rl) * 4 + (((kk >> 4) & 1) * 2 + ((n >> 4) & 1));
        const int     rn = 4 * (kk & 1) + 2 * ((kk >> 3) & 1) + ((n >> 3) & 1);
        out |= nib(ref[rw], rn) << (4 * nibble_of_row(e));
    }
    dst[w] = out;
}

inline unsigned blocks_for(int64_t n)
{
    return (unsigned)((n + kThreads - 1) / kThreads);
}

}  // namespace

namespace {

// one matrix's conversion: columns gathered as `cs` says, rows of K, quantisation groups; Q == nullptr: the weights alone
struct Matrix {
    ColumnSource cs;
    uint32_t *   A, *Q;
    int          m, k;
};

// Whole tiles: no tile straddles two sources or two heads, and every vector access is aligned.  Appends the matrix to a launch of
// `blocks` blocks so far, false if it (or the launch with it) has to go another way.
bool as_tiles(const Matrix& x, int group, int64_t& blocks, Conversion& c)
{
    auto aligned = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
    bool tiles   = aligned(x.A) && aligned(x.Q);
    for (int i = 0; i < 3; ++i)
        if (x.cs.width[i] > 0)
            tiles = tiles && (x.cs.interleave || x.cs.width[i] % kTileN == 0) && x.cs.rotary[i] % kTileN == 0 && aligned(x.cs.s[i]);
    const int     NT = x.m / kTileN, w_across = (2 * NT + 63) / 64, q_across = (NT + kThreads - 1) / kThreads;
    const int64_t w_blocks = (int64_t)(x.k / kGroup) * w_across;
    blocks += w_blocks + (x.Q ? (int64_t)(x.k / group) * q_across : 0);
    if (!tiles || blocks >= (1ll << 31)) return false;
    c = Conversion{x.cs, x.A, x.Q, NT, w_across, (int)w_blocks, q_across, (int)blocks};
    return true;
}

template<int M>
hipError_t launch_matrices(const Matrix (&x)[M], int group, hipStream_t st)
{
    Conversions<M> all;
    int64_t        blocks = 0;
    bool           tiles  = true;
    for (int i = 0; i < M; ++i) tiles = tiles && as_tiles(x[i], group, blocks, all.of[i]);
    if (tiles) return blocks ? launch_kernel(convert_tiles_kernel<M>, dim3((unsigned)blocks), dim3(kThreads), 0, st, all) : hipSuccess;
    hipError_t e = hipSuccess;
    for (int i = 0; i < M && e == hipSuccess; ++i) {
        if constexpr (M > 1) {
            const Matrix one[1] = {x[i]};
            e                   = launch_matrices(one, group, st);
        }
        else {
            const int64_t words = (int64_t)x[i].m * x[i].k / 8, entries = (int64_t)(x[i].k / group) * x[i].m;
            if (words == 0) continue;
            e = launch_kernel(deploy_weights_kernel, dim3(blocks_for(words)), dim3(kThreads), 0, st, x[i].A, x[i].cs, x[i].m, x[i].k);
            if (x[i].Q && e == hipSuccess)
                e = launch_kernel(deploy_q_kernel, dim3(blocks_for(entries)), dim3(kThreads), 0, st, x[i].Q, x[i].cs, x[i].m, x[i].k / group);
        }
    }
    return e;
}

Matrix plain(uint32_t* A_dst, uint32_t* Q_dst, const uint32_t* A_src, const uint16_t* scales, const uint32_t* qzeros, int m, int k)
{
    Matrix x{{}, A_dst, Q_dst, m, k};
    x.cs.qw[0] = A_src, x.cs.qz[0] = qzeros, x.cs.s[0] = scales, x.cs.width[0] = m;
    return x;
}

Matrix gathered(uint32_t* A_dst, uint32_t* Q_dst, const uint32_t* const qw[3], const uint32_t* const qz[3], const uint16_t* const s[3],
                const int width[3], const int rotary[3], int interleave, int k)
{
    Matrix x{{}, A_dst, Q_dst, 0, k};
    for (int i = 0; i < 3; ++i) {
        x.cs.qw[i] = qw[i], x.cs.qz[i] = qz[i], x.cs.s[i] = s[i];
        x.cs.width[i] = width[i], x.cs.rotary[i] = rotary[i];
        x.m += width[i];
    }
    x.cs.interleave = interleave;
    return x;
}

}  // namespace

hipError_t launch_convert(uint32_t* A_dst, uint32_t* Q_dst, const uint32_t* A_src, const uint16_t* scales,
                          const uint32_t* qzeros, int m, int k, int group, hipStream_t st)
{
    const Matrix one[1] = {plain(A_dst, Q_dst, A_src, scales, qzeros, m, k)};
    return launch_matrices(one, group, st);
}

hipError_t launch_deploy(uint32_t* A_dst, uint32_t* Q_dst, const uint32_t* const qw[3], const uint32_t* const qz[3],
                         const uint16_t* const s[3], const int width[3], const int rotary[3], int interleave, int k,
                         int group, hipStream_t st)
{
    const Matrix one[1] = {gathered(A_dst, Q_dst, qw, qz, s, width, rotary, interleave, k)};
    return launch_matrices(one, group, st);
}

hipError_t launch_deploy_layer(uint32_t* const A[4], uint32_t* const Q[4], const uint32_t* const qw[7], const uint32_t* const qz[7],
                               const uint16_t* const s[7], const int n[7], const int k[4], int size_per_head, int group, hipStream_t st)
{
    const uint32_t *const gate_up[3] = {qw[4], qw[5], nullptr}, *const gate_up_z[3] = {qz[4], qz[5], nullptr};
    const uint16_t* const gate_up_s[3] = {s[4], s[5], nullptr};
    const int             heads[3] = {size_per_head, size_per_head, 0}, none[3] = {0, 0, 0}, gate_up_n[3] = {n[4], n[5], 0};
    const Matrix          layer[4] = {gathered(A[0], Q[0], qw, qz, s, n, heads, 0, k[0]), plain(A[1], Q[1], qw[3], s[3], qz[3], n[3], k[1]),
                                      gathered(A[2], Q[2], gate_up, gate_up_z, gate_up_s, gate_up_n, none, 1, k[2]),
                                      plain(A[3], Q[3], qw[6], s[6], qz[6], n[6], k[3])};
    return launch_matrices(layer, group, st);
}

hipError_t launch_unpack(uint32_t* qweight, uint32_t* qzeros, uint16_t* scales, const uint32_t* A,
                         const uint32_t* Q, int m, int k, int group, hipStream_t st)
{
    const int64_t words = (int64_t)m * k / 8;
    const int64_t qw    = (int64_t)(k / group) * m / 8;
    if (words == 0) return hipSuccess;
    hipError_t e = hipSuccess;
    if (qweight) e = launch_kernel(unrepack_weights_kernel, dim3(blocks_for(words)), dim3(kThreads), 0, st, qweight, A, m, k);
    if ((qzeros || scales) && e == hipSuccess)
        e = launch_kernel(split_q_kernel, dim3(blocks_for(qw)), dim3(kThreads), 0, st, qzeros, scales, Q, qw);
    return e;
}

hipError_t launch_dequantize_repacked(uint16_t* W, const uint32_t* A, const uint32_t* Q, int m, int k, int group,
                                      hipStream_t st)
{
    const int64_t words = (int64_t)m * k / 8;
    if (words == 0) return hipSuccess;
    return launch_kernel(dequantize_repacked_kernel, dim3(blocks_for(words)), dim3(kThreads), 0, st, W, A, Q, m, k, group);
}

hipError_t launch_dequantize_s4(void* dst, const uint32_t* src, size_t count, hipStream_t st)
{
    if (count == 0) return hipSuccess;
    return launch_kernel(dequantize_s4_kernel, dim3(blocks_for((int64_t)count)), dim3(kThreads), 0, st, (uint4*)dst,
                         src, (int64_t)count);
}

hipError_t launch_fuse_w1_w3(uint32_t* dst, const uint32_t* src, int m, int k, hipStream_t st)
{
    const int64_t words = (int64_t)k * (2 * m / 8);
    if (words == 0) return hipSuccess;
    return launch_kernel(fuse_w1_w3_kernel, dim3(blocks_for(words)), dim3(kThreads), 0, st, dst, src, m, k);
}

hipError_t launch_transpose_qk(uint32_t* dst, const uint32_t* src, int m, int k, int size_per_head, hipStream_t st)
{
    const int64_t words = (int64_t)k * (m / 8);
    if (words == 0) return hipSuccess;
    return launch_kernel(transpose_qk_kernel, dim3(blocks_for(words)), dim3(kThreads), 0, st, dst, src, m, k,
                         size_per_head);
}

hipError_t launch_from_reference(uint32_t* dst, const uint32_t* ref, int m, int k, hipStream_t st)
{
    const int64_t words = (int64_t)m * k / 8;
    if (words == 0) return hipSuccess;
    return launch_kernel(from_reference_kernel, dim3(blocks_for(words)), dim3(kThreads), 0, st, dst, ref, m, k);
}

}  // namespace w4a16
