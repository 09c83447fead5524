// The whole-number arithmetic of csrc/w4a16_common.h that kernels and host share, as functions to call from a test, and what
// the members of a configuration are.
#include "../../lmdeploy_amd/csrc/w4a16_common.h"

extern "C" int arrive(int* counters, int tile, int splits, int epoch) { return w4a16::arrive_last(counters, tile, splits, epoch); }
extern "C" int layout(int which) { return (int)(which == 0 ? w4a16::kStaticCounters : which == 1 ? w4a16::kStaticTagged : w4a16::kEpochShift); }

extern "C" unsigned reciprocal_of(unsigned long long bound, unsigned d) { return w4a16::reciprocal(bound, d); }
extern "C" unsigned divide(unsigned n, unsigned d, unsigned by) { return w4a16::divide_by(n, d, by); }

// Workgroup `id` of a launch, with the reciprocals that the launch makes: (token tile, column tile or strip, split, first group, end)
extern "C" void tile_at(unsigned id, int tiles_t, int tiles_n, int groups, int splits, int split, int* out)
{
    const unsigned         by = w4a16::reciprocal((uint64_t)tiles_t * tiles_n, w4a16::tile_divisor(tiles_t, tiles_n));
    const w4a16::TilePlace p  = w4a16::tile_place((int)id, tiles_t, tiles_n, by, groups, split, w4a16::log2_of(splits));
    out[0] = p.tile_t, out[1] = p.tile_n, out[2] = split, out[3] = p.gbeg, out[4] = p.gend;
}
extern "C" void batch_at(unsigned id, unsigned strips, unsigned tiles_t, int splits, int* out)
{
    const unsigned          z = (unsigned)w4a16::log2_of(splits);
    const w4a16::BatchPlace p = w4a16::batch_place(id, strips, tiles_t, w4a16::by_batch_strips(strips, z), w4a16::by_batch_tiles(strips, tiles_t, z), z);
    out[0] = p.tile_t, out[1] = p.strip, out[2] = (int)p.split;
}

extern "C" void describe(const w4a16::Algo* a, int* out)
{
    out[0] = a->family == w4a16::kBatch ? 'b' : a->family == w4a16::kStrip ? 's' : 't';
    out[1] = a->tile_n, out[2] = a->tile_t, out[3] = a->bc.splits;
}
