// The whole-number arithmetic of csrc/w4a16_common.h that kernels and host share, as functions to call from a test.
#include "../../lmdeploy_amd/csrc/w4a16_common.h"

extern "C" int arrive(int* counters, int tile, int splits, int epoch) { return w4a16::arrive_last(counters, tile, splits, epoch); }
extern "C" int layout(int which) { return (int)(which == 0 ? w4a16::kStaticCounters : which == 1 ? w4a16::kStaticTagged : w4a16::kEpochShift); }
