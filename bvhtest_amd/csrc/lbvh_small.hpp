// One-workgroup key and sort stage of small LBVH builds (lbvh_small.hip).
#pragma once

#include "lbvh.hpp"
#include "runtime.hpp"

namespace bvht {

// Meshes of up to this many triangles take it: 8 per thread, what fits the
// registers (16 per thread spilled 101 of them and took 92.6 us for 12,000
// triangles, the large build's kernels 84.1).
constexpr uint32_t kSmallSortMax = 8192;

// Scene box (into prm), Morton keys and their stable sort: valsOut[p] is the
// triangle at sorted position p, keysOut (may be null) its key (uint64 for 63
// bits, uint32 for 30).  numFaces in [1, kSmallSortMax].  The words err become 0.
bool smallSort(const bvht_MeshRaw &mesh, int mortonBits, BuildParams *prm, void *keysOut, uint32_t *valsOut,
               uint32_t *const err[2]);

}  // namespace bvht
