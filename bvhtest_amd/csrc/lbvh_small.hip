// Small builds: scene box, Morton keys and sort of one mesh in one workgroup.
//
// A mesh of up to a few thousand triangles does not fill a launch of the
// large build's kernels: eight launches, each a workgroup or a few waiting on
// its own loads.  Here one workgroup of 1,024 threads keeps everything in
// registers and LDS: it loads the triangles (ITEMS per thread), reduces the
// box of the vertices they reference (the reference's box, so there is
// nothing to repair), makes the keys and sorts (key, index) with one stable
// 8-bit pass per digit; the indices leave in sorted order.
// Bound by latency and by the issue of one CU.  Whole builds, 30-bit keys, at
// 100 / 1,000 / 4,000 / 8,000 triangles: 12.7 / 16.9 / 26.3 / 38.1 us against
// 64.1 / 70.9 / 77.0 / 80.0 us with the large build's kernels; 63-bit keys
// 17.7 / 22.8 / 39.0 / 60.5 against 76.6 / 86.1 / 93.0 / 97.0.
#include "lbvh_small.hpp"
#include "lbvh_kernels.hpp"
#include "wave.hpp"

namespace bvht {

namespace {

constexpr int kSmallBlock = 1024, kSmallWaves = kSmallBlock / 64;

// PASSES 8-bit digits of the key; positions past n hold the largest key and
// stay behind every triangle (no Morton key has 255 as its top digit).
template <typename K, int PASSES, int ITEMS>
__global__ __launch_bounds__(kSmallBlock) void k_smallSort(const bvht_vec3 *__restrict__ vert,
                                                           const bvht_Triangle *__restrict__ faces, uint32_t n,
                                                           BuildParams *__restrict__ prm, K *__restrict__ keysOut,
                                                           uint32_t *__restrict__ valsOut, uint32_t *err,
                                                           uint32_t *errLong) {
  __shared__ K s_key[kSmallBlock * ITEMS];
  __shared__ uint16_t s_idx[kSmallBlock * ITEMS];
  __shared__ uint32_t s_wave[kSmallWaves][kSortRadix];
  __shared__ uint32_t s_start[kSortRadix], s_scan[kSortRadix / 64];
  __shared__ float s_red[6][kSmallWaves];
  static_assert(kSmallBlock * ITEMS <= 65536, "indices in 16 bits");
  const uint32_t tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const uint32_t first = wave * 64 * ITEMS + lane;  // item i is triangle first + 64 i

  // a repeat of triangle 0 past the end changes no min / max
  bvht_vec3 c[ITEMS];
  float mn[3] = {HUGE_VALF, HUGE_VALF, HUGE_VALF}, mx[3] = {-HUGE_VALF, -HUGE_VALF, -HUGE_VALF};
  bvht_Triangle t[ITEMS];
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) t[i] = faces[first + 64 * i < n ? first + 64 * i : 0u];
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    const bvht_vec3 a = vert[t[i].v1], b = vert[t[i].v2], d = vert[t[i].v3];
    c[i] = centroid(a, b, d);
    mn[0] = fminf(mn[0], fminf(fminf(a.x, b.x), d.x));
    mn[1] = fminf(mn[1], fminf(fminf(a.y, b.y), d.y));
    mn[2] = fminf(mn[2], fminf(fminf(a.z, b.z), d.z));
    mx[0] = fmaxf(mx[0], fmaxf(fmaxf(a.x, b.x), d.x));
    mx[1] = fmaxf(mx[1], fmaxf(fmaxf(a.y, b.y), d.y));
    mx[2] = fmaxf(mx[2], fmaxf(fmaxf(a.z, b.z), d.z));
  }
  shiftedBox(mn, mx);
  float box[6];
  blockBox(mn, mx, s_red, box);
  bvht_vec3 off, sc;
  mortonMapping(box, off, sc);
  if (tid == 0) {
    *err = *errLong = 0;  // an earlier staged sort's: this one has no wait to give up
    for (int a = 0; a < 3; ++a) {
      prm->sceneMin[a] = box[a];
      prm->sceneMax[a] = box[3 + a];
      prm->offset[a] = (&off.x)[a];
      prm->scale[a] = (&sc.x)[a];
    }
  }
  K key[ITEMS];
  uint32_t idx[ITEMS];
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    idx[i] = first + 64 * i;
    if constexpr (sizeof(K) == 8)
      key[i] = morton63(c[i], off, sc);
    else
      key[i] = morton30(c[i], off, sc);
    if (idx[i] >= n) key[i] = ~(K)0;
  }

  uint32_t *cnt = &s_wave[wave][0];
  const uint64_t lt = __lanemask_lt();
#pragma unroll 1
  for (int pass = 0; pass < PASSES; ++pass) {
    const uint32_t shift = pass * kSortRadixBits;
#pragma unroll
    for (uint32_t j = 0; j < kSortRadix / 64; ++j) cnt[lane + 64 * j] = 0;  // the wave's own counters
    memoryChanged();
    uint32_t at[ITEMS];
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {  // stable ranking, as in the onesweep passes
      const uint32_t d = (uint32_t)(key[i] >> shift) & (kSortRadix - 1);
      const uint64_t peers = matchDigit<kSortRadixBits>(d, ~0ull);
      const uint32_t lower = (uint32_t)__popcll(peers & lt);
      const uint32_t before = __hip_atomic_load(cnt + d, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      at[i] = before + lower;
      if (lower == 0)
        __hip_atomic_store(cnt + d, before + (uint32_t)__popcll(peers), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    __syncthreads();
    uint32_t total = 0, inc = 0;
    if (tid < (uint32_t)kSortRadix) {  // digit owners: offsets of each wave, then the digits' starts
#pragma unroll
      for (int w = 0; w < kSmallWaves; ++w) {
        const uint32_t x = s_wave[w][tid];
        s_wave[w][tid] = total;
        total += x;
      }
      inc = waveInclusiveScan(total);
      if (lane == 63) s_scan[wave] = inc;
    }
    __syncthreads();
    if (tid < (uint32_t)kSortRadix) {
      uint32_t before = 0;
      for (uint32_t w = 0; w < wave; ++w) before += s_scan[w];
      s_start[tid] = before + inc - total;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      const uint32_t d = (uint32_t)(key[i] >> shift) & (kSortRadix - 1);
      const uint32_t p = at[i] + s_start[d] + s_wave[wave][d];
      s_key[p] = key[i];
      s_idx[p] = (uint16_t)idx[i];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      key[i] = s_key[first + 64 * i];
      idx[i] = s_idx[first + 64 * i];
    }
    // the next pass writes s_key and s_idx after two more barriers; its
    // counters are the wave's own until then
  }
#pragma unroll
  for (int i = 0; i < ITEMS; ++i)
    if (first + 64 * i < n) {
      valsOut[first + 64 * i] = idx[i];
      if (keysOut) keysOut[first + 64 * i] = key[i];
    }
}

template <typename K, int PASSES, int ITEMS>
void launchSmall(const bvht_MeshRaw &mesh, BuildParams *prm, void *keysOut, uint32_t *valsOut, uint32_t *const err[2]) {
  k_smallSort<K, PASSES, ITEMS><<<1, kSmallBlock, 0, stream()>>>(mesh.vert, mesh.faces, mesh.numFaces, prm,
                                                                 static_cast<K *>(keysOut), valsOut, err[0], err[1]);
}

}  // namespace

bool smallSort(const bvht_MeshRaw &mesh, int mortonBits, BuildParams *prm, void *keysOut, uint32_t *valsOut,
               uint32_t *const err[2]) {
  const bool wide = mortonBits == 63;
  switch (divUp(mesh.numFaces, kSmallBlock)) {
#define BVHT_SMALL(I)                                                   \
  case I:                                                               \
    if (wide)                                                           \
      launchSmall<uint64_t, 8, I>(mesh, prm, keysOut, valsOut, err);    \
    else                                                                \
      launchSmall<uint32_t, 4, I>(mesh, prm, keysOut, valsOut, err);    \
    break;
    BVHT_SMALL(1)
    BVHT_SMALL(2)
    BVHT_SMALL(3)
    BVHT_SMALL(4)
    BVHT_SMALL(5)
    BVHT_SMALL(6)
    BVHT_SMALL(7)
    BVHT_SMALL(8)
#undef BVHT_SMALL
    default:
      setError("smallSort: %u triangles exceed %u", mesh.numFaces, kSmallSortMax);
      return false;
  }
  return checkLaunch("k_smallSort");
}

}  // namespace bvht
