// Ray generation and traversal for gfx950
// (reference: lib/tracer/CUDAKernels.cu:43-223, :386-417).
//
// Traversal visits nodes in the reference's order (Afra & Szirmay-Kalos
// 2014, the bit-trail algorithm of kTraceRay): at an inner node both children
// are tested against the current nearest hit, the nearer hit child is entered
// first and the other one later, without a second box test.  What makes it
// fast without changing that order:
//   * every node becomes one 64-byte record (k_packNodes): an inner node holds
//     its two children's boxes and references, a leaf its triangle as
//     (v0, e1, e2) (the same f32 subtractions the test makes), in leaf order,
//     so a visit is one record whichever kind it is;
//   * a reference is one word (node id, top bit: leaf), and the children still
//     to be entered are kept in a 24-entry per-lane LDS stack of them.  A ray
//     that needs a 25th starts over with the reference's 128-bit trail and its
//     parent links (slowWalk), so the common walk carries neither;
//   * the walk is bound by the L1's accesses and by vector issue (75% and 59%
//     of the cycles on primary rays at 1080p over 4.2M triangles, with 29 of 64
//     lanes active; 49%, 49% and 26 on secondary rays), so a step visits an
//     inner node and, if that leads to one, the leaf: a ray's last box test and
//     its triangle test take one step of the wave.  A lane's own sequence of
//     visits does not change.
// Measured against separate pair and triangle records, a 16-entry ring and a
// trail in every walk, one visit a step (1080p, 4.2M triangles; 512x512, 65k):
// primary rays 3.65 -> 3.27 ms and 278 -> 240 us, secondary rays 4.05 -> 4.00 ms
// and 681 -> 600 us.  Either kind in a step: 3.67 ms; the kind that more lanes
// wait for: 3.87 ms.  16, 20, 24, 32, 48 entries: 4.26 (rays that start over),
// 3.31, 3.27, 3.52, 4.10 ms (the LDS limits the waves).
// Arithmetic is f32 with no FMA contraction and IEEE division, so the visit
// order, hit triangle and distance are a pure function of the inputs (the
// oracle reproduces them exactly).  The 128-bit mask limits trees to depth
// 128, as the reference's trail does.
//
// Rays are generated in f64 from a camera basis computed in f64 on the host
// (the exact inverse of lookAtRH), then rounded once to f32.
#include "radix_sort.hpp"
#include "runtime.hpp"
#include "types.hpp"

#include <algorithm>
#include <cmath>

namespace bvht {

namespace {

constexpr uint32_t kNoHit = 0xFFFFFFFFu;

struct CamBasis {
  double s[3], u[3], f[3];
  float pos[3];
  float scale, ratio;
};

__device__ __forceinline__ void setRay(bvht_Ray &r, bvht_vec3 pos, bvht_vec3 dir, uint32_t x, uint32_t y) {
  // Ray::set -- lib/base/Ray.hpp:65-74
  r.pos = pos;
  r.dir = dir;
  r.px = x;
  r.py = y;
  r.invDir = {__fdiv_rn(1.0f, dir.x), __fdiv_rn(1.0f, dir.y), __fdiv_rn(1.0f, dir.z)};
  r.sign[0] = r.invDir.x < 0 ? 1 : 0;
  r.sign[1] = r.invDir.y < 0 ? 1 : 0;
  r.sign[2] = r.invDir.z < 0 ? 1 : 0;
  r._pad = 0;
}

// kGenerateRays -- CUDAKernels.cu:43-59.  A wave's 64 rays are consecutive
// and leave through LDS, as the records do in k_packNodes (1024x1024: 17.5 us
// with 48 bytes from each lane of 16x16 tiles, now 11.7).  `rays` starts at row y0.
__global__ __launch_bounds__(256) void k_genRays(bvht_Ray *__restrict__ rays, uint32_t w, uint32_t h, uint32_t y0,
                                                  uint32_t num, CamBasis cam) {
  static_assert(sizeof(bvht_Ray) == 48, "three 16-byte words a ray");
  __shared__ uint4 s_ray[4][64 * 3];
  const uint32_t i = blockIdx.x * 256 + threadIdx.x, lane = threadIdx.x & 63, first = i - lane;
  if (first >= num) return;
  const uint32_t row = i / w, x = i - row * w, y = y0 + row;
  const float px = (float)((2 * ((x + 0.5) / w) - 1) * cam.scale * cam.ratio);
  const float py = (float)((1 - 2 * ((y + 0.5) / h)) * cam.scale);
  double d[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) d[k] = (double)px * cam.s[k] + (double)py * cam.u[k] + cam.f[k];
  const double dl = sqrt(d[0] * d[0] + d[1] * d[1] + d[2] * d[2]);
  bvht_vec3 dir = {(float)(d[0] / dl), (float)(d[1] / dl), (float)(d[2] / dl)};
  bvht_Ray r;
  setRay(r, bvht_vec3{cam.pos[0], cam.pos[1], cam.pos[2]}, dir, x, y);
  uint4 *stage = s_ray[threadIdx.x / 64];
  uint4 words[3];
  __builtin_memcpy(words, &r, sizeof(r));
#pragma unroll
  for (int k = 0; k < 3; ++k) stage[3 * lane + k] = words[k];
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // its own wave's words only
  __builtin_amdgcn_wave_barrier();
  uint4 *out = reinterpret_cast<uint4 *>(rays + first);
  const uint32_t count = 3 * min(64u, num - first);
#pragma unroll
  for (uint32_t k = 0; k < 3; ++k)
    if (k * 64 + lane < count) out[k * 64 + lane] = stage[k * 64 + lane];
}

__device__ __forceinline__ bvht_vec3 vsub(bvht_vec3 a, bvht_vec3 b) { return {a.x - b.x, a.y - b.y, a.z - b.z}; }
__device__ __forceinline__ bvht_vec3 vcross(bvht_vec3 x, bvht_vec3 y) {
  return {x.y * y.z - y.y * x.z, x.z * y.x - y.z * x.x, x.x * y.y - y.x * x.y};
}
__device__ __forceinline__ float vdot(bvht_vec3 a, bvht_vec3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
// glm::normalize = v * (1 / sqrt(dot(v, v))), both operations correctly
// rounded.  sqrtf (not __fsqrt_rn, which maps to the 1-ulp v_sqrt_f32 on this
// toolchain) lowers to v_sqrt_f32 plus an fma residual correction.
__device__ __forceinline__ bvht_vec3 vnormalize(bvht_vec3 v) {
  float s = __fdiv_rn(1.0f, sqrtf(vdot(v, v)));
  return {v.x * s, v.y * s, v.z * s};
}

struct TraceOut {
  uint32_t tri;
  float t;
  uint16_t intCount;
};

// One node, 64 bytes.  Inner: a b c hold the left child's box, then the
// right's (min.xyz max.xyz each), d.x and d.y the children's references.
// Leaf: a = v0 and the first face, b = e1 = v1 - v0 and the face count,
// c = e2 = v2 - v0 (of that face).  d.z is 0.
struct NodeRec {
  float4 a, b, c;
  uint4 d;
};
static_assert(sizeof(NodeRec) == 64, "one record per visit");
constexpr uint32_t kLeafRef = 0x80000000u;  // the other bits: node id
// No child: past every reference, since prepareTrace takes fewer than kLeafRef
// nodes (up to 2^30 triangles).
constexpr uint32_t kNoChild = 0xFFFFFFFFu;
static_assert(((kLeafRef - 2) | kLeafRef) < kNoChild, "the last node of the largest tree has a reference of its own");
constexpr int kStackCap = 24;  // pending children per lane: 6 KiB of LDS a wave, 26 waves on a CU
// k_traceRaysDyn waves on a CU.  16, 20, 24, 26: 4.11, 3.99, 4.14, 4.13 ms at
// 1080p over 4.2M triangles, 685, 600, 608, 602 us at 512x512 over 65k (beyond
// 20 the waves displace each other's records from the L1).
constexpr uint32_t kTraceWavesPerCU = 20;
// Idle lanes that make a k_traceRaysDyn wave fetch rays.  8, 12, 16, 24, 32, 48: 4.37,
// 3.97, 3.98, 3.93, 3.94, 4.03 ms at 1080p over 4.2M triangles, 622, 612, 601, 585,
// 575, 554 us at 1024x1024 over 65k.
constexpr uint32_t kRefillAt = 32;

// One node's record.  A child index at or past `bound` becomes kNoChild with
// an empty box and raises *bad (the traversal then never reads past the
// arrays).
__device__ __forceinline__ NodeRec packNode(uint32_t i, const bvht_BVHNode *__restrict__ nodes, uint32_t bound,
                                            const bvht_Triangle *__restrict__ faces,
                                            const bvht_vec3 *__restrict__ vert, uint32_t numFaces,
                                            uint32_t *__restrict__ bad) {
  const uint4 *w = reinterpret_cast<const uint4 *>(nodes + i);
  const uint32_t left = w[1].w;
  const uint2 rf = *reinterpret_cast<const uint2 *>(w + 2);  // right, flags
  NodeRec p;
  p.d = make_uint4(0, 0, 0, 0);
  if ((rf.y & 0xFFFFu) != 0) {
    bvht_vec3 v0 = {0.f, 0.f, 0.f}, e1 = v0, e2 = v0;
    if (left < numFaces) {
      const bvht_Triangle t = faces[left];
      v0 = vert[t.v1];
      e1 = vsub(vert[t.v2], v0);
      e2 = vsub(vert[t.v3], v0);
    }
    p.a = make_float4(v0.x, v0.y, v0.z, __uint_as_float(left));
    p.b = make_float4(e1.x, e1.y, e1.z, __uint_as_float(rf.x));
    p.c = make_float4(e2.x, e2.y, e2.z, 0.f);
  } else {
    uint32_t child[2] = {left, rf.x};
    bvht_AABB box[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      if (child[k] < bound) {
        box[k] = nodes[child[k]].bbox;
        if (nodes[child[k]].isLeafFlag != 0) child[k] |= kLeafRef;
      } else {
        *bad = 1;
        box[k] = {{{0.f, 0.f, 0.f}, {-1.f, -1.f, -1.f}}};
        child[k] = kNoChild;
      }
    }
    p.a = make_float4(box[0].minMax[0].x, box[0].minMax[0].y, box[0].minMax[0].z, box[0].minMax[1].x);
    p.b = make_float4(box[0].minMax[1].y, box[0].minMax[1].z, box[1].minMax[0].x, box[1].minMax[0].y);
    p.c = make_float4(box[1].minMax[0].z, box[1].minMax[1].x, box[1].minMax[1].y, box[1].minMax[1].z);
    p.d.x = child[0];
    p.d.y = child[1];
  }
  return p;
}
// Packs every node below `bound`.  Bound by memory (1.1 GB at 4.2M triangles):
// a wave's 64 records go through LDS, word w of record r at slot
// 4 r + (w + r / 2) % 4 (eight lanes' 16-byte accesses then cover all the
// banks), and out as 4 KiB of consecutive bytes: 241 us, against 288 with 16
// bytes every 64 from each lane and 255 with workgroups of one wave.  The leaves
// (2i) and inner nodes (2i + 1) of the builder's order in one sequence cost the
// walks 15%: siblings then lie in two cache lines.
__global__ __launch_bounds__(256) void k_packNodes(const bvht_BVHNode *__restrict__ nodes, uint32_t bound,
                                                  const bvht_Triangle *__restrict__ faces,
                                                  const bvht_vec3 *__restrict__ vert, uint32_t numFaces,
                                                  NodeRec *__restrict__ recs, uint32_t *__restrict__ bad) {
  __shared__ float4 s_rec[4][64 * 4];
  const uint32_t i = blockIdx.x * 256 + threadIdx.x, lane = threadIdx.x & 63, first = i - lane;
  if (first >= bound) return;
  float4 *stage = s_rec[threadIdx.x / 64];
  if (i < bound) {
    const NodeRec p = packNode(i, nodes, bound, faces, vert, numFaces, bad);
    const uint32_t r = lane >> 1;
    stage[4 * lane + (r & 3)] = p.a;
    stage[4 * lane + ((r + 1) & 3)] = p.b;
    stage[4 * lane + ((r + 2) & 3)] = p.c;
    stage[4 * lane + ((r + 3) & 3)] =
        make_float4(__uint_as_float(p.d.x), __uint_as_float(p.d.y), __uint_as_float(p.d.z), __uint_as_float(p.d.w));
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // its own wave's words only
  __builtin_amdgcn_wave_barrier();
  float4 *out = reinterpret_cast<float4 *>(recs + first);
  const uint32_t words = 4 * min(64u, bound - first);
#pragma unroll
  for (uint32_t k = 0; k < 4; ++k) {
    const uint32_t x = k * 64 + lane, rec = x / 4;
    if (x < words) out[x] = stage[4 * rec + ((x + (rec >> 1)) & 3)];
  }
}

// Rays of a wave that all have the same signs (most tiles of an image) are
// walked by a loop made for them (OCT: the signs, x y z in bits 0 1 2): the near
// and far planes of a box are then named instead of selected, 12 of about 75
// instructions of a visit (primary rays, 1080p over 4.2M triangles 3.21 ->
// 3.15 ms, a 1024x1024 image of 65k 245 -> 234 us).  kAnyOct: any signs.  (Scalar
// loads where all of a wave's rays are at one node lost: 3.27 ms and 262 us.)
constexpr int kAnyOct = 8;

// A ray in registers; sx, sy, sz are its sign flags.
struct WalkRay {
  bvht_vec3 pos, dir, inv;
  bool sx, sy, sz;
};
__device__ __forceinline__ WalkRay walkRay(const bvht_Ray &r) {
  return WalkRay{r.pos, r.dir, r.invDir, r.sign[0] != 0, r.sign[1] != 0, r.sign[2] != 0};
}

// intersectRayAABB -- CUDAKernels.cu:66-85, on a packed box, against
// (0.01, t1).  The reference starts from x and takes y and z where they
// compare greater (near) or smaller (far): a NaN there is ignored, as max and
// min do, and a NaN in x makes the box missed, which the ordered compare adds.
template <int OCT>
__device__ __forceinline__ bool hitBox6(float mnx, float mny, float mnz, float mxx, float mxy, float mxz,
                                        const WalkRay &r, float t1, float &tmin) {
  const bool sx = OCT == kAnyOct ? r.sx : (OCT & 1) != 0, sy = OCT == kAnyOct ? r.sy : (OCT & 2) != 0,
             sz = OCT == kAnyOct ? r.sz : (OCT & 4) != 0;
  const float nx = ((sx ? mxx : mnx) - r.pos.x) * r.inv.x, fx = ((sx ? mnx : mxx) - r.pos.x) * r.inv.x;
  const float ny = ((sy ? mxy : mny) - r.pos.y) * r.inv.y, fy = ((sy ? mny : mxy) - r.pos.y) * r.inv.y;
  const float nz = ((sz ? mxz : mnz) - r.pos.z) * r.inv.z, fz = ((sz ? mnz : mxz) - r.pos.z) * r.inv.z;
  tmin = fmaxf(fmaxf(nx, ny), nz);
  const float tmax = fminf(fminf(fx, fy), fz);
  return !__builtin_isunordered(nx, fx) & (tmin < fminf(tmax, t1)) & (tmax > 0.01f);
}

// intersectRayTriangle2 -- CUDAKernels.cu:88-112, one-sided (the
// cudaFaceCulling default, meson_options.txt:1), on v0 and the two edges.
// IEEE 1/det replaces __fdividef; only hits divide.
__device__ __forceinline__ bool hitTri(const WalkRay &r, bvht_vec3 v0, bvht_vec3 e1, bvht_vec3 e2, float &dist) {
  const bvht_vec3 p = vcross(r.dir, e2);
  const float det = vdot(e1, p);
  const bvht_vec3 tv = vsub(r.pos, v0);
  const bvht_vec3 q = vcross(tv, e1);
  const float u = vdot(tv, p);
  const float v = vdot(r.dir, q);
  if (!((det > 0.0f) & (u >= 0.0f) & (u <= det) & (v >= 0.0f) & (u + v <= det))) return false;
  dist = vdot(e2, q) * __fdiv_rn(1.0f, det);
  return true;
}

struct TraceCtx {
  const NodeRec *recs;
  const bvht_BVHNode *nodes;  // parent links (dropped children)
  const bvht_Triangle *faces;
  const bvht_vec3 *vert;
  uint32_t bound;  // node count the packing covered
  uint32_t numFaces;
};

// One ray's walk (kTraceRay's loop, CUDAKernels.cu:146-204) between two visits.
struct Walk {
  uint32_t ref;    // the node to visit
  uint32_t sp;     // pending children on the stack; kStackCap + 1: one too many, see slowWalk
  uint32_t count;  // inner nodes visited
  uint32_t tri;
  uint32_t ahead;  // AHEAD: 0, from the children's records, taken at the next visit
  float nearest, t1;  // t1 = nearest + 0.01: boxes beyond are not entered
};

__device__ __forceinline__ void walkReset(Walk &s, uint32_t rootRef) {
  s.ref = rootRef;
  s.sp = s.count = s.ahead = 0;
  s.tri = kNoHit;
  s.nearest = s.t1 = HUGE_VALF;
}
__device__ __forceinline__ uint32_t rootRef(const TraceCtx &cx, uint32_t root) {
  return root | (cx.nodes[root].isLeafFlag != 0 ? kLeafRef : 0u);
}

// Goes to the next pending child; false: the walk has ended.
__device__ __forceinline__ bool walkPop(Walk &s, const uint32_t *stk) {
  if (s.sp == 0) return false;
  --s.sp;
  s.ref = stk[s.sp * 64];
  return true;
}

// The two children of an inner node: which one is entered now and which one
// waits (kNoChild: none).
template <int OCT>
__device__ __forceinline__ void innerChildren(const NodeRec *r, const WalkRay &ray, float t1, uint32_t &now,
                                              uint32_t &later) {
  const float4 a = r->a, b = r->b, c = r->c;
  const uint2 d = *reinterpret_cast<const uint2 *>(&r->d);
  float minL, minR;
  const bool hl = hitBox6<OCT>(a.x, a.y, a.z, a.w, b.x, b.y, ray, t1, minL);
  const bool hr = hitBox6<OCT>(b.z, b.w, c.x, c.y, c.z, c.w, ray, t1, minR);
  const bool both = hl & hr, left = hl & (!hr | (minL < minR));
  now = (hl | hr) ? (left ? d.x : d.y) : kNoChild;
  later = both ? (left ? d.y : d.x) : kNoChild;
}

// Visits an inner node; false: the walk has ended or gone past the stack.
// `stk` is this lane's column of a [kStackCap][64] LDS array.
// AHEAD: both children's records are asked for as soon as their references are
// known, beside the box tests (a word that is 0 in every record, added to the
// count a visit later), so the one that is visited next is on its way to the
// L1.  For launches that leave the GPU room, whose time is their longest walk's;
// see walksAhead.
template <int OCT, bool AHEAD>
__device__ __forceinline__ bool visitInner(Walk &s, const WalkRay &ray, const TraceCtx &cx, uint32_t *stk) {
  uint32_t now, later;
  const NodeRec *r = cx.recs + s.ref;
  if constexpr (AHEAD) {
    const uint2 d = *reinterpret_cast<const uint2 *>(&r->d);
    const uint32_t before = s.ahead, most = cx.bound - 1;
    s.ahead = cx.recs[min(d.x & ~kLeafRef, most)].d.z | cx.recs[min(d.y & ~kLeafRef, most)].d.z;
    s.count += before;
  }
  innerChildren<OCT>(r, ray, s.t1, now, later);
  s.count++;
  if (later != kNoChild) {
    if (s.sp >= (uint32_t)kStackCap) {
      s.sp = kStackCap + 1;
      return false;
    }
    stk[s.sp * 64] = later;
    ++s.sp;
  }
  if (now == kNoChild) return walkPop(s, stk);
  s.ref = now;
  return true;
}

// Visits a leaf.  MODE 0: reference triangle test.  MODE 1: hits need
// t > tMin and are not the triangle `skip` (secondary rays leaving a surface).
template <int MODE>
__device__ __forceinline__ void leafHit(Walk &s, uint32_t tri, float dist, float tMin, uint32_t skip) {
  if (MODE == 1 && !(dist > tMin && tri != skip)) return;
  if (dist < s.nearest) {
    s.nearest = dist;
    s.t1 = dist + 0.01f;
    s.tri = tri;
  }
}
template <int MODE>
__device__ __forceinline__ void leafTest(Walk &s, const WalkRay &ray, const TraceCtx &cx, float tMin, uint32_t skip) {
  const uint32_t node = s.ref & ~kLeafRef;
  if (node < cx.bound) {
    const NodeRec *r = cx.recs + node;
    const float4 a = r->a, b = r->b, c = r->c;
    const uint32_t first = __float_as_uint(a.w), count = __float_as_uint(b.w);
    float dist;
    if (count == 0 || first >= cx.numFaces) return;
    if (hitTri(ray, {a.x, a.y, a.z}, {b.x, b.y, b.z}, {c.x, c.y, c.z}, dist))
      leafHit<MODE>(s, first, dist, tMin, skip);
    for (uint32_t k = 1; k < count; ++k) {  // leaves of several triangles
      const uint32_t t = first + k;
      if (t >= cx.numFaces) break;
      const bvht_Triangle f = cx.faces[t];
      const bvht_vec3 v0 = cx.vert[f.v1];
      if (hitTri(ray, v0, vsub(cx.vert[f.v2], v0), vsub(cx.vert[f.v3], v0), dist))
        leafHit<MODE>(s, t, dist, tMin, skip);
    }
  }
}
template <int MODE>
__device__ __forceinline__ bool visitLeaf(Walk &s, const WalkRay &ray, const TraceCtx &cx, float tMin, uint32_t skip,
                                          const uint32_t *stk) {
  leafTest<MODE>(s, ray, cx, tMin, skip);
  return walkPop(s, stk);
}

// One step of a wave's walks.  `active` lanes have a node to visit.
template <int MODE, int OCT, bool AHEAD>
__device__ __forceinline__ void walkStep(bool &active, Walk &s, const WalkRay &ray, const TraceCtx &cx,
                                         float tMin, uint32_t skip, uint32_t *stk) {
  if (active && (s.ref & kLeafRef) == 0) active = visitInner<OCT, AHEAD>(s, ray, cx, stk);
  if (active && (s.ref & kLeafRef) != 0) active = visitLeaf<MODE>(s, ray, cx, tMin, skip, stk);
}

// A valid tree is walked in at most ~4 visits per node; this bound on the
// inner visits (looked at now and then) only ends walks of a malformed
// (cyclic) tree, whose every cycle passes inner nodes.
constexpr uint32_t kMaxSteps = 1u << 26, kCheckSteps = 1u << 20;

// The walk of a ray that had more than kStackCap children pending, from the
// start: the reference's 128-bit trail (a 1 marks a level whose second child
// is still pending) and, where the stack has dropped a child, its parent links.
// The stack keeps the last kStackCap of the pending children (a ring: `end`
// is the place of the next, `kept` of them are there).  Same visits.  (Trees of
// one path over 32, 64 and 120 triangles, one above the other, 640x480: 45, 114
// and 189 us, without the ring 45, 130 and 208, with a ring in every walk 57,
// 103 and 182.  A stack that goes on in scratch memory needs no start over, but
// took 490 us instead of 290 for a 1024x1024 image of 65k triangles and 12.7 ms
// instead of 7.1 for a 1080p frame of 4.2M.)
template <int MODE>
__device__ __forceinline__ TraceOut slowWalk(const WalkRay &ray, const TraceCtx &cx, uint32_t top, float tMin,
                                             uint32_t skip, uint32_t *stk) {
  Walk s;
  walkReset(s, top);
  uint32_t end = 0, kept = 0;
  uint64_t lo = 0, hi = 0;
  while (s.count < kMaxSteps) {
    const bool leaf = (s.ref & kLeafRef) != 0;
    if (leaf) {
      leafTest<MODE>(s, ray, cx, tMin, skip);
    } else {
      uint32_t now, later;
      innerChildren<kAnyOct>(cx.recs + s.ref, ray, s.t1, now, later);
      s.count++;
      if (now == kNoChild) {  // a missing child's empty box, met by a ray with wrong signs
        now = later;
        later = kNoChild;
      }
      if (now != kNoChild) {
        hi = (hi << 1) | (lo >> 63);
        lo <<= 1;
        if (later != kNoChild) {
          lo |= 1;
          stk[end * 64] = later;
          end = end + 1 == (uint32_t)kStackCap ? 0u : end + 1;
          kept = min(kept + 1, (uint32_t)kStackCap);
        }
        s.ref = now;
        continue;
      }
    }
    if ((lo | hi) == 0) break;
    uint32_t up;  // levels to the deepest node whose second child is pending
    if (lo != 0) {
      up = (uint32_t)__builtin_ctzll(lo);
      if (up) {
        lo = (lo >> up) | (hi << (64 - up));
        hi >>= up;
      }
    } else {
      up = 64 + (uint32_t)__builtin_ctzll(hi);
      lo = hi >> (up - 64);
      hi = 0;
    }
    lo ^= 1;
    if (kept > 0) {
      --kept;
      end = end == 0 ? (uint32_t)kStackCap - 1 : end - 1;
      s.ref = stk[end * 64];
      continue;
    }
    uint32_t node = s.ref & ~kLeafRef;
    for (uint32_t k = 0; k < up && node < cx.bound; ++k) node = cx.nodes[node].parent;
    if (node >= cx.bound) break;
    const uint32_t p = cx.nodes[node].parent;
    if (p >= cx.bound) break;
    node = cx.nodes[node].isLeft == 0 ? cx.nodes[p].left : cx.nodes[p].right;
    if (node >= cx.bound) break;
    s.ref = rootRef(cx, node);
  }
  return TraceOut{s.tri, s.nearest, (uint16_t)s.count};
}

template <int MODE, int OCT, bool AHEAD>
__device__ __forceinline__ void walkLoop(bool active, Walk &s, const WalkRay &ray, const TraceCtx &cx, float tMin,
                                         uint32_t skip, uint32_t *stk) {
  for (uint32_t it = 1;; ++it) {
    if (__ballot(active) == 0) break;
    walkStep<MODE, OCT, AHEAD>(active, s, ray, cx, tMin, skip, stk);
    if ((it & (kCheckSteps - 1)) == 0 && s.count >= kMaxSteps) active = false;
  }
}

// Walks one ray per lane to its end (every lane of the wave calls).
template <int MODE, bool AHEAD>
__device__ __forceinline__ TraceOut walkAll(bool active, const bvht_Ray &r, const TraceCtx &cx, uint32_t root,
                                            float tMin, uint32_t skip, uint32_t *stk) {
  const WalkRay ray = walkRay(r);
  const uint32_t top = root < cx.bound ? rootRef(cx, root) : 0u;
  Walk s;
  walkReset(s, top);
  active = active && root < cx.bound;
  const uint64_t act = __ballot(active);
  const uint64_t nx = __ballot(active && ray.sx), ny = __ballot(active && ray.sy), nz = __ballot(active && ray.sz);
  uint32_t oct = kAnyOct;
  if ((nx == 0 || nx == act) && (ny == 0 || ny == act) && (nz == 0 || nz == act))
    oct = (nx != 0 ? 1 : 0) | (ny != 0 ? 2 : 0) | (nz != 0 ? 4 : 0);
  switch (oct) {  // wave-uniform
    case 0: walkLoop<MODE, 0, AHEAD>(active, s, ray, cx, tMin, skip, stk); break;
    case 1: walkLoop<MODE, 1, AHEAD>(active, s, ray, cx, tMin, skip, stk); break;
    case 2: walkLoop<MODE, 2, AHEAD>(active, s, ray, cx, tMin, skip, stk); break;
    case 3: walkLoop<MODE, 3, AHEAD>(active, s, ray, cx, tMin, skip, stk); break;
    case 4: walkLoop<MODE, 4, AHEAD>(active, s, ray, cx, tMin, skip, stk); break;
    case 5: walkLoop<MODE, 5, AHEAD>(active, s, ray, cx, tMin, skip, stk); break;
    case 6: walkLoop<MODE, 6, AHEAD>(active, s, ray, cx, tMin, skip, stk); break;
    case 7: walkLoop<MODE, 7, AHEAD>(active, s, ray, cx, tMin, skip, stk); break;
    default: walkLoop<MODE, kAnyOct, AHEAD>(active, s, ray, cx, tMin, skip, stk); break;
  }
  if (s.sp > (uint32_t)kStackCap) return slowWalk<MODE>(ray, cx, top, tMin, skip, stk);
  return TraceOut{s.tri, s.nearest, (uint16_t)s.count};
}

// Shading of CUDAKernels.cu:208-218.
__device__ __forceinline__ bvht_CUDAPixel shade(const TraceOut &o, const bvht_Ray &ray, const bvht_vec3 *vert,
                                                const bvht_Triangle *faces, bvht_vec3 light) {
  bvht_CUDAPixel px = {0, 0, o.intCount};
  if (o.t < HUGE_VALF) {
    const bvht_Triangle tri = faces[o.tri];
    const bvht_vec3 v1 = vert[tri.v1], v2 = vert[tri.v2], v3 = vert[tri.v3];
    const bvht_vec3 n = vnormalize(vcross(vsub(v2, v1), vsub(v3, v1)));
    const bvht_vec3 hp = {ray.pos.x + ray.dir.x * o.t, ray.pos.y + ray.dir.y * o.t, ray.pos.z + ray.dir.z * o.t};
    const bvht_vec3 ld = vnormalize(vsub(light, hp));
    float diff = 1.0f + vdot(n, ld);
    diff = diff > 0.0f ? diff : 0.0f;
    px.hit = 1;
    px.diffuse = (uint8_t)(diff * 127.0f);
  }
  return px;
}

// Pixel of lane l in an 8x8 tile: 2x2 blocks of lanes are 2x2 blocks of
// pixels, so the four lanes whose accesses the L1 merges first are neighbours
// both ways.
__device__ __forceinline__ uint32_t tileX(uint32_t l) { return (l & 1) | ((l >> 1) & 2) | ((l >> 2) & 4); }
__device__ __forceinline__ uint32_t tileY(uint32_t l) { return tileX(l >> 1); }

// Image path: 8x8 pixel tiles per wave (kTraceRay launch shape, CUDAKernels.cu:409-416).
template <bool AHEAD>
__global__ __launch_bounds__(64) void k_traceImage(const bvht_Ray *__restrict__ rays,
                                                      bvht_CUDAPixel *__restrict__ img, TraceCtx cx, uint32_t root,
                                                      bvht_vec3 light, uint32_t w, uint32_t h) {
  __shared__ uint32_t s_stk[kStackCap * 64];
  const uint32_t x = blockIdx.x * 8 + tileX(threadIdx.x);
  const uint32_t y = blockIdx.y * 8 + tileY(threadIdx.x);
  const bool in = x < w && y < h;
  const size_t i = in ? (size_t)y * w + x : 0;
  const bvht_Ray ray = rays[i];
  const TraceOut o = walkAll<0, AHEAD>(in, ray, cx, root, 0.0f, kNoHit, s_stk + threadIdx.x);
  if (in) img[i] = shade(o, ray, cx.vert, cx.faces, light);
}

// Ray bundles (kTraceRayBundle, CUDAKernels.cu:240-383): the 64 rays of an
// 8x8 tile -- one wave -- walk one shared node sequence.  At an inner node
// each ray tests both children against its own nearest hit; the bundle
// enters every child some ray hits, the one a majority prefers first (ties:
// right), and backtracks on one shared trail.  Ballots replace the
// reference's shared-memory flags and reduction.  Every ray still finds its
// nearest hit (the shared walk covers its own); among triangles at exactly
// the same distance the first one met may differ from the per-ray order.
__global__ __launch_bounds__(64) void k_traceImageBundle(const bvht_Ray *__restrict__ rays,
                                                         bvht_CUDAPixel *__restrict__ img, TraceCtx cx, uint32_t root,
                                                         bvht_vec3 light, uint32_t w, uint32_t h) {
  __shared__ uint32_t s_stk[128];  // pending children: at most one per trail bit
  const uint32_t x = blockIdx.x * 8 + (threadIdx.x & 7);
  const uint32_t y = blockIdx.y * 8 + (threadIdx.x >> 3);
  const bool valid = x < w && y < h;
  const bvht_Ray ray = rays[valid ? (size_t)y * w + x : 0];
  const WalkRay wr = walkRay(ray);
  TraceOut o = {kNoHit, HUGE_VALF, 0};
  if (root < cx.bound) {
    uint64_t lo = 0, hi = 0;  // wave-uniform from here on
    uint32_t ref = rootRef(cx, root), sp = 0, ahead = 0;
    float nearest = HUGE_VALF, dist;
    for (uint32_t steps = 0; steps < (1u << 26); ++steps) {
      const uint32_t node = ref & ~kLeafRef;
      if ((ref & kLeafRef) == 0) {
        // both children's records are asked for beside the box tests, as in
        // visitInner; here it is one address a wave, and pays at every size: 65k / 0.9M
        // triangles, 160x120 1,059 / 2,796 -> 828 / 2,181 us, 640x480 395 / 1,422 ->
        // 322 / 1,207, 1024x1024 283 / 2,865 -> 277 / 2,532, 1920x1080 290 / 2,614 -> 289 / 2,367
        const uint2 d = *reinterpret_cast<const uint2 *>(&cx.recs[node].d);
        const uint32_t before = ahead, most = cx.bound - 1;
        ahead = cx.recs[min(d.x & ~kLeafRef, most)].d.z | cx.recs[min(d.y & ~kLeafRef, most)].d.z;
        o.intCount += 1 + before;
        const NodeRec pp = cx.recs[node];
        float minL = 0.0f, minR = 0.0f;
        const bool hl =
            valid && hitBox6<kAnyOct>(pp.a.x, pp.a.y, pp.a.z, pp.a.w, pp.b.x, pp.b.y, wr, nearest + 0.01f, minL);
        const bool hr =
            valid && hitBox6<kAnyOct>(pp.b.z, pp.b.w, pp.c.x, pp.c.y, pp.c.z, pp.c.w, wr, nearest + 0.01f, minR);
        const bool anyL = __ballot(hl) != 0, anyR = __ballot(hr) != 0;
        if (anyL || anyR) {
          hi = (hi << 1) | (lo >> 63);
          lo <<= 1;
          if (anyL && anyR) {
            lo |= 1;
            const bool wantL = hl && (minL < minR || !hr), wantR = hr && (minR < minL || !hl);
            const int vote = __popcll(__ballot(wantL)) - __popcll(__ballot(wantR));
            const bool leftFirst = vote > 0;
            if (sp < 128) s_stk[sp] = leftFirst ? pp.d.y : pp.d.x;
            ++sp;
            ref = leftFirst ? pp.d.x : pp.d.y;
          } else {
            ref = anyL ? pp.d.x : pp.d.y;
          }
          continue;
        }
      } else if (node < cx.bound) {
        const NodeRec pt = cx.recs[node];
        const uint32_t first = __float_as_uint(pt.a.w), count = __float_as_uint(pt.b.w);
        for (uint32_t k = 0; k < count; ++k) {
          const uint32_t t = first + k;
          if (t >= cx.numFaces) break;
          bvht_vec3 v0 = {pt.a.x, pt.a.y, pt.a.z}, e1 = {pt.b.x, pt.b.y, pt.b.z}, e2 = {pt.c.x, pt.c.y, pt.c.z};
          if (k > 0) {
            const bvht_Triangle f = cx.faces[t];
            v0 = cx.vert[f.v1];
            e1 = vsub(cx.vert[f.v2], v0);
            e2 = vsub(cx.vert[f.v3], v0);
          }
          if (valid && hitTri(wr, v0, e1, e2, dist) && dist < nearest) {
            nearest = dist;
            o.tri = t;
          }
        }
      }
      if (lo == 0 && hi == 0) break;
      if (lo != 0) {
        const uint32_t tz = (uint32_t)__builtin_ctzll(lo);
        if (tz) {
          lo = (lo >> tz) | (hi << (64 - tz));
          hi >>= tz;
        }
      } else {
        const uint32_t tz = 64 + (uint32_t)__builtin_ctzll(hi);
        lo = hi >> (tz - 64);
        hi = 0;
      }
      lo ^= 1;
      if (sp == 0 || sp > 128) break;  // a trail deeper than 128 levels (unsupported, as in the reference)
      ref = s_stk[--sp];
    }
    o.t = nearest;
  }
  if (valid) img[(size_t)y * w + x] = shade(o, ray, cx.vert, cx.faces, light);
}

template <int MODE, bool AHEAD>
__global__ __launch_bounds__(64) void k_traceRays(const bvht_Ray *__restrict__ rays, uint32_t num, TraceCtx cx,
                                                     uint32_t root, bvht_vec3 light, float tMin,
                                                     const uint32_t *__restrict__ skip, bvht_Hit *__restrict__ hits,
                                                     bvht_CUDAPixel *__restrict__ img,
                                                     const uint32_t *__restrict__ order, uint32_t imgW) {
  __shared__ uint32_t s_stk[kStackCap * 64];
  uint32_t i;
  bool in;
  if (imgW) {  // the rays of an imgW-wide image, row-major: one 8x8 pixel tile per wave
    const uint32_t tilesX = (imgW + 7) / 8;
    // workgroups go to the 8 XCDs round-robin: runs of 4 consecutive tiles
    // (neighbouring rays, shared nodes) go to one XCD's L2, and the runs of
    // the 8 XCDs interleave, so every XCD keeps sweeping the same band of
    // the image (one stripe of the image per XCD balanced the work badly:
    // 5.0 against 3.8 ms at 1080p); the last partial group keeps its order
    const uint32_t b = blockIdx.x, g0 = b / 32 * 32;
    const uint32_t t = g0 + 32 <= gridDim.x ? g0 + (b % 8) * 4 + (b / 8) % 4 : b;
    const uint32_t x = (t % tilesX) * 8 + tileX(threadIdx.x), y = (t / tilesX) * 8 + tileY(threadIdx.x);
    in = x < imgW && (uint64_t)y * imgW + x < num;
    i = y * imgW + x;
  } else {
    const uint32_t slot = blockIdx.x * 64 + threadIdx.x;
    in = slot < num;
    i = order && in ? order[slot] : slot;
  }
  if (!in) i = 0;
  const bvht_Ray ray = rays[i];
  const bool still = ray.dir.x == 0.0f && ray.dir.y == 0.0f && ray.dir.z == 0.0f;
  const TraceOut o = walkAll<MODE, AHEAD>(in && !still, ray, cx, root, tMin, skip ? skip[i] : kNoHit, s_stk + threadIdx.x);
  if (!in) return;
  if (hits) hits[i] = bvht_Hit{o.tri, o.t};
  if (img) img[i] = shade(o, ray, cx.vert, cx.faces, light);
}

// Rays of one call traced by resident waves that refill their idle lanes
// from a shared counter (`next`, zero at launch), so a wave does not idle
// behind its longest walk.  A wave takes at least kRefillAt rays at a time, in
// slot order (neighbouring rays stay together); each ray's walk is the
// same visit sequence as in k_traceRays.  Every wave ends once the counter
// has passed `num` and its lanes are idle.
template <int MODE>
__global__ __launch_bounds__(64) void k_traceRaysDyn(const bvht_Ray *__restrict__ rays, uint32_t num, TraceCtx cx,
                                                        uint32_t root, bvht_vec3 light, float tMin,
                                                        const uint32_t *__restrict__ skip, bvht_Hit *__restrict__ hits,
                                                        bvht_CUDAPixel *__restrict__ img,
                                                        const uint32_t *__restrict__ order,
                                                        uint32_t *__restrict__ next) {
  __shared__ uint32_t s_stk[kStackCap * 64];
  uint32_t *stk = s_stk + threadIdx.x;
  const uint64_t lt = __lanemask_lt();
  const uint32_t top = rootRef(cx, root);  // the caller has checked the root
  bool active = false, drained = false;
  uint32_t i = 0, skipTri = kNoHit;
  WalkRay ray = {};
  Walk s;
  walkReset(s, 0);
  for (uint32_t it = 1;; ++it) {
    uint64_t act = __ballot(active);
    const uint32_t nIdle = 64 - (uint32_t)__popcll(act);
    if (!drained && (nIdle >= kRefillAt)) {  // wave-uniform
      uint32_t base = 0;
      if (threadIdx.x == 0) base = atomicAdd(next, nIdle);
      base = __shfl(base, 0, 64);
      if (base + nIdle >= num) drained = true;
      if (!active) {
        const uint32_t slot = base + (uint32_t)__popcll(~act & lt);
        if (slot < num) {
          i = order ? order[slot] : slot;
          const bvht_Ray r = rays[i];
          ray = walkRay(r);
          skipTri = skip ? skip[i] : kNoHit;
          walkReset(s, top);
          active = !(r.dir.x == 0.0f && r.dir.y == 0.0f && r.dir.z == 0.0f);
          if (!active) {  // nothing to walk: a miss
            if (hits) hits[i] = bvht_Hit{kNoHit, HUGE_VALF};
            if (img) img[i] = bvht_CUDAPixel{0, 0, 0};
          }
        }
      }
      act = __ballot(active);
    }
    if (act == 0) {
      if (drained) break;
      continue;
    }
    const bool was = active;
    walkStep<MODE, kAnyOct, false>(active, s, ray, cx, tMin, skipTri, stk);
    if ((it & (kCheckSteps - 1)) == 0 && s.count >= kMaxSteps) active = false;
    if (was && !active) {
      TraceOut o = {s.tri, s.nearest, (uint16_t)s.count};
      if (s.sp > (uint32_t)kStackCap) o = slowWalk<MODE>(ray, cx, top, tMin, skipTri, stk);
      if (hits) hits[i] = bvht_Hit{o.tri, o.t};
      if (img) {
        bvht_Ray r = {};
        r.pos = ray.pos;
        r.dir = ray.dir;
        img[i] = shade(o, r, cx.vert, cx.faces, light);
      }
    }
  }
}

// kRefitLeafBVHTris (CUDAKernels.cu:492-525): leaf boxes from the current
// vertices (triangle box -+ FLT_EPSILON); like the reference, the leaf's
// surfaceArea is not rewritten.
__global__ __launch_bounds__(256) void k_refitLeafTris(const uint32_t *__restrict__ ids, uint32_t num,
                                                       bvht_BVHNode *__restrict__ nodes,
                                                       const bvht_Triangle *__restrict__ faces,
                                                       const bvht_vec3 *__restrict__ vert, uint32_t numFaces) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i >= num) return;
  const uint32_t id = ids[i];
  const uint32_t f = nodes[id].left;
  if (f >= numFaces) return;
  const bvht_Triangle t = faces[f];
  nodes[id].bbox = triangleBox(vert[t.v1], vert[t.v2], vert[t.v3]);  // exact min/max: the reference's box
}

// Counter-based hash RNG (splitmix64 finaliser) -> uniform floats in [0, 1).
__device__ __forceinline__ uint64_t mix64(uint64_t x) {
  x += 0x9E3779B97F4A7C15ull;
  x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
  x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
  return x ^ (x >> 31);
}

// One cosine-weighted bounce: origin hit + 1e-4 * n (n faces the incoming
// ray), direction sampled around n (Malley's method), orthonormal basis of
// Duff et al. 2017.
__global__ __launch_bounds__(256) void k_bounce(const bvht_Ray *__restrict__ prim, const bvht_Hit *__restrict__ hits,
                                                uint32_t num, const bvht_vec3 *__restrict__ vert,
                                                const bvht_Triangle *__restrict__ faces, uint32_t seed,
                                                bvht_Ray *__restrict__ out, uint32_t *__restrict__ skip) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i >= num) return;
  const bvht_Ray r = prim[i];
  const bvht_Hit hh = hits[i];
  bvht_Ray o;
  if (hh.triId == kNoHit) {
    o.pos = r.pos;
    o.dir = {0.0f, 0.0f, 0.0f};
    o.invDir = {0.0f, 0.0f, 0.0f};
    o.sign[0] = o.sign[1] = o.sign[2] = 0;
    o._pad = 0;
    o.px = r.px;
    o.py = r.py;
    out[i] = o;
    skip[i] = kNoHit;
    return;
  }
  const bvht_Triangle tri = faces[hh.triId];
  const bvht_vec3 v1 = vert[tri.v1], v2 = vert[tri.v2], v3 = vert[tri.v3];
  bvht_vec3 n = vnormalize(vcross(vsub(v2, v1), vsub(v3, v1)));
  if (vdot(n, r.dir) > 0.0f) n = {-n.x, -n.y, -n.z};
  const bvht_vec3 hp = {r.pos.x + r.dir.x * hh.t, r.pos.y + r.dir.y * hh.t, r.pos.z + r.dir.z * hh.t};
  const bvht_vec3 org = {hp.x + 1e-4f * n.x, hp.y + 1e-4f * n.y, hp.z + 1e-4f * n.z};
  const uint64_t h = mix64(((uint64_t)seed << 32) ^ (uint64_t)i);
  const float u1 = (float)(h >> 40) * (1.0f / 16777216.0f);
  const float u2 = (float)((h >> 16) & 0xFFFFFF) * (1.0f / 16777216.0f);
  const float rr = sqrtf(u1), phi = 6.28318530717958647692f * u2;
  const float lx = rr * cosf(phi), ly = rr * sinf(phi), lz = sqrtf(fmaxf(0.0f, 1.0f - u1));
  const float sg = n.z >= 0.0f ? 1.0f : -1.0f;
  const float a = -1.0f / (sg + n.z), b = n.x * n.y * a;
  const bvht_vec3 t1 = {1.0f + sg * n.x * n.x * a, sg * b, -sg * n.x};
  const bvht_vec3 t2 = {b, sg + n.y * n.y * a, -n.y};
  bvht_vec3 d = {lx * t1.x + ly * t2.x + lz * n.x, lx * t1.y + ly * t2.y + lz * n.y, lx * t1.z + ly * t2.z + lz * n.z};
  d = vnormalize(d);
  setRay(o, org, d, r.px, r.py);
  out[i] = o;
  skip[i] = hh.triId;
}

__device__ __forceinline__ uint32_t spread9(uint32_t v) {  // 9 bits -> every third bit of 27
  v &= 511u;
  v = (v | (v << 16)) & 0x030000FFu;
  v = (v | (v << 8)) & 0x0300F00Fu;
  v = (v | (v << 4)) & 0x030C30C3u;
  v = (v | (v << 2)) & 0x09249249u;
  return v;
}
__device__ __forceinline__ uint32_t cell9(float x, float lo, float inv) {
  const float q = (x - lo) * inv;
  return q <= 0.0f ? 0u : (q >= 511.0f ? 511u : (uint32_t)q);
}

// Ordering key of a secondary ray: its direction cell (4 bins per axis over
// [-1, 1]) above the Morton cell of its origin in the root box (8 bits per
// axis).  Rays that start close together and head the same way walk similar
// nodes, so a wave of them diverges less (measured on the 4.24M-triangle scene
// at 1080p, one-ray-per-lane tracing: bounce trace 5.6 ->
// 4.9 ms with the sort included; octant-only direction cells 4.9, origin-major
// keys 5.2).  A ray with no direction gets the largest key.  Plus the digit
// histograms of the 4 sort passes.
__global__ __launch_bounds__(256) void k_rayKeys(const bvht_Ray *__restrict__ rays, uint32_t num,
                                                 const bvht_BVHNode *__restrict__ nodes, uint32_t root,
                                                 uint32_t *__restrict__ keys, uint32_t *__restrict__ hist) {
  __shared__ uint32_t s_hist[4][kSortRadix];
  for (int p = 0; p < 4; ++p) s_hist[p][threadIdx.x] = 0;
  __syncthreads();
  const bvht_AABB box = nodes[root].bbox;
  const float ix = 512.0f / fmaxf(box.minMax[1].x - box.minMax[0].x, 1e-30f);
  const float iy = 512.0f / fmaxf(box.minMax[1].y - box.minMax[0].y, 1e-30f);
  const float iz = 512.0f / fmaxf(box.minMax[1].z - box.minMax[0].z, 1e-30f);
  for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < num; i += gridDim.x * 256) {
    const bvht_Ray r = rays[i];
    uint32_t key = (1u << 30) - 1;
    if (!(r.dir.x == 0.0f && r.dir.y == 0.0f && r.dir.z == 0.0f)) {
      // direction: 4 bins per axis over [-1, 1]; origin: 8 bits per axis
      const uint32_t dx = min((uint32_t)fmaxf((r.dir.x + 1.0f) * 2.0f, 0.0f), 3u);
      const uint32_t dy = min((uint32_t)fmaxf((r.dir.y + 1.0f) * 2.0f, 0.0f), 3u);
      const uint32_t dz = min((uint32_t)fmaxf((r.dir.z + 1.0f) * 2.0f, 0.0f), 3u);
      const uint32_t dcell = (dx << 4) | (dy << 2) | dz;
      const uint32_t o = (spread9(cell9(r.pos.x, box.minMax[0].x, ix) >> 1) << 2) |
                         (spread9(cell9(r.pos.y, box.minMax[0].y, iy) >> 1) << 1) |
                         spread9(cell9(r.pos.z, box.minMax[0].z, iz) >> 1);
      key = (dcell << 24) | o;
    }
    keys[i] = key;
#pragma unroll
    for (int p = 0; p < 4; ++p) atomicAdd(&s_hist[p][(key >> (8 * p)) & (kSortRadix - 1)], 1u);
  }
  __syncthreads();
  for (int p = 0; p < 4; ++p) {
    const uint32_t c = s_hist[p][threadIdx.x];
    if (c) atomicAdd(hist + p * kSortRadix + threadIdx.x, c);
  }
}

// Packed copy of the tree and its triangles, rebuilt by every trace call (the
// tree may have changed since the last one); the buffer only grows.
struct TraceCache {
  NodeRec *recs = nullptr;
  size_t recCap = 0;
  uint32_t *bad = nullptr;
  uint32_t *next = nullptr;  // ray counter of k_traceRaysDyn
  // the ray buffer generateRays last filled, as a w x h image
  const void *imgRays = nullptr;
  uint32_t imgW = 0, imgH = 0;
  // ray ordering (bvht_traceRays): keys and indices x2, sort scratch
  bool orderRays = false;  // measured: with lane refills the sort costs more than it saves
  uint32_t orderCap = 0;
  uint32_t *okeys[2] = {nullptr, nullptr}, *ovals[2] = {nullptr, nullptr}, *oscratch = nullptr;
};
TraceCache &traceCache() {
  static TraceCache c;
  return c;
}

// Node indices of the traced tree must lie below 2 * numFaces - 1 (every
// binary BVH over the mesh fits); children past that are reported through
// tracerDoCudaSync and traced as empty leaves.
bool prepareTrace(const bvht_BVHNode *nodes, const bvht_MeshRaw &mesh, TraceCtx &cx, const char *what) {
  if (!mesh.faces || !mesh.vert || mesh.numFaces == 0) {
    setError("%s: empty mesh", what);
    return false;
  }
  const uint64_t bound = 2ull * mesh.numFaces - 1;
  if (bound >= kLeafRef) {
    setError("%s: %u faces exceed the 31-bit node range", what, mesh.numFaces);
    return false;
  }
  TraceCache &c = traceCache();
  if (c.recCap < bound) {
    devFree(c.recs);
    c.recs = nullptr;
    c.recCap = 0;
    if (!devAlloc(&c.recs, bound, "trace node records")) return false;
    c.recCap = bound;
  }
  if (!c.bad && !devAlloc(&c.bad, 1, "trace flag")) return false;
  if (!fillU32(c.bad, 0u, 1)) return false;
  k_packNodes<<<divUp(bound, 256), 256, 0, stream()>>>(nodes, (uint32_t)bound, mesh.faces, mesh.vert, mesh.numFaces,
                                                       c.recs, c.bad);
  if (!checkLaunch("k_packNodes")) return false;
  cx = TraceCtx{c.recs, nodes, mesh.faces, mesh.vert, (uint32_t)bound, mesh.numFaces};
  return true;
}

// Whether a launch of so many waves has its walks load ahead (visitInner): up
// to ten waves per CU.  Plain against ahead, us, 65k triangles / 0.9M: 1 wave per
// CU 180 / 658 against 145 / 536, 4 waves 195 / 650 against 166 / 582, 10 waves
// 202 / 728 against 179 / 712, 18 waves 193 / 746 against 177 / 860, 64 waves
// 232 / 1,667 against 274 / 2,484 (the L1 is busy then).  Switching to it after a
// number of steps, or where few of a wave's lanes are left, lost everywhere.
bool walksAhead(uint64_t waves) { return waves <= (uint64_t)numCUs() * 10; }

// Sorts the rays by k_rayKeys and returns the trace order (nullptr on
// failure, with the error recorded).
const uint32_t *rayOrder(const bvht_Ray *rays, uint32_t num, const bvht_BVHNode *nodes, uint32_t root) {
  TraceCache &c = traceCache();
  const SortPlan plan = makeSortPlan(num, 4, 30);
  if (c.orderCap < num) {
    for (int b = 0; b < 2; ++b) {
      devFree(c.okeys[b]);
      devFree(c.ovals[b]);
      c.okeys[b] = c.ovals[b] = nullptr;
    }
    devFree(c.oscratch);
    c.oscratch = nullptr;
    c.orderCap = 0;
    if (!devAlloc(&c.okeys[0], num, "ray keys") || !devAlloc(&c.okeys[1], num, "ray keys") ||
        !devAlloc(&c.ovals[0], num, "ray order") || !devAlloc(&c.ovals[1], num, "ray order") ||
        !devMalloc(reinterpret_cast<void **>(&c.oscratch), sortScratchBytes(makeSortPlan(num, 4, 30)), "ray sort"))
      return nullptr;
    c.orderCap = num;
  }
  if (!sortReset(plan, c.oscratch)) return nullptr;
  const uint32_t blocks = std::min<uint32_t>(divUp(num, 256 * 4), (uint32_t)numCUs() * 2);
  k_rayKeys<<<blocks, 256, 0, stream()>>>(rays, num, nodes, root, c.okeys[0], sortHist(plan, c.oscratch));
  if (!checkLaunch("k_rayKeys")) return nullptr;
  void *keys[2] = {c.okeys[0], c.okeys[1]};
  const int r = sortRun(plan, keys, c.ovals, true, false, c.oscratch);
  return r < 0 ? nullptr : c.ovals[r];
}

}  // namespace

}  // namespace bvht

using namespace bvht;

extern "C" {

void bvht_setRayOrdering(bool enable) { traceCache().orderRays = enable; }

bool allocateRays(bvht_Ray **rays, uint32_t num) { return devAlloc(rays, num, "allocateRays"); }
bool allocateImage(bvht_CUDAPixel **img, uint32_t w, uint32_t h) {
  return devAlloc(img, (size_t)w * h, "allocateImage");
}
void freeRays(bvht_Ray **rays) {
  if (rays && *rays) {
    devFree(*rays);
    *rays = nullptr;
  }
}
void freeImage(bvht_CUDAPixel *img) { devFree(img); }

void generateRays(bvht_Ray *rays, uint32_t w, uint32_t h, bvht_vec3 pos, bvht_vec3 lookAt, bvht_vec3 up, float fov) {
  if (!rays || w == 0 || h == 0) {
    setError("generateRays: no ray buffer or empty image");
    return;
  }
  // inverse(lookAtRH(pos, lookAt, up)) has columns s, u, -f, pos
  CamBasis c;
  double P[3] = {pos.x, pos.y, pos.z};
  double f[3] = {lookAt.x - P[0], lookAt.y - P[1], lookAt.z - P[2]};
  double fl = std::sqrt(f[0] * f[0] + f[1] * f[1] + f[2] * f[2]);
  for (double &v : f) v /= fl;
  double U[3] = {up.x, up.y, up.z};
  double s[3] = {f[1] * U[2] - f[2] * U[1], f[2] * U[0] - f[0] * U[2], f[0] * U[1] - f[1] * U[0]};
  double sl = std::sqrt(s[0] * s[0] + s[1] * s[1] + s[2] * s[2]);
  for (double &v : s) v /= sl;
  double u[3] = {s[1] * f[2] - s[2] * f[1], s[2] * f[0] - s[0] * f[2], s[0] * f[1] - s[1] * f[0]};
  for (int k = 0; k < 3; ++k) {
    c.s[k] = s[k];
    c.u[k] = u[k];
    c.f[k] = f[k];
  }
  c.pos[0] = pos.x;
  c.pos[1] = pos.y;
  c.pos[2] = pos.z;
  c.ratio = (float)w / (float)h;
  c.scale = (float)std::tan((0.5 * (double)fov) * (M_PI / 180.0));  // tan(radians(0.5 * fov))
  const uint32_t rows = std::max(1u, (1u << 31) / w);  // rows of a launch: its rays are counted in 32 bits
  for (uint64_t y0 = 0; y0 < h; y0 += rows) {
    const uint32_t n = std::min<uint32_t>(rows, h - (uint32_t)y0) * w;
    k_genRays<<<divUp(n, 256), 256, 0, stream()>>>(rays + (size_t)y0 * w, w, h, (uint32_t)y0, n, c);
    if (!checkLaunch("k_genRays")) return;
  }
  TraceCache &tc = traceCache();
  tc.imgRays = rays;
  tc.imgW = w;
  tc.imgH = h;
}

void tracerImage(bvht_Ray *rays, bvht_CUDAPixel *img, bvht_BVHNode *nodes, uint32_t rootNode, bvht_MeshRaw mesh,
                 bvht_vec3 light, uint32_t w, uint32_t h, bool bundle) {
  if (!rays || !img || !nodes) {
    setError("tracerImage: missing rays, image or nodes");
    return;
  }
  TraceCtx cx;
  if (!prepareTrace(nodes, mesh, cx, "tracerImage")) return;
  dim3 grid(divUp(w, 8), divUp(h, 8));
  if (bundle)
    k_traceImageBundle<<<grid, 64, 0, stream()>>>(rays, img, cx, rootNode, light, w, h);
  else if (walksAhead((uint64_t)grid.x * grid.y))
    k_traceImage<true><<<grid, 64, 0, stream()>>>(rays, img, cx, rootNode, light, w, h);
  else
    k_traceImage<false><<<grid, 64, 0, stream()>>>(rays, img, cx, rootNode, light, w, h);
  checkLaunch(bundle ? "k_traceImageBundle" : "k_traceImage");
}

void copyImageToHost(bvht_CUDAPixel *hostPixel, bvht_CUDAPixel *cudaImg, uint32_t w, uint32_t h) {
  if (check(hipMemcpyAsync(hostPixel, cudaImg, sizeof(bvht_CUDAPixel) * (size_t)w * h, hipMemcpyDeviceToHost, stream()),
            "copyImageToHost"))
    check(hipStreamSynchronize(stream()), "copyImageToHost sync");
}

void tracerDoCudaSync(void) {
  if (!check(hipStreamSynchronize(stream()), "tracerDoCudaSync")) return;
  uint32_t bad = 0;
  TraceCache &c = traceCache();
  if (c.bad && check(hipMemcpy(&bad, c.bad, 4, hipMemcpyDeviceToHost), "tracerDoCudaSync flag") && bad)
    setError("tracer: a child index lies outside the 2 * numFaces - 1 nodes of the mesh");
}

bool bvht_traceRays(const bvht_Ray *rays, uint32_t num, bvht_BVHNode *nodes, uint32_t rootNode, bvht_MeshRaw mesh,
                    bvht_vec3 light, int mode, float tMin, const uint32_t *skipTri, bvht_Hit *hits,
                    bvht_CUDAPixel *img) {
  if (!rays || !nodes || (!hits && !img)) {
    setError("bvht_traceRays: missing rays, nodes or outputs");
    return false;
  }
  if (num == 0) return true;
  TraceCtx cx;
  if (!prepareTrace(nodes, mesh, cx, "bvht_traceRays")) return false;
  if (rootNode >= cx.bound) {
    setError("bvht_traceRays: root %u outside the %u nodes of the mesh", rootNode, cx.bound);
    return false;
  }
  // secondary rays only: primary rays of an image are coherent in their own order
  const uint32_t *order = nullptr;  // (measured: ordering primary rays costs more than it saves)
  if (mode == 1 && traceCache().orderRays && !(order = rayOrder(rays, num, nodes, rootNode))) return false;
  if (mode == 0) {  // primary rays: one ray per lane, neighbouring rays in a wave
    // Rays that generateRays wrote as an image are traced in 8x8 pixel tiles
    // (tighter bundles than 64-pixel rows); the order never changes a ray's
    // result, only which rays share a wave.
    const TraceCache &c = traceCache();
    const bool image = rays == c.imgRays && (uint64_t)num == (uint64_t)c.imgW * c.imgH;
    const uint32_t blocks = image ? divUp(c.imgW, 8) * divUp(c.imgH, 8) : divUp(num, 64);
    const uint32_t width = image ? c.imgW : 0u;
    if (walksAhead(blocks))
      k_traceRays<0, true><<<blocks, 64, 0, stream()>>>(rays, num, cx, rootNode, light, tMin, skipTri, hits, img, order,
                                                        width);
    else
      k_traceRays<0, false><<<blocks, 64, 0, stream()>>>(rays, num, cx, rootNode, light, tMin, skipTri, hits, img, order,
                                                         width);
    return checkLaunch("k_traceRays");
  }
  // secondary rays: resident waves refill idle lanes (walk lengths vary widely)
  TraceCache &c = traceCache();
  if (!c.next && !devAlloc(&c.next, 1, "trace ray counter")) return false;
  if (!fillU32(c.next, 0u, 1)) return false;
  // resident waves only
  const uint32_t waves = std::min<uint32_t>(divUp(num, 64), (uint32_t)numCUs() * kTraceWavesPerCU);
  k_traceRaysDyn<1><<<waves, 64, 0, stream()>>>(rays, num, cx, rootNode, light, tMin, skipTri,
                                                hits, img, order, c.next);
  return checkLaunch("k_traceRaysDyn");
}

void refitDynamicTris(bvht_CUDAMemoryBVHPointer *bvh, bvht_MeshRaw mesh, uint32_t *nodesToUpdate, uint32_t numNodes,
                      uint32_t blockSize) {
  (void)blockSize;
  if (!bvh || !bvh->nodes || (numNodes && !nodesToUpdate) || !mesh.faces || !mesh.vert) {
    setError("refitDynamicTris: missing tree, mesh or node list");
    return;
  }
  if (numNodes == 0) return;
  k_refitLeafTris<<<divUp(numNodes, 256), 256, 0, stream()>>>(nodesToUpdate, numNodes, bvh->nodes, mesh.faces,
                                                              mesh.vert, mesh.numFaces);
  checkLaunch("k_refitLeafTris");
}

bool bvht_makeBounceRays(const bvht_Ray *primary, const bvht_Hit *hits, uint32_t num, bvht_MeshRaw mesh, uint32_t seed,
                         bvht_Ray *outRays, uint32_t *outSkipTri) {
  if (!primary || !hits || !outRays || !outSkipTri) {
    setError("bvht_makeBounceRays: missing buffers");
    return false;
  }
  if (num == 0) return true;
  k_bounce<<<divUp(num, 256), 256, 0, stream()>>>(primary, hits, num, mesh.vert, mesh.faces, seed, outRays, outSkipTri);
  return checkLaunch("k_bounce");
}

}  // extern "C"
