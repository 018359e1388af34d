// Bittner et al. 2013 parallel SAH optimizer for gfx950
// (reference: lib/builder/Bittner13CUDA.cu, lib/base/BVHPatch.hpp).
//
// One step (bn13_doAlgorithmStep):
//   k_cost      removal priority of every inner node, SA^3*2/((L+R)*min(L,R))
//               (Bittner13CUDA.cu:480-500), as a descending sort key;
//   onesweep    stable sort of (priority, node id) -- the processing order;
//   per chunk of K nodes (bn13_rmAndReinsChunk):
//     k_search  one 64-lane wave per node: remove the node (patch), then two
//               reinsertions, each found by a wave-parallel exact branch and
//               bound over the patched view (the reference's findNode1 keeps
//               a 4096-entry heap per thread in local memory); the patch
//               reserves its nodes (round 1);
//     k_commit / k_resolveTail  deterministic reservations: exactly the
//               patches a rank-ordered first-come locking applies (the
//               reference's kCheckConflicts, timing-dependent there);
//               (beside them, the paths above the insertion points are walked);
//     k_contain a winner whose insertion point lies in a subtree another
//               winner moves is dropped (two such patches would form a cycle;
//               the reference has no guard); the others write their topology,
//               all locks are released;
//     k_refit   two-phase targeted refit from the 3 changed nodes of every
//               winner (the kFixTree3_1 / kFixTree3_2 result).  Boxes are
//               exact min/max, so this equals the reference's full refit
//               (kFixTree1).
// The root never moves (reinsertion at the root is refused, :310).
#include "mlp.hpp"
#include "radix_sort.hpp"
#include "refit.hpp"
#include "wave.hpp"

#include <algorithm>
#include <cstring>
#include <new>
#include <type_traits>
#include <vector>

namespace bvht {

namespace {

constexpr uint32_t NONE = 0xFFFFFFFFu;
constexpr int kNNode = 10;  // BVHPatch.hpp:40
constexpr uint32_t P_GRAND_PARENT = 0, P_1ST_ROOT = 1, P_1ST_BEST = 2, P_NODE = 3, P_1ST_INSERT = 4, P_2ND_ROOT = 5,
                   P_2ND_BEST = 6, P_2ND_INSERT = 7, P_SIBLING = 8, P_PARENT = 9;  // BVHPatch.hpp:44-53
constexpr uint32_t kStackCap = 1024;  // per-search frontier (findNode1 heap: 4096)
constexpr uint32_t kAltSlots = 16;  // findNode2's array (CUDA_ALT_QUEUE_SIZE, Bittner13CUDA.hpp:28)

// Stats words (device)
enum { ST_CONFLICT = 0, ST_FAILED, ST_CONTAIN, ST_OVERFLOW, ST_APPLIED, ST_UNRESOLVED, ST_RUNAWAY, ST_SORTERR, ST_WORDS = 8 };

// Patch states and node locks.  A lock holds key(round, rank): the upper word
// is ~round, so later rounds and applied patches (round kRoundWin, upper word
// 0) compare smaller.
constexpr uint64_t kLockFree = ~0ull;
constexpr uint32_t kRoundWin = 0xFFFFFFFFu;
// The last three: the patch won its nodes.
enum : uint32_t { REC_NONE = 0, REC_PENDING = 1, REC_LOST = 2, REC_CONTAINED = 3, REC_WON = 4, REC_APPLIED = 5 };

__device__ __forceinline__ uint64_t lockKey(uint32_t round, uint32_t k) {
  return ((uint64_t)(0xFFFFFFFFu - round) << 32) | k;
}

struct PatchRec {
  uint32_t node[kNNode];
  uint32_t parent[kNNode];
  uint32_t left[kNNode];
  uint32_t right[kNNode];
  uint32_t isLeft[kNNode];
  uint32_t moved[2];  // reinserted subtree roots
  uint32_t best[2];   // insertion points
  uint32_t fix[3];    // refit starts: grandparent, unused1, unused2
  uint32_t ok;
};

// BVHPatch (ENABLE_AABB_PATH == 0) in LDS, manipulated by lane 0.
struct Patch {
  uint32_t vPatch[kNNode];
  uint32_t parent[kNNode], left[kNNode], right[kNNode];
  uint16_t isLeaf[kNNode], isLeft[kNNode];
  uint32_t path[4];
  float box[4][6];
};

struct NodeView {
  uint32_t parent, left, right, isLeaf, isLeft;
};

__device__ __forceinline__ NodeView globalView(const bvht_BVHNode *nodes, uint32_t n) {
  const uint4 w = reinterpret_cast<const uint4 *>(nodes + n)[1];  // maxY maxZ parent left
  const uint4 z = reinterpret_cast<const uint4 *>(nodes + n)[2];  // right flags level sa
  return NodeView{w.z, w.w, z.x, z.y & 0xFFFFu, z.y >> 16};
}

__device__ __forceinline__ void globalBox(const bvht_BVHNode *nodes, uint32_t n, float b[6]) {
  const uint4 a = reinterpret_cast<const uint4 *>(nodes + n)[0];
  const uint4 w = reinterpret_cast<const uint4 *>(nodes + n)[1];
  b[0] = __uint_as_float(a.x);
  b[1] = __uint_as_float(a.y);
  b[2] = __uint_as_float(a.z);
  b[3] = __uint_as_float(a.w);
  b[4] = __uint_as_float(w.x);
  b[5] = __uint_as_float(w.y);
}

// A node as it stands in the array.
struct FullNode {
  NodeView v;
  float b[6];
  float sa;
};
__device__ __forceinline__ FullNode globalNode(const bvht_BVHNode *nodes, uint32_t n) {
  const uint4 a = reinterpret_cast<const uint4 *>(nodes + n)[0];
  const uint4 w = reinterpret_cast<const uint4 *>(nodes + n)[1];
  const uint4 z = reinterpret_cast<const uint4 *>(nodes + n)[2];
  return FullNode{{w.z, w.w, z.x, z.y & 0xFFFFu, z.y >> 16},
                  {__uint_as_float(a.x), __uint_as_float(a.y), __uint_as_float(a.z), __uint_as_float(a.w),
                   __uint_as_float(w.x), __uint_as_float(w.y)},
                  __uint_as_float(z.w)};
}

__device__ __forceinline__ FullNode selectNode(bool c, const FullNode &x, const FullNode &y) {  // field by field: no scratch
  FullNode f;
  f.v = NodeView{c ? x.v.parent : y.v.parent, c ? x.v.left : y.v.left, c ? x.v.right : y.v.right,
                 c ? x.v.isLeaf : y.v.isLeaf, c ? x.v.isLeft : y.v.isLeft};
#pragma unroll
  for (int k = 0; k < 6; ++k) f.b[k] = c ? x.b[k] : y.b[k];
  f.sa = c ? x.sa : y.sa;
  return f;
}

__device__ __forceinline__ void storeBox(bvht_BVHNode *nd, const float b[6], float sa) {
  reinterpret_cast<float4 *>(nd)[0] = make_float4(b[0], b[1], b[2], b[3]);
  reinterpret_cast<float2 *>(nd)[2] = make_float2(b[4], b[5]);
  nd->surfaceArea = sa;
}

__device__ __forceinline__ bvht_AABB boxOf(const float b[6]) { return bvht_AABB{{{b[0], b[1], b[2]}, {b[3], b[4], b[5]}}}; }

__device__ __forceinline__ float sa6(const float b[6]) { return surfaceArea(b[0], b[1], b[2], b[3], b[4], b[5]); }
__device__ __forceinline__ void merge6(float a[6], const float b[6]) {
  a[0] = mergeMin(a[0], b[0]);
  a[1] = mergeMin(a[1], b[1]);
  a[2] = mergeMin(a[2], b[2]);
  a[3] = mergeMax(a[3], b[3]);
  a[4] = mergeMax(a[4], b[4]);
  a[5] = mergeMax(a[5], b[5]);
}

// ---- patch operations (lane 0) -------------------------------------------

__device__ void patchClear(Patch &P) {
  for (int i = 0; i < kNNode; ++i) P.vPatch[i] = NONE;
  for (int i = 0; i < 4; ++i) P.path[i] = NONE;
}
__device__ __forceinline__ uint32_t patchIndex(const Patch &P, uint32_t n) {
  for (int i = 0; i < kNNode; ++i)
    if (P.vPatch[i] == n) return i;
  return NONE;
}
// patchIndexSubset -- BVHPatch.hpp:134-142
__device__ __forceinline__ uint32_t patchIndexSubset(const Patch &P, uint32_t n) {
  if (P.vPatch[0] == n) return 0;
  if (P.vPatch[1] == NONE) return NONE;
  if (P.vPatch[1] == n) return 1;
  if (P.vPatch[2] == n) return 2;
  if (P.vPatch[3] == n) return 3;
  return NONE;
}
__device__ __forceinline__ NodeView patchGetSubset(const Patch &P, const bvht_BVHNode *nodes, uint32_t n) {
  uint32_t i = patchIndexSubset(P, n);
  if (i == NONE) return globalView(nodes, n);
  return NodeView{P.parent[i], P.left[i], P.right[i], P.isLeaf[i], P.isLeft[i]};
}
__device__ __forceinline__ void patchNode(Patch &P, uint32_t n, const NodeView &v, uint32_t slot) {
  P.vPatch[slot] = n;
  P.parent[slot] = v.parent;
  P.left[slot] = v.left;
  P.right[slot] = v.right;
  P.isLeaf[slot] = (uint16_t)v.isLeaf;
  P.isLeft[slot] = (uint16_t)v.isLeft;
}
__device__ __forceinline__ void movePatch(Patch &P, uint32_t from, uint32_t to) {
  P.vPatch[to] = P.vPatch[from];
  P.vPatch[from] = NONE;
  P.parent[to] = P.parent[from];
  P.left[to] = P.left[from];
  P.right[to] = P.right[from];
  P.isLeaf[to] = P.isLeaf[from];
  P.isLeft[to] = P.isLeft[from];
}
// getAABB -- BVHPatch.hpp:319-325: b, the node's box in the array, becomes
// the first cached path box that matches.
__device__ __forceinline__ void patchBox(const Patch &P, uint32_t n, float b[6]) {
  uint32_t at = NONE;
#pragma unroll
  for (int i = 3; i >= 0; --i) at = P.path[i] == n ? (uint32_t)i : at;
  if (at == NONE) return;
#pragma unroll
  for (int k = 0; k < 6; ++k) b[k] = P.box[at][k];
}

// removeNode -- Bittner13CUDA.cu:267-305 (a patch that cannot be built is
// dropped whole instead of being applied half done), with the path boxes of
// patchAABBFrom (BVHPatch.hpp:293-316) from the grandparent.  Every lane
// runs it on the same node (lane 0 writes the patch): the loads come in five
// dependent rounds, each with everything that is known by then.  ins
// receives the two subtrees to reinsert, larger area first.
__device__ __forceinline__ bool removeNode(Patch &P, const bvht_BVHNode *__restrict__ nodes, uint32_t node, uint32_t root,
                           uint32_t ins[2], FullNode insNode[2], uint32_t &parentIdx, uint32_t &gpOut) {
  const NodeView nv = globalView(nodes, node);
  if (nv.isLeaf || node == root) return false;
  if (nv.parent == root) return false;
  parentIdx = nv.parent;
  const NodeView pn = globalView(nodes, parentIdx);
  const FullNode l = globalNode(nodes, nv.left), r = globalNode(nodes, nv.right);
  const uint32_t sib = nv.isLeft == 0 ? pn.left : pn.right, gp = pn.parent;
  const FullNode sn = globalNode(nodes, sib);
  NodeView gv = globalView(nodes, gp);
  const bool gpTop = gp == root;
  const uint32_t uncle = pn.isLeft != 0 ? gv.right : gv.left, up = gv.parent;
  float box[6], s[6];
  globalBox(nodes, uncle, s);
  const NodeView uv = globalView(nodes, gpTop ? gp : up);
  const uint32_t aunt = gv.isLeft != 0 ? uv.right : uv.left;
  float t[6];
  globalBox(nodes, gpTop ? gp : aunt, t);
  // the grandparent's box holds the sibling in the parent's place
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    const float lo = pn.isLeft != 0 ? sn.b[k] : s[k], hi = pn.isLeft != 0 ? s[k] : sn.b[k];
    box[k] = k < 3 ? mergeMin(lo, hi) : mergeMax(lo, hi);
  }
  gpOut = gp;
  const bool first = l.sa > r.sa;
  ins[0] = first ? nv.left : nv.right;
  ins[1] = first ? nv.right : nv.left;
  insNode[0] = selectNode(first, l, r);
  insNode[1] = selectNode(first, r, l);
  if (threadIdx.x != 0) return true;
  patchNode(P, node, nv, P_NODE);
  patchNode(P, sib, sn.v, P_SIBLING);
  patchNode(P, parentIdx, pn, P_PARENT);
  if (pn.isLeft != 0)
    gv.left = sib;
  else
    gv.right = sib;
  patchNode(P, gp, gv, P_GRAND_PARENT);
  P.isLeft[P_SIBLING] = pn.isLeft != 0 ? 1 : 0;
  P.parent[P_SIBLING] = gp;
  P.path[0] = gp;
#pragma unroll
  for (int k = 0; k < 6; ++k) P.box[0][k] = box[k];
  if (!gpTop) {
    merge6(box, t);
    P.path[1] = up;
#pragma unroll
    for (int k = 0; k < 6; ++k) P.box[1][k] = box[k];
  }
  return true;
}

// Splice of reinsert -- Bittner13CUDA.cu:312-355 (the search is done before).
// nodeFull and bestFull are the two nodes as they stand in the array; lane 0.
__device__ __forceinline__ void spliceAt(Patch &P, const bvht_BVHNode *__restrict__ nodes, uint32_t node, const FullNode &nodeFull,
                         uint32_t unusedIdx, uint32_t bestIdx, const FullNode &bestFull, bool update) {
  uint32_t bp = patchIndex(P, bestIdx);
  uint32_t bs;
  if (bp == NONE) {
    bs = update ? P_1ST_BEST : P_2ND_BEST;
    patchNode(P, bestIdx, bestFull.v, bs);
  } else if (bp == P_GRAND_PARENT) {
    bs = P_GRAND_PARENT;
  } else {
    bs = update ? P_1ST_BEST : P_2ND_BEST;
    movePatch(P, bp, bs);
  }
  const uint32_t ns = update ? P_1ST_INSERT : P_2ND_INSERT;
  patchNode(P, node, nodeFull.v, ns);
  const uint32_t us = update ? P_NODE : P_PARENT;
  const uint32_t rootIdx = P.parent[bs];
  uint32_t rp = patchIndex(P, rootIdx);
  uint32_t rs = update ? P_1ST_ROOT : P_2ND_ROOT;
  if (rp == NONE)
    patchNode(P, rootIdx, globalView(nodes, rootIdx), rs);
  else
    movePatch(P, rp, rs);
  // a move may have relocated the best node's slot
  if (P.vPatch[bs] != bestIdx) bs = patchIndex(P, bestIdx);
  if (P.isLeft[bs] != 0) {
    P.left[rs] = unusedIdx;
    P.isLeft[us] = 1;
  } else {
    P.right[rs] = unusedIdx;
    P.isLeft[us] = 0;
  }
  P.parent[us] = rootIdx;
  P.left[us] = bestIdx;
  P.right[us] = node;
  P.parent[bs] = unusedIdx;
  P.isLeft[bs] = 1;
  P.parent[ns] = unusedIdx;
  P.isLeft[ns] = 0;
  if (!update) return;
  // patchAABBFrom (BVHPatch.hpp:293-316) from the spliced-in node (never the
  // root, which is not removed): its box, then its parent's
  NodeView cur = patchGetSubset(P, nodes, unusedIdx);
  float box[6], s[6];
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    box[k] = bestFull.b[k];
    s[k] = nodeFull.b[k];
  }
  patchBox(P, bestIdx, box);
  patchBox(P, node, s);
  merge6(box, s);
#pragma unroll
  for (int k = 0; k < 6; ++k) P.box[2][k] = box[k];
  P.path[2] = unusedIdx;
  const bool wasLeft = cur.isLeft != 0;
  const uint32_t up = cur.parent;
  cur = patchGetSubset(P, nodes, up);
  const uint32_t sib = wasLeft ? cur.right : cur.left;
  globalBox(nodes, sib, s);
  patchBox(P, sib, s);
  merge6(box, s);
#pragma unroll
  for (int k = 0; k < 6; ++k) P.box[3][k] = box[k];
  P.path[3] = up;
}

// The patched view of a search: the ids that its nodes are compared with,
// the same in every lane.  patchIndexSubset (BVHPatch.hpp:134-142) looks at
// slots 1..3 only once slot 1 is in use.
struct SearchIds {
  uint32_t slot[4], path[4];
};
__device__ __forceinline__ SearchIds searchIds(const Patch &P) {
  SearchIds q;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    q.slot[i] = __builtin_amdgcn_readfirstlane(P.vPatch[i]);
    q.path[i] = __builtin_amdgcn_readfirstlane(P.path[i]);
  }
  if (q.slot[1] == NONE) q.slot[2] = q.slot[3] = NONE;
  return q;
}
// The links and box of node n in the patched view, from the node in the
// array.  Few nodes are patched: most steps only compare the ids.
__device__ __forceinline__ void patched(const Patch &P, const SearchIds &q, uint32_t n, FullNode &f) {
  const bool hit = (n == q.slot[0]) | (n == q.slot[1]) | (n == q.slot[2]) | (n == q.slot[3]) | (n == q.path[0]) |
                   (n == q.path[1]) | (n == q.path[2]) | (n == q.path[3]);
  if (!hit) return;
  const uint32_t slot = n == q.slot[0] ? 0u : n == q.slot[1] ? 1u : n == q.slot[2] ? 2u : n == q.slot[3] ? 3u : NONE;
  const uint32_t path = n == q.path[0] ? 0u : n == q.path[1] ? 1u : n == q.path[2] ? 2u : n == q.path[3] ? 3u : NONE;
  if (slot != NONE)
    f.v = NodeView{P.parent[slot], P.left[slot], P.right[slot], P.isLeaf[slot], P.isLeft[slot]};
  if (path != NONE) {
#pragma unroll
    for (int k = 0; k < 6; ++k) f.b[k] = P.box[path][k];
  }
}

// ---- wave-parallel branch and bound (findNode1, Bittner13CUDA.cu:141-191) --
//
// Exact: an entry is expanded only while induced + SA(x) < best, which is a
// lower bound of the cost of every node below it, so the returned node is a
// cost minimiser of the patched view (ties: the first step that reaches the
// minimum, smallest node id inside it).  Frontier: LDS stack, up to 64
// entries evaluated per step.  Every step pops at least one entry and a tree
// pushes each node at most once, so a search of a tree ends within `maxSteps`
// = node count steps; a search still running then (a patched view that is
// not a tree) returns NONE and its patch is dropped.
//
// A search is a chain of about 33 steps (1M triangles) with two or three
// waves per CU, so the length of a step is what counts: one load of the
// popped nodes, and little else.  The ids of the patched view sit in scalar
// registers, minima run through DPP, the workgroup is one wave whose LDS
// operations stay in order (no waits between steps).  k_search per chunk:
// 92 -> 49 us (65,536 triangles 75 -> 40, 4.2M 107 -> 58).
__device__ __forceinline__ uint32_t waveSearch(const Patch &P, const bvht_BVHNode *__restrict__ nodes,
                                               const FullNode &x, uint32_t root, uint2 *s_stk, uint32_t cap,
                                               uint32_t maxSteps, uint32_t *overflow, float &bestCost) {
  const uint32_t lane = threadIdx.x;
  const float sa = x.sa;
  const SearchIds q = searchIds(P);
  if (lane == 0) s_stk[0] = make_uint2(root, __float_as_uint(0.0f));
  memoryChanged();
  float best = HUGE_VALF;
  uint32_t bestNode = 0;
  const uint64_t lt = __lanemask_lt();
  uint32_t top = 1;
  for (uint32_t step = 0; top > 0; ++step) {
    if (step >= maxSteps) return NONE;  // uniform: step and top are wave-uniform
    const uint32_t m = top < 64 ? top : 64;
    const uint2 e = s_stk[lane < m ? top - 1 - lane : 0u];
    memoryChanged();
    const uint32_t newTop = top - m, node = e.x;
    const float ind = __uint_as_float(e.y);
    const bool eval = lane < m && (ind + sa) < best;
    float total = HUGE_VALF, newInd = 0.0f;
    FullNode f;
    if (eval) {
      f = globalNode(nodes, node);
      patched(P, q, node, f);
      newInd = -1.0f * sa6(f.b);
      merge6(f.b, x.b);
      total = ind + sa6(f.b);
      newInd += total;
    }
    const float mt = waveMinUniform(total == total ? total : HUGE_VALF);
    if (mt < best) {
      uint64_t tied = __ballot(eval && total == mt);
      bestNode = NONE;
      while (tied) {  // smallest node id among the tied lanes (mostly one)
        bestNode = min(bestNode, (uint32_t)__builtin_amdgcn_readlane(node, __builtin_ctzll(tied)));
        tied &= tied - 1;
      }
      best = mt;
    }
    const bool push = eval && f.v.isLeaf == 0 && (newInd + sa) < best;
    const uint64_t pm = __ballot(push);
    const uint32_t pos = newTop + 2u * (uint32_t)__popcll(pm & lt);
    const uint32_t cnt = 2u * (uint32_t)__popcll(pm);
    if (push && pos + 1 < cap) {
      s_stk[pos] = make_uint2(f.v.left, __float_as_uint(newInd));
      s_stk[pos + 1] = make_uint2(f.v.right, __float_as_uint(newInd));
    }
    uint32_t nt = __builtin_amdgcn_readfirstlane(newTop + cnt);
    if (nt > cap) {
      if (lane == 0) atomicAdd(overflow, 1u);
      nt = cap & ~1u;
    }
    top = nt;
    memoryChanged();
  }
  bestCost = best;
  return bestNode;
}

// ---- findNode2 (altFindNode), Bittner13CUDA.cu:194-264 ---------------------
//
// The reference's approximate search, exactly: a best-first search over a
// fixed array of 16 (node, induced cost) slots, held here by lanes 0..15 of
// the wave (one slot per lane).  Each iteration pops the slot of minimum
// cost; an expanded node's left child takes that slot and its right child
// the slot of maximum cost found by the previous scan (an empty slot holds
// HUGE_VALF, so it is the maximum while one is free; once the array is full
// the costliest entry is overwritten).  Both scans keep the first slot of
// their extreme (the reference's strict < and > loops); the maximum scan
// starts from 0 and keeps the previous slot when no cost is above 0.  NaN
// costs never compare, so they are mapped out of both scans.  One entry is
// popped per iteration and a tree pushes each node at most once, so a
// search of a tree ends within `maxIters` = node count iterations; a longer
// one (a patched view that is not a tree) returns NONE.
__device__ __forceinline__ uint32_t altSearch(const Patch &P, const bvht_BVHNode *__restrict__ nodes, const FullNode &x, uint32_t root,
                              uint32_t maxIters, float &bestCost) {
  const uint32_t lane = threadIdx.x;
  const bool slot = lane < kAltSlots;
  const float sa = x.sa;
  const SearchIds q = searchIds(P);
  uint32_t slotNode = root;
  float slotCost = lane == 0 ? 0.0f : HUGE_VALF;
  uint32_t minIdx = 0, maxIdx = 1;
  float best = HUGE_VALF, lMin = 0.0f;
  uint32_t bestNode = 0;
  for (uint32_t it = 0; lMin < HUGE_VALF; ++it) {  // lMin, minIdx, maxIdx are wave-uniform
    if (it >= maxIters) return NONE;
    const uint32_t cur = (uint32_t)__shfl((int)slotNode, (int)minIdx, 64);
    const float curCost = __shfl(slotCost, (int)minIdx, 64);
    if (lane == minIdx) slotCost = HUGE_VALF;
    if ((curCost + sa) >= best) break;
    FullNode f = globalNode(nodes, cur);
    patched(P, q, cur, f);
    const NodeView nv = f.v;
    float newInd = -1.0f * sa6(f.b);
    merge6(f.b, x.b);
    const float total = curCost + sa6(f.b);
    if (total < best) {
      best = total;
      bestNode = cur;
    }
    newInd += total;
    if ((newInd + sa) < best && nv.isLeaf == 0) {
      if (lane == minIdx) {
        slotNode = nv.left;
        slotCost = newInd;
      }
      if (lane == maxIdx) {  // written second: takes the slot if both are one
        slotNode = nv.right;
        slotCost = newInd;
      }
    }
    const bool num = slot && !__builtin_isnan(slotCost);
    const float cMin = num ? slotCost : HUGE_VALF, cMax = num ? slotCost : 0.0f;
    lMin = waveMin(cMin);
    const float lMax = waveMax(cMax);
    if (lMin < HUGE_VALF) minIdx = (uint32_t)__builtin_ctzll(__ballot(num && cMin == lMin));
    if (lMax > 0.0f) maxIdx = (uint32_t)__builtin_ctzll(__ballot(num && cMax == lMax));
  }
  bestCost = best;
  return bestNode;
}

// Destination of SAH-gain records (feat == nullptr: not recording).
struct RecordSink {
  const float *feat;  // features by inner-list position
  float *recFeat;     // [recMax][12]
  float *recGain;     // [recMax]
  uint32_t *recCount;
  uint32_t recMax;
};

// Gain of a patch in unit-cost SAH relative to the root: the areas of the
// two removed nodes plus the shrink of the two path boxes above the removal
// point, minus the two insertion costs the searches found.
__device__ float patchGain(const Patch &P, const bvht_BVHNode *nodes, uint32_t node, uint32_t parent, uint32_t root,
                           float c1, float c2) {
  float shrink = 0.0f;
  for (int i = 0; i < 2; ++i)
    if (P.path[i] != NONE) shrink += nodes[P.path[i]].surfaceArea - sa6(P.box[i]);
  const float g = nodes[node].surfaceArea + nodes[parent].surfaceArea + shrink - c1 - c2;
  const float sr = nodes[root].surfaceArea;
  return sr > 0.0f ? g / sr : 0.0f;
}

// PROBE: evaluate the patches of the nodes at inner-list positions
// order[blockIdx.x] and record their gains; nothing is reserved or applied.
template <bool PROBE>
__global__ __launch_bounds__(64) void k_search(const bvht_BVHNode *__restrict__ nodes, uint32_t root, uint32_t N,
                                               const uint32_t *__restrict__ order, const uint32_t *__restrict__ inner,
                                               uint32_t numInner, uint32_t chunk, uint32_t numChunks, uint32_t K,
                                               uint32_t offsetAccess, uint32_t alt, PatchRec *__restrict__ recs,
                                               uint64_t *locks, uint32_t *__restrict__ marks,
                                               uint32_t *__restrict__ stats, RecordSink sink,
                                               const uint32_t *__restrict__ sortErr) {
  __shared__ Patch P;
  __shared__ uint2 s_stk[kStackCap];  // node, induced cost
  const uint32_t k = blockIdx.x, lane = threadIdx.x;
  if (sortErr && k == 0 && lane == 0 && *sortErr) atomicAdd(stats + ST_SORTERR, 1u);
  PatchRec *rec = recs + k;
  const uint32_t pos = PROBE ? order[k] : order[offsetAccess ? k * numChunks + chunk : chunk * K + k];
  if (pos >= numInner) {  // block-uniform: altSort's entries past the selected, or a bad probe list
    if (!PROBE && lane == 0) rec->ok = REC_NONE;
    return;
  }
  const uint32_t nodeIdx = inner[pos];
  if (!PROBE && lane < 2) {  // takes the marks of the chunk before away (any mark is old here)
    const uint32_t was = rec->moved[lane];
    if (rec->ok >= REC_CONTAINED && was < N) marks[was] = NONE;
  }
  // The workgroup is one wave: everything below but the patch itself (lane 0
  // edits it) is computed by every lane alike.
  float cost[2] = {0.0f, 0.0f};
  uint32_t ins[2], best[2], parentIdx = 0, gp = 0;
  FullNode insNode[2];
  if (lane == 0) patchClear(P);
  memoryChanged();
  bool ok = removeNode(P, nodes, nodeIdx, root, ins, insNode, parentIdx, gp);
  const auto reinsert = [&](auto which) {
    constexpr int W = decltype(which)::value;
    memoryChanged();
    const uint32_t b =
        alt ? altSearch(P, nodes, insNode[W], root, N, cost[W])
            : waveSearch(P, nodes, insNode[W], root, s_stk, kStackCap, N, stats + ST_OVERFLOW, cost[W]);
    if (b == root || b == NONE) {
      if (b == NONE && lane == 0) atomicAdd(stats + ST_RUNAWAY, 1u);
      return false;
    }
    best[W] = b;
    if (lane == 0) spliceAt(P, nodes, ins[W], insNode[W], W == 0 ? nodeIdx : parentIdx, b, globalNode(nodes, b), W == 0);
    memoryChanged();
    return true;
  };
  ok = ok && reinsert(std::integral_constant<int, 0>()) && reinsert(std::integral_constant<int, 1>());
  if (!ok) {
    if (!PROBE && lane == 0) {
      rec->ok = REC_NONE;
      atomicAdd(stats + ST_FAILED, 1u);
    }
    return;
  }
  if (sink.feat && lane == 0) {
    const uint32_t slot = atomicAdd(sink.recCount, 1u);
    if (slot < sink.recMax) {
      for (int f = 0; f < kFeat; ++f) sink.recFeat[(size_t)slot * kFeat + f] = sink.feat[(size_t)pos * kFeat + f];
      sink.recGain[slot] = patchGain(P, nodes, nodeIdx, parentIdx, root, cost[0], cost[1]);
    }
  }
  if (PROBE) return;
  if (lane < (uint32_t)kNNode) {
    const uint32_t n = P.vPatch[lane];
    rec->node[lane] = n;
    rec->parent[lane] = P.parent[lane];
    rec->left[lane] = P.left[lane];
    rec->right[lane] = P.right[lane];
    rec->isLeft[lane] = P.isLeft[lane];
    // round-1 reservation of the deterministic conflict resolution
    if (n != NONE) atomicMin(reinterpret_cast<unsigned long long *>(locks + n), (unsigned long long)lockKey(1, k));
  }
  if (lane == 0) {
    rec->moved[0] = ins[0];
    rec->moved[1] = ins[1];
    rec->best[0] = best[0];
    rec->best[1] = best[1];
    rec->fix[0] = gp;
    rec->fix[1] = nodeIdx;
    rec->fix[2] = parentIdx;
    rec->ok = REC_PENDING;
  }
}

// ---- conflict resolution: deterministic reservations ---------------------
//
// kCheckConflicts (Bittner13CUDA.cu:567-609) lets patch k lock its nodes
// first come, first served; serialised in rank order this is the greedy rule
// "k is applied iff no node of k belongs to an applied patch of lower rank".
// That rule is computed here exactly and independently of timing: in round r
// every undecided patch reserves its nodes with atomicMin(key(r, k)); a patch
// that holds every reservation is applied (its nodes get key(WIN, k), smaller
// than any reservation), a patch that meets an applied patch's node loses,
// the rest retry in round r + 1.  The undecided patch of lowest rank always
// decides, so a round never leaves the set unchanged.
__device__ __forceinline__ void reserve(const PatchRec *r, uint32_t k, uint32_t round, uint64_t *locks) {
  const uint64_t key = lockKey(round, k);
  for (int i = 0; i < kNNode; ++i) {
    const uint32_t n = r->node[i];
    if (n != NONE) atomicMin(reinterpret_cast<unsigned long long *>(locks + n), (unsigned long long)key);
  }
}

// Returns REC_WON, REC_LOST or REC_PENDING and records a decision.
__device__ uint32_t decide(PatchRec *r, uint32_t k, uint32_t round, uint64_t *locks, uint32_t *marks,
                           uint32_t *skipped, uint32_t *stats) {
  const uint64_t mine = lockKey(round, k);
  bool holdAll = true, lost = false;
  for (int i = 0; i < kNNode; ++i) {
    const uint32_t n = r->node[i];
    if (n == NONE) continue;
    const uint64_t v = __hip_atomic_load(locks + n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if ((v >> 32) == 0) lost = true;  // node of an applied patch
    if (v != mine) holdAll = false;
  }
  if (lost) {
    r->ok = REC_LOST;
    skipped[k] += 1;
    atomicAdd(stats + ST_CONFLICT, 1u);
    return REC_LOST;
  }
  if (!holdAll) return REC_PENDING;
  const uint64_t win = lockKey(kRoundWin, k);
  for (int i = 0; i < kNNode; ++i) {
    const uint32_t n = r->node[i];
    if (n != NONE) atomicMin(reinterpret_cast<unsigned long long *>(locks + n), (unsigned long long)win);
  }
  r->ok = REC_WON;
  marks[r->moved[0]] = k;  // moved roots are patch nodes: one applied patch each
  marks[r->moved[1]] = k;
  return REC_WON;
}

// Sixteen lanes per patch for the kernels that touch every node of a patch:
// lane j holds node j, so the patch's node ids, their locks and the writes
// are one round trip each instead of ten in a row (a chunk has a few hundred
// to a few thousand patches, far too few to hide a chain of loads per
// thread).  1M triangles, 627 patches: round 1 13.3 -> 4.8 us,
// writing the topology 11.1 -> 4.8 us (a launch of its own then).
constexpr uint32_t kPatchLanes = 16, kPatchBlock = 256, kPatchesPerBlock = kPatchBlock / kPatchLanes;

// An undecided patch after round 1, as k_resolveTail reads it: its nodes, its
// rank and the roots it moves, one word per lane.
constexpr uint32_t kOpenWords = kPatchLanes, kOpenRank = 12, kOpenMoved = 13;
static_assert(kNNode <= (int)kOpenRank, "a patch's nodes lie below its rank");
constexpr uint32_t kCommitRounds = 3;  // k_commit launches of a chunk at most, an open list's length each

// Round 1 over every patch (the reservations were made by k_search), or, LATER,
// a further round over the entries that the one before left.  With `again` the
// undecided patches reserve their nodes for the next round at once: a patch
// that meets such a reservation in place of its own is only decided a round
// later.
template <bool LATER>
__global__ __launch_bounds__(kPatchBlock) void k_commit(PatchRec *__restrict__ recs, uint32_t K, uint64_t *locks,
                                                        uint32_t *__restrict__ marks, uint32_t *__restrict__ skipped,
                                                        uint32_t *__restrict__ stats, const uint32_t *__restrict__ openIn,
                                                        const uint32_t *__restrict__ numIn,
                                                        uint32_t *__restrict__ open, uint32_t *__restrict__ numPending,
                                                        uint32_t round, bool again) {
  const uint32_t at = blockIdx.x * kPatchesPerBlock + threadIdx.x / kPatchLanes, j = threadIdx.x % kPatchLanes;
  const bool in = at < (LATER ? *numIn : K);  // every lane stays for the ballots
  const bool mover = j == kOpenMoved || j == kOpenMoved + 1;
  uint32_t k = at, n, moved;
  bool undecided = in;
  if (LATER) {
    const uint32_t word = in ? openIn[(size_t)at * kOpenWords + j] : NONE;
    k = __shfl(word, kOpenRank, kPatchLanes);
    n = j < (uint32_t)kNNode ? word : NONE;
    moved = word;
  } else {
    PatchRec *r = recs + (in ? at : 0);
    n = in && j < (uint32_t)kNNode ? r->node[j] : NONE;
    moved = in && mover ? r->moved[j - kOpenMoved] : NONE;
    undecided = in && r->ok == REC_PENDING;
  }
  const bool use = undecided && n != NONE;
  const uint64_t mine = lockKey(round, k);
  const uint64_t v = use ? __hip_atomic_load(locks + n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : mine;
  const uint32_t group = threadIdx.x & 63u & ~(kPatchLanes - 1);
  const bool lost = ((__ballot((v >> 32) == 0) >> group) & 0xFFFFu) != 0;  // node of an applied patch
  const bool holdAll = ((__ballot(v != mine) >> group) & 0xFFFFu) == 0;
  if (!undecided) return;
  if (!lost && holdAll) {
    if (use)
      atomicMin(reinterpret_cast<unsigned long long *>(locks + n), (unsigned long long)lockKey(kRoundWin, k));
    if (mover) marks[moved] = k;  // moved roots are patch nodes: one applied patch each
    if (j == 0) recs[k].ok = REC_WON;
  } else if (lost) {
    if (j == 0) {
      recs[k].ok = REC_LOST;
      skipped[k] += 1;
      atomicAdd(stats + ST_CONFLICT, 1u);
    }
  } else {
    if (again && use)
      atomicMin(reinterpret_cast<unsigned long long *>(locks + n), (unsigned long long)lockKey(round + 1, k));
    uint32_t slot = 0;
    if (j == 0) slot = atomicAdd(numPending, 1u);
    slot = __shfl(slot, 0, kPatchLanes);
    open[(size_t)slot * kOpenWords + j] = j == kOpenRank ? k : mover ? moved : n;
  }
}

// The further rounds over the (few) undecided patches, in one workgroup.  At most
// `num + 1` rounds are needed; patches still undecided after that bound
// (never, unless memory ordering is broken) are dropped and counted.
//
// Up to kTailCap patches (two per thread, every node a table slot of its own
// at worst), the rounds run in LDS and registers: the nodes of the undecided
// patches go into an LDS hash table holding, per node, whether a winner took
// it (round 1's from its global lock, read once) and the lowest rank
// reserving it this round, and each thread keeps its patches' table slots in
// registers.  The table is built by 16 lanes a patch, from the entries that
// k_commit left (a line each): a node a lane, every load and every first
// probe of a thread in flight together (one thread a patch, node by node from
// its record: 22.0 against 13.3 us before the first round with 772 patches,
// 7.2 against 4.7 with 50).  A round is two barriers: a patch with a taken node loses, the
// others reserve their nodes; a patch that holds them all wins and takes
// them.  (A losing patch no longer reserves, which decides its neighbours no
// later.)  The reservations of a round are cleared by their own patches
// while the next round uses the other of two arrays; the two lie where the
// slots and the node ids were while the table was built.  Nothing
// is written to memory before the last round: a barrier would wait for it.
// Measured per chunk: 627 patches of 1M triangles 14.1 -> 10.4 us; 1,638
// patches of 65,536 triangles (10% per step) 48 -> 24 us in the mean; the
// first chunks of a step, whose more than 1,024 undecided patches took the
// global rounds before, 168 -> 47 us.
// Global locks keep their round-1 values (k_contain releases them all).
constexpr int kTailBlock = 1024;
constexpr uint32_t kTailSlotsLog = 14, kTailSlots = 1u << kTailSlotsLog;
constexpr uint32_t kTailCap = kTailSlots / kNNode;  // patches: the table never overflows
constexpr uint32_t kTailPer = 2;                    // patches per thread
constexpr uint32_t kTailEmpty = 0xFFFFFFFFu;
static_assert(kTailCap <= kTailPer * kTailBlock, "every patch of the LDS rounds has a thread");

__device__ __forceinline__ uint32_t tailHash(uint32_t n) { return (n * 0x9E3779B1u) >> (32 - kTailSlotsLog); }

// Slot of node n, inserted if absent, after a first probe at h found another
// node (the table never overflows).
__device__ __forceinline__ uint32_t tailInsert(uint32_t *keys, uint32_t n, uint32_t h) {
  for (uint32_t probe = 1; probe < kTailSlots; ++probe) {
    h = (h + 1) & (kTailSlots - 1);
    const uint32_t prev = atomicCAS(keys + h, kTailEmpty, n);
    if (prev == kTailEmpty || prev == n) return h;
  }
  return 0;  // unreachable
}

// The nodes from patch k's insertion point w up to the root, for k_contain:
// their number and then themselves, and of a path that does not fit, from its
// last stored node on, each node's parent at the node's place in `above` (a
// word per node; walks that share nodes write the same).  Without `paths`
// (allocateMemory), the parents from the insertion point on.
constexpr uint32_t kPathWords = 128;
__device__ void walkPath(const PatchRec *__restrict__ recs, uint32_t k, uint32_t w,
                         const bvht_BVHNode *__restrict__ nodes, uint32_t root, uint32_t N,
                         uint32_t *__restrict__ paths, uint32_t *above) {
  const uint32_t ok = recs[k].ok;  // another workgroup may be deciding it: undecided patches walk too
  if (ok == REC_NONE || ok == REC_LOST) return;
  uint32_t x = recs[k].best[w], len = 0;
  if (paths) {
    uint32_t *path = paths + (2 * (size_t)k + w) * kPathWords;
    while (true) {  // a store a level and no other: the wait for the next parent then leaves it in flight
      const uint32_t p = nodes[x].parent;
      path[++len] = x;
      if (x == root || len == kPathWords - 1) break;
      x = p;
    }
    path[0] = len;
  }
  for (; x != root && len < N; ++len) {
    const uint32_t p = nodes[x].parent;
    above[x] = p;
    x = p < N ? p : root;
  }
}

constexpr uint32_t kTailGroups = kTailBlock / kPatchLanes;                          // patches loaded at a time
constexpr uint32_t kTailTrips = (kTailCap + kTailGroups - 1) / kTailGroups;

__global__ __launch_bounds__(kTailBlock) void k_resolveTail(PatchRec *__restrict__ recs, uint64_t *locks,
                                                           uint32_t *__restrict__ marks,
                                                           uint32_t *__restrict__ skipped, uint32_t *__restrict__ stats,
                                                           const uint32_t *__restrict__ open, uint32_t *listA,
                                                           uint32_t *listB, const uint32_t *__restrict__ numPending,
                                                           uint32_t K, const bvht_BVHNode *__restrict__ nodes,
                                                           uint32_t root, uint32_t N, uint32_t *__restrict__ paths,
                                                           uint32_t *above, uint32_t walkers, uint32_t firstRound) {
  // lowest reserving rank per slot, rounds alternate; at first [1] holds the
  // node ids and [0] the patches' slots (16 bits each)
  __shared__ __align__(16) uint32_t s_min[2][kTailSlots];
  __shared__ __align__(16) uint32_t s_taken4[kTailSlots / 4];  // bytes: taken by a winner
  __shared__ uint32_t s_open[3];                 // undecided patches after a round (rounds rotate)
  __shared__ uint32_t s_cnt;
  uint8_t *s_taken = reinterpret_cast<uint8_t *>(s_taken4);
  uint16_t *s_slot = reinterpret_cast<uint16_t *>(&s_min[0][0]);
  if (blockIdx.x > 0) {  // workgroup-uniform
    const uint32_t at = (blockIdx.x - 1) * walkers + threadIdx.x;
    if (threadIdx.x < walkers && at / 2 < K) walkPath(recs, at / 2, at & 1, nodes, root, N, paths, above);
    return;
  }
  static_assert(kTailSlots <= 65535 && kTailCap * kNNode * 2 <= sizeof(s_min[0]), "the slots fit s_min[0]");
  uint32_t num = *numPending;
  if (num == 0) return;
  const uint32_t maxRound = num + firstRound;
  if (num <= kTailCap) {
    // 16 lanes per patch: a lane loads one node of each of up to kTailTrips
    // patches and its lock, all in flight together, and inserts it
    const uint32_t j = threadIdx.x % kPatchLanes, first = threadIdx.x / kPatchLanes;
    uint32_t n[kTailTrips], prev[kTailTrips], takenMask = 0;
#pragma unroll
    for (uint32_t i = 0; i < kTailTrips; ++i) {
      n[i] = NONE;
      if (i * kTailGroups < num && i * kTailGroups + first < num && j < (uint32_t)kNNode)
        n[i] = open[(i * kTailGroups + first) * kOpenWords + j];
    }
    uint4 rank[kTailPer];  // the patches of the rounds: rank and moved roots
#pragma unroll
    for (uint32_t q = 0; q < kTailPer; ++q) {
      const uint32_t at = threadIdx.x + q * kTailBlock;
      rank[q] = make_uint4(NONE, NONE, NONE, NONE);
      if (at < num) rank[q] = *reinterpret_cast<const uint4 *>(open + at * kOpenWords + kOpenRank);
    }
    uint4 *ids4 = reinterpret_cast<uint4 *>(&s_min[1][0]), *taken16 = reinterpret_cast<uint4 *>(s_taken4);
    for (uint32_t i = threadIdx.x; i < kTailSlots / 4; i += kTailBlock)
      ids4[i] = make_uint4(kTailEmpty, kTailEmpty, kTailEmpty, kTailEmpty);
    for (uint32_t i = threadIdx.x; i < kTailSlots / 16; i += kTailBlock) taken16[i] = make_uint4(0, 0, 0, 0);
    if (threadIdx.x < 3) s_open[threadIdx.x] = 0;
#pragma unroll
    for (uint32_t i = 0; i < kTailTrips; ++i) {  // a lock's upper half: 0 once a winner of round 1 holds it
      prev[i] = 1;
      if (i * kTailGroups < num && n[i] != NONE)
        prev[i] = loadRelaxedAgent(reinterpret_cast<const uint32_t *>(locks + n[i]) + 1);
    }
#pragma unroll
    for (uint32_t i = 0; i < kTailTrips; ++i) takenMask |= prev[i] == 0 ? 1u << i : 0u;
    static_assert(kTailTrips <= 32, "a bit per trip");
    __syncthreads();
#pragma unroll
    for (uint32_t i = 0; i < kTailTrips; ++i)  // the first probes go out together
      if (i * kTailGroups < num && n[i] != NONE) prev[i] = atomicCAS(&s_min[1][tailHash(n[i])], kTailEmpty, n[i]);
#pragma unroll
    for (uint32_t i = 0; i < kTailTrips; ++i) {
      if (i * kTailGroups >= num) continue;
      uint32_t h = 0xFFFFu;
      if (n[i] != NONE) {
        h = tailHash(n[i]);
        if (prev[i] != kTailEmpty && prev[i] != n[i]) h = tailInsert(&s_min[1][0], n[i], h);
        if (takenMask >> i & 1) s_taken[h] = 1;
      }
      n[i] = h;
      const uint32_t at = i * kTailGroups + first;
      if (at < num && j < (uint32_t)kNNode) s_slot[at * kNNode + j] = (uint16_t)h;
    }
    __syncthreads();
    uint32_t k[kTailPer], node[kTailPer][kNNode];  // slots
#pragma unroll
    for (uint32_t q = 0; q < kTailPer; ++q) {
      const uint32_t at = threadIdx.x + q * kTailBlock;
      k[q] = rank[q].x;
#pragma unroll
      for (int c = 0; c < kNNode; ++c) {
        const uint32_t h = at < num ? s_slot[at * kNNode + c] : 0xFFFFu;
        node[q][c] = h == 0xFFFFu ? NONE : h;
      }
    }
    __syncthreads();
    // the ids and the slots give way to reservations
#pragma unroll
    for (uint32_t i = 0; i < kTailTrips; ++i)
      if (i * kTailGroups < num && n[i] != 0xFFFFu) s_min[1][n[i]] = kTailEmpty;
    uint4 *min4 = reinterpret_cast<uint4 *>(&s_min[0][0]);
    for (uint32_t i = threadIdx.x; i < kTailSlots / 4; i += kTailBlock)
      min4[i] = make_uint4(kTailEmpty, kTailEmpty, kTailEmpty, kTailEmpty);
    uint32_t state[kTailPer];
    bool reserved[kTailPer];  // in the round before
#pragma unroll
    for (uint32_t q = 0; q < kTailPer; ++q) {
      state[q] = k[q] == NONE ? REC_NONE : REC_PENDING;
      reserved[q] = false;
    }
    __syncthreads();
    for (uint32_t round = 0; round <= maxRound; ++round) {
      uint32_t *cur = s_min[round & 1], *old = s_min[(round & 1) ^ 1];
      bool now[kTailPer];
#pragma unroll
      for (uint32_t q = 0; q < kTailPer; ++q) {
        now[q] = false;
        if (state[q] != REC_PENDING) continue;
        bool lost = false;
#pragma unroll
        for (int j = 0; j < kNNode; ++j) lost |= node[q][j] != NONE && s_taken[node[q][j]] != 0;
        if (lost) {
          state[q] = REC_LOST;
          continue;
        }
        now[q] = true;
#pragma unroll
        for (int j = 0; j < kNNode; ++j)
          if (node[q][j] != NONE) atomicMin(cur + node[q][j], k[q]);
      }
      if (threadIdx.x == 0) s_open[(round + 1) % 3] = 0;
      __syncthreads();
      uint32_t open = 0;
#pragma unroll
      for (uint32_t q = 0; q < kTailPer; ++q) {
        if (reserved[q]) {
#pragma unroll
          for (int j = 0; j < kNNode; ++j)
            if (node[q][j] != NONE) old[node[q][j]] = kTailEmpty;
        }
        reserved[q] = now[q];
        if (!now[q]) continue;
        bool holdAll = true;
#pragma unroll
        for (int j = 0; j < kNNode; ++j) holdAll &= node[q][j] == NONE || cur[node[q][j]] == k[q];
        if (!holdAll) {
          ++open;
          continue;
        }
        state[q] = REC_WON;
#pragma unroll
        for (int j = 0; j < kNNode; ++j)
          if (node[q][j] != NONE) s_taken[node[q][j]] = 1;
      }
      if (open) atomicAdd(&s_open[round % 3], open);
      __syncthreads();
      if (s_open[round % 3] == 0) break;  // workgroup-uniform
    }
    uint32_t conflicts = 0, unresolved = 0;
#pragma unroll
    for (uint32_t q = 0; q < kTailPer; ++q) {
      if (state[q] == REC_NONE) continue;
      PatchRec *r = recs + k[q];
      if (state[q] == REC_WON) {
        r->ok = REC_WON;
        marks[rank[q].y] = k[q];  // moved roots are patch nodes: one applied patch each
        marks[rank[q].z] = k[q];
        continue;
      }
      unresolved += state[q] == REC_PENDING;
      ++conflicts;
      r->ok = REC_LOST;
      skipped[k[q]] += 1;
    }
    if (conflicts) atomicAdd(stats + ST_CONFLICT, conflicts);
    if (unresolved) atomicAdd(stats + ST_UNRESOLVED, unresolved);
    return;
  }
  // more undecided patches than the LDS table takes: the rounds on the
  // global locks
  for (uint32_t i = threadIdx.x; i < num; i += kTailBlock) listA[i] = open[i * kOpenWords + kOpenRank];
  __syncthreads();
  uint32_t *cur = listA, *nxt = listB;
  for (uint32_t round = firstRound; num > 0 && round <= maxRound; ++round) {
    for (uint32_t i = threadIdx.x; i < num; i += kTailBlock) reserve(recs + cur[i], cur[i], round, locks);
    if (threadIdx.x == 0) s_cnt = 0;
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < num; i += kTailBlock) {
      const uint32_t k = cur[i];
      if (decide(recs + k, k, round, locks, marks, skipped, stats) == REC_PENDING) nxt[atomicAdd(&s_cnt, 1u)] = k;
    }
    __syncthreads();
    num = s_cnt;
    uint32_t *t = cur;
    cur = nxt;
    nxt = t;
    __syncthreads();
  }
  for (uint32_t i = threadIdx.x; i < num; i += kTailBlock) {
    PatchRec *r = recs + cur[i];
    r->ok = REC_LOST;
    skipped[cur[i]] += 1;
    atomicAdd(stats + ST_CONFLICT, 1u);
    atomicAdd(stats + ST_UNRESOLVED, 1u);
  }
}

// Whether node x is a root that a winner other than k moves.  A mark of an
// earlier chunk may be left at x (k_search takes most of them away): it counts
// only if its patch is a winner now and moves x.
__device__ __forceinline__ bool movedByOther(uint32_t m, uint32_t x, uint32_t k, uint32_t K, const PatchRec *recs) {
  if (m == NONE || m == k || m >= K) return false;
  const PatchRec *r = recs + m;
  return r->ok >= REC_CONTAINED && (r->moved[0] == x || r->moved[1] == x);
}

// Writes patch k's node j (the caller's lane): a winner's topology, released
// locks, the refit's starts.  Returns whether lane 0 of a patch dropped it (2)
// or applied it (1).
__device__ __forceinline__ uint32_t applyPatch(PatchRec *r, uint32_t k, uint32_t j, uint32_t ok, bool bad,
                                           bvht_BVHNode *__restrict__ nodes, uint64_t *__restrict__ locks,
                                           uint32_t *__restrict__ fixStarts, uint32_t *__restrict__ skipped) {
  const uint32_t jn = j < (uint32_t)kNNode ? j : 0u;
  const uint32_t n = r->node[jn], parent = r->parent[jn], left = r->left[jn], right = r->right[jn],
                 isLeft = r->isLeft[jn], fix = r->fix[j < 3 ? j : 0u];
  const bool win = ok == REC_WON && !bad;
  if (j < 3) fixStarts[3 * k + j] = win ? fix : NONE;
  if (ok == REC_NONE) return 0;
  if (j < (uint32_t)kNNode && n != NONE) {
    locks[n] = kLockFree;
    if (win) {  // MiniPatch::applyOne -- BVHPatch.hpp:72-80
      nodes[n].parent = parent;
      nodes[n].left = left;
      nodes[n].right = right;
      nodes[n].isLeft = (uint16_t)isLeft;
    }
  }
  if (j != 0 || ok != REC_WON) return 0;
  r->ok = win ? REC_APPLIED : REC_CONTAINED;
  if (!win) skipped[k] += 1;
  return win ? 1 : 2;
}

// Drops a winner whose insertion point lies below a node another winner moves;
// the other winners write their topology, and every patch releases its locks.
// The paths above the insertion points were walked while the conflicts were
// resolved (the tree does not change until here), so a patch's marks are one
// round trip for its 16 lanes, and nothing is read that another patch writes.
// Per chunk, with a launch for the walks and one to apply before: 627 patches
// of 1M triangles 12.3 + 4.8 -> 5.1 us, 2,648 of 4.2M 13.7 + 9.9 -> 7.8 us.
// A path longer than kPathWords goes on in `above`, the parents before this
// launch wrote any: two lanes of the patch, a round trip per level.  (One
// workgroup for a whole chunk with such a path: 7,503 patches below a path of
// 150 nodes 16.3 ms a step of four chunks, now 2.83.)
__global__ __launch_bounds__(kPatchBlock) void k_contain(PatchRec *__restrict__ recs, uint32_t K,
                                                         bvht_BVHNode *__restrict__ nodes, uint32_t root, uint32_t N,
                                                         const uint32_t *__restrict__ marks,
                                                         const uint32_t *__restrict__ paths,
                                                         const uint32_t *__restrict__ above, uint64_t *__restrict__ locks,
                                                         uint32_t *__restrict__ fixStarts,
                                                         uint32_t *__restrict__ skipped,
                                                         uint32_t *__restrict__ numPending,
                                                         uint32_t *__restrict__ stats) {
  const uint32_t j = threadIdx.x % kPatchLanes, group = threadIdx.x & 63u & ~(kPatchLanes - 1);
  if (blockIdx.x == 0 && threadIdx.x < kCommitRounds) numPending[threadIdx.x] = 0;
  const uint32_t k = blockIdx.x * kPatchesPerBlock + threadIdx.x / kPatchLanes;
  const bool in = k < K;  // every lane stays for the exchanges
  PatchRec *r = recs + (in ? k : 0);
  const uint32_t *path = paths + 2 * (size_t)(in ? k : 0) * kPathWords;
  constexpr uint32_t ROWS = 2;  // of 16 words, of each path, loaded before anything is known
  uint32_t x[2][ROWS];
#pragma unroll
  for (int w = 0; w < 2; ++w)
#pragma unroll
    for (uint32_t i = 0; i < ROWS; ++i) x[w][i] = paths ? path[w * kPathWords + i * kPatchLanes + j] : 0u;
  const uint32_t ok = in ? r->ok : (uint32_t)REC_NONE;  // read before lane 0 of the patch writes it
  bool bad = false;
  if (__ballot(ok == REC_WON) != 0) {
    uint32_t len[2];
#pragma unroll
    for (int w = 0; w < 2; ++w) {
      len[w] = __shfl(x[w][0], 0, kPatchLanes);
      if (ok != REC_WON) len[w] = 0;
    }
    uint32_t m[2][ROWS];
#pragma unroll
    for (int w = 0; w < 2; ++w)
#pragma unroll
      for (uint32_t i = 0; i < ROWS; ++i) {
        const uint32_t at = i * kPatchLanes + j;
        m[w][i] = at > 0 && at <= len[w] ? marks[x[w][i]] : NONE;
      }
    bool marked = false;
#pragma unroll
    for (int w = 0; w < 2; ++w)
#pragma unroll
      for (uint32_t i = 0; i < ROWS; ++i) {
        if (m[w][i] == k || m[w][i] >= K) m[w][i] = NONE;
        marked |= m[w][i] != NONE;
      }
    if (marked) {  // their patches' records, all in flight together
      uint32_t state[2][ROWS], root0[2][ROWS], root1[2][ROWS];
#pragma unroll
      for (int w = 0; w < 2; ++w)
#pragma unroll
        for (uint32_t i = 0; i < ROWS; ++i) {
          const PatchRec *o = recs + (m[w][i] != NONE ? m[w][i] : k);
          state[w][i] = o->ok;
          root0[w][i] = o->moved[0];
          root1[w][i] = o->moved[1];
        }
#pragma unroll
      for (int w = 0; w < 2; ++w)
#pragma unroll
        for (uint32_t i = 0; i < ROWS; ++i)
          bad |= m[w][i] != NONE && state[w][i] >= REC_CONTAINED && (root0[w][i] == x[w][i] || root1[w][i] == x[w][i]);
    }
    for (int w = 0; w < 2; ++w)
      for (uint32_t at = ROWS * kPatchLanes + j; at <= len[w]; at += kPatchLanes) {
        const uint32_t y = path[w * kPathWords + at];
        bad |= movedByOther(marks[y], y, k, K, recs);
      }
    if (j < 2 && (paths ? (j == 0 ? len[0] : len[1]) == kPathWords - 1 : ok == REC_WON)) {
      uint32_t y = paths ? path[j * kPathWords + kPathWords - 1] : r->best[j];
      if (!paths) bad |= movedByOther(marks[y], y, k, K, recs);  // a stored node's mark is done
      for (uint32_t steps = 0; steps < N && y != root; ++steps) {
        y = above[y];
        if (y >= N) break;  // not a tree
        const uint32_t m = marks[y];
        bad |= movedByOther(m, y, k, K, recs);
      }
    }
  }
  bad = ((__ballot(bad) >> group) & 0xFFFFu) != 0;
  const uint32_t did = in ? applyPatch(r, k, j, ok, bad, nodes, locks, fixStarts, skipped) : 0u;
  // counted per workgroup: one word takes an atomic every few ns
  const int applied = __syncthreads_count(did == 1), dropped = __syncthreads_count(did == 2);
  if (threadIdx.x == 0 && applied) atomicAdd(stats + ST_APPLIED, (uint32_t)applied);
  if (threadIdx.x == 0 && dropped) atomicAdd(stats + ST_CONTAIN, (uint32_t)dropped);
}

// ---- targeted refit (kFixTree3, Bittner13CUDA.cu:407-467) ------------------
//
// Two launches over the start nodes.  k_refitCount marks the paths from the
// starts to the root: a node's word holds how many of its children are on a
// path (bits 0-1), whether it is a start (bit 2), whether it is one more than
// once (bit 3) and, when both children are, the slot their walks meet in
// (bits 4..31: the index of the start whose walk arrived second and ended
// there, so no counter hands them out).  k_refitApply then walks up with the
// box of the node below in registers:
//   one child on a path   the other child's box does not change during the
//                         refit: a plain load that goes out beside the
//                         parent's links and word, one round trip per level;
//   both on a path        each walk exchanges its box into the slot.  The
//                         exchanged words carry the box and a tag, so one
//                         round trip tells a walk whether it came second and
//                         hands it the other's box; the first one ends.  The
//                         words of two walks may interleave: the walk that
//                         came second on word 0 goes on, and waits for the
//                         words that it reached first (the other walk has
//                         already issued them).
// Nothing else passes between walks, so boxes and words are written with
// plain stores.  Before, every level was an arrival count, coherent loads of
// both children's boxes and coherent stores that were waited for, three round
// trips past the L2: 1,881 starts in 1M triangles 59 -> 23 us, 100,000
// leaves of them 57 -> 37 us.
//
// Lists of more starts than there are slots take none: bit 4 of a word then
// says that a walk has arrived (kRefitArrived).
constexpr uint32_t kRefitChildren = 3u, kRefitStart = 4u, kRefitDup = 8u, kRefitSlotShift = 4u, kRefitArrived = 16u;
constexpr uint32_t kRefitBlock = 256;

template <bool SLOTS>
__global__ __launch_bounds__(kRefitBlock) void k_refitCount(const uint32_t *__restrict__ starts, uint32_t num,
                                                            uint32_t walks, const bvht_BVHNode *__restrict__ nodes, uint32_t N,
                                                            uint32_t *__restrict__ cnt) {
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t i = (blockIdx.x * (kRefitBlock / 64) + threadIdx.x / 64) * walks + lane;
  if (lane >= walks || i >= num) return;
  uint32_t node = starts[i];
  if (node >= N) return;
  uint32_t p = loadRelaxedAgent(&nodes[node].parent);  // issued beside the count: one round trip per level
  uint32_t old = atomicOr(cnt + node, kRefitStart);
  if (old & kRefitStart) atomicOr(cnt + node, kRefitDup);
  for (uint32_t steps = 0; steps < N && old == 0; ++steps) {  // the first to touch a node walks on
    if (p == node || p >= N) return;
    node = p;
    p = loadRelaxedAgent(&nodes[node].parent);
    old = atomicAdd(cnt + node, 1u);
    if (SLOTS && (old & kRefitChildren) == 1) atomicOr(cnt + node, i << kRefitSlotShift);
  }
}

// Words of a slot: three halfwords of payload below a 16-bit tag (0: empty,
// 1: from the left child, 2: from the right).
template <int WORDS>
__device__ __forceinline__ void packSlot(const uint32_t (&v)[6 + 2 * (WORDS - 4) / 2], uint32_t tag,
                                         uint64_t (&w)[WORDS]) {
  constexpr int VALS = 6 + 2 * (WORDS - 4) / 2;
#pragma unroll
  for (int i = 0; i < WORDS; ++i) {
    uint64_t x = (uint64_t)tag << 48;
#pragma unroll
    for (int h = 0; h < 3; ++h) {
      const int at = 3 * i + h;
      if (at < 2 * VALS) x |= (uint64_t)((v[at / 2] >> (16 * (at & 1))) & 0xFFFFu) << (16 * h);
    }
    w[i] = x;
  }
}
template <int WORDS>
__device__ __forceinline__ void unpackSlot(const uint64_t (&w)[WORDS], uint32_t (&v)[6 + 2 * (WORDS - 4) / 2]) {
  constexpr int VALS = 6 + 2 * (WORDS - 4) / 2;
#pragma unroll
  for (int k = 0; k < VALS; ++k) v[k] = 0;
#pragma unroll
  for (int at = 0; at < 2 * VALS; ++at)
    v[at / 2] |= (uint32_t)((w[at / 3] >> (16 * (at % 3))) & 0xFFFFu) << (16 * (at & 1));
}

// With FEAT (the learned priority's subtree features) the walk also keeps
// leaf counts and subtree areas exact: the nodes it recomputes are exactly
// those whose subtree changed.
//
// A walk is bound by latency, so a level is one round trip for every lane of
// the wave, whichever way its two children are: the next level's links, the
// other child's box (unused where it comes from the slot) and the exchanges
// go out together, and a node's own stores follow them (vector memory
// operations retire in order, so stores ahead of the loads would be waited
// for).  `walks` of a wave's lanes walk (the low ones): with few walks, fewer
// lanes a wave means fewer scattered accesses an instruction.
//
// NEAR: neighbours in the list are neighbours in the tree (a list of leaves
// in their order), and most walks meet inside their workgroup.  They do so
// in LDS first: the one that comes first leaves its box under the node's id
// and stops, the second takes it and goes on.  When every walk of the
// workgroup has stopped, those whose box nobody took meet other workgroups'
// walks in the slots.  Exchanging everything in the slots instead is bound
// by the exchanges themselves (100,000 leaves of 1M: 52 us against 37).
//
// By ids (NEAR lists of more than a quarter of the leaves): every node is a
// candidate, in the order of the ids, and the marked starts walk, so
// neighbours meet in LDS in whatever order the list names them.
//
// ARRIVE (by ids, more starts than slots): walks of two workgroups meet by
// arrival: the box is stored past the L2, then the arrival marked; the second
// loads the first one's box.  Three round trips, and no limit on the starts;
// workgroups of 1,024 leave fewer such meetings (4M leaves 530 -> 388 us).
//
// All of 20,000 leaves in order / mixed 38 / 40 us (40 / 63 with an arrival at
// every level, 101 / 199 in pieces of a quarter of the leaves), 100,000 48 / 56
// (59 / 113, 113 / 246), 1M 174 / 242 (316 / 472, 225 / 988), 4M 647 / 904
// (1,437 / 2,188, 623 / 4,114).
enum { kRefitScattered = 0, kRefitNear = 1, kRefitIds = 2, kRefitArrive = 3 };
constexpr uint32_t kSlotListMin = 1u << 17;
constexpr uint32_t refitBlock(int list) { return list == kRefitArrive ? 1024 : kRefitBlock; }
template <bool FEAT, int LIST>
__global__ __launch_bounds__(refitBlock(LIST)) void k_refitApply(const uint32_t *__restrict__ starts, uint32_t num,
                                                            uint32_t walks, bvht_BVHNode *__restrict__ nodes,
                                                            uint32_t N, uint32_t *__restrict__ cnt, uint64_t *slots,
                                                            uint32_t *__restrict__ leafCnt,
                                                            float *__restrict__ subSA, uint32_t *__restrict__ stats) {
  constexpr bool NEAR = LIST != kRefitScattered, IDS = LIST >= kRefitIds, ARRIVE = LIST == kRefitArrive;
  static_assert(!(FEAT && NEAR), "a near list keeps no features");
  constexpr int WORDS = FEAT ? 6 : 4;
  constexpr uint32_t BLOCK = refitBlock(LIST), kNearSlots = 2 * BLOCK;  // LDS table, at most half full
  __shared__ unsigned long long s_key[NEAR ? kNearSlots : 1];  // node id << 32 | thread that left its box
  __shared__ uint32_t s_box[6][NEAR ? BLOCK : 1];
  __shared__ uint32_t s_taken[NEAR ? BLOCK : 1];
  const uint32_t tid = threadIdx.x, lane = tid & 63u;
  const auto clearTable = [&] {
    for (uint32_t k = tid; k < kNearSlots; k += BLOCK) s_key[k] = ~0ull;
    s_taken[tid] = 0;
    __syncthreads();
  };
  if (NEAR && !IDS) clearTable();  // ahead of the loads: a barrier behind them would wait for them
  const uint32_t i = (blockIdx.x * (BLOCK / 64) + tid / 64) * walks + lane;
  uint32_t child = IDS ? i : lane < walks && i < num ? starts[i] : NONE;
  bool go = child < N;
  if (!go) child = 0;
  uint32_t c = cnt[child];
  // a walk from below recomputes the node (or has: its word is cleared)
  go = go && c != 0 && (c & kRefitChildren) == 0;
  if (IDS && __syncthreads_or(go) == 0) return;
  if (IDS) clearTable();
  NodeView nv = globalView(nodes, child);
  // one occurrence of a start named more than once goes on
  if (!IDS && go && (c & kRefitDup)) go = atomicExch(cnt + child, 0u) != 0;
  if (!NEAR && !go) return;
  uint32_t node = nv.parent;
  bool end = node == child || node >= N;
  NodeView nvUp = globalView(nodes, end ? child : node);
  uint32_t cUp = cnt[end ? child : node];
  // the node below (`child`): its box and area
  float b[6], sa, sub = 0.0f;
  uint32_t leaves = 0;
  if (nv.isLeaf == 0) {
    float r[6];
    globalBox(nodes, nv.left, b);
    globalBox(nodes, nv.right, r);
    merge6(b, r);
    sa = sa6(b);
    if (FEAT) {
      leaves = leafCnt[nv.left] + leafCnt[nv.right];
      sub = subSA[nv.left] + subSA[nv.right] + sa;
    }
  } else {  // a leaf start (dynamic refit) is not recomputed: it keeps its values
    globalBox(nodes, child, b);
    sa = nodes[child].surfaceArea;
    if (FEAT) {
      leaves = leafCnt[child];
      sub = subSA[child];
    }
  }
  // complete before the loop, whose waits then only count the loop's own loads
  asm volatile("" : "+v"(b[0]), "+v"(b[1]), "+v"(b[2]), "+v"(b[3]), "+v"(b[4]), "+v"(b[5]), "+v"(sa), "+v"(leaves),
                    "+v"(sub), "+v"(nvUp.parent), "+v"(nvUp.left), "+v"(nvUp.right), "+v"(cUp));
#pragma unroll
  for (int phase = NEAR ? 0 : 1; phase < 2; ++phase) {
    bool wait = false;  // stopped with its box left in LDS
    for (uint32_t steps = 0; go && steps <= N; ++steps) {
      nv = nvUp;
      c = cUp;
      const bool left = nv.left == child;
      const uint32_t sib = left ? nv.right : nv.left, p = nv.parent;
      const bool top = p == node || p >= N;
      const bool meet = !end && (c & kRefitChildren) != 1;
      const uint32_t at = c >> kRefitSlotShift;
      float s[6];
      uint32_t sibLeaves = 0;
      float sibSub = 0.0f;
      if (!end) {
        // the next level's links and word (both fixed until this walk arrives)
        nvUp = globalView(nodes, top ? node : p);
        cUp = cnt[top ? node : p];
        globalBox(nodes, sib, s);
        if (FEAT) {
          sibLeaves = leafCnt[sib];
          sibSub = subSA[sib];
        }
      }
      uint64_t w[WORDS];
      uint64_t *slot = slots + (size_t)at * WORDS;
      const bool bad = !ARRIVE && meet && at >= num;  // not a tree (more than two children on a path)
      const bool arrive = ARRIVE && phase == 1 && meet;
      if (!ARRIVE && phase == 1 && meet && !bad) {
        uint32_t v[6 + 2 * (WORDS - 4) / 2];
#pragma unroll
        for (int k = 0; k < 6; ++k) v[k] = __float_as_uint(b[k]);
        if constexpr (FEAT) {
          v[6] = leaves;
          v[7] = __float_as_uint(sub);
        }
        packSlot<WORDS>(v, left ? 1u : 2u, w);
#pragma unroll
        for (int k = 0; k < WORDS; ++k)
          w[k] = __hip_atomic_exchange(slot + k, w[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      if (arrive)
        storeBoxAgent(nodes + child, boxOf(b), sa);
      else
        storeBox(nodes + child, b, sa);
      if (FEAT) {
        leafCnt[child] = leaves;
        subSA[child] = sub;
      }
      cnt[child] = 0;
      if (end || bad) break;
      if (arrive) {
        waitVectorMemory();  // the box is out before the arrival
        const uint32_t seen = __hip_atomic_fetch_or(cnt + node, kRefitArrived, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if ((seen & kRefitArrived) == 0) break;  // first: the other walk goes on
        const bvht_AABB o = loadBoxAgent(nodes + sib);
        s[0] = o.minMax[0].x;
        s[1] = o.minMax[0].y;
        s[2] = o.minMax[0].z;
        s[3] = o.minMax[1].x;
        s[4] = o.minMax[1].y;
        s[5] = o.minMax[1].z;
      }
      if (phase == 0 && meet) {
#pragma unroll
        for (int k = 0; k < 6; ++k)
          __hip_atomic_store(&s_box[k][tid], __float_as_uint(b[k]), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        memoryChanged();  // the box before its key (LDS operations of a wave stay in order)
        uint32_t h = (node * 0x9E3779B1u) >> 16 & (kNearSlots - 1);
        uint32_t from = NONE;
        for (uint32_t probe = 0; probe < kNearSlots; ++probe) {
          const unsigned long long old = atomicCAS(s_key + h, ~0ull, ((unsigned long long)node << 32) | tid);
          if (old == ~0ull) break;
          if ((uint32_t)(old >> 32) == node) {
            from = (uint32_t)old;
            break;
          }
          h = (h + 1) & (kNearSlots - 1);
        }
        if (from == NONE) {
          wait = true;
          break;
        }
        s_taken[from] = 1;
        memoryChanged();
#pragma unroll
        for (int k = 0; k < 6; ++k)
          s[k] = __uint_as_float(
              __hip_atomic_load(&s_box[k][from], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
      }
      if (!ARRIVE && phase == 1 && meet) {
        if ((w[0] >> 48) == 0) break;  // first: the other walk goes on
        const uint32_t other = left ? 2u : 1u;
        for (uint32_t spins = 0;; ++spins) {
          bool missing = false;
#pragma unroll
          for (int k = 1; k < WORDS; ++k) missing |= (w[k] >> 48) != other;
          if (!missing) break;
          if (spins > (1u << 22)) {  // never, unless memory is broken: counted, the box is then wrong
            atomicAdd(stats + ST_UNRESOLVED, 1u);
            break;
          }
#pragma unroll
          for (int k = 1; k < WORDS; ++k)
            if ((w[k] >> 48) != other)
              w[k] = __hip_atomic_load(slot + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        uint32_t v[6 + 2 * (WORDS - 4) / 2];
        unpackSlot<WORDS>(w, v);
#pragma unroll
        for (int k = 0; k < 6; ++k) s[k] = __uint_as_float(v[k]);
        if constexpr (FEAT) {
          sibLeaves = v[6];
          sibSub = __uint_as_float(v[7]);
        }
#pragma unroll
        for (int k = 0; k < WORDS; ++k)
          __hip_atomic_store(slot + k, (uint64_t)0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      // the left child's box merges the right one's
#pragma unroll
      for (int k = 0; k < 6; ++k) {
        const float l = left ? b[k] : s[k], r = left ? s[k] : b[k];
        b[k] = k < 3 ? mergeMin(l, r) : mergeMax(l, r);
      }
      sa = sa6(b);
      if (FEAT) {
        leaves += sibLeaves;
        sub = sub + sibSub + sa;  // commutes: left + right + own
      }
      child = node;
      node = p;
      end = top;
    }
    if (phase == 0) {  // whose box nobody took goes on from the same node
      __syncthreads();
      go = wait && s_taken[tid] == 0;
      nvUp = nv;
      cUp = c;
    }
  }
}

// kCalcCost -- Bittner13CUDA.cu:480-500, written as an ascending sort key
// (~bits of the non-negative cost: descending cost, ties by input order).
// keys2 (optional) receives a second copy that the sort leaves untouched.
__global__ __launch_bounds__(256) void k_cost(const bvht_BVHNode *__restrict__ nodes, const uint32_t *__restrict__ ids,
                                              uint32_t num, uint32_t *__restrict__ keys, uint32_t *__restrict__ keys2,
                                              uint32_t *__restrict__ hist) {
  __shared__ uint32_t s_hist[4][kSortRadix];
  for (int p = 0; p < 4; ++p) s_hist[p][threadIdx.x] = 0;
  __syncthreads();
  for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < num; i += gridDim.x * 256) {
    const bvht_BVHNode nd = nodes[ids[i]];
    float cost = 0.0f;
    if (nd.isLeafFlag == 0) {
      const float s = nd.surfaceArea, l = nodes[nd.left].surfaceArea, r = nodes[nd.right].surfaceArea;
      cost = (s * s * s * 2.0f) / ((l + r) * (l < r ? l : r));
    }
    const uint32_t key = ~__float_as_uint(cost);
    keys[i] = key;
    if (keys2) keys2[i] = key;
#pragma unroll
    for (int p = 0; p < 4; ++p) atomicAdd(&s_hist[p][(key >> (8 * p)) & 255u], 1u);
  }
  __syncthreads();
  for (int p = 0; p < 4; ++p) {
    const uint32_t c = s_hist[p][threadIdx.x];
    if (c) atomicAdd(hist + p * kSortRadix + threadIdx.x, c);
  }
}

// Ordered-selection tiles: 16 consecutive positions per thread.
constexpr uint32_t kSelBlock = 256, kSelItems = 16, kSelTile = kSelBlock * kSelItems;

// ---- altSort selection (bn13_selectNodes with altSort, :682-699) ----------
//
// The costs sorted descending give the threshold t = sorted[used] (used =
// numChunks * chunkSize); every inner node with cost >= t is flagged
// (kGenerateFlags, :93-97) and the flagged inner-list positions are
// compacted in order (DeviceSelect::Flagged).  When `used` reaches the list
// length every node is flagged.  Costs are compared as floats, decoded from
// the ~bits sort keys.  Three launches: per-tile counts, one workgroup scans
// the tile counts (and fills the entries a step would take beyond the
// selected count with NONE), per-tile ordered writes.
constexpr uint32_t kAltTile = kSelTile;  // 4096 positions per workgroup

__device__ __forceinline__ bool altFlag(uint32_t key, bool all, float thr) {
  return all || __uint_as_float(~key) >= thr;
}

__device__ __forceinline__ void altThreshold(const uint32_t *sortedKeys, uint32_t num, uint32_t used, bool &all,
                                             float &thr) {
  all = used >= num;
  thr = all ? 0.0f : __uint_as_float(~sortedKeys[used]);
}

__global__ __launch_bounds__(kSelBlock) void k_altCount(const uint32_t *__restrict__ keys,
                                                        const uint32_t *__restrict__ sortedKeys, uint32_t num,
                                                        uint32_t used, uint32_t *__restrict__ counts) {
  __shared__ uint32_t s_scan[kSelBlock / 64];
  bool all;
  float thr;
  altThreshold(sortedKeys, num, used, all, thr);
  uint32_t c = 0;
  const uint32_t base = blockIdx.x * kAltTile + threadIdx.x * kSelItems;
  for (uint32_t j = 0; j < kSelItems; ++j)
    if (base + j < num && altFlag(keys[base + j], all, thr)) c++;
  const uint32_t ex = blockExclusiveScan<kSelBlock>(c, s_scan);
  if (threadIdx.x == kSelBlock - 1) counts[blockIdx.x] = ex + c;
}

constexpr int kAltScanBlock = 1024;
__global__ __launch_bounds__(kAltScanBlock) void k_altScan(uint32_t *__restrict__ counts, uint32_t numTiles,
                                                           uint32_t *__restrict__ order, uint32_t used) {
  __shared__ uint32_t s_scan[kAltScanBlock / 64];
  __shared__ uint32_t s_carry;
  if (threadIdx.x == 0) s_carry = 0;
  __syncthreads();
  for (uint32_t b = 0; b < numTiles; b += kAltScanBlock) {
    const uint32_t i = b + threadIdx.x;
    const uint32_t v = i < numTiles ? counts[i] : 0u;
    const uint32_t ex = blockExclusiveScan<kAltScanBlock>(v, s_scan);
    const uint32_t carry = s_carry;
    if (i < numTiles) counts[i] = carry + ex;
    __syncthreads();
    if (threadIdx.x == kAltScanBlock - 1) s_carry = carry + ex + v;
    __syncthreads();
  }
  for (uint32_t i = s_carry + threadIdx.x; i < used; i += kAltScanBlock) order[i] = NONE;
}

__global__ __launch_bounds__(kSelBlock) void k_altWrite(const uint32_t *__restrict__ keys,
                                                        const uint32_t *__restrict__ sortedKeys, uint32_t num,
                                                        uint32_t used, const uint32_t *__restrict__ offsets,
                                                        uint32_t *__restrict__ order) {
  __shared__ uint32_t s_scan[kSelBlock / 64];
  bool all;
  float thr;
  altThreshold(sortedKeys, num, used, all, thr);
  uint32_t c = 0;
  const uint32_t base = blockIdx.x * kAltTile + threadIdx.x * kSelItems;
  for (uint32_t j = 0; j < kSelItems; ++j)
    if (base + j < num && altFlag(keys[base + j], all, thr)) c++;
  uint32_t pos = offsets[blockIdx.x] + blockExclusiveScan<kSelBlock>(c, s_scan);
  for (uint32_t j = 0; j < kSelItems; ++j)
    if (base + j < num && altFlag(keys[base + j], all, thr)) order[pos++] = base + j;
}

// Order-preserving compactions (initData's two DeviceSelect::If calls,
// Bittner13CUDA.cu:962-978): per-block counts and a bit per item, a host-side
// scan of the (few) block counts, then an ordered write from the bits.  A
// wave's items are 64 consecutive ones at a time, so its loads and stores
// share lines, and the nodes are read once: a thread with 16 consecutive nodes,
// read by both launches, took 131 + 355 us for 8.4M nodes against 97 + 13.
constexpr uint32_t kSelWaveItems = kSelTile / (kSelBlock / 64), kSelTrips = kSelWaveItems / 64;
constexpr uint32_t kSelWords = kSelTile / 64;  // words of 64 bits per block
static_assert(kSelTrips <= 64, "a lane per word of a wave");

template <typename F>
__device__ __forceinline__ void selectCount(uint32_t num, F flag, uint64_t *__restrict__ bits,
                                            uint32_t *__restrict__ counts) {
  __shared__ uint32_t s_cnt[kSelBlock / 64];
  const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint32_t base = blockIdx.x * kSelTile + wave * kSelWaveItems + lane;
  bool in[kSelTrips];
#pragma unroll
  for (uint32_t t = 0; t < kSelTrips; ++t) in[t] = base + 64 * t < num && flag(base + 64 * t);
  uint64_t mine = 0;
  uint32_t c = 0;
#pragma unroll
  for (uint32_t t = 0; t < kSelTrips; ++t) {
    const uint64_t b = __ballot(in[t]);
    c += (uint32_t)__popcll(b);
    if (lane == t) mine = b;
  }
  if (lane < kSelTrips) bits[(size_t)blockIdx.x * kSelWords + wave * kSelTrips + lane] = mine;
  if (lane == 0) s_cnt[wave] = c;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (uint32_t w = 1; w < kSelBlock / 64; ++w) c += s_cnt[w];
    counts[blockIdx.x] = c;
  }
}

// put(item, in, items with their bit set before it)
template <typename F>
__device__ __forceinline__ void selectWrite(uint32_t num, const uint64_t *__restrict__ bits,
                                            const uint32_t *__restrict__ offsets, F put) {
  __shared__ uint32_t s_cnt[kSelBlock / 64];
  const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint64_t mine = lane < kSelTrips ? bits[(size_t)blockIdx.x * kSelWords + wave * kSelTrips + lane] : 0;
  const uint32_t own = (uint32_t)__popcll(mine), inc = waveInclusiveScan(own);
  if (lane == 63) s_cnt[wave] = inc;
  __syncthreads();
  uint32_t before = offsets[blockIdx.x];
  for (uint32_t w = 0; w < wave; ++w) before += s_cnt[w];
  const uint32_t base = blockIdx.x * kSelTile + wave * kSelWaveItems + lane;
  const uint64_t lt = __lanemask_lt();
#pragma unroll
  for (uint32_t t = 0; t < kSelTrips; ++t) {
    const uint64_t b = ((uint64_t)__builtin_amdgcn_readlane((int)(mine >> 32), t) << 32) |
                       (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)mine, t);
    const uint32_t first = before + __builtin_amdgcn_readlane((int)(inc - own), t);
    if (base + 64 * t < num) put(base + 64 * t, (b >> lane & 1) != 0, first + (uint32_t)__popcll(b & lt));
  }
}

__global__ __launch_bounds__(kSelBlock) void k_selCount(const bvht_BVHNode *__restrict__ nodes, uint32_t N,
                                                        uint64_t *__restrict__ bits, uint32_t *__restrict__ counts) {
  selectCount(N, [&](uint32_t i) { return nodes[i].isLeafFlag == 0; }, bits, counts);
}

__global__ __launch_bounds__(kSelBlock) void k_selWrite(uint32_t N, const uint64_t *__restrict__ bits,
                                                        const uint32_t *__restrict__ innerOffsets,
                                                        uint32_t *__restrict__ inner, uint32_t *__restrict__ leaves) {
  selectWrite(N, bits, innerOffsets, [&](uint32_t i, bool in, uint32_t before) {
    if (in)
      inner[before] = i;
    else
      leaves[i - before] = i;
  });
}

// Deterministic SA sums: one f64 partial per block, summed on the host.
__global__ __launch_bounds__(256) void k_sahPartials(const bvht_BVHNode *__restrict__ nodes, uint32_t N, uint32_t root,
                                                     float cInner, float cLeaf, int weighted,
                                                     double *__restrict__ partials) {
  __shared__ double s[256];
  double acc = 0.0;
  for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < N; i += gridDim.x * 256) {
    const bvht_BVHNode &nd = nodes[i];
    if (weighted) {
      if (i == root) continue;
      float c = nd.surfaceArea;
      c *= nd.isLeafFlag != 0 ? cLeaf : cInner;
      acc += c;
    } else {
      acc += nd.surfaceArea;
    }
  }
  s[threadIdx.x] = acc;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if (threadIdx.x < (uint32_t)o) s[threadIdx.x] += s[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) partials[blockIdx.x] = s[0];
}

// selectDynamicLeafNodes (CUDAKernels.cu:456-484): leaves whose first face
// is at or after `begin`, in leaf-list order (per-block counts, host scan,
// ordered write -- the order DeviceSelect::If keeps).
__global__ __launch_bounds__(kSelBlock) void k_dynCount(const bvht_BVHNode *__restrict__ nodes,
                                                        const uint32_t *__restrict__ leaves, uint32_t num,
                                                        uint32_t begin, uint64_t *__restrict__ bits,
                                                        uint32_t *__restrict__ counts) {
  selectCount(num, [&](uint32_t i) { return nodes[leaves[i]].left >= begin; }, bits, counts);
}
__global__ __launch_bounds__(kSelBlock) void k_dynWrite(const uint32_t *__restrict__ leaves, uint32_t num,
                                                        const uint64_t *__restrict__ bits,
                                                        const uint32_t *__restrict__ offsets,
                                                        uint32_t *__restrict__ out) {
  selectWrite(num, bits, offsets, [&](uint32_t i, bool in, uint32_t before) {
    if (in) out[before] = leaves[i];
  });
}

struct Internal {
  uint32_t N = 0, numLeaves = 0, numInner = 0, K = 0;
  uint32_t root = 0;
  uint32_t *inner = nullptr, *leaves = nullptr;
  uint32_t *keys[2] = {nullptr, nullptr};  // one allocation; once sorted, k_contain's `above`
  uint32_t *vals[2] = {nullptr, nullptr};
  uint32_t *keysAlt = nullptr;    // altSort: the keys the sort consumes (keys[0] keeps the unsorted costs)
  uint32_t *altCounts = nullptr;  // altSort: per-tile counts / offsets
  uint32_t *sortScratch = nullptr;
  SortPlan plan;
  uint32_t *sorted = nullptr;  // -> vals[result]
  PatchRec *recs = nullptr;
  // the words that initData sets, one allocation: `noneWords` of all ones
  // (locks, marks, fixStarts), then zeroes (the others)
  uint32_t *state = nullptr;
  size_t noneWords = 0, stateWords = 0;
  uint64_t *locks = nullptr;
  uint32_t *marks = nullptr, *cnt = nullptr, *refitCnt = nullptr;
  uint32_t *pending[2] = {nullptr, nullptr}, *numPending = nullptr, *paths = nullptr;
  uint32_t *fixStarts = nullptr;
  uint64_t *refitSlots = nullptr;  // where two refit walks meet (all zero between launches)
  size_t refitSlotWords = 0;
  uint32_t *skipped = nullptr;
  uint32_t *stats = nullptr;
  uint64_t *selBits = nullptr;    // a bit per item of a selection
  uint32_t *selCounts = nullptr;  // behind them: a count per block
  double *partials = nullptr;
  bool selected = false;
  // learned priority and SAH-gain records
  float *feat = nullptr;  // [numInner][12], inner-list order
  uint32_t *leafCnt = nullptr;
  float *subSA = nullptr;
  bool subValid = false;  // leafCnt/subSA match the tree (kept by the refit)
  unsigned long long *up = nullptr;  // computeDepth's pairs; computeSubtree's list before
  PriorityModel *model = nullptr;
  float *recFeat = nullptr, *recGain = nullptr;
  uint32_t *recCount = nullptr;
  uint32_t recMax = 0;
};

// Lays the per-node and per-patch words of `state` out; `words` receives
// their number (before the allocation the pointers mean nothing yet).
void carveState(Internal *in, size_t &words) {
  size_t off = 0;
  auto take = [&](size_t n) {
    uint32_t *p = in->state ? in->state + off : nullptr;
    off += (n + 3) & ~(size_t)3;  // 16-byte steps
    return p;
  };
  in->locks = reinterpret_cast<uint64_t *>(take(2 * (size_t)in->N));
  in->marks = take(in->N);
  in->fixStarts = take(3 * (size_t)in->K);
  in->noneWords = off;
  in->refitSlots = reinterpret_cast<uint64_t *>(take(2 * in->refitSlotWords));
  in->cnt = take(in->N);
  in->refitCnt = take(in->N);
  in->skipped = take(in->K);
  in->stats = take(ST_WORDS);
  in->numPending = take(kCommitRounds);
  words = off;
}

bool features(Internal *in, const bvht_CUDAMemoryBVHPointer *bvh) {
  // each for itself: a call that failed half way may be made again
  if ((!in->feat && !devAlloc(&in->feat, (size_t)in->numInner * kFeat, "bn13 features")) ||
      (!in->leafCnt && !devAlloc(&in->leafCnt, in->N, "bn13 leaf counts")) ||
      (!in->subSA && !devAlloc(&in->subSA, in->N, "bn13 subtree SA")) ||
      (!in->up && !devAlloc(&in->up, in->N, "bn13 depths")))
    return false;
  if (!in->subValid) {
    uint32_t *list = reinterpret_cast<uint32_t *>(in->up);
    if (!computeSubtree(bvh->nodes, in->N, in->leaves, in->numLeaves, in->leafCnt, in->subSA, in->refitCnt, list,
                        list + in->N))
      return false;
    in->subValid = true;
  }
  if (!computeDepth(bvh->nodes, in->N, in->root, in->inner, in->numInner, in->up)) return false;
  return computeFeatures(bvh->nodes, in->N, in->root, in->inner, in->numInner, in->leafCnt, in->subSA, in->up,
                         in->feat);
}

// Refit from `num` device start nodes.  near: a list of leaves in their order
// (no features kept); otherwise a chunk's scattered starts, 8 walks a wave
// (1,881 starts in 1M triangles: 23.2, 25.0, 26.3, 29.2 us with 8, 16, 32, 64),
// with the subtree features kept when they are in use.  More of those than
// slots are done in pieces: a node above starts of two pieces is recomputed by
// each, last with both its children final.
bool refitFrom(Internal *in, const bvht_CUDAMemoryBVHPointer *bvh, const uint32_t *starts, uint32_t num, bool near) {
  const bool feat = !near && in->subValid;
  const uint32_t walks = near ? 64 : 8;
  const uint32_t most = (uint32_t)std::min<size_t>(in->refitSlotWords / (feat ? 6 : 4), 1u << (32 - kRefitSlotShift));
  if (near && num > most) {
    k_refitCount<false><<<divUp(num, kRefitBlock), kRefitBlock, 0, stream()>>>(starts, num, walks, bvh->nodes, in->N, in->cnt);
    if (!checkLaunch("k_refitCount")) return false;
    constexpr uint32_t block = refitBlock(kRefitArrive);
    k_refitApply<false, kRefitArrive><<<divUp(in->N, block), block, 0, stream()>>>(
        nullptr, num, walks, bvh->nodes, in->N, in->cnt, nullptr, nullptr, nullptr, in->stats);
    return checkLaunch("k_refitApply");
  }
  for (uint32_t at = 0; at < num;) {
    const uint32_t n = std::min(most, num - at), blocks = divUp(n, walks * (kRefitBlock / 64));
    k_refitCount<true><<<blocks, kRefitBlock, 0, stream()>>>(starts + at, n, walks, bvh->nodes, in->N, in->cnt);
    if (!checkLaunch("k_refitCount")) return false;
    auto apply = [&](auto feat, auto list, uint32_t grid, uint32_t *leafCnt, float *subSA) {
      k_refitApply<decltype(feat)::value, decltype(list)::value><<<grid, kRefitBlock, 0, stream()>>>(
          starts + at, n, walks, bvh->nodes, in->N, in->cnt, in->refitSlots, leafCnt, subSA, in->stats);
    };
    if (near && n > in->numLeaves / 4)
      apply(std::false_type(), std::integral_constant<int, kRefitIds>(), divUp(in->N, kRefitBlock), nullptr, nullptr);
    else if (near)
      apply(std::false_type(), std::integral_constant<int, kRefitNear>(), blocks, nullptr, nullptr);
    else if (feat)
      apply(std::true_type(), std::integral_constant<int, kRefitScattered>(), blocks, in->leafCnt, in->subSA);
    else
      apply(std::false_type(), std::integral_constant<int, kRefitScattered>(), blocks, nullptr, nullptr);
    if (!checkLaunch("k_refitApply")) return false;
    at += n;
  }
  return true;
}

RecordSink sinkOf(const Internal *in) {
  RecordSink r{nullptr, in->recFeat, in->recGain, in->recCount, in->recMax};
  if (in->recMax) r.feat = in->feat;
  return r;
}

constexpr uint32_t kSahBlocks = 512;

Internal *inOf(bvht_GPUWorkingMemory *d) { return d ? reinterpret_cast<Internal *>(d->internal) : nullptr; }

bool validBVH(const bvht_CUDAMemoryBVHPointer *b, const char *what) {
  if (!b || !b->nodes || b->numNodes == 0) {
    setError("%s: no device BVH", what);
    return false;
  }
  return true;
}

double sahSum(const bvht_CUDAMemoryBVHPointer *b, double *partials, uint32_t root, float ci, float cl, int weighted) {
  k_sahPartials<<<kSahBlocks, 256, 0, stream()>>>(b->nodes, b->numNodes, root, ci, cl, weighted, partials);
  if (!checkLaunch("k_sahPartials")) return -1.0;
  std::vector<double> h(kSahBlocks);
  if (!check(hipMemcpyAsync(h.data(), partials, sizeof(double) * kSahBlocks, hipMemcpyDeviceToHost, stream()),
             "SAH partials") ||
      !check(hipStreamSynchronize(stream()), "SAH sync"))
    return -1.0;
  double s = 0.0;
  for (double x : h) s += x;
  return s;
}

double *sahScratch() {
  static double *p = nullptr;
  if (!p) devMalloc(reinterpret_cast<void **>(&p), sizeof(double) * kSahBlocks, "SAH scratch");
  return p;
}

float rootSA(const bvht_CUDAMemoryBVHPointer *b, uint32_t root) {
  float sa = 0.0f;
  if (check(hipMemcpyAsync(&sa, &b->nodes[root].surfaceArea, sizeof(float), hipMemcpyDeviceToHost, stream()), "root SA"))
    check(hipStreamSynchronize(stream()), "root SA sync");
  return sa;
}

}  // namespace

}  // namespace bvht

using namespace bvht;

extern "C" {

bvht_GPUWorkingMemory allocateMemory(bvht_CUDAMemoryBVHPointer *bvh, uint32_t batchSize, uint32_t numFaces) {
  bvht_GPUWorkingMemory m;
  std::memset(&m, 0, sizeof(m));
  if (!validBVH(bvh, "allocateMemory")) return m;
  if (bvh->numNodes != 2 * numFaces - 1 || numFaces < 2) {
    setError("allocateMemory: %u nodes do not form a binary BVH over %u faces", bvh->numNodes, numFaces);
    return m;
  }
  if (batchSize == 0) {
    setError("allocateMemory: batch size 0");
    return m;
  }
  Internal *in = new (std::nothrow) Internal();
  if (!in) {
    setError("allocateMemory: host allocation failed");
    return m;
  }
  m.internal = in;
  in->N = bvh->numNodes;
  in->numLeaves = numFaces;
  in->numInner = bvh->numNodes - numFaces;
  in->K = batchSize;
  in->plan = makeSortPlan(in->numInner, 4, 32);
  // a chunk's 3 starts per patch in one piece, and lists of up to a quarter of the leaves or 131,072 of them
  in->refitSlotWords = std::max<size_t>(6 * 3 * (size_t)batchSize,
                                        4 * (size_t)std::max(divUp(numFaces, 4), std::min(numFaces, kSlotListMin)));
  carveState(in, in->stateWords);
  const uint32_t selBlocks = divUp(in->N, kSelTile);
  // 1 KB a patch: not where they would take more than two thirds of the nodes' own 48 bytes each
  const bool storePaths = batchSize <= in->N / 32;
  const size_t keyStride = ((size_t)in->numInner + 4) & ~(size_t)3;  // both halves: at least N words, for k_contain
  m.numLeafNodes = in->numLeaves;
  m.numInnerNodes = in->numInner;
  m.numPatches = batchSize;
  m.numSkipped = batchSize;
  m.numNodesToFix = 3 * batchSize;
  m.numFlags = in->N;
  bool ok = devAlloc(&in->inner, in->numInner, "bn13 inner") && devAlloc(&in->leaves, in->numLeaves, "bn13 leaves") &&
            devAlloc(&in->keys[0], 2 * keyStride, "bn13 keys") &&
            devAlloc(&in->vals[0], in->numInner, "bn13 vals") && devAlloc(&in->vals[1], in->numInner, "bn13 vals") &&
            devMalloc(reinterpret_cast<void **>(&in->sortScratch), sortScratchBytes(in->plan), "bn13 sort") &&
            devAlloc(&in->recs, batchSize, "bn13 patches") && devAlloc(&in->state, in->stateWords, "bn13 state") &&
            devAlloc(&in->pending[0], (1 + kOpenWords) * (size_t)batchSize, "bn13 pending") && devAlloc(&in->pending[1], (1 + kOpenWords) * (size_t)batchSize, "bn13 pending") &&
            (!storePaths || devAlloc(&in->paths, 2 * kPathWords * (size_t)batchSize, "bn13 paths")) &&
            devAlloc(&in->selBits, (kSelWords + 1) * (size_t)selBlocks, "bn13 select") && devAlloc(&in->partials, kSahBlocks, "bn13 SAH");
  if (!ok) {
    freeMemory(&m);
    return m;
  }
  carveState(in, in->stateWords);
  in->keys[1] = in->keys[0] + keyStride;
  in->selCounts = reinterpret_cast<uint32_t *>(in->selBits + kSelWords * (size_t)selBlocks);
  m.result = true;
  return m;
}

void freeMemory(bvht_GPUWorkingMemory *data) {
  Internal *in = inOf(data);
  if (in) {
    devFree(in->inner);
    devFree(in->leaves);
    devFree(in->keys[0]);
    devFree(in->keysAlt);
    devFree(in->altCounts);
    devFree(in->vals[0]);
    devFree(in->vals[1]);
    devFree(in->sortScratch);
    devFree(in->recs);
    devFree(in->state);
    devFree(in->pending[0]);
    devFree(in->pending[1]);
    devFree(in->paths);
    devFree(in->selBits);
    devFree(in->partials);
    devFree(in->feat);
    devFree(in->leafCnt);
    devFree(in->subSA);
    devFree(in->up);
    devFree(in->recFeat);
    devFree(in->recGain);
    devFree(in->recCount);
    delete in;
  }
  if (data) {
    std::memset(data, 0, sizeof(*data));
  }
}

void initData(bvht_GPUWorkingMemory *data, bvht_CUDAMemoryBVHPointer *bvh, uint32_t blockSize) {
  (void)blockSize;
  Internal *in = inOf(data);
  if (!in || !validBVH(bvh, "initData")) {
    if (!in) setError("initData: working memory not allocated");
    return;
  }
  // root from the device header (the GPU optimizer keeps it fixed)
  bvht_BVH hdr;
  if (!check(hipMemcpyAsync(&hdr, bvh->bvh, sizeof(hdr), hipMemcpyDeviceToHost, stream()), "initData header") ||
      !check(hipStreamSynchronize(stream()), "initData sync"))
    return;
  in->root = hdr.vRootIndex;
  in->subValid = false;
  const uint32_t selBlocks = divUp(in->N, kSelTile);
  k_selCount<<<selBlocks, kSelBlock, 0, stream()>>>(bvh->nodes, in->N, in->selBits, in->selCounts);
  if (!checkLaunch("k_selCount")) return;
  std::vector<uint32_t> counts(selBlocks);
  if (!check(hipMemcpyAsync(counts.data(), in->selCounts, 4ull * selBlocks, hipMemcpyDeviceToHost, stream()),
             "initData counts") ||
      !check(hipStreamSynchronize(stream()), "initData sync"))
    return;
  uint32_t total = 0;
  for (auto &c : counts) {
    uint32_t t = c;
    c = total;
    total += t;
  }
  if (total != in->numInner) {
    setError("initData: %u inner nodes found, expected %u", total, in->numInner);
    return;
  }
  if (!check(hipMemcpyAsync(in->selCounts, counts.data(), 4ull * selBlocks, hipMemcpyHostToDevice, stream()),
             "initData offsets"))
    return;
  k_selWrite<<<selBlocks, kSelBlock, 0, stream()>>>(in->N, in->selBits, in->selCounts, in->inner, in->leaves);
  if (!checkLaunch("k_selWrite")) return;
  fillU32(in->state, NONE, in->noneWords);  // locks: kLockFree
  fillU32(in->state + in->noneWords, 0u, in->stateWords - in->noneWords);
  check(hipMemsetAsync(in->recs, 0, sizeof(PatchRec) * in->K, stream()), "initData patches");
  check(hipStreamSynchronize(stream()), "initData sync");
}

void fixTree1(bvht_GPUWorkingMemory *data, bvht_CUDAMemoryBVHPointer *bvh, uint32_t blockSize) {
  (void)blockSize;
  Internal *in = inOf(data);
  if (!in || !validBVH(bvh, "fixTree1")) return;
  in->subValid = false;  // boxes may change; the subtree features are recomputed when next needed
  refitFromLeaves(bvh->nodes, 0, in->numLeaves, in->leaves, in->refitCnt, in->N);
}

void fixTree3(bvht_GPUWorkingMemory *data, bvht_CUDAMemoryBVHPointer *bvh, uint32_t blockSize) {
  (void)blockSize;
  Internal *in = inOf(data);
  if (!in || !validBVH(bvh, "fixTree3")) return;
  refitFrom(in, bvh, in->fixStarts, 3 * in->K, false);
}

void selectDynamicLeafNodes(bvht_GPUWorkingMemory *data, bvht_CUDAMemoryBVHPointer *bvh, uint32_t *out,
                            uint32_t *numOut, uint32_t beginDynamicTriangle) {
  Internal *in = inOf(data);
  if (numOut) *numOut = 0;
  if (!in || !validBVH(bvh, "selectDynamicLeafNodes") || !out || !numOut) {
    if (!in) setError("selectDynamicLeafNodes: working memory not allocated");
    else if (!out || !numOut) setError("selectDynamicLeafNodes: no output");
    return;
  }
  const uint32_t blocks = divUp(in->numLeaves, kSelTile);
  k_dynCount<<<blocks, kSelBlock, 0, stream()>>>(bvh->nodes, in->leaves, in->numLeaves, beginDynamicTriangle,
                                                 in->selBits, in->selCounts);
  if (!checkLaunch("k_dynCount")) return;
  std::vector<uint32_t> counts(blocks);
  if (!check(hipMemcpyAsync(counts.data(), in->selCounts, 4ull * blocks, hipMemcpyDeviceToHost, stream()),
             "selectDynamicLeafNodes counts") ||
      !check(hipStreamSynchronize(stream()), "selectDynamicLeafNodes sync"))
    return;
  uint32_t total = 0;
  for (auto &c : counts) {
    const uint32_t t = c;
    c = total;
    total += t;
  }
  if (!check(hipMemcpyAsync(in->selCounts, counts.data(), 4ull * blocks, hipMemcpyHostToDevice, stream()),
             "selectDynamicLeafNodes offsets"))
    return;
  k_dynWrite<<<blocks, kSelBlock, 0, stream()>>>(in->leaves, in->numLeaves, in->selBits, in->selCounts, out);
  if (!checkLaunch("k_dynWrite") || !check(hipStreamSynchronize(stream()), "selectDynamicLeafNodes sync")) return;
  *numOut = total;
}

bool bvht_fixTreeFrom(bvht_GPUWorkingMemory *data, bvht_CUDAMemoryBVHPointer *bvh, const uint32_t *devStarts,
                      uint32_t num) {
  Internal *in = inOf(data);
  if (!in || !validBVH(bvh, "bvht_fixTreeFrom")) {
    if (!in) setError("bvht_fixTreeFrom: working memory not allocated");
    return false;
  }
  if (num == 0) return true;
  if (!devStarts) {
    setError("bvht_fixTreeFrom: no start nodes");
    return false;
  }
  in->subValid = false;  // leaf boxes may have changed (dynamic refit)
  return refitFrom(in, bvh, devStarts, num, true);
}

void bn13_selectNodes(bvht_GPUWorkingMemory *data, bvht_CUDAMemoryBVHPointer *bvh, bvht_AlgoCFG cfg) {
  Internal *in = inOf(data);
  if (!in || !validBVH(bvh, "bn13_selectNodes")) return;
  if (!cfg.sort) {  // Bittner13CUDA.cu:719
    setError("bn13_selectNodes: topKThElement is not supported (set option sort)");
    return;
  }
  if (cfg.priority > 1 || (cfg.priority == 1 && !in->model)) {
    setError("bn13_selectNodes: priority %u needs %s", cfg.priority,
             cfg.priority == 1 ? "a model (bvht_bn13_setModel)" : "0 (heuristic) or 1 (learned)");
    return;
  }
  if ((cfg.priority == 1 || in->recMax) && !features(in, bvh)) return;
  const bool alt = cfg.altSort != 0;
  if (alt && cfg.priority == 1) {
    setError("bn13_selectNodes: altSort selects by the heuristic priority only (priority 0)");
    return;
  }
  const uint64_t used = (uint64_t)cfg.numChunks * cfg.chunkSize;
  if (alt && used > in->numInner) {
    setError("bn13_selectNodes: altSort: %u chunks x %u exceed %u inner nodes", cfg.numChunks, cfg.chunkSize,
             in->numInner);
    return;
  }
  const uint32_t altTiles = divUp(in->numInner, kAltTile);
  if (alt && ((!in->keysAlt && !devAlloc(&in->keysAlt, in->numInner, "bn13 altSort keys")) ||
              (!in->altCounts && !devAlloc(&in->altCounts, altTiles, "bn13 altSort counts"))))
    return;
  uint32_t *scratch = in->sortScratch;
  if (!sortReset(in->plan, scratch)) return;
  if (cfg.priority == 1) {
    if (!mlpInfer(*in->model, in->feat, in->numInner, in->keys[0], sortHist(in->plan, scratch), nullptr)) return;
  } else {
    uint32_t blocks = divUp(in->numInner, 256 * 8);
    if (blocks > (uint32_t)numCUs() * 8) blocks = numCUs() * 8;
    k_cost<<<blocks, 256, 0, stream()>>>(bvh->nodes, in->inner, in->numInner, alt ? in->keysAlt : in->keys[0],
                                         alt ? in->keys[0] : nullptr, sortHist(in->plan, scratch));
    if (!checkLaunch("k_cost")) return;
  }
  if (alt) {
    // SortKeysDescending (:682-686): keysAlt and keys[1] ping-pong, keys[0]
    // keeps the unsorted costs for the flags
    void *keys[2] = {in->keysAlt, in->keys[1]};
    uint32_t *vals[2] = {in->vals[0], in->vals[1]};
    const int r = sortRun(in->plan, keys, vals, true, true, scratch);
    if (r < 0) return;
    const uint32_t *sortedKeys = reinterpret_cast<const uint32_t *>(keys[r]);
    uint32_t *order = in->vals[0];
    k_altCount<<<altTiles, kSelBlock, 0, stream()>>>(in->keys[0], sortedKeys, in->numInner, (uint32_t)used,
                                                     in->altCounts);
    if (!checkLaunch("k_altCount")) return;
    k_altScan<<<1, kAltScanBlock, 0, stream()>>>(in->altCounts, altTiles, order, (uint32_t)used);
    if (!checkLaunch("k_altScan")) return;
    k_altWrite<<<altTiles, kSelBlock, 0, stream()>>>(in->keys[0], sortedKeys, in->numInner, (uint32_t)used,
                                                     in->altCounts, order);
    if (!checkLaunch("k_altWrite")) return;
    in->sorted = order;
    in->selected = true;
    return;
  }
  void *keys[2] = {in->keys[0], in->keys[1]};
  uint32_t *vals[2] = {in->vals[0], in->vals[1]};
  // values: inner-list positions (identity); k_search maps them to node ids
  const int r = sortRun(in->plan, keys, vals, true, false, scratch);
  if (r < 0) return;
  in->sorted = in->vals[r];
  in->selected = true;
}

// Rounds over the whole GPU before the rest goes to one workgroup, which takes
// about 20 us for 800 undecided patches and more than its LDS holds much worse;
// a round costs a launch, 5 us.  Many patches, or many for the tree, leave enough
// of them.  Per chunk, us, with 1 / 2 / 3 rounds: K = 386 of N = 154k nodes
// 88.9 / 90.4 / 91.2, 965 of 154k 107.6 / 106.2 / 107.2, 1,134 of 1.8M
// 109.5 / 111.9 / 114.4, 2,269 of 1.8M 129.1 / 125.3 / 127.1, 5,105 of 8.2M
// 201 / 188 / 190, 10,210 of 8.2M 440 / 301 / 306, 11,349 of 1.8M 669 / 355 / 278.
static uint32_t commitRounds(uint32_t K, uint32_t N) {
  if (K >= 4096 && K >= N / 256) return 3;
  return K >= 2048 || (K >= 768 && K >= N / 512) ? 2 : 1;
}
static_assert(kCommitRounds >= 3, "a list length for every round");

void bn13_rmAndReinsChunk(bvht_GPUWorkingMemory *data, bvht_CUDAMemoryBVHPointer *bvh, bvht_AlgoCFG cfg, uint32_t chunk) {
  Internal *in = inOf(data);
  if (!in || !validBVH(bvh, "bn13_rmAndReinsChunk")) return;
  if (!in->selected) {
    setError("bn13_rmAndReinsChunk: call bn13_selectNodes first");
    return;
  }
  const uint32_t K = cfg.chunkSize;
  if (K == 0 || K > in->K || (uint64_t)cfg.numChunks * K > in->numInner || chunk >= cfg.numChunks) {
    setError("bn13_rmAndReinsChunk: chunk %u of %u x %u does not fit %u patches / %u inner nodes", chunk, cfg.numChunks,
             K, in->K, in->numInner);
    return;
  }
  // the first chunk of a step also counts a failed priority sort (its error
  // word is cleared with the sort state at the next selection)
  k_search<false><<<K, 64, 0, stream()>>>(bvh->nodes, in->root, in->N, in->sorted, in->inner, in->numInner, chunk,
                                          cfg.numChunks, K, cfg.offsetAccess ? 1u : 0u, cfg.altFindNode ? 1u : 0u,
                                          in->recs, in->locks, in->marks, in->stats, sinkOf(in),
                                          chunk == 0 ? in->sortScratch + in->plan.errOff : nullptr);
  if (!checkLaunch("k_search")) return;
  const uint32_t commitBlocks = divUp(K, kPatchesPerBlock), rounds = commitRounds(K, in->N);
  k_commit<false><<<commitBlocks, kPatchBlock, 0, stream()>>>(in->recs, K, in->locks, in->marks, in->skipped, in->stats,
                                                              nullptr, nullptr, in->pending[0], in->numPending, 1u,
                                                              rounds > 1);
  if (!checkLaunch("k_commit")) return;
  for (uint32_t r = 2; r <= rounds; ++r) {
    k_commit<true><<<commitBlocks, kPatchBlock, 0, stream()>>>(in->recs, K, in->locks, in->marks, in->skipped, in->stats,
                                                               in->pending[r & 1], in->numPending + r - 2,
                                                               in->pending[(r & 1) ^ 1], in->numPending + r - 1, r,
                                                               r < rounds);
    if (!checkLaunch("k_commit")) return;
  }
  const size_t lists = kOpenWords * (size_t)in->K;  // behind the open entries: room for k_resolveTail's lists
  // one wave of walks a workgroup (a CU each: its LDS is the tail's) while the
  // CUs take them all, else whole workgroups
  const uint32_t walkers = divUp(2ull * K, 64) < (uint32_t)numCUs() ? 64 : kTailBlock;
  k_resolveTail<<<1 + divUp(2ull * K, walkers), kTailBlock, 0, stream()>>>(
      in->recs, in->locks, in->marks, in->skipped, in->stats, in->pending[(rounds & 1) ^ 1],
      in->pending[0] + lists, in->pending[1] + lists, in->numPending + rounds - 1, K, bvh->nodes, in->root, in->N,
      in->paths, in->keys[0], walkers, rounds + 1);
  if (!checkLaunch("k_resolveTail")) return;
  k_contain<<<divUp(K, kPatchesPerBlock), kPatchBlock, 0, stream()>>>(in->recs, K, bvh->nodes, in->root, in->N, in->marks,
                                                                      in->paths, in->keys[0], in->locks, in->fixStarts,
                                                                      in->skipped, in->numPending, in->stats);
  if (!checkLaunch("k_contain")) return;
  refitFrom(in, bvh, in->fixStarts, 3 * K, false);
}

void bn13_doAlgorithmStep(bvht_GPUWorkingMemory *data, bvht_CUDAMemoryBVHPointer *bvh, bvht_AlgoCFG cfg) {
  bn13_selectNodes(data, bvh, cfg);
  for (uint32_t i = 0; i < cfg.numChunks; ++i) bn13_rmAndReinsChunk(data, bvh, cfg, i);
}

float CUDAcalcSAH(bvht_CUDAMemoryBVHPointer *bvh) {
  if (!validBVH(bvh, "CUDAcalcSAH")) return 0.0f;
  double *p = sahScratch();
  if (!p) return 0.0f;
  const double s = sahSum(bvh, p, 0, 1.0f, 1.0f, 0);
  const float r = rootSA(bvh, 0);  // the reference reads node 0 (Bittner13CUDA.cu:794)
  return (float)((s - (double)r) / (double)r);
}

double bvht_calcSAHWeighted(bvht_CUDAMemoryBVHPointer *bvh, float cInner, float cLeaf) {
  if (!validBVH(bvh, "bvht_calcSAHWeighted")) return 0.0;
  bvht_BVH hdr;
  if (!check(hipMemcpyAsync(&hdr, bvh->bvh, sizeof(hdr), hipMemcpyDeviceToHost, stream()), "SAH header") ||
      !check(hipStreamSynchronize(stream()), "SAH sync"))
    return 0.0;
  double *p = sahScratch();
  if (!p) return 0.0;
  const double s = sahSum(bvh, p, hdr.vRootIndex, cInner, cLeaf, 1);
  return s / (double)rootSA(bvh, hdr.vRootIndex);
}

void doCudaDevSync(void) { check(hipStreamSynchronize(stream()), "doCudaDevSync"); }

uint32_t calcNumSkipped(bvht_GPUWorkingMemory *data) {
  Internal *in = inOf(data);
  if (!in) return 0;
  std::vector<uint32_t> h(in->K);
  if (!check(hipMemcpyAsync(h.data(), in->skipped, 4ull * in->K, hipMemcpyDeviceToHost, stream()), "calcNumSkipped") ||
      !check(hipStreamSynchronize(stream()), "calcNumSkipped sync"))
    return 0;
  uint32_t s = 0;
  for (uint32_t x : h) s += x;
  return s;
}

// Counters of the optimizer (extension): conflicts, failed patches,
// containment drops, frontier overflows, applied patches, patches left
// undecided by the conflict resolution (always 0), searches stopped at the
// step bound (always 0 for a tree).
int bvht_bn13_stats(bvht_GPUWorkingMemory *data, uint32_t *out, int maxWords) {
  Internal *in = inOf(data);
  if (!in || !out) return 0;
  uint32_t h[ST_WORDS];
  if (!check(hipMemcpyAsync(h, in->stats, sizeof(h), hipMemcpyDeviceToHost, stream()), "bn13 stats") ||
      !check(hipStreamSynchronize(stream()), "bn13 stats sync"))
    return 0;
  int n = maxWords < 8 ? maxWords : 8;
  for (int i = 0; i < n; ++i) out[i] = h[i];
  return n;
}

// ---- learned priority and SAH-gain records (extension) -------------------

bool bvht_bn13_setModel(bvht_GPUWorkingMemory *data, bvht_PriorityModel *model) {
  Internal *in = inOf(data);
  if (!in) {
    setError("bvht_bn13_setModel: working memory not allocated");
    return false;
  }
  in->model = reinterpret_cast<PriorityModel *>(model);
  return true;
}

bool bvht_bn13_features(bvht_GPUWorkingMemory *data, bvht_CUDAMemoryBVHPointer *bvh, float *devFeat) {
  Internal *in = inOf(data);
  if (!in || !validBVH(bvh, "bvht_bn13_features") || !devFeat) {
    if (!in) setError("bvht_bn13_features: working memory not allocated");
    if (!devFeat) setError("bvht_bn13_features: no output buffer");
    return false;
  }
  if (!features(in, bvh)) return false;
  return check(hipMemcpyAsync(devFeat, in->feat, sizeof(float) * kFeat * (size_t)in->numInner,
                              hipMemcpyDeviceToDevice, stream()),
               "bvht_bn13_features");
}

bool bvht_bn13_setRecording(bvht_GPUWorkingMemory *data, uint32_t maxRecords) {
  Internal *in = inOf(data);
  if (!in) {
    setError("bvht_bn13_setRecording: working memory not allocated");
    return false;
  }
  devFree(in->recFeat);
  devFree(in->recGain);
  devFree(in->recCount);
  in->recFeat = in->recGain = nullptr;
  in->recCount = nullptr;
  in->recMax = 0;
  if (maxRecords == 0) return true;
  if (!devAlloc(&in->recFeat, (size_t)maxRecords * kFeat, "bn13 record features") ||
      !devAlloc(&in->recGain, maxRecords, "bn13 record gains") || !devAlloc(&in->recCount, 1, "bn13 record count") ||
      !fillU32(in->recCount, 0u, 1))
    return false;
  in->recMax = maxRecords;
  return true;
}

uint32_t bvht_bn13_records(bvht_GPUWorkingMemory *data, float **devFeat, float **devGain) {
  Internal *in = inOf(data);
  if (!in || !in->recMax) return 0;
  uint32_t n = 0;
  if (!check(hipMemcpyAsync(&n, in->recCount, 4, hipMemcpyDeviceToHost, stream()), "bvht_bn13_records") ||
      !check(hipStreamSynchronize(stream()), "bvht_bn13_records sync"))
    return 0;
  if (devFeat) *devFeat = in->recFeat;
  if (devGain) *devGain = in->recGain;
  return n < in->recMax ? n : in->recMax;
}

bool bvht_bn13_probe(bvht_GPUWorkingMemory *data, bvht_CUDAMemoryBVHPointer *bvh, bvht_AlgoCFG cfg,
                     const uint32_t *devPositions, uint32_t num) {
  Internal *in = inOf(data);
  if (!in || !validBVH(bvh, "bvht_bn13_probe")) {
    if (!in) setError("bvht_bn13_probe: working memory not allocated");
    return false;
  }
  if (!in->recMax) {
    setError("bvht_bn13_probe: enable recording first (bvht_bn13_setRecording)");
    return false;
  }
  if (num == 0) return true;
  if (!devPositions) {
    setError("bvht_bn13_probe: no positions");
    return false;
  }
  if (!features(in, bvh)) return false;
  k_search<true><<<num, 64, 0, stream()>>>(bvh->nodes, in->root, in->N, devPositions, in->inner, in->numInner, 0, 1,
                                          num, 0u, cfg.altFindNode ? 1u : 0u, in->recs, in->locks, in->marks,
                                          in->stats, sinkOf(in), nullptr);
  return checkLaunch("k_search (probe)");
}

}  // extern "C"
