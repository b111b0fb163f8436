// .svdag input: EncodedSVDAG::load + decode (encoded_svdag.cpp:43-66, 200-281).
//
// File: f32 min[3], f32 max[3], f32 rootSide, u32 levels, u32 nNodes,
// u32 firstLeafPtr, u32 count, u32 data[count].  Above the leaf level a node
// is its mask word followed by one absolute word index per child, child 7
// first; a leaf is its mask word.  The reference parses the words in order:
// a level begins at the smallest pointer seen in the level above, and a
// pointer becomes the target's node index in its level (words before the
// target minus pointer words before it).
//
// Device form, one level at a time from the root: the nodes of level l+1 are
// exactly the targets of level l's pointers (in a file written by the
// encoder every node is referenced), so marking the targets in the word range
// [smallest pointer, largest pointer] and scanning the marks numbers the nodes
// in file order.  A level has at most 8 times the nodes above it and a node 9
// words, so the marks to scan are bounded before the pointers are read, and a
// level needs one read-back (its range, error flags and the next level's
// size).  The decoded nodes must tile every level's word range and the
// leaf level must end at the last word; a file that breaks this (unreferenced
// or overlapping words, where a sequential parse could read differently) is
// rejected with SVD_ERR_FORMAT instead of being decoded differently.
#include <algorithm>
#include "svd_internal.hpp"

namespace svd {

namespace {

constexpr int kB = 256;

// Per level on the device: smallest and largest pointer, end of the level's
// words, error flags, nodes of the next level.
enum { kLo = 0, kHi, kEnd, kErr, kNext, kState };

__global__ void k_dec_init(uint32_t* __restrict__ st, uint32_t levels, uint32_t* __restrict__ root) {
  if (threadIdx.x < levels) {
    uint32_t* s = st + (uint64_t)threadIdx.x * kState;
    s[kLo] = 0xFFFFFFFFu;
    s[kHi] = s[kEnd] = s[kErr] = s[kNext] = 0u;
  }
  if (threadIdx.x == 0) *root = 0u;   // level 0: the root at word 0
}

// Node i of an inner level at word starts[i]: the 9-word record with raw
// (absolute word) child pointers; marks the targets; folds min/max pointer
// (one atomic each per workgroup).  Below the root a node without children
// never comes out of the encoder (buildSVO's cleanEmptyNodes and toDAG drop
// them), so it flags the file.
__global__ void __launch_bounds__(kB) k_dec_inner(const uint32_t* __restrict__ data, uint32_t count,
                                                  const uint32_t* __restrict__ starts, uint32_t n, uint32_t belowRoot,
                                                  uint32_t* __restrict__ rec, uint32_t* __restrict__ mark,
                                                  uint32_t* __restrict__ st) {
  __shared__ uint32_t wlo[kB / 64], whi[kB / 64];
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  uint32_t lo = 0xFFFFFFFFu, hi = 0;
  if (i < n) {
    const uint32_t w = starts[i];
    const uint32_t m = data[w] & 0xFFu;
    const uint32_t nc = (uint32_t)__popc(m);
    uint32_t* r = rec + (uint64_t)i * kRecWords;
    r[0] = m;
    mark[w] = 0u;        // from here on the marks are the next level's
    if (belowRoot && m == 0) atomicOr(&st[kErr], 4u);
    // tiling: this node ends where the next one starts
    const uint32_t end = w + 1 + nc;
    if (end > count || (i + 1 < n && starts[i + 1] != end)) {
      atomicOr(&st[kErr], 1u);
    } else {
      if (i + 1 == n) st[kEnd] = end;
      uint32_t k = 0;
      for (int c = 7; c >= 0; --c) {
        uint32_t v = kNull;
        if ((m >> c) & 1u) {
          v = data[w + 1 + k++];
          if (v >= count) { atomicOr(&st[kErr], 2u); v = kNull; }
          else {
            mark[v] = 1u;
            lo = min(lo, v);
            hi = max(hi, v);
          }
        }
        r[1 + c] = v;
      }
    }
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    lo = min(lo, (uint32_t)__shfl_xor(lo, o, 64));
    hi = max(hi, (uint32_t)__shfl_xor(hi, o, 64));
  }
  if ((threadIdx.x & 63) == 0) { wlo[threadIdx.x >> 6] = lo; whi[threadIdx.x >> 6] = hi; }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int q = 1; q < kB / 64; ++q) { lo = min(lo, wlo[q]); hi = max(hi, whi[q]); }
    if (lo != 0xFFFFFFFFu) { atomicMin(&st[kLo], lo); atomicMax(&st[kHi], hi); }
  }
}

__global__ void k_dec_leaf(const uint32_t* __restrict__ data, const uint32_t* __restrict__ starts, uint32_t n,
                           uint32_t count, uint32_t* __restrict__ rec, uint32_t* __restrict__ err) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint32_t w = starts[i];
  rec[i] = data[w] & 0xFFu;
  if ((data[w] & 0xFFu) == 0) atomicOr(err, 4u);
  const uint32_t next = i + 1 < n ? starts[i + 1] : count;
  if (next != w + 1) atomicOr(err, 1u);
}

// The next level's starts, from the marks (words lo .. lo + len - 1) and their
// scan from word from on; and raw pointers of this level -> node indices.
__global__ void k_dec_next(const uint32_t* __restrict__ mark, const uint32_t* __restrict__ pos, uint32_t from,
                           uint32_t lo, uint32_t len, uint32_t* __restrict__ starts, uint32_t* __restrict__ rec,
                           uint32_t n) {
  const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j < len && mark[lo + j]) starts[pos[lo + j - from]] = lo + j;
  if (j >= n) return;
  uint32_t* r = rec + (uint64_t)j * kRecWords;
  for (int c = 0; c < 8; ++c)
    if (r[1 + c] != kNull) r[1 + c] = pos[r[1 + c] - from];
}

}  // namespace

void octree_from_svdag(svd_octree* o, const uint8_t* file, uint64_t bytes, bool onDevice) {
  svd_ctx* c = o->ctx;
  constexpr uint64_t kHead = 40;
  if (bytes < kHead) throw Error{SVD_ERR_FORMAT, ".svdag: file shorter than its header"};
  uint8_t head[kHead + 4];
  if (bytes < kHead + 4) throw Error{SVD_ERR_FORMAT, ".svdag: file shorter than its header"};
  if (onDevice) {
    SVD_HIP(hipMemcpyAsync(head, file, kHead + 4, hipMemcpyDeviceToHost, c->stream));
    SVD_HIP(hipStreamSynchronize(c->stream));
  } else {
    memcpy(head, file, kHead + 4);
  }
  float bb[6], rootSide;
  uint32_t levels, nNodes, firstLeaf, count;
  memcpy(bb, head, 24);
  memcpy(&rootSide, head + 24, 4);
  memcpy(&levels, head + 28, 4);
  memcpy(&nNodes, head + 32, 4);
  memcpy(&firstLeaf, head + 36, 4);
  (void)firstLeaf;
  memcpy(&count, head + kHead, 4);
  if (levels < 2 || levels > (uint32_t)kMaxLevels) throw Error{SVD_ERR_LEVELS, ".svdag: unsupported level count"};
  if (bytes < kHead + 4 + 4ull * count || count == 0) throw Error{SVD_ERR_FORMAT, ".svdag: truncated word array"};
  uint32_t* data = dalloc<uint32_t>(c, (uint64_t)count + 1);
  SVD_HIP(hipMemcpyAsync(data, file + kHead + 4, 4ull * count, onDevice ? hipMemcpyDeviceToDevice
                                                                          : hipMemcpyHostToDevice, c->stream));
  uint32_t* mark = dalloc<uint32_t>(c, (uint64_t)count + 1);
  fill_u32(c, mark, 0u, count + 1);
  uint32_t* dev = dalloc<uint32_t>(c, (uint64_t)levels * kState);
  std::vector<Level> lv(levels);
  uint32_t* starts = dalloc<uint32_t>(c, 2);
  k_dec_init<<<1, 64, 0, c->stream>>>(dev, levels, starts);
  check_launch("k_dec_init");
  uint64_t n = 1, first = 0;                // nodes and first word of the level
  auto fail = [&](const std::string& what) {
    for (auto& x : lv) dfree(c, x.rec);
    dfree(c, data); dfree(c, mark); dfree(c, dev); dfree(c, starts);
    throw Error{SVD_ERR_FORMAT, ".svdag: " + what};
  };
  for (uint32_t l = 0; l < levels; ++l) {
    lv[l].n = n;
    lv[l].leaf = (l == levels - 1);
    uint32_t* st = dev + (uint64_t)l * kState;
    uint32_t h[kState];
    if (lv[l].leaf) {
      lv[l].rec = dalloc<uint32_t>(c, n + 1);
      k_dec_leaf<<<div_up(n, kB), kB, 0, c->stream>>>(data, starts, (uint32_t)n, count, lv[l].rec, st + kErr);
      check_launch("k_dec_leaf");
      read_u32s(c, st, h, kState);
      if (h[kErr] & 4u) fail("empty leaf node in level " + std::to_string(l));
      if (h[kErr]) fail("leaf words do not end the file");
      break;
    }
    lv[l].rec = dalloc<uint32_t>(c, n * kRecWords + 1);
    k_dec_inner<<<div_up(n, kB), kB, 0, c->stream>>>(data, count, starts, (uint32_t)n, l > 0 ? 1u : 0u, lv[l].rec,
                                                     mark, st);
    check_launch("k_dec_inner");
    // the next level begins after this one (n words at least) and its last
    // node starts at most 9 n + 72 n words on
    const uint64_t from = std::min<uint64_t>(first + n, count);
    const uint64_t upTo = std::min<uint64_t>(first + 81 * n, count);
    uint32_t* pos = dalloc<uint32_t>(c, upTo - from + 1);
    scan_exclusive(c, mark + from, pos, upTo - from, st + kNext);
    read_u32s(c, st, h, kState);
    auto stop = [&](const std::string& what) { dfree(c, pos); fail(what); };
    if (h[kErr] & 4u) stop("node without children below the root in level " + std::to_string(l));
    if (h[kErr] & 2u) stop("child pointer outside the word array");
    if (h[kErr]) stop("nodes do not tile level " + std::to_string(l));
    if (h[kLo] == 0xFFFFFFFFu) stop("level " + std::to_string(l) + " has no children");
    if (h[kLo] != h[kEnd]) stop("level " + std::to_string(l + 1) + " does not start where level " + std::to_string(l) +
                                " ends");
    if (h[kHi] >= upTo) stop("nodes do not tile level " + std::to_string(l + 1));
    const uint32_t lo = h[kLo], len = h[kHi] - h[kLo] + 1;
    const uint64_t nNext = h[kNext];
    dfree(c, starts);
    starts = dalloc<uint32_t>(c, nNext + 1);
    k_dec_next<<<div_up(std::max<uint64_t>(len, n), kB), kB, 0, c->stream>>>(mark, pos, (uint32_t)from, lo, len, starts,
                                                                             lv[l].rec, (uint32_t)n);
    check_launch("k_dec_next");
    dfree(c, pos);
    first = lo;
    n = nNext;
  }
  SVD_HIP(hipStreamSynchronize(c->stream));
  dfree(c, data); dfree(c, mark); dfree(c, dev); dfree(c, starts);
  o->levels = levels;
  for (int i = 0; i < 6; ++i) o->bbox[i] = bb[i];
  o->rootSide = rootSide;
  o->dag = lv;
  o->nNodesDAG = nNodes;   // the header's count (GeomOctree(NodeData, ...) takes stats.nNodesDAG)
  o->nVoxels = 0;          // EncodedSVDAG::load leaves _nVoxels at 0 and decode copies it
  o->state = SVD_S_DAG;
}

}  // namespace svd
