// CSVDAG cross-level merge on the device (geom_octree_extension.cpp:1192-1544).
//
// The reference walks a top-down frontier: every frontier node A of level levA
// is compared (compareSubtrees, :238-290) with the nodes of the levels above
// that share its hash (computeNodeHash, :34-74); the first equal one in
// (levB, index) order wins, A's whole subtree is recorded as corresponding to
// B's, and unmatched nodes send their children to the next frontier.  Then the
// levels are compacted bottom-up and pointers redirected (:1428-1498).
//
// compareSubtrees(A, B) is equality of the two subtrees cut at the depth of
// A's leaves: every pair of visited nodes has equal child masks.  Here that
// equality is a class number: cls_0(x) = mask(x), and cls_d(x) = the hash-table
// slot of (mask(x), cls_{d-1}(children)) over all nodes of levels 1..L-1-d, so
// cls_d(A) == cls_d(B) exactly when the depth-d subtrees are equal.  Equal
// subtrees have equal hashes (the hash depth never exceeds the compared
// depth), so the hash pre-filter drops nothing and is not needed.  The first
// match is then an atomicMin of (levB << 32 | index) per class.
//
// Recording: inside one comparison the reference's map keeps the last
// pre-order visit of a node; between matches of one round the earliest
// frontier node wins.  The last pre-order visit of x is its lexicographically
// largest child-slot path from A, so a top-down pass per level keeps, per
// node, the smallest matching frontier index and then the largest path
// (path * 8 + slot), and the winning parent writes B's descendant on the same
// path.  No subtree is walked per thread.
//
// The state of all levels lies in flat arrays (level l from base[l] on), so a
// step over several levels is one launch: a merge is bound by its launches
// and read-backs (2.8 us per launch at 200K nodes), not by its work.
#include "svd_internal.hpp"

namespace svd {

namespace {

constexpr int kB = 256;
constexpr uint32_t kMaxL = 21;

struct LevelPtrs {
  const uint32_t* rec[kMaxL];   // 9-word records (leaf level: 1 word)
  uint32_t n[kMaxL];
  uint64_t base[kMaxL + 1];     // flat index of a level's first node
  uint32_t leafLevel;
};

// Level and node of a flat index between levels lo and hi.
__device__ __forceinline__ uint32_t level_of(const LevelPtrs& P, uint64_t e, uint32_t lo, uint32_t hi, uint32_t& i) {
  uint32_t l = lo;
  while (l < hi && e >= P.base[l + 1]) ++l;
  i = (uint32_t)(e - P.base[l]);
  return l;
}

__device__ __forceinline__ uint32_t node_mask(const LevelPtrs& P, uint32_t lev, uint32_t i) {
  return lev == P.leafLevel ? (P.rec[lev][i] & 0xFFu) : (P.rec[lev][(uint64_t)i * kRecWords] & 0xFFu);
}
__device__ __forceinline__ uint32_t node_child(const LevelPtrs& P, uint32_t lev, uint32_t i, int c) {
  return lev == P.leafLevel ? kNull : P.rec[lev][(uint64_t)i * kRecWords + 1 + c];
}

// ---- truncated-subtree classes ---------------------------------------------
// keys of levels 1..top for depth d >= 1: mask, then the children's cls_{d-1}
// (clsChild == nullptr: d == 1, the children's masks).  Class and key arrays
// start at level 1.
__global__ void k_class_keys(LevelPtrs P, uint32_t top, const uint32_t* __restrict__ clsChild,
                             uint32_t* __restrict__ keys) {
  const uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= P.base[top + 1] - P.base[1]) return;
  uint32_t i;
  const uint32_t lev = level_of(P, e + P.base[1], 1, top, i);
  const uint32_t m = node_mask(P, lev, i);
  const uint64_t below = P.base[lev + 1] - P.base[1];
  uint32_t* k = keys + e * kRecWords;
  k[0] = m;
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    uint32_t v = kNull;
    if ((m >> c) & 1u) {
      const uint32_t ch = node_child(P, lev, i, c);
      v = clsChild ? clsChild[below + ch] : node_mask(P, lev + 1, ch);
    }
    k[1 + c] = v;
  }
}

// cls[i] = the slot that holds key i's value (one slot per distinct key)
__global__ void k_class_insert(const uint32_t* __restrict__ keys, uint64_t n, uint32_t* __restrict__ table,
                               uint32_t cmask, uint32_t* __restrict__ cls) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  uint32_t w[kRecWords];
#pragma unroll
  for (int k = 0; k < kRecWords; ++k) w[k] = keys[i * kRecWords + k];
  uint32_t h = (uint32_t)hash_rec(w) & cmask;
  while (true) {
    uint32_t v = __atomic_load_n(&table[h], __ATOMIC_RELAXED);
    if (v == kNone) {
      const uint32_t old = atomicCAS(&table[h], kNone, (uint32_t)i);
      if (old == kNone) { cls[i] = h; return; }
      v = old;
    }
    bool eq = true;
#pragma unroll
    for (int k = 0; k < kRecWords; ++k) eq = eq && keys[(uint64_t)v * kRecWords + k] == w[k];
    if (eq) { cls[i] = h; return; }
    h = (h + 1) & cmask;
  }
}

__device__ __forceinline__ uint32_t class_of(const LevelPtrs& P, uint32_t lev, uint32_t i,
                                             const uint32_t* __restrict__ cls) {
  return cls ? cls[i] : node_mask(P, lev, i);
}

// bestOf[class] = min over the nodes of levels 1..top of (level << 32 | index),
// at a depth with class numbers (from 1)
__global__ void k_class_best(LevelPtrs P, uint32_t top, const uint32_t* __restrict__ cls,
                             unsigned long long* __restrict__ bestOf) {
  const uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= P.base[top + 1] - P.base[1]) return;
  uint32_t j;
  const uint32_t levB = level_of(P, e + P.base[1], 1, top, j);
  const unsigned long long key = ((unsigned long long)levB << 32) | j;
  unsigned long long* b = &bestOf[cls[e]];
  if (key < __atomic_load_n(b, __ATOMIC_RELAXED)) atomicMin(b, key);
}

// The same at depth 0, where the class is the node's mask: folded in LDS
// first, as tens of thousands of nodes share a mask and the atomics of one
// address serialise (395K nodes: 142 us one by one, 8 so).
constexpr int kMaskBestT = 1024, kMaskBestGrid = 256;
__global__ void __launch_bounds__(kMaskBestT) k_mask_best(LevelPtrs P, uint32_t top,
                                                          unsigned long long* __restrict__ bestOf) {
  __shared__ unsigned long long fo[256];
  if (threadIdx.x < 256) fo[threadIdx.x] = ~0ull;
  __syncthreads();
  const uint64_t n = P.base[top + 1] - P.base[1], chunk = (n + gridDim.x - 1) / gridDim.x;
  const uint64_t lo = blockIdx.x * chunk, hi = lo + chunk < n ? lo + chunk : n;
  for (uint64_t e = lo + threadIdx.x; e < hi; e += kMaskBestT) {
    uint32_t j;
    const uint32_t levB = level_of(P, e + P.base[1], 1, top, j);
    const unsigned long long key = ((unsigned long long)levB << 32) | j;
    unsigned long long* b = &fo[node_mask(P, levB, j)];
    if (key < *b) atomicMin(b, key);
  }
  __syncthreads();
  const unsigned long long v = threadIdx.x < 256 ? fo[threadIdx.x] : ~0ull;
  if (v != ~0ull) atomicMin(&bestOf[threadIdx.x], v);
}

// Frontier nodes of levA take their class's first match; matched ones start
// the recording state (frontier index, empty path, B).
__global__ void k_frontier_best(LevelPtrs P, uint32_t levA, const uint8_t* __restrict__ front,
                                const uint32_t* __restrict__ cls, const unsigned long long* __restrict__ bestOf,
                                unsigned long long* __restrict__ best, uint32_t* __restrict__ sa,
                                uint64_t* __restrict__ sp, uint64_t* __restrict__ sb, uint32_t* __restrict__ nMatched) {
  const uint32_t a = blockIdx.x * blockDim.x + threadIdx.x;
  if (a >= P.n[levA]) return;
  unsigned long long b = ~0ull;
  if (front[a]) b = bestOf[class_of(P, levA, a, cls)];
  best[a] = b;
  sa[a] = b != ~0ull ? a : kNone;
  sp[a] = 0;
  sb[a] = b;
  // any match: the levels below are recorded (looked at first: stores of every
  // matched wavefront to the one address took up to half of the pass)
  if (b != ~0ull && !__hip_atomic_load(nMatched, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
    __hip_atomic_store(nMatched, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// One level of the recording pass: children (level lev+1) of recorded nodes.
__global__ void k_prop_min(LevelPtrs P, uint32_t lev, const uint32_t* __restrict__ sa, uint32_t* __restrict__ na) {
  const uint32_t x = blockIdx.x * blockDim.x + threadIdx.x;
  if (x >= P.n[lev]) return;
  const uint32_t a = sa[x];
  if (a == kNone) return;
  const uint32_t m = node_mask(P, lev, x);
  for (int c = 0; c < 8; ++c) {
    if (!((m >> c) & 1u)) continue;
    uint32_t* t = &na[node_child(P, lev, x, c)];
    if (a < __atomic_load_n(t, __ATOMIC_RELAXED)) atomicMin(t, a);
  }
}

__global__ void k_prop_path(LevelPtrs P, uint32_t lev, const uint32_t* __restrict__ sa, const uint64_t* __restrict__ sp,
                            const uint32_t* __restrict__ na, unsigned long long* __restrict__ np) {
  const uint32_t x = blockIdx.x * blockDim.x + threadIdx.x;
  if (x >= P.n[lev]) return;
  const uint32_t a = sa[x];
  if (a == kNone) return;
  const uint32_t m = node_mask(P, lev, x);
  const unsigned long long base = (unsigned long long)sp[x] << 3;
  for (int c = 0; c < 8; ++c) {
    if (!((m >> c) & 1u)) continue;
    const uint32_t y = node_child(P, lev, x, c);
    if (na[y] != a) continue;
    const unsigned long long v = base | (unsigned long long)c;
    if (v > __atomic_load_n(&np[y], __ATOMIC_RELAXED)) atomicMax(&np[y], v);
  }
}

__global__ void k_prop_write(LevelPtrs P, uint32_t lev, const uint32_t* __restrict__ sa, const uint64_t* __restrict__ sp,
                             const uint64_t* __restrict__ sb, const uint32_t* __restrict__ na,
                             const uint64_t* __restrict__ np, uint64_t* __restrict__ nb) {
  const uint32_t x = blockIdx.x * blockDim.x + threadIdx.x;
  if (x >= P.n[lev]) return;
  const uint32_t a = sa[x];
  if (a == kNone) return;
  const uint32_t m = node_mask(P, lev, x);
  const uint64_t base = sp[x] << 3;
  const uint32_t lb = (uint32_t)(sb[x] >> 32), b = (uint32_t)sb[x];
  for (int c = 0; c < 8; ++c) {
    if (!((m >> c) & 1u)) continue;
    const uint32_t y = node_child(P, lev, x, c);
    if (na[y] == a && np[y] == (base | (uint64_t)c))
      nb[y] = ((uint64_t)(lb + 1) << 32) | node_child(P, lb, b, c);
  }
}

// Merge this round into the global correspondence map: frontier matches of
// levA overwrite (operator[]), subtree entries only fill empty slots (insert).
__global__ void k_merge_self(uint32_t n, const uint8_t* __restrict__ front, const unsigned long long* __restrict__ best,
                             uint64_t* __restrict__ mlc, uint8_t* __restrict__ nextFront, const uint32_t* __restrict__ rec,
                             int leafLevel) {
  uint32_t a = blockIdx.x * blockDim.x + threadIdx.x;
  if (a >= n || !front[a]) return;
  if (best[a] != ~0ull) { mlc[a] = best[a]; return; }
  if (leafLevel || !nextFront) return;
  const uint32_t* r = rec + (uint64_t)a * kRecWords;
  for (int c = 0; c < 8; ++c)
    if ((r[0] >> c) & 1u) nextFront[r[1 + c]] = 1;
}

__global__ void k_merge_sub(uint64_t n, const uint64_t* __restrict__ cand, uint64_t* __restrict__ mlc) {
  const uint64_t x = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (x >= n) return;
  if (cand[x] != ~0ull && mlc[x] == ~0ull) mlc[x] = cand[x];
}

__global__ void k_fill64(uint64_t* d, uint64_t v, uint64_t n) {
  uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) d[i] = v;
}
// empty correspondences; the frontier holds level 1
__global__ void k_init(uint64_t* __restrict__ mlc, uint8_t* __restrict__ front, uint64_t n, uint64_t f0, uint64_t f1) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  mlc[i] = ~0ull;
  front[i] = i >= f0 && i < f1 ? 1 : 0;
}
// an empty recording state
__global__ void k_clear_record(uint32_t* __restrict__ sa, uint64_t* __restrict__ sp, uint64_t* __restrict__ cand,
                               uint64_t n) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  sa[i] = kNone;
  sp[i] = 0;
  cand[i] = ~0ull;
}

// ---- compaction (geom_octree_extension.cpp:1428-1498) ------------------------
// The reference compacts bottom-up and rewrites pointers after every level.
// A pointer's last value depends only on the final correspondences: a child
// with one becomes its B (level and compacted index), any other its own
// compacted index.  So all levels are numbered by one scan and written at once.
__global__ void k_keep_flags(const uint64_t* __restrict__ mlc, uint64_t n, uint32_t* __restrict__ flag) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) flag[i] = mlc[i] == ~0ull ? 1u : 0u;
}
// kept[l] = the scan at level l's start (l <= L; the total past the last level)
__global__ void k_level_starts(LevelPtrs P, uint32_t L, const uint32_t* __restrict__ pos,
                               const uint32_t* __restrict__ total, uint32_t* __restrict__ kept) {
  const uint32_t l = threadIdx.x;
  if (l <= L) kept[l] = P.base[l] < P.base[L] ? pos[P.base[l]] : *total;
}

struct OutLevels {
  uint32_t* rec[kMaxL];
  uint32_t* cl[kMaxL];
};
// pos: the scan of the keep flags; kept: its value at every level's start
__global__ void k_compact(LevelPtrs P, uint32_t L, const uint64_t* __restrict__ mlc, const uint32_t* __restrict__ pos,
                          const uint32_t* __restrict__ kept, OutLevels out, uint32_t* __restrict__ missing) {
  const uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= P.base[L] || mlc[e] != ~0ull) return;
  uint32_t i;
  const uint32_t lev = level_of(P, e, 0, L - 1, i);
  const uint32_t p = pos[e] - kept[lev];
  if (lev == P.leafLevel) { out.rec[lev][p] = P.rec[lev][i]; return; }
  const uint32_t* r = P.rec[lev] + (uint64_t)i * kRecWords;
  uint32_t* o = out.rec[lev] + (uint64_t)p * kRecWords;
  uint32_t* l = out.cl[lev] + (uint64_t)p * 8;
  const uint32_t m = r[0];
  o[0] = m;
  for (int c = 0; c < 8; ++c) {
    uint32_t v = r[1 + c], to = lev + 1;
    if ((m >> c) & 1u) {
      const uint64_t w = mlc[P.base[to] + v];
      if (w != ~0ull) { to = (uint32_t)(w >> 32); v = (uint32_t)w; }
      const uint64_t t = P.base[to] + v;
      if (mlc[t] == ~0ull) {
        v = pos[t] - kept[to];
      } else {
        v = kNone;
        atomicAdd(missing, 1u);
      }
    }
    o[1 + c] = v;
    l[c] = to;
  }
}

}  // namespace

void cross_level_merge(svd_octree* o) {
  svd_ctx* c = o->ctx;
  if (o->state != SVD_S_DAG) throw Error{SVD_ERR_STATE, "cross-level merge needs a DAG"};
  const uint32_t L = o->levels;
  if (L > kMaxL) throw Error{SVD_ERR_LEVELS, "too many levels"};
  LevelPtrs P{};
  P.leafLevel = L - 1;
  for (uint32_t l = 0; l < L; ++l) {
    P.rec[l] = o->dag[l].rec;
    P.n[l] = (uint32_t)o->dag[l].n;
    P.base[l + 1] = P.base[l] + o->dag[l].n;
  }
  const uint64_t N = P.base[L];
  uint64_t* mlc = dalloc<uint64_t>(c, N + 1);
  uint64_t* cand = dalloc<uint64_t>(c, N + 1);
  uint64_t* sp = dalloc<uint64_t>(c, N + 1);
  uint32_t* sa = dalloc<uint32_t>(c, N + 1);
  uint8_t* front = dalloc<uint8_t>(c, N + 1);
  if (N) k_init<<<div_up(N, kB), kB, 0, c->stream>>>(mlc, front, N, P.base[1], L > 1 ? P.base[2] : P.base[1]);
  // classes: cls[d] covers levels 1..L-1-d
  std::vector<uint32_t*> cls(L, nullptr);
  std::vector<uint32_t> capOf(L, 256);
  auto nodes = [&](uint32_t top) { return P.base[top + 1] - P.base[1]; };   // of levels 1..top
  if (L >= 3) {
    uint32_t* keys = dalloc<uint32_t>(c, (nodes(L - 2) + 1) * kRecWords);
    for (uint32_t d = 1; d + 2 <= L; ++d) {
      const uint32_t top = L - 1 - d;   // deepest level with d levels below it
      const uint64_t nd = nodes(top);
      uint64_t cap = 1024;
      while (cap < 2 * nd) cap <<= 1;
      if (cap > (1ull << 31)) throw Error{SVD_ERR_CAPACITY, "cross-level merge: too many nodes"};
      capOf[d] = (uint32_t)cap;
      cls[d] = dalloc<uint32_t>(c, nd + 1);
      uint32_t* table = dalloc<uint32_t>(c, cap);
      fill_u32(c, table, kNone, cap);
      if (nd) {
        k_class_keys<<<div_up(nd, kB), kB, 0, c->stream>>>(P, top, d == 1 ? nullptr : cls[d - 1], keys);
        k_class_insert<<<div_up(nd, kB), kB, 0, c->stream>>>(keys, nd, table, (uint32_t)(cap - 1), cls[d]);
      }
      check_launch("k_class");
      dfree(c, table);
    }
    dfree(c, keys);
  }

  uint32_t* matched = dalloc<uint32_t>(c, L);     // per levA: any match
  fill_u32(c, matched, 0u, L);
  for (uint32_t levA = 1; levA < L; ++levA) {
    const uint32_t D = L - 1 - levA;   // levels below A
    const uint32_t nA = P.n[levA];
    if (!nA) continue;
    const uint64_t bA = P.base[levA];
    unsigned long long* best = dalloc<unsigned long long>(c, nA);
    unsigned long long* bestOf = dalloc<unsigned long long>(c, capOf[D]);
    k_fill64<<<div_up(capOf[D], kB), kB, 0, c->stream>>>((uint64_t*)bestOf, ~0ull, capOf[D]);
    const uint32_t* cl = D ? cls[D] : nullptr;
    const uint64_t nb = nodes(levA - 1);
    if (nb && cl) k_class_best<<<div_up(nb, kB), kB, 0, c->stream>>>(P, levA - 1, cl, bestOf);
    else if (nb)
      k_mask_best<<<(uint32_t)std::min<uint64_t>(kMaskBestGrid, div_up(nb, kMaskBestT)), kMaskBestT, 0, c->stream>>>(
          P, levA - 1, bestOf);
    k_frontier_best<<<div_up(nA, kB), kB, 0, c->stream>>>(P, levA, front + bA, cl ? cl + (bA - P.base[1]) : nullptr,
                                                            bestOf, best, sa + bA, sp + bA, cand + bA, matched + levA);
    check_launch("k_frontier_best");
    if (levA + 1 < L && read_u32(c, matched + levA)) {
      const uint64_t b0 = P.base[levA + 1], nBelow = N - b0;
      if (nBelow) k_clear_record<<<div_up(nBelow, kB), kB, 0, c->stream>>>(sa + b0, sp + b0, cand + b0, nBelow);
      for (uint32_t l = levA; l + 1 < L; ++l) {
        if (!P.n[l]) continue;
        const uint32_t g = div_up(P.n[l], kB);
        const uint64_t x = P.base[l], y = P.base[l + 1];
        k_prop_min<<<g, kB, 0, c->stream>>>(P, l, sa + x, sa + y);
        k_prop_path<<<g, kB, 0, c->stream>>>(P, l, sa + x, sp + x, sa + y, (unsigned long long*)sp + y);
        k_prop_write<<<g, kB, 0, c->stream>>>(P, l, sa + x, sp + x, cand + x, sa + y, sp + y, cand + y);
        check_launch("cross-level record");
      }
      if (nBelow) k_merge_sub<<<div_up(nBelow, kB), kB, 0, c->stream>>>(nBelow, cand + b0, mlc + b0);
    }
    k_merge_self<<<div_up(nA, kB), kB, 0, c->stream>>>(nA, front + bA, best, mlc + bA,
                                                        levA + 1 < L ? front + P.base[levA + 1] : nullptr, P.rec[levA],
                                                        levA == L - 1 ? 1 : 0);
    check_launch("cross-level round");
    dfree(c, best); dfree(c, bestOf);
  }
  dfree(c, matched);
  for (auto* p : cls) dfree(c, p);

  // compaction: kept counts of every level (one read), then every level at once
  uint32_t* pos = dalloc<uint32_t>(c, N + 1);
  uint32_t* kept = dalloc<uint32_t>(c, L + 2);
  uint32_t* missing = dalloc<uint32_t>(c, 2);     // and the scan's total
  fill_u32(c, missing, 0u, 2);
  if (N) k_keep_flags<<<div_up(N, kB), kB, 0, c->stream>>>(mlc, N, pos);
  scan_exclusive(c, pos, pos, N, missing + 1);
  k_level_starts<<<1, 64, 0, c->stream>>>(P, L, pos, missing + 1, kept);
  check_launch("k_level_starts");
  std::vector<uint32_t> h(L + 1);
  read_u32s(c, kept, h.data(), L + 1);
  std::vector<Level> X(L);
  OutLevels out{};
  uint64_t nNodes = 1, merged = 0;
  for (uint32_t l = 0; l < L; ++l) {
    Level& x = X[l];
    x.n = h[l + 1] - h[l];
    x.leaf = o->dag[l].leaf;
    x.rec = dalloc<uint32_t>(c, (x.leaf ? x.n : x.n * kRecWords) + 1);
    if (!x.leaf) x.childLevels = dalloc<uint32_t>(c, 8 * x.n + 1);
    out.rec[l] = x.rec;
    out.cl[l] = x.childLevels;
    if (l) { nNodes += x.n; merged += P.n[l] - x.n; }
  }
  if (N) k_compact<<<div_up(N, kB), kB, 0, c->stream>>>(P, L, mlc, pos, kept, out, missing);
  check_launch("k_compact");
  const uint64_t nMissing = read_u32(c, missing);
  // replace the cross-level view
  for (auto& lv : o->xdag) { dfree(c, lv.rec); dfree(c, lv.childLevels); }
  o->xdag = X;
  o->hasX = true;
  o->nNodesX = nNodes;
  o->crossMerged = merged;
  dfree(c, mlc); dfree(c, cand); dfree(c, sp); dfree(c, sa); dfree(c, front);
  dfree(c, pos); dfree(c, kept); dfree(c, missing);
  for (auto& e : o->enc) e.valid = false;
  if (nMissing)
    throw Error{SVD_ERR_POINTER, "cross-level merge: " + std::to_string(nMissing) +
                                     " pointer(s) to a removed node (the reference prints 'Missing correspondence')"};
}

}  // namespace svd
