// Lossy DAG (LSVDAG) on the device: GeomOctree::toLossyDag
// (geom_octree_extension.cpp:797-1179) with a deterministic clustering rule in
// place of the reference's external MCL run (cluster.hpp:134-192).
//
// Per merged level (lev_hi down to lev_lo, bottom-up as in :882):
//   1. signatures: 512-bit occupancy of each node's cells three levels down
//      (bit c1*64 + c2*8 + c3 for the child-slot path; voxels at level L-3);
//   2. lists: for each candidate j (effective reference count <= max_refs,
//      :945) the first list_cap earlier nodes i < j with
//      popcount(sig_i ^ sig_j) <= bound -- exhaustively (all pairs inside the
//      bound's popcount window, their distances as a GEMM on the matrix
//      cores), or the list_cap nearest of them by (popcount, i) (ranked, an
//      LDS-tiled XOR-popcount scan), or among the learned proposals (kNN of
//      the MLP embeddings, sorted and de-duplicated);
//   3. verify: exact voxel difference of the two subtrees by a joint descent
//      with early abort that ends at 512-bit occupancies (the Hamming distance
//      above is a lower bound of it);
//   4. resolve: j walks its verified entries in order; a representative
//      becomes its target, an entry that merged earlier offers its own target
//      (taken when the exact difference to j is within the bound); resolved
//      in monotone rounds (each round settles at least the smallest
//      unresolved node, so the loop ends);
//   5. compact the level, remap the parent level's child pointers.
// Finally the whole DAG is re-deduplicated exactly (:1176).
#include <algorithm>
#include <type_traits>
#include "svd_internal.hpp"
#include <rocprim/device/device_radix_sort.hpp>

namespace svd {

namespace {

constexpr int kB = 256;
constexpr uint32_t kRounds = 3;      // resolution rounds between two looks at the unresolved flag
constexpr uint8_t kUnres = 0, kRep = 1, kMerged = 2;

struct LevelView {
  const uint32_t* rec[kMaxLevels];
  const uint64_t* vox[kMaxLevels];
  const uint32_t* occ;            // 512-bit occupancies (16 words) of every node of level occLev
  uint32_t occLev;
  uint32_t L;
};

__device__ __forceinline__ uint32_t mask_of(const LevelView& v, uint32_t lev, uint32_t n) {
  return (lev == v.L - 1 ? v.rec[lev][n] : v.rec[lev][(uint64_t)n * kRecWords]) & 0xFFu;
}
__device__ __forceinline__ uint32_t child_of(const LevelView& v, uint32_t lev, uint32_t n, int c) {
  return v.rec[lev][(uint64_t)n * kRecWords + 1 + c];
}

__global__ void k_fill_u64(uint64_t* d, uint64_t v, uint64_t n) {
  uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) d[i] = v;
}

// refs[child] += refs[parent] for every existing child (sortByEffectiveRefCount, :527-537)
__global__ void k_refs_level(const uint32_t* __restrict__ prec, uint64_t np, const uint64_t* __restrict__ pref,
                             unsigned long long* __restrict__ cref) {
  uint64_t p = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= np) return;
  const uint32_t* r = prec + p * kRecWords;
  const uint32_t m = r[0] & 0xFFu;
  const uint64_t v = pref[p];
  if (!v) return;
  for (int c = 0; c < 8; ++c)
    if (((m >> c) & 1u) && r[1 + c] != kNull) atomicAdd(&cref[r[1 + c]], (unsigned long long)v);
}

__global__ void k_vox_level(const uint32_t* __restrict__ rec, uint64_t n, int leaf, const uint64_t* __restrict__ cvox,
                            uint64_t* __restrict__ vox) {
  uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  if (leaf) { vox[i] = (uint64_t)__popc(rec[i] & 0xFFu); return; }
  const uint32_t* r = rec + i * kRecWords;
  const uint32_t m = r[0] & 0xFFu;
  uint64_t s = 0;
  for (int c = 0; c < 8; ++c)
    if ((m >> c) & 1u) s += cvox[r[1 + c]];
  vox[i] = s;
}

// 512-bit occupancies: the voxels of a node three levels down, bit c1 * 64 +
// c2 * 8 + c3.  Eight lanes per node, one per child: lane c1 reads the child's
// record and its children's masks in two round trips and stores words 2 c1 and
// 2 c1 + 1, so a wavefront stores whole lines.  One lane per node walked its 64
// grandchildren one load after the other (466K nodes 60 -> 33 us, 10K nodes 51 -> 9).
__global__ void k_signatures(LevelView v, uint32_t lev, uint64_t n, uint32_t* __restrict__ sig) {
  const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x, i = t >> 3;
  if (i >= n) return;                              // n * 8 lanes: a node's eight stay together
  const uint32_t c1 = (uint32_t)t & 7u;
  const bool in = (mask_of(v, lev, (uint32_t)i) >> c1) & 1u;
  uint64_t s = 0;
  if (lev + 2 < v.L) {
    if (in) {
      const uint32_t* b = v.rec[lev + 1] + (uint64_t)child_of(v, lev, (uint32_t)i, (int)c1) * kRecWords;
      uint32_t w[kRecWords], md[8];
#pragma unroll
      for (int k = 0; k < kRecWords; ++k) w[k] = b[k];
#pragma unroll
      for (int c2 = 0; c2 < 8; ++c2) md[c2] = ((w[0] >> c2) & 1u) ? mask_of(v, lev + 2, w[1 + c2]) : 0u;
#pragma unroll
      for (int c2 = 0; c2 < 8; ++c2) s |= (uint64_t)md[c2] << (8 * c2);
    }
  } else {                                         // one or two levels: bit c1, or byte c1, of the first 64 bits
    if (in) s = lev + 1 >= v.L ? 1ull << c1
                               : (uint64_t)mask_of(v, lev + 1, child_of(v, lev, (uint32_t)i, (int)c1)) << (8 * c1);
#pragma unroll
    for (int off = 1; off < 8; off <<= 1)
      s |= (uint64_t)__shfl_xor((uint32_t)(s >> 32), off, 64) << 32 | __shfl_xor((uint32_t)s, off, 64);
    if (c1) s = 0;
  }
  *reinterpret_cast<uint2*>(sig + i * 16 + 2 * c1) = make_uint2((uint32_t)s, (uint32_t)(s >> 32));
}

__device__ __forceinline__ uint32_t hamming512(const uint4* a, const uint32_t s[16]) {
  uint32_t h = 0;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const uint4 t = a[q];
    h += __popc(t.x ^ s[4 * q]) + __popc(t.y ^ s[4 * q + 1]) + __popc(t.z ^ s[4 * q + 2]) + __popc(t.w ^ s[4 * q + 3]);
  }
  return h;
}

typedef int i32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));

// One signature word as 32 fp4 (e2m1) values of a matrix operand: bit 4p + d
// becomes nibble p of dword d, 0 -> +1.0 (0x2), 1 -> -1.0 (0xA).  The order of
// the 512 positions along K is free as long as both operands share it.
__device__ __forceinline__ i32x4_t bits_to_fp4(uint32_t w) {
  constexpr uint32_t kOne = 0x22222222u, kSign = 0x88888888u;
  i32x4_t r;
  r[0] = (int)(((w << 3) & kSign) | kOne);
  r[1] = (int)(((w << 2) & kSign) | kOne);
  r[2] = (int)(((w << 1) & kSign) | kOne);
  r[3] = (int)((w & kSign) | kOne);
  return r;
}

// Order of the exhaustive scan: chunks of C consecutive nodes, by popcount
// within a chunk (stable).  Key = chunk * 513 + popcount.
constexpr uint32_t kPopBins = 513;
__global__ void k_list_keys(const uint32_t* __restrict__ sig, uint64_t n, uint32_t C, uint32_t* __restrict__ keys,
                            uint32_t* __restrict__ ids) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint4* p = reinterpret_cast<const uint4*>(sig + i * 16);
  uint32_t pc = 0;
#pragma unroll
  for (int q = 0; q < 4; ++q) { const uint4 t = p[q]; pc += __popc(t.x) + __popc(t.y) + __popc(t.z) + __popc(t.w); }
  keys[i] = (uint32_t)i / C * kPopBins + pc;
  ids[i] = (uint32_t)i;
}

// Signatures in scan order (four lanes each), and off[key] = the first
// position whose key is at least key (nKeys + 1 entries).
__global__ void k_list_gather(const uint32_t* __restrict__ sig, const uint32_t* __restrict__ ids,
                              const uint32_t* __restrict__ keys, uint64_t n, uint32_t nKeys,
                              uint4* __restrict__ ssig, uint32_t* __restrict__ off) {
  const uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const uint64_t p = e >> 2;
  if (p >= n) return;
  ssig[e] = reinterpret_cast<const uint4*>(sig + (uint64_t)ids[p] * 16)[e & 3];
  if (e & 3) return;
  const uint32_t key = keys[p];
  for (uint32_t k = p ? keys[p - 1] + 1 : 0; k <= key; ++k) off[k] = (uint32_t)p;
  if (p == n - 1)
    for (uint32_t k = key + 1; k <= nKeys; ++k) off[k] = (uint32_t)n;
}

// The entries of one j's list, cap in lists and cap more in spill, in no
// order, two per lane of a wavefront (at most 2 cap <= 128 of them).
__device__ __forceinline__ void load_list(const uint32_t* lists, const uint32_t* spill, uint64_t at, uint32_t cnt,
                                          uint32_t cap, int lane, uint32_t v[2]) {
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const uint32_t e = (uint32_t)lane + 64 * h;
    const uint32_t* p = e < cap ? lists + at + e : spill + at + (e - cap);
    v[h] = e < cnt ? __atomic_load_n(p, __ATOMIC_RELAXED) : kNone;
  }
}
// Their smallest cap go to lists, ascending.  Returns the largest one kept.
__device__ __forceinline__ uint32_t order_list(uint32_t* lists, uint64_t at, uint32_t cnt, uint32_t cap,
                                               const uint32_t v[2]) {
  uint32_t rank[2] = {0, 0};
  const int m = (int)(cnt < 64u ? cnt : 64u);
  for (int r = 0; r < m; ++r) {
    const uint32_t a = (uint32_t)__builtin_amdgcn_readlane((int)v[0], r);
    rank[0] += a < v[0] ? 1u : 0u;
    rank[1] += a < v[1] ? 1u : 0u;
  }
  for (int r = 64; r < (int)cnt; ++r) {
    const uint32_t a = (uint32_t)__builtin_amdgcn_readlane((int)v[1], r - 64);
    rank[0] += a < v[0] ? 1u : 0u;
    rank[1] += a < v[1] ? 1u : 0u;
  }
  const uint32_t keep = cnt < cap ? cnt : cap;
  uint32_t last = 0;
#pragma unroll
  for (int h = 0; h < 2; ++h)
    if (v[h] != kNone && rank[h] < keep) {
      lists[at + rank[h]] = v[h];
      if (rank[h] == keep - 1) last = v[h];
    }
  const unsigned long long w = __ballot(last != 0);   // one lane at most: node 0 alone gives 0
  return w ? (uint32_t)__builtin_amdgcn_readlane((int)last, __ffsll(w) - 1) : 0u;
}

// Exhaustive pre-filter lists on the matrix cores.  With bits as +-1 the dot
// product of two signatures is 512 - 2 Hamming, so popcount(a ^ b) <= bound is
// one comparison of an fp32 sum of +-1 (exact) with 512 - 2 bound, and the
// scan is a GEMM of fp4 operands (v_mfma_f32_32x32x64_f8f6f4: 8 of them per
// 32 x 32 pairs) that never leaves the registers.
//  - |popcount(a) - popcount(b)| <= Hamming: chunk by chunk in node order, a
//    workgroup's j (32 JT per wavefront, expanded as its B operand) meet only
//    the nodes whose popcount is within the bound of theirs.  Chunks keep the
//    scan to earlier nodes and let a j stop once the chunks behind it hold
//    cap matches (16 of them, or fewer of at least 512 nodes: on 10K nodes
//    0.30 ms against 0.46 ms for one chunk, on 466K nodes 4 to 64 chunks
//    measure the same).
//  - i streams through LDS in stages of 256 signatures, still as bits (rows
//    padded to 80 bytes: the 16-byte reads of eight lanes fall in distinct
//    banks), expanded as they are read (8 VALU operations per 32 positions).
//  - Accumulator element v of lane l is pair (i = 8 (v/4) + 4 (l/32) + v%4,
//    j = l%32) of a tile.  Matches are appended unordered, 2 cap of them at
//    most before the smallest cap are kept; k_list_order sorts at the end.
//  - Later j have more to scan, so the last workgroups start first.
// Bound by the matrix cores: on 466K nodes of the 2048^3 caves (bound 10, 36%
// of the pairs inside the popcount window) 8.6 - 9.0 ms at 66% of the MFMA cycles,
// against 19.3 ms without the window and 172 ms for an XOR/popcount scan.
template <int JT>
__global__ void __launch_bounds__(256, 3)
k_exhaustive_lists(const uint4* __restrict__ ssig, const uint32_t* __restrict__ ids, const uint32_t* __restrict__ keys,
                   const uint32_t* __restrict__ off, uint32_t n, uint32_t C, const uint64_t* __restrict__ refs,
                   uint64_t maxRefs, uint32_t bound, uint32_t cap, uint32_t* lists, uint32_t* spill,
                   uint32_t* __restrict__ counts) {
  constexpr int kStage = 256, kRow = 20;         // signatures per stage, dwords per LDS row
  __shared__ __attribute__((aligned(16))) uint32_t tile[2][kStage * kRow];
  __shared__ uint32_t tileId[2][kStage], tileMin[2][kStage / 32];   // node ids, the smallest of each 32
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, col = lane & 31, half = lane >> 5;
  const uint32_t j0 = (gridDim.x - 1 - blockIdx.x) * (128 * JT);
  const uint32_t jw = j0 + wave * (32 * JT);     // the wavefront's first position
  const float limit = bound >= 512u ? -513.f : 512.f - 2.f * (float)bound;
  i32x4_t b[JT][8];
  float thr[JT];                                 // +inf: inactive or full
  uint32_t cnt[JT], jid[JT], top[JT];            // matches held, node id, ids from top on are not needed
#pragma unroll
  for (int t = 0; t < JT; ++t) {
    const uint32_t j = jw + 32 * t + col;
    uint4 lo = make_uint4(0, 0, 0, 0), hi = lo;
    jid[t] = 0;
    if (j < n) {
      lo = ssig[(uint64_t)j * 4 + 2 * half];
      hi = ssig[(uint64_t)j * 4 + 2 * half + 1];
      jid[t] = ids[j];
    }
    const uint32_t w[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
#pragma unroll
    for (int k = 0; k < 8; ++k) b[t][k] = bits_to_fp4(w[k]);
    thr[t] = j < n && refs[jid[t]] <= maxRefs ? limit : __builtin_inff();
    cnt[t] = 0;
    top[t] = jid[t];
  }
  // 128 JT divides C: a workgroup's positions are of one chunk
  const uint32_t ch = j0 / C;
  const uint32_t jl = min(j0 + 128 * JT, n) - 1;
  const uint32_t pcLo = keys[j0] - ch * kPopBins, pcHi = keys[jl] - ch * kPopBins;
  const uint32_t binLo = pcLo > bound ? pcLo - bound : 0;
  const uint32_t binHi = bound >= 512u - pcHi ? 512u : pcHi + bound;
  int buf = 0;
  for (uint32_t q = 0; q <= ch; ++q) {
    bool live = false;
#pragma unroll
    for (int t = 0; t < JT; ++t) {
      if (cnt[t] >= cap) thr[t] = __builtin_inff();   // every later match has a larger id
      live |= thr[t] < __builtin_inff();
    }
    live = __any(live) != 0;
    const uint32_t iBeg = off[q * kPopBins + binLo], iEnd = off[q * kPopBins + binHi + 1];
    uint4 r[4];
    uint32_t rid = 0;
    auto load = [&](uint32_t i0) {
      const uint32_t i = i0 + tid;
#pragma unroll
      for (int x = 0; x < 4; ++x) r[x] = i < iEnd ? ssig[(uint64_t)i * 4 + x] : make_uint4(0, 0, 0, 0);
      rid = i < iEnd ? ids[i] : kNone;
    };
    load(iBeg);
    for (uint32_t i0 = iBeg; i0 < iEnd; i0 += kStage, buf ^= 1) {
      uint4* d = reinterpret_cast<uint4*>(&tile[buf][tid * kRow]);
#pragma unroll
      for (int x = 0; x < 4; ++x) d[x] = r[x];
      tileId[buf][tid] = rid;
      uint32_t mn = rid;
#pragma unroll
      for (int o = 16; o >= 1; o >>= 1) mn = min(mn, (uint32_t)__shfl_xor(mn, o, 64));
      if (col == 0) tileMin[buf][tid >> 5] = mn;
      if (!__syncthreads_or(live)) break;
      if (i0 + kStage < iEnd) load(i0 + kStage);
      if (!live) continue;
      for (uint32_t base = i0; base < i0 + kStage && base < iEnd; base += 32) {
        const uint4* a4 = reinterpret_cast<const uint4*>(&tile[buf][(base - i0 + col) * kRow + 8 * half]);
        const uint4 lo = a4[0], hi = a4[1];
        const uint32_t w[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
        f32x16_t acc[JT];
#pragma unroll
        for (int t = 0; t < JT; ++t)
#pragma unroll
          for (int v = 0; v < 16; ++v) acc[t][v] = 0.f;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          const i32x4_t a = bits_to_fp4(w[k]);
#pragma unroll
          for (int t = 0; t < JT; ++t)
            acc[t] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(
                __builtin_shufflevector(a, a, 0, 1, 2, 3, -1, -1, -1, -1),
                __builtin_shufflevector(b[t][k], b[t][k], 0, 1, 2, 3, -1, -1, -1, -1), acc[t], 4, 4, 0, 0, 0, 0);
        }
        const uint32_t least = tileMin[buf][(base - i0) >> 5];
        const uint32_t rows = iEnd - base < 32 ? (1u << (iEnd - base)) - 1u : 0xFFFFFFFFu;
#pragma unroll
        for (int t = 0; t < JT; ++t) {
          float m = acc[t][0];
#pragma unroll
          for (int v = 1; v < 16; ++v) m = fmaxf(m, acc[t][v]);
          const float th = least < top[t] ? thr[t] : __builtin_inff();
          if (!__any(m >= th)) continue;
          uint32_t hits = 0;
#pragma unroll
          for (int v = 0; v < 16; ++v) hits |= (acc[t][v] >= th ? 1u : 0u) << (8 * (v >> 2) + (v & 3));
          hits <<= 4 * half;
          hits |= __shfl_xor(hits, 32, 64);
          hits &= rows;
          const uint64_t at = (uint64_t)jid[t] * cap;
          while (true) {
            while (hits && cnt[t] < 2 * cap) {
              const uint32_t id = tileId[buf][base - i0 + (uint32_t)(__ffs(hits) - 1)];
              hits &= hits - 1;
              if (id < top[t]) {
                if (half == 0)
                  __atomic_store_n(cnt[t] < cap ? lists + at + cnt[t] : spill + at + (cnt[t] - cap), id,
                                   __ATOMIC_RELAXED);
                ++cnt[t];
              }
            }
            unsigned long long f = __ballot(half == 0 && cnt[t] == 2 * cap);
            if (!f) break;
            // full lists keep their smallest cap entries; four are loaded at a time
            __threadfence_block();
            while (f) {
              int l[4];
              uint32_t v[4][2];
#pragma unroll
              for (int x = 0; x < 4; ++x) {
                l[x] = f ? __ffsll(f) - 1 : -1;
                f &= f - 1;                                 // 0 stays 0
                if (l[x] >= 0)
                  load_list(lists, spill, (uint64_t)__builtin_amdgcn_readlane((int)jid[t], l[x]) * cap, 2 * cap, cap,
                            lane, v[x]);
              }
#pragma unroll
              for (int x = 0; x < 4; ++x) {
                if (l[x] < 0) break;
                const uint32_t last = order_list(
                    lists, (uint64_t)__builtin_amdgcn_readlane((int)jid[t], l[x]) * cap, 2 * cap, cap, v[x]);
                if (col == l[x]) { cnt[t] = cap; top[t] = last; }
              }
            }
            __threadfence_block();
          }
        }
      }
    }
  }
#pragma unroll
  for (int t = 0; t < JT; ++t) {
    const uint32_t j = jw + 32 * t + col;
    if (half == 0 && j < n) counts[jid[t]] = cnt[t];
  }
}

// Every list in ascending order, cut to cap: one wavefront per node.
__global__ void __launch_bounds__(256) k_list_order(uint64_t n, uint32_t cap, uint32_t* lists, uint32_t* spill,
                                                    uint32_t* counts) {
  const uint64_t j = (uint64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (j >= n) return;
  const int lane = threadIdx.x & 63;
  const uint32_t cnt = counts[j];
  if (cnt > 1) {
    uint32_t v[2];
    load_list(lists, spill, j * cap, cnt, cap, lane, v);
    order_list(lists, j * cap, cnt, cap, v);
  }
  if (cnt > cap && lane == 0) counts[j] = cap;
}

// Ranked pre-filter lists: every earlier node i < j within the bound, the K
// nearest kept by (hamming << 32 | i) in a sorted register list (an insertion
// bubbles the new key in and drops the largest).  Block = 256 consecutive j;
// the earlier nodes are streamed through LDS in tiles of 256 signatures (16
// KB) that every lane reads in the same order (LDS broadcast), to the end (no
// early stop).
template <int K>
__global__ void __launch_bounds__(256) k_ranked_lists(const uint32_t* __restrict__ sig, uint64_t n,
                                                      const uint64_t* __restrict__ refs, uint64_t maxRefs,
                                                      uint32_t bound, uint32_t cap, uint32_t* __restrict__ lists,
                                                      uint32_t* __restrict__ counts) {
  __shared__ uint4 tile[256 * 4];
  const uint64_t j0 = (uint64_t)blockIdx.x * 256;
  const uint64_t j = j0 + threadIdx.x;
  const bool active = j < n && refs[j] <= maxRefs;
  uint32_t s[16];
  if (j < n) {
    const uint4* p = reinterpret_cast<const uint4*>(sig + j * 16);
#pragma unroll
    for (int q = 0; q < 4; ++q) { const uint4 t = p[q]; s[4 * q] = t.x; s[4 * q + 1] = t.y; s[4 * q + 2] = t.z; s[4 * q + 3] = t.w; }
  }
  unsigned long long top[K];
#pragma unroll
  for (int q = 0; q < K; ++q) top[q] = ~0ull;
  uint32_t cnt = 0;
  const uint64_t jend = j0 + 256 < n ? j0 + 256 : n;
  for (uint64_t i0 = 0; i0 < jend; i0 += 256) {
    if (!__syncthreads_or(active)) break;
    for (int q = threadIdx.x; q < 256 * 4; q += 256) {
      const uint64_t i = i0 + (q >> 2);
      tile[q] = i < n ? reinterpret_cast<const uint4*>(sig + i * 16)[q & 3] : make_uint4(0, 0, 0, 0);
    }
    __syncthreads();
    if (active) {
      const uint64_t iend = i0 + 256 < j ? i0 + 256 : j;
      for (uint64_t i = i0; i < iend; ++i) {
        const uint32_t h = hamming512(&tile[(i - i0) * 4], s);
        if (h > bound) continue;
        unsigned long long x = ((unsigned long long)h << 32) | (unsigned long long)i;
        if (x >= top[K - 1]) continue;
#pragma unroll
        for (int q = 0; q < K; ++q) {
          const unsigned long long t = top[q];
          const bool lt = x < t;
          top[q] = lt ? x : t;
          x = lt ? t : x;
        }
        ++cnt;
      }
    }
    __syncthreads();
  }
  if (j >= n) return;
  const uint32_t m = active ? min(cnt, cap) : 0u;
#pragma unroll
  for (int q = 0; q < K; ++q)
    if ((uint32_t)q < m) lists[j * cap + q] = (uint32_t)top[q];
  counts[j] = m;
}

// Learned proposals -> keys hi << nb | lo (nodes below 2^nb); invalid entries
// get the bit above, so that the sort reads 2 nb + 1 bits.
__global__ void k_proposal_keys(const uint32_t* __restrict__ knn, uint64_t n, uint32_t k,
                                const uint32_t* __restrict__ sig, const uint64_t* __restrict__ refs, uint64_t maxRefs,
                                uint32_t bound, int nb, uint64_t* __restrict__ keys) {
  uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= n * k) return;
  const uint64_t x = e / k;
  const uint32_t y = knn[e];
  uint64_t key = 1ull << (2 * nb);
  if (y != kNone && (uint64_t)y != x && (uint64_t)y < n) {
    const uint64_t lo = x < y ? x : y, hi = x < y ? y : x;
    if (refs[hi] <= maxRefs) {
      uint32_t s[16];
      const uint4* p = reinterpret_cast<const uint4*>(sig + hi * 16);
#pragma unroll
      for (int q = 0; q < 4; ++q) { const uint4 t = p[q]; s[4 * q] = t.x; s[4 * q + 1] = t.y; s[4 * q + 2] = t.z; s[4 * q + 3] = t.w; }
      if (hamming512(reinterpret_cast<const uint4*>(sig + lo * 16), s) <= bound) key = (hi << nb) | lo;
    }
  }
  keys[e] = key;
}

// Sorted keys -> per hi node its first cap distinct lo (ascending).
__global__ void k_lists_from_sorted(const uint64_t* __restrict__ keys, uint64_t m, uint32_t cap, int nb,
                                    uint32_t* __restrict__ lists, uint32_t* __restrict__ counts) {
  uint64_t p = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= m) return;
  const uint64_t key = keys[p];
  if (key >> (2 * nb)) return;
  const uint64_t hi = key >> nb;
  if (p > 0 && (keys[p - 1] >> nb) == hi) return;
  uint32_t cnt = 0;
  uint64_t prev = ~0ull;
  for (uint64_t q = p; q < m && cnt < cap; ++q) {
    const uint64_t kq = keys[q];
    if ((kq >> nb) != hi) break;           // an invalid key's is above every node
    if (kq != prev) { lists[hi * cap + cnt++] = (uint32_t)(kq & ((1ull << nb) - 1)); prev = kq; }
  }
  counts[hi] = cnt;
}

__device__ __forceinline__ uint32_t occ_diff(const LevelView& v, uint32_t a, uint32_t b) {
  const uint4* pa = reinterpret_cast<const uint4*>(v.occ + (uint64_t)a * 16);
  const uint4* pb = reinterpret_cast<const uint4*>(v.occ + (uint64_t)b * 16);
  uint32_t h = 0;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const uint4 x = pa[q], y = pb[q];
    h += __popc(x.x ^ y.x) + __popc(x.y ^ y.y) + __popc(x.z ^ y.z) + __popc(x.w ^ y.w);
  }
  return h;
}

// Adds the voxel difference of the subtrees a, b (level lev, D levels above
// v.occLev) to acc; true once it exceeds the bound.  One nested loop per level
// keeps every index in registers.
template <int D>
__device__ __forceinline__ bool add_diff(const LevelView& v, uint32_t lev, uint32_t a, uint32_t b, uint32_t bound,
                                         uint64_t& acc) {
  if constexpr (D == 0) {
    acc += occ_diff(v, a, b);
  } else {
    const uint32_t* ra = v.rec[lev] + (uint64_t)a * kRecWords;
    const uint32_t* rb = v.rec[lev] + (uint64_t)b * kRecWords;
    const uint32_t ma = ra[0] & 0xFFu, mb = rb[0] & 0xFFu;
    for (uint32_t m = ma ^ mb; m; m &= m - 1) {          // one-sided children
      const int c = __ffs(m) - 1;
      acc += v.vox[lev + 1][((ma >> c) & 1u) ? ra[1 + c] : rb[1 + c]];
    }
    if (acc > bound) return true;
    for (uint32_t m = ma & mb; m; m &= m - 1) {
      const int c = __ffs(m) - 1;
      const uint32_t ca = ra[1 + c], cb = rb[1 + c];
      if (ca != cb && add_diff<D - 1>(v, lev + 1, ca, cb, bound, acc)) return true;
    }
  }
  return acc > bound;
}

// The same for any depth, with the path on a stack.
__device__ bool add_diff_deep(const LevelView& v, uint32_t lev0, uint32_t a0, uint32_t b0, uint32_t bound,
                              uint64_t& acc) {
  uint32_t sa[kMaxLevels], sb[kMaxLevels];
  uint8_t sc[kMaxLevels];
  int top = 0;
  sa[0] = a0; sb[0] = b0; sc[0] = 0;
  while (top >= 0) {
    const uint32_t lev = lev0 + (uint32_t)top;     // < occLev for every frame on the stack
    const uint32_t a = sa[top], b = sb[top];
    const uint32_t ma = mask_of(v, lev, a), mb = mask_of(v, lev, b);
    int c = sc[top];
    bool pushed = false;
    for (; c < 8 && !pushed; ++c) {
      const bool ea = (ma >> c) & 1u, eb = (mb >> c) & 1u;
      if (ea && eb) {
        const uint32_t ca = child_of(v, lev, a, c), cb = child_of(v, lev, b, c);
        if (ca == cb) continue;
        if (lev + 1 == v.occLev) {
          acc += occ_diff(v, ca, cb);
        } else {
          sc[top] = (uint8_t)(c + 1);
          ++top;
          sa[top] = ca; sb[top] = cb; sc[top] = 0;
          pushed = true;
        }
      } else if (ea || eb) {
        acc += v.vox[lev + 1][child_of(v, lev, ea ? a : b, c)];
      }
      if (acc > bound) return true;
    }
    if (!pushed) --top;
  }
  return false;
}

// Exact voxel difference of the subtrees a, b at level lev, capped at bound +
// 1 (the running total only grows, so the capped value does not depend on the
// visiting order).  The descent ends at level occLev: three levels above the
// bottom a node's occupancy is its voxels, so the difference of two such nodes
// is one 64-byte XOR/popcount instead of up to 73 records.  D = occLev - lev
// for up to kMaxD levels (0 from occLev down), D = kDeep beyond.
constexpr int kMaxD = 4, kDeep = kMaxD + 1;
template <int D>
__device__ __forceinline__ uint32_t subtree_diff(const LevelView& v, uint32_t lev, uint32_t a, uint32_t b,
                                                 uint32_t bound) {
  if (a == b) return 0;
  uint64_t acc = 0;
  bool over;
  if constexpr (D == kDeep) over = add_diff_deep(v, lev, a, b, bound, acc);
  else over = add_diff<D>(v, lev, a, b, bound, acc);
  return over ? bound + 1 : (uint32_t)acc;
}

// Sums of a workgroup of 256 added to two words, one atomic each: a grid
// strides over its work so that few workgroups meet at the address.
__device__ __forceinline__ void add_block(unsigned long long a, unsigned long long b, unsigned long long* da,
                                          unsigned long long* db) {
  __shared__ unsigned long long part[2][4];
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    a += __shfl_xor(a, o, 64);
    b += __shfl_xor(b, o, 64);
  }
  if ((threadIdx.x & 63) == 0) { part[0][threadIdx.x >> 6] = a; part[1][threadIdx.x >> 6] = b; }
  __syncthreads();
  if (threadIdx.x == 0) {
    a = part[0][0] + part[0][1] + part[0][2] + part[0][3];
    b = part[1][0] + part[1][1] + part[1][2] + part[1][3];
    if (a) atomicAdd(da, a);
    if (b) atomicAdd(db, b);
  }
}

template <int D>
__global__ void __launch_bounds__(256) k_verify(LevelView v, uint32_t lev, const uint32_t* __restrict__ lists,
                                                const uint32_t* __restrict__ counts, uint64_t n, uint32_t cap,
                                                uint32_t bound, uint32_t* __restrict__ dv,
                                                unsigned long long* __restrict__ stats) {
  unsigned long long listed = 0, kept = 0;
  for (uint64_t e = (uint64_t)blockIdx.x * 256 + threadIdx.x; e < n * cap; e += (uint64_t)gridDim.x * 256) {
    const uint64_t j = e / cap;
    const uint32_t t = (uint32_t)(e - j * cap);
    if (t >= counts[j]) continue;
    const uint32_t d = subtree_diff<D>(v, lev, lists[e], (uint32_t)j, bound);
    dv[e] = d;
    ++listed;
    kept += d <= bound ? 1 : 0;
  }
  add_block(listed, kept, &stats[0], &stats[1]);
}

// Node state word: state << 32 | target node (one 64-bit word, so a reader
// that sees "merged" also sees the target).
constexpr uint64_t kStRep = (uint64_t)kRep << 32, kStMerged = (uint64_t)kMerged << 32;

__global__ void __launch_bounds__(256) k_resolve_init(uint64_t n, const uint64_t* __restrict__ refs, uint64_t maxRefs,
                                                      unsigned long long* __restrict__ st,
                                                      uint32_t* __restrict__ tdist,
                                                      unsigned long long* __restrict__ stats) {
  unsigned long long cands = 0;
  for (uint64_t j = (uint64_t)blockIdx.x * 256 + threadIdx.x; j < n; j += (uint64_t)gridDim.x * 256) {
    const bool cand = refs[j] <= maxRefs;
    st[j] = cand ? (unsigned long long)kUnres << 32 : (unsigned long long)(kStRep | j);
    tdist[j] = 0;              // the walk's place in the list while j is unresolved
    cands += cand ? 1 : 0;
  }
  add_block(cands, 0, &stats[2], &stats[2]);
}

// One round: an unresolved j walks its verified entries in order.  A
// representative becomes its target; an entry that merged offers its own
// target (a representative), taken when the exact difference to j is within
// the bound; an unresolved entry makes j wait.  States only move away from
// "unresolved", so a stale read delays a node by one round and never changes
// its outcome, and an entry that was passed over stays passed over: j resumes
// where it waited (tdist[j] holds that place until j has its target).  The
// longest walk of dependent reads bounds a round, so four entries are read at a
// time, with (D == 0) the targets' occupancies.  *unresolved is set while a node waits.
template <int D>
__global__ void k_resolve(LevelView v, uint32_t lev, const uint32_t* __restrict__ lists,
                          const uint32_t* __restrict__ dv, const uint32_t* __restrict__ counts, uint64_t n,
                          uint32_t cap, uint32_t bound, unsigned long long* st, uint32_t* __restrict__ tdist,
                          uint32_t* __restrict__ unresolved) {
  uint64_t j = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= n) return;
  if ((__atomic_load_n(&st[j], __ATOMIC_RELAXED) >> 32) != kUnres) return;
  constexpr uint32_t kAhead = 4;
  const uint32_t cnt = counts[j];
  uint32_t own[16];
  if constexpr (D == 0) {
    const uint4* o = reinterpret_cast<const uint4*>(v.occ + j * 16);
#pragma unroll
    for (int q = 0; q < 4; ++q) { const uint4 x = o[q]; own[4 * q] = x.x; own[4 * q + 1] = x.y; own[4 * q + 2] = x.z; own[4 * q + 3] = x.w; }
  }
  for (uint32_t t = tdist[j]; t < cnt; t += kAhead) {
    uint32_t dd[kAhead], ii[kAhead];
    unsigned long long ww[kAhead];
#pragma unroll
    for (uint32_t k = 0; k < kAhead; ++k) {
      const uint64_t e = j * cap + min(t + k, cnt - 1);
      dd[k] = dv[e];
      ii[k] = lists[e];
    }
#pragma unroll
    for (uint32_t k = 0; k < kAhead; ++k) ww[k] = __atomic_load_n(&st[ii[k]], __ATOMIC_RELAXED);
    uint32_t td[kAhead];               // D == 0: differences to the targets of entries that merged
    if constexpr (D == 0) {
#pragma unroll
      for (uint32_t k = 0; k < kAhead; ++k) {
        const bool m = t + k < cnt && dd[k] <= bound && (uint32_t)(ww[k] >> 32) == kMerged;
        td[k] = hamming512(reinterpret_cast<const uint4*>(v.occ + (m ? (uint64_t)(uint32_t)ww[k] : j) * 16), own);
      }
    }
#pragma unroll
    for (uint32_t k = 0; k < kAhead; ++k) {
      if (t + k >= cnt || dd[k] > bound) continue;
      const uint32_t s = (uint32_t)(ww[k] >> 32);
      if (s == kUnres) {
        tdist[j] = t + k;
        // one address: a store from every wavefront with a waiting node took
        // most of a round (466K nodes: 256 us, looked at first 49)
        if (!__hip_atomic_load(unresolved, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
          __hip_atomic_store(unresolved, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return;
      }
      uint32_t r = ii[k], d = dd[k];
      if (s == kMerged) {
        r = (uint32_t)ww[k];
        if constexpr (D == 0) d = td[k];
        else d = subtree_diff<D>(v, lev, r, (uint32_t)j, bound);
        if (d > bound) continue;
      }
      tdist[j] = d;
      __atomic_store_n(&st[j], (unsigned long long)(kStMerged | r), __ATOMIC_RELAXED);
      return;
    }
  }
  __atomic_store_n(&st[j], (unsigned long long)(kStRep | j), __ATOMIC_RELAXED);
}

// Also clears hit[], which k_lossy_compact sets on every representative that
// takes in a merged node.
__global__ void k_rep_flag(const unsigned long long* __restrict__ st, uint64_t n, uint32_t* __restrict__ flag,
                           uint32_t* __restrict__ hit) {
  uint64_t j = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= n) return;
  flag[j] = (st[j] >> 32) == kRep ? 1u : 0u;
  hit[j] = 0u;
}

__global__ void __launch_bounds__(256)
k_lossy_compact(const uint32_t* __restrict__ rec, const uint64_t* __restrict__ vox,
                const unsigned long long* __restrict__ st, const uint32_t* __restrict__ tdist,
                const uint32_t* __restrict__ pos, const uint64_t* __restrict__ refs, uint64_t n,
                uint32_t* __restrict__ out, uint64_t* __restrict__ outVox, uint32_t* __restrict__ corr,
                uint32_t* __restrict__ hit, unsigned long long* __restrict__ stats) {
  unsigned long long err = 0, clusters = 0;
  for (uint64_t j = (uint64_t)blockIdx.x * 256 + threadIdx.x; j < n; j += (uint64_t)gridDim.x * 256) {
    const unsigned long long w = st[j];
    if ((w >> 32) == kRep) {
      const uint32_t p = pos[j];
      const uint32_t* s = rec + j * kRecWords;
      uint32_t* d = out + (uint64_t)p * kRecWords;
#pragma unroll
      for (int k = 0; k < kRecWords; ++k) d[k] = s[k];
      outVox[p] = vox[j];
      corr[j] = p;
    } else {
      corr[j] = pos[(uint32_t)w];
      err += (unsigned long long)tdist[j] * refs[j];
      // clusters: representatives with at least one member
      if (atomicExch(&hit[(uint32_t)w], 1u) == 0u) ++clusters;
    }
  }
  add_block(err, clusters, &stats[4], &stats[8]);
}

__global__ void k_remap_inplace(uint32_t* __restrict__ rec, uint64_t n, const uint32_t* __restrict__ corr) {
  uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  uint32_t* r = rec + i * kRecWords;
  const uint32_t m = r[0] & 0xFFu;
  for (int c = 0; c < 8; ++c)
    if ((m >> c) & 1u) r[1 + c] = corr[r[1 + c]];
}

// lists and spill hold cap entries per node each (spill is scratch).
void exhaustive_lists(svd_ctx* c, const uint32_t* sig, uint64_t n, const uint64_t* refs, uint64_t maxRefs,
                      uint32_t bound, uint32_t cap, uint32_t* lists, uint32_t* spill, uint32_t* counts) {
  const uint32_t chunks = (uint32_t)std::min<uint64_t>(16, std::max<uint64_t>(1, n / 512));
  const uint32_t C = div_up(div_up(n, chunks), 512) * 512;
  const uint32_t nKeys = div_up(n, C) * kPopBins;
  uint32_t bits = 1;
  while (nKeys >> bits) ++bits;
  uint32_t* keys = dalloc<uint32_t>(c, n);
  uint32_t* keys2 = dalloc<uint32_t>(c, n);
  uint32_t* ids = dalloc<uint32_t>(c, n);
  uint32_t* ids2 = dalloc<uint32_t>(c, n);
  uint32_t* off = dalloc<uint32_t>(c, (uint64_t)nKeys + 1);
  uint4* ssig = dalloc<uint4>(c, n * 4);
  k_list_keys<<<div_up(n, kB), kB, 0, c->stream>>>(sig, n, C, keys, ids);
  size_t bytes = 0;
  SVD_HIP(rocprim::radix_sort_pairs(nullptr, bytes, keys, keys2, ids, ids2, (size_t)n, 0, bits, c->stream));
  void* tmp = c->arena->get(bytes + 16);
  SVD_HIP(rocprim::radix_sort_pairs(tmp, bytes, keys, keys2, ids, ids2, (size_t)n, 0, bits, c->stream));
  c->arena->put(tmp);
  k_list_gather<<<div_up(n * 4, kB), kB, 0, c->stream>>>(sig, ids2, keys2, n, nKeys, ssig, off);
  // two j tiles per wavefront (256 nodes per workgroup) where that still gives
  // every CU the three workgroups it holds: one and two tiles took 7.1 and 5.7
  // ms on 372K nodes (2048^3 caves), 1.65 and 1.67 on 204K, 1.94 and 2.65 on
  // 126K, 1.20 and 1.77 on 68K
  if (n >= 768 * (uint64_t)std::max(c->numCU, 1))
    k_exhaustive_lists<2><<<div_up(n, 256), 256, 0, c->stream>>>(ssig, ids2, keys2, off, (uint32_t)n, C, refs, maxRefs,
                                                                 bound, cap, lists, spill, counts);
  else
    k_exhaustive_lists<1><<<div_up(n, 128), 256, 0, c->stream>>>(ssig, ids2, keys2, off, (uint32_t)n, C, refs, maxRefs,
                                                                 bound, cap, lists, spill, counts);
  k_list_order<<<div_up(n, 4), 256, 0, c->stream>>>(n, cap, lists, spill, counts);
  dfree(c, keys); dfree(c, keys2); dfree(c, ids); dfree(c, ids2); dfree(c, off); dfree(c, ssig);
}

LevelView make_view(const svd_octree* o, const std::vector<uint64_t*>& vox) {
  LevelView v = {};
  v.L = o->levels;
  for (uint32_t l = 0; l < o->levels; ++l) { v.rec[l] = o->dag[l].rec; v.vox[l] = vox[l]; }
  return v;
}

// fn(std::integral_constant<int, D>) for the level's depth above v.occLev
template <class F>
void with_depth(const LevelView& v, uint32_t lev, F fn) {
  const uint32_t d = lev < v.occLev ? v.occLev - lev : 0;
  static_assert(kMaxD == 4, "the cases below");
  switch (d) {
    case 0: return fn(std::integral_constant<int, 0>());
    case 1: return fn(std::integral_constant<int, 1>());
    case 2: return fn(std::integral_constant<int, 2>());
    case 3: return fn(std::integral_constant<int, 3>());
    case 4: return fn(std::integral_constant<int, 4>());
    default: return fn(std::integral_constant<int, kDeep>());
  }
}

struct PhaseClock {
  svd_ctx* c;
  std::vector<hipEvent_t> ev;
  explicit PhaseClock(svd_ctx* ctx, int n) : c(ctx), ev(n, nullptr) {
    for (auto& e : ev) SVD_HIP(hipEventCreate(&e));
  }
  ~PhaseClock() { for (auto& e : ev) if (e) (void)hipEventDestroy(e); }
  void mark(int i) { SVD_HIP(hipEventRecord(ev[i], c->stream)); }
  double ms(int a, int b) {
    float t = 0.f;
    SVD_HIP(hipEventSynchronize(ev[b]));
    SVD_HIP(hipEventElapsedTime(&t, ev[a], ev[b]));
    return (double)t;
  }
};

}  // namespace

// n u64 keys ascending by their low bits, through a scratch copy that takes
// their place: returns the array that holds them and frees the other.
static uint64_t* sort_u64(svd_ctx* c, uint64_t* keys, uint64_t n, int bits) {
  if (n < 2) return keys;
  uint64_t* sorted = dalloc<uint64_t>(c, n);
  size_t bytes = 0;
  SVD_HIP(rocprim::radix_sort_keys(nullptr, bytes, keys, sorted, (size_t)n, 0, bits, c->stream));
  void* tmp = c->arena->get(bytes + 16);
  SVD_HIP(rocprim::radix_sort_keys(tmp, bytes, keys, sorted, (size_t)n, 0, bits, c->stream));
  c->arena->put(tmp);
  dfree(c, keys);
  return sorted;
}

void lossy_signatures(svd_octree* o, uint32_t lev, uint32_t* sig) {
  if (o->state != SVD_S_DAG && o->state != SVD_S_SDAG) throw Error{SVD_ERR_STATE, "signatures need the DAG"};
  if (lev >= o->levels) throw Error{SVD_ERR_LEVELS, "level out of range"};
  std::vector<uint64_t*> vox(o->levels, nullptr);
  const LevelView v = make_view(o, vox);
  const uint64_t n = o->dag[lev].n;
  if (n) k_signatures<<<div_up(n * 8, kB), kB, 0, o->ctx->stream>>>(v, lev, n, sig);
  check_launch("k_signatures");
}

void lossy_merge(svd_octree* o, const svd_lossy_params* p, std::vector<svd_lossy_level_stats>& out) {
  svd_ctx* c = o->ctx;
  const uint32_t L = o->levels;
  if (o->state != SVD_S_DAG) throw Error{SVD_ERR_STATE, "toLossyDag: octree is not a DAG (geom_octree_extension.cpp:886-891)"};
  if (L < 3 || p->lev_lo < 1 || p->lev_lo > p->lev_hi || p->lev_hi > L - 2)
    throw Error{SVD_ERR_ARG, "lossy levels must satisfy 1 <= lev_lo <= lev_hi <= L-2"};
  if (p->list_cap < 1 || p->list_cap > 64) throw Error{SVD_ERR_ARG, "list_cap must be 1..64"};
  const bool learned = p->proposer == SVD_PROPOSER_LEARNED;
  const bool ranked = p->proposer == SVD_PROPOSER_RANKED;
  if (p->proposer > SVD_PROPOSER_RANKED) throw Error{SVD_ERR_ARG, "unknown proposer"};
  if (learned && (!p->model || p->knn_k < 1 || p->knn_k > 32 || p->knn_tables < 1 || p->knn_bits < 1 || p->knn_refine > 16 ||
                  p->knn_bits > 24 || p->knn_window < 1 || p->knn_window > 96))
    throw Error{SVD_ERR_ARG, "learned proposer needs a model, 1<=k<=32, tables>=1, 1<=bits<=24, 1<=window<=96"};
  const uint32_t cap = p->list_cap;
  const uint64_t maxRefs = p->max_refs;
  uint64_t recUsed = 0;

  // effective reference counts of levels 0..lev_hi on the input DAG
  std::vector<uint64_t*> refs(L, nullptr);
  refs[0] = dalloc<uint64_t>(c, o->dag[0].n + 1);
  k_fill_u64<<<div_up(o->dag[0].n + 1, kB), kB, 0, c->stream>>>(refs[0], 1ull, o->dag[0].n);
  for (uint32_t lev = 1; lev <= p->lev_hi; ++lev) {
    const uint64_t n = o->dag[lev].n;
    refs[lev] = dalloc<uint64_t>(c, n + 1);
    k_fill_u64<<<div_up(n + 1, kB), kB, 0, c->stream>>>(refs[lev], 0ull, n + 1);
    const uint64_t np = o->dag[lev - 1].n;
    if (np) k_refs_level<<<div_up(np, kB), kB, 0, c->stream>>>(o->dag[lev - 1].rec, np, refs[lev - 1],
                                                              (unsigned long long*)refs[lev]);
  }
  check_launch("effective refcounts");
  // voxel counts below the merged range
  std::vector<uint64_t*> vox(L, nullptr);
  for (int lev = (int)L - 1; lev > (int)p->lev_hi; --lev) {
    const uint64_t n = o->dag[lev].n;
    vox[lev] = dalloc<uint64_t>(c, n + 1);
    if (n) k_vox_level<<<div_up(n, kB), kB, 0, c->stream>>>(o->dag[lev].rec, n, lev == (int)L - 1,
                                                          lev + 1 < (int)L ? vox[lev + 1] : nullptr, vox[lev]);
  }
  check_launch("voxel counts");
  unsigned long long* dstats = dalloc<unsigned long long>(c, 9);
  uint32_t* unresolved = dalloc<uint32_t>(c, kRounds);
  uint32_t* bottom = nullptr;          // occupancies of level L-3, once the level is final
  // grid of the counting kernels: a resident wave of workgroups, one atomic each
  auto grid = [&](uint64_t work) { return std::min<uint32_t>(div_up(work, 256), 8 * (uint32_t)std::max(c->numCU, 1)); };
  PhaseClock clk(c, 7);

  for (int lev = (int)p->lev_hi; lev >= (int)p->lev_lo; --lev) {
    Level& lv = o->dag[lev];
    const uint64_t n = lv.n;
    svd_lossy_level_stats st = {};
    st.level = (uint64_t)lev;
    if (p->max_diff) st.bound = p->max_diff;
    else {
      const double d = (double)(L - (uint32_t)lev);
      st.bound = (uint64_t)std::llround(d * d * (double)p->diff_factor);
    }
    const uint32_t bound = st.bound > 0xFFFFFFF0ull ? 0xFFFFFFF0u : (uint32_t)st.bound;
    st.nodes_before = n;
    vox[lev] = dalloc<uint64_t>(c, n + 1);
    if (n) k_vox_level<<<div_up(n, kB), kB, 0, c->stream>>>(lv.rec, n, 0, vox[lev + 1], vox[lev]);
    k_fill_u64<<<1, 64, 0, c->stream>>>((uint64_t*)dstats, 0ull, 9);
    uint32_t* sig = dalloc<uint32_t>(c, (n + 1) * 16);
    uint32_t* lists = dalloc<uint32_t>(c, (n + 1) * cap);
    uint32_t* counts = dalloc<uint32_t>(c, n + 1);
    uint32_t* dv = dalloc<uint32_t>(c, (n + 1) * cap);
    unsigned long long* state = dalloc<unsigned long long>(c, n + 1);
    uint32_t* tdist = dalloc<uint32_t>(c, n + 1);
    uint32_t* pos = dalloc<uint32_t>(c, n + 1);
    uint32_t* total = dalloc<uint32_t>(c, 1);
    uint32_t* corr = dalloc<uint32_t>(c, n + 1);
    uint32_t* hit = dalloc<uint32_t>(c, n + 1);
    LevelView v = make_view(o, vox);
    clk.mark(0);
    if (n) k_signatures<<<div_up(n * 8, kB), kB, 0, c->stream>>>(v, (uint32_t)lev, n, sig);
    check_launch("k_signatures");
    clk.mark(1);
    if (!learned) {
      clk.mark(2);
      if (n && !ranked) exhaustive_lists(c, sig, n, refs[lev], maxRefs, bound, cap, lists, dv, counts);
      else if (n && cap <= 16)
        k_ranked_lists<16><<<div_up(n, 256), 256, 0, c->stream>>>(sig, n, refs[lev], maxRefs, bound, cap, lists,
                                                                   counts);
      else if (n && cap <= 32)
        k_ranked_lists<32><<<div_up(n, 256), 256, 0, c->stream>>>(sig, n, refs[lev], maxRefs, bound, cap, lists,
                                                                   counts);
      else if (n)
        k_ranked_lists<64><<<div_up(n, 256), 256, 0, c->stream>>>(sig, n, refs[lev], maxRefs, bound, cap, lists,
                                                                   counts);
      check_launch("pre-filter lists");
    } else {
      const uint32_t k = p->knn_k;
      float* emb = dalloc<float>(c, (n + 32) * 32);
      uint32_t* knn = dalloc<uint32_t>(c, (n + 1) * k);
      if (n) mlp_embed(p->model, sig, n, emb);
      clk.mark(2);
      if (n) knn_lsh(c, emb, n, k, p->knn_tables, p->knn_bits, p->knn_window, p->knn_seed, knn, sig);
      if (n) knn_refine(c, sig, n, k, p->knn_refine, knn);
      if (p->knn_record) {
        if (recUsed + n * k > p->knn_record_cap) throw Error{SVD_ERR_CAPACITY, "knn_record buffer too small"};
        if (n) SVD_HIP(hipMemcpyAsync(p->knn_record + recUsed, knn, n * k * 4, hipMemcpyDeviceToHost, c->stream));
        recUsed += n * k;
      }
      clk.mark(3);
      uint64_t* keys = dalloc<uint64_t>(c, n * k + 1);
      fill_u32(c, counts, 0u, n + 1);
      if (n) {
        int nb = 1;                        // n < 2^32 (32-bit node ids): at most 31 bits keep the flag in the key
        while (n >> nb) ++nb;
        if (nb > 31) throw Error{SVD_ERR_CAPACITY, "too many nodes in one level for the learned proposer"};
        k_proposal_keys<<<div_up(n * k, kB), kB, 0, c->stream>>>(knn, n, k, sig, refs[lev], maxRefs, bound, nb, keys);
        check_launch("k_proposal_keys");
        keys = sort_u64(c, keys, n * k, 2 * nb + 1);
        k_lists_from_sorted<<<div_up(n * k, kB), kB, 0, c->stream>>>(keys, n * k, cap, nb, lists, counts);
        check_launch("k_lists_from_sorted");
      }
      dfree(c, keys); dfree(c, knn); dfree(c, emb);
    }
    if (!learned) clk.mark(3);
    clk.mark(4);
    // the exact difference ends at the occupancies of level L-3 (or at the
    // level's own from there down)
    v.occ = sig;
    v.occLev = (uint32_t)lev;
    if ((uint32_t)lev + 3 < L) {
      if (!bottom) {
        const uint64_t nb = o->dag[L - 3].n;
        bottom = dalloc<uint32_t>(c, (nb + 1) * 16);
        if (nb) k_signatures<<<div_up(nb * 8, kB), kB, 0, c->stream>>>(v, L - 3, nb, bottom);
        check_launch("k_signatures");
      }
      v.occ = bottom;
      v.occLev = L - 3;
    }
    with_depth(v, (uint32_t)lev, [&](auto d) {
      if (n) k_verify<d()><<<grid(n * cap), 256, 0, c->stream>>>(v, (uint32_t)lev, lists, counts, n, cap, bound, dv,
                                                                 dstats + 5);
      check_launch("k_verify");
      clk.mark(5);
      if (n) k_resolve_init<<<grid(n), 256, 0, c->stream>>>(n, refs[lev], maxRefs, state, tdist, dstats + 5);
      check_launch("k_resolve_init");
      // kRounds rounds between looks: a round over settled nodes costs less
      // than a read-back (2 to 6 rounds settle the levels measured)
      for (uint64_t round = 0; n; round += kRounds) {
        fill_u32(c, unresolved, 0u, kRounds);
        for (uint32_t r = 0; r < kRounds; ++r)
          k_resolve<d()><<<div_up(n, kB), kB, 0, c->stream>>>(v, (uint32_t)lev, lists, dv, counts, n, cap, bound, state,
                                                              tdist, unresolved + r);
        check_launch("k_resolve");
        if (read_u32(c, unresolved + kRounds - 1) == 0) break;
        if (round > n) throw Error{SVD_ERR_DEVICE, "lossy resolution did not converge"};
      }
    });
    if (n) k_rep_flag<<<div_up(n, kB), kB, 0, c->stream>>>(state, n, pos, hit);
    scan_exclusive(c, pos, pos, n, total);
    const uint64_t kept = n ? read_u32(c, total) : 0;
    uint32_t* newRec = dalloc<uint32_t>(c, (kept + 1) * kRecWords);
    uint64_t* newVox = dalloc<uint64_t>(c, kept + 1);
    if (n) k_lossy_compact<<<grid(n), 256, 0, c->stream>>>(lv.rec, vox[lev], state, tdist, pos, refs[lev], n,
                                                              newRec, newVox, corr, hit, dstats);
    check_launch("k_lossy_compact");
    const uint64_t np = o->dag[lev - 1].n;
    if (np) k_remap_inplace<<<div_up(np, kB), kB, 0, c->stream>>>(o->dag[lev - 1].rec, np, corr);
    check_launch("k_remap_inplace");
    clk.mark(6);
    uint64_t hs[9];
    read_u32s(c, (const uint32_t*)dstats, (uint32_t*)hs, sizeof(hs) / 4);
    st.merged = n - kept;
    st.error_bound = hs[4];
    st.listed = hs[5];
    st.verified = hs[6];
    st.candidates = hs[7];
    st.clusters = hs[8];
    st.nodes_after = kept;
    st.ms_embed = learned ? clk.ms(1, 2) : 0.0;
    st.ms_knn = learned ? clk.ms(2, 3) : 0.0;
    st.ms_lists = learned ? clk.ms(3, 4) : clk.ms(2, 3);
    st.ms_verify = clk.ms(4, 5);
    st.ms_merge = clk.ms(5, 6);
    st.ms_total = clk.ms(0, 6);
    out.push_back(st);
    dfree(c, lv.rec);
    lv.rec = newRec;
    lv.n = kept;
    dfree(c, vox[lev]);
    vox[lev] = newVox;
    dfree(c, sig); dfree(c, lists); dfree(c, counts); dfree(c, dv); dfree(c, state); dfree(c, tdist);
    dfree(c, pos); dfree(c, total); dfree(c, corr); dfree(c, hit);
  }
  for (auto* r : refs) dfree(c, r);
  for (auto* x : vox) dfree(c, x);
  dfree(c, dstats); dfree(c, unresolved); dfree(c, bottom);
  // final exact dedup of every level (geom_octree_extension.cpp:1176)
  std::vector<Level> reduced;
  const uint64_t nn = dedup_all(c, L, o->dag, reduced);
  for (auto& lv : o->dag) dfree(c, lv.rec);
  o->dag = reduced;
  o->nNodesDAG = nn;
  SVD_HIP(hipStreamSynchronize(c->stream));
}

}  // namespace svd
