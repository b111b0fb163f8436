// k-nearest-neighbour search over 32-d embeddings for the learned lossy-DAG
// proposer: `tables` random-hyperplane LSH orderings; per ordering each point
// compares itself with the points within +-window sorted positions.  Exact,
// deterministic arithmetic (sequential fp32 sums, no contraction) so the CPU
// restatement reproduces the lists bit for bit:
//   key bit b of table t = dot(e, h[t][b]) > 0, h from a SplitMix64 stream
//   (component = ((z >> 40) * 2^-24) * 2 - 1);
//   stable sort by key; distance = sum_d (e_x[d] - e_y[d])^2;
//   result = the k smallest distinct (distance, index) pairs over all tables.
// With signatures given, the candidates are scored by the exact Hamming
// distance of the 512-bit occupancies instead (the embedding only decides
// which nodes meet in a window): the learned proposer's re-ranking.
#include <algorithm>
#include "svd_internal.hpp"
#include <rocprim/device/device_radix_sort.hpp>

namespace svd {

namespace {

constexpr int kDim = 32;
constexpr int kMaxK = 32;
constexpr int kTile = 256;
constexpr int kRow = kDim + 1;             // padded LDS row (no bank conflicts)

// Keys of `tables` orderings of every point: keys[t n + i] = t << bits | sign
// bits, so that one stable sort orders all of them.
__global__ void k_lsh_keys(const float* __restrict__ e, uint64_t n, const float* __restrict__ h, uint32_t bits,
                           uint32_t tables, uint32_t* __restrict__ keys, uint32_t* __restrict__ vals) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  float x[kDim];
#pragma unroll
  for (int d = 0; d < kDim; ++d) x[d] = e[i * kDim + d];
  for (uint32_t t = 0; t < tables; ++t) {
    uint32_t key = t << bits;
    for (uint32_t b = 0; b < bits; ++b) {
      const float* hp = h + ((uint64_t)t * bits + b) * kDim;
      float s = 0.f;
#pragma unroll
      for (int d = 0; d < kDim; ++d) { const float q = x[d] * hp[d]; s = s + q; }
      if (s > 0.f) key |= 1u << b;
    }
    keys[t * n + i] = key;
    vals[t * n + i] = (uint32_t)i;
  }
}

// ---- windows on the matrix cores (signatures, k <= 16, n <= 2^22) --------------
// The running list of a node is 16 ascending keys (Hamming << 22 | node), so
// (distance, index) order is integer order: 10 + 22 bits.
constexpr uint32_t kIdBits = 22, kIdMask = (1u << kIdBits) - 1u;
constexpr int kList = 16;
constexpr int kQ = 128;                    // queries per workgroup, 32 per wavefront
constexpr int kMaxW = 96;                  // the widest window
constexpr int kWinRows = kQ + 2 * kMaxW;   // rows a workgroup meets
constexpr int kSigRow = 20;                // dwords per LDS row (eight lanes' 16-byte reads in distinct banks)
constexpr int kHash = 1024;                // >= 3 x kWinRows
constexpr int kMaxTiles = (32 + 2 * kMaxW + 31) / 32;

typedef int i32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));

// One signature word as 32 fp4 values, bit 0 -> +1.0, 1 -> -1.0; bit 4p + d is
// nibble p of dword d (any order of the 512 positions serves).
__device__ __forceinline__ i32x4_t bits_to_fp4(uint32_t w) {
  constexpr uint32_t kOne = 0x22222222u, kSign = 0x88888888u;
  i32x4_t r;
  r[0] = (int)(((w << 3) & kSign) | kOne);
  r[1] = (int)(((w << 2) & kSign) | kOne);
  r[2] = (int)(((w << 1) & kSign) | kOne);
  r[3] = (int)((w & kSign) | kOne);
  return r;
}
__device__ __forceinline__ uint32_t med3(uint32_t a, uint32_t b, uint32_t c) {
  return max(min(a, b), min(max(a, b), c));
}

// One table's windows: a wavefront's 32 consecutive sorted positions (the
// columns) meet the 32 + 2W rows around them.  With bits as +-1 the dot
// product is 512 - 2 Hamming; a tile of 32 x 32 distances is 8 of
// v_mfma_f32_32x32x64_f8f6f4 (fp4, exact sums), which costs next to nothing.
// Accumulator element v of lane l is row 8 (v/4) + 4 (l/32) + v%4, column
// l%32: the two lanes of a column insert half of its rows each into a sorted
// list of 16 keys (16 medians, skipped while no lane has a key below its
// worst), the first starting from the running list, the second from copies of
// its worst key, and the 16 smallest of both are the new list.  Candidates
// that the running list already holds are masked out: the rows' ids are in a
// hash set, which every list entry looks itself up in.  Bound by the inserts.
// One lane per point with the window's XOR/popcounts took 0.66-1.22 ms per
// table on 466K nodes (W = 64), bound by a chain of some 2500 cycles per row.
__global__ void __launch_bounds__(256) k_window_keys(const uint32_t* __restrict__ sig,
                                                     const uint32_t* __restrict__ order, uint32_t n, uint32_t W,
                                                     int first, uint32_t* __restrict__ best) {
  __shared__ __attribute__((aligned(16))) uint32_t rows[kWinRows * kSigRow];
  __shared__ __attribute__((aligned(16))) uint32_t ids[kWinRows + 32];
  __shared__ uint32_t setId[kHash];
  __shared__ uint32_t setRow[kHash];
  __shared__ uint32_t dup[kQ][kMaxTiles];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, col = lane & 31, half = lane >> 5;
  const int64_t lo = (int64_t)blockIdx.x * kQ - (int64_t)W;     // sorted position of row 0
  const int nrows = kQ + 2 * (int)W;
  const int tiles = (32 + 2 * (int)W + 31) / 32;
  for (int r = tid; r < kWinRows + 32; r += 256) {
    const int64_t q = lo + r;
    ids[r] = r < nrows && q >= 0 && q < (int64_t)n ? order[q] : kNone;
  }
  if (!first) {
    for (int s = tid; s < kHash; s += 256) setId[s] = kNone;
    for (int s = tid; s < kQ * kMaxTiles; s += 256) (&dup[0][0])[s] = 0u;
  }
  __syncthreads();
  for (int t = tid; t < kWinRows * 4; t += 256) {
    const int r = t >> 2;
    const uint32_t id = ids[r];
    *reinterpret_cast<uint4*>(&rows[r * kSigRow + 4 * (t & 3)]) =
        id != kNone ? reinterpret_cast<const uint4*>(sig + (uint64_t)id * 16)[t & 3] : make_uint4(0, 0, 0, 0);
  }
  if (!first) {
    for (int r = tid; r < nrows; r += 256) {
      const uint32_t id = ids[r];
      if (id == kNone) continue;
      uint32_t h = (id * 2654435761u) >> 22;
      while (atomicCAS(&setId[h], kNone, id) != kNone) h = (h + 1) & (kHash - 1);   // ids are distinct
      setRow[h] = (uint32_t)r;
    }
  }
  __syncthreads();
  const int base = 32 * wave;                    // the wavefront's first row
  const uint32_t x = ids[base + col + (int)W];   // kNone past the last point
  uint32_t b[kList];
#pragma unroll
  for (int t = 0; t < kList; ++t) b[t] = kNone;
  if (!first && x != kNone) {
    const uint4* p = reinterpret_cast<const uint4*>(best + (uint64_t)x * kList);
#pragma unroll
    for (int t = 0; t < kList / 4; ++t) {
      const uint4 u = p[t];
      b[4 * t] = u.x; b[4 * t + 1] = u.y; b[4 * t + 2] = u.z; b[4 * t + 3] = u.w;
    }
    // each half looks its eight entries up
    const uint4 u = p[2 * half], w = p[2 * half + 1];
    const uint32_t mine[8] = {u.x, u.y, u.z, u.w, w.x, w.y, w.z, w.w};
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      const uint32_t key = mine[t];
      if (key == kNone) continue;
      const uint32_t id = key & kIdMask;
      uint32_t h = (id * 2654435761u) >> 22, got;
      while ((got = setId[h]) != kNone && got != id) h = (h + 1) & (kHash - 1);
      if (got == kNone) continue;
      const int r = (int)setRow[h] - base;
      if (r >= 0 && r < 32 * tiles) atomicOr(&dup[base + col][r >> 5], 1u << (r & 31));
    }
  }
  if (half) {
#pragma unroll
    for (int t = 0; t < kList; ++t) b[t] = b[kList - 1];
  }
  __syncthreads();
  i32x4_t qf[8];
  {
    const uint4* p = reinterpret_cast<const uint4*>(&rows[(base + col + (int)W) * kSigRow + 8 * half]);
    const uint4 u = p[0], w = p[1];
    const uint32_t q[8] = {u.x, u.y, u.z, u.w, w.x, w.y, w.z, w.w};
#pragma unroll
    for (int k = 0; k < 8; ++k) qf[k] = bits_to_fp4(q[k]);
  }
  for (int t = 0; t < tiles; ++t) {
    const int r0 = base + 32 * t;                // first row of the tile
    f32x16_t acc;
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[v] = 0.f;
    {
      const uint4* p = reinterpret_cast<const uint4*>(&rows[(r0 + col) * kSigRow + 8 * half]);
      const uint4 u = p[0], w = p[1];
      const uint32_t q[8] = {u.x, u.y, u.z, u.w, w.x, w.y, w.z, w.w};
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const i32x4_t a = bits_to_fp4(q[k]);
        acc = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(
            __builtin_shufflevector(a, a, 0, 1, 2, 3, -1, -1, -1, -1),
            __builtin_shufflevector(qf[k], qf[k], 0, 1, 2, 3, -1, -1, -1, -1), acc, 4, 4, 0, 0, 0, 0);
      }
    }
    // rows of the tile that this column may take: within W of it, not itself,
    // not listed already
    const int c = col - 32 * t;                  // row of the window's start, relative to the tile
    const int e = c + 2 * (int)W;                // and of its end
    uint32_t ok = 0;
    if (x != kNone && e >= 0 && c < 32)
      ok = (c > 0 ? 0xFFFFFFFFu << c : 0xFFFFFFFFu) & (e < 31 ? 0xFFFFFFFFu >> (31 - e) : 0xFFFFFFFFu);
    const int self = c + (int)W;
    if (self >= 0 && self < 32) ok &= ~(1u << self);
    if (!first) ok &= ~dup[base + col][t];
    const uint32_t bad = ~ok >> (4 * half);      // bit 8 (v/4) + v%4: accumulator element v is out
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const uint4 id4 = *reinterpret_cast<const uint4*>(&ids[r0 + 8 * g + 4 * half]);
      const uint32_t id[4] = {id4.x, id4.y, id4.z, id4.w};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t d = (uint32_t)(1073741824.f - 2097152.f * acc[4 * g + i]);   // Hamming << 22
        const uint32_t out = (uint32_t)((int)(bad << (31 - (8 * g + i))) >> 31);
        const uint32_t key = d | id[i] | out;    // an absent row's id is all ones
        if (!__any(key < b[kList - 1])) continue;
#pragma unroll
        for (int q = kList - 1; q > 0; --q) b[q] = med3(b[q - 1], key, b[q]);
        b[0] = min(b[0], key);
      }
    }
  }
  // the 16 smallest of the two halves' lists (a bitonic sequence), sorted
  uint32_t m[kList];
#pragma unroll
  for (int t = 0; t < kList; ++t) m[t] = min(b[t], (uint32_t)__shfl_xor(b[kList - 1 - t], 32, 64));
#pragma unroll
  for (int o = kList / 2; o >= 1; o >>= 1)
#pragma unroll
    for (int t = 0; t < kList; ++t)
      if (!(t & o)) {
        const uint32_t u = min(m[t], m[t + o]), w = max(m[t], m[t + o]);
        m[t] = u;
        m[t + o] = w;
      }
  if (half == 0 && x != kNone) {
    uint4* p = reinterpret_cast<uint4*>(best + (uint64_t)x * kList);
#pragma unroll
    for (int t = 0; t < kList / 4; ++t) p[t] = make_uint4(m[4 * t], m[4 * t + 1], m[4 * t + 2], m[4 * t + 3]);
  }
}

// The lists' first k nodes.
__global__ void k_window_ids(const uint32_t* __restrict__ best, uint64_t n, uint32_t k, uint32_t* __restrict__ out) {
  const uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= n * k) return;
  const uint32_t key = best[e / k * kList + e % k];
  out[e] = key == kNone ? kNone : key & kIdMask;
}

// Block = 256 consecutive sorted positions; the window's rows are staged in
// LDS.  Each lane keeps its point's running top-k (registers) across tables
// through best_d / best_i in HBM.  HAM = 0: squared L2 of the embeddings;
// HAM = 1: Hamming distance of the 512-bit signatures.
template <int HAM, int KM>
__global__ void __launch_bounds__(kTile) k_window_topk(const float* __restrict__ e, const uint32_t* __restrict__ sig,
                                                       const uint32_t* __restrict__ order, uint64_t n, uint32_t W,
                                                       uint32_t k, int first, float* __restrict__ best_d,
                                                       uint32_t* __restrict__ best_i) {
  constexpr int kWords = HAM ? 16 : kDim;
  constexpr int kR = kWords + 1;            // padded LDS row (no bank conflicts)
  extern __shared__ float rows[];           // (kTile + 2W) x kR
  uint32_t* urows = reinterpret_cast<uint32_t*>(rows);
  const uint64_t q0 = (uint64_t)blockIdx.x * kTile;
  const int64_t lo = (int64_t)q0 - (int64_t)W;
  const uint32_t nrows = kTile + 2 * W;
  for (uint32_t t = threadIdx.x; t < nrows * kWords; t += kTile) {
    const uint32_t rr = t / kWords, d = t % kWords;
    const int64_t q = lo + (int64_t)rr;
    const bool in = q >= 0 && q < (int64_t)n;
    if (HAM) urows[rr * kR + d] = in ? sig[(uint64_t)order[q] * 16 + d] : 0u;
    else rows[rr * kR + d] = in ? e[(uint64_t)order[q] * kDim + d] : 0.f;
  }
  __syncthreads();
  const uint64_t q = q0 + threadIdx.x;
  if (q >= n) return;
  const uint32_t x = order[q];
  float bd[KM];
  uint32_t bi[KM];
#pragma unroll
  for (int t = 0; t < KM; ++t) {
    bd[t] = first || t >= (int)k ? __builtin_inff() : best_d[(uint64_t)x * k + t];
    bi[t] = first || t >= (int)k ? 0xFFFFFFFFu : best_i[(uint64_t)x * k + t];
  }
  const uint32_t xr = (threadIdx.x + W) * kR;
  // the query row lives in registers
  uint32_t xs[HAM ? 16 : 1];
  float xe[HAM ? 1 : kDim];
  if (HAM) {
#pragma unroll
    for (int d = 0; d < (HAM ? 16 : 1); ++d) xs[d] = urows[xr + d];
  } else {
#pragma unroll
    for (int d = 0; d < (HAM ? 1 : kDim); ++d) xe[d] = rows[xr + d];
  }
  for (int64_t r = (int64_t)q - (int64_t)W; r <= (int64_t)q + (int64_t)W; ++r) {
    if (r < 0 || r >= (int64_t)n || r == (int64_t)q) continue;
    const uint32_t yr = (uint32_t)(r - lo) * kR;
    float s = 0.f;
    if (HAM) {
      uint32_t h = 0;
#pragma unroll
      for (int d = 0; d < (HAM ? 16 : 1); ++d) h += __popc(xs[d] ^ urows[yr + d]);
      s = (float)h;
    } else {
#pragma unroll
      for (int d = 0; d < (HAM ? 1 : kDim); ++d) { const float t = xe[d] - rows[yr + d]; const float sq = t * t; s = s + sq; }
    }
    // (s, y) < worst kept?
    float wd = bd[KM - 1];
    uint32_t wi = bi[KM - 1];
    if (KM != (int)k) {
#pragma unroll
      for (int t = 0; t < KM; ++t)
        if (t == (int)k - 1) { wd = bd[t]; wi = bi[t]; }
    }
    const uint32_t y = order[r];
    if (!(s < wd || (s == wd && y < wi))) continue;
    bool dup = false;
#pragma unroll
    for (int t = 0; t < KM; ++t) dup |= (t < (int)k) && bi[t] == y;
    if (dup) continue;
    // insert keeping (distance, index) ascending
    float cd = s;
    uint32_t ci = y;
#pragma unroll
    for (int t = 0; t < KM; ++t) {
      if (t < (int)k && (cd < bd[t] || (cd == bd[t] && ci < bi[t]))) {
        const float td = bd[t]; const uint32_t ti = bi[t];
        bd[t] = cd; bi[t] = ci;
        cd = td; ci = ti;
      }
    }
  }
#pragma unroll
  for (int t = 0; t < KM; ++t)
    if (t < (int)k) { best_d[(uint64_t)x * k + t] = bd[t]; best_i[(uint64_t)x * k + t] = bi[t]; }
}

// The smallest x of the wavefront, in every lane: a reduction by the VALU's
// lane shifts (rows of 16, then across rows), the result read from lane 63.
__device__ __forceinline__ uint32_t wave_min(uint32_t x) {
#define SVD_DPP_MIN(ctrl, rows) \
  x = min(x, (uint32_t)__builtin_amdgcn_update_dpp((int)x, (int)x, ctrl, rows, 0xf, false))
  SVD_DPP_MIN(0x111, 0xf);   // row_shr:1, 2, 4, 8
  SVD_DPP_MIN(0x112, 0xf);
  SVD_DPP_MIN(0x114, 0xf);
  SVD_DPP_MIN(0x118, 0xf);
  SVD_DPP_MIN(0x142, 0xa);   // row_bcast:15 into rows 1 and 3
  SVD_DPP_MIN(0x143, 0xc);   // row_bcast:31 into rows 2 and 3
#undef SVD_DPP_MIN
  return (uint32_t)__builtin_amdgcn_readlane((int)x, 63);
}
__device__ __forceinline__ uint64_t wave_min(uint64_t m) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const uint32_t lo = __shfl_xor((uint32_t)m, off, 64), hi = __shfl_xor((uint32_t)(m >> 32), off, 64);
    const uint64_t o = ((uint64_t)hi << 32) | lo;
    m = o < m ? o : m;
  }
  return m;
}

// One neighbour-of-neighbour round (NN-descent) on the signature Hamming
// metric: node x keeps the k smallest distinct (distance, index) among its
// own list and the lists of its neighbours.  Reads `in`, writes `out`.
// One wavefront per node: the k + k*k candidate ids are deduplicated through
// a hash set in LDS, each distinct candidate's signature is read once (by the
// lane whose insert won), and k wave-wide minima over the keys (distance <<
// IDB | index) take the k smallest.  The minima bound it: 32-bit keys (IDB =
// 22, up to 2^22 nodes) reduced by lane shifts took a round over 466K nodes
// from 1.28 ms (64-bit keys by shuffles, IDB = 32) to 0.85 - 1.03 ms.
template <int KM, typename Key>
__global__ void __launch_bounds__(256) k_knn_refine_wave(const uint32_t* __restrict__ sig, uint64_t n, uint32_t k,
                                                         const uint32_t* __restrict__ in, uint32_t* __restrict__ out) {
  constexpr int kCand = KM * (KM + 1);
  constexpr int kPer = (kCand + 63) / 64;                 // candidates per lane
  constexpr int kSlots = KM <= 16 ? 1024 : 4096;          // >= 2 * kCand, power of two
  constexpr int kShift = KM <= 16 ? 22 : 20;              // 32 - log2(kSlots): the product's high bits
  constexpr int IDB = sizeof(Key) == 4 ? (int)kIdBits : 32;
  constexpr Key kNoKey = ~(Key)0;
  __shared__ __attribute__((aligned(16))) uint32_t set[4][kSlots];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const uint64_t x = (uint64_t)blockIdx.x * 4 + wave;
  const bool live = x < n;
  uint32_t* S = set[wave];
  for (int j = lane; j < kSlots / 4; j += 64) reinterpret_cast<uint4*>(S)[j] = make_uint4(kNone, kNone, kNone, kNone);
  __syncthreads();
  const uint32_t nc = k + k * k;
  Key key[kPer];
#pragma unroll
  for (int p = 0; p < kPer; ++p) {
    key[p] = kNoKey;
    const uint32_t c = (uint32_t)(lane + 64 * p);
    if (!live || c >= nc) continue;
    uint32_t z;
    if (c < k) {
      z = in[x * k + c];
    } else {
      const uint32_t y = in[x * k + (c - k) / k];
      z = (y == kNone || (uint64_t)y >= n) ? kNone : in[(uint64_t)y * k + (c - k) % k];
    }
    if (z == kNone || (uint64_t)z == x || (uint64_t)z >= n) continue;
    uint32_t h = (z * 2654435761u) >> kShift;
    bool mine = false;
    while (true) {
      const uint32_t old = atomicCAS(&S[h], kNone, z);
      if (old == kNone) { mine = true; break; }
      if (old == z) break;
      h = (h + 1) & (kSlots - 1);
    }
    if (!mine) continue;
    const uint4* px = reinterpret_cast<const uint4*>(sig + x * 16);
    const uint4* pz = reinterpret_cast<const uint4*>(sig + (uint64_t)z * 16);
    uint32_t d = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const uint4 a = px[q], b = pz[q];
      d += __popc(a.x ^ b.x) + __popc(a.y ^ b.y) + __popc(a.z ^ b.z) + __popc(a.w ^ b.w);
    }
    key[p] = ((Key)d << IDB) | z;
  }
  Key mine = kNoKey;                 // lane t: the t-th smallest
  for (uint32_t t = 0; t < k; ++t) {
    Key m = key[0];
#pragma unroll
    for (int p = 1; p < kPer; ++p) m = key[p] < m ? key[p] : m;
    m = wave_min(m);
    if ((uint32_t)lane == t) mine = m;
#pragma unroll
    for (int p = 0; p < kPer; ++p)
      if (key[p] == m) key[p] = kNoKey;   // candidates are distinct: one lane holds m
  }
  if (live && (uint32_t)lane < k)
    out[x * k + lane] = mine == kNoKey ? kNone : (uint32_t)(mine & (((Key)1 << (IDB - 1) << 1) - 1));
}

}  // namespace

void knn_refine(svd_ctx* c, const uint32_t* sig, uint64_t n, uint32_t k, uint32_t rounds, uint32_t* knn) {
  if (!rounds || !n) return;
  if (k < 1 || k > (uint32_t)kMaxK) throw Error{SVD_ERR_ARG, "knn: k must be 1..32"};
  uint32_t* tmp = dalloc<uint32_t>(c, n * k);
  for (uint32_t r = 0; r < rounds; ++r) {
    const uint32_t* in = r & 1 ? tmp : knn;
    uint32_t* out = r & 1 ? knn : tmp;
    if (k <= 16 && n <= (1ull << kIdBits))
      k_knn_refine_wave<16, uint32_t><<<div_up(n, 4), 256, 0, c->stream>>>(sig, n, k, in, out);
    else if (k <= 16) k_knn_refine_wave<16, uint64_t><<<div_up(n, 4), 256, 0, c->stream>>>(sig, n, k, in, out);
    else k_knn_refine_wave<kMaxK, uint64_t><<<div_up(n, 4), 256, 0, c->stream>>>(sig, n, k, in, out);
  }
  check_launch("k_knn_refine");
  if (rounds & 1) SVD_HIP(hipMemcpyAsync(knn, tmp, n * k * 4, hipMemcpyDeviceToDevice, c->stream));
  dfree(c, tmp);
}

void knn_lsh(svd_ctx* c, const float* emb, uint64_t n, uint32_t k, uint32_t tables, uint32_t bits, uint32_t window,
             uint64_t seed, uint32_t* out, const uint32_t* sig) {
  if (k < 1 || k > (uint32_t)kMaxK) throw Error{SVD_ERR_ARG, "knn: k must be 1..32"};
  if (bits < 1 || bits > 24 || tables < 1 || window < 1 || window > 96) throw Error{SVD_ERR_ARG, "knn: bits 1..24, tables >= 1, window 1..96"};
  if (n >= 0xFFFFFFFFull) throw Error{SVD_ERR_CAPACITY, "knn: too many points"};
  if (n == 0) return;
  // hyperplanes of every table
  std::vector<float> h((size_t)tables * bits * kDim);
  uint64_t s = seed;
  for (auto& v : h) {
    s += 0x9E3779B97F4A7C15ull;
    uint64_t z = s;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
    v = (float)(z >> 40) * (1.0f / 16777216.0f) * 2.0f - 1.0f;
  }
  float* dh = dalloc<float>(c, h.size());
  SVD_HIP(hipMemcpyAsync(dh, h.data(), h.size() * 4, hipMemcpyHostToDevice, c->stream));
  // orderings are sorted several at a time, up to 2^22 keys (table << bits | key)
  const uint32_t group = (uint32_t)std::min<uint64_t>(std::min<uint64_t>(tables, 1ull << (32 - bits)),
                                                      std::max<uint64_t>(1, (1ull << 22) / n));
  uint32_t gbits = bits;
  while ((group - 1) >> (gbits - bits)) ++gbits;
  uint32_t* keys = dalloc<uint32_t>(c, n * group);
  uint32_t* keys2 = dalloc<uint32_t>(c, n * group);
  uint32_t* vals = dalloc<uint32_t>(c, n * group);
  uint32_t* orders = dalloc<uint32_t>(c, n * group);
  // the matrix-core windows need (distance, node) in 32 bits
  const bool mm = sig && k <= (uint32_t)kList && n <= (1ull << kIdBits);
  float* bd = mm ? nullptr : dalloc<float>(c, n * k);
  uint32_t* best = mm ? dalloc<uint32_t>(c, n * kList) : nullptr;
  size_t bytes = 0, last = 0;
  SVD_HIP(rocprim::radix_sort_pairs(nullptr, bytes, keys, keys2, vals, orders, (size_t)(n * group), 0, gbits, c->stream));
  if (tables % group)
    SVD_HIP(rocprim::radix_sort_pairs(nullptr, last, keys, keys2, vals, orders, (size_t)(n * (tables % group)), 0, gbits,
                                      c->stream));
  bytes = std::max(bytes, last);
  void* tmp = c->arena->get(bytes + 16);
  const size_t lds = (size_t)(kTile + 2 * window) * (sig ? 17 : kRow) * sizeof(float);
  for (uint32_t t = 0; t < tables; ++t) {
    const uint32_t inGroup = t % group;
    if (inGroup == 0) {
      const uint32_t m = std::min(group, tables - t);
      k_lsh_keys<<<div_up(n, 256), 256, 0, c->stream>>>(emb, n, dh + (size_t)t * bits * kDim, bits, m, keys, vals);
      SVD_HIP(rocprim::radix_sort_pairs(tmp, bytes, keys, keys2, vals, orders, (size_t)(n * m), 0, gbits, c->stream));
    }
    const uint32_t* order = orders + (uint64_t)inGroup * n;
    const dim3 g(div_up(n, kTile));
    if (mm) k_window_keys<<<div_up(n, kQ), 256, 0, c->stream>>>(sig, order, (uint32_t)n, window, t == 0, best);
    else if (sig && k == 16) k_window_topk<1, 16><<<g, kTile, lds, c->stream>>>(emb, sig, order, n, window, k, t == 0, bd, out);
    else if (sig) k_window_topk<1, kMaxK><<<g, kTile, lds, c->stream>>>(emb, sig, order, n, window, k, t == 0, bd, out);
    else if (k == 16) k_window_topk<0, 16><<<g, kTile, lds, c->stream>>>(emb, sig, order, n, window, k, t == 0, bd, out);
    else k_window_topk<0, kMaxK><<<g, kTile, lds, c->stream>>>(emb, sig, order, n, window, k, t == 0, bd, out);
    check_launch("knn table");
  }
  if (mm) {
    k_window_ids<<<div_up(n * k, 256), 256, 0, c->stream>>>(best, n, k, out);
    check_launch("k_window_ids");
  }
  c->arena->put(tmp);
  dfree(c, dh); dfree(c, keys); dfree(c, keys2); dfree(c, vals); dfree(c, orders); dfree(c, bd); dfree(c, best);
}

}  // namespace svd
