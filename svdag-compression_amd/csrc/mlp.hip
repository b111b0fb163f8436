// Learned candidate encoder for the lossy DAG: MLP 512 -> 256 -> 128 -> 32.
// bf16 weights and activations, fp32 accumulation on the CDNA matrix cores
// (v_mfma_f32_32x32x16_bf16 on LDS-staged tiles; the weight gradients split
// over the batch and summed in a fixed order by the optimizer), hand-written
// forward and backward passes, Adam.
// The reference has no learned part (its lossy path clusters an exhaustive
// similarity graph with MCL, geom_octree_extension.cpp:797-1179).
//
// Definitions (also stated by the CPU oracle the tests compare with):
//   z1 = x W1 + b1, h1 = bf16(relu(z1)); z2 = h1 W2 + b2, h2 = bf16(relu(z2));
//   e = h2 W3 + b3 (fp32).  x = the node's 512-bit occupancy, expanded to
//   0/1 inside the first GEMM's operand load (no expanded copy in HBM).
//   Pair p = batch rows (2p, 2p+1); d = |e_a - e_b|^2; y = min(H, 32);
//   loss = sum (d - y)^2 / P.  Each layer's delta is rounded to bf16 once and
//   feeds both its weight gradient and its bias gradient.
#include <algorithm>
#include <type_traits>
#include "svd_internal.hpp"
#include <rocprim/device/device_radix_sort.hpp>
#include <cmath>

namespace svd {

namespace {


constexpr int D0 = 512, D1 = 256, D2 = 128, D3 = 32;
constexpr uint64_t OFF_W1 = 0, OFF_B1 = OFF_W1 + D0 * D1, OFF_W2 = OFF_B1 + D1, OFF_B2 = OFF_W2 + D1 * D2,
                   OFF_W3 = OFF_B2 + D2, OFF_B3 = OFF_W3 + D2 * D3, N_PARAMS = OFF_B3 + D3;
// bf16 weights: W1 | W2 | W3 transposed ([out][in], the embedding's operand),
// then the training step's operands in fragment order: W1, W2, W3 for the
// forward products and W3, W2 transposed for the input gradients.
constexpr uint64_t WB_W1 = 0, WB_W2 = WB_W1 + D0 * D1, WB_W3 = WB_W2 + D1 * D2, N_WB = WB_W3 + D2 * D3;
constexpr uint64_t WF_W1 = N_WB, WF_W2 = WF_W1 + D0 * D1, WF_W3 = WF_W2 + D1 * D2, WF_W3T = WF_W3 + D2 * D3,
                   WF_W2T = WF_W3T + D3 * D2, N_WB_ALL = WF_W2T + D2 * D1;
constexpr float kHCap = 32.f;
static_assert(N_PARAMS == SVD_MLP_PARAMS, "parameter layout");

__device__ __forceinline__ uint16_t f2bf(float f) {   // round to nearest even (finite values)
  uint32_t u = __float_as_uint(f);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float bf2f(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));

// bf16 0/1 pair from the two low bits of w (element 0 in the low half)
__device__ __forceinline__ uint32_t bit_pair(uint32_t w) {
  return ((w & 1u) ? 0x3F80u : 0u) | ((w & 2u) ? 0x3F800000u : 0u);
}
// eight 0/1 values from the low byte of w
__device__ __forceinline__ uint4 bit_oct(uint32_t w) {
  return make_uint4(bit_pair(w), bit_pair(w >> 2), bit_pair(w >> 4), bit_pair(w >> 6));
}

// The embedding's layers: C = A (M x K) B (K x N) with bf16 operands and fp32
// accumulation, A[m][k] = bit k of signature m (AL_BITS, 16 words each) or
// a[m lda + k] (AL_MK), B[k][n] = b[n ldb + k]; out bf16(relu(C + bias)) or
// C + bias (fp32).
enum ALay { AL_BITS = 0, AL_MK = 1 };
enum Epi { E_BIAS_RELU_BF16 = 0, E_BIAS_F32 = 1 };

struct MmArgs {
  uint64_t M;
  int N, K;
  const uint32_t* abits;
  const uint16_t* a; int64_t lda;
  const uint16_t* b; int64_t ldb;
  const float* bias;
  uint16_t* outb; float* outf; int64_t ldo;
};

// Four wavefronts per workgroup, each a 32x32 sub-tile of a TM x TN tile
// (64x64 for WN = 2, 128x32 for WN = 1).  K runs in stages of KB: a stage is
// loaded from global memory into registers while the previous one feeds the
// matrix cores from LDS (two LDS buffers, one barrier per stage).  In LDS, A
// is kept [m][k] and B [n][k], rows padded by 16 bytes; bits are expanded to
// bf16 as they are stored.  Per 16 of K, lane l of a wavefront reads A[row
// l%32][k + 8(l/32) + i] and B[k + 8(l/32) + i][col l%32], i = 0..7 (16 bytes
// each), for one v_mfma_f32_32x32x16_bf16; accumulator element v of lane l is
// C[8(v/4) + 4(l/32) + v%4][l%32] of the wavefront's sub-tile.
template <int AL, int EP, int WN, int KB>
__global__ void __launch_bounds__(256) k_mm(MmArgs g) {
  constexpr int WM = 4 / WN, TM = 32 * WM, TN = 32 * WN, ROW = KB + 8;
  constexpr int A_CH = AL == AL_BITS ? TM * KB / 32 : TM * KB / 8;   // words or 16-byte chunks per stage
  constexpr int B_CH = TN * KB / 8;
  constexpr int NA = (A_CH + 255) / 256, NB = (B_CH + 255) / 256;
  __shared__ __attribute__((aligned(16))) uint16_t As[2][TM * ROW];
  __shared__ __attribute__((aligned(16))) uint16_t Bs[2][TN * ROW];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave % WM, wn = wave / WM;
  const uint64_t m0 = (uint64_t)blockIdx.x * TM;
  const int n0 = blockIdx.y * TN;
  uint4 ra[AL == AL_BITS ? 1 : NA];
  uint32_t rw[AL == AL_BITS ? NA : 1];
  uint4 rb[NB];

  auto load = [&](int k0) {
#pragma unroll
    for (int j = 0; j < NA; ++j) {
      const int c = tid + 256 * j;
      if (A_CH % 256 && c >= A_CH) continue;
      if (AL == AL_BITS) {
        const int r = c / (KB / 32), k = k0 + 32 * (c % (KB / 32));
        const uint64_t m = m0 + (uint64_t)r;
        rw[j] = m < g.M ? g.abits[m * 16 + (k >> 5)] : 0u;
      } else {
        const int r = c / (KB / 8), k = k0 + 8 * (c % (KB / 8));
        const uint64_t m = m0 + (uint64_t)r;
        ra[j] = m < g.M ? *reinterpret_cast<const uint4*>(g.a + (int64_t)m * g.lda + k) : make_uint4(0u, 0u, 0u, 0u);
      }
    }
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      const int c = tid + 256 * j;
      if (B_CH % 256 && c >= B_CH) continue;
      const int nn = c / (KB / 8), k = k0 + 8 * (c % (KB / 8));
      const uint4* p = reinterpret_cast<const uint4*>(g.b + (int64_t)(n0 + nn) * g.ldb + k);
      rb[j] = make_uint4(p->x, p->y, p->z, p->w);
    }
  };
  auto store = [&](int buf) {
    uint16_t* as = As[buf];
    uint16_t* bs = Bs[buf];
#pragma unroll
    for (int j = 0; j < NA; ++j) {
      const int c = tid + 256 * j;
      if (A_CH % 256 && c >= A_CH) continue;
      if (AL == AL_BITS) {
        const int r = c / (KB / 32), kc = 32 * (c % (KB / 32));
#pragma unroll
        for (int q = 0; q < 4; ++q)
          *reinterpret_cast<uint4*>(as + r * ROW + kc + 8 * q) = bit_oct(rw[j] >> (8 * q));
      } else {
        const int r = c / (KB / 8), kc = 8 * (c % (KB / 8));
        *reinterpret_cast<uint4*>(as + r * ROW + kc) = ra[j];
      }
    }
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      const int c = tid + 256 * j;
      if (B_CH % 256 && c >= B_CH) continue;
      const int nn = c / (KB / 8), kc = 8 * (c % (KB / 8));
      *reinterpret_cast<uint4*>(bs + nn * ROW + kc) = rb[j];
    }
  };

  const int n = n0 + wn * 32 + (lane & 31);
  const float bn = g.bias[n];        // loaded beside the first stage
  f32x16_t acc;
#pragma unroll
  for (int v = 0; v < 16; ++v) acc[v] = 0.f;
  const int nk = g.K / KB;
  load(0);
  store(0);
  __syncthreads();
  for (int t = 0; t < nk; ++t) {
    const int buf = t & 1;
    if (t + 1 < nk) load((t + 1) * KB);
    const uint16_t* ar = &As[buf][(wm * 32 + (lane & 31)) * ROW];
    const uint16_t* br = &Bs[buf][(wn * 32 + (lane & 31)) * ROW];
#pragma unroll
    for (int ks = 0; ks < KB; ks += 16) {
      const int kk = ks + 8 * (lane >> 5);
      const bf16x8_t a = *reinterpret_cast<const bf16x8_t*>(ar + kk);
      const bf16x8_t b = *reinterpret_cast<const bf16x8_t*>(br + kk);
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc, 0, 0, 0);
    }
    if (t + 1 < nk) store(buf ^ 1);
    __syncthreads();
  }
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    const uint64_t m = m0 + (uint64_t)(wm * 32 + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3));
    const float x = acc[v] + bn;
    if (m < g.M) {
      if constexpr (EP == E_BIAS_RELU_BF16) g.outb[(int64_t)m * g.ldo + n] = f2bf(x > 0.f ? x : 0.f);
      else g.outf[(int64_t)m * g.ldo + n] = x;
    }
  }
}

template <int AL, int EP, int WN, int KB>
void mm(svd_ctx* c, const MmArgs& g) {
  constexpr int TM = 128 / WN, TN = 32 * WN;
  if (g.N % TN || g.K % KB) throw Error{SVD_ERR_ARG, "mlp gemm: unsupported shape"};
  if (g.M == 0) return;
  const dim3 grid((uint32_t)div_up(g.M, (uint64_t)TM), (uint32_t)(g.N / TN));
  k_mm<AL, EP, WN, KB><<<grid, 256, 0, c->stream>>>(g);
}

// ---- the training step: three launches ------------------------------------------
// k_step: sampling, the three layers, the pair loss and the input gradients of
// 32 batch rows per workgroup, activations in LDS throughout; k_wgrad: the
// weight and bias gradients of all layers, split over the batch; k_adam: the
// optimizer and the bf16 weight copies.  One kernel per product took ten
// launches and 89 us per step of 4096 pairs, each bound by its own launch and
// load latency; the three take 41 us (19 + 12 + 9.5).
//
// What k_step leaves for k_wgrad is k-contiguous in the batch rows: matrices
// in row blocks of 32, element (n, row) at ((row / 32) N + n) 32 + row % 32,
// and the input bits as one word per (row block, input).  Batches are whole
// blocks (P is a multiple of 16).

// Fragment order of a B operand (K x N): the 8 values that lane l of the
// tile of columns t reads for K step s are element ((t K/16 + s) 64 + l) 8 + i.
__host__ __device__ inline uint64_t frag_pos(uint64_t k, uint64_t n, uint64_t K) {
  return (((n / 32) * (K / 16) + k / 16) * 64 + (n % 32) + 32 * ((k % 16) / 8)) * 8 + k % 8;
}

__device__ __forceinline__ uint64_t sm_next(uint64_t x) { return mix64(x + 0x9E3779B97F4A7C15ull); }

struct StepArgs {
  uint64_t P;                      // pairs
  // the batch: sampled from sig (n signatures, near-pair order and its
  // inverse, batch number *step), or given rows and labels (sig null)
  const uint32_t* sig; uint64_t n;
  const uint32_t* order; const uint32_t* pos;
  uint64_t seed; uint32_t nearPct;
  const uint32_t* step;
  const uint32_t* X; const uint32_t* labels;
  const uint16_t* wb; const float* params;
  uint32_t* xbits;                 // [block][512]
  uint16_t *h1, *h2, *dE, *dz2, *dz1;
  float* loss;                     // loss[*step] (loss[0] without step) += the batch loss
};

// The B fragments of one column tile, S K steps, in registers: loaded a stage
// ahead of their use, so that the weights' latency passes behind the work and
// the barriers before it.
template <int S>
struct Frags {
  bf16x8_t b[S];
  __device__ __forceinline__ void load(const uint16_t* frag, int lane) {
    const bf16x8_t* p = reinterpret_cast<const bf16x8_t*>(frag) + lane;
#pragma unroll
    for (int s = 0; s < S; ++s) b[s] = p[64 * s];
  }
  // the 32 x 32 tile with the A rows in LDS (row stride `ars` elements)
  __device__ __forceinline__ f32x16_t product(const uint16_t* arows, int ars, int lane) const {
    f32x16_t acc;
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[v] = 0.f;
    const uint16_t* ar = arows + (lane & 31) * ars + 8 * (lane >> 5);
#pragma unroll
    for (int s = 0; s < S; ++s)
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*reinterpret_cast<const bf16x8_t*>(ar + 16 * s), b[s], acc, 0, 0, 0);
    return acc;
  }
};

// Column n of a 32 x 32 tile (rounded values o[v] of a lane) into LDS rows
// (optional) and the row block's global column.
__device__ __forceinline__ void put_tile(const uint16_t o[16], int n, int N, uint64_t block, int half, uint16_t* lds,
                                         int rs, uint16_t* __restrict__ out) {
  uint16_t* col = out + (block * N + n) * 32 + 4 * half;
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const uint32_t lo = o[4 * g] | ((uint32_t)o[4 * g + 1] << 16), hi = o[4 * g + 2] | ((uint32_t)o[4 * g + 3] << 16);
    *reinterpret_cast<uint2*>(col + 8 * g) = make_uint2(lo, hi);
    if (lds) {
#pragma unroll
      for (int i = 0; i < 4; ++i) lds[(8 * g + 4 * half + i) * rs + n] = o[4 * g + i];
    }
  }
}

// Eight wavefronts, 16 pairs.  Layer 1 has a column tile per wavefront, layer
// 2 and its input gradient four, layer 3 one; every product reads the weights
// in fragment order straight from L2 (1 KB coalesced per K step).  256
// workgroups at 4096 pairs are one per CU, so the registers of two wavefronts
// per SIMD are free for the weights.
__global__ void __launch_bounds__(512, 2) k_step(StepArgs g) {
  constexpr int R0 = D0 + 8, R1 = D1 + 8, R2 = D2 + 8, R3 = D3 + 8;   // padded LDS rows
  __shared__ __attribute__((aligned(16))) uint16_t xs[32 * R0];
  __shared__ __attribute__((aligned(16))) uint16_t h1s[32 * R1];
  __shared__ __attribute__((aligned(16))) uint16_t h2s[32 * R2];
  __shared__ __attribute__((aligned(16))) uint16_t dEs[32 * R3];
  __shared__ __attribute__((aligned(16))) uint16_t dz2s[32 * R2];
  __shared__ __attribute__((aligned(16))) uint32_t bits[32][16];
  __shared__ uint32_t label[16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, half = lane >> 5;
  const uint64_t block = blockIdx.x, p0 = block * 16;
  const uint32_t step = g.step ? *g.step : 0u;
  const int w4 = wave & 3;           // the column tile of the four-tile products
  Frags<D0 / 16> f1;
  f1.load(g.wb + WF_W1 + (uint64_t)wave * 32 * D0, lane);
  const float bias1 = g.params[OFF_B1 + 32 * wave + (lane & 31)];
  if (tid < 64) {
    // four lanes per pair, a quarter of both signatures each
    const uint64_t p = p0 + (tid >> 2);
    const int q = tid & 3;
    uint4 u = make_uint4(0, 0, 0, 0), w = u;
    uint32_t lab = 0;
    if (g.sig) {
      // nearPct percent are neighbours (+-1..8) in the near-pair order, the
      // rest random
      const uint64_t gidx = (uint64_t)step * g.P + p;
      const uint64_t z1 = mix64(g.seed ^ ((gidx + 1) * 0x9E3779B97F4A7C15ull));
      const uint64_t z2 = sm_next(z1);
      const uint64_t a = z1 % g.n;
      uint64_t b;
      if ((p * 37u) % 100u >= g.nearPct) {
        b = z2 % g.n;
      } else {
        int64_t d = (int64_t)(z2 % 16) - 8;
        if (d >= 0) d += 1;
        int64_t o = (int64_t)g.pos[a] + d;
        o = o < 0 ? 0 : (o >= (int64_t)g.n ? (int64_t)g.n - 1 : o);
        b = g.order[o];
      }
      u = reinterpret_cast<const uint4*>(g.sig + a * 16)[q];
      w = reinterpret_cast<const uint4*>(g.sig + b * 16)[q];
      lab = __popc(u.x ^ w.x) + __popc(u.y ^ w.y) + __popc(u.z ^ w.z) + __popc(u.w ^ w.w);
    } else {
      u = reinterpret_cast<const uint4*>(g.X + 2 * p * 16)[q];
      w = reinterpret_cast<const uint4*>(g.X + (2 * p + 1) * 16)[q];
      lab = q == 0 ? g.labels[p] : 0u;
    }
    lab += __shfl_xor(lab, 1, 64);
    lab += __shfl_xor(lab, 2, 64);
    if (q == 0) label[tid >> 2] = lab;
    *reinterpret_cast<uint4*>(&bits[2 * (tid >> 2)][4 * q]) = u;
    *reinterpret_cast<uint4*>(&bits[2 * (tid >> 2) + 1][4 * q]) = w;
  }
  __syncthreads();
  {
    const uint32_t w = bits[tid >> 4][tid & 15];
    uint16_t* x = xs + (tid >> 4) * R0 + 32 * (tid & 15);
#pragma unroll
    for (int q = 0; q < 4; ++q) *reinterpret_cast<uint4*>(x + 8 * q) = bit_oct(w >> (8 * q));
    uint32_t t = 0;                  // input tid of the block's 32 rows
    for (int r = 0; r < 32; ++r) t |= ((bits[r][tid >> 5] >> (tid & 31)) & 1u) << r;
    g.xbits[block * D0 + tid] = t;
  }
  __syncthreads();
  uint16_t o[16];
  {
    const int n = 32 * wave + (lane & 31);
    const f32x16_t acc = f1.product(xs, R0, lane);
#pragma unroll
    for (int v = 0; v < 16; ++v) { const float z = acc[v] + bias1; o[v] = f2bf(z > 0.f ? z : 0.f); }
    put_tile(o, n, D1, block, half, h1s, R1, g.h1);
  }
  Frags<D1 / 16> f2;
  f2.load(g.wb + WF_W2 + (uint64_t)w4 * 32 * D1, lane);
  const float bias2 = g.params[OFF_B2 + 32 * w4 + (lane & 31)], bias3 = g.params[OFF_B3 + (lane & 31)];
  __syncthreads();
  Frags<D2 / 16> f3, f2t;
  Frags<D3 / 16> f3t;
  f3.load(g.wb + WF_W3, lane);
  f3t.load(g.wb + WF_W3T + (uint64_t)w4 * 32 * D3, lane);
  f2t.load(g.wb + WF_W2T + (uint64_t)wave * 32 * D2, lane);
  if (wave < D2 / 32) {
    const int n = 32 * wave + (lane & 31);
    const f32x16_t acc = f2.product(h1s, R1, lane);
#pragma unroll
    for (int v = 0; v < 16; ++v) { const float z = acc[v] + bias2; o[v] = f2bf(z > 0.f ? z : 0.f); }
    put_tile(o, n, D2, block, half, h2s, R2, g.h2);
  }
  __syncthreads();
  if (wave == 0) {
    // rows 2p and 2p+1 are accumulator elements v and v+1 (v even) of a lane;
    // d = |e_a - e_b|^2 is summed over the 32 lanes of a half-wavefront
    const int n = lane & 31;
    const float bn = bias3;
    const f32x16_t acc = f3.product(h2s, R2, lane);
    const float invP = 1.0f / (float)g.P;
    float lsum = 0.f;
#pragma unroll
    for (int v = 0; v < 16; v += 2) {
      const int m = 8 * (v >> 2) + 4 * half + (v & 3);
      const float diff = (acc[v] + bn) - (acc[v + 1] + bn);
      float d = diff * diff;
#pragma unroll
      for (int q = 16; q >= 1; q >>= 1) d += __shfl_xor(d, q, 64);
      const float y = fminf((float)label[m >> 1], kHCap);
      const float gr = 2.f * (d - y) * invP;
      o[v] = f2bf(2.f * gr * diff);
      o[v + 1] = (uint16_t)(o[v] ^ 0x8000u);     // bf16(-x) = -bf16(x)
      lsum += (d - y) * (d - y) * invP;
    }
    put_tile(o, n, D3, block, half, dEs, R3, g.dE);
    if (n == 0) atomicAdd(&g.loss[step], lsum);
  }
  __syncthreads();
  if (wave < D2 / 32) {
    const int n = 32 * wave + (lane & 31);
    const f32x16_t acc = f3t.product(dEs, R3, lane);
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int m = 8 * (v >> 2) + 4 * half + (v & 3);
      o[v] = bf2f(h2s[m * R2 + n]) > 0.f ? f2bf(acc[v]) : (uint16_t)0;
    }
    put_tile(o, n, D2, block, half, dz2s, R2, g.dz2);
  }
  __syncthreads();
  {
    const int n = 32 * wave + (lane & 31);
    const f32x16_t acc = f2t.product(dz2s, R2, lane);
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int m = 8 * (v >> 2) + 4 * half + (v & 3);
      o[v] = bf2f(h1s[m * R1 + n]) > 0.f ? f2bf(acc[v]) : (uint16_t)0;
    }
    put_tile(o, n, D1, block, half, nullptr, 0, g.dz1);
  }
}

// Weight gradients dW = A^T dz: M x N is small and K (the rows of the batch)
// long, so K is split over about kWgradBlocks workgroups; each split writes
// its partial tile and the optimizer (or the gradient read-out) sums the
// splits in order (deterministic, no atomics).
constexpr int kSplitUnit = 128;
constexpr uint64_t kWgradBlocks = 512;
constexpr int kMaxSplits = 32;
struct Split { int S, kPer; };
Split wgrad_split(uint64_t M, int N, int K, int TM, int TN) {
  const uint64_t tiles = div_up(M, (uint64_t)TM) * (uint64_t)(N / TN);
  const int maxS = M * (uint64_t)N <= 16384 ? 2 * kMaxSplits : kMaxSplits;   // small partials: split further
  int S = (int)std::min<uint64_t>(maxS, std::max<uint64_t>(1, kWgradBlocks / tiles));
  S = std::min(S, std::max(1, (K + kSplitUnit - 1) / kSplitUnit));
  int kPer = (K + S - 1) / S;
  kPer = (kPer + kSplitUnit - 1) / kSplitUnit * kSplitUnit;
  return Split{(K + kPer - 1) / kPer, kPer};
}

struct WgradArgs {
  int K;                           // batch rows
  const uint32_t* xbits;
  const uint16_t *h1, *h2, *dE, *dz2, *dz1;
  int kPer[3];
  uint32_t wgs[3];                 // workgroups of layers 1..3, in this order
  float* part[3];                  // split z: part + z M N (row-major)
  float* partBias[3];              // split z: + z N
  uint32_t* step;                  // optional: step[1] = step[0]++ (the optimizer's step and the next batch's)
};

// One TM x TN tile over the rows [kBeg, kEnd): four wavefronts of 32 x 32.
// The blocked layouts give every lane its fragments as 16-byte pieces of whole
// 64-byte rows, so both operands go from L2 straight to registers, several row
// blocks ahead, with no LDS and no barriers.  The bias gradient is the column
// sum of B, taken by the first row of wavefronts.
template <int M, int N, int WN, bool BITS>
__device__ __forceinline__ void wgrad_tile(const WgradArgs& g, const void* a, const uint16_t* b, int kPer, float* part,
                                           float* partBias, uint32_t wg) {
  constexpr int WM = 4 / WN, TM = 32 * WM, TN = 32 * WN;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, wm = wave % WM, wn = wave / WM, half = lane >> 5;
  const uint32_t mt = wg % (M / TM), nt = wg / (M / TM) % (N / TN), z = wg / ((M / TM) * (N / TN));
  const int m = (int)mt * TM + wm * 32 + (lane & 31), n = (int)nt * TN + wn * 32 + (lane & 31);
  const int kBeg = (int)z * kPer, kEnd = min(g.K, kBeg + kPer);
  const bool colSums = mt == 0 && wm == 0;
  f32x16_t acc;
#pragma unroll
  for (int v = 0; v < 16; ++v) acc[v] = 0.f;
  float colAcc = 0.f;
  const uint4* pb = reinterpret_cast<const uint4*>(b + (uint64_t)n * 32 + 8 * half);
  const uint4* pa = reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(a) + (uint64_t)m * 32 + 8 * half);
  const uint32_t* px = static_cast<const uint32_t*>(a) + m;
  // `count` row blocks from blk on, all their loads first
  auto blocks = [&](int blk, auto count) {
    constexpr int U = decltype(count)::value;
    uint4 a0[U], a1[U], b0[U], b1[U];
    uint32_t w[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint64_t k = (uint64_t)(blk + u);
      b0[u] = pb[k * (N * 4)];
      b1[u] = pb[k * (N * 4) + 2];
      if constexpr (BITS) {
        w[u] = px[k * M];
      } else {
        a0[u] = pa[k * (M * 4)];
        a1[u] = pa[k * (M * 4) + 2];
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if constexpr (BITS) {
        a0[u] = bit_oct(w[u] >> (8 * half));
        a1[u] = bit_oct(w[u] >> (16 + 8 * half));
      }
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a0[u]),
                                                    __builtin_bit_cast(bf16x8_t, b0[u]), acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a1[u]),
                                                    __builtin_bit_cast(bf16x8_t, b1[u]), acc, 0, 0, 0);
      if (colSums) {
        const uint32_t e[8] = {b0[u].x, b0[u].y, b0[u].z, b0[u].w, b1[u].x, b1[u].y, b1[u].z, b1[u].w};
#pragma unroll
        for (int i = 0; i < 8; ++i) colAcc += __uint_as_float(e[i] << 16) + __uint_as_float(e[i] & 0xFFFF0000u);
      }
    }
  };
  int blk = kBeg / 32;
  for (; blk + 4 <= kEnd / 32; blk += 4) blocks(blk, std::integral_constant<int, 4>());
  for (; blk < kEnd / 32; ++blk) blocks(blk, std::integral_constant<int, 1>());
  float* out = part + (uint64_t)z * M * N + (uint64_t)(m - (lane & 31)) * N + n;
#pragma unroll
  for (int v = 0; v < 16; ++v) out[(uint64_t)(8 * (v >> 2) + 4 * half + (v & 3)) * N] = acc[v];
  if (colSums) {
    colAcc += __shfl_xor(colAcc, 32, 64);
    if (half == 0) partBias[(uint64_t)z * N + n] = colAcc;
  }
}

// The three layers' tiles in one launch: 64 x 64 tiles for layers 1 and 2,
// 128 x 32 for layer 3.
__global__ void __launch_bounds__(256) k_wgrad(WgradArgs g) {
  uint32_t wg = blockIdx.x;
  if (g.step && wg == 0 && threadIdx.x == 0) {
    const uint32_t s = g.step[0];
    g.step[1] = s;
    g.step[0] = s + 1u;
  }
  if (wg < g.wgs[0]) return wgrad_tile<D0, D1, 2, true>(g, g.xbits, g.dz1, g.kPer[0], g.part[0], g.partBias[0], wg);
  wg -= g.wgs[0];
  if (wg < g.wgs[1]) return wgrad_tile<D1, D2, 2, false>(g, g.h1, g.dz2, g.kPer[1], g.part[1], g.partBias[1], wg);
  wgrad_tile<D2, D3, 1, false>(g, g.h2, g.dE, g.kPer[2], g.part[2], g.partBias[2], wg - g.wgs[1]);
}

// The split partial gradients of the three layers.
struct GradParts {
  const float* w[3];
  const float* b[3];
  uint32_t S[3];
};

__device__ __forceinline__ float grad_sum(const GradParts& gp, uint64_t i) {
  constexpr uint64_t offW[3] = {OFF_W1, OFF_W2, OFF_W3}, offB[3] = {OFF_B1, OFF_B2, OFF_B3};
  constexpr uint64_t dout[3] = {D1, D2, D3}, din[3] = {D0, D1, D2};
  const int l = i < OFF_W2 ? 0 : (i < OFF_W3 ? 1 : 2);
  const bool isB = i >= offB[l];
  const float* p = isB ? gp.b[l] + (i - offB[l]) : gp.w[l] + (i - offW[l]);
  const uint64_t stride = isB ? dout[l] : din[l] * dout[l];
  // splits in order; eight loads in flight at a time
  float s = 0.f;
  uint32_t z = 0;
  for (; z + 8 <= gp.S[l]; z += 8) {
    float x[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) x[q] = p[(z + q) * stride];
#pragma unroll
    for (int q = 0; q < 8; ++q) s += x[q];
  }
  for (; z < gp.S[l]; ++z) s += p[z * stride];
  return s;
}

__global__ void k_grad_sum(GradParts gp, float* __restrict__ grads) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < N_PARAMS) grads[i] = grad_sum(gp, i);
}

// bf16 copies of weight parameter i (a no-op for the biases, which stay fp32).
__device__ __forceinline__ void store_wb(uint16_t* __restrict__ wb, uint64_t i, float w) {
  constexpr uint64_t offW[3] = {OFF_W1, OFF_W2, OFF_W3}, offB[3] = {OFF_B1, OFF_B2, OFF_B3};
  constexpr uint64_t offWb[3] = {WB_W1, WB_W2, WB_W3}, offF[3] = {WF_W1, WF_W2, WF_W3};
  constexpr uint64_t dout[3] = {D1, D2, D3}, din[3] = {D0, D1, D2};
  const int l = i < OFF_W2 ? 0 : (i < OFF_W3 ? 1 : 2);
  if (i >= offB[l]) return;
  const uint64_t j = i - offW[l], k = j / dout[l], n = j % dout[l];
  const uint16_t v = f2bf(w);
  wb[offWb[l] + n * din[l] + k] = v;
  wb[offF[l] + frag_pos(k, n, din[l])] = v;
  // the input gradient's operand is the transpose: K = out, N = in
  if (l == 1) wb[WF_W2T + frag_pos(n, k, D2)] = v;
  if (l == 2) wb[WF_W3T + frag_pos(n, k, D3)] = v;
}

// Adam on the gradients summed from the split partials, at step
// step0 + *step + 1 (bias correction).
__global__ void k_adam(float* __restrict__ w, GradParts gp, float* __restrict__ m, float* __restrict__ v,
                       uint16_t* __restrict__ wb, const uint32_t* __restrict__ step, uint32_t step0, float lr) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= N_PARAMS) return;
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  const float t = (float)(step0 + *step + 1u);
  const float gi = grad_sum(gp, i);
  const float mi = b1 * m[i] + (1.f - b1) * gi;
  const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
  m[i] = mi; v[i] = vi;
  const float mh = mi / (1.f - powf(b1, t));
  const float vh = vi / (1.f - powf(b2, t));
  const float wn = w[i] - lr * mh / (sqrtf(vh) + eps);
  w[i] = wn;
  store_wb(wb, i, wn);
}

__global__ void k_refresh_wb(const float* __restrict__ w, uint16_t* __restrict__ wb) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < N_PARAMS) store_wb(wb, i, w[i]);
}

__global__ void k_set_u32(uint32_t* d, uint32_t v) { *d = v; }
__global__ void k_zero_f32(float* d, uint64_t n) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) d[i] = 0.f;
}

// Near-pair ordering key: popcount in the high bits, then 22 sampled bits.
__global__ void k_pair_keys(const uint32_t* __restrict__ sig, uint64_t n, const uint32_t* __restrict__ bitpos,
                            uint32_t* __restrict__ keys, uint32_t* __restrict__ vals) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint32_t* s = sig + i * 16;
  uint32_t pc = 0;
#pragma unroll
  for (int w = 0; w < 16; ++w) pc += __popc(s[w]);
  uint32_t k = pc << 22;
  for (int b = 0; b < 22; ++b) {
    const uint32_t q = bitpos[b];
    k |= ((s[q >> 5] >> (q & 31)) & 1u) << b;
  }
  keys[i] = k;
  vals[i] = (uint32_t)i;
}

__global__ void k_inverse_perm(const uint32_t* __restrict__ order, uint64_t n, uint32_t* __restrict__ pos) {
  const uint64_t q = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q < n) pos[order[q]] = (uint32_t)q;
}

// Working buffers of one forward/backward over R = 2P rows.
struct Work {
  uint64_t R = 0;              // rows, a multiple of 32
  uint32_t* xbits = nullptr;
  uint16_t *h1 = nullptr, *h2 = nullptr, *dE = nullptr, *dz2 = nullptr, *dz1 = nullptr;
  Split sp[3] = {};            // weight-gradient splits of layers 1..3
  uint32_t wgs[3] = {};
  float* partW[3] = {};
  float* partB[3] = {};
  void alloc(svd_ctx* c, uint64_t rows) {
    if (rows % 32 || rows > 0x7FFFFFFFull) throw Error{SVD_ERR_ARG, "a batch is a multiple of 16 pairs, below 2^30"};
    R = rows;
    xbits = dalloc<uint32_t>(c, R / 32 * D0);
    h1 = dalloc<uint16_t>(c, R * D1); h2 = dalloc<uint16_t>(c, R * D2);
    dE = dalloc<uint16_t>(c, R * D3); dz2 = dalloc<uint16_t>(c, R * D2); dz1 = dalloc<uint16_t>(c, R * D1);
    const int din[3] = {D0, D1, D2}, dout[3] = {D1, D2, D3};
    for (int l = 0; l < 3; ++l) {
      const int wn = dout[l] % 64 ? 1 : 2, tm = 128 / wn, tn = 32 * wn;
      sp[l] = wgrad_split(din[l], dout[l], (int)R, tm, tn);
      wgs[l] = (uint32_t)((din[l] / tm) * (dout[l] / tn) * sp[l].S);
      partW[l] = dalloc<float>(c, (uint64_t)sp[l].S * din[l] * dout[l]);
      partB[l] = dalloc<float>(c, (uint64_t)sp[l].S * dout[l]);
    }
  }
  GradParts parts() const {
    GradParts gp;
    for (int l = 0; l < 3; ++l) { gp.w[l] = partW[l]; gp.b[l] = partB[l]; gp.S[l] = (uint32_t)sp[l].S; }
    return gp;
  }
  void release(svd_ctx* c) {
    dfree(c, xbits); dfree(c, h1); dfree(c, h2); dfree(c, dE); dfree(c, dz2); dfree(c, dz1);
    for (int l = 0; l < 3; ++l) { dfree(c, partW[l]); dfree(c, partB[l]); }
  }
};

// Forward: the embeddings e (fp32) of `rows` signatures.
void forward(svd_mlp* m, const uint32_t* X, uint64_t rows, uint16_t* h1, uint16_t* h2, float* e) {
  svd_ctx* c = m->ctx;
  MmArgs g = {};
  g.M = rows; g.N = D1; g.K = D0;
  g.abits = X; g.b = m->wb + WB_W1; g.ldb = D0; g.bias = m->params + OFF_B1; g.outb = h1; g.ldo = D1;
  mm<AL_BITS, E_BIAS_RELU_BF16, 2, 128>(c, g);
  g = {};
  g.M = rows; g.N = D2; g.K = D1;
  g.a = h1; g.lda = D1; g.b = m->wb + WB_W2; g.ldb = D1; g.bias = m->params + OFF_B2; g.outb = h2; g.ldo = D2;
  mm<AL_MK, E_BIAS_RELU_BF16, 2, 128>(c, g);
  g = {};
  g.M = rows; g.N = D3; g.K = D2;
  g.a = h2; g.lda = D2; g.b = m->wb + WB_W3; g.ldb = D2; g.bias = m->params + OFF_B3; g.outf = e; g.ldo = D3;
  mm<AL_MK, E_BIAS_F32, 1, 128>(c, g);
}

// Forward, pair loss and backward of one batch into the split partial
// gradients of w.  s carries the batch; step (optional, two device words) is
// advanced for the optimizer.
void forward_backward(svd_mlp* m, StepArgs s, const Work& w, uint32_t* step) {
  svd_ctx* c = m->ctx;
  s.wb = m->wb; s.params = m->params; s.step = step;
  s.xbits = w.xbits; s.h1 = w.h1; s.h2 = w.h2; s.dE = w.dE; s.dz2 = w.dz2; s.dz1 = w.dz1;
  k_step<<<(uint32_t)(w.R / 32), 512, 0, c->stream>>>(s);
  WgradArgs g = {};
  g.K = (int)w.R;
  g.xbits = w.xbits; g.h1 = w.h1; g.h2 = w.h2; g.dE = w.dE; g.dz2 = w.dz2; g.dz1 = w.dz1;
  for (int l = 0; l < 3; ++l) { g.kPer[l] = w.sp[l].kPer; g.wgs[l] = w.wgs[l]; g.part[l] = w.partW[l]; g.partBias[l] = w.partB[l]; }
  g.step = step;
  k_wgrad<<<w.wgs[0] + w.wgs[1] + w.wgs[2], 256, 0, c->stream>>>(g);
}

}  // namespace

// Weights: Glorot uniform from a SplitMix64 stream (w = (2u - 1) a,
// u = (z >> 40) 2^-24, a = sqrt(6 / (fan_in + fan_out)) in fp32), zero biases.
void mlp_init(svd_mlp* m, uint64_t seed) {
  svd_ctx* c = m->ctx;
  std::vector<float> h(N_PARAMS, 0.f);
  const int dims[4] = {D0, D1, D2, D3};
  uint64_t state = seed, o = 0;
  for (int l = 0; l < 3; ++l) {
    const uint64_t fi = dims[l], fo = dims[l + 1], n = fi * fo;
    const float a = std::sqrt(6.0f / (float)(fi + fo));
    for (uint64_t i = 1; i <= n; ++i) {
      uint64_t z = state + i * 0x9E3779B97F4A7C15ull;
      z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
      z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
      z ^= z >> 31;
      const float u = (float)(z >> 40) * (1.0f / 16777216.0f);
      h[o + i - 1] = (u * 2.0f - 1.0f) * a;
    }
    state += n * 0x9E3779B97F4A7C15ull;
    o += n + fo;
  }
  SVD_HIP(hipMemcpyAsync(m->params, h.data(), N_PARAMS * 4, hipMemcpyHostToDevice, c->stream));
  k_refresh_wb<<<div_up(N_PARAMS, 256), 256, 0, c->stream>>>(m->params, m->wb);
  k_zero_f32<<<div_up(N_PARAMS, 256), 256, 0, c->stream>>>(m->m, N_PARAMS);
  k_zero_f32<<<div_up(N_PARAMS, 256), 256, 0, c->stream>>>(m->v, N_PARAMS);
  k_zero_f32<<<div_up(N_PARAMS, 256), 256, 0, c->stream>>>(m->grads, N_PARAMS);
  check_launch("mlp init");
  SVD_HIP(hipStreamSynchronize(c->stream));
  m->steps = 0;
}

void mlp_alloc(svd_mlp* m) {
  svd_ctx* c = m->ctx;
  m->params = dalloc<float>(c, N_PARAMS);
  m->grads = dalloc<float>(c, N_PARAMS);
  m->m = dalloc<float>(c, N_PARAMS);
  m->v = dalloc<float>(c, N_PARAMS);
  m->wb = dalloc<uint16_t>(c, N_WB_ALL);
}

void mlp_release(svd_mlp* m) {
  svd_ctx* c = m->ctx;
  dfree(c, m->params); dfree(c, m->grads); dfree(c, m->m); dfree(c, m->v); dfree(c, m->wb);
}

void mlp_set_params(svd_mlp* m, const float* host) {
  svd_ctx* c = m->ctx;
  SVD_HIP(hipMemcpyAsync(m->params, host, N_PARAMS * 4, hipMemcpyHostToDevice, c->stream));
  k_refresh_wb<<<div_up(N_PARAMS, 256), 256, 0, c->stream>>>(m->params, m->wb);
  check_launch("k_refresh_wb");
  SVD_HIP(hipStreamSynchronize(c->stream));
}

void mlp_get_params(svd_mlp* m, float* host) {
  svd_ctx* c = m->ctx;
  SVD_HIP(hipMemcpyAsync(host, m->params, N_PARAMS * 4, hipMemcpyDeviceToHost, c->stream));
  SVD_HIP(hipStreamSynchronize(c->stream));
}

void mlp_embed(svd_mlp* m, const uint32_t* sig, uint64_t n, float* emb) {
  svd_ctx* c = m->ctx;
  const uint64_t chunk = 1ull << 18;
  const uint64_t rows = n < chunk ? n : chunk;
  uint16_t* h1 = dalloc<uint16_t>(c, (rows + 32) * D1);
  uint16_t* h2 = dalloc<uint16_t>(c, (rows + 32) * D2);
  for (uint64_t r0 = 0; r0 < n; r0 += chunk) {
    const uint64_t r = n - r0 < chunk ? n - r0 : chunk;
    forward(m, sig + r0 * 16, r, h1, h2, emb + r0 * D3);
  }
  check_launch("mlp forward");
  dfree(c, h1); dfree(c, h2);
}

void mlp_loss_grad(svd_mlp* m, const uint32_t* X, const uint32_t* labels, uint64_t P, float* lossHost,
                   float* gradsHost) {
  svd_ctx* c = m->ctx;
  Work w;
  w.alloc(c, 2 * P);
  float* loss = dalloc<float>(c, 1);
  k_zero_f32<<<1, 32, 0, c->stream>>>(loss, 1);
  StepArgs s = {};
  s.P = P; s.X = X; s.labels = labels; s.loss = loss;
  forward_backward(m, s, w, nullptr);
  k_grad_sum<<<div_up(N_PARAMS, 256), 256, 0, c->stream>>>(w.parts(), m->grads);
  check_launch("mlp loss/grad");
  SVD_HIP(hipMemcpyAsync(lossHost, loss, 4, hipMemcpyDeviceToHost, c->stream));
  SVD_HIP(hipMemcpyAsync(gradsHost, m->grads, N_PARAMS * 4, hipMemcpyDeviceToHost, c->stream));
  SVD_HIP(hipStreamSynchronize(c->stream));
  dfree(c, loss);
  w.release(c);
}

// Pairs are drawn from the nodes of DAG levels lev_lo..lev_hi (signatures
// concatenated).  One step = sample -> forward -> loss -> backward -> Adam ->
// step counter, three launches.  They are enqueued one by one: the host runs
// ahead of a step's 40 us, while a captured step cost a gap of 8 - 11 us between
// two replays and its instantiation before the first.
void mlp_train(svd_mlp* m, svd_octree* o, const svd_mlp_train_params* p, svd_mlp_train_stats* st) {
  svd_ctx* c = m->ctx;
  if (o->state != SVD_S_DAG && o->state != SVD_S_SDAG) throw Error{SVD_ERR_STATE, "training needs the DAG"};
  if (p->lev_lo > p->lev_hi || p->lev_hi + 1 >= o->levels) throw Error{SVD_ERR_ARG, "training levels out of range"};
  if (p->pairs_per_step < 16 || p->pairs_per_step % 16 || p->steps < 1) throw Error{SVD_ERR_ARG, "pairs_per_step must be a multiple of 16, steps >= 1"};
  uint64_t n = 0;
  for (uint32_t l = p->lev_lo; l <= p->lev_hi; ++l) n += o->dag[l].n;
  if (n < 2) throw Error{SVD_ERR_ARG, "not enough nodes to sample pairs from"};
  if (n >= 0xFFFFFFFFull) throw Error{SVD_ERR_CAPACITY, "too many nodes"};
  const uint64_t P = p->pairs_per_step, R = 2 * P;
  const uint32_t nearPct = p->near_pct ? (p->near_pct > 100 ? 100 : p->near_pct) : 50;
  uint32_t* sig = dalloc<uint32_t>(c, n * 16);
  {
    uint64_t off = 0;
    for (uint32_t l = p->lev_lo; l <= p->lev_hi; ++l) {
      lossy_signatures(o, l, sig + off * 16);
      off += o->dag[l].n;
    }
  }
  // near-pair ordering
  uint32_t* keys = dalloc<uint32_t>(c, n);
  uint32_t* vals = dalloc<uint32_t>(c, n);
  uint32_t* keys2 = dalloc<uint32_t>(c, n);
  uint32_t* order = dalloc<uint32_t>(c, n);
  uint32_t* pos = dalloc<uint32_t>(c, n);
  uint32_t* bitpos = dalloc<uint32_t>(c, 22);
  uint32_t hb[22];                            // read by a copy of the stream: lives to the end
  {
    uint64_t s = p->seed ^ 0x5851F42D4C957F2Dull;
    for (int b = 0; b < 22; ++b) {
      s += 0x9E3779B97F4A7C15ull;
      uint64_t z = s;
      z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
      z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
      z ^= z >> 31;
      hb[b] = (uint32_t)(z % 512);
    }
    SVD_HIP(hipMemcpyAsync(bitpos, hb, sizeof(hb), hipMemcpyHostToDevice, c->stream));
    k_pair_keys<<<div_up(n, 256), 256, 0, c->stream>>>(sig, n, bitpos, keys, vals);
    size_t bytes = 0;
    SVD_HIP(rocprim::radix_sort_pairs(nullptr, bytes, keys, keys2, vals, order, (size_t)n, 0, 32, c->stream));
    void* tmp = c->arena->get(bytes + 16);
    SVD_HIP(rocprim::radix_sort_pairs(tmp, bytes, keys, keys2, vals, order, (size_t)n, 0, 32, c->stream));
    c->arena->put(tmp);
    k_inverse_perm<<<div_up(n, 256), 256, 0, c->stream>>>(order, n, pos);
    check_launch("pair ordering");
  }
  Work w;
  w.alloc(c, R);
  uint32_t* dstep = dalloc<uint32_t>(c, 2);   // batch counter, the current step's number
  float* lossHist = dalloc<float>(c, p->steps);
  k_zero_f32<<<div_up(p->steps, 256), 256, 0, c->stream>>>(lossHist, p->steps);
  k_set_u32<<<1, 1, 0, c->stream>>>(dstep, 0u);
  check_launch("train setup");
  // Adam's step index continues across calls (step0 + the batch counter),
  // the loss history starts at 0
  const uint32_t step0 = (uint32_t)m->steps;

  auto enqueue_step = [&]() {
    StepArgs s = {};
    s.P = P; s.sig = sig; s.n = n; s.order = order; s.pos = pos; s.seed = p->seed; s.nearPct = nearPct;
    s.loss = lossHist;
    forward_backward(m, s, w, dstep);
    k_adam<<<div_up(N_PARAMS, 256), 256, 0, c->stream>>>(m->params, w.parts(), m->m, m->v, m->wb, dstep + 1, step0,
                                                         p->lr);
  };
  {
    Timer t(c, "mlp_train");
    for (uint32_t s = 0; s < p->steps; ++s) enqueue_step();
  }
  check_launch("train steps");
  std::vector<float> hist(p->steps);
  SVD_HIP(hipMemcpyAsync(hist.data(), lossHist, p->steps * 4, hipMemcpyDeviceToHost, c->stream));
  SVD_HIP(hipStreamSynchronize(c->stream));
  m->steps += p->steps;
  if (st) {
    const uint32_t q = p->steps < 16 ? p->steps : 16;
    double a = 0, b = 0;
    for (uint32_t i = 0; i < q; ++i) { a += hist[i]; b += hist[p->steps - q + i]; }
    st->first_loss = (float)(a / q);
    st->last_loss = (float)(b / q);
    st->ms_train = timer_ms(c, "mlp_train");
    st->nodes = n;
    st->pairs = P * p->steps;
  }
  w.release(c);
  dfree(c, dstep); dfree(c, lossHist);
  dfree(c, sig); dfree(c, keys); dfree(c, vals); dfree(c, keys2); dfree(c, order); dfree(c, pos); dfree(c, bitpos);
}

}  // namespace svd
