// Learned warm start: kernels of the pressure-guess MLP (769 -> 512 -> 512 ->
// 256, GELU), BF16 operands on MFMA with FP32 accumulation, FP32 master
// weights.  No reference counterpart.
//
// GEMM: C[M x N] (fp32) = op(A) * op(B) (+ bias[N]) with op = identity or
// transpose, A/B bf16 row-major with leading dimensions, any M, N, K.
#include <hip/hip_runtime.h>

#include <stdint.h>

#include "cm_internal.h"

namespace cm {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;

__device__ __forceinline__ uint16_t f32_to_bf16(float x) {
  // round to nearest even; NaN kept quiet
  uint32_t u = __float_as_uint(x);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float bf16_to_f32(uint16_t h) { return __uint_as_float(((uint32_t)h) << 16); }

// GELU (tanh form) with the solver's tanh: g = 0.5 x (1 + tanh(c (x + 0.044715 x^3))).
__device__ __forceinline__ float gelu_tanh_arg(float x) { return 0.7978845608f * (x + 0.044715f * x * x * x); }
__device__ __forceinline__ float gelu(float x) { return 0.5f * x * (1.0f + tanhf(gelu_tanh_arg(x))); }
__device__ __forceinline__ float gelu_slope(float x) {
  const float t = tanhf(gelu_tanh_arg(x));
  const float dt = (1.0f - t * t) * 0.7978845608f * (1.0f + 3.0f * 0.044715f * x * x);
  return 0.5f * (1.0f + t) + 0.5f * x * dt;
}

// A workgroup owns a 64 x TN tile of C and walks K in steps of KS G: each of its
// G groups of 4 waves loads KS of them, and every element of C is one chain of
// products in the order of k, whatever G is (activations are rounded to BF16
// after the product: another order of its sum would move some of them by a whole
// BF16 step).  A step's elements are requested during the products of the step
// before it and reach LDS after them.  LDS holds both operands with k running
// along a row, as v_mfma_f32_16x16x32_bf16 takes them (8 consecutive k per lane,
// one 16-byte read); an operand that is contiguous the other way is loaded two k
// at a time and stored as pairs.  Words of a row are xor-ed with 8 x the row's
// block of 8: those stores, 8 rows apart from lane to lane, then reach all banks.
// Loads are 16 bytes at any alignment (769 inputs make odd leading dimensions), at
// the edges too, where they are moved inside the matrix and shifted back.
// Workgroups b, b + 8, ... of a launch share an XCD: they take consecutive tiles,
// so that its L2 reads few rows of A.
// Bound: the chain load -> LDS -> product of a step, 1 to 2 us when one wave per
// SIMD runs it.  The products of a training step have few tiles, so four groups
// load a 64 x 32 tile (16 waves, a quarter of the steps; eight of them then hold
// a 16 x 16 tile each) as long as every tile has a CU of its own: 104 KiB of LDS
// leave no room for a second.  With a tile more than that, 64 x 64 tiles by 4
// waves are faster.  M x 512 x 769: M = 1024 (256 tiles) 7.5 us against 10.4,
// M = 1536 (384) 12.9 against 10.4, M = 8192 46.9 against 23.2.
// Those take one step of 32 or 64 where K is no more: fewer loads, less LDS and, with
// no next step to hold, a quarter of the registers, so many more workgroups on a CU.
// 4096 x 4096 x 8 14.8 us (20.3 in steps of 64 with a next step), x 32 14.0 (19.5), x 64
// 15.1 (31.3 in steps of 128), 100000 x 256 x 32 17.9 (28.8); 2-byte loads and steps of 16
// took 16.1, 19.3, 26.9 and 29.0.
// Steps of 16 with 2-byte loads took 110 us at M = 1024; the eight products of a
// training step at batch 1024 take 47 us (713), 4096 x 4096 x 4096 0.32 ms.
constexpr int TM = 64, KPAD = 8;
// 32-bit words per LDS row of KS elements (32, 64 or 128)
constexpr int row_words(int KS) { return (KS + KPAD) / 2; }
template <int KS>
__device__ __forceinline__ int lds_word(int r, int c) {
  return r * row_words(KS) + (c ^ ((r >> 3 & (KS / 16 - 1)) << 3));
}

struct alignas(2) Elems8 {   // 8 elements at element alignment
  uint16_t v[8];
};
__device__ __forceinline__ uint4 vec8(const uint16_t *q) {
  return __builtin_bit_cast(uint4, *reinterpret_cast<const Elems8 *>(q));
}
// drop the first d of 8 elements, zeros move in
__device__ __forceinline__ uint4 drop(uint4 v, unsigned d) {
  uint64_t lo = (uint64_t)v.y << 32 | v.x, hi = (uint64_t)v.w << 32 | v.z;
  if (d >= 8) return make_uint4(0, 0, 0, 0);
  if (d >= 4) {
    lo = hi;
    hi = 0;
  }
  const unsigned n = 16 * (d & 3);
  if (n) {
    lo = lo >> n | hi << (64 - n);
    hi >>= n;
  }
  return make_uint4((uint32_t)lo, (uint32_t)(lo >> 32), (uint32_t)hi, (uint32_t)(hi >> 32));
}

// One operand's ROWS x KS tile: rows are m (or n), CONTIG_K when k runs along
// memory rows.  Each of a group's 256 threads holds kPieces pieces of 8 elements:
// along k, or (two k per thread) along the rows.  Rows past the matrix may hold
// anything, they reach no stored element; k past it is zero.
template <int ROWS, int KS, bool CONTIG_K>
struct Operand {
  static constexpr int kAll = ROWS * KS / 8 / 256;
  // two k at a time and one piece per thread: half of the threads hold two, the
  // others the same ones, which they do not store
  static constexpr bool kTwice = !CONTIG_K && kAll == 1;
  static constexpr int kPieces = kTwice ? 2 : kAll;
  static constexpr int kLanes = CONTIG_K ? KS / 8 : ROWS / 8;   // pieces along memory
  const uint16_t *p;
  int64_t ld;
  unsigned rows, K, r0;
  const uint16_t *at[kPieces];   // of the next step, all inside the matrix
  uint4 x[kPieces];

  __device__ __forceinline__ unsigned row(int i, int tid) const {
    return CONTIG_K ? r0 + (tid + 256 * i) / kLanes : r0 + 8 * (pair(i, tid) % kLanes);
  }
  __device__ __forceinline__ unsigned kofs(int i, int tid) const {
    return CONTIG_K ? 8 * ((tid + 256 * i) % kLanes) : 2 * (pair(i, tid) / kLanes) + (i & 1);
  }
  static __device__ __forceinline__ unsigned pair(int i, int tid) {
    return kTwice ? tid & 127 : tid + 256 * (i >> 1);
  }
  __device__ __forceinline__ void start(unsigned k0, int tid) {
#pragma unroll
    for (int i = 0; i < kPieces; ++i) {
      const unsigned r = row(i, tid), k = k0 + kofs(i, tid);
      at[i] = CONTIG_K ? p + (int64_t)(r < rows ? r : 0) * ld + k : p + (int64_t)k * ld + r;
    }
  }
  __device__ __forceinline__ void load(unsigned k0, int tid, int64_t advance) {
    if (k0 + KS <= K && (CONTIG_K || r0 + ROWS <= rows)) {
#pragma unroll
      for (int i = 0; i < kPieces; ++i) x[i] = vec8(at[i]);
    } else if (!CONTIG_K && r0 + ROWS <= rows) {   // whole lines, or none
#pragma unroll
      for (int i = 0; i < kPieces; ++i) {
        const unsigned r = row(i, tid), k = k0 + kofs(i, tid);
        x[i] = k < K ? vec8(p + (int64_t)k * ld + r) : make_uint4(0, 0, 0, 0);
      }
    } else {
#pragma unroll
      for (int i = 0; i < kPieces; ++i) {
        const unsigned r = row(i, tid), k = k0 + kofs(i, tid);
        x[i] = edge(CONTIG_K ? (r < rows ? r : 0) : r, k);
      }
    }
#pragma unroll
    for (int i = 0; i < kPieces; ++i) at[i] += advance;
  }
  // 8 elements from (r, k) along memory, zeros past its end or at k >= K
  __device__ __forceinline__ uint4 edge(unsigned r, unsigned k) const {
    const unsigned len = CONTIG_K ? K : rows, j = CONTIG_K ? k : r, line = CONTIG_K ? r : k < K ? k : 0;
    const uint16_t *q = p + (int64_t)line * ld;
    uint4 v;
    if (len >= 8) {
      const unsigned s = j + 8 <= len ? j : len - 8;
      v = drop(vec8(q + s), j - s);
    } else {
      uint32_t w[4] = {0, 0, 0, 0};
#pragma unroll
      for (unsigned e = 0; e < 8; ++e) w[e / 2] |= (j + e < len ? (uint32_t)q[j + e] : 0u) << 16 * (e & 1);
      v = make_uint4(w[0], w[1], w[2], w[3]);
    }
    return CONTIG_K || k < K ? v : make_uint4(0, 0, 0, 0);
  }
  __device__ __forceinline__ void store(uint32_t *lds, int tid) const {
    if (CONTIG_K) {
#pragma unroll
      for (int i = 0; i < kPieces; ++i) {
        const int e = tid + 256 * i;
        *reinterpret_cast<uint4 *>(lds + lds_word<KS>(e / kLanes, 4 * (e % kLanes))) = x[i];
      }
    } else if (!kTwice || tid < 128) {
#pragma unroll
      for (int i = 0; i < kPieces; i += 2) {
        const int e = tid + 256 * (i >> 1);
        uint32_t *q = lds + lds_word<KS>(8 * (e % kLanes), e / kLanes);
        const uint32_t a[4] = {x[i].x, x[i].y, x[i].z, x[i].w}, b[4] = {x[i + 1].x, x[i + 1].y, x[i + 1].z, x[i + 1].w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          q[(2 * j) * row_words(KS)] = __builtin_amdgcn_perm(b[j], a[j], 0x05040100u);       // low halves
          q[(2 * j + 1) * row_words(KS)] = __builtin_amdgcn_perm(b[j], a[j], 0x07060302u);   // high halves
        }
      }
    }
  }
};

// What a product's element becomes: itself, or with the activation of its layer
// (a pass over C and a launch less: 3.7 and 3.2 us each at 1024 x 512).
enum class End { plain, gelu, gelu_back };

struct GemmArgs {
  unsigned M, N, K;
  const uint16_t *A;
  int lda;
  const uint16_t *B;
  int ldb;
  float *C;
  int ldc;
  const float *bias;
  float beta;
  const float *Z;
  uint16_t *Cbf;
};
// Place of workgroup blk in the order of tiles that gives each XCD neighbours.
__device__ __forceinline__ unsigned xcd_order(unsigned blk, unsigned tiles) {
  const unsigned xcd = blk & 7, rem = tiles & 7;
  return xcd * (tiles >> 3) + (xcd < rem ? xcd : rem) + (blk >> 3);
}

template <int TN, int G, int KS, bool TA, bool TB, End END>
__device__ __forceinline__ void gemm_tile(const GemmArgs &g_, unsigned m0, unsigned n0) {
  const unsigned M = g_.M, N = g_.N, K = g_.K;
  if (KS < 128) __builtin_assume(K <= KS);   // one step
  const uint16_t *__restrict__ A = g_.A, *__restrict__ B = g_.B;
  const int lda = g_.lda, ldb = g_.ldb, ldc = g_.ldc;
  float *__restrict__ C = g_.C;
  const float *__restrict__ bias = g_.bias, *__restrict__ Z = g_.Z;
  const float beta = g_.beta;
  uint16_t *__restrict__ Cbf = g_.Cbf;
  constexpr int kTileWords = (TM + TN) * row_words(KS);
  // 16 x 16 tiles of a multiplying wave, and those waves' place in the tile
  constexpr int NI = G == 1 ? 2 : 1, NJ = G == 1 ? TN / 32 : 1, kWavesN = TN / (16 * NJ);
  constexpr int kWaves = TM / (16 * NI) * kWavesN;
  static_assert(kWaves <= 4 * G, "one wave per part of the tile");
  __shared__ __align__(16) uint32_t lds[G * kTileWords];
  const int tid = threadIdx.x & 255, lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), g = wave >> 2;
  const int wm = wave / kWavesN * 16 * NI, wn = wave % kWavesN * 16 * NJ;
  Operand<TM, KS, !TA> a{A, lda, M, K, m0, {}, {}};
  Operand<TN, KS, TB> b{B, ldb, N, K, n0, {}, {}};
  const int64_t adv_a = TA ? (int64_t)G * KS * lda : G * KS, adv_b = TB ? G * KS : (int64_t)G * KS * ldb;
  f32x4 acc[NI][NJ];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  uint32_t *const mine = lds + g * kTileWords;
  // lane l: A rows (B columns) l % 16, k = 8 (l / 16) .. + 7
  const int ar = wm + (lane & 15), br = wn + (lane & 15), kc = 4 * (lane >> 4);
  unsigned kg = g * KS;   // first k of this group's part of the step
  a.start(kg, tid);
  b.start(kg, tid);
  if (kg < K) {
    a.load(kg, tid, adv_a);
    b.load(kg, tid, adv_b);
  }
  for (unsigned k0 = 0; k0 < K; k0 += G * KS) {
    if (kg < K) {
      a.store(mine, tid);
      b.store(mine + TM * row_words(KS), tid);
    }
    kg += G * KS;
    __syncthreads();
    if (kg < K) {
      a.load(kg, tid, adv_a);
      b.load(kg, tid, adv_b);
    }
    if (wave < kWaves) {
#pragma unroll
      for (int h = 0; h < G; ++h) {
        if (k0 + h * KS >= K) break;
        const uint32_t *const ta = lds + h * kTileWords, *const tb = ta + TM * row_words(KS);
#pragma unroll
        for (int q = 0; q < KS / 32; ++q) {
          bf16x8 fa[NI], fb[NJ];
#pragma unroll
          for (int i = 0; i < NI; ++i)
            fa[i] =
                __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4 *>(ta + lds_word<KS>(ar + 16 * i, kc + 16 * q)));
#pragma unroll
          for (int j = 0; j < NJ; ++j)
            fb[j] =
                __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4 *>(tb + lds_word<KS>(br + 16 * j, kc + 16 * q)));
#pragma unroll
          for (int i = 0; i < NI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j)
              acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[i], fb[j], acc[i][j], 0, 0, 0);
        }
      }
    }
    __syncthreads();
  }
  if (wave >= kWaves) return;
  // lane l holds C rows 4*(l/16)..+3, column l%16 of each 16 x 16 tile
  const int cn = lane & 15, cm = (lane >> 4) * 4;
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const unsigned gm = m0 + wm + 16 * i + cm + q, gn = n0 + wn + 16 * j + cn;
        if (gm < M && gn < N) {
          float v = acc[i][j][q];
          const int64_t at = (int64_t)gm * ldc + gn;
          if constexpr (END == End::plain) {
            if (bias) v += bias[gn];
            C[at] = beta != 0.f ? beta * C[at] + v : v;
          } else if constexpr (END == End::gelu) {
            if (bias) v += bias[gn];
            C[at] = v;
            Cbf[at] = f32_to_bf16(gelu(v));
          } else {
            v *= gelu_slope(Z[at]);
            C[at] = v;
            Cbf[at] = f32_to_bf16(v);
          }
        }
      }
}

template <int TN, int G, int KS, bool TA, bool TB, End END>
__global__ __launch_bounds__(256 * G) void gemm_bf16_kernel(GemmArgs a) {
  const unsigned tile = xcd_order(blockIdx.y * gridDim.x + blockIdx.x, gridDim.x * gridDim.y);
  gemm_tile<TN, G, KS, TA, TB, END>(a, tile / gridDim.x * TM, tile % gridDim.x * TN);
}

// Up to kMany products A^T B (weight gradients) in one launch: none of a network's
// fills the chip, together they do.  At batch 1024 three launches took 20 us,
// this 11.
constexpr int kMany = 8;
struct GemmSet {
  GemmArgs a[kMany];
  unsigned first[kMany], cols[kMany];   // a product's first tile, and its tiles per row
};
template <int G>
__global__ __launch_bounds__(256 * G) void gemm_many_kernel(GemmSet s, int n) {
  const unsigned tile = xcd_order(blockIdx.x, gridDim.x);
  int k = 0;
  for (int i = 1; i < n; ++i)
    if (tile >= s.first[i]) k = i;
  const unsigned t = tile - s.first[k], cols = s.cols[k];
  gemm_tile<64, G, 128, true, false, End::plain>(s.a[k], t / cols * TM, t % cols * 64);
}

template <int TN, int G, int KS, bool TA, bool TB, End END>
void launch_tiles(const GemmArgs &a) {
  const unsigned cols = (a.N + TN - 1) / TN, rows = (a.M + TM - 1) / TM;
  hipLaunchKernelGGL((gemm_bf16_kernel<TN, G, KS, TA, TB, END>), dim3(cols, rows), dim3(256 * G), 0, stream(), a);
}
template <bool TA, bool TB, End END = End::plain>
int launch_gemm(const GemmArgs &a) {
  const int64_t tiles = (((int64_t)a.M + TM - 1) / TM) * (((int64_t)a.N + 31) / 32);
  if (tiles <= device_cus())
    launch_tiles<32, 4, 128, TA, TB, END>(a);
  else if (a.K <= 32)
    launch_tiles<64, 1, 32, TA, TB, END>(a);
  else if (a.K <= 64)
    launch_tiles<64, 1, 64, TA, TB, END>(a);
  else
    launch_tiles<64, 1, 128, TA, TB, END>(a);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

__global__ void gelu_fwd_kernel(const float *__restrict__ Z, uint16_t *__restrict__ Gbf, float *__restrict__ Gf,
                                int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float g = gelu(Z[i]);
  if (Gbf) Gbf[i] = f32_to_bf16(g);
  if (Gf) Gf[i] = g;
}

// dZ = dG * gelu'(Z), written as bf16 (next GEMM operand) and fp32 (bias grad).
__global__ void gelu_bwd_kernel(const float *__restrict__ dG, const float *__restrict__ Z, uint16_t *__restrict__ dZbf,
                                float *__restrict__ dZf, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float d = dG[i] * gelu_slope(Z[i]);
  if (dZbf) dZbf[i] = f32_to_bf16(d);
  if (dZf) dZf[i] = d;
}

__global__ void to_bf16_kernel(const float *__restrict__ x, uint16_t *__restrict__ y, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = f32_to_bf16(x[i]);
}

// column sums of dZ [M x N] -> db [N] (bias gradients), up to kMany matrices of
// M rows in one launch.  Every sum adds its rows in order, one after another from
// 0: the gradients of a training step, and what Adam makes of them, are then the
// same whatever the launch looks like (a sum in another order moves the biases by
// a rounding, and some steps later activations by whole BF16 steps).
// A workgroup takes 16 columns.  Its 1024 threads load tiles of 512 rows into two
// LDS buffers in turn, the next tile's loads in flight meanwhile, and 16 lanes of
// its first wave add a tile's rows, 32 per trip with the next trip's LDS reads in
// flight, four rows to a read (a column's rows lie next to each other; 4 words of
// padding spread the columns over the banks).  Rows past the matrix are zeros: a
// sum that starts at 0 is never -0, so adding them changes nothing.
// Bound: the chain of one addition per row, about 11 cycles each.  M x (512, 512,
// 256) in one launch: M = 1024 7.4 us, 8192 39; one thread per column took 94 us for
// 1024 x 512 alone, or 21 with eight loads in flight.
constexpr int kSumCols = 16, kSumRows = 512, kSumThreads = 1024;
constexpr int kSumLoads = kSumCols * kSumRows / kSumThreads, kSumStride = kSumRows + 4;
struct ColSums {
  const float *dZ[kMany];
  float *db[kMany];
  int N[kMany], first[kMany];   // columns; first group of kSumCols
};
__global__ __launch_bounds__(kSumThreads) void colsum_kernel(ColSums a, int n, int M, int groups) {
  __shared__ __align__(16) float tile[2][kSumCols * kSumStride];
  const int c = threadIdx.x % kSumCols, r = threadIdx.x / kSumCols;
  constexpr int kStep = kSumThreads / kSumCols;   // rows between a thread's loads
  for (int g = blockIdx.x; g < groups; g += gridDim.x) {
    int k = 0;
    for (int i = 1; i < n; ++i)
      if (g >= a.first[i]) k = i;
    const float *__restrict__ dZ = a.dZ[k];
    const int N = a.N[k];
    const int64_t col = (int64_t)(g - a.first[k]) * kSumCols + c;
    const int64_t step = (int64_t)kStep * N;
    // of this thread's first row in the next tile; a column past the matrix reads
    // the group's first one and is not stored
    const float *at = dZ + (int64_t)r * N + (col < N ? col : col - c);
    float x[kSumLoads];
    auto load = [&](int64_t row0) {
      if (row0 + kSumRows <= M) {
#pragma unroll
        for (int i = 0; i < kSumLoads; ++i) x[i] = at[i * step];
      } else {
#pragma unroll
        for (int i = 0; i < kSumLoads; ++i) x[i] = row0 + r + i * kStep < M ? at[i * step] : 0.0f;
      }
      at += kSumLoads * step;
    };
    load(0);
    float s = 0.0f;
    int half = 0;
    for (int64_t row0 = 0; row0 < M; row0 += kSumRows, half ^= 1) {
      float *t = tile[half];
#pragma unroll
      for (int i = 0; i < kSumLoads; ++i) t[c * kSumStride + r + i * kStep] = x[i];
      // one barrier per tile: a buffer is written again only after the next
      // tile's barrier, which the adding wave reaches when it is done with it
      __syncthreads();
      load(row0 + kSumRows);
      if (threadIdx.x < kSumCols) {
        const float4 *q = reinterpret_cast<const float4 *>(t + c * kSumStride);
        const int64_t left = M - row0;
        const int trips = (int)((left < kSumRows ? left : kSumRows) + 31) / 32;
        float4 v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = q[i];
        for (int j = 1; j <= trips; ++j) {
          float4 u[8];
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            u[i] = v[i];
            v[i] = q[8 * (j < trips ? j : 0) + i];   // in flight during the additions
          }
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            s += u[i].x;
            s += u[i].y;
            s += u[i].z;
            s += u[i].w;
          }
        }
      }
    }
    if (threadIdx.x < kSumCols && col < N) a.db[k][col] = s;
    __syncthreads();   // the next group's first tile may take the buffer added last
  }
}

// The same sums by one thread per column, 256 columns to a workgroup (`first` counts
// these): for few rows or very many columns (cm_colsums has the line).  Bound: one
// thread's loads, eight in flight, or the memory (1e6 columns of 1024 rows 5.8 TB/s).
constexpr int kWideCols = 256;
__global__ __launch_bounds__(kWideCols) void colsum_wide_kernel(ColSums a, int n, int M, int groups) {
  for (int g = blockIdx.x; g < groups; g += gridDim.x) {
    int k = 0;
    for (int i = 1; i < n; ++i)
      if (g >= a.first[i]) k = i;
    const int64_t N = a.N[k], col = (int64_t)(g - a.first[k]) * kWideCols + threadIdx.x;
    if (col >= N) continue;
    const float *__restrict__ at = a.dZ[k] + col;
    float s = 0.0f;
#pragma unroll 8
    for (int m = 0; m < M; ++m, at += N) s += *at;
    a.db[k][col] = s;
  }
}

// MSE loss gradient: dY = (2/(M*N)) (Y - T), loss partials per row.
__global__ void mse_grad_kernel(const float *__restrict__ Y, const float *__restrict__ T, float *__restrict__ dY,
                                uint16_t *__restrict__ dYbf, float *__restrict__ row_loss, int M, int N) {
  const int m = blockIdx.x;
  float part = 0.f;
  for (int n = threadIdx.x; n < N; n += blockDim.x) {
    const int64_t i = (int64_t)m * N + n;
    const float e = Y[i] - T[i];
    const float g = 2.0f * e / ((float)M * (float)N);
    dY[i] = g;
    if (dYbf) dYbf[i] = f32_to_bf16(g);
    part += e * e;
  }
  __shared__ float sh[256];
  sh[threadIdx.x] = part;
  __syncthreads();
  for (int t = blockDim.x >> 1; t >= 1; t >>= 1) {
    if ((int)threadIdx.x < t) sh[threadIdx.x] += sh[threadIdx.x + t];
    __syncthreads();
  }
  if (threadIdx.x == 0) row_loss[m] = sh[0];
}

// Adam on FP32 master weights; refreshes the BF16 copy.  Up to kMany arrays in one
// launch, each from its own block on: memory bound, and six arrays of a network
// one after another ran into each launch's latency (16 -> 7.7 us).
struct AdamSet {
  float *w[kMany], *m1[kMany], *m2[kMany];
  uint16_t *wbf[kMany];
  const float *g[kMany];
  int64_t n[kMany];
  float wd[kMany];
  unsigned first[kMany];
};
__global__ __launch_bounds__(256) void adam_kernel(AdamSet a, int count, float lr, float b1, float b2, float eps,
                                                   float bc1, float bc2) {
  int k = 0;
  for (int i = 1; i < count; ++i)
    if (blockIdx.x >= a.first[i]) k = i;
  const int64_t i = (int64_t)(blockIdx.x - a.first[k]) * 256 + threadIdx.x;
  if (i >= a.n[k]) return;
  float *__restrict__ w = a.w[k], *__restrict__ m1 = a.m1[k], *__restrict__ m2 = a.m2[k];
  const float gi = a.g[k][i] + a.wd[k] * w[i];
  const float m = b1 * m1[i] + (1.f - b1) * gi;
  const float v = b2 * m2[i] + (1.f - b2) * gi * gi;
  m1[i] = m;
  m2[i] = v;
  const float upd = lr * (m / bc1) / (sqrtf(v / bc2) + eps);
  const float nw = w[i] - upd;
  w[i] = nw;
  if (a.wbf[k]) a.wbf[k][i] = f32_to_bf16(nw);
}

}  // namespace cm

using namespace cm;

extern "C" {

int cm_gemm_bf16(int transA, int transB, int M, int N, int K, const void *A, int lda, const void *B, int ldb,
                 float *C, int ldc, const float *bias, float beta) {
  if (M <= 0 || N <= 0 || K <= 0 || !A || !B || !C) {
    set_error("cm_gemm_bf16: bad arguments");
    return -3;
  }
  const GemmArgs a{(unsigned)M, (unsigned)N, (unsigned)K, (const uint16_t *)A, lda, (const uint16_t *)B, ldb,
                   C, ldc, bias, beta, nullptr, nullptr};
  if (transA) return transB ? launch_gemm<true, true>(a) : launch_gemm<true, false>(a);
  return transB ? launch_gemm<false, true>(a) : launch_gemm<false, false>(a);
}

int cm_gemm_bf16_gelu(int M, int N, int K, const void *A, int lda, const void *B, int ldb, const float *bias, float *Z,
                      void *G, int ld) {
  if (M <= 0 || N <= 0 || K <= 0 || !A || !B || !Z || !G) {
    set_error("cm_gemm_bf16_gelu: bad arguments");
    return -3;
  }
  return launch_gemm<false, false, End::gelu>(
      GemmArgs{(unsigned)M, (unsigned)N, (unsigned)K, (const uint16_t *)A, lda, (const uint16_t *)B, ldb, Z, ld, bias,
               0.f, nullptr, (uint16_t *)G});
}

int cm_gemm_bf16_gelu_back(int M, int N, int K, const void *A, int lda, const void *B, int ldb, const float *Z,
                           float *dZ, void *dZbf, int ld) {
  if (M <= 0 || N <= 0 || K <= 0 || !A || !B || !Z || !dZ || !dZbf) {
    set_error("cm_gemm_bf16_gelu_back: bad arguments");
    return -3;
  }
  return launch_gemm<false, true, End::gelu_back>(
      GemmArgs{(unsigned)M, (unsigned)N, (unsigned)K, (const uint16_t *)A, lda, (const uint16_t *)B, ldb, dZ, ld,
               nullptr, 0.f, Z, (uint16_t *)dZbf});
}

int cm_weight_grads(int n, int K, const int *M, const int *N, const void *const *A, const void *const *B,
                    float *const *C) {
  if (n < 1 || n > kMany || K <= 0 || !M || !N || !A || !B || !C) {
    set_error("cm_weight_grads: 1 to %d products", kMany);
    return -3;
  }
  GemmSet s{};
  int64_t tiles = 0;
  for (int i = 0; i < n; ++i) {
    if (M[i] <= 0 || N[i] <= 0 || !A[i] || !B[i] || !C[i]) {
      set_error("cm_weight_grads: bad product %d", i);
      return -3;
    }
    s.a[i] = GemmArgs{(unsigned)M[i], (unsigned)N[i], (unsigned)K, (const uint16_t *)A[i], M[i],
                      (const uint16_t *)B[i], N[i], C[i], N[i], nullptr, 0.f, nullptr, nullptr};
    s.first[i] = (unsigned)tiles;
    s.cols[i] = ((unsigned)N[i] + 63) / 64;
    tiles += (((int64_t)M[i] + TM - 1) / TM) * s.cols[i];
  }
  if (tiles > INT32_MAX) {
    set_error("cm_weight_grads: too many tiles");
    return -3;
  }
  // sixteen waves per tile while every tile has a CU of its own, as for one product:
  // 200 tiles of K = 1024 11.0 us (four waves 15.8), 296 tiles 18.7 (18.5), 384 16.3 (13.4)
  if (tiles <= device_cus())
    hipLaunchKernelGGL((gemm_many_kernel<4>), dim3((unsigned)tiles), dim3(1024), 0, stream(), s, n);
  else
    hipLaunchKernelGGL((gemm_many_kernel<1>), dim3((unsigned)tiles), dim3(256), 0, stream(), s, n);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int cm_gelu_fwd(const float *Z, void *Gbf, float *Gf, int64_t n) {
  if (n <= 0) return 0;
  hipLaunchKernelGGL(gelu_fwd_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream(), Z, (uint16_t *)Gbf,
                     Gf, n);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int cm_gelu_bwd(const float *dG, const float *Z, void *dZbf, float *dZf, int64_t n) {
  if (n <= 0) return 0;
  hipLaunchKernelGGL(gelu_bwd_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream(), dG, Z,
                     (uint16_t *)dZbf, dZf, n);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int cm_to_bf16(const float *x, void *y, int64_t n) {
  if (n <= 0) return 0;
  hipLaunchKernelGGL(to_bf16_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream(), x, (uint16_t *)y, n);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int cm_colsums(int n, const float *const *dZ, float *const *db, int M, const int *N) {
  if (n < 1 || n > kMany || !dZ || !db || !N) {
    set_error("cm_colsums: 1 to %d matrices", kMany);
    return -3;
  }
  ColSums a{};
  int64_t groups = 0;   // of kSumCols columns
  for (int i = 0; i < n; ++i) {
    if (N[i] < 0) {
      set_error("cm_colsums: %d columns", N[i]);
      return -3;
    }
    a.dZ[i] = dZ[i];
    a.db[i] = db[i];
    a.N[i] = N[i];
    groups += ((int64_t)N[i] + kSumCols - 1) / kSumCols;
  }
  if (groups > INT32_MAX) {
    set_error("cm_colsums: too many columns");
    return -3;
  }
  // One thread per column for few rows, and for more of them where the columns
  // fill the chip: a workgroup of the tiled form takes 6 us whatever it adds, and
  // two fit on a CU.  us for tiles and threads: 512 columns of 128 rows 6.1 and
  // 4.5, of 256 6.6 and 6.9, of 1024 7.6 and 21.5; 32768 (4 rounds of the chip) of
  // 512 25 and 24, of 1024 44 and 46, of 4096 172 and 275; 131072 (16) of 4096 707
  // and 367.
  const int64_t rounds = (groups + 2 * device_cus() - 1) / (2 * device_cus());
  const bool wide = M <= 240 * rounds || rounds > 8;
  const int cols = wide ? kWideCols : kSumCols;
  groups = 0;
  for (int i = 0; i < n; ++i) {
    a.first[i] = (int)groups;
    groups += ((int64_t)N[i] + cols - 1) / cols;
  }
  const dim3 grid((unsigned)(groups < 65536 ? groups : 65536));
  if (wide)
    hipLaunchKernelGGL(colsum_wide_kernel, grid, dim3(kWideCols), 0, stream(), a, n, M, (int)groups);
  else
    hipLaunchKernelGGL(colsum_kernel, grid, dim3(kSumThreads), 0, stream(), a, n, M, (int)groups);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int cm_colsum(const float *dZ, float *db, int M, int N) { return cm_colsums(1, &dZ, &db, M, &N); }

int cm_mse_grad(const float *Y, const float *T, float *dY, void *dYbf, float *row_loss, int M, int N) {
  hipLaunchKernelGGL(mse_grad_kernel, dim3(M), dim3(256), 0, stream(), Y, T, dY, (uint16_t *)dYbf, row_loss, M, N);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int cm_adams(int count, float *const *w, void *const *wbf, const float *const *g, float *const *m1, float *const *m2,
             const int64_t *n, const float *wd, float lr, float b1, float b2, float eps, int step) {
  if (count < 1 || count > kMany || !w || !wbf || !g || !m1 || !m2 || !n || !wd) {
    set_error("cm_adams: 1 to %d arrays", kMany);
    return -3;
  }
  AdamSet a{};
  int64_t blocks = 0;
  for (int k = 0; k < count; ++k) {
    if (n[k] < 0) {
      set_error("cm_adams: negative size");
      return -3;
    }
    a.w[k] = w[k];
    a.wbf[k] = (uint16_t *)wbf[k];
    a.g[k] = g[k];
    a.m1[k] = m1[k];
    a.m2[k] = m2[k];
    a.n[k] = n[k];
    a.wd[k] = wd[k];
    a.first[k] = (unsigned)blocks;
    blocks += (n[k] + 255) / 256;
  }
  if (blocks > UINT32_MAX) {
    set_error("cm_adams: too many values");
    return -3;
  }
  const float bc1 = 1.f - powf(b1, (float)step), bc2 = 1.f - powf(b2, (float)step);
  hipLaunchKernelGGL(adam_kernel, dim3((unsigned)blocks), dim3(256), 0, stream(), a, count, lr, b1, b2, eps, bc1, bc2);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int cm_adam(float *w, void *wbf, const float *g, float *m1, float *m2, int64_t n, float lr, float b1, float b2,
            float eps, int step, float wd) {
  return cm_adams(1, &w, &wbf, &g, &m1, &m2, &n, &wd, lr, b1, b2, eps, step);
}

}  // extern "C"
