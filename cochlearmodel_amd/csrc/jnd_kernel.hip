// JND reductions of CudaCalculateJND (src/cochlea.cu:3703-4065) in one
// kernel: per-interval mean rate (GlobalCalculateMeanRate :3741-3771) and the
// Fisher AI / rate terms reduced over the 256 sections (GlobalCalculateJND
// :3773-3944).  One workgroup = 256 sections of one (interval, fiber group).
// The section reduction keeps the reference's halving tree (stride 128, 64,
// ..., 1) so the CPU oracle agrees bit for bit.
#include <hip/hip_runtime.h>

#include "cm_internal.h"

namespace cm {



// v of the threads 0..255 summed; every thread of the workgroup calls it.
__device__ __forceinline__ float halving_tree(float *sh, float v, int t) {
  if (t < CM_SECTIONS) sh[t] = v;
  for (int k = CM_SECTIONS >> 1; k >= 1; k >>= 1) {
    __syncthreads();
    if (t < k) sh[t] = sh[t] + sh[t + k];
  }
  __syncthreads();
  const float r = sh[0];
  __syncthreads();
  return r;
}

// Rows of one section, [row, row + N) of a run of `rows` rows from `base`;
// rows past it read as 0.
template <int N>
__device__ __forceinline__ void load_rows(const float *base, int64_t row, int64_t rows, int s, float (&x)[N]) {
  const int64_t left = rows - row;
  const auto desc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(base) + row * CM_SECTIONS, 0,
                                                      (int)(left < N ? (left > 0 ? left : 0) : N) * (CM_SECTIONS * 4),
                                                      0x00027000);
#pragma unroll
  for (int m = 0; m < N; ++m)
    x[m] = __builtin_bit_cast(float,
                              __builtin_amdgcn_raw_buffer_load_b32(desc, 4 * s + m * (CM_SECTIONS * 4), 0, 0));
}

// N / D as the compiler's correctly rounded FP64 division computes it, without
// its range scaling: for D within 2^+-200 and N a finite float, where nothing
// over- or underflows.
__device__ __forceinline__ double div_in_range(double n, double d) {
  double r = __builtin_amdgcn_rcp(d);
  r = __builtin_fma(__builtin_fma(-d, r, 1.0), r, r);
  r = __builtin_fma(__builtin_fma(-d, r, 1.0), r, r);
  const double q = n * r;
  return __builtin_fma(__builtin_fma(-d, q, n), r, q);
}

// One pass over the interval body of (interval, fiber group) and of its
// reference: both mean rates (FP64 sums in time order, as
// GlobalCalculateMeanRate takes them) and the AI Fisher sum (float, in time
// order), then the rate term and the two section reductions.  The reference's
// mean rate is summed again by every interval that uses it, in the same order,
// so it is the value its own workgroup writes.
//
// The three sums must stay serial in time; the Fisher terms (two divisions
// each, most of the work) need not.  So each 64 sections have 4 waves: all of
// them form the terms of a 32-row tile and put them into LDS, while one adds up
// the tile before it and two add up the rates, with fewer rows for these three
// (rows_of) so that all four reach the barrier together.
// Bound: instruction issue of one workgroup per CU.  41 intervals of 12.5 k
// rows: one thread per section doing everything in turn 6.01 ms, this 1.04 ms.
constexpr int kTileRows = 32;
constexpr int kMostRows = 10;
struct JndWave {
  const JndArgs &a;
  const float *c, *r;      // interval body, reference body: first row
  float *node_stage;
  int L, s, lane, stage;
  float dA;
  double inv_dA;

  // Fisher terms of N rows from row0 of the bodies into pre (64 lanes per row)
  template <int N>
  __device__ __forceinline__ void terms(const float (&cal)[kMostRows], const float (&ref)[kMostRows], int64_t row0,
                                        float *pre) const {
    bool in_range = a.Fs > 0x1p-100 && a.Fs < 0x1p100;
    float dl[N], sq[N];
#pragma unroll
    for (int m = 0; m < N; ++m) {
      // (cal - ref) / dA: the FP64 product with the reciprocal rounds to the
      // same float (a quotient of floats is 2^-49 from any midpoint of two; below
      // the normal range too unless dA is an even integer, and a dl of that size
      // squares to 0)
      dl[m] = dA > 0 ? (float)((double)(cal[m] - ref[m]) * inv_dA) : 0.0f;
      sq[m] = dl[m] * dl[m];
      in_range = in_range && (ref[m] > 0x1p-100f && ref[m] < 0x1p100f && sq[m] < __builtin_inff());
    }
    const bool fast = __builtin_amdgcn_ballot_w64(!in_range) == 0;
#pragma unroll
    for (int m = 0; m < N; ++m) {
      const double n = (double)sq[m], d = a.Fs * (double)ref[m];
      const float p = (float)(fast ? div_in_range(n, d) : n / d);
      pre[m * 64 + lane] = p;
      if (node_stage && row0 + m < L) node_stage[(row0 + m) * CM_SECTIONS + s] = stage == 3 ? dl[m] : p;
    }
  }
};

// first row and number of rows of a tile that each of the 4 waves forms
template <int Q>
struct RowsOf;
template <> struct RowsOf<0> { static constexpr int first = 0, n = 8; };     // adds up the Fisher terms
template <> struct RowsOf<1> { static constexpr int first = 8, n = 7; };     // adds up the interval's rates
template <> struct RowsOf<2> { static constexpr int first = 15, n = 7; };    // adds up the reference's rates
template <> struct RowsOf<3> { static constexpr int first = 22, n = 10; };

// The time loop of wave Q of a section group; returns its sum (0: in accv).
template <int Q>
__device__ __forceinline__ double jnd_time(const JndWave &w, float *pre, bool ai, float &accv) {
  constexpr int first = RowsOf<Q>::first, n = RowsOf<Q>::n;
  const int tiles = (w.L + kTileRows - 1) / kTileRows;
  constexpr int kHalf = kTileRows / 2;
  float cal[n], ref[n], rate[2][kHalf];
  double acc = 0.0;
  accv = 0.0f;
  const float *mine = Q == 1 ? w.c : w.r;
  if (ai) {
    load_rows(w.c, first, w.L, w.s, cal);
    load_rows(w.r, first, w.L, w.s, ref);
  }
  if (Q == 1 || Q == 2) {
    load_rows(mine, 0, w.L, w.s, rate[0]);
    load_rows(mine, kHalf, w.L, w.s, rate[1]);
  }
  for (int j = 0; j <= tiles; ++j) {
    const int64_t row = (int64_t)j * kTileRows;
    float *buf = pre + (j & 1) * kTileRows * 64;
    if (j < tiles) {
      if (ai) {
        float c0[kMostRows], r0[kMostRows];
#pragma unroll
        for (int m = 0; m < n; ++m) { c0[m] = cal[m]; r0[m] = ref[m]; }
        load_rows(w.c, row + kTileRows + first, w.L, w.s, cal);   // the next tile's, in flight meanwhile
        load_rows(w.r, row + kTileRows + first, w.L, w.s, ref);
        w.terms<n>(c0, r0, row + first, buf + first * 64);
      }
      if (Q == 1 || Q == 2) {
        // rows past the body read as 0
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
          for (int m = 0; m < kHalf; ++m) acc = acc + (double)rate[h][m];
          load_rows(mine, row + kTileRows + h * kHalf, w.L, w.s, rate[h]);
        }
      }
    }
    if (Q == 0 && ai && j > 0) {
      const float *last = pre + ((j - 1) & 1) * kTileRows * 64 + w.lane;
      const int64_t left = w.L - (row - kTileRows);
      if (left >= kTileRows) {
        float p[kTileRows];
#pragma unroll
        for (int m = 0; m < kTileRows; ++m) p[m] = last[m * 64];
#pragma unroll
        for (int m = 0; m < kTileRows; ++m) accv += p[m];
      } else {
        for (int m = 0; m < left; ++m) accv += last[m * 64];
      }
    }
    if (ai) __syncthreads();
  }
  return acc;
}

// A short body's sums by the thread of their section, in the same order: no tiles
// to fill, and a quarter of the threads.  Returns the Fisher sum.
__device__ __forceinline__ float jnd_short(const JndWave &w, bool ai, double &acc_c, double &acc_r) {
  float accv = 0.0f;
  acc_c = acc_r = 0.0;
  const float *c = w.c + w.s, *r = w.r + w.s;
  if (!ai) {
#pragma unroll 8
    for (int k = 0; k < w.L; ++k) {
      acc_c = acc_c + (double)c[(int64_t)k * CM_SECTIONS];
      acc_r = acc_r + (double)r[(int64_t)k * CM_SECTIONS];
    }
    return accv;
  }
#pragma unroll 4
  for (int k = 0; k < w.L; ++k) {
    const int64_t at = (int64_t)k * CM_SECTIONS;
    const float cal = c[at], ref = r[at];
    acc_c = acc_c + (double)cal;
    acc_r = acc_r + (double)ref;
    const float dl = w.dA > 0 ? (float)((double)(cal - ref) * w.inv_dA) : 0.0f;
    const float p = (float)((double)(dl * dl) / (w.a.Fs * (double)ref));
    accv += p;
    if (w.node_stage) w.node_stage[at + w.s] = w.stage == 3 ? dl : p;
  }
  return accv;
}

template <bool SHORT>
__global__ __launch_bounds__(SHORT ? CM_SECTIONS : 1024) void jnd_kernel(JndArgs a) {
  __shared__ float pre_lds[SHORT ? 1 : 4][SHORT ? 1 : 2 * kTileRows * 64];
  __shared__ double mean_lds[2][SHORT ? 1 : CM_SECTIONS];
  __shared__ float fisher_lds[SHORT ? 1 : CM_SECTIONS];
  __shared__ float sh[CM_SECTIONS];
  const int iv = blockIdx.x, li = blockIdx.y, t = threadIdx.x;
  const int ref = a.ref_index[iv];
  const float dAv = a.dA[iv];
  const int64_t c = ((int64_t)li * a.rows + (int64_t)iv * a.interval_nodes + a.head_nodes) * CM_SECTIONS;
  const int64_t r = ((int64_t)li * a.rows + (int64_t)ref * a.interval_nodes + a.head_nodes) * CM_SECTIONS;
  const int L = a.length_nodes;
  const int stage = a.buffer ? a.backup_stage : 0;
  // per-node stages 3 (dLambda) and 4 (preFisherAI) at the body's own lambda nodes
  float *node_stage = (stage == 3 || stage == 4) ? a.buffer + c : nullptr;
  float ai = 0.f, rms = 0.f;
  if (a.calc_ai || a.calc_rms) {
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6), group = SHORT ? wave : wave >> 2, role = wave & 3;
    const int lane = t & 63, s = group * 64 + lane;
    const JndWave w{a, a.lambda + c, a.lambda + r, node_stage, L, s, lane, stage, dAv, a.calc_ai ? 1.0 / (double)dAv : 0.0};
    float accv = 0.0f;
    double acc_c = 0.0, acc_r = 0.0;   // sums of section t
    if constexpr (SHORT) {
      accv = jnd_short(w, a.calc_ai, acc_c, acc_r);
    } else {
      if (role == 0) {
        jnd_time<0>(w, pre_lds[group], a.calc_ai, accv);
        fisher_lds[s] = accv;
      } else if (role == 1) {
        mean_lds[0][s] = jnd_time<1>(w, pre_lds[group], a.calc_ai, accv);
      } else if (role == 2) {
        mean_lds[1][s] = jnd_time<2>(w, pre_lds[group], a.calc_ai, accv);
      } else {
        jnd_time<3>(w, pre_lds[group], a.calc_ai, accv);
      }
      __syncthreads();
      if (t < CM_SECTIONS) {
        accv = fisher_lds[t];
        acc_c = mean_lds[0][t];
        acc_r = mean_lds[1][t];
      }
    }
    const int64_t ms = ((int64_t)li * a.n_intervals + iv) * CM_SECTIONS + t;   // mean-rate layout
    float mr = 0.0f, dMR = 0.0f, mref = 0.0f;
    if (t < CM_SECTIONS) {
      mr = (float)acc_c / (float)L;
      mref = (float)acc_r / (float)L;
      a.mean_rate[ms] = mr;
      dMR = (mr - mref) / dAv;
      if (stage == 2) a.buffer[ms] = dMR;
    }
    if (stage == 1 && a.calc_rms) {   // mean over the sections of this interval's mean rate
      const float sum = halving_tree(sh, mr, t);
      if (t == 0) a.buffer[(int64_t)li * a.n_intervals + iv] = sum / (float)CM_SECTIONS;
    }
    if (t < CM_SECTIONS) {
      if (a.calc_ai) {
        const float rs = 1.0f / __builtin_sqrtf(accv);
        ai = (float)((double)(a.T / a.Tlength) * a.nIHC[t] / (double)(rs * rs));
        if (stage == 5) a.buffer[ms] = ai;
      }
      if (a.calc_rms) {
        const float crlb = 1.0f / __builtin_sqrtf(((a.T / mref) * dMR) * dMR);
        rms = (float)(a.nIHC[t] / (double)(crlb * crlb));
        if (stage == 6) a.buffer[ms] = crlb;
      }
    }
  }
  const int64_t fi = (int64_t)li * a.out_stride + a.out_index[iv];
  if (a.calc_ai) {
    const float sum = halving_tree(sh, ai, t);
    if (t == 0) a.FisherAISum[fi] = sum * a.W[li];
  }
  if (a.calc_rms) {
    const float sum = halving_tree(sh, rms, t);
    if (t == 0) a.F_RA[fi] = sum * a.W[li];
  }
}

// cudaCalculateDA (src/cochlea.cu:3726-3739): dA = sqrt(max x^2) over the
// interval body of a non-generated input.
__global__ void calc_dA_kernel(const float *input, float *dA, int n, int interval_nodes, int head_nodes,
                               int length_nodes, int offset_start) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  float acc = 0.0f;
  const int64_t start = (int64_t)offset_start + (int64_t)i * interval_nodes + head_nodes;
  for (int64_t k = start; k < start + length_nodes; ++k) {
    float c = input[k];
    c = c * c;
    if (acc < c) acc = c;
  }
  dA[i] = __builtin_sqrtf(acc);
}

}  // namespace cm

// Which bodies are short.  With w workgroups per CU, a tile's barriers are hidden
// by other workgroups the better the fewer threads each has, so the longest short
// body grows with w; and a CU holds one workgroup of tiles at a time, so that just
// above 3 per CU the fourth round costs tiles more.  us for tiles and for short,
// Fisher and rate terms, each interval with another reference: 2 intervals of 8 rows
// 7.8 and 5.9, of 32 rows 8.0 and 10.1; 90 (w = 1.05) of 32 14.8 and 10.9, of 80 25.5
// and 33.4; 200 (2.3) of 80 40 and 35, of 96 40 and 41; 300 (3.5) of 96 53 and 44, of
// 160 73 and 69, of 256 104 and 107; 500 (5.9) of 160 111 and 77, of 256 164 and 164;
// 805 (9.4) of 256 270 and 289; 2000 (23) of 512 1158 and 1012.
// Rates alone leave tiles two of four waves: 41 (0.5) of 8820 361 and 682; 100 (1.2) of
// 700 68 and 56, of 8820 920 and 806 (with one reference for all, which stays in the
// caches, 737 and 783); 200 of 8820 1587 and 1585 (1163 and 1133); 805 of 1500 1062
// and 1069.
static bool short_bodies(const cm::JndArgs &a) {
  const int64_t n = a.n_intervals, L = a.length_nodes, cus = cm::device_cus();
  if (!a.calc_ai) return 3 * n > cus;
  if (L <= 16) return true;
  const int64_t over = (L - 24) * cus;
  return 3 * n > cus && (over <= 25 * 3 * n || (n > cus && L <= 240 && over <= 36 * 3 * n));
}

extern "C" int cm_launch_jnd(const cm::JndArgs *a, hipStream_t stream) {
  using namespace cm;
  if (a->n_intervals <= 0) return 0;
  if (a->n_intervals > 0x7fffffff) return -3;
  if (short_bodies(*a))
    hipLaunchKernelGGL((jnd_kernel<true>), dim3(a->n_intervals, 3), dim3(CM_SECTIONS), 0, stream, *a);
  else
    hipLaunchKernelGGL((jnd_kernel<false>), dim3(a->n_intervals, 3), dim3(1024), 0, stream, *a);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

extern "C" int cm_launch_calc_dA(const float *input, float *dA, int n, int interval_nodes, int head_nodes,
                                 int length_nodes, int offset_start, hipStream_t stream) {
  if (n <= 0) return 0;
  hipLaunchKernelGGL(cm::calc_dA_kernel, dim3((n + 255) / 256), dim3(256), 0, stream, input, dA, n, interval_nodes,
                     head_nodes, length_nodes, offset_start);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}
