// IHC and auditory-nerve rates (lambda) of the reference's RunIHCKernel
// (src/cochlea.cu:3573-3644): AC filter of BM velocity (FIR in
// CudaUnifiedCalcIHC :3431-3506 or IIR in CudaIIRFilter[Decoupled]
// :2840-2908), dS = (BM - AC)^2, box-car DC FIR, PRE_IHC = eta_AC*AC +
// eta_DC*DC, IHC = log10(max(10^IHC_Vector * PRE_IHC, 0) + 1e-20) and
// lambda_k = min(SAT, max(A_k * IHC, spont_k)) with section 0 at spont
// (CudaCalcLambda :3365-3408).
//
// Data layout: rows x 256 sections, section fastest; a wave is 64 sections of
// a run of rows, so every load and store is a coalesced row segment.  Work is
// described by an interval table: each interval is a run of rows whose FIR
// window follows min((k+1) mod per, taps) with the reference's per = L before
// the final regular division and the analysed length after it
// (src/cochlea.cu:2719-2728).  FIR sums accumulate in FP64 in tap order, as
// the reference does, so the CPU oracle agrees bit for bit; where a shorter
// computation stands in for one of those sums or for log10, it carries its
// error bound and the long one decides when the bound leaves two floats open.
#include <hip/hip_runtime.h>

#include "cm_internal.h"

namespace cm {

__device__ __forceinline__ int fir_window(int64_t k, const cm_ihc_interval &iv, int taps) {
  const int64_t sg = iv.frdp > 1 ? k / (iv.frdp - 1) : 1;
  const int64_t per = sg * iv.tla + (1 - sg) * iv.L;
  if (per <= 0) return 0;
  const int64_t w = (k + 1) % per;
  return (int)(w < taps ? w : taps);
}

constexpr int kRows = 16;   // outputs per thread (register block) = taps per chunk

// Row loaders of the FIR helpers: the value of one section at a row.
struct GlobalRows {   // rows x 256 in global memory, section s
  const float *__restrict__ src;
  uint32_t s;
  __device__ __forceinline__ float operator()(int64_t row) const { return src[row * CM_SECTIONS + s]; }
};
// General register-blocked FIR over the n <= kRows rows row_first.. of one
// section: inputs stream from the newest output row down, so each output
// accumulates fma(b[0],x[k]), fma(b[1],x[k-1]), ... in tap order; a tap
// outside an output's window contributes an exact zero.  No row past the
// block or before row 0 is read.
template <class Rows>
__device__ __forceinline__ void fir_block_general(const Rows &src, int64_t row_first, int n,
                                                  const double *__restrict__ b, int taps, const int (&w)[kRows],
                                                  double (&acc)[kRows]) {
#pragma unroll
  for (int i = 0; i < kRows; ++i) acc[i] = 0.0;
  const int top = n - 1;
  const int span = n + taps - 1;
  for (int jj = 0; jj < span; ++jj) {
    const int64_t row = row_first + top - jj;
    if (row < 0) break;
    const double x = (double)src(row);
#pragma unroll
    for (int i = 0; i < kRows; ++i) {
      const int t = jj - top + i;
      const bool in = t >= 0 && t < w[i];
      const double c = in ? b[t] : 0.0;
      acc[i] = __builtin_fma(c, x, acc[i]);
    }
  }
}

// Steady-state FIR (every output uses all taps): taps in chunks of kRows with
// a 2*kRows-1 row register window; coefficients are uniform per tap and the
// tap array is zero-padded to a whole number of chunks.  Output i takes tap
// t from row row_first + i - t, accumulated in ascending t.  Loads are
// clamped to [0, row_first + n - 1]; clamped rows only meet zero taps or
// outputs past n.  (Requesting the next chunk's rows ahead of the FMAs costs
// the two-pass kernels a wave per SIMD of occupancy: 114 -> 132 VGPRs, 9.1 ->
// 19.2 ms on 2.26 M rows.)
template <class Rows>
__device__ __forceinline__ void fir_block_steady(const Rows &src, int64_t row_first, int n,
                                                 const double *__restrict__ bpad, int chunks, double (&acc)[kRows]) {
#pragma unroll
  for (int i = 0; i < kRows; ++i) acc[i] = 0.0;
  const int64_t hi = row_first + n - 1;
  double X[2 * kRows - 1];   // X[m] = row row_first - 16c - 15 + m
#pragma unroll
  for (int m = kRows - 1; m < 2 * kRows - 1; ++m) {
    int64_t r = row_first - (kRows - 1) + m;
    r = r > hi ? hi : r;
    X[m] = (double)src(r);
  }
  for (int c = 0; c < chunks; ++c) {
#pragma unroll
    for (int m = 0; m < kRows; ++m) {
      int64_t r = row_first - (int64_t)kRows * c - (kRows - 1) + m;
      r = r < 0 ? 0 : r;
      X[m] = (double)src(r);
    }
    const double *bc = bpad + kRows * c;
#pragma unroll
    for (int u = 0; u < kRows; ++u) {
      const double coef = bc[u];
#pragma unroll
      for (int i = 0; i < kRows; ++i) acc[i] = __builtin_fma(coef, X[i - u + kRows - 1], acc[i]);
    }
#pragma unroll
    for (int m = 2 * kRows - 2; m >= kRows; --m) X[m] = X[m - kRows];
  }
}

// XCD-aware tile order.  Workgroups are dealt round-robin to the 8 XCDs of
// the MI355X, each with its own L2; consecutive row tiles share the FIR's tap
// window, so the linear workgroup id is remapped for every XCD to walk one
// contiguous range of tiles and find the window rows in its own L2.  Returns
// (tile x, interval y); a bijection on [0, gx * gy).
__device__ __forceinline__ void xcd_tile(int &tx, int &ty) {
  constexpr unsigned kXcd = 8;
  const unsigned gx = gridDim.x, total = gx * gridDim.y;
  const unsigned lid = blockIdx.x + blockIdx.y * gx;
  const unsigned x = lid % kXcd, k = lid / kXcd, per = total / kXcd, rem = total % kXcd;
  const unsigned logical = x < rem ? x * (per + 1) + k : rem * (per + 1) + (x - rem) * per + k;
  tx = (int)(logical % gx);
  ty = (int)(logical / gx);
}

// Window of kRows outputs starting at interval row r0; returns 1 when every
// output of the block uses all taps.
__device__ __forceinline__ int block_windows(const cm_ihc_interval &iv, int64_t r0, int n, int taps, int (&w)[kRows]) {
  int steady = 1;
#pragma unroll
  for (int i = 0; i < kRows; ++i) {
    w[i] = i < n ? fir_window(iv.kbase + r0 + i, iv, taps) : 0;
    if (i < n && w[i] != taps) steady = 0;
  }
  return steady;
}

// Two passes through an AC/dS workspace, for tables whose intervals continue a
// window (kbase > 0) and DC filters of more than kHalo + 1 taps.
// AC (FIR, or read back when an IIR pass already wrote it) and dS.
__global__ __launch_bounds__(256) void ac_ds_kernel(const float *__restrict__ bm, const cm_ihc_interval *__restrict__ ivs,
                                                    const double *__restrict__ b, const double *__restrict__ bpad,
                                                    int nb, float coefA, int ac_ready, float *__restrict__ AC,
                                                    float *__restrict__ dS) {
  int tx, ty;
  xcd_tile(tx, ty);
  const cm_ihc_interval iv = ivs[ty];
  const uint32_t s = threadIdx.x;
  const int64_t r0 = (int64_t)tx * kRows;
  if (r0 >= iv.len) return;
  const int n = iv.len - r0 < kRows ? (int)(iv.len - r0) : kRows;
  float ac[kRows];
  if (ac_ready) {
#pragma unroll
    for (int i = 0; i < kRows; ++i) ac[i] = i < n ? AC[(iv.row0 + r0 + i) * CM_SECTIONS + s] : 0.0f;
  } else {
    int w[kRows];
    double acc[kRows];
    const GlobalRows rows{bm, s};
    if (block_windows(iv, r0, n, nb, w))
      fir_block_steady(rows, iv.row0 + r0, n, bpad, (nb + kRows - 1) / kRows, acc);
    else
      fir_block_general(rows, iv.row0 + r0, n, b, nb, w, acc);
#pragma unroll
    for (int i = 0; i < kRows; ++i) {
      ac[i] = (float)acc[i];
      if (i < n) AC[(iv.row0 + r0 + i) * CM_SECTIONS + s] = ac[i];
    }
  }
#pragma unroll
  for (int i = 0; i < kRows; ++i) {
    if (i < n) {
      const int64_t o = (iv.row0 + r0 + i) * CM_SECTIONS + s;
      const float mid = __builtin_fmaf(bm[o], coefA, -ac[i]);
      dS[o] = mid * mid;
    }
  }
}

struct LambdaArgs {
  float *AC;
  const float *dS;
  const cm_ihc_interval *ivs;
  const double *dc;
  const double *dcpad;    // dc zero-padded to a multiple of kRows taps (two-pass path)
  int ndc;
  float etaAC;
  float etaDC;
  const double *damage;   // sets x 256
  const float *A;         // 3 x 256
  float spont[3];
  float sat;
  int64_t rows;           // lambda plane stride in rows
  float *lambda;          // 3 x rows x 256
  float *stages;          // optional 5 x rows x 256 (AC, dS, DC, PRE_IHC, IHC)
};

// Interval rows [lo, hi] of one section for a FIR block; other rows read as 0.
// In global memory through a buffer descriptor of just these rows, in scalar
// registers: a lane needs one offset register for 4 rows (64-bit addresses took
// two for each), and rows on either side are out of its range (below lo the
// unsigned offset is above it).
struct GlobalWindow {
  __amdgpu_buffer_rsrc_t desc;
  uint32_t at;   // byte offset of this lane's section in a row
  int lo;
  __device__ __forceinline__ GlobalWindow(float *rows, uint32_t s, int first, int last)
      : desc(__builtin_amdgcn_make_buffer_rsrc(rows + (int64_t)first * CM_SECTIONS, 0,
                                               (last - first + 1) * (CM_SECTIONS * 4), 0x00027000)),
        at(4 * s), lo(first) {}
  template <int N>
  __device__ __forceinline__ void load(int row, float (&x)[N]) const {
    if (row >= lo) {
      const uint32_t o = at + (uint32_t)(row - lo) * (CM_SECTIONS * 4);
#pragma unroll
      for (int m = 0; m < N; ++m) x[m] = get(o + m * (CM_SECTIONS * 4));
    } else {
#pragma unroll
      for (int m = 0; m < N; ++m) {
        uint32_t o = at + (uint32_t)(row + m - lo) * (CM_SECTIONS * 4);
        asm("" : "+v"(o));   // a whole offset per row: with a constant part split off, one below lo could wrap
        x[m] = get(o);
      }
    }
  }
  __device__ __forceinline__ float get(uint32_t o) const {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(desc, (int)o, 0, 0));
  }
  __device__ __forceinline__ void put(uint32_t o, float v) const {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), desc, (int)o, 0, 2);   // streaming
  }
};

// log10 of a double in (0, inf) to 1.5e-13.  v = m 2^e with m in [0.5, 1);
// c = 1/m to 7 fraction bits picks -log10(c) from a table of 129, and
// r = m c - 1 (|r| < 2^-8) leaves a cubic; the dropped r^5/5 log10(e) is at
// most 8e-14.  Where y -+ 1.5e-13 round to different floats, once in a million
// values, the caller takes the full log10, so the float is always the one that
// the full log10 rounds to.
constexpr int kLogCells = 129;
// The full log10 (a call: inlined, its constants would stay in registers).
__device__ __attribute__((noinline)) double log10_full(double v) { return log10(v); }
__device__ __forceinline__ void fill_log_table(double *tab, int tid, int n) {
  for (int i = tid; i < kLogCells; i += n) tab[i] = -log10_full(1.0 + (double)i * 0x1p-7);
}
__device__ __forceinline__ double log10_near(double v, const double *tab) {
  const double m = __builtin_amdgcn_frexp_mant(v);
  const int e = __builtin_amdgcn_frexp_exp(v);
  const uint32_t cb = (__float_as_uint(__builtin_amdgcn_rcpf((float)m)) + 0x8000u) & 0xffff0000u;
  const uint32_t cell = (cb - 0x3f800000u) >> 16;   // beyond the table only for an infinite v: y is NaN then
  const double r = __builtin_fma(m, (double)__uint_as_float(cb), -1.0);
  double q = __builtin_fma(r, -1.08573620475812959e-01, 1.44764827301083943e-01);
  q = __builtin_fma(r, q, -2.17147240951625914e-01);
  q = __builtin_fma(r, q, 4.34294481903251828e-01);
  const double base = __builtin_fma((double)e, 3.01029995663981195e-01, tab[cell < kLogCells ? cell : 0]);
  return __builtin_fma(r, q, base);
}

// PRE_IHC, IHC and the three lambdas of one node (CudaCalcIHCComposite /
// CudaCalcLambda).  The products of two floats that the reference takes in
// FP64 and rounds to float are one FP32 multiplication here (the same single
// rounding), and the clamps, which are floats, commute with that rounding.
struct LambdaNode {
  double dmg;
  float A3[3];
  int quiet;   // an IHC of at most 0 leaves every rate at its spontaneous value
  __device__ __forceinline__ void init(const LambdaArgs &a, int set, int s) {
    dmg = a.damage[(int64_t)set * CM_SECTIONS + s];
    bool q = !a.stages;
    for (int j = 0; j < 3; ++j) {
      A3[j] = a.A[j * CM_SECTIONS + s];
      q = q && A3[j] >= 0.0f && A3[j] <= 3.0e38f && a.spont[j] >= 0.0f;
    }
    quiet = __builtin_amdgcn_ballot_w64(!q) == 0;
  }
  __device__ __forceinline__ double drive(float pre) const { return fmax(dmg * (double)pre, 0.0) + 1e-20; }
  // section s of the n rows from `row`
  __device__ __forceinline__ void store(const LambdaArgs &a, const double *log_tab, int64_t row, uint32_t s, int n,
                                        const float (&ac)[kRows], const float (&ds)[kRows],
                                        const float (&dc)[kRows]) const {
    const int64_t plane = a.rows * CM_SECTIONS;
    const GlobalWindow lam0(a.lambda + row * CM_SECTIONS, s, 0, n - 1),
        lam1(a.lambda + plane + row * CM_SECTIONS, s, 0, n - 1),
        lam2(a.lambda + 2 * plane + row * CM_SECTIONS, s, 0, n - 1);
    // rows past n are outside the descriptors: their stores are dropped
    auto rates = [&](uint32_t o, float ihc) {
      auto rate = [&](int j) {
        return fminf(s != 0 ? a.sat : a.spont[j], fmaxf(A3[j] * ihc, a.spont[j]));   // section 0 stays at spont
      };
      lam0.put(o, rate(0));
      lam1.put(o, rate(1));
      lam2.put(o, rate(2));
    };
    float pre[kRows];
#pragma unroll
    for (int i = 0; i < kRows; ++i) pre[i] = __builtin_fmaf(ac[i], a.etaAC, dc[i] * a.etaDC);
    if (a.stages) {
#pragma unroll
      for (int i = 0; i < kRows; ++i) {
        if (i >= n) continue;
        float *st = a.stages + (row + i) * CM_SECTIONS;
        st[s] = ac[i];
        (st + plane)[s] = ds[i];
        (st + 2 * plane)[s] = dc[i];
        (st + 3 * plane)[s] = pre[i];
      }
    }
    uint32_t open = 0;   // rows whose float log10 is not settled in some lane
#pragma unroll
    for (int i = 0; i < kRows; ++i) {
      const double v = drive(pre[i]);
      float ihc = 0.0f;
      if (!quiet || __builtin_amdgcn_ballot_w64(v > 1.0) != 0) {
        const double y = log10_near(v, log_tab);
        ihc = (float)(y - 1.5e-13);
        if (__builtin_amdgcn_ballot_w64(ihc != (float)(y + 1.5e-13)) != 0) open |= 1u << i;
      }
      rates(lam0.at + i * (CM_SECTIONS * 4), ihc);
    }
    if (a.stages) open = 0xffffu;   // the stage dump takes every row's IHC from the loop below
    while (open) {
      const int k = __builtin_ctz(open);
      open &= open - 1;
      float p = pre[0];
#pragma unroll
      for (int i = 1; i < kRows; ++i) p = i == k ? pre[i] : p;
      const float ihc = (float)log10_full(drive(p));
      rates(lam0.at + k * (CM_SECTIONS * 4), ihc);
      if (a.stages && k < n) (a.stages + 4 * plane + (row + k) * CM_SECTIONS)[s] = ihc;
    }
  }
};

// IIR AC filter (DeviceCudaIIRFilter<float,float>, src/cochlea.cu:2742-2772):
// per row the feed-forward terms, then the feedback terms, each rounded to
// float; every interval starts from rest, and its last row's window is empty.
// General form, any order: one thread per section, serial over the interval.
__global__ __launch_bounds__(256) void ac_iir_kernel(const float *__restrict__ bm, const cm_ihc_interval *__restrict__ ivs,
                                                     const double *__restrict__ b, const double *__restrict__ a,
                                                     int taps, float *__restrict__ AC) {
  const cm_ihc_interval iv = ivs[blockIdx.x];
  const int s = threadIdx.x;
  const int64_t per = iv.len;
  for (int64_t k = 0; k < iv.len; ++k) {
    const int64_t row = iv.row0 + k;
    const int ob = per > 0 ? (int)(((k + 1) % per) < taps ? ((k + 1) % per) : taps) : 0;
    float y = 0.0f;
    for (int i = 0; i < ob; ++i) y = (float)((double)y + b[i] * (double)bm[(row - i) * CM_SECTIONS + s]);
    for (int i = 0; i < ob - 1; ++i) y = (float)((double)y - a[i + 1] * (double)AC[(row - i - 1) * CM_SECTIONS + s]);
    AC[row * CM_SECTIONS + s] = y;
  }
}

// Filters of up to kIirTaps taps in two kernels, because only the feedback is
// serial: the feed-forward sums run over all rows at once, then one wave per
// interval and 64 sections adds the feedback down the rows, its history in
// registers and the next rows' sums requested 16 rows ahead.
// Bound: the second kernel's serial chain, 4 FP64-rate instructions per tap and
// row for one wave per SIMD.  24 intervals of 4 to 9 k rows, 5 taps: 8.84 ms
// (history re-read from memory) -> 0.46 + 0.06 ms.
constexpr int kIirTaps = 9;

template <int N>
__global__ __launch_bounds__(256) void iir_feed_kernel(const float *__restrict__ bm,
                                                       const cm_ihc_interval *__restrict__ ivs,
                                                       const double *__restrict__ b, float *__restrict__ AC) {
  const cm_ihc_interval iv = ivs[blockIdx.y];
  const int k0 = blockIdx.x * kRows;
  if (k0 >= iv.len) return;
  const int n = iv.len - k0 < kRows ? iv.len - k0 : kRows;
  float x[kRows + N - 1];
  GlobalWindow(const_cast<float *>(bm) + iv.row0 * CM_SECTIONS, threadIdx.x, k0 > N - 1 ? k0 - (N - 1) : 0, k0 + n - 1)
      .load(k0 - (N - 1), x);
  const GlobalWindow out(AC + iv.row0 * CM_SECTIONS, threadIdx.x, k0, k0 + n - 1);
#pragma unroll
  for (int r = 0; r < kRows; ++r) {
    // rows before the interval are zeros here: adding a zero product changes nothing
    float y = 0.0f;
#pragma unroll
    for (int i = 0; i < N; ++i) y = (float)((double)y + b[i] * (double)x[r + N - 1 - i]);
    out.put(out.at + r * (CM_SECTIONS * 4), k0 + r + 1 < iv.len ? y : 0.0f);
  }
}

template <int N>
__global__ __launch_bounds__(64) void iir_feedback_kernel(const cm_ihc_interval *__restrict__ ivs,
                                                          const double *__restrict__ a, float *__restrict__ AC) {
  const cm_ihc_interval iv = ivs[blockIdx.x >> 2];
  if (iv.len <= 0) return;
  const uint32_t s = (blockIdx.x & 3) * 64 + threadIdx.x;
  float *rows = AC + iv.row0 * CM_SECTIONS;
  double c[N], h[N];   // h[i] = row k - 1 - i
#pragma unroll
  for (int i = 0; i < N - 1; ++i) {
    c[i] = a[i + 1];
    h[i] = 0.0;
  }
  float x[kRows];
  auto window = [&](int k) { return GlobalWindow(rows, s, k, k + kRows < iv.len ? k + kRows - 1 : iv.len - 1); };
  window(0).load(0, x);
  for (int k = 0; k < iv.len; k += kRows) {
    const GlobalWindow out = window(k);
    float y[kRows];
#pragma unroll
    for (int r = 0; r < kRows; ++r) y[r] = x[r];
    if (k + kRows < iv.len) window(k + kRows).load(k + kRows, x);
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
#pragma unroll
      for (int i = 0; i < N - 1; ++i) y[r] = (float)((double)y[r] - c[i] * h[i]);
#pragma unroll
      for (int i = N - 2; i > 0; --i) h[i] = h[i - 1];
      h[0] = (double)y[r];
      out.put(out.at + r * (CM_SECTIONS * 4), k + r + 1 < iv.len ? y[r] : 0.0f);
    }
  }
}

template <int N = 2>
int launch_iir(const float *bm, const cm_ihc_interval *d_ivs, int n_ivs, int max_len, const double *b, const double *a,
               int taps, float *AC, hipStream_t stream) {
  if constexpr (N <= kIirTaps) {
    if (taps != N || n_ivs > 65535) return launch_iir<N + 1>(bm, d_ivs, n_ivs, max_len, b, a, taps, AC, stream);
    if (max_len > 0) {
      hipLaunchKernelGGL((iir_feed_kernel<N>), dim3((max_len + kRows - 1) / kRows, n_ivs), dim3(256), 0, stream, bm,
                         d_ivs, b, AC);
      hipLaunchKernelGGL((iir_feedback_kernel<N>), dim3(4 * n_ivs), dim3(64), 0, stream, d_ivs, a, AC);
    }
  } else {
    hipLaunchKernelGGL(ac_iir_kernel, dim3(n_ivs), dim3(256), 0, stream, bm, d_ivs, b, a, taps, AC);
  }
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

// DC FIR, PRE_IHC, IHC and the three lambdas.
__global__ __launch_bounds__(256) void dc_lambda_kernel(LambdaArgs a) {
  __shared__ double log_tab[kLogCells];
  int tx, ty;
  xcd_tile(tx, ty);
  const cm_ihc_interval iv = a.ivs[ty];
  const uint32_t s = threadIdx.x;
  const int64_t r0 = (int64_t)tx * kRows;
  if (r0 >= iv.len) return;
  const int n = iv.len - r0 < kRows ? (int)(iv.len - r0) : kRows;
  fill_log_table(log_tab, s, CM_SECTIONS);
  LambdaNode node;
  node.init(a, iv.set, s);
  int w[kRows];
  double acc[kRows];
  const GlobalRows rows{a.dS, s};
  if (block_windows(iv, r0, n, a.ndc, w))
    fir_block_steady(rows, iv.row0 + r0, n, a.dcpad, (a.ndc + kRows - 1) / kRows, acc);
  else
    fir_block_general(rows, iv.row0 + r0, n, a.dc, a.ndc, w, acc);
  __syncthreads();
  float ac[kRows], ds[kRows], dc[kRows];
#pragma unroll
  for (int i = 0; i < kRows; ++i) {
    ac[i] = i < n ? (a.AC + (iv.row0 + r0 + i) * CM_SECTIONS)[s] : 0.0f;
    ds[i] = i < n ? (a.dS + (iv.row0 + r0 + i) * CM_SECTIONS)[s] : 0.0f;
    dc[i] = (float)acc[i];
  }
  node.store(a, log_tab, iv.row0 + r0, s, n, ac, ds, dc);
}

// ------------------------------------------------------ one pass --------
// The whole chain in one pass: BM -> AC FIR -> dS -> DC FIR -> PRE_IHC -> IHC
// -> 3 lambdas, with no AC / dS round trip through HBM.  A workgroup of 4 waves
// takes 64 sections of a tile of rows and walks down it 64 rows at a time,
// 16 to a wave: each wave filters its rows' AC, puts their dS and its sum into
// LDS rings, and after a barrier forms the DC of its rows from the rings, which
// hold the last 160 rows for all four waves.  The DC window reaches up to kHalo
// rows back, so a tile first runs AC and dS over the kHalo rows before it.
//
// Bound: instruction issue, FP64 first (4.2 to 4.8 cycles a wave instruction;
// the 76 AC taps are half of the time).  The default DC filter is a box car;
// its window sum is then not 88 multiply-adds per row but the sum of its whole
// 16-row blocks, two partial blocks and a running prefix and suffix, about 4
// additions per row (dc_boxcar).  A trip's first rows are requested before the
// second half of the trip before it.  Two workgroups per CU: 229 registers, so
// that nothing is spilled, whose reloads would wait behind the lambda stores.
// 847 k rows, 76 + 88 taps: 1.52 ms, 2.3 TB/s of the 16 B per node that the
// stage must move (HBM counters: 1.06 GB read, 2.54 GB written).
constexpr int kHalo = 96;                  // dS rows before a tile (DC taps <= 97)
constexpr int kStep = 4 * kRows;           // rows per trip of a workgroup
constexpr int kRingBlocks = 10;            // 16-row blocks of the rings: a trip's 4 and the 6 before it
constexpr int kInlineIvs = 4;

// An interval table of up to 4 entries travels in the kernel's arguments.
struct InlineIvs {
  cm_ihc_interval v[kInlineIvs];
};

// The period of a row: FIR windows of the rows k with lo <= k + 1 < lo + per
// (and before the row where the division into intervals changes) reach back to
// row lo, the row k = lo - 1 having none.  [from, next) are the rows of the
// period found last, so that a wave divides only where it leaves one.
struct Period {
  int lo = 0, from = 0, next = 0;
  __device__ __forceinline__ void find(const cm_ihc_interval &iv, int k) {
    if (k >= from && k < next) return;
    const int d = iv.frdp - 1;
    const int64_t sg = d > 0 ? (int64_t)((uint32_t)k / (uint32_t)d) : 1;
    const int64_t sg_end = d > 0 ? (sg + 1) * d : INT32_MAX;
    const int64_t per = sg * iv.tla + (1 - sg) * (int64_t)iv.L;
    from = k;
    int64_t end = sg_end;
    lo = INT32_MAX;                      // per <= 0: no window at all
    if (per > 0) {
      lo = per <= INT32_MAX ? (int)((uint32_t)(k + 1) / (uint32_t)per * (uint32_t)per) : 0;
      end = lo + per - 1 < sg_end ? lo + per - 1 : sg_end;
    }
    next = end < INT32_MAX ? (int)end : INT32_MAX;
  }
};

// The LDS ring of a workgroup's last 160 dS rows, one column per lane, in blocks
// of 16.  The last block is kept a second time before the first, so that the
// rows of two neighbouring blocks are always in ascending order; a row of
// zeros follows.
constexpr int kRingRows = kRingBlocks * kRows;
constexpr int kRingZero = kRingRows + kRows;
struct Ring {
  float *col;   // this lane's column
  __device__ __forceinline__ void put(int slot, int i, float v) const {
    col[((slot + 1) * kRows + i) * 64] = v;
    if (slot == kRingBlocks - 1) col[i * 64] = v;
  }
};
struct RingWindow {
  const float *col;
  int start, lo, hi;   // interval row of the ring's first block; rows in the window
  template <int N>
  __device__ __forceinline__ void load(int row, float (&x)[N]) const {
    asm("" : "+v"(row));   // in a vector register: N rows' selections would not fit the scalar ones
#pragma unroll
    for (int m = 0; m < N; ++m) {
      const int r = row + m;
      const int k = r >= lo && r <= hi ? kRows + (int)((uint32_t)(r - start) % kRingRows) : kRingZero;
      x[m] = col[k * 64];
    }
  }
};

// R outputs of a FIR at interval rows r0 .. r0 + R - 1, each in tap order from
// the newest row down.  A chunk of R taps needs 2 R - 1 rows, R - 1 of them the
// previous chunk's; the next chunk's R are requested before a chunk's products.
// The last chunk stops at a multiple of 4 taps.  x and up come in as rows
// r0 - R + 1 .. r0 and r0 + 1 .. r0 + R - 1.
template <int R, class Window>
__device__ __forceinline__ void fir_block(const Window &src, int r0, const double *__restrict__ b, int taps,
                                          float (&x)[R], const float (&up)[R - 1], double (&acc)[R]) {
  double X[2 * R - 1];   // X[m] = row r0 - t0 - (R - 1) + m
#pragma unroll
  for (int m = 0; m < R - 1; ++m) X[R + m] = (double)up[m];
#pragma unroll
  for (int i = 0; i < R; ++i) acc[i] = 0.0;
  int t0 = 0;
  for (; t0 + R <= taps; t0 += R) {
#pragma unroll
    for (int m = 0; m < R; ++m) X[m] = (double)x[m];
    if (t0 + R < taps) src.load(r0 - t0 - (2 * R - 1), x);
#pragma unroll
    for (int u = 0; u < R; ++u) {
      const double c = b[t0 + u];
#pragma unroll
      for (int i = 0; i < R; ++i) acc[i] = __builtin_fma(c, X[R - 1 + i - u], acc[i]);
    }
#pragma unroll
    for (int m = 2 * R - 2; m >= R; --m) X[m] = X[m - R];
  }
  const int left = taps - t0;
  if (left <= 0) return;
#pragma unroll
  for (int m = 0; m < R; ++m) X[m] = (double)x[m];
#pragma unroll
  for (int u0 = 0; u0 < R - 1; u0 += 4) {
    if (u0 >= left) break;
#pragma unroll
    for (int u = u0; u < u0 + 4; ++u) {
      const double c = u < left ? b[t0 + u] : 0.0;
#pragma unroll
      for (int i = 0; i < R; ++i) acc[i] = __builtin_fma(c, X[R - 1 + i - u], acc[i]);
    }
  }
}

// FIR outputs of rows r0 .. r0 + n - 1 (0 past them), each over its own period's
// window.  Nearly every block lies in one period; one that does not runs once
// for each.  window(lo) gives the rows from lo on; x and up hold the first
// period's rows already when `loaded`.
template <int R, class MakeWindow>
__device__ __forceinline__ void fir_rows(const MakeWindow &window, const cm_ihc_interval &iv, Period period, int r0,
                                         int n, const double *__restrict__ b, int taps, bool loaded, float (&x)[R],
                                         float (&up)[R - 1], float *out) {
#pragma unroll
  for (int i = 0; i < R; ++i) out[i] = 0.0f;
  for (int i0 = 0; i0 < n;) {
    period.find(iv, r0 + i0);
    const int i1 = period.next - r0 < n ? period.next - r0 : n;
    if (period.lo < r0 + i1) {
      const int low = r0 - (taps - 1), lo = period.lo > low ? period.lo : low;   // no window reaches below
      const auto win = window(lo);
      if (!loaded) {
        win.load(r0 - (R - 1), x);
        win.load(r0 + 1, up);
      }
      double acc[R];
      // Taps that reach below lo from every output would only add zeros, and short
      // intervals have few others: 30000 intervals of 16 rows took 5.92 ms with them
      // and take 2.65 (two passes 5.76), with an IIR filter 5.20 and 2.61 (4.51).
      fir_block<R>(win, r0, b, r0 + R - lo < taps ? r0 + R - lo : taps, x, up, acc);
#pragma unroll
      for (int i = 0; i < R; ++i) out[i] = i >= i0 && i < i1 ? (float)acc[i] : out[i];
    }
    loaded = false;
    i0 = i1;
  }
}

// Window sums of the 16 rows of ring block blk over the last `taps` dS rows
// each, 16 <= taps <= kHalo + 1, every window complete.  Common to all 16: the
// first row and the taps - 16 rows before it, which are whole blocks and the
// end (`part` rows) of one more.  Output i adds rows 1 .. i of the block and
// the 15 - i rows just before the common ones.  All LDS reads are requested
// together; the rows before the whole blocks ascend in the ring.  All terms are
// squares, so a sum's relative error is at most one unit of 2^-53 for each
// addition that a term goes through: 15 in its block's sum, one for each whole
// block and end row of the common ones (4 + 15 at 95 taps), 15 of the rows before
// for output 0, 49 in all.  The tap-order sum has one per tap.
constexpr int kWhole = (kHalo + 1 - kRows) / kRows;
constexpr int kBoxcarRoundings = (kRows - 1) + (kWhole + kRows - 1) + (kRows - 1);
// relative distance of the two sums, scaled by the tap: theirs and 3 for the
// product and the two ends of its range
constexpr double kBoxcarBound = 0x1p-45;
static_assert(kBoxcarRoundings + (kHalo + 1) + 3 <= 256, "the bound holds 256 units of 2^-53");
__device__ __forceinline__ void dc_boxcar(const float *col, const double *sums, int blk, int taps,
                                          const float (&ds)[kRows], double (&acc)[kRows]) {
  const int whole = (taps - kRows) / kRows, part = (taps - kRows) % kRows;
  double w[kWhole];
#pragma unroll
  for (int k = 0; k < kWhole; ++k) {
    const int slot = (int)((uint32_t)(blk - 1 - k + kRingBlocks) % kRingBlocks);
    w[k] = sums[(k < whole ? slot : kRingBlocks) * 64];
  }
  // rows just below the whole blocks, newest first: e[0 .. part) end the
  // common ones, the 15 below them are before[0 .. 14]
  const int top = ((int)((uint32_t)(blk - 1 - whole + kRingBlocks) % kRingBlocks) + 1) * kRows + kRows - 1;
  float e[kRows - 1], before[kRows - 1];
#pragma unroll
  for (int k = 0; k < kRows - 1; ++k) e[k] = col[(k < part ? top - k : kRingZero) * 64];
  const float *b = col + (top - part - (kRows - 2)) * 64;
#pragma unroll
  for (int k = 0; k < kRows - 1; ++k) before[k] = b[(kRows - 2 - k) * 64];
  double core = (double)ds[0];
#pragma unroll
  for (int k = 0; k < kWhole; ++k) core += w[k];
#pragma unroll
  for (int k = 0; k < kRows - 1; ++k) core += (double)e[k];
  acc[kRows - 1] = core;
#pragma unroll
  for (int i = kRows - 2; i >= 0; --i) acc[i] = acc[i + 1] + (double)before[kRows - 2 - i];
  double pre = 0.0;
#pragma unroll
  for (int i = 1; i < kRows; ++i) {
    pre += (double)ds[i];
    acc[i] += pre;
  }
}

// One pass for intervals of kbase 0 and DC filters of up to kHalo + 1 taps.
// FIR: the AC filter is run here; otherwise AC is read (an IIR pass wrote it).
template <bool FIR>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void ihc_lambda_kernel(
    float *__restrict__ bm, const double *__restrict__ b, int nb, float coefA, LambdaArgs a, int trips,
    InlineIvs inl) {
  __shared__ float ring_lds[(kRingZero + 1) * 64];
  __shared__ double sums_lds[(kRingBlocks + 1) * 64];   // of each block; the last is 0
  __shared__ double log_tab[kLogCells];
  int tx, ty;
  xcd_tile(tx, ty);
  cm_ihc_interval iv = inl.v[0];
  if (a.ivs) {
    iv = a.ivs[ty];
  } else {
#pragma unroll
    for (int k = 1; k < kInlineIvs; ++k)
      if (ty == k) iv = inl.v[k];
  }
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t s = (tx & 3) * 64 + lane;
  // interval rows are 32-bit: an interval holds fewer than 2^31 rows of
  // addressable memory
  const int tile = kStep * trips - kHalo;
  const int r_begin = (tx >> 2) * tile;
  if (r_begin >= iv.len) return;
  const int r_end = r_begin + tile < iv.len ? r_begin + tile : iv.len;
  const int start = r_begin > kHalo ? r_begin - kHalo : 0;
  fill_log_table(log_tab, threadIdx.x, 256);
  const Ring ring{ring_lds + lane};
  double *sums = sums_lds + lane;
  if (wave == 0) {
    ring.col[kRingZero * 64] = 0.0f;
    sums[kRingBlocks * 64] = 0.0;
  }
  // a box-car DC filter: every tap is the first one
  bool same = true;
  const double dc0 = a.ndc > 0 ? a.dc[0] : 0.0;
  for (int t = lane; t < a.ndc; t += 64) same = same && a.dc[t] == dc0;
  const bool boxcar = a.ndc >= kRows && __builtin_amdgcn_ballot_w64(!same) == 0;
  LambdaNode node;
  node.init(a, iv.set, s);
  float *rows = bm + iv.row0 * CM_SECTIONS;
  Period period;
  float x[kRows], up[kRows - 1];
  bool loaded = false;
  auto window = [&](int r0) {
    return [=](int lo) { return GlobalWindow(rows, s, lo, r0 + kRows < iv.len ? r0 + kRows : iv.len - 1); };
  };
  // rows of the block at r0 when one period covers its first row's window
  auto preload = [&](int r0) {
    loaded = false;
    if (!FIR || r0 >= r_end) return;
    period.find(iv, r0);
    if (period.lo > r0) return;
    const int low = r0 - (nb - 1);
    const GlobalWindow win = window(r0)(period.lo > low ? period.lo : low);
    win.load(r0 - (kRows - 1), x);
    win.load(r0 + 1, up);
    loaded = true;
  };
  preload(start + kRows * wave);
  int blk = wave;                                    // this wave's block, counted from start
  for (int first = start; first < r_end; first += kStep, blk += 4) {
    const int r0 = first + kRows * wave;
    const int n = r_end - r0 < kRows ? r_end - r0 : kRows;   // <= 0: past the tile
    const int slot = (int)((uint32_t)blk % kRingBlocks);
    bool fast = false;                               // every DC window complete, in one period
    float ac[kRows], ds[kRows];
    if (n > 0) {
      period.find(iv, r0);
      fast = boxcar && period.next >= r0 + n && r0 - (a.ndc - 1) >= period.lo;
      if constexpr (FIR) {
        fir_rows<kRows>(window(r0), iv, period, r0, n, b, nb, loaded, x, up, ac);
      } else {
        GlobalWindow(a.AC + iv.row0 * CM_SECTIONS, s, r0, r0 + n - 1).load(r0, ac);
      }
      float own[kRows];
      GlobalWindow(rows, s, r0, r0 + n - 1).load(r0, own);
      double sum = 0.0;
#pragma unroll
      for (int i = 0; i < kRows; ++i) {
        const float mid = __builtin_fmaf(own[i], coefA, -ac[i]);
        ds[i] = mid * mid;
        sum += (double)ds[i];
        ring.put(slot, i, ds[i]);
      }
      sums[slot * 64] = sum;
    }
    preload(r0 + kStep);                             // in flight during this trip's second half
    __syncthreads();
    if (n > 0 && r0 >= r_begin) {
      float dc[kRows];
      bool done = false;
      if (fast) {
        double acc[kRows];
        dc_boxcar(ring.col, sums, blk, a.ndc, ds, acc);
        // where the sums' distance leaves two floats open, the taps decide
        bool open = false;
#pragma unroll
        for (int i = 0; i < kRows; ++i) {
          const double y = acc[i] * dc0;
          dc[i] = (float)(y * (1.0 - kBoxcarBound));
          open = open || dc[i] != (float)(y * (1.0 + kBoxcarBound));
        }
        done = __builtin_amdgcn_ballot_w64(open) == 0;
      }
      if (!done) {
        // 8 rows at a time: the next block's rows and this block's AC stay in registers
        constexpr int kHalf = kRows / 2;
        float dx[kHalf], dup[kHalf - 1];
#pragma unroll
        for (int h = 0; h < kRows; h += kHalf)
          fir_rows<kHalf>([&](int lo) { return RingWindow{ring.col, start, lo, r0 + n - 1}; }, iv, period, r0 + h,
                          n - h < kHalf ? n - h : kHalf, a.dc, a.ndc, false, dx, dup, dc + h);
      }
      if (loaded) {   // wait for the next block's rows here: later, this block's stores would be waited for too
#pragma unroll
        for (int m = 0; m < kRows; ++m) asm volatile("" : "+v"(x[m]));
#pragma unroll
        for (int m = 0; m < kRows - 1; ++m) asm volatile("" : "+v"(up[m]));
      }
      node.store(a, log_tab, iv.row0 + r0, s, n, ac, ds, dc);
    }
    __syncthreads();   // the next trip's dS replaces the rings' oldest blocks
  }
}

}  // namespace cm

// Trips (64 rows each) of a one-pass workgroup's tile.  A tile of t trips
// yields 64 t - 96 rows, so long tiles waste less on their first kHalo rows and
// short ones spread a small batch over more of the chip: the estimate is the
// trips of a workgroup times the workgroups over the chip's places for them (2
// to a CU), which fill it at least once.  Measured: 4630 rows take 46 us at 2
// trips, 59 at 4 and 170 at 16; 847 k rows (96 intervals) 4151, 1859 and 1510.
static int tile_trips(const cm_ihc_interval *h_ivs, int n_ivs, int cus) {
  const int options[] = {2, 3, 4, 6, 8, 12, 16, 24, 32};
  int best = 0;
  int64_t best_cost = INT64_MAX;
  for (const int t : options) {
    const int64_t tile = cm::kStep * t - cm::kHalo;
    int64_t groups = 0;
    for (int i = 0; i < n_ivs; ++i) groups += (h_ivs[i].len + tile - 1) / tile * (CM_SECTIONS / 64);
    const int64_t cost = (groups > 2 * cus ? groups : 2 * cus) * t;
    if (cost < best_cost) {
      best_cost = cost;
      best = t;
    }
  }
  return best;
}

// Runs the whole IHC/lambda chain for one interval table.  One pass wherever
// every window starts in its interval (kbase 0), the DC window fits the tiles'
// halo and no output lies over the velocity: 16 B of HBM traffic per node, and the
// workspace d_scratch (2 x rows x 256 floats: AC, dS) is not touched unless an IIR
// AC filter writes its AC there first.  Other calls take two passes through the
// workspace.
// 847 k rows: one pass 1.52 ms, two passes (before the box-car sums and the
// shorter log10) 3.43 ms.
extern "C" int cm_launch_ihc_lambda(const float *d_bm, int64_t rows, const cm_ihc_interval *d_ivs,
                                    const cm_ihc_interval *h_ivs, int n_ivs, const cm_ihc_interval *d_iir_ivs,
                                    const cm_ihc_interval *h_iir_ivs, int n_iir_ivs, const double *d_ac_b, const double *d_ac_bpad,
                                    const double *d_ac_a, int n_ac, const double *d_dc, const double *d_dcpad, int n_dc, const double *d_damage, const float *d_A,
                                    const float *spont3, float lambda_sat, float eta_ac, float eta_dc, float scale_bm,
                                    float *d_scratch, float *d_lambda, float *d_stages, hipStream_t stream) {
  using namespace cm;
  if (n_ivs <= 0) return 0;
  int64_t max_len = 0;
  for (int i = 0; i < n_ivs; ++i) max_len = h_ivs[i].len > max_len ? h_ivs[i].len : max_len;
  const int64_t gx = (max_len + kRows - 1) / kRows;
  if (gx > 0x7fffffff || n_ivs > 65535) return -3;
  const int iir = d_ac_a != nullptr;
  LambdaArgs a;
  a.ivs = d_ivs;
  a.dc = d_dc;
  a.dcpad = d_dcpad;
  a.ndc = n_dc;
  a.etaAC = eta_ac;
  a.etaDC = eta_dc;
  a.damage = d_damage;
  a.A = d_A;
  for (int j = 0; j < 3; ++j) a.spont[j] = spont3[j];
  a.sat = lambda_sat;
  a.rows = rows;
  a.lambda = d_lambda;
  a.stages = d_stages;
  const bool one_pass = ihc_one_pass(h_ivs, n_ivs, n_dc, {d_bm, d_scratch, d_lambda, d_stages, rows});
  if (!d_scratch && (!one_pass || iir)) return -3;
  float *AC = d_scratch;
  float *dS = d_scratch ? d_scratch + rows * CM_SECTIONS : nullptr;
  a.AC = AC;
  a.dS = dS;
  if (iir) {
    int iir_len = 0;
    for (int i = 0; i < n_iir_ivs; ++i) iir_len = h_iir_ivs[i].len > iir_len ? h_iir_ivs[i].len : iir_len;
    if (launch_iir(d_bm, d_iir_ivs, n_iir_ivs, iir_len, d_ac_b, d_ac_a, n_ac, AC, stream)) return -1;
  }
  if (one_pass) {
    if (max_len <= 0) return 0;
    InlineIvs inl;
    if (!d_ivs)
      for (int i = 0; i < n_ivs; ++i) inl.v[i] = h_ivs[i];
    const int trips = tile_trips(h_ivs, n_ivs, device_cus());
    const int64_t tile = kStep * trips - kHalo;
    const dim3 grid((unsigned)((max_len + tile - 1) / tile * (CM_SECTIONS / 64)), n_ivs);
    if (iir)
      hipLaunchKernelGGL((ihc_lambda_kernel<false>), grid, dim3(256), 0, stream, const_cast<float *>(d_bm), d_ac_b, n_ac,
                         scale_bm, a, trips, inl);
    else
      hipLaunchKernelGGL((ihc_lambda_kernel<true>), grid, dim3(256), 0, stream, const_cast<float *>(d_bm), d_ac_b, n_ac,
                         scale_bm, a, trips, inl);
    return hipGetLastError() == hipSuccess ? 0 : -1;
  }
  hipLaunchKernelGGL(ac_ds_kernel, dim3((unsigned)gx, n_ivs), dim3(256), 0, stream, d_bm, d_ivs, d_ac_b, d_ac_bpad,
                     n_ac, scale_bm, iir, AC, dS);
  hipLaunchKernelGGL(dc_lambda_kernel, dim3((unsigned)gx, n_ivs), dim3(256), 0, stream, a);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

// Whether a call runs in one pass, and whether its table then travels in the
// kernel's arguments (d_ivs NULL) instead of through device memory.  One pass
// writes a tile's outputs while others still read the BM velocity around it, so
// outputs that lie over the velocity take two passes where there is a workspace:
// the second reads only that.
namespace cm {
static bool overlap(const float *a, int64_t na, const float *b, int64_t nb) {
  const uintptr_t x = (uintptr_t)a, y = (uintptr_t)b;
  return a && b && x < y + (uintptr_t)nb * sizeof(float) && y < x + (uintptr_t)na * sizeof(float);
}
bool ihc_one_pass(const cm_ihc_interval *h_ivs, int n_ivs, int n_dc, const IhcBuffers &b) {
  if (n_dc > kHalo + 1) return false;
  for (int i = 0; i < n_ivs; ++i)
    if (h_ivs[i].kbase != 0) return false;
  const int64_t plane = b.rows * CM_SECTIONS;
  return !b.scratch || !(overlap(b.bm, plane, b.lambda, 3 * plane) || overlap(b.bm, plane, b.stages, 5 * plane));
}
bool ihc_table_inline(const cm_ihc_interval *h_ivs, int n_ivs, int n_dc, const IhcBuffers &b) {
  return n_ivs <= kInlineIvs && ihc_one_pass(h_ivs, n_ivs, n_dc, b);
}
}  // namespace cm

// Spontaneous-rate fix-up of lambda loaded for a run that resumes from the
// lambda stage (CUDAFIXJND_Lambda, src/cochlea.cu:4512-4524): per fibre group
// k, buffer = max(spont_k, lambda) when kept, lambda = max(0, lambda - spont_k).
// Elementwise over [3][rows][256]; 16-byte accesses, grid-stride.
namespace cm {
__global__ __launch_bounds__(256) void fix_lambda_kernel(float4 *__restrict__ lam, float4 *__restrict__ buf,
                                                        int64_t plane4, float s0, float s1, float s2) {
  const int64_t n4 = 3 * plane4;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n4; i += stride) {
    const int k = (int)(i / plane4);
    const float s = k == 0 ? s0 : (k == 1 ? s1 : s2);
    const float4 v = lam[i];
    if (buf) buf[i] = make_float4(fmaxf(s, v.x), fmaxf(s, v.y), fmaxf(s, v.z), fmaxf(s, v.w));
    lam[i] = make_float4(fmaxf(0.0f, v.x - s), fmaxf(0.0f, v.y - s), fmaxf(0.0f, v.z - s), fmaxf(0.0f, v.w - s));
  }
}
}  // namespace cm

// lambda and buffer: [3][rows][256] floats (16-byte aligned device memory).
extern "C" int cm_launch_fix_lambda(float *d_lambda, float *d_buffer, int64_t rows, const float *spont3,
                                    hipStream_t stream) {
  if (rows <= 0) return 0;
  const int64_t plane4 = rows * (CM_SECTIONS / 4);
  int64_t blocks = (3 * plane4 + 255) / 256;
  if (blocks > 8192) blocks = 8192;
  hipLaunchKernelGGL(cm::fix_lambda_kernel, dim3((unsigned)blocks), dim3(256), 0, stream,
                     reinterpret_cast<float4 *>(d_lambda), reinterpret_cast<float4 *>(d_buffer), plane4, spont3[0],
                     spont3[1], spont3[2]);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}
