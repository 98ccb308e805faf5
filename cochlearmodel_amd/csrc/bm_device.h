// Device functions of the BM/OHC velocity solver with the semantics of the
// reference's kernel #17 (include/cochlea.cuh:13573-14245, launched from
// src/cochlea.cu:1436-1493), shared by the fused kernels (bm_kernel.hip,
// bm_split_kernel.hip) and the learned warm-start kernel.
//
// gfx950 layout: one wave64 integrates one time block; lane l holds the four
// consecutive sections 4l..4l+3 in registers.  The Jacobi pressure sweep
// exchanges the two lane-boundary pressures with DPP wave shifts, the three
// step-control reductions run interleaved as DPP trees, and accept/reject is a
// lane-uniform decision.  No LDS, no barriers.  The same functions also run a
// block over a workgroup of 4 or 8 waves (2 or 1 sections per lane), which carry
// their neighbours' sections and exchange pressures and totals through LDS
// (Lay<N> below); results are identical in every layout.
//
// Arithmetic contract (shared with the CPU oracle): FP32, every operation
// IEEE-rounded, no contraction (built with -ffp-contract=off), IEEE division
// where the reference uses __fdividef, tanh by tanh_slots below, and the fixed
// reduction tree (s0+s1)+(s2+s3) -> xor 1,2,4,8 -> (r0+r16)+(r32+r48).
#ifndef CM_BM_DEVICE_H
#define CM_BM_DEVICE_H

#include <hip/hip_runtime.h>

#include "cm_internal.h"

namespace cm {


// ----------------------------------------------------------- math ------
__device__ __forceinline__ float exp_reduced(float y) {
  const float log2e = 1.44269502e+00f;
  const float ln2_hi = 6.93145752e-01f;
  const float ln2_lo = 1.42860677e-06f;
  float k = __builtin_rintf(y * log2e);
  float r = __builtin_fmaf(-k, ln2_hi, y);
  r = __builtin_fmaf(-k, ln2_lo, r);
  float p = 2.48015873e-05f;
  p = __builtin_fmaf(p, r, 1.98412701e-04f);
  p = __builtin_fmaf(p, r, 1.38888892e-03f);
  p = __builtin_fmaf(p, r, 8.33333377e-03f);
  p = __builtin_fmaf(p, r, 4.16666679e-02f);
  p = __builtin_fmaf(p, r, 1.66666672e-01f);
  p = __builtin_fmaf(p, r, 5.00000000e-01f);
  p = __builtin_fmaf(p, r, 1.0f);
  p = __builtin_fmaf(p, r, 1.0f);
  return __builtin_ldexpf(p, (int)k);
}

// tanh of a lane's N values: odd series below 0.55, 1 - 2/(e^{2a}+1) below 10,
// 1 beyond.  The series runs for all N values together (independent chains, no
// branch per value; odd, so it needs no sign handling); the exponential form
// follows only when some lane of the wave holds an argument of 0.55 or more.
// There the divisor e + 1 lies in [2, 5e8], so the division is the correctly
// rounded sequence of reciprocal, Newton step and two residual corrections
// without range scaling.  (A NaN may leave as a NaN or, as beyond 10, as 1; it
// meets the same NaN again in psi's own term of the same sum.)
template <int N>
__device__ __forceinline__ void tanh_slots(const float (&x)[N], float (&r)[N]) {
  float q[N], z[N];
#pragma unroll
  for (int j = 0; j < N; ++j) {
    z[j] = x[j] * x[j];
    q[j] = __builtin_fmaf(-2.39129114e-04f, z[j], 5.90027441e-04f);
  }
  constexpr float c[7] = {-1.45583438e-03f, 3.59212812e-03f, -8.86323989e-03f, 2.18694881e-02f,
                          -5.39682540e-02f, 1.33333340e-01f, -3.33333343e-01f};
#pragma unroll
  for (int i = 0; i < 7; ++i)
#pragma unroll
    for (int j = 0; j < N; ++j) q[j] = __builtin_fmaf(q[j], z[j], c[i]);
  float m = __builtin_fabsf(x[0]);
#pragma unroll
  for (int j = 1; j < N; ++j) m = fmaxf(m, __builtin_fabsf(x[j]));
#pragma unroll
  for (int j = 0; j < N; ++j) r[j] = __builtin_fmaf(x[j] * z[j], q[j], x[j]);
  if (__builtin_amdgcn_ballot_w64(!(m < 0.55f)) != 0) {
#pragma unroll
    for (int j = 0; j < N; ++j) {
      const float a = __builtin_fabsf(x[j]);
      const float d = exp_reduced(a + a) + 1.0f;
      float y = __builtin_amdgcn_rcpf(d);
      y = __builtin_fmaf(__builtin_fmaf(-d, y, 1.0f), y, y);
      float t = 2.0f * y;
      t = __builtin_fmaf(__builtin_fmaf(-d, t, 2.0f), y, t);
      t = __builtin_fmaf(__builtin_fmaf(-d, t, 2.0f), y, t);
      const float big = a < 10.0f ? 1.0f - t : 1.0f;
      r[j] = a < 0.55f ? r[j] : __builtin_copysignf(big, x[j]);
    }
  }
}

// ------------------------------------------------------------ DPP ------
#define CM_DPP(x, ctrl) \
  __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), (ctrl), 0xF, 0xF, true))
// lane i <- lane i-1 (lane 0 <- 0)
__device__ __forceinline__ float wave_shr1(float x) { return CM_DPP(x, 0x138); }
// lane i <- lane i+1 (lane 63 <- 0)
__device__ __forceinline__ float wave_shl1(float x) { return CM_DPP(x, 0x130); }
__device__ __forceinline__ float quad_xor1(float x) { return CM_DPP(x, 0xB1); }
__device__ __forceinline__ float quad_xor2(float x) { return CM_DPP(x, 0x4E); }
__device__ __forceinline__ float row_half_mirror(float x) { return CM_DPP(x, 0x141); }
__device__ __forceinline__ float row_mirror(float x) { return CM_DPP(x, 0x140); }
__device__ __forceinline__ float readlane(float x, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), l));
}

// Row broadcasts: every row r >= 1 <- lane 15 of row r-1; rows 2 and 3 <-
// lane 31.  Only row 3 is read afterwards, so what the other rows receive
// does not matter and the full row mask lets the move fold into the add.
__device__ __forceinline__ float row_bcast15(float x) { return CM_DPP(x, 0x142); }
__device__ __forceinline__ float row_bcast31(float x) { return CM_DPP(x, 0x143); }

// Sum of 256 values, 4 per lane, with the fixed tree
// ((r0 + r1) + (r2 + r3)) of the row sums r_k.  After the xor steps every lane
// of row k holds r_k; the two row broadcasts leave (r3 + r2) + (r1 + r0) in
// row 3, which equals the tree because each addition is commutative.
__device__ __forceinline__ float tree_sum(float x0, float x1, float x2, float x3) {
  float s = (x0 + x1) + (x2 + x3);
  s = s + quad_xor1(s);
  s = s + quad_xor2(s);
  s = s + row_half_mirror(s);   // equals xor 4 once quads are uniform
  s = s + row_mirror(s);        // equals xor 8 once octets are uniform
  s = s + row_bcast15(s);
  s = s + row_bcast31(s);
  return readlane(s, 63);
}
// The cross-lane part of the tree for three (or two) per-lane values at once.
// A DPP operand needs two other instructions after the one that wrote it, so
// one tree alone waits in every step; three interleaved trees never do.  One
// asm block, because the compiler keeps the trees apart and, for the maximum,
// adds a canonicalising move and operation per step (values here come from
// arithmetic, so no operand is a signalling NaN).  Nor does the compiler see what
// a block wrote last, so each block ends with the wait states that a reader of it
// needs: two after v_readlane, for a vector instruction that reads the SGPR, and
// one after a VGPR, for v_readlane.
#define CM_SGPR_READY "\n\ts_nop 1"
#define CM_VGPR_READY "s_nop 0"
#define CM_TREE3(op0, op1, op2, ctrl)                                   \
  op0 " %0, %0, %0 " ctrl " row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t" \
  op1 " %1, %1, %1 " ctrl " row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t" \
  op2 " %2, %2, %2 " ctrl " row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
#define CM_TREE2(ctrl)                                                          \
  "v_add_f32_dpp %0, %0, %0 " ctrl " row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t" \
  "v_add_f32_dpp %1, %1, %1 " ctrl " row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t" \
  "s_nop 0\n\t"
#define CM_TREE_STEPS(step) \
  step("quad_perm:[1,0,3,2]") step("quad_perm:[2,3,0,1]") step("row_half_mirror") step("row_mirror") \
      step("row_bcast:15") step("row_bcast:31")
#define CM_TREE_MAX_SUM_SUM(ctrl) CM_TREE3("v_max_f32_dpp", "v_add_f32_dpp", "v_add_f32_dpp", ctrl)
#define CM_TREE_SUM3(ctrl) CM_TREE3("v_add_f32_dpp", "v_add_f32_dpp", "v_add_f32_dpp", ctrl)
#define CM_TREE_READ3 \
  "v_readlane_b32 %3, %0, 63\n\tv_readlane_b32 %4, %1, 63\n\tv_readlane_b32 %5, %2, 63" CM_SGPR_READY
__device__ __forceinline__ void tree_max_sum_sum(float &x, float &y, float &z) {
  float a, b, c;
  asm("s_nop 1\n\t" CM_TREE_STEPS(CM_TREE_MAX_SUM_SUM) CM_TREE_READ3
      : "+&v"(x), "+&v"(y), "+&v"(z), "=s"(a), "=s"(b), "=s"(c));
  x = a; y = b; z = c;
}
__device__ __forceinline__ void tree_sum3(float &x, float &y, float &z) {
  float a, b, c;
  asm("s_nop 1\n\t" CM_TREE_STEPS(CM_TREE_SUM3) CM_TREE_READ3
      : "+&v"(x), "+&v"(y), "+&v"(z), "=s"(a), "=s"(b), "=s"(c));
  x = a; y = b; z = c;
}
__device__ __forceinline__ void tree_sum2(float &x, float &y) {
  float a, b;
  asm("s_nop 1\n\t" CM_TREE_STEPS(CM_TREE2) "v_readlane_b32 %2, %0, 63\n\tv_readlane_b32 %3, %1, 63" CM_SGPR_READY
      : "+&v"(x), "+&v"(y), "=s"(a), "=s"(b));
  x = a; y = b;
}

#define UNROLL _Pragma("unroll")

// The four steps inside a row of 16 lanes, or the first three of them, for 1 to
// 3 values (MAX0: the first is a maximum), as above.
#define CM_TREE1(ctrl) \
  "s_nop 1\n\tv_add_f32_dpp %0, %0, %0 " ctrl " row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
#define CM_OCT_STEPS(step) step("quad_perm:[1,0,3,2]") step("quad_perm:[2,3,0,1]") step("row_half_mirror")
#define CM_ROW_STEPS(step) CM_OCT_STEPS(step) step("row_mirror")
template <int K, bool MAX0, bool ROW>
__device__ __forceinline__ void tree_row(float (&v)[K]) {
  static_assert(K >= 1 && K <= 3 && !(MAX0 && K != 3), "one to three sums, or a maximum and two sums");
  if constexpr (K == 1) {
    if constexpr (ROW) asm(CM_ROW_STEPS(CM_TREE1) CM_VGPR_READY : "+v"(v[0]));
    else asm(CM_OCT_STEPS(CM_TREE1) CM_VGPR_READY : "+v"(v[0]));
  } else if constexpr (K == 2) {   // CM_TREE2 ends with a wait state
    if constexpr (ROW) asm("s_nop 1\n\t" CM_ROW_STEPS(CM_TREE2) : "+v"(v[0]), "+v"(v[1]));
    else asm("s_nop 1\n\t" CM_OCT_STEPS(CM_TREE2) : "+v"(v[0]), "+v"(v[1]));
  } else if constexpr (MAX0) {
    if constexpr (ROW)
      asm("s_nop 1\n\t" CM_ROW_STEPS(CM_TREE_MAX_SUM_SUM) CM_VGPR_READY : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]));
    else
      asm("s_nop 1\n\t" CM_OCT_STEPS(CM_TREE_MAX_SUM_SUM) CM_VGPR_READY : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]));
  } else {
    if constexpr (ROW) asm("s_nop 1\n\t" CM_ROW_STEPS(CM_TREE_SUM3) CM_VGPR_READY : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]));
    else asm("s_nop 1\n\t" CM_OCT_STEPS(CM_TREE_SUM3) CM_VGPR_READY : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]));
  }
}

__device__ __forceinline__ float in_at(const BmLaunch &a, int64_t idx) {
  return (idx >= 0 && idx < a.input_len) ? a.input[idx] : 0.0f;
}

__device__ __forceinline__ float uniform(float x) {
  return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(x)));
}

template <int N>
__device__ __forceinline__ void ld_slots(const float *p, float (&o)[N]) {
  if constexpr (N == 4) {
    const float4 v = *reinterpret_cast<const float4 *>(p);
    o[0] = v.x; o[1] = v.y; o[2] = v.z; o[3] = v.w;
  } else if constexpr (N == 2) {
    const float2 v = *reinterpret_cast<const float2 *>(p);
    o[0] = v.x; o[1] = v.y;
  } else {
    o[0] = *p;
  }
}
template <int N>
__device__ __forceinline__ void st_slots(float *p, const float (&v)[N]) {
  if constexpr (N == 4)
    *reinterpret_cast<float4 *>(p) = make_float4(v[0], v[1], v[2], v[3]);
  else if constexpr (N == 2)
    *reinterpret_cast<float2 *>(p) = make_float2(v[0], v[1]);
  else
    *p = v[0];
}

// ------------------------------------------------ section layouts -------
// A block's 256 sections over the W waves of a workgroup, N consecutive ones
// per lane.
//
// N = 4 is one wave per block (W = 1): neighbour pressures move by DPP wave
// shifts, reductions run as DPP butterflies, nothing goes through LDS and there
// is no barrier.
//
// N = 2 and N = 1 spread a block over W = 4 and 8 waves, for launches that
// leave SIMDs without a wave.  A wave owns 32 N sections (two rows of lanes)
// and carries 16 N more on either side of them (on one side, twice as many, in
// the first and last wave, so that a wave's ends are the block's ends).  All
// its lanes do the same work, so a Jacobi sweep needs no exchange: each one
// spoils the outermost valid section only, and after up to kReach sweeps the
// owned sections are still those of the one-wave layout.  Then the owners'
// pressures pass to the others through LDS behind a workgroup barrier (share),
// and everything else follows from them in every lane that holds the section.
// Totals of the owned sections pass the same way.  The area has two halves used
// in turn, so one barrier per exchange suffices: a wave writes a half again
// only after the next exchange's barrier, which every wave reaches after its
// reads of that half.  Totals leave an exchange through readlane, so every
// branch that depends on them is a scalar branch, and every wave of a block
// forms the same totals bit for bit (the tree below) and takes the same
// branches: the barriers always match.
template <int N>
struct Lay {
  static_assert(N == 1 || N == 2 || N == 4, "1, 2 or 4 sections per lane");
  static constexpr int W = N == 4 ? 1 : 8 / N;
  static constexpr int kReach = N == 4 ? 1 << 30 : 16 * N - 1;   // sweeps between exchanges; one valid neighbour remains
  // bytes of a half: two vectors, 2 W part totals of up to 4 floats, and a place
  // for what lanes write that own nothing (a power of two: halves alternate by xor)
  static constexpr unsigned kVec = 4 * CM_SECTIONS, kParts = 2 * kVec, kIdle = kParts + 16 * 2 * W, kHalf = 4096;
  static_assert(kIdle + 4 * 64 * 4 <= kHalf, "a half holds its idle place");
  int lane;
  int wave;    // wave of the block (0 when W == 1)
  char *xa;    // exchange area: 2 halves (W > 1)
  float p0;    // section 0's pressure of the last share (W > 1)
  unsigned put_at, part_at, get_at, total_at;   // this lane's places in the half of the next exchange (W > 1)

  __device__ __forceinline__ Lay(int lane_, int wave_, char *xa_) : lane(lane_), wave(wave_), xa(xa_), p0(0.f) {
    if constexpr (W > 1) {
      const int rel = lane - own_lane();
      unsigned mine = 4 * base(), part = kParts + 16 * (2 * wave + (rel >> 4));
      asm volatile("" : "+v"(mine), "+v"(part));   // selected below, not branched around
      put_at = (unsigned)rel < 32u ? mine : kIdle + 4 * N * lane;
      part_at = (rel & ~16) == 0 ? part : kIdle + 16 * lane;
      get_at = mine;
      total_at = kParts + 16 * (lane & (2 * W - 1));
    }
  }

  // The lane, compared anew at each use (W > 1): masks of lanes kept over the
  // steps would take more scalar registers than there are.
  __device__ __forceinline__ int here() const {
    int l = lane;
    if constexpr (W > 1) asm volatile("" : "+v"(l));
    return l;
  }
  __device__ bool sec0() const { return (W == 1 || wave == 0) && here() == 0; }
  __device__ bool last() const { return (W == 1 || wave == W - 1) && here() == 63; }
  __device__ int base() const {
    if constexpr (W == 1) return N * lane;
    const int first = wave == 0 ? 0 : (wave == W - 1 ? CM_SECTIONS - 64 * N : 32 * N * wave - 16 * N);
    return first + N * lane;
  }
  // first of the 32 lanes whose sections this wave owns
  __device__ int own_lane() const { return wave == 0 ? 0 : (wave == W - 1 ? 32 : 16); }
  __device__ bool own() const { return W == 1 || (unsigned)(here() - own_lane()) < 32u; }
  // Slots that can hold section 254 or 255, whose lower coupling l_i is 0
  // (l_i = 1 elsewhere): slots 2 and 3 when N = 4, every slot otherwise.
  static constexpr bool has_low(int j) { return N == 4 ? j >= 2 : true; }
  __device__ float low() const {
    if (N == 4) return lane == 63 ? 0.0f : 1.0f;
    return base() + N - 1 >= 254 ? 0.0f : 1.0f;
  }

  // Pressures of the sections just before and after this lane's slots (0 past
  // either end of the wave), from every lane's last and first slot.
  __device__ __forceinline__ void nbrs(float last_v, float first_v, float &left, float &right) const {
    left = wave_shr1(last_v);
    right = wave_shl1(first_v);
  }

  // ---- exchanges (W > 1) ----
  // Writes of an exchange: the owned sections of vector `which`.
  __device__ __forceinline__ void put(const float (&x)[N], int which) const {
    st_slots<N>(reinterpret_cast<float *>(xa + put_at) + which * CM_SECTIONS, x);
  }
  // The one-wave tree is (s0 + s1) + (s2 + s3) over each lane's four sections,
  // then xor 1, 2, 4, 8 up to the 64-section sums R_k and (R0 + R1) + (R2 + R3).
  // Here a group of 4 sections spans 2 lanes (N = 2) or a quad (N = 1), a row of
  // lanes holds 16 N sections, and lane i continues with the total of row i of
  // the block: each step adds the same two partial sums as the matching one-wave
  // step (IEEE addition is commutative).
  template <int K, bool MAX0>
  __device__ __forceinline__ void put_parts(float (&v)[K]) const {
    tree_row<K, MAX0, true>(v);
    float *h = reinterpret_cast<float *>(xa + part_at);
    UNROLL for (int k = 0; k < K; ++k) h[k] = v[k];
  }
  // Ends the writes; returns the half to read from.  LDS only is waited for:
  // rows on their way to memory are not.
  struct Half {
    unsigned get_at, total_at;
  };
  __device__ __forceinline__ Half meet() {
    const Half h{get_at, total_at};
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    put_at ^= kHalf; part_at ^= kHalf; get_at ^= kHalf; total_at ^= kHalf;
    return h;
  }
  template <int K, bool MAX0>
  __device__ __forceinline__ void get_totals(const Half &h, float (&v)[K]) const {
    const float *t = reinterpret_cast<const float *>(xa + h.total_at);
    UNROLL for (int k = 0; k < K; ++k) v[k] = t[k];
    tree_row<K, MAX0, N == 1>(v);
    UNROLL for (int k = 0; k < K; ++k) v[k] = readlane(v[k], 0);
  }
  __device__ __forceinline__ void get(const Half &h, int which, float (&x)[N]) {
    ld_slots<N>(reinterpret_cast<const float *>(xa + h.get_at) + which * CM_SECTIONS, x);
    p0 = reinterpret_cast<const float *>(xa + (h.get_at & kHalf))[which * CM_SECTIONS];
  }
  // Every lane's pressures from their owners.
  __device__ __forceinline__ void share(float (&p)[N]) {
    if constexpr (W > 1) {
      put(p, 0);
      get(meet(), 0, p);
    }
  }
  template <int K, bool MAX0>
  __device__ __forceinline__ void totals(float (&v)[K]) {
    put_parts<K, MAX0>(v);
    get_totals<K, MAX0>(meet(), v);
  }
  static __device__ __forceinline__ float lane_sum(const float (&x)[N]) {
    if constexpr (N == 4) return (x[0] + x[1]) + (x[2] + x[3]);
    else if constexpr (N == 2) return x[0] + x[1];
    else return x[0];
  }
  static __device__ __forceinline__ float lane_max(const float (&x)[N]) {
    if constexpr (N == 4) return fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3]));
    else if constexpr (N == 2) return fmaxf(x[0], x[1]);
    else return x[0];
  }

  __device__ __forceinline__ float sum(const float (&x)[N]) {
    if constexpr (N == 4) {
      return tree_sum(x[0], x[1], x[2], x[3]);
    } else {
      float v[1] = {lane_sum(x)};
      totals<1, false>(v);
      return v[0];
    }
  }
  // reduce3 and share in one exchange (W > 1)
  __device__ __forceinline__ void reduce3_share(const float (&ex)[N], const float (&ey)[N], const float (&ez)[N],
                                                float (&p)[N], float &emax, float &esum, float &fsum) {
    float v[3] = {lane_max(ex), lane_sum(ey), lane_sum(ez)};
    put(p, 0);
    put_parts<3, true>(v);
    const Half h = meet();
    get(h, 0, p);
    get_totals<3, true>(h, v);
    emax = v[0]; esum = v[1]; fsum = v[2];
  }
  // max of ex, sums of ey and ez: the three step-control reductions
  __device__ __forceinline__ void reduce3(const float (&ex)[N], const float (&ey)[N], const float (&ez)[N],
                                          float &emax, float &esum, float &fsum) {
    float v[3] = {lane_max(ex), lane_sum(ey), lane_sum(ez)};
    if constexpr (N == 4) tree_max_sum_sum(v[0], v[1], v[2]);
    else totals<3, true>(v);
    emax = v[0]; esum = v[1]; fsum = v[2];
  }
  // sums of the squares of two or three vectors
  __device__ __forceinline__ void sum_sq2(const float (&x)[N], const float (&y)[N], float &sx, float &sy) {
    float a[N], b[N];
    UNROLL for (int j = 0; j < N; ++j) { a[j] = x[j] * x[j]; b[j] = y[j] * y[j]; }
    float v[2] = {lane_sum(a), lane_sum(b)};
    if constexpr (N == 4) tree_sum2(v[0], v[1]);
    else totals<2, false>(v);
    sx = v[0]; sy = v[1];
  }
  __device__ __forceinline__ void sum_sq3(const float (&x)[N], const float (&y)[N], const float (&z)[N], float &sx,
                                          float &sy, float &sz) {
    float a[N], b[N], c[N];
    UNROLL for (int j = 0; j < N; ++j) { a[j] = x[j] * x[j]; b[j] = y[j] * y[j]; c[j] = z[j] * z[j]; }
    float v[3] = {lane_sum(a), lane_sum(b), lane_sum(c)};
    if constexpr (N == 4) tree_sum3(v[0], v[1], v[2]);
    else totals<3, false>(v);
    sx = v[0]; sy = v[1]; sz = v[2];
  }
  // section 0's pressure in every lane (W > 1: of the last share)
  __device__ __forceinline__ float sec0_value(float x0) const {
    if constexpr (W == 1) return readlane(x0, 0);
    else return p0;
  }
};

// ------------------------------------------------- one time block -------
// Per-lane constants of an item: section parameters of this lane's N sections.
template <int N>
struct ItemConstN {
  float rsm[N], rmass[N], gam[N], R[N], S[N], Q[N], Sohc[N], Stm[N], Rtm[N], mf[N];
  float low;   // lower-coupling multiplier l_i of the Lay<N>::has_low slots
};

// Scalars shared by all lanes (uniform).
struct ItemScal {
  float w_ohc, alpha_r, Ts, al, Gme, a1, eta1, eta2, dt_min, dt_max, tso, mtt, mmspt;
  float al_over_as, dxdx, dxa0, neg_a2, neg_as, span;
  double inv_sigma_ow;
};

// One side of an integration step (include/cochlea.cuh:13620-13700 names:
// displacement, velocity, acceleration, psi, its derivative, xi's derivative
// and xi per section, and the oval window's displacement, velocity and
// acceleration).
template <int N>
struct HalfN {
  float d[N], v[N], a[N], psi[N], psid[N], xis[N], xi[N];
  float ow_d, ow_v, ow_a;
};

// Integration state of an item: two sides, the committed one and the one the
// passes of a step work on.  Which is which alternates from step to step, so
// a commit copies nothing.
template <int N>
struct ItemStateN {
  HalfN<N> A, B;
  float Ptm[N];
  float p[N];                                                          // resident pressure
  float dt, t, sx0, sx1;
  int in_s;
  float c_fail, c_dt, c_steps, c_passes;                               // sx[11], sx[12], sx[13], sx[15]
  int64_t n_steps, n_passes, n_sweeps;
  int32_t fb;
  float ctb, clb, cjb;
};
using ItemConst = ItemConstN<4>;
using ItemState = ItemStateN<4>;
using Half = HalfN<4>;

// The functions below take the per-lane section constants as K: ItemConstN<N>
// (every row in registers) or a type with the same members whose rarely read
// rows are pointers into LDS (the learned kernel's WsConst).

// a_i = l_i p_{i-1} + p_{i+1} of slot j (include/cochlea.cuh:13962-13982).  l_i
// is 0 or 1, so l_i p_{i-1} is exact and fma(l_i, p_{i-1}, p_{i+1}) rounds as
// the separate multiply and add do; the fma is used where both operands are
// in the lane (one instruction), the multiply and add where one comes from a
// DPP shift (which folds into the add).
template <int N>
__device__ __forceinline__ float coupling(int j, float low, float pl, float pr) {
  if (!Lay<N>::has_low(j)) return pl + pr;
  if (j > 0 && j < N - 1) return __builtin_fmaf(low, pl, pr);
  return low * pl + pr;
}

// One Jacobi sweep of the kernel convention, p_i <- (Y_i - a_i) / m_i with the
// reciprocal diagonal.
template <int N, class K>
__device__ __forceinline__ void jacobi_sweep(Lay<N> &L, const float (&Y)[N], const K &k,
                                             const float (&p)[N], float (&q)[N]) {
  float left, right;
  L.nbrs(p[N - 1], p[0], left, right);
  UNROLL for (int j = 0; j < N; ++j) {
    const float pl = j == 0 ? left : p[j - 1];
    const float pr = j == N - 1 ? right : p[j + 1];
    q[j] = (Y[j] - coupling<N>(j, k.low, pl, pr)) * k.rsm[j];
  }
}
// Sweeps of the one-wave layout in asm: 12 VALU instructions per sweep and no
// wait.  t <- sweep(p) reads p through DPP in its first two instructions, and
// the products that feed them (slots 0 and 3) come first among the previous
// sweep's last four, so every DPP operand is at least two instructions old;
// the compiler's loop took 13 and a wait.  The 13th was slot 3's coupling:
// l_255 = 0 and no section follows 255, so there it is l p_254 + 0, which does
// not change from sweep to sweep; %[a3]'s lane 63 holds it, and the shift
// without bound_ctrl leaves that lane alone.  (p_254 only enters it as 0 times
// itself; a non-finite p_254 still makes it NaN from the next call on.)
#define CM_SWEEP(p0, p1, p2, p3, t0, t1, t2, t3)                                                      \
  "v_add_f32_dpp %[" t0 "], %[" p3 "], %[" p1 "] wave_shr:1 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t" \
  "v_add_f32_dpp %[a3], %[" p0 "], %[" p2 "] wave_shl:1 row_mask:0xf bank_mask:0xf\n\t"              \
  "v_add_f32 %[" t1 "], %[" p0 "], %[" p2 "]\n\t"                                                    \
  "v_fma_f32 %[" t2 "], %[low], %[" p1 "], %[" p3 "]\n\t"                                            \
  "v_sub_f32 %[" t0 "], %[Y0], %[" t0 "]\n\t"                                                        \
  "v_sub_f32 %[" t3 "], %[Y3], %[a3]\n\t"                                                            \
  "v_sub_f32 %[" t1 "], %[Y1], %[" t1 "]\n\t"                                                        \
  "v_sub_f32 %[" t2 "], %[Y2], %[" t2 "]\n\t"                                                        \
  "v_mul_f32 %[" t0 "], %[r0], %[" t0 "]\n\t"                                                        \
  "v_mul_f32 %[" t3 "], %[r3], %[" t3 "]\n\t"                                                        \
  "v_mul_f32 %[" t1 "], %[r1], %[" t1 "]\n\t"                                                        \
  "v_mul_f32 %[" t2 "], %[r2], %[" t2 "]\n\t"
#define CM_SWEEP_PT CM_SWEEP("p0", "p1", "p2", "p3", "t0", "t1", "t2", "t3")
#define CM_SWEEP_TP CM_SWEEP("t0", "t1", "t2", "t3", "p0", "p1", "p2", "p3")
#define CM_SWEEP_IN                                                                                     \
  [Y0] "v"(Y[0]), [Y1] "v"(Y[1]), [Y2] "v"(Y[2]), [Y3] "v"(Y[3]), [r0] "v"(r[0]), [r1] "v"(r[1]),       \
      [r2] "v"(r[2]), [r3] "v"(r[3]), [low] "v"(low)
// J >= 0 sweeps; with TENS ten per trip as long as that many are left, the rest
// PAIRS (1 or 2) pairs per trip.
template <int PAIRS, bool TENS>
__device__ __forceinline__ void sweeps_asm(const float (&Y)[4], const float (&r)[4], float low, float (&p)[4], int J) {
  float a3 = low * p[2] + 0.0f;
  float t0, t1, t2, t3;
  if (TENS && __builtin_expect(J >= 10, 1)) {
    int n = J / 10;
    J -= 10 * n;
    asm("s_nop 1\n"
        "1:\n\t" CM_SWEEP_PT CM_SWEEP_TP CM_SWEEP_PT CM_SWEEP_TP CM_SWEEP_PT CM_SWEEP_TP CM_SWEEP_PT CM_SWEEP_TP
        CM_SWEEP_PT CM_SWEEP_TP "s_sub_i32 %[n], %[n], 1\n\ts_cmp_lg_u32 %[n], 0\n\ts_cbranch_scc1 1b\n\t"
        : [p0] "+&v"(p[0]), [p1] "+&v"(p[1]), [p2] "+&v"(p[2]), [p3] "+&v"(p[3]), [a3] "+&v"(a3), [n] "+&s"(n),
          [t0] "=&v"(t0), [t1] "=&v"(t1), [t2] "=&v"(t2), [t3] "=&v"(t3)
        : CM_SWEEP_IN
        : "scc");
    if (__builtin_expect(J == 0, 1)) return;
  }
  int n = J / (2 * PAIRS);
  if (n > 0) {
    if constexpr (PAIRS == 1)
      asm("s_nop 1\n"
          "1:\n\t" CM_SWEEP_PT CM_SWEEP_TP
          "s_sub_i32 %[n], %[n], 1\n\ts_cmp_lg_u32 %[n], 0\n\ts_cbranch_scc1 1b\n\t"
          : [p0] "+&v"(p[0]), [p1] "+&v"(p[1]), [p2] "+&v"(p[2]), [p3] "+&v"(p[3]), [a3] "+&v"(a3), [n] "+&s"(n),
            [t0] "=&v"(t0), [t1] "=&v"(t1), [t2] "=&v"(t2), [t3] "=&v"(t3)
          : CM_SWEEP_IN
          : "scc");
    else
      asm("s_nop 1\n"
          "1:\n\t" CM_SWEEP_PT CM_SWEEP_TP CM_SWEEP_PT CM_SWEEP_TP
          "s_sub_i32 %[n], %[n], 1\n\ts_cmp_lg_u32 %[n], 0\n\ts_cbranch_scc1 1b\n\t"
          : [p0] "+&v"(p[0]), [p1] "+&v"(p[1]), [p2] "+&v"(p[2]), [p3] "+&v"(p[3]), [a3] "+&v"(a3), [n] "+&s"(n),
            [t0] "=&v"(t0), [t1] "=&v"(t1), [t2] "=&v"(t2), [t3] "=&v"(t3)
          : CM_SWEEP_IN
          : "scc");
  }
  if (PAIRS == 2 && (J & 2))
    asm("s_nop 1\n\t" CM_SWEEP_PT CM_SWEEP_TP
        : [p0] "+&v"(p[0]), [p1] "+&v"(p[1]), [p2] "+&v"(p[2]), [p3] "+&v"(p[3]), [a3] "+&v"(a3), [t0] "=&v"(t0),
          [t1] "=&v"(t1), [t2] "=&v"(t2), [t3] "=&v"(t3)
        : CM_SWEEP_IN);
  if (TENS ? __builtin_expect(J & 1, 0) : J & 1) {
    asm("s_nop 1\n\t" CM_SWEEP_PT
        : [a3] "+&v"(a3), [t0] "=&v"(t0), [t1] "=&v"(t1), [t2] "=&v"(t2), [t3] "=&v"(t3)
        : [p0] "v"(p[0]), [p1] "v"(p[1]), [p2] "v"(p[2]), [p3] "v"(p[3]), CM_SWEEP_IN);
    p[0] = t0; p[1] = t1; p[2] = t2; p[3] = t3;
  }
}

// The spread layouts' sweeps.  Section 254 sits in a slot whose left neighbour
// comes through DPP, which cannot fold l_i: a move of the right neighbour and a
// multiply-add of l_i and the left one take its place (7 instructions for two
// sections, 4 and a wait for one).  Operands read through DPP are two
// instructions old, here and after the last sweep.
#define CM_SWEEP2(p0, p1, t0, t1)                                                                    \
  "v_mov_b32 %[" t0 "], %[" p1 "]\n\t"                                                               \
  "v_add_f32_dpp %[a1], %[" p0 "], %[" p0 "] wave_shl:1 row_mask:0xf bank_mask:0xf\n\t"              \
  "v_fmac_f32_dpp %[" t0 "], %[" p1 "], %[low] wave_shr:1 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t" \
  "v_sub_f32 %[" t1 "], %[Y1], %[a1]\n\t"                                                            \
  "v_sub_f32 %[" t0 "], %[Y0], %[" t0 "]\n\t"                                                        \
  "v_mul_f32 %[" t0 "], %[r0], %[" t0 "]\n\t"                                                        \
  "v_mul_f32 %[" t1 "], %[r1], %[" t1 "]\n\t"
#define CM_SWEEP1(p0, t0)                                                                            \
  "s_nop 1\n\t"                                                                                      \
  "v_mov_b32_dpp %[" t0 "], %[" p0 "] wave_shl:1 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"        \
  "v_fmac_f32_dpp %[" t0 "], %[" p0 "], %[low] wave_shr:1 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t" \
  "v_sub_f32 %[" t0 "], %[Y0], %[" t0 "]\n\t"                                                        \
  "v_mul_f32 %[" t0 "], %[r0], %[" t0 "]\n\t"
#define CM_PAIR2 CM_SWEEP2("p0", "p1", "t0", "t1") CM_SWEEP2("t0", "t1", "p0", "p1")
#define CM_PAIR1 CM_SWEEP1("p0", "t0") CM_SWEEP1("t0", "p0")
#define CM_LOOP(body) \
  "s_nop 1\n" "1:\n\t" body "s_sub_i32 %[n], %[n], 1\n\ts_cmp_lg_u32 %[n], 0\n\ts_cbranch_scc1 1b\n\t"
template <int PAIRS, bool TENS, int N>
__device__ __forceinline__ void sweeps_spread(const float (&Y)[N], const float (&r)[N], float low, float (&p)[N],
                                              int J) {
  if constexpr (N == 2) {
    // of the wave's last lane, which has no right neighbour (as a3 above)
    float a1 = low * p[0] + 0.0f, t0, t1;
#define CM_IO2 [p0] "+&v"(p[0]), [p1] "+&v"(p[1]), [a1] "+&v"(a1), [t0] "=&v"(t0), [t1] "=&v"(t1)
#define CM_IN2 [Y0] "v"(Y[0]), [Y1] "v"(Y[1]), [r0] "v"(r[0]), [r1] "v"(r[1]), [low] "v"(low)
    if (TENS && __builtin_expect(J >= 10, 1)) {
      int n = J / 10;
      J -= 10 * n;
      asm(CM_LOOP(CM_PAIR2 CM_PAIR2 CM_PAIR2 CM_PAIR2 CM_PAIR2) : CM_IO2, [n] "+&s"(n) : CM_IN2 : "scc");
      if (__builtin_expect(J == 0, 1)) return;
    }
    int n = J / (2 * PAIRS);
    if (n > 0) {
      if constexpr (PAIRS == 1) asm(CM_LOOP(CM_PAIR2) : CM_IO2, [n] "+&s"(n) : CM_IN2 : "scc");
      else asm(CM_LOOP(CM_PAIR2 CM_PAIR2) : CM_IO2, [n] "+&s"(n) : CM_IN2 : "scc");
    }
    if (PAIRS == 2 && (J & 2)) asm("s_nop 1\n\t" CM_PAIR2 "s_nop 1" : CM_IO2 : CM_IN2);
    if (TENS ? __builtin_expect(J & 1, 0) : J & 1) {
      asm("s_nop 1\n\t" CM_SWEEP2("p0", "p1", "t0", "t1") "s_nop 1" : CM_IO2 : CM_IN2);
      p[0] = t0; p[1] = t1;
    }
#undef CM_IO2
#undef CM_IN2
  } else {
    float t0;
#define CM_IO1 [p0] "+&v"(p[0]), [t0] "=&v"(t0)
#define CM_IN1 [Y0] "v"(Y[0]), [r0] "v"(r[0]), [low] "v"(low)
    if (TENS && __builtin_expect(J >= 10, 1)) {
      int n = J / 10;
      J -= 10 * n;
      asm(CM_LOOP(CM_PAIR1 CM_PAIR1 CM_PAIR1 CM_PAIR1 CM_PAIR1) : CM_IO1, [n] "+&s"(n) : CM_IN1 : "scc");
      if (__builtin_expect(J == 0, 1)) return;
    }
    int n = J / (2 * PAIRS);
    if (n > 0) {
      if constexpr (PAIRS == 1) asm(CM_LOOP(CM_PAIR1) : CM_IO1, [n] "+&s"(n) : CM_IN1 : "scc");
      else asm(CM_LOOP(CM_PAIR1 CM_PAIR1) : CM_IO1, [n] "+&s"(n) : CM_IN1 : "scc");
    }
    if (PAIRS == 2 && (J & 2)) asm(CM_PAIR1 "s_nop 1" : CM_IO1 : CM_IN1);
    if (TENS ? __builtin_expect(J & 1, 0) : J & 1) {
      asm(CM_SWEEP1("p0", "t0") "s_nop 1" : CM_IO1 : CM_IN1);
      p[0] = t0;
    }
#undef CM_IO1
#undef CM_IN1
  }
}

// J is wave-uniform: the count goes to a scalar register.  U (1, 2 or 4) is
// the unroll of the sweep loop, a launch knob of the autotuner: sweeps come in
// pairs (U = 2) or two pairs (U = 4) per trip, so the two iterates alternate
// between register sets; U = 1 copies the iterate back each sweep.  TENS (U = 4,
// the fixed sweeps of a slow pass, 20 in the reference method) first takes ten
// per trip: a taken branch keeps a lone wave waiting for about 26 cycles, as long
// as five instructions.  Every U performs the same sweeps in the same order, so
// results are identical.
template <int U = 2, bool TENS = false, int N, class K>
__device__ __forceinline__ void jacobi_sweeps(Lay<N> &L, const float (&Y)[N], const K &k, float (&p)[N],
                                              int J) {
  static_assert(U == 1 || U == 2 || U == 4, "unroll 1, 2 or 4");
  J = __builtin_amdgcn_readfirstlane(J);
  float r[N];
  if constexpr (U != 1) {
    UNROLL for (int j = 0; j < N; ++j) r[j] = k.rsm[j];
  }
  if constexpr (N == 4 && U != 1) {
    sweeps_asm<U / 2, TENS>(Y, r, k.low, p, J);
  } else {
    for (;;) {
      const int c = J < Lay<N>::kReach ? J : Lay<N>::kReach;
      if constexpr (U != 1) {
        sweeps_spread<U / 2, TENS>(Y, r, k.low, p, c);
      } else {
        float q[N];
        for (int i = 0; i < c; ++i) {
          jacobi_sweep(L, Y, k, p, q);
          UNROLL for (int j = 0; j < N; ++j) p[j] = q[j];
        }
      }
      J -= c;
      if (__builtin_expect(J <= 0, 1)) break;
      L.share(p);
    }
  }
}

// Residual Y - A p of the kernel convention, per lane, and its squared 2-norm
// with the fixed tree.
template <int N, class K>
__device__ __forceinline__ void resid_vec(Lay<N> &L, const float (&Y)[N], const K &k, const float (&p)[N],
                                          float (&r)[N]) {
  float left, right;
  L.nbrs(p[N - 1], p[0], left, right);
  UNROLL for (int j = 0; j < N; ++j) {
    const float pl = j == 0 ? left : p[j - 1];
    const float pr = j == N - 1 ? right : p[j + 1];
    r[j] = Y[j] - (coupling<N>(j, k.low, pl, pr) + k.mf[j] * p[j]);
  }
}
template <int N, class K>
__device__ __forceinline__ float resid2(Lay<N> &L, const float (&Y)[N], const K &k, const float (&p)[N]) {
  float r[N];
  resid_vec(L, Y, k, p, r);
  UNROLL for (int j = 0; j < N; ++j) r[j] = r[j] * r[j];
  return L.sum(r);
}
// Squared residual of p and, from the same couplings, the next sweep's iterate q
// (spread layouts: both owned sections only; take() picks one for all lanes).
template <int N, class K>
__device__ __forceinline__ float resid2_sweep(Lay<N> &L, const float (&Y)[N], const K &k, const float (&p)[N],
                                              float (&q)[N], typename Lay<N>::Half &h) {
  float left, right, r[N];
  L.nbrs(p[N - 1], p[0], left, right);
  UNROLL for (int j = 0; j < N; ++j) {
    const float pl = j == 0 ? left : p[j - 1];
    const float pr = j == N - 1 ? right : p[j + 1];
    const float c = coupling<N>(j, k.low, pl, pr);
    r[j] = Y[j] - (c + k.mf[j] * p[j]);
    r[j] = r[j] * r[j];
    q[j] = (Y[j] - c) * k.rsm[j];
  }
  if constexpr (N == 4) {
    return L.sum(r);
  } else {
    float v[1] = {L.lane_sum(r)};
    L.put(p, 0);
    L.put(q, 1);
    L.template put_parts<1, false>(v);
    h = L.meet();
    L.template get_totals<1, false>(h, v);
    return v[0];
  }
}
template <int N>
__device__ __forceinline__ void take(Lay<N> &L, const typename Lay<N>::Half &h, int which, float (&p)[N], const float (&x)[N]) {
  if constexpr (N == 4) {
    UNROLL for (int j = 0; j < N; ++j) p[j] = x[j];
  } else {
    L.get(h, which, p);
  }
}

template <bool TOL, int N>
__device__ __forceinline__ void load_consts(const BmLaunch &a, const cm_bm_item &it, const Lay<N> &L,
                                            ItemConstN<N> &k) {
  const int base = L.base();
  float mm[N];
  ld_slots<N>(a.sec + CM_SEC_MASS * CM_SECTIONS + base, mm);
  ld_slots<N>(a.sec + CM_SEC_RSM * CM_SECTIONS + base, k.rsm);
  ld_slots<N>(a.sec + CM_SEC_R * CM_SECTIONS + base, k.R);
  ld_slots<N>(a.sec + CM_SEC_S * CM_SECTIONS + base, k.S);
  ld_slots<N>(a.sec + CM_SEC_Q * CM_SECTIONS + base, k.Q);
  ld_slots<N>(a.sec + CM_SEC_SOHC * CM_SECTIONS + base, k.Sohc);
  ld_slots<N>(a.sec + CM_SEC_STM * CM_SECTIONS + base, k.Stm);
  ld_slots<N>(a.sec + CM_SEC_RTM * CM_SECTIONS + base, k.Rtm);
  ld_slots<N>(a.gamma + (int64_t)it.set * CM_SECTIONS + base, k.gam);
  UNROLL for (int j = 0; j < N; ++j) k.rmass[j] = 1.0f / mm[j];
  if (TOL) {
    ld_slots<N>(a.sec + CM_SEC_M * CM_SECTIONS + base, k.mf);
  } else {
    UNROLL for (int j = 0; j < N; ++j) k.mf[j] = 0.0f;
  }
  k.low = L.low();
}

template <bool TOL, int N>
__device__ __forceinline__ void item_setup(const BmLaunch &a, const cm_bm_item &it, const Lay<N> &L,
                                           ItemConstN<N> &k, ItemScal &c, ItemStateN<N> &s) {
  const cm_bm_scalars &sc = a.sc;
  load_consts<TOL>(a, it, L, k);

  c.w_ohc = sc.w_ohc; c.alpha_r = sc.alpha_r; c.Ts = sc.Ts;
  c.al = sc.alpha_l; c.Gme = sc.Gme; c.a1 = sc.a1;
  c.eta1 = sc.eta1; c.eta2 = sc.eta2;
  c.dt_min = sc.dt_min; c.dt_max = sc.dt_max; c.tso = sc.time_step_out;
  c.mtt = it.tol; c.mmspt = it.m1tol;
  c.al_over_as = sc.alpha_l / sc.alpha_s;
  c.dxdx = sc.delta_x * sc.delta_x;
  c.dxa0 = sc.delta_x * sc.a0;
  c.neg_a2 = -sc.a2; c.neg_as = -sc.alpha_s;
  c.span = (float)(it.mesi - it.mosi);
  c.inv_sigma_ow = 1.0 / (double)sc.sigma_ow;

  UNROLL for (int j = 0; j < N; ++j) {
    s.A.d[j] = 0; s.A.v[j] = 0; s.A.a[j] = 0; s.A.psi[j] = 0; s.A.psid[j] = 0; s.A.xis[j] = 0; s.A.xi[j] = 0;
    s.Ptm[j] = 0; s.p[j] = 0;
  }
  s.A.ow_d = 0; s.A.ow_v = 0; s.A.ow_a = 0;
  s.B = s.A;
  s.dt = sc.time_step;
  s.t = 0.0f;
  s.in_s = it.start;
  s.sx0 = in_at(a, s.in_s);
  s.sx1 = in_at(a, (int64_t)s.in_s + 1);
  s.c_fail = 0.f; s.c_dt = 0.f; s.c_steps = 0.f; s.c_passes = 0.f;
  s.n_steps = 0; s.n_passes = 0; s.n_sweeps = 0;
  s.fb = 0;
  s.ctb = 0.f; s.clb = 0.f; s.cjb = 0.f;
}

// Predictor (Euler) update of side n from the committed side o, :13770-13820.
// The trapezoids keep their own halving, ((a + b) 0.5) dt: folding it into
// 0.5 dt would save an instruction each and rounds alike except for sums below
// 2^-125, but the tails of decaying signals reach those.
template <int N>
__device__ __forceinline__ void predict(const HalfN<N> &o, HalfN<N> &n, float dt) {
  UNROLL for (int j = 0; j < N; ++j) {
    n.xi[j] = o.xis[j] * dt + o.xi[j];
    n.v[j] = o.a[j] * dt + o.v[j];
    n.d[j] = ((o.v[j] + n.v[j]) * 0.5f) * dt + o.d[j];
    n.psi[j] = o.psid[j] * dt + o.psi[j];
  }
  n.ow_d = o.ow_v * dt + o.ow_d;
  n.ow_v = o.ow_a * dt + o.ow_v;
}
// Corrector (trapezoid) update.
template <int N>
__device__ __forceinline__ void correct(const HalfN<N> &o, HalfN<N> &n, float dt) {
  UNROLL for (int j = 0; j < N; ++j) {
    n.v[j] = ((o.a[j] + n.a[j]) * 0.5f) * dt + o.v[j];
    n.d[j] = ((o.v[j] + n.v[j]) * 0.5f) * dt + o.d[j];
    n.xi[j] = ((o.xis[j] + n.xis[j]) * 0.5f) * dt + o.xi[j];
    n.psi[j] = ((o.psid[j] + n.psid[j]) * 0.5f) * dt + o.psi[j];
  }
  n.ow_d = ((o.ow_v + n.ow_v) * 0.5f) * dt + o.ow_d;
  n.ow_v = ((o.ow_a + n.ow_a) * 0.5f) * dt + o.ow_v;
}

// Forcing s(t), the same for every pass of a step.
template <int N>
__device__ __forceinline__ float forcing(const ItemScal &c, const ItemStateN<N> &s) {
  const float delta = s.t / c.Ts;
  return s.sx1 * delta + s.sx0 * (1.0f - delta);
}

// Terms of a pass that its end (pass_finish) uses again.
template <int N>
struct PassTerms {
  float eod[N];    // eta1 (xi - d)
  float wpsi[N];   // w_ohc psi
  float G[N];
};

// TM/OHC block (AUX: passes < 2, :13839-13898), G (:13905-13909) and the
// right-hand side with its boundaries (:13925-13954).
template <bool AUX, int N, class K>
__device__ __forceinline__ void pass_rhs(const K &k, const ItemScal &c, HalfN<N> &n, float (&Ptm)[N], float sf,
                                         const Lay<N> &L, PassTerms<N> &T, float (&Y)[N]) {
  UNROLL for (int j = 0; j < N; ++j) T.wpsi[j] = c.w_ohc * n.psi[j];
  float od[N];
  UNROLL for (int j = 0; j < N; ++j) {
    od[j] = n.xi[j] - n.d[j];
    T.eod[j] = c.eta1 * od[j];
  }
  if constexpr (AUX) {
    float x[N], th[N];
    UNROLL for (int j = 0; j < N; ++j) x[j] = c.al_over_as * n.psi[j];
    tanh_slots<N>(x, th);
    UNROLL for (int j = 0; j < N; ++j) {
      const float ohc_p = (k.gam[j] * k.Sohc[j]) * od[j];
      const float dL = c.neg_as * th[j];
      const float aux = c.al * (th[j] * th[j] - 1.0f);
      float m = (c.eta2 * n.v[j] + T.eod[j]) - T.wpsi[j];
      m = k.Stm[j] * dL + (m * k.Rtm[j]) * aux;
      const float sxi = k.Stm[j] * n.xi[j];
      m = (sxi + ohc_p) - k.gam[j] * m;
      float den = (k.gam[j] * aux) * c.eta2 - 1.0f;
      den = k.Rtm[j] * den;
      n.xis[j] = m / den;
      Ptm[j] = k.Rtm[j] * n.xis[j] + sxi;
    }
  }
  UNROLL for (int j = 0; j < N; ++j) {
    float g = n.v[j] * n.v[j];
    g = k.R[j] * (c.alpha_r * g + 1.0f);
    g = g * n.v[j] + k.S[j] * n.d[j];
    T.G[j] = -g - Ptm[j];
    Y[j] = (c.dxdx * T.G[j]) * k.Q[j];
  }
  const float Y0 = c.dxa0 * (((c.neg_a2 * n.ow_v) - c.a1 * n.ow_d) + c.Gme * sf);
  Y[0] = L.sec0() ? Y0 : Y[0];
  Y[N - 1] = L.last() ? 0.0f : Y[N - 1];
}

// Jacobi until |Y - A p|_2 <= tol |Y|_2 (checked every check_every sweeps,
// capped at max_sweeps); returns the sweeps done.  rr is |Y - A p|_2^2 of the
// incoming p (the guess selection has already computed it).  A check shares
// its couplings with the sweep that follows when it fails, and that sweep's
// other instructions fill the reduction's waits.
template <int U = 2, int N, class K>
__device__ __forceinline__ int jacobi_tol(Lay<N> &L, const cm_bm_scalars &sc, const K &k,
                                          const float (&Y)[N], float yy, float (&p)[N], float rr) {
  const float tau2 = sc.tol_rel * sc.tol_rel;
  const float lim = tau2 * yy;
  int J = 0;
  if (rr <= lim || J >= sc.max_sweeps) {
    L.share(p);
    return J;
  }
  int kk = sc.check_every < sc.max_sweeps ? sc.check_every : sc.max_sweeps;
  jacobi_sweeps<U>(L, Y, k, p, kk);
  for (;;) {
    J += kk;
    float q[N];
    typename Lay<N>::Half h{};
    rr = resid2_sweep(L, Y, k, p, q, h);
    if (rr <= lim || J >= sc.max_sweeps) {
      take(L, h, 0, p, p);
      return J;
    }
    kk = sc.check_every < sc.max_sweeps - J ? sc.check_every : sc.max_sweeps - J;
    take(L, h, 1, p, q);
    jacobi_sweeps<U>(L, Y, k, p, kk - 1);
  }
}

// Acceleration, oval-window acceleration and psi derivative, :13989-14013.
// The oval window's division by the constant sigma_ow is a product with its
// reciprocal in FP64: a quotient of two floats is at least 2^-49 (relative)
// from the midpoint of two floats, the product within 2^-52 of the quotient,
// so it rounds to the same float (below the normal range unless sigma_ow is an
// even integer: only then can a quotient lie on a midpoint there).
template <int N, class K>
__device__ __forceinline__ void pass_finish(Lay<N> &L, const K &k, const ItemScal &c, HalfN<N> &n,
                                            const float (&p)[N], const PassTerms<N> &T, float sf) {
  UNROLL for (int j = 0; j < N; ++j) n.a[j] = (p[j] + T.G[j]) * k.rmass[j];
  {
    const float p0 = L.sec0_value(p[0]);
    const float NN1 = c.neg_a2 * n.ow_v;
    const float NN2 = c.Gme * sf + p0;
    const float x = (NN1 + NN2) - c.a1 * n.ow_d;
    n.ow_a = (float)((double)x * c.inv_sigma_ow);
  }
  UNROLL for (int j = 0; j < N; ++j)
    n.psid[j] = (T.eod[j] + c.eta2 * (n.xis[j] - n.v[j])) - T.wpsi[j];
}

// Step control (:14021-14088); Q1 lane-0 semantics.  Returns whether the step
// needs another pass.  L = (emax dt) / esum only meets 6 and 0.5, so it is not
// divided out: the float quotient is above 6 where the exact one is above the
// midpoint 6 + 2^-22 (a tie rounds to 6), and below 0.5 where the exact one is
// below 0.5 - 2^-26; esum times either bound is exact in FP64.
// LONE: without branches, which cost a wave that has a SIMD to itself more than
// the operations they avoid.
template <bool LONE>
__device__ __forceinline__ bool step_control(const cm_bm_scalars &sc, const ItemScal &c, float &dt, float emax,
                                             float esum, float fsum) {
  if (sc.decision_mode == 1) { emax = 0.f; esum = 0.f; fsum = 0.f; }
  if constexpr (LONE) {
    const double e = esum, q = emax * dt;
    const bool moved = esum > c.mmspt;
    const bool above = moved & (q > e * (6.0 + 0x1p-22));       // L > 6
    const bool below = !moved | (q < e * (0.5 - 0x1p-26));      // L < 0.5
    const bool again = !above & ((fsum > 0.0f) | !below);
    const float half = dt * 0.5f, twice = dt * 2.0f;
    const float less = half < c.dt_min ? c.dt_min : half;
    const float more = twice > c.dt_max ? c.dt_max : twice;
    const float other = above ? less : more;
    dt = again ? dt : other;
    return again;
  }
  bool above = false, below = true;   // L > 6, L < 0.5
  if (esum > c.mmspt) {
    const double e = esum, q = emax * dt;
    above = q > e * (6.0 + 0x1p-22);
    below = q < e * (0.5 - 0x1p-26);
  }
  if (above) {
    dt = dt * 0.5f;
    if (dt < c.dt_min) dt = c.dt_min;
    return false;
  }
  if (fsum > 0.0f || !below) return true;
  dt = dt * 2.0f;
  if (dt > c.dt_max) dt = c.dt_max;
  return false;
}
// Its terms: the changes of acceleration and velocity since the last pass.
template <int N>
__device__ __forceinline__ void control_terms(const ItemScal &c, float dt, const float (&v)[N], const float (&a)[N],
                                              const float (&vref)[N], const float (&aref)[N], float (&ex)[N],
                                              float (&ey)[N], float (&ez)[N]) {
  UNROLL for (int j = 0; j < N; ++j) {
    ex[j] = __builtin_fabsf(aref[j] - a[j]);
    ey[j] = __builtin_fabsf(v[j] - vref[j]);
    ez[j] = ey[j] - fmaxf(c.mtt, v[j] * dt);
  }
}
template <bool LONE = false, int N>
__device__ __forceinline__ bool pass_control(Lay<N> &L, const cm_bm_scalars &sc, const ItemScal &c, float &dt,
                                             const HalfN<N> &n, const float (&vref)[N], const float (&aref)[N]) {
  float ex[N], ey[N], ez[N], emax, esum, fsum;
  control_terms(c, dt, n.v, n.a, vref, aref, ex, ey, ez);
  L.reduce3(ex, ey, ez, emax, esum, fsum);
  return step_control<LONE>(sc, c, dt, emax, esum, fsum);
}

// Commit of a step whose passes left side n: counters, sample advance with
// output row (:14130-14203) and local time (:14212-14230).
template <int N>
__device__ __forceinline__ void step_commit(const BmLaunch &a, const cm_bm_item &it, const ItemScal &c,
                                            ItemStateN<N> &s, const HalfN<N> &n, int out_loop, const Lay<N> &L) {
  s.c_steps += 1.0f;
  s.c_dt += s.dt;
  s.c_passes += (float)out_loop;
  s.n_steps++;
  s.n_passes += out_loop;
  if (s.t > c.tso) {
    s.t -= c.tso;
    s.sx0 = s.sx1;
    s.sx1 = in_at(a, (int64_t)s.in_s + 2);
    if (s.in_s + 1 >= it.mosi) {
      const float div_times = s.c_dt / s.c_steps;
      const float div_j = s.c_passes / s.c_steps;
      if (s.in_s >= it.write_start && s.in_s >= 0 && s.in_s < a.rows) {   // rows outside the buffer are dropped
        if (a.speeds) {
          // (one float4 per lane when N = 4, written out in full: the register
          // allocation of the learned kernel is tight enough that the generic
          // store costs it a spill)
          if constexpr (N == 4)
            *reinterpret_cast<float4 *>(a.speeds + (int64_t)s.in_s * CM_SECTIONS + 4 * L.lane) =
                make_float4(n.v[0], n.v[1], n.v[2], n.v[3]);
          else if (L.own())
            st_slots<N>(a.speeds + (int64_t)s.in_s * CM_SECTIONS + L.base(), n.v);
        }
        if (L.sec0()) {
          if (a.failed_nodes) a.failed_nodes[s.in_s] = (int32_t)s.c_fail;
          if (a.conv_time) a.conv_time[s.in_s] = div_times;
          if (a.conv_jacobi) a.conv_jacobi[s.in_s] = div_j;
          if (a.conv_loops) a.conv_loops[s.in_s] = s.c_steps;
        }
      }
      if (s.c_fail > 0.f) s.fb += 1;
      s.ctb += div_times / c.span;
      s.cjb += div_j / c.span;
      s.clb += s.c_steps / c.span;
    }
    s.c_fail = 0.f; s.c_dt = 0.f; s.c_steps = 0.f; s.c_passes = 0.f;
    s.in_s++;
  }
  s.t += s.dt;
}

template <int N>
__device__ __forceinline__ void item_final(const BmLaunch &a, const ItemStateN<N> &s, int item_index,
                                           const Lay<N> &L) {
  if (L.sec0()) {
    if (a.failed_blocks) a.failed_blocks[item_index] = s.fb;
    if (a.conv_time_blocks) a.conv_time_blocks[item_index] = s.ctb;
    if (a.conv_loops_blocks) a.conv_loops_blocks[item_index] = s.clb;
    if (a.conv_jacobi_blocks) a.conv_jacobi_blocks[item_index] = s.cjb;
    if (a.stats) {
      a.stats[item_index].steps = s.n_steps;
      a.stats[item_index].passes = s.n_passes;
      a.stats[item_index].sweeps = s.n_sweeps;
    }
  }
}

// Extrapolated predictor-pass guess: p <- p + (dt/dt_prev)(p - p_prev) when
// that lowers the residual (ties keep the previous pressure).  The previous
// step's pressure and dt_prev live in LDS (pold[lane], first N floats, and
// pold[64].x, one copy per wave).  Returns the squared residual of the plain
// guess; rre gets the extrapolation's and yy |Y|^2, and p holds the
// extrapolation on return when keep_lin, else the choice.
template <int N, class K>
__device__ __forceinline__ float extrapolate_guess(Lay<N> &L, const K &k, const float (&Y)[N], float dt,
                                                   float4 *pold, float (&p)[N], float &rre, float &yy,
                                                   bool keep_lin) {
  float *dt_prev = reinterpret_cast<float *>(pold + 64);
  float *mine = reinterpret_cast<float *>(pold + L.lane);
  const float rho = dt / *dt_prev;
  float po[N], r0[N], r1[N];
  ld_slots<N>(mine, po);
  st_slots<N>(mine, p);
  resid_vec(L, Y, k, p, r0);
  UNROLL for (int j = 0; j < N; ++j) p[j] = p[j] + rho * (p[j] - po[j]);
  resid_vec(L, Y, k, p, r1);
  float rr0;
  L.sum_sq3(r0, r1, Y, rr0, rre, yy);
  if (!keep_lin && !(rre < rr0)) ld_slots<N>(mine, p);
  if (L.lane == 0) *dt_prev = dt;
  return rr0;
}

// The pressure solve of a corrector pass: fixed sweeps, or to the tolerance
// from the resident pressure.
template <bool TOL, int U, bool SLOW = true, int N, class K>
__device__ __forceinline__ int solve_pass(Lay<N> &L, const cm_bm_scalars &sc, const K &k, const float (&Y)[N],
                                          float (&p)[N], int J_fixed) {
  if constexpr (TOL) {
    float r[N], yy, rr;
    resid_vec(L, Y, k, p, r);
    L.sum_sq2(r, Y, rr, yy);
    return jacobi_tol<U>(L, sc, k, Y, yy, p, rr);
  } else {
    jacobi_sweeps<U, SLOW && U == 4>(L, Y, k, p, J_fixed);
    L.share(p);
    return J_fixed;
  }
}

// The solve, end and control of a corrector pass.  The fixed sweeps of a spread
// block leave the owned pressures; these and the control's totals pass in one
// exchange.
template <bool TOL, int U, bool SLOW, int N>
__device__ __forceinline__ bool correct_end(const BmLaunch &a, Lay<N> &L, const ItemConstN<N> &k, const ItemScal &c,
                                            ItemStateN<N> &s, HalfN<N> &n, const PassTerms<N> &T, const float (&Y)[N],
                                            float sf, const float (&vref)[N], const float (&aref)[N], int J_fixed) {
  if constexpr (N == 4 || TOL) {
    s.n_sweeps += solve_pass<TOL, U, SLOW>(L, a.sc, k, Y, s.p, J_fixed);
    pass_finish(L, k, c, n, s.p, T, sf);
    return pass_control<!TOL && U == 4>(L, a.sc, c, s.dt, n, vref, aref);
  } else {
    jacobi_sweeps<U, SLOW && U == 4>(L, Y, k, s.p, J_fixed);
    s.n_sweeps += J_fixed;
    float acc[N], ex[N], ey[N], ez[N], emax, esum, fsum;
    UNROLL for (int j = 0; j < N; ++j) acc[j] = (s.p[j] + T.G[j]) * k.rmass[j];
    control_terms(c, s.dt, n.v, acc, vref, aref, ex, ey, ez);
    L.reduce3_share(ex, ey, ez, s.p, emax, esum, fsum);
    pass_finish(L, k, c, n, s.p, T, sf);
    return step_control<U == 4>(a.sc, c, s.dt, emax, esum, fsum);
  }
}

// One integration step, include/cochlea.cuh:13760-14230: committed side o to
// side n.  The predictor pass, the first corrector pass (which repeats the
// TM/OHC block) and the further ones are written out one after another, so
// that none carries the others' branches and selections.
// Bound: instruction issue.  One wave per SIMD issues an instruction every 5 to
// 6 cycles whatever it depends on; three reach about 3 cycles (FP32) and 4.2
// (DPP, FP64).  So the step is written for few instructions: per block-step of
// the reference method 1589 VALU and 122 SALU, where one pass loop for all
// kinds of pass, a branch per tanh, divided-out step control and copied states
// took 1793 and 246 (600 tones of 200 ms, 20-90 dB).  5 blocks: 141 -> 111 ms (85
// over four waves each, with ten sweeps a trip); 610 blocks, extrapolated guess:
// 183 -> 143 ms; 6000 blocks: 408 -> 380 ms.
template <int N, bool TOL, int WS, int U>
__device__ __forceinline__ void step(const BmLaunch &a, const cm_bm_item &it, Lay<N> &L, const ItemConstN<N> &k,
                                     const ItemScal &c, ItemStateN<N> &s, const HalfN<N> &o, HalfN<N> &n,
                                     float4 *pold) {
  const float sf = forcing(c, s);
  PassTerms<N> T;
  float Y[N];
  int J;
  predict(o, n, s.dt);
  pass_rhs<true>(k, c, n, s.Ptm, sf, L, T, Y);
  if constexpr (TOL && WS == 1) {
    float rre, yy;
    const float rr0 = extrapolate_guess(L, k, Y, s.dt, pold, s.p, rre, yy, false);
    J = jacobi_tol<U>(L, a.sc, k, Y, yy, s.p, rre < rr0 ? rre : rr0);   // residual of the guess kept
  } else {
    J = solve_pass<TOL, U>(L, a.sc, k, Y, s.p, a.sc.j_slow);
  }
  s.n_sweeps += J;
  pass_finish(L, k, c, n, s.p, T, sf);
  int passes = 1;
  bool another = passes < a.sc.max_passes;
  if (another) {
    float vref[N], aref[N];
    UNROLL for (int j = 0; j < N; ++j) { vref[j] = n.v[j]; aref[j] = n.a[j]; }
    correct(o, n, s.dt);
    pass_rhs<true>(k, c, n, s.Ptm, sf, L, T, Y);
    another = correct_end<TOL, U, true>(a, L, k, c, s, n, T, Y, sf, vref, aref, a.sc.j_slow);
    passes = 2;
    if (passes >= a.sc.max_passes) { another = false; s.c_fail = 1.f; }
    while (another) {
      UNROLL for (int j = 0; j < N; ++j) { vref[j] = n.v[j]; aref[j] = n.a[j]; }
      correct(o, n, s.dt);
      pass_rhs<false>(k, c, n, s.Ptm, sf, L, T, Y);
      another = correct_end<TOL, U, false>(a, L, k, c, s, n, T, Y, sf, vref, aref, a.sc.j_fast);
      ++passes;
      if (passes >= a.sc.max_passes) { another = false; s.c_fail = 1.f; }
    }
  } else {
    s.c_fail = 1.f;
  }
  step_commit(a, it, c, s, n, passes, L);
}

// One time block, include/cochlea.cuh:13620-14232.  TOL selects the
// sweep-to-tolerance Jacobi; otherwise the reference's fixed 20/2 sweeps.
// WS = 1 adds the extrapolated predictor-pass guess (tolerance mode only).
// U is the Jacobi sweep unroll, N the sections per lane.
template <int N, bool TOL, int WS, int U>
__device__ void run_item(const BmLaunch &a, int item_index, Lay<N> &L, float4 *pold) {
  const cm_bm_item it = a.items[item_index];
  ItemConstN<N> k;
  ItemScal c;
  ItemStateN<N> s;
  item_setup<TOL>(a, it, L, k, c, s);
  if (WS == 1) {
    pold[L.lane] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (L.lane == 0) reinterpret_cast<float *>(pold + 64)[0] = s.dt;
  }
  // two steps per trip: the sides change roles without a copy
  while (s.in_s < it.mesi) {
    step<N, TOL, WS, U>(a, it, L, k, c, s, s.A, s.B, pold);
    if (s.in_s >= it.mesi) break;
    step<N, TOL, WS, U>(a, it, L, k, c, s, s.B, s.A, pold);
  }
  item_final(a, s, item_index, L);
}

}  // namespace cm

#endif
