// What the list kernels (Viterbi, Forward, Backward: one target per wave or
// workgroup, taken from a list through its work queue) share.
#pragma once
#include "p7g_devfn.h"

// Where a list kernel finds its profile tables (template argument TM):
//   TM_LDS   the whole table in LDS, transitions pinned in registers
//   TM_PIN   the table in global memory (L2-resident), transitions pinned
//   TM_TLDS  transitions in LDS, read per row; emission rows from global memory
//   TM_GLOB  the table in global memory, transitions read per row
// Large models take the last two: B positions of every transition pinned in
// registers would not fit the register file, and the whole table not in LDS.
// The per-row reads go through an offset the compiler cannot see through, so
// that they are not hoisted out of the row loop into registers again.
enum { TM_LDS = 0, TM_PIN = 1, TM_TLDS = 2, TM_GLOB = 3 };

__device__ __forceinline__ int opaque_zero()
{
  int v = 0;
  asm volatile("" : "+v"(v));
  return v;
}

// The residues of a row loop, 64 rows at a time, as table offsets (residue *
// stride): while the loop's step s (0, 1, ...) runs, ahead(s & 63) is the offset
// of the step after it, so that its emission row can be loaded a row early; lane
// l of `cur` holds that of step s0 + l + 1. One vector load per 64 rows and one
// v_readlane per row; taking the bytes out of a 16-byte chunk in scalar registers
// cost six branches a row, about 200 cycles of a wave that runs alone. Step s
// reads residue s (ascending), or residue L-1-s (descending); steps past the end
// read the byte behind the target, which is always readable, or residue 0.
template <bool DESC>
struct RowRes {
  const uint8_t *sq;
  int L, z, s0, stride, cur, far;
  __device__ __forceinline__ int byte(int s) const { return (int) sq[DESC ? max(L - 1 - s, 0) : min(s, L)]; }
  __device__ __forceinline__ int init(const uint8_t *q, int len, int lane, int str)
  {
    sq = q; L = len; z = lane; s0 = 0; stride = str;
    const int x0 = uni(byte(0));
    cur = byte(1 + z) * stride; far = byte(65 + z);
    return x0 * stride;                          // the first step's offset
  }
  __device__ __forceinline__ int ahead(int u) const { return __builtin_amdgcn_readlane(cur, u); }
  __device__ __forceinline__ void advance() { s0 += 64; cur = far * stride; far = byte(s0 + 65 + z); }
};
// x > lim for a wave-uniform x held in a scalar register, as the float compare
// (false for NaN) on its bit pattern; lim is positive. A scalar compare and
// branch, where the vector compare took the branch through VCC.
__device__ __forceinline__ bool gt_bits(int xbits, int limbits)
{ return __builtin_expect((unsigned) (xbits - limbits - 1) <= 0x7f800000u - (unsigned) limbits - 1u, 0); }
#define BITS_1E4  0x461c4000      // 1.0e4f
#define BITS_1E16 0x5a0e1bca      // 1.0e16f
#define BITS_ONE  0x3f800000      // 1.0f

// Adds the logs of a block's row scales (lane u: row u's, 1 where the row was not
// rescaled) to totscale in row order. Once per 64 rows: with its logarithm in
// the row loop a parser held some twenty registers less for its rows (Backward's
// B = 5..7 spilled up to 23 of them, and B = 2 had five waves per SIMD for six).
__device__ __forceinline__ void add_scales(float &totscale, float s)
{
  unsigned long long m = __ballot(s > 1.0f);
  if (__builtin_expect(m != 0ull, 0)) {
    const double lg = log((double) s);
    const int lo = (int) __double2loint(lg), hi = (int) __double2hiint(lg);
    do {
      const int l = (int) __ffsll((long long) m) - 1;
      totscale = (float) ((double) totscale + __hiloint2double(__builtin_amdgcn_readlane(hi, l), __builtin_amdgcn_readlane(lo, l)));
      m &= m - 1;
    } while (m);
  }
}

// A workgroup barrier that orders LDS alone: global loads in flight (the next
// row's odds) stay in flight, where __syncthreads would wait for them.
__device__ __forceinline__ void lds_barrier()
{
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// How many waves of a list kernel's workgroup take targets: four, one per SIMD,
// while the list has no more than four targets per workgroup, else all. A wave
// alone on its SIMD issues an instruction in about 5 cycles, one of two in 8; the
// workgroups of a short list would fill a few compute units with two waves per
// SIMD and leave the others idle. Against all eight with a grid for eight, 200
// targets of 350: Backward at M = 86 | 400 | 700 284 | 413 | 533 -> 243 | 329 |
// 404 us; 1000 at M = 400: Viterbi 228 -> 192, Backward 437 -> 368 us. From about
// 4200 targets on there is no difference.
#define LIST_SIMDS 4
__device__ __forceinline__ int list_waves(int64_t count)
{
  const int w = (int) (blockDim.x >> 6);
  return (w > LIST_SIMDS && count <= (int64_t) LIST_SIMDS * gridDim.x) ? LIST_SIMDS : w;
}
// Their grid: enough workgroups for one wave per SIMD, none that cannot be resident.
static inline unsigned list_grid(const void *kernel, int64_t maxn, size_t lds_bytes, int wpb)
{
  const int64_t per = wpb < LIST_SIMDS ? wpb : LIST_SIMDS;
  return grid_for_waves_blk(kernel, (maxn + per - 1) / per * wpb, lds_bytes, wpb);
}

// Workgroup sizes of the list kernels: 8 waves, or 4 (one per SIMD, so that a
// wave may hold 512 registers with the accumulation registers) where the
// per-lane state of large models does not fit in 256.
#define VIT_THREADS(ND) ((ND) >= 40 ? 256 : 512)
#define FWD_THREADS(B)  ((B) >= 64 ? 256 : 512)
#define BCK_THREADS(B)  ((B) >= 28 ? 256 : 512)

// a*b + c*d in one rounding order, whatever the compiler would contract in the
// place it stands: the product of SW ? the first : the second pair is rounded,
// the other one fused onto it.
template <bool SW>
__device__ __forceinline__ float fma2(float a, float b, float c, float d)
{
#pragma clang fp contract(off)
  return SW ? __builtin_fmaf(c, d, a * b) : __builtin_fmaf(a, b, c * d);
}

// x = x * a + t, fused, in x's own register: left to itself the compiler adds onto
// t's and copies the sum back at the end of the row. What is left of t keeps it
// from that.
__device__ __forceinline__ void fma_onto(float &x, float a, float t)
{
  x = __builtin_fmaf(x, a, t);
  asm("" : "+v"(x) : "v"(t));
}

// v where the lane's bit of a constant mask is set, else w: one v_cndmask. The
// carry of a lane's 16-lane row is selected with these; left to itself the
// compiler branched over the lanes' rows inside the row loop.
__device__ __forceinline__ float lane_sel(float w, float v, unsigned long long mask)
{
  float r;
  asm("v_cndmask_b32_e64 %0, %1, %2, %3" : "=v"(r) : "v"(w), "v"(v), "s"(mask));
  return r;
}
#define LANES_ROW(r) (0xffffull << (16 * (r)))

// The D->D chain of a parser row as an affine scan: lane maps f(x) = P x + C
// composed over 16-lane rows with DPP, rows joined by readlane carries. The
// products P depend only on the profile's D->D odds: they are computed once
// per kernel (AffConst, with the same multiplications in the same order as a
// per-row computation would make), so a row costs the C recurrence alone.
struct AffConst {
  float w1, w2, w4, w8;      // window products the four row steps multiply by
  float prow;                // product over the row part the lane's window covers after the steps
  float pa, pb;              // wave-uniform row products used by the row carries
};

template <int B>
__device__ __forceinline__ void aff_fwd_setup(AffConst &k, const float (&a)[B])
{
  float P = 1.0f;
#pragma unroll
  for (int j = 0; j < B; j++) P *= a[j];
  k.w1 = P; P = P * dppf<ROW_SHR1>(1.0f, P);
  k.w2 = P; P = P * dppf<ROW_SHR2>(1.0f, P);
  k.w4 = P; P = P * dppf<ROW_SHR4>(1.0f, P);
  k.w8 = P; P = P * dppf<ROW_SHR8>(1.0f, P);
  k.prow = P; k.pa = readlanef(P, 31); k.pb = readlanef(P, 47);
}

template <int B>
__device__ __forceinline__ void aff_bck_setup(AffConst &k, const float (&a)[B])
{
  float P = 1.0f;
#pragma unroll
  for (int j = B-1; j >= 0; j--) P *= a[j];
  k.w1 = P; P = P * dppf<ROW_SHL1>(1.0f, P);
  k.w2 = P; P = P * dppf<ROW_SHL2>(1.0f, P);
  k.w4 = P; P = P * dppf<ROW_SHL4>(1.0f, P);
  k.w8 = P; P = P * dppf<ROW_SHL8>(1.0f, P);
  k.prow = P; k.pa = readlanef(P, 32); k.pb = readlanef(P, 16);
}

// C: the lane's map constant (carry-in 0); returns D at the end of lane z-1,
// resp. (towards smaller k) at the first position of lane z+1.
__device__ __forceinline__ float lane_carry_fwd(float C, const AffConst &k)
{
  C = C + k.w1 * dppz<ROW_SHR1>(C);
  C = C + k.w2 * dppz<ROW_SHR2>(C);
  C = C + k.w4 * dppz<ROW_SHR4>(C);
  C = C + k.w8 * dppz<ROW_SHR8>(C);
  {
    const float c1 = readlanef(C, 15);
    const float c2 = k.pa * c1 + readlanef(C, 31);
    const float c3 = k.pb * c2 + readlanef(C, 47);
    const float rc = lane_sel(lane_sel(lane_sel(0.0f, c1, LANES_ROW(1)), c2, LANES_ROW(2)), c3, LANES_ROW(3));
    C = C + k.prow * rc;
  }
  return dppz<WAVE_SHR1>(C);
}

__device__ __forceinline__ float lane_carry_bck(float C, const AffConst &k)
{
  C = C + k.w1 * dppz<ROW_SHL1>(C);
  C = C + k.w2 * dppz<ROW_SHL2>(C);
  C = C + k.w4 * dppz<ROW_SHL4>(C);
  C = C + k.w8 * dppz<ROW_SHL8>(C);
  {
    const float c2 = readlanef(C, 48);
    const float c1 = k.pa * c2 + readlanef(C, 32);
    const float c0 = k.pb * c1 + readlanef(C, 16);
    const float rc = lane_sel(lane_sel(lane_sel(0.0f, c2, LANES_ROW(2)), c1, LANES_ROW(1)), c0, LANES_ROW(0));
    C = C + k.prow * rc;
  }
  return dppz<WAVE_SHL1>(C);
}

template <int B>
__device__ __forceinline__ void affine_fwd_scan(float (&D)[B], const float (&a)[B], const AffConst &k)
{
  // D(j) = D0(j) + a(j) * D(j-1), carried across lanes in increasing k
  float C = D[0];
#pragma unroll
  for (int j = 1; j < B; j++) C = __builtin_fmaf(a[j], C, D[j]);
  float cur = lane_carry_fwd(C, k);
#pragma unroll
  for (int j = 0; j < B; j++) { cur = __builtin_fmaf(a[j], cur, D[j]); D[j] = cur; }
}

// a(j) gives the D->D odds of the lane's position j (read twice per call, so
// that large models need not hold them in registers through the scan).
template <int B, typename A>
__device__ __forceinline__ void affine_bck_scan(float (&D)[B], A a, const AffConst &k)
{
  // D(j) = c(j) + a(j) * D(j+1), carried across lanes in decreasing k
  float C = D[B-1];
#pragma unroll
  for (int j = B-2; j >= 0; j--) C = __builtin_fmaf(a(j), C, D[j]);
  float cur = lane_carry_bck(C, k);
#pragma unroll
  for (int j = B-1; j >= 0; j--) { cur = __builtin_fmaf(a(j), cur, D[j]); D[j] = cur; }
}

// The values of NT tables at a lane's B positions, read from memory where a row
// needs them (DESC: from the last position down), for models too large to hold
// or stage them: G positions at a time, the next group requested before this
// one is used. Bound by the latency of these loads: left to itself the compiler
// loads one position's values, waits and goes on. Decoding of 40 targets of
// M = 3500: Forward 18.9 ms, Backward 19.0 ms; position by position 70 and 120 ms.
template <int B, int NT, int G, bool DESC, typename F>
__device__ __forceinline__ void stream_tables(const float *const (&src)[NT], F f)
{
  constexpr int NG = (B + G - 1) / G;
  float v[2][NT][G];
  auto load = [&](int g) {
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
      for (int u = 0; u < G; u++)
        if (g * G + u < B) v[g & 1][t][u] = src[t][(DESC ? B - 1 - (g * G + u) : g * G + u) * 64];
  };
  load(0);
#pragma unroll
  for (int g = 0; g < NG; g++) {
    if (g + 1 < NG) load(g + 1);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < G; u++)
      if (g * G + u < B) {
        float x[NT];
#pragma unroll
        for (int t = 0; t < NT; t++) x[t] = v[g & 1][t][u];
        f(DESC ? B - 1 - (g * G + u) : g * G + u, x);
      }
  }
}

// Forward/Backward: the whole table in LDS up to B = 12 (150 KB); B = 14 reads
// the table from global memory with transitions pinned in registers;
// B = 16..48 keep the transitions in LDS (at most 160 KB) and read them per
// row; B = 64, 80 read everything from global memory per row.
#define FB_LDS_LIMIT (150 * 1024)
static inline int fb_mode(const DevProfile &p)
{
  if (p.fb_floats * 4 <= FB_LDS_LIMIT && p.fb_floats * 4 <= (size_t) lds_block_limit()) return TM_LDS;
  if (p.fb_B <= 14) return TM_PIN;
  if ((size_t) P7G_FB_NT * 64 * p.fb_B * 4 <= (size_t) lds_block_limit()) return TM_TLDS;
  return TM_GLOB;
}
static inline size_t fb_lds(const DevProfile &p, int tm)
{
  return (tm == TM_LDS) ? p.fb_floats * 4 : (tm == TM_TLDS) ? (size_t) P7G_FB_NT * 64 * p.fb_B * 4 : 0;
}
#define FB_CASES(X) \
  X(1, TM_LDS) X(2, TM_LDS) X(3, TM_LDS) X(4, TM_LDS) X(5, TM_LDS) X(6, TM_LDS) X(7, TM_LDS) X(8, TM_LDS) \
  X(10, TM_LDS) X(12, TM_LDS) X(14, TM_PIN) X(16, TM_TLDS) X(20, TM_TLDS) X(24, TM_TLDS) X(28, TM_TLDS) \
  X(32, TM_TLDS) X(40, TM_TLDS) X(48, TM_TLDS) X(64, TM_GLOB) X(80, TM_GLOB)
