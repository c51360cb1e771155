// Multidomain regions: region_trace_ensemble (HMMER/src/p7_domaindef.c:600-690)
// as p7_domaindef_ByPosteriorHeuristics runs it for a region that looks like
// more than one domain (:431-476), one workgroup per region:
//
//  1. p7_Forward over the region's residues with the profile in multihit
//     mode, length-configured to the whole target, keeping every row
//     (fwdback.c:258-465 with do_full). The sampled traces below are chaotic
//     in these values: a last-bit difference moves a choice, the random
//     stream then falls out of step, and every later trace differs. So the
//     matrix is computed in the reference's own operation order: its four
//     striped lanes (model position k = r*Q + q + 1) are lanes 0..3 here for
//     the sums that run along q (the row's E sum, the D->D passes), while the
//     cells' M and I values, which depend only on the row before, are spread
//     over the 64 lanes. The file is compiled without contraction into fused
//     multiply-adds and with flushed fp32 denormals, as the reference runs
//     with FTZ/DAZ set; each operation is written out in the reference's
//     order.
//  2. nsamples stochastic traces (impl_sse/stotrace.c:76-329) with Easel's
//     fast generator reset to the seed (esl_random.c:148-160, 215-230,
//     289-310). A step's candidate paths are lanes 0..3: one product each,
//     esl_vec_FNorm's float sum and division, esl_rnd_FChoose's double sums
//     and divisions, and the first lane whose threshold exceeds the roll.
//     select_e scans row i in the striped order with a double running sum.
//     Each sampled domain (p7_trace_Index, p7_trace.c:1173-1206) gets the null2
//     odds of its own trace segment (p7_Null2_ByTrace, impl_sse/null2.c:134-
//     205: every emitting M or I state counts at the M cell of its node), and
//     every residue of the region adds, per trace, that odds or 1 outside
//     domains; n2sc = logf(sum / nsamples).
//  3. The sampled domains are clustered by single linkage (esl_cluster.c:
//     136-185 with link_spsamples, p7_spensemble.c:191-222), clusters with
//     posterior >= 0.25 get the widest endpoints with >= 2% support
//     (p7_spensemble.c:282-411), sorted by start, and clusters dominated by an
//     overlapping one of higher posterior are dropped (p7_domaindef.c:650-682).
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include <algorithm>

#include "p7g_device.h"
#include "p7g_devfn.h"

// (also stated here, so that no build of this file contracts)
#pragma clang fp contract(off)

enum { MS_M = 1, MS_D, MS_I, MS_S, MS_N, MS_B, MS_E, MS_C, MS_T, MS_J };

// Bob Jenkins' 96-bit mix, as esl_random.c disperses a seed
__device__ __forceinline__ uint32_t md_mix3(uint32_t a, uint32_t b, uint32_t c)
{
  a = (a - b - c) ^ (c >> 13);
  b = (b - c - a) ^ (a << 8);
  c = (c - a - b) ^ (b >> 13);
  a = (a - b - c) ^ (c >> 12);
  b = (b - c - a) ^ (a << 16);
  c = (c - a - b) ^ (b >> 5);
  a = (a - b - c) ^ (c >> 3);
  b = (b - c - a) ^ (a << 10);
  c = (c - a - b) ^ (b >> 15);
  return c;
}

// the device Forward table's value of row `row` at model position k (0 past M)
__device__ __forceinline__ float md_tv(const DevProfile &p, int row, int k)
{
  if (k < 1 || k > p.M) return 0.0f;
  const int B = p.fb_B, zl = (k - 1) / B, j = (k - 1) - zl * B;
  return p.fb_tbl[((size_t) row * B + j) * 64 + zl];
}

// the device table row of the i-th staged transition row
__device__ __forceinline__ int md_trow(int i)
{
  switch (i) {
  case 0: return VT_BM; case 1: return VT_MM; case 2: return VT_IM; case 3: return VT_DM;
  case 4: return VT_MDS; case 5: return VT_DDS; case 6: return VT_MI; case 7: return VT_II;
  case 8: return FT_MD; default: return FT_DD;
  }
}

// esl_vec_FNorm then esl_rnd_FChoose's thresholds for n choices of weights
// v: the float sum and divisions, then the double running sums each divided
// by their total; the first n - 1 of them go to th (the last is 1)
__device__ __forceinline__ void md_thresholds(const float *v, int n, double *th)
{
  float s = 0.0f;
  for (int a = 0; a < n; a++) s = __fadd_rn(s, v[a]);
  double c[4], tot = 0.0;
  for (int a = 0; a < n; a++) {
    const float pa = (s != 0.0f) ? __fdiv_rn(v[a], s) : (float) (1.0 / (double) (float) n);
    tot = tot + (double) pa;
    c[a] = tot;
  }
  for (int a = 0; a < n - 1; a++) th[a] = c[a] / tot;
}

// Where one wavefront works alone, its LDS operations, and its loads and stores
// of one address, complete in the order it issues them: between lanes that
// exchange data so it is enough that the compiler moves no memory operation
// across this point (a workgroup barrier would also wait for the outstanding
// global stores, and waves that have left the workgroup could not reach it).
__device__ __forceinline__ void md_sync()
{
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

struct MdSeg { int idx, i, j, k, m; };

// link_spsamples: overlap >= 0.8 of the smaller segment in the sequence and in
// the model (the model overlap without the +1, as the reference has it), and
// start or end diagonals within 4
__device__ __forceinline__ bool md_linked(const MdSeg &a, const MdSeg &b)
{
  int nov = min(a.j, b.j) - max(a.i, b.i) + 1;
  int n = min(a.j - a.i + 1, b.j - b.i + 1);
  if (__fdiv_rn((float) nov, (float) n) < 0.8f) return false;
  nov = min(a.m, b.m) - max(a.k, b.k);
  n = min(a.m - a.k + 1, b.m - b.k + 1);
  if (__fdiv_rn((float) nov, (float) n) < 0.8f) return false;
  if (abs((a.i - a.k) - (b.i - b.k)) <= 4) return true;
  if (abs((a.j - a.m) - (b.j - b.m)) <= 4) return true;
  return false;
}

struct MdSig { int c, i, j, k, m; float prob; };

// The region's Forward matrix, one wave per region. The cells' M and I run on all
// lanes; what the reference's operation order makes serial along q runs on lanes
// 0..3 (its four SSE lanes), 10 cycles a step: the first D->D pass, beside which
// lanes 4..7 take the M sum, then each later pass's carries, and the row's D sum.
// Rows are kept per buffer in model order (cell (q, r) at r*QS + q), four steps to
// an LDS access. A later pass only adds its carries to the cells, which all lanes
// do; and where every D->D odds is at most 1 a pass is left out whose first
// carry is too small to change any cell, for then none of its carries does.
// Regions of up to 240 and 487 residues: M = 86 0.50 ms, M = 400 2.6 ms; with every
// pass run in full by four lanes, cell by cell between LDS waits, 1.15 and 5.9 ms.
// NU: models of up to 512 positions, NU cells per lane (c = 64 u + z), whose
// transitions, places and odds are in registers; a step over them loads all
// cells' operands before it stores any. 0: larger models, cell by cell.
template <int NU>
__global__ __launch_bounds__(64) void
k_md_fwd(const DevProfile p, const uint8_t *__restrict__ res, const MdJob *__restrict__ jobs, float *__restrict__ pool)
{
  extern __shared__ __attribute__((aligned(16))) float lds[];
  const int z = threadIdx.x;
  const MdJob J = jobs[blockIdx.x];
  const int M = p.M, Q = max(2, (M - 1) / 4 + 1), QS = (Q + 7) & ~7, Lr = J.Lr, L = J.Ltarget;
  const int TR = p.nrows;                                  // first transition row of the table
  const float xEmove = p.xfE_move, xEloop = p.xfE_loop, floop = p.xf_loop[L], fmove = p.xf_move[L];
  const uint8_t *dsq = res + J.res_off;                    // residue i (1-based) at dsq[i-1]
  float *mat = pool + J.area;                              // rows 0..Lr, [q][s][r], s = 0 M, 1 D, 2 I
  float *xmx = mat + (size_t) (Lr + 1) * 12 * Q;           // rows 0..Lr: E N J B C SCALE
  // The profile's transitions, staged in LDS when they fit (md_stage_t): rows
  // BM MM IM DM (into k), MDS DDS (into D_k), MI II, MD DD (out of k), each
  // [k = 0..M+1] with 0 outside 1..M
  const bool stage = md_stage_t(M);
  const int TW = M + 2;
  float *tl = lds;
  float *ph = lds + (stage ? md_stage_floats(M) : 0);       // the phases' own LDS
  if (stage)
    for (int c = z; c < 10 * TW; c += 64) tl[c] = md_tv(p, TR + md_trow(c / TW), c % TW);
  auto tv = [&](int row, int k) -> float {                 // row: 0..9 as staged
    if (stage) return tl[row * TW + k];
    return md_tv(p, TR + md_trow(row), k);
  };
  enum { T_BM = 0, T_MM, T_IM, T_DM, T_MDS, T_DDS, T_MI, T_II, T_MD, T_DD };

  // two rows of M, D, I; the D->D odds; a scratch row (odds of models above 512
  // positions; the carries of a pass); a zero cell, what precedes k = 1
  constexpr bool pre = NU > 0;
  constexpr int NC = pre ? NU : 1;
  const int N = pre ? 512 : 4 * QS;                        // a buffer's cells
  float *prev = ph, *cur = ph + 3 * N, *tdd = ph + 6 * N, *scr = ph + 7 * N;
  const int zero = (QS > Q && ! pre) ? 6 * N + Q : 8 * N;   // index in ph (md_row_floats): the odds' padding, or a cell of its own
  auto cell_k = [&](int c, int &q, int &r) { r = (c >= QS) + (c >= 2 * QS) + (c >= 3 * QS); q = c - r * QS; return r * Q + q + 1; };
  __syncthreads();
  for (int c = z; c < 3 * N; c += 64) prev[c] = cur[c] = 0.0f;
  for (int c = z; c < 12 * Q; c += 64) mat[c] = 0.0f;
  if (z == 0 && zero == 8 * N) ph[zero] = 0.0f;
  if (pre) for (int c = z; c < QS; c += 64) ph[8 * N + 4 + c] = 1.0f;      // odds of 1, for the M sum
  bool le1 = true;
  for (int c = z; c < N; c += 64) {
    int q, r;
    const int k = cell_k(c, q, r);
    const float t = (q < Q) ? tv(T_DD, min(k, M + 1)) : 0.0f;
    tdd[c] = t;
    scr[c] = 0.0f;
    // no odds above 1, and none out of the model's end into the cells behind it
    le1 = le1 && t >= 0.0f && t <= 1.0f && (k < M || t == 0.0f);
  }
  const bool skips = __all(le1);
  float xN = 1.0f, xJ = 0.0f, xB = fmove, xC = 0.0f, xE = 0.0f;
  if (z == 0) { xmx[0] = 0.0f; xmx[1] = xN; xmx[2] = xJ; xmx[3] = xB; xmx[4] = xC; xmx[5] = 1.0f; }
  __syncthreads();
  // the residues 64 rows at a time; a row's odds one row ahead
  const size_t xrow = (size_t) 64 * p.fb_B;
  float enext[NC], ecur[NC], tBMr[NC], tMMr[NC], tIMr[NC], tDMr[NC], tMIr[NC], tIIr[NC], tMDr[NC];
  int kr[NC], pr[NC], eo[NC], q0m = 0, xcur = 0;           // q0m: bit u where q = 0
  int ro[3 * NC];                                          // what the row's [q][s][r] copy takes from
  auto load_row = [&](int i1) {
    const int s = (i1 - 1) & 63;
    if (s == 0) xcur = dsq[min(i1 - 1 + z, Lr - 1)];
    const float *er = p.fb_tbl + (size_t) __builtin_amdgcn_readlane(xcur, s) * xrow;
#pragma unroll
    for (int u = 0; u < NC; u++) enext[u] = er[eo[u]];
  };
  if (pre) {
#pragma unroll
    for (int u = 0; u < NC; u++) {
      const int c = u * 64 + z;
      int q, r;
      const int k = cell_k(c, q, r), kk = min(k, M + 1);
      const bool in = q < Q;
      kr[u] = in ? k : 0;
      // model position k in the device table (past M: any, not used)
      const int kz = min(max(k, 1), M) - 1, zl = kz / p.fb_B;
      eo[u] = (kz - zl * p.fb_B) * 64 + zl;
      q0m |= (int) (q == 0) << u;
      // row i-1's predecessor, as an index from prev (none: far out, see cells)
      pr[u] = (q > 0) ? c - 1 : (r > 0) ? (r - 1) * QS + Q - 1 : -1;
      tBMr[u] = in ? tv(T_BM, kk) : 0.0f; tMMr[u] = in ? tv(T_MM, kk) : 0.0f;
      tIMr[u] = in ? tv(T_IM, kk) : 0.0f; tDMr[u] = in ? tv(T_DM, kk) : 0.0f;
      tMIr[u] = in ? tv(T_MI, kk) : 0.0f; tIIr[u] = in ? tv(T_II, kk) : 0.0f;
      tMDr[u] = (in && q > 0) ? tv(T_MD, min(k - 1, M + 1)) : 0.0f;
    }
#pragma unroll
    for (int v = 0; v < 3 * NC; v++) {
      const int c = min(v * 64 + z, 12 * Q - 1), q = c / 12, s = (c - 12 * q) >> 2;
      ro[v] = s * N + (c & 3) * QS + q;
    }
    load_row(1);
  }
  // M and I of a cell from row i-1 (esl_sse_rightshift_ps at q = 0)
  auto cell_m = [&](float mp, float dp, float ip, float e, float bm, float mm, float im, float dm) {
    float sv = __fmul_rn(xB, bm);
    sv = __fadd_rn(sv, __fmul_rn(mp, mm));
    sv = __fadd_rn(sv, __fmul_rn(ip, im));
    sv = __fadd_rn(sv, __fmul_rn(dp, dm));
    return __fmul_rn(sv, e); };
  auto cell_i = [&](float m, float i, float mi, float ii) { return __fadd_rn(__fmul_rn(m, mi), __fmul_rn(i, ii)); };
  // A chain along q over one or two arrays, eight steps' values loaded while the
  // eight before run. f(q, u, a, b): the step, from a = A[q], b = T[q]; what it
  // returns goes to dst[q] where there is one.
  auto chain = [&](const float *A, const float *T, float *dst, auto f) {
    auto ld = [&](const float *x, int q, float (&v)[8]) {
      const float4 *w = (const float4 *) (x + q);
      const float4 w0 = w[0], w1 = w[1];
      v[0] = w0.x; v[1] = w0.y; v[2] = w0.z; v[3] = w0.w; v[4] = w1.x; v[5] = w1.y; v[6] = w1.z; v[7] = w1.w; };
    auto run = [&](int q, const float (&a)[8], const float (&b)[8]) {
      float o[8];
#pragma unroll
      for (int u = 0; u < 8; u++) o[u] = f(a[u], T ? b[u] : 0.0f);
      if (dst) {
        float4 *w = (float4 *) (dst + q);
        w[0] = make_float4(o[0], o[1], o[2], o[3]); w[1] = make_float4(o[4], o[5], o[6], o[7]);
      } };
    auto tail = [&](int q, const float (&a)[8], const float (&b)[8]) {
#pragma unroll
      for (int u = 0; u < 7; u++)
        if (q + u < Q) { const float o = f(a[u], T ? b[u] : 0.0f); if (dst) dst[q + u] = o; } };
    float a0[8], b0[8], a1[8], b1[8];
    ld(A, 0, a0); if (T) ld(T, 0, b0);
    int q = 0;
    for (; q + 16 <= Q; q += 16) {
      ld(A, q + 8, a1); if (T) ld(T, q + 8, b1);
      run(q, a0, b0);
      const int qn = min(q + 16, QS - 8);
      ld(A, qn, a0); if (T) ld(T, qn, b0);
      run(q + 8, a1, b1);
    }
    if (q + 8 <= Q) {
      const int qn = min(q + 8, QS - 8);
      ld(A, qn, a1); if (T) ld(T, qn, b1);
      run(q, a0, b0);
      tail(q + 8, a1, b1);
    } else tail(q, a0, b0);
  };
  for (int i = 1; i <= Lr; i++) {
    if (pre) {
#pragma unroll
      for (int u = 0; u < NC; u++) ecur[u] = ((unsigned) (kr[u] - 1) < (unsigned) M) ? enext[u] : 0.0f;
      if (i < Lr) load_row(i + 1);
      md_sync();
      float mp[NC], dp[NC], ip[NC], m0[NC], i0[NC];
#pragma unroll
      for (int u = 0; u < NC; u++) {
        const float *P = (pr[u] >= 0) ? prev + pr[u] : ph + zero;
        const int dn = (pr[u] >= 0) ? N : 0;
        mp[u] = P[0]; dp[u] = P[dn]; ip[u] = P[2 * dn]; m0[u] = prev[u * 64 + z]; i0[u] = prev[2 * N + u * 64 + z];
      }
#pragma unroll
      for (int u = 0; u < NC; u++) {
        m0[u] = cell_i(m0[u], i0[u], tMIr[u], tIIr[u]);
        mp[u] = cell_m(mp[u], dp[u], ip[u], ecur[u], tBMr[u], tMMr[u], tIMr[u], tDMr[u]);
      }
#pragma unroll
      for (int u = 0; u < NC; u++) { cur[u * 64 + z] = mp[u]; cur[2 * N + u * 64 + z] = m0[u]; }
      md_sync();
      // D before the D->D passes: cell q holds M(q-1)·tMD (the q loop's dcv); q = 0 holds 0
#pragma unroll
      for (int u = 0; u < NC; u++) mp[u] = cur[max(pr[u], 0)];
#pragma unroll
      for (int u = 0; u < NC; u++) cur[N + u * 64 + z] = (((q0m >> u) & 1) || kr[u] == 0) ? 0.0f : __fmul_rn(mp[u], tMDr[u]);
    } else {
      const int x = dsq[i - 1];
      for (int c0 = 0; c0 < N; c0 += 64 * 8) {             // this residue's odds
        float e[8];
#pragma unroll
        for (int u = 0; u < 8; u++) { const int c = c0 + u * 64 + z; int q, r; const int k = cell_k(c, q, r); e[u] = md_tv(p, x, (c < N && q < Q) ? k : 0); }
#pragma unroll
        for (int u = 0; u < 8; u++) { const int c = c0 + u * 64 + z; if (c < N) scr[c] = e[u]; }
      }
      md_sync();
      for (int c = z; c < N; c += 64) {
        int q, r;
        const int k = cell_k(c, q, r), kk = min(k, M + 1), pc = (q > 0) ? c - 1 : (r > 0) ? (r - 1) * QS + Q - 1 : -1;
        if (q < Q) {
          const float *P = (pc >= 0) ? prev + pc : ph + zero;
          const int dn = (pc >= 0) ? N : 0;
          const float m = cell_m(P[0], P[dn], P[2 * dn], scr[c], tv(T_BM, kk), tv(T_MM, kk), tv(T_IM, kk), tv(T_DM, kk));
          cur[2 * N + c] = cell_i(prev[c], prev[2 * N + c], tv(T_MI, kk), tv(T_II, kk));
          cur[c] = m;
        }
      }
      md_sync();
      for (int c = z; c < N; c += 64) {
        int q, r;
        const int k = cell_k(c, q, r);
        if (q < Q) cur[N + c] = q ? __fmul_rn(cur[c - 1], tv(T_MD, min(k - 1, M + 1))) : 0.0f;
      }
    }
    md_sync();
    const int r4 = z & 3;
    float dcv = 0.0f, xm;
    if (z < 8) {
      // lanes 0..3: D(q) = dcv + D0(q), dcv = D(q)·tDD(q); lanes 4..7: the M sum
      // in the same steps, with odds of 1, its partial sums to the scratch row
      const bool dl = z < 4;
      const float end = __fmul_rn(cur[r4 * QS + Q - 1], tv(T_MD, min(r4 * Q + Q, M + 1)));
      const float sh = __shfl(end, (z + 3) & 3, 4);
      float acc = (dl && r4) ? sh : 0.0f;
      chain(cur + (dl ? N : 0) + r4 * QS, (dl || ! pre) ? tdd + r4 * QS : ph + 8 * N + 4, (dl ? cur + N : scr) + r4 * QS, [&](float d, float t) {
        const float o = __fadd_rn(acc, d);
        acc = __fmul_rn(o, (pre || dl) ? t : 1.0f);
        return o; });
      dcv = acc;
    }
    xm = __shfl(dcv, 4 + r4, 64);                          // lane r: the M sum of its lane
    md_sync();
    for (int pass = 1; pass < 4; pass++) {
      const float sh = __shfl(dcv, (z + 3) & 3, 4);
      dcv = (z < 4 && r4) ? sh : 0.0f;
      if (skips && pass > 1) {
        // the carry against the smallest D of the cells it can reach (positive
        // values, whose bit patterns order as integers)
        int big = 0;
        auto take = [&](int k, float d) { if (k > Q && k <= M) big = max(big, 0x7f800000 - __float_as_int(d)); };
        if (pre) {
          float d[NC];
#pragma unroll
          for (int u = 0; u < NC; u++) d[u] = cur[N + u * 64 + z];
#pragma unroll
          for (int u = 0; u < NC; u++) take(kr[u], d[u]);
        } else
          for (int c = z; c < N; c += 64) { int q, r; const int k = cell_k(c, q, r); if (q < Q) take(k, cur[N + c]); }
        const float dmin = __int_as_float(0x7f800000 - uni(wave_max_i(big)));
        if (__all(dcv == 0.0f || (dcv > 0.0f && dcv < dmin * 0x1p-26f && dmin >= 0x1p-90f && dmin < INFINITY))) break;
      }
      if (z < 4) {
        float acc = dcv;
        chain(tdd + z * QS, nullptr, scr + z * QS, [&](float t, float) { const float o = acc; acc = __fmul_rn(acc, t); return o; });
        dcv = acc;
      }
      md_sync();
      bool changed = false;
      if (pre) {
        float d[NC], g[NC];
#pragma unroll
        for (int u = 0; u < NC; u++) { d[u] = cur[N + u * 64 + z]; g[u] = scr[u * 64 + z]; }
#pragma unroll
        for (int u = 0; u < NC; u++) {
          const float dd = (kr[u] > 0) ? __fadd_rn(g[u], d[u]) : 0.0f;
          changed = changed || dd > d[u];
          cur[N + u * 64 + z] = dd;
        }
      } else
        for (int c = z; c < N; c += 64) {
          int q, r;
          (void) cell_k(c, q, r);
          if (q < Q) {
            const float d = cur[N + c], dd = __fadd_rn(scr[c], d);
            changed = changed || dd > d;
            cur[N + c] = dd;
          }
        }
      md_sync();
      if (M >= 100 && ! __any(changed)) break;
    }
    float xe = 0.0f;
    if (z < 4) {                                           // the row's sum: the M sum, then D in q order
      xe = xm;
      chain(cur + N + z * QS, nullptr, nullptr, [&](float d, float) { xe = __fadd_rn(d, xe); return 0.0f; });
    }
    // esl_sse_hsum_ps: (e0 + e1) + (e2 + e3)
    xE = __fadd_rn(__fadd_rn(readlanef(xe, 0), readlanef(xe, 1)), __fadd_rn(readlanef(xe, 2), readlanef(xe, 3)));
    xN = __fmul_rn(xN, floop);
    xC = __fadd_rn(__fmul_rn(xC, floop), __fmul_rn(xE, xEmove));
    xJ = __fadd_rn(__fmul_rn(xJ, floop), __fmul_rn(xE, xEloop));
    xB = __fadd_rn(__fmul_rn(xJ, fmove), __fmul_rn(xN, fmove));
    float scale = 1.0f;
    md_sync();
    if (xE > 1.0e4f) {
      xN = __fdiv_rn(xN, xE); xC = __fdiv_rn(xC, xE); xJ = __fdiv_rn(xJ, xE); xB = __fdiv_rn(xB, xE);
      const float inv = (float) (1.0 / (double) xE);
      for (int c = z; c < 3 * N; c += 64) cur[c] = __fmul_rn(cur[c], inv);
      scale = xE;
      xE = 1.0f;
      md_sync();
    }
    float *row = mat + (size_t) i * 12 * Q;
    if (pre) {                                             // [q][s][r]
      float v[3 * NC];
#pragma unroll
      for (int j = 0; j < 3 * NC; j++) v[j] = cur[ro[j]];
#pragma unroll
      for (int j = 0; j < 3 * NC; j++) if (j * 64 + z < 12 * Q) row[j * 64 + z] = v[j];
    } else
      for (int c = z; c < 12 * Q; c += 64) {
        const int q = c / 12, s = (c - 12 * q) >> 2;
        row[c] = cur[s * N + (c & 3) * QS + q];
      }
    if (z == 0) {
      float *xr = xmx + (size_t) i * 6;
      xr[0] = xE; xr[1] = xN; xr[2] = xJ; xr[3] = xB; xr[4] = xC; xr[5] = scale;
    }
    float *t = prev; prev = cur; cur = t;
    md_sync();
  }
}

// The comparison of a draw x with a threshold th in (0, 1], as the walk makes
// it on integers: x / 2^32 < th is x < T, T = ceil(2^32 th), or always when T is
// 2^32 (bit a of the cell's flags). T = 0 for thresholds that no draw is under,
// NaN among them.
__device__ __forceinline__ uint32_t md_thr_word(double th, int a, uint32_t &flags)
{
  const double v = ceil(th * 4294967296.0);
  if (! (v >= 1.0)) return 0u;
  if (v > 4294967295.0) { flags |= 1u << a; return 0u; }
  return (uint32_t) v;
}
enum { MD_NAN_M = 5, MD_NAN_D = 6, MD_NAN_I = 7 };         // flag bits: the cell's weights gave NaN

// The traces' walks: one wave per region. A walk is a chain of dependent
// steps, each a random draw against the thresholds of the state it is in, and
// its loads' latency bounds the stage: nothing else is done here. In a state
// that can repeat (M along its diagonal, D along its row, I, C and J down their
// column) lane l takes the step that follows l repeats, with the (l+1)-th draw
// from here (the generator's jump) and that cell's thresholds; the first lane
// whose step leaves the state (or fails) is the step the walk takes after those
// repeats. What a sampled domain's steps mean (its counts, null2 odds, ends) is
// left to k_md_replay, for which each run goes to the log: bits 0-6 the
// repeats, 7-9 the state it leads to (0: the run goes on), 10 whether that I
// or D state steps back to M at once; a domain starts with its last node and
// state. Regions of up to 240 and 487 residues, walk + replay: M = 86 3.1 + 1.7 ms,
// M = 400 6.2 + 1.2 ms; with the steps' bookkeeping and the null2 sums of each
// domain in the walk's chain, one wave a region, it was 9.1 and 13.7 ms.
__global__ __launch_bounds__(64) void
k_md_walk(const DevProfile p, const MdJob *__restrict__ jobs, MdOut *__restrict__ out, float *__restrict__ pool,
          int nsamples, uint32_t seed, int first)
{
  const int z = threadIdx.x;
  const MdJob J = jobs[blockIdx.x];
  MdOut *O = out + blockIdx.x;
  const int M = p.M, Q = max(2, (M - 1) / 4 + 1), Lr = J.Lr;
  float *area = pool + J.area;
  const float *mat = area, *xmx = mat + (size_t) (Lr + 1) * 12 * Q;
  const double *xthr = (const double *) (area + md_xthr_at(M, Lr, J.segcap));
  const double *ecum = (const double *) (area + md_ecum_at(M, Lr, J.segcap));
  const uint2 *thr = (const uint2 *) (area + md_thr_at(M, Lr, J.segcap));
  uint16_t *lg = (uint16_t *) (area + md_log_at(M, Lr, J.segcap));
  MdSeg *segs = (MdSeg *) (area + md_seg_at(M, Lr));
  int *dlog = (int *) (area + md_clu_at(M, Lr, J.segcap)), *drow = dlog + J.segcap;
  uint32_t rng;
  int t = 0, nseg = 0, status = 0;
  if (first) {
    rng = md_mix3(seed, 87654321u, 12345678u);
    if (rng == 0) rng = 42;
  } else {
    status = O->status; t = O->trace; nseg = O->nseg; rng = O->rng;
    if (status || t >= nsamples) return;
  }
  rng = (uint32_t) uni((int) rng); t = uni(t); nseg = uni(nseg);
  // lane l's jump: l + 1 draws of x -> 69069 x + 1 are x -> jA x + jC
  uint32_t jA = 1u, jC = 0u;
  for (int l = 0; l <= z; l++) { jA *= 69069u; jC = jC * 69069u + 1u; }
  const int64_t max_steps = 64 * ((int64_t) Lr + M + 16);
  const int64_t log_end = md_log_entries(M, Lr) - md_log_trace(M, Lr);
  int lbuf = 0;                                            // lane u: the log's entry n with n mod 64 = u
  int n = 0;
  auto put = [&](int v) {
    lbuf = (z == (n & 63)) ? v : lbuf;
    if ((n & 63) == 63) lg[n - 63 + z] = (uint16_t) lbuf;
    n++;
  };
  for (; t < nsamples && ! status && n <= log_end; t++) {
    int i = Lr, k = 0, nd = 0;
    int64_t steps = 0;
    bool over = false;
    int col = 0;                                           // 0 the C state, 1 J
    for (;;) {
      // down C's or J's column to an E
      for (;;) {
        const uint32_t xl = jA * rng + jC;
        const double roll = (double) xl / 4294967296.0;
        const int li = i - z;
        int sl = -1;                                       // 0 stays, 1 E
        if (li >= 1) {
          const double th = xthr[(size_t) li * 3 + col];
          sl = (roll < th) ? 0 : (th == th) ? 1 : -1;
        }
        const unsigned long long stop = __ballot(sl != 0);
        const int f = stop ? (int) __ffsll((long long) stop) - 1 : 64;
        i -= f;
        steps += f;
        if (f == 64) {
          rng = (uint32_t) __builtin_amdgcn_readlane((int) xl, 63);
          if (steps > max_steps) { status = 1; break; }
          continue;
        }
        rng = (uint32_t) __builtin_amdgcn_readlane((int) xl, f);
        if (++steps > max_steps || __builtin_amdgcn_readlane(sl, f) < 0) status = 1;
        break;
      }
      if (status) break;
      // E: one roll; the first running sum above it
      if (++steps > max_steps || i < 1) { status = 1; break; }
      int s = -1;
      {
        rng = rng * 69069u + 1u;
        const double roll = (double) rng / 4294967296.0;
        // the row's running sums are kept at every 64th element (ecum,
        // md_ncp per row): the first checkpoint above the roll names the
        // chunk, whose sums are formed again from the checkpoint before it
        const int NCP = md_ncp(Q);
        const double *cp = ecum + (size_t) i * NCP;
        int c = -1;
        for (int c0 = 0; c0 < NCP && c < 0; c0 += 64) {
          const int cc = c0 + z;
          const double v = cp[min(cc, NCP - 1)];
          const unsigned long long m = __ballot(cc < NCP && roll < v);
          if (m) c = c0 + (int) __ffsll((long long) m) - 1;
        }
        int found = -1;
        const float nf = (float) (1.0 / (double) xmx[(size_t) i * 6 + 0]);
        if (c >= 0) {
          const int j = 64 * c + z, q = j >> 3;
          const float u = (j < 8 * Q) ? __fmul_rn(mat[((size_t) i * Q + q) * 12 + (j & 7)], nf) : 0.0f;
          double sum = c ? cp[c - 1] : 0.0;
          // eight sums to a test (they do not fall: a roll under one of them is
          // under the last, unless that is no number)
          for (int l0 = 0; l0 < 64 && found < 0; l0 += 8) {
            double s8[8];
#pragma unroll
            for (int l = 0; l < 8; l++) { sum = sum + (double) readlanef(u, l0 + l); s8[l] = sum; }
            if (! (roll >= s8[7])) {
#pragma unroll
              for (int l = 7; l >= 0; l--) if (roll < s8[l]) found = 64 * c + l0 + l;
            }
          }
        }
        if (found >= 0) {
          k = (found & 3) * Q + (found >> 3) + 1;
          s = ((found >> 2) & 1) ? MS_D : MS_M;
        } else {
          // the reference scans the row again, the sum going on from its total
          double sum = cp[NCP - 1];
          for (int pass = 1; pass < 4 && s < 0; pass++)
            for (int q0 = 0; q0 < Q && s < 0; q0 += 8) {
              const int q = q0 + (z >> 3), sm = (z >> 2) & 1, r = z & 3;
              const float u = (q < Q) ? __fmul_rn(mat[(((size_t) i * Q + q) * 3 + sm) * 4 + r], nf) : 0.0f;
              for (int l = 0; l < 64; l++) {
                sum = sum + (double) readlanef(u, l);
                if (roll < sum) { k = (l & 3) * Q + q0 + (l >> 3) + 1; s = ((l >> 2) & 1) ? MS_D : MS_M; break; }
              }
            }
        }
      }
      if (s < 0 || k < 1 || k > M) { status = 1; break; }
      if (nseg + nd < J.segcap) {
        if (z == 0) { dlog[nseg + nd] = n; drow[nseg + nd] = i; segs[nseg + nd].idx = t; }
      } else over = true;
      put(k | (s == MS_D ? 0x8000 : 0));
      // the domain's runs, to its B
      while (s != MS_B) {
        const uint32_t xl = jA * rng + jC;
        const int li = (s == MS_D) ? i : i - z, lk = (s == MS_I) ? k : k - z;
        int sl = -1;
        // An M run's step to I or D is most often followed by one step back
        // to M. Lane l also takes that step ahead, as if it stopped here:
        // the I or D cell is lane l+1's, whose thresholds that lane loads
        // anyway, and the draw the next one. spec: that step leads to M
        // (and its M cell is inside the matrix).
        bool spec = false;
        if (s == MS_M) {
          const bool in = (li >= 1 && lk >= 1);
          uint2 ta = make_uint2(0u, 0u), tb = ta, tc = ta;
          if (in) {
            const uint2 *c = thr + ((size_t) li * (M + 1) + lk) * 3;
            ta = c[0]; tb = c[1]; tc = c[2];
          }
          const uint32_t F = tc.y;
          if (in)
            sl = (xl < ta.x || (F & 1u)) ? MS_B : (xl < ta.y || (F & 2u)) ? MS_M : (xl < tb.x || (F & 4u)) ? MS_I
                 : (F >> MD_NAN_M & 1u) ? -1 : MS_D;
          // cell (li - 1, lk - 1): lane 63 has no next lane
          const uint32_t n3 = (uint32_t) wave_shl1((int) tb.y, 0), n4 = (uint32_t) wave_shl1((int) tc.x, 0);
          const uint32_t nF = (uint32_t) wave_shl1((int) F, 0);
          const bool nin = wave_shl1((int) in, 0) != 0;
          const uint32_t x2 = 69069u * xl + 1u;
          // back to M at (li - 2, lk - 1) from I, (li - 1, lk - 2) from D
          if (sl == MS_I) spec = nin && (x2 < n4 || (nF & 16u)) && li - 2 >= 1;
          if (sl == MS_D) spec = nin && (x2 < n3 || (nF & 8u)) && lk - 2 >= 1;
        } else if (li >= 1 && lk >= 1) {
          const uint2 *c = thr + ((size_t) li * (M + 1) + lk) * 3;
          const uint2 tb = c[1], tc = c[2];
          const uint32_t tt = (s == MS_D) ? tb.y : tc.x;
          const uint32_t F = tc.y, all = (s == MS_D) ? 8u : 16u, nan = 1u << ((s == MS_D) ? MD_NAN_D : MD_NAN_I);
          sl = (xl < tt || (F & all)) ? MS_M : (F & nan) ? -1 : s;
        }
        const unsigned long long stop = __ballot(sl != s);
        const int f = stop ? (int) __ffsll((long long) stop) - 1 : 64;
        if (s != MS_D) i -= f;
        if (s != MS_I) k -= f;
        steps += f;
        if (f == 64) {
          rng = (uint32_t) __builtin_amdgcn_readlane((int) xl, 63);
          if (steps > max_steps) { status = 1; break; }
          put(64);
          continue;
        }
        rng = (uint32_t) __builtin_amdgcn_readlane((int) xl, f);
        const int s1 = __builtin_amdgcn_readlane(sl, f);
        const bool back = (s == MS_M) && __builtin_amdgcn_readlane((int) spec, f) != 0;
        if (++steps > max_steps || s1 < 0) { status = 1; break; }
        if (s != MS_D) i--;
        if (s != MS_I) k--;
        if (s1 != MS_B && (k < 1 || k > M || i < 1)) { status = 1; break; }
        put(f | (s1 << 7) | ((int) back << 10));
        s = s1;
        // the I or D state's step back to M, taken ahead in the M run's ballot:
        // its draw, then the M element at (i - 1, k) from I, (i, k - 1) from D
        if (back) {
          rng = rng * 69069u + 1u;
          if (s1 == MS_I) i--; else k--;
          if (++steps > max_steps || k < 1 || k > M || i < 1) { status = 1; break; }
          s = MS_M;
        }
      }
      if (status) break;
      if (nd >= MD_TSEG) { status = 5; break; }
      nd++;
      // B: N (which repeats down to row 0 without draws) or J
      if (++steps > max_steps) { status = 1; break; }
      rng = rng * 69069u + 1u;
      const double roll = (double) rng / 4294967296.0, th = xthr[(size_t) i * 3 + 2];
      if (roll < th) { if (++steps > max_steps) status = 1; break; }
      if (! (th == th)) { status = 1; break; }
      col = 1;
    }
    if (! status && over) status = 5;
    if (! status) nseg += nd;
  }
  if ((n & 63) && z < (n & 63)) lg[(n & ~63) + z] = (uint16_t) lbuf;
  if (z == 0) {
    O->status = status; O->trace = t; O->nseg = nseg; O->rng = rng;
    if (first) { O->nc = 0; O->rtrace = 0; O->rdom = 0; O->done = 0; }
  }
}

// What the walked traces mean: one workgroup per region. Each sampled domain
// (p7_trace_Index, p7_trace.c:1173-1206) is replayed from the log by one wave:
// its ends in the sequence and the model, and the null2 odds of its own trace
// segment (p7_Null2_ByTrace, impl_sse/null2.c:134-205: every emitting M or I
// state counts at the M cell of its node). MD_CHUNK domains at a time; then
// every residue adds, per trace in trace order, the odds of the domain that
// holds it or 1 outside domains. After the last trace: n2sc = logf(sum /
// nsamples), and the clustering.
__global__ __launch_bounds__(64 * MD_REPLAY_WAVES) void
k_md_replay(const DevProfile p, const uint8_t *__restrict__ res, const MdJob *__restrict__ jobs, MdOut *__restrict__ out,
            float *__restrict__ pool, int nsamples)
{
  extern __shared__ float lds[];
  const int tid = threadIdx.x, z = tid & 63, wv = tid >> 6, NT = blockDim.x, NW = NT >> 6;
  const MdJob J = jobs[blockIdx.x];
  MdOut *O = out + blockIdx.x;
  const int M = p.M, Q = max(2, (M - 1) / 4 + 1), Lr = J.Lr;
  const uint8_t *dsq = res + J.res_off;                    // residue i (1-based) at dsq[i-1]
  float *area = pool + J.area;
  float *xmx = area + (size_t) (Lr + 1) * 12 * Q;
  float *acc = xmx + (size_t) 6 * (Lr + 1);                // residues 0..Lr
  int   *hist = (int *) (acc + (Lr + 1));                  // max(Lr, M) + 2 endpoint counts
  MdSeg *segs = (MdSeg *) (area + md_seg_at(M, Lr));       // the ensemble, J.segcap entries
  const uint16_t *lg = (const uint16_t *) (area + md_log_at(M, Lr, J.segcap));
  const int *dlog = (const int *) (area + md_clu_at(M, Lr, J.segcap)), *drow = dlog + J.segcap;
  int status = O->status;
  const int ntr = O->trace, nseg = O->nseg, dom0 = O->rdom;
  if (O->done) return;
  if (status) { if (tid == 0) { O->nc = 0; O->done = 1; } return; }
  const bool last = (ntr >= nsamples);
  float *n2v = lds;                                        // [MD_CHUNK][32]
  int4  *drec = (int4 *) (lds + MD_CHUNK * 32);            // trace, sqfrom, sqto, last of its trace
  float *cnt = lds + md_rec_floats() + wv * 4 * Q;         // [q][r] counts of this wave's domain
  const bool em_lds = md_em_lds(M) && p.K <= 20;
  float *em = lds + md_rec_floats() + NW * 4 * Q;          // [x][q][r] odds, when em_lds
  if (em_lds)
    for (int c = tid; c < p.K * 4 * Q; c += NT) {
      const int x = c / (4 * Q), rem = c - x * 4 * Q;
      em[c] = md_tv(p, x, min((rem & 3) * Q + (rem >> 2) + 1, M + 1));
    }
  auto cnt_at = [&](int k) {                               // the count cell of model position k
    const int r = (k - 1 >= Q) + (k - 1 >= 2 * Q) + (k - 1 >= 3 * Q);
    return (k - 1 - r * Q) * 4 + r; };
  if (O->rtrace == 0) for (int pos = tid; pos <= Lr; pos += NT) acc[pos] = 0.0f;
  for (int c = z; c < 4 * Q; c += 64) cnt[c] = 0.0f;
  int hi0 = Lr, tr0 = -1;                                  // the domain before the chunk: its sqfrom and trace
  __syncthreads();
  for (int c0 = dom0; c0 < nseg; c0 += MD_CHUNK) {
    const int nc = min(MD_CHUNK, nseg - c0);
    for (int d = wv; d < nc; d += NW) {
      const int e = c0 + d, t = uni(segs[e].idx);
      int at = uni(dlog[e]), i = uni(drow[e]);
      int w = (int) lg[at + z];                            // 64 entries ahead (the log has room past its end)
      int o = 0;
      auto next = [&]() {
        if (o == 64) { at += 64; w = (int) lg[at + z]; o = 0; }
        return __builtin_amdgcn_readlane(w, o++);
      };
      const int v0 = next();
      int k = v0 & 0x7fff, s = (v0 & 0x8000) ? MS_D : MS_M;
      int sqfrom = 0, sqto = 0, hmmfrom = 0, hmmto = 0, Ld = 0, kmin = 0x7fffffff, kmax = 0;
      auto emit = [&](bool m) {                            // an M (m) or I element at (i, k)
        if (z == 0) cnt[cnt_at(k)] += 1.0f;
        kmin = min(kmin, k); kmax = max(kmax, k);
        Ld++;
        if (m) { if (sqto == 0) { sqto = i; hmmto = k; } sqfrom = i; hmmfrom = k; }
        md_sync();
      };
      if (s == MS_M) emit(true);
      while (s != MS_B) {
        const int v = next(), f = v & 0x7f, s1 = (v >> 7) & 7;
        if (f > 0) {                                       // the repeats: M and I states emit
          if (s == MS_M) {
            if (z < f) cnt[cnt_at(k - 1 - z)] += 1.0f;
            kmin = min(kmin, k - f); kmax = max(kmax, k - 1);
            Ld += f;
            if (sqto == 0) { sqto = i - 1; hmmto = k - 1; }
            sqfrom = i - f; hmmfrom = k - f;
            i -= f; k -= f;
          } else if (s == MS_I) {
            if (z == 0) cnt[cnt_at(k)] += (float) f;
            kmin = min(kmin, k); kmax = max(kmax, k);
            Ld += f;
            i -= f;
          } else k -= f;
          md_sync();
        }
        if (s1 == 0) continue;                             // the run goes on
        if (s != MS_D) i--;
        if (s != MS_I) k--;
        if (s1 == MS_M) emit(true);
        else if (s1 == MS_I) emit(false);
        s = s1;
        if (v & 0x400) {
          if (s1 == MS_I) i--; else k--;
          emit(true);
          s = MS_M;
        }
      }
      // four striped sums over q per canonical residue, their hsum; degenerate
      // codes the mean. Lane z sums x = z / 4 and, x + 16 (the same lane r, so
      // the same counts): two chains per lane, one pass
      float *nv = n2v + d * 32;
      const float nrm = (float) (1.0 / (double) (float) Ld);
      for (int base = 0; base < p.K * 4; base += 128) {
        const int xr = base + z, x = xr >> 2, r = xr & 3, x2 = x + 16;
        const bool h1 = x < p.K, h2 = x2 < p.K;
        float sv = 0.0f, sv2 = 0.0f;
        if (h1) {
          // positions kmin..kmax in lane r: the other cells' counts are 0, and
          // adding their products (+0) leaves the striped sum unchanged
          const int q0 = max(0, kmin - 1 - r * Q), q1 = min(Q - 1, kmax - 1 - r * Q);
          for (int qa = q0; qa <= q1; qa += 8) {
            float e1[8], e2[8], cq[8];
#pragma unroll
            for (int u = 0; u < 8; u++) cq[u] = cnt[min(qa + u, Q - 1) * 4 + r];
            if (em_lds) {
#pragma unroll
              for (int u = 0; u < 8; u++) {
                e1[u] = em[(x * Q + min(qa + u, Q - 1)) * 4 + r];
                e2[u] = h2 ? em[(x2 * Q + min(qa + u, Q - 1)) * 4 + r] : 0.0f;
              }
            } else {
#pragma unroll
              for (int u = 0; u < 8; u++) {
                e1[u] = md_tv(p, x, min(r * Q + qa + u + 1, M + 1));
                e2[u] = h2 ? md_tv(p, x2, min(r * Q + qa + u + 1, M + 1)) : 0.0f;
              }
            }
            // a zero count adds +0.0, which leaves the non-negative sums as
            // they are: no branch per cell
#pragma unroll
            for (int u = 0; u < 8; u++) {
              const float wt = __fmul_rn(qa + u <= q1 ? cq[u] : 0.0f, nrm);
              sv = __fadd_rn(sv, __fmul_rn(wt, e1[u]));
              sv2 = __fadd_rn(sv2, __fmul_rn(wt, e2[u]));
            }
          }
        }
        // lanes 4x..4x+3 hold x's lane sums
        const float s01 = __fadd_rn(sv, __shfl_down(sv, 1, 4)), s23 = __shfl_down(s01, 2, 4);
        if (h1 && r == 0) nv[x] = __fadd_rn(__fadd_rn(s01, s23), 0.0f);
        const float t01 = __fadd_rn(sv2, __shfl_down(sv2, 1, 4)), t23 = __shfl_down(t01, 2, 4);
        if (h2 && r == 0) nv[x2] = __fadd_rn(__fadd_rn(t01, t23), 0.0f);
      }
      md_sync();
      {                                                    // degenerate codes: one lane each
        const int xx = p.K + 1 + z;
        if (xx <= p.Kp - 3) {
          const uint32_t dm = p.degen[xx];
          float rr = 0.0f;
          for (int y = 0; y < p.K; y++) if ((dm >> y) & 1u) rr = __fadd_rn(rr, nv[y]);
          nv[xx] = __fdiv_rn(rr, (float) (dm >> 24));
        }
        if (z == 0) { nv[p.K] = 1.0f; nv[p.Kp - 2] = 1.0f; nv[p.Kp - 1] = 1.0f; }
      }
      for (int c = z; c < 4 * Q; c += 64) cnt[c] = 0.0f;
      md_sync();
      // the trace's domains join the ensemble in sequence order: the walk met
      // them last first
      int b0 = e, b1 = e;
      while (b0 > 0 && segs[b0 - 1].idx == t) b0--;
      while (b1 + 1 < nseg && segs[b1 + 1].idx == t) b1++;
      if (z == 0) {
        MdSeg &sg = segs[b0 + b1 - e];
        sg.i = sqfrom; sg.j = sqto; sg.k = hmmfrom; sg.m = hmmto;
        drec[d] = make_int4(t, sqfrom, sqto, e == b1);
      }
    }
    __syncthreads();
    // residues (sqto, hi] are outside domains (1), (sqfrom, sqto] take the odds;
    // hi is the sqfrom of the trace's domain before, or Lr
    for (int pos = tid + 1; pos <= Lr; pos += NT) {
      float a = acc[pos];
      const int x = dsq[pos - 1];
      int hi = hi0, tp = tr0;
      for (int d = 0; d < nc; d++) {
        const int4 r = drec[d];
        if (r.x != tp) hi = Lr;
        if (pos > r.y && pos <= hi) a = __fadd_rn(a, pos > r.z ? 1.0f : n2v[d * 32 + x]);
        if (r.w && pos <= r.y) a = __fadd_rn(a, 1.0f);
        hi = r.y; tp = r.x;
      }
      acc[pos] = a;
    }
    hi0 = drec[nc - 1].y; tr0 = drec[nc - 1].x;
    __syncthreads();
  }
  if (! last) { if (tid == 0) { O->rtrace = ntr; O->rdom = nseg; } return; }
  for (int pos = tid + 1; pos <= Lr; pos += NT) acc[pos] = logf(__fdiv_rn(acc[pos], (float) nsamples));
  if (tid == 0) { O->rtrace = ntr; O->rdom = nseg; O->done = 1; }
  __syncthreads();
  if (wv != 0) return;                                     // the rest is one wave's work, without barriers
  auto l2_sync = []() { __threadfence(); md_sync(); };     // around counts made by atomics at L2

  // ---------------- 3. clustering ----------------
  // the two stacks of the linkage in LDS; each element's cluster and each
  // cluster's trace count in the region's area
  int *av = (int *) lds, *bv = av + J.segcap;
  int *asg = (int *) (area + md_clu_at(M, Lr, J.segcap)), *ninc = asg + J.segcap;
  unsigned long long *lk = (unsigned long long *) (bv + J.segcap);   // link bits of one pass
  MdSig *sig = (MdSig *) (lk + (J.segcap + 63) / 64);
  const int n = nseg;
  for (int v = z; v < n; v += 64) { av[v] = n - v - 1; ninc[v] = 0; }
  l2_sync();
  int na = n, nb = 0, ncl = 0;
  while (na > 0) {
    na--;
    if (z == 0) bv[nb] = av[na];
    nb++;
    md_sync();
    while (nb > 0) {
      nb--;
      const int v = bv[nb];
      if (z == 0) asg[v] = ncl;
      const MdSeg sv = segs[v];
      const int nw = (na + 63) / 64;
      for (int w = 0; w < nw; w++) {
        const int a = w * 64 + z;
        const bool l = (a < na) && md_linked(sv, segs[av[a]]);
        const unsigned long long m = __ballot(l);
        if (z == 0) lk[w] = m;
      }
      md_sync();
      // the linked slots, highest first: each leaves by taking the top's element
      for (int w = nw - 1; w >= 0; w--) {
        unsigned long long m = lk[w];
        while (m) {
          const int bit = 63 - __clzll((long long) m);
          m &= ~(1ull << bit);
          const int a = w * 64 + bit;
          if (z == 0) { const int we = av[a]; av[a] = av[na - 1]; bv[nb] = we; }
          na--; nb++;
          md_sync();
        }
      }
      md_sync();
    }
    ncl++;
  }
  md_sync();
  // posterior of each cluster: the traces with a member (members of one trace are adjacent)
  for (int h = z; h < n; h += 64) {
    bool first = true;
    for (int h2 = h - 1; h2 >= 0 && segs[h2].idx == segs[h].idx; h2--) if (asg[h2] == asg[h]) first = false;
    if (first) atomicAdd(&ninc[asg[h]], 1);
  }
  l2_sync();
  int nsig = 0;
  for (int c = 0; c < ncl; c++) {
    const int ni = __hip_atomic_load(&ninc[c], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // counted at L2
    if (__fdiv_rn((float) ni, (float) nsamples) < 0.25f) continue;
    int lo[4], hi4[4];
    for (int e = 0; e < 4; e++) { lo[e] = 0x7fffffff; hi4[e] = -1; }
    for (int h = z; h < n; h += 64) if (asg[h] == c) {
      const int v4[4] = { segs[h].i, segs[h].j, segs[h].k, segs[h].m };
      for (int e = 0; e < 4; e++) { lo[e] = min(lo[e], v4[e]); hi4[e] = max(hi4[e], v4[e]); }
    }
    for (int e = 0; e < 4; e++) { lo[e] = -wave_max_i(-lo[e]); hi4[e] = wave_max_i(hi4[e]); }
    const int thr = (int) ceilf(__fmul_rn((float) ni, 0.02f));
    int best[4];
    for (int e = 0; e < 4; e++) {                          // i, j, k, m: leftmost start, rightmost end with support
      const int w = hi4[e] - lo[e] + 1;
      for (int b = z; b < w; b += 64) hist[b] = 0;
      l2_sync();
      for (int h = z; h < n; h += 64) if (asg[h] == c) {
        const int v = (e == 0) ? segs[h].i : (e == 1) ? segs[h].j : (e == 2) ? segs[h].k : segs[h].m;
        atomicAdd(&hist[v - lo[e]], 1);
      }
      l2_sync();
      // the counts were made by atomics at L2: read them there too
      auto hcount = [&](int o) { return __hip_atomic_load(&hist[o], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
      int b = -1;
      const bool up = (e == 0 || e == 2);
      for (int base = 0; base < w && b < 0; base += 64) {
        const int o = up ? base + z : w - 1 - base - z;
        const unsigned long long m = __ballot(o >= 0 && o < w && hcount(o) >= thr);
        if (m) b = up ? base + (int) __ffsll((long long) m) - 1 : w - 1 - base - ((int) __ffsll((long long) m) - 1);
      }
      if (b < 0) {                                         // esl_vec_IArgMax: the first maximum
        int bc = -1, bi = 0x7fffffff;
        for (int o = z; o < w; o += 64) { const int h = hcount(o); if (h > bc) { bc = h; bi = o; } }
        const int mc = wave_max_i(bc);
        b = -wave_max_i(bc == mc ? -bi : -0x7fffffff);
      }
      best[e] = lo[e] + b;
      md_sync();
    }
    if (best[0] > best[1] || best[2] > best[3]) continue;
    if (nsig >= MD_MAXSIG) { status = 5; break; }
    if (z == 0) sig[nsig] = MdSig{ c, best[0], best[1], best[2], best[3], __fdiv_rn((float) ni, (float) nsamples) };
    nsig++;
  }
  md_sync();
  if (status) { if (z == 0) { O->status = status; O->nc = 0; O->nseg = nseg; } return; }
  if (z == 0) {
    for (int a = 1; a < nsig; a++) {                       // start order; equal starts keep their order
      const MdSig v = sig[a];
      int b = a - 1;
      while (b >= 0 && sig[b].i > v.i) { sig[b + 1] = sig[b]; b--; }
      sig[b + 1] = v;
    }
    int dom[MD_MAXSIG];
    for (int d = 0; d < nsig; d++) dom[d] = 0;
    for (int d = 0; d < nsig; d++)
      for (int d2 = d + 1; d2 < nsig; d2++) {
        const int nov = min(sig[d].j, sig[d2].j) - max(sig[d].i, sig[d2].i) + 1;
        if (nov == 0) break;
        const int nn = min(sig[d].j - sig[d].i + 1, sig[d2].j - sig[d2].i + 1);
        if ((double) __fdiv_rn((float) nov, (float) nn) >= 0.8) {
          if (sig[d].prob > sig[d2].prob) dom[d2] = 1; else dom[d] = 1;
        }
      }
    int nc = 0;
    for (int d = 0; d < nsig; d++) {
      if (dom[d]) continue;
      if (nc < MD_MAXC) { O->ci[nc] = sig[d].i; O->cj[nc] = sig[d].j; }
      nc++;
    }
    O->status = (nc > MD_MAXC) ? 5 : 0;
    O->nc = min(nc, MD_MAXC);
    O->nseg = nseg;
  }
}

// LDS of one region's workgroup: the Forward's two rows and D->D odds, the
// replay's odds and counts, or the clustering's stacks
static size_t md_fwd_lds(int M)
{ return (size_t) ((md_stage_t(M) ? md_stage_floats(M) : 0) + md_row_floats(M)) * 4; }
static size_t md_replay_lds(int M, int segcap)
{
  const size_t clu = (size_t) 2 * segcap * 4 + (size_t) (segcap + 63) / 64 * 8 + (size_t) MD_MAXSIG * sizeof(MdSig);
  return std::max((size_t) md_replay_floats(M) * 4, clu);
}
size_t md_lds_bytes(int M, int segcap) { return std::max(md_fwd_lds(M), md_replay_lds(M, segcap)); }

// The traces' cell thresholds of every region (md_thresholds over each cell
// of its finished Forward matrix): a grid of gridDim.x workgroups of
// MD_THR_NT threads per region (blockIdx.y). Every choice a trace can make
// depends only on the finished matrix, so its thresholds are computed first,
// with the same operations p7_StochasticTrace performs at the step
// (md_thresholds); a step is then one draw and one to three comparisons.
// thr[(i, k)]: M's three (B | M | I | D), D's one (M | D), I's one (M | I), as
// the integers a draw is compared with (md_thr_word), and their flags. A pass's
// six-word records go out through LDS, so that the stores of a wave are
// contiguous. The rows' thresholds are k_md_rows'.
#define MD_THR_NT 256
#define MD_THR_CELLS 2                                     // cells per thread per pass
#define MD_THR_LDS_OUT ((size_t) 4 * MD_THR_CELLS * MD_THR_NT * MD_THR_WORDS)
static __host__ __device__ inline size_t md_thr_tl_bytes(int M)      // the staged transitions, when they fit
{
  const size_t b = ((size_t) 10 * (M + 2) * 4 + 7) & ~(size_t) 7;
  return (b + MD_THR_LDS_OUT <= P7G_LDS_MAX) ? b : 0;
}

__global__ __launch_bounds__(MD_THR_NT) void
k_md_thr(const DevProfile p, const MdJob *__restrict__ jobs, float *__restrict__ pool)
{
  const int t = threadIdx.x, NT = MD_THR_NT;
  const MdJob J = jobs[blockIdx.y];
  const int M = p.M, Q = max(2, (M - 1) / 4 + 1), Lr = J.Lr;
  const int TR = p.nrows;
  float *mat = pool + J.area;
  float *xmx = mat + (size_t) (Lr + 1) * 12 * Q;
  extern __shared__ double ldsd[];
  const int TW = M + 2;
  const size_t tlb = md_thr_tl_bytes(M);
  float *tl = (float *) ldsd;
  uint32_t *ob = (uint32_t *) (ldsd + tlb / 8);            // the outgoing words
  if (tlb) {
    for (int c = t; c < 10 * TW; c += NT) tl[c] = md_tv(p, TR + md_trow(c / TW), c % TW);
    __syncthreads();
  }
  auto tv = [&](int row, int k) -> float { return tlb ? tl[row * TW + k] : md_tv(p, TR + md_trow(row), k); };
  enum { T_BM = 0, T_MM, T_IM, T_DM, T_MDS, T_DDS, T_MI, T_II, T_MD, T_DD };
#define CELL(i_, q_, s_, r_) mat[(((size_t) (i_) * Q + (q_)) * 3 + (s_)) * 4 + (r_)]
  uint32_t *thr = (uint32_t *) (pool + J.area + md_thr_at(M, Lr, J.segcap));
  auto cellk = [&](int i, int k, int s) {                  // the cell of model position k (1..4Q) in row i
    const int r = (k - 1 >= Q) + (k - 1 >= 2 * Q) + (k - 1 >= 3 * Q), q = k - 1 - r * Q;
    return CELL(i, q, s, r); };
  // cells c = (i - 1) M + (k - 1): each pass MD_THR_CELLS * NT of them, their
  // matrix values loaded before the threshold arithmetic of any of them
  const int64_t LM = (int64_t) Lr * M;
  constexpr int CU = MD_THR_CELLS;
  // a cell's row and column from the pass's first cell (one 64-bit division
  // per pass) and its offset o < CU * NT: x = r0 + o < M + CU * NT, divided
  // by M through a float reciprocal and corrected by one
  const float invM = 1.0f / (float) M;
  for (int64_t c0 = (int64_t) blockIdx.x * CU * NT; c0 < LM; c0 += (int64_t) gridDim.x * CU * NT) {
    const int a0 = (int) (c0 / M), r0 = (int) (c0 - (int64_t) a0 * M);
    const int olast = (int) min((int64_t) CU * NT - 1, LM - 1 - c0);
    auto rowcol = [&](int o, int &i, int &k) {
      const int x = r0 + o;
      int qd = (int) ((float) x * invM);
      if (qd * M > x) qd--; else if ((qd + 1) * M <= x) qd++;
      i = 1 + a0 + qd; k = 1 + x - qd * M;
    };
    float in[CU][8];
#pragma unroll
    for (int u = 0; u < CU; u++) {
      int i, k;
      rowcol(min(u * NT + t, olast), i, k);
      in[u][0] = xmx[(size_t) (i - 1) * 6 + 3];
      in[u][1] = k > 1 ? cellk(i - 1, k - 1, 0) : 0.0f;
      in[u][2] = k > 1 ? cellk(i - 1, k - 1, 2) : 0.0f;
      in[u][3] = k > 1 ? cellk(i - 1, k - 1, 1) : 0.0f;
      in[u][4] = k > 1 ? cellk(i, k - 1, 0) : 0.0f;
      in[u][5] = k > 1 ? cellk(i, k - 1, 1) : 0.0f;
      in[u][6] = cellk(i - 1, k, 0);
      in[u][7] = cellk(i - 1, k, 2);
    }
#pragma unroll
    for (int u = 0; u < CU; u++) {
      int i, k;
      rowcol(min(u * NT + t, olast), i, k);
      uint32_t *ow = ob + (size_t) (u * NT + t) * MD_THR_WORDS;
      double o[5];
      float v[4];
      v[0] = __fmul_rn(in[u][0], tv(T_BM, k));
      v[1] = __fmul_rn(in[u][1], tv(T_MM, k));
      v[2] = __fmul_rn(in[u][2], tv(T_IM, k));
      v[3] = __fmul_rn(in[u][3], tv(T_DM, k));
      md_thresholds(v, 4, o);
      v[0] = (k > 1) ? __fmul_rn(in[u][4], tv(T_MDS, k)) : 0.0f;
      v[1] = (k > 1) ? __fmul_rn(in[u][5], tv(T_DDS, k)) : 0.0f;
      md_thresholds(v, 2, o + 3);
      v[0] = __fmul_rn(in[u][6], tv(T_MI, k));
      v[1] = __fmul_rn(in[u][7], tv(T_II, k));
      md_thresholds(v, 2, o + 4);
      uint32_t fl = 0u;
#pragma unroll
      for (int a = 0; a < 5; a++) ow[a] = md_thr_word(o[a], a, fl);
      ow[5] = fl | (isnan(o[0]) ? 1u << MD_NAN_M : 0u) | (isnan(o[3]) ? 1u << MD_NAN_D : 0u) | (isnan(o[4]) ? 1u << MD_NAN_I : 0u);
    }
    __syncthreads();
    // the pass's cells are consecutive in row-major order, each row's cells at
    // (i (M + 1) + k) MD_THR_WORDS: the stores run along them
    for (int d = t; d < CU * NT * MD_THR_WORDS; d += NT) {
      const int o = d / MD_THR_WORDS;
      if (o <= olast) {
        int i, k;
        rowcol(o, i, k);
        thr[((size_t) i * (M + 1) + k) * MD_THR_WORDS + (d - o * MD_THR_WORDS)] = ob[d];
      }
    }
    __syncthreads();
  }
#undef CELL
}

// The rows' thresholds of every region: C's (C | E), J's (J | E) and B's
// (N | J), and the E state's running-sum checkpoints (every 64th cell and
// the last, md_ncp per row). One wave per 64 rows (blockIdx.x) of a region
// (blockIdx.y). A row's sum is a chain of 8Q double additions that its lane
// runs; the wave loads the 64 rows' M and D values eight q at a time into
// LDS, so that its loads run along the rows.
__global__ __launch_bounds__(64) void
k_md_rows(const DevProfile p, const MdJob *__restrict__ jobs, float *__restrict__ pool)
{
  const int t = threadIdx.x;
  const MdJob J = jobs[blockIdx.y];
  const int M = p.M, Q = max(2, (M - 1) / 4 + 1), Lr = J.Lr, L = J.Ltarget;
  const int r0 = blockIdx.x * 64;
  if (r0 > Lr) return;
  const float xEmove = p.xfE_move, xEloop = p.xfE_loop, floop = p.xf_loop[L], fmove = p.xf_move[L];
  const float *mat = pool + J.area;
  const float *xmx = mat + (size_t) (Lr + 1) * 12 * Q;
  double *xthr = (double *) (pool + J.area + md_xthr_at(M, Lr, J.segcap));
  double *ecum = (double *) (pool + J.area + md_ecum_at(M, Lr, J.segcap));
  __shared__ float4 tile[64 * 17];                         // [row][q][M, D halves], 17 float4 a row
  const int i = r0 + t;
  const bool row = (i >= 1 && i <= Lr);
  float nf = 0.0f;
  if (i <= Lr) {
    float v[2];
    if (i >= 1) {
      v[0] = __fmul_rn(xmx[(size_t) (i - 1) * 6 + 4], floop);
      v[1] = __fmul_rn(__fmul_rn(xmx[(size_t) i * 6 + 0], xEmove), xmx[(size_t) i * 6 + 5]);
      md_thresholds(v, 2, xthr + (size_t) i * 3 + 0);
      v[0] = __fmul_rn(xmx[(size_t) (i - 1) * 6 + 2], floop);
      v[1] = __fmul_rn(__fmul_rn(xmx[(size_t) i * 6 + 0], xEloop), xmx[(size_t) i * 6 + 5]);
      md_thresholds(v, 2, xthr + (size_t) i * 3 + 1);
      // select_e: norm = 1/E(i) in double, the products in float, summed in double
      nf = (float) (1.0 / (double) xmx[(size_t) i * 6 + 0]);
    }
    v[0] = __fmul_rn(xmx[(size_t) i * 6 + 1], fmove);
    v[1] = __fmul_rn(xmx[(size_t) i * 6 + 2], fmove);
    md_thresholds(v, 2, xthr + (size_t) i * 3 + 2);
  }
  const int NCP = md_ncp(Q);
  double sum = 0.0;
  for (int q0 = 0; q0 < Q; q0 += 8) {
    // lane t loads parts j = t + 64 m: row j / 16, q q0 + (j % 16) / 2, half j % 2
#pragma unroll
    for (int m = 0; m < 16; m++) {
      const int j = t + 64 * m, rw = j >> 4, part = j & 15;
      const int ii = min(r0 + rw, Lr), q = min(q0 + (part >> 1), Q - 1);   // past the ends: a valid cell, unused
      tile[rw * 17 + part] = *(const float4 *) (mat + ((size_t) ii * Q + q) * 12 + (part & 1) * 4);
    }
    __syncthreads();
    if (row) {
#pragma unroll
      for (int a = 0; a < 8; a++)
        if (q0 + a < Q) {
          const float4 x0 = tile[t * 17 + 2 * a], x1 = tile[t * 17 + 2 * a + 1];
          sum = sum + (double) __fmul_rn(x0.x, nf); sum = sum + (double) __fmul_rn(x0.y, nf);
          sum = sum + (double) __fmul_rn(x0.z, nf); sum = sum + (double) __fmul_rn(x0.w, nf);
          sum = sum + (double) __fmul_rn(x1.x, nf); sum = sum + (double) __fmul_rn(x1.y, nf);
          sum = sum + (double) __fmul_rn(x1.z, nf); sum = sum + (double) __fmul_rn(x1.w, nf);
        }
      ecum[(size_t) i * NCP + (q0 >> 3)] = sum;                 // after element min(8 (q0 + 8), 8Q) - 1
    }
    __syncthreads();
  }
}

// floats of one region's area in the pool: matrix, specials, residue sums,
// endpoint counts, the ensemble, the traces' thresholds, the walk's log (and 64
// entries past it, which the replay may read)
int64_t md_area_floats(int M, int Lr, int segcap)
{
  const int64_t f = md_log_at(M, Lr, segcap) + (md_log_entries(M, Lr) + 1) / 2 + 32;
  return (f + 63) & ~(int64_t) 63;
}

hipError_t launch_md_regions(const DevProfile &p, const uint8_t *res, const MdJob *jobs, MdOut *out, int njobs,
                             float *pool, int segcap, int nsamples, uint32_t seed, int max_lr, hipStream_t st,
                             hipEvent_t thr_done)
{
  if (njobs <= 0) return hipSuccess;
  const size_t lds0 = md_fwd_lds(p.M), lds = md_replay_lds(p.M, segcap);
  if (std::max(lds0, lds) > P7G_LDS_MAX) return hipErrorInvalidValue;
  void *kf;
  switch (4 * md_qs(p.M) <= 512 ? (4 * md_qs(p.M) + 63) / 64 : 0) {
    case 1: kf = (void *) k_md_fwd<1>; break;
    case 2: kf = (void *) k_md_fwd<2>; break;
    case 3: case 4: kf = (void *) k_md_fwd<4>; break;
    case 5: case 6: kf = (void *) k_md_fwd<6>; break;
    case 7: case 8: kf = (void *) k_md_fwd<8>; break;
    default: kf = (void *) k_md_fwd<0>; break;
  }
  hipError_t e = hipFuncSetAttribute((const void *) kf, hipFuncAttributeMaxDynamicSharedMemorySize, (int) lds0);
  if (e == hipSuccess) e = hipFuncSetAttribute((const void *) k_md_replay, hipFuncAttributeMaxDynamicSharedMemorySize, (int) lds);
  if (e != hipSuccess) return e;
  // the Forward matrices (one wave per region, the Forward's LDS only), the
  // thresholds (the whole device), then the traces' walks and replays
  {
    void *args[] = { (void *) &p, (void *) &res, (void *) &jobs, (void *) &pool };
    if ((e = hipLaunchKernel(kf, dim3(njobs), dim3(64), args, lds0, st)) != hipSuccess) return e;
  }
  for (int j0 = 0; j0 < njobs; j0 += 65535) {
    const int nj = std::min(njobs - j0, 65535);
    hipLaunchKernelGGL(k_md_thr, dim3(32, nj), dim3(MD_THR_NT), md_thr_tl_bytes(p.M) + MD_THR_LDS_OUT, st, p, jobs + j0, pool);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    hipLaunchKernelGGL(k_md_rows, dim3((max_lr + 1 + 63) / 64, nj), dim3(64), 0, st, p, jobs + j0, pool);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  if (thr_done && (e = hipEventRecord(thr_done, st)) != hipSuccess) return e;
  // as many launches as a region needs whose every trace fills its share of
  // the log: one for M above some 150, and mostly the first does everything
  const int passes = std::max(md_passes(p.M, max_lr, nsamples), md_passes(p.M, 1, nsamples));
  for (int a = 0; a < passes; a++) {
    hipLaunchKernelGGL(k_md_walk, dim3(njobs), dim3(64), 0, st, p, jobs, out, pool, nsamples, seed, (int) (a == 0));
    if ((e = hipGetLastError()) != hipSuccess) return e;
    hipLaunchKernelGGL(k_md_replay, dim3(njobs), dim3(64 * md_replay_waves(p.M)), lds, st, p, res, jobs, out, pool, nsamples);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  return hipSuccess;
}

// Residue copies of the envelopes the clusters define, from their regions'
// copies: one block per envelope, padded to 16 bytes plus 16 with the pad code
// as the region copies are.
__global__ void k_md_copy(uint8_t *__restrict__ res, const int64_t *__restrict__ src, const int64_t *__restrict__ dst,
                          const int32_t *__restrict__ len, int n)
{
  const int e = blockIdx.x;
  if (e >= n) return;
  const int Ld = len[e];
  const int64_t need = (((int64_t) Ld + 15) & ~(int64_t) 15) + 16;
  for (int64_t b = threadIdx.x; b < need; b += blockDim.x)
    res[dst[e] + b] = (b < Ld) ? res[src[e] + b] : (uint8_t) P7G_PADCODE;
}

// The regions' residue null2 scores (their areas' residues 1..Lr), gathered
// in job order for one copy to the host: one workgroup per region.
__global__ void k_md_n2_gather(const MdJob *__restrict__ jobs, const float *__restrict__ pool, int M,
                               float *__restrict__ dst)
{
  const MdJob J = jobs[blockIdx.x];
  const float *src = pool + J.area + md_n2sc_at(M, J.Lr) + 1;
  for (int i = threadIdx.x; i < J.Lr; i += blockDim.x) dst[(size_t) J.n2o + i] = src[i];
}

hipError_t launch_md_n2_gather(const MdJob *jobs, int njobs, const float *pool, int M, float *dst, hipStream_t st)
{
  if (njobs <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_md_n2_gather, dim3(njobs), dim3(256), 0, st, jobs, pool, M, dst);
  return hipGetLastError();
}

hipError_t launch_md_copy(uint8_t *res, const int64_t *src, const int64_t *dst, const int32_t *len, int n, hipStream_t st)
{
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_md_copy, dim3(n), dim3(256), 0, st, res, src, dst, len, n);
  return hipGetLastError();
}
