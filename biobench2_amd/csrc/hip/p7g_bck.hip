// gfx950 kernels of the Backward parser (HMMER/src/impl_sse/fwdback.c:238-256,
// 470-735), with Forward's scale factors.
#include "p7g_list.h"

/*****************************************************************
 * 8. Backward parser (one target per wave), with Forward's scale factors
 *****************************************************************/
// MODE 0: the parser. MODE 1: the special-state rows also go to the caller's
// matrix (one target) or to the domain decoding pool (a separate instance, so
// that the plain parser keeps its register budget). MODE 2: envelopes.
// At B <= 2 six waves per SIMD (80 registers) leave room for a third workgroup.
template <int B, int TM, int MODE>
__global__ __launch_bounds__(BCK_THREADS(B)) __attribute__((amdgpu_waves_per_eu((B) <= 2 ? 6 : (B) <= 7 ? 4 : 1)))
void k_bck(const DevProfile p, const uint8_t *__restrict__ res, const int64_t *__restrict__ off,
           const int32_t *__restrict__ len, const int32_t *__restrict__ list, const int32_t *__restrict__ count,
           DevResults r, const float *__restrict__ pool, const int64_t *__restrict__ scale_off,
           const float *__restrict__ fwd_xmx, float *__restrict__ xmx_out, LenCfg lc, DomBufs dom, DevLists l)
{
  constexpr bool PIN = (TM == TM_LDS || TM == TM_PIN);
  const int lw = list_waves(*count);
  if ((int64_t) blockIdx.x * lw >= *count) return;
  extern __shared__ float ldsf[];
  const size_t rowf = (size_t) 64 * B;
  const float *tbl = p.fb_tbl;                           // emission rows
  if (TM == TM_LDS) { stage_table(ldsf, p.fb_tbl, p.fb_floats); tbl = ldsf; }
  if (TM == TM_TLDS) stage_table(ldsf, p.fb_tbl + (size_t) p.nrows * rowf, (size_t) P7G_FB_NT * rowf);
  const int z = threadIdx.x & 63;
  const float *tr = ((TM == TM_TLDS) ? ldsf : tbl + (size_t) p.nrows * rowf) + z;
  float tBM[B], tMMN[B], tIMN[B], tDMN[B], tMD[B], tDD[B], tMI[B], tII[B];
  if (PIN) {
#pragma unroll
    for (int j = 0; j < B; j++) {
      tBM[j] = tr[VT_BM*rowf + j*64]; tMMN[j] = tr[FT_MMN*rowf + j*64]; tIMN[j] = tr[FT_IMN*rowf + j*64]; tDMN[j] = tr[FT_DMN*rowf + j*64];
      tMD[j] = tr[FT_MD*rowf + j*64]; tDD[j] = tr[FT_DD*rowf + j*64]; tMI[j] = tr[VT_MI*rowf + j*64]; tII[j] = tr[VT_II*rowf + j*64];
    }
  }
  AffConst akc;
  {
    float tdd[B];
#pragma unroll
    for (int j = 0; j < B; j++) tdd[j] = tr[FT_DD*rowf + j*64];
    aff_bck_setup<B>(akc, tdd);
  }
#define BTR(A, T, j) (PIN ? A[j] : trr[(T) * rowf + (j) * 64])
  constexpr bool DOM = (MODE == 1), ENV = (MODE == 2), STREAM = (TM == TM_GLOB), PF = ! STREAM;
  // which product of I's and M's update is rounded first (as FP in k_fwd: the order
  // each size was first compiled with, the same in every mode)
  constexpr bool FI = (B == 1 || (B >= 6 && B <= 8)), FM = (B == 1 || (B >= 7 && B <= 8));
  const int64_t n = ENV ? min((int64_t) *count, dom.env_cap) : (int64_t) *count;
  const float eMove = ENV ? 1.0f : p.xfE_move, eLoop = ENV ? 0.0f : p.xfE_loop;

  int32_t *queue = (int32_t *) count + P7G_QOFF;
  if ((int) (threadIdx.x >> 6) >= lw) return;
  for (int64_t t = queue_next(queue, 1); t < n; t = queue_next(queue, 1)) {
    const int slot = uni(list[t]);
    const int L = uni(len[slot]);
    const uint8_t *sq = res + off[slot];
    const float floop = ENV ? dom.env_loop[slot] : lc.on ? lc.floop : p.xf_loop[L];
    const float fmove = ENV ? dom.env_move[slot] : lc.on ? lc.fmove : p.xf_move[L];
    const float *fsc = nullptr;       // forward row scale factors, fsc[i], i = 0..L
    int fstride = 1;
    float *cells = nullptr;           // envelope Backward for null2: its M and I rows
    float *xo = xmx_out;
    if (ENV) {
      const int64_t so = dom.n2soff[slot];
      if (so < 0) {                   // the envelope-score pass found no room for its scales
        if (z == 0) { r.bcksc[slot] = NAN; r.fstatus[slot] = 5; }
        continue;
      }
      fsc = dom.n2scl + (((int64_t) (unsigned) uni((int) (so >> 32)) << 32) | (unsigned) uni((int) so));
      const int64_t o = dom.n2off[slot];
      float *area = dom.n2pool + (((int64_t) (unsigned) uni((int) (o >> 32)) << 32) | (unsigned) uni((int) o));
      xo = area;
      cells = xo + n2_xrows_floats(L) + z;
    } else if (fwd_xmx) { fsc = fwd_xmx + 5; fstride = 6; }
    else {
      const int64_t so = scale_off[slot];
      if (so < 0) {
        if (z == 0) { r.bcksc[slot] = NAN; r.fstatus[slot] = 5; }
        continue;
      }
      fsc = pool + so;
    }
    // the special-state rows: the caller's matrix (one target), or the
    // target's decoding entry that the Forward parser reserved
    if (DOM && dom.pool) {
      const int64_t bo = dom.boff[slot];
      const int64_t bu = ((int64_t) (unsigned) uni((int) (bo >> 32)) << 32) | (unsigned) uni((int) bo);
      xo = (bu >= 0) ? dom.pool + bu : nullptr;
    }
    float M[B], I[B], D[B];
    float xJ = 0.0f, xB = 0.0f, xN = 0.0f;
    float xC = fmove;
    float xE = xC * eMove;
#pragma unroll
    for (int j = 0; j < B; j++) { M[j] = xE; D[j] = xE; I[j] = 0.0f; }
    {
      const float *trr = tr + (PIN ? 0 : opaque_zero());
      affine_bck_scan<B>(D, [&](int j) { return BTR(tDD, FT_DD, j); }, akc);
      const float dS = dppz<WAVE_SHL1>(D[0]);
#pragma unroll
      for (int j = 0; j < B; j++) M[j] = M[j] + (j < B-1 ? D[j+1] : dS) * BTR(tMD, FT_MD, j);
    }
    int own = 0;
    float totscale;
    {
      const float s = fsc[(size_t) L * fstride];
      if (s > 1.0f) {
        xE = xE / s; xN = xN / s; xC = xC / s; xJ = xJ / s; xB = xB / s;
        const float inv = (float) (1.0 / (double) s);
#pragma unroll
        for (int j = 0; j < B; j++) { M[j] *= inv; D[j] *= inv; I[j] *= inv; }
      }
      totscale = (float) log((double) s);
      if (xo && z == 0) {
        float *xr = xo + (size_t) L * 6;
        xr[0] = xE; xr[1] = xN; xr[2] = xJ; xr[3] = xB; xr[4] = xC; xr[5] = s;
      }
      if (ENV && L > 0) {
        float *cr = cells + (size_t) (L-1) * 2 * rowf;
#pragma unroll
        for (int j = 0; j < B; j++) { cr[j*64] = M[j]; cr[rowf + j*64] = I[j]; }
      }
    }
    // One row, as in k_fwd: the emission odds come a row ahead (PF), Forward's
    // scale factors and the residues 64 rows at a time, and the row's specials
    // leave 64 rows at a time. A row of one target alone, M = 20 | 86 | 400 |
    // 803: 188 | 195 | 301 | 499 ns (before 422 | 455 | 525 | 740 ns).
    float bE = 0.0f, bN = 0.0f, bJ = 0.0f, bB = 0.0f, bC = 0.0f, bS = 0.0f;
    float e[B];
    auto row = [&](int xoff, int xnext, int fsbits, int i, int u) {
      const float *er = tbl + xoff + z;
      const float *trr = tr + (PIN ? 0 : opaque_zero());
      float xBl = 0.0f;
      if constexpr (STREAM) {
        // M(j) * e(j), its share of the B sum, then the update
        stream_tables<B, 2, 32, false>({ er, trr + VT_BM*rowf }, [&](int j, const float (&x)[2]) {
          M[j] = M[j] * x[0];
          xBl = __builtin_fmaf(M[j], x[1], xBl); });
        const float mS = dppz<WAVE_SHL1>(M[0]);
        stream_tables<B, 4, 16, false>({ trr + VT_II*rowf, trr + FT_IMN*rowf, trr + VT_MI*rowf, trr + FT_MMN*rowf },
                                       [&](int j, const float (&x)[4]) {
          const float ms = (j < B-1) ? M[j < B-1 ? j+1 : 0] : mS, ip = I[j];
          I[j] = fma2<FI>(ip, x[0], ms, x[1]);
          D[j] = ms;
          M[j] = fma2<FM>(ip, x[2], ms, x[3]); });
      } else {
        // mn(j) = M(j) * e(j), formed one position ahead of the update that
        // overwrites M(j); xBl sums mn(j) * tBM(j) in increasing j
        const float mn = M[0] * e[0];
        xBl = __builtin_fmaf(mn, BTR(tBM, VT_BM, 0), xBl);
        const float mS = dppz<WAVE_SHL1>(mn);
#pragma unroll
        for (int j = 0; j < B; j++) {
          float ms = mS;
          if (j < B-1) { ms = M[j+1] * e[j+1]; xBl = __builtin_fmaf(ms, BTR(tBM, VT_BM, j+1), xBl); }
          const float ip = I[j];
          M[j] = fma2<FM>(ip, BTR(tMI, VT_MI, j), ms, BTR(tMMN, FT_MMN, j));   // before I: ip in place, no copy
          if (FI || ! PIN) I[j] = fma2<FI>(ip, BTR(tII, VT_II, j), ms, BTR(tIMN, FT_IMN, j));
          else fma_onto(I[j], BTR(tII, VT_II, j), ms * BTR(tIMN, FT_IMN, j));
          D[j] = ms;
        }
        const float *el = tbl + xnext + z;
#pragma unroll
        for (int j = 0; j < B; j++) e[j] = el[j * 64];
      }
      xB = wave_sum_f(xBl);
      xC = xC * floop;
      xJ = fma2<true>(xB, fmove, xJ, floop);
      xN = fma2<true>(xB, fmove, xN, floop);
      xE = fma2<false>(xC, eMove, xJ, eLoop);
      if constexpr (STREAM) {
        float C = 0.0f, mdl = 0.0f;
        stream_tables<B, 2, 32, true>({ trr + FT_DMN*rowf, trr + FT_DD*rowf }, [&](int j, const float (&x)[2]) {
          D[j] = __builtin_fmaf(D[j], x[0], xE);
          C = (j == B-1) ? D[j] : __builtin_fmaf(x[1], C, D[j]); });
        float cur = lane_carry_bck(C, akc);
        stream_tables<B, 2, 32, true>({ trr + FT_DD*rowf, trr + FT_MD*rowf }, [&](int j, const float (&x)[2]) {
          if (j < B-1) M[j] = __builtin_fmaf(D[j < B-1 ? j+1 : 0], x[1], M[j] + xE);
          else mdl = x[1];
          D[j] = cur = __builtin_fmaf(x[0], cur, D[j]); });
        M[B-1] = __builtin_fmaf(dppz<WAVE_SHL1>(D[0]), mdl, M[B-1] + xE);
      } else {
#pragma unroll
        for (int j = 0; j < B; j++) D[j] = __builtin_fmaf(D[j], BTR(tDMN, FT_DMN, j), xE);
        affine_bck_scan<B>(D, [&](int j) { return BTR(tDD, FT_DD, j); }, akc);
        const float dS = dppz<WAVE_SHL1>(D[0]);
#pragma unroll
        for (int j = 0; j < B; j++) M[j] = __builtin_fmaf(j < B-1 ? D[j+1] : dS, BTR(tMD, FT_MD, j), M[j] + xE);
      }
      // the row's scale: Forward's, or its own; bits in scalar registers
      const int xBbits = uni(__float_as_int(xB));
      if (gt_bits(xBbits, BITS_1E16)) own = 1;
      if (own) fsbits = gt_bits(xBbits, BITS_1E4) ? xBbits : BITS_ONE;
      const float fs = __int_as_float(fsbits);
      if (gt_bits(fsbits, BITS_ONE)) {
        const float s = fs;
        xE /= s; xN /= s; xJ /= s; xB /= s; xC /= s;
        const float inv = (float) (1.0 / (double) s);
#pragma unroll
        for (int j = 0; j < B; j++) { M[j] *= inv; D[j] *= inv; I[j] *= inv; }
        if (MODE == 0) bS = (z == u) ? s : bS;
      }
      if (MODE != 0) {
        const bool me = (z == u);
        bE = me ? xE : bE; bN = me ? xN : bN; bJ = me ? xJ : bJ; bB = me ? xB : bB; bC = me ? xC : bC;
        bS = me ? fs : bS;
      }
      if (ENV) {
        float *cr = cells + (size_t) (i-1) * 2 * rowf;
#pragma unroll
        for (int j = 0; j < B; j++) { cr[j*64] = M[j]; cr[rowf + j*64] = I[j]; }
      }
    };
    int xoff = P7G_PADCODE * (int) rowf;                 // the step's emission row
    if (L > 0) {
      RowRes<true> rr;
      xoff = rr.init(sq, L, z, (int) rowf);
      if (PF) {
#pragma unroll
        for (int j = 0; j < B; j++) e[j] = tbl[xoff + z + j * 64];
      }
      // Forward's scale factors of the block's rows: lane u holds row L-1-s0-u's
      auto scales = [&](int s0) { return fsc[(size_t) max(L - 1 - s0 - z, 0) * fstride]; };
      float sc0 = scales(0), sc1 = scales(64);
      for (int s0 = 0; s0 < L - 1; s0 += 64) {
        const int cnt = uni(min(64, L - 1 - s0)), i0 = L - 1 - s0;
        bS = 1.0f;
        for (int u = 0; u < cnt; u++) {
          const int xnext = rr.ahead(u);
          row(xoff, xnext, __builtin_amdgcn_readlane(__float_as_int(sc0), u), i0 - u, u);
          xoff = xnext;
        }
        add_scales(totscale, bS);
        if (MODE != 0 && xo && z < cnt) {
          float *xr = xo + (size_t) (i0 - z) * 6;
          xr[0] = bE; xr[1] = bN; xr[2] = bJ; xr[3] = bB; xr[4] = bC; xr[5] = bS;
        }
        rr.advance();
        sc0 = sc1; sc1 = scales(s0 + 128);
      }
    }
    {
      const float *e = tbl + xoff + z;
      const float *trr = tr + (PIN ? 0 : opaque_zero());
      float xBl = 0.0f;
#pragma unroll
      for (int j = 0; j < B; j++) xBl += (M[j] * e[j * 64]) * BTR(tBM, VT_BM, j);
      xB = unif(wave_sum_f(xBl));
      xN = (xB * fmove) + (xN * floop);
    }
    if (z == 0) {
      if (xo) {
        xo[0] = 0.0f; xo[1] = xN; xo[2] = 0.0f; xo[3] = xB; xo[4] = 0.0f; xo[5] = 1.0f;
      }
      int status = 0;
      float sc;
      if (isnan(xN) || (L > 0 && xN == 0.0f) || isinf(xN)) { status = 16; sc = NAN; }
      else sc = (float) ((double) totscale + log((double) xN));
      r.bcksc[slot] = sc;
      r.fstatus[slot] = status | (own ? 0x100 : 0);
    }
  }
}
#undef BTR

// Backward parser for large models, W waves per target: the slices of
// k_fwd_wg, traversed the other way. The D->D chain runs towards smaller k
// (slice constants, lanes composed from their last slice, scanned across lanes
// from lane 63 down). A row takes two barriers: one for the slices' chain
// constants, one for the waves' parts of the B sum and the slices' first M; the
// next slice's D at its first position is the chain's carry into this one, and
// every wave updates the special states by itself.
// Bound by the row's chain of dependent steps; M = 2600 (B = 48, W = 4): 761 ns
// a row, where four barriers and odds loaded in the row made it 1250 ns.
__device__ __forceinline__ void aff_setup_lane_bck(AffConst &k, float P)
{
  k.w1 = P; P = P * dppf<ROW_SHL1>(1.0f, P);
  k.w2 = P; P = P * dppf<ROW_SHL2>(1.0f, P);
  k.w4 = P; P = P * dppf<ROW_SHL4>(1.0f, P);
  k.w8 = P; P = P * dppf<ROW_SHL8>(1.0f, P);
  k.prow = P; k.pa = readlanef(P, 32); k.pb = readlanef(P, 16);
}

// ROWS: the special-state rows go to the caller's matrix (one target), and
// Forward's scale factors come from its matrix.
template <int B, int W, bool ROWS>
__global__ __launch_bounds__(64 * W)
void k_bck_wg(const DevProfile p, const uint8_t *__restrict__ res, const int64_t *__restrict__ off,
              const int32_t *__restrict__ len, const int32_t *__restrict__ list, const int32_t *__restrict__ count,
              DevResults r, const float *__restrict__ pool, const int64_t *__restrict__ scale_off, LenCfg lc,
              const float *__restrict__ fwd_xmx, float *__restrict__ xmx_out)
{
  static_assert(B % W == 0, "slices of equal width");
  constexpr int BW = B / W;
  __shared__ float sh_m0[W][65];     // M at each slice's first position (lane 64: none, for the last slice)
  __shared__ float sh_c[W][64];      // the slices' D-chain constants
  __shared__ float sh_x[W];          // the waves' parts of the B sum
  __shared__ int64_t sh_t;
  if ((int64_t) blockIdx.x >= *count) return;
  const int wv = threadIdx.x >> 6, z = threadIdx.x & 63;
  const int j0 = wv * BW;
  const size_t rowf = (size_t) 64 * B;
  const float *tbl = p.fb_tbl;
  const float *tr = tbl + (size_t) p.nrows * rowf + z;
  float tBM[BW], tMMN[BW], tIMN[BW], tDMN[BW], tMD[BW], tDD[BW], tMI[BW], tII[BW];
#pragma unroll
  for (int j = 0; j < BW; j++) {
    const size_t c = (size_t) (j0 + j) * 64;
    tBM[j] = tr[VT_BM*rowf + c]; tMMN[j] = tr[FT_MMN*rowf + c]; tIMN[j] = tr[FT_IMN*rowf + c]; tDMN[j] = tr[FT_DMN*rowf + c];
    tMD[j] = tr[FT_MD*rowf + c]; tDD[j] = tr[FT_DD*rowf + c]; tMI[j] = tr[VT_MI*rowf + c]; tII[j] = tr[VT_II*rowf + c];
  }
  // the position after the slice's last one: the next slice's first (for the
  // last slice the next lane's)
  const bool none = (wv == W-1 && z == 63);
  const int hoff = none ? 0 : (wv < W-1) ? (j0 + BW) * 64 : 1;
  const int nw = (wv < W-1) ? wv + 1 : 0, nz = (wv < W-1) ? z : z + 1;     // where its M is in sh_m0
  float Pv[W];
#pragma unroll
  for (int v = 0; v < W; v++) {
    float P = 1.0f;
    for (int j = BW-1; j >= 0; j--) P *= tr[FT_DD*rowf + (size_t) (v * BW + j) * 64];
    Pv[v] = P;
  }
  AffConst akl;
  {
    float P = 1.0f;
#pragma unroll
    for (int v = W-1; v >= 0; v--) P *= Pv[v];
    aff_setup_lane_bck(akl, P);
  }
  if (threadIdx.x < W) sh_m0[threadIdx.x][64] = 0.0f;
  const int64_t n = *count;
  int32_t *queue = (int32_t *) count + P7G_QOFF;

  // the D->D chain of the row in D (towards smaller k), then M += (D of the
  // next position) * tMD; one barrier. The chain's carry into a slice is D at
  // the next slice's first position.
  auto dchain_and_m = [&](float (&M)[BW], float (&D)[BW], float add) {
    {
      float C = 0.0f;
#pragma unroll
      for (int j = BW-1; j >= 0; j--) C = __builtin_fmaf(tDD[j], C, D[j]);
      sh_c[wv][z] = C;
    }
    lds_barrier();
    float cv[W];
#pragma unroll
    for (int v = 0; v < W; v++) cv[v] = sh_c[v][z];
    float Cl = 0.0f;
#pragma unroll
    for (int v = W-1; v >= 0; v--) Cl = __builtin_fmaf(Pv[v], Cl, cv[v]);
    float c = lane_carry_bck(Cl, akl);
#pragma unroll
    for (int v = W-1; v > 0; v--) if (v > wv) c = __builtin_fmaf(Pv[v], c, cv[v]);
    float cur = c;
#pragma unroll
    for (int j = BW-1; j >= 0; j--) { cur = __builtin_fmaf(tDD[j], cur, D[j]); D[j] = cur; }
#pragma unroll
    for (int j = 0; j < BW; j++) M[j] = __builtin_fmaf(j < BW-1 ? D[j+1] : c, tMD[j], M[j] + add);
  };

  for (;;) {
    if (threadIdx.x == 0) sh_t = (int64_t) atomicAdd(queue, 1);
    __syncthreads();
    const int64_t t = sh_t;
    if (t >= n) break;
    const int slot = list[t];
    const int L = len[slot];
    const uint8_t *sq = res + off[slot];
    const float floop = lc.on ? lc.floop : p.xf_loop[L], fmove = lc.on ? lc.fmove : p.xf_move[L];
    const float *fsc;
    constexpr int fstride = ROWS ? 6 : 1;
    if (ROWS) fsc = fwd_xmx + 5;
    else {
      const int64_t so = scale_off[slot];
      if (so < 0) {
        if (threadIdx.x == 0) { r.bcksc[slot] = NAN; r.fstatus[slot] = 5; }
        __syncthreads();
        continue;
      }
      fsc = pool + so;
    }
    float M[BW], I[BW], D[BW];
    float xJ = 0.0f, xB = 0.0f, xN = 0.0f;
    float xC = fmove;
    float xE = xC * p.xfE_move;
#pragma unroll
    for (int j = 0; j < BW; j++) { M[j] = xE; D[j] = xE; I[j] = 0.0f; }
    dchain_and_m(M, D, 0.0f);
    int own = 0;
    float totscale;
    {
      const float s = fsc[(size_t) L * fstride];
      if (s > 1.0f) {
        xE = xE / s; xN = xN / s; xC = xC / s; xJ = xJ / s; xB = xB / s;
        const float inv = (float) (1.0 / (double) s);
#pragma unroll
        for (int j = 0; j < BW; j++) { M[j] *= inv; D[j] *= inv; I[j] *= inv; }
      }
      totscale = (float) log((double) s);
      if (ROWS && threadIdx.x == 0) {
        float *xr = xmx_out + (size_t) L * 6;
        xr[0] = xE; xr[1] = xN; xr[2] = xJ; xr[3] = xB; xr[4] = xC; xr[5] = s;
      }
    }
    // a row's odds (the slice's and the next position's) and its share of the B
    // sum, M(j) * e(j) * tBM(j) in increasing j
    float e[BW], eh;
    auto odds = [&](int xo) {
      const float *q = tbl + xo + z;
#pragma unroll
      for (int j = 0; j < BW; j++) e[j] = q[(size_t) (j0 + j) * 64];
      eh = q[hoff];
    };
    auto bsum = [&]() {
      float xBl = 0.0f;
#pragma unroll
      for (int j = 0; j < BW; j++) { M[j] = M[j] * e[j]; xBl = __builtin_fmaf(M[j], tBM[j], xBl); }
      const float ws = wave_sum_f(xBl);
      if (z == 0) sh_x[wv] = ws;
      lds_barrier();                                    // the parts (and the slices' first M) are written
      xB = 0.0f;
#pragma unroll
      for (int v = 0; v < W; v++) xB += sh_x[v];
    };
    int xlast = P7G_PADCODE * (int) rowf;
    if (L > 0) {
      RowRes<true> rr;
      xlast = rr.init(sq, L, z, (int) rowf);
      odds(xlast);
      auto scales = [&](int s0) { return fsc[(size_t) max(L - 1 - s0 - z, 0) * fstride]; };
      float sc0 = scales(0), sc1 = scales(64);
      float bE = 0.0f, bN = 0.0f, bJ = 0.0f, bB = 0.0f, bC = 0.0f, bS = 0.0f;
      for (int s0 = 0; s0 < L - 1; s0 += 64) {
        const int cnt = min(64, L - 1 - s0), i0 = L - 1 - s0;
        for (int u = 0; u < cnt; u++) {
          xlast = rr.ahead(u);
          float fs = readlanef(sc0, u);
          sh_m0[wv][z] = M[0];
          const float eh1 = eh;
          bsum();                                       // M now holds M * e
          const float mS = none ? 0.0f : sh_m0[nw][nz] * eh1;
          odds(xlast);
#pragma unroll
          for (int j = 0; j < BW; j++) {
            const float ms = (j < BW-1) ? M[j+1] : mS;
            const float ip = I[j];
            I[j] = fma2<false>(ip, tII[j], ms, tIMN[j]);
            D[j] = ms;
            M[j] = fma2<false>(ip, tMI[j], ms, tMMN[j]);
          }
          xC = xC * floop;
          xJ = fma2<true>(xB, fmove, xJ, floop);
          xN = fma2<true>(xB, fmove, xN, floop);
          xE = fma2<false>(xC, p.xfE_move, xJ, p.xfE_loop);
#pragma unroll
          for (int j = 0; j < BW; j++) D[j] = __builtin_fmaf(D[j], tDMN[j], xE);
          dchain_and_m(M, D, xE);
          if (gt_bits(uni(__float_as_int(xB)), BITS_1E16)) own = 1;
          if (__builtin_expect(own, 0)) fs = (xB > 1.0e4f) ? xB : 1.0f;
          if (gt_bits(uni(__float_as_int(fs)), BITS_ONE)) {
            const float s = fs;
            xE /= s; xN /= s; xJ /= s; xB /= s; xC /= s;
            const float inv = (float) (1.0 / (double) s);
#pragma unroll
            for (int j = 0; j < BW; j++) { M[j] *= inv; D[j] *= inv; I[j] *= inv; }
            totscale = (float) ((double) totscale + log((double) s));
          }
          if (ROWS) {
            const bool me = (z == u);
            bE = me ? xE : bE; bN = me ? xN : bN; bJ = me ? xJ : bJ; bB = me ? xB : bB; bC = me ? xC : bC;
            bS = me ? fs : bS;
          }
        }
        if (ROWS && wv == 0 && z < cnt) {
          float *xr = xmx_out + (size_t) (i0 - z) * 6;
          xr[0] = bE; xr[1] = bN; xr[2] = bJ; xr[3] = bB; xr[4] = bC; xr[5] = bS;
        }
        rr.advance();
        sc0 = sc1; sc1 = scales(s0 + 128);
      }
    } else odds(xlast);
    bsum();
    xN = (xB * fmove) + (xN * floop);
    if (threadIdx.x == 0) {
      if (ROWS) {
        xmx_out[0] = 0.0f; xmx_out[1] = xN; xmx_out[2] = 0.0f; xmx_out[3] = xB; xmx_out[4] = 0.0f; xmx_out[5] = 1.0f;
      }
      int status = 0;
      float sc;
      if (isnan(xN) || (L > 0 && xN == 0.0f) || isinf(xN)) { status = 16; sc = NAN; }
      else sc = (float) ((double) totscale + log((double) xN));
      r.bcksc[slot] = sc;
      r.fstatus[slot] = status | (own ? 0x100 : 0);
    }
    __syncthreads();                                    // the target is done before the next one is taken
  }
}

// the parser that keeps no rows; from B = 16 on k_bck_wg takes these calls
template <int B, int TM> static void *bck_plain()
{
  if constexpr (B < 16) return (void *) k_bck<B, TM, 0>;
  else return nullptr;
}
#define BCK_CASE(N, T) case N * 4 + T: k = dom.env_loop ? (void *) k_bck<N, T, 2> : (dom.pool || xmx_out) ? (void *) k_bck<N, T, 1> \
                                          : bck_plain<N, T>(); nthr = BCK_THREADS(N); break;

#define BCK_WG_CASE(N, W) case N: kw = xmx_out ? (void *) k_bck_wg<N, W, true> : (void *) k_bck_wg<N, W, false>; ww = W; break;
hipError_t launch_bck(const DevProfile &p, const DevSeqs &s, const int32_t *list, const int32_t *count, int64_t maxn,
                      DevResults r, const float *scale_pool, const int64_t *scale_off, const float *fwd_xmx,
                      float *xmx_out, LenCfg lc, hipStream_t st, const DomBufs &dom, DevLists l)
{
  if (maxn <= 0) return hipSuccess;
  // large models run the parser with several waves per target, as Forward does
  // (a single target's row of M = 1000 | 2600: 528 | 761 ns, one wave 922 | 3267 ns)
  void *kw = nullptr;
  int ww = 0;
  if (! dom.pool && ! dom.env_loop) {
    switch (p.fb_B) {
      BCK_WG_CASE(16, 4)
      BCK_WG_CASE(20, 4)
      BCK_WG_CASE(24, 4)
      BCK_WG_CASE(28, 4)
      BCK_WG_CASE(32, 4)
      BCK_WG_CASE(40, 4)
      BCK_WG_CASE(48, 4)
      BCK_WG_CASE(64, 8)
      BCK_WG_CASE(80, 8)
      default: break;
    }
  }
  if (kw) {
    const unsigned grid = grid_for_waves_blk(kw, maxn * ww, 0, ww);
    void *args[] = { (void *) &p, (void *) &s.res, (void *) &s.off, (void *) &s.len, (void *) &list, (void *) &count,
                     &r, (void *) &scale_pool, (void *) &scale_off, &lc, (void *) &fwd_xmx, &xmx_out };
    return launch(kw, grid, 64 * ww, args, 0, st);
  }
  const int tm = fb_mode(p);
  void *k = nullptr;
  int nthr = LIST_BLOCK;
  switch (p.fb_B * 4 + tm) {
    FB_CASES(BCK_CASE)
    default: return hipErrorInvalidValue;
  }
  if (! k) return hipErrorInvalidValue;
  const size_t lds = fb_lds(p, tm);
  const unsigned grid = list_grid(k, maxn, lds, nthr / 64);
  void *args[] = { (void *) &p, (void *) &s.res, (void *) &s.off, (void *) &s.len, (void *) &list, (void *) &count,
                   &r, (void *) &scale_pool, (void *) &scale_off, (void *) &fwd_xmx, &xmx_out, &lc, (void *) &dom, &l };
  return launch(k, grid, nthr, args, lds, st);
}

