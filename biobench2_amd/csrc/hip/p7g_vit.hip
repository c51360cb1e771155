// gfx950 kernels of the Viterbi filter (HMMER/src/impl_sse/vitfilter.c:84-249):
// int16 pairs with v_pk_add_i16 clamp = _mm_adds_epi16 and v_pk_max_i16 =
// _mm_max_epi16. The D->D closure of a row is a max-plus prefix scan across the
// wave. Where the profile's ddbound bounds every D->D path (vf_free, as the
// conversion sets it) each row is closed; else the lazy-F condition
// (Dmax + ddbound > xB) is evaluated per row exactly as the reference does.
#include "p7g_list.h"

/*****************************************************************
 * 6. Viterbi filter (one target per wave, 64 lanes, int16 pairs)
 *****************************************************************/
// D->D closure of one Viterbi row: D(k) = max(D0(k), D(k-1) + tDD(k-1)).
// Every tDD <= 0 and the int16 floor at -32768 absorbs, so a saturating chain
// equals the int32 maximum over paths floored at -32768. Inside a lane both
// halves run as packed int16 chains; across lanes the lane maps
// x -> max(C, x + A) are composed by an int32 max-plus scan whose window sums
// depend only on the profile and are set up once per kernel.
template <int ND>
struct DDConst {
  int t[ND];                   // tDD pairs: position d (low half), position d+ND (high half)
  int alo, ahi;                // int32 sums of the two halves
  int k1, k2, k4, k8;          // row-scan window sums; -2^28 where the step has no source lane
  int arow;                    // sum of lane totals from the row start to this lane
  int arow31, arow47;          // the same at lanes 31 and 47 (wave-uniform)
  int send;                    // sum of lane totals from lane 0 to this lane
};

template <int ND>
__device__ __forceinline__ void dd_setup(DDConst<ND> &c, const int *__restrict__ tdd, int z)
{
  const int NEG = -(1 << 28);
  int alo = 0, ahi = 0;
#pragma unroll
  for (int d = 0; d < ND; d++) { c.t[d] = tdd[d * 64]; alo += lo16(c.t[d]); ahi += hi16(c.t[d]); }
  c.alo = alo; c.ahi = ahi;
  const int r = z & 15;
  int pre = alo + ahi;                      // inclusive prefix over the lanes of this row
#pragma unroll
  for (int s = 1; s < 16; s <<= 1) { const int v = __shfl_up(pre, s, 16); if (r >= s) pre += v; }
  auto back = [&](int s) { const int v = __shfl_up(pre, s, 16); return (r >= s) ? pre - v : NEG; };
  c.k1 = back(1); c.k2 = back(2); c.k4 = back(4); c.k8 = back(8);
  c.arow = pre;
  c.arow31 = __builtin_amdgcn_readlane(pre, 31);
  c.arow47 = __builtin_amdgcn_readlane(pre, 47);
  const int r0 = __builtin_amdgcn_readlane(pre, 15), r1 = c.arow31, r2 = c.arow47;
  c.send = pre + (z >= 16 ? r0 : 0) + (z >= 32 ? r1 : 0) + (z >= 48 ? r2 : 0);
}

template <int CTRL>
__device__ __forceinline__ int dpp0(int v) { return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xf, 0xf, true); }

template <int ND>
__device__ __forceinline__ void dd_closure(int (&D)[ND], const DDConst<ND> &c, int z)
{
  const int NEG = -(1 << 28);
  // chains inside the lane, no carry in
  int P[ND];
  P[0] = D[0];
#pragma unroll
  for (int d = 1; d < ND; d++) P[d] = max2(D[d], adds2(P[d-1], c.t[d]));
  const int plo = lo16(P[ND-1]), phi = hi16(P[ND-1]);
  // the lane as x -> max(C, x + A), A = alo + ahi; scanned over 16-lane rows
  int C = max(phi, plo + c.ahi);
  C = max(C, dpp0<ROW_SHR1>(C) + c.k1);
  C = max(C, dpp0<ROW_SHR2>(C) + c.k2);
  C = max(C, dpp0<ROW_SHR4>(C) + c.k4);
  C = max(C, dpp0<ROW_SHR8>(C) + c.k8);
  {
    const int c1 = __builtin_amdgcn_readlane(C, 15);
    const int c2 = max(c1 + c.arow31, __builtin_amdgcn_readlane(C, 31));
    const int c3 = max(c2 + c.arow47, __builtin_amdgcn_readlane(C, 47));
    const int row = z >> 4;
    const int rc = (row == 0) ? NEG : (row == 1) ? c1 : (row == 2) ? c2 : c3;
    C = max(C, rc + c.arow);
  }
  const int cin = dppi<WAVE_SHR1>(NEG, C);
  // carries into the low half (from the lane before) and the high half (end of the low half)
  const int clo = max(cin, -32768);
  const int chi = max(plo, max(cin + c.alo, -32768));
  int Q = (int) (((unsigned) clo & 0xffffu) | ((unsigned) chi << 16));
#pragma unroll
  for (int d = 0; d < ND; d++) { Q = adds2(Q, c.t[d]); D[d] = max2(P[d], Q); }
}

// The same closure with the lane maps taken as a prefix maximum: with S(k) the
// sum of tDD up to position k, a path from j to k adds S(k) - S(j), so D(k) -
// S(k) is the running maximum of D0(j) - S(j). A scan step is then one maximum
// with a DPP operand, where composed maps take a move, an add and a maximum
// (S spans at most 5120 * 32768, well inside 32 bits).
template <int ND>
__device__ __forceinline__ int dd_closure_max(int (&D)[ND], const DDConst<ND> &c)
{
  int P[ND];
  P[0] = D[0];
#pragma unroll
  for (int d = 1; d < ND; d++) P[d] = max2(D[d], adds2(P[d-1], c.t[d]));
  const int plo = lo16(P[ND-1]), phi = hi16(P[ND-1]);
  int C = max(phi, plo + c.ahi) - c.send;
  C = max(C, dppi<ROW_SHR1>(INT_NEG, C));
  C = max(C, dppi<ROW_SHR2>(INT_NEG, C));
  C = max(C, dppi<ROW_SHR4>(INT_NEG, C));
  C = max(C, dppi<ROW_SHR8>(INT_NEG, C));
  C = max(C, dppi<ROW_BCAST15, 0xa>(INT_NEG, C));
  C = max(C, dppi<ROW_BCAST31, 0xc>(INT_NEG, C));
  const int cin = dppi<WAVE_SHR1>(-(1 << 28), C + c.send);
  const int clo = max(cin, -32768);
  const int chi = max(plo, max(cin + c.alo, -32768));
  int Q = (int) __builtin_amdgcn_perm((unsigned) chi, (unsigned) clo, 0x05040100u);
#pragma unroll
  for (int d = 0; d < ND; d++) { Q = adds2(Q, c.t[d]); D[d] = max2(P[d], Q); }
  // D at the position before the lane's first ones: the lane before's last, and
  // the end of the lane's own low half
  return (int) __builtin_amdgcn_perm((unsigned) D[ND-1], (unsigned) clo, 0x05040100u);
}

// The same closure, found by passes that stop at the fixed point (the lazy-F
// passes of vitfilter.c:200-225, over half-lanes instead of SSE segments).
// Each half of a lane is first closed on its own; then the carries into the
// halves (the previous lane's last position into the low half, the lane's own
// low half into its high half) are applied while any of them raises a first
// position. A chain closed inside each half is raised somewhere only if it is
// raised at its first position, so that one comparison per half decides.
// Rows whose D->D paths reach past DD_LAZY_PASSES half-lane boundaries finish
// with the scan above, which gives the same closure from any partly closed row.
#define DD_LAZY_PASSES 2
template <int ND>
__device__ __forceinline__ void dd_closure_lazy(int (&D)[ND], const DDConst<ND> &c, int z)
{
#pragma unroll
  for (int d = 1; d < ND; d++) D[d] = max2(D[d], adds2(D[d-1], c.t[d]));
  for (int pass = 0; ; pass++) {
    const int nb = dppi<WAVE_SHR1>((int) NEG_PAIR, D[ND-1]);       // lane 0: no lane before, -infinity
    int Q = adds2((int) __builtin_amdgcn_alignbit((unsigned) D[ND-1], (unsigned) nb, 16), c.t[0]);
    const int m0 = max2(D[0], Q);
    if (__ballot(m0 != D[0]) == 0ull) return;
    if (pass == DD_LAZY_PASSES) { dd_closure<ND>(D, c, z); return; }
    D[0] = m0;
#pragma unroll
    for (int d = 1; d < ND; d++) { Q = adds2(Q, c.t[d]); D[d] = max2(D[d], Q); }
  }
}


template <int ND, int TM>
__global__ __launch_bounds__(VIT_THREADS(ND))
void k_vit(const DevProfile p, const uint8_t *__restrict__ res, const int64_t *__restrict__ off,
           const int32_t *__restrict__ len, const int32_t *__restrict__ list, const int32_t *__restrict__ count,
           DevResults r, DevLists l, GateThresh g, int gating, LenCfg lc, int32_t above)
{
#pragma clang fp contract(off)
  static_assert(TM == TM_LDS || TM == TM_TLDS, "Viterbi tables are in LDS, whole or transitions only");
  constexpr bool PIN = (TM == TM_LDS), PMDS = (ND < 10 && ND != 6);
  const int lw = list_waves(*count);
  if (((ND == 12 || ND == 16) && *count <= above) || (int64_t) blockIdx.x * lw >= *count) return;
  extern __shared__ int lds[];
  const size_t rowd = (size_t) 64 * ND;
  const int *tbl = p.vf_tbl;                             // emission rows
  if (TM == TM_LDS) { stage_table(lds, p.vf_tbl, p.vf_dwords); tbl = lds; }
  else stage_table(lds, p.vf_tbl + (size_t) p.nrows * rowd, (size_t) P7G_VF_NT * rowd);
  const int z = threadIdx.x & 63;
  const int *tr = ((TM == TM_LDS) ? lds + (size_t) p.nrows * rowd : lds) + z;
  int tMM[ND], tIM[ND], tDM[ND], tMDS[ND], tMI[ND], tII[ND];
  if (PIN) {
#pragma unroll
    for (int d = 0; d < ND; d++) {
      tMM[d] = tr[VT_MM*rowd + d*64]; tIM[d] = tr[VT_IM*rowd + d*64]; tDM[d] = tr[VT_DM*rowd + d*64];
      tMDS[d] = tr[VT_MDS*rowd + d*64]; tMI[d] = tr[VT_MI*rowd + d*64]; tII[d] = tr[VT_II*rowd + d*64];
    }
  }
  DDConst<ND> ddc;
  dd_setup<ND>(ddc, tr + VT_DDS*rowd, z);
  const bool loops0 = (p.xwN_loop == 0 && p.xwC_loop == 0 && p.xwJ_loop == 0);
  const int64_t n = *count;

  int32_t *queue = (int32_t *) count + P7G_QOFF;
  if ((int) (threadIdx.x >> 6) >= lw) return;
  for (int64_t t = queue_next(queue, 1); t < n; t = queue_next(queue, 1)) {
    const int slot = uni(list[t]);
    const int L = uni(len[slot]);
    const uint8_t *sq = res + off[slot];
    const int xmove = lc.on ? lc.xmove : (int) p.xw_move[L];
    int xN = p.base_w;
    int xB = (int16_t) (xN + xmove);
    int xB2 = pair16(xB);
    int xJ = -32768, xC = -32768;
    int M[ND], I[ND], D[ND];
#pragma unroll
    for (int d = 0; d < ND; d++) { M[d] = I[d] = D[d] = (int) NEG_PAIR; }
    int status = 0;
    // DPP destinations: lane 0 never has a source and keeps the -infinity fill
    int nbM = (int) NEG_PAIR, nbI = (int) NEG_PAIR, nbD = (int) NEG_PAIR;
    int ms0 = (int) NEG_PAIR;                     // M(i-1, k-1) for the lane's first position
    if (PIN && p.vf_free && xmove <= 0 && L > 0) {
      // Every row closes its D->D paths (see vf_free), and M's part that does
      // not come through D is formed for the next row already, in the shadow of
      // the closure's scan: a row's chain is M from D, D from M, the scan. Bound
      // by that chain, and from ND = 4 on by the instructions of a lone wave
      // (one in 4-5 cycles, about 18 per dword). A row of one target, M = 86 |
      // 400 | 803 (ND = 1 | 4 | 8): 121 | 232 | 379 ns; with the lazy test, the
      // residues, odds and thresholds handled in the row 238 | 368 | 583 ns.
      // 16,384 targets of 350: M = 400 1110 us (1189 before), 803 1704 (1891),
      // 1500 2447 (2945). Where the closure hardly ever ran, a full chip pays for
      // it: 60,000 targets at M = 20 1443 us (1314).
      int bm[ND], part[ND], e[ND];
      // xB and the specials change only on a row whose xE exceeds a threshold,
      // found by a ballot on the lanes' packed maxima; xB does not fall then
      int th2;
      auto raise = [&]() {
        xB2 = pair16(xB);
        th2 = pair16(max(min(min(xC - p.xwE_move, xJ - p.xwE_loop), 32766), -32768));
#pragma unroll
        for (int d = 0; d < ND; d++) bm[d] = adds2(xB2, tr[VT_BM*rowd + d*64]);
      };
      auto ahead = [&]() {
        nbI = dppi<WAVE_SHR1>(nbI, I[ND-1]);
        const int is0 = (int) __builtin_amdgcn_alignbit((unsigned) I[ND-1], (unsigned) nbI, 16);
#pragma unroll
        for (int d = ND-1; d >= 0; d--) {
          part[d] = max2(max2(bm[d], adds2(d ? M[d-1] : ms0, tMM[d])), adds2(d ? I[d-1] : is0, tIM[d]));
          I[d] = max2(adds2(M[d], tMI[d]), adds2(I[d], tII[d]));
        }
      };
      raise();
      ahead();
      int ds0 = (int) NEG_PAIR;
      RowRes<false> rr;
      const int x0 = rr.init(sq, L, z, (int) rowd);
#pragma unroll
      for (int d = 0; d < ND; d++) e[d] = tbl[x0 + z + d * 64];
      for (int i0 = 0; i0 < L && status == 0; i0 += 64) {
        const int cnt = min(64, L - i0);
        for (int u = 0; u < cnt; u++) {
          int xE = (int) NEG_PAIR;
#pragma unroll
          for (int d = ND-1; d >= 0; d--) {
            M[d] = adds2(max2(part[d], adds2(d ? D[d-1] : ds0, tDM[d])), e[d]);
            xE = max2(xE, M[d]);
          }
          // M -> D scores that are not pinned come before the next row's odds:
          // LDS answers in order
          int md[PMDS ? 1 : ND];
          if (! PMDS) {
            const int *trr = tr + opaque_zero();
#pragma unroll
            for (int d = 0; d < ND; d++) md[d] = trr[VT_MDS*rowd + d*64];
          }
          const int *en = tbl + rr.ahead(u) + z;
#pragma unroll
          for (int d = 0; d < ND; d++) e[d] = en[d * 64];
          const unsigned long long hit = __ballot(max2(xE, th2) != th2);
          nbM = dppi<WAVE_SHR1>(nbM, M[ND-1]);
          ms0 = (int) __builtin_amdgcn_alignbit((unsigned) M[ND-1], (unsigned) nbM, 16);
#pragma unroll
          for (int d = 0; d < ND; d++) D[d] = adds2(d ? M[d-1] : ms0, PMDS ? tMDS[d] : md[d]);
          ahead();
          ds0 = dd_closure_max<ND>(D, ddc);
          if (__builtin_expect(hit != 0ull, 0)) {
            const int xEs = uni(wave_max_i(max(lo16(xE), hi16(xE))));
            if (xEs >= 32767) { status = 16; break; }
            xC = max(xC, xEs + p.xwE_move);
            xJ = max(xJ, xEs + p.xwE_loop);
            xB = (int16_t) max(xJ + xmove, xN + xmove);
            raise();
#pragma unroll
            for (int d = 0; d < ND; d++) part[d] = max2(part[d], bm[d]);
          }
        }
        rr.advance();
      }
    } else {
      ResAsc rd;
      if (L > 0) rd.init(sq);

      for (int i = 0; i < L; i++) {
        const int x = rd.at(i);
        const int *e = tbl + (size_t) x * rowd + z;
        const int *trr = tr + opaque_zero();
#define VTR(A, T, d) (PIN ? A[d] : trr[(T) * rowd + (d) * 64])
        nbI = dppi<WAVE_SHR1>(nbI, I[ND-1]);
        nbD = dppi<WAVE_SHR1>(nbD, D[ND-1]);
        const int is0 = (int) __builtin_amdgcn_alignbit((unsigned) I[ND-1], (unsigned) nbI, 16);
        const int ds0 = (int) __builtin_amdgcn_alignbit((unsigned) D[ND-1], (unsigned) nbD, 16);
        const int xB2 = pair16(xB);
        int xE = (int) NEG_PAIR;
#pragma unroll
        for (int d = ND-1; d >= 0; d--) {
          const int mp = d ? M[d-1] : ms0, ip = d ? I[d-1] : is0, dp = d ? D[d-1] : ds0;
          int sv = adds2(xB2, trr[VT_BM * rowd + d * 64]);
          sv = max2(sv, adds2(mp, VTR(tMM, VT_MM, d)));
          sv = max2(sv, adds2(ip, VTR(tIM, VT_IM, d)));
          sv = max2(sv, adds2(dp, VTR(tDM, VT_DM, d)));
          sv = adds2(sv, e[d * 64]);
          xE = max2(xE, sv);
          I[d] = max2(adds2(M[d], VTR(tMI, VT_MI, d)), adds2(I[d], VTR(tII, VT_II, d)));
          M[d] = sv;
        }
        // D(k) <- M(k-1) + tMD(k-1) on the new row; the shifted row is also the next row's M(i-1, k-1)
        nbM = dppi<WAVE_SHR1>(nbM, M[ND-1]);
        ms0 = (int) __builtin_amdgcn_alignbit((unsigned) M[ND-1], (unsigned) nbM, 16);
        int Dm = (int) NEG_PAIR;
#pragma unroll
        for (int d = 0; d < ND; d++) { D[d] = adds2(d ? M[d-1] : ms0, trr[VT_MDS * rowd + d * 64]); Dm = max2(Dm, D[d]); }
#undef VTR
        // With the N, C and J loops at zero (as the conversion sets them,
        // p7_oprofile.c:888-897) the specials only change, and the overflow test
        // only fires, when the row's xE exceeds th; that holds if it holds on
        // any lane, so a ballot stands in for the wave maximum on other rows.
        const int xel = max(lo16(xE), hi16(xE));
        const int th = loops0 ? min(min(xC - p.xwE_move, xJ - p.xwE_loop), 32766) : -(1 << 30);
        if (__ballot(xel > th) != 0ull) {
          const int xEs = uni(wave_max_i(xel));
          if (xEs >= 32767) { status = 16; break; }
          xN = (int16_t) (xN + p.xwN_loop);
          xC = (int16_t) max(xC + p.xwC_loop, xEs + p.xwE_move);
          xJ = (int16_t) max(xJ + p.xwJ_loop, xEs + p.xwE_loop);
          xB = (int16_t) max(xJ + xmove, xN + xmove);
        }
        // the lazy-F test Dmax + ddbound > xB (vitfilter.c:198-199) holds if it
        // holds on any lane: a ballot instead of a wave maximum
        const int dml = max(lo16(Dm), hi16(Dm));
        if (__ballot(dml + p.ddbound_w > xB) != 0ull) dd_closure_lazy<ND>(D, ddc, z);
      }
    }
    if (z == 0) {
      float sc;
      if (status == 16) sc = INFINITY;
      else if (xC > -32768) {
        sc = (float) xC + (float) xmove - (float) p.base_w;
        sc = __fdiv_rn(sc, p.scale_w);
        sc = (float) ((double) sc - 3.0);
      } else sc = -INFINITY;
      r.vfsc[slot] = sc;
      r.vstatus[slot] = status;
      if (gating) {
        const float seq = (float) __ddiv_rn((double) (sc - r.filtersc[slot]), LOG2_D);
        if (seq >= g.T2v) r.stage[slot] = 3;
        else r.stage[slot] = 2;
      }
    }
  }
}

// Viterbi filter for large models, four waves per target, where vf_free holds.
// Each lane's ND dwords (positions d and d+ND of the lane as int16 pairs) are
// split into slices of ND/4; wave V owns slice V of every lane, with its
// transitions pinned in registers. What precedes a slice's first dword is the
// slice before's last dword, and for slice 0 the last dword of the lane before
// (low half) and of its own lane (high half).
// A row takes one barrier. Every wave forms the M and I before its slice again
// (its halo), for which the slice before publishes M and I at its last dword
// but one; every wave composes the lane's D->D map from all slices' chain ends,
// scans the lanes by itself, and takes from the scan the carries into its slice
// (D at the halo) and into the one before (D at the dword before the halo).
// The exchange alternates between two buffers, so that a row may be written
// while the row before is still read. As in the one-wave kernel the next row's
// M but for its D part is formed in the shadow of the exchange. Scores equal
// the one-wave kernel's bit for bit. Bound by the row's chain; M = 2600 | 5000:
// 475 | 620 ns a row, 1207 ns at 2600 with three barriers, the lazy test and
// residues and odds fetched in the row.
#define VIT_W 4
template <int ND>
__global__ __launch_bounds__(64 * VIT_W)
void k_vit_wg(const DevProfile p, const uint8_t *__restrict__ res, const int64_t *__restrict__ off,
              const int32_t *__restrict__ len, const int32_t *__restrict__ list, const int32_t *__restrict__ count,
              DevResults r, DevLists l, GateThresh g, int gating, LenCfg lc, int32_t upto)
{
#pragma clang fp contract(off)
  constexpr int W = VIT_W, NW = ND / W;
  static_assert(ND % W == 0 && NW >= 2, "slices of equal width, of two dwords at least");
  // lane z at z + 1: index 0 is what precedes lane 0
  __shared__ int4 sh_x[2][W][65];        // the row's M, I and D chain at each slice's last dword but one
  __shared__ int4 sh_p[2][64];           // the slices' chain ends
  __shared__ int4 sh_f[2][64];           // lanes whose M exceeds the specials' threshold
  __shared__ int sh_e[W];
  __shared__ int64_t sh_t;
  if (*count > upto || (int64_t) blockIdx.x >= *count) return;
  const int wv = uni(threadIdx.x >> 6), z = threadIdx.x & 63;
  const int d0 = wv * NW;
  const size_t rowd = (size_t) 64 * ND;
  const int *tbl = p.vf_tbl;
  const int *tr = tbl + (size_t) p.nrows * rowd + z;
  // the dword before d (d = 0: the last one, halves of this lane and the one before)
  const unsigned hsel = (wv > 0) ? 0x07060504u : 0x05040302u;
  auto before = [&](int own) {
    return (int) __builtin_amdgcn_perm((unsigned) own, (unsigned) dppi<WAVE_SHR1>((int) NEG_PAIR, own), hsel); };
  const int hd = (wv > 0) ? d0 - 1 : ND - 1;
  int tMM[NW], tIM[NW], tDM[NW], tMDS[NW], tMI[NW], tII[NW], tDD[NW], tBM[NW];
#pragma unroll
  for (int j = 0; j < NW; j++) {
    const size_t c = (size_t) (d0 + j) * 64;
    tBM[j] = tr[VT_BM*rowd + c]; tMM[j] = tr[VT_MM*rowd + c]; tIM[j] = tr[VT_IM*rowd + c]; tDM[j] = tr[VT_DM*rowd + c];
    tMDS[j] = tr[VT_MDS*rowd + c]; tMI[j] = tr[VT_MI*rowd + c]; tII[j] = tr[VT_II*rowd + c]; tDD[j] = tr[VT_DDS*rowd + c];
  }
  const size_t hc = (size_t) hd * 64;
  const int hBM = before(tr[VT_BM*rowd + hc]), hMM = before(tr[VT_MM*rowd + hc]), hIM = before(tr[VT_IM*rowd + hc]);
  const int hDM = before(tr[VT_DM*rowd + hc]), hMI = before(tr[VT_MI*rowd + hc]), hII = before(tr[VT_II*rowd + hc]);
  // nothing precedes lane 0's low half: M stays -infinity there
  const bool first = (wv == 0 && z == 0);
  const int hand = first ? (int) 0xffff0000 : -1, hor = first ? 0x8000 : 0;
  // int32 sums of the D->D steps, per half: of each slice of this lane, and of
  // the slice before this one without its last dword
  int alo[W], ahi[W], blo, bhi;
#pragma unroll
  for (int v = 0; v < W; v++) {
    int x = 0, y = 0;
    for (int j = 0; j < NW; j++) { const int t = tr[VT_DDS*rowd + (size_t) (v * NW + j) * 64]; x += lo16(t); y += hi16(t); }
    alo[v] = x; ahi[v] = y;
  }
  {
    int x = 0, y = 0;
    for (int j = 0; j < NW - 1; j++) { const int t = tr[VT_DDS*rowd + (size_t) (hd - NW + 1 + j) * 64]; x += lo16(t); y += hi16(t); }
    blo = (wv > 0) ? x : dppi<WAVE_SHR1>(0, y);
    bhi = (wv > 0) ? y : x;
  }
  DDConst<ND> ddc;
  dd_setup<ND>(ddc, tr + VT_DDS*rowd, z);
  if (z == 0)
    for (int q = 0; q < 2; q++) sh_x[q][wv][0] = make_int4((int) NEG_PAIR, (int) NEG_PAIR, (int) NEG_PAIR, 0);
  const int64_t n = *count;
  int32_t *queue = (int32_t *) count + P7G_QOFF;

  for (;;) {
    if (threadIdx.x == 0) sh_t = (int64_t) atomicAdd(queue, 1);
    __syncthreads();
    const int64_t t = sh_t;
    if (t >= n) break;
    const int slot = uni(list[t]);
    const int L = uni(len[slot]);
    const uint8_t *sq = res + off[slot];
    const int xmove = lc.on ? lc.xmove : (int) p.xw_move[L];
    const int xN = p.base_w;
    int xB = (int16_t) (xN + xmove);
    int xJ = -32768, xC = -32768;
    int status = 0;
    auto rows = [&](auto vc) {
      constexpr int V = decltype(vc)::value;
      constexpr int PV = (V + W - 1) % W;                  // the slice before
      int M[NW], I[NW], D[NW], bm[NW], part[NW], e[NW];
      int hM = (int) NEG_PAIR, hI = (int) NEG_PAIR, hD = (int) NEG_PAIR, gD = (int) NEG_PAIR;   // halo; D before it
      int hbm, hpart, he;
#pragma unroll
      for (int j = 0; j < NW; j++) { M[j] = I[j] = D[j] = (int) NEG_PAIR; }
      int th2;
      auto raise = [&]() {
        const int xB2 = pair16(xB);
        th2 = pair16(max(min(min(xC - p.xwE_move, xJ - p.xwE_loop), 32766), -32768));
#pragma unroll
        for (int j = 0; j < NW; j++) bm[j] = adds2(xB2, tBM[j]);
        hbm = adds2(xB2, hBM);
      };
      auto ahead = [&]() {                                 // the slice's own cells
#pragma unroll
        for (int j = NW-1; j >= 0; j--) {
          part[j] = max2(max2(bm[j], adds2(j ? M[j-1] : hM, tMM[j])), adds2(j ? I[j-1] : hI, tIM[j]));
          I[j] = max2(adds2(M[j], tMI[j]), adds2(I[j], tII[j]));
        }
      };
      auto ahead_halo = [&](int m, int i) {
        hpart = max2(max2(hbm, adds2(m, hMM)), adds2(i, hIM));
        hI = max2(adds2(hM, hMI), adds2(hI, hII));
      };
      raise(); ahead(); ahead_halo((int) NEG_PAIR, (int) NEG_PAIR);
      RowRes<false> rr;
      const int x0 = rr.init(sq, L, z, (int) rowd);
      auto odds = [&](int x) {
        const int *en = tbl + x + z;
#pragma unroll
        for (int j = 0; j < NW; j++) e[j] = en[(V * NW + j) * 64];
        he = en[(V > 0 ? V * NW - 1 : ND - 1) * 64];
      };
      odds(x0);
      for (int i0 = 0; i0 < L && status == 0; i0 += 64) {
        const int cnt = min(64, L - i0);
        for (int u = 0; u < cnt; u++) {
          const int q = u & 1;                             // 64 is even: the buffers alternate
          int xE = (int) NEG_PAIR;
#pragma unroll
          for (int j = NW-1; j >= 0; j--) {
            M[j] = adds2(max2(part[j], adds2(j ? D[j-1] : hD, tDM[j])), e[j]);
            xE = max2(xE, M[j]);
          }
          hM = adds2(max2(hpart, adds2(gD, hDM)), V > 0 ? he : before(he));
          if (V == 0) hM = (hM & hand) | hor;
          // the slice's D, closed but for what comes from before it
#pragma unroll
          for (int j = 0; j < NW; j++) D[j] = adds2(j ? M[j-1] : hM, tMDS[j]);
#pragma unroll
          for (int j = 1; j < NW; j++) D[j] = max2(D[j], adds2(D[j-1], tDD[j]));
          sh_x[q][V][z + 1] = make_int4(M[NW-2], I[NW-2], D[NW-2], 0);
          ((int *) &sh_p[q][z])[V] = D[NW-1];
          ((int *) &sh_f[q][z])[V] = max2(xE, th2) ^ th2;
          odds(rr.ahead(u));
          lds_barrier();
          const int4 P4 = sh_p[q][z], F4 = sh_f[q][z], X = sh_x[q][PV][z + 1];
          int4 Y = X;
          if (V == 0) Y = sh_x[q][PV][z];
          ahead();
          const int P[W] = { P4.x, P4.y, P4.z, P4.w };
          // what reaches each slice's halves from the lane's own D alone, and the lane's end
          int cl[W + 1], ch[W + 1];
          cl[0] = ch[0] = -(1 << 28);
#pragma unroll
          for (int v = 0; v < W; v++) { cl[v+1] = max(lo16(P[v]), cl[v] + alo[v]); ch[v+1] = max(hi16(P[v]), ch[v] + ahi[v]); }
          int Alo = 0, Ahi = 0, AloV = 0, AhiV = 0, AloP = 0, AhiP = 0;      // constants of the row loop
#pragma unroll
          for (int v = 0; v < W; v++) {
            if (v == V) { AloV = Alo; AhiV = Ahi; }
            if (v == PV) { AloP = Alo; AhiP = Ahi; }
            Alo += alo[v]; Ahi += ahi[v];
          }
          int C = max(ch[W], cl[W] + Ahi) - ddc.send;
          C = max(C, dppi<ROW_SHR1>(INT_NEG, C));
          C = max(C, dppi<ROW_SHR2>(INT_NEG, C));
          C = max(C, dppi<ROW_SHR4>(INT_NEG, C));
          C = max(C, dppi<ROW_SHR8>(INT_NEG, C));
          C = max(C, dppi<ROW_BCAST15, 0xa>(INT_NEG, C));
          C = max(C, dppi<ROW_BCAST31, 0xc>(INT_NEG, C));
          const int cin = dppi<WAVE_SHR1>(-(1 << 28), C + ddc.send);
          const int mid = max(cl[W], cin + Alo);           // the end of the low halves
          // carries into the halves of this slice and of the one before
          const int vlo = max(cl[V], cin + AloV), vhi = max(ch[V], mid + AhiV);
          const int plo = max(cl[PV], cin + AloP), phi = max(ch[PV], mid + AhiP);
          auto pack = [](int lo, int hi) { return (int) __builtin_amdgcn_perm((unsigned) max(hi, -32768), (unsigned) max(lo, -32768), 0x05040100u); };
          int Q = hD = pack(vlo, vhi);
#pragma unroll
          for (int j = 0; j < NW; j++) { Q = adds2(Q, tDD[j]); D[j] = max2(D[j], Q); }
          // the dword before the halo: slice PV's last but one; for slice 0 the
          // lane before's high half and this lane's low half
          const unsigned ysel = 0x05040302u;
          auto mix = [&](int x, int y) { return (V > 0) ? x : (int) __builtin_amdgcn_perm((unsigned) x, (unsigned) y, ysel); };
          gD = max2(mix(X.z, Y.z), (V > 0) ? pack(plo + blo, phi + bhi)
                                          : pack(dppi<WAVE_SHR1>(-(1 << 28), phi) + blo, plo + bhi));
          ahead_halo(mix(X.x, Y.x), mix(X.y, Y.y));
          if (__builtin_expect(__ballot((F4.x | F4.y | F4.z | F4.w) != 0) != 0ull, 0)) {
            const int xel = wave_max_i(max(lo16(xE), hi16(xE)));
            if (z == 0) sh_e[V] = xel;
            lds_barrier();
            int xEs = sh_e[0];
#pragma unroll
            for (int v = 1; v < W; v++) xEs = max(xEs, sh_e[v]);
            xEs = uni(xEs);
            if (xEs >= 32767) { status = 16; break; }
            xC = max(xC, xEs + p.xwE_move);
            xJ = max(xJ, xEs + p.xwE_loop);
            xB = (int16_t) max(xJ + xmove, xN + xmove);
            raise();
#pragma unroll
            for (int j = 0; j < NW; j++) part[j] = max2(part[j], bm[j]);
            hpart = max2(hpart, hbm);
          }
        }
        rr.advance();
      }
    };
    if (L > 0)
      switch (wv) {
        case 0: rows(std::integral_constant<int, 0>()); break;
        case 1: rows(std::integral_constant<int, 1>()); break;
        case 2: rows(std::integral_constant<int, 2>()); break;
        default: rows(std::integral_constant<int, 3>()); break;
      }
    if (threadIdx.x == 0) {
      float sc;
      if (status == 16) sc = INFINITY;
      else if (xC > -32768) {
        sc = (float) xC + (float) xmove - (float) p.base_w;
        sc = __fdiv_rn(sc, p.scale_w);
        sc = (float) ((double) sc - 3.0);
      } else sc = -INFINITY;
      r.vfsc[slot] = sc;
      r.vstatus[slot] = status;
      if (gating) {
        const float seq = (float) __ddiv_rn((double) (sc - r.filtersc[slot]), LOG2_D);
        if (seq >= g.T2v) r.stage[slot] = 3;
        else r.stage[slot] = 2;
      }
    }
    __syncthreads();                                     // sh_t and the exchange are free for the next target
  }
}

// Viterbi: the whole table in LDS while it fits (ND <= 16 at 160 KB), else the
// transitions in LDS and emission rows from global memory.
// The cooperative kernel takes models of ND >= 20, and of ND = 12 and 16 short
// lists: its row is the shorter one (M = 1500 383 against 595 ns, 2000 416 against
// 930 ns), but its waves repeat the scan, and a full chip does less (us for 512 |
// 4096 targets of 350, M = 2000: 320 | 1514 against 550 | 1072). Lists given by a
// caller: up to VIT_WG_FEW targets. Lists behind the gates have a search's lengths,
// whose longest targets keep the longer row waiting: up to VIT_WG_FEW_GATED (us at
// M = 1500 for 1546 | 7975 of them: 845 | 2283 against 1240 | 1964; M = 2000, 1175 |
// 5632: 1094 | 1899 against 1250 | 2019). Their number is not known on the host: both
// kernels are launched, and the count on the device decides which leaves at once
// (4 us). At ND = 8 the row gains little (350 against 386 ns). P7G_VIT_WG=0 selects
// the one-wave kernel (for comparisons).
#define VIT_WG_FEW 1024
#define VIT_WG_FEW_GATED 4096
static bool vit_wg_on()
{
  static const bool on = [] { const char *v = getenv("P7G_VIT_WG"); return ! (v && v[0] == '0'); }();
  return on;
}
#define VIT_CASE(N, T) case N: k = (void *) k_vit<N, T>; lds = (T == TM_LDS) ? p.vf_dwords * 4 : (size_t) P7G_VF_NT * 64 * N * 4; \
  nthr = VIT_THREADS(N); break;
hipError_t launch_vit(const DevProfile &p, const DevSeqs &s, const int32_t *list, const int32_t *count, int64_t maxn,
                      DevResults r, DevLists l, GateThresh g, int gating, LenCfg lc, hipStream_t st)
{
  if (maxn <= 0) return hipSuccess;
  // large models run the filter with several waves per target
  void *kw = nullptr;
  int32_t upto = INT32_MAX;
  switch (p.vf_ND) {
    case 12: kw = (void *) k_vit_wg<12>; upto = gating ? VIT_WG_FEW_GATED : VIT_WG_FEW; break;
    case 16: kw = (void *) k_vit_wg<16>; upto = gating ? VIT_WG_FEW_GATED : VIT_WG_FEW; break;
    case 20: kw = (void *) k_vit_wg<20>; break;
    case 24: kw = (void *) k_vit_wg<24>; break;
    case 32: kw = (void *) k_vit_wg<32>; break;
    case 40: kw = (void *) k_vit_wg<40>; break;
    default: break;
  }
  int32_t above = 0;
  if (kw && p.vf_free && ! (lc.on && lc.xmove > 0) && vit_wg_on() && (gating || maxn <= upto)) {   // a caller's list holds maxn
    const unsigned grid = grid_for_waves_blk(kw, std::min<int64_t>(maxn, upto) * VIT_W, 0, VIT_W);
    void *args[] = { (void *) &p, (void *) &s.res, (void *) &s.off, (void *) &s.len, (void *) &list, (void *) &count,
                     &r, &l, &g, &gating, &lc, &upto };
    const hipError_t e = launch(kw, grid, 64 * VIT_W, args, 0, st);
    if (e != hipSuccess || maxn <= upto) return e;
    above = upto;
  }
  void *k = nullptr;
  size_t lds = 0;
  int nthr = LIST_BLOCK;
  switch (p.vf_ND) {
    VIT_CASE(1, TM_LDS) VIT_CASE(2, TM_LDS) VIT_CASE(3, TM_LDS) VIT_CASE(4, TM_LDS) VIT_CASE(5, TM_LDS)
    VIT_CASE(6, TM_LDS) VIT_CASE(8, TM_LDS) VIT_CASE(10, TM_LDS) VIT_CASE(12, TM_LDS) VIT_CASE(16, TM_LDS)
    VIT_CASE(20, TM_TLDS) VIT_CASE(24, TM_TLDS) VIT_CASE(32, TM_TLDS) VIT_CASE(40, TM_TLDS)
    default: return hipErrorInvalidValue;
  }
  const unsigned grid = list_grid(k, maxn, lds, nthr / 64);
  void *args[] = { (void *) &p, (void *) &s.res, (void *) &s.off, (void *) &s.len, (void *) &list, (void *) &count,
                   &r, &l, &g, &gating, &lc, &above };
  return launch(k, grid, nthr, args, lds, st);
}

