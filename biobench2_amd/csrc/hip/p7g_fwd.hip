// gfx950 kernels of the Forward parser (HMMER/src/impl_sse/fwdback.c:134-465):
// fp32, the D->D chain as an affine prefix scan across the wave, sparse
// rescaling when xE > 1e4; the same pass over region copies gives the envelope
// scores and, with the stored Backward rows, null2 and the optimal accuracy fill.
#include "p7g_list.h"

/*****************************************************************
 * 7. Forward parser (one target per wave, fp32, B positions per lane)
 *****************************************************************/

// The end of an envelope's null2 pass (MODE 3 of k_fwd), one wave: the
// posterior sums accM/accI (this lane's B positions) and pN/pJ/pC over the
// envelope's L rows become weights (times 1/L); null2[x] for canonical x is
// the weighted sum of the positions' match odds, plus the insert weights
// (odds 1) and the N, C, J weights (impl_sse/null2.c:80-107); a degenerate
// code's value is the average over the residues it stands for
// (esl_alphabet.c:1331-1341), and gap, '*' and '~' get 1. Lane x holds
// null2[x]. The correction is sum over the envelope's residues of
// logf(null2[x]) (p7_domaindef.c:925-931). A scale product that ended
// infinite is the decoding's range error: status 16, no correction.
template <int B>
__device__ __forceinline__ void null2_epilogue(const DevProfile &p, const float *tbl, size_t rowf, int z,
                                               float (&accM)[B], float (&accI)[B], float pN, float pJ, float pC,
                                               float sp, const uint8_t *sq, int L, float *dc_out, int32_t *st_out)
{
  if (isinf(sp)) {
    if (z == 0) { *dc_out = NAN; *st_out = 16; }
    return;
  }
  const float norm = (float) (1.0 / (double) L);
  float iw = 0.0f;
#pragma unroll
  for (int j = 0; j < B; j++) { accM[j] = __fmul_rn(accM[j], norm); iw = __fadd_rn(iw, __fmul_rn(accI[j], norm)); }
  const float xfac = __builtin_fmaf(pJ, norm, fma2<true>(pN, norm, pC, norm));
  float v = 1.0f;
  for (int x = 0; x < p.K; x++) {
    const float *e = tbl + (size_t) x * rowf + z;
    float part = iw;
#pragma unroll
    for (int j = 0; j < B; j++) part = __fadd_rn(part, __fmul_rn(accM[j], e[j * 64]));
    const float s = wave_sum_f(part);
    if (z == x) v = __fadd_rn(s, xfac);
  }
  {
    const uint32_t dg = (z < 32) ? p.degen[z] : 0u;
    float r = 0.0f;
    for (int y = 0; y < p.K; y++) {
      const float vy = __shfl(v, y);
      if ((dg >> y) & 1u) r = __fadd_rn(r, vy);
    }
    if (z > p.K && z <= p.Kp - 3) v = __fdiv_rn(r, (float) (dg >> 24));
  }
  float part = 0.0f;
  for (int b0 = 0; b0 < L; b0 += 64) {
    const int pos = b0 + z;
    const int x = (pos < L) ? sq[pos] : 0;
    const float vx = __shfl(v, x & 63);
    if (pos < L) part = __fadd_rn(part, logf(vx));
  }
  const float dc = wave_sum_f(part);
  if (z == 0) { *dc_out = dc; *st_out = 0; }
}

// p7_alidisplay_EncodePostProb (p7_alidisplay.c:520-524) as a number: '*' is 10
__device__ __forceinline__ int pp_code(float p)
{
  const double q = (double) p + 0.05;
  return (q >= 1.0) ? 10 : (int) (q * 10.0);
}

// One row of the optimal accuracy fill (p7_OptimalAccuracy, impl_sse/
// optacc.c:60-175) inside the null2 Forward pass, from the row's posteriors,
// with the traceback's choices (select_m/d/i/e/c/j/b, optacc.c:288-423) made
// here from the same values and stored for k_oa_trace: four bits per cell
// (lane-minor words), one word per row. Backward's M and I values of the row
// come in registers (pbM, pbI: PRE, loaded by the caller before the row's
// Forward part) or are loaded here from cr, eight positions at a time, so
// that the row waits on memory once per eight positions, not once per cell.
// As in the SSE code, a predecessor
// behind a transition of probability 0 contributes +0.0 to the fill's maximum
// and -infinity to the traceback's choice; D(1) is -infinity; the reference's
// striped padding cells (model positions M+1..4Q) hold 0.0 and take part in
// E's maximum and in select_e's scan, which runs in the striped order
// (k = r*Q + q + 1, q outer), an M replacing on >= and a D on >. Values are
// -infinity or >= 0, so their bit patterns order as integers. The profile is
// in unihit mode (E move 1, E loop 0; N, J, C loop floop and move fmove).
template <int B, int NW, bool PIN, bool PRE>
__device__ __forceinline__ void oa_row(const DevProfile &p, int z, int i,
                                       const float (&tBM)[B], const float (&tMM)[B], const float (&tIM)[B],
                                       const float (&tDM)[B], const float (&tMDS)[B], const float (&tMI)[B],
                                       const float (&tII)[B], const float *trr, size_t rowf,
                                       const float (&fM)[B], const float (&fI)[B], const float *cr,
                                       const float *pbM, const float *pbI, float totr,
                                       float (&accM)[B], float (&accI)[B], float qN, float qJ, float qC, float sp,
                                       float floop, float fmove, float (&oaM)[B], float (&oaI)[B], float (&oaD)[B],
                                       float &oaN, float &oaJ, float &oaB, float &oaC, uint32_t *obits, uint32_t *orow,
                                       uint8_t *opp)
{
#define OTR(A, T, j) (PIN ? A[j] : trr[(T) * rowf + (j) * 64])
  const float NI = -INFINITY;
  const int M = p.M;
  const int Q = max(2, (M - 1) / 4 + 1);
  uint32_t nib[NW];
#pragma unroll
  for (int w = 0; w < NW; w++) nib[w] = 0u;
  constexpr int CH = 8;
  float cbM[CH], cbI[CH];
  uint32_t ppw = 0u;
  uint32_t *opw = (uint32_t *) opp + (size_t) (i - 1) * n2_pp_words(B) * 64 + z;
  // row i-1's values at the lane's first position's predecessor (lane z-1's last)
  const float mpL = dppf<WAVE_SHR1>(NI, oaM[B-1]), ipL = dppf<WAVE_SHR1>(NI, oaI[B-1]), dpL = dppf<WAVE_SHR1>(NI, oaD[B-1]);
  // M and I in place, last position first: position j reads row i-1 at j-1 and j
#pragma unroll
  for (int j = B - 1; j >= 0; j--) {
    const int k = z * B + j + 1;
    const bool first = (k == 1);
    const int c8 = (B - 1 - j) % CH;
    if (! PRE && c8 == 0) {
#pragma unroll
      for (int u = 0; u < CH; u++)
        if (j - u >= 0) { cbM[u] = cr[(j - u) * 64]; cbI[u] = cr[rowf + (j - u) * 64]; }
    }
    const float bm = PRE ? pbM[j] : cbM[c8], bi = PRE ? pbI[j] : cbI[c8];
    // the posteriors of row i: (f * b) * (scaleproduct * scale_i), summed for null2
    // (fused onto the sums where the larger models' registers allow; the
    // products alone rounded for the codes)
    const float fbm = __fmul_rn(fM[j], bm), fbi = __fmul_rn(fI[j], bi);
    const float pm = __fmul_rn(fbm, totr), pi = __fmul_rn(fbi, totr);
    {
#pragma clang fp contract(off)
      accM[j] = (B > 1 && B <= 16) ? __builtin_fmaf(fbm, totr, accM[j]) : pm + accM[j];
      accI[j] = (B > 1 && B <= 12) ? __builtin_fmaf(fbi, totr, accI[j]) : pi + accI[j];
    }
    // the cell's posterior probability codes for the alignment display
    ppw |= (uint32_t) (pp_code(pm) | (pp_code(pi) << 4)) << ((j % 4) * 8);
    if (j % 4 == 0) { opw[(j / 4) * 64] = ppw; ppw = 0u; }
    const float mp = j ? oaM[j-1] : mpL, ip = j ? oaI[j-1] : ipL, dp = j ? oaD[j-1] : dpL;
    const bool tb = OTR(tBM, VT_BM, j) > 0.0f, tm = OTR(tMM, VT_MM, j) > 0.0f;
    const bool ti = OTR(tIM, VT_IM, j) > 0.0f, td = OTR(tDM, VT_DM, j) > 0.0f;
    // select_m: paths M, I, D, B; the first maximum wins; node 0 reads 0.0
    const float p0 = tm ? (first ? 0.0f : mp) : NI, p1 = ti ? (first ? 0.0f : ip) : NI;
    const float p2 = td ? (first ? 0.0f : dp) : NI, p3 = tb ? oaB : NI;
    int c = 0;
    float bv = p0;
    if (p1 > bv) { c = 1; bv = p1; }
    if (p2 > bv) { c = 2; bv = p2; }
    if (p3 > bv) { c = 3; }
    float v = tb ? oaB : 0.0f;
    v = fmaxf(v, tm ? mp : 0.0f);
    v = fmaxf(v, ti ? ip : 0.0f);
    v = fmaxf(v, td ? dp : 0.0f);
    // select_i: M over I on ties
    const bool tmi = OTR(tMI, VT_MI, j) > 0.0f, tii = OTR(tII, VT_II, j) > 0.0f;
    const int ci = ((tmi ? oaM[j] : NI) >= (tii ? oaI[j] : NI)) ? 0 : 1;
    {
#pragma clang fp contract(off)
      const float vi = fmaxf(tmi ? oaM[j] : 0.0f, tii ? oaI[j] : 0.0f);
      oaI[j] = (B > 1) ? __builtin_fmaf(fbi, totr, vi) : vi + pi;
    }
    oaM[j] = __builtin_fmaf(fbm, totr, v);
    nib[j / 8] |= (uint32_t) (c | (ci << 2)) << ((j % 8) * 4);
  }
  // D(k) = max(tMD(k-1) ? M(k-1) : 0, tDD(k-1) ? D(k-1) : 0), D(1) = -infinity:
  // per position the map x -> max(c, p ? x : -inf), composed along the lane,
  // scanned across the lanes, then applied from the carry of the lanes before
  const float mL = dppf<WAVE_SHR1>(NI, oaM[B-1]);
  float C = NI;
  int P = 1;
#pragma unroll
  for (int j = 0; j < B; j++) {
    const int k = z * B + j + 1;
    const bool tmd = OTR(tMDS, VT_MDS, j) > 0.0f, tdd = trr[VT_DDS * rowf + j * 64] > 0.0f;
    const float A = tmd ? (j ? oaM[j-1] : mL) : 0.0f;
    const int pj = (k != 1 && tdd) ? 1 : 0;
    const float cj = (k == 1) ? NI : (tdd ? A : fmaxf(A, 0.0f));
    C = fmaxf(cj, pj ? C : NI);
    P &= pj;
  }
  // x -> max(C, x + W) with W = 0 (pass) or -infinity: an exact max-plus scan
  float W = P ? 0.0f : NI;
  wave_maxplus_scan(C, W);
  float cur = dppf<WAVE_SHR1>(NI, C);
#pragma unroll
  for (int j = 0; j < B; j++) {
    const int k = z * B + j + 1;
    const float mprev = j ? oaM[j-1] : mL;
    const bool tmd = OTR(tMDS, VT_MDS, j) > 0.0f, tdd = trr[VT_DDS * rowf + j * 64] > 0.0f;
    // select_d: M over D on ties; node 1 has neither
    const float a0 = (k == 1) ? NI : (tmd ? mprev : NI), a1 = (k == 1) ? NI : (tdd ? cur : NI);
    nib[j / 8] |= (uint32_t) ((a0 >= a1) ? 0 : 1) << ((j % 8) * 4 + 3);
    const float A = tmd ? mprev : 0.0f;
    const float cj = (k == 1) ? NI : (tdd ? A : fmaxf(A, 0.0f));
    cur = fmaxf(cj, (k != 1 && tdd) ? cur : NI);
    oaD[j] = cur;
  }
  // E(i): the row maximum over the model's cells (and the striped padding's 0.0)
  float el = NI;
#pragma unroll
  for (int j = 0; j < B; j++) if (z * B + j + 1 <= M) el = fmaxf(el, fmaxf(oaM[j], oaD[j]));
  const bool refpad = 4 * Q > M;
  float V = __int_as_float(wave_max_i(__float_as_int(el)));
  if (refpad) V = fmaxf(V, 0.0f);
  // select_e: the last M cell of value V in the striped order, else the first D cell
  auto key = [Q](int k) {                       // k - 1 < 4Q: the lane r by three compares
    const int r = (k - 1 >= Q) + (k - 1 >= 2 * Q) + (k - 1 >= 3 * Q);
    return (k - 1 - r * Q) * 4 + r; };
  int km = -1, kd = 0x7fffffff;
#pragma unroll
  for (int j = 0; j < B; j++) {
    const int k = z * B + j + 1;
    if (k <= M && oaM[j] == V) km = max(km, key(k));
    if (k <= M && oaD[j] == V) kd = min(kd, key(k));
  }
  int kmax = wave_max_i(km);
  int fail = 0, es = 0, ek = 0;
  // padding M cells hold V too, and the last of them (k = 4Q, key 4Q - 1)
  // comes after every model cell in the striped order
  if (refpad && V == 0.0f) fail = 1;
  if (kmax >= 0) { ek = (kmax & 3) * Q + (kmax >> 2) + 1; }
  else {
    const int kmin = -wave_max_i(-kd);
    if (kmin == 0x7fffffff) fail = 1;
    else { es = 1; ek = (kmin & 3) * Q + (kmin >> 2) + 1; }
  }
  // specials (unihit: E loop 0, E move 1), with select_j/c/b's choices
  const float eLoop = 0.0f, eMove = 1.0f;
  const float oaJp = __builtin_fmaf(qJ, sp, oaJ), oaCp = __builtin_fmaf(qC, sp, oaC);
  const float j0 = (floop == 0.0f) ? 0.0f : oaJp, j1 = (eLoop == 0.0f) ? 0.0f : V;
  const int bj = (((floop == 0.0f) ? NI : oaJp) > ((eLoop == 0.0f) ? NI : V)) ? 1 : 0;
  const float nJ = fmaxf(j0, j1);
  const float c0 = (floop == 0.0f) ? 0.0f : oaCp, c1 = (eMove == 0.0f) ? 0.0f : V;
  const int bc = (((floop == 0.0f) ? NI : oaCp) > ((eMove == 0.0f) ? NI : V)) ? 1 : 0;
  const float nC = fmaxf(c0, c1);
  const float nN = (floop == 0.0f) ? 0.0f : __builtin_fmaf(qN, sp, oaN);
  const float b0 = (fmove == 0.0f) ? 0.0f : nN, b1 = (fmove == 0.0f) ? 0.0f : nJ;
  const int bb = (((fmove == 0.0f) ? NI : nN) > ((fmove == 0.0f) ? NI : nJ)) ? 1 : 0;
  oaJ = nJ; oaC = nC; oaN = nN; oaB = fmaxf(b0, b1);
#pragma unroll
  for (int w = 0; w < NW; w++) obits[((size_t) (i - 1) * NW + w) * 64 + z] = nib[w];
  if (z == 0)
    orow[i] = (uint32_t) ek | ((uint32_t) es << OA_ESTATE) | ((uint32_t) bc << OA_CBIT) | ((uint32_t) bj << OA_JBIT) |
              ((uint32_t) bb << OA_BBIT) | ((uint32_t) fail << OA_EFAIL);
#undef OTR
}

// The null2 pass (MODE 3) runs in workgroups of four waves, one per SIMD, whose
// waves may hold 512 registers; with 256 the rows of B > 12 spilled up to 1100
// of them (null2 pass of M = 1500 | 2600: 34 | 215 ms, now 15 | 140 ms).
#define NULL2_THREADS 256
// MODE 0: the parser. MODE 1: the special-state rows also go to the caller's
// matrix (one target) or to the domain decoding pool (a separate instance, so
// that the plain parser keeps its register budget).
// MODE 2: envelope scores: the list is of region copies, each scored in unihit
// mode (E move 1, E loop 0) with the N/J/C odds of its whole target's length;
// its row scales go to the scale pool when one is given.
// MODE 3: the same Forward pass again for null2: each row's posteriors
// (p7_Decoding, impl_sse/decoding.c:109-139) from this row and the stored
// Backward row, summed over the rows; then the null2 odds
// (p7_Null2_ByExpectation, impl_sse/null2.c:59-118) and the envelope's
// correction sum_pos logf(null2[x_pos]) (p7_domaindef.c:925-931).
template <int B, int TM, int MODE>
__global__ __launch_bounds__(MODE == 3 && B > 12 ? NULL2_THREADS : FWD_THREADS(B))
void k_fwd(const DevProfile p, const uint8_t *__restrict__ res, const int64_t *__restrict__ off,
           const int32_t *__restrict__ len, const int32_t *__restrict__ list, const int32_t *__restrict__ count,
           DevResults r, DevLists l, GateThresh g, int gating, LenCfg lc,
           float *__restrict__ pool, int64_t pool_size, int64_t *__restrict__ scale_off, float *__restrict__ xmx_out,
           DomBufs dom)
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
  float tBM[B], tMM[B], tIM[B], tDM[B], tMDS[B], tMI[B], tII[B];
  if (PIN) {
#pragma unroll
    for (int j = 0; j < B; j++) {
      tBM[j] = tr[VT_BM*rowf + j*64]; tMM[j] = tr[VT_MM*rowf + j*64]; tIM[j] = tr[VT_IM*rowf + j*64]; tDM[j] = tr[VT_DM*rowf + j*64];
      tMDS[j] = tr[VT_MDS*rowf + j*64]; tMI[j] = tr[VT_MI*rowf + j*64]; tII[j] = tr[VT_II*rowf + j*64];
    }
  }
  // PF: a row's emission odds are loaded a row ahead (not where the positions
  // of a large model, or the alignment's state, already fill the registers).
  // PIND: the D->D odds are pinned too. STREAM: nothing is (see stream_tables).
  // FP: which product of xB * tBM + M * tMM is rounded before the other is fused
  // onto it. The choice is the one each size was first compiled with, kept so that
  // results stay; it depends on B alone, because the null2 pass must rescale the
  // same rows as the envelope-score pass, whose scales Backward has taken.
  constexpr bool FP = (B == 1);
  constexpr int EG = (MODE == 3) ? 8 : 16;
  constexpr bool STREAM = (TM == TM_GLOB && MODE != 3), PF = (MODE != 3 && B <= 28), PIND = (PIN && MODE != 3 && B <= 4);
  AffConst akc;
  float tDDP[B];
#pragma unroll
  for (int j = 0; j < B; j++) tDDP[j] = tr[VT_DDS*rowf + j*64];
  aff_fwd_setup<B>(akc, tDDP);
  constexpr bool DOM = (MODE == 1);
  constexpr bool ENV = (MODE >= 2);
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
    float *scl = nullptr;
    // null2: the region's area (Backward special rows, Backward M/I rows)
    float *area = nullptr;
    if (MODE == 3) {
      const int64_t o = dom.n2off[slot];
      area = dom.n2pool + (((int64_t) (unsigned) uni((int) (o >> 32)) << 32) | (unsigned) uni((int) o));
    }
    const float *xb = nullptr, *cells = nullptr;
    float sp = 0.0f, pN = 0.0f, pJ = 0.0f, pC = 0.0f;
    int own = 0;
    if (MODE == 3) {
      const int bs = uni(dom.n2st[slot]);
      if ((bs & 0xff) != 0 || L < 1) {            // the envelope's Backward failed
        if (z == 0) { dom.n2dc[slot] = NAN; dom.n2st[slot] = 16; }
        continue;
      }
      own = (bs & 0x100) != 0;
      xb = area;
      cells = xb + n2_xrows_floats(L) + z;
      sp = (float) (1.0 / (double) xb[1]);        // 1 / Backward's N at row 0
    }
    float accM[B], accI[B];
#pragma unroll
    for (int j = 0; j < B; j++) accM[j] = accI[j] = 0.0f;
    // optimal accuracy alignment (MODE 3): the OA rows (row 0: -infinity in
    // the cells; N 0, J -infinity, B 0, C -infinity) and where the traceback's
    // choices go
    constexpr int NW = (B + 7) / 8;
    float oaM[B], oaI[B], oaD[B];
    float oaN = 0.0f, oaJ = -INFINITY, oaB = 0.0f, oaC = -INFINITY;
    uint32_t *obits = nullptr, *orow = nullptr;
    uint8_t *opp = nullptr;
    if (MODE == 3) {
#pragma unroll
      for (int j = 0; j < B; j++) oaM[j] = oaI[j] = oaD[j] = -INFINITY;
      obits = (uint32_t *) (area + n2_oa_bits_at(L, B));
      orow  = (uint32_t *) (area + n2_oa_rows_at(L, B));
      opp   = (uint8_t *) (area + n2_pp_at(L, B));
      if (z == 0) orow[0] = 1u << OA_BBIT;        // B(0) comes from N(0)
    }
    if (MODE != 3 && pool) {
      unsigned long long a64 = 0;
      if (z == 0) a64 = atomicAdd(l.cursor, (unsigned long long) (L + 1));
      const int64_t at = ((int64_t) (unsigned) uni((int) (a64 >> 32)) << 32) | (unsigned) uni((int) a64);
      if (at + L + 1 <= pool_size) { scl = pool + at; if (z == 0) scale_off[slot] = at; }
      else { if (z == 0) { scale_off[slot] = -1; atomicExch(&l.counts[6], 1); } }
    }
    // the special-state rows go to the caller's matrix (one target) or, for
    // domain decoding, to the target's entry in the decoding pool
    float *xo = DOM ? xmx_out : nullptr;
    if (DOM && dom.pool) {
      const int64_t need = 6 * (int64_t) (L + 1);
      unsigned long long a64 = 0;
      if (z == 0) a64 = atomicAdd(l.cursor + 1, (unsigned long long) need);
      const int64_t at = ((int64_t) (unsigned) uni((int) (a64 >> 32)) << 32) | (unsigned) uni((int) a64);
      if (at + need <= dom.size) { xo = dom.pool + at; if (z == 0) dom.doff[slot] = at; }
      else { xo = nullptr; if (z == 0) { dom.doff[slot] = -1; atomicOr(&l.counts[7], 1); } }
    }
    float M[B], I[B], D[B];
#pragma unroll
    for (int j = 0; j < B; j++) M[j] = I[j] = D[j] = 0.0f;
    float xN = 1.0f, xJ = 0.0f, xC = 0.0f, xB = fmove, xE = 0.0f;
    float totscale = 0.0f;
    if (xo && z == 0) {
      xo[0] = 0.0f; xo[1] = 1.0f; xo[2] = 0.0f; xo[3] = xB; xo[4] = 0.0f; xo[5] = 1.0f;
    }
    if (scl && z == 0) scl[0] = 1.0f;

    float mL = 0.0f;                            // M(i-1, k-1) of the lane's first position
    // One row. A wave that runs alone is bound by the row's chain of
    // dependent instructions, so nothing in a row waits on memory or takes a
    // branch that it can do without: the next row's emission odds take this
    // row's registers once M is done (PF), a row's scale and specials go to
    // registers of lane u and leave 64 rows at a time, and the rescaling test
    // is a scalar one. A row of one target alone, M = 20 | 86 | 400 | 803: 198 |
    // 209 | 352 | 513 ns (with odds, residues and scales fetched in the row and
    // the branches 305 | 329 | 451 | 656 ns).
    float sbuf = 1.0f;                          // lane u: the scale of the block's row u
    float bE = 0.0f, bN = 0.0f, bJ = 0.0f, bB = 0.0f, bC = 0.0f;
    float e[PF ? B : 1];
    auto row = [&](int xoff, int xnext, int i, int u) {
      const float *er = (const float *) ((const char *) tbl + xoff) + z;
      const float *trr = tr + (PIN ? 0 : opaque_zero());
      const float pxN = xN, pxJ = xJ, pxC = xC;          // row i-1
      // null2 (MODE 3): Backward's specials and, for up to eight positions
      // per lane, its M and I values of row i, loaded before the row's
      // Forward part so that their latency overlaps it
      constexpr bool PRE = (MODE == 3 && B <= 8);
      float bx1 = 0.0f, bx2 = 0.0f, bx4 = 0.0f, bx5 = 1.0f;
      float pbM[PRE ? B : 1], pbI[PRE ? B : 1];
      if (MODE == 3) {
        const float *xr = xb + (size_t) i * 6;
        bx1 = xr[1]; bx2 = xr[2]; bx4 = xr[4]; bx5 = xr[5];
        if (PRE) {
          const float *cr = cells + (size_t) (i-1) * 2 * rowf;
#pragma unroll
          for (int j = 0; j < (PRE ? B : 1); j++) { pbM[j] = cr[j*64]; pbI[j] = cr[rowf + j*64]; }
        }
      }

#define FTR(A, T, j) (PIN ? A[j] : trr[(T) * rowf + (j) * 64])
      const float iL = dppz<WAVE_SHR1>(I[B-1]), dL = dppz<WAVE_SHR1>(D[B-1]);
      float xEl = 0.0f;
      auto cell = [&](int j, float ej, float bm, float mm, float im, float dm, float mi, float ii) {
        const float mp = j ? M[j ? j-1 : 0] : mL, ip = j ? I[j ? j-1 : 0] : iL, dp = j ? D[j ? j-1 : 0] : dL;
        const float In = fma2<false>(M[j], mi, I[j], ii);
        float sv = fma2<FP>(xB, bm, mp, mm);
        sv = __builtin_fmaf(ip, im, sv);
        sv = __builtin_fmaf(dp, dm, sv);
        M[j] = sv * ej; I[j] = In;
        xEl = (B > 1 && j == B-1) ? M[j] : __builtin_fmaf(sv, ej, xEl);   // B = 1: no product left to fuse with D
      };
      if constexpr (STREAM) {
        stream_tables<B, 7, 8, true>({ er, trr + VT_BM*rowf, trr + VT_MM*rowf, trr + VT_IM*rowf, trr + VT_DM*rowf,
                                        trr + VT_MI*rowf, trr + VT_II*rowf },
                                      [&](int j, const float (&x)[7]) { cell(j, x[0], x[1], x[2], x[3], x[4], x[5], x[6]); });
        mL = dppz<WAVE_SHR1>(M[B-1]);
        float C = 0.0f;
        stream_tables<B, 2, 32, false>({ trr + VT_MDS*rowf, trr + VT_DDS*rowf }, [&](int j, const float (&x)[2]) {
          D[j] = (j ? M[j ? j-1 : 0] : mL) * x[0];
          C = j ? __builtin_fmaf(x[1], C, D[j]) : D[j]; });
        float cur = lane_carry_fwd(C, akc);
        stream_tables<B, 1, 32, false>({ trr + VT_DDS*rowf }, [&](int j, const float (&x)[1]) {
          D[j] = cur = __builtin_fmaf(x[0], cur, D[j]); });
      } else {
        float eg[EG];                            // without PF the odds come EG positions at a time
#pragma unroll
        for (int j = B-1; j >= 0; j--) {
          if (! PF && (B - 1 - j) % EG == 0) {
#pragma unroll
            for (int v = 0; v < EG; v++) if (j - v >= 0) eg[v] = er[(j - v) * 64];
          }
          cell(j, PF ? e[PF ? j : 0] : eg[(B - 1 - j) % EG], FTR(tBM, VT_BM, j), FTR(tMM, VT_MM, j), FTR(tIM, VT_IM, j),
               FTR(tDM, VT_DM, j), FTR(tMI, VT_MI, j), FTR(tII, VT_II, j));
        }
        if (PF) {
          const float *el = (const float *) ((const char *) tbl + xnext) + z;
#pragma unroll
          for (int j = 0; j < (PF ? B : 1); j++) e[j] = el[j * 64];
        }
        mL = dppz<WAVE_SHR1>(M[B-1]);
#pragma unroll
        for (int j = 0; j < B; j++) D[j] = (j ? M[j-1] : mL) * FTR(tMDS, VT_MDS, j);
#undef FTR
        if (PIND) affine_fwd_scan<B>(D, tDDP, akc);
        else {
          // the D->D odds are read per row, not pinned in registers: this keeps
          // the kernel at 128 VGPRs, four waves per SIMD
          float tDDS[B];
#pragma unroll
          for (int j = 0; j < B; j++) tDDS[j] = trr[VT_DDS*rowf + j*64];
          affine_fwd_scan<B>(D, tDDS, akc);
        }
      }
#pragma unroll
      for (int j = 0; j < B; j++) xEl += D[j];
      xE = wave_sum_f(xEl);
      xN = xN * floop;
      fma_onto(xC, floop, xE * eMove);
      fma_onto(xJ, floop, xE * eLoop);
      xB = fma2<true>(xJ, fmove, xN, fmove);
      float scale = 1.0f;
      if (gt_bits(uni(__float_as_int(xE)), BITS_1E4)) {
        xN = xN / xE; xC = xC / xE; xJ = xJ / xE; xB = xB / xE;
        const float inv = (float) (1.0 / (double) xE);
#pragma unroll
        for (int j = 0; j < B; j++) { M[j] *= inv; D[j] *= inv; I[j] *= inv; }
        mL *= inv;
        scale = xE;
        if (MODE != 3) {
          sbuf = (z == u) ? xE : sbuf;
          totscale = (float) ((double) totscale + log((double) xE));
        }
        xE = 1.0f;
        if (TM == TM_LDS && MODE != 3) {
          // the pinned odds are read again, so that they need no registers
          // beside the logarithm's on this rare path (B = 7 keeps its 128)
          const float *t2 = tr + opaque_zero();
#pragma unroll
          for (int j = 0; j < B; j++) {
            tBM[j] = t2[VT_BM*rowf + j*64]; tMM[j] = t2[VT_MM*rowf + j*64]; tIM[j] = t2[VT_IM*rowf + j*64]; tDM[j] = t2[VT_DM*rowf + j*64];
            tMDS[j] = t2[VT_MDS*rowf + j*64]; tMI[j] = t2[VT_MI*rowf + j*64]; tII[j] = t2[VT_II*rowf + j*64];
          }
        }
      }
      if (DOM) {
        const bool me = (z == u);
        bE = me ? xE : bE; bN = me ? xN : bN; bJ = me ? xJ : bJ; bB = me ? xB : bB; bC = me ? xC : bC;
      }
      if (MODE == 3) {
        // posteriors of row i: (f * b) * (scaleproduct * scale_i); N, J, C
        // from Forward's row i-1 and Backward's row i
        const float totr = sp * scale;
        const float *cr = cells + (size_t) (i-1) * 2 * rowf;
        const float qN = __fmul_rn(__fmul_rn(pxN, bx1), floop);
        const float qJ = __fmul_rn(__fmul_rn(pxJ, bx2), floop);
        const float qC = __fmul_rn(__fmul_rn(pxC, bx4), floop);
        const float spi = sp;
        {
#pragma clang fp contract(off)
          pN = pN + qN * spi; pJ = pJ + qJ * spi; pC = pC + qC * spi;
        }
        if (own) sp = __fmul_rn(sp, __fdiv_rn(scale, bx5));
        // the row's posteriors (summed for null2) and its optimal accuracy row
        oa_row<B, NW, PIN, PRE>(p, z, i, tBM, tMM, tIM, tDM, tMDS, tMI, tII, tr + (PIN ? 0 : opaque_zero()), rowf,
                                M, I, cr, pbM, pbI, totr, accM, accI, qN, qJ, qC, spi, floop, fmove, oaM, oaI, oaD,
                                oaN, oaJ, oaB, oaC, obits, orow, opp);
      }
    };
    if constexpr (MODE == 3) {
      // long rows that keep many registers: a scalar residue each, no row ahead
      ResAsc rd;
      rd.init(sq);
      for (int i = 1; i <= L; i++) row(rd.at(i - 1) * (int) rowf * 4, 0, i, 0);
    } else if (L > 0) {
      RowRes<false> rr;
      int xoff = rr.init(sq, L, z, (int) rowf * 4);      // in bytes: one instruction a row less
      if (PF) {
#pragma unroll
        for (int j = 0; j < (PF ? B : 1); j++) e[j] = ((const float *) ((const char *) tbl + xoff))[z + j * 64];
      }
      for (int i0 = 0; i0 < L; i0 += 64) {
        const int cnt = uni(min(64, L - i0));
        sbuf = 1.0f;
        for (int u = 0; u < cnt; u++) {
          const int xnext = rr.ahead(u);
          row(xoff, xnext, i0 + u + 1, u);
          xoff = xnext;
        }
        if (z < cnt) {
          if (scl) scl[i0 + 1 + z] = sbuf;
          if (DOM && xo) {
            float *xr = xo + (size_t) (i0 + 1 + z) * 6;
            xr[0] = bE; xr[1] = bN; xr[2] = bJ; xr[3] = bB; xr[4] = bC; xr[5] = sbuf;
          }
        }
        rr.advance();
      }
    }
    if (MODE == 3) {
      if (z == 0) dom.n2oa[slot] = oaC;          // p7_OptimalAccuracy's *ret_e = C(L)
      null2_epilogue<B>(p, tbl, rowf, z, accM, accI, pN, pJ, pC, sp, sq, L, dom.n2dc + slot, dom.n2st + slot);
      continue;
    }
    if (z == 0) {
      int status = 0;
      float sc;
      if (isnan(xC) || (L > 0 && xC == 0.0f) || isinf(xC)) { status = 16; sc = NAN; }
      else sc = (float) ((double) totscale + log((double) (xC * fmove)));
      r.fwdsc[slot] = sc;
      r.fstatus[slot] = status;
      bool pass = false;
      if (gating) {
        const float seq = (float) __ddiv_rn((double) (sc - r.filtersc[slot]), LOG2_D);
        pass = (status == 0 && seq >= g.T3f);
        r.stage[slot] = pass ? 4 : 3;
      }
      // an F3 survivor's decoding entry: the Backward rows, then btot, etot, mocc
      if (DOM && dom.pool) {
        int64_t bo = -1;
        if (pass && xo) {
          const int64_t need = 9 * (int64_t) (L + 1);
          const int64_t at = (int64_t) atomicAdd(l.cursor + 1, (unsigned long long) need);
          if (at + need <= dom.size) bo = at;
          else atomicOr(&l.counts[7], 1);
        }
        dom.boff[slot] = bo;
      }
    }
  }
}

// Forward parser for large models, W waves per target. Each lane's B table
// positions are split into W slices of B/W; wave w owns slice w of every lane,
// with its transitions pinned in registers (one wave alone would have to read
// them from memory every row). The D->D chain is composed per slice (constants
// of the row), per lane (the W slices in order), then scanned across the
// lanes. A row takes two barriers: one for the slices' chain constants, one for
// the waves' parts of the row sum and the slices' last positions, which the
// next slice's first position continues from (in row i+1 and, through M of the
// position before it, which every wave forms again, in its own row's D). Every
// wave updates the special states and rescales by itself, from the same sum.
// Bound by the row's chain of dependent steps; M = 2600 (B = 48, W = 4): 832 ns
// a row, where four barriers and odds loaded in the row made it 1083 ns.
__device__ __forceinline__ void aff_setup_lane(AffConst &k, float P)
{
  k.w1 = P; P = P * dppf<ROW_SHR1>(1.0f, P);
  k.w2 = P; P = P * dppf<ROW_SHR2>(1.0f, P);
  k.w4 = P; P = P * dppf<ROW_SHR4>(1.0f, P);
  k.w8 = P; P = P * dppf<ROW_SHR8>(1.0f, P);
  k.prow = P; k.pa = readlanef(P, 31); k.pb = readlanef(P, 47);
}

// ROWS: the special-state rows go to the caller's matrix (one target).
template <int B, int W, bool ROWS>
__global__ __launch_bounds__(64 * W)
void k_fwd_wg(const DevProfile p, const uint8_t *__restrict__ res, const int64_t *__restrict__ off,
              const int32_t *__restrict__ len, const int32_t *__restrict__ list, const int32_t *__restrict__ count,
              DevResults r, DevLists l, GateThresh g, int gating, LenCfg lc,
              float *__restrict__ pool, int64_t pool_size, int64_t *__restrict__ scale_off, float *__restrict__ xmx_out)
{
  static_assert(B % W == 0 && B / W >= 2, "slices of equal width, of two positions at least");
  constexpr int BW = B / W;
  // a row's M, I and D at each slice's last position (0..2) and the one before
  // it (3..5); lane z at z + 1, so that slice 0 reads lane z - 1 at z (0: none)
  __shared__ float sh_p[6][W][65];
  __shared__ float sh_c[W][64];                               // this row's slice D-chain constants
  __shared__ float sh_e[W];                                   // the waves' parts of the row sum
  __shared__ int64_t sh_t, sh_at;
  if ((int64_t) blockIdx.x >= *count) return;
  const int wv = threadIdx.x >> 6, z = threadIdx.x & 63;
  const int j0 = wv * BW;
  const size_t rowf = (size_t) 64 * B;
  const float *tbl = p.fb_tbl;
  const float *tr = tbl + (size_t) p.nrows * rowf + z;
  float tBM[BW], tMM[BW], tIM[BW], tDM[BW], tMDS[BW], tMI[BW], tII[BW], tDD[BW];
#pragma unroll
  for (int j = 0; j < BW; j++) {
    const size_t c = (size_t) (j0 + j) * 64;
    tBM[j] = tr[VT_BM*rowf + c]; tMM[j] = tr[VT_MM*rowf + c]; tIM[j] = tr[VT_IM*rowf + c]; tDM[j] = tr[VT_DM*rowf + c];
    tMDS[j] = tr[VT_MDS*rowf + c]; tMI[j] = tr[VT_MI*rowf + c]; tII[j] = tr[VT_II*rowf + c]; tDD[j] = tr[VT_DDS*rowf + c];
  }
  // the position before the slice's first one: the previous slice's last (for
  // slice 0 the previous lane's); its M of every row is formed here again
  const bool none = (wv == 0 && z == 0);
  const int hoff = none ? 0 : (wv > 0) ? (j0 - 1) * 64 : (B - 1) * 64 - 1;
  const float hBM = tr[VT_BM*rowf + hoff], hMM = tr[VT_MM*rowf + hoff], hIM = tr[VT_IM*rowf + hoff], hDM = tr[VT_DM*rowf + hoff];
  const int pw = (wv > 0) ? wv - 1 : W - 1, pz = (wv > 0) ? z + 1 : z;     // where its values are in sh_p
  // the D->D products of every slice of this lane, and of the whole lane
  float Pv[W];
#pragma unroll
  for (int v = 0; v < W; v++) {
    float P = 1.0f;
    for (int j = 0; j < BW; j++) P *= tr[VT_DDS*rowf + (size_t) (v * BW + j) * 64];
    Pv[v] = P;
  }
  AffConst akl;
  {
    float P = 1.0f;
#pragma unroll
    for (int v = 0; v < W; v++) P *= Pv[v];
    aff_setup_lane(akl, P);
  }
  if (threadIdx.x < 6 * W) sh_p[threadIdx.x / W][threadIdx.x % W][0] = 0.0f;
  const int64_t n = *count;
  int32_t *queue = (int32_t *) count + P7G_QOFF;

  for (;;) {
    if (threadIdx.x == 0) sh_t = (int64_t) atomicAdd(queue, 1);
    __syncthreads();
    const int64_t t = sh_t;
    if (t >= n) break;
    const int slot = list[t];
    const int L = len[slot];
    const uint8_t *sq = res + off[slot];
    const float floop = lc.on ? lc.floop : p.xf_loop[L], fmove = lc.on ? lc.fmove : p.xf_move[L];
    if (threadIdx.x == 0) {
      int64_t at = -1;
      if (pool) {
        at = (int64_t) atomicAdd(l.cursor, (unsigned long long) (L + 1));
        if (at + L + 1 > pool_size) { at = -1; atomicExch(&l.counts[6], 1); }
        scale_off[slot] = at;
      }
      sh_at = at;
    }
    __syncthreads();
    float *scl = (pool && sh_at >= 0) ? pool + sh_at : nullptr;
    float M[BW], I[BW], D[BW];
#pragma unroll
    for (int j = 0; j < BW; j++) M[j] = I[j] = D[j] = 0.0f;
    float m1 = 0.0f, i1 = 0.0f, d1 = 0.0f, m2 = 0.0f, i2 = 0.0f, d2 = 0.0f;   // row i-1 at the two positions before
    float xN = 1.0f, xJ = 0.0f, xC = 0.0f, xB = fmove, xE = 0.0f;
    float totscale = 0.0f;
    if (scl && threadIdx.x == 0) scl[0] = 1.0f;
    if (ROWS && threadIdx.x == 0) {
      xmx_out[0] = 0.0f; xmx_out[1] = 1.0f; xmx_out[2] = 0.0f; xmx_out[3] = xB; xmx_out[4] = 0.0f; xmx_out[5] = 1.0f;
    }
    if (L > 0) {
      RowRes<false> rr;
      const int x0 = rr.init(sq, L, z, (int) rowf);
      // the odds of the slice and of the position before it, a row ahead: they
      // come from L2, which took a quarter of the row when waited for
      float e[BW], eh;
      auto odds = [&](int xo) {
        const float *q = tbl + xo + z;
#pragma unroll
        for (int j = 0; j < BW; j++) e[j] = q[(size_t) (j0 + j) * 64];
        eh = q[hoff];
      };
      odds(x0);
      float sbuf = 1.0f;
      float bE = 0.0f, bN = 0.0f, bJ = 0.0f, bB = 0.0f, bC = 0.0f;
      for (int i0 = 0; i0 < L; i0 += 64) {
        const int cnt = min(64, L - i0);
        sbuf = 1.0f;
        for (int u = 0; u < cnt; u++) {
          const int xnext = rr.ahead(u);
          // this row's M at the position before the slice, as its own slice forms it
          float mh = fma2<false>(xB, hBM, m2, hMM);
          mh = __builtin_fmaf(i2, hIM, mh);
          mh = __builtin_fmaf(d2, hDM, mh);
          mh = mh * eh;
          float xEl = 0.0f;
#pragma unroll
          for (int j = BW-1; j >= 0; j--) {
            const float mp = j ? M[j-1] : m1, ip = j ? I[j-1] : i1, dp = j ? D[j-1] : d1;
            const float In = fma2<false>(M[j], tMI[j], I[j], tII[j]);
            float sv = fma2<false>(xB, tBM[j], mp, tMM[j]);
            sv = __builtin_fmaf(ip, tIM[j], sv);
            sv = __builtin_fmaf(dp, tDM[j], sv);
            M[j] = sv * e[j]; I[j] = In;
            xEl = __builtin_fmaf(sv, e[j], xEl);
          }
          odds(xnext);
          const float mS = none ? 0.0f : mh;
#pragma unroll
          for (int j = 0; j < BW; j++) D[j] = (j ? M[j-1] : mS) * tMDS[j];
          {
            float C = 0.0f;
#pragma unroll
            for (int j = 0; j < BW; j++) C = __builtin_fmaf(tDD[j], C, D[j]);
            sh_c[wv][z] = C;
          }
          lds_barrier();                                // the slices' chain constants are written
          {
            float cv[W];
#pragma unroll
            for (int v = 0; v < W; v++) cv[v] = sh_c[v][z];
            float Cl = 0.0f;
#pragma unroll
            for (int v = 0; v < W; v++) Cl = __builtin_fmaf(Pv[v], Cl, cv[v]);
            float c = lane_carry_fwd(Cl, akl);
#pragma unroll
            for (int v = 0; v < W - 1; v++) if (v < wv) c = __builtin_fmaf(Pv[v], c, cv[v]);
            float cur = c;
#pragma unroll
            for (int j = 0; j < BW; j++) { cur = __builtin_fmaf(tDD[j], cur, D[j]); D[j] = cur; }
          }
#pragma unroll
          for (int j = 0; j < BW; j++) xEl += D[j];
          sh_p[0][wv][z + 1] = M[BW-1]; sh_p[1][wv][z + 1] = I[BW-1]; sh_p[2][wv][z + 1] = D[BW-1];
          sh_p[3][wv][z + 1] = M[BW-2]; sh_p[4][wv][z + 1] = I[BW-2]; sh_p[5][wv][z + 1] = D[BW-2];
          {
            const float ws = wave_sum_f(xEl);
            if (z == 0) sh_e[wv] = ws;
          }
          lds_barrier();                                // the row's slice ends and sum parts are written
          m1 = sh_p[0][pw][pz]; i1 = sh_p[1][pw][pz]; d1 = sh_p[2][pw][pz];
          m2 = sh_p[3][pw][pz]; i2 = sh_p[4][pw][pz]; d2 = sh_p[5][pw][pz];
          xE = 0.0f;
#pragma unroll
          for (int v = 0; v < W; v++) xE += sh_e[v];
          xN = xN * floop;
          xC = fma2<false>(xC, floop, xE, p.xfE_move);
          xJ = fma2<false>(xJ, floop, xE, p.xfE_loop);
          xB = fma2<true>(xJ, fmove, xN, fmove);
          if (gt_bits(uni(__float_as_int(xE)), BITS_1E4)) {
            xN = xN / xE; xC = xC / xE; xJ = xJ / xE; xB = xB / xE;
            const float inv = (float) (1.0 / (double) xE);
#pragma unroll
            for (int j = 0; j < BW; j++) { M[j] *= inv; D[j] *= inv; I[j] *= inv; }
            m1 *= inv; i1 *= inv; d1 *= inv; m2 *= inv; i2 *= inv; d2 *= inv;
            sbuf = (z == u) ? xE : sbuf;
            totscale = (float) ((double) totscale + log((double) xE));
            xE = 1.0f;
          }
          if (ROWS) {
            const bool me = (z == u);
            bE = me ? xE : bE; bN = me ? xN : bN; bJ = me ? xJ : bJ; bB = me ? xB : bB; bC = me ? xC : bC;
          }
        }
        if (wv == 0 && z < cnt) {
          if (scl) scl[i0 + 1 + z] = sbuf;
          if (ROWS) {
            float *xr = xmx_out + (size_t) (i0 + 1 + z) * 6;
            xr[0] = bE; xr[1] = bN; xr[2] = bJ; xr[3] = bB; xr[4] = bC; xr[5] = sbuf;
          }
        }
        rr.advance();
      }
    }
    if (threadIdx.x == 0) {
      int status = 0;
      float sc;
      if (isnan(xC) || (L > 0 && xC == 0.0f) || isinf(xC)) { status = 16; sc = NAN; }
      else sc = (float) ((double) totscale + log((double) (xC * fmove)));
      r.fwdsc[slot] = sc;
      r.fstatus[slot] = status;
      bool pass = false;
      if (gating) {
        const float seq = (float) __ddiv_rn((double) (sc - r.filtersc[slot]), LOG2_D);
        pass = (status == 0 && seq >= g.T3f);
        r.stage[slot] = pass ? 4 : 3;
      }
    }
    __syncthreads();                                    // the target is done before the next one is taken
  }
}

// the parser that keeps no rows; from B = 16 on k_fwd_wg takes these calls
template <int B, int TM> static void *fwd_plain()
{
  if constexpr (B < 16) return (void *) k_fwd<B, TM, 0>;
  else return nullptr;
}
#define FWD_CASE(N, T) case N * 4 + T: k = dom.env_loop ? (dom.n2mode == 2 ? (void *) k_fwd<N, T, 3> : (void *) k_fwd<N, T, 2>) \
                                          : (dom.pool || xmx_out) ? (void *) k_fwd<N, T, 1> : fwd_plain<N, T>(); \
                                          nthr = FWD_THREADS(N); break;

#define FWD_WG_CASE(N, W) case N: kw = xmx_out ? (void *) k_fwd_wg<N, W, true> : (void *) k_fwd_wg<N, W, false>; ww = W; break;
hipError_t launch_fwd(const DevProfile &p, const DevSeqs &s, const int32_t *list, const int32_t *count, int64_t maxn,
                      DevResults r, DevLists l, GateThresh g, int gating, LenCfg lc,
                      float *scale_pool, int64_t pool_size, int64_t *scale_off, float *xmx_out, hipStream_t st,
                      const DomBufs &dom)
{
  if (maxn <= 0) return hipSuccess;
  // large models run the parser with several waves per target (4 up to 48
  // positions per lane, 8 above), also for a single target, whose row of
  // M = 1000 | 2600 takes 617 | 832 ns instead of one wave's 1028 | 2778 ns
  void *kw = nullptr;
  int ww = 0;
  if (! dom.pool && ! dom.env_loop) {
    switch (p.fb_B) {
      FWD_WG_CASE(16, 4)
      FWD_WG_CASE(20, 4)
      FWD_WG_CASE(24, 4)
      FWD_WG_CASE(28, 4)
      FWD_WG_CASE(32, 4)
      FWD_WG_CASE(40, 4)
      FWD_WG_CASE(48, 4)
      FWD_WG_CASE(64, 8)
      FWD_WG_CASE(80, 8)
      default: break;
    }
  }
  if (kw) {
    const unsigned grid = grid_for_waves_blk(kw, maxn * ww, 0, ww);
    void *args[] = { (void *) &p, (void *) &s.res, (void *) &s.off, (void *) &s.len, (void *) &list, (void *) &count,
                     &r, &l, &g, &gating, &lc, &scale_pool, &pool_size, &scale_off, &xmx_out };
    return launch(kw, grid, 64 * ww, args, 0, st);
  }
  const int tm = fb_mode(p);
  void *k = nullptr;
  int nthr = LIST_BLOCK;
  switch (p.fb_B * 4 + tm) {
    FB_CASES(FWD_CASE)
    default: return hipErrorInvalidValue;
  }
  if (! k) return hipErrorInvalidValue;
  // the null2 pass in workgroups of four waves (one per SIMD), so that one of
  // them fits on a compute unit beside a multidomain region's wave
  if (dom.env_loop && dom.n2mode == 2) nthr = std::min(nthr, NULL2_THREADS);
  const size_t lds = fb_lds(p, tm);
  const unsigned grid = list_grid(k, maxn, lds, nthr / 64);
  void *args[] = { (void *) &p, (void *) &s.res, (void *) &s.off, (void *) &s.len, (void *) &list, (void *) &count,
                   &r, &l, &g, &gating, &lc, &scale_pool, &pool_size, &scale_off, &xmx_out, (void *) &dom };
  return launch(k, grid, nthr, args, lds, st);
}

