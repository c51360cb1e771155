// gfx950 kernels of the HMMER3 filter pipeline.
//
// Layout shared by all DP kernels: a target's model positions k = 1..M are
// split into contiguous blocks, one block per lane of a G-lane group
// (G = 16 or 64). Lane z owns positions z*B + 1 .. z*B + B, so the row-to-row
// dependency M(i,k) <- M(i-1,k-1) stays inside a lane except at block starts,
// where one DPP lane shift (row_shr / wave_shr) brings the neighbour's last
// value. The integer stages hold two positions per dword as int16 halves:
// dword d carries positions j = d (low half) and j = d + ND (high half), so a
// whole row shifts with one DPP move plus one v_alignbit on the last dword.
//
// MSV stage (HMMER/src/impl_sse/msvfilter.c:76-210): the uchar recurrence
//   sv = subs_u8(adds_u8(max(M(i-1,k-1), xB), bias), rbv[x][k])
// is evaluated exactly, in two passes:
//   1. k_ssv: while the J state is unused xB is a per-target constant, and with
//      Z = max(M, xB) - xB the row update becomes Z(i,k) = max(Z(i-1,k-1) + r, 0),
//      r = bias - rbv. Holding Z - 32768 in int16, the floor at 0 is exactly the
//      saturation of v_pk_add_i16 ... clamp, so a cell costs one packed add and
//      one packed max (the running maximum). The pass records max Z per target.
//   2. k_msv_classify decides per target: overflow (some row reaches
//      xE + bias >= 255), exact score (J never above base, xJ = max xE - tec), or
//      "needs the J state" -> k_msv_full runs the row-serial recurrence.
// This file holds the MSV stage's decision and full recurrence, the bias filter,
// domain decoding and the stages' compaction; Viterbi, Forward and Backward are in
// files of their own.
#include "p7g_list.h"

/*****************************************************************
 * 2. MSV stage: per-target decision after the ungapped pass
 *****************************************************************/
__global__ void k_msv_classify(const DevProfile p, const int32_t *__restrict__ len, const int32_t *__restrict__ slots,
                               int64_t n, const uint16_t *__restrict__ zmax, int16_t *__restrict__ xj,
                               int32_t *__restrict__ full_list, int32_t *__restrict__ full_count, LenCfg lc)
{
  for (int64_t t = (int64_t) blockIdx.x * blockDim.x + threadIdx.x; t < n; t += (int64_t) gridDim.x * blockDim.x) {
    const int64_t slot = slots ? (int64_t) slots[t] : t;
    const int L    = len[slot];
    const int tjbm = ((lc.on ? lc.tjb : (int) p.tjb[L]) + p.tbm) & 0xff;
    const int xB   = max(p.base - tjbm, 0);
    const int zm   = zmax[slot];
    int v;
    if (zm == 0)                          v = -2;          // no cell above the B floor: rescore exactly
    else if (xB + zm + p.bias >= 255)     v = -1;          // some row overflows (MSV values only grow with xB)
    else if (xB + zm > p.base + p.tec)    v = -2;          // the J state would raise xB
    else                                  v = max(xB + zm - p.tec, 0);
    if (slots) {                                   // explicit slot list: append here
      list_append(v == -2, (int32_t) slot, full_list, full_count);
      if (v == -2) v = 0;
    }
    xj[slot] = (int16_t) v;                        // -2 marks "full recurrence" for the compaction
  }
}

/*****************************************************************
 * 3. MSV stage, full recurrence (one target per wave, 64 lanes)
 *****************************************************************/
// The score table is staged in LDS (models of ND <= 16; larger ones run
// k_msv_full_wg). Bound by the row's chain of a long target alone: residues come
// 64 rows at a time and the scores a row ahead. Lists of 60,013 targets, M = 86: 95 us; 5,003 targets with longer
// ones, M = 50: 88 us (217 and 205 us with both fetched in the row, the floor at
// 0 as an instruction and a wave maximum every row).
template <int ND>
__global__ __launch_bounds__(512)
void k_msv_full(const DevProfile p, const int *__restrict__ tbl, int tbl_dwords,
                const uint8_t *__restrict__ res, const int64_t *__restrict__ off, const int32_t *__restrict__ len,
                const int32_t *__restrict__ list, const int32_t *__restrict__ count, int16_t *__restrict__ xj, LenCfg lc)
{
  const int lw = list_waves(*count);
  if ((int64_t) blockIdx.x * lw >= *count) return;
  extern __shared__ int lds[];
  const int *rows = lds;
  stage_table(lds, tbl, (size_t) tbl_dwords);
  const int z = threadIdx.x & 63;
  const int64_t n = *count;
  int32_t *queue = (int32_t *) count + P7G_QOFF;

  if ((int) (threadIdx.x >> 6) >= lw) return;
  for (int64_t t = queue_next(queue, 1); t < n; t = queue_next(queue, 1)) {
    const int slot = uni(list[t]);
    const int L = uni(len[slot]);
    const uint8_t *sq = res + off[slot];
    const int tjbm = ((lc.on ? lc.tjb : (int) p.tjb[L]) + p.tbm) & 0xff;
    int xJ = 0;
    int xB = max(p.base - tjbm, 0);
    // Values are held as M - 32768 in int16, so that the floor at 0 is the
    // saturation of the add. xJ (and so xB) only changes, and the overflow test
    // only fires, when the row's xE exceeds min(xJ + tec, 254 - bias): a ballot
    // on the lanes' packed maxima decides whether the wave maximum is needed.
    int mp[ND], e[ND];
#pragma unroll
    for (int d = 0; d < ND; d++) mp[d] = (int) NEG_PAIR;
    bool overflow = false;
    int xB2 = pair16(xB - 32768), th2 = pair16(min(xJ + p.tec, 254 - p.bias) - 32768);
    if (L > 0) {
      RowRes<false> rr;
      const int x0 = rr.init(sq, L, z, ND * 64);
#pragma unroll
      for (int d = 0; d < ND; d++) e[d] = rows[x0 + z + d * 64];
      for (int i0 = 0; i0 < L && ! overflow; i0 += 64) {
        const int cnt = min(64, L - i0);
        for (int u = 0; u < cnt; u++) {
          const int *en = rows + rr.ahead(u) + z;
          const int s0 = shift_in<64>(mp[ND-1], (int) NEG_PAIR);
          int E = (int) NEG_PAIR;
#pragma unroll
          for (int d = ND-1; d >= 0; d--) {
            const int tv = adds2(max2(d > 0 ? mp[d-1] : s0, xB2), e[d]);
            E = max2(E, tv);
            mp[d] = tv;
          }
          // the next row's scores, a row ahead
#pragma unroll
          for (int d = 0; d < ND; d++) e[d] = en[d * 64];
          if (__builtin_expect(__ballot(max2(E, th2) != th2) != 0ull, 0)) {
            const int xE = uni(wave_max_i(max(lo16(E), hi16(E)))) + 32768;
            if (xE + p.bias >= 255) { overflow = true; break; }
            xJ = max(xJ, max(xE - p.tec, 0));
            xB = max(max(p.base, xJ) - tjbm, 0);
            xB2 = pair16(xB - 32768); th2 = pair16(min(xJ + p.tec, 254 - p.bias) - 32768);
          }
        }
        rr.advance();
      }
    }
    if (z == 0) xj[slot] = (int16_t) (overflow ? -1 : xJ);
  }
}

// The full MSV recurrence for large models, W waves per target: wave w owns
// dwords [w·ND/W, (w+1)·ND/W) of every lane. A slice's first dword takes the
// previous row's last dword of the slice before it (slice 0: of the last
// slice, joined across lanes as shift_in does) from LDS, double-buffered by
// row parity, so one barrier per row orders the exchange. The lanes' row
// maxima travel in the same buffers, and xJ and xB are updated from them at
// the top of the next row (or after the last), in the same order as the
// one-wave kernel; results are bit-identical. Bound by the row's exchange;
// M = 2600, a target of 35,000 residues: 3.1 ms, 5.4 ms with the maxima reduced
// in every wave and residues and scores fetched in the row.
template <int ND, int W>
__global__ __launch_bounds__(64 * W)
void k_msv_full_wg(const DevProfile p, const int *__restrict__ tbl, const uint8_t *__restrict__ res,
                   const int64_t *__restrict__ off, const int32_t *__restrict__ len, const int32_t *__restrict__ list,
                   const int32_t *__restrict__ count, int16_t *__restrict__ xj, LenCfg lc)
{
  static_assert(ND % W == 0, "slices of equal width");
  constexpr int NW = ND / W;
  __shared__ int sh_end[2][W][65];       // each slice's last dword, by row parity; lane z at z + 1 (0: none)
  __shared__ int sh_el[2][W][64];        // each wave's row maxima per lane, by row parity
  __shared__ int64_t sh_t;
  if ((int64_t) blockIdx.x >= *count) return;
  const int wv = uni(threadIdx.x >> 6), z = threadIdx.x & 63;
  const int d0 = wv * NW;
  const int64_t n = *count;
  int32_t *queue = (int32_t *) count + P7G_QOFF;
  if (z == 0) sh_end[0][wv][0] = sh_end[1][wv][0] = (int) NEG_PAIR;

  for (;;) {
    if (threadIdx.x == 0) sh_t = (int64_t) atomicAdd(queue, 1);
    __syncthreads();
    const int64_t t = sh_t;
    if (t >= n) break;
    const int slot = uni(list[t]);
    const int L = uni(len[slot]);
    const uint8_t *sq = res + off[slot];
    const int tjbm = ((lc.on ? lc.tjb : (int) p.tjb[L]) + p.tbm) & 0xff;
    int xJ = 0;
    int xB = max(p.base - tjbm, 0);
    // values as M - 32768, and the threshold of a change of xJ, as in k_msv_full
    int mp[NW], e[NW];
#pragma unroll
    for (int j = 0; j < NW; j++) mp[j] = (int) NEG_PAIR;
    sh_end[1][wv][z + 1] = (int) NEG_PAIR;             // row -1
    bool overflow = false;
    int xB2 = pair16(xB - 32768), th2 = pair16(min(xJ + p.tec, 254 - p.bias) - 32768);
    // the update of xJ and xB when a row's maximum, left per lane in buffer b,
    // exceeds the threshold
    auto update = [&](int b) {
      int E = sh_el[b][0][z];
#pragma unroll
      for (int v = 1; v < W; v++) E = max2(E, sh_el[b][v][z]);
      if (__builtin_expect(__ballot(max2(E, th2) != th2) == 0ull, 1)) return;
      const int xE = uni(wave_max_i(max(lo16(E), hi16(E)))) + 32768;
      if (xE + p.bias >= 255) { overflow = true; return; }
      xJ = max(xJ, max(xE - p.tec, 0));
      xB = max(max(p.base, xJ) - tjbm, 0);
      xB2 = pair16(xB - 32768); th2 = pair16(min(xJ + p.tec, 254 - p.bias) - 32768);
    };
    if (L > 0) {
      RowRes<false> rr;
      const int x0 = rr.init(sq, L, z, ND * 64);
      const int *tz = tbl + (size_t) d0 * 64 + z;
#pragma unroll
      for (int j = 0; j < NW; j++) e[j] = tz[x0 + j * 64];
      for (int i0 = 0; i0 < L && ! overflow; i0 += 64) {
        const int cnt = min(64, L - i0);
        for (int u = 0; u < cnt; u++) {
          const int q = u & 1;                         // 64 is even: the buffers alternate
          lds_barrier();                               // the previous row's slice ends and maxima are written
          int s0;
          if (wv > 0) s0 = sh_end[q ^ 1][wv-1][z + 1];
          else s0 = (int) __builtin_amdgcn_alignbit((unsigned) sh_end[q ^ 1][W-1][z + 1], (unsigned) sh_end[q ^ 1][W-1][z], 16);
          if (i0 + u > 0) { update(q ^ 1); if (overflow) break; }
          int E = (int) NEG_PAIR;
#pragma unroll
          for (int j = NW-1; j >= 0; j--) {
            const int tv = adds2(max2(j ? mp[j-1] : s0, xB2), e[j]);
            E = max2(E, tv);
            mp[j] = tv;
          }
          const int *en = tz + rr.ahead(u);            // the next row's scores, a row ahead
#pragma unroll
          for (int j = 0; j < NW; j++) e[j] = en[j * 64];
          sh_end[q][wv][z + 1] = mp[NW-1];
          sh_el[q][wv][z] = E;
        }
        rr.advance();
      }
      if (! overflow) {
        lds_barrier();
        update((L - 1) & 1);
      }
    }
    if (threadIdx.x == 0) xj[slot] = (int16_t) (overflow ? -1 : xJ);
    __syncthreads();                                   // sh_t and the buffers are free for the next target
  }
}

// MSV scores of listed targets from their final xJ (msvfilter.c:203-207,
// with the per-target length model): ((xJ - tjb) - base) / scale_b - 3 nats
// in float, the last step in double as the reference's `-= 3.0`; +inf and
// status 16 (eslERANGE) where the recurrence overflowed.
__global__ void k_msv_scores(const DevProfile p, const int32_t *__restrict__ len, const int32_t *__restrict__ slots,
                             int64_t n, const int16_t *__restrict__ xj, float *__restrict__ sc, int *__restrict__ st)
{
#pragma clang fp contract(off)
  for (int64_t t = (int64_t) blockIdx.x * blockDim.x + threadIdx.x; t < n; t += (int64_t) gridDim.x * blockDim.x) {
    const int slot = slots[t];
    const int v = xj[slot];
    if (v < 0) { sc[t] = __int_as_float(0x7f800000); st[t] = 16; continue; }
    float f = (float) (v - (int) p.tjb[len[slot]]) - (float) p.base;
    f = __fdiv_rn(f, p.scale_b);
    sc[t] = (float) ((double) f - 3.0);
    st[t] = 0;
  }
}

/*****************************************************************
 * 4. MSV gate: score, null score, F1 (and F2 when the bias filter is off)
 *****************************************************************/
__global__ void k_msv_gate(const DevProfile p, const int32_t *__restrict__ len, int64_t n,
                           const int16_t *__restrict__ xj, DevResults r, DevLists l, GateThresh g)
{
#pragma clang fp contract(off)
  for (int64_t slot = (int64_t) blockIdx.x * blockDim.x + threadIdx.x; slot < n; slot += (int64_t) gridDim.x * blockDim.x) {
    const int L = len[slot];
    const int v = xj[slot];
    const float nullsc = p.nullsc[L];
    float usc;
    if (v < 0) usc = INFINITY;
    else {
      usc = __fdiv_rn((float) (v - (int) p.tjb[L]) - (float) p.base, p.scale_b);
      usc = (float) ((double) usc - 3.0);
    }
    r.usc[slot] = usc;
    r.nullsc[slot] = nullsc;
    uint8_t stage = 0;
    bool to_bias = false, to_vit = false, to_fwd = false;
    if (L > 0) {
      const float seq = (float) __ddiv_rn((double) (usc - nullsc), LOG2_D);
      if (seq >= g.T1m) {
        stage = 1;
        if (g.do_bias) to_bias = true;
        else {
          r.filtersc[slot] = nullsc;
          if (seq >= g.T2m) { to_fwd = true; stage = 3; }
          else              { to_vit = true; stage = 2; }
        }
      }
    }
    (void) to_bias; (void) to_vit; (void) to_fwd;   // the next lists are compacted from stage[]
    r.stage[slot] = stage;
  }
}

/*****************************************************************
 * 5. Bias-composition filter: 2-state HMM Forward with per-row max
 *    normalisation (easel/esl_hmm.c:351-409, HMMER/src/p7_bg.c:473-484).
 *    Float arithmetic in the reference's order, in two passes:
 *    k_bias runs the recurrence, one target per pair of lanes, and stores each
 *    row's normaliser; k_bias_sum takes the logs of a target's normalisers
 *    on all lanes at once and adds them in row order, as the reference does.
 *    The log is off the recurrence's serial chain, which bounds the stage.
 *****************************************************************/
__device__ __forceinline__ void bias_finish(const DevProfile &p, DevResults &r, const GateThresh &g, int gating,
                                            const LenCfg &lc, int slot, int L, float logsc)
{
#pragma clang fp contract(off)
  // with a caller-supplied length model the host adds the length terms
  const float filtersc = lc.on ? logsc : (logsc + p.flen_a[L]) + p.flen_b[L];
  r.filtersc[slot] = filtersc;
  if (gating) {
    const float seq = (float) __ddiv_rn((double) (r.usc[slot] - filtersc), LOG2_D);
    if (seq < g.T1m)       r.stage[slot] = 1;
    else if (seq >= g.T2m) r.stage[slot] = 3;       // the lists of the next stages are compacted from stage[]
    else                   r.stage[slot] = 2;
  }
}

// n / m, correctly rounded, for n <= m in the range that bias_ok and the length
// model's test set up: no intermediate is subnormal, so that the residuals are
// exact and no operand needs scaling. The quotient is corrected twice by its
// exact residual (P. Markstein, Computation of elementary functions on the IBM
// RISC System/6000, IBM J. Res. Dev. 34, 1990).
__device__ __forceinline__ float div_in_range(float n, float m)
{
  float y = __builtin_amdgcn_rcpf(m);
  y = __builtin_fmaf(__builtin_fmaf(-m, y, 1.0f), y, y);
  float q = n * y;
  q = __builtin_fmaf(__builtin_fmaf(-m, q, n), y, q);
  return __builtin_fmaf(__builtin_fmaf(-m, q, n), y, q);
}

// Two lanes per target: the even lane holds state 0, the odd one state 1, and a
// row takes the other state's value with a DPP operand. A target's rows are one
// serial chain and a wave runs alone on its SIMD for most lists, so the stage is
// bound by the instructions of a row, 15 here. A row of one target: 104 ns with
// both states and both divisions in one lane, 47 ns now.
__global__ __launch_bounds__(64)
void k_bias(const DevProfile p, const uint8_t *__restrict__ res, const int64_t *__restrict__ off,
            const int32_t *__restrict__ len, const int32_t *__restrict__ list, const int32_t *__restrict__ count,
            DevResults r, GateThresh g, int gating, LenCfg lc,
            float *__restrict__ rowmax, int64_t rowmax_size, unsigned long long *cursor, int64_t *__restrict__ defer_off)
{
#pragma clang fp contract(off)
  constexpr int OTHER = 0xB1;                    // quad_perm [1, 0, 3, 2]: the pair's other lane
  // the two states' odds of every residue code, in LDS
  __shared__ float eo2[2 * P7G_NROWS];
  for (int x = threadIdx.x; x < 2 * P7G_NROWS; x += blockDim.x) eo2[x] = p.eo[x];
  __syncthreads();
  const int64_t n = *count;
  const int lane = threadIdx.x & 63, s = lane & 1;
  for (int64_t t0 = (int64_t) blockIdx.x * 32; t0 < n; t0 += (int64_t) gridDim.x * 32) {
    const int64_t t = t0 + (lane >> 1);
    const bool valid = t < n;
    const int slot = valid ? list[t] : 0;
    const int L = valid ? len[slot] : 0;
    // room for L row normalisers and the final sum: one bump of the cursor per wave
    int64_t base = -1;
    if (rowmax) {
      // whole 16-row blocks and the closing sum, in 16-byte aligned pieces
      const int64_t need = valid ? 16 * (((int64_t) L + 15) >> 4) + 4 : 0;
      int64_t incl = s ? 0 : need;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) { const int64_t v = __shfl_up(incl, o, 64); if (lane >= o) incl += v; }
      unsigned long long b0 = 0;
      if (lane == 63) b0 = atomicAdd(cursor, (unsigned long long) incl);
      b0 = __shfl(b0, 63, 64);
      const int64_t mine = (int64_t) b0 + incl - need;
      if (valid && mine + need <= rowmax_size) base = mine;
    }
    if (! valid) continue;
    const uint8_t *sq = res + off[slot];
    const float p1  = lc.on ? lc.p1 : __fdiv_rn((float) L, (float) (L + 1));
    const float t00 = p1, t01 = lc.on ? lc.q1 : 1.0f - p1;
    // this state's transitions from itself and from the other state
    const float ts = s ? p.ft1_1 : t00, to = s ? t01 : p.ft1_0;
    float *rm = (base >= 0) ? rowmax + base : nullptr;
    float logsc = 0.0f;
    // Row 0 runs the same arithmetic as the others with the identity for the
    // transitions and (pi0, pi1) for the previous row: ((0 + pi0*1) + pi1*0)
    // * e0 is exactly pi0 * e0, the reference's first row.
    float d = s ? p.pi1 : p.pi0;
    float Ts = 1.0f, To = 0.0f;
    float fin = d;                               // d after the target's last row
    float mx;
    // a row in the reference's order for any odds
    auto row_any = [&](float e) {
      const float ds = d * Ts, dot = dppz<OTHER>(d) * To;
      const float nn = ((0.0f + (s ? dot : ds)) + (s ? ds : dot)) * e;
      const float no = dppz<OTHER>(nn), n0 = s ? no : nn, n1 = s ? nn : no;
      mx = 0.0f; mx = (n0 > mx) ? n0 : mx; mx = (n1 > mx) ? n1 : mx;
      d = __fdiv_rn(nn, mx);
      Ts = ts; To = to;
    };
    // the same for odds and transitions in range, all positive, so that the
    // values' bit patterns order as integers
    auto row_fast = [&](float e) {
      const float nn = (d * Ts + dppz<OTHER>(d) * To) * e;
      const int ni = __float_as_int(nn);
      mx = __int_as_float(max(ni, dppi<OTHER>(0, ni)));
      d = div_in_range(nn, mx);
    };
    const uint4 *pc = (const uint4 *) sq;
    const int nblk = (L + 15) >> 4;
    const bool ok = p.bias_ok && t00 >= 0x1p-2f && t00 <= 1.0f && t01 >= 0x1p-32f && t01 <= 1.0f;
    if (rm && __all(ok)) {
      // Straight-line blocks of 16 rows, so that the compiler can count the
      // memory operations in flight. At the top of block bk every access in
      // flight was issued a whole block earlier: the block's residue chunk,
      // and the stores of block bk-2's normalisers. The block then reads its
      // odds from LDS, requests the next chunk, stores block bk-1's
      // normalisers (block 0 writes its own slot, rewritten a block later),
      // and runs its rows. Rows past the end compute values no one reads,
      // into the target's own whole-block room.
      uint4 cn = pc[0];
      const float *es = eo2 + s;
      float qp[16];
#pragma unroll
      for (int u = 0; u < 16; u++) qp[u] = 0.0f;
      auto put = [&](int bk) {
        if (s) return;
        float4 *o = (float4 *) (rm + bk * 16);
        o[0] = make_float4(qp[0], qp[1], qp[2], qp[3]);     o[1] = make_float4(qp[4], qp[5], qp[6], qp[7]);
        o[2] = make_float4(qp[8], qp[9], qp[10], qp[11]);   o[3] = make_float4(qp[12], qp[13], qp[14], qp[15]);
      };
      auto block = [&](int bk, auto last) {
        float eb[16];
#pragma unroll
        for (int u = 0; u < 16; u++) eb[u] = es[2 * chunk_byte(cn, u)];
        cn = pc[min(bk + 1, nblk)];             // the chunk after the target is still readable
        put(max(bk - 1, 0));
#pragma unroll
        for (int u = 0; u < 16; u++) {
          row_fast(eb[u]);
          qp[u] = mx;
          if (u == 0) { Ts = ts; To = to; }
          if (decltype(last)::value) fin = (bk * 16 + u == L - 1) ? d : fin;
        }
      };
      for (int bk = 0; bk < nblk - 1; bk++) block(bk, std::false_type());
      if (nblk > 0) { block(nblk - 1, std::true_type()); put(nblk - 1); }
    } else if (rm) {
      // odds out of range: row by row
      for (int i = 0; i < L; i++) {
        row_any(eo2[2 * chunk_byte(pc[i >> 4], i) + s]);
        if (! s) rm[i] = mx;
      }
      fin = d;
    } else {
      // no room for the normalisers (pool exhausted): their logs are summed here
      for (int i = 0; i < L; i++) {
        row_any(eo2[2 * chunk_byte(pc[i >> 4], i) + s]);
        logsc += (float) log((double) mx);
      }
      fin = d;
    }
    // the closing sum; an empty target scores log(pi_end) = log(0) (esl_hmm.c:360-364)
    const float fo = dppz<OTHER>(fin);
    float sfin = 0.0f;
    if (L > 0) { sfin += (s ? fo : fin) * 1.0f; sfin += (s ? fin : fo) * 1.0f; }
    if (s) continue;
    if (rm) {
      rm[L] = sfin;                            // after the block stores of the same lane
      defer_off[slot] = base;                  // k_bias_log + k_bias_sum finish it
      continue;
    }
    if (rowmax) defer_off[slot] = -1;
    logsc += (float) log((double) sfin);
    bias_finish(p, r, g, gating, lc, slot, L, logsc);
  }
}

// Every stored value replaced by float(log(double(v))), in parallel.
__global__ __launch_bounds__(256)
void k_bias_log(float *__restrict__ rowmax, const unsigned long long *__restrict__ used, int64_t cap)
{
  const int64_t n = min((int64_t) *used, cap);
  for (int64_t i = (int64_t) blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t) gridDim.x * blockDim.x)
    rowmax[i] = (float) log((double) rowmax[i]);
}

// One target per wave: its L+1 logs added in row order, as esl_hmm_Forward
// sums sc[1..L+1] (esl_hmm.c:403-405), so the order of the float additions is the
// reference's and their latency bounds a long target. The wave loads 256 terms
// ahead and passes them through LDS 64 at a time, from which every lane reads
// them back four at a time and adds them all: an addition and a quarter of a
// read per term. 35,000 terms: 121 us, 661 us with each term taken out of its
// lane by v_readlane.
__global__ __launch_bounds__(256)
void k_bias_sum(const DevProfile p, const int32_t *__restrict__ len, const int32_t *__restrict__ list,
                const int32_t *__restrict__ count, DevResults r, GateThresh g, int gating, LenCfg lc,
                const float *__restrict__ rowmax, const int64_t *__restrict__ defer_off)
{
#pragma clang fp contract(off)
  __shared__ __attribute__((aligned(16))) float sh[4][2][64];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int64_t n = *count;
  for (int64_t t = wave_id(); t < n; t += wave_cnt()) {
    const int slot = uni(list[t]);
    const int64_t o0 = defer_off[slot];
    const int64_t o = ((int64_t) (unsigned) uni((int) (o0 >> 32)) << 32) | (unsigned) uni((int) o0);
    if (o < 0) continue;                       // finished in the first pass
    const int L = uni(len[slot]);
    const int nv = L + 1;                      // L row terms and the closing sum
    const float *rw = rowmax + o;
    float logsc = 0.0f;
    float v[4], nx[4];
#pragma unroll
    for (int j = 0; j < 4; j++) v[j] = rw[min(64 * j + lane, L)];
    for (int base = 0; base < nv; base += 256) {
#pragma unroll
      for (int j = 0; j < 4; j++) nx[j] = rw[min(base + 256 + 64 * j + lane, L)];
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const int cnt = min(64, nv - base - 64 * j);
        float *w = sh[wv][j & 1];
        w[lane] = v[j];
        // a wave's LDS operations complete in order: only the compiler is held
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
        if (cnt == 64) {
          float x[64];
#pragma unroll
          for (int k = 0; k < 64; k++) x[k] = w[k];
#pragma unroll
          for (int k = 0; k < 64; k++) logsc += x[k];
        } else
          for (int k = 0; k < cnt; k++) logsc += readlanef(v[j], k);
        v[j] = nx[j];
      }
    }
    if (lane == 0) bias_finish(p, r, g, gating, lc, slot, L, logsc);
  }
}

/*****************************************************************
 * 9. Domain decoding and regions (F3 survivors, one target per wave)
 *****************************************************************/
// p7_DomainDecoding (HMMER/src/impl_sse/decoding.c:166-197) from the two
// parsers' special rows: btot[i] / etot[i], the expected B / E visits up to
// row i, and mocc[i], the probability that residue i is emitted by the core
// model. Each row's terms are the reference's float products; the running
// sums over rows are taken 64 rows at a time by a wave scan (the reference
// adds them one by one, so the sums may differ in the last bits). When the
// Backward parser used its own scale factors the scale product changes from
// row to row, and the first lane walks the rows in the reference's order.
// Then the region loop of p7_domaindef_ByPosteriorHeuristics
// (p7_domaindef.c:409-489): its three occupancy tests are evaluated for 64
// rows at once into ballots, and the loop's state machine steps through
// their bits; a region's is_multidomain_region test (:534-547) is a wave
// maximum over its split points. Thresholds rt1/rt2/rt3 of
// p7_domaindef_Create (:109-111). Regions are appended as {slot, i, j,
// multidomain} records, each with a 16-byte aligned copy of its residues and
// the unihit N/J/C odds of its target's length, for the envelope scores that
// k_fwd (MODE 2) computes next.
#define DOM_RT1 0.25f
#define DOM_RT2 0.10f
#define DOM_RT3 0.20f
__global__ __launch_bounds__(256)
void k_domains(const DevProfile p, const uint8_t *__restrict__ res, const int64_t *__restrict__ off,
               const int32_t *__restrict__ len, const int32_t *__restrict__ list,
               const int32_t *__restrict__ count, const int *__restrict__ fstatus, DevLists l, LenCfg lc,
               DomBufs dom, DomOut out)
{
#pragma clang fp contract(off)
  enum { E = 0, N = 1, J = 2, Bx = 3, C = 4, S = 5 };
  const int lane = threadIdx.x & 63;
  const int64_t n = *count;
  for (int64_t t = wave_id(); t < n; t += wave_cnt()) {
    const int slot = uni(list[t]);
    const int L = uni(len[slot]);
    const int64_t fo = dom.doff[slot], bo = dom.boff[slot];
    if (fo < 0 || bo < 0) {
      if (lane == 0) { out.nexp[slot] = NAN; out.nreg[slot] = -1; out.nclu[slot] = -1; }
      continue;
    }
    const float *fx = dom.pool + fo;
    const float *bx = dom.pool + bo;
    float *btot = dom.pool + bo + 6 * (int64_t) (L + 1), *etot = btot + (L + 1), *mocc = etot + (L + 1);
    const bool own = (fstatus[slot] & 0x100) != 0;
    const float loop = lc.on ? lc.floop : p.xf_loop[L];     // N, J and C loops are equal after ReconfigLength
    // N/J/C odds of p7_oprofile_ReconfigUnihit(om, L) (impl_sse/p7_oprofile.c:1176-1186,
    // 1113-1114: nj = 0) for the envelope scores of this target's regions
    const float umove = __fdiv_rn(2.0f + 0.0f, (float) L + 2.0f + 0.0f), uloop = 1.0f - umove;
    const float sp0 = __fdiv_rn(1.0f, bx[N]);
    if (lane == 0) { btot[0] = 0.0f; etot[0] = 0.0f; mocc[0] = 0.0f; }
    if (! own) {
      float cb = 0.0f, ce = 0.0f;                           // btot, etot at the row before the block
      for (int base = 0; base < L; base += 64) {
        const int i = base + lane + 1;
        float db = 0.0f, de = 0.0f, mo = 0.0f;
        if (i <= L) {
          const float *f0 = fx + (size_t) (i - 1) * 6, *f1 = fx + (size_t) i * 6;
          const float *b0 = bx + (size_t) (i - 1) * 6, *b1 = bx + (size_t) i * 6;
          db = f0[Bx] * b0[Bx] * f0[S] * sp0;
          de = f1[E] * b1[E] * f1[S] * sp0;
          float njcp = f0[N] * b1[N] * loop * sp0;
          njcp += f0[J] * b1[J] * loop * sp0;
          njcp += f0[C] * b1[C] * loop * sp0;
          mo = 1.0f - njcp;
        }
        const float bt = cb + wave_scan_f(db), et = ce + wave_scan_f(de);
        if (i <= L) { btot[i] = bt; etot[i] = et; mocc[i] = mo; }
        cb = readlanef(bt, 63); ce = readlanef(et, 63);
      }
    } else if (lane == 0) {
      float sp = sp0, bt = 0.0f, et = 0.0f;
      for (int i = 1; i <= L; i++) {
        const float *f0 = fx + (size_t) (i - 1) * 6, *f1 = fx + (size_t) i * 6;
        const float *b0 = bx + (size_t) (i - 1) * 6, *b1 = bx + (size_t) i * 6;
        bt = bt + (f0[Bx] * b0[Bx] * f0[S] * sp);
        sp *= __fdiv_rn(f0[S], b0[S]);
        et = et + (f1[E] * b1[E] * f1[S] * sp);
        float njcp = f0[N] * b1[N] * loop * sp;
        njcp += f0[J] * b1[J] * loop * sp;
        njcp += f0[C] * b1[C] * loop * sp;
        btot[i] = bt; etot[i] = et; mocc[i] = 1.0f - njcp;
      }
    }
    __threadfence_block();                                  // the rows above are read back by other lanes
    if (lane == 0) out.nexp[slot] = btot[L];

    int nreg = 0, nclu = 0, i0 = -1;
    bool triggered = false;
    for (int base = 0; base < L; base += 64) {
      const int j = base + lane + 1;
      bool cs = false, ct = false, ce = false;
      if (j <= L) {
        const float mo = mocc[j];
        cs = mo - (btot[j] - btot[j-1]) < DOM_RT2;
        ct = mo >= DOM_RT1;
        ce = mo - (etot[j] - etot[j-1]) < DOM_RT2;
      }
      const unsigned long long ms = __ballot(cs), mt = __ballot(ct), me = __ballot(ce);
      const int nr = min(64, L - base);
      for (int r = 0; r < nr; r++) {                       // the loop's steps, on wave-uniform values
        const int jj = base + r + 1;
        if (! triggered) {
          if      ((ms >> r) & 1ull) i0 = jj;
          else if (i0 == -1)         i0 = jj;
          if      ((mt >> r) & 1ull) triggered = true;
        } else if ((me >> r) & 1ull) {
          // is_multidomain_region(i0, jj): max over split points z of
          // min(etot[z] - etot[i0-1], btot[jj] - btot[z-1])
          const float e0 = etot[i0 - 1], bj = btot[jj];
          float mx = -1.0f;
          for (int z0 = i0; z0 <= jj; z0 += 64) {
            const int z = z0 + lane;
            float en = -1.0f;
            if (z <= jj) {
              const float a = etot[z] - e0, b = bj - btot[z - 1];
              en = (a < b) ? a : b;
            }
            mx = fmaxf(mx, en);
          }
          {
            float v = mx;
            v = fmaxf(v, __shfl_xor(v, 1, 64)); v = fmaxf(v, __shfl_xor(v, 2, 64)); v = fmaxf(v, __shfl_xor(v, 4, 64));
            v = fmaxf(v, __shfl_xor(v, 8, 64)); v = fmaxf(v, __shfl_xor(v, 16, 64)); v = fmaxf(v, __shfl_xor(v, 32, 64));
            mx = unif(v);
          }
          const int multi = (mx >= DOM_RT3) ? 1 : 0;
          // record the region, and copy its residues for the envelope score
          const int Ld = jj - i0 + 1;
          const int64_t need = (((int64_t) Ld + 15) & ~(int64_t) 15) + 16;
          int k = 0;
          unsigned long long ro64 = 0;
          if (lane == 0) {
            k = atomicAdd(&out.ecount[0], 1);
            if (multi) atomicAdd(out.nclu_total, 1);
            if (k < out.reg_cap) ro64 = atomicAdd(l.cursor + 2, (unsigned long long) need);
          }
          k = uni(k);
          const int64_t ro = ((int64_t) (unsigned) uni((int) (ro64 >> 32)) << 32) | (unsigned) uni((int) ro64);
          if (k >= out.reg_cap) { if (lane == 0) atomicOr(&l.counts[7], 2); }
          else {
            const bool fits = ro + need <= out.res_cap;
            if (fits) {
              const uint8_t *src = res + off[slot] + (i0 - 1);
              for (int64_t b = lane; b < need; b += 64) out.res[ro + b] = (b < Ld) ? src[b] : (uint8_t) P7G_PADCODE;
            }
            if (lane == 0) {
              out.regs[k] = make_int4(slot, i0, jj, multi);
              out.v_off[k] = fits ? ro : 0; out.v_len[k] = fits ? Ld : 0; out.v_list[k] = k;
              out.env_loop[k] = uloop; out.env_move[k] = umove;
              if (! fits) atomicOr(&l.counts[7], 4);
            }
          }
          nreg++; nclu += multi;
          i0 = -1; triggered = false;
        }
      }
    }
    if (lane == 0) { out.nreg[slot] = nreg; out.nclu[slot] = nclu; }
  }
}


__global__ void k_fill32(uint32_t *__restrict__ p, uint32_t v, int64_t n)
{
  for (int64_t i = (int64_t) blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t) gridDim.x * blockDim.x) p[i] = v;
}

__global__ void k_copy32(uint32_t *__restrict__ d, const uint32_t *__restrict__ s, int64_t n)
{
  for (int64_t i = (int64_t) blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t) gridDim.x * blockDim.x) d[i] = s[i];
}

/*****************************************************************
 * Launchers
 *****************************************************************/
hipError_t launch_fill32(void *p, uint32_t v, int64_t nwords, hipStream_t st)
{
  if (nwords <= 0) return hipSuccess;
  const unsigned grid = (unsigned) std::min<int64_t>((nwords + 255) / 256, 4096);
  hipLaunchKernelGGL(k_fill32, dim3(grid), dim3(256), 0, st, (uint32_t *) p, v, nwords);
  return hipGetLastError();
}

// The start of a single-target call, one launch in place of seven copies and
// fills with a synchronisation among them: its residues and, when given, a second
// array, read from pinned host memory in 16-byte words; the target's offset and
// length; the cleared counts and cursor; and the stage's list of slot 0. The
// single targets' fixed cost is the launches and copies around their stages:
// five calls of 350 residues at M = 86 took 690 us, and 384 us with these kernels.
__global__ __launch_bounds__(256)
void k_single_in(SingleIn a)
{
  const int64_t i0 = (int64_t) blockIdx.x * blockDim.x + threadIdx.x, step = (int64_t) gridDim.x * blockDim.x;
  for (int64_t i = i0; i < a.n1; i += step) ((uint4 *) a.dst1)[i] = ((const uint4 *) a.src1)[i];
  for (int64_t i = i0; i < a.n2; i += step) ((uint4 *) a.dst2)[i] = ((const uint4 *) a.src2)[i];
  if (i0 < 16) {
    a.counts[i0] = (a.list && i0 == a.which) ? 1 : 0;
    ((uint32_t *) a.cursor)[i0] = 0u;
  }
  if (i0 == 0) {
    *a.off = 0; *a.len = a.L;
    if (a.list) a.list[0] = 0;
  }
}
// Its end: two result words and, when given, rows of floats, to pinned host memory.
__global__ __launch_bounds__(256)
void k_single_out(SingleOut a)
{
  const int64_t i0 = (int64_t) blockIdx.x * blockDim.x + threadIdx.x, step = (int64_t) gridDim.x * blockDim.x;
  for (int64_t i = i0; i < a.n; i += step) a.dst[i] = a.src[i];
  if (i0 == 0) { a.words[0] = a.half ? (int32_t) *(const int16_t *) a.w0 : *(const int32_t *) a.w0; a.words[1] = a.w1 ? *a.w1 : 0; }
}

hipError_t launch_single_in(const SingleIn &a, hipStream_t st)
{
  const unsigned grid = (unsigned) std::min<int64_t>((std::max(a.n1, a.n2) + 255) / 256 + 1, 64);
  hipLaunchKernelGGL(k_single_in, dim3(grid), dim3(256), 0, st, a);
  return hipGetLastError();
}
hipError_t launch_single_out(const SingleOut &a, hipStream_t st)
{
  const unsigned grid = (unsigned) std::min<int64_t>(a.n / 256 + 1, 64);
  hipLaunchKernelGGL(k_single_out, dim3(grid), dim3(256), 0, st, a);
  return hipGetLastError();
}

hipError_t launch_copy32(void *dst, const void *src, int64_t nwords, hipStream_t st)
{
  if (nwords <= 0) return hipSuccess;
  const unsigned grid = (unsigned) std::min<int64_t>((nwords + 255) / 256, 4096);
  hipLaunchKernelGGL(k_copy32, dim3(grid), dim3(256), 0, st, (uint32_t *) dst, (const uint32_t *) src, nwords);
  return hipGetLastError();
}

// p7_OATrace (impl_sse/optacc.c:227-276) over the choices the null2 pass
// stored (oa_row), one wave per region, from C at the region's last residue
// back to S; keeps the first and last M states (p7_alidisplay_Create's
// hmmfrom/hmmto/sqfrom/sqto, p7_alidisplay.c:74-145), and writes the
// alignment itself for the display, from its last M state back to its first
// (p7_alidisplay_Create's z2 down to z1), one word per state: state (0 M,
// 1 I, 2 D) in bits 0-1, model position in bits 2-18, the cell's posterior
// probability code in bits 19-22, the residue code in bits 23-27; at most
// n2pcap words at n2path + n2poff[region], their number to n2pn[region]
// (0 without an alignment).
//
// The walk is one thread's, kept uniform over the wave; the wave's lanes
// speculate on runs: in M, lane l loads the choice at (i-l, k-l), and the
// leading lanes whose choice is M -> M take their steps at once, each writing
// its state's word; in C, lane l reads row i-l's C -> C bit likewise. A run's
// lanes stop wherever the step-by-step walk would fail (bounds, the word
// cap, the step guard), so that the walk itself meets every failure.
__global__ void __launch_bounds__(64) k_oa_trace(const DevProfile p, const int32_t *__restrict__ list, int64_t n,
                           const int32_t *__restrict__ vlen, const uint8_t *__restrict__ vres,
                           const int64_t *__restrict__ voff, DomBufs dom)
{
  enum { S_S = 0, S_N, S_B, S_M, S_I, S_D, S_E, S_J, S_C };
  const int64_t t = (int64_t) blockIdx.x;
  const int lane = (int) threadIdx.x;
  if (t >= n) return;
  const int slot = list[t];
  int4 out = make_int4(0, 0, 0, 0);
  if (dom.n2st[slot] != 0) {                           // no decoding, no trace
    if (lane == 0) { dom.n2ali[slot] = out; dom.n2pn[slot] = 0; }
    return;
  }
  const int L = vlen[slot], B = p.fb_B, NW = n2_oa_words(B);
  const float *area = dom.n2pool + dom.n2off[slot];
  const uint32_t *bits = (const uint32_t *) (area + n2_oa_bits_at(L, B));
  const uint32_t *rows = (const uint32_t *) (area + n2_oa_rows_at(L, B));
  const uint32_t *pp = (const uint32_t *) (area + n2_pp_at(L, B));
  const uint8_t *sq = vres + voff[slot];               // residue i at sq[i-1]
  uint32_t *path = dom.n2path + dom.n2poff[slot];
  const int pcap = L + p.M + 2;
  auto cell = [&](int i, int k) -> uint32_t {
    const int z = (k - 1) / B, j = (k - 1) % B;
    return (bits[((size_t) (i - 1) * NW + j / 8) * 64 + z] >> ((j % 8) * 4)) & 15u;
  };
  const int NP = n2_pp_words(B);
  auto ppat = [&](int i, int k) -> uint32_t {
    const int z = (k - 1) / B, j = (k - 1) % B;
    return (pp[((size_t) (i - 1) * NP + j / 4) * 64 + z] >> ((j % 4) * 8)) & 0xffu;
  };
  int i = L, k = 0, s0 = S_C, nm = 0, ok = 1, nw = 0, last = 0;
  bool rec = false;                    // s0 is a display state still to be written
  bool spec = true;                    // a run may start here (false just after a broken run)
  const int guard = 4 * (L + p.M) + 8;
  for (int step = 0; s0 != S_S; step++) {
    int s1;
    if (step > guard || i < 0) { ok = 0; break; }
    if (spec && s0 == S_M && rec) {
      // M -> M steps from (i, k): the one from (i-l, k-l) needs both cells in
      // the model and the matrix, its record below the cap, its step within
      // the guard; each writes the word of the state it leaves
      const int lim = min(min(64, pcap - nw - 1), guard - step + 1);
      const int ii = i - lane, kk = k - lane;
      bool go = false;
      uint32_t wd = 0;
      if (lane < lim && ii >= 2 && kk >= 2 && kk <= p.M) {
        const uint32_t c = cell(ii, kk), b = ppat(ii, kk), x = (uint32_t) sq[ii - 1];
        go = (c & 3u) == 0u;
        wd = ((uint32_t) kk << 2) | ((b & 15u) << 19) | (x << 23);
      }
      const unsigned long long stop = __ballot(! go);
      const int r = stop ? (int) __ffsll((long long) stop) - 1 : 64;
      if (r > 0) {
        if (lane < r) path[nw + lane] = wd;
        nw += r; last = nw; nm += r; i -= r; k -= r;
        out.x = k; out.z = i;
        spec = (r == 64);
        step += r - 1;
        continue;
      }
    }
    if (spec && s0 == S_C) {
      // C -> C steps from row i down: row i-l's C bit, the next row in the
      // matrix, the step within the guard
      const int lim = min(64, guard - step + 1);
      const int ii = i - lane;
      const bool go = lane < lim && ii >= 1 && ((rows[ii] >> OA_CBIT) & 1u);
      const unsigned long long stop = __ballot(! go);
      const int r = stop ? (int) __ffsll((long long) stop) - 1 : 64;
      if (r > 0) {
        i -= r;
        spec = (r == 64);
        step += r - 1;
        continue;
      }
    }
    spec = true;
    // the display word of s0 (entered last step) is written here, so that its
    // loads and s0's choice loads go out together
    const bool mid = (s0 == S_M || s0 == S_I || s0 == S_D) && i >= 1 && k >= 1 && k <= p.M;
    const uint32_t cw = mid ? cell(i, k) : 0u;
    if (rec) {
      const uint32_t b = (s0 == S_D) ? 0u : ppat(i, k);
      const uint32_t st = (s0 == S_M) ? 0u : (s0 == S_I) ? 1u : 2u;
      const uint32_t code = (s0 == S_M) ? (b & 15u) : (s0 == S_I) ? (b >> 4) : 0u;
      const uint32_t x = (s0 == S_D) ? 0u : (uint32_t) sq[i - 1];
      if (lane == 0) path[nw] = st | ((uint32_t) k << 2) | (code << 19) | (x << 23);
      nw++;
      if (s0 == S_M) last = nw;
      rec = false;
    }
    switch (s0) {
      case S_C: s1 = ((rows[i] >> OA_CBIT) & 1u) ? S_C : S_E; break;
      case S_E: {
        const uint32_t r = rows[i];
        if ((r >> OA_EFAIL) & 1u) { ok = 0; break; }
        s1 = ((r >> OA_ESTATE) & 1u) ? S_D : S_M;
        k = (int) (r & 0xffffu);
        break;
      }
      case S_M: {
        if (i < 1 || k < 1 || k > p.M) { ok = 0; break; }
        const int c = (int) (cw & 3u);
        s1 = (c == 0) ? S_M : (c == 1) ? S_I : (c == 2) ? S_D : S_B;
        k--; i--;
        break;
      }
      case S_D:
        if (i < 1 || k < 1 || k > p.M) { ok = 0; break; }
        s1 = ((cw >> 3) & 1u) ? S_D : S_M;
        k--;
        break;
      case S_I:
        if (i < 1 || k < 1 || k > p.M) { ok = 0; break; }
        s1 = ((cw >> 2) & 1u) ? S_I : S_M;
        i--;
        break;
      case S_B: s1 = ((rows[i] >> OA_BBIT) & 1u) ? S_N : S_J; break;
      case S_N: s1 = (i == 0) ? S_S : S_N; break;
      case S_J: s1 = ((rows[i] >> OA_JBIT) & 1u) ? S_J : S_E; break;
      default: ok = 0; s1 = S_S; break;
    }
    if (! ok) break;
    if (s1 == S_M) {                     // walking back: the first M is the alignment's last
      if (nm == 0) { out.y = k; out.w = i; }
      out.x = k; out.z = i;
      nm++;
    }
    // the display's states: from the first M walked back to (states before
    // it are the E -> D end, not shown) to the last (B precedes it)
    if ((s1 == S_M || ((s1 == S_I || s1 == S_D) && nm > 0))) {
      if (i < 1 || k < 1 || k > p.M || nw >= pcap) { ok = 0; break; }
      rec = true;                        // its word, at the next step
    }
    if ((s1 == S_N || s1 == S_J || s1 == S_C) && s1 == s0) i--;
    s0 = s1;
  }
  if (! ok || nm == 0) { out = make_int4(0, 0, 0, 0); last = 0; }
  if (lane == 0) { dom.n2ali[slot] = out; dom.n2pn[slot] = last; }
}

hipError_t launch_oa_trace(const DevProfile &p, const DevSeqs &s, const int32_t *list, int64_t n, const DomBufs &dom,
                           hipStream_t st)
{
  if (n <= 0) return hipSuccess;
  if (n > 0x7fffffff) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_oa_trace, dim3((unsigned) n), dim3(64), 0, st, p, list, n, s.len, s.res, s.off, dom);
  return hipGetLastError();
}

hipError_t launch_msv_scores(const DevProfile &p, const DevSeqs &s, const int32_t *slots, int64_t n,
                             const int16_t *xj, float *sc, int *st, hipStream_t stream)
{
  if (n <= 0) return hipSuccess;
  unsigned grid = (unsigned) ((n + 255) / 256); if (grid > 65536) grid = 65536;
  hipLaunchKernelGGL(k_msv_scores, dim3(grid), dim3(256), 0, stream, p, s.len, slots, n, xj, sc, st);
  return hipGetLastError();
}

hipError_t launch_msv_classify(const DevProfile &p, const DevSeqs &s, const int32_t *slots, int64_t n,
                               const uint16_t *zmax, int16_t *xj, int32_t *full_list, int32_t *full_count,
                               LenCfg lc, hipStream_t st)
{
  if (n <= 0) return hipSuccess;
  unsigned grid = (unsigned) ((n + 255) / 256); if (grid > 65536) grid = 65536;
  hipLaunchKernelGGL(k_msv_classify, dim3(grid), dim3(256), 0, st, p, s.len, slots, n, zmax, xj, full_list, full_count, lc);
  return hipGetLastError();
}

#define MF_CASE(N) case N: k = (void *) k_msv_full<N>; break;
hipError_t launch_msv_full(const DevProfile &p, const DevSeqs &s, const int32_t *list, const int32_t *count,
                           int64_t maxn, int16_t *xj, LenCfg lc, hipStream_t st)
{
  if (maxn <= 0) return hipSuccess;
  // large models run the recurrence with several waves per target
  void *kw = nullptr;
  int ww = 0;
  switch (p.mf_ND) {
    case 20: kw = (void *) k_msv_full_wg<20, 4>; ww = 4; break;
    case 24: kw = (void *) k_msv_full_wg<24, 4>; ww = 4; break;
    case 32: kw = (void *) k_msv_full_wg<32, 8>; ww = 8; break;
    case 40: kw = (void *) k_msv_full_wg<40, 8>; ww = 8; break;
    default: break;
  }
  if (kw) {
    const unsigned grid = grid_for_waves_blk(kw, maxn * ww, 0, ww);
    void *args[] = { (void *) &p, (void *) &p.mf_tbl, (void *) &s.res, (void *) &s.off, (void *) &s.len,
                     (void *) &list, (void *) &count, &xj, &lc };
    return launch(kw, grid, 64 * ww, args, 0, st);
  }
  void *k = nullptr;
  switch (p.mf_ND) {
    MF_CASE(1) MF_CASE(2) MF_CASE(3) MF_CASE(4) MF_CASE(5) MF_CASE(6) MF_CASE(8) MF_CASE(10) MF_CASE(12) MF_CASE(16)
    default: return hipErrorInvalidValue;
  }
  const size_t lds = p.mf_dwords * 4;
  const unsigned grid = list_grid(k, maxn, lds, LIST_BLOCK / 64);
  int tbl_dwords = (int) p.mf_dwords;
  void *args[] = { (void *) &p, (void *) &p.mf_tbl, &tbl_dwords, (void *) &s.res, (void *) &s.off, (void *) &s.len,
                   (void *) &list, (void *) &count, &xj, &lc };
  return launch(k, grid, LIST_BLOCK, args, lds, st);
}

hipError_t launch_msv_gate(const DevProfile &p, const DevSeqs &s, int64_t n, const int16_t *xj, DevResults r,
                           DevLists l, GateThresh g, hipStream_t st)
{
  if (n <= 0) return hipSuccess;
  unsigned grid = (unsigned) ((n + 255) / 256); if (grid > 65536) grid = 65536;
  hipLaunchKernelGGL(k_msv_gate, dim3(grid), dim3(256), 0, st, p, s.len, n, xj, r, l, g);
  return hipGetLastError();
}

hipError_t launch_bias(const DevProfile &p, const DevSeqs &s, const int32_t *list, const int32_t *count, int64_t maxn,
                       DevResults r, DevLists l, GateThresh g, int gating, LenCfg lc,
                       float *rowmax, int64_t rowmax_size, int64_t *defer_off, hipStream_t st)
{
  if (maxn <= 0) return hipSuccess;
  unsigned grid = (unsigned) ((maxn + 31) / 32); if (grid > 8192) grid = 8192;
  hipLaunchKernelGGL(k_bias, dim3(grid), dim3(64), 0, st, p, s.res, s.off, s.len, list, count, r, g, gating, lc,
                     rowmax, rowmax_size, l.cursor, defer_off);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || ! rowmax) return e;
  dev_props();
  hipLaunchKernelGGL(k_bias_log, dim3(ncu() * 8), dim3(256), 0, st, rowmax, (const unsigned long long *) l.cursor, rowmax_size);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  const unsigned wgrid = (unsigned) std::min<int64_t>((maxn + 3) / 4, 8192);
  hipLaunchKernelGGL(k_bias_sum, dim3(wgrid), dim3(256), 0, st, p, s.len, list, count, r, g, gating, lc,
                     (const float *) rowmax, (const int64_t *) defer_off);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  // the scale-factor pool's cursor starts from zero again for the Forward stage
  return launch_fill32(l.cursor, 0u, 2, st);
}

hipError_t launch_domains(const DevProfile &p, const DevSeqs &s, const int32_t *list, const int32_t *count, int64_t maxn,
                          const DevResults &r, DevLists l, LenCfg lc, const DomBufs &dom, const DomOut &out,
                          hipStream_t st)
{
  if (maxn <= 0) return hipSuccess;
  if (! dom.pool || ! dom.doff || ! dom.boff || ! out.nexp || ! out.nreg || ! out.nclu || ! out.regs || ! out.ecount ||
      ! out.res || ! out.v_off || ! out.v_len || ! out.v_list || ! out.env_loop || ! out.env_move) return hipErrorInvalidValue;
  const unsigned grid = (unsigned) std::min<int64_t>((maxn + 3) / 4, 8192);
  hipLaunchKernelGGL(k_domains, dim3(grid), dim3(256), 0, st, p, s.res, s.off, s.len, list, count, (const int *) r.fstatus,
                     l, lc, dom, out);
  return hipGetLastError();
}

/*****************************************************************
 * Pipeline counters and caller-order outputs
 *****************************************************************/
__global__ __launch_bounds__(256)
void k_stats(const int32_t *__restrict__ len, const uint8_t *__restrict__ stage, int64_t n,
             const int32_t *__restrict__ vit, const int32_t *__restrict__ fwd, const int32_t *__restrict__ counts,
             unsigned long long *__restrict__ out)
{
  unsigned long long a[8] = { 0, 0, 0, 0, 0, 0, 0, 0 };
  const int64_t i0 = (int64_t) blockIdx.x * blockDim.x + threadIdx.x, step = (int64_t) gridDim.x * blockDim.x;
  for (int64_t slot = i0; slot < n; slot += step) {
    const int sg = stage[slot];
    const unsigned long long L = (unsigned long long) len[slot];
    a[0] += sg >= 1; a[1] += sg >= 2; a[2] += sg >= 3; a[3] += sg >= 4;
    a[4] += sg >= 1 ? L : 0ull;
    a[5] += sg >= 4 ? L : 0ull;
  }
  const int64_t nv = counts[2], nf = counts[3];
  for (int64_t t = i0; t < nv; t += step) a[6] += (unsigned long long) len[vit[t]];
  for (int64_t t = i0; t < nf; t += step) a[7] += (unsigned long long) len[fwd[t]];
  __shared__ unsigned long long red[8][4];
  const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
#pragma unroll
  for (int k = 0; k < 8; k++) {
    unsigned long long v = a[k];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    if (lane == 0) red[k][wv] = v;
  }
  __syncthreads();
  if (threadIdx.x < 8) {
    const unsigned long long v = red[threadIdx.x][0] + red[threadIdx.x][1] + red[threadIdx.x][2] + red[threadIdx.x][3];
    if (v) atomicAdd(&out[threadIdx.x], v);
  }
}

__global__ void k_scatter32(const int32_t *__restrict__ perm, const uint32_t *__restrict__ src, uint32_t *__restrict__ dst, int64_t n)
{
  for (int64_t s = (int64_t) blockIdx.x * blockDim.x + threadIdx.x; s < n; s += (int64_t) gridDim.x * blockDim.x)
    dst[perm[s]] = src[s];
}
__global__ void k_scatter8(const int32_t *__restrict__ perm, const uint8_t *__restrict__ src, uint8_t *__restrict__ dst, int64_t n)
{
  for (int64_t s = (int64_t) blockIdx.x * blockDim.x + threadIdx.x; s < n; s += (int64_t) gridDim.x * blockDim.x)
    dst[perm[s]] = src[s];
}

hipError_t launch_stats(const DevSeqs &s, const uint8_t *stage, int64_t n, const int32_t *vit, const int32_t *fwd,
                        const int32_t *counts, unsigned long long *out, hipStream_t st)
{
  if (n <= 0) return hipSuccess;
  unsigned grid = (unsigned) std::min<int64_t>((n + 255) / 256, (int64_t) ncu() * 2);
  hipLaunchKernelGGL(k_stats, dim3(grid), dim3(256), 0, st, s.len, stage, n, vit, fwd, counts, out);
  return hipGetLastError();
}
// each region record's caller index and target length, taken while the
// database is at hand, so that the run's results outlive it
__global__ void k_rec_gather(const int4 *__restrict__ regs, int64_t n, const int32_t *__restrict__ perm,
                             const int32_t *__restrict__ len, int32_t *__restrict__ rseq, int32_t *__restrict__ rlen)
{
  for (int64_t r = (int64_t) blockIdx.x * blockDim.x + threadIdx.x; r < n; r += (int64_t) gridDim.x * blockDim.x) {
    const int slot = regs[r].x;
    rseq[r] = perm[slot];
    rlen[r] = len[slot];
  }
}
hipError_t launch_rec_gather(const DevSeqs &s, const int4 *regs, int64_t n, int32_t *rseq, int32_t *rlen, hipStream_t st)
{
  if (n <= 0) return hipSuccess;
  unsigned grid = (unsigned) std::min<int64_t>((n + 255) / 256, 4096);
  hipLaunchKernelGGL(k_rec_gather, dim3(grid), dim3(256), 0, st, regs, n, s.perm, s.len, rseq, rlen);
  return hipGetLastError();
}
hipError_t launch_scatter32(const DevSeqs &s, const void *src, void *dst, int64_t n, hipStream_t st)
{
  if (n <= 0) return hipSuccess;
  unsigned grid = (unsigned) std::min<int64_t>((n + 255) / 256, 65536);
  hipLaunchKernelGGL(k_scatter32, dim3(grid), dim3(256), 0, st, s.perm, (const uint32_t *) src, (uint32_t *) dst, n);
  return hipGetLastError();
}
hipError_t launch_scatter8(const DevSeqs &s, const uint8_t *src, uint8_t *dst, int64_t n, hipStream_t st)
{
  if (n <= 0) return hipSuccess;
  unsigned grid = (unsigned) std::min<int64_t>((n + 255) / 256, 65536);
  hipLaunchKernelGGL(k_scatter8, dim3(grid), dim3(256), 0, st, s.perm, src, dst, n);
  return hipGetLastError();
}

/*****************************************************************
 * Order-preserving compaction of the survivor lists
 *****************************************************************/
#define CT_TILE 4096     // slots per block: 256 threads x 16 consecutive slots

template <typename T>
__device__ __forceinline__ int tile_flags(const T *__restrict__ f, int value, int64_t base, int64_t n, unsigned &mask)
{
  mask = 0u;
#pragma unroll
  for (int u = 0; u < 16; u++) {
    const int64_t s = base + u;
    if (s < n && (int) f[s] == value) mask |= 1u << u;
  }
  return __popc(mask);
}

template <typename T>
__global__ __launch_bounds__(256)
void k_compact_count(const T *__restrict__ f, int value, int64_t n, int32_t *__restrict__ tilecnt)
{
  __shared__ int part[4];
  unsigned m;
  int c = tile_flags(f, value, (int64_t) blockIdx.x * CT_TILE + threadIdx.x * 16, n, m);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o, 64);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = c;
  __syncthreads();
  if (threadIdx.x == 0) tilecnt[blockIdx.x] = part[0] + part[1] + part[2] + part[3];
}

template <typename T>
__global__ __launch_bounds__(256)
void k_compact_scatter(const T *__restrict__ f, int value, int64_t n, const int32_t *__restrict__ tilecnt,
                       int32_t *__restrict__ list, int32_t *__restrict__ count)
{
  __shared__ int part[4];
  __shared__ int wsum[4];
  // start of this tile's output: the counts of the tiles before it
  int before = 0;
  for (int b = threadIdx.x; b < (int) blockIdx.x; b += blockDim.x) before += tilecnt[b];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) before += __shfl_xor(before, o, 64);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = before;
  // this thread's 16 slots, and an exclusive scan of the counts over the block
  unsigned m;
  const int64_t base = (int64_t) blockIdx.x * CT_TILE + threadIdx.x * 16;
  const int c = tile_flags(f, value, base, n, m);
  const int lane = threadIdx.x & 63;
  int incl = c;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) { const int v = __shfl_up(incl, o, 64); if (lane >= o) incl += v; }
  if (lane == 63) wsum[threadIdx.x >> 6] = incl;
  __syncthreads();
  const int start = part[0] + part[1] + part[2] + part[3];
  int woff = 0;
  for (int w = 0; w < (int) (threadIdx.x >> 6); w++) woff += wsum[w];
  int at = start + woff + incl - c;
#pragma unroll
  for (int u = 0; u < 16; u++) if (m & (1u << u)) list[at++] = (int32_t) (base + u);
  if (blockIdx.x == gridDim.x - 1 && threadIdx.x == blockDim.x - 1) *count = start + woff + incl;
}

template <typename T>
static hipError_t launch_compact(const T *f, int value, int64_t n, int32_t *list, int32_t *count, int32_t *tilecnt,
                                 hipStream_t st)
{
  if (n <= 0) return launch_fill32(count, 0u, 1, st);
  const unsigned tiles = (unsigned) ((n + CT_TILE - 1) / CT_TILE);
  hipLaunchKernelGGL(k_compact_count<T>, dim3(tiles), dim3(256), 0, st, f, value, n, tilecnt);
  hipLaunchKernelGGL(k_compact_scatter<T>, dim3(tiles), dim3(256), 0, st, f, value, n, (const int32_t *) tilecnt, list, count);
  return hipGetLastError();
}
hipError_t launch_compact_u8(const uint8_t *flags, int value, int64_t n, int32_t *list, int32_t *count,
                             int32_t *tilecnt, hipStream_t st)
{
  return launch_compact<uint8_t>(flags, value, n, list, count, tilecnt, st);
}
hipError_t launch_compact_i16(const int16_t *flags, int value, int64_t n, int32_t *list, int32_t *count,
                              int32_t *tilecnt, hipStream_t st)
{
  return launch_compact<int16_t>(flags, value, n, list, count, tilecnt, st);
}

