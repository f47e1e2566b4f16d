// batched.hip -- many independent DM-QR factorisations in one persistent
// launch: each workgroup factorises whole matrices, one after another,
// taking the next one (in decreasing flop count, ordered by the host) from a
// device counter, with the DM state of the current matrix in LDS.
//
// The arithmetic of a step is the plain path's (src/dgeqrdm_work.c:694-787):
// the same device routines for the norms (wave_nrm2), the top-k order
// (wave_sort64 / wave_merge64), the greedy acceptance and permute_marked
// plan (select_wave), and the panel in either of the plain path's forms --
// on panels of at least gram_rows rows the Gram-based one (chol1_core,
// recon_core: CholeskyQR2 with Householder reconstruction, T from V^T V),
// otherwise dgeqr2_mia column by column (panel_exact_body) with dlarft
// (larft_recurrence).  The candidate Gram, the panel's products and Grams
// and the trailing update run on the FP64 matrix cores inside the
// workgroup.  Limits: n <= BT_NMAX (the per-column state lives in LDS); m
// is free.

namespace qrdm {

constexpr int BT_NMAX = BATCH_NMAX;
constexpr double kEpsD = 1.1102230246251565e-16;  // LAPACK dlamch('E') = 2^-53

// One matrix of a batch; layout of qrdm_batch_item (include/qrdm_amd.h).
struct BatchItem {
  int m, n, lda, pad;
  long long a_off, tau_off, col_off;
};

struct BatchParams {
  double delta, tau_dm, eta3, tol3z;
  int nb, stop_mode;
  const PolicyNet* policy;  // learned (tau, delta) per step, or nullptr
  float* trace;             // per-step training records (POL_REC floats), or nullptr
  unsigned* trace_count;    // records written (may exceed trace_cap)
  int trace_cap;
  float tau_lo, tau_hi, delta_lo, delta_hi;  // label normalisation
  int gram_rows;  // panels of at least this many rows (and 2+ columns) take the Gram-based form
};

template <int NW>
struct BatchLds {
  double work[BT_NMAX], wold[BT_NMAX];
  int jp[BT_NMAX];
  union {
    struct {
      double lv[NW][KMAX];
      int li[NW][KMAX];
    } tk;                       // the top-k's per-wave lists
    double E[2][KMAX][LDP];     // the Gram-based panel's matrices
  } u;
  double R1[KMAX * LDP];  // candidate Gram / V^T V (the panel's scratch after it)
  double Ts[KMAX * LDP];  // T (column-major, leading dimension KMAX)
  double ts[KMAX], tmp[KMAX];
  double rinv[KMAX], dsg[KMAX], tl[KMAX], scv[KMAX];
  double red[16];
  int perm[4 * KMAX + KMAX];
  int s_done, s_why;
  DevState st;
  float feat[POL_IN];
  float hbuf[POL_H];
  int hist[POL_BINS];
};

// Unit lower trapezoidal V of the panel at column j: V(row, c) for c < kk.
__device__ __forceinline__ double bt_v(const double* a, int lda, int j, int kk, int row, int c,
                                       int m) {
  const int rr = row - j;
  if (c >= kk || row >= m || rr < c) return 0.0;
  return rr == c ? 1.0 : a[(size_t)(j + c) * lda + row];
}

// C := C - V T^T V^T C on rows [j, m), columns [c0, n), 128 columns at a time, a
// wave two groups of 16: P = V^T C down the rows, W = T^T P, C -= V W back up the
// rows (the last rows of C are still in the L2).  V goes through LDS in 32-row
// chunks (E's space, two buffers) as the merged pass of trailing.hip keeps it; a
// wave holds its whole columns' P, so W follows in registers (the layout of one
// product's result is the next one's operand).
//
// Memory bounds it, through the loads in flight: the matrices of a launch exceed
// the caches, and one wave per SIMD (LDS holds one workgroup per CU) hides
// nothing.  So two chunks of V and C are on their way to registers beside the
// one in LDS, and 128 columns share a reading of V.  Per CU of a launch over 1024
// matrices up to 1024 x 512 (8.87 -> 7.08 ms): 2.2 ms, about 11 GB in all, against
// 2.95 with V read per wave and no loads in flight across chunks, and 4.7 with one
// chunk in flight and 64 columns.
//
// P is summed in pieces of two chunks, as in the merged pass: one running sum down
// the rows was off by 1.2e-15 of the result at 1024 x 512, this by 5.4e-16 (four
// waves' sums 7.2e-16), for 0.06 ms of the launch above.
template <int NW>
__device__ __forceinline__ void bt_trailing(double* a, int lda, int j, int m, int kk, int c0, int n,
                            BatchLds<NW>& L) {
  static_assert(NW == 4, "a chunk of V is staged by four waves");
  FuChunk* S = reinterpret_cast<FuChunk*>(&L.u.E[0][0][0]);
  static_assert(sizeof(L.u.E) >= 2 * sizeof(FuChunk), "V's chunks lie in E");
  constexpr int U = 2;  // column groups per wave
  const int tid = local_tid(), lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, li = lane & 15;
  const int nch = (m - j + FU_CH - 1) / FU_CH;
  struct Regs {
    fu_pair v[4], c[U][4];
  };
  for (int cb = c0; cb < n; cb += 64 * U) {
    double* Cc[U];
    bool on[U], cok[U];  // the wave has columns of the group; the lane's one exists
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int col = cb + 64 * u + 16 * wave + li;
      on[u] = cb + 64 * u + 16 * wave < n;
      cok[u] = col < n;
      Cc[u] = a + (size_t)min(col, n - 1) * lda;
    }
    // chunk ch: V's columns 16 wave + 4 i + g, rows 2 li, 2 li + 1; C's rows
    // j + 32 ch + 8 v + 2 g + (0, 1) of the lane's columns
    auto load = [&](int ch, Regs& x) {
      if (ch < 0 || ch >= nch) return;
      const int r0 = j + FU_CH * ch;
      if (r0 + FU_CH <= m) {  // whole: plain loads, back to back
#pragma unroll
        for (int i = 0; i < 4; i++)
          x.v[i] = *reinterpret_cast<const fu_pair*>(
              a + (size_t)(j + min(16 * wave + 4 * i + g, kk - 1)) * lda + r0 + 2 * li);
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
          for (int v = 0; v < 4; v++)
            x.c[u][v] = *reinterpret_cast<const fu_pair*>(Cc[u] + r0 + 8 * v + 2 * g);
        return;
      }
      // the last one: rows from m on read as the last row (every load in flight
      // before any is used)
      double lo[4 + 4 * U], hi[4 + 4 * U];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const double* col = a + (size_t)(j + min(16 * wave + 4 * i + g, kk - 1)) * lda;
        lo[i] = col[min(r0 + 2 * li, m - 1)];
        hi[i] = col[min(r0 + 2 * li + 1, m - 1)];
      }
#pragma unroll
      for (int u = 0; u < U; u++)
#pragma unroll
        for (int v = 0; v < 4; v++) {
          lo[4 + 4 * u + v] = Cc[u][min(r0 + 8 * v + 2 * g, m - 1)];
          hi[4 + 4 * u + v] = Cc[u][min(r0 + 8 * v + 2 * g + 1, m - 1)];
        }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < 4; i++) x.v[i] = (fu_pair){lo[i], hi[i]};
#pragma unroll
      for (int u = 0; u < U; u++)
#pragma unroll
        for (int v = 0; v < 4; v++)
          x.c[u][v] = (fu_pair){lo[4 + 4 * u + v], hi[4 + 4 * u + v]};
    };
    auto store_v = [&](int ch, const fu_pair (&x)[4]) {
      if (ch < 0 || ch >= nch) return;
      if (ch > 1 && kk == KMAX && j + FU_CH * (ch + 1) <= m) {  // below the top block, whole
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const int c = 16 * wave + 4 * i + g;
          S[ch & 1][c][li ^ (c & 15)] = make_double2(x[i].x, x[i].y);
        }
        return;
      }
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int c = 16 * wave + 4 * i + g, pr = FU_CH * ch + 2 * li;
        double2 v;
        v.x = (c < kk && j + pr < m) ? (pr > c ? x[i].x : (pr == c ? 1.0 : 0.0)) : 0.0;
        v.y = (c < kk && j + pr + 1 < m) ? (pr + 1 > c ? x[i].y : (pr + 1 == c ? 1.0 : 0.0)) : 0.0;
        S[ch & 1][c][li ^ (c & 15)] = v;
      }
    };
    dbl4 acc[U][4], tot[U][4];  // P of two chunks, of all
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
      for (int t = 0; t < 4; t++) acc[u][t] = tot[u][t] = (dbl4){0.0, 0.0, 0.0, 0.0};
    // chunk ch's products; x0: chunk ch (V stored already), x1: ch + 1, which
    // follows into LDS; ch + 2 is fetched over x0
    auto down = [&](int ch, Regs& x0, Regs& x1) {
      lds_barrier();  // chunk ch is in LDS; the other buffer is read
      fu_pair c[U][4];
#pragma unroll
      for (int u = 0; u < U; u++)
#pragma unroll
        for (int v = 0; v < 4; v++) c[u][v] = x0.c[u][v];
      load(ch + 2, x0);
      const FuChunk& V = S[ch & 1];
#pragma unroll
      for (int v = 0; v < 4; v++) {
        double2 x[4];
#pragma unroll
        for (int t = 0; t < 4; t++) x[t] = V[16 * t + li][(g + 4 * v) ^ li];
#pragma unroll
        for (int u = 0; u < U; u++)
          if (on[u]) {
#pragma unroll
            for (int t = 0; t < 4; t++)
              acc[u][t] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[t].x, c[u][v].x, acc[u][t], 0, 0, 0);
#pragma unroll
            for (int t = 0; t < 4; t++)
              acc[u][t] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[t].y, c[u][v].y, acc[u][t], 0, 0, 0);
          }
      }
      store_v(ch + 1, x1.v);
    };
    Regs xa, xb;
    load(0, xa);
    load(1, xb);
    store_v(0, xa.v);
    for (int ch = 0; ch < nch; ch += 2) {
      down(ch, xa, xb);
      if (ch + 1 < nch) down(ch + 1, xb, xa);
#pragma unroll
      for (int u = 0; u < U; u++)
#pragma unroll
        for (int t = 0; t < 4; t++) {
          tot[u][t] += acc[u][t];
          acc[u][t] = (dbl4){0.0, 0.0, 0.0, 0.0};
        }
    }
    // back from the last chunk, in LDS still
    load(nch - 1, xa);
    load(nch - 2, xb);
    // P's rows 16 t + g + 4 v in tot[u][t][v], -W's in w[u][t][v]: W_t = sum over
    // the blocks k <= t of T_kt^T P_k
    dbl4 w[U][4];
#pragma unroll
    for (int t = 0; t < 4; t++) {
#pragma unroll
      for (int u = 0; u < U; u++) w[u][t] = (dbl4){0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int k = 0; k <= t; k++)
#pragma unroll
        for (int v = 0; v < 4; v++) {
          const double x = -L.Ts[(16 * k + g + 4 * v) + (16 * t + li) * KMAX];
#pragma unroll
          for (int u = 0; u < U; u++)
            w[u][t] = __builtin_amdgcn_mfma_f64_16x16x4f64(x, tot[u][k][v], w[u][t], 0, 0, 0);
        }
    }
    auto up = [&](int ch, Regs& x0, Regs& x1) {
      fu_pair c[U][4];
#pragma unroll
      for (int u = 0; u < U; u++)
#pragma unroll
        for (int v = 0; v < 4; v++) c[u][v] = x0.c[u][v];
      load(ch - 2, x0);
      const FuChunk& V = S[ch & 1];
      dbl4 d[U][2];
#pragma unroll
      for (int u = 0; u < U; u++) d[u][0] = d[u][1] = (dbl4){0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int s = 0; s < 16; s++) {
        const double2 x = V[4 * s + g][li ^ (4 * (s & 3) + g)];
#pragma unroll
        for (int u = 0; u < U; u++)
          if (on[u]) {
            d[u][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(x.x, w[u][s >> 2][s & 3], d[u][0], 0, 0, 0);
            d[u][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(x.y, w[u][s >> 2][s & 3], d[u][1], 0, 0, 0);
          }
      }
      if (j + FU_CH * (ch + 1) <= m) {
#pragma unroll
        for (int u = 0; u < U; u++)
          if (cok[u]) {
#pragma unroll
            for (int v = 0; v < 4; v++)
              *reinterpret_cast<fu_pair*>(Cc[u] + j + FU_CH * ch + 8 * v + 2 * g) =
                  (fu_pair){c[u][v].x + d[u][0][v], c[u][v].y + d[u][1][v]};
          }
      } else
#pragma unroll
      for (int u = 0; u < U; u++)
        if (cok[u]) {
#pragma unroll
          for (int v = 0; v < 4; v++) {
            const int r = j + FU_CH * ch + 8 * v + 2 * g;
            const fu_pair o = {c[u][v].x + d[u][0][v], c[u][v].y + d[u][1][v]};
            if (r + 1 < m) *reinterpret_cast<fu_pair*>(Cc[u] + r) = o;
            else if (r < m) Cc[u][r] = o.x;
          }
        }
      store_v(ch - 1, x1.v);
      lds_barrier();
    };
    for (int ch = nch - 1; ch >= 0; ch -= 2) {
      up(ch, xa, xb);
      if (ch > 0) up(ch - 1, xb, xa);
    }
  }
}

// S = the sum of the four waves' tile Grams gt (in wave order), both
// triangles; four waves.  Ends with a barrier.
__device__ __forceinline__ void bt_gram_store(double (*S)[LDP], const dbl4p (&gt)[10]) {
  const int t = local_tid(), lane = t & 63, wv = t >> 6, g = lane >> 4, li = lane & 15;
  for (int e = t; e < KMAX * KMAX; e += 256) S[e >> 6][e & 63] = 0.0;
  lds_barrier();
  for (int w = 0; w < 4; w++) {
    if (wv == w) {
      int p = 0;
#pragma unroll
      for (int u = 0; u < 4; u++)
#pragma unroll
        for (int u2 = u; u2 < 4; u2++) {
#pragma unroll
          for (int v = 0; v < 4; v++) S[16 * u + g + 4 * v][16 * u2 + li] += gt[p][v];
          p++;
        }
    }
    lds_barrier();
  }
  // the diagonal tiles are whole; mirror the tiles below them
  for (int e = t; e < KMAX * KMAX; e += 256) {
    const int r = e >> 6, c = e & 63;
    if ((r >> 4) > (c >> 4)) S[r][c] = S[c][r];
  }
  lds_barrier();
}

// Gram X^T X of up to 64 columns over rows [r0, m), X(r, c) = colval(c, r),
// into R1 (both triangles, leading dimension KMAX + 1); four waves.  Each
// wave takes its own 16-row blocks (rows r0 + 16 wv, then every 64th), reads
// them straight into the matrix cores' operand layout and accumulates the
// upper tiles in registers (bt_gram_tiles); no barrier until the waves' sums
// go into R1 in wave order.
template <int NW, typename ColFn>
__device__ __forceinline__ void bt_gram(int r0, int m, int ncols, ColFn colval, BatchLds<NW>& L) {
  static_assert(NW == 4, "the Gram's tiles are spread over four waves");
  const int tid = local_tid(), lane = tid & 63, wv = tid >> 6, g = lane >> 4, li = lane & 15;
  dbl4p gt[10];
#pragma unroll
  for (int p = 0; p < 10; p++) gt[p] = (dbl4p){0.0, 0.0, 0.0, 0.0};
  dbl4p xn[4];  // the next block, on its way while this one is multiplied
  auto load = [&](int rb) {
#pragma unroll
    for (int u = 0; u < 4; u++)
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const int c = 16 * u + li, r = rb + g + 4 * v;
        xn[u][v] = (c < ncols && r < m) ? colval(c, r) : 0.0;
      }
  };
  load(r0 + 16 * wv);
  for (int rb = r0 + 16 * wv; rb < m; rb += NW * 16) {
    dbl4p xb[4];
#pragma unroll
    for (int u = 0; u < 4; u++) xb[u] = xn[u];
    if (rb + NW * 16 < m) load(rb + NW * 16);
    gram_tiles(xb, gt);
  }
  bt_gram_store(reinterpret_cast<double (*)[LDP]>(L.R1), gt);
}

// The Gram-based panel (panel.hip's tall-panel form) by the workgroup: R1 =
// chol of the panel's Gram, gathered from the candidate Gram in L.R1 through
// the ranks select_wave left in perm[4 KMAX ..] (chol1_core); Q = P R1^-1
// and G2 = Q^T Q over 64-row slabs; the reconstruction (recon_core: R, V1,
// tau, M); V2 = P_bottom M written into the panel, with V^T V; then tau and
// T from V^T V (the compact WY identity, as k_reduce_t), T into L.Ts.
// Returns the columns kept, or -1 with A and tau unchanged when the form
// falls back (the caller then runs the column-by-column panel).
template <int NW>
__device__ __forceinline__ int bt_panel_gram(double* a, int lda, int j, int m, int fjb, double tau_dm,
                             double* tau, BatchLds<NW>& L) {
  static_assert(NW == 4, "the one-workgroup factorisations run on four waves");
  const int tid = local_tid(), lane = tid & 63, wv = tid >> 6;
  double (*E0)[LDP] = L.u.E[0];
  double (*E1)[LDP] = L.u.E[1];
  double (*RT)[LDP] = reinterpret_cast<double (*)[LDP]>(L.R1);
  double (*TS)[LDP] = reinterpret_cast<double (*)[LDP]>(L.Ts);
  auto Yof = [](double* p) { return reinterpret_cast<double (*)[BLK][BLK + 1]>(p); };
  // 1. R1 and R1^-1 (E0, E1; zero outside k1 x k1)
  const int* rank = L.perm + 4 * KMAX;
  if (tid < KMAX) {
    const int rk = tid < fjb ? rank[tid] : 0;
    L.tmp[tid] = tid < fjb ? L.R1[rk * (KMAX + 2)] : 0.0;  // G(rk, rk)
  }
  for (int e = tid; e < KMAX * KMAX; e += NW * 64) {
    const int r = e >> 6, c = e & 63;
    E0[r][c] = (r < fjb && c < fjb) ? L.R1[rank[r] + rank[c] * (KMAX + 1)] : (r == c ? 1.0 : 0.0);
  }
  lds_barrier();
  const int k1 = chol1_core(E0, E1, Yof(L.Ts), L.rinv, L.tmp, fjb, tau_dm, &L.s_done, &L.s_why);
  if (k1 < 0) return -1;
  for (int e = tid; e < KMAX * KMAX; e += NW * 64) {
    const int r = e >> 6, c = e & 63;
    if (!(r < k1 && c < k1)) {
      E0[r][c] = 0.0;
      E1[r][c] = 0.0;
    }
  }
  lds_barrier();
  // 2. G2 = (P R1^-1)^T (P R1^-1): each wave takes its own 16-row blocks (rows
  // j + 16 wv, then every 64th) with no barrier: Q_blk = P_blk R1^-1 on the
  // matrix cores, P read straight into the A operand; Q_blk^T Q_blk from the
  // product's own layout (bt_gram_tiles).  The waves' sums go into RT in wave
  // order; identity beyond k1.
  const int g = lane >> 4, li = lane & 15;
  dbl4p gt[10];
#pragma unroll
  for (int p = 0; p < 10; p++) gt[p] = (dbl4p){0.0, 0.0, 0.0, 0.0};
  double pn[KMAX / 4];  // the next block's P
  auto load_p = [&](int rb, int kc) {
    const int ra = rb + li;
#pragma unroll
    for (int t = 0; t < KMAX / 4; t++)
      pn[t] = (ra < m && 4 * t + g < kc) ? a[(size_t)(j + 4 * t + g) * lda + ra] : 0.0;
  };
  load_p(j + 16 * wv, k1);
  for (int rb = j + 16 * wv; rb < m; rb += NW * 16) {
    double pa[KMAX / 4];
#pragma unroll
    for (int t = 0; t < KMAX / 4; t++) pa[t] = pn[t];
    if (rb + NW * 16 < m) load_p(rb + NW * 16, k1);
    dbl4p qb[4];
#pragma unroll
    for (int u = 0; u < 4; u++) qb[u] = (dbl4p){0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int t = 0; t < KMAX / 4; t++)
#pragma unroll
      for (int u = t / 4; u < 4; u++)
        qb[u] = __builtin_amdgcn_mfma_f64_16x16x4f64(pa[t], E1[4 * t + g][16 * u + li], qb[u], 0, 0,
                                                     0);
    gram_tiles(qb, gt);
  }
  bt_gram_store(RT, gt);
  if (tid >= k1 && tid < KMAX) RT[tid][tid] = 1.0;
  lds_barrier();
  // 3. the reconstruction: SR = E0, SA = E1 (R1^-1), SW = TS (also its
  // scratch Y, and M out), SX = RT
  double* Mf = &TS[0][0];  // M(q, c) at Mf[q + c * KMAX]
  const int k = recon_core(
      E0, E1, TS, RT, Yof(L.Ts), L.rinv, L.dsg, L.tl, L.scv, &L.s_done, &L.s_why,
      [&](double(*S)[LDP]) {  // E1 holds R1^-1: S takes it before E1 is overwritten
        for (int e = tid; e < KMAX * KMAX; e += NW * 64) S[e & 63][e >> 6] = E1[e & 63][e >> 6];
        lds_barrier();
      },
      [&](double(*S)[LDP]) { load_slab(S, a, lda, j, j, j + k1, k1); }, a, lda, j, fjb, k1, tau_dm,
      tau + j, Mf);
  if (k < 0) return -1;
  __syncthreads();  // the top block the reconstruction wrote to A is read below
  for (int e = tid; e < KMAX * KMAX; e += NW * 64) E0[e & 63][e >> 6] = Mf[e];  // M, padded
  lds_barrier();
  // 4. V2 = P_bottom M: each wave its own 16-row blocks as in 2, P straight
  // into the A operand, M (E0) the B operand; the top block's rows take V1
  // (unit lower, written into A by the reconstruction), V2's rows are
  // written into the panel, and V^T V accumulates from the product's layout
  // (summed into E1 in wave order).
#pragma unroll
  for (int p = 0; p < 10; p++) gt[p] = (dbl4p){0.0, 0.0, 0.0, 0.0};
  load_p(j + 16 * wv, k);
  for (int rb = j + 16 * wv; rb < m; rb += NW * 16) {
    double pa[KMAX / 4];
#pragma unroll
    for (int t = 0; t < KMAX / 4; t++) pa[t] = pn[t];
    if (rb + NW * 16 < m) load_p(rb + NW * 16, k);
    dbl4p vb[4];
#pragma unroll
    for (int u = 0; u < 4; u++) vb[u] = (dbl4p){0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int t = 0; t < KMAX / 4; t++)
#pragma unroll
      for (int u = t / 4; u < 4; u++)
        vb[u] = __builtin_amdgcn_mfma_f64_16x16x4f64(pa[t], E0[4 * t + g][16 * u + li], vb[u], 0, 0,
                                                     0);
#pragma unroll
    for (int u = 0; u < 4; u++)
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const int r = rb + g + 4 * v, c = 16 * u + li, pr = r - j;
        double x = vb[u][v];
        if (c >= k || r >= m) x = 0.0;
        else if (pr < k) x = (pr < c) ? 0.0 : (pr == c ? 1.0 : a[(size_t)(j + c) * lda + r]);
        else a[(size_t)(j + c) * lda + r] = x;
        vb[u][v] = x;
      }
    gram_tiles(vb, gt);
  }
  bt_gram_store(E1, gt);
  // 5. tau_i = 2 / S_ii and T = (striu(S) + diag(S) / 2)^-1 from S = V^T V
  for (int e = tid; e < KMAX * KMAX; e += NW * 64) {
    const int r = e & 63, c = e >> 6;
    const double sv = E1[r][c];
    E0[r][c] = (r < k && c < k) ? ((r < c) ? sv : (r == c ? 0.5 * sv : 0.0)) : (r == c ? 1.0 : 0.0);
  }
  lds_barrier();
  if (tid < k) tau[j + tid] = 1.0 / E0[tid][tid];
  upper_inverse(E0, E1, L.rinv, Yof(L.R1));  // E1 = T (upper)
  for (int e = tid; e < KMAX * KMAX; e += NW * 64) {
    const int r = e & 63, c = e >> 6;
    L.Ts[r + c * KMAX] = (r < k && c < k && r <= c) ? E1[r][c] : 0.0;
  }
  __syncthreads();  // V2 in A and T in LDS, for the trailing update
  return k;
}

// The norms of columns c, c + step, c + 2 step, c + 3 step (below n), each
// summed as wave_nrm2 does, the four columns' loads in flight together (one
// column at a time waits for memory 1.5 us per column and wave).
__device__ __forceinline__ void bt_nrm2x4(const double* a, int lda, int c, int step, int n, int m,
                                          double (&nr)[4]) {
  const int lane = local_tid() & 63;
  const double* x[4];
#pragma unroll
  for (int q = 0; q < 4; q++) x[q] = a + (size_t)min(c + q * step, n - 1) * lda;
  double s[4][4];
#pragma unroll
  for (int q = 0; q < 4; q++)
#pragma unroll
    for (int u = 0; u < 4; u++) s[q][u] = 0.0;
  int i = lane;
  for (; i + 192 < m; i += 256) {
    double v[4][4];
#pragma unroll
    for (int q = 0; q < 4; q++)
#pragma unroll
      for (int u = 0; u < 4; u++) v[q][u] = x[q][i + 64 * u];
#pragma unroll
    for (int q = 0; q < 4; q++)
#pragma unroll
      for (int u = 0; u < 4; u++) s[q][u] = fma(v[q][u], v[q][u], s[q][u]);
  }
  for (; i < m; i += 64) {
    double v[4];
#pragma unroll
    for (int q = 0; q < 4; q++) v[q] = x[q][i];
#pragma unroll
    for (int q = 0; q < 4; q++) s[q][0] = fma(v[q], v[q], s[q][0]);
  }
#pragma unroll
  for (int q = 0; q < 4; q++) nr[q] = wave_sum((s[q][0] + s[q][1]) + (s[q][2] + s[q][3]));
#pragma unroll
  for (int q = 0; q < 4; q++) {
    if (nr[q] >= 1e-280 && nr[q] <= 1e280) nr[q] = sqrt(nr[q]);
    else if (c + q * step < n) nr[q] = wave_nrm2(x[q], m);
  }
}

// One DM-QR (dgeqrdm semantics, free columns) of the matrix it by the whole
// workgroup.  Returns info (0, or -13 for a non-finite entry, A untouched).
template <int NW>
__device__ __forceinline__ int bt_factor(const BatchItem& it, double* A, double* tau_all, int* jp_all,
                         int* nc_all, const BatchParams& P, BatchLds<NW>& L) {
  constexpr int NT = 64 * NW;
  const int tid = local_tid(), lane = tid & 63, wave = tid >> 6;
  const int m = it.m, n = it.n, lda = it.lda;
  double* a = A + it.a_off;
  double* tau = tau_all + it.tau_off;
  const int minmn = m < n ? m : n;
  // initial norms (src/dgeqrdm_work.c:670-682), as k_init_norms
  double mx = 0.0, bad = 0.0;
  for (int c = wave; c < n; c += 4 * NW) {
    double nr4[4];
    bt_nrm2x4(a, lda, c, NW, n, m, nr4);
#pragma unroll
    for (int q = 0; q < 4; q++) {
      if (c + NW * q >= n) break;
      const double nr = nr4[q];
      if (lane == 0) {
        L.work[c + NW * q] = nr;
        L.wold[c + NW * q] = nr;
      }
      if (!(nr <= DBL_MAX)) bad = 1.0;
      else mx = fmax(mx, nr);
    }
  }
  for (int c = tid; c < n; c += NT) L.jp[c] = c + 1;
  const double maxnrm0 = block_max(mx, L.red);
  if (block_max(bad, L.red) != 0.0) return -13;
  double eta = 0.0;
  const int enable_stop = P.stop_mode;
  if (P.stop_mode == 1) eta = kEpsD * n;
  else if (P.stop_mode == 2) eta = kEpsD * sqrt((double)n);
  else if (P.stop_mode == 3) eta = P.eta3;
  eta *= maxnrm0;
  int j = 0, itn = 0;
  while (j < minmn) {
    // the workitem id afresh for each step: what the step derives from it is
    // not held in registers across the steps
    const int tid = local_tid(), lane = tid & 63, wave = tid >> 6;
    const int nsub = n - j;
    int kmax = P.nb < KMAX ? P.nb : KMAX;
    if (m - j < kmax) kmax = m - j;
    if (nsub < kmax) kmax = nsub;
    // --- candidates: the first kmax keys of work[j..n) in qsort/cmpStruct
    // order (value descending, position ascending), count > tau * max
    {
      double v = -1.0;
      int ix = 0x7fffffc0 + lane;  // a sorted list of padding keys
      for (int b = wave; 64 * b < nsub; b += NW) {
        const int t = 64 * b + lane;
        double bv = (t < nsub) ? L.work[j + t] : -1.0;
        bv = bv == bv ? bv : 0.0;  // (as k_topk)
        int bi = (t < nsub) ? t : 0x40000000 + t;
        wave_sort64(bv, bi);
        wave_merge64(v, ix, bv, bi);
      }
      L.u.tk.lv[wave][lane] = v;
      L.u.tk.li[wave][lane] = ix;
      __syncthreads();
      block_merge_lists<NW>(L.u.tk.lv, L.u.tk.li, v, ix);
      if (wave == 0) {
        const double cv = L.u.tk.lv[0][lane];
        const int ci = L.u.tk.li[0][lane];
        L.st.cand_val[lane] = lane < kmax ? cv : 0.0;
        L.st.cand_idx[lane] = lane < kmax ? ci : -1;
        const double lim = P.tau_dm * L.u.tk.lv[0][0];
        const int nc = __popcll(__ballot(lane < kmax && cv > lim));
        if (lane == 0) {
          L.st.nc = nc;
          L.st.kmax = kmax;
          L.st.j = j;
          L.st.halt = 0;
          L.st.policy_on = 0;
          L.st.tau_step = P.tau_dm;
          L.st.delta_step = P.delta;
        }
      }
      __syncthreads();
      // the learned proposal (k_policy's arithmetic), and the inputs of a
      // training record
      if (P.policy || P.trace)
        policy_features(L.work + j, nsub, L.st.cand_val[0], j, m, n, L.feat, L.hist);
      if (P.policy && wave == 0) {
        const double cv = L.u.tk.lv[0][lane];
        const float2 y = policy_forward(P.policy, L.feat, L.hbuf);
        double tp = P.policy->tau_lo + (P.policy->tau_hi - P.policy->tau_lo) * (double)y.x;
        double dp = P.policy->delta_lo + (P.policy->delta_hi - P.policy->delta_lo) * (double)y.y;
        if (!(tp >= 0.0 && tp <= 1.0 && dp >= 0.0 && dp <= 1.0)) {
          tp = P.tau_dm;
          dp = P.delta;
        }
        const int nc2 = __popcll(__ballot(lane < kmax && cv > tp * L.u.tk.lv[0][0]));
        if (lane == 0) {
          L.st.nc = nc2;
          L.st.policy_on = 1;
          L.st.tau_step = tp;
          L.st.delta_step = dp;
        }
      }
      __syncthreads();
    }
    const int nc = L.st.nc;
    // --- cosines (src/dgeqrdm_work.c:365-379): Gram of the candidate
    // columns over rows j..m, scaled by the reciprocal norms in select_wave
    // (over all kmax candidates when a training record scores other tau)
    const int ng = P.trace ? kmax : nc;
    if (ng > 1) {
      const DevState& st = L.st;
      bt_gram<NW>(j, m, ng,
                  [&](int c, int r) { return a[(size_t)(j + st.cand_idx[c]) * lda + r]; }, L);
    }
    if (P.trace && wave == 0) {
      unsigned slot = 0;
      if (lane == 0) slot = atomicAdd(P.trace_count, 1u);
      slot = (unsigned)__builtin_amdgcn_readfirstlane((int)slot);
      if (slot < (unsigned)P.trace_cap)
        label_record(L.R1, L.st.cand_val, kmax, P.tau_dm, P.delta, L.Ts, L.feat, j, nsub,
                     P.tau_lo, P.tau_hi, P.delta_lo, P.delta_hi,
                     P.trace + (size_t)slot * POL_REC);
    }
    // --- greedy acceptance and the permute_marked plan
    if (wave == 0) select_wave(L.R1, select_inputs(&L.st, P.delta), m, n, INT_MAX, 1, L.perm, &L.st);
    __syncthreads();
    const int fjb = L.st.fjb, npair = L.st.npair;
    // --- column moves (whole columns; work and jpvt with them, not workold)
    if (npair > 0) {
      // a wave takes 32-row blocks: lane (h, r) row r of the pairs 2 p + h, every
      // pair read before any is written, no barrier (with 8 elements a thread and
      // two barriers per round over all rows 0.90 ms per CU of the launch above; 0.50)
      constexpr int MV = 2 * KMAX / 2;  // pairs per lane at most
      const int h = lane >> 5;
      for (int r0 = 32 * wave; r0 < m; r0 += 32 * NW) {
        const int r = r0 + (lane & 31);
        double v[MV];
#pragma unroll
        for (int p0 = 0; p0 < MV; p0 += 8)
          if (2 * p0 < npair) {
#pragma unroll
            for (int p = p0; p < p0 + 8; p++) {
              const int pp = min(2 * p + h, npair - 1);
              v[p] = a[(size_t)L.perm[2 * pp + 1] * lda + min(r, m - 1)];
            }
          }
#pragma unroll
        for (int p0 = 0; p0 < MV; p0 += 8)
          if (2 * p0 < npair) {
#pragma unroll
            for (int p = p0; p < p0 + 8; p++)
              if (2 * p + h < npair && r < m) a[(size_t)L.perm[2 * (2 * p + h)] * lda + r] = v[p];
          }
      }
      double wv = 0.0;
      int jv = 0;
      if (tid < npair) {
        wv = L.work[L.perm[2 * tid + 1]];
        jv = L.jp[L.perm[2 * tid + 1]];
      }
      __syncthreads();
      if (tid < npair) {
        L.work[L.perm[2 * tid]] = wv;
        L.jp[L.perm[2 * tid]] = jv;
      }
      __syncthreads();
    }
    // --- dgeqr2_mia with truncation (src/dgeqrdm_work.c:735-738): the
    // Gram-based form on tall panels (T from its V^T V; the trailing update
    // also reaches the rejected in-block columns, as dlarf_ did inside the
    // reference's panel), else, or when it falls back, column by column
    int kk = -1, c0 = 0;
    if (fjb >= 2 && m - j >= P.gram_rows) {
      kk = bt_panel_gram<NW>(a, lda, j, m, fjb, P.tau_dm, tau, L);
      c0 = j + kk;
    }
    if (kk < 0) {
      kk = panel_exact_body<4>(a, lda, j, m, fjb, P.tau_dm, 1, tau + j, L.red);
      __syncthreads();
      c0 = j + fjb;
      // --- dlarft from S = V^T V (src/dgeqrdm_work.c:751-754)
      if (c0 < n) {
        bt_gram<NW>(j, m, kk, [&](int c, int r) { return bt_v(a, lda, j, kk, r, c, m); }, L);
        // R1 holds S with leading dimension KMAX + 1: repack to KMAX for the recurrence
        double sv[KMAX * KMAX / NT];
#pragma unroll
        for (int q = 0; q < KMAX * KMAX / NT; q++) {
          const int e = tid + NT * q;
          sv[q] = L.R1[(e & 63) + (e >> 6) * (KMAX + 1)];
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < KMAX * KMAX / NT; q++) {
          const int e = tid + NT * q;
          L.R1[e] = sv[q];
          L.Ts[e] = 0.0;
        }
        if (tid < KMAX) L.ts[tid] = tid < kk ? tau[j + tid] : 0.0;
        __syncthreads();
        larft_recurrence(L.R1, L.Ts, L.ts, L.tmp, kk);
        __syncthreads();
      }
    }
    // --- dlarfb on columns c0..n (src/dgeqrdm_work.c:762-767)
    if (c0 < n) {
      bt_trailing<NW>(a, lda, j, m, kk, c0, n, L);
      __syncthreads();
    }
    // --- norm_update (src/dgeqrdm_work.c:80-109), as k_norm_update
    double nmx = 0.0;
    const int mrem = m - j - kk;
    // a wave's columns j + kk + wave + NW i, i < 64: their sums by the wave, eight
    // columns' loads in flight, then lane i does column i's arithmetic
    for (int cb = j + kk + wave; cb < n; cb += 64 * NW) {
      const int nc64 = min(64, (n - cb + NW - 1) / NW);
      double s2 = 0.0;
      for (int i0 = 0; i0 < nc64; i0 += 8) {
        double x[8];
#pragma unroll
        for (int q = 0; q < 8; q++)
          x[q] = (lane < kk) ? a[(size_t)min(cb + NW * (i0 + q), n - 1) * lda + j + lane] : 0.0;
#pragma unroll
        for (int q = 0; q < 8; q++) x[q] = wave_sum(x[q] * x[q]);
#pragma unroll
        for (int q = 0; q < 8; q++) s2 = lane == i0 + q ? x[q] : s2;
      }
      const int col = cb + NW * lane;
      const bool mine = lane < nc64;
      double wk = mine ? L.work[col] : 0.0;
      const bool live = wk != 0.0;  // (also not for a lane without a column)
      bool again = false;
      if (live) {
        double temp = sqrt(fabs(s2)) / wk;
        const double d2 = (temp + 1.0) * (1.0 - temp);
        temp = (0.0 >= d2) ? 0.0 : d2;
        const double d1 = wk / L.wold[col];
        const double temp2 = temp * (d1 * d1);
        again = temp2 <= P.tol3z;
        if (!again) wk *= sqrt(temp);
      }
      for (unsigned long long left = __ballot(again); left; left &= left - 1) {
        const int i = __builtin_ctzll(left);
        const double nr =
            (mrem > 0) ? wave_nrm2(a + (size_t)(cb + NW * i) * lda + j + kk, mrem) : 0.0;
        if (lane == i) {
          wk = nr;
          L.wold[col] = nr;
        }
      }
      if (live) {
        L.work[col] = wk;
        if (wk == wk) nmx = fmax(nmx, wk);
      }
    }
    const double maxnrm = block_max(nmx, L.red);
    // --- step end (src/dgeqrdm_work.c:740, :780-785)
    if (tid == 0) nc_all[it.col_off + itn] = kk;
    itn++;
    int done = (j + kk >= minmn) ? 1 : 0;
    if (enable_stop && maxnrm * sqrt((double)(n - j - kk)) <= eta) done = 1;
    j += kk;
    __syncthreads();
    if (done) break;
  }
  for (int c = tid; c < n; c += NT) jp_all[it.col_off + c] = L.jp[c];
  return 0;
}

// Persistent batch kernel: the workgroups factorise the matrices
// order[0 .. count), each taking the next index from queue[0].
template <int NW>
__global__ __launch_bounds__(64 * NW) void k_dm_batch(const BatchItem* __restrict__ items,
                                                      const int* __restrict__ order, int count,
                                                      int* queue, double* A, double* tau,
                                                      int* jpvt, int* ncols, int* info,
                                                      BatchParams P) {
  __shared__ BatchLds<NW> L;
  __shared__ int s_next;
  // Each workgroup takes the next matrix of order (decreasing flop count)
  // until none is left: list scheduling on the actual durations.  A
  // matrix's arithmetic does not depend on the workgroup that runs it.
  for (;;) {
    if (threadIdx.x == 0) s_next = atomicAdd(&queue[0], 1);
    __syncthreads();
    const int b = s_next;
    if (b >= count) break;  // every thread read the same s_next
    const int idx = order[b];
    const BatchItem it = items[idx];
    const int r = bt_factor<NW>(it, A, tau, jpvt, ncols, P, L);
    if (threadIdx.x == 0) info[idx] = r;
    __syncthreads();  // s_next is read by all before thread 0 takes the next
  }
  // the last workgroup out zeroes the queue for the next launch (a graph
  // replay included): every other workgroup has taken its last index
  if (threadIdx.x == 0 && atomicAdd(&queue[1], 1) == (int)gridDim.x - 1) {
    atomicExch(&queue[0], 0);
    atomicExch(&queue[1], 0);
  }
}

int launch_dm_batch(int waves, int grid, const void* items, const int* order, int count,
                     int* queue, double* A, double* tau, int* jpvt, int* ncols,
                     int* info, int nb, double delta, double tau_dm, int stop_mode, double eta3,
                     double tol3z, const void* policy, float* trace, unsigned* trace_count,
                     int trace_cap, const float* ranges, int gram_rows, hipStream_t s) {
  BatchParams P{delta, tau_dm, eta3, tol3z, nb, stop_mode,
                static_cast<const PolicyNet*>(policy), trace, trace_count, trace_cap,
                ranges ? ranges[0] : 0.f, ranges ? ranges[1] : 1.f,
                ranges ? ranges[2] : 0.f, ranges ? ranges[3] : 1.f,
                gram_rows > 0 ? gram_rows : INT_MAX};
  const BatchItem* it = static_cast<const BatchItem*>(items);
  // Only the 4-wave shape is instantiated: runs of k_dm_batch<8> on a
  // 4096-matrix batch ended in host-heap aborts of unidentified cause.
  if (waves != 4) return -1;
  hipLaunchKernelGGL(k_dm_batch<4>, dim3(grid), dim3(256), 0, s, it, order, count, queue, A,
                     tau, jpvt, ncols, info, P);
  return 0;
}

}  // namespace qrdm
