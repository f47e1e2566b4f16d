// regpanel.hip -- the column-by-column Householder panel (dgeqr2_mia,
// src/dgeqr2.c:144-191, with dlarfg_mia, src/dlarfg.c:116-185) with the panel
// held in registers.
//
// What bounds it: 64 columns that each wait on the one before.  A panel kept
// in memory (panel_exact_body) costs every column three round trips to the L2
// (norm, scaling, update).  Here a workgroup keeps RP_ROWS rows x 64 columns in
// registers (a wave 16 QH rows, a lane 4 QH rows of four columns), so that a
// column costs one pass of products, one LDS exchange and one barrier:
//
//   x = column i below the diagonal; s_c = x^T (column c) for all 64 columns
//   in one reduction: s_i = ||x||^2 gives beta, tau and the scale
//   sc = 1 / (alpha - beta); for c > i, w_c = tau (a_ic + sc s_c) is dlarf_'s
//   product v^T (column c); for c < i, a_ic + sc s_c = (V^T v_i)_c is the entry
//   of V^T V that T needs.
//
// Row i leaves the registers when column i is done (R to the right of the
// diagonal, V to the left), through LDS; the rest is written once, at the end,
// with the dense V of the trailing update.  One wave that holds no rows builds
// T's diagonal blocks from those entries beside the others' updates.  Panels of
// more than RP_ROWS rows take a workgroup per RP_HALF (or RP_ROWS) rows: every
// column's partial sums pass between the workgroups through memory, each in a slot
// that holds a sentinel until it is written.
//
// The workgroups of such a panel wait for each other, so all of them have to be on
// the chip at once.  They meet before column 0 (rp_all_here), while nothing is
// written: where one does not arrive in time -- another kernel or process holds the
// CUs -- all of them decline, and the memory-based panel, one workgroup that waits
// for nobody, takes it.  Once all have met they stay, and every later wait ends.
// Devices with fewer CUs than the panel has workgroups, and streams with a CU mask,
// go to the memory-based panel at once.
//
// Measured for 64 columns, with V and T (rocprofv3): up to 128 rows 67 us, up to 336
// rows 87, up to 448 rows 105 us (memory-based: about 180 us for 64 rows, with T another
// 60), 1024 rows on five workgroups 136 us, 4096 rows on nineteen 160 us
// (memory-based 3.8 ms; on ten workgroups over all XCDs 189).  A column costs
// about 2500 cycles at 128 rows and 3600 at 448, of which the reflector's scalars
// take 280; between workgroups the exchange adds 2000 to 2500.  The loop is
// unrolled over the four column groups so that every register index is static:
// with uniform branches in their place the 448-row panel took 163 us.  Unpivoted
// QR of 1024 x 1024 15.5 -> 2.3 ms, of 4096 x 2048 129 -> 6.6 ms; 2048 x 1024 DM
// with 128-column blocks 68.2 -> 4.25 ms; 64 x 48 DM 0.51 -> 0.22 ms.
//
// Sums of squares are taken plainly: where one leaves [1e-280, 1e280] (or is
// not a number) the panel is declined before anything is written, and the
// memory-based panel, which scales, takes it.  So are panels with a column below
// that range that may never be summed itself.
#include <stdlib.h>
#include <string.h>

#include <algorithm>

#include "qrdm_internal.h"

namespace qrdm {

constexpr int RP_ROWS = 448;  // rows per workgroup (seven waves of 64, and the one for T)
constexpr int RP_SMALL = 128;  // panels up to this many rows: four waves of 32
constexpr int RP_MID = 336;    // up to this many: seven waves of 48
constexpr int RP_WGS = 64;     // workgroups of one panel at most
constexpr int RP_HALF = 224;   // rows per workgroup while that leaves RP_XCD of them at most
// Up to this many workgroups (one per CU: an XCD has 32) every eighth of the grid
// works, which puts them on one XCD, whose L2 then carries the exchange: a round
// among ten took 1900 cycles against 2700 over all XCDs (3000 with a fresh slot for
// every column, which is read from memory first).  Only speed depends on it.
constexpr int RP_XCD = 28;

// A slot not yet written: a NaN pattern no published value takes (published
// NaNs are made the canonical one).
__device__ constexpr unsigned long long kRpEmpty = 0x7ff4a5a5c3c30f0full;
// Polls of one slot before a workgroup gives the panel up (about seconds; only a
// workgroup that is gone could keep one empty).
constexpr int RP_POLLS = 1 << 22;
// Polls for the workgroups not here yet before all decline: a few milliseconds, about
// what the memory-based panel takes at 4096 rows.
constexpr int RP_MEET = 1 << 12;
// The meeting's word (the first of the slots' space): how many are here, and whether
// one has declined for all.
constexpr unsigned kRpDeclined = 0x80000000u;

// Two doubles at any multiple of eight bytes.
typedef double rp_pair __attribute__((ext_vector_type(2), aligned(8)));

// QH: 16-row groups per data wave; NW: data waves.  One more wave builds T.
template <int QH, int NW>
struct RegPanelLds {
  double x[NW][16 * QH];        // column i's rows, per wave
  double red[2][NW][KMAX];      // partial sums, by column
  double all[2][NW + 2][KMAX];  // their sums over shares of the workgroups, and row i
  double row[2][KMAX];          // row i
  double out[KMAX][LDP];        // the top block: R, V below the diagonal
  double S[KMAX][LDP];          // V^T V above the diagonal, else zero
  double X[KMAX][LDP];          // T
  double Y[4][BLK][BLK + 1];
  double tau[KMAX];
  int here;
};

// (lane 16 g + li) := the sum over the four lane groups of s[g], column 16 g + li.
__device__ __forceinline__ double group_sums(const double (&s)[4]) {
  auto halves = [](double a, double b) {  // lanes < 32: a's two halves summed, else b's
    const long long x = __double_as_longlong(a), y = __double_as_longlong(b);
    const auto lo = __builtin_amdgcn_permlane32_swap((int)x, (int)y, false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap((int)(x >> 32), (int)(y >> 32), false, false);
    return __longlong_as_double(((long long)(int)hi[0] << 32) | (unsigned)lo[0]) +
           __longlong_as_double(((long long)(int)hi[1] << 32) | (unsigned)lo[1]);
  };
  auto rows = [](double a, double b) {  // even rows of 16: a's row pair summed, odd rows: b's
    const long long x = __double_as_longlong(a), y = __double_as_longlong(b);
    const auto lo = __builtin_amdgcn_permlane16_swap((int)x, (int)y, false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap((int)(x >> 32), (int)(y >> 32), false, false);
    return __longlong_as_double(((long long)(int)hi[0] << 32) | (unsigned)lo[0]) +
           __longlong_as_double(((long long)(int)hi[1] << 32) | (unsigned)lo[1]);
  };
  return rows(halves(s[0], s[2]), halves(s[1], s[3]));
}

// f[u] := the value of lane 16 u + li in lane 16 g + li.
__device__ __forceinline__ void group_values(double v, double (&f)[4]) {
  const long long b = __double_as_longlong(v);
  int w[4][2];
#pragma unroll
  for (int h = 0; h < 2; h++) {
    const int x = h ? (int)(b >> 32) : (int)b;
    const auto p = __builtin_amdgcn_permlane16_swap(x, x, false, false);  // rows 0022, 1133
    const auto e = __builtin_amdgcn_permlane32_swap(p[0], p[0], false, false);  // 0000, 2222
    const auto o = __builtin_amdgcn_permlane32_swap(p[1], p[1], false, false);  // 1111, 3333
    w[0][h] = e[0];
    w[1][h] = o[0];
    w[2][h] = e[1];
    w[3][h] = o[1];
  }
#pragma unroll
  for (int u = 0; u < 4; u++)
    f[u] = __longlong_as_double(((long long)w[u][1] << 32) | (unsigned)w[u][0]);
}

__device__ __forceinline__ double rp_publishable(double v) {
  return v == v ? v : __longlong_as_double(0x7ff8000000000000ll);
}

// Whether any of the n values is not zero (a wave).
__device__ __forceinline__ bool rp_nonzero(const double* v, int n) {
  bool any = false;
  for (int e = local_tid() & 63; e < n; e += 64) any |= v[e] != 0.0;
  return __any(any) != 0;
}

// v := the sum, in order, of the slots first, first + step, ... < n (each of
// KMAX values, this lane's); false when one stayed empty for RP_POLLS polls.
// The slots' loads are in flight together.
__device__ __forceinline__ bool rp_collect(const double* slots, int first, int step, int n,
                                           double& v) {
  constexpr int BATCH = 4;
  const int lane = local_tid() & 63;
  v = 0.0;
  for (int b0 = first; b0 < n; b0 += BATCH * step) {
    unsigned long long w[BATCH];
    int polls = 0;
    for (;;) {
      bool empty = false;
#pragma unroll
      for (int q = 0; q < BATCH; q++) {
        const int b = b0 + q * step;
        w[q] = 0ull;
        if (b < n)
          w[q] = __hip_atomic_load(
              reinterpret_cast<const unsigned long long*>(slots) + b * KMAX + lane,
              __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
#pragma unroll
      for (int q = 0; q < BATCH; q++) empty |= w[q] == kRpEmpty;
      if (!__any(empty)) break;
      if (++polls == RP_POLLS) return false;
    }
#pragma unroll
    for (int q = 0; q < BATCH; q++)
      if (b0 + q * step < n) v += __longlong_as_double((long long)w[q]);
  }
  return true;
}

// Whether all nwg workgroups, each counted into *word, are here; false for all of
// them when one has waited RP_MEET polls in vain.  (One thread.  The word goes from
// "not all here" to one of the two answers once, by the last arrival's count or by
// the exchange, and every workgroup, a late one too, reads that answer.)
__device__ __forceinline__ bool rp_all_here(unsigned* word, unsigned nwg) {
  for (int polls = 0;; polls++) {
    unsigned v = __hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (v & kRpDeclined) return false;
    if (v == nwg) return true;
    if (polls >= RP_MEET)
      __hip_atomic_compare_exchange_strong(word, &v, v | kRpDeclined, __ATOMIC_RELAXED,
                                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// The panel's columns [0, fjb) at P (leading dimension lda, msub rows) by nwg
// workgroups, this one the rows from wg * 16 QH NW.  Truncation: 5e-14 is the
// bound of the columns after the first (tau_dm > 0: tau_dm |R(0, 0)| once
// column 0 is done), unless truncate is 0; truncate = 2: beta0 is the block's
// R(0, 0), and every column is tested.  slots (GRID): the meeting's word, in which
// this workgroup is counted, and, from KMAX values on, four columns' sets
// of (nwg + 1) x KMAX values, empty on entry; column i uses set i mod 4 and
// empties its own slot of column i + 2, whose values (of column i - 2) every
// workgroup has read before any publishes column i - 1.  Returns the columns reduced with
// everything written -- the panel, tau, rows [-z0, msub) of the dense V (zero
// above the panel) and T, or with T_out null T^-1 as the merged trailing pass
// takes it -- or -1, declined, with nothing written.  Every
// workgroup returns the same (one that gives up waiting sets flags bit 3,
// which fails the call).
template <int QH, int NW, bool GRID>
__device__ __forceinline__ int reg_panel(double* P, int lda, int msub, int fjb, double tau_dm,
                                         int truncate, double beta0, double* tau, double* V,
                                         int ldv, int z0, double* T_out, double* S_out,
                                         double* slots, int nwg, int wg, bool scales,
                                         DevState* st, RegPanelLds<QH, NW>& L) {
  constexpr int WR = 16 * QH, NQ = 4 * QH, NT = 64 * (NW + 1);
  const int tid = local_tid(), lane = tid & 63, g = lane >> 4, li = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool data = wave < NW;  // the last wave builds T
  const int row0 = data ? wg * WR * NW + wave * WR : 0;  // this wave's first row
  // the lane's rows: row0 + 16 (q / 4) + 4 g + q % 4
  double a[4][NQ];
#pragma unroll
  for (int u = 0; u < 4; u++)
#pragma unroll
    for (int h = 0; h < QH; h++) {
      const int r = row0 + 16 * h + 4 * g, c = 16 * u + li;
      const double* p = P + (size_t)c * lda + r;
      rp_pair lo = {0.0, 0.0}, hi = {0.0, 0.0};
      if (data && c < fjb) {
        if (r + 3 < msub) {
          lo = *reinterpret_cast<const rp_pair*>(p);
          hi = *reinterpret_cast<const rp_pair*>(p + 2);
        } else {
          if (r < msub) lo.x = p[0];
          if (r + 1 < msub) lo.y = p[1];
          if (r + 2 < msub) hi.x = p[2];
        }
      }
      a[u][4 * h] = lo.x;
      a[u][4 * h + 1] = lo.y;
      a[u][4 * h + 2] = hi.x;
      a[u][4 * h + 3] = hi.y;
    }
  if constexpr (GRID) {
    if (tid == 0) L.here = rp_all_here(reinterpret_cast<unsigned*>(slots), nwg) ? 1 : 0;
    lds_barrier();
    if (!L.here) return -1;
    slots += KMAX;
  }
  // column 16 u + ii to LDS: its owner lanes' rows, zero on and above the diagonal
  auto put_column = [&](int u, int ii) {
    if (li == ii) {
#pragma unroll
      for (int q = 0; q < NQ; q += 2)
        *reinterpret_cast<double2*>(&L.x[wave][16 * (q >> 2) + 4 * g + (q & 3)]) =
            make_double2(a[u][q], a[u][q + 1]);
    }
    if (wg == 0 && wave <= u / QH && lane < WR && lane <= 16 * u + ii - row0)
      L.x[wave][lane] = 0.0;
  };
  // row 16 ur + ii, before its step, from the lanes that hold it
  auto put_row = [&](int ur, int ii) {
    if (wg != 0 || wave != ur / QH) return;
    const int h = 4 * (ur % QH), ql = ii & 3;
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const double lo = ql & 1 ? a[u][h + 1] : a[u][h], hi = ql & 1 ? a[u][h + 3] : a[u][h + 2];
      if (g == ii >> 2) L.row[ii & 1][16 * u + li] = ql & 2 ? hi : lo;
    }
  };
  const bool cont = truncate == 2;
  const double thr0 = cont && tau_dm > 0.0 ? tau_dm * beta0 : 5e-14;
  double thr2 = truncate && cont ? thr0 * thr0 : -1.0;  // nothing is below -1
  int k = fjb;
  bool ok = true;
  // After the data waves' partial sums of column i: sum := x^T (column lane),
  // rv := row i's entry there.  (i = -1: any sums, before column 0's.)
  auto exchange = [&](int i, double& sum, double& rv) {
    const int buf = i & 1;
    lds_barrier();
    if constexpr (GRID) {
      // this workgroup's sums (and row i, from the one that holds it) to the
      // others; wave w then collects workgroups w, w + NW + 1, ... in order
      double* sl = slots + (size_t)(i & 3) * (nwg + 1) * KMAX;
      double* s2 = slots + (size_t)((i + 2) & 3) * (nwg + 1) * KMAX;
      const double none = __longlong_as_double((long long)kRpEmpty);
      handoff_wait();  // the slot emptied a column ago is empty for everyone
      if (wave == 0) {
        double t = L.red[buf][0][lane];
#pragma unroll
        for (int w = 1; w < NW; w++) t += L.red[buf][w][lane];
        if (rdlane(t, i) == 0.0 && rp_nonzero(&L.x[0][0], NW * WR) && lane == i) t = 1e-300;
        st_dev(sl + wg * KMAX + lane, rp_publishable(t));
        st_dev(s2 + wg * KMAX + lane, none);
      }
      if (wg == 0 && wave == 1) {
        st_dev(sl + nwg * KMAX + lane, rp_publishable(L.row[buf][lane]));
        st_dev(s2 + nwg * KMAX + lane, none);
      }
      double t = 0.0, rr = 0.0;
      bool got = rp_collect(sl, wave, NW + 1, nwg, t);
      if (wave == NW) got &= rp_collect(sl, nwg, 1, nwg + 1, rr);
      if (!got) {
        if (lane == 0) atomicOr(&st->flags, 8);  // given up: the call fails
        t = __longlong_as_double(0x7ff8000000000000ll);
      }
      L.all[buf][wave][lane] = t;
      if (wave == NW) L.all[buf][NW + 1][lane] = rr;
      lds_barrier();
      rv = L.all[buf][NW + 1][lane];
      sum = L.all[buf][0][lane];
#pragma unroll
      for (int w = 1; w < NW + 1; w++) sum += L.all[buf][w][lane];
    } else {
      rv = L.row[buf][lane];
      sum = L.red[buf][0][lane];
#pragma unroll
      for (int w = 1; w < NW; w++) sum += L.red[buf][w][lane];
    }
  };
  // dlarfg of column i (every wave computes the same): tau, beta, 1 / (alpha -
  // beta); false ends the panel before column i.  y = 1 / sqrt(t2) by one
  // third-order step from the hardware's estimate; the reciprocal of alpha -
  // beta likewise, its estimate taken beside y's step.
  auto reflect = [&](int i, double sum, double rv, double& taui, double& beta, double& sc) {
    const double si = rdlane(sum, i), alpha = rdlane(rv, i);
    const double aa = fabs(alpha), t2 = fma(alpha, alpha, si);
    if (si >= 1e-280 && t2 <= 1e280 && si >= thr2) {
      double y = __builtin_amdgcn_rsq(t2);
      double e = __builtin_amdgcn_rcp(fma(t2, y, aa));
      const double h = fma(-t2 * y, y, 1.0);
      y = fma(y * h, fma(0.375, h, 0.5), y);
      double b = t2 * y;
      b = fma(fma(-b, b, t2), 0.5 * y, b);
      taui = fma(aa, y, 1.0);  // (beta - alpha) / beta
      const double r = fma(-(aa + b), e, 1.0);
      e = fma(fma(r, r, r), e, e);
      sc = alpha >= 0 ? e : -e;
      beta = alpha >= 0 ? -b : b;
    } else {
      // a zero column (tau = 0), the truncation, or out of range
      bool zero = si == 0.0;
      if (!GRID && zero) {
        zero = !rp_nonzero(&L.x[0][0], NW * WR);
        lds_barrier();  // every wave has looked
      }
      if (!zero && !(si >= 1e-280 && t2 <= 1e280)) {
        ok = false;
        return false;
      }
      // (a column of one row is not tested: dlarfg_mia returns before the test)
      if (msub - i > 1 && si < thr2) {
        k = i;
        return false;
      }
      taui = 0.0;
      beta = alpha;
      sc = 1.0;
    }
    if (truncate && i == 0 && !cont) {
      const double thr = tau_dm > 0.0 && fjb > 1 ? tau_dm * beta : thr0;
      thr2 = thr * thr;
    }
    return true;
  };
  // A column whose entries are all so small that their products with an accepted
  // column could be lost (each entry counts 1 from 1e-140 on, below that 2^-30): the
  // panel is declined.
  if (scales) {
    if (data) {
      double s[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int u = 0; u < 4; u++)
#pragma unroll
        for (int q = 0; q < NQ; q++)
          s[u] += fabs(a[u][q]) >= 1e-140 ? 1.0 : (a[u][q] != 0.0 ? 0x1p-30 : 0.0);
      L.red[1][wave][lane] = group_sums(s);
    }
    double sum, rv;
    exchange(-1, sum, rv);
    if (__any(sum > 0.0 && sum < 1.0)) return -1;
  }
  if (data) {
    put_column(0, 0);
    put_row(0, 0);
    bool go = true;
#pragma unroll
    for (int ui = 0; ui < 4; ui++) {
      for (int ii = 0; go && ii < 16 && 16 * ui + ii < fjb; ii++) {
        const int i = 16 * ui + ii;
        wave_lds_sync();
        double x[NQ];
#pragma unroll
        for (int q = 0; q < NQ; q += 2) {
          const double2 t =
              *reinterpret_cast<const double2*>(&L.x[wave][16 * (q >> 2) + 4 * g + (q & 3)]);
          x[q] = t.x;
          x[q + 1] = t.y;
        }
        // eight independent chains
        double s[4] = {0.0, 0.0, 0.0, 0.0}, s1[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int q = 0; q < NQ; q += 2)
#pragma unroll
          for (int u = 0; u < 4; u++) {
            s[u] = fma(x[q], a[u][q], s[u]);
            s1[u] = fma(x[q + 1], a[u][q + 1], s1[u]);
          }
#pragma unroll
        for (int u = 0; u < 4; u++) s[u] += s1[u];
        L.red[i & 1][wave][lane] = group_sums(s);  // column `lane`
        double sum, rv, taui, beta, sc;
        exchange(i, sum, rv);
        go = reflect(i, sum, rv, taui, beta, sc);
        if (!go) break;
        // c > i: v^T (column c); c < i: (V^T V)(c, i)
        const double vc = fma(sc, sum, rv);
        double f[4];
        group_values(lane > i ? -(taui * sc) * vc : (lane == i ? sc : 0.0), f);
        if (li == ii) {
#pragma unroll
          for (int q = 0; q < NQ; q++) a[ui][q] = 0.0;  // becomes v = sc x
        }
#pragma unroll
        for (int u = ui; u < 4; u++) {
#pragma unroll
          for (int q = 0; q < NQ; q++) a[u][q] = fma(x[q], f[u], a[u][q]);
          // the next column's way through LDS runs beside the other groups
          if (u == ui && ii < 15) put_column(ui, ii + 1);
          if (u == ui + 1 && ii == 15) put_column(ui + 1, 0);
        }
        if (ii < 15) put_row(ui, ii + 1);
        else if (ui < 3) put_row(ui + 1, 0);
        if (wg == 0 && wave == 0)
          L.out[i][lane] = lane < i ? rv : (lane == i ? beta : fma(-taui, vc, rv));
      }
    }
  } else {
    if (wg == 0) {
      for (int r = 0; r < KMAX; r++) L.S[r][lane] = L.X[r][lane] = 0.0;
    }
    // T's 16 x 16 diagonal blocks by dlarft's recurrence, lane p its row p
    // (z = V^T v_i by row broadcasts); the other blocks follow from them
    double tb[BLK];
    for (int i = 0; i < fjb; i++) {
      const int ui = i >> 4, ii = i & 15;
      double sum, rv, taui, beta, sc;
      exchange(i, sum, rv);
      if (!reflect(i, sum, rv, taui, beta, sc)) break;
      if (wg != 0) continue;
      const double vc = fma(sc, sum, rv);
      if (ii == 0) {
#pragma unroll
        for (int t = 0; t < BLK; t++) tb[t] = 0.0;
      }
      double t0 = 0.0, t1 = 0.0;
#pragma unroll
      for (int t = 0; t < BLK; t += 2) {
        t0 = fma(tb[t], row_bcast(vc, t), t0);
        t1 = fma(tb[t + 1], row_bcast(vc, t + 1), t1);
      }
      const double v = li < ii ? -taui * (t0 + t1) : (li == ii ? taui : 0.0);
#pragma unroll
      for (int t = 0; t < BLK; t++) tb[t] = t == ii ? v : tb[t];
      if (g == ui) L.X[lane][i] = v;
      if (lane < i) L.S[lane][i] = vc;
      if (lane == 0) L.tau[i] = taui;
    }
  }
  lds_barrier();
  if (!ok) return -1;
  // the rows below the top k: V left of column k, updated columns right of it
#pragma unroll
  for (int u = 0; u < 4; u++)
#pragma unroll
    for (int h = 0; h < QH; h++) {
      const int r = row0 + 16 * h + 4 * g, c = 16 * u + li;
      double* p = P + (size_t)c * lda + r;
      double* pv = V + (size_t)c * ldv + r;
      const bool in = c < fjb, on = c < k;
      if (data && r >= k && r + 3 < msub) {
        const rp_pair lo = {a[u][4 * h], a[u][4 * h + 1]}, hi = {a[u][4 * h + 2], a[u][4 * h + 3]};
        const rp_pair zero = {0.0, 0.0};
        if (in) {
          *reinterpret_cast<rp_pair*>(p) = lo;
          *reinterpret_cast<rp_pair*>(p + 2) = hi;
        }
        *reinterpret_cast<rp_pair*>(pv) = on ? lo : zero;
        *reinterpret_cast<rp_pair*>(pv + 2) = on ? hi : zero;
      } else if (data) {
#pragma unroll
        for (int q = 0; q < 4; q++)
          if (r + q >= k && r + q < msub) {
            if (in) p[q] = a[u][4 * h + q];
            pv[q] = on ? a[u][4 * h + q] : 0.0;
          }
      }
    }
  if (wg != 0) return k;
  if (T_out) inverse_merge(L.S, L.X, L.Y);  // T = (striu(V^T V) + diag(1 / tau))^-1
  const int tid2 = local_tid();
  for (int e = tid2; e < KMAX * KMAX; e += NT) {
    const int r = e & 63, c = e >> 6;
    if (r < k) {
      const double v = L.out[r][c];
      if (c < fjb) P[(size_t)c * lda + r] = v;
      V[(size_t)c * ldv + r] = c < k ? (r > c ? v : (r == c ? 1.0 : 0.0)) : 0.0;
    }
    if (r < z0) V[(size_t)c * ldv + r - z0] = 0.0;
    if (T_out)
      T_out[r + c * KMAX] = r <= c && c < k ? L.X[r][c] : 0.0;
    else
      S_out[r + c * KMAX] = c < k ? (r < c ? L.S[r][c] : (r == c ? L.tau[c] : 0.0)) : 0.0;
  }
  if (tid2 < k) tau[tid2] = L.tau[tid2];
  return k;
}

// Panels (RUN_ALWAYS: host j, fjb, the first V buffer; RUN_EXACT: j and fjb
// from st, tau indexed from column 0, V of the step's parity).  The dense V,
// T and the slots lie in the workspace behind st (ws_v, ws_mat, ws_slots).
// truncate = 2: the panel continues a wider block (wide.hip), whose first
// pivot st->pan_beta bounds every column, the first included.  A declined
// panel sets DevState::flags bit 2 for k_panel_slow, queued behind.
template <int QH, int NW, bool GRID>
__global__ __launch_bounds__(64 * (NW + 1)) void k_panel_reg(double* A, int lda, int j, int m, int fjb,
                                                       double tau_dm, int truncate, double* tau,
                                                       DevState* st, int mode, int stride) {
  __shared__ RegPanelLds<QH, NW> L;
  if (!step_runs(st, mode)) return;
  const int ldv = ws_ldv(m);
  double* V = ws_v(st, m);
  if (mode != RUN_ALWAYS) {
    j = st->j;
    fjb = st->fjb;
    tau += j;
    if (st->fused) V += (size_t)(st->it & 1) * ldv * KMAX;
  }
  const int msub = m - j;
  const int nwg = GRID ? (msub + 16 * QH * NW - 1) / (16 * QH * NW) : 1;
  const int wg = blockIdx.x / stride;
  // one workgroup in stride works; the grid is sized for the lowest j
  if (wg * stride != (int)blockIdx.x || wg >= nwg) return;
  // Columns that no test of their own reaches: those the truncation rejects, and one
  // with a single row left.  As DM candidates they are above tau_dm times the first
  // column's norm, which is tested; otherwise the panel looks at their scale first.
  const bool picked = truncate && tau_dm >= 1e-20 && !(mode != RUN_ALWAYS && st->policy_on);
  const bool scales = (truncate || fjb >= msub) && !picked;
  // (counted first: the panel's loads run beside the wait for the others)
  if (GRID && threadIdx.x == 0)
    __hip_atomic_fetch_add(reinterpret_cast<unsigned*>(ws_slots(st)), 1u, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
  const double beta0 = truncate == 2 ? st->pan_beta : 0.0;
  const int k = reg_panel<QH, NW, GRID>(A + j + (size_t)j * lda, lda, msub, fjb, tau_dm, truncate,
                                        beta0, tau, V + j, ldv, min(j, KMAX),
                                        mode != RUN_ALWAYS && st->fused ? nullptr
                                                                        : ws_mat(st, WS_T),
                                        ws_mat(st, WS_S), ws_slots(st), nwg, wg, scales, st,
                                        L);
  if (wg == 0 && threadIdx.x == 0) {
    if (k < 0) {
      atomicOr(&st->flags, 4);
    } else {
      if (truncate != 2) st->pan_beta = L.out[0][0];
      st->fjb_cmp = k;
      // the rejected columns j + k .. j + fjb are already updated (as dlarf_
      // does inside the reference's panel); the trailing update starts after
      st->c0 = j + fjb;
    }
  }
}

// The panel in memory, column by column (panel_exact_body: norms with
// dnrm2's scaling, any number of rows), then V and T, by one workgroup: runs
// when the register-held form declined (flags bit 2), or with force.
__global__ __launch_bounds__(1024) void k_panel_slow(double* A, int lda, int j, int m, int fjb,
                                                     double tau_dm, int truncate, double* tau,
                                                     DevState* st, int mode, int force) {
  __shared__ double Ss[KMAX * KMAX];
  __shared__ double Ts[KMAX * KMAX];
  __shared__ double tmp[KMAX], ts[KMAX], red[16];
  if (!step_runs(st, mode) || !(force || (st->flags & 4))) return;
  const int ldv = ws_ldv(m);
  double* V = ws_v(st, m);
  if (mode != RUN_ALWAYS) {
    j = st->j;
    fjb = st->fjb;
    tau += j;
    if (st->fused) V += (size_t)(st->it & 1) * ldv * KMAX;
  }
  const double beta0 = truncate == 2 ? st->pan_beta : 0.0;
  const int k = panel_exact_body<1>(A, lda, j, m, fjb, tau_dm, truncate, tau, red, beta0);
  __syncthreads();
  const int tid = local_tid(), lane = tid & 63, wave = tid >> 6, g = lane >> 4, li = lane & 15;
  for (int c = wave; c < KMAX; c += 16)
    for (int r = max(j - KMAX, 0) + lane; r < m; r += 64)
      V[(size_t)c * ldv + r] = (c >= k || r < j + c) ? 0.0
                               : (r == j + c ? 1.0 : A[(size_t)(j + c) * lda + r]);
  for (int e = tid; e < KMAX * KMAX; e += 1024) Ss[e] = Ts[e] = 0.0;
  if (tid < KMAX) ts[tid] = tid < k ? tau[tid] : 0.0;
  __syncthreads();
  // S = V^T V: wave w takes the 16-row blocks w, w + 16, ...; summed in wave order
  dbl4 gt[10];
#pragma unroll
  for (int p = 0; p < 10; p++) gt[p] = (dbl4){0.0, 0.0, 0.0, 0.0};
  for (int rb = j + 16 * wave; rb < m; rb += 256) {
    dbl4 xb[4];
#pragma unroll
    for (int u = 0; u < 4; u++)
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const int r = rb + g + 4 * v;
        xb[u][v] = r < m ? V[(size_t)(16 * u + li) * ldv + r] : 0.0;
      }
    gram_tiles(xb, gt);
  }
  for (int w = 0; w < 16; w++) {
    if (wave == w) {
      int p = 0;
#pragma unroll
      for (int u = 0; u < 4; u++)
#pragma unroll
        for (int u2 = u; u2 < 4; u2++) {
#pragma unroll
          for (int v = 0; v < 4; v++) Ss[(16 * u + g + 4 * v) + (16 * u2 + li) * KMAX] += gt[p][v];
          p++;
        }
    }
    __syncthreads();
  }
  larft_recurrence(Ss, Ts, ts, tmp, k);
  for (int e = tid; e < KMAX * KMAX; e += 1024) {
    const int r = e & 63, c = e >> 6;
    ws_mat(st, WS_T)[e] = Ts[e];
    ws_mat(st, WS_S)[e] = c < k ? (r < c ? Ss[e] : (r == c ? ts[c] : 0.0)) : 0.0;
  }
  if (tid == 0) {
    if (truncate != 2) st->pan_beta = A[(size_t)j * lda + j];
    st->fjb_cmp = k;
    st->c0 = j + fjb;
    st->flags &= ~4;
  }
}

// The meeting's word (nobody here, or declined), and every slot of a panel by several
// workgroups empty (see kRpEmpty).
__global__ __launch_bounds__(256) void k_panel_slots(DevState* st, int n, int mode,
                                                     unsigned word) {
  if (!step_runs(st, mode)) return;
  unsigned long long* s = reinterpret_cast<unsigned long long*>(ws_slots(st));
  for (int e = blockIdx.x * 256 + threadIdx.x; e < KMAX + n; e += gridDim.x * 256)
    s[e] = e < KMAX ? word : kRpEmpty;
}

// The CUs that a panel's workgroups can count on: the device's, or none with a mask
// on the stream.
static int panel_cus(hipStream_t s) {
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
    return 0;
  // (the default streams have no mask, and the call is not for the named ones)
  if (s == nullptr || s == hipStreamLegacy || s == hipStreamPerThread) return cus;
  uint32_t mask[32] = {0};
  if (hipExtStreamGetCUMask(s, 32, mask) != hipSuccess) {
    (void)hipGetLastError();
    return cus;  // (the meeting decides)
  }
  int on = 0;
  for (uint32_t w : mask) on += __builtin_popcount(w);
  return on < cus ? 0 : cus;
}

// The form by the panel's rows (m - j, j the lowest the step can have): up to
// RP_SMALL rows four waves of 32 rows, up to RP_MID seven of 48, up to RP_ROWS
// seven of 64 in one workgroup, then RP_HALF or RP_ROWS rows per workgroup, at most
// RP_WGS of them and no more than there are CUs for.  Larger ones stay in memory.
// (QRDM_PANEL=alone: the panels of several workgroups decline where they meet.)
void launch_panel_exact(double* A, int lda, int j, int m, int fjb, double tau_dm,
                        int truncate, double* tau, DevState* st, hipStream_t s, int mode) {
  if (truncate == PANEL_GIVEN) {
    launch_given_panel(A, lda, j, m, fjb, tau, st, s);
    return;
  }
  const int rows = m - j, nwg = (rows + RP_ROWS - 1) / RP_ROWS;
  const int half = (rows + RP_HALF - 1) / RP_HALF;
  bool in_memory = nwg > RP_WGS;
  auto grid = [&](auto kernel, int n) {
    const int cus = panel_cus(s);
    in_memory = n > cus;
    if (in_memory) return;
    const int stride = n <= std::min(RP_XCD, cus / 8) ? 8 : 1;
    const char* pe = getenv("QRDM_PANEL");
    const unsigned word = pe && strcmp(pe, "alone") == 0 ? kRpDeclined : 0u;
    hipLaunchKernelGGL(k_panel_slots, dim3(n + 2), dim3(256), 0, s, st, 4 * KMAX * (n + 1), mode,
                       word);
    hipLaunchKernelGGL(kernel, dim3(n * stride), dim3(512), 0, s, A, lda, j, m, fjb, tau_dm,
                       truncate, tau, st, mode, stride);
  };
  if (rows <= RP_SMALL)
    hipLaunchKernelGGL((k_panel_reg<2, 4, false>), dim3(1), dim3(320), 0, s, A, lda, j, m, fjb,
                       tau_dm, truncate, tau, st, mode, 1);
  else if (rows <= RP_MID)
    hipLaunchKernelGGL((k_panel_reg<3, 7, false>), dim3(1), dim3(512), 0, s, A, lda, j, m, fjb,
                       tau_dm, truncate, tau, st, mode, 1);
  else if (nwg == 1)
    hipLaunchKernelGGL((k_panel_reg<4, 7, false>), dim3(1), dim3(512), 0, s, A, lda, j, m, fjb,
                       tau_dm, truncate, tau, st, mode, 1);
  else if (half <= RP_XCD)
    grid(k_panel_reg<2, 7, true>, half);
  else if (nwg <= RP_WGS)
    grid(k_panel_reg<4, 7, true>, nwg);
  hipLaunchKernelGGL(k_panel_slow, dim3(1), dim3(1024), 0, s, A, lda, j, m, fjb, tau_dm,
                     truncate, tau, st, mode, in_memory ? 1 : 0);
}

}  // namespace qrdm
