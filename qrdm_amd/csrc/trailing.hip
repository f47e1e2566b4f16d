// trailing.hip -- the DM loop's trailing update as one pass over C per step.
//
// The reference applies each DM step's block reflector to the trailing
// matrix in one dlarfb call (src/dgeqrdm_work.c:762-767, src/dlarfb.c:142):
// W = T^T V^T C, then C -= V W -- three sweeps of C per step (read for W,
// read and write for the update).  Here the update of step s is deferred and
// merged with the next step's first product, so that C is read and written
// once per step:
//
//   k_fused (step s+1):  C -= V_s W_s            (step s's update, deferred)
//                        Wp[slab] = V_{s+1}^T C  (step s+1's partial products
//                                                 on the updated C)
//   k_wsum_norm (s+1):   W_{s+1} = T^T sum_slab Wp; the step's R12 rows
//                        C_top - V_top W_{s+1} (final R rows, written); the
//                        norm downdate of every trailing column from them
//                        (src/dgeqrdm_work.c:80-109); columns whose norm must
//                        be recomputed get the update at once (all rows) and
//                        their W column is cleared.
//
// What the next step needs before its V exists is brought forward: the R12
// rows and the norms (above), and the candidate columns, which the candidate
// Gram kernel updates as it reads them (their W columns are then cleared).
// Columns that move in the step's permutation carry their W column with
// them.  W is stored by absolute column (64 x n per buffer, a column's 64
// entries contiguous); V and W of two consecutive steps alternate between two
// buffers (st->it & 1).
//
// Rounding: V W is summed from zero and then added to C, in every pass and at the
// step's end (R12, the recomputed columns): an entry of C is rounded once.  Summed
// into C on the matrix cores formq 4096 x 2048 was off by 2.3e-15 of its norm instead
// of 1.7e-15, and a recomputed column's small rows by several units in the last
// place instead of half a unit, at the same speed.
#include "qrdm_internal.h"

#include <algorithm>
#include <climits>

namespace qrdm {

constexpr int FU_CH = 32;         // rows per chunk: two interleaved 16-row tiles
constexpr int FU_NWG = 4;         // waves per workgroup
constexpr int FU_MAX_SPLIT = 64;  // row slabs of the partial products at most
constexpr int FU_GC = 16 * FU_NWG;  // columns of a workgroup
constexpr int FU_OCC = 2;         // workgroups per CU (64 KB of LDS each)

// Two doubles at any multiple of eight bytes (a column of any leading dimension).
typedef double fu_pair __attribute__((ext_vector_type(2), aligned(8)));

// Geometry of one fused pass over rows [r_lo, m) and columns [c0, n):
// chunks of FU_CH rows from the FU_CH-row boundary at or below r_lo, split into
// ns slabs of whole chunks, and column groups of FU_GC columns.
struct FuGeom {
  int base, nchunk, slab_ch, cgroups;
};

__host__ __device__ __forceinline__ FuGeom fused_geom(int r_lo, int m, int c0, int n, int ns) {
  FuGeom g;
  g.base = r_lo & ~(FU_CH - 1);
  g.nchunk = (m - g.base + FU_CH - 1) / FU_CH;
  if (g.nchunk < 0) g.nchunk = 0;
  g.slab_ch = (g.nchunk + ns - 1) / ns;
  if (g.slab_ch < 1) g.slab_ch = 1;
  g.cgroups = (n - c0 + FU_GC - 1) / FU_GC;
  if (g.cgroups < 0) g.cgroups = 0;
  return g;
}

// Workgroups of a fused pass per XCD: the (slab, column group) pairs, slab by slab,
// in eight equal runs, so that every XCD has work however few column groups there
// are and reads only its slabs' part of V.  (With a column group's slabs all on one
// XCD every XCD read the whole V, and narrow C left some idle: 16384 x 1024 took
// 86 us a pass.)
__host__ __device__ __forceinline__ int fused_per_xcd(int ns, int cgroups) {
  return (ns * cgroups + 7) / 8;
}

// Row slabs of a fused pass, at most one round of the chip's 64 workgroups per
// XCD (two per CU): the cost of a count in chunks -- a slab's chunks and two for its
// start and its partial tile, 1.7 times as long with a second workgroup on the CU,
// and a twentieth per slab for the step's end -- in twentieths, or INT_MAX where Wp
// (16 x 64 x n values) does not hold the partials.  Whole numbers: the pass and the
// step's end each choose, and have to agree, and counts tie (72608 x 448: 36 and 64
// slabs; in floats the choice there depends on how the sum is rounded).  Measured
// (us by workgroups per XCD, 4096 x 4096): 32 87, 48 104, 56 92, 64 79; 16384 x 512:
// 16 87, 32 50, 64 49; 1024 x 1024: 16 16, 32 12, 64 15.  (Waves of 32 columns: 312
// against 317 at 8192 x 8192, 169 against 160 at 8192 x 4096; groups of 96 or 128
// columns were slower throughout.)
__host__ __device__ __forceinline__ int fused_cost(int ns, int nchunk, int cgroups, int ncol,
                                                   int n) {
  const int per = fused_per_xcd(ns, cgroups);
  if (ns > 1 && (per > 32 * FU_OCC || ns > nchunk || (long long)ns * ncol > 16LL * n))
    return INT_MAX;
  const int chunks = (nchunk + ns - 1) / ns + 2;
  return (per > 32 ? 34 : 20) * chunks + ns;
}

// The count with the least cost, by a wave (lane: count lane + 1): the DM loop's
// steps choose theirs on the device, from their own j and c0.  Chosen by the host
// from the column reached at the last readback, up to sixteen steps before, the
// last passes over 16384 x 1024 took as long as the first, 84 us.
__device__ __forceinline__ int fused_slabs_wave(int r_lo, int m, int c0, int n) {
  static_assert(FU_MAX_SPLIT == 64, "a lane per count");
  const FuGeom g = fused_geom(r_lo, m, c0, n, 1);
  if (g.cgroups <= 0 || g.nchunk <= 0) return 1;
  const int ns = (local_tid() & 63) + 1;
  int best = fused_cost(ns, g.nchunk, g.cgroups, n - c0, n), arg = ns;  // ties: fewer slabs
  auto take = [&](int ob, int oa) {
    const bool t = ob < best || (ob == best && oa < arg);
    best = t ? ob : best;
    arg = t ? oa : arg;
  };
  take(xor_lane<1>(best), xor_lane<1>(arg));
  take(xor_lane<2>(best), xor_lane<2>(arg));
  take(xor_lane<4>(best), xor_lane<4>(arg));
  take(xor_lane<8>(best), xor_lane<8>(arg));
  take(xor_lane<16>(best), xor_lane<16>(arg));
  take(xor_lane<32>(best), xor_lane<32>(arg));
  return __builtin_amdgcn_readfirstlane(arg);
}

// A 32 x 64 chunk of V in LDS as 16-byte units of two rows: unit (row pair
// rp, column c) at [c][rp ^ (c % 16)].  The 16 lanes that share a column and
// the 16 that share a row pair both read 16 different units of a 256-byte
// line: no bank conflicts in either product.
typedef double2 FuChunk[KMAX][FU_CH / 2];

// The step's T^-1 (ws_mat WS_S) and tau from k_v2's partial V^T V, after a
// Gram-based panel: eight entries of the upper triangle at a time per
// workgroup, the slabs over 32 threads each; every workgroup of the launch
// takes its share.
__device__ __forceinline__ void sum_gram(const DevState* st, int m) {
  __shared__ double part[FU_NWG][8];
  if (!st->fast || (st->flags & 2)) return;
  DevState* ws = const_cast<DevState*>(st);  // the workspace's head
  const double* __restrict__ p = ws_slots(ws);
  const int j = st->j, k = st->fjb_cmp, nslab = (m - j + PR_ROWS - 1) / PR_ROWS;
  const int tid = local_tid(), el = tid & 7, sl = tid >> 3;
  for (int b = blockIdx.x; b < 288; b += gridDim.x) {
    // unit b: eight rows of one column on or above the diagonal; the columns
    // 8 q .. 8 q + 7 have q + 1 units each
    int q = 0;
    while (b >= 4 * (q + 1) * (q + 2)) q++;
    const int u = b - 4 * q * (q + 1);
    const int r = 8 * (u % (q + 1)) + el, c = 8 * q + u / (q + 1), e = r + KMAX * c;
    double s = 0.0;
    for (int q0 = sl; q0 < nslab; q0 += 128) {
      double v[4];
#pragma unroll
      for (int q = 0; q < 4; q++)
        v[q] = p[(size_t)(q0 + 32 * q < nslab ? q0 + 32 * q : sl) * KMAX * KMAX + e];
#pragma unroll
      for (int q = 0; q < 4; q++) s += q0 + 32 * q < nslab ? v[q] : 0.0;
    }
    s += __shfl_xor(s, 8, 64);
    s += __shfl_xor(s, 16, 64);
    s += __shfl_xor(s, 32, 64);
    if ((tid & 63) < 8) part[tid >> 6][el] = s;
    lds_barrier();
    if (tid < 8) {
      const double x = (part[0][el] + part[1][el]) + (part[2][el] + part[3][el]);
      const bool diag = r == c && c < k;
      const double t = !diag ? 0.0 : (st->given_k ? st->tau_base[j + r] : 2.0 / x);
      ws_mat(ws, WS_S)[e] = c < k && r < c ? x : t;
      if (diag && !st->given_k) st->tau_base[j + r] = t;
    }
    lds_barrier();
  }
}

// One pass.  APPLY: C -= Vp Wprev (Vp, Wprev of the previous step) before
// the products; ACCUM: Wp[slab] = Vn^T C.  Rows [r_lo, m) of columns
// [c0, n) are written (APPLY only).
//
// What bounds it: the FP64 matrix cores (64 cycles per 16 x 16 x 4 product, 256
// flops per 16 bytes of C with 64 columns of V), if loads, LDS and barriers
// stay out of their way.  A wave owns 16 columns and a chunk of 32 rows is two
// 16-row tiles, even rows and odd rows: a lane's two consecutive rows are one
// 16-byte element of C and one 16-byte unit of V, so one LDS read feeds two
// products and independent accumulators keep the cores busy.  The tile
// of C in the output layout of product 1 is the B operand of product 2.  The
// next chunk of V goes from memory straight to the other LDS buffer and the
// next chunk of C to registers while this one is multiplied (64 products per
// wave and barrier), so nothing waits for a load issued in the same chunk.
// Measured: the first pass at 8192 x 8192 325 us, 52 TF/s of products, the matrix
// cores busy in 75 % of the cycles, 62 % over all passes (117 us on average); per 8192
// x 8192 factorisation 15.1 ms, against 18.2 with 16-row chunks, V stored to LDS
// through registers and a barrier every 32 products, 16384 x 1024 0.85 against 1.64.
// Odd leading dimensions run here too (3001 x 1777 DM 6.53 -> 6.06 ms against the
// three-kernel form with 8-byte loads).
//
// V^T C is summed in pieces of two chunks: the error of one running sum grows with
// its rows, and how many row slabs there are follows from the chip, not from that
// (2 to 4 for 8192 columns and more, 2048 rows and more in one sum).  Relative error
// of an update, pieces of 64 rows / slabs in one sum: Q C with C
// 8192 x 8192, 256 reflectors 2.0e-16 / 6.6e-16, unpivoted QR 4096 x 8192 2.7e-16 /
// 9.7e-16, DM 8192 x 8192 3.4e-16 / 1.3e-15; a pass takes as long with as without.
//
// V is zero above its panel (within 64 rows) and past m, which the callers
// keep so: no masks in the products, only the stores look at r_lo and m.  W is
// indexed by absolute columns; the partials, ns slabs, by the columns from c0 on (a
// narrow C leaves room for more slabs).  With st (the DM loop) r_lo, c0, ns and the
// buffers come from st; surplus workgroups of the grid return.
//
// On the way, beside the first loads, the workgroups sum V^T V of a Gram-based
// panel from k_v2's slabs (fixed order) into the step's T^-1, and tau_i =
// 2 / S_ii from it: the pass needs neither, its end needs both, and a launch of
// their own with the inverse took 14 us a step.  (The reconstruction's own tau
// and T agree with these only to about eps times the square of the panel's
// condition number; the block reflector has to be orthogonal for the V stored.)
template <bool APPLY, bool ACCUM>
__global__ __launch_bounds__(64 * FU_NWG, FU_OCC) void k_fused(double* A, int lda, int r_lo, int m,
                                                               int c0, int n, StepBufs bufs,
                                                               double* Wp, int ns, int cur,
                                                               const DevState* st) {
  // the chunks of V_s and V_{s+1}, two buffers each (arrays of their own, so
  // that a load on its way into one does not hold up reads of the other)
  __shared__ FuChunk vp0, vp1, vn0, vn1;
  if (st) {
    const int stopped = st->done | st->halt, given = st->given_k, j = st->j, sc0 = st->c0,
              it = st->it;
    asm volatile("" ::"s"(stopped), "s"(given), "s"(j), "s"(sc0), "s"(it));  // one round trip
    if (stopped) return;
    if (!given) {
      r_lo = j;
      c0 = sc0;
      cur = it & 1;
      ns = fused_slabs_wave(r_lo, m, c0, n);
    }
  }
  const int ldw = n - c0;
  const int ldv = bufs.ldv;
  const double* Vn = bufs.V + (size_t)cur * bufs.vstride;
  const double* Vp = bufs.V + (size_t)(cur ^ 1) * bufs.vstride;
  const double* Wprev = bufs.W + (size_t)(cur ^ 1) * bufs.wstride;
  const FuGeom G = fused_geom(r_lo, m, c0, n, ns);
  const int per = fused_per_xcd(ns, G.cgroups);
  const int xcd = blockIdx.x & 7, kx = blockIdx.x >> 3;
  const int pair = xcd * per + kx;
  const int slab = G.cgroups > 0 ? pair / G.cgroups : ns, cgrp = pair - slab * G.cgroups;
  const bool active = kx < per && slab < ns;
  if (!active) {
    if (ACCUM && st) sum_gram(st, m);
    return;
  }
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, li = lane & 15;
  const int ncol = n - c0;
  const int cbw = cgrp * FU_GC + wave * 16;  // this wave's columns (relative to c0)
  const int ch0 = slab * G.slab_ch;
  const int ch1 = min(ch0 + G.slab_ch, G.nchunk);
  // the lane's column c0 + cbw + li (past ncol: a valid column, never stored)
  const bool cok = cbw + li < ncol, won = cbw < ncol;  // (won: some lane's)
  double* Cc = A + (size_t)(c0 + min(cbw + li, ncol - 1)) * lda;
  // the previous step's W tile, negated: wr[s] = -W(4s + g, column li) (lane
  // group g takes the k index 4s + g of step s of product 1)
  // (every load unconditional and in flight together: a load under a condition,
  // negated at once, waited for memory sixteen times in a row, about 10 us)
  double wr[16];
  if (APPLY) {
    const double* wc = Wprev + (size_t)(c0 + min(cbw + li, ncol - 1)) * KMAX + g;
#pragma unroll
    for (int s = 0; s < 16; s++) wr[s] = wc[4 * s];
#pragma unroll
    for (int s = 0; s < 16; s++) wr[s] = cok ? -wr[s] : 0.0;
  }
  dbl4 acc[4], tot[4];  // V^T C of two chunks, of the slab
#pragma unroll
  for (int t = 0; t < 4; t++) acc[t] = tot[t] = (dbl4){0.0, 0.0, 0.0, 0.0};
  // chunk c of V into LDS: a wave takes the columns 16 w .. 16 w + 15, four
  // per load (lane: column lane / 16, unit lane % 16): the lane's byte offsets
  // from the load's first column
  unsigned voff[4];
#pragma unroll
  for (int i = 0; i < 4; i++)
    voff[i] = 8u * ((unsigned)g * (unsigned)ldv + 2u * (unsigned)(li ^ (4 * i + g)));
  auto load_v = [&](const double* V, FuChunk& S, int c) {
    const double* col = V + (size_t)(16 * wave) * ldv + G.base + FU_CH * c;
#pragma unroll
    for (int i = 0; i < 4; i++)
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) void*)(
              reinterpret_cast<const char*>(col + (size_t)(4 * i) * ldv) + voff[i]),
          (__attribute__((address_space(3))) void*)&S[16 * wave + 4 * i][0], 16, 0, 0);
  };
  // chunk c of C as it lies in memory: rows base + 32c + 8v + 2g + (0, 1) in
  // x[v] (taken apart into the tiles where they are used: a move here would
  // wait for the load)
  auto load_c = [&](int c, fu_pair (&x)[4]) {
    const int r0 = G.base + FU_CH * c;
    if (r0 + FU_CH <= m) {
#pragma unroll
      for (int v = 0; v < 4; v++)
        x[v] = *reinterpret_cast<const fu_pair*>(Cc + r0 + 8 * v + 2 * g);
    } else {
#pragma unroll
      for (int v = 0; v < 4; v++)
#pragma unroll
        for (int h = 0; h < 2; h++) x[v][h] = Cc[min(r0 + 8 * v + 2 * g + h, m - 1)];
    }
  };
  // One chunk: the next one's loads, product 1 and the store of its rows,
  // product 2.  Tile h of C: rows 8v + 2g + h in cc[h][v].
  auto step = [&](int c, FuChunk& sp, FuChunk& sn, FuChunk& np, FuChunk& nn, fu_pair (&x)[4]) {
    dbl4 cc[2], cx[2];
#pragma unroll
    for (int v = 0; v < 4; v++)
#pragma unroll
      for (int h = 0; h < 2; h++) {
        cx[h][v] = x[v][h];
        cc[h][v] = APPLY ? 0.0 : x[v][h];
      }
    if (c + 1 < ch1) {
      if (APPLY) load_v(Vp, np, c + 1);
      if (ACCUM) load_v(Vn, nn, c + 1);
      load_c(c + 1, x);
    }
    __builtin_amdgcn_sched_barrier(0);  // the loads are issued before the stores
    // the products first: of the two waves on a SIMD one multiplies while the other
    // is between chunks (8192 x 8192: 117 -> 113 us a pass)
    __builtin_amdgcn_s_setprio(1);
    bool four = false;  // the wave's last four memory operations are its stores
    if (APPLY) {
#pragma unroll
      for (int s = 0; s < 16; s++) {
        const double2 a = sp[4 * s + g][li ^ (4 * (s & 3) + g)];
        cc[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x, wr[s], cc[0], 0, 0, 0);
        cc[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a.y, wr[s], cc[1], 0, 0, 0);
      }
      cc[0] += cx[0];
      cc[1] += cx[1];
      const int r0 = G.base + FU_CH * c;
      if (r0 >= r_lo && r0 + FU_CH <= m) {
        four = won;
        if (cok) {
#pragma unroll
          for (int v = 0; v < 4; v++)
            *reinterpret_cast<fu_pair*>(Cc + r0 + 8 * v + 2 * g) = (fu_pair){cc[0][v], cc[1][v]};
        }
      } else if (cok) {
#pragma unroll
        for (int v = 0; v < 4; v++)
#pragma unroll
          for (int h = 0; h < 2; h++) {
            const int r = r0 + 8 * v + 2 * g + h;
            if (r >= r_lo && r < m) Cc[r] = cc[h][v];
          }
      }
    }
    if (ACCUM) {
#pragma unroll
      for (int v = 0; v < 4; v++) {
        double2 a[4];
#pragma unroll
        for (int t = 0; t < 4; t++) a[t] = sn[16 * t + li][(g + 4 * v) ^ li];
#pragma unroll
        for (int t = 0; t < 4; t++)
          acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[t].x, cc[0][v], acc[t], 0, 0, 0);
#pragma unroll
        for (int t = 0; t < 4; t++)
          acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[t].y, cc[1][v], acc[t], 0, 0, 0);
      }
    }
    // the next chunk of V is in LDS once every wave's loads have arrived; the
    // stores behind them (vector memory operations complete in order) may still
    // be on their way
    __builtin_amdgcn_s_setprio(0);
    if (four) __builtin_amdgcn_s_waitcnt(0x0F74);  // vmcnt(4)
    else __builtin_amdgcn_s_waitcnt(0x0F70);       // vmcnt(0)
    lds_barrier();
  };
  fu_pair x[4];
  if (ch1 > ch0) {
    if (APPLY) load_v(Vp, vp0, ch0);
    if (ACCUM) load_v(Vn, vn0, ch0);
    load_c(ch0, x);
  }
  if (ACCUM && st) sum_gram(st, m);
  __syncthreads();
#pragma clang loop unroll(disable)
  for (int c = ch0; c < ch1; c += 2) {
    step(c, vp0, vn0, vp1, vn1, x);
    if (c + 1 < ch1) step(c + 1, vp1, vn1, vp0, vn0, x);
    if (ACCUM) {
#pragma unroll
      for (int t = 0; t < 4; t++) {
        tot[t] += acc[t];
        acc[t] = (dbl4){0.0, 0.0, 0.0, 0.0};
      }
    }
  }
  if (!ACCUM || !cok) return;
  // partial tile: row 16t + g + 4w of the lane's column
  double* out = Wp + (size_t)slab * KMAX * ldw + (cbw + li);
#pragma unroll
  for (int t = 0; t < 4; t++)
#pragma unroll
    for (int w = 0; w < 4; w++) out[(size_t)(16 * t + g + 4 * w) * ldw] = tot[t][w];
}

int fused_slabs(int r_lo, int m, int c0, int n) {
  const FuGeom g = fused_geom(r_lo, m, c0, n, 1);
  if (g.cgroups <= 0 || g.nchunk <= 0) return 1;
  int best = 1;
  for (int ns = 2; ns <= FU_MAX_SPLIT; ns++)
    if (fused_cost(ns, g.nchunk, g.cgroups, n - c0, n) <
        fused_cost(best, g.nchunk, g.cgroups, n - c0, n))
      best = ns;
  return best;
}

void launch_fused(double* A, int lda, int r_lo, int m, int c0, int n, const StepBufs& bufs,
                  double* Wp, int ns, int apply, int accum, int cur, hipStream_t s,
                  const DevState* st) {
  if (n - c0 <= 0 || m - r_lo <= 0 || !(apply || accum)) return;
  const FuGeom g = fused_geom(r_lo, m, c0, n, ns);
  // with st the device chooses the slabs, at most one round (or a pair per chunk)
  int per = fused_per_xcd(ns, g.cgroups);
  if (st) {
    const long long most = ((long long)g.nchunk * g.cgroups + 7) / 8;
    per = std::max(per, (int)std::min(most, (long long)std::max(32 * FU_OCC, (g.cgroups + 7) / 8)));
  }
  const dim3 grid(8 * per), block(64 * FU_NWG);
  if (apply && accum)
    hipLaunchKernelGGL((k_fused<true, true>), grid, block, 0, s, A, lda, r_lo, m, c0, n, bufs, Wp,
                       ns, cur, st);
  else if (accum)
    hipLaunchKernelGGL((k_fused<false, true>), grid, block, 0, s, A, lda, r_lo, m, c0, n, bufs,
                       Wp, ns, cur, st);
  else
    hipLaunchKernelGGL((k_fused<true, false>), grid, block, 0, s, A, lda, r_lo, m, c0, n, bufs,
                       Wp, ns, cur, st);
}

// ---------------------------------------------------------------------------
// The end of a fused step, one 16-column tile of [j + kk, n) per workgroup
// (256 threads): W = T^T sum_slab Wp (the fused pass's partials, summed in
// slab order; zero for the columns below c0, which the column-by-column panel
// already updated), the step's R12 rows R12 = C_top - V_top W (rows j..j+kk,
// final, written), then the norm downdate of src/dgeqrdm_work.c:80-109 from
// them: s = sum of the kk squares (as the reference's loop, :84-86), temp =
// max(0, (1 + t)(1 - t)) with t = sqrt(|s|) / work, temp2 = temp (work /
// workold)^2; temp2 <= tol3z recomputes the norm from the rows below -- such a
// column receives the whole update now (rows j + kk .. m, C -= V W on the
// matrix cores) and its W column is zero, so the next fused pass leaves it --
// otherwise work *= sqrt(temp).  The running max into st (maxnrm).  W goes to
// the step's W buffer.
//
// Latency bounds it: one round of loads, then a chain of products.  Tiles of
// 16 columns instead of 64 give every CU a workgroup from 4096 columns on and
// a quarter of the loads in flight per thread; T is not formed: T^-T W = P is
// solved by blocks of 16 rows with the inverses of T^-1's diagonal blocks, 40
// products of one wave, whose output layout is the next one's operand layout.
constexpr int WN_TC = 16;

// S1 (64 x 16): P in, W out; U = T^-1 and D the inverses of U's 16 x 16 diagonal
// blocks; one wave.  TRANS: U^T W = P, W_i = D_i^T (P_i - sum_{k < i} U_ki^T W_k);
// otherwise U W = P, W_i = D_i (P_i - sum_{k > i} U_ik W_k).
template <bool TRANS>
__device__ __forceinline__ void wy_solve(const double (*Us)[LDP], const double (*Di)[LDP],
                                         double (*S1)[WN_TC + 1]) {
  const int lane = local_tid() & 63, g = lane >> 4, li = lane & 15;
  dbl4 w[4];  // w[i][v]: row 16 i + g + 4 v
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const int i = TRANS ? q : 3 - q;
    dbl4 p;
#pragma unroll
    for (int v = 0; v < 4; v++) p[v] = S1[16 * i + g + 4 * v][li];
#pragma unroll
    for (int h = 0; h < q; h++) {
      const int k = TRANS ? h : 3 - h;
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const double u = TRANS ? Us[16 * k + g + 4 * v][16 * i + li]
                               : Us[16 * i + li][16 * k + g + 4 * v];
        p = __builtin_amdgcn_mfma_f64_16x16x4f64(-u, w[k][v], p, 0, 0, 0);
      }
    }
    w[i] = (dbl4){0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const int r = g + 4 * v;
      const double d = TRANS ? (r <= li ? Di[16 * i + r][16 * i + li] : 0.0)
                             : (li <= r ? Di[16 * i + li][16 * i + r] : 0.0);
      w[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(d, p[v], w[i], 0, 0, 0);
    }
  }
#pragma unroll
  for (int i = 0; i < 4; i++)
#pragma unroll
    for (int v = 0; v < 4; v++) S1[16 * i + g + 4 * v][li] = w[i][v];
}

__global__ __launch_bounds__(256) void k_wsum_norm(double* A, int lda, int m, int n,
                                                   const double* __restrict__ Wp,
                                                   StepBufs bufs, double* work, double* workold,
                                                   DevState* st, double tol3z) {
  __shared__ double Us[KMAX][LDP];             // T^-1
  __shared__ double Di[KMAX][LDP];             // the inverses of its diagonal blocks
  __shared__ double S1[KMAX][WN_TC + 1];       // the partials' sum, then W
  __shared__ double s_rd[KMAX];
  __shared__ double s_ss[4][WN_TC];
  __shared__ double s_wk[WN_TC], s_wo[WN_TC];  // work, workold of the tile's columns
  __shared__ unsigned long long s_rows[4];
  __shared__ int s_rec[WN_TC];
  const int j = st->j, kk = st->fjb_cmp, c0 = st->c0, it = st->it;
  const int stopped = st->done | st->halt;
  asm volatile("" ::"s"(j), "s"(kk), "s"(c0), "s"(it), "s"(stopped));  // one round trip
  if (stopped) return;
  // the step's end is pending from here on (run by the next k_topk or k_step_end)
  if (blockIdx.x == 0 && threadIdx.x == 0) st->pend = 1;
  const int jn = j + kk;
  const int cb = jn + blockIdx.x * WN_TC;
  if (cb >= n) return;
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, li = lane & 15;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const double* V = bufs.V + (size_t)(it & 1) * bufs.vstride;
  double* W = bufs.W + (size_t)(it & 1) * bufs.wstride;
  const int ldv = bufs.ldv, ldw = n - c0, ns = fused_slabs_wave(j, m, c0, n);
  const int col = cb + li, cl = min(col, n - 1);  // the lane's column
  // every global read of the prologue in flight together: T^-1, the first
  // slabs' partials (thread: column li, rows i0 + 16 q), V's and C's top rows
  double us[KMAX * KMAX / 256];
#pragma unroll
  for (int q = 0; q < KMAX * KMAX / 256; q++) us[q] = ws_mat(st, WS_S)[tid + 256 * q];
  const int i0 = tid >> 4;
  const double* wp = Wp + (size_t)i0 * ldw + max(cl - c0, 0);
  constexpr int YB = 8;  // slabs per round
  double pv[YB][4];
  auto load_p = [&](int y0) {
#pragma unroll
    for (int y = 0; y < YB; y++)
#pragma unroll
      for (int q = 0; q < 4; q++)
        pv[y][q] = wp[((size_t)min(y0 + y, ns - 1) * KMAX + 16 * q) * ldw];
  };
  load_p(0);
  // V(j + 16 wv + li, 4t + g): product operand; C's rows 16 wv + g + 4v
  double va[KMAX / 4];
  const int rt = 16 * wv + li;
#pragma unroll
  for (int t = 0; t < KMAX / 4; t++) va[t] = V[(size_t)(4 * t + g) * ldv + min(j + rt, ldv - 1)];
  dbl4 r12;
#pragma unroll
  for (int v = 0; v < 4; v++) {
    const int r = 16 * wv + g + 4 * v;
    r12[v] = r < kk ? A[(size_t)cl * lda + j + r] : 0.0;
  }
  if (tid < WN_TC) {
    s_wk[tid] = cb + tid < n ? work[cb + tid] : 0.0;
    s_wo[tid] = cb + tid < n ? workold[cb + tid] : 1.0;
    s_rec[tid] = 0;
  }
#pragma unroll
  for (int q = 0; q < KMAX * KMAX / 256; q++) {
    const int e = tid + 256 * q, r = e & 63, c = e >> 6;
    Us[r][c] = us[q];
    if (r == c) s_rd[r] = us[q];
  }
  lds_barrier();
#pragma unroll
  for (int t = 0; t < KMAX / 4; t++) va[t] = rt < kk ? va[t] : 0.0;
  // one wave inverts the diagonal blocks while the others wait for their loads
  if (wv == 3) diag_inverse(Us, s_rd, Di);
  {
    double sum[4] = {0.0, 0.0, 0.0, 0.0};
    for (int y0 = 0; y0 < ns; y0 += YB) {
#pragma unroll
      for (int y = 0; y < YB; y++)
#pragma unroll
        for (int q = 0; q < 4; q++) sum[q] += y0 + y < ns ? pv[y][q] : 0.0;
      if (y0 + YB < ns) load_p(y0 + YB);
    }
    const int c = tid & 15;
    const bool in = cb + c >= c0 && cb + c < n;
#pragma unroll
    for (int q = 0; q < 4; q++) S1[i0 + 16 * q][c] = in ? sum[q] : 0.0;
  }
  lds_barrier();
  if (wv == 0) wy_solve<true>(Us, Di, S1);
  lds_barrier();
  dbl4 vw = (dbl4){0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int t = 0; t < KMAX / 4; t++)
    vw = __builtin_amdgcn_mfma_f64_16x16x4f64(va[t], S1[4 * t + g][li], vw, 0, 0, 0);
  r12 -= vw;
  double sq = 0.0;
#pragma unroll
  for (int v = 0; v < 4; v++) {
    const int r = 16 * wv + g + 4 * v;
    if (r < kk && col < n) A[(size_t)col * lda + j + r] = r12[v];
    sq = r < kk ? fma(r12[v], r12[v], sq) : sq;
  }
  // norm downdate: the sum of squares of column c's kk R12 entries, four
  // waves' parts added in a fixed order
  sq += __shfl_xor(sq, 16, 64);
  sq += __shfl_xor(sq, 32, 64);
  if (g == 0) s_ss[wv][li] = sq;
  lds_barrier();
  double mx = 0.0;
  if (tid < WN_TC) {
    const int c = tid;
    const double wk = s_wk[c];
    if (cb + c < n && wk != 0.0) {
      const double s2 = (s_ss[0][c] + s_ss[1][c]) + (s_ss[2][c] + s_ss[3][c]);
      double temp = sqrt(fabs(s2)) / wk;
      const double d2 = (temp + 1.0) * (1.0 - temp);
      temp = (0.0 >= d2) ? 0.0 : d2;
      const double d1 = wk / s_wo[c];
      const double temp2 = temp * (d1 * d1);
      if (temp2 <= tol3z) {
        s_rec[c] = 1;
      } else {
        const double nw = wk * sqrt(temp);
        s_wk[c] = nw;
        if (nw == nw) mx = nw;
      }
    }
  }
  lds_barrier();
  const bool rec = s_rec[li] != 0;
  unsigned long long rows = 0;
  if (__any(rec)) {
    // the recomputed columns take the update on rows [jn, m) now.  Each wave
    // runs its own 16-row blocks (rows jn + 16 wv, then every 64th): D =
    // V_blk W on the matrix cores, V read straight into the A operand, W from
    // LDS, no workgroup barrier inside the loop.  Lane (g, li) keeps the sum
    // of squares of its column over its rows g + 4 v of each block.
    double ps = 0.0;
    for (int rb = jn + 16 * wv; rb < m; rb += 4 * 16) {
      const int ra = rb + li;  // the lane's row of the A operand
      double vb[KMAX / 4];
#pragma unroll
      for (int t = 0; t < KMAX / 4; t++)
        vb[t] = V[(size_t)(4 * t + g) * ldv + min(ra, m - 1)];  // V(ra, 4t + g)
      dbl4 x, d = (dbl4){0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const int r = rb + g + 4 * v;
        x[v] = A[(size_t)cl * lda + min(r, m - 1)];
      }
#pragma unroll
      for (int t = 0; t < KMAX / 4; t++)
        d = __builtin_amdgcn_mfma_f64_16x16x4f64(vb[t], S1[4 * t + g][li], d, 0, 0, 0);
      x -= d;
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const int r = rb + g + 4 * v;
        if (rec && r < m) {
          A[(size_t)cl * lda + r] = x[v];
          ps = fma(x[v], x[v], ps);
        }
      }
    }
    ps += __shfl_xor(ps, 16, 64);
    ps += __shfl_xor(ps, 32, 64);
    lds_barrier();  // the downdate's sums are read
    if (g == 0) s_ss[wv][li] = ps;
    // the columns' updated rows, for a norm taken again below
    __syncthreads();
    // norms of the recomputed columns (the scaled form where the plain sum
    // of squares leaves the safe range, as dnrm2's scaling does)
    const int mrem = m - jn;
    for (int q = 0; q < WN_TC / 4; q++) {
      const int c = (WN_TC / 4) * wv + q;
      if (!s_rec[c] || cb + c >= n) continue;
      const double s2 = (s_ss[0][c] + s_ss[1][c]) + (s_ss[2][c] + s_ss[3][c]);
      double nr;
      if (mrem <= 0) nr = 0.0;
      else if (s2 >= 1e-280 && s2 <= 1e280) nr = sqrt(s2);
      else nr = wave_nrm2(A + (size_t)(cb + c) * lda + jn, mrem);
      if (lane == 0) {
        s_wk[c] = nr;
        workold[cb + c] = nr;
      }
      if (nr == nr) mx = fmax(mx, nr);
      rows += (unsigned long long)(mrem > 0 ? mrem : 0);
    }
  }
  lds_barrier();
  // the tile's norms, and its W (zero for the recomputed columns), column-major
  if (tid < WN_TC && cb + tid < n) work[cb + tid] = s_wk[tid];
#pragma unroll
  for (int q = 0; q < WN_TC / 4; q++) {
    const int c = wv + 4 * q;
    if (cb + c < n) W[(size_t)(cb + c) * KMAX + lane] = s_rec[c] ? 0.0 : S1[lane][c];
  }
  if (lane == 0) s_rows[wv] = rows;
  // (a lane of wave 0 holds its own column's norm: the wave's maximum goes in)
  block_max_atomic(wave_max(mx), 0, st);
  if (tid == 0) {
    const unsigned long long r = s_rows[0] + s_rows[1] + s_rows[2] + s_rows[3];
    if (r) atomicAdd(&st->recomp_rows, r);
  }
}

void launch_wsum_norm(double* A, int lda, int j0, int m, int n, const double* T,
                      const double* Wp, int ns, const StepBufs& bufs, double* work,
                      double* workold, DevState* st, double tol3z, hipStream_t s) {
  // (T, ns: what the three-kernel update's W takes; here T^-1 lies behind the state
  // (ws_mat WS_S) and the slabs are as the pass chose them)
  (void)T;
  (void)ns;
  // tiles of [j + kk, n), j + kk >= j0 + 1; one workgroup at least (it marks
  // the step's end pending).
  int tiles = (n - j0 - 1 + WN_TC - 1) / WN_TC;
  if (tiles < 1) tiles = 1;
  hipLaunchKernelGGL(k_wsum_norm, dim3(tiles), dim3(256), 0, s, A, lda, m, n, Wp,
                     bufs, work, workold, st, tol3z);
}

// W = op(T) sum_slab Wp from a merged pass, without the norm downdate: ormqr's
// blocks (GIVEN: from T^-1 behind st, as above) and the blocks of the unpivoted
// QR and of the wide steps (from T).  One 16-column tile per workgroup, latency
// bound as the step's end; W by absolute column.  With GIVEN the workgroups past the
// tiles prepare the next block, which none of this needs (4096 x 2048: 9.7 us a block
// against 7.3 and 9.3 in turn; the whole 1.87 -> 1.66 ms).
template <bool GIVEN>
__global__ __launch_bounds__(256) void k_wsum_fused(int c0, int n, const double* __restrict__ T,
                                                    int trans, const double* __restrict__ Wp,
                                                    int ns, double* W, int jnext, int m,
                                                    const DevState* st) {
  __shared__ union {
    struct {
      double Us[KMAX][LDP];  // T^-1, or T
      double Di[KMAX][LDP];
      double S1[KMAX][WN_TC + 1];
      double s_rd[KMAX];
    } w;
    double Gp[4][10][4][64];
  } L;
  const int tiles = (n - c0 + WN_TC - 1) / WN_TC;
  if (GIVEN && (int)blockIdx.x >= tiles) {  // the next block's V and V^T V
    given_panel(jnext, m, blockIdx.x - tiles, const_cast<DevState*>(st), L.Gp);
    return;
  }
  double (*Us)[LDP] = L.w.Us;
  double (*Di)[LDP] = L.w.Di;
  double (*S1)[WN_TC + 1] = L.w.S1;
  double* s_rd = L.w.s_rd;
  const int cb = c0 + blockIdx.x * WN_TC;
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, li = lane & 15;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ldw = n - c0;
  const double* U = GIVEN ? ws_mat(const_cast<DevState*>(st), WS_S) : T;
  double us[KMAX * KMAX / 256];
#pragma unroll
  for (int q = 0; q < KMAX * KMAX / 256; q++) us[q] = U[tid + 256 * q];
  const int i0 = tid >> 4;
  const double* wp = Wp + (size_t)i0 * ldw + min(cb + li, n - 1) - c0;
  constexpr int YB = 8;  // slabs per round
  double pv[YB][4];
  auto load_p = [&](int y0) {
#pragma unroll
    for (int y = 0; y < YB; y++)
#pragma unroll
      for (int q = 0; q < 4; q++)
        pv[y][q] = wp[((size_t)min(y0 + y, ns - 1) * KMAX + 16 * q) * ldw];
  };
  load_p(0);
#pragma unroll
  for (int q = 0; q < KMAX * KMAX / 256; q++) {
    const int e = tid + 256 * q, r = e & 63, c = e >> 6;
    Us[r][c] = us[q];
    if (r == c) s_rd[r] = us[q];
  }
  lds_barrier();
  if (GIVEN && wv == 3) diag_inverse(Us, s_rd, Di);
  {
    double sum[4] = {0.0, 0.0, 0.0, 0.0};
    for (int y0 = 0; y0 < ns; y0 += YB) {
#pragma unroll
      for (int y = 0; y < YB; y++)
#pragma unroll
        for (int q = 0; q < 4; q++) sum[q] += y0 + y < ns ? pv[y][q] : 0.0;
      if (y0 + YB < ns) load_p(y0 + YB);
    }
#pragma unroll
    for (int q = 0; q < 4; q++) S1[i0 + 16 * q][li] = sum[q];
  }
  lds_barrier();
  if (GIVEN) {
    if (wv == 0) {
      if (trans) wy_solve<true>(Us, Di, S1);
      else wy_solve<false>(Us, Di, S1);
    }
  } else {
    // rows 16 wv .. of op(T) S1
    dbl4 w = (dbl4){0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int t = 0; t < KMAX / 4; t++) {
      const int k = 4 * t + g, r = 16 * wv + li;
      w = __builtin_amdgcn_mfma_f64_16x16x4f64(trans ? Us[k][r] : Us[r][k], S1[k][li], w, 0, 0, 0);
    }
    lds_barrier();
#pragma unroll
    for (int v = 0; v < 4; v++) S1[16 * wv + g + 4 * v][li] = w[v];
  }
  lds_barrier();
#pragma unroll
  for (int q = 0; q < WN_TC / 4; q++) {
    const int c = wv + 4 * q;
    if (cb + c < n) W[(size_t)(cb + c) * KMAX + lane] = S1[lane][c];
  }
}

void launch_wsum_fused(int c0, int n, const double* T, int trans, const double* Wp, double* W,
                       int ns, int jnext, int m, hipStream_t s, const DevState* st) {
  if (n - c0 <= 0) return;
  const int tiles = (n - c0 + WN_TC - 1) / WN_TC;
  // (the next block's slabs; past the given columns they return at once)
  const int slabs = !T && jnext >= 0 && jnext < m ? (m - jnext + PR_ROWS - 1) / PR_ROWS : 0;
  if (T)
    hipLaunchKernelGGL(k_wsum_fused<false>, dim3(tiles), dim3(256), 0, s, c0, n, T, trans, Wp, ns,
                       W, jnext, m, st);
  else
    hipLaunchKernelGGL(k_wsum_fused<true>, dim3(tiles + slabs), dim3(256), 0, s, c0, n, T, trans,
                       Wp, ns, W, jnext, m, st);
}

// A block reflector on its own: V^T C, W = op(T) V^T C, C -= V W.
void launch_larfb(double* A, int lda, int j, int m, int c0, int n, const double* V, int ldv,
                  const double* T, int trans, double* Wp, double* W, int nsplit, hipStream_t s) {
  (void)nsplit;  // the three-kernel update's slabs: fused_slabs chooses those here
  if (n - c0 <= 0 || m - j <= 0) return;
  const StepBufs bufs{const_cast<double*>(V), 0, ldv, W, 0};
  const int ns = fused_slabs(j, m, c0, n);
  launch_fused(A, lda, j, m, c0, n, bufs, Wp, ns, 0, 1, 0, s, nullptr);
  launch_wsum_fused(c0, n, T, trans, Wp, W, ns, -1, m, s, nullptr);
  launch_fused(A, lda, j, m, c0, n, bufs, Wp, ns, 1, 0, 0, s, nullptr);
}

}  // namespace qrdm
