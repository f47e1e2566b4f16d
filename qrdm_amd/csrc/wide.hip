// wide.hip -- DM steps wider than 64 columns (nb > 64), driven from the host.
//
// The reference accepts any nb > 0 (src/dgeqrdm_work.c:572-574) and takes up
// to k_max = min(nb, m - j, n - j) candidates per step (:703).  The device
// loop of kernels.hip, panel.hip and trailing.hip is built around one
// 64-column tile per step; a call with 64 < nb <= KW runs each step with the
// kernels below and the host walking the step (one synchronisation per
// step):
//   k_topk_wide    the top k_max of the partial norms (value descending,
//                  position ascending, the order of the reference's qsort):
//                  passes over lists of 1024 keys, each keeping its first
//                  k_max keys, until one list holds them all;
//   k_gram_wide    the candidates' Gram over rows j..m on the matrix cores, a
//                  64 x 64 tile pair of a row slab per workgroup, then the
//                  slabs' sum in a fixed order;
//   k_select_wide  the candidate count (> tau * max) and the greedy cosine
//                  acceptance (:354-403), with the cosine of the 64-wide
//                  path: |G(q, t) / norm_q / norm_t| >= delta marks a conflict;
//   k_swap_pairs   the column moves of permute_marked's walk (computed on the
//                  host, src/dgeqrdm_work.c:149-262), with work and jpvt;
// then the column-by-column panel (regpanel.hip), 64 columns at a time, the block
// reflector applied in 64-column chunks of the kept reflectors (the same product
// H_0 .. H_{k-1} as one dlarfb of width k), and the norm downdate over the step's
// fjb_cmp new rows.
#include "qrdm_internal.h"

#include <climits>

namespace qrdm {

constexpr int WT_KEYS = 1024;  // keys per list of a sort pass
constexpr int WT_OWN = 64;     // keys a workgroup places

// One pass over list b, the keys [1024 b, 1024 (b + 1)) of the L input keys
// (key_before's order, then position; index idx_in[g], or g itself when idx_in is
// null; missing keys sort last): its first K keys in order to out[b K ..].  A
// key's place is the number of keys before it, counted against the whole list in
// LDS: 16 workgroups per list, each placing 64 keys with four threads a key, 256
// comparisons a thread.  (A bitonic sort by one workgroup, 55 stages with a
// barrier each, took 26 us a step; this takes 12.)
__global__ __launch_bounds__(256) void k_topk_wide(const double* __restrict__ val_in,
                                                   const int* __restrict__ idx_in, int L,
                                                   double* val_out, int* idx_out, int K) {
  __shared__ double sv[WT_KEYS];
  __shared__ int si[WT_KEYS];
  const int tid = threadIdx.x;
  const int list = blockIdx.x, base = list * WT_KEYS;
#pragma unroll
  for (int u = 0; u < WT_KEYS / 256; u++) {
    const int e = tid + 256 * u, g = base + e;
    const bool in = g < L;
    const double v = val_in[min(g, L - 1)];
    const int i = idx_in ? idx_in[min(g, L - 1)] : g;
    // norms are >= 0; one that overflowed to a NaN counts as 0 (with a NaN among the
    // keys they have no order, and places stay empty)
    sv[e] = !in ? -1.0 : (v == v ? v : 0.0);
    si[e] = in ? i : INT_MAX;
  }
  __syncthreads();
  // thread: key 64 blockIdx.y + lane, against the quarter of the list of its wave
  const int own = WT_OWN * blockIdx.y + (tid & 63), q0 = (tid >> 6) * (WT_KEYS / 4);
  const double v = sv[own];
  const int ix = si[own];
  int before = 0;
#pragma unroll 8
  for (int q = q0; q < q0 + WT_KEYS / 4; q++) {
    const double vq = sv[q];
    const int iq = si[q];
    // key_before, then position (bitwise: no branch per comparison)
    before += (int)(vq > v) | ((int)(vq == v) & ((int)(iq < ix) | ((int)(iq == ix) & (int)(q < own))));
  }
  __shared__ int cnt[4][64];
  cnt[tid >> 6][tid & 63] = before;
  __syncthreads();
  if (tid < 64) {
    const int at = (cnt[0][tid] + cnt[1][tid]) + (cnt[2][tid] + cnt[3][tid]);
    if (at < K) {
      val_out[(size_t)list * K + at] = v;
      idx_out[(size_t)list * K + at] = ix;
    }
  }
}

// Row slabs of the candidate Gram: as many 64-row blocks as the scratch behind G
// (768 x ldg values) holds partial tiles for, at most about two workgroups per CU.
struct GwGeom {
  int pairs, ns, rows;
};
static GwGeom gram_wide_geom(int rows, int nc, int ldg) {
  const int nt = (nc + 63) / 64;
  GwGeom g;
  g.pairs = nt * (nt + 1) / 2;
  int ns = (rows + 63) / 64;
  const int room = (int)((long long)768 * ldg / (4096 * g.pairs));
  if (ns > room) ns = room;
  if (ns > 512 / g.pairs) ns = 512 / g.pairs;
  if (ns < 1) ns = 1;
  g.rows = ((rows + ns - 1) / ns + 63) / 64 * 64;
  g.ns = (rows + g.rows - 1) / g.rows;
  if (g.ns < 1) g.ns = 1;
  return g;
}
__device__ __forceinline__ void gram_wide_tile(int t, int nt, int& ti, int& tj) {
  ti = 0;
  while (t >= nt - ti) {
    t -= nt - ti;
    ti++;
  }
  tj = ti + t;
}

// G(p, q) = sum_{r = j..m-1} A(r, j + idx[p]) A(r, j + idx[q]) for the 64 x 64
// tile pair (ti <= tj) blockIdx.x, rows of slab blockIdx.y: the partial tile to
// part (one slab: G itself).  64-row chunks through LDS, the next one's loads in
// flight during the products; wave w accumulates tile rows 16w..16w+15 on the
// matrix cores.  Latency bounds it (a slab is a few chunks): one workgroup per
// tile pair walking all rows left three CUs working, 400 us a step at 2048 rows
// and 128 candidates, against 9 with the slabs and 3 for their sum.
__global__ __launch_bounds__(256) void k_gram_wide(const double* __restrict__ A, int lda, int j,
                                                   int m, const int* __restrict__ idx, int nc,
                                                   double* G, int ldg, double* part, int ns,
                                                   int rows) {
  __shared__ double X[64][65];
  __shared__ double Y[64][65];
  int ti, tj;
  gram_wide_tile(blockIdx.x, (nc + 63) / 64, ti, tj);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, g = lane >> 4, li = lane & 15;
  dbl4 acc[4];
#pragma unroll
  for (int cb = 0; cb < 4; cb++) acc[cb] = (dbl4){0.0, 0.0, 0.0, 0.0};
  // thread: row lane of the chunk, columns wave + 4 q
  const double* px[16];
  const double* py[16];
#pragma unroll
  for (int q = 0; q < 16; q++) {
    const int pc = 64 * ti + wave + 4 * q, qc = 64 * tj + wave + 4 * q;
    px[q] = A + (size_t)(j + idx[min(pc, nc - 1)]) * lda;
    py[q] = A + (size_t)(j + idx[min(qc, nc - 1)]) * lda;
  }
  const int rs = j + blockIdx.y * rows, re = min(rs + rows, m);
  double x[16], y[16];
  auto load = [&](int r0) {
    const int r = r0 + lane, rc = min(r, m - 1);
#pragma unroll
    for (int q = 0; q < 16; q++) {
      x[q] = px[q][rc];
      y[q] = py[q][rc];
    }
#pragma unroll
    for (int q = 0; q < 16; q++) {
      x[q] = r < re ? x[q] : 0.0;
      y[q] = r < re ? y[q] : 0.0;
    }
  };
  if (rs < re) load(rs);
  for (int r0 = rs; r0 < re; r0 += 64) {
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 16; q++) {
      X[lane][wave + 4 * q] = x[q];
      Y[lane][wave + 4 * q] = y[q];
    }
    __syncthreads();
    if (r0 + 64 < re) load(r0 + 64);
#pragma unroll 4
    for (int k0 = 0; k0 < 64; k0 += 4) {
      const double a = X[k0 + g][16 * wave + li];
#pragma unroll
      for (int cb = 0; cb < 4; cb++)
        acc[cb] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, Y[k0 + g][16 * cb + li], acc[cb], 0, 0,
                                                       0);
    }
  }
  double* out = part + ((size_t)blockIdx.y * gridDim.x + blockIdx.x) * 4096;
#pragma unroll
  for (int cb = 0; cb < 4; cb++)
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const int r = 16 * wave + g + 4 * v, c = 16 * cb + li;
      const int p = 64 * ti + r, q = 64 * tj + c;
      if (ns > 1) out[r + 64 * c] = acc[cb][v];
      else if (p < nc && q < nc) G[p + (size_t)q * ldg] = acc[cb][v];
    }
}

// The slabs' sum, in slab order, into G: 64 entries (one tile column) per
// workgroup, the slabs over its four waves.
__global__ __launch_bounds__(256) void k_gram_wide_sum(const double* __restrict__ part, int pairs,
                                                       int ns, int nc, double* G, int ldg) {
  __shared__ double sm[4][64];
  int ti, tj;
  gram_wide_tile(blockIdx.x, (nc + 63) / 64, ti, tj);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, c = blockIdx.y;
  const double* p = part + (size_t)blockIdx.x * 4096 + 64 * c + lane;
  double s = 0.0;
  for (int b0 = w; b0 < ns; b0 += 32) {
    double v[8];
#pragma unroll
    for (int u = 0; u < 8; u++)
      v[u] = p[(size_t)(b0 + 4 * u < ns ? b0 + 4 * u : w) * pairs * 4096];
#pragma unroll
    for (int u = 0; u < 8; u++) s += b0 + 4 * u < ns ? v[u] : 0.0;
  }
  sm[w][lane] = s;
  __syncthreads();
  const int r = 64 * ti + lane, q = 64 * tj + c;
  if (w == 0 && r < nc && q < nc)
    G[r + (size_t)q * ldg] = (sm[0][lane] + sm[1][lane]) + (sm[2][lane] + sm[3][lane]);
}

// The step's selection from the sorted candidates (val: their norms, the
// first kmax): out[0] = nc (> tau * val[0], at most kmax), out[1] = fjb,
// out[2 + s] = the candidate rank accepted s-th.  Candidate 0 is always
// accepted; candidate i after it when |cos| < delta against every accepted
// one and fewer than kmax are accepted.  The conflicts as bit words, a wave per
// word (consecutive lanes: consecutive rows of G), then one thread's walk over
// them in LDS (49 us a step with a thread per candidate and the count from
// memory one by one; 13 so).
__global__ __launch_bounds__(1024) void k_select_wide(const double* __restrict__ G, int ldg,
                                                      const double* __restrict__ val, int kmax,
                                                      double tau, double delta, int* out) {
  __shared__ unsigned long long conf[KW][KW / 64];
  __shared__ double r[KW];
  __shared__ int sel[KW];
  __shared__ int s_nc, s_nsel;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  if (t == 0) s_nc = kmax;
  __syncthreads();
  const double lim = tau * val[0];
  if (t < kmax) {
    const double v = val[t];
    r[t] = 1.0 / v;
    if (!(v > lim)) atomicMin(&s_nc, t);  // the first one not above
  }
  __syncthreads();
  const int nc = s_nc, nw = (nc + 63) / 64;
  constexpr int NL = 8;  // words in flight
  for (int e0 = wave; e0 < nc * nw; e0 += 16 * NL) {
    double v[NL];
    int row[NL], word[NL];
#pragma unroll
    for (int u = 0; u < NL; u++) {
      const int e = min(e0 + 16 * u, nc * nw - 1);
      row[u] = e / nw;
      word[u] = e - row[u] * nw;
      v[u] = G[min(64 * word[u] + lane, row[u]) + (size_t)row[u] * ldg];
    }
#pragma unroll
    for (int u = 0; u < NL; u++) {
      const int i = row[u], q = 64 * word[u] + lane;
      // G(q, i), q < i
      const unsigned long long bits =
          __ballot(q < i && fabs(v[u] * r[min(q, KW - 1)] * r[i]) >= delta);
      if (lane == 0) conf[i][word[u]] = bits;
    }
  }
  __syncthreads();
  if (t == 0) {
    unsigned long long acc[KW / 64];
#pragma unroll
    for (int w = 0; w < KW / 64; w++) acc[w] = 0ull;
    acc[0] = 1ull;
    int nsel = 1;
    sel[0] = 0;
    unsigned long long nx[KW / 64];  // the next candidate's words
#pragma unroll
    for (int w = 0; w < KW / 64; w++) nx[w] = conf[1][w];
    for (int i = 1; i < nc; i++) {
      unsigned long long hit = 0ull;
#pragma unroll
      for (int w = 0; w < KW / 64; w++) {
        hit |= (w < nw ? nx[w] : 0ull) & acc[w];
        nx[w] = conf[min(i + 1, KW - 1)][w];
      }
      if (hit == 0ull && nsel < kmax) {
#pragma unroll
        for (int w = 0; w < KW / 64; w++) acc[w] |= w == (i >> 6) ? 1ull << (i & 63) : 0ull;
        sel[nsel] = i;
        nsel++;
      }
    }
    s_nsel = nsel;
  }
  __syncthreads();
  if (t == 0) {
    out[0] = nc;
    out[1] = s_nsel;
  }
  if (t < s_nsel) out[2 + t] = sel[t];
}

// Position swaps (relative to column j), in order: whole columns of A, work
// and jpvt.  SW_BATCH swaps at a time with their loads in flight together where
// no column occurs twice among them (the walk's swaps nearly always), else one
// by one; 64 rows per workgroup.  (One by one throughout, 256 rows per
// workgroup: 44 us a step with 128 swaps of 2048 rows; 22 so.)
constexpr int SW_BATCH = 16;
__global__ __launch_bounds__(64) void k_swap_pairs(double* A, int lda, int m, int j,
                                                   double* work, int* jp,
                                                   const int* __restrict__ pairs, int np) {
  const int lane = threadIdx.x, r = blockIdx.x * 64 + lane;
  const bool own = blockIdx.x == 0;  // work and jpvt too
  // lane 2 p + s: column s of swap p (the next batch's in flight with this one's)
  int nxt = lane < 2 * min(SW_BATCH, np) ? pairs[lane] : 0;
  for (int p0 = 0; p0 < np; p0 += SW_BATCH) {
    const int nb = min(SW_BATCH, np - p0);
    const int col = lane < 2 * nb ? nxt : -1 - lane;
    const int p1 = p0 + SW_BATCH;
    nxt = lane < 2 * min(SW_BATCH, np - p1) ? pairs[2 * p1 + lane] : 0;
    bool twice = false;
#pragma unroll
    for (int d = 1; d < 2 * SW_BATCH; d++)
      twice |= lane < 2 * SW_BATCH && col == __shfl(col, (lane + d) & (2 * SW_BATCH - 1), 64);
    if (!__any(twice)) {
      double a[SW_BATCH], b[SW_BATCH];
      double* pa[SW_BATCH];
      double* pb[SW_BATCH];
#pragma unroll
      for (int p = 0; p < SW_BATCH; p++) {
        const int q = p < nb ? p : 0;
        pa[p] = A + (size_t)(j + __builtin_amdgcn_readlane(col, 2 * q)) * lda + min(r, m - 1);
        pb[p] = A + (size_t)(j + __builtin_amdgcn_readlane(col, 2 * q + 1)) * lda + min(r, m - 1);
        a[p] = *pa[p];
        b[p] = *pb[p];
      }
#pragma unroll
      for (int p = 0; p < SW_BATCH; p++)
        if (p < nb && r < m) {
          *pa[p] = b[p];
          *pb[p] = a[p];
        }
      if (own && lane < 2 * nb) {
        const int other = __shfl(col, lane ^ 1, 64);
        const double w = work[j + other];
        const int q = jp[j + other];
        work[j + col] = w;
        jp[j + col] = q;
      }
      if (own) __threadfence_block();  // the next batch's lanes read them
    } else {
      for (int p = 0; p < nb; p++) {
        const int ca = j + __builtin_amdgcn_readlane(col, 2 * p);
        const int cb = j + __builtin_amdgcn_readlane(col, 2 * p + 1);
        if (r < m) {
          const double x = A[(size_t)ca * lda + r];
          A[(size_t)ca * lda + r] = A[(size_t)cb * lda + r];
          A[(size_t)cb * lda + r] = x;
        }
        if (own && lane == 0) {
          const double w = work[ca];
          work[ca] = work[cb];
          work[cb] = w;
          const int q = jp[ca];
          jp[ca] = jp[cb];
          jp[cb] = q;
        }
      }
    }
  }
}

// The state the host-driven kernels read: the step's column and width, a
// fresh maximum norm.
__global__ void k_wide_state(DevState* st, int j, int kk) {
  st->j = j;
  st->fjb_cmp = kk;
  st->maxnrm_bits = 0ull;
  st->done = 0;
  st->halt = 0;
}

int wide_sort_keys(int n) { return ((n + WT_KEYS - 1) / WT_KEYS) * KW; }

void launch_topk_wide(const double* work, int nsub, int kmax, double* val[2], int* idx[2],
                      const double** out_val, hipStream_t s) {
  const double* vin = work;
  const int* iin = nullptr;
  int L = nsub, b = 0, grid;
  do {
    grid = (L + WT_KEYS - 1) / WT_KEYS;
    hipLaunchKernelGGL(k_topk_wide, dim3(grid, WT_KEYS / WT_OWN), dim3(256), 0, s, vin, iin, L, val[b], idx[b],
                       kmax);
    vin = val[b];
    iin = idx[b];
    L = grid * kmax;
    b ^= 1;
  } while (grid > 1);
  *out_val = vin;
}

const int* wide_topk_idx(double* val[2], int* idx[2], const double* out_val) {
  return out_val == val[0] ? idx[0] : idx[1];
}

void launch_gram_wide(const double* A, int lda, int j, int m, const int* idx, int nc, double* G,
                      int ldg, hipStream_t s) {
  if (nc <= 0) return;
  const GwGeom g = gram_wide_geom(m - j, nc, ldg);
  double* part = G + (size_t)KW * ldg;
  hipLaunchKernelGGL(k_gram_wide, dim3(g.pairs, g.ns), dim3(256), 0, s, A, lda, j, m, idx, nc, G,
                     ldg, part, g.ns, g.rows);
  if (g.ns > 1)
    hipLaunchKernelGGL(k_gram_wide_sum, dim3(g.pairs, 64), dim3(256), 0, s, part, g.pairs, g.ns,
                       nc, G, ldg);
}

void launch_select_wide(const double* G, int ldg, const double* val, int kmax, double tau,
                        double delta, int* out, hipStream_t s) {
  hipLaunchKernelGGL(k_select_wide, dim3(1), dim3(1024), 0, s, G, ldg, val, kmax, tau, delta,
                     out);
}

void launch_swap_pairs(double* A, int lda, int m, int j, double* work, int* jp, const int* pairs,
                       int np, hipStream_t s) {
  if (np <= 0) return;
  hipLaunchKernelGGL(k_swap_pairs, dim3((m + 63) / 64), dim3(64), 0, s, A, lda, m, j, work, jp,
                     pairs, np);
}

void launch_wide_state(DevState* st, int j, int kk, hipStream_t s) {
  hipLaunchKernelGGL(k_wide_state, dim3(1), dim3(1), 0, s, st, j, kk);
}

}  // namespace qrdm
