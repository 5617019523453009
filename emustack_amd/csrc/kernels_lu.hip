// Multifrontal sparse LU of K - shift*M on the GPU, batched over instances
// that share one mesh (replaces UMFPACK umf4znum / umf4zsol, reference
// backend/fortran/valpr_umf_64.f:198 and :340).
//
// Every front is a dense column-major f x f block [S | U] (S = own,
// fully-summed variables, U = update variables).  The numeric phase walks
// the assembly tree level by level (deepest first); within a level all
// fronts of all instances are processed by the same launches:
//   panel  : NB columns of partial-pivoting LU (pivots restricted to S rows)
//   apply  : row interchanges of the other columns, U12 block row <- L11^{-1}
//            U12, update rows of the panel <- U11^{-1}
//   gemm   : trailing update F22 -= L21 U12 (64 x 64 tiles)
//   extend : child Schur complement added into its parent (slot 0, then 1:
//            no two tasks of one launch touch the same parent -> no atomics)
// The factors are then rewritten into an inverted-factor form and the solves
// walk the same tree as dense matrix-vector products: forward elimination
// bottom-up with update vectors passed to the parent (deterministic,
// atomic-free), back substitution top-down.
#include <type_traits>

#include "engine.h"

namespace emu {

constexpr int NB = 32;     // panel width
constexpr int TILE = 64;   // gemm tile
constexpr int EA_COLS = 8; // columns per extend-add task

struct FrontArrays {
  const int32_t *s, *u, *f, *b, *parent;
  const int64_t *off, *uoff, *pivoff, *ioff, *fvoff;
  const int32_t *uidx, *pmap, *cmap;
};

static FrontArrays fa(DevMesh &dm) {
  FrontArrays a;
  a.s = dm.fs.p; a.u = dm.fu.p; a.f = dm.ff.p; a.b = dm.fb.p; a.parent = dm.fparent.p;
  a.off = dm.foff.p; a.uoff = dm.fuoff.p; a.pivoff = dm.fpivoff.p;
  a.ioff = dm.fioff.p; a.fvoff = dm.ffvoff.p;
  a.uidx = dm.uidx.p; a.pmap = dm.pmap.p; a.cmap = dm.cmap.p;
  return a;
}

__global__ void k_fill(zd *__restrict__ p, int64_t n, zd v) {
  int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  int64_t st = (int64_t)gridDim.x * blockDim.x;
  for (; i < n; i += st) p[i] = v;
}

void launch_fill(zd *p, int64_t n, zd v, hipStream_t s) {
  if (n <= 0) return;
  int64_t blocks = std::min<int64_t>((n + 255) / 256, 65536);
  hipLaunchKernelGGL(k_fill, dim3((unsigned)blocks), dim3(256), 0, s, p, n, v);
  EMU_LAUNCH_CHECK();
}

// pool[b][nnz2front[k]] = mat1[b][k]
__global__ void k_scatter_fronts(int64_t nnz, int64_t pool, const int64_t *__restrict__ map,
                                 const zd *__restrict__ mat1, zd *__restrict__ P) {
  int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  int b = blockIdx.y;
  if (k >= nnz) return;
  P[b * pool + map[k]] = mat1[b * nnz + k];
}

// Panel step of any number of rows, the panel in memory: fronts with more
// than 4,096 pivot candidates (k_panel_reg covers the rest).
__global__ __launch_bounds__(256) void k_panel(const int32_t *__restrict__ tasks, int k0,
                                               FrontArrays A, zd *__restrict__ pool, int64_t psz,
                                               int32_t *__restrict__ piv, int64_t npiv,
                                               int32_t *__restrict__ pflag, int32_t *__restrict__ sig,
                                               int4 *__restrict__ gx, double pert) {
  const int t = tasks[blockIdx.x];
  const int b = blockIdx.y;
  const int tid = threadIdx.x;
  const int s = A.s[t], f = A.f[t];
  zd *F = pool + b * psz + A.off[t];
  int32_t *pv = piv + b * npiv + A.pivoff[t];
  int32_t *pf = pflag + b * npiv + A.pivoff[t];
  int32_t *sg = sig + b * npiv + A.pivoff[t];
  const int w = min(NB, s - k0);
  // the rows are exchanged here, in every column: none left to k_panel_apply
  if (tid < w) gx[b * npiv + A.pivoff[t] + k0 + tid] = make_int4(k0 + tid, -1, 0, 0);
  if (k0 == 0) {
    for (int i = tid; i < s; i += 256) sg[i] = i;
    __syncthreads();
  }
  __shared__ double redv[4];
  __shared__ int redi[4];
  __shared__ zd urow[NB];
  const int lane = tid & 63, wave = tid >> 6;
  for (int jj = 0; jj < w; ++jj) {
    const int k = k0 + jj;
    double best = -1.0;
    int bi = k;
    for (int r = k + tid; r < s; r += 256) {
      double a = zabs1(F[r + (int64_t)k * f]);
      if (a > best) { best = a; bi = r; }
    }
    // pivot search: largest |.|_1, smallest row on ties (wave shuffles, then
    // the four waves' winners through LDS: two barriers per column)
#pragma unroll
    for (int m = 32; m > 0; m >>= 1) {
      const double a = __shfl_xor(best, m, 64);
      const int ai = __shfl_xor(bi, m, 64);
      if (a > best || (a == best && ai < bi)) {
        best = a;
        bi = ai;
      }
    }
    if (lane == 0) {
      redv[wave] = best;
      redi[wave] = bi;
    }
    __syncthreads();
    int p = redi[0];
    {
      double pb = redv[0];
      for (int q = 1; q < 4; ++q)
        if (redv[q] > pb || (redv[q] == pb && redi[q] < p)) {
          pb = redv[q];
          p = redi[q];
        }
    }
    if (p != k)
      for (int c = tid; c < f; c += 256) {
        zd a = F[k + (int64_t)c * f];
        F[k + (int64_t)c * f] = F[p + (int64_t)c * f];
        F[p + (int64_t)c * f] = a;
      }
    __syncthreads();
    zd d = F[k + (int64_t)k * f];
    const bool zero = (d.x == 0.0 && d.y == 0.0);
    if (zero) d = zmk(pert, 0.0);
    if (tid == 0) {
      pv[k] = p;
      pf[k] = zero ? 1 : 0;
      if (p != k) {
        const int32_t a = sg[k];
        sg[k] = sg[p];
        sg[p] = a;
      }
      if (zero) F[k + (int64_t)k * f] = d;
    }
    const zd dinv = zdiv(zmk(1.0, 0.0), d);
    const int nrest = w - jj - 1;
    for (int c = tid; c < nrest; c += 256) urow[c] = F[k + (int64_t)(k + 1 + c) * f];
    __syncthreads();
    for (int r = k + 1 + tid; r < s; r += 256) {
      zd l = zmul(F[r + (int64_t)k * f], dinv);
      F[r + (int64_t)k * f] = l;
      // rank-1 update of the row's remaining panel columns, eight at a time
      // (all eight loads in flight before the updates)
      zd *pr = &F[r + (int64_t)(k + 1) * f];
      for (int c0 = 0; c0 < nrest; c0 += 8) {
        zd v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = pr[(int64_t)min(c0 + u, nrest - 1) * f];
#pragma unroll
        for (int u = 0; u < 8; ++u)
          if (c0 + u < nrest) pr[(int64_t)(c0 + u) * f] = zfms(l, urow[c0 + u], v[u]);
      }
    }
    __syncthreads();
  }
}

// Orders a wavefront's own LDS writes before its later reads (no other wave
// takes part).
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

__device__ __forceinline__ double wave_max(double v) {
  // prefix maxima along the four 16-lane rows, then across the rows: lane 63
  // ends with the maximum of the wavefront
#define EMU_DPP_MAX(ctrl, rows)                                                                        \
  {                                                                                                    \
    const int lo = __double2loint(v), hi = __double2hiint(v);                                          \
    v = fmax(v, __hiloint2double(__builtin_amdgcn_update_dpp(hi, hi, ctrl, rows, 0xf, false),          \
                                 __builtin_amdgcn_update_dpp(lo, lo, ctrl, rows, 0xf, false)));        \
  }
  EMU_DPP_MAX(0x111, 0xf)  // row_shr:1
  EMU_DPP_MAX(0x112, 0xf)  // row_shr:2
  EMU_DPP_MAX(0x114, 0xf)  // row_shr:4
  EMU_DPP_MAX(0x118, 0xf)  // row_shr:8
  EMU_DPP_MAX(0x142, 0xa)  // row_bcast:15 into rows 1 and 3
  EMU_DPP_MAX(0x143, 0xc)  // row_bcast:31 into rows 2 and 3
#undef EMU_DPP_MAX
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), 63),
                          __builtin_amdgcn_readlane(__double2loint(v), 63));
}

// 1 / d, Smith's division without its branch: the bits of zdiv(1, d), which the
// update rows and k_panel use.  (One reciprocal of |d|^2 is a shorter chain by
// 1 to 2 % of a panel, but its other rounding decides near ties of the pivot
// search differently, and with them the rounding of the complex64 factor.)
__device__ __forceinline__ zd zrecip(zd d) {
  const bool xl = fabs(d.x) >= fabs(d.y);
  const double p = xl ? d.x : d.y, q = xl ? d.y : d.x;
  const double r = q / p, den = p + q * r;
  const double u = 1.0 / den, v = r / den;
  return xl ? zmk(u, -v) : zmk(v, -u);
}

// Panel step with the panel in registers (up to 64 NW RPT pivot-candidate
// rows).  Thread (lane, wave) owns the rows k0 + tid + 64 NW q and holds CW
// columns of each; the 32-column panel is CW columns at a time.  A column
// step is a serial chain (pivot search, broadcast of the pivot row,
// multipliers, rank-1 update) and latency-bound, so the chain is kept short:
//  * pivoting is implicit: rows stay where they are and each carries the
//    position it would have after the interchanges (pos), so no row data is
//    exchanged; positions settle ties (largest |.|_1, smallest position);
//  * every thread forms the reciprocal of its own candidate while the search
//    runs, each wave reduces its candidates with DPP moves and its winner posts
//    its row and reciprocal to the wave's LDS slot; one barrier (none when
//    NW = 1), then every thread picks the winner among the NW slots.  There are
//    two sets of slots, by the parity of the column in its chunk: a wave that
//    is a step ahead posts to the set that no other wave still reads, and it
//    cannot be two ahead, as that takes the next step's barrier (a chunk ends
//    with barriers of its own);
//  * half a chunk's columns at a time are a ring: a step uses entry 0, writes
//    the updated entry c to c - 1 and the multiplier (or the finished U entry)
//    to the last place, so that register indices are compile-time without
//    unrolling the steps; entries of finished columns meet a zero in the update.
// At the end of a chunk the rows are written to their positions and the
// threads take over the row at their own position (from: its place when the
// panel began).  gx records the net interchange (x: source row of position k;
// y, z: a row outside the panel and its source, y = -1: none) for
// k_panel_apply, which moves the other columns' entries in one gather instead
// of up to 32 dependent swaps.
// Measured, mean per launch (k_panel in brackets): the dense LUs of a 64-point
// 200-mode cascade 44 us (85), the 8,000-triangle mesh with 2 instances 61 us
// (164).
template <int NW, int RPT, int CW>
__global__ __launch_bounds__(64 * NW) void k_panel_reg(const int32_t *__restrict__ tasks, int k0, FrontArrays A,
                                                       zd *__restrict__ pool, int64_t psz, int32_t *__restrict__ piv,
                                                       int64_t npiv, int32_t *__restrict__ pflag,
                                                       int32_t *__restrict__ sig, int4 *__restrict__ gx,
                                                       double pert) {
  constexpr int NT = 64 * NW;
  constexpr int G = CW < 4 ? CW : 4;  // divides CW, so also every c0
  constexpr int HC = CW / 2;
  const int t = tasks[blockIdx.x];
  const int b = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int s = A.s[t], f = A.f[t];
  zd *F = pool + b * psz + A.off[t];
  const int64_t po = b * npiv + A.pivoff[t];
  const int w = min(NB, s - k0);
  // the waves' candidates: row (entry 0 first), reciprocal of entry 0, and a
  // zero for the entries of finished columns
  __shared__ zd slot[2][NW][CW + 2];
  __shared__ double sval[2][NW];
  __shared__ int spos[2][NW];
  __shared__ zd Ush[NB][CW];
  __shared__ int perm[NT * RPT];
  __shared__ int nout, outr[NB], outs[NB];
  __shared__ int2 spiv[NB];  // (position, replaced): global stores would be waited for at every barrier
  int row[RPT], from[RPT], pos[RPT];
#pragma unroll
  for (int q = 0; q < RPT; ++q) row[q] = from[q] = k0 + tid + NT * q;
  if (tid == 0) nout = 0;
  if (tid < NB) {
    outr[tid] = -1;
    outs[tid] = k0;
  }
  if (lane == 0) slot[0][wave][CW + 1] = slot[1][wave][CW + 1] = zmk(0, 0);
  for (int c0 = 0; c0 < w; c0 += CW) {
    const int cw = min(CW, w - c0);
    zd xa[RPT][HC], xb[RPT][HC];
#pragma unroll
    for (int q = 0; q < RPT; ++q) {
      const zd *Fr = F + min(from[q], s - 1) + (int64_t)(k0 + c0) * f;
#pragma unroll
      for (int i = 0; i < HC; ++i) xa[q][i] = Fr[(int64_t)min(i, cw - 1) * f];
#pragma unroll
      for (int i = 0; i < HC; ++i) xb[q][i] = Fr[(int64_t)min(HC + i, cw - 1) * f];
      pos[q] = row[q];
    }
    if (c0 > 0) {
      // the finished columns [0, c0) applied to these: wave 0 solves the
      // rows of the panel's upper triangle in order and posts them, the other
      // rows follow once all are posted (the multipliers are read back)
      if (wave == 0)
        for (int kb = 0; kb < c0; kb += G) {
          zd l[RPT][G];
#pragma unroll
          for (int q = 0; q < RPT; ++q)
#pragma unroll
            for (int u = 0; u < G; ++u) l[q][u] = F[min(row[q], s - 1) + (int64_t)(k0 + kb + u) * f];
#pragma unroll
          for (int u = 0; u < G; ++u) {
            if (lane == kb + u)
#pragma unroll
              for (int i = 0; i < HC; ++i) {
                Ush[kb + u][i] = xa[0][i];
                Ush[kb + u][HC + i] = xb[0][i];
              }
            wave_sync();
#pragma unroll
            for (int q = 0; q < RPT; ++q) {
              const zd lm = row[q] > k0 + kb + u ? l[q][u] : zmk(0, 0);
#pragma unroll
              for (int i = 0; i < HC; ++i) {
                xa[q][i] = zfms(lm, Ush[kb + u][i], xa[q][i]);
                xb[q][i] = zfms(lm, Ush[kb + u][HC + i], xb[q][i]);
              }
            }
          }
        }
      if (NW > 1) {
        __syncthreads();
        if (wave != 0)
#pragma unroll
          for (int q = 0; q < RPT; ++q)
            for (int kb = 0; kb < c0; kb += G) {
              zd l[G];
#pragma unroll
              for (int u = 0; u < G; ++u) l[u] = F[min(row[q], s - 1) + (int64_t)(k0 + kb + u) * f];
#pragma unroll
              for (int u = 0; u < G; ++u)
#pragma unroll
                for (int i = 0; i < HC; ++i) {
                  xa[q][i] = zfms(l[u], Ush[kb + u][i], xa[q][i]);
                  xb[q][i] = zfms(l[u], Ush[kb + u][HC + i], xb[q][i]);
                }
            }
      }
    }
    // one column step: A holds the ring that the column is taken from, B the
    // columns after it that are not in the ring (HB of them, 0 in the second
    // half of the chunk)
    auto steps = [&](auto &A_, auto &B_, auto hb, const int j0) {
      constexpr int HB = decltype(hb)::value;
#pragma unroll 1
      for (int jj = 0; jj < HC; ++jj) {
        if (j0 + jj >= cw) {  // short last chunk: only bring the ring back in order
#pragma unroll
          for (int q = 0; q < RPT; ++q) {
            const zd v = A_[q][0];
#pragma unroll
            for (int i = 1; i < HC; ++i) A_[q][i - 1] = A_[q][i];
            A_[q][HC - 1] = v;
          }
          continue;
        }
        const int k = k0 + c0 + j0 + jj, pb = (j0 + jj) & 1;
        // this wave's largest candidate; NaN counts as the smallest value of a
        // row, absent and finished rows below it
        double best = -2.0, a[RPT];
        zd rec[RPT];
#pragma unroll
        for (int q = 0; q < RPT; ++q) {
          const double v = zabs1(A_[q][0]);
          a[q] = (pos[q] >= k && row[q] < s) ? (v >= 0.0 ? v : -1.0) : -2.0;
          best = fmax(best, a[q]);
          rec[q] = zrecip(v == 0.0 ? zmk(pert, 0.0) : A_[q][0]);
        }
        const double wmax = wave_max(best);
        int wpos = INT32_MAX, wlane = -1, wq = -1;
        if (wmax > -2.0) {
#pragma unroll
          for (int q = 0; q < RPT; ++q)
            for (uint64_t m = __ballot(a[q] == wmax); m; m &= m - 1) {  // one bit but for ties
              const int l = (int)__builtin_ctzll(m), pl = __builtin_amdgcn_readlane(pos[q], l);
              if (pl < wpos) {
                wpos = pl;
                wlane = l;
                wq = q;
              }
            }
        }
#pragma unroll
        for (int q = 0; q < RPT; ++q)
          if (q == wq && lane == wlane) {
#pragma unroll
            for (int i = 0; i < HC; ++i) slot[pb][wave][i] = A_[q][i];
#pragma unroll
            for (int i = 0; i < HB; ++i) slot[pb][wave][HC + i] = B_[q][i];
            slot[pb][wave][CW] = rec[q];
          }
        int win = 0, p = wpos;
        if (NW > 1) {
          if (lane == 0) {
            sval[pb][wave] = wmax;
            spos[pb][wave] = wpos;
          }
          __syncthreads();
          double bv = sval[pb][0];
          p = spos[pb][0];
#pragma unroll
          for (int q = 1; q < NW; ++q) {
            const double v = sval[pb][q];
            const int r = spos[pb][q];
            if (v > bv || (v == bv && r < p)) {
              bv = v;
              p = r;
              win = q;
            }
          }
        } else {
          wave_sync();
        }
        const zd *u = slot[pb][win];
        const zd d = u[0], dinv = u[CW];
        const bool zero = d.x == 0.0 && d.y == 0.0;
        if (tid == 0) spiv[k - k0] = make_int2(p, zero ? 1 : 0);
#pragma unroll
        for (int q = 0; q < RPT; ++q) {
          pos[q] = pos[q] == p ? k : (pos[q] == k ? p : pos[q]);
          const bool below = pos[q] > k;
          const zd l = zmul(A_[q][0], dinv);
          const zd lm = below ? l : zmk(0, 0);
          const zd last = below ? l : (zero && pos[q] == k ? zmk(pert, 0.0) : A_[q][0]);
#pragma unroll
          for (int i = 1; i < HC; ++i) A_[q][i - 1] = zfms(lm, u[i < HC - jj ? i : CW + 1], A_[q][i]);
#pragma unroll
          for (int i = 0; i < HB; ++i) B_[q][i] = zfms(lm, u[HC + i], B_[q][i]);
          A_[q][HC - 1] = last;
        }
        if (NW == 1) wave_sync();
      }
    };
    steps(xa, xb, std::integral_constant<int, HC>(), 0);
    if (cw > HC) steps(xb, xa, std::integral_constant<int, 0>(), HC);
    // the chunk's columns to the rows' positions; the panel's earlier columns
    // follow the chunk's interchanges (read before any is written)
#pragma unroll
    for (int q = 0; q < RPT; ++q) {
      perm[pos[q] - k0] = from[q];
      if (row[q] < s)
#pragma unroll
        for (int i = 0; i < HC; ++i) {
          if (i < cw) F[pos[q] + (int64_t)(k0 + c0 + i) * f] = xa[q][i];
          if (HC + i < cw) F[pos[q] + (int64_t)(k0 + c0 + HC + i) * f] = xb[q][i];
        }
    }
    for (int e = 0; e < c0; e += HC) {
#pragma unroll
      for (int q = 0; q < RPT; ++q)
        if (pos[q] != row[q])
#pragma unroll
          for (int i = 0; i < HC; ++i) xa[q][i] = F[row[q] + (int64_t)(k0 + e + i) * f];
      __syncthreads();
#pragma unroll
      for (int q = 0; q < RPT; ++q)
        if (pos[q] != row[q])
#pragma unroll
          for (int i = 0; i < HC; ++i) F[pos[q] + (int64_t)(k0 + e + i) * f] = xa[q][i];
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < RPT; ++q) from[q] = perm[row[q] - k0];
    __syncthreads();
  }
  // pivot order and the net interchange
  int so[RPT];
#pragma unroll
  for (int q = 0; q < RPT; ++q) so[q] = k0 == 0 ? from[q] : sig[po + min(from[q], s - 1)];
  __syncthreads();
#pragma unroll
  for (int q = 0; q < RPT; ++q)
    if (row[q] < s) {
      sig[po + row[q]] = so[q];
      if (row[q] >= k0 + w && from[q] != row[q]) {
        const int i = atomicAdd(&nout, 1);
        outr[i] = row[q];
        outs[i] = from[q];
      }
    }
  __syncthreads();
  if (tid < w) {
    gx[po + k0 + tid] = make_int4(from[0], outr[tid], outs[tid], 0);
    piv[po + k0 + tid] = spiv[tid].x;
    pflag[po + k0 + tid] = spiv[tid].y;
  }
}

// The rest of a panel step outside the panel, one 64-thread workgroup per
// task (front, position, kind):
//   kind 0  64 update rows s <= r < f (not pivot candidates) of the panel's
//           columns: a row-wise triangular solve against the factored w x w
//           block U (incl. the possibly perturbed diagonal), x U = a_r, with
//           the operations the column steps would apply to the row, in the
//           same order (l = x_j / U_jj via the reciprocal, then
//           x_c -= l U_jc).  One thread per row.
//   kind 1  64 columns outside the panel: the panel's net row interchange
//           (gx) as one gather and, right of the panel, the unit lower
//           triangular solve of the U12 block row.  One thread per column; the
//           interchange only ever moves rows of [k0, k0 + w) out of the panel,
//           so the rows outside are written from the panel's old rows.
// Both kinds are independent and latency-bound at the few-front levels, so
// they share one launch.
//
// The 32 steps of a solve run in two rolled loops of 16 on a ring of
// registers (as in k_panel_reg), the first also applied to the second half:
// unrolled, the 496 coefficients are 100 KB of code, more than the
// instruction cache.  A short panel is padded with the identity.
template <bool ROWS>
__device__ __forceinline__ void apply_half(const zd (*__restrict__ P)[NB + 1], const zd *__restrict__ dinv, int j0,
                                           zd (&a)[NB / 2], zd (&b)[NB / 2]) {
  constexpr int H = NB / 2;
#pragma unroll 1
  for (int jj = 0; jj < H; ++jj) {
    const int j = j0 + jj;
    const zd l = ROWS ? zmul(a[0], dinv[j]) : a[0];
#pragma unroll
    for (int i = 1; i < H; ++i) {
      const zd u = i < H - jj ? P[j][(j + i) & (NB - 1)] : zmk(0, 0);
      a[i - 1] = ROWS ? zfms(l, u, a[i]) : zfms(u, l, a[i]);
    }
    a[H - 1] = l;
    if (j0 == 0)
#pragma unroll
      for (int i = 0; i < H; ++i) b[i] = ROWS ? zfms(l, P[j][H + i], b[i]) : zfms(P[j][H + i], l, b[i]);
  }
}

__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2, 8)))
void k_panel_apply(const int32_t *__restrict__ tasks, int k0, FrontArrays A, zd *__restrict__ pool, int64_t psz,
                   const int4 *__restrict__ gx, int64_t npiv) {
  constexpr int H = NB / 2;
  const int t = tasks[3 * blockIdx.x], p0 = tasks[3 * blockIdx.x + 1], kind = tasks[3 * blockIdx.x + 2];
  const int b = blockIdx.y;
  const int tid = threadIdx.x;
  const int s = A.s[t], f = A.f[t];
  zd *F = pool + b * psz + A.off[t];
  const int w = min(NB, s - k0);
  // P[j][c]: coefficient of step j on entry c (U for the rows, L transposed
  // for the columns)
  __shared__ zd P[NB][NB + 1];
  __shared__ zd dinv[NB];
  const bool left = kind == 1 && p0 < k0;
  if (!left) {
    for (int idx = tid; idx < NB * NB; idx += 64) {
      const int i = idx % NB, j = idx / NB;
      const zd v = F[(k0 + min(i, w - 1)) + (int64_t)(k0 + min(j, w - 1)) * f];
      const zd e = (i < w && j < w) ? v : zmk(i == j ? 1.0 : 0.0, 0.0);
      if (kind == 0) P[i][j] = e;
      else P[j][i] = e;
    }
    __syncthreads();
  }
  zd xa[H], xb[H];
  if (kind == 0) {
    if (tid < NB) dinv[tid] = zdiv(zmk(1.0, 0.0), P[tid][tid]);
    __syncthreads();
    const int r = p0 + tid;
    zd *row = F + min(r, f - 1) + (int64_t)k0 * f;
#pragma unroll
    for (int j = 0; j < H; ++j) xa[j] = row[(int64_t)min(j, w - 1) * f];
#pragma unroll
    for (int j = 0; j < H; ++j) xb[j] = row[(int64_t)min(H + j, w - 1) * f];
    apply_half<true>(P, dinv, 0, xa, xb);
    if (w > H) apply_half<true>(P, dinv, H, xb, xa);
    if (r < f) {
#pragma unroll
      for (int j = 0; j < H; ++j)
        if (j < w) row[(int64_t)j * f] = xa[j];
#pragma unroll
      for (int j = 0; j < H; ++j)
        if (H + j < w) row[(int64_t)(H + j) * f] = xb[j];
    }
    return;
  }
  const int4 *g = gx + b * npiv + A.pivoff[t] + k0;  // wave-uniform: scalar loads
  const int c = p0 + tid;
  const bool ok = left ? c < k0 : c < f;
  zd *col = F + (int64_t)(ok ? c : p0) * f;
#pragma unroll
  for (int i = 0; i < H; ++i) xa[i] = col[g[min(i, w - 1)].x];
#pragma unroll
  for (int i = 0; i < H; ++i) xb[i] = col[g[min(H + i, w - 1)].x];
  // the rows leaving the panel (a prefix of the list), from its old rows
  for (int i = 0; i < w && g[i].y >= 0; i += 4) {
    const int4 e0 = g[i], e1 = g[min(i + 1, w - 1)], e2 = g[min(i + 2, w - 1)], e3 = g[min(i + 3, w - 1)];
    const zd v0 = col[e0.z], v1 = col[e1.z], v2 = col[e2.z], v3 = col[e3.z];
    if (ok) {  // entries past the list repeat the last one or have y = -1
      col[e0.y] = v0;
      if (e1.y >= 0) col[e1.y] = v1;
      if (e2.y >= 0) col[e2.y] = v2;
      if (e3.y >= 0) col[e3.y] = v3;
    }
  }
  if (!left) {
    apply_half<false>(P, dinv, 0, xa, xb);
    if (w > H) apply_half<false>(P, dinv, H, xb, xa);
  }
  if (ok) {
#pragma unroll
    for (int i = 0; i < H; ++i)
      if (i < w) col[k0 + i] = xa[i];
#pragma unroll
    for (int i = 0; i < H; ++i)
      if (H + i < w) col[k0 + H + i] = xb[i];
  }
}

// C -= L21 U12 on one 64 x 64 tile of the trailing block.  The panel's K = w
// <= 32 columns are staged through LDS in two halves of 16 (32 KB of LDS, so
// that four workgroups share a CU); thread (tx, ty) owns rows tx + 16 i and
// columns ty + 16 j, so a wave's C accesses cover 16 consecutive rows of 4
// columns; the 16 reads of C are issued together from clamped addresses
// before any is used, the stores are masked.
constexpr int GK = 16;  // K staged per round
__global__ __launch_bounds__(256) void k_gemm_update(const int32_t *__restrict__ tasks, int k0,
                                                     FrontArrays A, zd *__restrict__ pool,
                                                     int64_t psz) {
  const int t = tasks[3 * blockIdx.x], r0 = tasks[3 * blockIdx.x + 1], c0 = tasks[3 * blockIdx.x + 2];
  const int b = blockIdx.y;
  const int tid = threadIdx.x;
  const int s = A.s[t], f = A.f[t];
  zd *F = pool + b * psz + A.off[t];
  const int w = min(NB, s - k0);
  __shared__ zd As[GK][TILE];
  __shared__ zd Bs[GK][TILE];
  const int tx = tid % 16, ty = tid / 16;
  zd acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = zmk(0, 0);
  for (int kb = 0; kb < w; kb += GK) {
    if (kb > 0) __syncthreads();
    // staging: unconditional loads from clamped addresses (a load inside a
    // branch is waited for before the branch merges, which would serialise
    // the tile's loads), out-of-range entries zeroed afterwards
#pragma unroll
    for (int u = 0; u < GK * TILE / 256; ++u) {
      const int idx = tid + 256 * u, i = idx % TILE, kk = idx / TILE, r = r0 + i;
      const zd v = F[min(r, f - 1) + (int64_t)(k0 + min(kb + kk, w - 1)) * f];
      As[kk][i] = (kb + kk < w && r < f) ? v : zmk(0, 0);
    }
#pragma unroll
    for (int u = 0; u < GK * TILE / 256; ++u) {
      const int idx = tid + 256 * u, kk = idx % GK, jj = idx / GK, c = c0 + jj;
      const zd v = F[(k0 + min(kb + kk, w - 1)) + (int64_t)min(c, f - 1) * f];
      Bs[kk][jj] = (kb + kk < w && c < f) ? v : zmk(0, 0);
    }
    __syncthreads();
    const int kn = min(GK, w - kb);
    for (int kk = 0; kk < kn; ++kk) {
      zd a[4], bb[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = As[kk][tx + 16 * i];
#pragma unroll
      for (int j = 0; j < 4; ++j) bb[j] = Bs[kk][ty + 16 * j];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = zfma(a[i], bb[j], acc[i][j]);
    }
  }
  // in two halves of 8 entries (fewer live registers)
#pragma unroll
  for (int jh = 0; jh < 4; jh += 2) {
    zd cv[4][2];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        cv[i][j] = F[min(r0 + tx + 16 * i, f - 1) + (int64_t)min(c0 + ty + 16 * (jh + j), f - 1) * f];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int c = c0 + ty + 16 * (jh + j);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = r0 + tx + 16 * i;
        if (r < f && c < f) F[r + (int64_t)c * f] = zsub(cv[i][j], acc[i][jh + j]);
      }
    }
  }
}

__global__ __launch_bounds__(256) void k_extend_add(const int32_t *__restrict__ tasks, FrontArrays A,
                                                    zd *__restrict__ pool, int64_t psz) {
  const int t = tasks[2 * blockIdx.x], c0 = tasks[2 * blockIdx.x + 1];
  const int b = blockIdx.y;
  const int s = A.s[t], u = A.u[t], f = A.f[t];
  const int p = A.parent[t];
  const int fp = A.f[p];
  const zd *C = pool + b * psz + A.off[t];
  zd *P = pool + b * psz + A.off[p];
  const int32_t *mp = A.pmap + A.uoff[t];
  for (int cc = 0; cc < EA_COLS; ++cc) {
    int c = c0 + cc;
    if (c >= u) break;
    int64_t pc = (int64_t)mp[c] * fp;
    const zd *src = C + (int64_t)(s + c) * f + s;
    for (int r = threadIdx.x; r < u; r += blockDim.x) {
      zd *d = P + pc + mp[r];
      *d = zadd(*d, src[r]);
    }
  }
}

// Forward gather records, one per pivot: the right-hand-side index of the
// pivot's row (fb + j, j = sig[k]) and the two child update entries that add
// into that row (-1: none).  The solves of one factorisation then fetch a
// front's inputs with one dependent load instead of three.
__global__ __launch_bounds__(64) void k_gather_index(FrontArrays A, const int32_t *__restrict__ sig, int64_t npiv,
                                                     int4 *__restrict__ gx) {
  const int t = blockIdx.x, b = blockIdx.y;
  const int s = A.s[t], fb = A.b[t];
  const int64_t po = A.pivoff[t], fvo = A.fvoff[t];
  const int32_t *sg = sig + b * npiv + po;
  int4 *g = gx + b * npiv + po;
  for (int k = threadIdx.x; k < s; k += 64) {
    const int j = sg[k];
    g[k] = make_int4(fb + j, A.cmap[2 * (fvo + j)], A.cmap[2 * (fvo + j) + 1], 0);
  }
}

// The panel kernel by the largest number of pivot candidates in the launch:
// one wavefront up to 128 rows (no barrier, and the small fronts of the lower
// levels then keep four times as many panels in flight), one row per thread
// up to the 1,024 threads of a workgroup, then more rows per thread and
// fewer columns at a time, within the 128 registers that 1,024 threads leave.
static void launch_panel(const int32_t *tasks, unsigned cnt, int nb, int k0, int rows, const FrontArrays &A, zd *pool,
                         int64_t psz, int32_t *piv, int64_t npiv, int32_t *pflag, int32_t *sig, int4 *gx,
                         hipStream_t s) {
  const double pert = 1e-13;
  const dim3 g(cnt, nb);
#define EMU_PANEL(NW, RPT, CW)                                                                              \
  hipLaunchKernelGGL((k_panel_reg<NW, RPT, CW>), g, dim3(64 * NW), 0, s, tasks, k0, A, pool, psz, piv, npiv, \
                     pflag, sig, gx, pert)
  if (rows <= 64) EMU_PANEL(1, 1, 16);
  else if (rows <= 128) EMU_PANEL(1, 2, 8);
  else if (rows <= 256) EMU_PANEL(4, 1, 16);
  else if (rows <= 512) EMU_PANEL(8, 1, 16);
  else if (rows <= 1024) EMU_PANEL(16, 1, 8);
  else if (rows <= 2048) EMU_PANEL(16, 2, 4);
  else if (rows <= 4096) EMU_PANEL(16, 4, 2);
  else
    hipLaunchKernelGGL(k_panel, g, dim3(256), 0, s, tasks, k0, A, pool, psz, piv, npiv, pflag, sig, gx, pert);
#undef EMU_PANEL
}

void lu_factor(DevMesh &dm, int nb, const zd *mat1, zd *pool, int32_t *piv, int32_t *pflag, int32_t *sig,
               int32_t *gx, zd *inv, zd *wt, hipStream_t s) {
  const Symbolic &sy = dm.host.sym;
  const int64_t psz = sy.pool;
  FrontArrays A = fa(dm);
  launch_fill(pool, psz * nb, zmk(0, 0), s);
  {
    int64_t nnz = dm.host.nnz;
    dim3 g((unsigned)((nnz + 255) / 256), nb);
    hipLaunchKernelGGL(k_scatter_fronts, g, dim3(256), 0, s, nnz, psz, dm.nnz2front.p, mat1, pool);
    EMU_LAUNCH_CHECK();
  }
  for (const LevelSched &L : dm.sched) {
    for (const StepPlan &st : L.steps) {
      if (st.panel_cnt)
        launch_panel(dm.tasks.p + st.panel_off, (unsigned)st.panel_cnt, nb, st.k0, st.rows, A, pool, psz, piv,
                     sy.npiv, pflag, sig, reinterpret_cast<int4 *>(gx), s);
      if (st.apply_cnt)
        hipLaunchKernelGGL(k_panel_apply, dim3((unsigned)st.apply_cnt, nb), dim3(64), 0, s,
                           dm.tasks.p + st.apply_off, st.k0, A, pool, psz, reinterpret_cast<const int4 *>(gx),
                           sy.npiv);
      if (st.gemm_cnt)
        hipLaunchKernelGGL(k_gemm_update, dim3((unsigned)st.gemm_cnt, nb), dim3(256), 0, s,
                           dm.tasks.p + st.gemm_off, st.k0, A, pool, psz);
    }
    for (int sl = 0; sl < 2; ++sl)
      if (L.ea_cnt[sl])
        hipLaunchKernelGGL(k_extend_add, dim3((unsigned)L.ea_cnt[sl], nb), dim3(256), 0, s,
                           dm.tasks.p + L.ea_off[sl], A, pool, psz);
    EMU_LAUNCH_CHECK();
  }
  lu_invert(dm, nb, pool, inv, wt, s);
  const int nf = (int)sy.fronts.size();
  if (nf)
    hipLaunchKernelGGL(k_gather_index, dim3((unsigned)nf, nb), dim3(64), 0, s, A, sig, sy.npiv,
                       reinterpret_cast<int4 *>(gx));
  EMU_LAUNCH_CHECK();
}

// ------------------------------------------------- inverted-factor form
//
// After the numeric factorisation every front is rewritten, out of place,
// into the form the solves use:
//   forward block  (f x s, ld f):  [ L11^{-1} ; -L21 L11^{-1} ]
//   backward block (s x f, ld s):  [ U11^{-1} , -U11^{-1} U12 ]
// so that one front's forward step is y = Fwd * (P r_S) (+ r_U on the update
// rows) and its backward step is x_S = Bwd * [y_S ; x_U]: dense matrix-vector
// products that split over row tiles across the whole GPU instead of a
// column-sequential substitution inside one workgroup.  P is the front's
// row-pivot permutation, applied as a gather (the gx records).

// The triangular inverses are formed by doubling: k_tri_diag inverts the
// 64 x 64 diagonal blocks, then for h = 64, 128, ... each pair of inverted
// diagonal blocks A (h) and C gets its off-diagonal block B' = -C^-1 (B A^-1)
// (lower) or -A^-1 (B C^-1) (upper) as two products of 64 x 64 tiles
// (k_inv_gemm), all pairs of all fronts in one launch each, and two more that
// correct it by its residual: U11 is ill-conditioned (1e6 on the case-1 cell)
// and the plain products would leave solve residuals up to ten times those of
// a substitution (8e-9 against 1e-9; 1e-9 with the correction).  The two
// off-diagonal blocks of the inverted form follow as tiles of the same kernel.
// Column-block substitution (one workgroup per 32 columns walking down the
// front) was a serial chain of s / 32 products and 32-step solves.  Both parts
// per factorisation: 8,000-triangle mesh, 2 / 8 instances, 6.4 / 15.5 ms, now
// 2.9 / 8.8 ms; 64 dense matrices of order 98 and 200 (mean) 403 us, now 194 us.
typedef double v4d __attribute__((ext_vector_type(4)));

// acc += A B on 16 x 16 x 4 complex blocks: a = A[i][k] in lane i + 16 k,
// x = B[k][j] in lane j + 16 k; result D[i][j] in lane j + 16 (i mod 4),
// register i / 4.
__device__ __forceinline__ void mfma_z(v4d &re, v4d &im, zd a, zd x) {
  re = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x, x.x, re, 0, 0, 0);
  im = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x, x.y, im, 0, 0, 0);
  re = __builtin_amdgcn_mfma_f64_16x16x4f64(-a.y, x.y, re, 0, 0, 0);
  im = __builtin_amdgcn_mfma_f64_16x16x4f64(a.y, x.x, im, 0, 0, 0);
}

// Eight steps of the substitution of k_tri_diag, from row j0 of the block at
// o: the ring a holds rows j0 .. j0 + 7, b the eight rows after them (FIRST).
template <bool FIRST>
__device__ __forceinline__ void tri_half(const zd (*__restrict__ T)[65], const zd *__restrict__ dinv, int o, int j0,
                                         zd (&a)[8], zd (&b)[8]) {
#pragma unroll 1
  for (int jj = 0; jj < 8; ++jj) {
    const int j = j0 + jj;
    const zd l = zmul(a[0], dinv[j]);
#pragma unroll
    for (int i = 1; i < 8; ++i) {
      const zd u = i < 8 - jj ? T[min(j + i, 63)][j] : zmk(0, 0);
      a[i - 1] = zfms(u, l, a[i]);
    }
    a[7] = l;
    if (FIRST)
#pragma unroll
      for (int i = 0; i < 8; ++i) b[i] = zfms(T[o + 8 + i][j], l, b[i]);
  }
}

// One workgroup per (front, 64-row diagonal block J, kind, instance): the
// block's inverse, zeros of the other triangle included (the solves and the
// products below read nothing outside the diagonal 64-blocks and the
// triangle).  kind 0: L11 (unit lower); kind 1: U11, handled as a lower
// triangle by reversing rows and columns.  The block sits in LDS, padded with
// the identity, and X = T^-1 replaces it 16 rows at a time: the product of
// the rows with the finished rows of X on the matrix cores, then a substitution
// with the 16 x 16 diagonal block, one lane per column.  (Multiplying by an
// inverted diagonal block instead would be shorter, but U11's blocks are
// ill-conditioned, 1e6 on the case-1 cell, and its rounding then grows to ten
// times that of the substitution.)
__global__ __launch_bounds__(256) void k_tri_diag(const int32_t *__restrict__ tasks, FrontArrays A,
                                                  const zd *__restrict__ pool, int64_t psz, zd *__restrict__ inv,
                                                  int64_t isz) {
  constexpr int D = 64, E = 16;
  const int t = tasks[3 * blockIdx.x], J = tasks[3 * blockIdx.x + 1], kind = tasks[3 * blockIdx.x + 2];
  const int b = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int s = A.s[t], f = A.f[t];
  const int j0 = J * D, w = min(D, s - j0);
  const zd *F = pool + b * psz + A.off[t] + j0 + (int64_t)j0 * f;
  const int64_t ldo = kind ? s : f;
  zd *O = inv + b * isz + A.ioff[t] + (kind ? (int64_t)f * s : 0) + j0 + j0 * ldo;
  __shared__ zd T[D][D + 1];
  __shared__ zd dinv[D];
  for (int idx = tid; idx < D * D; idx += 256) {
    const int i = idx % D, j = idx / D;
    const int fi = kind ? w - 1 - i : i, fj = kind ? w - 1 - j : j;
    const zd v = F[min(max(fi, 0), w - 1) + (int64_t)min(max(fj, 0), w - 1) * f];
    T[i][j] = (i < w && j <= i) ? v : zmk(0, 0);
  }
  __syncthreads();
  if (tid < D) dinv[tid] = kind && tid < w ? zdiv(zmk(1, 0), T[tid][tid]) : zmk(1, 0);
  __syncthreads();
  const int fi = lane & 15, fk = lane >> 4;
#pragma unroll 1
  for (int o = 0; o < w; o += E) {
    // rows o .. o + 15 of -T X over the finished rows of X: wave v the columns
    // 16 v .. 16 v + 15, written over the entries of T that they come from
    const int cv = E * wave;
    v4d re = {0, 0, 0, 0}, im = {0, 0, 0, 0};
    if (cv < o)
      for (int k = cv; k < o; k += 4) mfma_z(re, im, T[o + fi][k + fk], T[k + fk][cv + fi]);
    __syncthreads();
    if (cv < o)
#pragma unroll
      for (int r = 0; r < 4; ++r) T[o + fk + 4 * r][cv + fi] = zmk(-re[r], -im[r]);
    __syncthreads();
    if (wave == 0) {  // lane = column: substitution with the 16 x 16 diagonal block
      constexpr int H = E / 2;
      zd xa[H], xb[H];
#pragma unroll
      for (int i = 0; i < H; ++i) {
        const zd va = T[o + i][lane], vb = T[o + H + i][lane];
        xa[i] = lane < o ? va : zmk(lane == o + i ? 1.0 : 0.0, 0.0);
        xb[i] = lane < o ? vb : zmk(lane == o + H + i ? 1.0 : 0.0, 0.0);
      }
      tri_half<true>(T, dinv, o, o, xa, xb);
      tri_half<false>(T, dinv, o, o + H, xb, xa);
      wave_sync();
      if (lane < o + E)
#pragma unroll
        for (int i = 0; i < H; ++i) {
          T[o + i][lane] = xa[i];
          T[o + H + i][lane] = xb[i];
        }
    }
    __syncthreads();
  }
  for (int idx = tid; idx < w * w; idx += 256) {
    const int i = idx % w, j = idx / w;
    const int ti = kind ? w - 1 - i : i, tj = kind ? w - 1 - j : j;
    O[i + j * ldo] = ti >= tj ? T[ti][tj] : zmk(0, 0);
  }
}

// One 64 x 64 tile C = A B, -A B, C + A B or C - A B of the inversion (InvTile:
// base arrays, offsets, leading dimensions, extents).  As k_zgemm_nn: 16-deep K rounds in
// LDS, the next round fetched from clamped addresses meanwhile, wave w owns
// columns 16 w .. 16 w + 15; 16-column blocks and the lower
// half beyond the tile's extents are skipped
// (most fronts are smaller than a tile).  FLOP-bound: a full tile takes 64 x 64
// x 16 x 8 flops / 128 per clock = 4,096 clocks a round.
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3, 4))) void k_inv_gemm(const InvTile *__restrict__ tiles, const zd *__restrict__ pool,
                                                  int64_t psz, zd *__restrict__ inv, int64_t isz,
                                                  zd *__restrict__ wt, int64_t wsz) {
  const InvTile R = tiles[blockIdx.x];
  const int b = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  zd *const base1 = inv + b * isz, *const base2 = wt + b * wsz;
  const zd *Ab = (R.abase == 0 ? pool + b * psz : R.abase == 1 ? (const zd *)base1 : base2) + R.aoff;
  const zd *Bb = (R.bbase == 0 ? pool + b * psz : R.bbase == 1 ? (const zd *)base1 : base2) + R.boff;
  zd *Cb = (R.cbase == 1 ? base1 : base2) + R.coff;
  __shared__ zd As[GK][TILE + 1];
  __shared__ zd Bs[GK][TILE + 1];
  const int am = tid & 63, ak = tid >> 6;  // A: row am, K columns ak + 4 i
  const int bk = tid & 15, bn = tid >> 4;  // B: K row bk, columns bn + 16 i
  zd ra[4], rb[4];
  auto fetch = [&](int k0) {
#pragma unroll
    for (int i = 0; i < 4; ++i) ra[i] = Ab[min(am, R.M - 1) + (int64_t)min(k0 + ak + 4 * i, R.K - 1) * R.lda];
    const int kb = min(k0 + bk, R.K - 1);
#pragma unroll
    for (int i = 0; i < 4; ++i) rb[i] = Bb[kb + (int64_t)min(bn + 16 * i, R.N - 1) * R.ldb];
  };
  v4d re[4], im[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    re[t] = (v4d){0, 0, 0, 0};
    im[t] = (v4d){0, 0, 0, 0};
  }
  const int fi = lane & 15, fk = lane >> 4;
  fetch(0);
  for (int k0 = 0; k0 < R.K; k0 += GK) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int kk = ak + 4 * i, d = k0 + kk - am - R.doff;  // columns right of the diagonal
      bool ok = k0 + kk < R.K && am < R.M;
      if (R.tri == 1) ok = ok && d < 0;
      if (R.tri == 2) ok = ok && d >= 0;
      As[kk][am] = ok ? ra[i] : zmk(R.tri == 1 && d == 0 ? 1.0 : 0.0, 0);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) Bs[bk][bn + 16 * i] = (k0 + bk < R.K && bn + 16 * i < R.N) ? rb[i] : zmk(0, 0);
    __syncthreads();
    if (k0 + GK < R.K) fetch(k0 + GK);
    if (16 * wv < R.N) {
      if (R.M > 32) {
#pragma unroll
        for (int ks = 0; ks < GK / 4; ++ks) {
          const int kk = ks * 4 + fk;
          const zd xb = Bs[kk][16 * wv + fi];
#pragma unroll
          for (int t = 0; t < 4; ++t) mfma_z(re[t], im[t], As[kk][16 * t + fi], xb);
        }
      } else {
#pragma unroll
        for (int ks = 0; ks < GK / 4; ++ks) {
          const int kk = ks * 4 + fk;
          const zd xb = Bs[kk][16 * wv + fi];
#pragma unroll
          for (int t = 0; t < 2; ++t) mfma_z(re[t], im[t], As[kk][16 * t + fi], xb);
        }
      }
    }
  }
  const int n = 16 * wv + fi;
  if (n >= R.N) return;
  Cb += (int64_t)n * R.ldc;
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int m = 16 * t + fk + 4 * r;
      if (m < R.M) {
        zd v = R.neg ? zmk(-re[t][r], -im[t][r]) : zmk(re[t][r], im[t][r]);
        if (R.acc) v = zadd(Cb[m], v);
        Cb[m] = v;
      }
    }
}

void lu_invert(DevMesh &dm, int nb, const zd *pool, zd *inv, zd *wt, hipStream_t s) {
  const Symbolic &sy = dm.host.sym;
  FrontArrays A = fa(dm);
  if (dm.tri_cnt)
    hipLaunchKernelGGL(k_tri_diag, dim3((unsigned)dm.tri_cnt, nb), dim3(256), 0, s, dm.tasks.p + dm.tri_off, A, pool,
                       sy.pool, inv, dm.isz);
  EMU_LAUNCH_CHECK();
  for (const auto &r : dm.inv_phases)
    if (r.second > 0)
      hipLaunchKernelGGL(k_inv_gemm, dim3((unsigned)r.second, nb), dim3(256), 0, s, dm.inv_tiles.p + r.first, pool,
                         sy.pool, inv, dm.isz, wt, dm.wsz);
  EMU_LAUNCH_CHECK();
}

// ---------------------------------------------------------------- solves
//
// Rows of a front are cut into 64-row tiles, one per wavefront.  A workgroup
// (4 waves) takes `tpw` consecutive tiles of one front (task (front, r0,
// tpw), tpw = 4, 2 or 1 chosen per front on the host); the 4 / tpw waves that
// share a tile split its column range and add their partial sums through
// LDS.  Small-front levels thus keep all waves busy on distinct rows, the
// few large fronts of the top levels get the column split.  The front's
// input vector is staged through LDS in chunks of KC entries, gathered on
// the fly (forward: b at the pivot rows in pivot order plus the children's
// update vectors; backward: y at the own rows, x at the ancestors' rows).
// Structural zeros of the triangular inverses are skipped per tile.  Tasks
// of one level never write what another reads, so a level is one launch.

constexpr int KC = 64;  // staged input chunk

// Storage of the inverted factor read by the solves: complex128 (zd), or
// complex64 (float2, the mixed-precision form), widened to double on load;
// the arithmetic is FP64 either way.
template <typename FT>
struct FactorLd;
template <>
struct FactorLd<zd> {
  static constexpr uint32_t kBytes = 16;
  static __device__ __forceinline__ zd ld(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
    return buf_ld_stream(r, voff, soff);
  }
};
template <>
struct FactorLd<float2> {
  static constexpr uint32_t kBytes = 8;
  static __device__ __forceinline__ zd ld(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
    typedef float f2 __attribute__((ext_vector_type(2)));
    const f2 v = __builtin_bit_cast(f2, __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 2));
    return zmk((double)v.x, (double)v.y);
  }
};

template <int RC, typename FT>
__global__ __launch_bounds__(256) void k_fwd(const SolveTask *__restrict__ tasks, const int32_t *__restrict__ cmap,
                                             const FT *__restrict__ inv, int64_t isz, const int4 *__restrict__ gx,
                                             int64_t npiv, int nrhs, int64_t n, int64_t nw,
                                             const zd *__restrict__ bv, zd *__restrict__ y, zd *__restrict__ wbuf,
                                             zd *__restrict__ part, int nslot, int span) {
  const SolveTask T = tasks[blockIdx.x];
  const int b = blockIdx.y;
  const int q0 = blockIdx.z * RC;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform: column offsets in SGPRs
  const int ks = 4 / T.tpw, tile = wave / ks, kp = wave - tile * ks;
  const int s = T.s, f = T.f;
  const FT *Fw = inv + b * isz + T.ioff;
  constexpr uint32_t EB = FactorLd<FT>::kBytes;
  const int4 *gi = gx + b * npiv + T.pivoff;
  const int nq = min(RC, nrhs - q0);
  const int64_t col0 = (int64_t)b * nrhs + q0;
  const int row0 = T.r0 + 64 * tile;  // first row of this wave's tile
  const int row = row0 + lane;
  const int rowc = min(row, f - 1);   // clamped: addresses stay inside the front
  const uint32_t rowb = (uint32_t)rowc * EB;  // byte offset of the row in a column
  // columns of this task: the workgroup's range, cut to [kb, kb + span)
  // for a split task; lower-triangular rows need k <= row
  int kbeg = 0, kend = min(s, T.r0 + 64 * T.tpw);
  if (T.kb >= 0) {
    kbeg = T.kb;
    kend = min(kend, T.kb + span);
  }
  const int kend_w = row0 < f ? min(kend, min(s, row0 + 64)) : 0;
  // child update entries of this row (static), added by the epilogue on the
  // update rows; requested now so that the epilogue waits for one load only
  const int2 cr = reinterpret_cast<const int2 *>(cmap)[T.fvoff + rowc];
  __shared__ zd xin[KC][RC];
  __shared__ zd red[3][64][RC];
  zd acc[RC];
#pragma unroll
  for (int q = 0; q < RC; ++q) acc[q] = zmk(0, 0);
  // Load order per chunk: gather records, then this wave's first 8 columns,
  // then the input values (which depend on the records); the column loads are
  // thus in flight during the gather, and each later batch of 8 is requested
  // before the previous one is used.  All loads are unconditional from
  // clamped addresses, unused values zeroed or discarded afterwards.
  for (int kc = kbeg; kc < kend; kc += KC) {
    const int k = tid & (KC - 1), qg = tid / KC;
    const int kk = kc + k;
    const bool okk = kk < kend;
    const int4 g = gi[okk ? kk : kbeg];
    const int kl = min(KC, kend_w - kc);
    const int nk = kl > kp ? (kl - kp + ks - 1) / ks : 0;  // this wave's columns kp, kp + ks, ...
    // column c of the wave's rows: byte c f EB + rowb of the front's block
    const __amdgpu_buffer_rsrc_t Fcol = buf_view(Fw, (uint32_t)f * (uint32_t)s * EB);
    // column indices clamped into [0, s): an idle wave (nk = 0) reads a
    // valid column and discards it, so the loads need no branch (a branch
    // would make the gather below wait for them)
    const int cbase = kc + kp, clast = min(kc + kp + max(nk - 1, 0) * ks, s - 1);
    zd a[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) a[u] = FactorLd<FT>::ld(Fcol, rowb, (uint32_t)(min(cbase + u * ks, clast) * f) * EB);
    constexpr int NG = (RC + 3) / 4;  // right-hand sides gathered per thread
    zd gv[NG], g0[NG], g1[NG];
#pragma unroll
    for (int u = 0; u < NG; ++u) {
      const int64_t cq = col0 + min(min(qg + 4 * u, RC - 1), nq - 1);
      gv[u] = bv[cq * n + g.x];
      g0[u] = wbuf[cq * nw + max(g.y, 0)];
      g1[u] = wbuf[cq * nw + max(g.z, 0)];
    }
#pragma unroll
    for (int u = 0; u < NG; ++u) {
      const int qq = qg + 4 * u;
      // selects, not branches: a branch would let the compiler sink the
      // load into it and wait there for every load in flight
      const zd v = zadd(zadd(gv[u], g.y >= 0 ? g0[u] : zmk(0, 0)), g.z >= 0 ? g1[u] : zmk(0, 0));
      if (qq < RC) xin[k][qq] = (okk && qq < nq) ? v : zmk(0, 0);
    }
    __syncthreads();
    // full batches: the next batch is requested before this one is used (no
    // branch around the loads: a branch join would wait for them at once)
    int t0 = 0;
    for (; t0 + 8 < nk; t0 += 8) {
      zd nx[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) nx[u] = FactorLd<FT>::ld(Fcol, rowb, (uint32_t)(min(cbase + (t0 + 8 + u) * ks, clast) * f) * EB);
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int kx = kp + (t0 + u) * ks;
#pragma unroll
        for (int q = 0; q < RC; ++q) acc[q] = zfma(a[u], xin[kx][q], acc[q]);
      }
#pragma unroll
      for (int u = 0; u < 8; ++u) a[u] = nx[u];
    }
    // the last, possibly partial, batch
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (t0 + u < nk) {
        const int kx = kp + (t0 + u) * ks;
#pragma unroll
        for (int q = 0; q < RC; ++q) acc[q] = zfma(a[u], xin[kx][q], acc[q]);
      }
    __syncthreads();
  }
  if (ks > 1) {
    if (kp > 0)
#pragma unroll
      for (int q = 0; q < RC; ++q) red[wave - 1][lane][q] = acc[q];
    __syncthreads();
    if (kp == 0)
      for (int j = 1; j < ks; ++j)
#pragma unroll
        for (int q = 0; q < RC; ++q) acc[q] = zadd(acc[q], red[wave + j - 1][lane][q]);
  }
  if (kp != 0) return;
  if (T.slot >= 0) {  // split task: partial sums of the tile, added by k_fwd_red
#pragma unroll
    for (int q = 0; q < RC; ++q)
      if (q < nq) part[((col0 + q) * nslot + T.slot) * 64 + lane] = acc[q];
    return;
  }
  if (row < f) {
    if (row < s) {
#pragma unroll
      for (int q = 0; q < RC; ++q)
        if (q < nq) y[(col0 + q) * n + T.fb + row] = acc[q];
    } else {
      zd w0[RC], w1[RC];
#pragma unroll
      for (int q = 0; q < RC; ++q) {
        const int64_t cq = col0 + min(q, nq - 1);
        w0[q] = wbuf[cq * nw + max(cr.x, 0)];
        w1[q] = wbuf[cq * nw + max(cr.y, 0)];
      }
#pragma unroll
      for (int q = 0; q < RC; ++q) {
        const zd v = zadd(zadd(acc[q], cr.x >= 0 ? w0[q] : zmk(0, 0)), cr.y >= 0 ? w1[q] : zmk(0, 0));
        if (q < nq) wbuf[(col0 + q) * nw + T.uoff + (row - s)] = v;
      }
    }
  }
}

// Sum of the partial sums of a split forward tile (task: front, r0, first
// slot, count; one lane per row, the four waves take every fourth
// right-hand side), then the forward epilogue of k_fwd.  The slot loads of a
// right-hand side are issued eight at a time from clamped slots and added in
// slot order.
template <int RC>
__global__ __launch_bounds__(256) void k_fwd_red(const int32_t *__restrict__ tasks, FrontArrays A, int nrhs,
                                                 int64_t n, int64_t nw, const zd *__restrict__ part, int nslot,
                                                 zd *__restrict__ y, zd *__restrict__ wbuf) {
  const int32_t *tk = tasks + 4 * blockIdx.x;
  const int t = tk[0], r0 = tk[1], p0 = tk[2], np = tk[3];
  const int b = blockIdx.y, q0 = blockIdx.z * RC;
  const int lane = threadIdx.x & 63, qg = threadIdx.x >> 6;
  const int s = A.s[t], f = A.f[t], fb = A.b[t];
  const int32_t *cm = A.cmap + 2 * A.fvoff[t];
  const int64_t uo = A.uoff[t];
  const int nq = min(RC, nrhs - q0);
  const int64_t col0 = (int64_t)b * nrhs + q0;
  const int row = r0 + lane;
  if (row >= f) return;
  const int c0i = row >= s ? cm[2 * row] : -1, c1i = row >= s ? cm[2 * row + 1] : -1;
#pragma unroll
  for (int u = 0; u < (RC + 3) / 4; ++u) {
    const int q = qg + 4 * u;
    if (q >= nq) break;
    const zd *pp = part + ((col0 + q) * nslot + p0) * 64 + lane;
    zd v = zmk(0, 0);
    for (int c = 0; c < np; c += 8) {
      zd h[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) h[i] = pp[(int64_t)min(c + i, np - 1) * 64];
#pragma unroll
      for (int i = 0; i < 8; ++i)
        if (c + i < np) v = zadd(v, h[i]);
    }
    if (row < s) {
      y[(col0 + q) * n + fb + row] = v;
    } else {
      const zd w0 = wbuf[(col0 + q) * nw + max(c0i, 0)], w1 = wbuf[(col0 + q) * nw + max(c1i, 0)];
      if (c0i >= 0) v = zadd(v, w0);
      if (c1i >= 0) v = zadd(v, w1);
      wbuf[(col0 + q) * nw + uo + (row - s)] = v;
    }
  }
}

template <int RC, typename FT>
__global__ __launch_bounds__(256) void k_bwd(const SolveTask *__restrict__ tasks, const int32_t *__restrict__ uidx,
                                             const FT *__restrict__ inv, int64_t isz, int nrhs, int64_t n,
                                             const zd *__restrict__ y, zd *__restrict__ x, int64_t sx,
                                             zd *__restrict__ part, int nslot, int span) {
  const SolveTask T = tasks[blockIdx.x];
  const int b = blockIdx.y;
  const int q0 = blockIdx.z * RC;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform: column offsets in SGPRs
  const int ks = 4 / T.tpw, tile = wave / ks, kp = wave - tile * ks;
  const int s = T.s, f = T.f;
  const FT *Bw = inv + b * isz + T.ioff + (int64_t)f * s;
  constexpr uint32_t EB = FactorLd<FT>::kBytes;
  const int32_t *ui = uidx + T.uoff;
  const int nq = min(RC, nrhs - q0);
  const int64_t col0 = (int64_t)b * nrhs + q0;
  // this instance's input y (nrhs columns of n) and output x (instance
  // stride sx: the solve may write straight into a slot of a larger array)
  const zd *yb = y + (int64_t)b * nrhs * n;
  zd *xb = x + (int64_t)b * sx;
  const int row = T.r0 + 64 * tile;  // first row of this wave's tile
  const int rowl = row + lane;
  const int rowc = min(rowl, s - 1);
  const uint32_t rowb = (uint32_t)max(rowc, 0) * EB;  // byte offset of the row in a column
  // columns: [r0, f) for the workgroup (upper-triangular rows need k >= row),
  // cut to [kb, kb + span) for a split task
  int kbeg = T.r0, kend = f;
  if (T.kb >= 0) {
    kbeg = T.kb;
    kend = min(f, T.kb + span);
  }
  __shared__ zd xin[KC][RC];
  __shared__ zd red[3][64][RC];
  zd acc[RC];
#pragma unroll
  for (int q = 0; q < RC; ++q) acc[q] = zmk(0, 0);
  // load order as in k_fwd: input index, first 8 columns, input values
  for (int kc = kbeg; kc < kend; kc += KC) {
    const int k = tid & (KC - 1), qg = tid / KC;
    const int kk = kc + k;
    const bool okk = kk < kend;
    const int kkc = okk ? kk : kbeg;
    // input row kkc: y of this front or x of an ancestor
    const int64_t off = kkc < s ? (int64_t)T.fb + kkc : (int64_t)ui[kkc - s];
    const int klo = max(0, row - kc), khi = min(KC, kend - kc);
    const int kst = klo + kp;
    const int nk = (row < s && khi > kst) ? (khi - kst + ks - 1) / ks : 0;
    // column c of the wave's rows: byte c s EB + rowb of the front's block
    const __amdgpu_buffer_rsrc_t Fcol = buf_view(Bw, (uint32_t)f * (uint32_t)s * EB);
    // column indices clamped into [0, f) (see k_fwd)
    const int cbase = kc + kst, clast = min(kc + kst + max(nk - 1, 0) * ks, f - 1);
    zd a[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) a[u] = FactorLd<FT>::ld(Fcol, rowb, (uint32_t)(min(cbase + u * ks, clast) * s) * EB);
    const zd *src = kkc < s ? yb : xb;
    constexpr int NG = (RC + 3) / 4;
    zd gv[NG];
#pragma unroll
    for (int u = 0; u < NG; ++u) gv[u] = src[(q0 + min(min(qg + 4 * u, RC - 1), nq - 1)) * n + off];
#pragma unroll
    for (int u = 0; u < NG; ++u) {
      const int qq = qg + 4 * u;
      if (qq < RC) xin[k][qq] = (okk && qq < nq) ? gv[u] : zmk(0, 0);
    }
    __syncthreads();
    // full batches: the next batch is requested before this one is used (no
    // branch around the loads: a branch join would wait for them at once)
    int t0 = 0;
    for (; t0 + 8 < nk; t0 += 8) {
      zd nx[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) nx[u] = FactorLd<FT>::ld(Fcol, rowb, (uint32_t)(min(cbase + (t0 + 8 + u) * ks, clast) * s) * EB);
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int kx = kst + (t0 + u) * ks;
#pragma unroll
        for (int q = 0; q < RC; ++q) acc[q] = zfma(a[u], xin[kx][q], acc[q]);
      }
#pragma unroll
      for (int u = 0; u < 8; ++u) a[u] = nx[u];
    }
    // the last, possibly partial, batch
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (t0 + u < nk) {
        const int kx = kst + (t0 + u) * ks;
#pragma unroll
        for (int q = 0; q < RC; ++q) acc[q] = zfma(a[u], xin[kx][q], acc[q]);
      }
    __syncthreads();
  }
  if (ks > 1) {
    if (kp > 0)
#pragma unroll
      for (int q = 0; q < RC; ++q) red[wave - 1][lane][q] = acc[q];
    __syncthreads();
    if (kp == 0)
      for (int j = 1; j < ks; ++j)
#pragma unroll
        for (int q = 0; q < RC; ++q) acc[q] = zadd(acc[q], red[wave + j - 1][lane][q]);
  }
  if (kp != 0) return;
  if (T.slot >= 0) {  // split task: partial sums, added by k_bwd_red
#pragma unroll
    for (int q = 0; q < RC; ++q)
      if (q < nq) part[((col0 + q) * nslot + T.slot) * 64 + lane] = acc[q];
    return;
  }
  if (rowl < s)
#pragma unroll
    for (int q = 0; q < RC; ++q)
      if (q < nq) xb[(int64_t)(q0 + q) * n + T.fb + rowl] = acc[q];
}

template <int RC>
__global__ __launch_bounds__(256) void k_bwd_red(const int32_t *__restrict__ tasks, FrontArrays A, int nrhs,
                                                 int64_t n, const zd *__restrict__ part, int nslot,
                                                 zd *__restrict__ x, int64_t sx) {
  const int32_t *tk = tasks + 4 * blockIdx.x;
  const int t = tk[0], r0 = tk[1], p0 = tk[2], np = tk[3];
  const int b = blockIdx.y, q0 = blockIdx.z * RC;
  const int lane = threadIdx.x & 63, qg = threadIdx.x >> 6;
  const int s = A.s[t], fb = A.b[t];
  const int nq = min(RC, nrhs - q0);
  const int64_t col0 = (int64_t)b * nrhs + q0;
  const int row = r0 + lane;
  if (row >= s) return;
#pragma unroll
  for (int u = 0; u < (RC + 3) / 4; ++u) {
    const int q = qg + 4 * u;
    if (q >= nq) break;
    const zd *pp = part + ((col0 + q) * nslot + p0) * 64 + lane;
    zd v = zmk(0, 0);
    for (int c = 0; c < np; c += 8) {
      zd h[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) h[i] = pp[(int64_t)min(c + i, np - 1) * 64];
#pragma unroll
      for (int i = 0; i < 8; ++i)
        if (c + i < np) v = zadd(v, h[i]);
    }
    x[(int64_t)b * sx + (int64_t)(q0 + q) * n + fb + row] = v;
  }
}

// RHS columns per workgroup: as many as there are (at most 8) unless the level
// then has fewer than 128 workgroups.  A chunk of fewer columns makes more
// workgroups, but each chunk reads the level's factor again, from another XCD's
// L2 or HBM: with the limit at 1,024 (4 columns, 2 to 4 passes over most levels'
// factors) one light on 8,000 triangles took 387 ms instead of 361, two on 1,500
// 97.9 instead of 93.3, three concurrent solves on 1,000 211 instead of 193; 64
// and 256 measure the same as 128.
static int pick_rc(int nrhs, int64_t tasks, int nb) {
  int rc = 8;
  while (rc > nrhs) rc >>= 1;
  while (rc > 1 && tasks * nb * ((nrhs + rc - 1) / rc) < 128) rc >>= 1;
  return rc;
}

template <int RC, typename FT>
static void launch_fwd(const SolveTasks &T, DevMesh &dm, FrontArrays A, int nb, int nrhs, const FT *inv,
                       const int32_t *gx, const zd *bnew, zd *y, zd *w, zd *part, hipStream_t s, KTime kt) {
  const Symbolic &sy = dm.host.sym;
  const unsigned nz = (unsigned)((nrhs + RC - 1) / RC);
  const int64_t nw = std::max<int64_t>(sy.nw, 1);
  hipExtLaunchKernelGGL(k_fwd<RC, FT>, dim3((unsigned)T.cnt, nb, nz), dim3(256), 0, s, kt.a, kt.b, 0,
                        reinterpret_cast<const SolveTask *>(dm.tasks.p + T.off), dm.cmap.p, inv, dm.isz,
                        reinterpret_cast<const int4 *>(gx), sy.npiv, nrhs, sy.n, nw, bnew, y, w, part,
                        (int)T.nslot, (int)std::min<int64_t>(T.span, INT32_MAX));
  if (T.rcnt > 0)
    hipLaunchKernelGGL(k_fwd_red<RC>, dim3((unsigned)T.rcnt, nb, nz), dim3(256), 0, s, dm.tasks.p + T.roff, A, nrhs,
                       sy.n, nw, part, (int)T.nslot, y, w);
}

template <int RC, typename FT>
static void launch_bwd(const SolveTasks &T, DevMesh &dm, FrontArrays A, int nb, int nrhs, const FT *inv,
                       const zd *y, zd *x, int64_t sx, zd *part, hipStream_t s, KTime kt) {
  const Symbolic &sy = dm.host.sym;
  const unsigned nz = (unsigned)((nrhs + RC - 1) / RC);
  hipExtLaunchKernelGGL(k_bwd<RC, FT>, dim3((unsigned)T.cnt, nb, nz), dim3(256), 0, s, kt.a, kt.b, 0,
                        reinterpret_cast<const SolveTask *>(dm.tasks.p + T.off), dm.uidx.p, inv, dm.isz, nrhs,
                        sy.n, y, x, sx, part, (int)T.nslot, (int)std::min<int64_t>(T.span, INT32_MAX));
  if (T.rcnt > 0)
    hipLaunchKernelGGL(k_bwd_red<RC>, dim3((unsigned)T.rcnt, nb, nz), dim3(256), 0, s, dm.tasks.p + T.roff, A, nrhs,
                       sy.n, part, (int)T.nslot, x, sx);
}

// The top levels of a tree of small fronts (a grating's separators), forward to
// the root and back down, in one launch: a workgroup of 16 waves per instance
// and right-hand side, a wave per 64-row tile, a barrier per level.  These
// launches took 3.2 to 4.2 us each however few tiles they had (a grating of
// 1,990 unknowns at one wavelength 17.9 -> 15.5 ms, at 16 43.0 -> 40.5 ms).  y, x and w are
// written by some waves and read by others after the barrier, so none of their
// pointers is restrict or read-only here.
template <typename FT>
__global__ __launch_bounds__(1024) void k_top(const SolveTask *__restrict__ tasks, TopLevels L,
                                              const int32_t *__restrict__ cmap, const int32_t *__restrict__ uidx,
                                              const FT *__restrict__ inv, int64_t isz, const int4 *__restrict__ gx,
                                              int64_t npiv, int nrhs, int64_t n, int64_t nw, const zd *__restrict__ bv,
                                              zd *y, zd *w, zd *x, int64_t sx) {
  constexpr uint32_t EB = FactorLd<FT>::kBytes;
  constexpr int NB8 = 8;  // factor columns in flight
  const int b = blockIdx.x, q = blockIdx.y;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const zd *bq = bv + ((int64_t)b * nrhs + q) * n;
  zd *yq = y + ((int64_t)b * nrhs + q) * n, *wq = w + ((int64_t)b * nrhs + q) * nw;
  zd *xq = x + (int64_t)b * sx + (int64_t)q * n;
  // acc += F[:, c0 + k] v_k for k = 0..cnt-1, v_k in lane k
  auto columns = [&](__amdgpu_buffer_rsrc_t F, uint32_t rowb, int ld, int c0, int cnt, zd v, zd acc) {
    for (int k = 0; k < cnt; k += NB8) {
      zd a[NB8];
#pragma unroll
      for (int u = 0; u < NB8; ++u) a[u] = FactorLd<FT>::ld(F, rowb, (uint32_t)((c0 + min(k + u, cnt - 1)) * ld) * EB);
#pragma unroll
      for (int u = 0; u < NB8; ++u)
        if (k + u < cnt) acc = zfma(a[u], zmk(__shfl(v.x, k + u, 64), __shfl(v.y, k + u, 64)), acc);
    }
    return acc;
  };
  for (int l = 0; l < L.n; ++l) {
    for (int t = wave; t < L.cnt[0][l]; t += 16) {
      const SolveTask T = tasks[L.off[0][l] + t];
      const int s = T.s, f = T.f, row = T.r0 + lane, rowc = min(row, f - 1);
      const __amdgpu_buffer_rsrc_t F = buf_view(inv + b * isz + T.ioff, (uint32_t)f * (uint32_t)s * EB);
      const int2 cr = reinterpret_cast<const int2 *>(cmap)[T.fvoff + rowc];
      const int4 g = gx[b * npiv + T.pivoff + min(lane, s - 1)];
      zd v = bq[g.x];
      if (g.y >= 0) v = zadd(v, wq[g.y]);
      if (g.z >= 0) v = zadd(v, wq[g.z]);
      zd acc = columns(F, (uint32_t)rowc * EB, f, 0, s, v, zmk(0, 0));
      if (row < s) {
        yq[T.fb + row] = acc;
      } else if (row < f) {
        if (cr.x >= 0) acc = zadd(acc, wq[cr.x]);
        if (cr.y >= 0) acc = zadd(acc, wq[cr.y]);
        wq[T.uoff + (row - s)] = acc;
      }
    }
    __syncthreads();
  }
  for (int l = L.n - 1; l >= 0; --l) {
    for (int t = wave; t < L.cnt[1][l]; t += 16) {
      const SolveTask T = tasks[L.off[1][l] + t];
      const int s = T.s, f = T.f, row = T.r0 + lane;
      const __amdgpu_buffer_rsrc_t F =
          buf_view(inv + b * isz + T.ioff + (int64_t)f * s, (uint32_t)f * (uint32_t)s * EB);
      zd acc = zmk(0, 0);
      for (int kc = T.r0; kc < f; kc += 64) {
        const int k = min(kc + lane, f - 1);
        const zd v = k < s ? yq[T.fb + k] : xq[uidx[T.uoff + k - s]];
        acc = columns(F, (uint32_t)min(row, s - 1) * EB, s, kc, min(64, f - kc), v, acc);
      }
      if (row < s) xq[T.fb + row] = acc;
    }
    __syncthreads();
  }
}

int64_t solve_ws(const DevMesh &dm) { return std::max<int64_t>(dm.host.sym.nw, 1) + dm.part_rhs; }

// The split task lists for the Krylov solves (one block of at most 8
// right-hand sides: the grid has no RHS dimension to fill the GPU with); the
// plain ones for many right-hand sides (dense solves of the cascade), where
// RHS chunks already give a large grid and partial sums would only add
// traffic.
static const SolveTasks &pick_tasks(const SolveTasks *v, int nrhs) { return nrhs <= 8 ? v[1] : v[0]; }

template <typename FT>
static void lu_solve_t(DevMesh &dm, int nb, int nrhs, const FT *inv, const int32_t *gx, const zd *bnew, zd *y,
                       zd *x, zd *w, hipStream_t s, Profiler *prof, int64_t sx) {
  FrontArrays A = fa(dm);
  if (sx < 0) sx = (int64_t)nrhs * dm.host.sym.n;
  const double vecs = (double)nb * nrhs;
  const double fscale = FactorLd<FT>::kBytes / 16.0;  // factor bytes per entry relative to complex128
  // partial sums of split tasks live behind the update vectors in w
  zd *part = w + (int64_t)nb * nrhs * std::max<int64_t>(dm.host.sym.nw, 1);
  // the dense solves' many right-hand sides fill the launches by themselves,
  // and a profile times the levels one by one
  const size_t ntop = prof || nrhs > 8 ? 0 : dm.top.n, nlow = dm.sched.size() - ntop;
  for (size_t l = 0; l < nlow; ++l) {
    const LevelSched &L = dm.sched[l];
    const SolveTasks &T = pick_tasks(L.fwd, nrhs);
    const int rc = pick_rc(nrhs, T.cnt, nb);
    KTime kt = prof ? prof->time(0, L.fwd_mat * fscale * nb + L.fwd_vec * vecs) : KTime{};
    switch (rc) {
      case 8: launch_fwd<8>(T, dm, A, nb, nrhs, inv, gx, bnew, y, w, part, s, kt); break;
      case 4: launch_fwd<4>(T, dm, A, nb, nrhs, inv, gx, bnew, y, w, part, s, kt); break;
      case 2: launch_fwd<2>(T, dm, A, nb, nrhs, inv, gx, bnew, y, w, part, s, kt); break;
      default: launch_fwd<1>(T, dm, A, nb, nrhs, inv, gx, bnew, y, w, part, s, kt); break;
    }
  }
  EMU_LAUNCH_CHECK();
  if (ntop > 0) {
    hipLaunchKernelGGL(k_top<FT>, dim3(nb, nrhs), dim3(1024), 0, s, reinterpret_cast<const SolveTask *>(dm.tasks.p),
                       dm.top, dm.cmap.p, dm.uidx.p, inv, dm.isz, reinterpret_cast<const int4 *>(gx), dm.host.sym.npiv,
                       nrhs, dm.host.sym.n, std::max<int64_t>(dm.host.sym.nw, 1), bnew, y, w, x, sx);
    EMU_LAUNCH_CHECK();
  }
  for (auto it = dm.sched.rbegin() + ntop; it != dm.sched.rend(); ++it) {
    const SolveTasks &T = pick_tasks(it->bwd, nrhs);
    const int rc = pick_rc(nrhs, T.cnt, nb);
    KTime kt = prof ? prof->time(1, it->bwd_mat * fscale * nb + it->bwd_vec * vecs) : KTime{};
    switch (rc) {
      case 8: launch_bwd<8>(T, dm, A, nb, nrhs, inv, y, x, sx, part, s, kt); break;
      case 4: launch_bwd<4>(T, dm, A, nb, nrhs, inv, y, x, sx, part, s, kt); break;
      case 2: launch_bwd<2>(T, dm, A, nb, nrhs, inv, y, x, sx, part, s, kt); break;
      default: launch_bwd<1>(T, dm, A, nb, nrhs, inv, y, x, sx, part, s, kt); break;
    }
  }
  EMU_LAUNCH_CHECK();
}

void lu_solve(DevMesh &dm, int nb, int nrhs, const zd *inv, const int32_t *gx, const zd *bnew, zd *y, zd *x,
              zd *w, hipStream_t s, Profiler *prof, int64_t sx) {
  lu_solve_t<zd>(dm, nb, nrhs, inv, gx, bnew, y, x, w, s, prof, sx);
}

void lu_solve(DevMesh &dm, int nb, int nrhs, const float2 *inv32, const int32_t *gx, const zd *bnew, zd *y, zd *x,
              zd *w, hipStream_t s, Profiler *prof, int64_t sx) {
  lu_solve_t<float2>(dm, nb, nrhs, inv32, gx, bnew, y, x, w, s, prof, sx);
}

// complex64 copy of the inverted factor (round to nearest)
__global__ void k_narrow(int64_t n, const zd *__restrict__ src, float2 *__restrict__ dst) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const zd v = src[i];
    dst[i] = make_float2((float)v.x, (float)v.y);
  }
}

void lu_narrow(const DevMesh &dm, int nb, const zd *inv, float2 *inv32, hipStream_t s) {
  const int64_t n = (int64_t)nb * dm.isz;
  if (n <= 0) return;
  const unsigned g = (unsigned)std::min<int64_t>((n + 255) / 256, 65536);
  hipLaunchKernelGGL(k_narrow, dim3(g), dim3(256), 0, s, n, inv, inv32);
  EMU_LAUNCH_CHECK();
}

// dst[b][c][new] = src[b][c][perm[new]]  (to_new) or dst[b][c][perm[new]] = src[b][c][new]
__global__ void k_permute_vec(int64_t n, int ncol, const int32_t *__restrict__ perm,
                              const zd *__restrict__ src, zd *__restrict__ dst, int to_new) {
  int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  int64_t bc = blockIdx.y;
  if (i >= n) return;
  const zd *sp = src + bc * n;
  zd *dp = dst + bc * n;
  if (to_new) dp[i] = sp[perm[i]];
  else dp[perm[i]] = sp[i];
}

void launch_permute_vec(DevMesh &dm, int nb, int ncol, const zd *src, zd *dst, bool to_new,
                        hipStream_t s) {
  int64_t n = dm.host.neq;
  dim3 g((unsigned)((n + 255) / 256), nb * ncol);
  hipLaunchKernelGGL(k_permute_vec, g, dim3(256), 0, s, n, ncol, dm.perm.p, src, dst, to_new ? 1 : 0);
  EMU_LAUNCH_CHECK();
}

}  // namespace emu
