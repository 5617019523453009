// Dense / vector kernels of the Krylov-Schur eigensolver and of the overlap
// contractions, batched over instances (blockIdx.y / blockIdx.z = instance).
#include <map>
#include <mutex>
#include <string>

#include "engine.h"

namespace emu {

// --------------------------------------------------------------- SpMM (CSR)
// y[b][c][r] = sum_k A[b][r][k] x[b][c][k] for a block of SM_C columns.
// Eight lanes share a row: each lane walks every eighth nonzero (coalesced
// value / index reads, one read of the row per column block), accumulates
// the SM_C column sums, and the eight partial sums are combined with
// cross-lane shuffles; lane j then writes column j.  A wavefront covers 8
// rows, a workgroup 32.  Workgroups are dealt to the 8 XCDs round-robin by
// launch index, so the kernel maps launch index p to row block
// (p % 8) * per + p / 8: each XCD works through one contiguous eighth of the
// rows and, the rows being in nested-dissection order, gathers x from a
// compact range that stays in its own L2 instead of every L2 fetching all of
// x.
constexpr int SM_C = 8;

__device__ __forceinline__ zd shfl_z(zd v, int lane) { return zmk(__shfl(v.x, lane, 64), __shfl(v.y, lane, 64)); }
__device__ __forceinline__ zd shfl_xor_z(zd v, int m) {
  return zmk(__shfl_xor(v.x, m, 64), __shfl_xor(v.y, m, 64));
}

__global__ __launch_bounds__(256) void k_spmm(int64_t n, int ncol, const int64_t *__restrict__ rp,
                                              const int32_t *__restrict__ ci, const zd *__restrict__ vals,
                                              int64_t vstride, const zd *__restrict__ x, int64_t xstride,
                                              zd *__restrict__ y, int64_t ystride, int per) {
  const int lane8 = threadIdx.x & 7;
  const int64_t blk = (int64_t)(blockIdx.x & 7) * per + (blockIdx.x >> 3);
  const int64_t r = blk * 32 + (threadIdx.x >> 3);
  const int b = blockIdx.y;
  const int c0 = blockIdx.z * SM_C;
  const int nc = min(SM_C, ncol - c0);
  const zd *v = vals + b * vstride;
  const zd *xb = x + b * xstride + (int64_t)c0 * n;
  zd acc[SM_C];
#pragma unroll
  for (int c = 0; c < SM_C; ++c) acc[c] = zmk(0, 0);
  const int64_t k0 = r < n ? rp[r] : 0, k1 = r < n ? rp[r + 1] : 0;
  if (k1 > k0) {  // rows >= n and empty rows read nothing
    // The value and column index of the lane's next nonzero are requested
    // before this one's gathers (indices clamped to the row), so each step
    // waits for one round of loads; the gathers are unconditional (clamped
    // column, unused columns multiply zero) so that all are in flight together.
    int64_t k = k0 + lane8;
    const int64_t klast = max(k1 - 1, k0);
    zd a = ld_stream(v + min(k, klast));
    int64_t col = ld_stream(ci + min(k, klast));
    for (; k < k1; k += 8) {
      const zd an = ld_stream(v + min(k + 8, klast));
      const int64_t coln = ld_stream(ci + min(k + 8, klast));
      zd xv[SM_C];
#pragma unroll
      for (int c = 0; c < SM_C; ++c) xv[c] = xb[(int64_t)min(c, nc - 1) * n + col];
      // keep the scheduler from interleaving each gather with its use (it
      // otherwise reuses one register quad and waits for every load in turn)
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int c = 0; c < SM_C; ++c) acc[c] = zfma(c < nc ? a : zmk(0, 0), xv[c], acc[c]);
      a = an;
      col = coln;
    }
  }
#pragma unroll
  for (int c = 0; c < SM_C; ++c) {
    acc[c] = zadd(acc[c], shfl_xor_z(acc[c], 1));
    acc[c] = zadd(acc[c], shfl_xor_z(acc[c], 2));
    acc[c] = zadd(acc[c], shfl_xor_z(acc[c], 4));
  }
  zd out = acc[0];
#pragma unroll
  for (int c = 1; c < SM_C; ++c)
    if (lane8 == c) out = acc[c];
  if (r < n && lane8 < nc) y[b * ystride + (int64_t)(c0 + lane8) * n + r] = out;
}

// ------------------------------------------ SpMM with many columns (modes)
// Post-processing multiplies M (or K - shift M) by all nval mode vectors at
// once.  The mode block is first transposed to row-major (xi[col][c], one
// pass through LDS tiles), so that a nonzero's nval values are one
// contiguous run; a wavefront then owns a row and its lanes the columns
// (lane, lane + 64, ...), reads the row's values and column indices once
// (wave-uniform) and streams the column runs coalesced, four nonzeros at a
// time.  A workgroup's 8 rows are gathered in LDS and written back column by
// column (128-byte runs).  Column chunks of 256 (grid z) bound the LDS tile.
constexpr int SR_ROWS = 8, SR_COLS = 256;

__global__ __launch_bounds__(256) void k_transpose_rm(int64_t n, int ncol, const zd *__restrict__ X, int64_t ldx,
                                                      int64_t sX, zd *__restrict__ xi, int64_t sI) {
  __shared__ zd T[32][33];
  const int b = blockIdx.z;
  const int64_t r0 = (int64_t)blockIdx.x * 32;
  const int c0 = blockIdx.y * 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // 32 x 8
  const zd *x = X + b * sX;
  for (int k = ty; k < 32; k += 8) {
    const int c = c0 + k;
    const int64_t r = r0 + tx;
    if (c < ncol && r < n) T[k][tx] = x[r + (int64_t)c * ldx];
  }
  __syncthreads();
  zd *o = xi + b * sI;
  for (int k = ty; k < 32; k += 8) {
    const int64_t r = r0 + k;
    const int c = c0 + tx;
    if (c < ncol && r < n) o[r * ncol + c] = T[tx][k];
  }
}

__global__ __launch_bounds__(256) void k_spmm_rows(int64_t n, int ncol, const int64_t *__restrict__ rp,
                                                   const int32_t *__restrict__ ci, const zd *__restrict__ vals,
                                                   int64_t vstride, const zd *__restrict__ xi, int64_t sI,
                                                   zd *__restrict__ y, int64_t ldy, int64_t sY) {
  __shared__ zd Ys[SR_ROWS][SR_COLS + 1];
  const int b = blockIdx.y;
  const int c0 = blockIdx.z * SR_COLS;
  const int nc = min(SR_COLS, ncol - c0);
  const int64_t rbase = (int64_t)blockIdx.x * SR_ROWS;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const zd *v = vals + b * vstride;
  const zd *xb = xi + b * sI + c0;
  for (int i = 0; i < SR_ROWS / 4; ++i) {
    const int rr = (SR_ROWS / 4) * w + i;
    const int64_t r = rbase + rr;
    zd acc[SR_COLS / 64];
#pragma unroll
    for (int q = 0; q < SR_COLS / 64; ++q) acc[q] = zmk(0, 0);
    if (r < n) {
      const int64_t k0 = rp[r], k1 = rp[r + 1];
      // four nonzeros per step: their column runs are all requested before
      // the first is used
      for (int64_t kb = k0; kb < k1; kb += 4) {
        zd a[4], xv[4][SR_COLS / 64];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int64_t k = min(kb + u, k1 - 1);
          a[u] = kb + u < k1 ? v[k] : zmk(0, 0);
          const zd *xr = xb + (int64_t)ci[k] * ncol;
#pragma unroll
          for (int q = 0; q < SR_COLS / 64; ++q) xv[u][q] = xr[min(lane + 64 * q, nc - 1)];
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
          for (int q = 0; q < SR_COLS / 64; ++q) acc[q] = zfma(a[u], xv[u][q], acc[q]);
      }
    }
#pragma unroll
    for (int q = 0; q < SR_COLS / 64; ++q) Ys[rr][lane + 64 * q] = acc[q];
  }
  __syncthreads();
  zd *yb = y + b * sY + (int64_t)c0 * ldy;
  for (int idx = tid; idx < SR_ROWS * nc; idx += 256) {
    const int c = idx / SR_ROWS, rr = idx % SR_ROWS;
    const int64_t r = rbase + rr;
    if (r < n) yb[(int64_t)c * ldy + r] = Ys[rr][c];
  }
}

void launch_spmm(int nb, int64_t n, int ncol, const int64_t *rp, const int32_t *ci, const zd *vals,
                 int64_t vstride, const zd *x, int64_t xstride, zd *y, int64_t ystride, hipStream_t s, KTime kt,
                 zd *xi) {
  if (xi && ncol > 8) {  // many columns: row-major copy, then one wavefront per row
    dim3 gt((unsigned)((n + 31) / 32), (unsigned)((ncol + 31) / 32), nb);
    hipLaunchKernelGGL(k_transpose_rm, gt, dim3(256), 0, s, n, ncol, x, n, xstride, xi, n * ncol);
    EMU_LAUNCH_CHECK();
    dim3 g((unsigned)((n + SR_ROWS - 1) / SR_ROWS), nb, (unsigned)((ncol + SR_COLS - 1) / SR_COLS));
    hipExtLaunchKernelGGL(k_spmm_rows, g, dim3(256), 0, s, kt.a, kt.b, 0, n, ncol, rp, ci, vals, vstride, xi,
                          n * ncol, y, n, ystride);
    EMU_LAUNCH_CHECK();
    return;
  }
  // 8 * per launch indices cover the (n + 31) / 32 row blocks; rows >= n idle
  const int per = (int)(((n + 31) / 32 + 7) / 8);
  dim3 g((unsigned)(8 * per), nb, (unsigned)((ncol + SM_C - 1) / SM_C));
  hipExtLaunchKernelGGL(k_spmm, g, dim3(256), 0, s, kt.a, kt.b, 0, n, ncol, rp, ci, vals, vstride, x, xstride, y,
                        ystride, per);
  EMU_LAUNCH_CHECK();
}


// ------------------------------------------- SpMM on a row-interleaved block
// The Krylov loop multiplies M by one B-column block per step.  Gathering
// x[col] of B columns stored n apart touches B cache lines per nonzero; with
// the block stored row-interleaved (xi[B col + c]) the B values of a nonzero's
// column are one run (a 128-byte line at B = 8), read whole.  The block is
// interleaved by k_trmm_right as it is written, or by one pass
// (k_interleave, 2 x 16 n bytes per column block) before the product.
template <int B>
__global__ __launch_bounds__(256) void k_interleave(int64_t n, const zd *__restrict__ X, int64_t sX,
                                                    zd *__restrict__ xi, int64_t sI) {
  const int64_t r = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  const int b = blockIdx.y;
  if (r >= n) return;
  const zd *x = X + b * sX;
  zd v[B];
#pragma unroll
  for (int c = 0; c < B; ++c) v[c] = ld_stream(x + (int64_t)c * n + r);
  zd *o = xi + b * sI + B * r;
#pragma unroll
  for (int c = 0; c < B; ++c) o[c] = v[c];
}

template <int B>
__global__ __launch_bounds__(256) void k_spmm_il(int64_t n, const int64_t *__restrict__ rp,
                                                 const int32_t *__restrict__ ci, const zd *__restrict__ vals,
                                                 int64_t vstride, const zd *__restrict__ xi, int64_t xstride,
                                                 zd *__restrict__ y, int64_t ystride, int per) {
  // Eight lanes share a row.  Per step the group takes the row's next eight
  // nonzeros (lane j loads value and column of nonzero j, coalesced).  B = 8:
  // lane c owns output column c and for each of the nonzeros loads x[col][c]:
  // the group reads one 128-byte line per nonzero, eight lines per wavefront
  // load, and accumulates without a final cross-lane reduction.  B < 8: the
  // lanes are 8 / B sets of B columns, each set takes every (8 / B)-th nonzero,
  // and the sets' sums are added at the end.
  constexpr int NS = 8 / B;
  const int lane8 = threadIdx.x & 7, col8 = lane8 % B, set = lane8 / B;
  const int gbase = threadIdx.x & 63 & ~7;  // first lane of the group in the wavefront
  const int64_t blk = (int64_t)(blockIdx.x & 7) * per + (blockIdx.x >> 3);
  const int64_t r = blk * 32 + (threadIdx.x >> 3);
  const int b = blockIdx.y;
  const zd *v = vals + b * vstride;
  const zd *xb = xi + b * xstride;
  zd acc = zmk(0, 0);
  const int64_t k0 = r < n ? rp[r] : 0, k1 = r < n ? rp[r + 1] : 0;
  for (int64_t kb = k0; kb < k1; kb += 8) {
    const int64_t k = kb + lane8;
    const bool ok = k < k1;
    const int64_t kc = ok ? k : k1 - 1;
    zd a = ld_stream(v + kc);
    const int col = ld_stream(ci + kc);
    if (!ok) a = zmk(0, 0);
    const int cnt = (int)min((int64_t)8, k1 - kb);
    zd xv[B], av[B];
#pragma unroll
    for (int q = 0; q < B; ++q) {
      const int src = gbase + NS * q + set;
      const int cq = __shfl(col, src, 64);
      av[q] = zmk(__shfl(a.x, src, 64), __shfl(a.y, src, 64));
      xv[q] = xb[B * (int64_t)cq + col8];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < B; ++q)
      if (NS * q + set < cnt) acc = zfma(av[q], xv[q], acc);
  }
#pragma unroll
  for (int m = B; m < 8; m *= 2) acc = zadd(acc, shfl_xor_z(acc, m));
  if (r < n && set == 0) y[b * ystride + (int64_t)col8 * n + r] = acc;
}

void launch_spmm_il(int nb, int64_t n, int bq, const int64_t *rp, const int32_t *ci, const zd *vals, int64_t vstride,
                    const zd *x, int64_t xstride, zd *xi, zd *y, int64_t ystride, hipStream_t s, KTime kt,
                    bool xi_ready) {
  const int per = (int)(((n + 31) / 32 + 7) / 8);
  const dim3 gi((unsigned)((n + 255) / 256), nb), g((unsigned)(8 * per), nb);
#define EMU_SPMM_IL(B)                                                                                               \
  do {                                                                                                               \
    if (!xi_ready) hipLaunchKernelGGL(k_interleave<B>, gi, dim3(256), 0, s, n, x, xstride, xi, B * n);               \
    hipExtLaunchKernelGGL(k_spmm_il<B>, g, dim3(256), 0, s, kt.a, kt.b, 0, n, rp, ci, vals, vstride, xi, B * n, y,   \
                          ystride, per);                                                                             \
  } while (0)
  switch (bq) {
    case 2: EMU_SPMM_IL(2); break;
    case 4: EMU_SPMM_IL(4); break;
    case 8: EMU_SPMM_IL(8); break;
    default: throw HipError("spmm_il: block size must be 2, 4 or 8");
  }
#undef EMU_SPMM_IL
  EMU_LAUNCH_CHECK();
}

typedef double v4d __attribute__((ext_vector_type(4)));

// -------------------------------- C = op(A)^T B, wide, on the matrix cores
// Mode overlaps and plane-wave contractions: M, N of tens to hundreds, K the
// DOF count.  A workgroup owns a 64 x 64 output tile and one K chunk; per
// 32-row step it stages the 32 x 64 tiles of A and B in LDS (the next pair is
// fetched into registers meanwhile), and wave w accumulates output columns
// 16 w .. 16 w + 15 against all 64 rows with FP64 16x16x4 MFMAs (four real
// products per complex one).  Partials per chunk: part[b][chunk][n][m].
template <bool CONJ>
__global__ __launch_bounds__(256) void k_atb_mfma_wide(int64_t K, int M, int N, int64_t kchunk,
                                                       const zd *__restrict__ A, int64_t lda, int64_t sA,
                                                       const zd *__restrict__ B, int64_t ldb, int64_t sB,
                                                       zd *__restrict__ part, int tilesM) {
  constexpr int TT = 64, TK = 32;
  // The output tiles of one (K chunk, instance) read the same rows of A and
  // B: the linear workgroup id is renumbered (a bijection of [0, T)) so that
  // each of the 8 XCDs, which take workgroups round-robin and have an L2
  // each, runs a contiguous range of the tile order.
  const unsigned T = gridDim.x * gridDim.y * gridDim.z;
  const unsigned Lin = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
  const unsigned xcd = Lin & 7u, q8 = T >> 3, r8 = T & 7u;
  const unsigned Lg = xcd * q8 + min(xcd, r8) + (Lin >> 3);
  const int bx = (int)(Lg % gridDim.x);
  const int tm = bx % tilesM, tn = bx / tilesM;
  const int m0 = tm * TT, n0 = tn * TT;
  const int chunk = (int)((Lg / gridDim.x) % gridDim.y), nchunk = gridDim.y;
  const int b = (int)(Lg / (gridDim.x * gridDim.y));
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const zd *Ab = A + b * sA;
  const zd *Bb = B + b * sB;
  __shared__ zd As[TK][TT + 1];
  __shared__ zd Bs[TK][TT + 1];
  const int64_t kb = chunk * kchunk, ke = min(K, kb + kchunk);
  const int lr = tid & 31, lc = tid >> 5;  // staging: row lr, columns lc + 8 i
  zd ra[8], rb[8];
  auto fetch = [&](int64_t k0) {
    const int64_t k = k0 + lr;
    const int64_t kc = k < ke ? k : ke - 1;
#pragma unroll
    for (int i = 0; i < 8; ++i) ra[i] = Ab[kc + (int64_t)min(m0 + lc + 8 * i, M - 1) * lda];
#pragma unroll
    for (int i = 0; i < 8; ++i) rb[i] = Bb[kc + (int64_t)min(n0 + lc + 8 * i, N - 1) * ldb];
  };
  v4d pr[4], pi[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    pr[t] = (v4d){0, 0, 0, 0};
    pi[t] = (v4d){0, 0, 0, 0};
  }
  if (kb < ke) fetch(kb);
  const int fi = lane & 15, fk = lane >> 4;
  for (int64_t k0 = kb; k0 < ke; k0 += TK) {
    __syncthreads();
    const bool okk = k0 + lr < ke;
#pragma unroll
    for (int i = 0; i < 8; ++i) As[lr][lc + 8 * i] = (okk && m0 + lc + 8 * i < M) ? ra[i] : zmk(0, 0);
#pragma unroll
    for (int i = 0; i < 8; ++i) Bs[lr][lc + 8 * i] = (okk && n0 + lc + 8 * i < N) ? rb[i] : zmk(0, 0);
    __syncthreads();
    if (k0 + TK < ke) fetch(k0 + TK);
#pragma unroll
    for (int ks = 0; ks < TK / 4; ++ks) {
      const int kk = ks * 4 + fk;
      const zd xb = Bs[kk][16 * wv + fi];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const zd va = As[kk][16 * t + fi];
        pr[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(va.x, xb.x, pr[t], 0, 0, 0);
        pi[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(va.x, xb.y, pi[t], 0, 0, 0);
      }
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const zd va = As[kk][16 * t + fi];
        // CONJ: Re += ar br + ai bi, Im += ar bi - ai br
        pr[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(CONJ ? va.y : -va.y, xb.y, pr[t], 0, 0, 0);
        pi[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(CONJ ? -va.y : va.y, xb.x, pi[t], 0, 0, 0);
      }
    }
  }
  const int nn = n0 + 16 * wv + fi;
  if (nn < N) {
    zd *pp = part + (((int64_t)b * nchunk + chunk) * N + nn) * M;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = m0 + 16 * t + fk + 4 * r;
        if (m < M) pp[m] = zmk(pr[t][r], pi[t][r]);
      }
  }
}

// ------------------------------------------ C = op(A)^T b for one vector
// The Gram-Schmidt projection h = V^H w: A (K x M) is the Krylov basis, read
// once from HBM; B is the new vector.  A workgroup owns 64 columns of A and one
// K chunk.  Per 32-row step it stages the 32 x 64 tile of A (read along the
// rows, coalesced) and 32 values of B in LDS; lane c of each wave then
// accumulates column c over the rows of its wave (rows w, w + 4, ...).  The next
// tile is fetched into registers while the current one is used.  At the end the
// four waves' sums are combined in LDS and written as the chunk's partial
// product, added by k_atb_reduce or k_cgs_sub.
__global__ __launch_bounds__(256) void k_atb_tall(int64_t K, int M, int64_t kchunk, const zd *__restrict__ A,
                                                  int64_t lda, int64_t sA, const zd *__restrict__ B, int64_t sB,
                                                  int conjA, zd *__restrict__ part) {
  constexpr int TM = 64, TK = 32;
  const int m0 = blockIdx.x * TM;
  const int chunk = blockIdx.y, nchunk = gridDim.y;
  const int b = blockIdx.z;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const zd *Ab = A + b * sA;
  const zd *Bb = B + b * sB;
  __shared__ zd As[TK][TM + 1];
  __shared__ zd Bs[TK];
  const int64_t kb = chunk * kchunk, ke = min(K, kb + kchunk);
  const int lr = tid % TK, lc = tid / TK;  // staging: row lr, columns lc + 8 i
  zd ra[8], rb;
  // Loads are unconditional from clamped (in-range) addresses, and the
  // out-of-range values are zeroed afterwards: a load inside a branch makes
  // the compiler wait for it before the branch merges, which serialises the
  // tile's loads instead of keeping them all in flight.
  auto fetch = [&](int64_t k0) {
    const int64_t k = k0 + lr;
    const bool okk = k < ke;
    const int64_t kc = okk ? k : ke - 1;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int m = m0 + lc + 8 * i;
      const zd v = Ab[kc + (int64_t)min(m, M - 1) * lda];
      ra[i] = (okk && m < M) ? v : zmk(0, 0);
    }
    const zd v = Bb[kc];
    rb = okk ? v : zmk(0, 0);
  };
  zd acc = zmk(0, 0);
  if (kb < ke) fetch(kb);
  for (int64_t k0 = kb; k0 < ke; k0 += TK) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 8; ++i) As[lr][lc + 8 * i] = conjA ? zconj(ra[i]) : ra[i];
    if (lc == 0) Bs[lr] = rb;
    __syncthreads();
    if (k0 + TK < ke) fetch(k0 + TK);
#pragma unroll
    for (int kk = wv; kk < TK; kk += 4) acc = zfma(As[kk][lane], Bs[kk], acc);
  }
  __syncthreads();
  zd *red = &As[0][0];
  red[wv * 64 + lane] = acc;
  __syncthreads();
  if (wv == 0 && m0 + lane < M)
    part[((int64_t)b * nchunk + chunk) * M + m0 + lane] =
        zadd(zadd(zadd(acc, red[64 + lane]), red[128 + lane]), red[192 + lane]);
}

// Exchange two equal ranges (the data of two batch slots).
template <typename T>
__global__ __launch_bounds__(256) void k_swap(int64_t n, T *__restrict__ a, T *__restrict__ b) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const T t = a[i];
    a[i] = b[i];
    b[i] = t;
  }
}

void launch_swap(int64_t n, zd *a, zd *b, hipStream_t s) {
  if (n <= 0 || a == b) return;
  const unsigned g = (unsigned)std::min<int64_t>((n + 255) / 256, 65536);
  hipLaunchKernelGGL(k_swap<zd>, dim3(g), dim3(256), 0, s, n, a, b);
  EMU_LAUNCH_CHECK();
}

void launch_swap_f2(int64_t n, float2 *a, float2 *b, hipStream_t s) {
  if (n <= 0 || a == b) return;
  const unsigned g = (unsigned)std::min<int64_t>((n + 255) / 256, 65536);
  hipLaunchKernelGGL(k_swap<float2>, dim3(g), dim3(256), 0, s, n, a, b);
  EMU_LAUNCH_CHECK();
}

void launch_swap_i32(int64_t n, int32_t *a, int32_t *b, hipStream_t s) {
  if (n <= 0 || a == b) return;
  const unsigned g = (unsigned)std::min<int64_t>((n + 255) / 256, 65536);
  hipLaunchKernelGGL(k_swap<int32_t>, dim3(g), dim3(256), 0, s, n, a, b);
  EMU_LAUNCH_CHECK();
}


// The projection of the delayed Gram-Schmidt on the matrix cores: A^H B with B
// of N <= 16 columns (padded with zeros to 16), as four real
// v_mfma_f64_16x16x4f64 per 16 x 16 x 4 complex block (real and imaginary
// parts).  A workgroup stages a 32-row x 64-column tile of A and the 32 x 16
// tile of B in LDS (as k_atb_tall); wave w multiplies rows 8w .. 8w + 7 of the
// tile (two k-steps of 4) into four 16 x 16 output tiles, and the waves' sums
// are added through LDS at the end (one partial per K chunk, added by
// k_atb_reduce).  Fragment layouts (FP64 16x16x4): A[i][k] in lane i + 16 k,
// B[k][j] in lane j + 16 k, D[i][j] in lane j + 16 (i % 4), register i / 4.
// three waves per SIMD (164 registers, no spills): more loads in flight
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3, 3)))
void k_atb_mfma16(int64_t K, int M, int N, int64_t kchunk, const zd *__restrict__ A, int64_t lda, int64_t sA,
                  const zd *__restrict__ B, int64_t ldb, int64_t sB, zd *__restrict__ part) {
  constexpr int TM = 64, TK = 32, NQ = 16;
  // The column tiles of one (K chunk, instance) all read the same rows of B.
  // Workgroups go to the 8 XCDs round-robin by linear id, each XCD with its
  // own L2, so the linear id is renumbered to give consecutive tiles to one
  // XCD (XCD x takes a contiguous range of the tile order, in order): B's
  // rows are then fetched from HBM once per chunk instead of once per tile.
  // The renumbering is a bijection of [0, T) whatever the hardware's
  // placement, so it affects only locality.
  const unsigned T = gridDim.x * gridDim.y * gridDim.z;
  const unsigned Lin = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
  const unsigned xcd = Lin & 7u, q = T >> 3, r = T & 7u;
  const unsigned Lg = xcd * q + min(xcd, r) + (Lin >> 3);
  const int m0 = (int)(Lg % gridDim.x) * TM;
  const int chunk = (int)((Lg / gridDim.x) % gridDim.y), nchunk = gridDim.y;
  const int b = (int)(Lg / (gridDim.x * gridDim.y));
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const zd *Ab = A + b * sA;
  const zd *Bb = B + b * sB;
  __shared__ zd As[TK][TM + 1];
  __shared__ zd Bs[TK][NQ + 1];
  const int64_t kb = chunk * kchunk, ke = min(K, kb + kchunk);
  const int lr = tid & 31, lc = tid >> 5;  // staging: row lr, columns lc + 8 i
  zd ra[8], rb[2];
  // unconditional loads from clamped addresses (see k_atb_tall); the
  // out-of-range values are zeroed when they are stored to LDS, not here: a
  // select right after the load would make the wave wait for the prefetch
  // before the matrix-core phase instead of during it
  auto fetch = [&](int64_t k0) {
    const int64_t k = k0 + lr;
    const int64_t kc = k < ke ? k : ke - 1;
#pragma unroll
    for (int i = 0; i < 8; ++i) ra[i] = Ab[kc + (int64_t)min(m0 + lc + 8 * i, M - 1) * lda];
#pragma unroll
    for (int i = 0; i < 2; ++i) rb[i] = Bb[kc + (int64_t)min(lc + 8 * i, N - 1) * ldb];
  };
  v4d pr[4], pi[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    pr[t] = (v4d){0, 0, 0, 0};
    pi[t] = (v4d){0, 0, 0, 0};
  }
  if (kb < ke) fetch(kb);
  const int fi = lane & 15, fk = lane >> 4;
  for (int64_t k0 = kb; k0 < ke; k0 += TK) {
    __syncthreads();
    const bool okk = k0 + lr < ke;
#pragma unroll
    for (int i = 0; i < 8; ++i) As[lr][lc + 8 * i] = (okk && m0 + lc + 8 * i < M) ? ra[i] : zmk(0, 0);
#pragma unroll
    for (int i = 0; i < 2; ++i) Bs[lr][lc + 8 * i] = (okk && lc + 8 * i < N) ? rb[i] : zmk(0, 0);
    __syncthreads();
    if (k0 + TK < ke) fetch(k0 + TK);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const int kk = wv * 8 + ks * 4 + fk;
      const zd xb = Bs[kk][fi];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const zd va = As[kk][16 * t + fi];
        // conjugated: Re += ar br + ai bi, Im += ar bi - ai br
        pr[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(va.x, xb.x, pr[t], 0, 0, 0);
        pr[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(va.y, xb.y, pr[t], 0, 0, 0);
        pi[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(va.x, xb.y, pi[t], 0, 0, 0);
        pi[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(-va.y, xb.x, pi[t], 0, 0, 0);
      }
    }
  }
  // the four waves' sums, one output tile at a time through As (wave, register,
  // lane: 1,024 of its 2,080 entries)
  zd *red = &As[0][0];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; ++i) red[(wv * 4 + i) * 64 + lane] = zmk(pr[t][i], pi[t][i]);
    __syncthreads();
    // thread (register wv, lane) adds the waves' values of that entry
    zd sum = red[wv * 64 + lane];
#pragma unroll
    for (int w = 1; w < 4; ++w) sum = zadd(sum, red[(w * 4 + wv) * 64 + lane]);
    const int m = m0 + 16 * t + fk + 4 * wv;
    if (m < M && fi < N) part[(((int64_t)b * nchunk + chunk) * N + fi) * M + m] = sum;
  }
}

// C[b][m + nn ldc] = sum over chunks of part[b][chunk][nn][m]: 64 outputs per
// workgroup, its four waves summing every fourth chunk, combined in LDS.
__global__ __launch_bounds__(256) void k_atb_reduce(int M, int N, int nchunk, const zd *__restrict__ part,
                                                    zd *__restrict__ C, int64_t ldc, int64_t sC) {
  __shared__ zd red[4][64];
  const int b = blockIdx.y;
  const int lane = threadIdx.x & 63, g = threadIdx.x >> 6;
  const int64_t idx = blockIdx.x * 64ll + lane, tot = (int64_t)M * N;
  zd acc = zmk(0, 0);
  if (idx < tot)
    for (int c = g; c < nchunk; c += 4) acc = zadd(acc, part[((int64_t)b * nchunk + c) * tot + idx]);
  red[g][lane] = acc;
  __syncthreads();
  if (g == 0 && idx < tot) {
    const int m = (int)(idx % M), nn = (int)(idx / M);
    C[b * sC + m + (int64_t)nn * ldc] = zadd(zadd(red[0][lane], red[1][lane]), zadd(red[2][lane], red[3][lane]));
  }
}

// Partial products A^H b of the K chunks (part[b][chunk][M]), at most `most`
// chunks; returns their number.
static int atb_partials(int nb, int64_t K, int M, const zd *A, int64_t lda, int64_t sA, const zd *B, int64_t sB,
                        bool conjA, int64_t most, zd *scratch, size_t scratch_elems, hipStream_t s,
                        KTime kt) {
  const int kstep = 32;
  const int tiles = (M + 63) / 64;
  const int64_t per = (int64_t)nb * M;
  const int64_t maxchunk = std::max<int64_t>(1, (int64_t)(scratch_elems / std::max<int64_t>(per, 1)));
  const int64_t want = std::max<int64_t>(1, 2048 / std::max(1, tiles * nb));
  int64_t nchunk = std::min<int64_t>(std::min<int64_t>(want, maxchunk), (K + kstep - 1) / kstep);
  nchunk = std::max<int64_t>(1, std::min<int64_t>(nchunk, most));
  int64_t kchunk = (K + nchunk - 1) / nchunk;
  kchunk = ((kchunk + kstep - 1) / kstep) * kstep;
  nchunk = (K + kchunk - 1) / kchunk;
  if ((size_t)(nchunk * per) > scratch_elems) throw HipError("atb: scratch too small");
  hipExtLaunchKernelGGL(k_atb_tall, dim3((unsigned)tiles, (unsigned)nchunk, nb), dim3(256), 0, s, kt.a, kt.b, 0, K, M,
                        kchunk, A, lda, sA, B, sB, conjA ? 1 : 0, scratch);
  EMU_LAUNCH_CHECK();
  return (int)nchunk;
}

void launch_atb(int nb, int64_t K, int M, int N, const zd *A, int64_t lda, int64_t sA, const zd *B,
                int64_t ldb, int64_t sB, zd *C, int64_t ldc, int64_t sC, bool conjA, zd *scratch,
                size_t scratch_elems, hipStream_t s, KTime kt) {
  if (M <= 0 || N <= 0 || nb <= 0) return;
  const bool tall = N == 1;
  if (!tall) {  // wide products (mode overlaps, J contractions): 64 x 64 MFMA tiles, split over K
    const int tilesM = (M + 63) / 64, tiles = tilesM * ((N + 63) / 64);
    const int64_t per = (int64_t)nb * M * N;
    const int64_t maxchunk = std::max<int64_t>(1, (int64_t)(scratch_elems / std::max<int64_t>(per, 1)));
    const int64_t want = std::max<int64_t>(1, 2048 / std::max(1, tiles * nb));
    int64_t nchunk = std::min<int64_t>(std::min<int64_t>(want, maxchunk), (K + 31) / 32);
    nchunk = std::max<int64_t>(1, std::min<int64_t>(nchunk, 65535));
    int64_t kchunk = (K + nchunk - 1) / nchunk;
    kchunk = ((kchunk + 31) / 32) * 32;
    nchunk = (K + kchunk - 1) / kchunk;
    if ((size_t)(nchunk * per) > scratch_elems) throw HipError("atb: scratch too small");
    // the kernel renumbers the linear id of the whole grid in 32 bits
    if ((int64_t)tiles * nchunk * nb > 0xffffffffLL) throw HipError("atb: grid too large");
    dim3 g((unsigned)tiles, (unsigned)nchunk, nb);
    if (conjA)
      hipLaunchKernelGGL(k_atb_mfma_wide<true>, g, dim3(256), 0, s, K, M, N, kchunk, A, lda, sA, B, ldb, sB, scratch,
                         tilesM);
    else
      hipLaunchKernelGGL(k_atb_mfma_wide<false>, g, dim3(256), 0, s, K, M, N, kchunk, A, lda, sA, B, ldb, sB,
                         scratch, tilesM);
    EMU_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_atb_reduce, dim3((unsigned)((per / nb + 63) / 64), nb), dim3(256), 0, s, M, N, (int)nchunk,
                       scratch, C, ldc, sC);
    EMU_LAUNCH_CHECK();
    return;
  }
  const int nchunk = atb_partials(nb, K, M, A, lda, sA, B, sB, conjA, 256, scratch, scratch_elems, s, kt);
  hipLaunchKernelGGL(k_atb_reduce, dim3((unsigned)((M + 63) / 64), nb), dim3(256), 0, s, M, N, nchunk, scratch, C, ldc,
                     sC);
  EMU_LAUNCH_CHECK();
}


// The delayed Gram-Schmidt projection: C[b] (M x N) = A[b]^H B[b] for N <= 16
// on the matrix cores.  K is cut into enough chunks for about 2,048
// workgroups, but at least 128 rows each: every chunk writes M x N partial
// sums, which at 32 rows per chunk (n = 6,072, 2 instances) were more bytes
// than the basis itself.
void launch_proj(int nb, int64_t K, int M, int N, const zd *A, int64_t lda, int64_t sA, const zd *B, int64_t ldb,
                 int64_t sB, zd *C, int64_t ldc, int64_t sC, zd *scratch, size_t scratch_elems, hipStream_t s, KTime kt) {
  if (N > 16) throw HipError("proj: at most 16 columns");
  const int tiles = (M + 63) / 64;
  const int64_t per = (int64_t)nb * M * N;
  int64_t nchunk = std::max<int64_t>(1, 2048 / std::max(1, tiles * nb));
  nchunk = std::min<int64_t>({nchunk, (int64_t)(scratch_elems / std::max<int64_t>(per, 1)), (K + 127) / 128, 256});
  nchunk = std::max<int64_t>(1, nchunk);
  int64_t kchunk = (K + nchunk - 1) / nchunk;
  kchunk = ((kchunk + 31) / 32) * 32;
  nchunk = (K + kchunk - 1) / kchunk;
  if ((size_t)(nchunk * per) > scratch_elems) throw HipError("proj: scratch too small");
  // the kernel renumbers the linear id of the whole grid in 32 bits
  if ((int64_t)tiles * nchunk * nb > 0xffffffffLL) throw HipError("proj: grid too large");
  hipExtLaunchKernelGGL(k_atb_mfma16, dim3((unsigned)tiles, (unsigned)nchunk, nb), dim3(256), 0, s, kt.a, kt.b, 0, K, M,
                        N, kchunk, A, lda, sA, B, ldb, sB, scratch);
  EMU_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_atb_reduce, dim3((unsigned)(((int64_t)M * N + 63) / 64), nb), dim3(256), 0, s, M, N,
                     (int)nchunk, scratch, C, ldc, sC);
  EMU_LAUNCH_CHECK();
}

// ------------------------------------------------ C = alpha A B + beta C (NN)
// Batched complex GEMM on the FP64 matrix cores, for the restart combination
// V Q, the Ritz vectors V W, H S in the delayed Gram-Schmidt and the
// star-product cascade.  A workgroup owns a 64 x 64 tile of C; per 16-deep K
// step it stages the 64 x 16 tile of A (loaded along the columns of A,
// coalesced) and the 16 x 64 tile of B in LDS (33 KB, four workgroups per
// CU), and wave w accumulates the 64 x 16 slice of columns 16 w .. 16 w + 15
// with 16x16x4 FP64 MFMAs (four real products per complex one, the two
// products of each accumulator issued apart).  The next pair of tiles is fetched into
// registers while the current one is multiplied.  Launch order runs the N
// tiles of one M tile next to each other, so A's rows are shared in L2.
template <bool BETA>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3, 3)))
void k_zgemm_nn(int64_t M, int N, int K, zd alpha, const zd *__restrict__ A,
                                                  int64_t lda, int64_t sA, const zd *__restrict__ B, int64_t ldb,
                                                  int64_t sB, zd beta, zd *__restrict__ C, int64_t ldc, int64_t sC,
                                                  int tilesN) {
  constexpr int TT = 64, TK = 16;
  const int64_t tm = blockIdx.x / tilesN;
  const int tn = blockIdx.x % tilesN;
  const int64_t m0 = tm * TT;
  const int n0 = tn * TT;
  const int b = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const zd *Ab = A + b * sA;
  const zd *Bb = B + b * sB;
  __shared__ zd As[TK][TT + 1];
  __shared__ zd Bs[TK][TT + 1];
  // A tile: row am = tid & 63 of the tile, K columns ak + 4 i; B tile: K row
  // bk = tid & 15, columns bn + 16 i
  const int am = tid & 63, ak = tid >> 6;
  const int bk = tid & 15, bn = tid >> 4;
  const int64_t arow = min(m0 + am, M - 1);
  zd ra[4], rb[4];
  auto fetch = [&](int k0) {
#pragma unroll
    for (int i = 0; i < 4; ++i) ra[i] = Ab[arow + (int64_t)min(k0 + ak + 4 * i, K - 1) * lda];
    const int kb = min(k0 + bk, K - 1);
#pragma unroll
    for (int i = 0; i < 4; ++i) rb[i] = Bb[kb + (int64_t)min(n0 + bn + 16 * i, N - 1) * ldb];
  };
  v4d pr[4], pi[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    pr[t] = (v4d){0, 0, 0, 0};
    pi[t] = (v4d){0, 0, 0, 0};
  }
  fetch(0);
  const int fi = lane & 15, fk = lane >> 4;
  for (int k0 = 0; k0 < K; k0 += TK) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int kk = ak + 4 * i;
      As[kk][am] = (k0 + kk < K && m0 + am < M) ? ra[i] : zmk(0, 0);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) Bs[bk][bn + 16 * i] = (k0 + bk < K && n0 + bn + 16 * i < N) ? rb[i] : zmk(0, 0);
    __syncthreads();
    if (k0 + TK < K) fetch(k0 + TK);
#pragma unroll
    for (int ks = 0; ks < TK / 4; ++ks) {
      const int kk = ks * 4 + fk;
      const zd xb = Bs[kk][16 * wv + fi];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const zd va = As[kk][16 * t + fi];
        pr[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(va.x, xb.x, pr[t], 0, 0, 0);
        pi[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(va.x, xb.y, pi[t], 0, 0, 0);
      }
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const zd va = As[kk][16 * t + fi];
        pr[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(-va.y, xb.y, pr[t], 0, 0, 0);
        pi[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(va.y, xb.x, pi[t], 0, 0, 0);
      }
    }
  }
  const int nn = n0 + 16 * wv + fi;
  if (nn >= N) return;
  zd *Cb = C + b * sC + (int64_t)nn * ldc;
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int64_t m = m0 + 16 * t + fk + 4 * r;
      if (m < M) {
        zd v = zmul(alpha, zmk(pr[t][r], pi[t][r]));
        if (BETA) v = zfma(beta, Cb[m], v);
        Cb[m] = v;
      }
    }
}

// Tall products (M = the DOF count: restart combination, Ritz vectors): a
// 128 x 64 tile per workgroup, waves in a 2 x 2 grid of 64 x 32 slices, so
// that every A fragment read from LDS feeds two column blocks (six LDS reads
// per 32 MFMAs instead of five per 16) and B is staged once per 128 rows.
template <bool BETA>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2)))
void k_zgemm_nn_tall(int64_t M, int N, int K, zd alpha, const zd *__restrict__ A,
                                                       int64_t lda, int64_t sA, const zd *__restrict__ B,
                                                       int64_t ldb, int64_t sB, zd beta, zd *__restrict__ C,
                                                       int64_t ldc, int64_t sC, int tilesN) {
  constexpr int TM = 128, TN = 64, TK = 16;
  // The tilesN column tiles of a row tile read the same 128 rows of A: the
  // linear workgroup id is renumbered (a bijection of [0, T)) so that each
  // of the 8 XCDs, which take workgroups round-robin and have an L2 each,
  // runs a contiguous range of the tile order, row tile by row tile.
  const unsigned T = gridDim.x * gridDim.y;
  const unsigned Lin = blockIdx.x + gridDim.x * blockIdx.y;
  const unsigned xcd = Lin & 7u, q = T >> 3, r = T & 7u;
  const unsigned Lg = xcd * q + min(xcd, r) + (Lin >> 3);
  const unsigned bx = Lg % gridDim.x;
  const int64_t tm = bx / tilesN;
  const int tn = bx % tilesN;
  const int64_t m0 = tm * TM;
  const int n0 = tn * TN;
  const int b = (int)(Lg / gridDim.x);
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int wm = wv & 1, wn = wv >> 1;
  const zd *Ab = A + b * sA;
  const zd *Bb = B + b * sB;
  __shared__ zd As[TK][TM + 1];
  __shared__ zd Bs[TK][TN + 1];
  // A tile: row am = tid & 127, K columns ak + 2 i; B tile: K row bk =
  // tid & 15, columns bn + 16 i
  const int am = tid & 127, ak = tid >> 7;
  const int bk = tid & 15, bn = tid >> 4;
  const int64_t arow = min(m0 + am, M - 1);
  zd ra[8], rb[4];
  auto fetch = [&](int k0) {
#pragma unroll
    for (int i = 0; i < 8; ++i) ra[i] = Ab[arow + (int64_t)min(k0 + ak + 2 * i, K - 1) * lda];
    const int kb = min(k0 + bk, K - 1);
#pragma unroll
    for (int i = 0; i < 4; ++i) rb[i] = Bb[kb + (int64_t)min(n0 + bn + 16 * i, N - 1) * ldb];
  };
  v4d pr[4][2], pi[4][2];
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      pr[t][j] = (v4d){0, 0, 0, 0};
      pi[t][j] = (v4d){0, 0, 0, 0};
    }
  fetch(0);
  const int fi = lane & 15, fk = lane >> 4;
  for (int k0 = 0; k0 < K; k0 += TK) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int kk = ak + 2 * i;
      As[kk][am] = (k0 + kk < K && m0 + am < M) ? ra[i] : zmk(0, 0);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) Bs[bk][bn + 16 * i] = (k0 + bk < K && n0 + bn + 16 * i < N) ? rb[i] : zmk(0, 0);
    __syncthreads();
    if (k0 + TK < K) fetch(k0 + TK);
#pragma unroll
    for (int ks = 0; ks < TK / 4; ++ks) {
      const int kk = ks * 4 + fk;
      zd xb[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) xb[j] = Bs[kk][32 * wn + 16 * j + fi];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const zd va = As[kk][64 * wm + 16 * t + fi];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          pr[t][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(va.x, xb[j].x, pr[t][j], 0, 0, 0);
          pi[t][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(va.x, xb[j].y, pi[t][j], 0, 0, 0);
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          pr[t][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(-va.y, xb[j].y, pr[t][j], 0, 0, 0);
          pi[t][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(va.y, xb[j].x, pi[t][j], 0, 0, 0);
        }
      }
    }
  }
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int nn = n0 + 32 * wn + 16 * j + fi;
    if (nn >= N) continue;
    zd *Cb = C + b * sC + (int64_t)nn * ldc;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t m = m0 + 64 * wm + 16 * t + fk + 4 * r;
        if (m < M) {
          zd v = zmul(alpha, zmk(pr[t][j][r], pi[t][j][r]));
          if (BETA) v = zfma(beta, Cb[m], v);
          Cb[m] = v;
        }
      }
  }
}

void launch_gemm_nn(int nb, int64_t M, int N, int K, zd alpha, const zd *A, int64_t lda, int64_t sA,
                    const zd *B, int64_t ldb, int64_t sB, zd beta, zd *C, int64_t ldc, int64_t sC,
                    hipStream_t s) {
  if (M <= 0 || N <= 0 || nb <= 0) return;
  if (K <= 0) throw HipError("gemm_nn: K must be positive");
  if (M >= 4096 && N >= 64) {  // tall: 128 x 64 tiles
    const int tilesN = (N + 63) / 64;
    const int64_t tiles = ((M + 127) / 128) * tilesN;
    // the kernel renumbers the linear id of the whole grid in 32 bits
    if (tiles * nb > 0xffffffffLL || nb > 65535) throw HipError("gemm_nn: grid too large");
    dim3 g((unsigned)tiles, nb), t(256);
    if (beta.x == 0.0 && beta.y == 0.0)
      hipLaunchKernelGGL(k_zgemm_nn_tall<false>, g, t, 0, s, M, N, K, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc,
                         sC, tilesN);
    else
      hipLaunchKernelGGL(k_zgemm_nn_tall<true>, g, t, 0, s, M, N, K, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc,
                         sC, tilesN);
    EMU_LAUNCH_CHECK();
    return;
  }
  const int tilesN = (N + 63) / 64;
  const int64_t tiles = ((M + 63) / 64) * tilesN;
  if (tiles > 0x7fffffff || nb > 65535) throw HipError("gemm_nn: grid too large");
  dim3 g((unsigned)tiles, nb), t(256);
  if (beta.x == 0.0 && beta.y == 0.0)
    hipLaunchKernelGGL(k_zgemm_nn<false>, g, t, 0, s, M, N, K, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc, sC,
                       tilesN);
  else
    hipLaunchKernelGGL(k_zgemm_nn<true>, g, t, 0, s, M, N, K, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc, sC,
                       tilesN);
  EMU_LAUNCH_CHECK();
}

__global__ void k_copy(int64_t n, const zd *__restrict__ src, int64_t ss, zd *__restrict__ dst, int64_t sd) {
  int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  int b = blockIdx.y;
  if (i < n) dst[b * sd + i] = src[b * ss + i];
}

void launch_copy(int nb, int64_t n, const zd *src, int64_t ss, zd *dst, int64_t sd, hipStream_t s) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_copy, dim3((unsigned)((n + 255) / 256), nb), dim3(256), 0, s, n, src, ss, dst, sd);
  EMU_LAUNCH_CHECK();
}

}  // namespace emu

namespace emu {

// ---------------------------------------------- block Gram-Schmidt helpers
// w[b] -= sum_{c<k} V[b][:, c] h[b][c]  (thread per row, h staged through LDS 64 values at a time)
__global__ __launch_bounds__(256) void k_sub_vh(int64_t n, int k, const zd *__restrict__ V, int64_t ldv, int64_t sV,
                                                const zd *__restrict__ h, int64_t sh, zd *__restrict__ w,
                                                int64_t sw) {
  __shared__ zd hs[64];
  const int b = blockIdx.y;
  const int64_t r = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  const zd *Vb = V + b * sV;
  zd acc = r < n ? w[b * sw + r] : zmk(0, 0);
  for (int c0 = 0; c0 < k; c0 += 64) {
    const int cn = min(64, k - c0);
    __syncthreads();
    if (threadIdx.x < 64) hs[threadIdx.x] = (int)threadIdx.x < cn ? h[b * sh + c0 + threadIdx.x] : zmk(0, 0);
    __syncthreads();
    if (r < n)
      for (int c = 0; c < cn; ++c) acc = zfms(Vb[r + (int64_t)(c0 + c) * ldv], hs[c], acc);
  }
  if (r < n) w[b * sw + r] = acc;
}

void launch_sub_vh(int nb, int64_t n, int k, const zd *V, int64_t ldv, int64_t sV, const zd *h, int64_t sh, zd *w,
                   int64_t sw, hipStream_t s, KTime kt) {
  hipExtLaunchKernelGGL(k_sub_vh, dim3((unsigned)((n + 255) / 256), nb), dim3(256), 0, s, kt.a, kt.b, 0, n, k, V, ldv,
                        sV, h, sh, w, sw);
  EMU_LAUNCH_CHECK();
}

// Two-pass Gram-Schmidt of one vector against k columns on small batches, in
// five dependent launches instead of ten: the projection's partial sums
// (k_atb_tall), then k_cgs_sub, in which every workgroup adds them up for
// itself (k x nchunk values from L2) and subtracts, once more of both, and
// k_cgs_norm.  A launch in this chain takes 2 to 6 us however little it does
// (a step of two instances of 1,990 unknowns 92 -> 76 us, of 32 166 -> 157 us).
// A workgroup has 64 rows; its four waves take every fourth column and add
// through LDS.  h1: the first pass's coefficients.  LAST: the second pass
// stores the sum of both to H and its rows' part of |w|^2 to npart.
template <bool LAST>
__global__ __launch_bounds__(256) void k_cgs_sub(int n, int k, const zd *__restrict__ V, int64_t sV,
                                                 const zd *__restrict__ part, int nchunk, zd *__restrict__ h1,
                                                 int64_t sh, zd *__restrict__ H, int64_t sH, zd *__restrict__ w,
                                                 int64_t sw, double *__restrict__ npart) {
  __shared__ zd hs[256], red[3][64];
  const int b = blockIdx.y, tid = threadIdx.x, lane = tid & 63, g = tid >> 6;
  const int row = blockIdx.x * 64 + lane, rc = min(row, n - 1);
  const zd *Vb = V + b * sV + rc, *pb = part + (int64_t)b * nchunk * k;
  const zd w0 = w[b * sw + rc];
  zd acc = zmk(0, 0);
  for (int c0 = 0; c0 < k; c0 += 256) {
    const int cn = min(256, k - c0), e = c0 + min(tid, cn - 1);
    zd h = zmk(0, 0);
    for (int q = 0; q < nchunk; q += 8) {
      zd v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = pb[(int64_t)min(q + u, nchunk - 1) * k + e];
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (q + u < nchunk) h = zadd(h, v[u]);
    }
    __syncthreads();
    hs[tid] = tid < cn ? h : zmk(0, 0);
    if (blockIdx.x == 0 && tid < cn) {
      if (LAST) H[b * sH + e] = zadd(h1[b * sh + e], h);
      else h1[b * sh + e] = h;
    }
    __syncthreads();
    for (int c = g; c < cn; c += 32) {
      zd v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = Vb[(int64_t)(c0 + min(c + 4 * u, cn - 1)) * n];
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (c + 4 * u < cn) acc = zfma(v[u], hs[c + 4 * u], acc);
    }
  }
  if (g > 0) red[g - 1][lane] = acc;
  __syncthreads();
  if (g > 0) return;
#pragma unroll
  for (int q = 0; q < 3; ++q) acc = zadd(acc, red[q][lane]);
  const zd x = zsub(w0, acc);
  if (row < n) w[b * sw + row] = x;
  if (LAST) {
    double d = row < n ? x.x * x.x + x.y * x.y : 0.0;
#pragma unroll
    for (int m = 32; m > 0; m >>= 1) d += __shfl_xor(d, m, 64);
    if (lane == 0) npart[(int64_t)b * gridDim.x + blockIdx.x] = d;
  }
}

// w /= |w| from the sums of k_cgs_sub; |w| to *hn (a length of zero is replaced
// by a tiny one and counted, as in k_cholqr)
__global__ __launch_bounds__(256) void k_cgs_norm(int n, int nparts, const double *__restrict__ npart,
                                                  zd *__restrict__ w, int64_t sw, zd *__restrict__ hn, int64_t sH,
                                                  int32_t *__restrict__ bad) {
  __shared__ double red[4];
  const int b = blockIdx.y, tid = threadIdx.x;
  double d = 0;
  for (int i = tid; i < nparts; i += 256) d += npart[(int64_t)b * nparts + i];
#pragma unroll
  for (int m = 32; m > 0; m >>= 1) d += __shfl_xor(d, m, 64);
  if ((tid & 63) == 0) red[tid >> 6] = d;
  __syncthreads();
  d = (red[0] + red[1]) + (red[2] + red[3]);
  const bool zero = !(d > 0.0);
  if (zero) d = 1e-300;
  const double r = sqrt(d), inv = 1.0 / r;
  const int row = blockIdx.x * 256 + tid;
  if (row < n) w[b * sw + row] = zscale(w[b * sw + row], inv);
  if (blockIdx.x == 0 && tid == 0) {
    hn[b * sH] = zmk(r, 0.0);
    if (zero) bad[b] += 1;
  }
}

// Where the vectors' 64-row pieces are at most 1,280 workgroups (a fuller chip
// is bound by the basis' bytes, and the partial sums read again by every
// workgroup only add to them).  False: not for this size, nothing done.
bool launch_cgs1(int nb, int64_t n, int k, const zd *V, int64_t sV, zd *w, int64_t sw, zd *scratch,
                 size_t scratch_elems, zd *h1, int64_t sh, zd *H, int64_t sH, double *npart, int32_t *bad,
                 hipStream_t s, const KTime *kp, const KTime *ks) {
  const int64_t blocks = (n + 63) / 64;
  if (blocks * nb > 1280 || n > INT32_MAX - 256) return false;
  for (int pass = 0; pass < 2; ++pass) {
    const int nchunk = atb_partials(nb, n, k, V, n, sV, w, sw, true, 32, scratch, scratch_elems, s, kp[pass]);
    const KTime kt = ks[pass];
    if (pass == 0)
      hipExtLaunchKernelGGL(k_cgs_sub<false>, dim3((unsigned)blocks, nb), dim3(256), 0, s, kt.a, kt.b, 0, (int)n, k, V,
                            sV, scratch, nchunk, h1, sh, H, sH, w, sw, npart);
    else
      hipExtLaunchKernelGGL(k_cgs_sub<true>, dim3((unsigned)blocks, nb), dim3(256), 0, s, kt.a, kt.b, 0, (int)n, k, V,
                            sV, scratch, nchunk, h1, sh, H, sH, w, sw, npart);
    EMU_LAUNCH_CHECK();
  }
  hipLaunchKernelGGL(k_cgs_norm, dim3((unsigned)((n + 255) / 256), nb), dim3(256), 0, s, (int)n, (int)blocks, npart, w,
                     sw, H + k, sH, bad);
  EMU_LAUNCH_CHECK();
  return true;
}

// ------------------------------- delayed block Gram-Schmidt (one pass per block)
// Block Arnoldi where the second Gram-Schmidt pass of block j is delayed into
// the projection of block j + 1 (the low-synchronisation "DCGS2" scheme of
// Swirydowicz et al., Numer. Linear Algebra Appl. 28 (2021), here in block
// form): the operator is applied to the provisional block Z (projected once),
// and a single read of the basis Vt = V[:, :j] gives both Vt^H Z (Z's
// reorthogonalisation) and Vt^H W (W = OP Z's first projection), so each
// block costs two passes over the basis instead of four.  The Arnoldi
// relation OP V[:, :j] = V[:, :j+B] H[:j+B, :j] is kept exact by correcting
// row block j of H when Z is reorthogonalised and by removing OP Vt S (known
// from H) from W.  B = 2, 4 or 8 columns per block.
//
// One step's small dense work is spread over the row blocks of the basis
// (k_dcgs_pre, k_dcgs_coef) and the Gram matrices of Cholesky-QR are formed
// by the kernels that write the block (k_combine, k_trmm_right): at a few
// thousand unknowns the step is a chain of launches of a few microseconds
// each, and at 100,000 these kernels still take their time one after the
// other.  Measured per step of 8 columns without the projection and the update
// themselves (500-triangle cell, 2 instances / 8,000-triangle cell, 2
// instances): 49 / 100 us, from 165 / 310 us with one workgroup per instance
// for the coefficients, sequential 8 x 8 factorisations, a tiled GEMM for H S
// and separate Gram and copy kernels.

// Rows of the basis per workgroup in k_dcgs_pre and k_dcgs_coef.
constexpr int DR = 32;

// Gram matrix of B columns over the rows of a 256-thread workgroup, row r held
// by thread r's w (gram_thread_rows) or already in ws.  The
// rows are staged 128 at a time (18 KB of LDS at B = 8): thread (p + B q, g) sums conj(w_p) w_q over rows g,
// g + G, ..., and the G partial sums are added pairwise.  Threads < B^2 return
// output p + B q.
constexpr int GR = 128;
template <int B>
struct GramLds {
  zd ws[GR][B + 1];
  zd red[256];
};
template <int B>
__device__ __forceinline__ zd gram_acc(const GramLds<B> &g, int rows, zd acc) {
  constexpr int G = 256 / (B * B);
  const int tid = threadIdx.x, o = tid % (B * B), p = o % B, q = o / B;
#pragma unroll 8
  for (int r = tid / (B * B); r < rows; r += G) acc = zcfma(g.ws[r][p], g.ws[r][q], acc);
  return acc;
}
template <int B>
__device__ __forceinline__ zd gram_sum(GramLds<B> &g, zd acc) {
  constexpr int G = 256 / (B * B);
  const int tid = threadIdx.x, o = tid % (B * B);
  g.red[tid] = acc;
#pragma unroll
  for (int h = G / 2; h > 0; h /= 2) {
    __syncthreads();
    if (tid < h * B * B) g.red[tid] = zadd(g.red[tid], g.red[tid + h * B * B]);
  }
  return g.red[o];  // threads < B^2 read what they wrote
}
template <int B>
__device__ __forceinline__ zd gram_thread_rows(GramLds<B> &g, const zd *w) {
  zd acc = zmk(0, 0);
#pragma unroll
  for (int h = 0; h < 256; h += GR) {
    if (h > 0) __syncthreads();
    if ((int)threadIdx.x >= h && (int)threadIdx.x < h + GR)
#pragma unroll
      for (int q = 0; q < B; ++q) g.ws[threadIdx.x - h][q] = w[q];
    __syncthreads();
    acc = gram_acc<B>(g, GR, acc);
  }
  return gram_sum<B>(g, acc);
}

// W[b] (n x NQ, in place) = W[b] L[b] - V[b][:, :k] E[b] (L: NQ x NQ, column-
// major; E: k x NQ, row-major so that the NQ coefficients of basis column c
// are contiguous).  The coefficients of a column are the same for every lane,
// so they are read with scalar loads straight into SGPRs and used as FMA
// operands: no LDS traffic in the main loop.  GRAM: also the Gram matrix of
// the last NQ / 2 columns over the workgroup's rows, gpart[b][block].
// QS = 1: a thread per row (bandwidth-bound on V).  QS = 4: 64 rows per
// workgroup and NQ / 4 columns per wave, for problems whose rows alone leave
// most SIMDs idle: a row's NQ FMAs per basis column are a serial stream of
// 256 clocks at NQ = 16.
template <int NQ, int QS, bool GRAM>
__global__ __launch_bounds__(256) void k_combine(int64_t n, int k, const zd *__restrict__ V, int64_t ldv,
                                                 int64_t sV, const zd *__restrict__ E, int64_t sE,
                                                 const zd *__restrict__ L, zd *__restrict__ W, int64_t ldw,
                                                 int64_t sW, zd *__restrict__ gpart) {
  constexpr int R = 256 / QS, C = NQ / QS, B = NQ / 2;
  __shared__ zd ls[NQ][NQ];
  const int b = blockIdx.y;
  const int lrow = threadIdx.x % R;
  const int q0 = QS == 1 ? 0 : C * __builtin_amdgcn_readfirstlane(threadIdx.x / R);
  const int r = blockIdx.x * R + lrow, nr = (int)n;  // n < 2^31 (checked by the launcher)
  const int rr = min(r, nr - 1);                     // clamped row: loads stay in bounds, the store is skipped
  const zd *Vb = V + b * sV + rr;
  const zd *Eb = E + b * sE + q0;
  for (int idx = threadIdx.x; idx < NQ * NQ; idx += blockDim.x) ls[idx % NQ][idx / NQ] = L[(int64_t)b * NQ * NQ + idx];
  __syncthreads();
  zd acc[C];
#pragma unroll
  for (int q = 0; q < C; ++q) acc[q] = zmk(0, 0);
  // acc = W L, W read in halves of NQ / 2 columns, each half's loads all in
  // flight before the first use (the scheduler would otherwise wait for each
  // in turn); halves keep the live registers within four waves per SIMD
#pragma unroll
  for (int h = 0; h < NQ; h += NQ / 2) {
    zd x[NQ / 2];
#pragma unroll
    for (int p = 0; p < NQ / 2; ++p) x[p] = W[b * sW + (h + p) * ldw + rr];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < C; ++q)
#pragma unroll
      for (int p = 0; p < NQ / 2; ++p) acc[q] = zfma(x[p], ls[h + p][q0 + q], acc[q]);
  }
  if (QS > 1) __syncthreads();  // W is read by every wave before any writes it
#pragma unroll QS == 1 ? 2 : 8
  for (int c = 0; c < k; ++c) {
    const zd v = Vb[(int64_t)c * ldv];
    const zd *ec = Eb + (int64_t)c * NQ;
#pragma unroll
    for (int q = 0; q < C; ++q) acc[q] = zfms(v, ec[q], acc[q]);
  }
  if (r < nr)
#pragma unroll
    for (int q = 0; q < C; ++q) W[b * sW + (q0 + q) * ldw + r] = acc[q];
  if constexpr (GRAM) {
    static_assert(R <= GR, "the workgroup's rows fit the staging");
    __shared__ GramLds<B> gl;
    if (r >= nr)
#pragma unroll
      for (int q = 0; q < C; ++q) acc[q] = zmk(0, 0);
#pragma unroll
    for (int q = 0; q < C; ++q)
      if (q0 + q >= B) gl.ws[lrow][q0 + q - B] = acc[q];
    __syncthreads();
    const zd g = gram_sum<B>(gl, gram_acc<B>(gl, R, zmk(0, 0)));
    if (threadIdx.x < B * B) gpart[((int64_t)b * gridDim.x + blockIdx.x) * B * B + threadIdx.x] = g;
  }
}

// Split columns where the rows alone fill at most about one wave per SIMD
// (1,024 SIMDs); NQ = 16, split against not: 190 waves (n = 6,072, 2 instances)
// 14 / 36 us, 1,116 waves (n = 17,832, 4) 46 / 70 us, 3,006 waves (n = 96,168,
// 2) 267 / 202 us.
// Only the split form adds the Gram matrix: with it the other one needs a
// 129th register, hence three instead of four waves per SIMD (805 -> 1,340 us
// at 96,168 unknowns and 8 instances), while k_gram takes 24 us there.
int64_t launch_combine(int nb, int64_t n, int k, int nq, const zd *V, int64_t ldv, int64_t sV, const zd *E,
                       int64_t sE, const zd *L, zd *W, int64_t ldw, int64_t sW, zd *gpart, hipStream_t s, KTime kt) {
  if (n > INT32_MAX - 256) throw HipError("combine: too many rows");
  const bool split = nq >= 4 && (n + 63) / 64 * nb <= 1280;
  const unsigned blocks = (unsigned)(split ? (n + 63) / 64 : (n + 255) / 256);
  dim3 g(blocks, nb), t(256);
#define EMU_COMBINE(NQ, QS, GR) \
  hipExtLaunchKernelGGL((k_combine<NQ, QS, GR>), g, t, 0, s, kt.a, kt.b, 0, n, k, V, ldv, sV, E, sE, L, W, ldw, sW, gpart)
#define EMU_COMBINE_NQ(NQ)                    \
  if (!split) EMU_COMBINE(NQ, 1, false);      \
  else if (gpart) EMU_COMBINE(NQ, 4, true);   \
  else EMU_COMBINE(NQ, 4, false);
  switch (nq) {
    case 2: EMU_COMBINE(2, 1, false); break;
    case 4: EMU_COMBINE_NQ(4) break;
    case 8: EMU_COMBINE_NQ(8) break;
    case 16: EMU_COMBINE_NQ(16) break;
    default: throw HipError("combine: 2, 4, 8 or 16 columns");
  }
#undef EMU_COMBINE_NQ
#undef EMU_COMBINE
  EMU_LAUNCH_CHECK();
  return split && gpart ? blocks : 0;
}

// Cholesky factor R (upper, real diagonal) of the B x B Gram matrix C and its
// inverse, by one wavefront: lane p + B q holds entry (p, q), each of the B
// steps is a few cross-lane moves.  A non-positive pivot (rank-deficient block)
// is replaced by a tiny value and counted.
template <int B>
__device__ __forceinline__ int chol_inv(zd c, double gmax, int lane, zd &R, zd &Ri) {
  const int p = lane % B, q = (lane / B) % B;
  int nbad = 0;
  R = zmk(0, 0);
  double dinv[B];
#pragma unroll
  for (int k = 0; k < B; ++k) {
    double d = __shfl(c.x, k + B * k, 64);
    if (!(d > 1e-28 * gmax)) {
      d = 1e-28 * gmax + 1e-300;
      ++nbad;
    }
    const double rk = sqrt(d);
    dinv[k] = 1.0 / rk;
    const zd cp = shfl_z(c, k + B * p), cq = shfl_z(c, k + B * q);  // row k of C at columns p and q
    const zd rp = zscale(cp, dinv[k]), rq = zscale(cq, dinv[k]);
    if (p == k && q == k) R = zmk(rk, 0.0);
    else if (p == k && q > k) R = rq;
    else if (p > k && q > k) c = zsub(c, zmul(zconj(rp), rq));
  }
  // X = R^-1: rows from the last; acc = (delta - sum over finished rows)
  Ri = zmk(p == q ? 1.0 : 0.0, 0.0);
#pragma unroll
  for (int k = B - 1; k >= 0; --k) {
    if (p == k) Ri = zscale(Ri, dinv[k]);
    const zd xk = shfl_z(Ri, k + B * q), rik = shfl_z(R, p + B * k);
    if (p < k) Ri = zfms(rik, xk, Ri);
  }
  if (p > q) Ri = zmk(0, 0);
  return nbad;
}

// First half of a step's coefficients: per 32 rows i of the basis,
//   A0[i, :] = H[i, :j] S,
// and over these rows the partial sums of S^H S, S^H T and u = H[j:j+B, c0:j] S
// (part[b][block][3][B][B], row index first).  P = [Vt Z W]^H [Z W]
// ((j + 2B) x 2B, ld ldp): S = P[:j, :B], T = P[:j, B:].  FIN (P = [Vt Z]^H Z):
// S^H S only.
template <int B, bool FIN>
__global__ __launch_bounds__(256) void k_dcgs_pre(int j, int c0, const zd *__restrict__ P, int64_t ldp, int64_t sP,
                                                  const zd *__restrict__ H, int64_t ldh, int64_t sH,
                                                  zd *__restrict__ A0, int64_t lda, int64_t sA,
                                                  zd *__restrict__ part) {
  constexpr int KG = 256 / DR, KB = 64;  // k groups, k per round
  const int b = blockIdx.y, tid = threadIdx.x, i0 = blockIdx.x * DR;
  const zd *Pb = P + b * sP, *Hb = H + b * sH;
  __shared__ zd Ps[DR][2 * B + 1], Hr[B][DR + 1];
  for (int idx = tid; idx < DR * 2 * B; idx += 256) {
    const int r = idx % DR, c = idx / DR;
    const zd v = Pb[min(i0 + r, j - 1) + (int64_t)(FIN ? c % B : c) * ldp];
    Ps[r][c] = i0 + r < j ? v : zmk(0, 0);
  }
  if (!FIN)
    for (int idx = tid; idx < DR * B; idx += 256) {
      const int p = idx % B, r = idx / B, c = i0 + r;
      const zd v = Hb[j + p + (int64_t)min(c, j - 1) * ldh];
      Hr[p][r] = (c >= c0 && c < j) ? v : zmk(0, 0);
    }
  __syncthreads();
  for (int o = tid; o < (FIN ? 1 : 3) * B * B; o += 256) {
    const int which = o / (B * B), p = o % B, q = o / B % B;
    zd acc = zmk(0, 0);
#pragma unroll 8
    for (int r = 0; r < DR; ++r) {
      if (which == 2) acc = zfma(Hr[p][r], Ps[r][q], acc);
      else acc = zcfma(Ps[r][p], Ps[r][which * B + q], acc);
    }
    part[(((int64_t)b * gridDim.x + blockIdx.x) * 3 + which) * B * B + p + B * q] = acc;
  }
  if (FIN) return;
  // A0: thread (row r, group g) sums k = g, g + KG, ... of every round
  __shared__ zd Ss[KB][B + 1];
  __shared__ zd red[KG][DR][B + 1];
  const int r = tid % DR, g = tid / DR;
  zd acc[B];
#pragma unroll
  for (int q = 0; q < B; ++q) acc[q] = zmk(0, 0);
  for (int k0 = 0; k0 < j; k0 += KB) {
    zd h[KB / KG];
#pragma unroll
    for (int u = 0; u < KB / KG; ++u) h[u] = Hb[min(i0 + r, j - 1) + (int64_t)min(k0 + g + KG * u, j - 1) * ldh];
    __syncthreads();
    for (int idx = tid; idx < KB * B; idx += 256) {
      const int k = idx % KB, q = idx / KB;
      const zd v = Pb[min(k0 + k, j - 1) + (int64_t)q * ldp];
      Ss[k][q] = k0 + k < j ? v : zmk(0, 0);
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < KB / KG; ++u)
#pragma unroll
      for (int q = 0; q < B; ++q) acc[q] = zfma(h[u], Ss[g + KG * u][q], acc[q]);
  }
#pragma unroll
  for (int q = 0; q < B; ++q) red[g][r][q] = acc[q];
  __syncthreads();
  for (int idx = tid; idx < DR * B; idx += 256) {
    const int rr = idx % DR, q = idx / DR;
    zd v = red[0][rr][q];
#pragma unroll
    for (int k = 1; k < KG; ++k) v = zadd(v, red[k][rr][q]);
    if (i0 + rr < j) A0[b * sA + i0 + rr + (int64_t)q * lda] = v;
  }
}

// Second half, one workgroup per 32 rows of the basis (at least one):
//   G = P[j:j+2B, :] = [Z W]^H [Z W];  row block j of H (rows j .. j+B-1) is
//   nonzero in columns [c0, j).
// Z's reorthogonalisation: C = Z^H Z - S^H S = R^H R, Q = (Z - Vt S) R^-1,
// H[:j, c0:j] += S H[j:j+B, c0:j], H[j:j+B, c0:j] <- R H[j:j+B, c0:j].
// W's first projection against [Vt, Q] with OP Vt S = [Vt, Q] H S removed:
//   u = H_old[j:j+B, :j] S, a = A0 + S u, b = R u,
//   cV = (T - a) R^-1, cQ = R^-H (Z^H W - S^H T) R^-1 - b R^-1  (column j of H),
//   D = b R^-1 + cQ, E = [S R^-1, a R^-1 + cV - S R^-1 D],
//   L = [[R^-1, -R^-1 D], [0, R^-1]], so that [Q, Zraw] = [Z W] L - Vt E.
// FIN (no W; the last provisional block of an expansion; P = [Vt Z]^H Z):
// only Z's reorthogonalisation, E = S R^-1 (j x B), L = R^-1.
// Every workgroup forms the B x B quantities for itself (a few microseconds,
// less than another launch) and applies them to its rows; R H[j:j+B, c0:j] goes
// to Hrow (B x j) because the other workgroups read the old rows: k_cholqr
// (or, FIN, k_hrow) stores it.
template <int B, bool FIN>
__global__ __launch_bounds__(256) void k_dcgs_coef(int j, int c0, const zd *__restrict__ P, int64_t ldp, int64_t sP,
                                                   const zd *__restrict__ A0, int64_t lda, int64_t sA,
                                                   const zd *__restrict__ part, int nblk, zd *__restrict__ H,
                                                   int64_t ldh, int64_t sH, zd *__restrict__ E, int64_t sE,
                                                   zd *__restrict__ L, zd *__restrict__ Hrow, int64_t sR,
                                                   int32_t *__restrict__ bad) {
  constexpr int NG = FIN ? B : 2 * B, BB = B * B;
  const int b = blockIdx.y, tid = threadIdx.x, lane = tid & 63;
  const zd *Pb = P + b * sP;
  zd *Hb = H + b * sH;
  zd *Eb = E + b * sE;
  __shared__ zd Gs[NG][NG], S3[3][BB], R[B][B], Ri[B][B], Bm[B][B], Dm[B][B], T1[B][B], T2[B][B];
  for (int idx = tid; idx < NG * NG; idx += 256) Gs[idx % NG][idx / NG] = Pb[(j + idx % NG) + (int64_t)(idx / NG) * ldp];
  for (int o = tid; o < (FIN ? 1 : 3) * BB; o += 256) {
    const zd *pp = part + (int64_t)b * nblk * 3 * BB + o;
    zd acc = zmk(0, 0);
    for (int k = 0; k < nblk; k += 4) {
      zd v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) v[u] = pp[(int64_t)min(k + u, nblk - 1) * 3 * BB];
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (k + u < nblk) acc = zadd(acc, v[u]);
    }
    S3[o / BB][o % BB] = acc;
  }
  __syncthreads();
  const int p = lane % B, q = lane / B % B;
  if (tid < 64) {
    double gmax = 0;
#pragma unroll
    for (int i = 0; i < B; ++i) gmax = fmax(gmax, Gs[i][i].x);
    zd r, ri;
    const int nbad = chol_inv<B>(zsub(Gs[p][q], S3[0][p + B * q]), gmax, lane, r, ri);
    if (lane < BB) {
      R[p][q] = r;
      Ri[p][q] = ri;
    }
    if (tid == 0 && blockIdx.x == 0 && nbad) bad[b] += nbad;
  }
  __syncthreads();
  if (!FIN) {
    if (tid < BB) {
      zd acc = zmk(0, 0);
      for (int k = p; k < B; ++k) acc = zfma(R[p][k], S3[2][k + B * q], acc);
      Bm[p][q] = acc;  // b = R u
      T1[p][q] = zsub(Gs[p][B + q], S3[1][p + B * q]);
    }
    __syncthreads();
    if (tid < BB) {
      zd acc = zmk(0, 0);
      for (int k = 0; k <= q; ++k) acc = zfma(T1[p][k], Ri[k][q], acc);
      T2[p][q] = acc;
    }
    __syncthreads();
    if (tid < BB) {
      zd acc = zmk(0, 0), bri = zmk(0, 0);
      for (int k = 0; k <= p; ++k) acc = zcfma(Ri[k][p], T2[k][q], acc);
      for (int k = 0; k <= q; ++k) bri = zfma(Bm[p][k], Ri[k][q], bri);
      Dm[p][q] = acc;                                                 // D = R^-H T1 R^-1
      if (blockIdx.x == 0) Hb[(j + p) + (int64_t)(j + q) * ldh] = zsub(acc, bri);  // cQ
    }
    __syncthreads();
  }
  // this workgroup's rows: E, column block j of H, and the row correction
  __shared__ zd Ps[DR][2 * B + 1], sa[DR][B], se[DR][B];
  const int i0 = blockIdx.x * DR;
  if (i0 < j) {
    for (int idx = tid; idx < DR * NG; idx += 256) {
      const int r = idx % DR, c = idx / DR;
      Ps[r][c] = Pb[min(i0 + r, j - 1) + (int64_t)c * ldp];
    }
    __syncthreads();
    for (int idx = tid; idx < DR * B; idx += 256) {
      const int rr = idx / B, c = idx % B, i = i0 + rr;
      zd e1 = zmk(0, 0), av = zmk(0, 0);
      for (int k = 0; k <= c; ++k) e1 = zfma(Ps[rr][k], Ri[k][c], e1);
      if (i < j) Eb[(int64_t)i * NG + c] = e1;
      if (!FIN) {
        av = A0[b * sA + min(i, j - 1) + (int64_t)c * lda];
#pragma unroll
        for (int k = 0; k < B; ++k) av = zfma(Ps[rr][k], S3[2][k + B * c], av);
      }
      se[rr][c] = e1;
      sa[rr][c] = av;
    }
    __syncthreads();
    if (!FIN)
      for (int idx = tid; idx < DR * B; idx += 256) {
        const int rr = idx / B, c = idx % B, i = i0 + rr;
        zd cv = zmk(0, 0), e2 = zmk(0, 0);
        for (int k = 0; k <= c; ++k) {
          cv = zfma(zsub(Ps[rr][B + k], sa[rr][k]), Ri[k][c], cv);
          e2 = zfma(sa[rr][k], Ri[k][c], e2);
        }
#pragma unroll
        for (int k = 0; k < B; ++k) e2 = zfms(se[rr][k], Dm[k][c], e2);
        if (i < j) {
          Hb[i + (int64_t)(j + c) * ldh] = cv;
          Eb[(int64_t)i * NG + B + c] = zadd(e2, cv);
        }
      }
    const int rr = tid % DR;
    if (i0 + rr < j)
      for (int c = c0 + tid / DR; c < j; c += 256 / DR) {
        zd hr[B];
#pragma unroll
        for (int k = 0; k < B; ++k) hr[k] = Hb[(j + k) + (int64_t)c * ldh];
        zd acc = Hb[i0 + rr + (int64_t)c * ldh];
#pragma unroll
        for (int k = 0; k < B; ++k) acc = zfma(Ps[rr][k], hr[k], acc);
        Hb[i0 + rr + (int64_t)c * ldh] = acc;
      }
  }
  if (blockIdx.x != 0) return;
  for (int c = c0 + tid; c < j; c += 256) {
    zd h[B];
#pragma unroll
    for (int k = 0; k < B; ++k) h[k] = Hb[(j + k) + (int64_t)c * ldh];
#pragma unroll
    for (int i = 0; i < B; ++i) {
      zd acc = zmk(0, 0);
#pragma unroll
      for (int k = i; k < B; ++k) acc = zfma(R[i][k], h[k], acc);
      Hrow[b * sR + i + (int64_t)c * B] = acc;
    }
  }
  zd *Lb = L + (int64_t)b * NG * NG;
  if (tid < BB) {
    Lb[p + q * NG] = Ri[p][q];
    if (!FIN) {
      zd rd = zmk(0, 0);
      for (int k = p; k < B; ++k) rd = zfma(Ri[p][k], Dm[k][q], rd);
      Lb[p + (B + q) * NG] = zsub(zmk(0, 0), rd);
      Lb[(B + p) + q * NG] = zmk(0, 0);
      Lb[(B + p) + (B + q) * NG] = Ri[p][q];
    }
  }
}

// Row block j of H from Hrow (the last step of an expansion; otherwise k_cholqr
// does it)
template <int B>
__global__ __launch_bounds__(256) void k_hrow(int j, int c0, const zd *__restrict__ Hrow, int64_t sR,
                                              zd *__restrict__ H, int64_t ldh, int64_t sH) {
  const int b = blockIdx.y, idx = blockIdx.x * 256 + threadIdx.x;
  if (idx >= (j - c0) * B) return;
  const int p = idx % B, c = c0 + idx / B;
  H[b * sH + j + p + (int64_t)c * ldh] = Hrow[b * sR + p + (int64_t)c * B];
}

void launch_dcgs(int nb, int bq, bool fin, int j, int c0, const zd *P, int64_t ldp, int64_t sP, zd *A0, int64_t lda,
                 int64_t sA, zd *part, zd *H, int64_t ldh, int64_t sH, zd *E, int64_t sE, zd *L, zd *Hrow, int64_t sR,
                 int32_t *bad, hipStream_t s) {
  const int nblk = (j + DR - 1) / DR;
  const dim3 gp((unsigned)nblk, nb), gc((unsigned)std::max(nblk, 1), nb);
#define EMU_DCGS(B, FIN)                                                                                            \
  do {                                                                                                              \
    if (nblk)                                                                                                       \
      hipLaunchKernelGGL((k_dcgs_pre<B, FIN>), gp, dim3(256), 0, s, j, c0, P, ldp, sP, H, ldh, sH, A0, lda, sA, part); \
    hipLaunchKernelGGL((k_dcgs_coef<B, FIN>), gc, dim3(256), 0, s, j, c0, P, ldp, sP, A0, lda, sA, part, nblk, H,   \
                       ldh, sH, E, sE, L, Hrow, sR, bad);                                                           \
    if (FIN && j > c0)                                                                                              \
      hipLaunchKernelGGL(k_hrow<B>, dim3((unsigned)(((j - c0) * B + 255) / 256), nb), dim3(256), 0, s, j, c0, Hrow, \
                         sR, H, ldh, sH);                                                                           \
  } while (0)
#define EMU_DCGS_B(B)           \
  if (fin) EMU_DCGS(B, true);   \
  else EMU_DCGS(B, false);
  switch (bq) {
    case 2: EMU_DCGS_B(2) break;
    case 4: EMU_DCGS_B(4) break;
    case 8: EMU_DCGS_B(8) break;
    default: throw HipError("dcgs: block size must be 2, 4 or 8");
  }
#undef EMU_DCGS_B
#undef EMU_DCGS
  EMU_LAUNCH_CHECK();
}

int64_t dcgs_part_elems(int bq, int m) { return (int64_t)((m + DR - 1) / DR) * 3 * bq * bq; }

// Gram matrix of a block (n x B, ld ldw) over 256 rows per workgroup:
// gpart[b][block][B][B], as k_combine and k_trmm_right write it
template <int B>
__global__ __launch_bounds__(256) void k_gram(int64_t n, const zd *__restrict__ W, int64_t ldw, int64_t sW,
                                              zd *__restrict__ gpart) {
  __shared__ GramLds<B> gl;
  const int b = blockIdx.y;
  const int64_t r = blockIdx.x * (int64_t)256 + threadIdx.x, rr = r < n ? r : n - 1;
  zd w[B];
#pragma unroll
  for (int q = 0; q < B; ++q) {
    const zd v = W[b * sW + q * ldw + rr];
    w[q] = r < n ? v : zmk(0, 0);
  }
  const zd g = gram_thread_rows<B>(gl, w);
  if (threadIdx.x < B * B) gpart[((int64_t)b * gridDim.x + blockIdx.x) * B * B + threadIdx.x] = g;
}

int64_t launch_gram(int nb, int64_t n, int bq, const zd *W, int64_t ldw, int64_t sW, zd *gpart, hipStream_t s) {
  const unsigned blocks = (unsigned)((n + 255) / 256);
  const dim3 g(blocks, nb);
  switch (bq) {
    case 1: hipLaunchKernelGGL(k_gram<1>, g, dim3(256), 0, s, n, W, ldw, sW, gpart); break;
    case 2: hipLaunchKernelGGL(k_gram<2>, g, dim3(256), 0, s, n, W, ldw, sW, gpart); break;
    case 4: hipLaunchKernelGGL(k_gram<4>, g, dim3(256), 0, s, n, W, ldw, sW, gpart); break;
    case 8: hipLaunchKernelGGL(k_gram<8>, g, dim3(256), 0, s, n, W, ldw, sW, gpart); break;
    default: throw HipError("gram: block size must be 1, 2, 4 or 8");
  }
  EMU_LAUNCH_CHECK();
  return blocks;
}

// Cholesky-QR factor of a block from its Gram partials (gpart[b][nchunk][B][B]):
// G = R^H R, Rinv = R^-1, Racc = R Rprev (Rprev = identity when null).  One
// workgroup per instance: 1,024 threads add the partials, one wavefront
// factorises.  With H the results of the block step go there as well: Racc to
// rows j + B .. of column block j, Hrow to columns [c0, j) of row block j.
template <int B>
__global__ __launch_bounds__(1024) void k_cholqr(int nchunk, const zd *__restrict__ gpart, zd *__restrict__ Rinv,
                                                 const zd *__restrict__ Rprev, zd *__restrict__ Racc, int j, int c0,
                                                 const zd *__restrict__ Hrow, int64_t sR, zd *__restrict__ H,
                                                 int64_t ldh, int64_t sH, int32_t *__restrict__ bad) {
  constexpr int BB = B * B, G = 1024 / BB < 64 ? 1024 / BB : 64;
  const int b = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
  __shared__ zd red[G][BB], Rs[B][B], Gs[B][B];
  if (tid < G * BB) {
    const int o = tid % BB, g = tid / BB;
    const zd *pp = gpart + (int64_t)b * nchunk * BB + o;
    zd acc = zmk(0, 0);
    for (int k = g; k < nchunk; k += 4 * G) {
      zd v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) v[u] = pp[(int64_t)min(k + u * G, nchunk - 1) * BB];
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (k + u * G < nchunk) acc = zadd(acc, v[u]);
    }
    red[g][o] = acc;
  }
  if (H)
    for (int idx = tid; idx < (j - c0) * B; idx += 1024) {
      const int p = idx % B, c = c0 + idx / B;
      H[b * sH + j + p + (int64_t)c * ldh] = Hrow[b * sR + p + (int64_t)c * B];
    }
  __syncthreads();
  if (tid >= 64) return;
  const int p = lane % B, q = lane / B % B;
  zd c = zmk(0, 0);
  if (lane < BB) {
    for (int g = 0; g < G; ++g) c = zadd(c, red[g][lane]);
    Gs[p][q] = c;
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  double gmax = 0;
#pragma unroll
  for (int i = 0; i < B; ++i) gmax = fmax(gmax, Gs[i][i].x);
  zd R, Ri;
  const int nbad = chol_inv<B>(Gs[p][q], gmax, lane, R, Ri);
  if (lane == 0 && nbad) bad[b] += nbad;
  if (lane >= BB) return;
  Rs[p][q] = R;
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  const int64_t o = (int64_t)b * BB;
  Rinv[o + lane] = Ri;
  zd acc = zmk(0, 0);
#pragma unroll
  for (int k = 0; k < B; ++k) {
    const zd rp = Rprev ? Rprev[o + k + q * B] : zmk(k == q ? 1.0 : 0.0, 0.0);
    if (k >= p) acc = zfma(Rs[p][k], rp, acc);
  }
  Racc[o + lane] = acc;
  if (H) H[b * sH + j + B + p + (int64_t)(j + q) * ldh] = acc;
}

void launch_cholqr(int nb, int bq, int64_t nchunk, const zd *gpart, zd *Rinv, const zd *Rprev, zd *Racc, int32_t *bad,
                   hipStream_t s, int j, int c0, const zd *Hrow, int64_t sR, zd *H, int64_t ldh, int64_t sH) {
#define EMU_CHOLQR(B)                                                                                               \
  hipLaunchKernelGGL(k_cholqr<B>, dim3(nb), dim3(1024), 0, s, (int)nchunk, gpart, Rinv, Rprev, Racc, j, c0, Hrow, sR, \
                     H, ldh, sH, bad)
  switch (bq) {
    case 1: EMU_CHOLQR(1); break;
    case 2: EMU_CHOLQR(2); break;
    case 4: EMU_CHOLQR(4); break;
    case 8: EMU_CHOLQR(8); break;
    default: throw HipError("cholqr: block size must be 1, 2, 4 or 8");
  }
#undef EMU_CHOLQR
  EMU_LAUNCH_CHECK();
}

// O[b][:, 0:B] = W[b][:, 0:B] * Rinv[b]  (B x B upper triangular, in place
// allowed); with xi, the row-interleaved copy of O as well (xi[b][B r + j], the
// operand of the next Krylov block's SpMM, saving k_interleave's pass); with
// gpart, the Gram matrix of O over the workgroup's 256 rows
template <int B>
__global__ __launch_bounds__(256) void k_trmm_right(int64_t n, const zd *W, int64_t ldw, int64_t sW,
                                                    const zd *__restrict__ Ri, zd *O, int64_t ldo,
                                                    int64_t sO, zd *__restrict__ xi, zd *__restrict__ gpart) {
  __shared__ zd rs[B][B];
  __shared__ GramLds<B> gl;
  const int b = blockIdx.y;
  for (int idx = threadIdx.x; idx < B * B; idx += blockDim.x) rs[idx % B][idx / B] = Ri[(int64_t)b * B * B + idx];
  __syncthreads();
  const int64_t r = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  const int64_t rr = r < n ? r : n - 1;
  zd w[B], o[B];
#pragma unroll
  for (int q = 0; q < B; ++q) w[q] = W[b * sW + q * ldw + rr];
#pragma unroll
  for (int j = 0; j < B; ++j) {
    zd acc = zmk(0, 0);
#pragma unroll
    for (int k = 0; k <= j; ++k) acc = zfma(w[k], rs[k][j], acc);
    o[j] = acc;
    if (r < n) O[b * sO + j * ldo + r] = acc;
  }
  if (xi && r < n) {
    zd *xr = xi + (int64_t)b * B * n + (int64_t)B * r;
#pragma unroll
    for (int j = 0; j < B; ++j) xr[j] = o[j];
  }
  if (gpart) {
    if (r >= n)
#pragma unroll
      for (int j = 0; j < B; ++j) o[j] = zmk(0, 0);
    const zd g = gram_thread_rows<B>(gl, o);
    if (threadIdx.x < B * B) gpart[((int64_t)b * gridDim.x + blockIdx.x) * B * B + threadIdx.x] = g;
  }
}

int64_t launch_trmm_right(int nb, int64_t n, int bq, const zd *W, int64_t ldw, int64_t sW, const zd *Ri, zd *O,
                          int64_t ldo, int64_t sO, hipStream_t s, zd *xi, zd *gpart) {
  const unsigned blocks = (unsigned)((n + 255) / 256);
  dim3 g(blocks, nb);
#define EMU_TRMM(B) hipLaunchKernelGGL(k_trmm_right<B>, g, dim3(256), 0, s, n, W, ldw, sW, Ri, O, ldo, sO, xi, gpart)
  switch (bq) {
    case 1: EMU_TRMM(1); break;
    case 2: EMU_TRMM(2); break;
    case 4: EMU_TRMM(4); break;
    case 8: EMU_TRMM(8); break;
    default: throw HipError("trmm_right: block size must be 1, 2, 4 or 8");
  }
#undef EMU_TRMM
  EMU_LAUNCH_CHECK();
  return blocks;
}

// Dst[b][i + j*ldd] (+)= Src[b][i + j*lds] for i < rows, j < cols
__global__ void k_block_copy(int rows, int cols, const zd *__restrict__ S, int64_t lds, int64_t sS,
                             zd *__restrict__ D, int64_t ldd, int64_t sD, int add) {
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  const int b = blockIdx.y;
  if (idx >= rows * cols) return;
  const int i = idx % rows, j = idx / rows;
  zd v = S[b * sS + i + (int64_t)j * lds];
  zd *d = &D[b * sD + i + (int64_t)j * ldd];
  *d = add ? zadd(*d, v) : v;
}

void launch_block_copy(int nb, int rows, int cols, const zd *S, int64_t lds, int64_t sS, zd *D, int64_t ldd,
                       int64_t sD, bool add, hipStream_t s) {
  if (rows <= 0 || cols <= 0) return;
  hipLaunchKernelGGL(k_block_copy, dim3((rows * cols + 255) / 256, nb), dim3(256), 0, s, rows, cols, S, lds, sS,
                     D, ldd, sD, add ? 1 : 0);
  EMU_LAUNCH_CHECK();
}

}  // namespace emu
