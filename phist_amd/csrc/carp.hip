// carp.hip -- Kaczmarz (CARP) sweeps on the device by multicolouring.
//
// PHIST's CARP kernels (phist_kernels_carp_decl.h:35-102) leave the
// parallelisation to the kernel library.  Here the rows are coloured so that
// two rows of one colour never touch the same entry of x (greedy distance-2
// colouring of the row graph, a row's support being its columns plus its own
// index, which the shift term updates); the rows of a colour then update in
// parallel, a lane per row and vector of columns of X, and a sweep runs the colours
// forward and then backward.  Each colour's rows keep their entries in a
// chunked column-major copy (coalesced reads across the rows of a wave).
// The per-row arithmetic is that of builtin's
// kacz_sub_def.h:27-139 (shifted row product, row norm corrected for the
// shift, scaled projection with relaxation omega_j), with fused multiply-adds
// in a fixed place so that a sequential sweep in colour order reproduces it
// exactly.  RC: real matrix, complex shifts sigma_r + i sigma_i and complex
// solution X_r + i X_i (kacz_sub_def.h under KACZ_RC_VARIANT).
#include "amd_device.hpp"
#include <algorithm>
#include <vector>

namespace phx {

// Rows of one colour in chunks of kCarpChunk (in colour order), each chunk's
// entries stored column-major (entry k of chunk row rr at chunk_ptr + k*kCarpChunk
// + rr, padded to the chunk's longest row), so the rows a wave updates at once
// read their matrix entries in coalesced segments.
constexpr int kCarpChunk = 32;

template <typename T>
struct CarpWork {
  int64_t n = 0;
  int nshifts = 0;
  int ncolors = 0;
  int32_t max_len = 0;               // entries of the longest row
  std::vector<int64_t> color_ptr;    // rows of colour c: rows[color_ptr[c] .. color_ptr[c+1])
  std::vector<int64_t> color_chunk;  // first chunk of colour c
  std::vector<int32_t> h_rows;
  int32_t* rows = nullptr;       // device: rows in colour order
  int32_t* rlen = nullptr;       // device: their lengths
  int64_t* chunk_ptr = nullptr;  // device: first slot of every chunk
  int32_t* col = nullptr;        // device: chunked entries
  T* val = nullptr;
};

// shifts and relaxation factors of up to kCarpCols columns, passed by value
constexpr int kCarpCols = 64;
template <typename T>
struct CarpCoef {
  T sr[kCarpCols], si[kCarpCols], w[kCarpCols];
};

// One colour.  A lane owns VPL consecutive columns of X (a 16-byte vector
// where the layout allows) in one row, nvec / VPL lanes per row.  A row's
// entries are taken in batches of LB: all of a batch's indices and values go
// out together, then all its x rows, so a row of up to LB entries (ONE: every
// row of the matrix) costs three dependent round trips - row data, entries, x
// - whatever its length, and its entries and x rows stay in registers for the
// projection.  Rows of one colour have no x entry in common, so a launch
// reuses nothing but the other half of a cache line; each XCD takes a
// contiguous range of the colour's rows to keep that half in its L2.
// What bounds it: the x lines that each colour reads and writes (2048 x 2048
// sheet, counters: 271 MB read and 189 MB written a launch in 99 us, 4.7 TB/s,
// the rate of a copy); one round trip less, with the entries' place computed
// instead of loaded, gave 2 %.
// 1024 x 1024 graphene sheet with 13 entries per row, 8 columns, FP64, 19
// colours: 41 -> 25 us a launch, 1571 -> 963 us a sweep against one lane per
// (row, column) that read entry after entry and read all of them twice.
// A column that a row stores more than once (the entries are sorted, so the
// repeats are neighbours) continues from the value the entry before it wrote,
// and the diagonal entry from the x_i that the shift term has updated.
template <typename T, bool RC, int VPL, int LB, bool ONE>
__global__ void __launch_bounds__(kBlock)
    k_kacz(const int32_t* __restrict__ rows, const int32_t* __restrict__ rlen, const int64_t* __restrict__ cptr,
           int64_t nr, int64_t ntiles, const int32_t* __restrict__ ci, const T* __restrict__ va, int lpr,
           const CarpCoef<T> coef, const T* __restrict__ b, int64_t ldb, T* xr, T* xi, int64_t ldx) {
  const uint32_t rpt = kBlock / (uint32_t)lpr;  // rows per tile (lanes beyond rpt * lpr stay idle)
  const uint32_t rl = threadIdx.x / (uint32_t)lpr;
  if (rl >= rpt) return;
  const int c0 = (int)(threadIdx.x - rl * (uint32_t)lpr) * VPL;
  T s_r[VPL], s_i[VPL], w[VPL];
#pragma unroll
  for (int e = 0; e < VPL; e++) {
    s_r[e] = coef.sr[c0 + e];
    s_i[e] = RC ? coef.si[c0 + e] : T(0);
    w[e] = coef.w[c0 + e];
  }
  const TileWalk tw = xcd_tiles(ntiles);
  for (int64_t t = tw.t; t < tw.end; t += tw.stride) {
    const int64_t r = t * rpt + rl;
    if (r >= nr) continue;
    const int64_t i = rows[r];
    const int len = rlen[r];
    const int64_t k0 = cptr[r / kCarpChunk] + (r % kCarpChunk);
    T xri[VPL], xii[VPL], bv[VPL], tr[VPL], ti[VPL];
    vload<T, VPL>(xr + i * ldx + c0, xri);
    if (RC) vload<T, VPL>(xi + i * ldx + c0, xii);
    if (b) vload<T, VPL>(b + i * ldb + c0, bv);
    int32_t cj[LB];
    T a[LB], xg[LB][VPL], yg[RC ? LB : 1][VPL];
    auto load = [&](int q0) {
#pragma unroll
      for (int q = 0; q < LB; q++)
        if (q0 + q < len) {
          cj[q] = ci[k0 + (int64_t)(q0 + q) * kCarpChunk];
          a[q] = va[k0 + (int64_t)(q0 + q) * kCarpChunk];
        }
#pragma unroll
      for (int q = 0; q < LB; q++)
        if (q0 + q < len) {
          vload<T, VPL>(xr + (int64_t)cj[q] * ldx + c0, xg[q]);
          if constexpr (RC) vload<T, VPL>(xi + (int64_t)cj[q] * ldx + c0, yg[q]);
        }
    };
#pragma unroll
    for (int e = 0; e < VPL; e++) {
      if (RC) {
        tr[e] = fma(s_i[e], xii[e], -s_r[e] * xri[e]);
        ti[e] = fma(-s_i[e], xri[e], -s_r[e] * xii[e]);
      } else {
        tr[e] = -s_r[e] * xri[e];
      }
    }
    T d = T(0), nrm0 = T(0);
    for (int q0 = 0; q0 < (ONE ? 1 : len); q0 += LB) {
      load(q0);
#pragma unroll
      for (int q = 0; q < LB; q++)
        if (q0 + q < len) {
#pragma unroll
          for (int e = 0; e < VPL; e++) {
            tr[e] = fma(a[q], xg[q][e], tr[e]);
            if constexpr (RC) ti[e] = fma(a[q], yg[q][e], ti[e]);
          }
          nrm0 = fma(a[q], a[q], nrm0);
          if (cj[q] == i) d = a[q];
        }
    }
#pragma unroll
    for (int e = 0; e < VPL; e++) {
      if (b) tr[e] = tr[e] - bv[e];
      T nrm = fma(s_r[e], s_r[e], fma(T(-2) * d, s_r[e], nrm0));
      if (RC) nrm = fma(s_i[e], s_i[e], nrm);
      if (nrm == T(0)) nrm = T(1);
      tr[e] = (tr[e] * w[e]) / nrm;
      if (RC) ti[e] = (ti[e] * w[e]) / nrm;
      // projection: the shift term of x_i first, then every column of the row
      if (RC) {
        xri[e] = xri[e] + fma(ti[e], s_i[e], tr[e] * s_r[e]);
        xii[e] = xii[e] + fma(-tr[e], s_i[e], ti[e] * s_r[e]);
      } else {
        xri[e] = fma(tr[e], s_r[e], xri[e]);
      }
    }
    vstore<T, VPL>(xr + i * ldx + c0, xri);
    if (RC) vstore<T, VPL>(xi + i * ldx + c0, xii);
    int32_t jp = -1;
    T px[VPL], py[VPL];  // what the entry before wrote, to column jp
    for (int q0 = 0; q0 < (ONE ? 1 : len); q0 += LB) {
      if (!ONE) load(q0);
#pragma unroll
      for (int q = 0; q < LB; q++)
        if (q0 + q < len) {
          const bool again = cj[q] == jp, own = cj[q] == i;
#pragma unroll
          for (int e = 0; e < VPL; e++) {
            px[e] = fma(-tr[e], a[q], again ? px[e] : (own ? xri[e] : xg[q][e]));
            if constexpr (RC) py[e] = fma(-ti[e], a[q], again ? py[e] : (own ? xii[e] : yg[q][e]));
          }
          jp = cj[q];
          vstore<T, VPL>(xr + (int64_t)cj[q] * ldx + c0, px);
          if constexpr (RC) vstore<T, VPL>(xi + (int64_t)cj[q] * ldx + c0, py);
        }
    }
  }
}

// greedy distance-2 colouring in row order: a row takes the smallest colour
// not used by any row sharing one of its columns (its own index included)
static void color_rows(const std::vector<int64_t>& ptr, const std::vector<int32_t>& col, int64_t n,
                       std::vector<int>& color, int& ncolors) {
  // transpose structure: rows touching each column (own index included)
  std::vector<int64_t> cp(n + 1, 0);
  for (int64_t i = 0; i < n; i++) {
    cp[i + 1]++;
    for (int64_t k = ptr[i]; k < ptr[i + 1]; k++)
      if (col[k] != i) cp[(int64_t)col[k] + 1]++;
  }
  for (int64_t i = 0; i < n; i++) cp[i + 1] += cp[i];
  std::vector<int64_t> fill(cp.begin(), cp.end() - 1);
  std::vector<int32_t> rr(cp[n]);
  for (int64_t i = 0; i < n; i++) {
    rr[fill[i]++] = (int32_t)i;
    for (int64_t k = ptr[i]; k < ptr[i + 1]; k++)
      if (col[k] != i) rr[fill[col[k]]++] = (int32_t)i;
  }
  color.assign(n, -1);
  std::vector<int64_t> mark;  // mark[c] == i: colour c is taken next to row i
  ncolors = 0;
  auto forbid_column = [&](int64_t j, int64_t i) {
    for (int64_t q = cp[j]; q < cp[j + 1]; q++) {
      const int c = color[rr[q]];
      if (c >= 0) mark[c] = i;
    }
  };
  for (int64_t i = 0; i < n; i++) {
    forbid_column(i, i);
    for (int64_t k = ptr[i]; k < ptr[i + 1]; k++)
      if (col[k] != i) forbid_column(col[k], i);
    int c = 0;
    while (c < ncolors && mark[c] == i) c++;
    if (c == ncolors) {
      ncolors++;
      mark.push_back(-1);
    }
    color[i] = c;
  }
}

template <typename T>
void* carp_setup(const SparseMat<T>* A, int nshifts) {
  PHX_REQUIRE(A->nrows == A->ncols, PHIST_INVALID_INPUT, "CARP needs a square matrix");
  PHX_REQUIRE(nshifts >= 1, PHIST_INVALID_INPUT, "numShifts %d", nshifts);
  auto* W = new CarpWork<T>();
  W->n = A->nrows;
  W->nshifts = nshifts;
  std::vector<int> color;
  color_rows(A->crs_ptr, A->crs_col, W->n, color, W->ncolors);
  W->color_ptr.assign(W->ncolors + 1, 0);
  for (int64_t i = 0; i < W->n; i++) W->color_ptr[color[i] + 1]++;
  for (int c = 0; c < W->ncolors; c++) W->color_ptr[c + 1] += W->color_ptr[c];
  W->h_rows.resize(W->n);
  std::vector<int64_t> fill(W->color_ptr.begin(), W->color_ptr.end() - 1);
  for (int64_t i = 0; i < W->n; i++) W->h_rows[fill[color[i]]++] = (int32_t)i;
  // chunked entry layout, colour by colour (entries of a row in CRS order)
  std::vector<int32_t> rlen(W->n);
  std::vector<int64_t> cptr;
  W->color_chunk.assign(W->ncolors + 1, 0);
  int64_t slots = 0;
  for (int c = 0; c < W->ncolors; c++) {
    W->color_chunk[c] = (int64_t)cptr.size();
    for (int64_t r0 = W->color_ptr[c]; r0 < W->color_ptr[c + 1]; r0 += kCarpChunk) {
      const int64_t r1 = std::min<int64_t>(W->color_ptr[c + 1], r0 + kCarpChunk);
      int32_t wmax = 0;
      for (int64_t r = r0; r < r1; r++) {
        const int64_t i = W->h_rows[r];
        rlen[r] = (int32_t)(A->crs_ptr[i + 1] - A->crs_ptr[i]);
        wmax = std::max(wmax, rlen[r]);
      }
      W->max_len = std::max(W->max_len, wmax);
      cptr.push_back(slots);
      slots += (int64_t)wmax * kCarpChunk;
    }
  }
  W->color_chunk[W->ncolors] = (int64_t)cptr.size();
  cptr.push_back(slots);
  std::vector<int32_t> ccol((size_t)std::max<int64_t>(1, slots), 0);
  std::vector<T> cval((size_t)std::max<int64_t>(1, slots), T(0));
  for (int c = 0; c < W->ncolors; c++)
    for (int64_t r = W->color_ptr[c]; r < W->color_ptr[c + 1]; r++) {
      const int64_t rl = r - W->color_ptr[c];
      const int64_t base = cptr[W->color_chunk[c] + rl / kCarpChunk] + rl % kCarpChunk;
      const int64_t i = W->h_rows[r];
      for (int32_t q = 0; q < rlen[r]; q++) {
        ccol[base + (int64_t)q * kCarpChunk] = A->crs_col[A->crs_ptr[i] + q];
        cval[base + (int64_t)q * kCarpChunk] = A->crs_val[A->crs_ptr[i] + q];
      }
    }
  hipStream_t st = rt().stream;
  PHX_HIP(hipMalloc(&W->rows, sizeof(int32_t) * std::max<int64_t>(1, W->n)));
  PHX_HIP(hipMalloc(&W->rlen, sizeof(int32_t) * std::max<int64_t>(1, W->n)));
  PHX_HIP(hipMalloc(&W->chunk_ptr, sizeof(int64_t) * cptr.size()));
  PHX_HIP(hipMalloc(&W->col, sizeof(int32_t) * ccol.size()));
  PHX_HIP(hipMalloc(&W->val, sizeof(T) * cval.size()));
  if (W->n) {
    PHX_HIP(hipMemcpyAsync(W->rows, W->h_rows.data(), sizeof(int32_t) * W->n, hipMemcpyHostToDevice, st));
    PHX_HIP(hipMemcpyAsync(W->rlen, rlen.data(), sizeof(int32_t) * W->n, hipMemcpyHostToDevice, st));
  }
  PHX_HIP(hipMemcpyAsync(W->chunk_ptr, cptr.data(), sizeof(int64_t) * cptr.size(), hipMemcpyHostToDevice, st));
  PHX_HIP(hipMemcpyAsync(W->col, ccol.data(), sizeof(int32_t) * ccol.size(), hipMemcpyHostToDevice, st));
  PHX_HIP(hipMemcpyAsync(W->val, cval.data(), sizeof(T) * cval.size(), hipMemcpyHostToDevice, st));
  sync_stream();  // the host staging vectors die here
  return W;
}

template <typename T>
void carp_destroy(void* work) {
  auto* W = static_cast<CarpWork<T>*>(work);
  if (!W) return;
  sync_stream();
  if (W->rows) PHX_HIP(hipFree(W->rows));
  if (W->rlen) PHX_HIP(hipFree(W->rlen));
  if (W->chunk_ptr) PHX_HIP(hipFree(W->chunk_ptr));
  if (W->col) PHX_HIP(hipFree(W->col));
  if (W->val) PHX_HIP(hipFree(W->val));
  delete W;
}

template <typename T, bool RC, int VPL, int LB, bool ONE, typename... Args>
void kacz_go(const int32_t* rows, const int32_t* rlen, const int64_t* cptr, int64_t nr, const int32_t* ci, const T* va,
             int lpr, Args... args) {
  const int64_t rpt = kBlock / lpr, ntiles = (nr + rpt - 1) / rpt;
  const int grid = persistent_blocks(k_kacz<T, RC, VPL, LB, ONE>, 0, ntiles);
  hipLaunchKernelGGL((k_kacz<T, RC, VPL, LB, ONE>), dim3(grid), dim3(kBlock), 0, rt().stream, rows, rlen, cptr, nr,
                     ntiles, ci, va, lpr, args...);
  PHX_HIP(hipGetLastError());
}

// one colour on nc columns: vector lanes where every block's rows are whole
// 16-byte vectors (real shifts; the complex update holds twice the values),
// and the batch that takes the longest row at once, up to 16 entries
template <typename T>
void kacz_launch(const int32_t* rows, const int32_t* rlen, const int64_t* cptr, int64_t nr, int32_t max_len,
                 const int32_t* ci, const T* va, int nc, const CarpCoef<T>& coef, const T* b, int64_t ldb, T* xr,
                 T* xi, int64_t ldx) {
  constexpr int V = 16 / sizeof(T);
  auto al = [](const T* p, int64_t ld) { return ((uintptr_t)p & 15) == 0 && ld % V == 0; };
  const bool vec = !xi && nc % V == 0 && al(xr, ldx) && (!b || al(b, ldb));
#define PHX_KACZ(RC, VPL)                                                                                            \
  (max_len <= 8    ? kacz_go<T, RC, VPL, 8, true>(rows, rlen, cptr, nr, ci, va, nc / VPL, coef, b, ldb, xr, xi, ldx)  \
   : max_len <= 16 ? kacz_go<T, RC, VPL, 16, true>(rows, rlen, cptr, nr, ci, va, nc / VPL, coef, b, ldb, xr, xi, ldx) \
                   : kacz_go<T, RC, VPL, 8, false>(rows, rlen, cptr, nr, ci, va, nc / VPL, coef, b, ldb, xr, xi, ldx))
  if (xi)
    PHX_KACZ(true, 1);
  else if (vec)
    PHX_KACZ(false, V);
  else
    PHX_KACZ(false, 1);
#undef PHX_KACZ
}

// forward then backward sweep over the colours; B may be null (b = 0),
// si and Xi null for real shifts
template <typename T>
void carp_sweep(const SparseMat<T>* A, void* work, const T* sr, const T* si, const Mvec<T>* B, Mvec<T>* Xr,
                Mvec<T>* Xi, const T* omega) {
  auto* W = static_cast<CarpWork<T>*>(work);
  PHX_REQUIRE(W, PHIST_INVALID_INPUT, "CARP work object is NULL (call carp_setup first)");
  PHX_REQUIRE(W->n == A->nrows, PHIST_INVALID_INPUT, "CARP work object belongs to another matrix");
  const int nvec = Xr->nvec;
  PHX_REQUIRE(sr && omega, PHIST_INVALID_INPUT, "sigma and omega must hold one entry per column of X");
  PHX_REQUIRE(Xr->nrows == W->n && (!B || (B->nrows == W->n && B->nvec == nvec)), PHIST_INVALID_INPUT,
              "vector shapes do not match the matrix");
  PHX_REQUIRE(!Xi || (Xi->nrows == W->n && Xi->nvec == nvec && Xi->lda == Xr->lda), PHIST_INVALID_INPUT,
              "X_i must match X_r");
  ktimer_begin();  // whole sweep (all colour launches) when the kernel timer is on
  // columns are independent: blocks of up to kCarpCols columns sweep one after another
  for (int c0 = 0; c0 < nvec; c0 += kCarpCols) {
    const int nc = std::min(kCarpCols, nvec - c0);
    CarpCoef<T> coef{};
    for (int c = 0; c < nc; c++) {
      coef.sr[c] = sr[c0 + c];
      coef.si[c] = si ? si[c0 + c] : T(0);
      coef.w[c] = omega[c0 + c];
    }
    const T* bp = B ? B->dev() + c0 : nullptr;
    const int64_t ldb = B ? B->lda : 0;
    T* xr = Xr->dev() + c0;
    T* xi = Xi ? Xi->dev() + c0 : nullptr;
    auto run = [&](int c) {
      const int64_t r0 = W->color_ptr[c], nr = W->color_ptr[c + 1] - r0;
      if (nr == 0) return;
      kacz_launch<T>(W->rows + r0, W->rlen + r0, W->chunk_ptr + W->color_chunk[c], nr, W->max_len, W->col, W->val, nc,
                     coef, bp, ldb, xr, xi, Xr->lda);
    };
    for (int c = 0; c < W->ncolors; c++) run(c);
    for (int c = W->ncolors - 1; c >= 0; c--) run(c);
  }
  ktimer_end();
}

template <typename T>
void carp_colors(void* work, int* ncolors, int64_t* color_ptr, int32_t* rows) {
  auto* W = static_cast<CarpWork<T>*>(work);
  PHX_REQUIRE(W, PHIST_INVALID_INPUT, "NULL work object");
  *ncolors = W->ncolors;
  if (color_ptr) std::copy(W->color_ptr.begin(), W->color_ptr.end(), color_ptr);
  if (rows) std::copy(W->h_rows.begin(), W->h_rows.end(), rows);
}

#define PHX_INST(T)                                                                                           \
  template void* carp_setup<T>(const SparseMat<T>*, int);                                                     \
  template void carp_destroy<T>(void*);                                                                       \
  template void carp_sweep<T>(const SparseMat<T>*, void*, const T*, const T*, const Mvec<T>*, Mvec<T>*, Mvec<T>*, \
                              const T*);                                                                      \
  template void carp_colors<T>(void*, int*, int64_t*, int32_t*);
PHX_INST(double)
PHX_INST(float)
#undef PHX_INST

}  // namespace phx
