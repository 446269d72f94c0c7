// k_spmm.hip — CSR x dense (SpMM) kernels for gfx950.
//
// C = alpha*A*B + beta*C with the reference's rules
// (spmm_rowwise_csr_blocked_m_kernel, src/compressed_sparse_rows.cpp:1699-1745,
// and the C zeroing of src/matmul.cpp:596-605): beta == 0 never reads C.
//
// B and C are row-major (the entry points lay others out again first): k_spmm_tile or
// k_spmm_lds where a block of rows shares its B rows, else k_spmm_gather.
#include <algorithm>
#include <type_traits>

#include "k_common.hpp"
#include "plsparse.hpp"

namespace plk {

// Rows whose B rows are not shared within a block (scattered columns), and
// k < 8: C rows accumulated straight from the gathered B rows.  A window of
// G * VW columns is read by G lanes, VW adjacent columns each: 16 bytes where
// k allows, with element alignment only, so odd k and ld take the same path
// (the lane that would run past column k starts at k - VW and stores only its
// own columns).  S lane groups share a row, each taking every S-th pair of
// non-zeros, and fold with xor shuffles.  S * kGatherPairs pairs cover a row
// of the mean length in one step (quarter or double S measured 1.2-1.9x slower
// at k <= 16 on the 27-point stencil).  A row of more than pls::kSpmmLongRow
// non-zeros has a workgroup of its own, the first nlong of the grid, so the
// longest rows start first.  Bound: latency of row pointer -> entries -> B rows
// for short products, the MALL rate of the gathered B rows for large ones
// (power-law 262,144 rows, FP32 k = 64: 1.35 GB of B rows in 0.22 ms, 6.0
// TB/s).  One lane group per row with 4 non-zeros in flight and scalar B loads
// took 1.19 ms there (the longest row, ~1,100 non-zeros, outlasted the rest),
// and row blocks staged in LDS (k <= 16) 0.36 ms against 0.067 at k = 8.
template <int G> constexpr int kGatherPairs = G <= 2 ? 2 : 4;

template <int G, int VW, class V, class X, bool BETA>
__global__ __launch_bounds__(kBlock) void k_spmm_gather(
    int32_t row0, int32_t m, int32_t k, int32_t win0, int32_t S, int32_t nlong,
    const int32_t *__restrict__ longrow, const int32_t *__restrict__ rp,
    const int32_t *__restrict__ ci, const V *__restrict__ val, const X *__restrict__ B,
    int64_t ldb, X *__restrict__ Cm, int64_t ldc, acc_t<X> alpha, acc_t<X> beta) {
  using A = acc_t<X>;
  typedef X XV __attribute__((ext_vector_type(VW), aligned(sizeof(X))));
  constexpr int U = kGatherPairs<G>;  // entry pairs in flight per lane
  __shared__ A red[kBlock / 64][G * VW];
  const bool whole = int32_t(blockIdx.x) < nlong;  // the workgroup shares one long row
  const int tid = threadIdx.x, lane = tid & (G - 1);
  if (whole) S = 64 / G;
  const int sub = (tid & (G * S - 1)) / G;
  int64_t row;
  if (whole) row = longrow[blockIdx.x];
  else row = row0 + (int64_t(xcd_swizzle(blockIdx.x - nlong, gridDim.x - nlong)) * kBlock + tid) / (G * S);
  // the lane's first column, and where its vector starts
  const int64_t own = int64_t(win0 + int32_t(blockIdx.y)) * (G * VW) + lane * VW;
  const int64_t c0 = min(own, int64_t(k - VW));
  bool live = whole || row < m;
  uint32_t p0 = 0, p1 = 0;
  if (live) {
    p0 = uint32_t(rp[row]);
    p1 = uint32_t(rp[row + 1]);
    live = whole || p1 - p0 <= uint32_t(pls::kSpmmLongRow);  // else another workgroup's
  }
  A acc[VW];
#pragma unroll
  for (int t = 0; t < VW; ++t) acc[t] = A(0);
  if (live && p0 < p1) {
    // entries in aligned pairs (one 8-byte index load, one 2-value load; the
    // plan's arrays end with one padding entry), those outside the row masked
    const uint32_t step = 2 * (whole ? S * (kBlock / 64) : S), last = (p1 - 1) & ~1u;
    const X *Bc = B + c0;
    for (uint32_t p = (p0 & ~1u) + 2 * (sub + (whole ? (tid >> 6) * S : 0)); p < p1;
         p += U * step) {
      int32_t c[U][2];
      A a[U][2];
#pragma unroll
      for (int u = 0; u < U; ++u) ld_pair(ci, val, int32_t(min(p + u * step, last)), c[u], a[u]);
      XV b[U][2];
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int h = 0; h < 2; ++h)
          b[u][h] = *reinterpret_cast<const XV *>(Bc + int64_t(c[u][h]) * ldb);
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const uint32_t q = p + u * step + h;
          const bool ok = q >= p0 && q < p1;
          const A w = alpha * a[u][h];
#pragma unroll
          for (int t = 0; t < VW; ++t) acc[t] = ok ? acc[t] + w * A(b[u][h][t]) : acc[t];
        }
    }
  }
  for (int o = G; o < G * S; o <<= 1)
#pragma unroll
    for (int t = 0; t < VW; ++t) acc[t] += __shfl_xor(acc[t], o);
  if (whole) {
    if (sub == 0)
#pragma unroll
      for (int t = 0; t < VW; ++t) red[tid >> 6][lane * VW + t] = acc[t];
    __syncthreads();
    if (tid >= G) return;
#pragma unroll
    for (int t = 0; t < VW; ++t)
      acc[t] = (red[0][lane * VW + t] + red[1][lane * VW + t]) +
               (red[2][lane * VW + t] + red[3][lane * VW + t]);
  }
  if (!live || sub != 0 || own >= k) return;
  X *c = Cm + row * ldc + c0;
  if (c0 == own) {
    XV o;
    if (BETA) o = *reinterpret_cast<const XV *>(c);
#pragma unroll
    for (int t = 0; t < VW; ++t) {
      A r = acc[t];
      if (BETA) r += beta * A(o[t]);
      o[t] = X(r);
    }
    *reinterpret_cast<XV *>(c) = o;
  } else {
#pragma unroll
    for (int t = 0; t < VW; ++t)
      if (c0 + t >= own) {
        A r = acc[t];
        if (BETA) r += beta * A(c[t]);
        c[t] = X(r);
      }
  }
}

// One element of C.
template <class X, bool BETA>
__device__ __forceinline__ void store_one(X *c, acc_t<X> v, acc_t<X> alpha, acc_t<X> beta) {
  acc_t<X> r = alpha * v;
  if (BETA) r += beta * acc_t<X>(*c);
  *c = X(r);
}

// x[i] of an array in registers.
template <int N> __device__ __forceinline__ int64_t pick(const uint32_t (&x)[N], int32_t i) {
  uint32_t v = x[0];
#pragma unroll
  for (int j = 1; j < N; ++j) v = i == j ? x[j] : v;
  return v;
}

// VW columns of one C row from column c0 on; the lane owns those from `own` on.
template <int VW, class X, bool BETA>
__device__ __forceinline__ void store_cols(X *crow, int64_t c0, int64_t own, int32_t k,
                                           const acc_t<X> (&v)[VW], acc_t<X> alpha,
                                           acc_t<X> beta) {
  using A = acc_t<X>;
  typedef X XV __attribute__((ext_vector_type(VW), aligned(sizeof(X))));
  if (own >= k) return;
  X *c = crow + c0;
  if (c0 == own) {
    XV o;
    if (BETA) o = *reinterpret_cast<const XV *>(c);
#pragma unroll
    for (int t = 0; t < VW; ++t) {
      A r = alpha * v[t];
      if (BETA) r += beta * A(o[t]);
      o[t] = X(r);
    }
    *reinterpret_cast<XV *>(c) = o;
  } else {
#pragma unroll
    for (int t = 0; t < VW; ++t)
      if (c0 + t >= own) {
        A r = alpha * v[t];
        if (BETA) r += beta * A(c[t]);
        c[t] = X(r);
      }
  }
}

// The same in a wave with a NaN among its results (redo): an element that is NaN
// is not stored; the returned bits name them.
template <int VW, class X, bool BETA>
__device__ __forceinline__ uint32_t store_or_mark(bool redo, X *crow, int64_t c0, int64_t own,
                                                  int32_t k, const acc_t<X> (&v)[VW],
                                                  acc_t<X> alpha, acc_t<X> beta) {
  uint32_t nans = 0;
  if (!redo) {
    store_cols<VW, X, BETA>(crow, c0, own, k, v, alpha, beta);
  } else {
#pragma unroll
    for (int e = 0; e < VW; ++e) {
      if (c0 + e < own) continue;
      if (v[e] == v[e]) store_one<X, BETA>(crow + c0 + e, v[e], alpha, beta);
      else nans |= 1u << e;
    }
  }
  return nans;
}

// Row tiles (pls::spmm_on_tiles: operands whose rows share columns, k > 16): one
// wave multiplies a tile of up to 32 rows, two halves of 16, by a window of NW *
// 16 * VW columns of B on the matrix cores.  The tile's distinct columns are
// listed four to a step; a step's B rows are read once, VW adjacent columns per
// lane (the columns of a window are permuted), and serve both halves through
// v_mfma_f64_16x16x4 / v_mfma_f32_16x16x4.  alpha is multiplied into the values, as
// in the other CSR kernels.  The values stay compressed: per step
// and half the non-zero ones in lane order behind a 64-bit mask of the lanes
// that have one.  They are copied to the wave's LDS slice with full-width loads
// one group of G steps ahead, and each lane picks its own by counting mask bits
// (picked straight from global memory, and with 16 rows per tile, the texture
// path was busy 74% of the kernel and FP64 k = 32 took 129 us below).  Columns
// of one half alone come first and last, so those steps skip the other half.
// Windows are the slow grid index and the grid a multiple of 8, so an XCD sweeps
// its own tiles one window at a time and the B rows of a sweep stay in its L2
// (two windows at k = 128 side by side: 446 us against 421).
// Bound: 27-point stencil 96^3, FP64 k = 32, 203 us (floor 156 at the copy rate,
// matrix cores 106), k = 128 on 80^3 408 us (floor 257): matrix cores about half
// busy and 2.5 GB moved for 1.2 GB, B rows fetched again across grid planes.
// k_spmm_lds took 275 and 553 us there, with its present staging 497 at k = 128.
// An element that comes out NaN is computed again entry by entry: a column some
// row of the tile does not have is multiplied by zero for that row, which changes
// nothing unless the B value is infinite or NaN, and then leaves NaN in that
// element.  A wave with such elements stores the others, lists these in its LDS
// slice and takes one per lane, up to the first NaN (27-point 80^3, FP64 k = 32,
// 122 us: one bad entry 124, a column of NaN 181, of infinities 274, all of B NaN
// 269; all elements of such waves one after the other 221 / 1488 / 1488 / 1486).
template <class X> struct TileAcc;
template <> struct TileAcc<double> {
  typedef double T __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ T mma(double a, double b, T c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int kk, int r) { return 4 * r + kk; }
};
template <> struct TileAcc<float> {
  typedef float T __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ T mma(float a, float b, T c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int kk, int r) { return 4 * kk + r; }
};

// One element of alpha*A*B from its entries, four in flight, up to the first NaN.
template <class V, class X>
__device__ __forceinline__ acc_t<X> csr_dot(acc_t<X> alpha, int32_t p0, int32_t p1, int64_t c,
                                            const int32_t *ci, const V *val, const X *Bm,
                                            int64_t ldb) {
  using A = acc_t<X>;
  A s = 0;
  for (int32_t p = p0; p < p1 && s == s; p += 4) {
    A a[4], b[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int32_t q = min(p + u, p1 - 1);
      a[u] = alpha * A(ldv(val, q));
      b[u] = A(Bm[int64_t(ci[q]) * ldb + c]);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) s = p + u < p1 ? s + a[u] * b[u] : s;
  }
  return s;
}
template <int NW, int VW, class V, class X, bool BETA>
__global__ __launch_bounds__(kBlock, 4) void k_spmm_tile(
    int32_t tile0, int32_t ntiles, int32_t win0, int32_t k, const pls::SpmmTile *__restrict__ tiles,
    const int32_t *__restrict__ trow, const uint64_t *__restrict__ mask,
    const int32_t *__restrict__ tcol, const V *__restrict__ tval, const int32_t *__restrict__ rp,
    const int32_t *__restrict__ ci, const V *__restrict__ val, const X *__restrict__ Bm,
    int64_t ldb, X *__restrict__ Cm, int64_t ldc, acc_t<X> alpha, acc_t<X> beta) {
  using A = acc_t<X>;
  using M = TileAcc<X>;
  typedef X XV __attribute__((ext_vector_type(VW), aligned(sizeof(X))));
  constexpr int G = 4;       // steps in flight
  constexpr int PF = G / 2;  // prefetched value registers: 64 values each
  __shared__ A lds[kBlock / 64][G * 128];  // the values of G steps
  const int lane = threadIdx.x & 63, n = lane & 15, kk = lane >> 4;
  A *av = lds[threadIdx.x >> 6];
  const int32_t tile = tile0 + int32_t(xcd_swizzle(blockIdx.x, gridDim.x)) * (kBlock / 64) +
                       __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (tile >= ntiles) return;
  const int32_t pass = win0 + int32_t(blockIdx.y);
  const pls::SpmmTile t0 = tiles[tile], t1 = tiles[tile + 1];
  uint32_t own[NW];  // below 2^31 + a window
  int32_t c0[NW];    // -1 where a window of one column (k = 1) is the rest of a wider B
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    own[w] = (uint32_t(pass) * NW + w) * (16 * VW) + n * VW;
    c0[w] = int32_t(min(int64_t(own[w]), int64_t(k - VW)));
  }
  typename M::T acc[2][NW][VW];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int w = 0; w < NW; ++w)
#pragma unroll
      for (int e = 0; e < VW; ++e) acc[h][w][e] = typename M::T{0, 0, 0, 0};
  const V *tv = tval + t0.val0;
  const uint32_t ld = uint32_t(ldb);
  A pf[PF];
#pragma unroll
  for (int i = 0; i < PF; ++i) pf[i] = A(ldv(tv, lane + 64 * i));
  for (int32_t q0 = t0.step0; q0 < t1.step0; q0 += 16) {
    // columns of the next 16 steps, one per lane (past the last: the last
    // one), and their masks, two per step (past the last: 0)
    const int32_t ns = min(t1.step0 - q0, 16);
    const int32_t cv = ldi(tcol, 4 * int64_t(q0) + min(lane, 4 * ns - 1));
    const uint64_t mv = lane < 2 * ns ? mask[2 * int64_t(q0) + lane] : 0;
    for (int32_t s = 0; s < ns; s += G) {
      XV b[G][NW];
#pragma unroll
      for (int u = 0; u < G; ++u) {
        const uint32_t col = __builtin_amdgcn_ds_bpermute(kk * 4 + s * 16 + u * 16, cv);
        const X *bp = Bm + uint64_t(col) * ld;
#pragma unroll
        for (int w = 0; w < NW; ++w) b[u][w] = *reinterpret_cast<const XV *>(bp + c0[w]);
      }
      uint64_t m[G][2];
      int32_t nv = 0;
#pragma unroll
      for (int u = 0; u < G; ++u)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const uint32_t hi = __builtin_amdgcn_readlane(uint32_t(mv >> 32), 2 * (s + u) + h),
                         lo = __builtin_amdgcn_readlane(uint32_t(mv), 2 * (s + u) + h);
          m[u][h] = uint64_t(hi) << 32 | lo;
          nv += __builtin_popcountll(m[u][h]);
        }
#pragma unroll
      for (int i = 0; i < PF; ++i) av[lane + 64 * i] = alpha * pf[i];
      for (int32_t i = 64 * PF; i < nv; i += 64) av[lane + i] = alpha * A(ldv(tv, lane + i));
      tv += nv;
#pragma unroll
      for (int i = 0; i < PF; ++i) pf[i] = A(ldv(tv, lane + 64 * i));
      __builtin_amdgcn_wave_barrier();
      const A *ap = av;
#pragma unroll
      for (int u = 0; u < G; ++u)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          if (m[u][h] == 0) continue;
          A a = ap[__builtin_amdgcn_mbcnt_hi(uint32_t(m[u][h] >> 32),
                                             __builtin_amdgcn_mbcnt_lo(uint32_t(m[u][h]), 0))];
          a = __builtin_amdgcn_inverse_ballot_w64(m[u][h]) ? a : A(0);
          ap += __builtin_popcountll(m[u][h]);
#pragma unroll
          for (int w = 0; w < NW; ++w)
#pragma unroll
            for (int e = 0; e < VW; ++e) acc[h][w][e] = M::mma(a, A(b[u][w][e]), acc[h][w][e]);
        }
      __builtin_amdgcn_wave_barrier();
    }
  }
  const int32_t nrows = t1.row0 - t0.row0;
  bool nan = false;
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int w = 0; w < NW; ++w)
#pragma unroll
      for (int e = 0; e < VW; ++e)
#pragma unroll
        for (int r = 0; r < 4; ++r) nan = nan || acc[h][w][e][r] != acc[h][w][e][r];
  const bool redo = __any(nan);
  uint64_t nans = 0;  // the lane's elements to be computed again
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int32_t i = M::row(kk, r) + (h ? t0.half : 0);
      if (i >= (h ? nrows : t0.half)) continue;
      const int32_t row = trow[t0.row0 + i];
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        A out[VW];
#pragma unroll
        for (int e = 0; e < VW; ++e) out[e] = acc[h][w][e][r];
        nans |= uint64_t(store_or_mark<VW, X, BETA>(redo, Cm + int64_t(row) * ldc, c0[w], own[w], k,
                                                    out, A(1), beta))
                << (((h * 4 + r) * NW + w) * VW);
      }
    }
  if (!redo) return;
  // listed in the wave's LDS slice as lane + 64 * element, a lane for each
  constexpr int CAP = sizeof(A) * G * 128 / 4, NE = 8 * NW * VW;
  uint32_t *list = reinterpret_cast<uint32_t *>(av);
  int32_t cnt = 0;
  for (int32_t s = 0; s < NE; ++s) {
    const bool mine = nans >> s & 1;
    const uint64_t all = __ballot(mine);
    if (mine)
      list[cnt + int32_t(__builtin_amdgcn_mbcnt_hi(
                     uint32_t(all >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(all), 0)))] =
          uint32_t(lane + 64 * s);
    cnt += __builtin_popcountll(all);
    if (s + 1 < NE && cnt + 64 <= CAP) continue;
    __builtin_amdgcn_wave_barrier();
    for (int32_t j = lane; j < cnt; j += 64) {
      const int32_t l = int32_t(list[j] & 63u), el = int32_t(list[j] >> 6);
      const int32_t e = el % VW, w = el / VW % NW, r = el / (VW * NW) & 3, h = el / (VW * NW * 4);
      const int32_t row = trow[t0.row0 + M::row(l >> 4, r) + (h ? t0.half : 0)];
      const int64_t c = min((int64_t(pass) * NW + w) * (16 * VW) + (l & 15) * VW, int64_t(k - VW)) + e;
      store_one<X, BETA>(Cm + int64_t(row) * ldc + c,
                         csr_dot<V, X>(alpha, rp[row], rp[row + 1], c, ci, val, Bm, ldb), A(1), beta);
    }
    __builtin_amdgcn_wave_barrier();
    cnt = 0;
  }
}

// Column-compressed row blocks (k >= 8 when the plan's block lists are short
// enough, see build_spmm_blocks, and the product is not one for the row tiles
// above): one workgroup per block of rows, consecutive ones or (brow !=
// nullptr) the rows brow lists for the block, whose non-zeros the plan keeps in
// block order (prp, lval, lidx: one contiguous range per block, like
// consecutive rows).  The block's alpha-scaled values and list positions are
// staged in LDS once (loaded in aligned pairs); then, KC columns at a time,
// every B row the block needs is loaded into LDS once (coalesced, KC contiguous
// elements per row, 16 bytes per lane) and each row of C is accumulated from
// LDS by a group of KC / CPL lanes (CPL adjacent columns each, written as one
// vector), 8 non-zeros in flight per lane.  On the 27-point stencil a staged B
// row feeds about 5 non-zeros of a block of clustered rows (2.6 with
// consecutive rows), so L2 -> CU traffic for B falls by that factor against the
// direct kernels, which fetch a B row per non-zero.
// Bound by the block's chain of loads and barriers and by the instructions per
// non-zero (FP32, k = 8: vector units busy 70% of the time when every step of 8
// masked its tail).  So a block's record is one load, and every load of its row
// starts, rows, list and entries is in flight before the first LDS store; a row
// is walked in steps of 8, 4, 2 and 1 without masks (from 4 where a lane's
// columns take more than 16 bytes: the registers of 8 cost FP64 k = 16 a
// workgroup per CU, 98 -> 109 us); and FP32 chunks of up to 16 columns keep an
// entry as one 8-byte LDS read, value and byte offset of its B row (PACK; chunks
// of 32 lose a workgroup by the larger entries, 7-point 80^3 k = 32 47 -> 49 us).
// us, masked steps of 8 -> unmasked -> loads in flight together: 27-point 80^3
// FP32 k = 8 / 16 59.1 / 66.7 -> 54.6 / 60.0 -> 44.6 / 51.5, FP64 68.0 / 100.1 ->
// 64.9 / 97.7 -> 52.9 / 82.2; 5-point 1000^2 FP32 k = 8 / 32 34.2 / 66.2 -> 32.0 /
// 63.3 -> 28.0 / 51.4; 8 x 8 block stencil FP64 k = 16 50.1 -> 42.8 -> 38.1.
// Slower: a row's parts summed in contiguous pieces or four columns per lane at
// k = 8 (FP64 64.9 -> 77), a persistent launch that prefetches the next block
// (FP32 k = 8 / 16 61 / 83: it loses its occupancy), the first chunk's B loads
// addressed from registers before the first barrier (FP64 k = 16 82 -> 99).
// A block without a list (one row with more than UMAX distinct columns or
// lb_nnz_per_ucol(UMAX) * UMAX non-zeros) spreads its non-zeros over the
// workgroup's lane groups, reads B directly and sums the groups through LDS.
template <int KC, int UMAX, int CPL, class V, class X, bool BETA>
__global__ __launch_bounds__(kBlock) void k_spmm_lds(
    const pls::SpmmBlock *__restrict__ blocks, const int32_t *__restrict__ ucol,
    const uint8_t *__restrict__ lidx,
    const int32_t *__restrict__ brow, const int32_t *__restrict__ prp,
    const V *__restrict__ lval, int32_t k, const int32_t *__restrict__ rp,
    const int32_t *__restrict__ ci, const V *__restrict__ val, const X *__restrict__ B,
    int64_t ldb, X *__restrict__ Cm, int64_t ldc, acc_t<X> alpha, acc_t<X> beta) {
  using A = acc_t<X>;
  constexpr int NG = kBlock / KC;  // lane groups (rows in flight) per workgroup
  __shared__ __align__(16) A sB[UMAX * KC];
  constexpr int NNZ = pls::lb_nnz_per_ucol(UMAX) * UMAX;
  constexpr bool PACK = KC <= 16 && sizeof(A) == 4;
  __shared__ uint2 s_e[PACK ? NNZ : 1];  // an entry's value and byte offset of its B row
  __shared__ A s_a[PACK ? 1 : NNZ];
  __shared__ uint8_t s_l[PACK ? 1 : NNZ];
  __shared__ int32_t s_rp[pls::kLbRows + 1];
  __shared__ int32_t s_uc[UMAX];
  __shared__ int32_t s_row[pls::kLbRows];  // clustered blocks: the rows' indices
  const uint32_t blk = xcd_swizzle(blockIdx.x, gridDim.x);
  const int tid = threadIdx.x, lane = tid % KC, grp = tid / KC;
  const pls::SpmmBlock bk = blocks[blk];
  const int32_t r0 = bk.r0, nrows = bk.nrows, nu = bk.nu, e0 = bk.e0, nnz = bk.nnz;
  // block-order arrays (the CSR arrays for consecutive rows)
  const int32_t *brp = brow ? prp : rp;
  const V *bval = brow ? lval : val;

  if (nu == 0 && nnz > 0) {  // one long row without a list: B read directly
    const int32_t row = brow ? brow[r0] : r0, f0 = rp[row];  // its CSR non-zeros
    for (int32_t c0 = 0; c0 < k; c0 += KC) {
      const int32_t col = c0 + lane;
      A acc = 0;
      if (col < k)
        for (int32_t p = grp; p < nnz; p += NG)
          acc += alpha * A(ldv(val, f0 + p)) * A(B[int64_t(ldi(ci, f0 + p)) * ldb + col]);
      sB[grp * KC + lane] = acc;
      __syncthreads();
      if (grp == 0 && col < k) {
        A r = 0;
        for (int g = 0; g < NG; ++g) r += sB[g * KC + lane];
        X *c = Cm + int64_t(row) * ldc + col;
        if (BETA) r += beta * A(*c);
        *c = X(r);
      }
      __syncthreads();
    }
    return;
  }

  {
    // every load of the block's row starts, rows, list and entries in flight
    // before the first LDS store; values and list positions in aligned pairs
    // from the even index at or below e0 (both arrays end with one padding entry)
    constexpr int NP = NNZ / 2 / kBlock + 1;
    static_assert(pls::kLbRows < kBlock && UMAX <= kBlock);
    typedef uint8_t L2 __attribute__((ext_vector_type(2)));
    const int32_t start = brp[r0 + min(tid, nrows)];
    const int32_t row = brow ? brow[r0 + min(tid, nrows - 1)] : 0;
    const int32_t uc = nu > 0 ? ucol[bk.u0 + min(tid, nu - 1)] : 0;
    const int32_t a0 = e0 & ~1, sh = e0 - a0, last = (e0 + nnz - 1) & ~1;
    A v[NP][2];
    L2 l[NP];
    if (nnz > 0)
#pragma unroll
      for (int u = 0; u < NP; ++u) {
        const int32_t j = min(a0 + 2 * (tid + u * kBlock), last);
        ld_val_pair(bval, j, v[u]);
        l[u] = *reinterpret_cast<const L2 *>(lidx + j);
      }
    if (tid <= nrows) s_rp[tid] = start - e0;
    if (brow && tid < nrows) s_row[tid] = row;
    if (tid < nu) s_uc[tid] = uc;
    auto put = [&](int32_t at, A a, uint8_t pos) {
      if (at < 0 || at >= nnz) return;
      if constexpr (PACK) {
        s_e[at] = make_uint2(__float_as_uint(alpha * a), pos * uint32_t(KC * sizeof(A)));
      } else {
        s_a[at] = alpha * a;
        s_l[at] = pos;
      }
    };
#pragma unroll
    for (int u = 0; u < NP; ++u) {
      const int32_t q = 2 * (tid + u * kBlock) - sh;
      put(q, v[u][0], l[u].x);
      put(q + 1, v[u][1], l[u].y);
    }
  }
  __syncthreads();
  // compute mapping: G = KC / CPL lanes per row group, CPL adjacent columns
  // per lane (read from LDS as one vector); S groups of one wave share a row
  // when the block has few (long) rows, each taking every S-th non-zero, and
  // xor shuffles fold them
  constexpr int G = KC / CPL, NGC = kBlock / G;
  int S = 1;
  while (S * 2 * G <= 64 && nrows * S * 2 <= NGC) S *= 2;
  const int lc = tid % G, sub = (tid % (G * S)) / G;
  for (int32_t c0 = 0; c0 < k; c0 += KC) {
    {
      // B rows of the list, columns [c0, c0 + KC), 16 bytes per lane with
      // element alignment only: half (FP64) or a quarter (FP32) of the load
      // instructions of one element per lane
      constexpr int VW = 16 / sizeof(X), LR = KC / VW, NGV = kBlock / LR;
      constexpr int NIFV = UMAX / NGV < 1 ? 1 : UMAX / NGV < 8 ? UMAX / NGV : 8;
      typedef X XV __attribute__((ext_vector_type(VW)));
      typedef X XU __attribute__((ext_vector_type(VW), aligned(sizeof(X))));
      const int lv = tid % LR;
      const int32_t cv = c0 + lv * VW;
      const bool full = cv + VW <= k;
      for (int32_t i0 = tid / LR; i0 < nu; i0 += NIFV * NGV) {
        XV t[NIFV];
#pragma unroll
        for (int s = 0; s < NIFV; ++s) {
          const X *src = B + int64_t(s_uc[min(i0 + s * NGV, nu - 1)]) * ldb + cv;
          if (full) {
            t[s] = *reinterpret_cast<const XU *>(src);
          } else {
#pragma unroll
            for (int e = 0; e < VW; ++e) t[s][e] = cv + e < k ? src[e] : X(0);
          }
        }
#pragma unroll
        for (int s = 0; s < NIFV; ++s)
          if (i0 + s * NGV < nu) *reinterpret_cast<XV *>(&sB[(i0 + s * NGV) * KC + lv * VW]) = t[s];
      }
    }
    __syncthreads();
    for (int32_t rr = tid / (G * S); rr < nrows; rr += kBlock / (G * S)) {
      const int32_t p0 = s_rp[rr], p1 = s_rp[rr + 1];
      A acc[CPL];
#pragma unroll
      for (int t = 0; t < CPL; ++t) acc[t] = 0;
      if constexpr (PACK) {
        // 8, 4, 2 and 1 entries at a time: no clamped index and no select
        const char *bl = reinterpret_cast<const char *>(&sB[lc * CPL]);
        auto run = [&](int32_t p, auto n) {
          constexpr int N = decltype(n)::value;
          typedef A XC __attribute__((ext_vector_type(CPL)));
          uint2 e[N];
          XC x[N];
#pragma unroll
          for (int u = 0; u < N; ++u) e[u] = s_e[p + u * S];
#pragma unroll
          for (int u = 0; u < N; ++u) x[u] = *reinterpret_cast<const XC *>(bl + e[u].y);
#pragma unroll
          for (int u = 0; u < N; ++u)
#pragma unroll
            for (int t = 0; t < CPL; ++t) acc[t] += __uint_as_float(e[u].x) * x[u][t];
          return p + N * S;
        };
        int32_t p = p0 + sub;
        while (p + 7 * S < p1) p = run(p, std::integral_constant<int, 8>{});
        if (p + 3 * S < p1) p = run(p, std::integral_constant<int, 4>{});
        if (p + S < p1) p = run(p, std::integral_constant<int, 2>{});
        if (p < p1) run(p, std::integral_constant<int, 1>{});
      } else {
        auto run = [&](int32_t p, auto n) {
          constexpr int N = decltype(n)::value;
          using A2 = std::conditional_t<sizeof(A) == 8, double2, float2>;
          A a[N];
          int32_t l[N];
#pragma unroll
          for (int u = 0; u < N; ++u) a[u] = s_a[p + u * S];
#pragma unroll
          for (int u = 0; u < N; ++u) l[u] = s_l[p + u * S];
#pragma unroll
          for (int u = 0; u < N; ++u) {
            const A *b = &sB[l[u] * KC + lc * CPL];
#pragma unroll
            for (int h = 0; h < CPL / 2; ++h) {
              const A2 v = reinterpret_cast<const A2 *>(b)[h];
              acc[2 * h] += a[u] * v.x;
              acc[2 * h + 1] += a[u] * v.y;
            }
          }
          return p + N * S;
        };
        int32_t p = p0 + sub;
        if constexpr (CPL * sizeof(A) <= 16)
          while (p + 7 * S < p1) p = run(p, std::integral_constant<int, 8>{});
        while (p + 3 * S < p1) p = run(p, std::integral_constant<int, 4>{});
        if (p + S < p1) p = run(p, std::integral_constant<int, 2>{});
        if (p < p1) run(p, std::integral_constant<int, 1>{});
      }
#pragma unroll
      for (int t = 0; t < CPL; ++t)
        for (int o = G; o < G * S; o <<= 1) acc[t] += __shfl_xor(acc[t], o);
      if (sub == 0) {
        X *c = Cm + int64_t(brow ? s_row[rr] : r0 + rr) * ldc;
        const int32_t cb = c0 + lc * CPL;
        if (cb + CPL <= k) {  // the lane's CPL columns as one vector
          typedef X XC __attribute__((ext_vector_type(CPL), aligned(sizeof(X))));
          XC o;
          if (BETA) o = *reinterpret_cast<const XC *>(c + cb);
#pragma unroll
          for (int t = 0; t < CPL; ++t) {
            A r = acc[t];
            if (BETA) r += beta * A(o[t]);
            o[t] = X(r);
          }
          *reinterpret_cast<XC *>(c + cb) = o;
        } else {
#pragma unroll
          for (int t = 0; t < CPL; ++t) {
            const int32_t cc = cb + t;
            if (cc < k) {
              A r = acc[t];
              if (BETA) r += beta * A(c[cc]);
              c[cc] = X(r);
            }
          }
        }
      }
    }
    __syncthreads();
  }
}

// Few right-hand sides (n < 5, the range where the reference repeats SpMV per
// column, src/matmul.cpp:42-89): the CSR-vector mapping (L lanes per row, L
// from the mean row length) with NR column sums per lane, so A is read once
// for all columns.  op(B) arrives as a row-major block with rows of P >= NR
// values (P in {1, 2, 4}, packed by the caller when its own layout is
// strided), so each non-zero gathers one contiguous piece of B; C is written
// through its strides (for the column-major C the reference materialises,
// lanes of consecutive rows store consecutive addresses of each column).
template <int P, class X> struct Piece;
template <class X> struct Piece<1, X> {
  static __device__ __forceinline__ void load(const X *b, acc_t<X> (&v)[1]) { v[0] = b[0]; }
};
template <class X> struct Piece<2, X> {
  typedef X v2 __attribute__((ext_vector_type(2)));
  static __device__ __forceinline__ void load(const X *b, acc_t<X> (&v)[2]) {
    const v2 t = *reinterpret_cast<const v2 *>(b);
    v[0] = t.x;
    v[1] = t.y;
  }
};
template <class X> struct Piece<4, X> {
  typedef X v4 __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ void load(const X *b, acc_t<X> (&v)[4]) {
    const v4 t = *reinterpret_cast<const v4 *>(b);
    v[0] = t.x;
    v[1] = t.y;
    v[2] = t.z;
    v[3] = t.w;
  }
};

template <int L, int NR, int P, class V, class X, bool BETA>
__global__ __launch_bounds__(kBlock) void k_csr_few_rhs(
    int32_t m, const int32_t *__restrict__ rp, const int32_t *__restrict__ ci,
    const V *__restrict__ val, const X *__restrict__ B, X *__restrict__ Cm, int64_t c_sr,
    int64_t c_sc, acc_t<X> alpha, acc_t<X> beta) {
  using A = acc_t<X>;
  const int64_t t = int64_t(xcd_swizzle(blockIdx.x, gridDim.x)) * kBlock + threadIdx.x;
  const int64_t row = t / L;
  const int lane = threadIdx.x & (L - 1);
  A s[NR];
#pragma unroll
  for (int r = 0; r < NR; ++r) s[r] = A(0);
  if (row < m) {
    // the row's entries in aligned pairs (the CSR plan's arrays end with one
    // padding entry), two pairs in flight per lane; entries outside the row
    // multiply by zero
    const int32_t rs = rp[row], e = rp[row + 1];
    const int32_t last = (e - 1) & ~1;
    constexpr int U = 2;
    for (int32_t j = (rs & ~1) + 2 * lane; j <= last && rs < e; j += 2 * U * L) {
      int32_t c[U][2];
      A a[U][2];
#pragma unroll
      for (int u = 0; u < U; ++u) ld_pair(ci, val, min(j + 2 * u * L, last), c[u], a[u]);
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int32_t q = j + 2 * u * L + h;
          const A w = q >= rs && q < e ? a[u][h] : A(0);
          A b[P];
          Piece<P, X>::load(B + int64_t(c[u][h]) * P, b);
#pragma unroll
          for (int r = 0; r < NR; ++r) s[r] += w * b[r];
        }
    }
  }
#pragma unroll
  for (int r = 0; r < NR; ++r) s[r] = group_sum_c<L>(s[r]);
  if (row < m && lane == 0) {
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      X *c = Cm + row * c_sr + r * c_sc;
      A v = alpha * s[r];
      if (BETA) v += beta * A(*c);
      *c = X(v);
    }
  }
}

// Native BSR x dense (b = 4 or 8, row-major B and C) on the matrix cores: one
// wave per block row and window of B columns, the blocks multiplied as 4 x 4
// tiles by v_mfma_f64_4x4x4 (4 independent products: 70 TFLOP/s measured, the
// scalar FMA rate without its operand traffic; v_mfma_f64_16x16x4 would be
// half padding) or v_mfma_f32_4x4x1 (16 independent products).  The products
// of one instruction are split over NB column tiles and PB blocks of the row,
// so a block value reaches NB lanes and a B value one lane, both 16 bytes of
// adjacent values at a time (permuting the columns of a window or of a block
// costs nothing).  No LDS and few registers: occupancy hides the latency.
// Bound: the block stream and the B rows re-fetched across grid planes.  27
// blocks per row, 8 x 8, block grid 32^3, FP64 k = 8 / 32 / 128: 94 / 168 / 483
// us (4.9 TB/s at k = 8); FP32 37 / 89 / 284.  Scalar FMAs on a b x CPL register
// tile, with the block broadcast from LDS and a select per product for stored
// zeros, took 151 / 292 / 993 and 103 / 159 / 500.
// Loads need element alignment only; a lane that would run past column k
// starts at k - VW and stores only its own columns.
//
// A stored zero adds nothing, as in the zero-dropped CSR product of the
// reference (src/matmul.cpp:619-649), even against an infinite or NaN B value.
// The tiles do multiply stored zeros: 0 * finite adds a zero, which changes
// nothing, and 0 * Inf or 0 * NaN makes the accumulator NaN.  So an element that
// comes out NaN is computed again entry by entry, skipping zeros, up to the first
// NaN, after the wave has stored its others (8 x 8 24^3, FP64 k = 8, 40 us: a
// column of NaN 48, all of B NaN 56; with all elements of such waves computed
// again to their last entry 1812 and 1809).
template <int BS, bool CM, class V, class X>
__device__ __forceinline__ acc_t<X> bsr_dot_nonzero(int32_t p0, int32_t p1, int32_t r, int64_t c,
                                                    const int32_t *ci, const V *val, const X *Bm,
                                                    int64_t ldb) {
  acc_t<X> s = 0;
  for (int32_t p = p0; p < p1 && s == s; ++p) {  // up to the first NaN
    acc_t<X> a[BS], b[BS];
    const X *Bc = Bm + int64_t(ci[p]) * BS * ldb + c;
#pragma unroll
    for (int j = 0; j < BS; ++j) {
      a[j] = acc_t<X>(ldv(val, int64_t(p) * (BS * BS) + (CM ? j * BS + r : r * BS + j)));
      b[j] = acc_t<X>(Bc[j * ldb]);
    }
#pragma unroll
    for (int j = 0; j < BS; ++j) s = a[j] != acc_t<X>(0) ? s + a[j] * b[j] : s;
  }
  return s;
}

// Block values, kept in the caches: several loads share a line (the rows or
// columns of a block, neighbouring block rows of a wave), and one that is not kept
// is fetched again for each (us non-temporal / kept, k = 8: 4 x 4, 9 per row, FP32
// column-major 58 / 23, row-major 33 / 22, FP64 51 / 39; 8 x 8 block grid 32^3 FP32
// 61 / 37).  FP64 blocks are streamed past them in windows of 64 columns and more,
// where the B rows need the room (8 x 8, 7 per row, k = 64 92 / 97), and when they
// are more than the MALL holds (k = 8, 8 x 8 269 MB 64 / 54, 405 MB 91 / 95, 4 x 4
// 349 MB 96 / 99; column-major 8 x 8 blocks, of which a load takes single columns,
// 405 MB 110 / 96), and where few blocks share a row (k = 32, 8 x 8, 3 per row 50 /
// 54, 4 x 4, 7 per row 79 / 83; block-diagonal 4 x 4, k = 24 54 / 60).
template <bool KEEP, class T> __device__ __forceinline__ T ld_block(const T *p) {
  if constexpr (KEEP) return *p;
  else return __builtin_nontemporal_load(p);
}
// N adjacent ones (1, 2, 4; aligned to their size) as one load.
template <int N, class V>
__device__ __forceinline__ void ld_adjacent(const V *p, float (&x)[N]) {
  typedef V VN __attribute__((ext_vector_type(N)));
  const VN t = ld_block<true>(reinterpret_cast<const VN *>(p));
#pragma unroll
  for (int i = 0; i < N; ++i) {
    if constexpr (sizeof(V) == 2) x[i] = __uint_as_float(uint32_t(V(t[i])) << 16);
    else x[i] = t[i];
  }
}

// Blocks a wave steps through: a block row's, or (ROWS) the longest of the
// block rows of its lanes, which differ at the lane bits from FROM to below TO.
template <bool ROWS, int FROM, int TO>
__device__ __forceinline__ int32_t bsr_steps(int32_t n) {
  if (ROWS)
#pragma unroll
    for (int o = FROM; o < TO; o <<= 1) n = max(n, __shfl_xor(n, o));
  return n;
}
// The block of lane group pb at a step: the step's own of its block row (ROWS),
// else one of PB adjacent ones of the wave's, whose columns civ holds.  Past
// the end (on = false) it is a block that exists.
struct BsrAt {
  int32_t p, col;
  bool on;
};
template <bool ROWS, int PB>
__device__ __forceinline__ BsrAt bsr_at(int32_t s, int32_t u, int32_t pb, int32_t nq, int32_t q0,
                                        int32_t p0, int32_t p1, int32_t civ, const int32_t *ci) {
  BsrAt r;
  if (ROWS) {
    const int32_t n = p1 - p0, at = q0 + s + u;
    r.on = at < n;
    r.p = n > 0 ? p0 + min(at, n - 1) : 0;
    r.col = ci[r.p];
  } else {
    const int32_t at = s + u * PB + pb, q = min(at, nq - 1);
    r.on = at < nq;
    r.p = p0 + q0 + q;
    r.col = PB == 1 ? __builtin_amdgcn_readlane(civ, min(s + u, nq - 1)) : __shfl(civ, q);
  }
  return r;
}

// FP64: lane = n + 4 * (nb + NB * pb) + 16 * kk holds A(row i = n, column kk)
// and B(row kk, column n) of product (nb, pb); its result is C(row lane / 16,
// column n).  8 x 8 blocks are T x T = 2 x 2 tiles; the tile of a lane's value
// pair (16 bytes of the block) is chosen by parity: columns 2 kk + kt of
// row-major blocks, rows 2 i + it of column-major ones.
// Block rows per lane of the short-row FP64 kernel.
template <int BS, int NW> constexpr int bsr_rows_f64 = BS == 8 ? 1 : NW == 1 ? 4 : 2;

template <int BS, int NB, int NW, int VW, bool ROWS, bool CM, bool KEEP, bool BETA>
__global__ __launch_bounds__(kBlock) void k_bsr_mfma_f64(
    int64_t unit0, int64_t units, int32_t npass, int32_t mb, int32_t k, const int32_t *__restrict__ rp,
    const int32_t *__restrict__ ci, const double *__restrict__ val, const double *__restrict__ Bm,
    int64_t ldb, double *__restrict__ Cm, int64_t ldc, double alpha, double beta) {
  constexpr int T = BS / 4, PB = 4 / NB, BB = BS * BS;
  // R block rows per lane, or U steps of one, in flight together
  constexpr int R = ROWS ? bsr_rows_f64<BS, NW> : 1, U = ROWS || BS == 8 ? 1 : 2;
  typedef double XV __attribute__((ext_vector_type(VW), aligned(8)));
  typedef double D2 __attribute__((ext_vector_type(2)));
  const int lane = threadIdx.x & 63;
  const int64_t unit = unit0 + int64_t(xcd_swizzle(blockIdx.x, gridDim.x)) * (kBlock / 64) +
                       __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (unit >= units) return;
  const int32_t pass = int32_t(unit % npass);
  const int n = lane & 3, nb = (lane >> 2) % NB, pb = ((lane >> 2) & 3) / NB, kk = lane >> 4;
  const int32_t br = int32_t(unit / npass) * (ROWS ? PB * R : 1) + (ROWS ? pb : 0);
  uint32_t own[NW], c0[NW];  // below 2^31 + a window
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    own[w] = (uint32_t(pass) * NW + w) * (4 * NB * VW) + (nb * 4 + n) * VW;
    c0[w] = min(own[w], uint32_t(k - VW));
  }
  int32_t p0[R], p1[R], steps = 0;
  double acc[R][T][NW][VW];
#pragma unroll
  for (int i = 0; i < R; ++i) {  // block rows br + i * PB
    const bool live = br + i * PB < mb;
    p0[i] = live ? rp[br + i * PB] : 0;
    p1[i] = live ? rp[br + i * PB + 1] : 0;
    steps = max(steps, p1[i] - p0[i]);
#pragma unroll
    for (int it = 0; it < T; ++it)
#pragma unroll
      for (int w = 0; w < NW; ++w)
#pragma unroll
        for (int e = 0; e < VW; ++e) acc[i][it][w][e] = 0.0;
  }
  steps = bsr_steps<ROWS, 4 * NB, 16>(steps);
  for (int32_t q0 = 0; q0 < steps; q0 += 64) {
    const int32_t nq = min(steps - q0, 64);
    int32_t civ = 0;  // the next 64 block columns
    if (!ROWS) civ = ldi(ci, p0[0] + q0 + min(lane, nq - 1));
    for (int32_t s = 0; s < nq; s += (ROWS ? 1 : PB) * U) {
      constexpr int F = R * U;  // blocks in flight: u is a block row or a step
      double a[F][T][T];
      XV b[F][T][NW];
#pragma unroll
      for (int u = 0; u < F; ++u) {
        const int i = u % R;
        const BsrAt at = bsr_at<ROWS, PB>(s, u / R, pb, nq, q0, p0[i], p1[i], civ, ci);
        const double *v = val + int64_t(at.p) * BB;
        const int32_t col = at.col;
        const bool on = at.on;
        if constexpr (T == 2) {
#pragma unroll
          for (int t = 0; t < 2; ++t) {
            const D2 x = ld_block<KEEP>(reinterpret_cast<const D2 *>(
                v + (CM ? (2 * kk + t) * BS + 2 * n : (t * 4 + n) * BS + 2 * kk)));
            a[u][CM ? 0 : t][CM ? t : 0] = on ? x.x : 0.0;
            a[u][CM ? 1 : t][CM ? t : 1] = on ? x.y : 0.0;
          }
        } else {
          const double x = ld_block<KEEP>(v + (CM ? kk * BS + n : n * BS + kk));
          a[u][0][0] = on ? x : 0.0;
        }
#pragma unroll
        for (int kt = 0; kt < T; ++kt)
#pragma unroll
          for (int w = 0; w < NW; ++w)
            b[u][kt][w] = *reinterpret_cast<const XV *>(
                Bm + (int64_t(col) * BS + T * kk + kt) * ldb + c0[w]);
      }
#pragma unroll
      for (int u = 0; u < F; ++u)
#pragma unroll
        for (int kt = 0; kt < T; ++kt)
#pragma unroll
          for (int it = 0; it < T; ++it)
#pragma unroll
            for (int w = 0; w < NW; ++w)
#pragma unroll
              for (int e = 0; e < VW; ++e)
                acc[u % R][it][w][e] = __builtin_amdgcn_mfma_f64_4x4x4f64(
                    a[u][it][kt], b[u][kt][w][e], acc[u % R][it][w][e], 0, 0, 0);
    }
  }
  bool nan = false;
#pragma unroll
  for (int i = 0; i < R; ++i)
#pragma unroll
    for (int it = 0; it < T; ++it)
#pragma unroll
      for (int w = 0; w < NW; ++w)
#pragma unroll
        for (int e = 0; e < VW; ++e) {
          if (!ROWS)
#pragma unroll
            for (int o = 4 * NB; o < 16; o <<= 1)
              acc[i][it][w][e] += __shfl_xor(acc[i][it][w][e], o);
          nan = nan || acc[i][it][w][e] != acc[i][it][w][e];
        }
  const bool redo = __any(nan);
  uint32_t nans = 0;  // the lane's elements to be computed again
#pragma unroll
  for (int i = 0; i < R; ++i) {
    if (br + i * PB >= mb || !(ROWS || pb == 0)) continue;
#pragma unroll
    for (int it = 0; it < T; ++it) {
      const int32_t r = T == 2 ? (CM ? 2 * kk + it : it * 4 + kk) : kk;
#pragma unroll
      for (int w = 0; w < NW; ++w)
        nans |= store_or_mark<VW, double, BETA>(redo, Cm + (int64_t(br + i * PB) * BS + r) * ldc,
                                                c0[w], own[w], k, acc[i][it][w], alpha, beta)
                << (((i * T + it) * NW + w) * VW);
    }
  }
  if (!redo) return;
  for (int32_t s = 0; s < R * T * NW * VW; ++s)
    if (nans >> s & 1) {
      const int32_t e = s % VW, w = s / VW % NW, it = s / (VW * NW) % T, row = br + s / (VW * NW * T) * PB;
      const int32_t r = T == 2 ? (CM ? 2 * kk + it : it * 4 + kk) : kk;
      const int64_t c = pick(c0, w) + e;
      store_one<double, BETA>(Cm + (int64_t(row) * BS + r) * ldc + c,
                              bsr_dot_nonzero<BS, CM, double, double>(rp[row], rp[row + 1], r, c, ci, val, Bm, ldb),
                              alpha, beta);
    }
}

// FP32 (and BF16 values): lane = n + 4 * (nb + NB * (kk + KL * pb)) holds
// A(row i = n, column j) and B(row j, column n) of products of depth one, for
// the KT = BS / KL block columns j = KT * kk + kt, one instruction each (a
// lane's KT values of a row-major block row are one load); register r of the
// results is C(row r, column n), summed over the lanes (kk, pb) at the end,
// which leaves BS of them one row each.
template <int BS, int NB, int NW, int KL, int VW, bool ROWS, bool CM, class V, bool BETA>
__global__ __launch_bounds__(kBlock) void k_bsr_mfma_f32(
    int64_t unit0, int64_t units, int32_t npass, int32_t mb, int32_t k, const int32_t *__restrict__ rp,
    const int32_t *__restrict__ ci, const V *__restrict__ val, const float *__restrict__ Bm,
    int64_t ldb, float *__restrict__ Cm, int64_t ldc, float alpha, float beta) {
  constexpr int T = BS / 4, KT = BS / KL, PB = 16 / (KL * NB), BB = BS * BS;
  static_assert(KL * PB >= BS, "a lane for every row of the block row");
  typedef float XV __attribute__((ext_vector_type(VW), aligned(4)));
  typedef float F4 __attribute__((ext_vector_type(4)));
  const int lane = threadIdx.x & 63;
  const int64_t unit = unit0 + int64_t(xcd_swizzle(blockIdx.x, gridDim.x)) * (kBlock / 64) +
                       __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (unit >= units) return;
  const int32_t pass = int32_t(unit % npass);
  const int n = lane & 3, nb = (lane >> 2) % NB, g = (lane >> 2) / NB, kk = g % KL, pb = g / KL;
  const int32_t br = int32_t(unit / npass) * (ROWS ? PB : 1) + (ROWS ? pb : 0);
  uint32_t own[NW], c0[NW];  // below 2^31 + a window
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    own[w] = (uint32_t(pass) * NW + w) * (4 * NB * VW) + (nb * 4 + n) * VW;
    c0[w] = min(own[w], uint32_t(k - VW));
  }
  const bool live = br < mb;
  const int32_t p0 = live ? rp[br] : 0, p1 = live ? rp[br + 1] : 0;
  const int32_t steps = bsr_steps<ROWS, 4 * NB * KL, 64>(p1 - p0);
  F4 acc[T][NW][VW];
#pragma unroll
  for (int it = 0; it < T; ++it)
#pragma unroll
    for (int w = 0; w < NW; ++w)
#pragma unroll
      for (int e = 0; e < VW; ++e) acc[it][w][e] = F4{0.f, 0.f, 0.f, 0.f};
  for (int32_t q0 = 0; q0 < steps; q0 += 64) {
    const int32_t nq = min(steps - q0, 64);
    int32_t civ = 0;
    if (!ROWS) civ = ldi(ci, p0 + q0 + min(lane, nq - 1));
    for (int32_t s = 0; s < nq; s += ROWS ? 1 : PB) {
      float a[T][KT];
      XV b[KT][NW];
      const BsrAt at = bsr_at<ROWS, PB>(s, 0, pb, nq, q0, p0, p1, civ, ci);
      const V *v = val + int64_t(at.p) * BB;
      const int32_t col = at.col;
      const bool on = at.on;
      // block row it * 4 + n (row-major) or T * n + it (column-major)
      if constexpr (CM) {
#pragma unroll
        for (int kt = 0; kt < KT; ++kt) {
          float x[T];
          ld_adjacent<T>(v + (KT * kk + kt) * BS + T * n, x);
#pragma unroll
          for (int it = 0; it < T; ++it) a[it][kt] = on ? x[it] : 0.f;
        }
      } else {
#pragma unroll
        for (int it = 0; it < T; ++it) {
          float x[KT];
          ld_adjacent<KT>(v + (it * 4 + n) * BS + KT * kk, x);
#pragma unroll
          for (int kt = 0; kt < KT; ++kt) a[it][kt] = on ? x[kt] : 0.f;
        }
      }
#pragma unroll
      for (int kt = 0; kt < KT; ++kt)
#pragma unroll
        for (int w = 0; w < NW; ++w)
          b[kt][w] = *reinterpret_cast<const XV *>(
              Bm + (int64_t(col) * BS + KT * kk + kt) * ldb + c0[w]);
#pragma unroll
      for (int kt = 0; kt < KT; ++kt)
#pragma unroll
        for (int it = 0; it < T; ++it)
#pragma unroll
          for (int w = 0; w < NW; ++w)
#pragma unroll
            for (int e = 0; e < VW; ++e)
              acc[it][w][e] = __builtin_amdgcn_mfma_f32_4x4x1f32(a[it][kt], b[kt][w][e],
                                                                 acc[it][w][e], 0, 0, 0);
    }
  }
  constexpr int L = 4 * NB;  // lane distance of g's lowest bit
  bool nan = false;
  if constexpr (ROWS) {
    // a block row's lanes kk (KL = T of them) exchange tiles: lane kk keeps tile kk
    static_assert(KL == T, "one tile for each lane of a block row");
#pragma unroll
    for (int w = 0; w < NW; ++w)
#pragma unroll
      for (int e = 0; e < VW; ++e)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          if (T == 2) {
            const float keep = kk ? acc[T - 1][w][e][r] : acc[0][w][e][r];
            acc[0][w][e][r] = keep + __shfl_xor(kk ? acc[0][w][e][r] : acc[T - 1][w][e][r], L);
          }
          nan = nan || acc[0][w][e][r] != acc[0][w][e][r];
        }
    const bool redo = __any(nan);
    if (!live) return;
    uint32_t nans = 0;  // the lane's elements to be computed again
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = CM ? T * i + kk : kk * 4 + i;
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        float out[VW];
#pragma unroll
        for (int e = 0; e < VW; ++e) out[e] = acc[0][w][e][i];
        nans |= store_or_mark<VW, float, BETA>(redo, Cm + (int64_t(br) * BS + r) * ldc, c0[w], own[w],
                                               k, out, alpha, beta)
                << ((i * NW + w) * VW);
      }
    }
    if (!redo) return;
    for (int32_t s = 0; s < 4 * NW * VW; ++s)
      if (nans >> s & 1) {
        const int32_t e = s % VW, w = s / VW % NW, i = s / (VW * NW), r = CM ? T * i + kk : kk * 4 + i;
        const int64_t c = pick(c0, w) + e;
        store_one<float, BETA>(Cm + (int64_t(br) * BS + r) * ldc + c,
                               bsr_dot_nonzero<BS, CM, V, float>(p0, p1, r, c, ci, val, Bm, ldb), alpha, beta);
      }
    return;
  }
  // sum over the lanes g = (kk, pb): at each of the low bits a lane keeps half
  // of its rows and sends the other half, so lane g ends with register (and
  // tile) number g % BS
  float out[NW][VW];
#pragma unroll
  for (int w = 0; w < NW; ++w)
#pragma unroll
    for (int e = 0; e < VW; ++e) {
      F4 h = acc[0][w][e];
      if constexpr (T == 2) {
        const bool up = g & 4;
        const F4 keep = up ? acc[1][w][e] : acc[0][w][e], give = up ? acc[0][w][e] : acc[1][w][e];
#pragma unroll
        for (int r = 0; r < 4; ++r) h[r] = keep[r] + __shfl_xor(give[r], 4 * L);
      }
      const bool u2 = g & 2, u1 = g & 1;
      const float g0 = (u2 ? h[2] : h[0]) + __shfl_xor(u2 ? h[0] : h[2], 2 * L);
      const float g1 = (u2 ? h[3] : h[1]) + __shfl_xor(u2 ? h[1] : h[3], 2 * L);
      float f = (u1 ? g1 : g0) + __shfl_xor(u1 ? g0 : g1, L);
#pragma unroll
      for (int o = L * BS; o < 64; o <<= 1) f += __shfl_xor(f, o);
      out[w][e] = f;
      nan = nan || f != f;
    }
  const bool redo = __any(nan);
  const int gr = g % BS, r = CM ? T * (gr % 4) + gr / 4 : gr;  // the lane's block row
  if (g >= BS) return;
  uint32_t nans = 0;
#pragma unroll
  for (int w = 0; w < NW; ++w)
    nans |= store_or_mark<VW, float, BETA>(redo, Cm + (int64_t(br) * BS + r) * ldc, c0[w], own[w], k,
                                           out[w], alpha, beta)
            << (w * VW);
  if (!redo) return;
  for (int32_t s = 0; s < NW * VW; ++s)
    if (nans >> s & 1) {
      const int32_t e = s % VW, w = s / VW;
      const int64_t c = pick(c0, w) + e;
      store_one<float, BETA>(Cm + (int64_t(br) * BS + r) * ldc + c,
                             bsr_dot_nonzero<BS, CM, V, float>(p0, p1, r, c, ci, val, Bm, ldb), alpha, beta);
    }
}

template <class X>
__global__ __launch_bounds__(kBlock) void k_scale_dense(int64_t m, int64_t n, acc_t<X> beta,
                                                        X *Cm, int64_t sr, int64_t sc) {
  const int64_t t = int64_t(blockIdx.x) * kBlock + threadIdx.x;
  if (t >= m * n) return;
  X *c = Cm + (t / n) * sr + (t % n) * sc;
  *c = beta == acc_t<X>(0) ? X(0) : X(beta * acc_t<X>(*c));
}

template <class X>
__global__ __launch_bounds__(kBlock) void k_strided_copy(int64_t n, const X *src, int64_t ss,
                                                         X *dst, int64_t ds) {
  const int64_t i = int64_t(blockIdx.x) * kBlock + threadIdx.x;
  if (i < n) dst[i * ds] = src[i * ss];
}

namespace {
template <int G, int VW, class V, class X>
void launch_gather(const pls::DevCsr &A, int32_t k, double alpha, const void *B, int64_t ldb,
                   double beta, void *C, int64_t ldc, hipStream_t s, bool direct) {
  // direct: only the rows that the tiles leave out, a workgroup each
  const int32_t m = direct ? 0 : A.m, nlong = direct ? A.t_ndirect : A.nlong;
  const int32_t *longrow = (direct ? A.t_direct : A.longrow).template as<int32_t>();
  const double mean = double(A.nnz) / A.m;
  int32_t S = 1;  // lane groups per row
  while (2 * S * G <= 64 && 2 * kGatherPairs<G> * S <= mean) S *= 2;
  const int64_t windows = (int64_t(k) + G * VW - 1) / (G * VW);
  const int32_t slice = (1 << 30) / (G * S);  // rows per launch: fewer than 2^32 threads
  auto go = [&](auto kern) {
    for (int64_t w = 0; w < windows; w += 65535)
      for (int64_t r = 0; r < std::max(m, 1); r += slice) {
        const int32_t rows = int32_t(std::min<int64_t>(slice, m - r)), nl = r == 0 ? nlong : 0;
        const dim3 grid(unsigned(nl) + grid_for(int64_t(rows) * (G * S)),
                        unsigned(std::min<int64_t>(65535, windows - w)));
        if (grid.x == 0) continue;
        kern<<<grid, kBlock, 0, s>>>(int32_t(r), int32_t(r) + rows, k, int32_t(w), S, nl, longrow,
                                     A.rp.as<int32_t>(), A.ci.as<int32_t>(), A.vals.as<V>(),
                                     (const X *)B, ldb, (X *)C, ldc, acc_t<X>(alpha),
                                     acc_t<X>(beta));
      }
  };
  if (beta != 0.0) go(k_spmm_gather<G, VW, V, X, true>);
  else go(k_spmm_gather<G, VW, V, X, false>);
}

template <int VW, class V, class X>
void gather_lanes(const pls::DevCsr &A, int32_t k, double alpha, const void *B, int64_t ldb,
                  double beta, void *C, int64_t ldc, hipStream_t s, bool direct) {
  const int32_t lanes = (k + VW - 1) / VW;
  if (lanes <= 1) launch_gather<1, VW, V, X>(A, k, alpha, B, ldb, beta, C, ldc, s, direct);
  else if (lanes <= 2) launch_gather<2, VW, V, X>(A, k, alpha, B, ldb, beta, C, ldc, s, direct);
  else if (lanes <= 4) launch_gather<4, VW, V, X>(A, k, alpha, B, ldb, beta, C, ldc, s, direct);
  else if (lanes <= 8) launch_gather<8, VW, V, X>(A, k, alpha, B, ldb, beta, C, ldc, s, direct);
  else if (lanes <= 16) launch_gather<16, VW, V, X>(A, k, alpha, B, ldb, beta, C, ldc, s, direct);
  else if (lanes <= 32) launch_gather<32, VW, V, X>(A, k, alpha, B, ldb, beta, C, ldc, s, direct);
  else launch_gather<64, VW, V, X>(A, k, alpha, B, ldb, beta, C, ldc, s, direct);
}

// VW: 16 bytes of columns per lane, fewer when B has fewer columns.
template <class V, class X>
void dispatch_gather(const pls::DevCsr &A, int32_t k, double alpha, const void *B, int64_t ldb,
                     double beta, void *C, int64_t ldc, hipStream_t s, bool direct) {
  if (sizeof(X) == 4 && k >= 4)
    gather_lanes<(sizeof(X) == 4 ? 4 : 2), V, X>(A, k, alpha, B, ldb, beta, C, ldc, s, direct);
  else if (k >= 2) gather_lanes<2, V, X>(A, k, alpha, B, ldb, beta, C, ldc, s, direct);
  else launch_gather<1, 1, V, X>(A, k, alpha, B, ldb, beta, C, ldc, s, direct);
}

template <int NW, int VW, class V, class X>
void launch_tile(const pls::DevCsr &A, int32_t k, double alpha, const void *B, int64_t ldb,
                 double beta, void *C, int64_t ldc, hipStream_t s) {
  constexpr int WCOLS = 16 * VW * NW;  // columns of one wave
  const int64_t windows = (int64_t(k) + WCOLS - 1) / WCOLS;
  const int64_t slice = int64_t(1) << 25;  // tiles per launch
  auto go = [&](auto kern) {
    for (int64_t w = 0; w < windows; w += 65535)
      for (int64_t t = 0; t < A.ntiles; t += slice) {
        const int32_t n = int32_t(std::min(slice, A.ntiles - t));
        // a multiple of 8 workgroups per window: a tile's windows run on one XCD
        const dim3 grid((grid_for(int64_t(n) * 64) + 7) / 8 * 8,
                        unsigned(std::min<int64_t>(65535, windows - w)));
        kern<<<grid, kBlock, 0, s>>>(
            int32_t(t), int32_t(t) + n, int32_t(w), k, A.t_tiles.as<pls::SpmmTile>(), A.t_row.as<int32_t>(),
            A.t_mask.as<uint64_t>(), A.t_col.as<int32_t>(), A.t_val.as<V>(), A.rp.as<int32_t>(),
            A.ci.as<int32_t>(), A.vals.as<V>(), (const X *)B, ldb, (X *)C, ldc, acc_t<X>(alpha),
            acc_t<X>(beta));
      }
  };
  if (beta != 0.0) go(k_spmm_tile<NW, VW, V, X, true>);
  else go(k_spmm_tile<NW, VW, V, X, false>);
}
template <class V, class X>
void dispatch_tile(const pls::DevCsr &A, int32_t k, double alpha, const void *B, int64_t ldb,
                   double beta, void *C, int64_t ldc, hipStream_t s) {
  if constexpr (sizeof(X) == 8) {
    // A rest of at most 32 columns behind windows of 64 gets a window of 32
    // (27-point 80^3, k = 65 / 96 391 / 380 -> 339 / 344 us, banded 200k rows 234 /
    // 227 -> 205 / 201), unless a second launch of so few tiles costs more (28^3
    // k = 65 25 -> 32).  Its lanes may read columns of the windows before it.
    const int32_t c = k > 64 && pls::spmm_tile_cols(A, true, k) % 64 != 0 ? k / 64 * 64 : k;
    if (k <= 32) launch_tile<1, 2, V, X>(A, k, alpha, B, ldb, beta, C, ldc, s);
    else launch_tile<2, 2, V, X>(A, c, alpha, B, ldb, beta, C, ldc, s);
    if (c < k)
      launch_tile<1, 2, V, X>(A, k - c, alpha, static_cast<const X *>(B) + c, ldb, beta,
                              static_cast<X *>(C) + c, ldc, s);
  } else {
    if (k <= 32) launch_tile<1, 2, V, X>(A, k, alpha, B, ldb, beta, C, ldc, s);
    else if (k <= 64) launch_tile<1, 4, V, X>(A, k, alpha, B, ldb, beta, C, ldc, s);
    else launch_tile<2, 4, V, X>(A, k, alpha, B, ldb, beta, C, ldc, s);
  }
}

template <class V, class X>
void launch_lds(const pls::DevCsr &A, int32_t k, double alpha, const void *B, int64_t ldb,
                double beta, void *C, int64_t ldc, hipStream_t s) {
  auto go = [&](auto kc, auto um) {
    constexpr int KC = decltype(kc)::value, UMAX = decltype(um)::value;
    const auto *blocks = A.lb_block.as<pls::SpmmBlock>();
    const auto *ucol = A.lb_ucol.as<int32_t>();
    const auto *lidx = A.lb_lidx.as<uint8_t>();
    // clustered blocks (nullptr for consecutive rows): row order, block-order
    // row starts and values
    const auto *brow = A.lb_brow.as<int32_t>();
    const auto *prp = A.lb_prp.as<int32_t>();
    const auto *lval = A.lb_val.as<V>();
    if (beta != 0.0)
      k_spmm_lds<KC, UMAX, (KC >= 16 ? 4 : 2), V, X, true><<<A.lb_nblocks, kBlock, 0, s>>>(
          blocks, ucol, lidx, brow, prp, lval, k, A.rp.as<int32_t>(), A.ci.as<int32_t>(),
          A.vals.as<V>(), (const X *)B, ldb, (X *)C, ldc, acc_t<X>(alpha), acc_t<X>(beta));
    else
      k_spmm_lds<KC, UMAX, (KC >= 16 ? 4 : 2), V, X, false><<<A.lb_nblocks, kBlock, 0, s>>>(
          blocks, ucol, lidx, brow, prp, lval, k, A.rp.as<int32_t>(), A.ci.as<int32_t>(),
          A.vals.as<V>(), (const X *)B, ldb, (X *)C, ldc, acc_t<X>(alpha), acc_t<X>(0));
  };
  // Column chunks: 8 for k <= 8 and for FP64 lists of 256, then 16 (FP64) or
  // 16 / 32 (FP32) columns; at most 16 KB of staged FP64 B, so six workgroups
  // share a CU (the best measured shapes on the 27-point stencil and its 8 x 8
  // block form)
  using S_ = std::integral_constant<int, pls::kLbUcolsSmall>;
  using L_ = std::integral_constant<int, pls::kLbUcolsLarge>;
  using C8 = std::integral_constant<int, 8>;
  using C16 = std::integral_constant<int, 16>;
  using C32 = std::integral_constant<int, 32>;
  const bool large = A.lb_umax > pls::kLbUcolsSmall;
  if (k <= 8 || (large && sizeof(X) == 8)) {
    large ? go(C8{}, L_{}) : go(C8{}, S_{});
  } else if (sizeof(X) == 8 || k <= 16) {
    large ? go(C16{}, L_{}) : go(C16{}, S_{});
  } else {
    large ? go(C32{}, L_{}) : go(C32{}, S_{});
  }
}

}  // namespace

hipError_t csr_spmm(const pls::DevCsr &A, bool dbl, pls::SpmmForm form, int32_t k, double alpha,
                    const void *B, int64_t ldb, double beta, void *C, int64_t ldc, hipStream_t s) {
  if (A.m == 0 || k == 0) return hipSuccess;
  auto run = [&](auto vtag, auto xtag) -> hipError_t {
    using V = std::remove_const_t<std::remove_pointer_t<decltype(vtag)>>;
    using X = std::remove_pointer_t<decltype(xtag)>;
    if (form == pls::SpmmForm::Tiles) {
      dispatch_tile<V, X>(A, k, alpha, B, ldb, beta, C, ldc, s);
      dispatch_gather<V, X>(A, k, alpha, B, ldb, beta, C, ldc, s, true);
    } else if (form == pls::SpmmForm::Lds) {
      launch_lds<V, X>(A, k, alpha, B, ldb, beta, C, ldc, s);
    } else {
      dispatch_gather<V, X>(A, k, alpha, B, ldb, beta, C, ldc, s, false);
    }
    return hipGetLastError();
  };
  if (dbl) {
    if (A.vs != pls::VStore::F64) return hipErrorInvalidValue;
    return run((const double *)nullptr, (double *)nullptr);
  }
  if (A.vs == pls::VStore::F32) return run((const float *)nullptr, (float *)nullptr);
  if (A.vs == pls::VStore::BF16) return run((const uint16_t *)nullptr, (float *)nullptr);
  return hipErrorInvalidValue;
}

namespace {
template <int L, int NR, int P, class V, class X>
void launch_few(const pls::DevCsr &A, double alpha, const void *B, double beta, void *C,
                int64_t c_sr, int64_t c_sc, hipStream_t s) {
  const unsigned grid = grid_for(int64_t(A.m) * L);
  if (grid == 0) return;
  if (beta != 0.0)
    k_csr_few_rhs<L, NR, P, V, X, true><<<grid, kBlock, 0, s>>>(
        A.m, A.rp.as<int32_t>(), A.ci.as<int32_t>(), A.vals.as<V>(), (const X *)B, (X *)C, c_sr,
        c_sc, acc_t<X>(alpha), acc_t<X>(beta));
  else
    k_csr_few_rhs<L, NR, P, V, X, false><<<grid, kBlock, 0, s>>>(
        A.m, A.rp.as<int32_t>(), A.ci.as<int32_t>(), A.vals.as<V>(), (const X *)B, (X *)C, c_sr,
        c_sc, acc_t<X>(alpha), acc_t<X>(0));
}
template <int NR, int P, class V, class X>
void few_lanes(const pls::DevCsr &A, double alpha, const void *B, double beta, void *C,
               int64_t c_sr, int64_t c_sc, hipStream_t s) {
  // a lane reads entry pairs: half the lanes per row of one-entry lanes
  switch (std::max(A.vec_lanes / 2, 1)) {
    case 1: launch_few<1, NR, P, V, X>(A, alpha, B, beta, C, c_sr, c_sc, s); break;
    case 2: launch_few<2, NR, P, V, X>(A, alpha, B, beta, C, c_sr, c_sc, s); break;
    case 4: launch_few<4, NR, P, V, X>(A, alpha, B, beta, C, c_sr, c_sc, s); break;
    case 8: launch_few<8, NR, P, V, X>(A, alpha, B, beta, C, c_sr, c_sc, s); break;
    case 16: launch_few<16, NR, P, V, X>(A, alpha, B, beta, C, c_sr, c_sc, s); break;
    case 32: launch_few<32, NR, P, V, X>(A, alpha, B, beta, C, c_sr, c_sc, s); break;
    default: launch_few<64, NR, P, V, X>(A, alpha, B, beta, C, c_sr, c_sc, s); break;
  }
}
}  // namespace

int few_rhs_pitch(int32_t n) { return n <= 1 ? 1 : n == 2 ? 2 : 4; }

hipError_t csr_spmm_few(const pls::DevCsr &A, bool dbl, int32_t n, double alpha, const void *B,
                        double beta, void *C, int64_t c_sr, int64_t c_sc, hipStream_t s) {
  if (A.m == 0 || n <= 0) return hipSuccess;
  if (n > 4) return hipErrorInvalidValue;
  auto run = [&](auto vtag, auto xtag) -> hipError_t {
    using V = std::remove_const_t<std::remove_pointer_t<decltype(vtag)>>;
    using X = std::remove_pointer_t<decltype(xtag)>;
    switch (n) {
      case 1: few_lanes<1, 1, V, X>(A, alpha, B, beta, C, c_sr, c_sc, s); break;
      case 2: few_lanes<2, 2, V, X>(A, alpha, B, beta, C, c_sr, c_sc, s); break;
      case 3: few_lanes<3, 4, V, X>(A, alpha, B, beta, C, c_sr, c_sc, s); break;
      default: few_lanes<4, 4, V, X>(A, alpha, B, beta, C, c_sr, c_sc, s); break;
    }
    return hipGetLastError();
  };
  if (dbl) {
    if (A.vs != pls::VStore::F64) return hipErrorInvalidValue;
    return run((const double *)nullptr, (double *)nullptr);
  }
  if (A.vs == pls::VStore::F32) return run((const float *)nullptr, (float *)nullptr);
  if (A.vs == pls::VStore::BF16) return run((const uint16_t *)nullptr, (float *)nullptr);
  return hipErrorInvalidValue;
}

namespace {
template <int BS, int NB, int NW, int VW, bool ROWS, class V, class X>
void launch_bsr_mfma(const pls::DevBsr &A, int32_t k, double alpha, const void *B, int64_t ldb,
                     double beta, void *C, int64_t ldc, hipStream_t s) {
  constexpr int WCOLS = 4 * NB * VW * NW;  // columns of one wave
  const int32_t npass = (k + WCOLS - 1) / WCOLS;
  // block rows per wave
  constexpr int RPW = !ROWS ? 1 : sizeof(X) == 8 ? 4 / NB * bsr_rows_f64<BS, NW> : 64 / (NB * BS);
  const int64_t units = (int64_t(A.mb) + RPW - 1) / RPW * npass, slice = int64_t(1) << 25;
  auto go = [&](auto kern) {
    for (int64_t u = 0; u < units; u += slice)
      kern<<<grid_for(std::min(slice, units - u) * 64), kBlock, 0, s>>>(
          u, std::min(units, u + slice), npass, A.mb, k, A.rp.as<int32_t>(), A.ci.as<int32_t>(),
          A.vals.as<V>(), (const X *)B, ldb, (X *)C, ldc, acc_t<X>(alpha), acc_t<X>(beta));
  };
  auto by_type = [&](auto ctag, auto btag) {
    constexpr bool CM = decltype(ctag)::value, BETA = decltype(btag)::value;
    if constexpr (sizeof(X) == 4) go(k_bsr_mfma_f32<BS, NB, NW, BS / 4, VW, ROWS, CM, V, BETA>);
    else if (WCOLS <= 32 && A.nnzb >= (WCOLS <= 16 ? 2 : 8) * int64_t(A.mb) &&
             (A.vals.bytes() <= size_t(288) << 20 || (BS == 8 && CM)))  // see ld_block
      go(k_bsr_mfma_f64<BS, NB, NW, VW, ROWS, CM, WCOLS <= 32, BETA>);
    else go(k_bsr_mfma_f64<BS, NB, NW, VW, ROWS, CM, false, BETA>);
  };
  using T_ = std::true_type;
  using F_ = std::false_type;
  if (A.layout == PERFLIBS_COL_MAJOR) beta != 0.0 ? by_type(T_{}, T_{}) : by_type(T_{}, F_{});
  else beta != 0.0 ? by_type(F_{}, T_{}) : by_type(F_{}, F_{});
}
template <int BS, class V, class X>
void dispatch_bsr_spmm(const pls::DevBsr &A, int32_t k, double alpha, const void *B, int64_t ldb,
                       double beta, void *C, int64_t ldc, hipStream_t s) {
  // Window (columns of one wave) by k: the smallest that holds k, since block
  // values are read once per window and a wider one wastes its tail.  Its split
  // into column tiles (NB) and accumulators per lane (NW): measured best of 1-4
  // x 1-4, e.g. 8 x 8 FP64 k = 32 as NB x NW 4 x 1 / 2 x 2 / 1 x 4: 186 / 168 /
  // 193 us, k = 128 in windows of 32 / 64 / 128: 612 / 525 / 486.  FP32 lanes
  // per block row KL = BS / 4 (16-byte block loads), k = 32 with KL = 8 / 4 / 2:
  // 143 / 99 / 92; two windows per wave at k = 64 measured 189 against 172 (all
  // with non-temporal block loads, before ld_block).  Few columns take 1 or 2 per
  // lane, so that no lane repeats another's (4 x 4, 9 per row, FP32 k = 4 / 7 in
  // windows of 16: 33 / 45 us, of 4 and 8: 29 / 37), and short 4 x 4 block rows at
  // k = 9 to 16 two column tiles (46 / 40 at k = 9).
  auto go = [&](auto rtag) {
    constexpr bool R = decltype(rtag)::value;
    if constexpr (sizeof(X) == 8) {
      if (k <= 4) launch_bsr_mfma<BS, 1, 1, 1, R, V, X>(A, k, alpha, B, ldb, beta, C, ldc, s);
      else if (k <= 8) launch_bsr_mfma<BS, 1, 1, 2, R, V, X>(A, k, alpha, B, ldb, beta, C, ldc, s);
      else if (k <= 16) launch_bsr_mfma<BS, 1, 2, 2, R, V, X>(A, k, alpha, B, ldb, beta, C, ldc, s);
      else if (k <= 32) launch_bsr_mfma<BS, 2, 2, 2, R, V, X>(A, k, alpha, B, ldb, beta, C, ldc, s);
      else if (k <= 64 || (k > 128 && (k - 1) % 128 < 64))
        launch_bsr_mfma<BS, 2, 4, 2, R, V, X>(A, k, alpha, B, ldb, beta, C, ldc, s);
      else launch_bsr_mfma<BS, 4, 4, 2, false, V, X>(A, k, alpha, B, ldb, beta, C, ldc, s);
    } else {
      if (k <= 4) launch_bsr_mfma<BS, 1, 1, 1, R, V, X>(A, k, alpha, B, ldb, beta, C, ldc, s);
      else if (k <= 8) launch_bsr_mfma<BS, 1, 1, 2, R, V, X>(A, k, alpha, B, ldb, beta, C, ldc, s);
      else if (k <= 16 && BS == 4 && R)
        launch_bsr_mfma<BS, 2, 1, 2, R, V, X>(A, k, alpha, B, ldb, beta, C, ldc, s);
      else if (k <= 16) launch_bsr_mfma<BS, 1, 1, 4, R, V, X>(A, k, alpha, B, ldb, beta, C, ldc, s);
      else if (k <= 32 || BS == 8)
        launch_bsr_mfma<BS, 2, 1, 4, R, V, X>(A, k, alpha, B, ldb, beta, C, ldc, s);
      else launch_bsr_mfma<BS, BS == 4 ? 4 : 2, 1, 4, R, V, X>(A, k, alpha, B, ldb, beta, C, ldc, s);
    }
  };
  // Short block rows: one lane group per block row instead of several sharing
  // one, where there are rows enough for that (a wave takes 4 to 16 of them).  Mean
  // lengths below which it is faster, by block rows (us shared / own, k = 8): 4 x 4
  // FP64 60,000 rows, 12 blocks per row 28.5 / 22.6, 50,000, 16 25.0 / 26.5; 20,000,
  // 9 11.4 / 10.1, 12 11.9 / 13.5; 8,000, 4 4.7 / 4.9, 7 5.1 / 6.0.  FP32 60,000, 12
  // 22.5 / 14.9, 20,000, 12 8.2 / 7.4; 8,000, 7 5.3 / 5.1, 9 4.7 / 5.6.  8 x 8 FP64
  // 20,000, 5 15.1 / 12.4; 30,000, 7 21.6 / 24.1; 2,000, 3 5.4 / 5.3, 5 4.9 / 5.8.
  // FP32 20,000, 12 15.5 / 14.9, 15,000, 16 13.4 / 16.2; 8,000, 7 5.8 / 5.8, 12 7.1 /
  // 7.6; 2,000, 4 5.2 / 5.2, 9 5.0 / 6.1.
  const int32_t mb = A.mb;
  const int32_t few = BS == 4 ? (sizeof(X) == 8 ? (mb >= 49152 ? 13 : mb >= 16384 ? 10 : 5)
                                                : (mb >= 16384 ? 13 : 7))
                      : mb < 4096 ? 4 : sizeof(X) == 8 ? 6 : mb >= 16384 ? 12 : 8;
  if (A.nnzb < int64_t(A.mb) * few) go(std::true_type{});
  else go(std::false_type{});
}
}  // namespace

hipError_t bsr_spmm(const pls::DevBsr &A, bool dbl, int32_t k, double alpha, const void *B,
                    int64_t ldb, double beta, void *C, int64_t ldc, hipStream_t s) {
  if (A.mb == 0 || k == 0) return hipSuccess;
  if (!(A.b == 4 || A.b == 8)) return hipErrorInvalidValue;
  auto run = [&](auto vtag, auto xtag) -> hipError_t {
    using V = std::remove_const_t<std::remove_pointer_t<decltype(vtag)>>;
    using X = std::remove_pointer_t<decltype(xtag)>;
    if (A.b == 8) dispatch_bsr_spmm<8, V, X>(A, k, alpha, B, ldb, beta, C, ldc, s);
    else dispatch_bsr_spmm<4, V, X>(A, k, alpha, B, ldb, beta, C, ldc, s);
    return hipGetLastError();
  };
  if (dbl) {
    if (A.vs != pls::VStore::F64) return hipErrorInvalidValue;
    return run((const double *)nullptr, (double *)nullptr);
  }
  if (A.vs == pls::VStore::F32) return run((const float *)nullptr, (float *)nullptr);
  if (A.vs == pls::VStore::BF16) return run((const uint16_t *)nullptr, (float *)nullptr);
  return hipErrorInvalidValue;
}

hipError_t strided_copy(bool dbl, int64_t n, const void *src, int64_t ss, void *dst, int64_t ds,
                        hipStream_t s) {
  if (n <= 0) return hipSuccess;
  if (dbl) k_strided_copy<double><<<grid_for(n), kBlock, 0, s>>>(n, (const double *)src, ss, (double *)dst, ds);
  else k_strided_copy<float><<<grid_for(n), kBlock, 0, s>>>(n, (const float *)src, ss, (float *)dst, ds);
  return hipGetLastError();
}

hipError_t scale_dense(bool dbl, int64_t m, int64_t n, double beta, void *C, int64_t sr,
                       int64_t sc, hipStream_t s) {
  if (m * n <= 0) return hipSuccess;
  const unsigned grid = grid_for(m * n);
  if (dbl) k_scale_dense<double><<<grid, kBlock, 0, s>>>(m, n, beta, (double *)C, sr, sc);
  else k_scale_dense<float><<<grid, kBlock, 0, s>>>(m, n, float(beta), (float *)C, sr, sc);
  return hipGetLastError();
}

}  // namespace plk
