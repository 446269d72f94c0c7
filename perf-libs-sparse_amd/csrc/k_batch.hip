// k_batch.hip — one launch over a batch of independent CSR
// products Y_p = alpha * A_p * X_p + beta * Y_p (X_p: n_p x k_p, Y_p: m_p x k_p,
// row-major; k_p = 1 is SpMV).
//
// The host cuts every problem into row tiles of bounded nnz and sorts the
// tiles by estimated cost, largest first; workgroup b takes tiles b, b + G,
// b + 2G, ... (G = resident workgroups; one tile each when the device holds them
// all at once), a static greedy schedule that needs no queue counter, so the
// launch can be captured in a hipGraph and replayed as is.  Inside a tile a row
// is handled by a group of `lanes` lanes (a power of two): the k_p right-hand-side
// columns are split over k_p / cpl lanes (cpl consecutive columns per lane, read as
// one contiguous piece of the X row), and the row's non-zeros over the remaining
// lanes / (k_p / cpl) subsets, folded with xor shuffles.  The shape (lanes, cpl) is
// chosen per k class by the batch autotuner.  Same per-row arithmetic as the
// single-matrix CSR kernels (src/compressed_sparse_rows.cpp:1114-1138 for k = 1 and
// the row-blocked SpMM, src/compressed_sparse_rows.cpp:1699-1763, for k > 1).
#include <algorithm>
#include <type_traits>

#include "k_batch.hpp"
#include "k_common.hpp"

namespace plk {

// Staged tiles (k_batch.hpp: at most kBatchStage non-zeros and
// batch_staged_rows() rows) let the per-row loops wait only for the X rows they
// gather; a tile that does not fit (a row longer than kBatchStage) reads the
// matrix from HBM directly.
template <class A> constexpr int kBatchRows = batch_staged_rows(sizeof(A) == 8);

template <class A> struct BatchLds {
  int32_t ci[kBatchStage];
  A a[kBatchStage];
  int32_t rp[kBatchRows<A> + 1];
};

// A tile on its way into LDS: a thread's entry pairs and row offsets.
template <class A> struct BatchRegs {
  static constexpr int NP = kBatchStage / kBlock / 2;
  static constexpr int NR = kBatchRows<A> / kBlock + 1;
  int32_t c[NP][2];
  A a[NP][2];
  int32_t r[NR];
};

// SELL-C-sigma arrays of the batch.
template <class V> struct BatchSell {
  const BatchSellChunk *chunks;
  const int32_t *ci;
  const V *val;
  const int32_t *perm;
};

template <class A> __device__ __forceinline__ bool batch_staged(const BatchTile &tl) {
  return tl.nnz <= kBatchStage && tl.nrows <= kBatchRows<A>;
}

// Loads a staged tile's entries in pairs (one 8-byte index load, one 2-value
// load) from the even index at or below its first; the batch arrays end with
// one padding entry, so the last pair stays in bounds.
template <class V, class A>
__device__ __forceinline__ void batch_load(const BatchTile &tl, const int32_t *__restrict__ rp_all,
                                           const int32_t *__restrict__ ci_all,
                                           const V *__restrict__ val_all, BatchRegs<A> &g) {
  const int tid = threadIdx.x;
  if (!batch_staged<A>(tl)) return;
  const int32_t *rp = rp_all + tl.rp0;
#pragma unroll
  for (int u = 0; u < BatchRegs<A>::NR; ++u) g.r[u] = rp[min(tid + u * kBlock, tl.nrows)];
  if (tl.nnz == 0) return;
  const int32_t sh = int32_t(tl.nz0 & 1);
  const int32_t *cia = ci_all + (tl.nz0 - sh);
  const V *vaa = val_all + (tl.nz0 - sh);
  const int32_t lastp = (tl.nnz + sh - 1) & ~1;  // last pair holding a tile entry
#pragma unroll
  for (int u = 0; u < BatchRegs<A>::NP; ++u)
    ld_pair(cia, vaa, min(2 * (tid + u * kBlock), lastp), g.c[u], g.a[u]);
}

template <class V, class A>
__device__ __forceinline__ void batch_store(const BatchTile &tl, const int32_t *__restrict__ ci_all,
                                            const V *__restrict__ val_all, A alpha,
                                            const BatchRegs<A> &g, BatchLds<A> &lds) {
  const int tid = threadIdx.x;
  if (!batch_staged<A>(tl)) return;
#pragma unroll
  for (int u = 0; u < BatchRegs<A>::NR; ++u)
    if (tid + u * kBlock <= tl.nrows) lds.rp[tid + u * kBlock] = g.r[u] - tl.e0;
  const int32_t sh = int32_t(tl.nz0 & 1);
#pragma unroll
  for (int u = 0; u < BatchRegs<A>::NP; ++u) {
    const int32_t q = 2 * (tid + u * kBlock) - sh;  // tile position of the pair's first entry
#pragma unroll
    for (int h = 0; h < 2; ++h)
      if (q + h >= 0 && q + h < tl.nnz) {
        lds.ci[q + h] = g.c[u][h];
        lds.a[q + h] = alpha * g.a[u][h];
      }
  }
  // a full tile from an odd index has one entry past the pairs
  if (sh && tid == 0 && tl.nnz == kBatchStage) {
    lds.ci[tl.nnz - 1] = ldi(ci_all, tl.nz0 + tl.nnz - 1);
    lds.a[tl.nnz - 1] = alpha * A(ldv(val_all, tl.nz0 + tl.nnz - 1));
  }
}

template <int CPL, bool STAGED, class V, class X, bool BETA>
__device__ __forceinline__ void batch_rows(const BatchTile &tl, int G,
                                           const int32_t *__restrict__ rp_all,
                                           const int32_t *__restrict__ ci_all,
                                           const V *__restrict__ val_all,
                                           const X *__restrict__ xp, X *__restrict__ yp,
                                           acc_t<X> alpha, acc_t<X> beta,
                                           const BatchLds<acc_t<X>> &lds) {
  using A = acc_t<X>;
  typedef X XV __attribute__((ext_vector_type(CPL), aligned(sizeof(X))));
  const int k = tl.k;
  const int kc = k / CPL;  // lanes spanning one row's k columns
  const int S = G / kc;    // non-zero subsets per row
  const int32_t *rp = rp_all + tl.rp0;
  const int32_t *ci = ci_all + tl.nz0;
  const V *va = val_all + tl.nz0;
  const int tid = threadIdx.x;
  const int lane = tid & (G - 1), grp = tid / G;
  const int sub = lane / kc, cb = (lane % kc) * CPL;
  const int rows_per_pass = kBlock / G;
  const bool products = alpha != A(0);
  for (int32_t base = 0; base < tl.nrows; base += rows_per_pass) {
    const int32_t rr = base + grp;
    A acc[CPL];
#pragma unroll
    for (int t = 0; t < CPL; ++t) acc[t] = A(0);
    if (rr < tl.nrows && products) {
      const int32_t p0 = STAGED ? lds.rp[rr] : rp[rr] - tl.e0;
      const int32_t p1 = STAGED ? lds.rp[rr + 1] : rp[rr + 1] - tl.e0;
      constexpr int U = CPL >= 4 ? 4 : 8;  // non-zeros in flight per lane
      for (int32_t j = p0 + sub; j < p1; j += U * S) {
        int32_t c[U];
        A a[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int32_t jj = min(j + u * S, p1 - 1);
          c[u] = STAGED ? lds.ci[jj] : ldi(ci, jj);
          a[u] = STAGED ? lds.a[jj] : alpha * A(ldv(va, jj));
        }
        XV x[U];
#pragma unroll
        for (int u = 0; u < U; ++u)
          x[u] = *reinterpret_cast<const XV *>(xp + int64_t(c[u]) * k + cb);
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const bool ok = j + u * S < p1;
#pragma unroll
          for (int t = 0; t < CPL; ++t) acc[t] = ok ? acc[t] + a[u] * A(x[u][t]) : acc[t];
        }
      }
    }
    for (int o = kc; o < G; o <<= 1)
#pragma unroll
      for (int t = 0; t < CPL; ++t) acc[t] += __shfl_xor(acc[t], o);
    if (rr < tl.nrows && sub == 0) {
      XV *yr = reinterpret_cast<XV *>(yp + int64_t(tl.r0 + rr) * k + cb);
      XV o;
      if (BETA) o = *yr;
#pragma unroll
      for (int t = 0; t < CPL; ++t) {
        A r = acc[t];
        if (BETA) r += beta * A(o[t]);
        o[t] = X(r);
      }
      *yr = o;
    }
  }
}

// SELL-C-sigma tile of a k = 1 problem: C lanes per chunk (one row per lane),
// 64 / C chunks per wave, every wave of the workgroup on its own chunks.  The
// column / value slices of a chunk are contiguous across its lanes, so each
// step of the row loop is one coalesced load per array; padding slots hold
// value 0 and column 0 of the problem.  Four non-zeros in flight per lane.
// Many of them run in a kernel of their own after the CSR tiles': it needs no LDS
// and a quarter of their registers (256 banded problems, all k = 1, C = 32: FP64 /
// FP32 379 / 297 us as tiles of one kernel, 261 / 192 on its own; the two
// launches as parallel branches of the graph took 615 us where one after the
// other take 496).  Few of them run beside the CSR tiles (batch_sell_beside).
template <int C, class V, class X, bool BETA>
__device__ __forceinline__ void batch_sell(const BatchTile &tl, const BatchSell<V> &sell,
                                           const X *const *__restrict__ xs,
                                           X *const *__restrict__ ys, acc_t<X> alpha,
                                           acc_t<X> beta) {
  using A = acc_t<X>;
  const X *xp = xs[tl.prob];
  X *yp = ys[tl.prob];
  const int tid = threadIdx.x, r = tid % C;
  for (int32_t c = tl.r0 + tid / C; c < tl.r1; c += kBlock / C) {
    const BatchSellChunk ch = sell.chunks[c];
    A acc = 0;
    if (alpha != A(0)) {
      const int32_t *cc = sell.ci + ch.off + r;
      const V *vv = sell.val + ch.off + r;
      int32_t j = 0;
      for (; j + 4 <= ch.width; j += 4) {
        int32_t col[4];
        A a[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          col[u] = ldi(cc, int64_t(j + u) * C);
          a[u] = A(ldv(vv, int64_t(j + u) * C));
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) acc += a[u] * A(xp[col[u]]);
      }
      for (; j < ch.width; ++j) acc += A(ldv(vv, int64_t(j) * C)) * A(xp[ldi(cc, int64_t(j) * C)]);
    }
    const int32_t row = sell.perm[ch.slot0 + r];
    if (row >= 0) {
      A res = alpha * acc;
      if (BETA) res += beta * A(yp[row]);
      yp[row] = X(res);
    }
  }
}
template <int C, class V, class X, bool BETA>
__global__ __launch_bounds__(kBlock) void k_batch_sell(const BatchTile *__restrict__ tiles,
                                                       BatchSell<V> sell,
                                                       const X *const *__restrict__ xs,
                                                       X *const *__restrict__ ys, acc_t<X> alpha,
                                                       acc_t<X> beta) {
  batch_sell<C, V, X, BETA>(tiles[blockIdx.x], sell, xs, ys, alpha, beta);
}

// LOOP: a persistent workgroup has its next tile's record, entries and row
// offsets on their way (in registers) while it computes the current one from LDS:
// a tile then waits for its X rows only (256 banded problems, FP64 / FP32: 546 /
// 317 -> 505 / 295 us).  That takes 125 VGPRs in FP64, so four workgroups share a
// CU; five or six spill and take 792 / 952 us.  Without LOOP each has one tile and
// six share a CU: for batches that then run all at once, 1.5 times what the
// persistent ones hold (16 / 12 problems, 1,424 / 1,299 tiles, k = 16, FP32 27.1 ->
// 22.9 / 26.3 -> 21.9 us, FP64, 8 problems, 1,180 tiles, 36.5 -> 33.2; at 2,109
// tiles it is 33.0 -> 34.4).
template <int SELLC, bool LOOP, class V, class X, bool BETA>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(LOOP ? 4 : 6))) void k_batch(
    int32_t ntiles, const BatchTile *__restrict__ tiles, const int32_t *__restrict__ rp_all,
    const int32_t *__restrict__ ci_all, const V *__restrict__ val_all,
    const X *const *__restrict__ xs, X *const *__restrict__ ys, acc_t<X> alpha, acc_t<X> beta,
    BatchShape shape, int32_t grid, BatchSell<V> sell) {
  using A = acc_t<X>;
  __shared__ BatchLds<A> lds;
  BatchRegs<A> g;
  int32_t t = blockIdx.x;
  if constexpr (SELLC > 0)  // the workgroups past the CSR tiles' grid: a SELL tile each
    if (t >= grid) {
      batch_sell<SELLC, V, X, BETA>(tiles[ntiles + t - grid], sell, xs, ys, alpha, beta);
      return;
    }
  if (t >= ntiles) return;
  BatchTile tl = tiles[t];
  const X *xp = xs[tl.prob];
  X *yp = ys[tl.prob];
  batch_load(tl, rp_all, ci_all, val_all, g);
  for (;;) {
    const int32_t nt = t + grid;
    const bool more = LOOP && nt < ntiles;
    BatchTile next = tl;
    if (more) next = tiles[nt];
    __syncthreads();  // the previous tile is done with the LDS
    batch_store(tl, ci_all, val_all, alpha, g, lds);
    if (more) batch_load(next, rp_all, ci_all, val_all, g);
    __syncthreads();
    const int G = shape.lanes[tl.kclass];
    const int cpl = shape.cpl[tl.kclass];
    auto rows = [&](auto ctag) {
      constexpr int CPL = decltype(ctag)::value;
      if (batch_staged<A>(tl))
        batch_rows<CPL, true, V, X, BETA>(tl, G, rp_all, ci_all, val_all, xp, yp, alpha, beta, lds);
      else
        batch_rows<CPL, false, V, X, BETA>(tl, G, rp_all, ci_all, val_all, xp, yp, alpha, beta, lds);
    };
    if (cpl == 1) rows(std::integral_constant<int, 1>{});
    else if (cpl == 2) rows(std::integral_constant<int, 2>{});
    else rows(std::integral_constant<int, 4>{});
    if (!more) return;
    tl = next;
    t = nt;
    xp = xs[tl.prob];
    yp = ys[tl.prob];
  }
}

namespace {
template <class F> hipError_t batch_types(pls::VStore vs, bool dbl, F &&f) {
  if (dbl) {
    if (vs != pls::VStore::F64) return hipErrorInvalidValue;
    return f((const double *)nullptr, (double *)nullptr);
  }
  if (vs == pls::VStore::F32) return f((const float *)nullptr, (float *)nullptr);
  if (vs == pls::VStore::BF16) return f((const uint16_t *)nullptr, (float *)nullptr);
  return hipErrorInvalidValue;
}
}  // namespace

// Whether the SELL-C-sigma tiles share the CSR tiles' launch.  Beside them they fill
// the CUs that the persistent workgroups leave, and there is one launch, but four
// workgroups to a CU; after them there are eight.  The line is a few rounds of the
// chip, farther out for C = 64 (half the loads per row in a wave) unless most tiles
// are SELL (banded problems, k = 1, 4, 16 mixed, tile 2048, us beside / after: FP64, C
// = 32, 16 / 32 / 48 / 256 problems 30 / 49 / 76 / 479 against 38 / 57 / 73 / 471; C =
// 64 29 / 47 / 69 / 453 against 38 / 55 / 76 / 478; 7 of 8 problems k = 1, C = 32 26 /
// 41 / 69 / 409 against 32 / 40 / 61 / 312, C = 64 23 / 34 / 57 / 346 against 31 / 43 /
// 65 / 336; BF16, C = 64, 256 problems 262 against 261, 4096 4160 against 3830).
static bool batch_sell_beside(const BatchLaunch &L) {
  const int64_t nsell = L.ntiles - L.ncsr;
  if (nsell <= 0 || L.ncsr <= 0) return false;
  return L.sell_C == 32 ? nsell <= 3 * int64_t(L.resident)
                        : nsell <= 6 * int64_t(L.resident) ||
                              (nsell <= L.ncsr && nsell <= 16 * int64_t(L.resident));
}

hipError_t batch_launch(const BatchLaunch &L, hipStream_t s) {
  if (L.ntiles == 0 || L.grid == 0) return hipSuccess;
  return batch_types(L.vs, L.dbl, [&](auto vtag, auto xtag) -> hipError_t {
    using V = std::remove_const_t<std::remove_pointer_t<decltype(vtag)>>;
    using X = std::remove_pointer_t<decltype(xtag)>;
    const auto *xs = static_cast<const X *const *>(L.xs);
    auto *ys = static_cast<X *const *>(L.ys);
    const auto *sv = static_cast<const V *>(L.svals);
    const auto *tiles = L.tiles;
    const BatchSell<V> sl{L.chunks, L.sci, sv, L.perm};
    const bool upd = L.beta != 0.0;
    const bool loop = 2 * int64_t(L.ncsr) > 3 * int64_t(L.resident);
    const int32_t grid = loop ? std::min(L.grid, L.ncsr) : L.ncsr, nsell = L.ntiles - L.ncsr;
    auto with = [&](auto sell_c, auto lp, int32_t more) {
      constexpr int C = decltype(sell_c)::value;
      constexpr bool LOOP = decltype(lp)::value;
      auto go = [&](auto kern) {
        kern<<<grid + more, kBlock, 0, s>>>(L.ncsr, tiles, L.rp, L.ci, static_cast<const V *>(L.vals),
                                            xs, ys, acc_t<X>(L.alpha), acc_t<X>(L.beta), L.shape, grid, sl);
      };
      upd ? go(k_batch<C, LOOP, V, X, true>) : go(k_batch<C, LOOP, V, X, false>);
    };
    auto csr = [&](auto sell_c, int32_t more) {
      loop ? with(sell_c, std::true_type{}, more) : with(sell_c, std::false_type{}, more);
    };
    auto sell = [&](auto kern) {
      kern<<<nsell, kBlock, 0, s>>>(tiles + L.ncsr, sl, xs, ys, acc_t<X>(L.alpha),
                                    acc_t<X>(L.beta));
    };
    const bool beside = batch_sell_beside(L);
    if (beside && L.sell_C == 32) csr(std::integral_constant<int, 32>{}, nsell);
    else if (beside) csr(std::integral_constant<int, 64>{}, nsell);
    else if (L.ncsr > 0) csr(std::integral_constant<int, 0>{}, 0);
    if (nsell > 0 && !beside) {
      if (L.sell_C == 32) upd ? sell(k_batch_sell<32, V, X, true>) : sell(k_batch_sell<32, V, X, false>);
      else upd ? sell(k_batch_sell<64, V, X, true>) : sell(k_batch_sell<64, V, X, false>);
    }
    return hipGetLastError();
  });
}

int batch_occupancy(bool dbl, pls::VStore vs) {
  int nb = 0;
  hipError_t e = batch_types(vs, dbl, [&](auto vtag, auto xtag) -> hipError_t {
    using V = std::remove_const_t<std::remove_pointer_t<decltype(vtag)>>;
    using X = std::remove_pointer_t<decltype(xtag)>;
    const void *kern = reinterpret_cast<const void *>(&k_batch<0, true, V, X, false>);
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, kern, kBlock, 0);
  });
  return e == hipSuccess ? nb : 0;
}

}  // namespace plk
