// spmm_blocks.cpp — row blocks of the column-compressed SpMM kernels: which rows
// belong together, the distinct columns each block lists once, and every
// non-zero's position in its block's list.  Two device forms are made from the
// cut on first use: the blocks as they are, a workgroup each (k_spmm_lds), and
// their rows in tiles of up to 32, a wave each (k_spmm_tile).
//
// Two cuts are made and the one with the shorter lists kept:
//  * consecutive: rows in order, a block closed before the row that would
//    exceed a limit;
//  * clustered: a block grows from its first unassigned row by repeatedly
//    adding the row that brings the fewest columns not yet listed (ties: the
//    row adjacent to the most rows already in the block, then the lowest row
//    index), so the rows of a block share their columns.  On the 27-point
//    stencil of a 128^3 grid a block becomes a compact patch of neighbouring
//    grid points instead of a segment of one grid line: 6.2 instead of 10.4
//    listed columns per row with lists of 128, i.e. 40% fewer B rows staged
//    in LDS per product (k = 128 FP64 product 3.39 -> 2.83 ms measured on
//    the symmetrically permuted matrix before the kernel took row lists).
// A clustered block's rows are listed in `brow` (the kernel reads them from
// there); consecutive blocks leave it empty.
#include <algorithm>
#include <exception>
#include <mutex>
#include <new>
#include <system_error>
#include <thread>

#include "plsparse.hpp"

namespace pls {

struct LbHost {
  std::vector<int32_t> row0{0};  // block b: entries [row0[b], row0[b+1]) of the row order
  std::vector<int32_t> uoff{0};  // block b: list entries [uoff[b], uoff[b+1]) of ucol
  std::vector<int32_t> ucol;     // distinct columns of each block, in list order
  std::vector<int32_t> brow;     // row order (empty: consecutive rows)
  std::vector<uint8_t> lidx;     // list position of every non-zero (CSR order)
  int64_t direct = 0;            // non-zeros of rows without a list
  int64_t cost() const { return int64_t(ucol.size()) + direct; }
};

namespace {
template <class F> void parallel_ranges(int64_t n, int64_t min_per_range, int64_t max_ranges, F &&fn) {
  const unsigned hw = std::thread::hardware_concurrency();
  const int64_t nt =
      std::max<int64_t>(1, std::min<int64_t>({hw ? hw : 1, max_ranges, n / min_per_range}));
  if (nt <= 1) {
    fn(0, int64_t(0), n);
    return;
  }
  // an exception on a thread (no memory) is the caller's, not the program's end
  std::vector<std::thread> th;
  std::exception_ptr error;
  std::mutex mu;
  auto run = [&](int t, int64_t lo, int64_t hi) {
    try {
      fn(t, lo, hi);
    } catch (...) {
      const std::lock_guard<std::mutex> lock(mu);
      error = std::current_exception();
    }
  };
  th.reserve(size_t(nt));
  const int64_t step = (n + nt - 1) / nt;
  for (int64_t t = 0; t < nt; ++t) {
    const int64_t lo = t * step, hi = std::min(n, lo + step);
    if (lo >= hi) break;
    try {
      th.emplace_back(run, int(t), lo, hi);
    } catch (const std::system_error &) {  // no further thread: this one does it
      run(int(t), lo, hi);
    }
  }
  for (auto &t : th) t.join();
  if (error) std::rethrow_exception(error);
}

// Greedy cut of consecutive rows into blocks of at most umax distinct
// columns, lb_nnz_per_ucol(umax) * umax non-zeros and kLbRows rows; a row that
// alone exceeds a limit becomes a block without a column list.
void cut_consecutive(const Operand &o, int32_t umax, LbHost &h) {
  const int32_t nnz_max = lb_nnz_per_ucol(umax) * umax;
  const int32_t m = o.m;
  const int32_t *rp = o.prp, *ci = o.pci;
  const int32_t base = rp[0];
  const int64_t nnz = int64_t(rp[m]) - base;
  const size_t ncols = size_t(std::max(o.n, 1));
  h.lidx.assign(size_t(std::max<int64_t>(nnz, 1)), 0);
  // inblk[c] == bid: column c is in the current block's list at pos[c];
  // seen[c] == pass: column c was counted by the current counting pass
  std::vector<int32_t> inblk(ncols, -1), pos(ncols, 0), seen(ncols, -1);
  int32_t bid = 0, pass = 0, u = 0, rows = 0;
  int64_t bnnz = 0;
  auto close = [&](int32_t r) {  // the current block ends before row r
    h.row0.push_back(r);
    h.uoff.push_back(int32_t(h.ucol.size()));
    ++bid;
    u = rows = 0;
    bnnz = 0;
  };
  auto count_fresh = [&](int64_t j0, int64_t j1) {  // distinct columns not in the list
    ++pass;
    int32_t f = 0;
    for (int64_t j = j0; j < j1; ++j) {
      const int32_t c = ci[j] - base;
      if (inblk[size_t(c)] != bid && seen[size_t(c)] != pass) {
        seen[size_t(c)] = pass;
        ++f;
      }
    }
    return f;
  };
  for (int32_t r = 0; r < m; ++r) {
    const int64_t j0 = int64_t(rp[r]) - base, j1 = int64_t(rp[r + 1]) - base;
    int32_t fresh = count_fresh(j0, j1);
    if (rows > 0 && !(u + fresh <= umax && bnnz + (j1 - j0) <= nnz_max && rows < kLbRows)) {
      close(r);
      fresh = count_fresh(j0, j1);
    }
    if (fresh > umax || j1 - j0 > nnz_max) {
      close(r + 1);  // rows == 0: the row is a block of its own without a list
      h.direct += j1 - j0;
      continue;
    }
    for (int64_t j = j0; j < j1; ++j) {
      const int32_t c = ci[j] - base;
      if (inblk[size_t(c)] != bid) {
        inblk[size_t(c)] = bid;
        pos[size_t(c)] = u++;
        h.ucol.push_back(c);
      }
      h.lidx[size_t(j)] = uint8_t(pos[size_t(c)]);
    }
    bnnz += j1 - j0;
    ++rows;
  }
  if (rows > 0) close(m);
}

// Columns whose rows are not followed when scoring candidates (a column shared
// by very many rows says little about which rows belong together, and following
// it would make the candidate sets large).
constexpr int32_t kDegreeCap = 256;

// Rows of each column of the operand's pattern (0-based, rows ascending).
void rows_by_column(const Operand &o, std::vector<int32_t> &cp, std::vector<int32_t> &cr) {
  const int32_t m = o.m, n = o.n, base = o.prp[0];
  const int64_t nnz = int64_t(o.prp[m]) - base;
  cp.assign(size_t(n) + 1, 0);
  cr.resize(size_t(std::max<int64_t>(nnz, 1)));
  for (int64_t j = 0; j < nnz; ++j) ++cp[size_t(o.pci[j] - base) + 1];
  for (int32_t c = 0; c < n; ++c) cp[size_t(c) + 1] += cp[size_t(c)];
  std::vector<int32_t> next(cp.begin(), cp.end() - 1);
  for (int32_t r = 0; r < m; ++r)
    for (int64_t j = int64_t(o.prp[r]) - base; j < int64_t(o.prp[r + 1]) - base; ++j)
      cr[size_t(next[size_t(o.pci[j] - base)]++)] = r;
}

// Over up to 256 evenly spaced non-empty rows: the mean of the largest
// fraction of a row's non-zeros whose columns one other row shares (near 0 for
// scattered columns: no block can share columns, so clustering is skipped; 2/3
// on the 27-point stencil), and the fraction of rows whose best partner lies
// within m / 32 rows of it (row ranges can then be clustered independently).
struct Overlap {
  double shared = 0, near = 0;
};
Overlap sampled_overlap(const Operand &o, const std::vector<int32_t> &cp,
                        const std::vector<int32_t> &cr) {
  const int32_t m = o.m, base = o.prp[0];
  std::vector<int32_t> cnt(size_t(m), 0), hit;
  double sum = 0;
  int32_t ns = 0, near = 0;
  const int32_t step = std::max(1, m / 256);
  for (int32_t r = 0; r < m; r += step) {
    const int64_t j0 = int64_t(o.prp[r]) - base, j1 = int64_t(o.prp[r + 1]) - base;
    if (j1 == j0) continue;
    int32_t best = 0, partner = r;
    for (int64_t j = j0; j < j1; ++j) {
      const int32_t c = o.pci[j] - base;
      if (cp[size_t(c) + 1] - cp[size_t(c)] > kDegreeCap) continue;
      for (int32_t q = cp[size_t(c)]; q < cp[size_t(c) + 1]; ++q) {
        const int32_t s = cr[size_t(q)];
        if (s == r) continue;
        if (cnt[size_t(s)]++ == 0) hit.push_back(s);
        if (cnt[size_t(s)] > best) {
          best = cnt[size_t(s)];
          partner = s;
        }
      }
    }
    for (int32_t s : hit) cnt[size_t(s)] = 0;
    hit.clear();
    sum += double(best) / double(j1 - j0);
    near += std::abs(int64_t(partner) - r) <= m / 32;
    ++ns;
  }
  Overlap v;
  if (ns) {
    v.shared = sum / ns;
    v.near = double(near) / ns;
  }
  return v;
}

// Column -> list position of the block being grown (open addressing; at most
// kLbUcolsLarge columns at a quarter load).
class ColMap {
 public:
  ColMap() : key_(kCap, -1), val_(kCap, 0) { used_.reserve(kCap); }
  int32_t find(int32_t c) const {
    for (uint32_t i = hash(c);; i = (i + 1) & (kCap - 1)) {
      if (key_[i] == c) return val_[i];
      if (key_[i] < 0) return -1;
    }
  }
  void insert(int32_t c, int32_t v) {
    uint32_t i = hash(c);
    while (key_[i] >= 0) i = (i + 1) & (kCap - 1);
    key_[i] = c;
    val_[i] = v;
    used_.push_back(i);
  }
  void clear() {
    for (uint32_t i : used_) key_[i] = -1;
    used_.clear();
  }

 private:
  static constexpr uint32_t kCap = 4 * kLbUcolsLarge;
  static uint32_t hash(int32_t c) { return (uint32_t(c) * 2654435761u) >> 22; }  // 10 bits
  std::vector<int32_t> key_, val_;
  std::vector<uint32_t> used_;
};
static_assert(4 * kLbUcolsLarge == 1024, "ColMap hashes to 10 bits");

// One range of rows clustered on its own (ranges run in parallel).
struct RangeBlocks {
  std::vector<int32_t> order, nrow, nu, ucol;
  int64_t direct = 0;
  bool ok = true;
};

// Clustered cut over up to `ranges` row ranges clustered in parallel; false
// when the candidate scans exceed their work budget (48 steps per non-zero of a
// range: the greedy then gives up and the consecutive cut is used).
bool cut_clustered(const Operand &o, int32_t umax, const std::vector<int32_t> &cp,
                   const std::vector<int32_t> &cr, int64_t ranges, LbHost &h) {
  const int32_t nnz_max = lb_nnz_per_ucol(umax) * umax;
  const int32_t m = o.m, base = o.prp[0];
  const int32_t *rp = o.prp, *ci = o.pci;
  const int64_t nnz = int64_t(rp[m]) - base;
  h.lidx.assign(size_t(std::max<int64_t>(nnz, 1)), 0);
  // per row, written only by the range that owns the row: assigned to a
  // block; listed columns shared with the block; rows of the block it is
  // adjacent to (its index appears among their columns)
  std::vector<uint8_t> assigned(size_t(m), 0);
  std::vector<int32_t> ov(size_t(m), 0), adj(size_t(m), 0);
  std::vector<RangeBlocks> parts(16);
  auto len = [&](int32_t r) { return rp[r + 1] - rp[r]; };
  parallel_ranges(m, 4096, ranges, [&](int t, int64_t lo64, int64_t hi64) {
    const int32_t lo = int32_t(lo64), hi = int32_t(hi64);
    RangeBlocks &P = parts[size_t(t)];
    const int64_t budget = 48 * (int64_t(rp[hi]) - rp[lo]) + 65536;
    int64_t work = 0;
    ColMap cm;
    std::vector<int32_t> touched, empties;
    auto own = [&](int32_t r) { return r >= lo && r < hi && !assigned[size_t(r)]; };
    auto note = [&](int32_t r) {
      if (ov[size_t(r)] == 0 && adj[size_t(r)] == 0) touched.push_back(r);
    };
    auto flush_empties = [&] {
      if (empties.empty()) return;
      P.order.insert(P.order.end(), empties.begin(), empties.end());
      P.nrow.push_back(int32_t(empties.size()));
      P.nu.push_back(0);
      empties.clear();
    };
    for (int32_t seed = lo; seed < hi; ++seed) {
      if (assigned[size_t(seed)]) continue;
      const int32_t sl = len(seed);
      if (sl == 0) {  // empty rows share blocks of their own (C = beta * C)
        assigned[size_t(seed)] = 1;
        empties.push_back(seed);
        if (int32_t(empties.size()) == kLbRows) flush_empties();
        continue;
      }
      cm.clear();
      int32_t fresh = 0;  // distinct columns, counted up to umax + 1
      for (int64_t j = int64_t(rp[seed]) - base; j < int64_t(rp[seed + 1]) - base && fresh <= umax; ++j)
        if (cm.find(ci[j] - base) < 0) cm.insert(ci[j] - base, fresh++);
      cm.clear();
      if (fresh > umax || sl > nnz_max) {  // a block of its own without a list
        assigned[size_t(seed)] = 1;
        P.order.push_back(seed);
        P.nrow.push_back(1);
        P.nu.push_back(0);
        P.direct += sl;
        continue;
      }
      int32_t u = 0, rows = 0, cur = seed;
      int64_t bnnz = 0;
      touched.clear();
      for (;;) {
        assigned[size_t(cur)] = 1;
        P.order.push_back(cur);
        ++rows;
        bnnz += len(cur);
        for (int64_t j = int64_t(rp[cur]) - base; j < int64_t(rp[cur + 1]) - base; ++j) {
          const int32_t c = ci[j] - base;
          if (c < m && own(c)) {
            note(c);
            ++adj[size_t(c)];
          }
          int32_t p = cm.find(c);
          if (p < 0) {
            p = u++;
            cm.insert(c, p);
            P.ucol.push_back(c);
            const int32_t q0 = cp[size_t(c)], q1 = cp[size_t(c) + 1];
            if (q1 - q0 <= kDegreeCap) {
              work += q1 - q0;
              for (int32_t q = q0; q < q1; ++q) {
                const int32_t r = cr[size_t(q)];
                if (!own(r)) continue;
                note(r);
                ++ov[size_t(r)];
              }
            }
          }
          h.lidx[size_t(j)] = uint8_t(p);
        }
        if (rows >= kLbRows) break;
        // the candidate bringing the fewest unlisted columns (len - shared is
        // an upper bound on them, so the limits hold), then the most adjacent
        // block rows, then the lowest index
        int32_t best = -1, bnew = 0, badj = 0;
        work += int64_t(touched.size());
        for (const int32_t r : touched) {
          if (assigned[size_t(r)]) continue;
          const int32_t l = len(r), nw = l - ov[size_t(r)];
          if (l == 0 || u + nw > umax || bnnz + l > nnz_max) continue;
          const int32_t a = adj[size_t(r)];
          if (best < 0 || nw < bnew || (nw == bnew && (a > badj || (a == badj && r < best)))) {
            best = r;
            bnew = nw;
            badj = a;
          }
        }
        if (best < 0) break;
        cur = best;
      }
      for (const int32_t r : touched) ov[size_t(r)] = adj[size_t(r)] = 0;
      P.nrow.push_back(rows);
      P.nu.push_back(u);
      if (work > budget) {
        P.ok = false;
        return;
      }
    }
    flush_empties();
  });
  for (const RangeBlocks &P : parts)
    if (!P.ok) return false;
  h.brow.reserve(size_t(m));
  for (const RangeBlocks &P : parts) {
    h.brow.insert(h.brow.end(), P.order.begin(), P.order.end());
    h.ucol.insert(h.ucol.end(), P.ucol.begin(), P.ucol.end());
    for (size_t b = 0; b < P.nrow.size(); ++b) {
      h.row0.push_back(h.row0.back() + P.nrow[b]);
      h.uoff.push_back(h.uoff.back() + P.nu[b]);
    }
    h.direct += P.direct;
  }
  return int32_t(h.brow.size()) == m;
}

// The copies and the value gather of a form's build, waited for before the form is
// used: a product on any stream finds its form written.  (The plan's values
// themselves are complete: their uploads and updates wait.)  They run on the library
// stream, or, while that is being captured, on one of their own (making one takes
// about as long as the build of a small plan).
class BuildStream {
 public:
  BuildStream() : s_(stream()) {
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    own_ = hipStreamIsCapturing(s_, &st) != hipSuccess || st != hipStreamCaptureStatusNone;
    if (own_) e_ = hipStreamCreateWithFlags(&s_, hipStreamNonBlocking);
    if (e_ != hipSuccess) s_ = nullptr;
  }
  ~BuildStream() {
    if (own_ && s_) (void)hipStreamDestroy(s_);
  }
  BuildStream(const BuildStream &) = delete;
  BuildStream &operator=(const BuildStream &) = delete;
  // The host arrays must live until wait().
  void alloc(DevBuf &dst, size_t bytes) {
    if (e_ == hipSuccess) e_ = dst.alloc(std::max<size_t>(bytes, 8));
  }
  void copy(void *dst, const void *host, size_t bytes) {
    if (e_ == hipSuccess && bytes) e_ = hipMemcpyAsync(dst, host, bytes, hipMemcpyHostToDevice, s_);
  }
  template <class T> void upload(DevBuf &dst, const std::vector<T> &host) {
    alloc(dst, sizeof(T) * host.size());
    copy(dst.get(), host.data(), sizeof(T) * host.size());
  }
  void gather(const DevCsr &d, DevBuf &dst, const DevBuf &epos, int64_t n) {
    if (e_ == hipSuccess)
      e_ = plk::gather_vals(d.vs, dst.get(), d.vals.get(), epos.as<int32_t>(), n, s_);
  }
  hipError_t wait() {
    const hipError_t w = own_ && !s_ ? hipSuccess : hipStreamSynchronize(s_);
    if (e_ == hipSuccess) e_ = w;
    return e_;
  }

 private:
  hipStream_t s_;
  bool own_;
  hipError_t e_ = hipSuccess;
};

// Clustered blocks also keep their non-zeros in block order: first non-zero
// of each entry of the row order (prp), list positions, the CSR position of
// each (epos) and the values gathered through it on the device.
hipError_t upload_blocks(const Operand &o, const LbHost &h, DevCsr &d) {
  d.lb_brow.reset();
  d.lb_prp.reset();
  d.lb_epos.reset();
  d.lb_val.reset();
  std::vector<int32_t> prp;  // clustered: first non-zero of each entry of the row order
  // list positions and block-order values end with one padding entry (the
  // kernel stages them in aligned pairs); the CSR plan's values carry theirs
  const size_t nnz = h.lidx.size();
  std::vector<int32_t> epos;
  std::vector<uint8_t> lidx;
  if (h.brow.empty()) {
    lidx = h.lidx;
    lidx.push_back(0);
  } else {
    const int32_t m = o.m, base = o.prp[0];
    prp.assign(size_t(m) + 1, 0);
    epos.assign(nnz + 1, 0);
    lidx.assign(nnz + 1, 0);
    for (int32_t i = 0; i < m; ++i) {
      const int32_t r = h.brow[size_t(i)];
      prp[size_t(i) + 1] = prp[size_t(i)] + (o.prp[r + 1] - o.prp[r]);
    }
    parallel_ranges(m, 65536, 16, [&](int, int64_t lo, int64_t hi) {
      for (int64_t i = lo; i < hi; ++i) {
        const int32_t r = h.brow[size_t(i)], j0 = o.prp[r] - base;
        const int32_t q0 = prp[size_t(i)], len = prp[size_t(i) + 1] - q0;
        for (int32_t t = 0; t < len; ++t) {
          epos[size_t(q0 + t)] = j0 + t;
          lidx[size_t(q0 + t)] = h.lidx[size_t(j0 + t)];
        }
      }
    });
    // the padding entry gathers the CSR plan's own padding value (zero)
    epos[nnz] = int32_t(nnz);
  }
  const auto first = [&](int32_t r) { return h.brow.empty() ? o.prp[r] - o.prp[0] : prp[size_t(r)]; };
  std::vector<SpmmBlock> blocks(h.row0.size() - 1);
  for (size_t b = 0; b < blocks.size(); ++b) {
    const int32_t r0 = h.row0[b], r1 = h.row0[b + 1], u0 = h.uoff[b];
    blocks[b] = {r0, r1 - r0, u0, h.uoff[b + 1] - u0, first(r0), first(r1) - first(r0)};
  }
  BuildStream to;
  to.upload(d.lb_ucol, h.ucol);
  to.upload(d.lb_lidx, lidx);
  to.upload(d.lb_block, blocks);
  if (!h.brow.empty()) {
    const size_t es = d.vs == VStore::F64 ? 8 : d.vs == VStore::F32 ? 4 : 2;
    to.upload(d.lb_brow, h.brow);
    to.upload(d.lb_prp, prp);
    to.upload(d.lb_epos, epos);
    to.alloc(d.lb_val, es * (nnz + 1));
    to.gather(d, d.lb_val, d.lb_epos, int64_t(nnz + 1));
  }
  const hipError_t e = to.wait();
  d.lb_lds = e == hipSuccess;
  if (e != hipSuccess)
    for (DevBuf *b : {&d.lb_ucol, &d.lb_lidx, &d.lb_block, &d.lb_brow, &d.lb_prp, &d.lb_epos, &d.lb_val})
      b->reset();
  return e;
}

// Row tiles of the blocks: each block's rows in runs of at most 32, the run's
// distinct columns four to a step, the step's values half by half in lane
// order (row + 16 * column) behind masks of the lanes that have one.  A column
// a row stores twice is listed twice.  Rows without a list stay outside.
struct TileHost {
  std::vector<SpmmTile> tiles;
  std::vector<int32_t> row, col, epos, direct;
  std::vector<uint64_t> mask;
};
hipError_t upload_tiles(const Operand &o, const LbHost &h, DevCsr &d) {
  const int32_t base = o.prp[0];
  const int64_t nb = int64_t(h.row0.size()) - 1;
  std::vector<TileHost> parts(16);
  parallel_ranges(nb, 64, 16, [&](int part, int64_t lo, int64_t hi) {
    TileHost &P = parts[size_t(part)];
    // list position -> tile column; tile slot (column * 32 + row) -> CSR position
    std::vector<int32_t> pos, slot;
    std::vector<uint8_t> halves;  // which halves of the run use a listed column
    for (int64_t b = lo; b < hi; ++b) {
      const int32_t r0 = h.row0[size_t(b)], nr = h.row0[size_t(b) + 1] - r0;
      const int32_t u0 = h.uoff[size_t(b)], nu = h.uoff[size_t(b) + 1] - u0;
      if (nu == 0 && nr == 1) {
        const int32_t r = h.brow.empty() ? r0 : h.brow[size_t(r0)];
        if (o.prp[r + 1] > o.prp[r]) {  // no list
          P.direct.push_back(r);
          continue;
        }
      }
      const int32_t runs = (nr + 31) / 32;
      for (int32_t t = 0; t < runs; ++t) {
        const int32_t a = int32_t(int64_t(nr) * t / runs), e = int32_t(int64_t(nr) * (t + 1) / runs);
        const int32_t half = e - a <= 16 ? e - a : (e - a + 1) / 2;
        P.tiles.push_back({int32_t(P.row.size()), int32_t(P.mask.size() / 2), int32_t(P.epos.size()), half});
        const size_t c0 = P.col.size();
        // columns of the first half alone, of both, of the second alone: the
        // steps at the ends skip a half
        halves.assign(size_t(nu), 0);
        for (int32_t i = a; i < e; ++i) {
          const int32_t r = h.brow.empty() ? r0 + i : h.brow[size_t(r0 + i)];
          P.row.push_back(r);
          for (int32_t j = o.prp[r] - base; j < o.prp[r + 1] - base; ++j)
            halves[h.lidx[size_t(j)]] |= i - a < half ? 1 : 2;
        }
        pos.assign(size_t(nu), -1);
        for (const uint8_t cls : {1, 3, 2})
          for (int32_t p = 0; p < nu; ++p)
            if (halves[size_t(p)] == cls) {
              pos[size_t(p)] = int32_t(P.col.size() - c0);
              P.col.push_back(h.ucol[size_t(u0 + p)]);
            }
        slot.assign((P.col.size() - c0) * 32, -1);
        for (int32_t i = a; i < e; ++i) {
          const int32_t r = h.brow.empty() ? r0 + i : h.brow[size_t(r0 + i)];
          const int32_t l = i - a < half ? i - a : 16 + i - a - half;  // half 1 from 16 on
          for (int32_t j = o.prp[r] - base; j < o.prp[r + 1] - base; ++j) {
            int32_t c = pos[h.lidx[size_t(j)]];
            if (slot[size_t(c) * 32 + size_t(l)] >= 0) {  // stored twice: listed again
              c = int32_t(P.col.size() - c0);
              P.col.push_back(h.ucol[size_t(u0) + h.lidx[size_t(j)]]);
              slot.resize(slot.size() + 32, -1);
            }
            slot[size_t(c) * 32 + size_t(l)] = j;
          }
        }
        while ((P.col.size() - c0) % 4 != 0) {
          P.col.push_back(P.col.back());
          slot.resize(slot.size() + 32, -1);
        }
        for (size_t s = 0; s < slot.size(); s += 128)
          for (int hf = 0; hf < 2; ++hf) {
            uint64_t m = 0;
            for (int l = 0; l < 64; ++l) {
              const int32_t j = slot[s + size_t(l / 16) * 32 + size_t(hf * 16 + l % 16)];
              if (j < 0) continue;
              m |= uint64_t(1) << l;
              P.epos.push_back(j);
            }
            P.mask.push_back(m);
          }
      }
    }
  });
  size_t nt = 0, nr = 0, nc = 0, nv = 0, nd = 0;
  for (TileHost &P : parts) {  // positions in the whole arrays
    for (SpmmTile &t : P.tiles) {
      t.row0 += int32_t(nr);
      t.step0 += int32_t(nc / 4);
      t.val0 += int32_t(nv);
    }
    nt += P.tiles.size();
    nr += P.row.size();
    nc += P.col.size();
    nv += P.epos.size();
    nd += P.direct.size();
  }
  // the kernel reads whole groups of values ahead: padding (the CSR plan's own
  // padding value)
  TileHost end;
  end.tiles.push_back({int32_t(nr), int32_t(nc / 4), int32_t(nv), 0});
  end.epos.assign(size_t(kTilePad), int32_t(int64_t(o.prp[o.m]) - base));
  parts.push_back(std::move(end));
  const size_t es = d.vs == VStore::F64 ? 8 : d.vs == VStore::F32 ? 4 : 2;
  BuildStream to;
  auto put = [&](DevBuf &dst, auto member) {
    size_t bytes = 0;
    for (const TileHost &P : parts) bytes += (P.*member).size() * sizeof((P.*member)[0]);
    to.alloc(dst, bytes);
    size_t at = 0;
    for (const TileHost &P : parts) {
      const size_t n = (P.*member).size() * sizeof((P.*member)[0]);
      to.copy(static_cast<char *>(dst.get()) + at, (P.*member).data(), n);
      at += n;
    }
  };
  put(d.t_tiles, &TileHost::tiles);
  put(d.t_row, &TileHost::row);
  put(d.t_mask, &TileHost::mask);
  put(d.t_col, &TileHost::col);
  put(d.t_epos, &TileHost::epos);
  put(d.t_direct, &TileHost::direct);
  to.alloc(d.t_val, es * (nv + size_t(kTilePad)));
  d.t_nnz = int64_t(nv);
  d.t_ndirect = int32_t(nd);
  to.gather(d, d.t_val, d.t_epos, d.t_nnz + kTilePad);
  const hipError_t e = to.wait();
  d.ntiles = e == hipSuccess ? int32_t(nt) : -1;
  if (e != hipSuccess)
    for (DevBuf *b : {&d.t_tiles, &d.t_row, &d.t_mask, &d.t_col, &d.t_epos, &d.t_direct, &d.t_val})
      b->reset();
  return e;
}
}  // namespace

// Lists of at most 128 columns keep the kernel's LDS small enough for six
// workgroups per CU (measured 1.3x faster than 256 on the 27-point stencil at
// k = 32 and 128); lists of 256 serve operands whose rows alone have more
// distinct columns (e.g. 8 x 8 block rows).  The blocks are used when their
// lists plus the non-zeros of list-less rows are at most 60% of nnz (a B row
// loaded into LDS then feeds 1.7 non-zeros or more); otherwise the direct
// kernels, which read B for every non-zero, run.
namespace {
// The blocks the plan uses (true), or the last cut tried when no list length
// limit gives enough reuse (false); umax = the limit of the returned cut.
bool choose_blocks(const Operand &o, int rows, LbHost &out, int32_t &umax_out) {
  const int64_t nnz = int64_t(o.prp[o.m]) - o.prp[0];
  std::vector<int32_t> cp, cr;
  Overlap ov;
  // the column -> rows structure and the sampled overlap are built on a thread
  // of their own while the consecutive cut runs
  const bool may_cluster = rows != 1 && o.m >= 2;
  std::thread pre;
  if (may_cluster)
    pre = std::thread([&] {
      rows_by_column(o, cp, cr);
      ov = sampled_overlap(o, cp, cr);
    });
  int overlap = -1;     // 1: rows share enough columns for clustering to pay
  int64_t ranges = 16;  // row ranges clustered in parallel
  bool used = false;
  for (const int32_t umax : {kLbUcolsSmall, kLbUcolsLarge}) {
    LbHost h;
    cut_consecutive(o, umax, h);
    if (may_cluster && double(h.direct) < 0.4 * double(nnz)) {
      if (overlap < 0) {
        pre.join();
        overlap = rows == 2 || ov.shared >= 0.25 ? 1 : 0;
        // rows whose partners are far apart (a scattered row order) are
        // clustered as one range when that stays quick
        if (ov.near < 0.5 && o.m <= (1 << 18)) ranges = 1;
      }
      LbHost c;
      if (overlap == 1 && cut_clustered(o, umax, cp, cr, ranges, c) &&
          (rows == 2 || double(c.cost()) < 0.9 * double(h.cost())))
        h = std::move(c);
    }
    used = double(h.cost()) <= 0.6 * double(nnz);
    out = std::move(h);
    umax_out = umax;
    if (used) break;
  }
  if (pre.joinable()) pre.join();
  return used;
}
}  // namespace

void build_spmm_blocks(const Operand &o, DevCsr &d, int rows) {
  auto h = std::make_shared<LbHost>();
  int32_t umax = 0;
  const bool used = choose_blocks(o, rows, *h, umax);
  d.lb_nblocks = int32_t(h->row0.size() - 1);
  d.lb_ucols = int64_t(h->ucol.size());
  d.lb_umax = umax;
  d.lb_clustered = !h->brow.empty();
  d.lb_lds = d.lb_failed = false;
  d.ntiles = -1;
  d.lb_host = used ? std::move(h) : nullptr;
  d.lb_state = used ? 1 : -1;
}

hipError_t upload_spmm_form(const Operand &o, DevCsr &d, bool tiles) {
  if (d.lb_state != 1 || (tiles ? d.ntiles >= 0 : d.lb_lds)) return hipSuccess;
  hipError_t e;
  try {
    e = tiles ? upload_tiles(o, *d.lb_host, d) : upload_blocks(o, *d.lb_host, d);
  } catch (const std::bad_alloc &) {  // host memory: as on the device
    e = hipErrorOutOfMemory;
  }
  // the cut (a byte per non-zero, the lists and the row order) until both are there
  if (d.has_form(true) && d.has_form(false)) d.lb_host.reset();
  return e;
}

int spmm_blocks_host(const Operand &o, int rows, int32_t *nblocks, int32_t *list_max,
                     int64_t *list_total, int32_t *clustered, int32_t *row_order,
                     int32_t *block_starts) {
  LbHost h;
  int32_t umax = 0;
  const bool used = choose_blocks(o, rows, h, umax);
  const int32_t nb = int32_t(h.row0.size() - 1);
  if (nblocks) *nblocks = nb;
  if (list_max) *list_max = umax;
  if (list_total) *list_total = int64_t(h.ucol.size());
  if (clustered) *clustered = h.brow.empty() ? 0 : 1;
  if (row_order)
    for (int32_t i = 0; i < o.m; ++i) row_order[i] = h.brow.empty() ? i : h.brow[size_t(i)];
  if (block_starts) std::copy(h.row0.begin(), h.row0.end(), block_starts);
  return used ? 1 : -1;
}

hipError_t refresh_block_values(DevCsr &d) {
  hipError_t e = hipSuccess;
  if (d.lb_state != 1) return e;
  if (d.lb_lds && d.lb_clustered)
    e = plk::gather_vals(d.vs, d.lb_val.get(), d.vals.get(), d.lb_epos.as<int32_t>(), d.nnz + 1,
                         stream());
  if (e == hipSuccess && d.ntiles >= 0)
    e = plk::gather_vals(d.vs, d.t_val.get(), d.vals.get(), d.t_epos.as<int32_t>(),
                         d.t_nnz + kTilePad, stream());
  return e;
}

}  // namespace pls
