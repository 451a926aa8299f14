// hmvm_multi_plan.cpp -- builds the multi-RHS schedule from the value layout.
#include "hmvm_multi_plan.hpp"

#include <algorithm>
#include <climits>
#include <cstddef>
#include <cstdint>
#include <map>
#include <utility>

namespace hmvm {

namespace {

// The value layout by factor, from the repack records.
struct Piece {  // rows of a stage-1 stack: ranks k0.. of a leaf
  int leaf, k0, n;
};
struct Band {  // rows of a stage-1 stack stored together: all of it, or one band
  int64_t base;
  int ld, row0, rows;
};
struct Stack {  // the stacked a1 factors of a column cluster
  int ncols, col0;
  int rows = 0;
  std::vector<Piece> pieces;
  std::vector<Band> bands;
};
struct Factor {  // dense leaf or a2 factor: columns of a row cluster
  int64_t base;
  int ncols, v, leaf;
  bool t;  // columns multiply t rows v.. (else X rows v..)
};
struct Cluster {
  int row0, rows, ld;
  std::vector<Factor> factors;
};

// Columns of an item under construction: their slices, and the pack records
// (dst: slice index within the item until the item is placed).
struct Columns {
  std::vector<MultiSlice> slices;
  std::vector<MultiPack> pack;
};

struct Builder {
  const int KS;
  MultiPlan &M;
  Builder(int storage, MultiPlan &m) : KS(multi_slice_cols(storage)), M(m) {}

  // The slices of n columns that multiply rows v.. of X or t.
  void add_slices(Columns &c, int n, int v, bool t) const {
    for (int k = 0; k < n; k += KS)
      c.slices.push_back({v + k, std::min(KS, n - k) | (t ? kSliceT : 0)});
  }
  // The slices of a chunk of n columns of BF16 stage 1 (ordered_column).
  void add_ordered(Columns &c, int n, int v) const {
    for (int k = 0; k < n; k += 2 * kStep)
      for (int s = 0; s < kMultiBatch; s++) {
        auto in_use = [&](int first) { return std::max(0, std::min(kHalf, n - first)); };
        const int first = k + s * kHalf;
        // (a slice without columns stays inside the vector)
        c.slices.push_back({first < n ? v + first : v,
                            in_use(first) | in_use(first + kStep) << 4 | (k + 2 * kStep >= n ? kSliceEnd : 0)});
      }
  }
  // Places the columns of an item of nrows rows: {a0, slice0, batches}.
  struct Place {
    int64_t a0;
    int slice0, nbatch;
  };
  Place place(Columns &c, int nrows) {
    Place p;
    p.a0 = M.nvals;
    p.slice0 = (int)M.slices.size();
    const int n = (int)c.slices.size(), pad = (kMultiBatch - n % kMultiBatch) % kMultiBatch;
    p.nbatch = (n + pad) / kMultiBatch;
    M.slices.insert(M.slices.end(), c.slices.begin(), c.slices.end());
    M.slices.insert(M.slices.end(), pad, MultiSlice{0, 0});
    for (MultiPack &r : c.pack) {
      const int last = (int)r.dst + (r.cols + KS - 1) / KS;
      if (!r.ordered) r.pad = last == n ? pad : 0;  // the records of the last columns also write the item's padding
      r.dst = p.a0 + r.dst * nrows * KS;
      r.nrows = nrows;
      M.pack.push_back(r);
    }
    M.nvals += (int64_t)(n + pad) * nrows * KS;
    return p;
  }
};

// Relative cost of a batch over `rows` rows: the loads of X and the fixed
// work of a batch, then the rows in steps of 16.
double batch_cost(int rows) { return 2.0 + (rows + 15) / 16; }

// Workgroup w of a launch runs on XCD w % kMultiXcds: MI355X hands the workgroups
// of a grid to its 8 XCDs round robin, and each XCD has its own L2.  Sorted
// by the vector rows they read (key), the groups are cut into kMultiXcds runs of
// equal cost and laid out so that the workgroups of XCD k take run k's
// groups, costliest first: each XCD then reads about one kMultiXcds-th of the
// vector, which its L2 holds, instead of all of it.  A workgroup whose run is
// used up takes a group of the run with the most left.
std::vector<size_t> xcd_order(const std::vector<int32_t> &key, const std::vector<double> &cost) {
  const size_t n = key.size();
  std::vector<size_t> idx(n);
  for (size_t i = 0; i < n; i++) idx[i] = i;
  std::stable_sort(idx.begin(), idx.end(), [&](size_t a, size_t b) { return key[a] < key[b]; });
  double total = 0;
  for (double c : cost) total += c;
  std::vector<std::vector<size_t>> run(kMultiXcds);
  double cum = 0;
  for (size_t i : idx) {
    const int r = total > 0 ? std::min(kMultiXcds - 1, (int)((cum + 0.5 * cost[i]) * kMultiXcds / total)) : 0;
    run[r].push_back(i);
    cum += cost[i];
  }
  for (auto &r : run)
    std::stable_sort(r.begin(), r.end(), [&](size_t a, size_t b) { return cost[a] > cost[b]; });
  std::vector<size_t> out;
  out.reserve(n);
  std::vector<size_t> pos(kMultiXcds, 0);
  for (int w = 0; out.size() < n; w++) {
    int r = w % kMultiXcds;
    if (pos[r] == run[r].size())  // run used up: the run with the most groups left
      for (int q = 0; q < kMultiXcds; q++)
        if (run[q].size() - pos[q] > run[r].size() - pos[r]) r = q;
    out.push_back(run[r][pos[r]++]);
  }
  return out;
}

// Groups under construction, put into dispatch order at the end.
struct GroupList {
  std::vector<MultiGroup> groups;
  std::vector<MultiWave> waves;
  std::vector<int32_t> key;  // first vector row read
  std::vector<double> cost;
  void finish(int nw, std::vector<MultiGroup> *g, std::vector<MultiWave> *w) const {
    for (size_t i : xcd_order(key, cost)) {
      g->push_back(groups[i]);
      w->insert(w->end(), waves.begin() + (std::ptrdiff_t)(i * nw), waves.begin() + (std::ptrdiff_t)((i + 1) * nw));
    }
  }
};

}  // namespace

// Sizes by matrix order, measured on generated matrices of 1,000 to 101,250
// rows in all storages (ms of the product; best of rows 16 / 32 / 64, waves 2
// / 4 / 8, wave_cols 32 / 256):
//   rows   a group of 64 reads X and t least often, but 16,384 rows are 256
//          such groups, one per CU; below, shorter groups fill the chip
//          (N=12,007, FP64, 32 right-hand sides: 64 rows 0.104, 32 rows
//          0.073; N=1,000: 32 rows 0.019, 16 rows 0.014; N=30,011: 32 rows
//          0.172, 64 rows 0.167);
//   waves  more waves a group shorten the chain of batches of each (N=1,000: 2
//          waves 0.021, 8 waves 0.014); from about 80,000 rows on there are
//          groups enough, and fewer waves start and end less often (2 / 4
//          waves, us, 16 and 64 right-hand sides: N=60,013 FP64 272 / 261 and
//          610 / 489, FP32 168 / 152 and 371 / 313, BF16 113 / 111 and 159 / 152;
//          N=70,003 302 / 293 and 595 / 540, 178 / 177 and 377 / 347, 105 / 110
//          and 171 / 177; N=82,007 337 / 331 and 627 / 605, 198 / 200 and 408 /
//          384, 129 / 129 and 187 / 203; N=101,250 454 / 456 and 860 / 843, 267 /
//          274 and 556 / 542, 160 / 173 and 258 / 289; N=160,003 783 / 810 and
//          1437 / 1408, 446 / 461 and 911 / 894, 256 / 272 and 387 / 411: BF16
//          and 16 right-hand sides gain, 64 in FP64 and FP32 lose 2 to 4%);
//   wave_cols  one wave a stack saves the sum over the waves, but a launch of
//          a small matrix then lasts as long as its longest stack (N=4,096,
//          FP64, 16 right-hand sides: 256 columns 0.038, 32 columns 0.025;
//          N=101,250: 32 columns 0.548, 256 columns 0.542);
//   cols1  stacks up to so many columns need no slots and no t sum; beyond
//          2048 a launch lasts as long as its widest stacks (32 right-hand
//          sides, 1024 / 2048 / 4096 / 8192 columns, us: N=20,011 FP32 120 /
//          118 / 117 / 117, BF16 81 / 77 / 78 / 78; N=101,250 FP64 547 / 545 /
//          545 / 614, BF16 with 16 164 / 161 / 163 / 192).
MultiOptions multi_options(const Plan &P) {
  MultiOptions o;
  o.rows = P.nd >= 16384 ? 64 : P.nd >= 2048 ? 32 : 16;
  o.rows_a = P.nd >= 16384 ? 64 : P.nd >= 2048 ? 32 : 16;
  o.waves = P.nd >= 81920 ? 2 : P.nd >= 2048 ? 4 : 8;
  o.wave_cols = P.nd >= 8192 ? 256 : 32;
  return o;
}

std::string build_multi_plan(const Plan &P, int storage, const int *nstrtl, const int *nstrtt,
                             const MultiOptions &opt, MultiPlan *out) {
  MultiPlan &M = *out;
  M = MultiPlan();
  M.waves = opt.waves;
  if (opt.rows < 1 || opt.rows > kMultiRows || opt.rows_a < 1 || opt.rows_a > kMultiRows || opt.waves < 1 ||
      opt.cols1 < 1)
    return "bad multi-RHS options";
  Builder B(storage, M);
  // (address space alone: what is not used is never touched)
  M.slices.reserve((size_t)(P.nvals / (16 * B.KS)) + 64);
  M.pack.reserve(4 * P.repack.size());
  M.items.reserve(4 * P.repack.size());
  const int nw = opt.waves;
  const bool bf16 = storage == kBF16;

  // ---- the layout ----------------------------------------------------------------
  std::vector<Stack> stacks;
  std::vector<Cluster> clusters;
  std::vector<int> t_idx(P.nlf, -1), kdone(P.nlf, 0);
  for (const RepackDesc &r : P.repack) {
    if (r.rows == 0 || r.cols == 0) continue;
    const int leaf = r.factor / 2;
    if (r.factor % 2 == 0) {
      const int col0 = nstrtt[leaf] - 1;
      if (stacks.empty() || stacks.back().ncols != r.cols || stacks.back().col0 != col0)
        stacks.push_back({r.cols, col0, 0, {}, {}});
      Stack &s = stacks.back();
      if (s.bands.empty() || s.bands.back().ld != r.dst_cs || s.bands.back().base + s.bands.back().rows != r.dst_off)
        s.bands.push_back({r.dst_off, r.dst_cs, s.rows, 0});
      s.bands.back().rows += r.rows;
      s.pieces.push_back({leaf, kdone[leaf], r.rows});
      s.rows += r.rows;
      kdone[leaf] += r.rows;
    } else {
      const int row0 = nstrtl[leaf] - 1;
      if (clusters.empty() || clusters.back().row0 != row0 || clusters.back().rows != r.rows)
        clusters.push_back({row0, r.rows, r.dst_cs, {}});
      Factor f;
      f.base = r.dst_off;
      f.ncols = r.cols;
      f.leaf = leaf;
      f.t = kdone[leaf] > 0;  // a low-rank leaf: its a1 records come first
      if (f.t) {
        t_idx[leaf] = (int)M.n_t;
        M.n_t += r.cols;
        if (M.n_t > INT32_MAX) return kMultiTooLarge;
      }
      f.v = f.t ? t_idx[leaf] : nstrtt[leaf] - 1;
      clusters.back().factors.push_back(f);
    }
  }
  M.t_factor.assign((size_t)M.n_t, 0);
  for (const Cluster &c : clusters)
    for (const Factor &f : c.factors)
      if (f.t)
        for (int k = 0; k < f.ncols; k++) M.t_factor[(size_t)f.v + k] = 2 * f.leaf;

  GroupList A, Bl;
  // Adds a workgroup: each wave's own items, then its share of the kept
  // batches, which go to the waves, `unit` at a time, so that all end together.
  auto add_group = [&](GroupList &L, MultiKind kind, int64_t out_row, int key, const Builder::Place &kept, int nrows,
                       const std::vector<std::vector<MultiItem>> &own, const std::vector<double> &load, int unit = 1) {
    std::vector<int> take(nw, 0);  // in units, the last of which may be shorter
    std::vector<double> l = load;
    const double c = batch_cost(nrows);
    double total = kept.nbatch * c;
    for (double v : l) total += v;
    int left = (kept.nbatch + unit - 1) / unit;
    for (int w = 0; w < nw && left > 0; w++) {
      const int n = std::min(left, std::max(0, (int)((total / nw - l[w]) / (c * unit))));
      take[w] = n;
      l[w] += n * c * unit;
      left -= n;
    }
    while (left > 0) {
      const int w = (int)(std::min_element(l.begin(), l.end()) - l.begin());
      take[w]++;
      l[w] += c * unit;
      left--;
    }
    int b = 0;
    for (int w = 0; w < nw; w++) {
      L.waves.push_back({(int32_t)M.items.size(), (int32_t)own[w].size() + 1});
      M.items.insert(M.items.end(), own[w].begin(), own[w].end());
      const int n = std::min(take[w] * unit, kept.nbatch - b);
      M.items.push_back({kept.a0 + (int64_t)b * kMultiBatch * nrows * B.KS, kept.slice0 + b * kMultiBatch, n, nrows, -1,
                         kItemKept, 0});
      b += n;
    }
    L.groups.push_back({nrows, kind, (int32_t)out_row, 0});
    L.key.push_back(key);
    L.cost.push_back(total);
  };
  const std::vector<std::vector<MultiItem>> none(nw);
  const std::vector<double> idle(nw, 0.0);

  // ---- stage 1 ---------------------------------------------------------------------
  Columns col;
  struct Single {
    MultiItem it;
    int key;
  };
  std::vector<Single> single;  // stacks that one wave takes
  // rows r0.. and columns c0.. of a stack from an item's slice `first` on, a
  // record per band; pad >= 0: ordered
  auto pack_stack = [&](const Stack &s, int r0, int nr, int c0, int nc, int first, int pad) {
    for (const Band &q : s.bands) {
      const int a = std::max(q.row0, r0), e = std::min(q.row0 + q.rows, r0 + nr);
      if (a < e)
        col.pack.push_back({q.base + (a - q.row0) + (int64_t)c0 * q.ld, first, q.ld, e - a, nc, a - r0, 0,
                            std::max(pad, 0), -1, pad >= 0 ? 1 : 0});
    }
  };
  for (const Stack &s : stacks) {
    std::vector<int32_t> trow((size_t)s.rows);
    {
      int r = 0;
      for (const Piece &p : s.pieces)
        for (int k = 0; k < p.n; k++) {
          if (t_idx[p.leaf] < 0) return "stage-1 rows of a leaf without a2";
          trow[(size_t)r++] = t_idx[p.leaf] + p.k0 + k;
        }
    }
    if (bf16) {
      // row groups as Plan::chunk_rows has them: a leaf that fits starts a
      // group where it would straddle two
      std::vector<int> size(1, 0);
      for (size_t i = 0; i < s.pieces.size();) {
        int kt = 0;
        for (const int leaf = s.pieces[i].leaf; i < s.pieces.size() && s.pieces[i].leaf == leaf; i++) kt += s.pieces[i].n;
        for (int done = 0; done < kt;) {
          const int full = size.back();
          if (full == P.chunk_rows ||
              (done == 0 && full > 0 && full + kt > P.chunk_rows && kt <= P.chunk_rows))
            size.push_back(0);
          const int take = std::min(kt - done, P.chunk_rows - size.back());
          size.back() += take;
          done += take;
        }
      }
      const int rows = std::min(opt.rows_a, kOrderedRows);
      int g0 = 0;
      for (const int n : size) {
        const int C = std::min(s.ncols, chunk_cols(n, P.chunk_w));
        const int unit = (C + 2 * kStep - 1) / (2 * kStep);  // batches of a chunk
        const int step = std::max({opt.cols1, s.ncols / 32768, C}) / C * C;  // (at most 32768 groups)
        const bool direct = step >= s.ncols;
        for (int r0 = g0; r0 < g0 + n; r0 += rows) {
          const int nr = std::min(rows, g0 + n - r0);
          const int64_t slot0 = M.n_slots;
          int groups = 0;
          for (int c0 = 0; c0 < s.ncols; c0 += step, groups++) {
            const int end = std::min(s.ncols, c0 + step);
            col.slices.clear();
            col.pack.clear();
            for (int c = c0; c < end; c += C) {
              const int nc = std::min(C, end - c), first = (int)col.slices.size();
              B.add_ordered(col, nc, s.col0 + c);
              pack_stack(s, r0, nr, c, nc, first, (int)col.slices.size() - first - (nc + B.KS - 1) / B.KS);
            }
            const Builder::Place b = B.place(col, nr);
            const int64_t map = (int64_t)M.tmap.size();
            if (direct && s.ncols <= opt.wave_cols)
              single.push_back({{b.a0, b.slice0, b.nbatch, nr, (int32_t)map, kItemT, 0}, s.col0});
            else
              add_group(A, direct ? kMultiT : kMultiTSlot, direct ? map : M.n_slots, s.col0 + c0, b, nr, none, idle,
                        unit);
            if (!direct) M.n_slots += nr;
            if (M.n_slots > INT32_MAX) return kMultiTooLarge;
          }
          if (direct)
            M.tmap.insert(M.tmap.end(), trow.begin() + r0, trow.begin() + r0 + nr);
          else
            for (int r = 0; r < nr; r++) M.tsum.push_back({(int32_t)(slot0 + r), groups, nr, trow[(size_t)r0 + r]});
        }
        g0 += n;
      }
      continue;
    }
    const int cols1 = std::max(opt.cols1, s.ncols / 32768);  // (at most 65535 chunks)
    const int nch = (s.ncols + cols1 - 1) / cols1;
    const int step = ((s.ncols + nch - 1) / nch + B.KS - 1) / B.KS * B.KS;
    const bool direct = step >= s.ncols;
    for (int r0 = 0; r0 < s.rows; r0 += opt.rows_a) {
      const int nr = std::min(opt.rows_a, s.rows - r0);
      const int64_t slot0 = M.n_slots;
      int chunks = 0;
      for (int c0 = 0; c0 < s.ncols; c0 += step, chunks++) {
        const int nc = std::min(s.ncols - c0, step);
        col.slices.clear();
        col.pack.clear();
        pack_stack(s, r0, nr, c0, nc, 0, -1);
        B.add_slices(col, nc, s.col0 + c0, false);
        const Builder::Place b = B.place(col, nr);
        if (direct && s.ncols <= opt.wave_cols)
          single.push_back({{b.a0, b.slice0, b.nbatch, nr, (int32_t)M.tmap.size(), kItemT, 0}, s.col0});
        else
          add_group(A, direct ? kMultiT : kMultiTSlot, direct ? (int64_t)M.tmap.size() : M.n_slots, s.col0 + c0, b, nr,
                    none, idle);
        if (direct)
          M.tmap.insert(M.tmap.end(), trow.begin() + r0, trow.begin() + r0 + nr);
        else
          M.n_slots += nr;
        if (M.n_slots > INT32_MAX) return kMultiTooLarge;
      }
      if (!direct)
        for (int r = 0; r < nr; r++)
          M.tsum.push_back({(int32_t)(slot0 + r), chunks, nr, trow[(size_t)r0 + r]});
    }
  }
  if (M.tmap.size() > (size_t)INT32_MAX) return kMultiTooLarge;
  // one-wave stacks of like cost share a workgroup
  std::stable_sort(single.begin(), single.end(), [](const Single &x, const Single &y) {
    return x.it.nbatch * batch_cost(x.it.nrows) > y.it.nbatch * batch_cost(y.it.nrows);
  });
  for (size_t i = 0; i < single.size(); i += nw) {
    A.groups.push_back({1, kMultiNone, 0, 0});
    A.key.push_back(single[i].key);
    A.cost.push_back(0.0);
    for (int w = 0; w < nw; w++) {
      const bool on = i + w < single.size();
      A.waves.push_back({(int32_t)M.items.size(), on ? 1 : 0});
      if (!on) continue;
      M.items.push_back(single[i + w].it);
      A.cost.back() = std::max(A.cost.back(), single[i + w].it.nbatch * batch_cost(single[i + w].it.nrows) * nw);
    }
  }
  std::sort(M.tsum.begin(), M.tsum.end(),
            [](const MultiPlan::TSum &a, const MultiPlan::TSum &b) { return a.entry < b.entry; });

  // ---- rows of y -----------------------------------------------------------------------
  // cuts: the ends of clusters taller than a group are cuts always, other
  // cluster ends where a group would get too tall
  std::vector<char> cut((size_t)P.nd + 1, 0);  // 1: some cluster starts or ends here, 2: one taller than a group
  cut[0] = cut[(size_t)P.nd] = 2;
  for (const Cluster &c : clusters)
    for (int r : {c.row0, c.row0 + c.rows}) cut[(size_t)r] = std::max(cut[(size_t)r], (char)(c.rows > opt.rows ? 2 : 1));
  std::vector<int> start;  // first row of every group, and nd
  for (int r = 0; r < P.nd;) {
    start.push_back(r);
    int e = r + 1, soft = -1;
    while (e < P.nd && cut[(size_t)e] != 2 && e - r < opt.rows) {
      if (cut[(size_t)e] == 1) soft = e;
      e++;
    }
    if (e < P.nd && cut[(size_t)e] == 0 && soft > 0) e = soft;  // back to the last cluster end
    r = e;
  }
  start.push_back(P.nd);
  const int nblk = (int)start.size() - 1;
  struct Part {
    int cluster, lo, hi;  // rows of the group the cluster covers
  };
  std::vector<std::vector<Part>> parts(nblk);
  for (int ci = 0; ci < (int)clusters.size(); ci++) {
    const Cluster &c = clusters[ci];
    int b = (int)(std::upper_bound(start.begin(), start.end(), c.row0) - start.begin()) - 1;
    for (; b < nblk && start[b] < c.row0 + c.rows; b++)
      parts[b].push_back({ci, std::max(0, c.row0 - start[b]),
                          std::min(start[b + 1], c.row0 + c.rows) - start[b]});
  }
  M.yptr.assign(2 * (size_t)P.nd, 0);
  struct Dense {  // rows [lo, hi) of a dense leaf's columns [v, v + ncols)
    int v, ncols, lo, hi;
    int64_t src;
    int ld, leaf;
  };
  std::vector<Dense> dense;
  std::vector<MultiItem> small;
  std::vector<int> lo_of;
  for (int b = 0; b < nblk; b++) {
    const int r0 = start[b], nr = start[b + 1] - r0;
    col.slices.clear();
    col.pack.clear();
    std::map<std::pair<int, int>, Columns> partial;
    auto columns_of = [&](int lo, int hi) -> Columns & { return lo == 0 && hi == nr ? col : partial[{lo, hi}]; };
    // dense columns: the leaves of one column cluster that follow each other
    // in the rows are taken as one
    dense.clear();
    for (const Part &p : parts[b]) {
      const Cluster &c = clusters[p.cluster];
      for (const Factor &F : c.factors)
        if (!F.t) dense.push_back({F.v, F.ncols, p.lo, p.hi, F.base + (r0 + p.lo - c.row0), c.ld, F.leaf});
    }
    std::sort(dense.begin(), dense.end(), [](const Dense &x, const Dense &y) {
      if (x.v != y.v) return x.v < y.v;
      if (x.ncols != y.ncols) return x.ncols < y.ncols;
      return x.lo != y.lo ? x.lo < y.lo : x.leaf < y.leaf;
    });
    for (size_t i = 0; i < dense.size();) {
      size_t j = i + 1;
      while (j < dense.size() && dense[j].v == dense[i].v && dense[j].ncols == dense[i].ncols &&
             dense[j].lo == dense[j - 1].hi)
        j++;
      const int lo = dense[i].lo, hi = dense[j - 1].hi;
      Columns &c = columns_of(lo, hi);
      for (size_t q = i; q < j; q++)
        c.pack.push_back({dense[q].src, (int64_t)c.slices.size(), dense[q].ld, dense[q].hi - dense[q].lo, dense[q].ncols,
                          dense[q].lo - lo, 0, 0, bf16 ? 2 * dense[q].leaf + 1 : -1, 0});
      B.add_slices(c, dense[i].ncols, dense[i].v, false);
      i = j;
    }
    // columns of t: a2 factors back to back with their t rows in order are one factor
    for (const Part &p : parts[b]) {
      const Cluster &c = clusters[p.cluster];
      for (size_t q = 0; q < c.factors.size(); q++) {
        const Factor &F = c.factors[q];
        if (!F.t) continue;
        int n = F.ncols;
        while (q + 1 < c.factors.size() && c.factors[q + 1].t &&
               c.factors[q + 1].base == F.base + (int64_t)n * c.ld && c.factors[q + 1].v == F.v + n)
          n += c.factors[++q].ncols;
        Columns &cc = columns_of(p.lo, p.hi);
        cc.pack.push_back({F.base + (r0 + p.lo - c.row0), (int64_t)cc.slices.size(), c.ld, p.hi - p.lo, n, 0, 0, 0, -1, 0});
        B.add_slices(cc, n, F.v, true);
      }
    }
    // partial items, the large ones split so that one wave does not outlast the others
    auto nbatch_of = [](const Columns &c) { return (int)((c.slices.size() + kMultiBatch - 1) / kMultiBatch); };
    double total = nbatch_of(col) * batch_cost(nr);
    for (const auto &kv : partial) total += nbatch_of(kv.second) * batch_cost(kv.first.second - kv.first.first);
    small.clear();
    lo_of.clear();
    for (auto &kv : partial) {
      const int lo = kv.first.first, n = kv.first.second - lo;
      const Builder::Place bb = B.place(kv.second, n);
      const int np = std::max(1, std::min(bb.nbatch, (int)(bb.nbatch * batch_cost(n) / (total / nw) + 0.75)));
      for (int q = 0; q < np; q++) {
        const int q0 = (int)((int64_t)bb.nbatch * q / np), q1 = (int)((int64_t)bb.nbatch * (q + 1) / np);
        small.push_back({bb.a0 + (int64_t)q0 * kMultiBatch * n * B.KS, bb.slice0 + q0 * kMultiBatch, q1 - q0, n,
                         (int32_t)M.n_slots, kItemSlot, 0});
        lo_of.push_back(lo);
        M.n_slots += n;
        if (M.n_slots > INT32_MAX) return kMultiTooLarge;
      }
    }
    // y lists: rows between two ends of partial items add the same slots
    if (!small.empty()) {
      std::vector<int> ends = {0, nr};
      for (size_t q = 0; q < small.size(); q++) {
        ends.push_back(lo_of[q]);
        ends.push_back(lo_of[q] + small[q].nrows);
      }
      std::sort(ends.begin(), ends.end());
      ends.erase(std::unique(ends.begin(), ends.end()), ends.end());
      for (size_t e = 0; e + 1 < ends.size(); e++) {
        const int32_t p0 = (int32_t)M.ylist.size();
        for (size_t q = 0; q < small.size(); q++)
          if (lo_of[q] <= ends[e] && ends[e] < lo_of[q] + small[q].nrows)
            M.ylist.push_back(small[q].out - (r0 + lo_of[q]));
        for (int r = ends[e]; r < ends[e + 1]; r++) {
          M.yptr[2 * ((size_t)r0 + r)] = p0;
          M.yptr[2 * ((size_t)r0 + r) + 1] = (int32_t)M.ylist.size();
        }
      }
      if (M.ylist.size() > (size_t)INT32_MAX) return kMultiTooLarge;
    }
    // partial items to the waves, largest first to the least loaded
    std::vector<int> ord(small.size());
    for (size_t q = 0; q < ord.size(); q++) ord[q] = (int)q;
    std::sort(ord.begin(), ord.end(), [&](int x, int y) {
      const double cx = small[x].nbatch * batch_cost(small[x].nrows), cy = small[y].nbatch * batch_cost(small[y].nrows);
      return cx != cy ? cx > cy : x < y;
    });
    std::vector<std::vector<MultiItem>> own(nw);
    std::vector<double> load(nw, 0.0);
    for (int q : ord) {
      const int w = (int)(std::min_element(load.begin(), load.end()) - load.begin());
      own[w].push_back(small[q]);
      load[w] += small[q].nbatch * batch_cost(small[q].nrows) + 2.0;
    }
    add_group(Bl, kMultiY, r0, r0, B.place(col, nr), nr, own, load);
  }
  if (M.slices.size() > (size_t)INT32_MAX || M.items.size() > (size_t)INT32_MAX) return kMultiTooLarge;
  A.finish(nw, &M.groups_a, &M.waves_a);
  Bl.finish(nw, &M.groups_b, &M.waves_b);
  return "";
}

std::string window_multi_plan(int storage, int64_t cap, MultiPlan *Mp, std::vector<MultiWindow> *out) {
  MultiPlan &M = *Mp;
  out->clear();
  const int KS = multi_slice_cols(storage), nw = M.waves;
  size_t rec = 0;
  for (int list = 0; list < 2; list++) {
    std::vector<MultiGroup> &gl = list == 0 ? M.groups_a : M.groups_b;
    std::vector<MultiWave> &wl = list == 0 ? M.waves_a : M.waves_b;
    struct Range {
      int64_t a, b;
      size_t g;
    };
    std::vector<Range> rg;
    for (size_t g = 0; g < gl.size(); g++) {
      Range r{INT64_MAX, 0, g};
      for (int w = 0; w < nw; w++) {
        const MultiWave &wv = wl[g * nw + w];
        for (int i = wv.item0; i < wv.item0 + wv.nitems; i++) {
          const MultiItem &it = M.items[(size_t)i];
          if (it.nbatch == 0) continue;
          r.a = std::min(r.a, it.a0);
          r.b = std::max(r.b, it.a0 + (int64_t)it.nbatch * kMultiBatch * it.nrows * KS);
        }
      }
      if (r.a > r.b) r.a = r.b;  // a group without values
      rg.push_back(r);
    }
    std::stable_sort(rg.begin(), rg.end(), [](const Range &x, const Range &y) { return x.a < y.a; });
    std::vector<MultiGroup> ng;
    std::vector<MultiWave> nwv;
    for (size_t i = 0; i < rg.size();) {
      MultiWindow win{rg[i].a, list, (int32_t)ng.size(), 0, (int32_t)rec, 0};
      int64_t end = rg[i].b;
      size_t j = i;
      while (j < rg.size() && std::max(end, rg[j].b) - win.a0 <= cap) end = std::max(end, rg[j++].b);
      if (j == i) return "a group's values exceed the window";
      std::vector<size_t> in;
      for (size_t q = i; q < j; q++) in.push_back(rg[q].g);
      std::sort(in.begin(), in.end());
      for (size_t g : in) {
        ng.push_back(gl[g]);
        nwv.insert(nwv.end(), wl.begin() + (std::ptrdiff_t)(g * nw), wl.begin() + (std::ptrdiff_t)((g + 1) * nw));
      }
      while (rec < M.pack.size() && M.pack[rec].dst < end) rec++;
      win.ngroups = (int32_t)in.size();
      win.npack = (int32_t)rec - win.pack0;
      out->push_back(win);
      i = j;
    }
    gl.swap(ng);
    wl.swap(nwv);
  }
  if (rec != M.pack.size()) return "pack records outside the windows";
  // what the kernels of a window address lies inside its buffer
  for (const MultiWindow &w : *out) {
    auto outside = [&](int64_t a, int64_t n) { return a < w.a0 || a + n > w.a0 + cap; };
    for (int32_t i = w.pack0; i < w.pack0 + w.npack; i++) {
      const MultiPack &r = M.pack[(size_t)i];
      if (outside(r.dst, ((r.cols + KS - 1) / KS + r.pad) * (int64_t)r.nrows * KS)) return "pack record outside its window";
    }
    const std::vector<MultiWave> &wl = w.launch == 0 ? M.waves_a : M.waves_b;
    for (size_t k = (size_t)w.group0 * nw; k < (size_t)(w.group0 + w.ngroups) * nw; k++)
      for (int i = wl[k].item0; i < wl[k].item0 + wl[k].nitems; i++) {
        const MultiItem &it = M.items[(size_t)i];
        if (it.nbatch > 0 && outside(it.a0, (int64_t)it.nbatch * kMultiBatch * it.nrows * KS)) return "item outside its window";
      }
  }
  return "";
}

std::string verify_multi_plan(const Plan &P, int storage, const MultiPlan &M) {
  const int KS = multi_slice_cols(storage);
  const int64_t nslice = (int64_t)M.slices.size();
  // packing: sources inside the values, each element once
  int64_t packed = 0;
  for (const MultiPack &r : M.pack) {
    if (r.rows < 1 || r.cols < 1 || r.row0 < 0 || r.row0 + r.rows > r.nrows || r.pad < 0) return "pack record shape";
    if (r.src < 0 || r.ld < 1 || r.src + r.rows - 1 + (int64_t)(r.cols - 1) * r.ld >= P.nvals)
      return "pack source outside the values";
    if (r.factor >= P.nfactors) return "pack factor";
    packed += (int64_t)r.rows * r.cols;
  }
  if (packed != P.len) return "packing does not cover the leaves";
  // the records of the same slices cover the item's rows, one after the
  // other, and the slices follow each other up to the last value
  std::vector<int32_t> order(M.pack.size());
  for (size_t i = 0; i < order.size(); i++) order[i] = (int32_t)i;
  auto before = [&](int32_t x, int32_t y) {
    const MultiPack &p = M.pack[(size_t)x], &q = M.pack[(size_t)y];
    return p.dst != q.dst ? p.dst < q.dst : p.row0 < q.row0;
  };
  if (!std::is_sorted(order.begin(), order.end(), before)) std::sort(order.begin(), order.end(), before);
  int64_t end = 0;
  for (size_t i = 0; i < order.size();) {
    const MultiPack &f = M.pack[(size_t)order[i]];
    const int64_t ns = (f.cols + KS - 1) / KS + f.pad;
    int row = 0;
    if (f.dst != end) return "packed values overlap or have gaps";
    for (; i < order.size() && M.pack[(size_t)order[i]].dst == f.dst; i++) {
      const MultiPack &r = M.pack[(size_t)order[i]];
      if (r.row0 != row || r.nrows != f.nrows || (r.cols + KS - 1) / KS + r.pad != ns)
        return "pack records of the same slices disagree";
      row += r.rows;
    }
    if (row != f.nrows) return "packed rows missing";
    end += ns * f.nrows * KS;
  }
  if (end != M.nvals) return "packing does not cover the packed values";
  // every packed element is read by one item: the items' values follow each other
  std::vector<std::pair<int64_t, int64_t>> read;
  for (const MultiItem &it : M.items)
    if (it.nbatch > 0) read.push_back({it.a0, it.a0 + (int64_t)it.nbatch * kMultiBatch * it.nrows * KS});
  std::sort(read.begin(), read.end());
  end = 0;
  for (const auto &r : read) {
    if (r.first != end) return "items overlap or leave packed values out";
    end = r.second;
  }
  if (end != M.nvals) return "items leave packed values out";
  int64_t covered = 0;
  std::vector<char> t_seen((size_t)M.n_t, 0), y_seen((size_t)P.nd, 0), slot_seen((size_t)M.n_slots, 0);
  for (int list = 0; list < 2; list++) {
    const std::vector<MultiGroup> &gl = list == 0 ? M.groups_a : M.groups_b;
    const std::vector<MultiWave> &wl = list == 0 ? M.waves_a : M.waves_b;
    if (wl.size() != gl.size() * (size_t)M.waves) return "waves of the groups";
    for (size_t gi = 0; gi < gl.size(); gi++) {
      const MultiGroup &g = gl[gi];
      if (g.nrows < 1 || g.nrows > kMultiRows || g.out < 0) return "group shape";
      for (int w = 0; w < M.waves; w++) {
        const MultiWave &wv = wl[gi * (size_t)M.waves + w];
        if (wv.item0 < 0 || wv.nitems < (g.kind == kMultiNone ? 0 : 1) ||
            (int64_t)wv.item0 + wv.nitems > (int64_t)M.items.size())
          return "wave items out of range";
        for (int i = wv.item0; i < wv.item0 + wv.nitems; i++) {
          const MultiItem &it = M.items[(size_t)i];
          if (it.nrows < 1 || it.nrows > (storage == kBF16 && list == 0 ? kOrderedRows : kMultiRows)) return "item rows";
          if (it.slice0 < 0 || it.nbatch < 0 || (int64_t)it.slice0 + (int64_t)it.nbatch * kMultiBatch > nslice)
            return "item slices";
          if (it.a0 < 0 || it.a0 + (int64_t)it.nbatch * kMultiBatch * it.nrows * KS > M.nvals)
            return "item outside the packed values";
          const bool last = g.kind != kMultiNone && i == wv.item0 + wv.nitems - 1;
          if (last != (it.kind == kItemKept) || (last && it.nrows != g.nrows)) return "kept item not last";
          for (int r = 0; r < it.nrows && !last; r++) {
            if (it.kind == kItemSlot) {
              if (it.out < 0 || (int64_t)it.out + r >= M.n_slots) return "item slot out of range";
              if (slot_seen[(size_t)it.out + r]++) return "slot written twice";
            } else if (it.kind == kItemT && list == 0) {
              if (it.out < 0 || (int64_t)it.out + r >= (int64_t)M.tmap.size()) return "t map out of range";
              const int32_t e = M.tmap[(size_t)it.out + r];
              if (e < 0 || e >= M.n_t || t_seen[(size_t)e]++) return "t row out of range or written twice";
            } else {
              return "item kind";
            }
          }
          for (int64_t s = it.slice0; s < it.slice0 + (int64_t)it.nbatch * kMultiBatch; s++) {
            const MultiSlice &q = M.slices[(size_t)s];
            const bool t = (q.info & kSliceT) != 0, ordered = storage == kBF16 && list == 0;
            const int n1 = q.info & 15, n2 = ordered ? (q.info >> 4) & 15 : 0, n = n1 + n2;
            if (n > KS || (ordered && (n1 > kHalf || n2 > kHalf)) || (t && list == 0)) return "slice";
            // a wave's columns end with a chunk, and a batch's slices agree
            if (ordered && (q.info & kSliceEnd) != (M.slices[(size_t)((s / kMultiBatch) * kMultiBatch)].info & kSliceEnd))
              return "chunk end";
            if (ordered && s == it.slice0 + (int64_t)it.nbatch * kMultiBatch - 1 && !(q.info & kSliceEnd))
              return "columns end inside a chunk";
            if (q.v < 0 || (int64_t)q.v + (n2 > 0 ? kStep + n2 : n1) > (t ? M.n_t : (int64_t)P.nd))
              return "slice outside its vector";
            covered += (int64_t)n * it.nrows;
          }
        }
      }
      for (int r = 0; r < g.nrows && g.kind != kMultiNone; r++) {
        if (g.kind == kMultiT && list == 0) {
          if ((int64_t)g.out + r >= (int64_t)M.tmap.size()) return "t map out of range";
          const int32_t e = M.tmap[(size_t)g.out + r];
          if (e < 0 || e >= M.n_t || t_seen[(size_t)e]++) return "t row out of range or written twice";
        } else if (g.kind == kMultiTSlot && list == 0) {
          if ((int64_t)g.out + r >= M.n_slots || slot_seen[(size_t)g.out + r]++) return "t slot";
        } else if (g.kind == kMultiY && list == 1) {
          if ((int64_t)g.out + r >= P.nd || y_seen[(size_t)g.out + r]++) return "y row out of range or written twice";
        } else {
          return "group kind";
        }
      }
    }
  }
  if (covered != P.len) return "items do not cover the leaves";
  for (const MultiPlan::TSum &t : M.tsum) {
    if (t.entry < 0 || t.entry >= M.n_t || t_seen[(size_t)t.entry]++) return "t sum entry";
    if (t.nch < 1 || t.first < 0 || t.stride < 0 || (int64_t)t.first + (int64_t)(t.nch - 1) * t.stride >= M.n_slots)
      return "t sum slots out of range";
    if (t.nch > 0xFFFF || t.stride > 0xFFFF) return "t sum with more than 65535 chunks";
    for (int c = 0; c < t.nch; c++)
      if (!slot_seen[(size_t)t.first + (size_t)c * t.stride]) return "t sum reads a slot nothing writes";
  }
  for (char c : t_seen)
    if (!c) return "t row never written";
  for (char c : y_seen)
    if (!c) return "y row never written";
  if (M.yptr.size() != 2 * (size_t)P.nd) return "y lists";
  for (int r = 0; r < P.nd; r++) {
    const int b = M.yptr[2 * (size_t)r], e = M.yptr[2 * (size_t)r + 1];
    if (b < 0 || e < b || e > (int64_t)M.ylist.size()) return "y list range";
    for (int i = b; i < e; i++) {
      const int64_t s = (int64_t)M.ylist[(size_t)i] + r;
      if (s < 0 || s >= M.n_slots || !slot_seen[(size_t)s]) return "y list slot";
    }
  }
  return "";
}

std::string verify_multi_values(const Plan &P, int storage, const int *nstrtl, const int *nstrtt, const MultiPlan &M) {
  const int KS = multi_slice_cols(storage);
  // the repack record of every element of the value layout, and its first
  // rank row or column in the factor
  std::vector<int32_t> owner((size_t)P.nvals, -1);
  std::vector<int> first(P.repack.size(), 0), kdone(P.nlf, 0);
  for (size_t i = 0; i < P.repack.size(); i++) {
    const RepackDesc &r = P.repack[i];
    if (r.rows == 0 || r.cols == 0) continue;
    if (r.factor % 2 == 0) {
      first[i] = kdone[r.factor / 2];
      kdone[r.factor / 2] += r.rows;
    }
    for (int c = 0; c < r.cols; c++)
      for (int k = 0; k < r.rows; k++) owner[(size_t)(r.dst_off + k + (int64_t)c * r.dst_cs)] = (int32_t)i;
  }
  std::vector<int> t_idx(P.nlf, -1);
  for (int64_t e = M.n_t; e-- > 0;) t_idx[(size_t)M.t_factor[(size_t)e] / 2] = (int)e;
  // where the rows of every item go: a row of t (launch A) or of y
  struct Read {
    int64_t a0, end;
    int32_t item, row0;  // row0: first row of y or index in t_of
    int list;
  };
  std::vector<int32_t> t_of(M.tmap), slot_t((size_t)M.n_slots, -1);
  for (const MultiPlan::TSum &t : M.tsum)
    for (int c = 0; c < t.nch; c++) slot_t[(size_t)t.first + (size_t)c * t.stride] = t.entry;
  std::vector<int32_t> slot_y((size_t)M.n_slots, -1);
  std::vector<char> added((size_t)M.n_slots, 0);
  for (int r = 0; r < P.nd; r++)
    for (int i = M.yptr[2 * (size_t)r]; i < M.yptr[2 * (size_t)r + 1]; i++) {
      const size_t q = (size_t)M.ylist[(size_t)i] + r;
      if (added[q]++) return "slot added to y twice";
      slot_y[q] = r;
    }
  std::vector<Read> read;
  for (int list = 0; list < 2; list++) {
    const std::vector<MultiGroup> &gl = list == 0 ? M.groups_a : M.groups_b;
    const std::vector<MultiWave> &wl = list == 0 ? M.waves_a : M.waves_b;
    for (size_t k = 0; k < wl.size(); k++)
      for (int i = wl[k].item0; i < wl[k].item0 + wl[k].nitems; i++) {
        const MultiItem &it = M.items[(size_t)i];
        const MultiGroup &g = gl[k / (size_t)M.waves];
        if (it.nbatch == 0) continue;
        Read r{it.a0, it.a0 + (int64_t)it.nbatch * kMultiBatch * it.nrows * KS, i, 0, list};
        const bool slots = it.kind == kItemSlot || (it.kind == kItemKept && g.kind == kMultiTSlot);
        const int out = it.kind == kItemKept ? g.out : it.out;
        if (list == 0 && !slots) {
          r.row0 = out;
        } else if (list == 0) {
          r.row0 = (int32_t)t_of.size();
          for (int q = 0; q < it.nrows; q++) t_of.push_back(slot_t[(size_t)out + q]);
        } else if (slots) {
          r.row0 = slot_y[(size_t)out];
          for (int q = 0; q < it.nrows; q++)
            if (slot_y[(size_t)out + q] != r.row0 + q || r.row0 < 0) return "slot added to another row of y";
        } else {
          r.row0 = out;
        }
        read.push_back(r);
      }
  }
  std::sort(read.begin(), read.end(), [](const Read &x, const Read &y) { return x.a0 < y.a0; });
  for (const MultiPack &r : M.pack) {
    const int64_t step = (int64_t)r.nrows * KS;  // of a slice
    for (int s = 0; s < (r.cols + KS - 1) / KS + r.pad; s++) {
      const int64_t at = r.dst + s * step;
      auto rd = std::upper_bound(read.begin(), read.end(), at, [](int64_t a, const Read &x) { return a < x.a0; });
      if (rd == read.begin()) return "packed slice without an item";
      --rd;
      const MultiItem &it = M.items[(size_t)rd->item];
      if (at >= rd->end || it.nrows != r.nrows || (at - rd->a0) % step) return "packed slice beside its item";
      const MultiSlice &q = M.slices[(size_t)it.slice0 + (size_t)((at - rd->a0) / step)];
      const bool ordered = storage == kBF16 && rd->list == 0;
      if (ordered != (r.ordered != 0)) return "order of a pack record";
      const int n1 = q.info & 15, n2 = ordered ? (q.info >> 4) & 15 : 0;
      for (int j = 0; j < KS; j++) {
        const int c = ordered ? ordered_column(s, j) : s * KS + j;
        const bool in_use = ordered && j >= kHalf ? j - kHalf < n2 : j < n1;
        if (in_use != (c < r.cols)) return "columns of a slice in use";
        if (!in_use) continue;
        const int v = q.v + (ordered && j >= kHalf ? kStep + j - kHalf : j);
        for (int k = 0; k < r.rows; k++) {
          const int64_t p = r.src + k + (int64_t)c * r.ld;
          const int32_t o = owner[(size_t)p];
          if (o < 0) return "element packed twice, or none";
          owner[(size_t)p] = -1;
          const RepackDesc &d = P.repack[(size_t)o];
          const int leaf = d.factor / 2, row = (int)((p - d.dst_off) % d.dst_cs), col = (int)((p - d.dst_off) / d.dst_cs);
          const bool a1 = d.factor % 2 == 0, a2 = !a1 && kdone[(size_t)leaf] > 0;
          if (a1 != (rd->list == 0) || a2 != ((q.info & kSliceT) != 0)) return "factor in the wrong launch";
          if (v != (a2 ? t_idx[(size_t)leaf] : nstrtt[leaf] - 1) + col) return "element meets another vector entry";
          const int out = a1 ? t_of[(size_t)rd->row0 + r.row0 + k] : rd->row0 + r.row0 + k;
          if (out != (a1 ? t_idx[(size_t)leaf] + first[(size_t)o] : nstrtl[leaf] - 1) + row) return "element goes to another row";
          if (r.factor >= 0 && r.factor != d.factor) return "scale of another factor";
          if (storage == kBF16 && !a1 && !a2 && r.factor < 0) return "dense leaf without its scale";
        }
      }
    }
  }
  for (int32_t o : owner)
    if (o >= 0) return "element never packed";
  return "";
}

}  // namespace hmvm
