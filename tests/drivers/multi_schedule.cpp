// The multi-RHS schedule on the CPU: built, checked and executed in FP64 as the
// kernels read it (packed values, batches of slices, items, groups, t sums, y
// lists), against the leaves; and damaged in ways that keep all totals, which
// the checks have to report.
//   usage: multi_schedule hmatrix_1.bin storage t_mode windows
// (windows: 1 in windows as small as the largest group allows, 0 all values packed at once)
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <functional>
#include <string>
#include <utility>
#include <vector>

#include "hacapk.h"
#include "hmvm_multi_plan.hpp"

using namespace hmvm;

static std::vector<double> leaves(const matrix2 &m, const std::vector<double> &x) {
  std::vector<double> y((size_t)m.nd, 0.0);
  for (int i = 0; i < m.nlf; i++) {
    const int nl = m.ndl[i], nt = m.ndt[i], r0 = m.nstrtl[i] - 1, c0 = m.nstrtt[i] - 1;
    const double *a1 = m.rowmat + m.a1[i], *a2 = m.rowmat + m.a2[i];
    if (m.ltmtx[i] == 2) {
      for (int il = 0; il < nl; il++)
        for (int it = 0; it < nt; it++) y[r0 + il] += a1[il * nt + it] * x[c0 + it];
      continue;
    }
    for (int k = 0; k < m.kt[i]; k++) {
      double t = 0;
      for (int it = 0; it < nt; it++) t += a1[k * nt + it] * x[c0 + it];
      for (int il = 0; il < nl; il++) y[r0 + il] += a2[k * nl + il] * t;
    }
  }
  return y;
}

// The rows of one item, in FP64.
static std::vector<double> item_sum(const MultiPlan &M, int KS, int E, bool ordered, const MultiItem &it,
                                    const std::vector<double> &vals, const std::vector<double> &x,
                                    const std::vector<double> &t) {
  std::vector<double> s((size_t)it.nrows, 0.0);
  for (int q = 0; q < it.nbatch * kMultiBatch; q++) {
    const MultiSlice &sl = M.slices[(size_t)it.slice0 + q];
    const int n1 = sl.info & 15, n2 = ordered ? (sl.info >> 4) & 15 : 0;
    for (int j = 0; j < KS; j++) {
      const bool second = ordered && j >= kHalf;
      if (second ? j - kHalf >= n2 : j >= n1) continue;
      const double v = (sl.info & kSliceT ? t : x)[(size_t)sl.v + (second ? kStep + j - kHalf : j)];
      for (int r = 0; r < it.nrows; r++)
        s[r] += vals[(size_t)(it.a0 + ((int64_t)q * (KS / E) + j / E) * it.nrows * E + r * E + j % E)] * v;
    }
  }
  return s;
}

// launch: which groups; window: pack records from base on into `vals`.
static void run(const MultiPlan &M, int KS, int E, bool bf16, int launch, size_t g0, size_t ng, const std::vector<double> &vals,
                const std::vector<double> &x, std::vector<double> &t, std::vector<double> &slots, std::vector<double> &y) {
  const std::vector<MultiGroup> &gl = launch == 0 ? M.groups_a : M.groups_b;
  const std::vector<MultiWave> &wl = launch == 0 ? M.waves_a : M.waves_b;
  for (size_t g = g0; g < g0 + ng; g++) {
    std::vector<double> kept((size_t)gl[g].nrows, 0.0);
    for (int w = 0; w < M.waves; w++) {
      const MultiWave &wv = wl[g * (size_t)M.waves + w];
      for (int i = wv.item0; i < wv.item0 + wv.nitems; i++) {
        const MultiItem &it = M.items[(size_t)i];
        const std::vector<double> s = item_sum(M, KS, E, bf16 && launch == 0, it, vals, x, t);
        for (int r = 0; r < it.nrows; r++) {
          if (it.kind == kItemKept) kept[r] += s[r];
          else if (it.kind == kItemSlot) slots[(size_t)it.out + r] = s[r];
          else t[(size_t)M.tmap[(size_t)it.out + r]] = s[r];
        }
      }
    }
    for (int r = 0; r < gl[g].nrows && gl[g].kind != kMultiNone; r++) {
      const size_t o = (size_t)gl[g].out + r;
      if (gl[g].kind == kMultiT) t[(size_t)M.tmap[o]] = kept[r];
      else if (gl[g].kind == kMultiTSlot) slots[o] = kept[r];
      else {
        y[o] = kept[r];
        for (int q = M.yptr[2 * o]; q < M.yptr[2 * o + 1]; q++) y[o] += slots[(size_t)M.ylist[q] + o];
      }
    }
  }
}

int main(int argc, char **argv) {
  if (argc < 5) return 2;
  const int storage = std::atoi(argv[2]), t_mode = std::atoi(argv[3]), window = std::atoi(argv[4]);
  matrix mat;
  matrix2 m;
  if (loadHmatrix(argv[1], &mat, &m)) return 2;
  std::vector<int64_t> a1(m.a1, m.a1 + m.nlf), a2(m.a2, m.a2 + m.nlf);
  LeafArrays la{};
  la.nd = m.nd, la.nlf = m.nlf, la.ltmtx = m.ltmtx, la.kt = m.kt, la.ndl = m.ndl, la.ndt = m.ndt;
  la.nstrtl = m.nstrtl, la.nstrtt = m.nstrtt, la.src_a1 = a1.data(), la.src_a2 = a2.data(), la.src_len = m.len;
  PlanOptions po;
  po.storage = storage;
  po.t_mode = t_mode < 0 ? 1 : t_mode;
  po.bands = t_mode < 0;
  po.w1 = 2000;
  po.chunk_w = 1500;
  Plan P;
  MultiPlan M;
  MultiOptions opt = multi_options(P);
  std::string err = build_plan(la, po, &P);
  if (err.empty()) opt = multi_options(P);
  if (window > 0) opt.wave_cols = 0;
  if (err.empty()) err = build_multi_plan(P, storage, m.nstrtl, m.nstrtt, opt, &M);
  std::vector<MultiWindow> win;
  if (err.empty() && window > 0) {
    // the least window there is: doubled from one value until the groups fit
    const MultiPlan all = M;
    int64_t cap = 1;
    while (!(err = window_multi_plan(storage, cap, &M, &win)).empty() && cap < M.nvals) {
      M = all;
      cap *= 2;
    }
  }
  auto check = [&](const MultiPlan &Q) {
    std::string e = verify_multi_plan(P, storage, Q);
    return e.empty() ? verify_multi_values(P, storage, m.nstrtl, m.nstrtt, Q) : e;
  };
  if (err.empty()) err = check(M);
  if (!err.empty()) return std::printf("refused: %s\n", err.c_str()), 1;

  // ---- replay --------------------------------------------------------------------
  std::vector<double> x((size_t)m.nd), t((size_t)M.n_t, 0.0), slots((size_t)M.n_slots, 0.0), y((size_t)m.nd, 0.0);
  for (size_t i = 0; i < x.size(); i++) x[i] = std::sin((double)(i + 1));
  std::vector<double> layout((size_t)P.nvals, 0.0);
  for (const RepackDesc &r : P.repack)
    for (int c = 0; c < r.cols; c++)
      for (int k = 0; k < r.rows; k++)
        layout[(size_t)(r.dst_off + k + (int64_t)c * r.dst_cs)] =
            m.rowmat[(size_t)(r.src_off + (int64_t)k * r.src_rs + (int64_t)c * r.src_cs)];
  const int KS = multi_slice_cols(storage), E = multi_word(storage);
  std::vector<double> vals((size_t)M.nvals);
  auto pack = [&](size_t r0, size_t n) {
    for (size_t i = r0; i < r0 + n; i++) {
      const MultiPack &r = M.pack[i];
      for (int s = 0; s < (r.cols + KS - 1) / KS + r.pad; s++)
        for (int k = 0; k < r.rows; k++)
          for (int j = 0; j < KS; j++) {
            const int c = r.ordered ? ordered_column(s, j) : s * KS + j;
            vals[(size_t)(r.dst + (int64_t)s * r.nrows * KS + (int64_t)(j / E) * r.nrows * E + (r.row0 + k) * E + j % E)] =
                c < r.cols ? layout[(size_t)(r.src + k + (int64_t)c * r.ld)] : 0.0;
          }
    }
  };
  const bool bf16 = storage == kBF16;
  for (int launch = 0; launch < 2; launch++) {
    if (win.empty()) {
      if (launch == 0) std::fill(vals.begin(), vals.end(), NAN), pack(0, M.pack.size());
      run(M, KS, E, bf16, launch, 0, (launch == 0 ? M.groups_a : M.groups_b).size(), vals, x, t, slots, y);
    }
    for (const MultiWindow &w : win) {
      if (w.launch != launch) continue;
      std::fill(vals.begin(), vals.end(), NAN);
      pack((size_t)w.pack0, (size_t)w.npack);
      run(M, KS, E, bf16, launch, (size_t)w.group0, (size_t)w.ngroups, vals, x, t, slots, y);
    }
    if (launch == 0)
      for (const MultiPlan::TSum &s : M.tsum) {
        t[(size_t)s.entry] = 0;
        for (int c = 0; c < s.nch; c++) t[(size_t)s.entry] += slots[(size_t)s.first + (size_t)c * s.stride];
      }
  }
  const std::vector<double> ref = leaves(m, x);
  double d = 0, n = 0;
  for (size_t i = 0; i < y.size(); i++) d += (y[i] - ref[i]) * (y[i] - ref[i]), n += ref[i] * ref[i];
  const double rel = std::sqrt(d) / std::sqrt(n);
  std::printf("windows %zu tsum %zu slots %lld rel %.3e\n", win.size(), M.tsum.size(), (long long)M.n_slots, rel);
  if (!(rel <= 1e-13)) return 1;

  // ---- damage --------------------------------------------------------------------
  int missed = 0;
  auto damage = [&](const char *what, const std::function<bool(MultiPlan &)> &f) {
    MultiPlan Q = M;
    if (!f(Q)) return (void)std::printf("%s: nothing to damage\n", what);
    const std::string e = check(Q);
    std::printf("%s: %s\n", what, e.empty() ? "MISSED" : e.c_str());
    missed += e.empty();
  };
  auto same_shape = [](const MultiPack &a, const MultiPack &b) {
    return a.rows == b.rows && a.cols == b.cols && a.nrows == b.nrows && a.pad == b.pad && a.ordered == b.ordered &&
           a.src != b.src;
  };
  auto pair_of = [&](const std::function<bool(size_t, size_t)> &ok, size_t count) {
    for (size_t i = 0; i < count; i++)
      for (size_t j = i + 1; j < std::min(count, i + 200); j++)
        if (ok(i, j)) return std::make_pair(i, j);
    return std::make_pair(size_t(0), size_t(0));
  };
  damage("sources of two records swapped", [&](MultiPlan &Q) {
    auto p = pair_of([&](size_t i, size_t j) { return same_shape(Q.pack[i], Q.pack[j]); }, Q.pack.size());
    std::swap(Q.pack[p.first].src, Q.pack[p.second].src);
    return p.second > 0;
  });
  damage("record packed over another", [&](MultiPlan &Q) {
    auto p = pair_of([&](size_t i, size_t j) { return same_shape(Q.pack[i], Q.pack[j]) && Q.pack[i].dst != Q.pack[j].dst; },
                     Q.pack.size());
    Q.pack[p.second].dst = Q.pack[p.first].dst;
    return p.second > 0;
  });
  damage("source packed twice", [&](MultiPlan &Q) {
    auto p = pair_of([&](size_t i, size_t j) { return same_shape(Q.pack[i], Q.pack[j]); }, Q.pack.size());
    Q.pack[p.second].src = Q.pack[p.first].src;
    return p.second > 0;
  });
  damage("slice of other columns", [&](MultiPlan &Q) {
    for (MultiSlice &s : Q.slices)
      if ((s.info & 15) > 0 && !(s.info & kSliceT) && s.v > 0) return s.v--, true;
    return false;
  });
  damage("items read each other's values", [&](MultiPlan &Q) {
    auto p = pair_of([&](size_t i, size_t j) {
      const MultiItem &a = Q.items[i], &b = Q.items[j];
      return a.nbatch > 0 && a.nbatch == b.nbatch && a.nrows == b.nrows && a.a0 != b.a0;
    }, Q.items.size());
    std::swap(Q.items[p.first].a0, Q.items[p.second].a0);
    return p.second > 0;
  });
  damage("rows of t swapped", [&](MultiPlan &Q) {
    if (Q.tmap.size() < 2) return false;
    std::swap(Q.tmap[0], Q.tmap[1]);
    return true;
  });
  damage("t sums swapped", [&](MultiPlan &Q) {
    if (Q.tsum.size() < 2) return false;
    std::swap(Q.tsum[0].entry, Q.tsum[1].entry);
    return true;
  });
  damage("slot added to another row", [&](MultiPlan &Q) {
    for (size_t r = 0; r + 1 < (size_t)m.nd; r++)
      for (int q = Q.yptr[2 * r]; q < Q.yptr[2 * r + 1]; q++) return Q.ylist[q]++, true;
    return false;
  });
  return missed ? 1 : 0;
}
