// Geometric nested dissection and interface labelling (host, integer work).
// Reference: partition.cpp:54-157 (helpers, rows2clusters, rmap2cmap),
// 241-348 (bissect_geo, GeometricPartitionAtA), 506-578 (getInterfacesUsingA);
// tree.cpp:46-163 (initPermutation, form_rmap).
#include "partition.hpp"

#include "parallel.hpp"

#include <algorithm>
#include <cmath>
#include <limits>
#include <numeric>

namespace spq {

CscMat csc_transpose(const CscMat& A) {
  CscMat T;
  T.m = A.n;
  T.n = A.m;
  T.p.assign(A.m + 1, 0);
  for (int r : A.i) T.p[r + 1]++;
  std::partial_sum(T.p.begin(), T.p.end(), T.p.begin());
  T.i.resize(A.nnz());
  T.x.resize(A.nnz());
  std::vector<int> fill(T.p.begin(), T.p.end() - 1);
  for (int c = 0; c < A.n; ++c)
    for (int q = A.p[c]; q < A.p[c + 1]; ++q) {
      const int dst = fill[A.i[q]]++;
      T.i[dst] = c;
      T.x[dst] = A.x[q];
    }
  return T;
}

// B(r, c) = A(rperm[r], cperm[c]) (either permutation may be null).
CscMat csc_permute(const CscMat& A, const std::vector<int>* rperm, const std::vector<int>* cperm) {
  CscMat B;
  B.m = A.m;
  B.n = A.n;
  B.p.assign(A.n + 1, 0);
  B.i.resize(A.nnz());
  B.x.resize(A.nnz());
  std::vector<int> rinv;
  if (rperm) {
    rinv.resize(A.m);
    for (int r = 0; r < A.m; ++r) rinv[(*rperm)[r]] = r;
  }
  for (int c = 0; c < A.n; ++c) {
    const int src = cperm ? (*cperm)[c] : c;
    B.p[c + 1] = B.p[c] + (A.p[src + 1] - A.p[src]);
  }
  parallel_for(A.n, 4096, [&](int, int b, int e) {
    std::vector<std::pair<int, double>> col;
    for (int c = b; c < e; ++c) {
      const int src = cperm ? (*cperm)[c] : c;
      col.clear();
      for (int q = A.p[src]; q < A.p[src + 1]; ++q) col.push_back({rperm ? rinv[A.i[q]] : A.i[q], A.x[q]});
      if (rperm) std::sort(col.begin(), col.end(), [](const auto& a, const auto& b) { return a.first < b.first; });
      int at = B.p[c];
      for (auto& v : col) { B.i[at] = v.first; B.x[at++] = v.second; }
    }
  });
  return B;
}

std::vector<double> tensor_coordinates(int n, int dim) {
  int64_t N = 1;
  for (int d = 0; d < dim; ++d) N *= n;
  std::vector<double> X((size_t)dim * N);
  for (int64_t id = 0; id < N; ++id) {
    int64_t rem = id;
    for (int d = dim - 1; d >= 0; --d) {  // coordinate 0 varies slowest
      X[(size_t)id * dim + d] = (double)(rem % n);
      rem /= n;
    }
  }
  return X;
}

namespace {

// Median split of the columns [b, e) of `ord` along the coordinate with the
// largest range (first such coordinate on ties): X <= median value goes to the
// front, else to the back, each in its order; returns where the back begins.
int split_geo(std::vector<int>& ord, int b, int e, const std::vector<double>& X, int dim, std::vector<double>& vals,
              std::vector<int>& back) {
  if (b == e) return b;
  int best = -1;
  double range = -1.0;
  for (int d = 0; d < dim; ++d) {
    double mx = std::numeric_limits<double>::lowest(), mn = std::numeric_limits<double>::max();
    for (int q = b; q < e; ++q) {
      const double c = X[(size_t)ord[q] * dim + d];
      mx = std::max(mx, c);
      mn = std::min(mn, c);
    }
    if (mx - mn > range) { range = mx - mn; best = d; }
  }
  vals.clear();
  for (int q = b; q < e; ++q) vals.push_back(X[(size_t)ord[q] * dim + best]);
  const size_t mid = vals.size() / 2;
  std::nth_element(vals.begin(), vals.begin() + mid, vals.end());
  const double cut = vals[mid];
  back.clear();
  int at = b;
  for (int q = b; q < e; ++q) {
    const int v = ord[q];
    if (X[(size_t)v * dim + best] <= cut) ord[at++] = v;
    else back.push_back(v);
  }
  std::copy(back.begin(), back.end(), ord.begin() + at);
  return at;
}

// Pattern of A^T: the columns of each row, sorted.  Chunks of rows are filled
// by a scan of all columns each.
struct Pattern { std::vector<int> p, i; };
Pattern row_pattern(const CscMat& A) {
  Pattern T;
  T.p.assign(A.m + 1, 0);
  for (int r : A.i) T.p[r + 1]++;
  std::partial_sum(T.p.begin(), T.p.end(), T.p.begin());
  T.i.resize(A.nnz());
  const int nch = A.nnz() < 65536 ? 1 : std::min(host_threads(), 8);
  std::vector<int> fill(T.p.begin(), T.p.end() - 1);
  parallel_for(nch, 1, [&](int, int b, int e) {
    const int r0 = (int)((int64_t)b * A.m / nch), r1 = (int)((int64_t)e * A.m / nch);
    for (int c = 0; c < A.n; ++c)
      for (int q = A.p[c]; q < A.p[c + 1]; ++q) {
        const int r = A.i[q];
        if (r >= r0 && r < r1) T.i[fill[r]++] = c;
      }
  });
  return T;
}

SepID climb_common(SepID a, SepID b) {  // partition.cpp:63-86
  while (a.lvl < b.lvl) { a.lvl++; a.sep /= 2; }
  while (b.lvl < a.lvl) { b.lvl++; b.sep /= 2; }
  while (a.sep != b.sep) { a.lvl++; a.sep /= 2; b.lvl++; b.sep /= 2; }
  return a;
}
SepID lower_of(SepID a, SepID b) { return a.lvl < b.lvl ? a : b; }  // partition.cpp:88-100

// Row labels of a rectangular matrix: each row joins the column cluster whose
// entries in that row carry the largest sum of squares (tree.cpp:57-98).
void rows_by_weight(const CscMat& A, const std::vector<CID>& cpermed, const std::vector<int>& cperm,
                    std::vector<CID>& rlab) {
  CscMat rowsP = csc_transpose(csc_permute(A, nullptr, &cperm));  // column r = row r, entries by permuted column
  const CID last = cpermed[A.n - 1];
  for (int r = 0; r < A.m; ++r) {
    if (rlab[r] != CID()) continue;
    double bestw = -1;
    CID pick = rlab[r];
    int q = rowsP.p[r];
    const int e = rowsP.p[r + 1];
    while (q < e) {
      const CID g = cpermed[rowsP.i[q]];
      double w = 0;
      int t = q;
      while (t < e && cpermed[rowsP.i[t]] == g) { w += rowsP.x[t] * rowsP.x[t]; ++t; }
      if (w > bestw) { bestw = w; pick = g; }
      q = t;
    }
    rlab[r] = (pick == CID()) ? last : pick;
  }
}

}  // namespace

std::vector<CID> geometric_labels(const CscMat& A, int nlevels, const std::vector<double>& X, int dim) {
  const int n = A.n;
  const Pattern R = row_pattern(A);
  constexpr int grain = 4096;
  // recursive bisection of all columns (nlevels - 1 times): `ord` holds them
  // part after part, in column order
  std::vector<int> part(n, 0), ord(n), at{0, n};
  std::iota(ord.begin(), ord.end(), 0);
  for (int depth = 0; depth < nlevels - 1; ++depth) {
    const int nparts = 1 << depth;
    std::vector<int> next(2 * nparts + 1, n);
    parallel_for(nparts, 1, [&](int, int b, int e) {
      std::vector<double> vals;
      std::vector<int> back;
      for (int g = b; g < e; ++g) {
        next[2 * g] = at[g];
        next[2 * g + 1] = split_geo(ord, at[g], at[g + 1], X, dim, vals, back);
      }
    });
    at = std::move(next);
  }
  parallel_for((int)at.size() - 1, 16, [&](int, int b, int e) {
    for (int g = b; g < e; ++g)
      for (int q = at[g]; q < at[g + 1]; ++q) part[ord[q]] = g;
  });
  // separators: from the top level down, a still-unlabelled column in an even
  // subtree becomes a separator of level l when an unlabelled column of the
  // adjacent odd subtree is its neighbour in the graph of A^T A.  (Columns of
  // odd subtrees keep their state within a level, so the columns of one can be
  // looked at in any order.)
  std::vector<CID> lab(n);
  std::vector<int> slvl(n, -1);
  for (int depth = 0; depth < nlevels - 1; ++depth) {
    const int l = nlevels - depth - 1;
    parallel_for(n, grain, [&](int, int b, int e) {
      for (int v = b; v < e; ++v) {
        if (slvl[v] != -1) continue;
        const int pv = part[v] >> (l - 1);
        if (pv & 1) continue;
        bool sep = false;
        for (int q = A.p[v]; q < A.p[v + 1] && !sep; ++q) {
          const int row = A.i[q];
          for (int t = R.p[row]; t < R.p[row + 1]; ++t) {
            const int u = R.i[t];
            if ((part[u] >> (l - 1)) == pv + 1 && slvl[u] == -1) { sep = true; break; }
          }
        }
        if (sep) {
          slvl[v] = l;
          lab[v].self = SepID(l, pv / 2);
        }
      }
    });
  }
  parallel_for(n, grain, [&](int, int b, int e) {
    for (int v = b; v < e; ++v)
      if (slvl[v] == -1) {
        lab[v].self = SepID(0, part[v]);
        lab[v].l = lab[v].self;
        lab[v].r = lab[v].self;
      }
  });
  // row labels
  std::vector<CID> rlab(A.m);
  if (A.m != A.n) {
    std::vector<int> cperm(n);
    std::iota(cperm.begin(), cperm.end(), 0);
    std::stable_sort(cperm.begin(), cperm.end(), [&](int a, int b) { return lab[a] < lab[b]; });
    std::vector<CID> cpermed(n);
    for (int c = 0; c < n; ++c) cpermed[c] = lab[cperm[c]];
    rows_by_weight(A, cpermed, cperm, rlab);
  } else {
    rlab = lab;
  }
  // interfaces (partition.cpp:506-578): pass 1 from lower-level neighbours
  parallel_for(A.m, grain, [&](int, int b, int e) {
    for (int r = b; r < e; ++r) {
      const SepID self = rlab[r].self;
      if (self.lvl <= 0) continue;
      SepID left, right;
      for (int t = R.p[r]; t < R.p[r + 1]; ++t) {
        const SepID nb = lab[R.i[t]].self;
        if (nb.lvl >= self.lvl) continue;
        const int side = nb.sep >> (self.lvl - nb.lvl - 1);
        if (side % 2 == 0) left = (left.lvl == -1) ? nb : lower_of(nb, left);
        else right = (right.lvl == -1) ? nb : lower_of(nb, right);
      }
      rlab[r].l = left;
      rlab[r].r = right;
    }
  });
  std::vector<CID> clab = rlab;  // row i matched to column i
  // pass 2: a missing side is borrowed from same-separator neighbours
  parallel_for(A.m, grain, [&](int, int b, int e) {
    for (int r = b; r < e; ++r) {
      const SepID self = rlab[r].self;
      SepID left = rlab[r].l, right = rlab[r].r;
      if (right == SepID()) {
        for (int t = R.p[r]; t < R.p[r + 1]; ++t) {
          const CID& c = clab[R.i[t]];
          if (c.self == self && c.r != SepID()) right = (right == SepID()) ? c.r : climb_common(right, c.r);
        }
      } else if (left == SepID()) {
        for (int t = R.p[r]; t < R.p[r + 1]; ++t) {
          const CID& c = clab[R.i[t]];
          if (c.self == self && c.l != SepID()) left = (left == SepID()) ? c.l : climb_common(left, c.l);
        }
      }
      rlab[r].l = left;
      rlab[r].r = right;
    }
  });
  for (auto& c : rlab) {
    if (c.l == SepID()) c.l = c.self;
    if (c.r == SepID()) c.r = c.self;
  }
  return rlab;
}

// Columns by their labels: the order that stable sorts by the label and then by
// its merged form at each level leave, so the last level's form counts first.
// There are far fewer labels than columns: those are sorted, and the columns
// counted into their places.
void order_columns(int nlevels, const std::vector<CID>& labels, std::vector<int>& cperm) {
  const int n = (int)cperm.size();
  auto mix = [](const CID& c) {
    size_t h = 1469598103934665603ull;
    for (int v : {c.self.lvl, c.self.sep, c.l.lvl, c.l.sep, c.r.lvl, c.r.sep, c.part, c.section})
      h = (h ^ (size_t)(unsigned)v) * 1099511628211ull;
    return h ^ (h >> 29);
  };
  // distinct labels, in order of appearance
  std::vector<CID> key;
  std::vector<int> id(labels.size()), table(1024, -1);
  std::vector<size_t> hash;
  for (size_t v = 0; v < labels.size(); ++v) {
    if (v > 0 && labels[v] == labels[v - 1]) { id[v] = id[v - 1]; continue; }
    const size_t h = mix(labels[v]);
    size_t q = h & (table.size() - 1);
    while (table[q] >= 0 && !(hash[table[q]] == h && key[table[q]] == labels[v])) q = (q + 1) & (table.size() - 1);
    if (table[q] < 0) {
      table[q] = (int)key.size();
      key.push_back(labels[v]);
      hash.push_back(h);
      if (2 * key.size() > table.size()) {
        table.assign(2 * table.size(), -1);
        for (size_t d = 0; d < key.size(); ++d) {
          size_t t = hash[d] & (table.size() - 1);
          while (table[t] >= 0) t = (t + 1) & (table.size() - 1);
          table[t] = (int)d;
        }
        id[v] = (int)key.size() - 1;
        continue;
      }
    }
    id[v] = table[q];
  }
  const int nd = (int)key.size();
  std::vector<int> order(nd);
  std::iota(order.begin(), order.end(), 0);
  auto by_key = [&key](int a, int b) { return key[a] < key[b]; };
  std::sort(order.begin(), order.end(), by_key);
  for (int lvl = 1; lvl < nlevels; ++lvl) {
    parallel_for(nd, 1024, [&](int, int b, int e) {
      for (int d = b; d < e; ++d) key[d] = cid_merge_if(key[d], lvl);
    });
    if (!std::is_sorted(order.begin(), order.end(), by_key)) std::stable_sort(order.begin(), order.end(), by_key);
  }
  // cperm's columns by rank, in cperm's order
  std::vector<int> rank(nd), at(nd + 1, 0), out(n);
  for (int q = 0; q < nd; ++q) rank[order[q]] = q;
  for (int c : cperm) at[rank[id[c]] + 1]++;
  std::partial_sum(at.begin(), at.end(), at.begin());
  for (int c : cperm) out[at[rank[id[c]]]++] = c;
  cperm = std::move(out);
}

void order_rows_ls(const CscMat& Ap, const std::vector<CID>& cpermed, std::vector<int>& rperm,
                   std::vector<int>& rows_per_col) {
  const int m = Ap.m, n = Ap.n;
  const CscMat R = csc_transpose(Ap);
  std::vector<std::vector<int>> owned(n);
  rows_per_col.assign(n, 0);
  for (int r = 0; r < m; ++r) {
    double bestw = -1;
    int pick = -1;
    int q = R.p[r];
    const int e = R.p[r + 1];
    while (q < e) {
      const CID& g = cpermed[R.i[q]];
      double w = 0;
      int t = q;
      while (t < e && cpermed[R.i[t]] == g) { w += R.x[t] * R.x[t]; ++t; }
      if (w > bestw) { bestw = w; pick = R.i[q]; }
      q = t;
    }
    if (pick == -1) pick = n - 1;
    rows_per_col[pick]++;
    owned[pick].push_back(r);
  }
  rperm.clear();
  rperm.reserve(m);
  for (int c = 0; c < n; ++c)
    for (int r : owned[c]) rperm.push_back(r);
}

}  // namespace spq
