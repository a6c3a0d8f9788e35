#include "gdtp_ldlt.h"

#include <algorithm>
#include <array>
#include <cmath>
#include <functional>
#include <limits>

namespace gdtp {

// Recursive bisection at the middle breadth-first level from a pseudo-peripheral vertex; the
// separator is the part of that level adjacent to the next level, ordered last.
void NestedDissectionOrder(const Csr& A, std::vector<int>& perm) {
  const int n = A.rows;
  perm.clear();
  perm.reserve(n);
  std::vector<int> stamp(n, -1), level(n, -1), inSet(n, -1);
  int setId = 0, bfsId = 0;
  std::vector<int> queue;
  queue.reserve(n);
  auto bfs = [&](int src, int sid) {  // levels within set `sid`; returns vertices in BFS order
    queue.clear();
    int id = bfsId++;
    stamp[src] = id, level[src] = 0;
    queue.push_back(src);
    for (size_t h = 0; h < queue.size(); h++) {
      int v = queue[h];
      for (int k = A.rowptr[v]; k < A.rowptr[v + 1]; k++) {
        int u = A.col[k];
        if (u == v || inSet[u] != sid || stamp[u] == id) continue;
        stamp[u] = id, level[u] = level[v] + 1;
        queue.push_back(u);
      }
    }
  };
  // explicit work stack of vertex sets; a set is split into (A, B, S) and S is emitted after A and B.
  struct Item { std::vector<int> verts; bool emit; };
  std::vector<Item> stack;
  stack.push_back({std::vector<int>(n), false});
  for (int i = 0; i < n; i++) stack.back().verts[i] = i;
  const size_t kLeaf = 48;
  while (!stack.empty()) {
    Item it = std::move(stack.back());
    stack.pop_back();
    if (it.emit || it.verts.size() <= kLeaf) {
      perm.insert(perm.end(), it.verts.begin(), it.verts.end());
      continue;
    }
    int sid = setId++;
    for (int v : it.verts) inSet[v] = sid;
    bfs(it.verts[0], sid);
    if (queue.size() < it.verts.size()) {  // disconnected: split off this component
      std::vector<int> comp(queue.begin(), queue.end()), rest;
      int id = bfsId - 1;
      for (int v : it.verts)
        if (stamp[v] != id) rest.push_back(v);
      stack.push_back({std::move(rest), false});
      stack.push_back({std::move(comp), false});
      continue;
    }
    int far = queue.back();
    bfs(far, sid);
    far = queue.back();
    bfs(far, sid);
    int maxLevel = level[queue.back()];
    if (maxLevel < 2) {
      perm.insert(perm.end(), it.verts.begin(), it.verts.end());
      continue;
    }
    std::vector<int> cnt(maxLevel + 2, 0);
    for (int v : queue) cnt[level[v]]++;
    int half = (int)queue.size() / 2, acc = 0, mid = 1;
    for (int l = 0; l <= maxLevel; l++) {
      acc += cnt[l];
      if (acc >= half) { mid = std::max(1, std::min(l, maxLevel - 1)); break; }
    }
    std::vector<int> a, b, s;
    for (int v : queue) {
      int l = level[v];
      if (l < mid) a.push_back(v);
      else if (l > mid) b.push_back(v);
      else {
        bool touchesNext = false;
        for (int k = A.rowptr[v]; k < A.rowptr[v + 1]; k++) {
          int u = A.col[k];
          if (inSet[u] == sid && level[u] == mid + 1) { touchesNext = true; break; }
        }
        (touchesNext ? s : a).push_back(v);
      }
    }
    stack.push_back({std::move(s), true});
    stack.push_back({std::move(b), false});
    stack.push_back({std::move(a), false});
  }
}

int FactorLdlt(const Csr& A, Ldlt& F, std::string& err) {
  const int n = A.rows;
  F.n = n;
  NestedDissectionOrder(A, F.perm);
  F.iperm.assign(n, 0);
  for (int i = 0; i < n; i++) F.iperm[F.perm[i]] = i;
  // lower triangle of the permuted matrix by rows: C[k][i] (i <= k)
  std::vector<Triplet> t;
  t.reserve(A.col.size() / 2 + n);
  for (int r = 0; r < n; r++)
    for (int k = A.rowptr[r]; k < A.rowptr[r + 1]; k++) {
      int pr = F.iperm[r], pc = F.iperm[A.col[k]];
      if (pc <= pr) t.push_back({pr, pc, A.val[k]});
    }
  Csr C = Csr::FromTriplets(n, n, t);
  // symbolic: elimination tree and column counts
  std::vector<int> parent(n, -1), flag(n, -1), lnz(n, 0);
  for (int k = 0; k < n; k++) {
    flag[k] = k;
    for (int p = C.rowptr[k]; p < C.rowptr[k + 1]; p++)
      for (int i = C.col[p]; i < k && flag[i] != k; i = parent[i]) {
        if (parent[i] == -1) parent[i] = k;
        lnz[i]++;
        flag[i] = k;
      }
  }
  std::vector<int64_t> Lp(n + 1, 0);
  for (int k = 0; k < n; k++) Lp[k + 1] = Lp[k] + lnz[k];
  if (Lp[n] > (int64_t)2000000000) { err = "LDL^T factor too large"; return 0; }
  std::vector<int> Li(Lp[n]);
  std::vector<double> Lx(Lp[n]);
  std::vector<double> y(n, 0.0);
  std::vector<int> pattern(n), fill(n, 0);
  F.D.assign(n, 0.0);
  std::fill(flag.begin(), flag.end(), -1);
  // numeric: up-looking, row k of L by a sparse triangular solve over the etree reach
  for (int k = 0; k < n; k++) {
    int top = n;
    flag[k] = k;
    for (int p = C.rowptr[k]; p < C.rowptr[k + 1]; p++) {
      int i = C.col[p];
      y[i] += C.val[p];
      int len = 0;
      for (; flag[i] != k; i = parent[i]) pattern[len++] = i, flag[i] = k;
      while (len > 0) pattern[--top] = pattern[--len];
    }
    double d = y[k];
    y[k] = 0.0;
    for (; top < n; top++) {
      int i = pattern[top];
      double yi = y[i];
      y[i] = 0.0;
      int64_t p2 = Lp[i] + fill[i];
      for (int64_t p = Lp[i]; p < p2; p++) y[Li[p]] -= Lx[p] * yi;
      double lki = yi / F.D[i];
      d -= lki * yi;
      Li[p2] = k, Lx[p2] = lki;
      fill[i]++;
    }
    if (!(d > 0.0) || !std::isfinite(d)) { err = "matrix is not positive definite (LDL^T pivot " + std::to_string(d) + ")"; return 0; }
    F.D[k] = d;
  }
  // L by columns and by rows
  Csr& Lc = F.Lcols;
  Lc.rows = n, Lc.cols = n;
  Lc.rowptr.assign(n + 1, 0);
  for (int k = 0; k < n; k++) Lc.rowptr[k + 1] = (int)Lp[k + 1];
  Lc.col = Li, Lc.val = Lx;
  F.Lrows = Lc.Transpose();
  return 1;
}

void BuildLdltStages(const Ldlt& F, LdltStages& S, int topRows) {
  const int n = F.n;
  S = LdltStages();
  S.n = n;
  if (n == 0) return;
  // elimination tree (a column's first entry below the diagonal) and subtree sizes
  std::vector<int> parent(n, -1), size(n, 1);
  for (int i = 0; i < n; i++) {
    int p = n;
    for (int k = F.Lcols.rowptr[i]; k < F.Lcols.rowptr[i + 1]; k++) p = std::min(p, F.Lcols.col[k]);
    if (p < n) parent[i] = p;
  }
  for (int i = 0; i < n; i++)
    if (parent[i] >= 0) size[parent[i]] += size[i];
  // stage limits: rows whose subtree exceeds the last limit form the top
  std::vector<int> limit;
  if (n > std::min(topRows, kLdltDenseRows))
    for (long s = kLdltLeafRows, last = n;; s *= kLdltStageGrowth) {
      long above = 0;
      for (int i = 0; i < n; i++) above += size[i] > s;
      // no row left for the top: what the last stage left is the top unless that is far too many
      if (above == 0 && !limit.empty() && last <= 2 * (long)topRows) break;
      limit.push_back((int)std::min<long>(s, n));
      if (above <= topRows) break;
      last = above;
    }
  const int nStages = (int)limit.size() + 1;
  std::vector<int> stage(n), comp(n), compStage;
  for (int i = 0; i < n; i++) stage[i] = (int)(std::lower_bound(limit.begin(), limit.end(), size[i]) - limit.begin());
  // components: a row joins its parent's when both are of one stage; the top is one component
  for (int i = n - 1, top = -1; i >= 0; i--) {
    if (stage[i] == nStages - 1 && top >= 0) comp[i] = top;
    else if (stage[i] < nStages - 1 && parent[i] >= 0 && stage[parent[i]] == stage[i]) comp[i] = comp[parent[i]];
    else {
      comp[i] = (int)compStage.size();
      compStage.push_back(stage[i]);
      if (stage[i] == nStages - 1) top = comp[i];
    }
  }
  // new numbering: components by stage, rows of a component in elimination order
  const int nComp = (int)compStage.size();
  std::vector<int> order(nComp), rank(nComp), count(nComp, 0);
  for (int c = 0; c < nComp; c++) order[c] = c;
  std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return compStage[a] < compStage[b]; });
  for (int c = 0; c < nComp; c++) rank[order[c]] = c;
  for (int i = 0; i < n; i++) count[rank[comp[i]]]++;
  S.compPtr.assign(nComp + 1, 0);
  for (int c = 0; c < nComp; c++) S.compPtr[c + 1] = S.compPtr[c] + count[c];
  std::vector<int> next(S.compPtr.begin(), S.compPtr.end() - 1), rowOf(n), at(n);
  for (int i = 0; i < n; i++) {
    at[i] = next[rank[comp[i]]]++;
    rowOf[at[i]] = i;
  }
  S.stages.assign(nStages, LdltStage());
  for (int c = 0, s = 0; s < nStages; s++) {
    LdltStage& T = S.stages[s];
    T.compBegin = c;
    while (c < nComp && compStage[order[c]] == s) T.wide = T.wide || count[c] > kLdltNarrowRows, c++;
    T.compEnd = c;
    T.rowBegin = S.compPtr[T.compBegin], T.rowEnd = S.compPtr[T.compEnd];
    // the top, and every stage after a wide one
    T.wide = T.wide || s == nStages - 1 || (s > 0 && S.stages[s - 1].wide);
  }
  S.wideBegin = n;
  for (int s = nStages - 1; s >= 0 && S.stages[s].wide; s--) S.wideBegin = S.stages[s].rowBegin;
  S.perm.resize(n), S.dinv.resize(n);
  for (int w = 0; w < n; w++) S.perm[w] = F.perm[rowOf[w]], S.dinv[w] = 1.0 / F.D[rowOf[w]];
  auto couplings = [&](const Csr& L, std::vector<int>& ptr, std::vector<int>& col, std::vector<double>& val) {
    ptr.assign(n + 1, 0);
#pragma omp parallel for schedule(static)
    for (int w = 0; w < n; w++) {
      const int i = rowOf[w];
      for (int k = L.rowptr[i]; k < L.rowptr[i + 1]; k++) ptr[w + 1] += comp[L.col[k]] != comp[i];
    }
    for (int w = 0; w < n; w++) ptr[w + 1] += ptr[w];
    col.resize(ptr[n]), val.resize(ptr[n]);
#pragma omp parallel for schedule(static)
    for (int w = 0; w < n; w++) {
      const int i = rowOf[w];
      int p = ptr[w];
      for (int k = L.rowptr[i]; k < L.rowptr[i + 1]; k++)
        if (comp[L.col[k]] != comp[i]) col[p] = at[L.col[k]], val[p] = L.val[k], p++;
    }
  };
  couplings(F.Lrows, S.fwdPtr, S.fwdCol, S.fwdVal);
  couplings(F.Lcols, S.bwdPtr, S.bwdCol, S.bwdVal);
  // inverses of the components' unit-lower blocks
  S.fwdMatPtr.assign(nComp + 1, 0), S.bwdMatPtr.assign(nComp + 1, 0);
  std::vector<char> wide(nComp, 0);
  for (const LdltStage& T : S.stages)
    for (int c = T.compBegin; c < T.compEnd; c++) wide[c] = T.wide;
  for (int c = 0; c < nComp; c++) {
    const int m = count[c];
    long f = 0, b = 0;
    if (wide[c]) f = b = (long)m * LdltWideStride(m);
    else
      for (int r0 = 0; r0 < m; r0 += kLdltBlock) {
        const int nr = std::min(kLdltBlock, m - r0);
        f += (long)nr * (r0 + nr), b += (long)nr * (m - r0);
      }
    S.fwdMatPtr[c + 1] = S.fwdMatPtr[c] + f, S.bwdMatPtr[c + 1] = S.bwdMatPtr[c] + b;
  }
  S.fwdMat.Allocate(S.fwdMatPtr[nComp]), S.bwdMat.Allocate(S.bwdMatPtr[nComp]);
  S.fwdLow.Allocate(S.fwdMat.size()), S.bwdLow.Allocate(S.bwdMat.size());
  static_assert(std::numeric_limits<long double>::digits >= 64, "the inverses' low parts come from 64-bit significands");
  auto split = [](long double v, double& high, float& low) { high = (double)v, low = (float)(v - high); };
  // a component's block of L by rows without its unit diagonal, and each row's parent in it (or -1)
  struct Block {
    std::vector<int> ptr, col, up;
    std::vector<double> val;
  };
  auto load = [&](int c, Block& L) {
    const int w0 = S.compPtr[c];
    L.ptr.assign(1, 0), L.col.clear(), L.up.clear(), L.val.clear();
    for (int a = 0; a < count[c]; a++) {
      const int i = rowOf[w0 + a];
      for (int k = F.Lrows.rowptr[i]; k < F.Lrows.rowptr[i + 1]; k++)
        if (comp[F.Lrows.col[k]] == comp[i]) L.col.push_back(at[F.Lrows.col[k]] - w0), L.val.push_back(F.Lrows.val[k]);
      L.ptr.push_back((int)L.col.size());
      L.up.push_back(parent[i] >= 0 && comp[parent[i]] == comp[i] ? at[parent[i]] - w0 : -1);
    }
  };
  // Columns j0 .. j1 - 1 (at most kColumns, each the next one's child) of the block's inverse by forward
  // substitution from the unit vectors: z[a][j - j0] for row a.  A column's rows are its ancestors; z is zero
  // before and elsewhere.
  constexpr int kColumns = 4;
  using Row = std::array<long double, kColumns>;
  auto group = [](const Block& L, int m, int j0) {
    int j1 = j0 + 1;
    while (j1 < m && j1 < j0 + kColumns && L.up[j1 - 1] == j1) j1++;
    return j1;
  };
  auto columns = [](const Block& L, int j0, int j1, std::vector<Row>& z) {
    for (int a = j0; a >= 0; a = L.up[a]) {
      Row v{};
      if (a < j1) v[a - j0] = 1.0L;
      const int end = L.ptr[a + 1];  // entries in columns before j0 meet zeros
      for (int p = (int)(std::lower_bound(L.col.begin() + L.ptr[a], L.col.begin() + end, j0) - L.col.begin()); p < end; p++) {
        const Row& x = z[L.col[p]];
        for (int q = 0; q < kColumns; q++) v[q] -= L.val[p] * x[q];
      }
      z[a] = v;
    }
  };
  const int nNarrow = (int)(std::find(wide.begin(), wide.end(), 1) - wide.begin());
#pragma omp parallel for schedule(dynamic, 8)
  for (int c = 0; c < nNarrow; c++) {
    const int m = count[c];
    Block L;
    std::vector<double> high((size_t)m * m, 0.0);
    std::vector<float> low((size_t)m * m, 0.0f);
    std::vector<Row> z(m, Row{});
    load(c, L);
    for (int j0 = 0, j1; j0 < m; j0 = j1) {  // high, low: the inverse by columns
      j1 = group(L, m, j0);
      columns(L, j0, j1, z);
      for (int a = j0; a >= 0; a = L.up[a]) {
        for (int j = j0; j < j1; j++) split(z[a][j - j0], high[(size_t)j * m + a], low[(size_t)j * m + a]);
        z[a] = Row{};
      }
    }
    double *f = S.fwdMat.data() + S.fwdMatPtr[c], *b = S.bwdMat.data() + S.bwdMatPtr[c];
    float *fl = S.fwdLow.data() + S.fwdMatPtr[c], *bl = S.bwdLow.data() + S.bwdMatPtr[c];
    for (int r0 = 0; r0 < m; r0 += kLdltBlock) {
      const int nr = std::min(kLdltBlock, m - r0);
      for (int j = 0; j < r0 + nr; j++)
        for (int r = 0; r < nr; r++) *f++ = high[(size_t)j * m + r0 + r], *fl++ = low[(size_t)j * m + r0 + r];
      for (int j = r0; j < m; j++)
        for (int r = 0; r < nr; r++) *b++ = high[(size_t)(r0 + r) * m + j], *bl++ = low[(size_t)(r0 + r) * m + j];
    }
  }
  for (int c = nNarrow; c < nComp; c++) {  // few and large: in parallel over the columns
    const int m = count[c];
    const size_t stride = LdltWideStride(m);
    Block L;
    load(c, L);
    double *f = S.fwdMat.data() + S.fwdMatPtr[c], *b = S.bwdMat.data() + S.bwdMatPtr[c];
    float *fl = S.fwdLow.data() + S.fwdMatPtr[c], *bl = S.bwdLow.data() + S.bwdMatPtr[c];
    std::vector<int> start;  // first column of each group
    for (int j = 0; j < m; j = group(L, m, j)) start.push_back(j);
    start.push_back(m);
#pragma omp parallel
    {
      std::vector<Row> z(m, Row{});
#pragma omp for schedule(dynamic, 4)
      for (int g = 0; g < (int)start.size() - 1; g++) {  // a column is a row of the transposed inverse
        columns(L, start[g], start[g + 1], z);
        std::fill(b + start[g] * stride, b + start[g + 1] * stride, 0.0), std::fill(bl + start[g] * stride, bl + start[g + 1] * stride, 0.0f);
        for (int a = start[g]; a >= 0; a = L.up[a]) {
          for (int j = start[g]; j < start[g + 1]; j++) split(z[a][j - start[g]], b[j * stride + a], bl[j * stride + a]);
          z[a] = Row{};
        }
      }
#pragma omp for schedule(static)
      for (int r = 0; r < m; r++) {
        for (int j = 0; j <= r; j++) f[r * stride + j] = b[j * stride + r], fl[r * stride + j] = bl[j * stride + r];
        std::fill(f + r * stride + r + 1, f + (r + 1) * stride, 0.0), std::fill(fl + r * stride + r + 1, fl + (r + 1) * stride, 0.0f);
      }
    }
  }
}

void SolveLdlt(const Ldlt& F, const double* b, double* x, int ncols, int ld) {
  const int n = F.n;
  std::vector<double> y(n);
  for (int c = 0; c < ncols; c++) {
    for (int k = 0; k < n; k++) {
      double s = b[(size_t)c * ld + F.perm[k]];
      for (int p = F.Lrows.rowptr[k]; p < F.Lrows.rowptr[k + 1]; p++) s -= F.Lrows.val[p] * y[F.Lrows.col[p]];
      y[k] = s;
    }
    for (int k = 0; k < n; k++) y[k] /= F.D[k];
    for (int i = n - 1; i >= 0; i--) {
      double s = y[i];
      for (int p = F.Lcols.rowptr[i]; p < F.Lcols.rowptr[i + 1]; p++) s -= F.Lcols.val[p] * y[F.Lcols.col[p]];
      y[i] = s;
    }
    for (int k = 0; k < n; k++) x[(size_t)c * ld + F.perm[k]] = y[k];
  }
}

}  // namespace gdtp
