// The staged triangular solves evaluated on the host as the GPU kernels do, against substitution.
// Usage: ldlt_stages MATRIX TOP_ROWS, MATRIX a file of rows, entries (int64), rowptr, columns (int32), values.
// Prints one line per stage (rows, components, rows of the largest component, wide) and a line of errors of the
// staged solve and of substitution against a solution refined in extended precision.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <string>

#include "gdtp_ldlt.h"

using namespace gdtp;

struct Sum2 {
  double v = 0.0, e = 0.0;
  void AddProduct(double high, float low, double x) {
    const double p = high * x, t = v + p, z = t - v;
    e += std::fma(high, x, -p);
    e = std::fma((double)low, x, e);
    e += (v - (t - z)) + (p - z);
    v = t;
  }
};

static std::vector<double> Staged(const LdltStages& S, const std::vector<double>& b) {
  std::vector<double> y(S.n), x(S.n);
  auto component = [&](int c, bool forward, bool wide) {
    const int w0 = S.compPtr[c], m = S.compPtr[c + 1] - w0;
    const auto &ptr = forward ? S.fwdPtr : S.bwdPtr, &col = forward ? S.fwdCol : S.bwdCol;
    const auto& val = forward ? S.fwdVal : S.bwdVal;
    std::vector<double> r(m);
    for (int i = 0; i < m; i++) {
      double s = 0.0;
      for (int p = ptr[w0 + i]; p < ptr[w0 + i + 1]; p++) s += val[p] * y[col[p]];
      r[i] = (forward ? b[S.perm[w0 + i]] : y[w0 + i] * S.dinv[w0 + i]) - s;
    }
    const size_t at = forward ? S.fwdMatPtr[c] : S.bwdMatPtr[c];
    const double* high = (forward ? S.fwdMat : S.bwdMat).data() + at;
    const float* low = (forward ? S.fwdLow : S.bwdLow).data() + at;
    std::vector<Sum2> sum(m);
    if (wide) {
      const size_t stride = LdltWideStride(m);
      for (int i = 0; i < m; i++)
        for (int j = forward ? 0 : i; j < (forward ? i + 1 : m); j++) sum[i].AddProduct(high[i * stride + j], low[i * stride + j], r[j]);
    } else {
      for (int r0 = 0; r0 < m; r0 += kLdltBlock) {
        const int nr = std::min(kLdltBlock, m - r0);
        for (int j = forward ? 0 : r0; j < (forward ? r0 + nr : m); j++)
          for (int i = 0; i < nr; i++) sum[r0 + i].AddProduct(*high++, *low++, r[j]);
      }
    }
    for (int i = 0; i < m; i++) y[w0 + i] = sum[i].v + sum[i].e;
  };
  for (const LdltStage& T : S.stages)
    for (int c = T.compBegin; c < T.compEnd; c++) component(c, true, T.wide);
  for (int k = (int)S.stages.size() - 1; k >= 0; k--)
    for (int c = S.stages[k].compBegin; c < S.stages[k].compEnd; c++) component(c, false, S.stages[k].wide);
  for (int w = 0; w < S.n; w++) x[S.perm[w]] = y[w];
  return x;
}

int main(int argc, char** argv) {
  if (argc != 3) return 2;
  Csr A;
  int64_t head[2];
  FILE* f = std::fopen(argv[1], "rb");
  bool ok = f && std::fread(head, sizeof head, 1, f) == 1;
  if (ok) {
    A.rows = A.cols = (int)head[0];
    A.rowptr.resize(head[0] + 1), A.col.resize(head[1]), A.val.resize(head[1]);
    ok = std::fread(A.rowptr.data(), 4, A.rowptr.size(), f) == A.rowptr.size() && std::fread(A.col.data(), 4, A.col.size(), f) == A.col.size() &&
         std::fread(A.val.data(), 8, A.val.size(), f) == A.val.size();
  }
  if (f) std::fclose(f);
  Ldlt F;
  std::string err = "cannot read the matrix";
  if (!ok || !FactorLdlt(A, F, err)) return std::fprintf(stderr, "%s\n", err.c_str()), 1;
  LdltStages S;
  BuildLdltStages(F, S, std::atoi(argv[2]));
  const int n = A.rows, columns = 4;
  std::vector<int> seen(n, 0);
  for (int p : S.perm) seen[p]++;
  if (std::count(seen.begin(), seen.end(), 1) != n) return std::fprintf(stderr, "not a permutation\n"), 1;
  for (const LdltStage& T : S.stages) {
    int largest = 0;
    for (int c = T.compBegin; c < T.compEnd; c++) largest = std::max(largest, S.compPtr[c + 1] - S.compPtr[c]);
    std::printf("stage %d %d %d %d\n", T.rowEnd - T.rowBegin, T.compEnd - T.compBegin, largest, (int)T.wide);
  }
  // b - A x (less what b's own rounding leaves) and A x in extended precision
  auto product = [&](int i, auto&& x) {
    long double s = 0.0L;
    for (int k = A.rowptr[i]; k < A.rowptr[i + 1]; k++) s += (long double)A.val[k] * x(A.col[k]);
    return s;
  };
  double log[2][2] = {};  // staged, substitution; residual, error in A's norm
  for (int t = 0; t < columns; t++) {
    std::mt19937_64 gen(t + 1);
    std::uniform_real_distribution<double> uniform(0.0, 1.0);
    std::vector<double> u(n), b(n), d(n), e(n);
    for (double& v : u) v = uniform(gen);
    for (int i = 0; i < n; i++) b[i] = (double)product(i, [&](int j) { return (long double)u[j]; });
    std::vector<long double> want(n, 0.0L);
    for (int step = 0; step < 3; step++) {
      for (int i = 0; i < n; i++) d[i] = (double)(b[i] - product(i, [&](int j) { return want[j]; }));
      SolveLdlt(F, d.data(), e.data(), 1, n);
      for (int i = 0; i < n; i++) want[i] += e[i];
    }
    for (int which = 0; which < 2; which++) {
      std::vector<double> x(n);
      if (which == 0) x = Staged(S, b);
      else SolveLdlt(F, b.data(), x.data(), 1, n);
      long double residual = 0.0L, error = 0.0L;
      for (int i = 0; i < n; i++) {
        const long double r = b[i] - product(i, [&](int j) { return (long double)x[j]; });
        residual += r * r;
        error += (x[i] - want[i]) * product(i, [&](int j) { return (long double)x[j] - want[j]; });
      }
      log[which][0] += std::log(std::max((double)std::sqrt(residual), 1e-300)) / columns, log[which][1] += std::log(std::max((double)std::sqrt(error), 1e-300)) / columns;
    }
  }
  std::printf("ratio %.6g %.6g\n", std::exp(log[0][0] - log[1][0]), std::exp(log[0][1] - log[1][1]));
  return 0;
}
