// Sparse LDL^T factorisation (host) of symmetric positive-definite matrices, with a
// nested-dissection ordering so that the triangular solves have shallow dependency levels.
//
// Replaces the reference's exact boundary and coarse solvers, Eigen SimplicialLDLT
// (include/Src/Solver.h:145-259).  Factorisation: up-looking LDL^T (T. A. Davis, "Algorithm 849:
// a concise sparse Cholesky factorization package", ACM TOMS 31(4), 2005).  Ordering: recursive
// breadth-first-level bisection (A. George, "Nested dissection of a regular finite element mesh",
// SIAM J. Numer. Anal. 10, 1973).
#pragma once
#include <memory>
#include <string>

#include "gdtp_sparse.h"

namespace gdtp {

struct Ldlt {
  int n = 0;
  std::vector<int> perm;      // new index -> old index
  std::vector<int> iperm;     // old index -> new index
  Csr Lrows;                  // strictly lower triangular L by rows (row k: entries l_ki, i < k), permuted space
  Csr Lcols;                  // the same entries by columns (row of L^T)
  std::vector<double> D;      // diagonal
};

// The triangular solves of an LDL^T factor as a few passes whose rows are all independent, for the
// GPU (partitioned inverses: F. L. Alvarado and R. Schreiber, "Optimal parallel solution of sparse
// triangular systems", SIAM J. Sci. Comput. 14, 1993).  The elimination tree is cut by subtree size
// into stages; a stage's connected pieces ("components") do not couple with each other, so a stage is
// one gather of couplings with the stages already solved and one product with each component's
// explicit inverse of its unit-lower block.  The last stage (the top of the tree) is one component.
// Rows are renumbered by (stage, component, row): a component is a contiguous range.
constexpr int kLdltLeafRows = 128;     // largest subtree of the first stage
constexpr int kLdltStageGrowth = 8;    // each further stage takes subtrees this many times larger
constexpr int kLdltTopRows = 2048;     // stages are added until the top has at most this many rows
// Matrices up to this size are the top alone.  (At 2048 a system of 1536 and 768 boundary rows, a 128^2 cube,
// took 13 ms to create or to update instead of 7, for dense inverses of 70 MB; its V-cycle 296 us against 292.)
constexpr int kLdltDenseRows = 512;
constexpr int kLdltNarrowRows = 256;   // components up to this size are solved by one workgroup
constexpr int kLdltBlock = 64;         // rows per block of a narrow component's inverse

struct LdltStage {
  int rowBegin = 0, rowEnd = 0;        // rows (new numbering)
  int compBegin = 0, compEnd = 0;      // components
  bool wide = false;                   // some component has more than kLdltNarrowRows rows (or the top)
};

constexpr int LdltWideStride(int rows) { return (rows + 1) / 2 * 2; }  // even: rows are read in pairs

// Values that the threads filling them touch first (a vector's one thread would clear them before).
template <class T>
struct LdltArray {
  std::unique_ptr<T[]> values;
  size_t count = 0;
  void Allocate(size_t n) { values.reset(new T[n]), count = n; }
  T* data() { return values.get(); }
  const T* data() const { return values.get(); }
  size_t size() const { return count; }
};

struct LdltStages {
  int n = 0;
  std::vector<LdltStage> stages;       // in forward order; the last is the top
  std::vector<int> perm;               // new row -> row of the original matrix
  std::vector<double> dinv;            // 1 / D
  std::vector<int> compPtr;            // first row of each component (one more than components)
  // couplings with other stages: of a row of L with the earlier stages, of a row of L^T with the later
  std::vector<int> fwdPtr, fwdCol, bwdPtr, bwdCol;
  std::vector<double> fwdVal, bwdVal;
  // Inverses, a rounded part and what the rounding left (Low; single precision is enough for it): a product
  // with the rounded inverse alone, summed in double, is not backward stable, and where L's block is badly
  // conditioned (texels with a support of 1e-12 of the others) its error was up to 21 times that of
  // substitution.  With both parts and a compensated sum it is no larger.
  // Narrow component: for each block of kLdltBlock rows the columns its rows can reach (forward: columns
  // before the block's end; backward: from its begin), column-major, the block's rows contiguous.  Wide
  // component: the whole matrix row-major (backward: transposed), rows of LdltWideStride values.
  std::vector<long> fwdMatPtr, bwdMatPtr;  // per component
  LdltArray<double> fwdMat, bwdMat;
  LdltArray<float> fwdLow, bwdLow;
  int wideBegin = 0;                   // first row of the first wide stage (the later stages are all wide)
};

void NestedDissectionOrder(const Csr& A, std::vector<int>& perm);
int FactorLdlt(const Csr& A, Ldlt& F, std::string& err);
// The staged form of F's triangular solves; topRows: the largest top (kLdltTopRows, smaller in tests).
void BuildLdltStages(const Ldlt& F, LdltStages& S, int topRows = kLdltTopRows);
// Solve A x = b for ncols column-major vectors (host reference path).
void SolveLdlt(const Ldlt& F, const double* b, double* x, int ncols, int ld);

}  // namespace gdtp
