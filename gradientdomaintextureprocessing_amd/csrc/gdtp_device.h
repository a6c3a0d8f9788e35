// Device-resident multigrid system and the HIP V-cycle (internal interface of libgdtp).
#pragma once
#include <hip/hip_runtime.h>

#include <string>
#include <vector>

#include "gdtp_galerkin.h"
#include "gdtp_vectorfield.h"

namespace gdtp {

#define GDTP_HIP(call)                                                                 \
  do {                                                                                 \
    hipError_t e_ = (call);                                                            \
    if (e_ != hipSuccess) throw std::runtime_error(std::string(#call) + ": " + hipGetErrorString(e_)); \
  } while (0)

// A row of a wide stage: its component's first row and size, and where its rows of the two inverses begin.
struct LdltWideRow {
  int begin, rows;
  long mat[2];  // forward, backward
};

// Exact triangular solves of an LDL^T factor on the device: the staged form (LdltStages).
struct DevLdlt {
  int n = 0, wideBegin = 0;
  std::vector<LdltStage> stages;
  int* perm = nullptr;
  double* dinv = nullptr;
  int* compPtr = nullptr;
  int *fwdPtr = nullptr, *fwdCol = nullptr, *bwdPtr = nullptr, *bwdCol = nullptr;
  double *fwdVal = nullptr, *bwdVal = nullptr;
  long *fwdMatPtr = nullptr, *bwdMatPtr = nullptr;
  double *fwdMat = nullptr, *bwdMat = nullptr;
  float *fwdLow = nullptr, *bwdLow = nullptr;
  LdltWideRow* wideRows = nullptr;  // of each row of the wide stages (row - wideBegin)
  double* wideBuf = nullptr;   // [2][kcap][n - wideBegin]: right-hand sides of the wide products
  // boundary factors: the texel of each row, and A_BD's rows in the factor's numbering
  int *texel = nullptr, *rhsPtr = nullptr, *rhsCol = nullptr;
  double* rhsVal = nullptr;
  int kcap = 0;
};

struct DevCsr {
  int rows = 0, nnz = 0;
  int *rowptr = nullptr, *col = nullptr;
  double* val = nullptr;
};

struct DevLevel {
  int N = 0, D = 0, B = 0;
  double* coef = nullptr;      // reciprocal (levels < L-1) deep stencil, SoA [10][D]
  double* coefRaw = nullptr;   // raw deep stencil A, SoA [10][D]
  double* coefSym = nullptr;   // level 0: A's deep couplings in symmetric five-word form, SoA [5][N] over global
                               // indices (slots 0-3: lower neighbours k = 0..3, slot 4: diagonal)
  int* bgi = nullptr;          // boundary -> global
  DevCsr brestr;               // boundary restriction to level+1
  DevCsr rows;                 // A_BB's and (from rowMid on) A_BD's entries row by row, global columns
  int* rowMid = nullptr;
  // band tasks
  int nTasks = 0;
  int* taskPtr = nullptr;
  int* blockRow = nullptr;                           // first row of each block in bandRows
  BandRow* bandRows = nullptr;
  int4* pairs = nullptr;                             // BandPair
  long nPairs = 0;
  int nRaster = 0, nRestr = 0, nProl = 0;
  int *raster = nullptr, *restr = nullptr, *prol = nullptr;  // 5, 5, 6 ints per line
  DevLdlt factor;              // boundary factor (levels < L-1) or full coarse factor (level L-1)
  // work vectors for up to `kcap` columns
  double *x = nullptr, *b = nullptr, *r = nullptr, *y = nullptr;
};

struct DeviceSystem {
  int levels = 0, kcap = 0;
  std::vector<DevLevel> L;
  DevLevel mass0, stiff0;      // level-0 mass and stiffness (raw stencils and boundary rows only; the rows share their columns)
  std::vector<void*> allocations;
  size_t bytes = 0;
  hipStream_t stream = nullptr;
  ~DeviceSystem();
};

// Upload an LDL^T factor's staged triangular solves; LdltSolve solves for K columns (at most kcap); dst
// may be src.  y: [K][n] scratch.
void UploadLdlt(std::vector<void*>& allocations, const Ldlt& F, DevLdlt& d, int kcap, const Csr* bd = nullptr,
                const std::vector<int>* bgi = nullptr);
// Bytes uploaded / allocated by this thread's device uploads so far (monotone counter).
size_t UploadByteCounter();
void LdltSolve(DevLdlt& F, const double* src, int lds, double* dst, int ldd, double* y, int K, hipStream_t s);

void UploadSystem(const Hierarchy& h, const OperatorHierarchy& oh, const FineOperator& op, int kcap, DeviceSystem& ds);

// One V-cycle of the reference schedule on level-0 vectors x (in/out) and b, K <= kcap columns,
// column stride ld (IterativeSolvers.inl:1211-1333).
void VCycleReference(DeviceSystem& ds, double* x, const double* b, int K, int ld, hipStream_t s);

// Building blocks, exported for kernel-level parity tests.
void RelaxLevel(DeviceSystem& ds, int level, double* x, const double* b, double* r, int K, int ld, bool withResidual, hipStream_t s);
void BandSweepLevel(DeviceSystem& ds, int level, double* x, const double* b, double* r, int K, int ld, hipStream_t s);
void RestrictLevel(DeviceSystem& ds, int level, const double* rFine, double* bCoarse, int K, int ldF, int ldC, hipStream_t s);
void ProlongAddLevel(DeviceSystem& ds, int level, const double* xCoarse, double* xFine, int K, int ldC, int ldF, hipStream_t s);
void BoundarySolveLevel(DeviceSystem& ds, int level, const double* rhs, double* sol, int K, int ld, hipStream_t s);
void CoarseSolve(DeviceSystem& ds, const double* rhs, double* sol, int K, int ld, hipStream_t s);
// y = A x with raw (non-reciprocal) coefficients of `level`; residual r = b - A x.
void ApplyLevel(DeviceSystem& ds, int level, const double* x, double* y, int K, int ld, hipStream_t s);
void ApplyOperator(DeviceSystem& ds, DevLevel& op, const double* x, double* y, int K, int ld, hipStream_t s);
// Squared 2-norms of K columns (stride ld) accumulated into dNorms[0..K) (zeroed first).
void SquaredNorms(const double* v, int N, int K, int ld, double* dNorms, hipStream_t s);
void ResidualLevel(DeviceSystem& ds, int level, const double* x, const double* b, double* r, int K, int ld, hipStream_t s);
// Squared norms of the level-0 residual b - A x and of b for K columns: out[2c] = ||b_c - A x_c||^2,
// out[2c + 1] = ||b_c||^2 (device, 2K doubles); `parts` is a device scratch of NormPartsSize(K)
// doubles, every entry of which the call overwrites.
constexpr int kNormParts = 512;
constexpr size_t NormPartsSize(int K) { return (size_t)2 * K * kNormParts; }
// weights: null, or two per column (host): column c's operator is weights[2c] M + weights[2c + 1] S.
void ResidualNorms(DeviceSystem& ds, const double* x, const double* b, int K, int ld, double* parts, double* out, hipStream_t s,
                   const double* weights = nullptr);
// The same with the scratch in a static device array (no allocation): at most kNoAllocMaxCols
// columns; the 2 K squared norms are copied to hostSquares and the stream is synchronised.
constexpr int kNoAllocMaxCols = 64;
void ResidualNormsNoAlloc(DeviceSystem& ds, const double* x, const double* b, int K, int ld, double* hostSquares, hipStream_t s);

// Normalised-gradient integration samples on the device (cell samples SoA [13][n]).
struct DevVectorField {
  long nCell = 0;
  int nGen = 0;
  int* cellCorners = nullptr;  // 4 per sample
  float* cellData = nullptr;   // SoA [13][nCell]
  double invCellW = 0, invCellH = 0;
  int *genPtr = nullptr, *genTexel = nullptr;
  float *genTensor = nullptr, *genG = nullptr, *genV = nullptr;
  std::vector<void*> allocations;
  ~DevVectorField();
};
void UploadVectorField(const VectorFieldSamples& vs, DevVectorField& d);
// rhs[:, t] = sum over samples of < -grad u / |grad u|_g , v(t) > for K columns of level-0 vectors
// (IntergrateNormalizedVectorFieldFromSamples, VectorFieldIntergration.inl:452-582); rhs is
// overwritten.
void VectorFieldDivergence(const DevVectorField& d, const double* u, int ldu, double* rhs, int ldr, int N, int K, hipStream_t s);

// Per-cell modulated stiffness of fixed signal columns (the sharpening brush's right-hand side,
// CellStiffnessToTexelStiffness, IterativeSolvers.inl:1170-1208): t_k = sum_c mask_c S_c f_k.
struct DevModulation {
  int K = 0, N = 0, D = 0, B = 0, numCells = 0;
  long nnz = 0;
  double* deep = nullptr;       // [K][4D]: the four cells around each deep texel
  int* deepCells = nullptr;     // [2D]: cells (i-1,j-1) and (i-1,j) of deep texel d
  int* deepGlobal = nullptr;    // [D]
  int *bRowptr = nullptr, *bCell = nullptr, *bGlobal = nullptr;
  double* bVal = nullptr;       // [K][nnz]
  size_t bytes = 0;
  std::vector<void*> allocations;
  ~DevModulation();
};
void UploadModulation(const Level& L0, const CellStiffnessRhs& c, DevModulation& m);
// out[k][t] = sum over the cells c of texel t of mask[c] * (S_c f_k)_t for every level-0 texel t
// (out is [K][N], overwritten; mask has one weight per active cell).
void ModulatedStiffness(const DevModulation& m, const double* mask, double* out, hipStream_t s);

}  // namespace gdtp
