// HIP kernels of the texel multigrid (CDNA4 / gfx950) and their host orchestration.
//
// Vectors are column-major: column c of a level-l vector starts at c*ld.  Deep stencils are
// stored structure-of-arrays, [10][D], so every stencil slot is a coalesced stream.
#include <algorithm>
#include <stdexcept>

#include "gdtp_device.h"
#include "gdtp_tiles.h"

#include <mutex>

namespace gdtp {

static constexpr int kWave = 64;
static constexpr int kBandColumns = 3;  // most columns of a band workgroup

// ------------------------------------------------------------------ band Gauss-Seidel
// The reference smoother (IterativeSolvers.inl:398-558 with residual, :174-395 without):
// per band task, blocks left to right; inside a block, three lagged passes over the block's deep
// rows (at step j rows j, j-1, j-2), each row a left-to-right Gauss-Seidel sweep of its deep segments.
// The reference also computes a row's residual inside the sweep, from final values only; it equals
// b - A x after the sweep, which is one streaming pass over the level (ResidualLevel).
//
// One workgroup per band task and chunk of KC columns.  The sweep is a chain: rows x passes of a block,
// blocks one after another.  Within a block three waves run the passes as a pipeline, one row per wave
// per step (step t: wave 0 row t first pass, wave 1 row t - 2 second, wave 2 row t - 4 third): each
// operation sees exactly the values it sees in the reference's order, rows of one step are disjoint,
// and a block of 16 rows takes 20 steps.  What bounds a launch is therefore the latency of a step, so
// a step touches no memory but LDS on its chain: the rows' values live in a ring of eight LDS rows
// (rows t - 5 .. t + 1 are read at step t, row t + 2 is filled meanwhile), a fourth wave streams the
// rows in two steps ahead, a pass loads its next row's stencil and right-hand side as soon as the
// current ones are used, and only the third pass stores.  The barrier of a step waits for LDS alone.
// The in-row dependence x_i = beta_i - c3_i x_{i-1} is a first-order linear recurrence: two texels per
// lane, then a wavefront scan by DPP moves.
// (Measured, us per sweep of both colours, 4096^2 icosphere, three columns: level 0 739, level 1 274,
// level 2 99; with x read and written through the L2, loads behind branches, the scan by LDS permutes
// and the residual rows as a fourth pass 2690, 1015, 408 (3.5-6 us a step).  Tried: a load per line that
// brings the next rows' stencils into the L2 ahead of the first pass (level 0 865 against 777 then), and
// nine pass waves of one column each instead of three of three (level 0 1346, level 1 467: the stencil
// loads of nine waves).  A lane's two neighbouring words as one 16-byte load: level 0 777 to 765.)
constexpr int kBandRing = 8;  // ring rows, of kBandRowMax texels
static_assert(kBandPairs == kWave, "a pair per lane");

// Wave-wide DPP move of a double; lanes without a source (and rows masked out) get `old`, or with kZero
// zero (for unmasked moves: no initial value to set up).
template <int kCtrl, int kRowMask = 0xf, bool kZero = false>
__device__ __forceinline__ double DppMove(double v, double old) {
  const unsigned long long u = __builtin_bit_cast(unsigned long long, v), o = __builtin_bit_cast(unsigned long long, old);
  unsigned lo, hi;
  if constexpr (kZero) {
    lo = __builtin_amdgcn_mov_dpp((int)u, kCtrl, kRowMask, 0xf, true);
    hi = __builtin_amdgcn_mov_dpp((int)(u >> 32), kCtrl, kRowMask, 0xf, true);
  } else {
    lo = __builtin_amdgcn_update_dpp((int)o, (int)u, kCtrl, kRowMask, 0xf, false);
    hi = __builtin_amdgcn_update_dpp((int)(o >> 32), (int)(u >> 32), kCtrl, kRowMask, 0xf, false);
  }
  return __builtin_bit_cast(double, (unsigned long long)hi << 32 | lo);
}
// One step of the inclusive scan of the maps x -> A x + B over the lanes (identity where no source).
template <int kCtrl, int kRowMask, int KC>
__device__ __forceinline__ void ScanStep(double& A, double (&B)[KC]) {
  const double Au = DppMove<kCtrl, kRowMask>(A, 1.0);
#pragma unroll
  for (int c = 0; c < KC; c++) B[c] += A * DppMove<kCtrl, kRowMask, kRowMask == 0xf>(B[c], 0.0);
  A *= Au;
}

// Two neighbouring doubles of a lane in one load (a pair starts at any texel: 8-byte alignment).
struct __attribute__((packed, aligned(8))) Double2 {
  double a, b;
};
__device__ __forceinline__ void LoadPair(const double* p, double& a, double& b) {
  const Double2 v = *reinterpret_cast<const Double2*>(p);
  a = v.a, b = v.b;
}

// All waves' LDS accesses before this point are done; global loads and stores stay in flight.
__device__ __forceinline__ void LdsBarrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

template <int KC>
__global__ __launch_bounds__(256) void KBandGs(int color, int nTasks, const int* __restrict__ taskPtr, const int* __restrict__ blockRow,
                                               const BandRow* __restrict__ rows, const int4* __restrict__ pairs,
                                               const double* __restrict__ coef, int D, double* x, const double* __restrict__ b, int K, int ld) {
  __shared__ double S[KC][kBandRing][kBandRowMax];
  const int task = 2 * blockIdx.x + color;
  if (task >= nTasks) return;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave), lane = threadIdx.x % kWave;
  // column of each slot of the chunk; the last chunk's slots past K repeat column K - 1 (same values)
  size_t col[KC];
#pragma unroll
  for (int c = 0; c < KC; c++) col[c] = (size_t)min((int)blockIdx.y * KC + c, K - 1) * ld;
  for (int blk = taskPtr[task]; blk < taskPtr[task + 1]; blk++) {
    // rows R[0 .. nr + 1]: the chart rows of the block's deep rows 1 .. nr and one row either side
    const BandRow* R = rows + blockRow[blk];
    const int nr = blockRow[blk + 1] - blockRow[blk] - 2, steps = nr + 4;
    __syncthreads();  // the block before this one has stored its rows
    if (wave == 3) {
      constexpr int kLoads = (KC * kBandRowMax + kWave - 1) / kWave;
      const double* from[kLoads];  // a lane's columns and places in a row, the same for every row
      double* to[kLoads];
      int at[kLoads];
#pragma unroll
      for (int k = 0; k < kLoads; k++) {
        const int e = min(lane + kWave * k, KC * kBandRowMax - 1), c = e / kBandRowMax;
        at[k] = e % kBandRowMax, to[k] = &S[c][0][at[k]];
        from[k] = x + (c == 0 ? col[0] : c == 1 ? col[KC > 1 ? 1 : 0] : col[KC - 1]);
      }
      // (a row's places past its texels repeat the last one; their values are not used)
      auto load = [&](int r, double (&v)[kLoads]) {
        const BandRow W = R[min(r, nr + 1)];
#pragma unroll
        for (int k = 0; k < kLoads; k++) v[k] = from[k][W.base + min(at[k], max(W.len - 1, 0))];
      };
      auto put = [&](int r, const double (&v)[kLoads]) {
#pragma unroll
        for (int k = 0; k < kLoads; k++) to[k][(r % kBandRing) * kBandRowMax] = v[k];
      };
      double v0[kLoads], v1[kLoads], v2[kLoads];
      load(0, v0), load(1, v1), load(2, v2);
      put(0, v0), put(1, v1), put(2, v2);
      load(3, v0), load(4, v1);
      LdsBarrier();
      for (int t = 0; t < steps; t += 2) {
        put(t + 3, v0);
        load(t + 5, v0);
        LdsBarrier();
        if (t + 1 == steps) break;
        put(t + 4, v1);
        load(t + 6, v1);
        LdsBarrier();
      }
      continue;
    }
    // pair of this lane in row r: texels g, g + 1 with stencils d, d + 1 (first: g starts a segment;
    // two: both are deep) and the LDS places of g, of the texel above g - 1 and of the one below g - 1
    auto pairOf = [&](const BandRow& W) { return pairs[lane < W.pairs ? W.pair0 + lane : 0]; };
    double c0[9], c1[9], b0[KC], b1[KC];
    auto operands = [&](const int4& P) {
#pragma unroll
      for (int k = 0; k < 9; k++) LoadPair(coef + (size_t)k * D + P.y, c0[k], c1[k]);
#pragma unroll
      for (int c = 0; c < KC; c++) LoadPair(b + col[c] + P.x, b0[c], b1[c]);
    };
    int n0 = R[1].pairs;
    int4 P0 = pairOf(R[1]);
    operands(P0);
    BandRow W1 = R[min(2, nr + 1)];
    int4 P1 = pairOf(W1);
    LdsBarrier();
    for (int t = 0; t < steps; t++) {
      const int r = t + 1 - 2 * wave;
      if (r >= 1 && r <= nr) {
        const BandRow W2 = R[min(r + 2, nr + 1)];
        const int4 P2 = pairOf(W2);
        const bool first = P0.w & 1, two = P0.w & 2, active = lane < n0;
        const int og = P0.z & 255, oa = (P0.z >> 8) & 255, ob = (P0.z >> 16) & 255;
        const double a0 = first ? 0.0 : -c0[3], a1 = two ? -c1[3] : 0.0;
        double beta0[KC], beta1[KC];
#pragma unroll
        for (int c = 0; c < KC; c++) {
          double* own = &S[c][r % kBandRing][og];
          const double* up = &S[c][(r - 1) % kBandRing][oa];
          const double* dn = &S[c][(r + 1) % kBandRing][ob];
          const double u0 = up[0], u1 = up[1], u2 = up[2], u3 = up[3], w0 = dn[0], w1 = dn[1], w2 = dn[2], w3 = dn[3];
          const double left = own[-1], right = own[1], far = own[2];
          const double s0 = u0 * c0[0] + u1 * c0[1] + u2 * c0[2] + right * c0[5] + w0 * c0[6] + w1 * c0[7] + w2 * c0[8];
          const double s1 = u1 * c1[0] + u2 * c1[1] + u3 * c1[2] + far * c1[5] + w1 * c1[6] + w2 * c1[7] + w3 * c1[8];
          double v = b0[c] * c0[4] - s0;
          if (first) v -= left * c0[3];
          beta0[c] = v;
          beta1[c] = two ? b1[c] * c1[4] - s1 : 0.0;
        }
        operands(P1);  // the next row's, in flight until the next step
        // the lane's two texels as one map, then an inclusive scan over the wave
        double A = a1 * a0, B[KC];
#pragma unroll
        for (int c = 0; c < KC; c++) B[c] = a1 * beta0[c] + beta1[c];
        ScanStep<0x111, 0xf, KC>(A, B);  // row_shr:1, 2, 4, 8 within 16 lanes
        ScanStep<0x112, 0xf, KC>(A, B);
        ScanStep<0x114, 0xf, KC>(A, B);
        ScanStep<0x118, 0xf, KC>(A, B);
        ScanStep<0x142, 0xa, KC>(A, B);  // row_bcast:15 into rows 1 and 3
        ScanStep<0x143, 0xc, KC>(A, B);  // row_bcast:31 into rows 2 and 3
#pragma unroll
        for (int c = 0; c < KC; c++) {
          const double prev = DppMove<0x138, 0xf, true>(B[c], 0.0);  // wave_shr:1
          const double x0 = a0 * prev + beta0[c], x1 = a1 * x0 + beta1[c];
          if (active) {
            double* own = &S[c][r % kBandRing][og];
            own[0] = x0;
            if (two) own[1] = x1;
            if (wave == 2) {
              x[col[c] + P0.x] = x0;
              if (two) x[col[c] + P0.x + 1] = x1;
            }
          }
        }
        P0 = P1, P1 = P2, n0 = W1.pairs, W1 = W2;
      }
      LdsBarrier();
    }
  }
}

// ------------------------------------------------------------------ exact LDL^T solves
// The staged triangular solves (LdltStages): forward stages r = src[perm] - L y(earlier stages),
// y = inv(L_cc) r per component, then backward r = y / D - L^T x(later stages), x = inv(L_cc)^T r.
//
// What bounds them: a dependency chain.  The level-scheduled solve they replace walked the elimination
// tree's 250-450 levels (subtree teams of one workgroup, a barrier per level, one thread per row), each
// level a round trip to memory: 1.75 ms for the 175,580 boundary rows of a 4096^2 atlas and three
// columns, 0.25 ms for 3840 rows; the stages take 0.25 and 0.03 ms.  Explicit inverses of components of up
// to 128 (first stage) or a few hundred rows leave two passes per stage, each a gather and a product with
// loads that wait for nothing.  Inverses and couplings are 5 to 13 times the bytes of a boundary factor's L by
// rows and by columns (2048^2 icosphere 183 MB against 34, 1200^2 cube 89 against 7), twice those of a
// direct solve's (840 k texels: 5.0 GB against 2.4).

// Lanes' sum over groups of G lanes.
template <int G>
__device__ __forceinline__ double GroupSum(double v) {
#pragma unroll
  for (int o = G / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, G);
  return v;
}
// A sum in two doubles, v and what its additions rounded away, e (compensated summation: T. Ogita,
// S. M. Rump and S. Oishi, "Accurate sum and dot product", SIAM J. Sci. Comput. 26, 2005).
struct Sum2 {
  double v, e;
  // (the error terms are differences of rounded values: nothing here may be contracted)
  __device__ __forceinline__ void Add(double b) {
#pragma clang fp contract(off)
    const double t = v + b, z = t - v;
    e += (v - (t - z)) + (b - z);
    v = t;
  }
  __device__ __forceinline__ void Add(const Sum2& s) {
    Add(s.v);
    e += s.e;
  }
  // + (high + low) x, the product's own rounding kept too.  (Add with the unrounded product in one fused
  // step, three operations fewer, is not exact where the product exceeds the sum: residual 3 times larger.)
  __device__ __forceinline__ void AddProduct(double high, float low, double x) {
#pragma clang fp contract(off)
    const double p = high * x;
    e += __builtin_fma(high, x, -p);
    e = __builtin_fma((double)low, x, e);
    Add(p);
  }
  __device__ __forceinline__ double Value() const { return v + e; }
};
// A DPP move of a sum (zero where no source).
template <int kCtrl, int kRowMask>
__device__ __forceinline__ Sum2 DppMove(const Sum2& s) {
  return {DppMove<kCtrl, kRowMask, kRowMask == 0xf>(s.v, 0.0), DppMove<kCtrl, kRowMask, kRowMask == 0xf>(s.e, 0.0)};
}
// The wave's sum in lane 63, by DPP moves.
__device__ __forceinline__ double WaveSumLast(Sum2 s) {
  s.Add(DppMove<0x111, 0xf>(s));
  s.Add(DppMove<0x112, 0xf>(s));
  s.Add(DppMove<0x114, 0xf>(s));
  s.Add(DppMove<0x118, 0xf>(s));
  s.Add(DppMove<0x142, 0xa>(s));
  s.Add(DppMove<0x143, 0xc>(s));
  return s.Value();
}

// The tables of one direction and the vectors of a solve.
struct LdltPass {
  const int* compPtr;
  const long* matPtr;
  const double* mat;
  const float* low;
  const int *ptr, *col;  // couplings with the stages solved before
  const double* val;
  const int* index;      // of each row in the right-hand side (forward) or the solution (backward)
  const double* dinv;
  // the relaxation's right-hand side b - A_BD x is formed by the forward stages: A_BD's rows
  const int *rhsPtr, *rhsCol;
  const double *rhsVal, *rhsX;
};

// A group of G lanes adds val y[col] over entries [p0, p1) to s, for up to KC columns.
template <int G, int KC>
__device__ __forceinline__ void CouplingTerms(const int* __restrict__ col, const double* __restrict__ val, int p0, int p1, int lane,
                                              const double* y, size_t n, int kc, double (&s)[KC]) {
  for (int p = p0 + lane; p < p1; p += G) {
    const double v = val[p];
    const int j = col[p];
#pragma unroll
    for (int c = 0; c < KC; c++) s[c] += v * y[min(c, kc - 1) * n + j];
  }
}

// Row w's right-hand side of a stage in lane c (of the group) for column c: what is known of it
// (forward: b, backward: y / D) less its couplings with the stages solved before.
template <bool kForward, bool kRhs, int G, int KC>
__device__ __forceinline__ double StageRhs(const LdltPass& P, int w, int lane, const double* src, int lds, const double* y, int n, int c0,
                                           int kc) {
  double s[KC] = {};
  // column slots past kc repeat the last column, so that no load is behind a branch
  const int c = min(min(lane, KC - 1), kc - 1);
  const double known = kForward ? src[(size_t)(c0 + c) * lds + P.index[w]] : y[(size_t)c * n + w] * P.dinv[w];
  CouplingTerms<G, KC>(P.col, P.val, P.ptr[w], P.ptr[w + 1], lane, y, n, kc, s);
  if constexpr (kRhs) CouplingTerms<G, KC>(P.rhsCol, P.rhsVal, P.rhsPtr[w], P.rhsPtr[w + 1], lane, P.rhsX + (size_t)c0 * lds, lds, kc, s);
  double mine = 0.0;
#pragma unroll
  for (int k = 0; k < KC; k++) {
    const double t = GroupSum<G>(s[k]);
    if (k == c) mine = t;
  }
  return known - mine;
}

// The 16 waves of a narrow component's workgroup are divided over its row blocks (at most four) in
// proportion to the blocks' columns (forward: later blocks have more; backward: mirrored).
__device__ __constant__ const unsigned char kWaveSplit[4][5] = {{0, 16, 16, 16, 16}, {0, 5, 16, 16, 16}, {0, 3, 8, 16, 16}, {0, 2, 5, 10, 16}};
static constexpr int kEarlyColumns = 13; // loaded ahead: all of them for components of up to 128 rows

// A narrow stage: one workgroup of 16 waves per component of at most kLdltNarrowRows rows and chunk of
// up to KC columns.  A wave owns one row per lane and a share of its block's columns, so the inverse's
// loads are whole lines that wait for nothing; they go out first and are in flight while the
// component's right-hand side is gathered into LDS.  The waves' parts are added in a fixed order.
// What bounds a launch: HBM where components are many (1981 of them, three columns: 55 us forward with rounded
// inverses, 86 with both parts), else the chain of one workgroup, the FP64 additions of its sums among
// it (52 components: 10.7 us with three columns a workgroup, 8.4 with one).
template <bool kForward, bool kRhs, int G, int KC>
__global__ __launch_bounds__(1024) void KLdltNarrow(int comp0, LdltPass P, const double* src, int lds, double* y, int n, double* dst, int ldd,
                                                    int K) {
  __shared__ double R[KC][kLdltNarrowRows];
  __shared__ Sum2 Q[16][KC][kLdltBlock];
  const int comp = comp0 + blockIdx.x, w0 = P.compPtr[comp], m = P.compPtr[comp + 1] - w0;
  const int c0 = blockIdx.y * KC, kc = min(KC, K - c0);
  y += (size_t)c0 * n;
  const int blocks = (m + kLdltBlock - 1) / kLdltBlock, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave), lane = threadIdx.x % kWave;
  // this wave's block: the split's k-th (backward: mirrored, so that the widest block gets the most waves)
  int k = 0;
  while (wave >= kWaveSplit[blocks - 1][k + 1]) k++;
  const int part = wave - kWaveSplit[blocks - 1][k], parts = kWaveSplit[blocks - 1][k + 1] - kWaveSplit[blocks - 1][k];
  const int rb = kForward ? k : blocks - 1 - k, r0 = rb * kLdltBlock, nr = min(kLdltBlock, m - r0);
  const int j0 = kForward ? 0 : r0, cols = kForward ? r0 + nr : m - r0;
  // the blocks before this one: kLdltBlock rows each (only the last is shorter)
  const long off = P.matPtr[comp] + (kForward ? (long)kLdltBlock * kLdltBlock * (rb * (rb + 1) / 2)
                                              : (long)kLdltBlock * rb * m - (long)kLdltBlock * kLdltBlock * (rb * (rb - 1) / 2));
  const double* M = P.mat + off + min(lane, nr - 1);
  const float* Ml = P.low + off + min(lane, nr - 1);
  double early[kEarlyColumns];
  float earlyLow[kEarlyColumns];
#pragma unroll
  for (int q = 0; q < kEarlyColumns; q++) {
    const size_t o = (size_t)min(part + q * parts, cols - 1) * nr;
    early[q] = M[o], earlyLow[q] = Ml[o];
  }
  const int outRow = min((int)threadIdx.x, m * KC - 1) % m;
  const int out = kForward ? 0 : P.index[w0 + outRow];
  for (int i = threadIdx.x / G; i < m; i += 1024 / G) {
    const int gl = threadIdx.x % G;
    const double v = StageRhs<kForward, kRhs, G, KC>(P, w0 + i, gl, src, lds, y, n, c0, kc);
    if (gl < KC) R[gl][i] = v;
  }
  __syncthreads();
  Sum2 acc[KC] = {};
#pragma unroll
  for (int q = 0; q < kEarlyColumns; q++) {
    const int j = part + q * parts;
    if (j >= cols) break;
#pragma unroll
    for (int c = 0; c < KC; c++) acc[c].AddProduct(early[q], earlyLow[q], R[c][j0 + j]);
  }
#pragma unroll 4
  for (int j = part + kEarlyColumns * parts; j < cols; j += parts) {
    const double a = M[(size_t)j * nr];
    const float al = Ml[(size_t)j * nr];
#pragma unroll
    for (int c = 0; c < KC; c++) acc[c].AddProduct(a, al, R[c][j0 + j]);
  }
#pragma unroll
  for (int c = 0; c < KC; c++) Q[wave][c][lane] = acc[c];
  __syncthreads();
  static_assert(kLdltNarrowRows * 4 <= 1024, "one result per thread");
  if ((int)threadIdx.x < m * kc) {
    const int c = threadIdx.x / m, i = outRow, b = i / kLdltBlock, kk = kForward ? b : blocks - 1 - b;
    Sum2 sum = {};
    for (int q = kWaveSplit[blocks - 1][kk]; q < kWaveSplit[blocks - 1][kk + 1]; q++) sum.Add(Q[q][c][i % kLdltBlock]);
    const double s = sum.Value();
    y[(size_t)c * n + w0 + i] = s;
    if (!kForward) dst[(size_t)(c0 + c) * ldd + out] = s;
  }
}

// A wide stage's right-hand sides (its rows [row0, row1), one wave per row and chunk of columns).
template <bool kForward, bool kRhs, int KC>
__global__ __launch_bounds__(256) void KLdltCouple(int row0, int row1, int wideBegin, LdltPass P, const double* src, int lds, const double* y,
                                                   int n, double* buf, int nWide, int K) {
  const int w = row0 + blockIdx.x * (256 / kWave) + (int)threadIdx.x / kWave, lane = threadIdx.x % kWave;
  if (w >= row1) return;
  const int c0 = blockIdx.y * KC, kc = min(KC, K - c0);
  const double v = StageRhs<kForward, kRhs, kWave, KC>(P, w, lane, src, lds, y + (size_t)c0 * n, n, c0, kc);
  if (lane < kc) buf[(size_t)(c0 + lane) * nWide + w - wideBegin] = v;
}

// A wide stage's product with its components' inverses, one wave per row and chunk of columns, two
// entries per lane and load: the forward result to y, or for the top scaled by 1 / D to `top` (the
// backward product's input); the backward result to y and dst.  (1920 rows, three columns: forward
// 26 and backward 20 us with one entry per load and the component looked up first, 13 and 8 us so; with
// compensated sums 35 and 33 us with three columns a wave, 20 and 19 with one.)
template <bool kForward, int KC>
__global__ __launch_bounds__(256) void KLdltWide(int row0, int row1, int wideBegin, const LdltWideRow* __restrict__ wideRows, LdltPass P,
                                                 const double* __restrict__ buf, int nWide, double* y, int n, double* top, double* dst, int ldd,
                                                 int K) {
  const int w = row0 + blockIdx.x * (256 / kWave) + (int)threadIdx.x / kWave, lane = threadIdx.x % kWave;
  if (w >= row1) return;
  const LdltWideRow T = wideRows[w - wideBegin];
  const int i = w - T.begin, m = T.rows;
  const int c0 = blockIdx.y * KC, kc = min(KC, K - c0);
  const double* row = P.mat + T.mat[kForward ? 0 : 1];
  const float* low = P.low + T.mat[kForward ? 0 : 1];
  const double* in = buf + (size_t)c0 * nWide + T.begin - wideBegin;
  const double dinv = P.dinv[w];
  const int out = kForward ? 0 : P.index[w];
  Sum2 acc[KC] = {};
  const int j1 = kForward ? i + 1 : m;
#pragma unroll 4
  for (int j = (kForward ? 0 : i / 2 * 2) + 2 * lane; j < j1; j += 2 * kWave) {  // backward: entries before i are zero
    double a0, a1;
    LoadPair(row + j, a0, a1);
    const float l0 = low[j], l1 = low[j + 1];
    const bool both = j + 1 < m;  // (a row of odd length is padded with a zero; the vector is not)
#pragma unroll
    for (int c = 0; c < KC; c++) {
      double v0, v1;
      LoadPair(in + (size_t)min(c, kc - 1) * nWide + j, v0, v1);
      acc[c].AddProduct(a0, l0, v0);
      if (both) acc[c].AddProduct(a1, l1, v1);
    }
  }
#pragma unroll
  for (int c = 0; c < KC; c++) {
    const double s = WaveSumLast(acc[c]);
    if (lane != kWave - 1 || c >= kc) continue;
    if (kForward && top) top[(size_t)(c0 + c) * nWide + w - wideBegin] = s * dinv;
    else y[(size_t)(c0 + c) * n + w] = s;
    if (!kForward) dst[(size_t)(c0 + c) * ldd + out] = s;
  }
}

// ------------------------------------------------------------------ transfers
// Sparse rows (boundary rows of an operator, of the restriction): kRowLanes lanes per row, so that a
// row's entries are read together instead of one round trip after another.
static constexpr int kRowLanes = 8;
static constexpr int kRowBatch = 4 * kRowLanes;  // entries staged at a time
static constexpr int kRowThreads = 128;          // threads of the kernels that take sparse rows and lines
template <int KC, int kThreads>
struct RowTerms {
  double val[kThreads / kRowLanes][kRowBatch + 1], x[kThreads / kRowLanes][KC][kRowBatch + 1];
};

// Sum over entries [k0, mid) plus sum over [mid, k1) of val x[col] for column (lane of the row's group),
// up to KC columns (lane < kc).  Seam rows cancel, so both the order of the additions and their single
// rounding are kept: the lanes stage an entry's value and its columns' x in LDS, and lane c takes column
// c's in the row's order, one fused multiply-add each.  (Staged as products, each rounded before it is added,
// the result differs in its last bits: rows of texels with a support of 1e-12 of the others then moved a
// mixed solve to a tolerance of 1e-6 by up to 1.6e-2 on a 48,614-texel atlas.)
template <int KC, int kThreads>
__device__ __forceinline__ double RowSum(int k0, int mid, int k1, const int* __restrict__ cl, const double* __restrict__ vl,
                                         const double* __restrict__ x, size_t ld, int kc, RowTerms<KC, kThreads>& terms) {
  double(&V)[kRowBatch + 1] = terms.val[threadIdx.x / kRowLanes];
  double(&X)[KC][kRowBatch + 1] = terms.x[threadIdx.x / kRowLanes];
  const int lane = threadIdx.x % kRowLanes;
  double first = 0.0, second = 0.0;
  for (int at = k0; at < k1; at += kRowBatch) {
    double v[kRowBatch / kRowLanes], xv[kRowBatch / kRowLanes][KC];
#pragma unroll
    for (int q = 0; q < kRowBatch / kRowLanes; q++) {
      const int k = min(at + lane + kRowLanes * q, k1 - 1);
      const int g = cl[k];
      v[q] = vl[k];
#pragma unroll
      for (int c = 0; c < KC; c++) xv[q][c] = x[(size_t)min(c, kc - 1) * ld + g];
    }
#pragma unroll
    for (int q = 0; q < kRowBatch / kRowLanes; q++) {
      V[lane + kRowLanes * q] = v[q];
#pragma unroll
      for (int c = 0; c < KC; c++) X[c][lane + kRowLanes * q] = xv[q][c];
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // the group's lanes are of one wave
    if (lane < kc) {
      const int n = min(kRowBatch, k1 - at), m = min(max(mid - at, 0), n);
      const double* t = X[lane];
#pragma unroll 8
      for (int k = 0; k < m; k++) first = fma(V[k], t[k], first);
#pragma unroll 8
      for (int k = m; k < n; k++) second = fma(V[k], t[k], second);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  }
  return first + second;
}

// Restriction into the next level in one launch (blockIdx.y = chunk of KC columns): blocks [0, rowBlocks)
// take the coarse boundary rows (R_B r, IterativeSolvers.inl:1027-1030), the others one restriction line
// each, coarse deep texels by 3x3 full weighting around the fine texel 2c (:1034-1050).  With `zero` the
// coarse vector there is set to zero as well (the coarse correction of a V-cycle starts from zero).
template <int KC>
__global__ __launch_bounds__(kRowThreads) void KRestrict(int rowBlocks, int rows, const int* __restrict__ outMap, const int* __restrict__ rp,
                                                         const int* __restrict__ cl, const double* __restrict__ vl, int nLines,
                                                         const int* __restrict__ lines, const double* __restrict__ in, int ldi, double* out,
                                                         double* zero, int ldo, int K) {
  const int c0 = blockIdx.y * KC, kc = min(KC, K - c0);
  in += (size_t)c0 * ldi, out += (size_t)c0 * ldo;
  if (zero) zero += (size_t)c0 * ldo;
  if ((int)blockIdx.x < rowBlocks) {
    __shared__ RowTerms<KC, kRowThreads> terms;
    const int row = (blockIdx.x * kRowThreads + (int)threadIdx.x) / kRowLanes, c = threadIdx.x % kRowLanes;
    if (row >= rows) return;  // whole row groups leave together
    const double s = RowSum(rp[row], rp[row + 1], rp[row + 1], cl, vl, in, ldi, kc, terms);
    if (c < kc) {
      const size_t o = (size_t)c * ldo + outMap[row];
      out[o] = s;
      if (zero) zero[o] = 0.0;
    }
    return;
  }
  const int* L = lines + 5 * (blockIdx.x - rowBlocks);
  const int start = L[0], end = L[1], prev = L[2], next = L[3], outStart = L[4];
  const int len = (end - start) / 2 + 1;
  for (int i = threadIdx.x; i < len; i += kRowThreads) {
    const int j = 2 * i;
    double v[KC][9];
#pragma unroll
    for (int c = 0; c < KC; c++) {
      const double* X = in + (size_t)min(c, kc - 1) * ldi;
#pragma unroll
      for (int k = 0; k < 9; k++) v[c][k] = X[(k < 3 ? prev : k < 6 ? start : next) + j + k % 3 - 1];
    }
#pragma unroll
    for (int c = 0; c < KC; c++)
      if (c < kc) {
        const double* R = v[c];
        out[(size_t)c * ldo + outStart + i] = R[4] + (R[1] + R[3] + R[5] + R[7]) * 0.5 + (R[0] + R[2] + R[6] + R[8]) * 0.25;
        if (zero) zero[(size_t)c * ldo + outStart + i] = 0.0;
      }
  }
}

// x_fine += P x_coarse, bilinear along prolongation lines (IterativeSolvers.inl:1122-1168)
__global__ void KProlongAdd(int nLines, const int* __restrict__ lines, const double* __restrict__ in, int ldi, double* out, int ldo, int K) {
  const int l = blockIdx.x;
  if (l >= nLines) return;
  const int* L = lines + 6 * l;
  const int start = L[0], len = L[1], center = L[2], prev = L[3], next = L[4], off = L[5] ? 0 : 1;
  for (int i = threadIdx.x; i < len; i += blockDim.x) {
    const int a = (i + off) / 2, bq = (i + off + 1) / 2;
    for (int c = 0; c < K; c++) {
      const double* X = in + (size_t)c * ldi;
      double v = center != -1 ? (X[center + a] + X[center + bq]) * 0.5 : (X[prev + a] + X[prev + bq] + X[next + a] + X[next + bq]) * 0.25;
      out[(size_t)c * ldo + start + i] += v;
    }
  }
}

// ------------------------------------------------------------------ operator application
// y = A x with raw stencils (MultiplyBySystemMatrix_NoReciprocals, IterativeSolvers.inl:881-950), or with
// `b` the residual b - A x, in one launch: first the boundary rows (rowBlocks blocks per chunk of KC
// columns, all of whose loads are in flight together), then a raster line and chunk per workgroup.
// (A small apply is its launches and round trips: one launch with kRowLanes lanes per row and global
// columns took 6,936 texels x 3 columns from 14.1 to 4.4 us of kernels (13.2 to 9.9 a call) against a thread
// per row and column that looked its A_BB columns up, beside the deep rows' own launch.  A large one is bound
// by memory: a line's chunks and its neighbours in one XCD's L2 (TileOf) took 3.3 M texels x 16 columns from
// 551 to 484 us.)
template <int KC>
__global__ __launch_bounds__(kRowThreads) void KApply(int rowBlocks, int nLines, int B, const int* __restrict__ bgi, const int* __restrict__ rp,
                                                      const int* __restrict__ mid, const int* __restrict__ cl, const double* __restrict__ vl, const int* __restrict__ lines,
                                                      const double* __restrict__ coef, int D, const double* __restrict__ x,
                                                      const double* __restrict__ b, double* y, int K, int ld) {
  const int rowWork = rowBlocks * ((K + KC - 1) / KC);
  const bool onBoundary = (int)blockIdx.x < rowWork;
  const TileChunk v0 = onBoundary ? TileOf<KC>(blockIdx.x, rowBlocks, K) : TileOf<KC>(blockIdx.x - rowWork, nLines, K);
  const int c0 = v0.c0, kc = min(KC, K - c0);
  x += (size_t)c0 * ld, y += (size_t)c0 * ld;
  if (b) b += (size_t)c0 * ld;
  if (onBoundary) {
    __shared__ RowTerms<KC, kRowThreads> terms;
    const int row = (v0.tile * kRowThreads + (int)threadIdx.x) / kRowLanes, c = threadIdx.x % kRowLanes;
    if (row >= B) return;  // whole row groups leave together
    const double s = RowSum(rp[row], mid[row], rp[row + 1], cl, vl, x, ld, kc, terms);
    if (c < kc) {
      const size_t o = (size_t)c * ld + bgi[row];
      y[o] = b ? b[o] - s : s;
    }
    return;
  }
  const int* L = lines + 5 * v0.tile;
  const int start = L[0], len = L[1] - L[0] + 1, prev = L[2], next = L[3], d0 = L[4];
  for (int i = threadIdx.x; i < len; i += kRowThreads) {
    double a[9], v[KC][9], bv[KC];
#pragma unroll
    for (int k = 0; k < 9; k++) a[k] = coef[(size_t)k * D + d0 + i];
#pragma unroll
    for (int c = 0; c < KC; c++) {
      const size_t o = (size_t)min(c, kc - 1) * ld;
#pragma unroll
      for (int k = 0; k < 9; k++) v[c][k] = x[o + (k < 3 ? prev : k < 6 ? start : next) + i + k % 3 - 1];
      bv[c] = b ? b[o + start + i] : 0.0;
    }
#pragma unroll
    for (int c = 0; c < KC; c++)
      if (c < kc) {
        double s = v[c][0] * a[0];
#pragma unroll
        for (int k = 1; k < 9; k++) s += v[c][k] * a[k];
        y[(size_t)c * ld + start + i] = b ? bv[c] - s : s;
      }
  }
}

// Squared 2-norm of column blockIdx.y: a bounded grid strides over the column so that only a
// few hundred blocks add into the column's accumulator.
__global__ __launch_bounds__(256) void KSquaredNorm(int N, const double* __restrict__ v, int ld, double* out) {
  const int c = blockIdx.y;
  double a = 0.0;
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < N; i += (long)gridDim.x * blockDim.x) {
    const double t = v[(long)c * ld + i];
    a += t * t;
  }
  for (int o = 32; o > 0; o >>= 1) a += __shfl_xor(a, o, 64);
  __shared__ double part[4];
  if (threadIdx.x % 64 == 0) part[threadIdx.x / 64] = a;
  __syncthreads();
  if (threadIdx.x == 0) atomicAdd(out + c, part[0] + part[1] + part[2] + part[3]);
}

__global__ void KZero(long n, double* x) {
  long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) x[i] = 0.0;
}

// ------------------------------------------------------------------ host side
static inline unsigned Blocks(long n, int bs) { return (unsigned)((n + bs - 1) / bs); }

DeviceSystem::~DeviceSystem() {
  for (void* p : allocations) (void)hipFree(p);
}

// ------------------------------------------------------------------ normalised-gradient integration
// One thread per cell sample: the bilinear gradient at the sample from its 4 corners, normalised in
// the metric, dotted with the 4 integrated basis gradients and added to the corners' rhs.
// Atomic adds bound it: a triangle's samples run along its rows of cells, so the next lane's left corners
// are mostly this lane's right ones, and the lane takes their terms along (DPP) before adding.
// (4.4 M samples x 64 columns: 14.8 ms with four adds per sample, 11.6 so; sorted by texel 23.6.)
__global__ __launch_bounds__(256) void KVfCell(long n, const int* __restrict__ corners, const float* __restrict__ data, double invW, double invH,
                                               const double* __restrict__ u, int ldu, double* rhs, int ldr, int K) {
  const long at = (long)blockIdx.x * blockDim.x + threadIdx.x, s = min(at, n - 1);
  const bool active = at < n;  // every lane takes part in the moves
  int cn[4];
  for (int k = 0; k < 4; k++) cn[k] = corners[4 * s + k];
  const double x = data[s], y = data[n + s], t00 = data[2 * n + s], t01 = data[3 * n + s], t11 = data[4 * n + s];
  double vx[4], vy[4];
  for (int k = 0; k < 4; k++) vx[k] = data[(5 + 2 * k) * n + s], vy[k] = data[(6 + 2 * k) * n + s];
  // corners 1 and 2 (right) against the next lane's 0 and 3 (left); -1 where there is none
  const int next0 = __builtin_amdgcn_update_dpp(-1, active ? cn[0] : -1, 0x130, 0xf, 0xf, false);  // wave_shl:1
  const int next3 = __builtin_amdgcn_update_dpp(-1, active ? cn[3] : -1, 0x130, 0xf, 0xf, false);
  const int take1 = active && next0 == cn[1], take2 = active && next3 == cn[2];
  const int give0 = __builtin_amdgcn_update_dpp(0, take1, 0x138, 0xf, 0xf, false), give3 = __builtin_amdgcn_update_dpp(0, take2, 0x138, 0xf, 0xf, false);
  for (int ch = 0; ch < K; ch++) {
    const double* U = u + (long)ch * ldu;
    const double c0 = U[cn[0]], c1 = U[cn[1]], c2 = U[cn[2]], c3 = U[cn[3]];
    // the bilinear gradient in difference form: exactly zero for a constant potential
    const double nx = -((1 - y) * (c1 - c0) + y * (c2 - c3)) * invW;
    const double ny = -((1 - x) * (c3 - c0) + x * (c2 - c1)) * invH;
    const double ax = t00 * nx + t01 * ny, ay = t01 * nx + t11 * ny;
    const double len2 = nx * ax + ny * ay;
    const bool any = active && len2 > 0;
    const double il = any ? 1.0 / sqrt(len2) : 0.0;
    double v[4];
    for (int k = 0; k < 4; k++) v[k] = any ? (ax * vx[k] + ay * vy[k]) * il : 0.0;
    const double n0 = DppMove<0x130, 0xf, true>(v[0], 0.0), n3 = DppMove<0x130, 0xf, true>(v[3], 0.0);
    if (take1) v[1] += n0;
    if (take2) v[2] += n3;
    double* R = rhs + (long)ch * ldr;
    if (v[1] != 0.0) atomicAdd(&R[cn[1]], v[1]);
    if (v[2] != 0.0) atomicAdd(&R[cn[2]], v[2]);
    if (!give0 && v[0] != 0.0) atomicAdd(&R[cn[0]], v[0]);
    if (!give3 && v[3] != 0.0) atomicAdd(&R[cn[3]], v[3]);
  }
}

// One thread per general sample (quadratic seam elements): gradient from its texel entries.
__global__ void KVfGeneral(int n, const int* __restrict__ ptr, const int* __restrict__ texel, const float* __restrict__ G,
                           const float* __restrict__ V, const float* __restrict__ T, const double* __restrict__ u, int ldu, double* rhs,
                           int ldr, int K) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n) return;
  const int e0 = ptr[s], e1 = ptr[s + 1];
  const double t00 = T[3 * s], t01 = T[3 * s + 1], t11 = T[3 * s + 2];
  for (int ch = 0; ch < K; ch++) {
    const double* U = u + (long)ch * ldu;
    // the entries' G sum to zero: differences to the first entry's value keep a constant exact
    const double u0 = U[texel[e0]];
    double nx = 0, ny = 0;
    for (int e = e0 + 1; e < e1; e++) {
      const double du = U[texel[e]] - u0;
      nx -= G[2 * e] * du, ny -= G[2 * e + 1] * du;
    }
    const double ax = t00 * nx + t01 * ny, ay = t01 * nx + t11 * ny;
    const double len2 = nx * ax + ny * ay;
    if (!(len2 > 0)) continue;
    const double il = 1.0 / sqrt(len2);
    double* R = rhs + (long)ch * ldr;
    for (int e = e0; e < e1; e++) atomicAdd(&R[texel[e]], (ax * V[2 * e] + ay * V[2 * e + 1]) * il);
  }
}

__global__ void KZeroStrided(int N, double* x, int ld, int K) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (long)N * K) return;
  x[(t / N) * ld + t % N] = 0.0;
}

static thread_local size_t g_uploadBytes = 0;
size_t UploadByteCounter() { return g_uploadBytes; }

template <class V, class T = std::decay_t<decltype(*std::declval<const V&>().data())>>
static T* UploadTo(std::vector<void*>& allocs, const V& v) {
  if (v.size() == 0) return nullptr;
  T* p = nullptr;
  GDTP_HIP(hipMalloc(&p, v.size() * sizeof(T)));
  allocs.push_back(p);
  g_uploadBytes += v.size() * sizeof(T);
  GDTP_HIP(hipMemcpy(p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice));
  return p;
}

template <class T>
static T* Upload(DeviceSystem& ds, const std::vector<T>& v) {
  return UploadTo(ds.allocations, v);
}

static double* Alloc(DeviceSystem& ds, size_t n) {
  double* p = nullptr;
  GDTP_HIP(hipMalloc(&p, std::max<size_t>(n, 1) * sizeof(double)));
  g_uploadBytes += std::max<size_t>(n, 1) * sizeof(double);
  ds.allocations.push_back(p);
  GDTP_HIP(hipMemset(p, 0, std::max<size_t>(n, 1) * sizeof(double)));
  return p;
}

static DevCsr UploadCsr(DeviceSystem& ds, const Csr& m) {
  DevCsr d;
  d.rows = m.rows, d.nnz = (int)m.col.size();
  d.rowptr = Upload(ds, m.rowptr);
  d.col = Upload(ds, m.col);
  d.val = Upload(ds, m.val);
  return d;
}

// An operator's boundary rows with global columns: A_BB's entries, then A_BD's (from rowMid on).
static void UploadBoundaryRows(DeviceSystem& ds, DevLevel& d, const Csr& bb, const Csr& bd, const std::vector<int>& bgi) {
  Csr m;
  std::vector<int> mid;
  m.rows = bb.rows, m.cols = bd.cols;
  m.col.reserve(bb.col.size() + bd.col.size()), m.val.reserve(m.col.capacity());
  for (int r = 0; r < bb.rows; r++) {
    for (int k = bb.rowptr[r]; k < bb.rowptr[r + 1]; k++) m.col.push_back(bgi[bb.col[k]]), m.val.push_back(bb.val[k]);
    mid.push_back((int)m.col.size());
    for (int k = bd.rowptr[r]; k < bd.rowptr[r + 1]; k++) m.col.push_back(bd.col[k]), m.val.push_back(bd.val[k]);
    m.rowptr.push_back((int)m.col.size());
  }
  d.rows = UploadCsr(ds, m);
  d.rowMid = Upload(ds, mid);
}

static std::vector<double> SoA10(const std::vector<double>& aos) {
  size_t D = aos.size() / 10;
  std::vector<double> s(aos.size());
  for (size_t d = 0; d < D; d++)
    for (int k = 0; k < 10; k++) s[k * D + d] = aos[10 * d + k];
  return s;
}

// Level-0 deep stencils in symmetric five-word form (the mixed path's FP64 residual): slot k < 4 of
// texel g holds its coupling to its lower neighbour k (k = 3(dj+1) + (di+1): (-1,-1), (0,-1),
// (+1,-1), (-1,0)), slot 4 the diagonal, SoA [5][N] over global indices.  A deep row reads its upper
// coupling k = 5..8 from slot 8-k of the upper neighbour (g+1, next-1, next, next+1); a neighbour
// that is not deep gets that slot from the deep row's own stencil.  Assembled couplings agree with
// their mirror to rounding (within 1 ulp), so this is A up to 1 ulp in some off-diagonal entries.
static std::vector<double> SymStencil(const std::vector<double>& aos, const std::vector<Line5>& lines, int N) {
  std::vector<double> s(5 * (size_t)N, 0.0);
  std::vector<char> deep(N, 0);
  const long nl = (long)lines.size();
  bool bad = false;
#pragma omp parallel for schedule(dynamic, 256) reduction(|| : bad)
  for (long r = 0; r < nl; r++) {
    const Line5& x = lines[r];
    if (x.start < 0 || x.end >= N) bad = true;
    else
      for (int g = x.start; g <= x.end; g++) deep[g] = 1;
  }
  // every (slot, texel) has one writer: a deep texel its own slots, a non-deep texel's slot 8-k the
  // deep row below it in direction k
#pragma omp parallel for schedule(dynamic, 256) reduction(|| : bad)
  for (long r = 0; r < nl; r++) {
    const Line5& x = lines[r];
    for (int i = 0; i <= x.end - x.start && !bad; i++) {
      const size_t d = (size_t)x.coeff + i;
      const int cur = x.start + i, next = x.next + i;
      if (cur + 1 >= N || next - 1 < 0 || next + 1 >= N) { bad = true; break; }
      for (int k = 0; k < 5; k++) s[k * (size_t)N + cur] = aos[10 * d + k];
      const int up[4] = {cur + 1, next - 1, next, next + 1};
      for (int k = 5; k < 9; k++)
        if (!deep[up[k - 5]]) s[(8 - k) * (size_t)N + up[k - 5]] = aos[10 * d + k];
    }
  }
  if (bad) throw std::runtime_error("deep raster line outside the level or without its upper neighbours");
  return s;
}

// bd, bgi (boundary factors; null for others): A_BD and the boundary texels, so that LdltRelaxSolve can
// form its right-hand side itself and write into a level vector.
void UploadLdlt(std::vector<void*>& ds, const Ldlt& F, DevLdlt& d, int kcap, const Csr* bd, const std::vector<int>* bgi) {
  LdltStages S;
  BuildLdltStages(F, S);
  d.n = S.n, d.wideBegin = S.wideBegin, d.kcap = kcap;
  d.stages = S.stages;
  d.perm = UploadTo(ds, S.perm), d.dinv = UploadTo(ds, S.dinv), d.compPtr = UploadTo(ds, S.compPtr);
  d.fwdPtr = UploadTo(ds, S.fwdPtr), d.fwdCol = UploadTo(ds, S.fwdCol), d.fwdVal = UploadTo(ds, S.fwdVal);
  d.bwdPtr = UploadTo(ds, S.bwdPtr), d.bwdCol = UploadTo(ds, S.bwdCol), d.bwdVal = UploadTo(ds, S.bwdVal);
  d.fwdMatPtr = UploadTo(ds, S.fwdMatPtr), d.bwdMatPtr = UploadTo(ds, S.bwdMatPtr);
  d.fwdMat = UploadTo(ds, S.fwdMat), d.bwdMat = UploadTo(ds, S.bwdMat);
  d.fwdLow = UploadTo(ds, S.fwdLow), d.bwdLow = UploadTo(ds, S.bwdLow);
  std::vector<LdltWideRow> wide(S.n - S.wideBegin);
  for (size_t c = 0; c + 1 < S.compPtr.size(); c++)
    for (int w = std::max(S.compPtr[c], S.wideBegin); w < S.compPtr[c + 1]; w++) {
      const int m = S.compPtr[c + 1] - S.compPtr[c];
      const long o = (long)(w - S.compPtr[c]) * LdltWideStride(m);
      wide[w - S.wideBegin] = {S.compPtr[c], m, {S.fwdMatPtr[c] + o, S.bwdMatPtr[c] + o}};
    }
  d.wideRows = UploadTo(ds, wide);
  if (kcap > 0 && !wide.empty())  // (one double more: a row of odd length is read in pairs)
    d.wideBuf = UploadTo(ds, std::vector<double>(2 * (size_t)kcap * wide.size() + 1, 0.0));
  if (!bd) return;
  Csr rhs;
  rhs.rows = S.n, rhs.cols = bd->cols;
  std::vector<int> texel(S.n);
  for (int w = 0; w < S.n; w++) {
    const int r = S.perm[w];
    rhs.col.insert(rhs.col.end(), bd->col.begin() + bd->rowptr[r], bd->col.begin() + bd->rowptr[r + 1]);
    rhs.val.insert(rhs.val.end(), bd->val.begin() + bd->rowptr[r], bd->val.begin() + bd->rowptr[r + 1]);
    rhs.rowptr.push_back((int)rhs.col.size());
    texel[w] = (*bgi)[r];
  }
  d.texel = UploadTo(ds, texel);
  d.rhsPtr = UploadTo(ds, rhs.rowptr), d.rhsCol = UploadTo(ds, rhs.col), d.rhsVal = UploadTo(ds, rhs.val);
}

void UploadSystem(const Hierarchy& h, const OperatorHierarchy& oh, const FineOperator& op, int kcap, DeviceSystem& ds) {
  const int nl = (int)h.levels.size();
  ds.levels = nl, ds.kcap = kcap;
  g_uploadBytes = 0;
  ds.L.assign(nl, DevLevel());
  for (int l = 0; l < nl; l++) {
    const Level& H = h.levels[l];
    const LevelOperator& O = oh.levels[l];
    DevLevel& d = ds.L[l];
    d.N = H.numTexels, d.D = H.numDeep, d.B = H.numBoundary;
    d.coef = Upload(ds, SoA10(O.deepRecip));
    d.coefRaw = Upload(ds, SoA10(O.deepRaw));
    if (l == 0) d.coefSym = Upload(ds, SymStencil(O.deepRaw, H.rasterLines, H.numTexels));
    d.bgi = Upload(ds, H.boundaryGlobalIndex);
    UploadBoundaryRows(ds, d, O.bb, O.bd, H.boundaryGlobalIndex);
    if (l + 1 < nl) d.brestr = UploadCsr(ds, H.boundaryRestriction);
    d.nTasks = (int)H.tasks.taskPtr.size() - 1;
    d.taskPtr = Upload(ds, H.tasks.taskPtr);
    {
      BandTables t;
      BuildBandTables(H.tasks, t);
      d.blockRow = Upload(ds, t.blockRow), d.bandRows = Upload(ds, t.rows);
      static_assert(sizeof(BandPair) == sizeof(int4), "a pair is loaded as four words");
      d.pairs = reinterpret_cast<int4*>(Upload(ds, t.pairs)), d.nPairs = (long)t.pairs.size();
    }
    std::vector<int> rl;
    for (auto& x : H.rasterLines) rl.insert(rl.end(), {x.start, x.end, x.prev, x.next, x.coeff});
    d.nRaster = (int)H.rasterLines.size();
    d.raster = Upload(ds, rl);
    rl.clear();
    for (auto& x : H.restrictionLines) rl.insert(rl.end(), {x.start, x.end, x.prev, x.next, x.coeff});
    d.nRestr = (int)H.restrictionLines.size();
    d.restr = Upload(ds, rl);
    rl.clear();
    for (auto& x : H.prolongationLines) rl.insert(rl.end(), {x.start, x.length, x.center, x.prev, x.next, x.aligned});
    d.nProl = (int)H.prolongationLines.size();
    d.prol = Upload(ds, rl);
    if (l + 1 < nl) UploadLdlt(ds.allocations, oh.boundaryFactor[l], d.factor, kcap, &O.bd, &H.boundaryGlobalIndex);
    else UploadLdlt(ds.allocations, oh.coarseFactor, d.factor, kcap);
    d.x = Alloc(ds, (size_t)d.N * kcap);
    d.b = Alloc(ds, (size_t)d.N * kcap);
    d.r = Alloc(ds, (size_t)d.N * kcap);
    d.y = Alloc(ds, (size_t)std::max(d.factor.n, 1) * kcap);
  }
  for (int which = 0; which < 2; which++) {
    DevLevel& d = which == 0 ? ds.mass0 : ds.stiff0;
    const DevLevel& l0 = ds.L[0];
    d.N = l0.N, d.D = l0.D, d.B = l0.B, d.bgi = l0.bgi, d.nRaster = l0.nRaster, d.raster = l0.raster;
    d.coefRaw = Upload(ds, SoA10(which == 0 ? op.deepMass : op.deepStiffness));
    d.coefSym = Upload(ds, SymStencil(which == 0 ? op.deepMass : op.deepStiffness, h.levels[0].rasterLines, l0.N));
  }
  {  // one pattern for both (an entry only one of them has: zero in the other)
    const std::vector<int>& bgi = h.levels[0].boundaryGlobalIndex;
    auto widened = [](const Csr& m, const Csr& other) {
      return m.rowptr == other.rowptr && m.col == other.col ? m : m.Combine(1.0, other, 0.0);
    };
    UploadBoundaryRows(ds, ds.mass0, widened(op.bbMass, op.bbStiffness), widened(op.bdMass, op.bdStiffness), bgi);
    const Csr bbS = widened(op.bbStiffness, op.bbMass), bdS = widened(op.bdStiffness, op.bdMass);
    std::vector<double> val;
    val.reserve(bbS.val.size() + bdS.val.size());
    for (int r = 0; r < bbS.rows; r++) {
      val.insert(val.end(), bbS.val.begin() + bbS.rowptr[r], bbS.val.begin() + bbS.rowptr[r + 1]);
      val.insert(val.end(), bdS.val.begin() + bdS.rowptr[r], bdS.val.begin() + bdS.rowptr[r + 1]);
    }
    ds.stiff0.rows = ds.mass0.rows, ds.stiff0.rowMid = ds.mass0.rowMid;
    ds.stiff0.rows.val = Upload(ds, val);
  }
  ds.bytes = g_uploadBytes;
}

// Columns in chunks of KC = min(K, 4), or one column per workgroup where a stage has so few workgroups that
// the chip is not full; a stage's launches cover all chunks.  index: of each row in src and dst; rhsX (kRhs):
// src is b, and A_BD rhsX is subtracted from it.
// (V-cycle on a 512^2 cube 570 us with chunks everywhere, 501 so; on the 4096^2 icosphere 5274, 5049; the same bits.)
static constexpr long kLdltNarrowSplit = 256, kLdltWideSplit = 2048;  // workgroups: one and eight per CU
template <bool kRhs, int KC>
static void LdltSolveChunks(DevLdlt& F, const double* src, int lds, double* dst, int ldd, const int* index, const double* rhsX, double* y, int K,
                            hipStream_t s) {
  const int n = F.n, nWide = n - F.wideBegin, last = (int)F.stages.size() - 1;
  double *buf = F.wideBuf, *top = F.wideBuf + (size_t)F.kcap * nWide;
  const LdltPass fwd{F.compPtr, F.fwdMatPtr, F.fwdMat, F.fwdLow, F.fwdPtr, F.fwdCol, F.fwdVal, index, F.dinv, F.rhsPtr, F.rhsCol, F.rhsVal, rhsX};
  const LdltPass bwd{F.compPtr, F.bwdMatPtr, F.bwdMat, F.bwdLow, F.bwdPtr, F.bwdCol, F.bwdVal, index, F.dinv, nullptr, nullptr, nullptr, nullptr};
  // launch(columns per workgroup, grid) with the workgroups of one chunk of T
  auto chunked = [&](const LdltStage& T, auto&& launch) {
    const unsigned groups = T.wide ? Blocks(T.rowEnd - T.rowBegin, 256 / kWave) : (unsigned)(T.compEnd - T.compBegin);
    if ((long)groups * K <= (T.wide ? kLdltWideSplit : kLdltNarrowSplit)) launch(std::integral_constant<int, 1>(), dim3(groups, K));
    else launch(std::integral_constant<int, KC>(), dim3(groups, (K + KC - 1) / KC));
  };
  for (int k = 0; k <= last; k++) {
    const LdltStage& T = F.stages[k];
    if (T.rowBegin == T.rowEnd) continue;
    chunked(T, [&](auto columns, dim3 grid) {
      constexpr int C = decltype(columns)::value;
      if (!T.wide) {
        // the first stage has no couplings; the next stages' rows have tens (C2 level 0: 43 on average)
        const auto kernel = k == 0 ? KLdltNarrow<true, kRhs, 8, C> : KLdltNarrow<true, kRhs, 16, C>;
        kernel<<<grid, 1024, 0, s>>>(T.compBegin, fwd, src, lds, y, n, nullptr, 0, K);
        return;
      }
      KLdltCouple<true, kRhs, C><<<grid, 256, 0, s>>>(T.rowBegin, T.rowEnd, F.wideBegin, fwd, src, lds, y, n, buf, nWide, K);
      KLdltWide<true, C><<<grid, 256, 0, s>>>(T.rowBegin, T.rowEnd, F.wideBegin, F.wideRows, fwd, buf, nWide, y, n, k == last ? top : nullptr, nullptr, 0, K);
    });
  }
  for (int k = last; k >= 0; k--) {
    const LdltStage& T = F.stages[k];
    if (T.rowBegin == T.rowEnd) continue;
    chunked(T, [&](auto columns, dim3 grid) {
      constexpr int C = decltype(columns)::value;
      if (!T.wide) {
        KLdltNarrow<false, false, 8, C><<<grid, 1024, 0, s>>>(T.compBegin, bwd, nullptr, 0, y, n, dst, ldd, K);
        return;
      }
      if (k < last) KLdltCouple<false, false, C><<<grid, 256, 0, s>>>(T.rowBegin, T.rowEnd, F.wideBegin, bwd, nullptr, 0, y, n, buf, nWide, K);
      KLdltWide<false, C><<<grid, 256, 0, s>>>(T.rowBegin, T.rowEnd, F.wideBegin, F.wideRows, bwd, k == last ? top : buf, nWide, y, n, nullptr, dst, ldd, K);
    });
  }
}

template <bool kRhs>
static void LdltSolveAny(DevLdlt& F, const double* src, int lds, double* dst, int ldd, const int* index, const double* rhsX, double* y, int K,
                         hipStream_t s) {
  if (F.n == 0) return;
  if (K < 1 || K > F.kcap) throw std::runtime_error("column count outside [1, capacity]");
  switch (std::min(K, 4)) {
    case 1: LdltSolveChunks<kRhs, 1>(F, src, lds, dst, ldd, index, rhsX, y, K, s); break;
    case 2: LdltSolveChunks<kRhs, 2>(F, src, lds, dst, ldd, index, rhsX, y, K, s); break;
    case 3: LdltSolveChunks<kRhs, 3>(F, src, lds, dst, ldd, index, rhsX, y, K, s); break;
    default: LdltSolveChunks<kRhs, 4>(F, src, lds, dst, ldd, index, rhsX, y, K, s); break;
  }
}

void LdltSolve(DevLdlt& F, const double* src, int lds, double* dst, int ldd, double* y, int K, hipStream_t s) {
  LdltSolveAny<false>(F, src, lds, dst, ldd, F.perm, nullptr, y, K, s);
}

// The boundary part of a relaxation: x_B = A_BB^-1 (b_B - A_BD x) on level vectors of stride ld
// (IterativeSolvers.inl:410-419; the forward stages form the right-hand side, deep texels are read only).
static void LdltRelaxSolve(DevLdlt& F, double* x, const double* b, int ld, double* y, int K, hipStream_t s) {
  LdltSolveAny<true>(F, b, ld, x, ld, F.texel, x, y, K, s);
}

static void CheckK(const DeviceSystem& ds, int K) {
  if (K < 1 || K > ds.kcap) throw std::runtime_error("column count outside [1, capacity]");
}

void BoundarySolveLevel(DeviceSystem& ds, int l, const double* rhs, double* sol, int K, int ld, hipStream_t s) {
  CheckK(ds, K);
  DevLevel& d = ds.L[l];
  if (l + 1 >= ds.levels) throw std::runtime_error("the coarsest level has no boundary solver");
  LdltSolve(d.factor, rhs, ld, sol, ld, d.y, K, s);
}

void CoarseSolve(DeviceSystem& ds, const double* rhs, double* sol, int K, int ld, hipStream_t s) {
  CheckK(ds, K);
  DevLevel& d = ds.L[ds.levels - 1];
  LdltSolve(d.factor, rhs, ld, sol, ld, d.y, K, s);
}

// The band sweep of a level's deep rows, columns in chunks of up to kBandColumns, every chunk a workgroup
// of its own (columns are independent).  A step's latency grows with its columns (0.5 us with one, 1.0
// with three) and each chunk reads the stencil again, so a launch takes one column per workgroup as long
// as it then has at most two workgroups per CU (us per sweep, one / three columns per workgroup, K = 3:
// 30 tasks a launch 59 / 102, 160 tasks 99 / 158, 320 tasks 346 / 274).
static constexpr long kBandSplit = 512;
static void BandSweep(DevLevel& d, double* x, const double* b, int K, int ld, hipStream_t s) {
  if (d.nTasks == 0 || d.nPairs == 0) return;
  const int chunks = (K + kBandColumns - 1) / kBandColumns;
  const int kc = (d.nTasks + 1) / 2 * (long)K <= kBandSplit ? 1 : (K + chunks - 1) / chunks;
  for (int color = 0; color < 2; color++) {
    const int tasks = color == 0 ? (d.nTasks + 1) / 2 : d.nTasks / 2;
    if (tasks == 0) continue;
    const dim3 grid(tasks, (K + kc - 1) / kc);
    const auto kernel = kc == 1 ? KBandGs<1> : kc == 2 ? KBandGs<2> : KBandGs<3>;
    kernel<<<grid, 256, 0, s>>>(color, d.nTasks, d.taskPtr, d.blockRow, d.bandRows, d.pairs, d.coef, d.D, x, b, K, ld);
  }
}

// y = A x of an operator's rows, or with `b` the residual b - A x; boundary: its boundary rows too.
static void ApplyRows(DevLevel& d, const double* x, const double* b, double* y, int K, int ld, bool boundary, hipStream_t s) {
  const int rowBlocks = boundary ? (int)Blocks((long)d.B * kRowLanes, kRowThreads) : 0;
  if (rowBlocks + d.nRaster == 0) return;
  // three columns at a time: 27 values of x in registers
  const int chunks = (K + 2) / 3, kc = (K + chunks - 1) / chunks;
  const auto kernel = kc == 1 ? KApply<1> : kc == 2 ? KApply<2> : KApply<3>;
  kernel<<<(unsigned)((long)(rowBlocks + d.nRaster) * ((K + kc - 1) / kc)), kRowThreads, 0, s>>>(rowBlocks, d.nRaster, d.B, d.bgi, d.rows.rowptr, d.rowMid, d.rows.col, d.rows.val,
                                                                                d.raster, d.coefRaw, d.D, x, b, y, K, ld);
}

void BandSweepLevel(DeviceSystem& ds, int l, double* x, const double* b, double* r, int K, int ld, hipStream_t s) {
  CheckK(ds, K);
  BandSweep(ds.L[l], x, b, K, ld, s);
  if (r) ApplyRows(ds.L[l], x, b, r, K, ld, false, s);
}

void RelaxLevel(DeviceSystem& ds, int l, double* x, const double* b, double* r, int K, int ld, bool withResidual, hipStream_t s) {
  CheckK(ds, K);
  DevLevel& d = ds.L[l];
  LdltRelaxSolve(d.factor, x, b, ld, d.y, K, s);
  BandSweep(d, x, b, K, ld, s);
  if (withResidual) ResidualLevel(ds, l, x, b, r, K, ld, s);
}

// Restriction of level l's residual; zeroC (may be null): a level l + 1 vector set to zero with it.
static void Restrict(DeviceSystem& ds, int l, const double* rF, double* bC, double* zeroC, int K, int ldF, int ldC, hipStream_t s) {
  DevLevel &f = ds.L[l], &c = ds.L[l + 1];
  const int rowBlocks = (int)Blocks((long)c.B * kRowLanes, kRowThreads);
  if (rowBlocks + c.nRestr == 0) return;
  const int chunks = (K + 2) / 3, kc = (K + chunks - 1) / chunks;
  const auto kernel = kc == 1 ? KRestrict<1> : kc == 2 ? KRestrict<2> : KRestrict<3>;
  kernel<<<dim3(rowBlocks + c.nRestr, (K + kc - 1) / kc), kRowThreads, 0, s>>>(rowBlocks, c.B, c.bgi, f.brestr.rowptr, f.brestr.col, f.brestr.val,
                                                                              c.nRestr, c.restr, rF, ldF, bC, zeroC, ldC, K);
}

void RestrictLevel(DeviceSystem& ds, int l, const double* rF, double* bC, int K, int ldF, int ldC, hipStream_t s) {
  CheckK(ds, K);
  Restrict(ds, l, rF, bC, nullptr, K, ldF, ldC, s);
}

void ProlongAddLevel(DeviceSystem& ds, int l, const double* xC, double* xF, int K, int ldC, int ldF, hipStream_t s) {
  CheckK(ds, K);
  DevLevel& f = ds.L[l];
  if (f.nProl > 0) KProlongAdd<<<f.nProl, 128, 0, s>>>(f.nProl, f.prol, xC, ldC, xF, ldF, K);
}

void ApplyLevel(DeviceSystem& ds, int l, const double* x, double* y, int K, int ld, hipStream_t s) {
  ApplyOperator(ds, ds.L[l], x, y, K, ld, s);
}

void ApplyOperator(DeviceSystem& ds, DevLevel& d, const double* x, double* y, int K, int ld, hipStream_t s) {
  CheckK(ds, K);
  ApplyRows(d, x, nullptr, y, K, ld, true, s);
}

void SquaredNorms(const double* v, int N, int K, int ld, double* dNorms, hipStream_t s) {
  KZero<<<1, 64, 0, s>>>(K, dNorms);
  KSquaredNorm<<<dim3(std::min(Blocks(N, 256), 512u), K), 256, 0, s>>>(N, v, ld, dNorms);
}

void ResidualLevel(DeviceSystem& ds, int l, const double* x, const double* b, double* r, int K, int ld, hipStream_t s) {
  CheckK(ds, K);
  ApplyRows(ds.L[l], x, b, r, K, ld, true, s);
}

void VCycleReference(DeviceSystem& ds, double* x, const double* b, int K, int ld, hipStream_t s) {
  CheckK(ds, K);
  const int nl = ds.levels;
  auto X = [&](int l) { return l == 0 ? x : ds.L[l].x; };
  auto Bv = [&](int l) { return l == 0 ? const_cast<double*>(b) : ds.L[l].b; };
  auto LD = [&](int l) { return l == 0 ? ld : ds.L[l].N; };
  for (int l = 0; l + 1 < nl; l++) {
    RelaxLevel(ds, l, X(l), Bv(l), ds.L[l].r, K, LD(l), true, s);
    // the level residual lives in r with the level's own stride
    Restrict(ds, l, ds.L[l].r, ds.L[l + 1].b, ds.L[l + 1].x, K, LD(l), ds.L[l + 1].N, s);
  }
  CoarseSolve(ds, ds.L[nl - 1].b, ds.L[nl - 1].x, K, ds.L[nl - 1].N, s);
  for (int l = nl - 2; l >= 0; l--) {
    ProlongAddLevel(ds, l, ds.L[l + 1].x, X(l), K, ds.L[l + 1].N, LD(l), s);
    RelaxLevel(ds, l, X(l), Bv(l), nullptr, K, LD(l), false, s);
  }
}

DevVectorField::~DevVectorField() {
  for (void* p : allocations) (void)hipFree(p);
}

void UploadVectorField(const VectorFieldSamples& vs, DevVectorField& d) {
  d.nCell = (long)vs.numCellSamples();
  d.nGen = (int)vs.numGeneralSamples();
  d.invCellW = vs.invCellW, d.invCellH = vs.invCellH;
  std::vector<float> soa(13 * (size_t)d.nCell);
  for (long s = 0; s < d.nCell; s++)
    for (int f = 0; f < 13; f++) soa[(size_t)f * d.nCell + s] = vs.cellData[13 * (size_t)s + f];
  d.cellCorners = UploadTo(d.allocations, vs.cellCorners);
  d.cellData = UploadTo(d.allocations, soa);
  d.genPtr = UploadTo(d.allocations, vs.genPtr), d.genTexel = UploadTo(d.allocations, vs.genTexel);
  d.genTensor = UploadTo(d.allocations, vs.genTensor), d.genG = UploadTo(d.allocations, vs.genG), d.genV = UploadTo(d.allocations, vs.genV);
}

void VectorFieldDivergence(const DevVectorField& d, const double* u, int ldu, double* rhs, int ldr, int N, int K, hipStream_t s) {
  KZeroStrided<<<(unsigned)(((long)N * K + 255) / 256), 256, 0, s>>>(N, rhs, ldr, K);
  if (d.nCell > 0)
    KVfCell<<<(unsigned)((d.nCell + 255) / 256), 256, 0, s>>>(d.nCell, d.cellCorners, d.cellData, d.invCellW, d.invCellH, u, ldu, rhs, ldr,
                                                              K);
  if (d.nGen > 0)
    KVfGeneral<<<(unsigned)((d.nGen + 255) / 256), 256, 0, s>>>(d.nGen, d.genPtr, d.genTexel, d.genG, d.genV, d.genTensor, u, ldu, rhs,
                                                                ldr, K);
}

// ------------------------------------------------------------------ modulated stiffness
// Deep texels: the four cell products weighted by the masks of the cells (i-1,j-1), (i,j-1),
// (i-1,j), (i,j), summed in that order (IterativeSolvers.inl:1184-1192).
__global__ __launch_bounds__(256) void KModulatedDeep(int D, const int* __restrict__ deepGlobal, const int* __restrict__ cells,
                                                      const double* __restrict__ coef, const double* __restrict__ mask, double* out, int N,
                                                      int K) {
  const int d = blockIdx.x * blockDim.x + threadIdx.x;
  if (d >= D) return;
  const int cp = cells[2 * d], cn = cells[2 * d + 1];
  const double m0 = mask[cp], m1 = mask[cp + 1], m2 = mask[cn], m3 = mask[cn + 1];
  const long g = deepGlobal[d];
  for (int k = 0; k < K; k++) {
    const double* c = coef + (long)k * 4 * D + 4L * d;
    out[(long)k * N + g] = c[0] * m0 + c[1] * m1 + c[2] * m2 + c[3] * m3;
  }
}

// Boundary texels: a sparse row over cells (IterativeSolvers.inl:1177-1181).
__global__ __launch_bounds__(256) void KModulatedBoundary(int B, const int* __restrict__ bGlobal, const int* __restrict__ rp,
                                                          const int* __restrict__ cell, const double* __restrict__ val, long nnz,
                                                          const double* __restrict__ mask, double* out, int N, int K) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= B) return;
  const int e0 = rp[r], e1 = rp[r + 1];
  const long g = bGlobal[r];
  for (int k = 0; k < K; k++) {
    const double* v = val + (long)k * nnz;
    double s = 0.0;
    for (int e = e0; e < e1; e++) s += v[e] * mask[cell[e]];
    out[(long)k * N + g] = s;
  }
}

DevModulation::~DevModulation() {
  for (void* p : allocations) (void)hipFree(p);
}

void UploadModulation(const Level& L0, const CellStiffnessRhs& c, DevModulation& m) {
  m.K = c.K, m.N = L0.numTexels, m.D = L0.numDeep, m.B = L0.numBoundary, m.numCells = c.numCells;
  m.nnz = (long)c.bCell.size();
  const size_t before = g_uploadBytes;
  m.deep = UploadTo(m.allocations, c.deep);
  m.deepCells = UploadTo(m.allocations, c.deepCells);
  m.deepGlobal = UploadTo(m.allocations, L0.deepGlobalIndex);
  m.bRowptr = UploadTo(m.allocations, c.bRowptr), m.bCell = UploadTo(m.allocations, c.bCell);
  m.bGlobal = UploadTo(m.allocations, L0.boundaryGlobalIndex);
  m.bVal = UploadTo(m.allocations, c.bVal);
  m.bytes = g_uploadBytes - before;
}

void ModulatedStiffness(const DevModulation& m, const double* mask, double* out, hipStream_t s) {
  if (m.D > 0)
    KModulatedDeep<<<(unsigned)((m.D + 255) / 256), 256, 0, s>>>(m.D, m.deepGlobal, m.deepCells, m.deep, mask, out, m.N, m.K);
  if (m.B > 0)
    KModulatedBoundary<<<(unsigned)((m.B + 255) / 256), 256, 0, s>>>(m.B, m.bGlobal, m.bRowptr, m.bCell, m.bVal, m.nnz, mask, out, m.N,
                                                                     m.K);
}

// ------------------------------------------------------------------ residual norms
// ||b - A x||^2 and ||b||^2 per column on level 0 without storing the residual: a fixed grid of
// kNormParts blocks strides over the raster lines (deep rows, raw stencil) and the boundary rows,
// each block writes one partial per (column, quantity), and a second pass adds the partials of a
// column in a fixed order, so repeated calls give bitwise identical norms.
// kPair: column c's operator is w.m[c] M + w.s[c] S (coef, vl: M's; coefS, vlS: S's).  Memory bounds it:
// both stencils (144 bytes a texel) once per four columns.  (3.3 M texels x 16 columns: 710 us; the two products
// written, combined and summed in passes of their own 3.2 ms.)
template <int KC>
struct PairWeights {
  double m[KC], s[KC];
};
template <int KC, bool kPair>
__global__ __launch_bounds__(256) void KResidualNormParts(int nLines, const int* __restrict__ lines, const double* __restrict__ coef, int D,
                                                          int B, const int* __restrict__ bgi, const int* __restrict__ rp,
                                                          const int* __restrict__ mid, const int* __restrict__ cl,
                                                          const double* __restrict__ vl,
                                                          const double* __restrict__ x, const double* __restrict__ b, int ld, int c0,
                                                          double* parts, const double* __restrict__ coefS, const double* __restrict__ vlS,
                                                          PairWeights<KC> w) {
  double rr[KC], bn[KC];
#pragma unroll
  for (int c = 0; c < KC; c++) rr[c] = 0.0, bn[c] = 0.0;
  for (int l = blockIdx.x; l < nLines; l += gridDim.x) {
    const int* L = lines + 5 * l;
    const int start = L[0], len = L[1] - L[0] + 1, prev = L[2], next = L[3], d0 = L[4];
    for (int i = threadIdx.x; i < len; i += blockDim.x) {
      double cf[9], cs[9];
#pragma unroll
      for (int k = 0; k < 9; k++) cf[k] = coef[(size_t)k * D + d0 + i];
      if constexpr (kPair)
#pragma unroll
        for (int k = 0; k < 9; k++) cs[k] = coefS[(size_t)k * D + d0 + i];
#pragma unroll
      for (int c = 0; c < KC; c++) {
        const double* X = x + (size_t)(c0 + c) * ld;
        if constexpr (kPair) {
          double sm = 0.0, ss = 0.0;
#pragma unroll
          for (int k = 0; k < 9; k++) {
            const double v = X[(k < 3 ? prev : k < 6 ? start : next) + i + k % 3 - 1];
            sm += v * cf[k], ss += v * cs[k];
          }
          const double t = b[(size_t)(c0 + c) * ld + start + i], r = t - w.m[c] * sm - w.s[c] * ss;
          rr[c] += r * r, bn[c] += t * t;
          continue;
        }
        const double s = X[prev + i - 1] * cf[0] + X[prev + i] * cf[1] + X[prev + i + 1] * cf[2] + X[start + i - 1] * cf[3] +
                         X[start + i] * cf[4] + X[start + i + 1] * cf[5] + X[next + i - 1] * cf[6] + X[next + i] * cf[7] +
                         X[next + i + 1] * cf[8];
        const double t = b[(size_t)(c0 + c) * ld + start + i], r = t - s;
        rr[c] += r * r, bn[c] += t * t;
      }
    }
  }
  // boundary rows: kRowLanes lanes each; lane c of a row's group adds column c's terms
  __shared__ RowTerms<KC, 256> terms;
  const int lane = threadIdx.x % kRowLanes;
  for (int i = (int)((blockIdx.x * blockDim.x + threadIdx.x) / kRowLanes); i < B; i += (int)(gridDim.x * blockDim.x / kRowLanes)) {
    const double s = RowSum(rp[i], mid[i], rp[i + 1], cl, vl, x + (size_t)c0 * ld, ld, KC, terms);
    const double bv = b[(size_t)(c0 + min(lane, KC - 1)) * ld + bgi[i]];
    double r = bv - s;
    if constexpr (kPair) {
      const double t = RowSum(rp[i], mid[i], rp[i + 1], cl, vlS, x + (size_t)c0 * ld, ld, KC, terms);
      double wm = w.m[0], ws = w.s[0];
#pragma unroll
      for (int c = 1; c < KC; c++) wm = lane == c ? w.m[c] : wm, ws = lane == c ? w.s[c] : ws;
      r = bv - wm * s - ws * t;
    }
#pragma unroll
    for (int c = 0; c < KC; c++) rr[c] += lane == c ? r * r : 0.0, bn[c] += lane == c ? bv * bv : 0.0;
  }
  __shared__ double part[2 * KC][4];
#pragma unroll
  for (int c = 0; c < KC; c++) {
    double a = rr[c], e = bn[c];
    for (int o = 32; o > 0; o >>= 1) a += __shfl_xor(a, o, 64), e += __shfl_xor(e, o, 64);
    if (threadIdx.x % 64 == 0) part[2 * c][threadIdx.x / 64] = a, part[2 * c + 1][threadIdx.x / 64] = e;
  }
  __syncthreads();
  if (threadIdx.x < 2 * KC) {
    const int c = threadIdx.x / 2, w = threadIdx.x % 2;
    const double* p = part[threadIdx.x];
    parts[((size_t)(c0 + c) * 2 + w) * gridDim.x + blockIdx.x] = (p[0] + p[1]) + (p[2] + p[3]);
  }
}

// out[q] = sum of the nParts partials of row q (q = 2 c + w), in a fixed order.
__global__ __launch_bounds__(256) void KNormPartsSum(const double* __restrict__ parts, int nParts, double* out) {
  const int q = blockIdx.x;
  double a = 0.0;
  for (int i = threadIdx.x; i < nParts; i += blockDim.x) a += parts[(size_t)q * nParts + i];
  for (int o = 32; o > 0; o >>= 1) a += __shfl_xor(a, o, 64);
  __shared__ double w[4];
  if (threadIdx.x % 64 == 0) w[threadIdx.x / 64] = a;
  __syncthreads();
  if (threadIdx.x == 0) out[q] = (w[0] + w[1]) + (w[2] + w[3]);
}

// weights (host, 2 per column: M's and S's) or null for the system's operator
template <int KC>
static void NormParts(DeviceSystem& ds, const double* x, const double* b, int c0, int ld, double* parts, const double* weights, hipStream_t s) {
  const DevLevel &d = ds.L[0], &M = ds.mass0, &S = ds.stiff0;
  PairWeights<KC> w = {};
  if (weights) {
    for (int c = 0; c < KC; c++) w.m[c] = weights[2 * (c0 + c)], w.s[c] = weights[2 * (c0 + c) + 1];
    KResidualNormParts<KC, true><<<kNormParts, 256, 0, s>>>(d.nRaster, d.raster, M.coefRaw, d.D, d.B, d.bgi, M.rows.rowptr, M.rowMid, M.rows.col,
                                                            M.rows.val, x, b, ld, c0, parts, S.coefRaw, S.rows.val, w);
  } else {
    KResidualNormParts<KC, false><<<kNormParts, 256, 0, s>>>(d.nRaster, d.raster, d.coefRaw, d.D, d.B, d.bgi, d.rows.rowptr, d.rowMid, d.rows.col,
                                                             d.rows.val, x, b, ld, c0, parts, nullptr, nullptr, w);
  }
}

void ResidualNorms(DeviceSystem& ds, const double* x, const double* b, int K, int ld, double* parts, double* out, hipStream_t s,
                   const double* weights) {
  for (int c0 = 0; c0 < K; c0 += 4) {
    switch (std::min(4, K - c0)) {
      case 4: NormParts<4>(ds, x, b, c0, ld, parts, weights, s); break;
      case 3: NormParts<3>(ds, x, b, c0, ld, parts, weights, s); break;
      case 2: NormParts<2>(ds, x, b, c0, ld, parts, weights, s); break;
      default: NormParts<1>(ds, x, b, c0, ld, parts, weights, s); break;
    }
  }
  KNormPartsSum<<<2 * K, 256, 0, s>>>(parts, kNormParts, out);
}

// ------------------------------------------------------------------ residual norms without allocation
// For callers that cannot allocate device memory: the partial sums and squared norms of
// ResidualNorms live in this file-scope array (one copy per GPU, held until the process ends).
// Host code never passes `scratch` itself to a kernel: its device address, looked up once per
// device with hipGetSymbolAddress, is kept in g_scratchAddr.  Every call on one GPU shares the
// array, so calls that overlap on one GPU race; each call overwrites every entry it reads.
static __device__ __align__(256) double scratch[NormPartsSize(kNoAllocMaxCols) + 2 * kNoAllocMaxCols];
static constexpr int kMaxDevices = 64;
static std::mutex g_scratchLock;
static double* g_scratchAddr[kMaxDevices] = {};

static double* ScratchAddress() {
  int dev = 0;
  GDTP_HIP(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices) throw std::runtime_error("device ordinal beyond the no-allocation scratch table");
  std::lock_guard<std::mutex> lock(g_scratchLock);
  if (!g_scratchAddr[dev]) {
    void* p = nullptr;
    GDTP_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    g_scratchAddr[dev] = static_cast<double*>(p);
  }
  return g_scratchAddr[dev];
}

void ResidualNormsNoAlloc(DeviceSystem& ds, const double* x, const double* b, int K, int ld, double* hostSquares, hipStream_t s) {
  if (K < 1 || K > kNoAllocMaxCols) throw std::invalid_argument("column count outside the no-allocation scratch");
  double* p = ScratchAddress();
  double* out = p + NormPartsSize(kNoAllocMaxCols);
  ResidualNorms(ds, x, b, K, ld, p, out, s);
  GDTP_HIP(hipMemcpyAsync(hostSquares, out, 2 * (size_t)K * sizeof(double), hipMemcpyDeviceToHost, s));
  GDTP_HIP(hipStreamSynchronize(s));
}

}  // namespace gdtp
