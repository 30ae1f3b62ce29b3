// Cholesky QR with regularised pivots: the pieces shared by the
// one-workgroup QR of small matrices and the wide panels of large ones.
//
// A pass takes P to P L^-T with L L^T the Cholesky factor of P^T P, and
// passes repeat until the Gram matrix a pass starts from is within 0.1 of the
// identity (that pass leaves an orthonormal Q at rounding level). A pivot at
// or below tau times its column's squared norm is replaced by that bound and
// eliminates nothing: the column (a direction the Gram matrix cannot resolve)
// keeps its components along the earlier ones, scaled up, and the next pass,
// whose Gram matrix is formed from those scaled columns, resolves it. So
// graded and numerically rank-deficient matrices need three or four passes
// instead of two and no other algorithm. A column that vanishes exactly has a
// zero row in R and any direction will do for Q: it is filled with
// pseudo-random numbers after the first pass. P - Q R stays at rounding level in every pass because P is
// solved against L, not multiplied by its inverse: 16-wide blocks by forward
// substitution, the inverse only of the diagonal blocks and corrected once by
// the residual where a block may be ill conditioned.
//
// All block products are FP64 16x16x4 MFMAs. With lr = lane % 16 and lk =
// lane / 16 the result's element v sits at (lk + 4 v, lr), which is the place
// the next product's right operand of step v is read from, so chains of
// products T_1 (T_2 (... Z)) stay in registers: a wave keeps the transpose of
// its 16 matrix rows as blocks Z_j and the triangular solve L Z = P^T needs
// no exchange between lanes. The products' index q stands for row (or column)
// qc_at(q) = 4 (q % 4) + q / 4 of a block, so that a lane's four elements of a
// block are neighbours in the matrix row: element v of Z_j is P(lr, 16 j + 4 lk
// + v). (In place order the lanes read 32 bytes of a row at a time: the panel
// kernel took 19 us at 2048 x 128, 6.4 of them for these loads and 3 for the
// stores.)
#pragma once
#include "tnx_common.h"

namespace tnx {

typedef double qc_f64x2 __attribute__((ext_vector_type(2)));
typedef double qc_f64x4 __attribute__((ext_vector_type(4)));

constexpr int kQcXLd = 17;       // row stride of the diagonal blocks' inverses
constexpr double kQcTau1 = 1e-11;  // pivot bound of the first pass ...
constexpr double kQcTau2 = 1e-12;  // ... and of the later ones
constexpr int kQcPasses = 6;

__device__ __forceinline__ qc_f64x4 qc_mfma(double a, double b, qc_f64x4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// Entry (i, c) of the filling of a zero column: even in (-1, 1), from the
// position alone (splitmix64), so the factorisation is reproducible.
__device__ __forceinline__ double qc_fill(unsigned i, unsigned c) {
  unsigned long long z = ((unsigned long long)c << 32 | i) + 0x9e3779b97f4a7c15ull;
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
  z ^= z >> 31;
  return (double)(long long)z * 0x1p-63;
}

// Lane i's value as a wave-uniform scalar; i must be wave-uniform.
__device__ __forceinline__ double qc_lane(double v, int i) {
  const long long u = __double_as_longlong(v);
  const unsigned lo = __builtin_amdgcn_readlane((int)(u & 0xffffffffll), i);
  const unsigned hi = __builtin_amdgcn_readlane((int)(u >> 32), i);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

__device__ __forceinline__ int qc_at(int q) { return 4 * (q & 3) + (q >> 2); }

// One 16-wide column block of the factorisation in one wave's registers, one
// row per lane: lanes 0..15 the diagonal block, lanes 16..31 (inv) the columns
// of the identity, which the same eliminations turn into the inverse of the
// diagonal factor, the other lanes rows below. d0: in lane j < 16 the
// column's squared norm. ill is set when a pivot falls below 1e-2 of it.
__device__ __forceinline__ void qc_chol16(double (&a)[16], double d0, double tau, bool& ill) {
  const int lane = threadIdx.x & 63;
  const bool inv = lane >= 16 && lane < 32;
  // The pivot of step j + 1 is ready after one of step j's updates, so its
  // reciprocal root overlaps the rest of them. Selects, no branches: those
  // would split the register array. (Bound by instruction issue, 270 cycles a
  // column. The multipliers through LDS instead of lane reads took as long,
  // and an LDL^T form with one root at the end 330.)
  double d, rs, mul, low = 1.0;
  auto pivot = [&](int j) {
    const double g0 = qc_lane(d0, j), x = qc_lane(a[j], j), thr = tau * g0;
    d = fmax(x, thr);
    rs = rsqrt_nr(d);
    mul = inv || x > thr ? rs : 0.0;
    low = fmin(low, fma(-1e-2, g0, x));
  };
  pivot(0);
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    a[j] = lane == j ? d * rs : a[j] * mul;
    if (j + 1 < 16) {
      a[j + 1] = fma(-a[j], qc_lane(a[j], j + 1), a[j + 1]);
      pivot(j + 1);
    }
#pragma unroll
    for (int c = j + 2; c < 16; ++c) a[c] = fma(-a[j], qc_lane(a[j], c), a[c]);
    __builtin_amdgcn_sched_barrier(0);
  }
  ill = ill || !(low > 0.0);
}

// Cholesky factor of the 16 nb x 16 nb matrix in LDS (lower triangle of G, row
// stride ld) by all NT threads: L over G's lower triangle (zeros above the
// diagonal in the diagonal blocks), the inverses of L's diagonal blocks to X
// (16 rows of stride kQcXLd each). d0: the squared column norms. All
// waves factor the diagonal block of a step (16 columns, no barrier between
// them), each with up to 32 of the rows below; NT / 2 >= 16 nb.
// Returns ill (above) for the whole workgroup.
template <int NT, int ld>
__device__ __forceinline__ bool qc_cholesky(double* G, int nb, const double* d0, double tau, double* X, int* flag) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, lr = lane & 15, lk = lane >> 4;
  constexpr int NW = NT / 64;
  bool ill = false;
  if (tid == 0) *flag = 0;
  // tile (i, j) minus the product of its rows in block column kb
  auto update = [&](int i, int j, int kb) {
    const double* Gi = G + (16 * i + lr) * ld + 16 * kb + lk;
    const double* Gj = G + (16 * j + lr) * ld + 16 * kb + lk;
    double* C = G + (16 * i + lk) * ld + 16 * j + lr;
    qc_f64x4 g;
#pragma unroll
    for (int v = 0; v < 4; ++v) g[v] = C[4 * v * ld];
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) g = qc_mfma(-Gi[4 * kk], Gj[4 * kk], g);
#pragma unroll
    for (int v = 0; v < 4; ++v) C[4 * v * ld] = g[v];
  };
  for (int kb = 0; kb < nb; ++kb) {
    const int base = 16 * kb, below = base + 16 + 32 * wave;
    const int row = lane < 16 ? base + lane : below + lane - 32;
    const bool on = lane < 16 || (lane >= 32 && row < 16 * nb);
    const int nf = max(1, (16 * (nb - kb - 1) + 31) / 32);  // waves with rows
    double a[16];
    if (wave < nf) {
      const double* src = G + (on ? row : base) * ld + base;
#pragma unroll
      for (int c = 0; c < 16; ++c) {
        const double x = src[c];
        a[c] = on ? x : (lane - 16 == c ? 1.0 : 0.0);
      }
      qc_chol16(a, lane < 16 ? d0[base + lane] : 0.0, tau, ill);
      if (lane >= 32 && on) {
#pragma unroll
        for (int c = 0; c < 16; ++c) G[row * ld + base + c] = a[c];
      }
    } else if (kb > 0) {
      // the other waves meanwhile finish the update by the block column before
      const int left = nb - kb - 1, tiles = left * (left + 1) / 2;
      for (int t = wave - nf; t < tiles; t += NW - nf) {
        int i = 0, j = t;
        while (j > i) { j -= i + 1; ++i; }
        update(kb + 1 + i, kb + 1 + j, kb - 1);
      }
    }
    __syncthreads();
    // every wave has read the diagonal block, and the updates do not
    if (wave == 0 && lane < 32) {
      double* dst = lane < 16 ? G + row * ld + base : X + base * kQcXLd + lane - 16;
      const int step = lane < 16 ? 1 : kQcXLd;
#pragma unroll
      for (int c = 0; c < 16; ++c) dst[c * step] = lane >= 16 || c <= lane ? a[c] : 0.0;
    }
    // what the next step factors: block column kb + 1
    for (int i = kb + 1 + (NW - 1 - wave); i < nb; i += NW) update(i, kb + 1, kb);
    __syncthreads();
  }
  if (ill && wave == 0 && lane == 0) *flag = 1;
  __syncthreads();
  return *flag != 0;
}

// Solves L Z = P^T for one 16-row tile of P held as blocks Z (registers, P^T
// on entry). L (row stride ld) and the diagonal inverses X in LDS or global
// memory; refine corrects every diagonal solve by its residual.
template <int NB, int ld>
__device__ __forceinline__ void qc_trsm(qc_f64x4 (&Z)[NB], int nb, const double* L, const double* X, bool refine) {
  const int lane = threadIdx.x & 63, at = qc_at(lane & 15), lk = lane >> 4;
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    if (j >= nb) break;
    const double* Lj = L + (16 * j + at) * ld + 4 * lk;
    qc_f64x4 acc = Z[j];
#pragma unroll
    for (int k = 0; k < j; ++k)
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) acc = qc_mfma(-Lj[16 * k + kk], Z[k][kk], acc);
    const double* Xj = X + (16 * j + at) * kQcXLd + 4 * lk;
    qc_f64x4 z = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) z = qc_mfma(Xj[kk], acc[kk], z);
    if (refine) {
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) acc = qc_mfma(-Lj[16 * j + kk], z[kk], acc);
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) z = qc_mfma(Xj[kk], acc[kk], z);
    }
    Z[j] = z;
    __builtin_amdgcn_sched_barrier(0);  // keeps later blocks' operand loads from piling up in registers
  }
}

// R <- L^T R for one block column w of the upper triangular R held as blocks
// R_0 .. R_w (registers, element v of R_k is R(16 k + 4 lk + v, 16 w + lr)); L
// in LDS.
template <int NB, int ld>
__device__ __forceinline__ void qc_update_r(qc_f64x4 (&R)[NB], int w, const double* L) {
  const int lane = threadIdx.x & 63, at = qc_at(lane & 15), lk = lane >> 4;
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    if (i > w) break;
    qc_f64x4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int k = i; k < NB; ++k) {
      if (k > w) break;
#pragma unroll
      for (int kk = 0; kk < 4; ++kk)
        acc = qc_mfma(L[(16 * k + 4 * lk + kk) * ld + 16 * i + at], R[k][kk], acc);
    }
    R[i] = acc;
    __builtin_amdgcn_sched_barrier(0);
  }
}

}  // namespace tnx
