// QR and the untruncated gauge moves of one-site DMRG.
//
// The reference moves the orthogonality centre with an untruncated SVD
// (tnpy/matrix_product_state.py:187-225 via tnpy/linalg.py:9-23): site <- U,
// neighbour <- (s V^T) * neighbour. Any factorisation psi = Q X with Q an
// isometry leaves the state unchanged and the site left-orthonormal; Q R is
// the cheapest. Site tensors are often rank deficient (product-like states,
// e.g. the ferromagnetic XXZ chain), so the Cholesky QR used for it (qr_chol.h;
// in LDS for small matrices, in wide panels for large ones) repeats its passes
// until Q is orthonormal. Householder QR remains for what it leaves.
//
// Layout: A is row-major m x n (m >= n). R has a non-negative diagonal.
#include "qr_chol.h"
#include "tnx_common.h"

#include <algorithm>
#include <vector>

namespace tnx {

__device__ __forceinline__ double wsum(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// Sum K per-thread values over the block; result in out[0..K-1] (LDS),
// visible to all threads on return.
template <int NT, int K>
__device__ __forceinline__ void block_reduce(const double (&v)[K], double* red, double* out) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  constexpr int NW = NT / 64;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const double t = wsum(v[k]);
    if (lane == 0) red[wv * K + k] = t;
  }
  __syncthreads();
  if ((int)threadIdx.x < K) {
    double s = 0.0;
#pragma unroll
    for (int w = 0; w < NW; ++w) s += red[w * K + threadIdx.x];
    out[threadIdx.x] = s;
  }
  __syncthreads();
}

// Panels of NB columns factored by one workgroup that holds its rows in
// registers (two block reductions per column: the column norm, then the
// reflector products with the other panel columns fused with the V^T v Gram
// entries that build the compact-WY factor T); trailing updates and the
// explicit Q are GEMMs: A_trail -= V (T^T (V^T A_trail)), Q_sub -= V (T (V^T
// Q_sub)). Factor the panel A[jb:m, jb:jb+b] (b <= NB). Writes R and the reflectors
// back to A, the explicit V (unit diagonal, zeros above) to Vall at the same
// positions, and the b x b upper-triangular T (row-major, ld NB) to Tp.
template <int NT, int RPT, int NB>
__global__ __launch_bounds__(NT) void qr_panel_kernel(double* __restrict__ A, int m, int n,
                                                     int jb, int b, double* __restrict__ Vall,
                                                     double* __restrict__ Tp) {
  __shared__ double red[(NT / 64) * NB];
  __shared__ double dots[NB];
  __shared__ double sig[1];
  __shared__ double alpha_s[1];
  __shared__ double T[NB * NB];
  const int tid = threadIdx.x;
  const int mp = m - jb;
  double P[RPT][NB];
#pragma unroll
  for (int r = 0; r < RPT; ++r) {
    const int rho = tid + NT * r;
#pragma unroll
    for (int c = 0; c < NB; ++c)
      P[r][c] = (rho < mp && c < b) ? A[(int64_t)(jb + rho) * n + jb + c] : 0.0;
  }
  for (int t = tid; t < NB * NB; t += NT) T[t] = 0.0;

  // The column loop is a runtime loop; every access to P uses a compile-time
  // column index (select on c == j) so the panel stays in registers.
  for (int j = 0; j < b; ++j) {
    // --- column norm below the diagonal, and alpha = P[j][j]
    double part[1] = {0.0};
#pragma unroll
    for (int r = 0; r < RPT; ++r) {
      const int rho = tid + NT * r;
      double pj = 0.0;
#pragma unroll
      for (int c = 0; c < NB; ++c) pj = (c == j) ? P[r][c] : pj;
      if (rho > j && rho < mp) part[0] += pj * pj;
      if (rho == j) alpha_s[0] = pj;
    }
    block_reduce<NT, 1>(part, red, sig);
    const double sigma = sig[0];
    const double alpha = alpha_s[0];
    double tau, beta, scale;
    if (sigma == 0.0) {
      tau = 0.0; beta = alpha; scale = 0.0;
    } else {
      const double nrm = sqrt(alpha * alpha + sigma);
      beta = alpha >= 0.0 ? -nrm : nrm;
      tau = (beta - alpha) / beta;
      scale = 1.0 / (alpha - beta);
    }
    // v_j: 1 at rho == j, P*scale below (kept in column j); R diag = beta
    double vj[RPT];
#pragma unroll
    for (int r = 0; r < RPT; ++r) {
      const int rho = tid + NT * r;
      const bool below = rho > j && rho < mp;
      double pj = 0.0;
#pragma unroll
      for (int c = 0; c < NB; ++c) pj = (c == j) ? P[r][c] : pj;
      vj[r] = below ? pj * scale : (rho == j ? 1.0 : 0.0);
#pragma unroll
      for (int c = 0; c < NB; ++c)
        if (c == j) P[r][c] = below ? vj[r] : (rho == j ? beta : P[r][c]);
    }
    // --- one reduction: c > j: v_j . P[:, c] (reflector application);
    //     c < j: v_j . v_c (Gram entries for T). Below the diagonal of a
    //     column c < j, P[.][c] holds v_c, and rho >= j > c covers the
    //     whole support of v_j.
    {
      // streamed: one wave reduction per column keeps a single partial live
      const int lane = tid & 63, wv = tid >> 6;
#pragma unroll
      for (int c = 0; c < NB; ++c) {
        double pd = 0.0;
#pragma unroll
        for (int r = 0; r < RPT; ++r) {
          const int rho = tid + NT * r;
          if (c != j && c < b && rho >= j && rho < mp) pd += vj[r] * P[r][c];
        }
        pd = wsum(pd);
        if (lane == 0) red[wv * NB + c] = pd;
      }
      __syncthreads();
      if (tid < NB) {
        double acc = 0.0;
#pragma unroll
        for (int w = 0; w < NT / 64; ++w) acc += red[w * NB + tid];
        dots[tid] = acc;
      }
      __syncthreads();
    }
    if (tau != 0.0) {
#pragma unroll
      for (int c = 0; c < NB; ++c) {
        if (c > j && c < b) {
          const double f = tau * dots[c];
#pragma unroll
          for (int r = 0; r < RPT; ++r) {
            const int rho = tid + NT * r;
            if (rho >= j && rho < mp) P[r][c] -= f * vj[r];
          }
        }
      }
    }
    // T[0:j, j] = -tau T[0:j, 0:j] y,  y_i = v_i . v_j ;  T[j][j] = tau
    if (tid == 0) {
      for (int i = 0; i < j; ++i) {
        double acc = 0.0;
        for (int l = i; l < j; ++l) acc += T[i * NB + l] * dots[l];
        T[i * NB + j] = -tau * acc;
      }
      T[j * NB + j] = tau;
    }
    __syncthreads();
  }
  // write back R / reflectors, explicit V, and T
#pragma unroll
  for (int r = 0; r < RPT; ++r) {
    const int rho = tid + NT * r;
    if (rho < mp) {
#pragma unroll
      for (int c = 0; c < NB; ++c) {
        if (c < b) {
          const int64_t off = (int64_t)(jb + rho) * n + jb + c;
          A[off] = P[r][c];
          Vall[off] = rho < c ? 0.0 : (rho == c ? 1.0 : P[r][c]);
        }
      }
    }
  }
  for (int t = tid; t < NB * NB; t += NT) Tp[t] = T[t];
}

// R[i][c] = A[i][c] for c >= i, else 0   (n x n, row-major)
__global__ void extract_r_kernel(const double* A, int n, double* R) {
  const int64_t nn = (int64_t)n * n;
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < nn;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t i = e / n, c = e % n;
    R[e] = c >= i ? A[i * n + c] : 0.0;
  }
}

// A (m x n) <- [I_n ; 0]
__global__ void eye_kernel(double* A, int m, int n) {
  const int64_t mn = (int64_t)m * n;
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < mn;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t i = e / n, c = e % n;
    A[e] = (i == c) ? 1.0 : 0.0;
  }
}

// Sign convention of every QR here: R with a non-negative diagonal (a
// column j with R_jj < 0 flips column j of Q and row j of R), so every path
// returns the same factorisation of a full-rank matrix.
__global__ void qr_signs_kernel(const double* __restrict__ R, int n, double* __restrict__ sg) {
  for (int j = blockIdx.x * blockDim.x + threadIdx.x; j < n; j += gridDim.x * blockDim.x)
    sg[j] = R[(int64_t)j * n + j] < 0.0 ? -1.0 : 1.0;
}

__global__ void qr_apply_signs_kernel(double* __restrict__ Q, int m, double* __restrict__ R, int n,
                                      const double* __restrict__ sg) {
  const int64_t mn = (int64_t)m * n, nn = (int64_t)n * n;
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < mn + nn;
       e += (int64_t)gridDim.x * blockDim.x) {
    if (e < mn) {
      Q[e] *= sg[e % n];
    } else {
      const int64_t f = e - mn;
      R[f] *= sg[f / n];
    }
  }
}

static int qr_fix_signs(double* Q, int m, double* R, int n, double* sg, hipStream_t s) {
  hipLaunchKernelGGL(qr_signs_kernel, dim3((n + 255) / 256), dim3(256), 0, s, R, n, sg);
  TNX_LAUNCH_CHECK();
  const int64_t tot = (int64_t)m * n + (int64_t)n * n;
  const int nb = (int)std::min<int64_t>((tot + 255) / 256, 8192);
  hipLaunchKernelGGL(qr_apply_signs_kernel, dim3(nb), dim3(256), 0, s, Q, m, R, n, sg);
  TNX_LAUNCH_CHECK();
  return TNX_OK;
}

struct QrCfg { int nt, rpt, nb; };

static bool qr_config(int m, QrCfg* c) {
  if (m <= 512) { *c = {512, 1, 16}; return true; }
  if (m <= 1024) { *c = {512, 2, 16}; return true; }
  if (m <= 2048) { *c = {512, 4, 16}; return true; }
  if (m <= 4096) { *c = {1024, 4, 8}; return true; }
  if (m <= 8192) { *c = {1024, 8, 4}; return true; }
  return false;
}

static size_t al(size_t x) { return (x + 255) & ~(size_t)255; }

template <int NT>
__device__ __forceinline__ double block_sum(double v, double* red) {
  constexpr int NW = NT / 64;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  v = wsum(v);
  __syncthreads();
  if (lane == 0) red[wv] = v;
  __syncthreads();
  double t = 0.0;
#pragma unroll
  for (int w = 0; w < NW; ++w) t += red[w];
  return t;
}

// Householder QR of the m x n (m >= n) matrix held in LDS (row stride ld):
// R on and above the diagonal, the reflector tails below it, tau_s[j].
template <int NT>
__device__ void lds_householder(double* S, int ld, int m, int n, double* tau_s, double* red) {
  constexpr int NW = NT / 64;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int j = 0; j < n; ++j) {
    double part = 0.0;
    for (int i = j + 1 + tid; i < m; i += NT) part += S[i * ld + j] * S[i * ld + j];
    const double sigma = block_sum<NT>(part, red);
    const double alpha = S[j * ld + j];
    double tj = 0.0, beta = alpha, scale = 0.0;
    if (sigma != 0.0) {
      const double nrm = sqrt(alpha * alpha + sigma);
      beta = alpha >= 0.0 ? -nrm : nrm;
      tj = (beta - alpha) / beta;
      scale = 1.0 / (alpha - beta);
    }
    __syncthreads();
    for (int i = j + 1 + tid; i < m; i += NT) S[i * ld + j] *= scale;
    if (tid == 0) { S[j * ld + j] = beta; tau_s[j] = tj; }
    __syncthreads();
    if (tj != 0.0) {
      for (int c = j + 1 + wave; c < n; c += NW) {
        double acc = 0.0;
        for (int i = j + lane; i < m; i += 64) acc += (i == j ? 1.0 : S[i * ld + j]) * S[i * ld + c];
        const double w = tj * wsum(acc);
        for (int i = j + lane; i < m; i += 64) S[i * ld + c] -= (i == j ? 1.0 : S[i * ld + j]) * w;
      }
    }
    __syncthreads();
  }
}

static size_t householder_ws_bytes(int m, int n) {
  QrCfg c;
  if (!qr_config(m, &c)) c = {1024, 8, 4};
  const int np = (n + c.nb - 1) / c.nb;
  size_t b = al((size_t)m * n * 8);                 // Vall
  b += al((size_t)np * c.nb * c.nb * 8);            // T factors
  b += 2 * al((size_t)c.nb * n * 8);                // W, W2
  b += al((size_t)32 * c.nb * 8);                   // split-K partials of one-column products
  b += al((size_t)n * 8);                           // R diagonal signs
  return b + 256;
}

static int launch_panel(const QrCfg& c, double* A, int m, int n, int jb, int b, double* Vall,
                        double* Tp, hipStream_t s) {
#define TNX_PANEL(NT_, RPT_, NB_)                                                        \
  if (c.nt == NT_ && c.rpt == RPT_ && c.nb == NB_) {                                     \
    hipLaunchKernelGGL((qr_panel_kernel<NT_, RPT_, NB_>), dim3(1), dim3(NT_), 0, s, A, m, n, \
                       jb, b, Vall, Tp);                                                 \
    TNX_LAUNCH_CHECK();                                                                  \
    return TNX_OK;                                                                       \
  }
  TNX_PANEL(512, 1, 16)
  TNX_PANEL(512, 2, 16)
  TNX_PANEL(512, 4, 16)
  TNX_PANEL(1024, 4, 8)
  TNX_PANEL(1024, 8, 4)
#undef TNX_PANEL
  set_error("qr: no panel configuration");
  return TNX_ERR_UNSUPPORTED;
}

// Householder QR with one-workgroup panels: only for what the Cholesky QR
// below leaves (numbers whose squares leave the range).
static int qr_householder(double* A, int m, int n, double* R, void* ws, hipStream_t s) {
  QrCfg c;
  if (!qr_config(m, &c)) {
    set_error("qr: m=%d rows exceeds the supported 8192", m);
    return TNX_ERR_UNSUPPORTED;
  }
  const int NB = c.nb;
  const int np = (n + NB - 1) / NB;
  char* p = (char*)(((uintptr_t)ws + 255) & ~(uintptr_t)255);
  double* Vall = (double*)p; p += al((size_t)m * n * 8);
  double* Tall = (double*)p; p += al((size_t)np * NB * NB * 8);
  double* Wb = (double*)p; p += al((size_t)NB * n * 8);
  double* W2 = (double*)p; p += al((size_t)NB * n * 8);
  double* part = (double*)p; p += al((size_t)32 * NB * 8);
  double* sg = (double*)p;
  const size_t part_bytes = al((size_t)32 * NB * 8);

  // ---- factorisation
  for (int pi = 0; pi < np; ++pi) {
    const int jb = pi * NB;
    const int b = std::min(NB, n - jb);
    const int mp = m - jb;
    double* Tp = Tall + (size_t)pi * NB * NB;
    TNX_TRY(launch_panel(c, A, m, n, jb, b, Vall, Tp, s));
    const int nt = n - jb - b;
    if (nt <= 0) continue;
    const double* Vp = Vall + (size_t)jb * n + jb;
    double* At = A + (size_t)jb * n + jb + b;
    // W = V^T A_trail   (b x nt)
    GemmDesc g{};
    g.M = b; g.N = nt; g.K = mp; g.batch = 1;
    g.A = Vp; g.ta = DT::F64; g.lda = n; g.sA = 0; g.a_kcontig = false;
    g.B = At; g.tb = DT::F64; g.ldb = n; g.sB = 0; g.b_ncontig = true;
    g.C = Wb; g.tc = DT::F64; g.ldc = nt; g.sC = 0;
    g.alpha = 1.0; g.beta = 0.0; g.prec = Prec::F64;
    g.splitk_ws = part; g.splitk_ws_bytes = part_bytes;
    TNX_TRY(gemm(g, s));
    // W2 = T^T W
    GemmDesc g2{};
    g2.M = b; g2.N = nt; g2.K = b; g2.batch = 1;
    g2.A = Tp; g2.ta = DT::F64; g2.lda = NB; g2.sA = 0; g2.a_kcontig = false;
    g2.B = Wb; g2.tb = DT::F64; g2.ldb = nt; g2.sB = 0; g2.b_ncontig = true;
    g2.C = W2; g2.tc = DT::F64; g2.ldc = nt; g2.sC = 0;
    g2.alpha = 1.0; g2.beta = 0.0; g2.prec = Prec::F64;
    TNX_TRY(gemm(g2, s));
    // A_trail -= V W2
    GemmDesc g3{};
    g3.M = mp; g3.N = nt; g3.K = b; g3.batch = 1;
    g3.A = Vp; g3.ta = DT::F64; g3.lda = n; g3.sA = 0; g3.a_kcontig = true;
    g3.B = W2; g3.tb = DT::F64; g3.ldb = nt; g3.sB = 0; g3.b_ncontig = true;
    g3.C = At; g3.tc = DT::F64; g3.ldc = n; g3.sC = 0;
    g3.alpha = -1.0; g3.beta = 1.0; g3.prec = Prec::F64;
    TNX_TRY(gemm(g3, s));
  }
  // ---- R, then Q = H_0 ... H_{np-1} [I; 0] accumulated backwards into A
  {
    const int64_t nn = (int64_t)n * n;
    const int blocks = (int)std::min<int64_t>((nn + 255) / 256, 4096);
    hipLaunchKernelGGL(extract_r_kernel, dim3(blocks), dim3(256), 0, s, A, n, R);
    TNX_LAUNCH_CHECK();
    const int64_t mn = (int64_t)m * n;
    const int b2 = (int)std::min<int64_t>((mn + 255) / 256, 4096);
    hipLaunchKernelGGL(eye_kernel, dim3(b2), dim3(256), 0, s, A, m, n);
    TNX_LAUNCH_CHECK();
  }
  for (int pi = np - 1; pi >= 0; --pi) {
    const int jb = pi * NB;
    const int b = std::min(NB, n - jb);
    const int mp = m - jb;
    const int nq = n - jb;
    const double* Tp = Tall + (size_t)pi * NB * NB;
    const double* Vp = Vall + (size_t)jb * n + jb;
    double* Qs = A + (size_t)jb * n + jb;
    GemmDesc g{};
    g.M = b; g.N = nq; g.K = mp; g.batch = 1;
    g.A = Vp; g.ta = DT::F64; g.lda = n; g.sA = 0; g.a_kcontig = false;
    g.B = Qs; g.tb = DT::F64; g.ldb = n; g.sB = 0; g.b_ncontig = true;
    g.C = Wb; g.tc = DT::F64; g.ldc = nq; g.sC = 0;
    g.alpha = 1.0; g.beta = 0.0; g.prec = Prec::F64;
    g.splitk_ws = part; g.splitk_ws_bytes = part_bytes;
    TNX_TRY(gemm(g, s));
    GemmDesc g2{};
    g2.M = b; g2.N = nq; g2.K = b; g2.batch = 1;
    g2.A = Tp; g2.ta = DT::F64; g2.lda = NB; g2.sA = 0; g2.a_kcontig = true;
    g2.B = Wb; g2.tb = DT::F64; g2.ldb = nq; g2.sB = 0; g2.b_ncontig = true;
    g2.C = W2; g2.tc = DT::F64; g2.ldc = nq; g2.sC = 0;
    g2.alpha = 1.0; g2.beta = 0.0; g2.prec = Prec::F64;
    TNX_TRY(gemm(g2, s));
    GemmDesc g3{};
    g3.M = mp; g3.N = nq; g3.K = b; g3.batch = 1;
    g3.A = Vp; g3.ta = DT::F64; g3.lda = n; g3.sA = 0; g3.a_kcontig = true;
    g3.B = W2; g3.tb = DT::F64; g3.ldb = nq; g3.sB = 0; g3.b_ncontig = true;
    g3.C = Qs; g3.tc = DT::F64; g3.ldc = n; g3.sC = 0;
    g3.alpha = -1.0; g3.beta = 1.0; g3.prec = Prec::F64;
    TNX_TRY(gemm(g3, s));
  }
  return qr_fix_signs(A, m, R, n, sg, s);
}

// ---- QR in LDS -----------------------------------------------------------------
// Householder QR of `batch` small m x n matrices (m >= n), one workgroup per
// matrix held in LDS (row stride n + 1). trans = 0: matrix p is A_p, m x n
// row-major. trans = 1: matrix p is A_p^T, where A_p is n x m row-major (the
// leftward gauge move: A = (Q R)^T). On exit A_p holds the thin Q (Q^T when
// trans) and R_p = R (n x n, upper triangular). Same reflector convention as
// the blocked path (beta = -sign(alpha) |x|).
constexpr int kQrSmallBig = 16640;   // m * (n + 1) doubles: 130 KiB of LDS

// Householder QR of the matrix at A (trans as above) by the whole workgroup
// in the LDS buffer S (m (n + 1) + 2 n + 16 doubles).
template <int NT>
__device__ void qr_lds_householder(double* __restrict__ A, int m, int n, int trans, double* __restrict__ R,
                                   double* S) {
  constexpr int NW = NT / 64;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int ld = n + 1, mn = m * n;
  double* tau_s = S + m * ld;
  double* sgn = tau_s + n;
  double* red = sgn + n;
  for (int e = tid; e < mn; e += NT) {
    int i, c;
    if (trans) { c = e / m; i = e - c * m; } else { i = e / n; c = e - i * n; }
    S[i * ld + c] = A[e];
  }
  __syncthreads();
  lds_householder<NT>(S, ld, m, n, tau_s, red);
  // ---- R, with a non-negative diagonal (same convention as the blocked QR)
  for (int j = tid; j < n; j += NT) sgn[j] = S[j * ld + j] < 0.0 ? -1.0 : 1.0;
  __syncthreads();
  for (int e = tid; e < n * n; e += NT) {
    const int i = e / n, c = e - i * n;
    R[e] = (c >= i) ? sgn[i] * S[i * ld + c] : 0.0;
  }
  __syncthreads();
  // ---- thin Q = H_0 ... H_{n-1} [I; 0], formed in place from the last column
  for (int j = n - 1; j >= 0; --j) {
    const double tj = tau_s[j];
    if (tj != 0.0) {
      for (int c = j + 1 + wave; c < n; c += NW) {
        double acc = 0.0;
        for (int i = j + lane; i < m; i += 64) acc += (i == j ? 1.0 : S[i * ld + j]) * S[i * ld + c];
        const double w = tj * wsum(acc);
        for (int i = j + lane; i < m; i += 64) S[i * ld + c] -= (i == j ? 1.0 : S[i * ld + j]) * w;
      }
    }
    __syncthreads();
    for (int i = tid; i < m; i += NT)
      S[i * ld + j] = (i < j) ? 0.0 : (i == j ? 1.0 - tj : -tj * S[i * ld + j]);
    __syncthreads();
  }
  for (int e = tid; e < mn; e += NT) {
    int i, c;
    if (trans) { c = e / m; i = e - c * m; } else { i = e / n; c = e - i * n; }
    A[e] = sgn[c] * S[i * ld + c];
  }
}

__global__ __launch_bounds__(256) void qr_small_kernel(double* __restrict__ A, int m, int n, int trans,
                                                       double* __restrict__ R) {
  __shared__ double S[kQrSmallBig + 2 * 256 + 16];
  qr_lds_householder<256>(A + (int64_t)blockIdx.x * m * n, m, n, trans, R + (int64_t)blockIdx.x * n * n, S);
}

// The same factorisation by Cholesky QR (qr_chol.h), where the matrix, its
// Gram matrix and the diagonal inverses fit in LDS together (up to about
// 144 x 72): two to four passes of Gram, Cholesky and triangular solve on the
// matrix cores instead of a chain of 2 n column steps with a block reduction
// each. A matrix whose Gram matrix leaves the range of the numbers is read again
// and takes the Householder steps. R's block column w stays in
// wave w's registers. Bound by the chain of pivots (16 n per pass) and one
// CU's matrix rate. The gauge move of a 60 x 2 x 60 site, with R times the
// neighbour: 162 us with two panels of a many-workgroup path, 54 us so (49 in
// this kernel); 16 sites of 64 x 2 x 64 took 683 us in the Householder kernel
// above, 66 here.
constexpr int kQcLdsBig = 20200, kQcLdsLittle = 4864;  // 158 and 38 KiB

template <int CAP, int NT, int NB>
__global__ __launch_bounds__(NT) void qr_chol_kernel(double* __restrict__ A, int m, int n, int trans,
                                                     double* __restrict__ R) {
  __shared__ double S[CAP];
  __shared__ int flag[3];
  __shared__ unsigned zero[3];  // the columns that vanish, a bit each
  constexpr int NW = NT / 64;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, lr = lane & 15, lk = lane >> 4;
  constexpr int nb = NB, ld = 16 * NB + 1;
  const int mt = (m + 15) / 16;
  double* G = S + 16 * mt * ld;
  double* X = G + 16 * nb * ld;
  double* d0 = X + 16 * nb * kQcXLd;
  double* Ap = A + (int64_t)blockIdx.x * m * n;
  double* Rp = R + (int64_t)blockIdx.x * n * n;
  for (int e = tid; e < 16 * mt * ld; e += NT) S[e] = 0.0;
  if (tid < 3) zero[tid] = 0;
  __syncthreads();
  if (trans) {
    for (int c = wave; c < n; c += NW)
#pragma unroll 4
      for (int i = lane; i < m; i += 64) S[i * ld + c] = Ap[c * m + i];
  } else {
#pragma unroll 4
    for (int i = wave; i < m; i += NW)
      for (int c = lane; c < n; c += 64) S[i * ld + c] = Ap[i * n + c];
  }
  qc_f64x4 Rb[NB];
  bool done = false;
  for (int p = 0; p < kQcPasses && !done; ++p) {
    if (tid < 2) flag[tid] = 0;
    __syncthreads();
    // ---- Gram matrix, lower 16 x 16 tiles; identity in the padding
    bool far = false, bad = false;
    for (int t = wave; t < nb * (nb + 1) / 2; t += NW) {
      int bi = 0, bj = t;
      while (bj > bi) { bj -= bi + 1; ++bi; }
      const double* Si = S + lk * ld + 16 * bi + lr;
      const double* Sj = S + lk * ld + 16 * bj + lr;
      qc_f64x4 g = {0.0, 0.0, 0.0, 0.0}, h = g;
      for (int k = 0; k < 16 * mt; k += 16) {
        g = qc_mfma(Si[k * ld], Sj[k * ld], g);
        h = qc_mfma(Si[(k + 4) * ld], Sj[(k + 4) * ld], h);
        g = qc_mfma(Si[(k + 8) * ld], Sj[(k + 8) * ld], g);
        h = qc_mfma(Si[(k + 12) * ld], Sj[(k + 12) * ld], h);
      }
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int i = 16 * bi + lk + 4 * v, c = 16 * bj + lr;
        double x = g[v] + h[v];
        if (i == c) {
          if (i >= n) x = 1.0;
          if (p == 0 && x == 0.0) {
            atomicOr(&zero[i >> 5], 1u << (i & 31));
            x = 1.0;
          }
          d0[i] = x;
          bad = bad || !(x > 1e-290 && x < 1e290);
        }
        if (c <= i) far = far || !(fabs(x - (i == c ? 1.0 : 0.0)) <= 0.1);
        G[i * ld + c] = x;
      }
    }
    if (far) flag[0] = 1;
    if (bad) flag[1] = 1;
    __syncthreads();
    done = p > 0 && flag[0] == 0;
    if (flag[1]) break;
    const bool ill = qc_cholesky<NT, ld>(G, NB, d0, p == 0 ? kQcTau1 : kQcTau2, X, &flag[2]);
    if (wave < nb) {
      if (p == 0) {
#pragma unroll
        for (int k = 0; k < NB; ++k)
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const int i = 16 * k + 4 * lk + v;
            const bool on = k <= wave && !(zero[i >> 5] >> (i & 31) & 1);
            Rb[k][v] = on ? G[(16 * wave + lr) * ld + i] : 0.0;
          }
      } else {
        qc_update_r<NB, ld>(Rb, wave, G);
      }
    }
    for (int t = wave; t < mt; t += NW) {
      double* St = S + (16 * t + lr) * ld + 4 * lk;
      qc_f64x4 Z[NB];
#pragma unroll
      for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v) Z[j][v] = St[16 * j + v];
      qc_trsm<NB, ld>(Z, NB, G, X, ill);
#pragma unroll
      for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v) St[16 * j + v] = Z[j][v];
    }
    __syncthreads();
    if (p == 0 && (zero[0] | zero[1] | zero[2])) {
      for (int c = wave; c < n; c += NW)
        if (zero[c >> 5] >> (c & 31) & 1)
          for (int i = lane; i < m; i += 64) S[i * ld + c] = qc_fill(i, c);
      __syncthreads();
    }
  }
  if (!done) {
    qr_lds_householder<NT>(Ap, m, n, trans, Rp, S);
    return;
  }
  if (wave < nb) {
    const int c = 16 * wave + lr;
#pragma unroll
    for (int k = 0; k < NB; ++k)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int i = 16 * k + 4 * lk + v;
        if (i < n && c < n) Rp[i * n + c] = Rb[k][v];
      }
  }
  if (trans) {
    for (int c = wave; c < n; c += NW)
#pragma unroll 4
      for (int i = lane; i < m; i += 64) Ap[c * m + i] = S[i * ld + c];
  } else {
#pragma unroll 4
    for (int i = wave; i < m; i += NW)
      for (int c = lane; c < n; c += 64) Ap[i * n + c] = S[i * ld + c];
  }
}

static int64_t qr_chol_need(int m, int n) {
  const int64_t m16 = (m + 15) / 16 * 16, n16 = (n + 15) / 16 * 16;
  return (m16 + n16) * (n16 + 1) + (kQcXLd + 1) * n16;
}

static bool qr_chol_fits(int m, int n) { return m >= n && n >= 1 && n <= 80 && qr_chol_need(m, n) <= kQcLdsBig; }

static int qr_chol(double* A, int m, int n, int trans, double* R, int batch, hipStream_t s) {
  const int nb = (n + 15) / 16;
  // the little form (four waves) leaves room for several matrices on a CU
  const bool little = nb <= 3 && qr_chol_need(m, n) <= kQcLdsLittle;
#define TNX_QRC(NB_, CAP_, NT_)                                                                               \
  case NB_:                                                                                                   \
    hipLaunchKernelGGL((qr_chol_kernel<CAP_, NT_, NB_>), dim3(batch), dim3(NT_), 0, s, A, m, n, trans, R);    \
    break;
  if (little) {
    switch (nb) {
      TNX_QRC(1, kQcLdsLittle, 256)
      TNX_QRC(2, kQcLdsLittle, 256)
      TNX_QRC(3, kQcLdsLittle, 256)
    }
  } else {
    switch (nb) {
      TNX_QRC(1, kQcLdsBig, 512)
      TNX_QRC(2, kQcLdsBig, 512)
      TNX_QRC(3, kQcLdsBig, 512)
      TNX_QRC(4, kQcLdsBig, 512)
      TNX_QRC(5, kQcLdsBig, 512)
    }
  }
#undef TNX_QRC
  TNX_LAUNCH_CHECK();
  return TNX_OK;
}

static bool qr_small_fits(int m, int n) {
  return m >= n && n >= 1 && n <= 256 && (int64_t)m * (n + 1) <= kQrSmallBig;
}

static int qr_small_b(double* A, int m, int n, int trans, double* R, int batch, hipStream_t s) {
  TNX_CHECK_ARG(qr_small_fits(m, n), "qr_batched: %d x %d exceeds the LDS-resident limit", m, n);
  TNX_CHECK_ARG(batch >= 1 && batch <= 2147483647, "qr_batched: bad batch %d", batch);
  if (qr_chol_fits(m, n)) return qr_chol(A, m, n, trans, R, batch, s);
  hipLaunchKernelGGL(qr_small_kernel, dim3(batch), dim3(256), 0, s, A, m, n, trans, R);
  TNX_LAUNCH_CHECK();
  return TNX_OK;
}

// ---- Cholesky QR in wide panels ----------------------------------------------------
// Larger matrices in panels of up to kWpW columns, by block Gram-Schmidt with
// reorthogonalisation, every factor a Cholesky factor as in qr_chol.h. Panel
// P (columns j0 .. j0 + w of A, already reduced by the panels before):
//   pass 0:   G = P^T P, P <- P L^-T;
//   pass 1:   [C; G] = [Q_<  P]^T P, P <- (P - Q_< C) L^-T,
//             R_<p += C R_p, R_p <- L^T R_p;
//   pass 2, 3: the same again, needed while the pass before has started from
//             |G - I| > 0.1 or |C| > kWpFar (below it the C^T C that G leaves
//             out is at rounding level: its n terms are squares of entries
//             that are well below the largest);
//   then R_p,> = P^T A_> and A_> -= P R_p,> for the columns behind.
// Q replaces A in place and needs no backward formation, so a panel costs one
// workgroup's 128-wide factorisation (wp_factor) and GEMMs, where 32-wide
// Householder panels took four of everything and rebuilt their reflectors.
// Well-conditioned panels take two passes, graded and rank-deficient ones
// three or four (zero columns included, see qc_fill). The host queues two, and
// from the saved copy all four where a panel has asked for them; a panel then
// leaves out on the device what it does not need, for 4.5 us a launch (280 us
// at n = 1024, why they are not queued at once). What does not converge in four
// (numbers out of the Gram matrix's range) is factored by Householder panels.
constexpr int kWpW = 128, kWpNB = kWpW / 16, kWpLd = kWpW + 1;
constexpr int kWpPasses = 4;
constexpr double kWpFar = 2e-9;
// flags of a panel: [p] pass p is needed (p = 2, 3), [kWpPasses] it did not
// converge, [kWpIll] the current factor's ill, [kWpZero ..] zero columns
constexpr int kWpIll = 6, kWpZero = 8, kWpFlags = 16;

struct WpBuf {
  double* S;      // n x kWpW: [C; G] of the current pass
  double* L;      // kWpW x kWpW: its Cholesky factor
  double* X;      // the inverses of L's diagonal blocks
  double* Rp[2];  // R_p before and after a pass
  int* flags;     // kWpFlags of the current panel
};

// The Cholesky factor of a pass, by one workgroup. Close to the identity it is
// I + Phi(E), the lower half of E = G - I with half its diagonal, up to E^2.
__global__ __launch_bounds__(512) void wp_factor_kernel(WpBuf b, int j0, int w, int p) {
  __shared__ double G[kWpW * kWpLd];
  __shared__ double X[kWpW * kQcXLd];
  __shared__ double d0[kWpW];
  __shared__ int sh[3];  // far from I, not close to I, out of range
  __shared__ int flag;
  __shared__ unsigned zero[4];
  if (p >= 2 && b.flags[p] == 0) return;
  const int tid = threadIdx.x;
  if (tid < 3) sh[tid] = 0;
  if (tid < 4) zero[tid] = 0;
  __syncthreads();
  bool far = false, wide = false, bad = false;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    double v[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      const int e = tid + 512 * (16 * h + u), i = e >> 7, c = e & 127;
      const double x = b.S[(size_t)(j0 + min(i, w - 1)) * kWpW + c];
      v[u] = i < w && c <= i ? x : (i == c ? 1.0 : 0.0);
    }
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      const int e = tid + 512 * (16 * h + u), i = e >> 7, c = e & 127;
      const double off = fabs(v[u] - (i == c ? 1.0 : 0.0));
      far = far || !(off <= 0.1);
      wide = wide || !(off <= 1e-9);
      G[i * kWpLd + c] = v[u];
    }
  }
  __syncthreads();
  if (tid < kWpW) {
    double x = G[tid * kWpLd + tid];
    if (p == 0 && x == 0.0) {
      atomicOr(&zero[tid >> 5], 1u << (tid & 31));
      x = G[tid * kWpLd + tid] = 1.0;
    }
    d0[tid] = x;
    bad = !(x > 1e-290 && x < 1e290);
  }
  if (far) sh[0] = 1;
  if (wide) sh[1] = 1;
  if (bad) sh[2] = 1;
  __syncthreads();
  if (p == 0 && tid < 4) b.flags[kWpZero + tid] = (int)zero[tid];
  if (tid == 0) {
    if (sh[2]) b.flags[kWpPasses] = 1;
    if (p >= 1 && sh[0]) b.flags[p + 1] = 1;
  }
  const int nb = (w + 15) / 16;
  bool ill = false;
  if (p >= 1 && !sh[1]) {
    for (int e = tid; e < kWpW * 16; e += 512) {
      const int i = e >> 4, c = e & 15, gc = (i & ~15) + c;
      const double x = G[i * kWpLd + gc];
      X[i * kQcXLd + c] = gc < i ? -x : (gc == i ? 1.5 - 0.5 * x : 0.0);
    }
    __syncthreads();
    if (tid < kWpW) G[tid * kWpLd + tid] = 0.5 + 0.5 * G[tid * kWpLd + tid];
    __syncthreads();
  } else {
    ill = qc_cholesky<512, kWpLd>(G, nb, d0, p == 0 ? kQcTau1 : kQcTau2, X, &flag);
  }
  if (tid == 0) b.flags[kWpIll] = ill ? 1 : 0;
#pragma unroll 8
  for (int e = tid; e < kWpW * kWpW; e += 512) {
    const int i = e >> 7, c = e & 127;
    b.L[e] = c <= i ? G[i * kWpLd + c] : 0.0;
  }
  if (p == 0) {
#pragma unroll 8
    for (int e = tid; e < kWpW * kWpW; e += 512) {
      const int i = e >> 7, c = e & 127;
      b.Rp[0][e] = c >= i && !(zero[i >> 5] >> (i & 31) & 1) ? G[c * kWpLd + i] : 0.0;
    }
  }
  for (int e = tid; e < kWpW * kQcXLd; e += 512) b.X[e] = X[e];
}

// The rest of a pass, 16 rows per wave: the first nrow workgroups solve the
// rows of P against L; the next ones, from pass 1 on, take C's rows, R_<p += C
// R_p, and ask for another pass where C is not small; the last two take R_p <-
// L^T R_p, one block column per wave.
__global__ __launch_bounds__(256) void wp_rows_kernel(double* __restrict__ A, int m, int n, int j0, int w, bool pairs,
                                                      double* __restrict__ R, WpBuf b, int p, int nrow) {
  __shared__ double T[kWpW * kWpLd];
  __shared__ double X[kWpW * kQcXLd];
  if (p >= 2 && b.flags[p] == 0) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, lr = lane & 15, lk = lane >> 4;
  const int nb = (w + 15) / 16, nc = (j0 + 63) / 64, blk = blockIdx.x;
  const bool rows = blk < nrow, crow = !rows && blk < nrow + nc;
  const double* Ro = b.Rp[(p - 1) & 1];
  const int r0 = 64 * (rows ? blk : blk - nrow) + 16 * wave, row = r0 + lr;
  const int cb = 4 * (blk - nrow - nc) + wave;  // block column of R_p
  const bool in = row < (rows ? m : j0);        // j0 is a whole number of tiles
  double* Ap = (rows ? A : R) + (int64_t)(in ? row : 0) * n + j0 + 4 * lk;
  qc_f64x4 Z[kWpNB], Y[kWpNB];
  int ill = 0, z[4];
  {
    // the 36 tiles of L's lower triangle, or R_p's upper one for the rows of
    // C, the diagonal inverses and the rows of P: all loads in flight before
    // the first LDS store
    ill = b.flags[kWpIll];
#pragma unroll
    for (int q = 0; q < 4; ++q) z[q] = b.flags[kWpZero + q];
    const double* src = crow ? Ro : b.L;
    constexpr int kX = (kWpW * kQcXLd + 255) / 256, kT = kWpNB * (kWpNB + 1) / 2;
    double t[kT], x[kX];
    if (rows) {
#pragma unroll
      for (int u = 0; u < kX; ++u) x[u] = b.X[min(tid + 256 * u, kWpW * kQcXLd - 1)];
    }
    if (rows || crow) {
      // the rows of P, or of C with those of R_<p
      const double* Cp = b.S + (size_t)(in ? row : 0) * kWpW + 4 * lk;
#pragma unroll
      for (int j = 0; j < kWpNB; ++j) {
        qc_f64x4 a, e = {0.0, 0.0, 0.0, 0.0};
        if (pairs) {  // rows of whole blocks on even places: two loads each
          const double* Aj = Ap + min(16 * j, w - 16);
          const qc_f64x2 a0 = *reinterpret_cast<const qc_f64x2*>(Aj), a1 = *reinterpret_cast<const qc_f64x2*>(Aj + 2);
          a = qc_f64x4{a0[0], a0[1], a1[0], a1[1]};
        } else {
#pragma unroll
          for (int v = 0; v < 4; ++v) a[v] = Ap[min(16 * j + v, w - 1 - 4 * lk)];
        }
        if (crow) {
#pragma unroll
          for (int v = 0; v < 4; ++v) e[v] = Cp[16 * j + v];
        }
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const bool on = in && 16 * j + 4 * lk + v < w;
          Z[j][v] = on ? (crow ? e[v] : a[v]) : 0.0;
          Y[j][v] = on ? a[v] : 0.0;
        }
      }
    } else {
#pragma unroll
      for (int k = 0; k < kWpNB; ++k)
#pragma unroll
        for (int v = 0; v < 4; ++v) Z[k][v] = k <= cb ? Ro[(16 * k + 4 * lk + v) * kWpW + 16 * (cb & 7) + lr] : 0.0;
    }
#pragma unroll
    for (int bi = 0, q = 0; bi < kWpNB; ++bi)
#pragma unroll
      for (int bj = 0; bj <= bi; ++bj, ++q) {
        const int r = crow ? bj : bi, c = crow ? bi : bj;
        t[q] = bi < nb ? src[(16 * r + (tid >> 4)) * kWpW + 16 * c + (tid & 15)] : 0.0;
      }
#pragma unroll
    for (int bi = 0, q = 0; bi < kWpNB; ++bi)
#pragma unroll
      for (int bj = 0; bj <= bi; ++bj, ++q) {
        const int r = crow ? bj : bi, c = crow ? bi : bj;
        T[(16 * r + (tid >> 4)) * kWpLd + 16 * c + (tid & 15)] = t[q];
      }
    if (rows) {
#pragma unroll
      for (int u = 0; u < kX; ++u)
        if (tid + 256 * u < kWpW * kQcXLd) X[tid + 256 * u] = x[u];
    }
  }
  __syncthreads();
  auto put = [&](const qc_f64x4(&V)[kWpNB]) {
#pragma unroll
    for (int j = 0; j < kWpNB; ++j) {
      if (pairs) {
        if (in && 16 * j < w) {
          *reinterpret_cast<qc_f64x2*>(Ap + 16 * j) = qc_f64x2{V[j][0], V[j][1]};
          *reinterpret_cast<qc_f64x2*>(Ap + 16 * j + 2) = qc_f64x2{V[j][2], V[j][3]};
        }
      } else {
#pragma unroll
        for (int v = 0; v < 4; ++v)
          if (in && 16 * j + 4 * lk + v < w) Ap[16 * j + v] = V[j][v];
      }
    }
  };
  if (rows) {
    if (r0 >= m) return;
    qc_trsm<kWpNB, kWpLd>(Z, nb, T, X, ill != 0);
    if (p == 0) {
      if (z[0] | z[1] | z[2] | z[3]) {
        const double sc = sqrt(3.0 / m);
#pragma unroll
        for (int j = 0; j < kWpNB; ++j)
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const int c = 16 * j + 4 * lk + v;
            if ((unsigned)z[j >> 1] >> (c & 31) & 1) Z[j][v] = sc * qc_fill(row, j0 + c);
          }
      }
    }
    put(Z);
    return;
  }
  if (crow) {
    if (r0 >= j0) return;
    bool far = false;
#pragma unroll
    for (int j = 0; j < kWpNB; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) far = far || !(fabs(Z[j][v]) <= kWpFar);
    if (far) b.flags[p + 1] = 1;
#pragma unroll
    for (int j = 0; j < kWpNB; ++j) {
      if (j >= nb) break;
#pragma unroll
      for (int k = 0; k <= j; ++k)
#pragma unroll
        for (int kk = 0; kk < 4; ++kk)
          Y[j] = qc_mfma(T[(16 * k + 4 * lk + kk) * kWpLd + 16 * j + qc_at(lr)], Z[k][kk], Y[j]);
      __builtin_amdgcn_sched_barrier(0);
    }
    put(Y);
    return;
  }
  if (cb >= nb) return;
  qc_update_r<kWpNB, kWpLd>(Z, cb, T);
  double* Rn = b.Rp[p & 1];
#pragma unroll
  for (int k = 0; k < kWpNB; ++k)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int i = 16 * k + 4 * lk + v, c = 16 * cb + lr;
      Rn[i * kWpW + c] = Z[k][v];
      if (i < w && c < w) R[(int64_t)(j0 + i) * n + j0 + c] = Z[k][v];
    }
}

__global__ void wp_init_kernel(double* __restrict__ R, int64_t nn, int* __restrict__ flags, int nf) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  for (int64_t e = t; e < nn; e += (int64_t)gridDim.x * blockDim.x) R[e] = 0.0;
  for (int64_t e = t; e < nf; e += (int64_t)gridDim.x * blockDim.x) flags[e] = 0;
}

static int wp_panels(int n) { return (n + kWpW - 1) / kWpW; }

static size_t wp_ws_bytes(int n) {
  size_t b = al((size_t)n * kWpW * 8);          // S
  b += 3 * al((size_t)kWpW * kWpW * 8);         // L, R_p twice
  b += al((size_t)kWpW * kQcXLd * 8);           // X
  b += al((size_t)wp_panels(n) * kWpFlags * sizeof(int));
  return b;
}

// Queues the factorisation; flags is the device array of every panel's flags.
static int wp_queue(double* A, int m, int n, double* R, void* ws, int passes, int** flags, hipStream_t s) {
  char* p = (char*)ws;
  WpBuf b;
  b.S = (double*)p; p += al((size_t)n * kWpW * 8);
  b.L = (double*)p; p += al((size_t)kWpW * kWpW * 8);
  b.Rp[0] = (double*)p; p += al((size_t)kWpW * kWpW * 8);
  b.Rp[1] = (double*)p; p += al((size_t)kWpW * kWpW * 8);
  b.X = (double*)p; p += al((size_t)kWpW * kQcXLd * 8);
  *flags = (int*)p;
  // panels of about the same width, whole 16-wide blocks
  const int np = wp_panels(n), width = ((n + np - 1) / np + 15) / 16 * 16;
  const int64_t nn = (int64_t)n * n;
  hipLaunchKernelGGL(wp_init_kernel, dim3((int)std::min<int64_t>((nn + 255) / 256, 2048)), dim3(256), 0, s, R, nn,
                     *flags, np * kWpFlags);
  TNX_LAUNCH_CHECK();
  GemmDesc t{};
  t.batch = 1; t.prec = Prec::F64;
  t.ta = t.tb = t.tc = DT::F64;
  for (int j0 = 0, pi = 0; j0 < n; j0 += width, ++pi) {
    const int w = std::min(width, n - j0), nt = n - j0 - w;
    // 16-byte accesses: whole blocks, even row starts in A and R (R and the
    // other buffers are 256-byte aligned when the caller's A and R are)
    const bool pairs = w % 16 == 0 && n % 2 == 0 && (((uintptr_t)A | (uintptr_t)R) & 15) == 0;
    b.flags = *flags + pi * kWpFlags;
    for (int q = 0; q < passes; ++q) {
      const int top = q == 0 ? j0 : 0;  // the first pass has no use for C
      GemmDesc g = t;
      g.gate = q >= 2 ? b.flags + q : nullptr;
      g.M = j0 + w - top; g.N = w; g.K = m;
      g.A = A + top; g.lda = n; g.a_kcontig = false;
      g.B = A + j0; g.ldb = n; g.b_ncontig = true;
      g.C = b.S + (size_t)top * kWpW; g.ldc = kWpW;
      g.alpha = 1.0; g.beta = 0.0;
      TNX_TRY(gemm(g, s));
      hipLaunchKernelGGL(wp_factor_kernel, dim3(1), dim3(512), 0, s, b, j0, w, q);
      TNX_LAUNCH_CHECK();
      if (q > 0 && j0 > 0) {  // P -= Q_< C
        GemmDesc u = t;
        u.gate = g.gate;
        u.M = m; u.N = w; u.K = j0;
        u.A = A; u.lda = n; u.a_kcontig = true;
        u.B = b.S; u.ldb = kWpW; u.b_ncontig = true;
        u.C = A + j0; u.ldc = n;
        u.alpha = -1.0; u.beta = 1.0;
        TNX_TRY(gemm(u, s));
      }
      const int nrow = (m + 63) / 64, more = q > 0 ? (j0 + 63) / 64 + 2 : 0;
      hipLaunchKernelGGL(wp_rows_kernel, dim3(nrow + more), dim3(256), 0, s, A, m, n, j0, w, pairs, R, b, q, nrow);
      TNX_LAUNCH_CHECK();
    }
    if (nt <= 0) continue;
    double* Rt = R + (int64_t)j0 * n + j0 + w;
    GemmDesc g = t;  // R_p,> = P^T A_>
    g.M = w; g.N = nt; g.K = m;
    g.A = A + j0; g.lda = n; g.a_kcontig = false;
    g.B = A + j0 + w; g.ldb = n; g.b_ncontig = true;
    g.C = Rt; g.ldc = n;
    g.alpha = 1.0; g.beta = 0.0;
    TNX_TRY(gemm(g, s));
    GemmDesc u = t;  // A_> -= P R_p,>
    u.M = m; u.N = nt; u.K = w;
    u.A = A + j0; u.lda = n; u.a_kcontig = true;
    u.B = Rt; u.ldb = n; u.b_ncontig = true;
    u.C = A + j0 + w; u.ldc = n;
    u.alpha = -1.0; u.beta = 1.0;
    TNX_TRY(gemm(u, s));
  }
  return TNX_OK;
}

size_t qr_ws_bytes(int m, int n) {
  // a copy of A for a second factorisation, then either one's buffers
  return al((size_t)m * n * 8) + std::max(wp_ws_bytes(n), householder_ws_bytes(m, n)) + 256;
}

// QR, then what uses Q and R (`after` queues it on the same stream). The wide
// panels' flags go to a pinned block behind the last panel; the host waits for
// them with `after` already queued, and queues it again where A had to be
// factored a second time.
template <class After>
static int qr_then(double* A, int m, int n, double* R, void* ws, size_t ws_bytes, hipStream_t s, QrUse use,
                   After after) {
  TNX_CHECK_ARG(A && R, "qr: null pointer");
  TNX_CHECK_ARG(m >= 1 && n >= 1 && m >= n, "qr: need m >= n >= 1 (m=%d n=%d)", m, n);
  QrCfg c;
  if (!qr_chol_fits(m, n) && !qr_config(m, &c)) {
    set_error("qr: m=%d rows exceeds the supported 8192", m);
    return TNX_ERR_UNSUPPORTED;
  }
  TNX_CHECK_ARG(ws && ws_bytes >= qr_ws_bytes(m, n), "qr: workspace too small");
  if (qr_chol_fits(m, n)) {
    TNX_TRY(qr_chol(A, m, n, 0, R, 1, s));
    return after();
  }
  char* p = (char*)(((uintptr_t)ws + 255) & ~(uintptr_t)255);
  double* save = (double*)p; p += al((size_t)m * n * 8);
  TNX_TRY(copy_f64(A, save, (int64_t)m * n, s));
  // A thread whose last matrix of the same use took more than two passes queues
  // all four at once: the results are the same, and a wrong guess costs a second
  // factorisation (two queued, four wanted) or the gated launches. One use says
  // nothing of the next: a truncation factors its matrix, the graded factor of
  // that and an almost orthonormal basis in turn (one guess for the three: 8.15
  // ms at n = 512, 70.7 at 2048; one each: 7.7, 68.0).
  static thread_local bool more_of[(int)QrUse::Count] = {};
  bool& more = more_of[(int)use];
  const int nf = wp_panels(n) * kWpFlags;
  PinnedLease pin((size_t)(nf + 1) / 2);
  StepEvent fev;
  std::vector<int> plain;
  int* hf = reinterpret_cast<int*>(pin.get());
  if (!hf || !fev.e) {
    plain.resize(nf);
    hf = plain.data();
  }
  auto any = [&](int f) {
    for (int i = f; i < nf; i += kWpFlags)
      if (hf[i] != 0) return true;
    return false;
  };
  for (bool four = more;; four = true) {
    int* flags = nullptr;
    TNX_TRY(wp_queue(A, m, n, R, p, four ? kWpPasses : 2, &flags, s));
    TNX_HIP(hipMemcpyAsync(hf, flags, (size_t)nf * sizeof(int), hipMemcpyDeviceToHost, s));
    if (plain.empty()) {
      TNX_HIP(hipEventRecord(fev.e, s));
      const int st = after();
      // the copy must land before the block goes back to the pool
      const hipError_t we = hipEventSynchronize(fev.e);
      TNX_TRY(st);
      TNX_HIP(we);
    } else {
      TNX_HIP(hipStreamSynchronize(s));
    }
    more = any(2) || any(kWpPasses);
    const bool failed = four ? any(kWpPasses) : more;
    if (!failed) return plain.empty() ? TNX_OK : after();
    TNX_TRY(copy_f64(save, A, (int64_t)m * n, s));
    if (four) break;
  }
  TNX_TRY(qr_householder(A, m, n, R, p, s));
  return after();
}

int qr(double* A, int m, int n, double* R, void* ws, size_t ws_bytes, hipStream_t s, QrUse use) {
  return qr_then(A, m, n, R, ws, ws_bytes, s, use, [] { return TNX_OK; });
}

// ---- gauge moves -------------------------------------------------------------
size_t gauge_ws_bytes(int chil, int d, int chir) {
  const int64_t m1 = (int64_t)chil * d, n1 = chir;          // rightward
  const int64_t m2 = (int64_t)d * chir, n2 = chil;          // leftward (transposed)
  size_t a = 0, b = 0;
  if (m1 >= n1) a = al((size_t)n1 * n1 * 8) + qr_ws_bytes((int)m1, (int)n1);
  if (m2 >= n2) b = al((size_t)m2 * n2 * 8) + al((size_t)n2 * n2 * 8) + qr_ws_bytes((int)m2, (int)n2);
  return std::max(a, b) + 256;
}

int gauge_right(double* A, const double* next, double* next_out, int chil, int d, int chir,
                int next_cols, void* ws, size_t ws_bytes, hipStream_t s) {
  TNX_CHECK_ARG(A && next && next_out && next != next_out, "gauge_right: bad pointers");
  TNX_CHECK_ARG(chil > 0 && d > 0 && chir > 0 && next_cols > 0, "gauge_right: bad dims");
  const int m = chil * d, n = chir;
  TNX_CHECK_ARG(m >= n, "gauge_right: chil*d=%d < chir=%d (bond would shrink)", m, n);
  TNX_CHECK_ARG(ws && ws_bytes >= gauge_ws_bytes(chil, d, chir), "gauge_right: workspace too small");
  char* p = (char*)(((uintptr_t)ws + 255) & ~(uintptr_t)255);
  double* R = (double*)p; p += al((size_t)n * n * 8);
  return qr_then(A, m, n, R, p, qr_ws_bytes(m, n), s, QrUse::GaugeRight, [&]() -> int {
    // next_out = R * next
    GemmDesc g{};
    g.M = n; g.N = next_cols; g.K = n; g.batch = 1;
    g.A = R; g.ta = DT::F64; g.lda = n; g.sA = 0; g.a_kcontig = true;
    g.B = next; g.tb = DT::F64; g.ldb = next_cols; g.sB = 0; g.b_ncontig = true;
    g.C = next_out; g.tc = DT::F64; g.ldc = next_cols; g.sC = 0;
    g.alpha = 1.0; g.beta = 0.0; g.prec = Prec::F64;
    return gemm(g, s);
  });
}

int gauge_left(double* A, const double* prev, double* prev_out, int chil, int d, int chir,
               int prev_rows, void* ws, size_t ws_bytes, hipStream_t s) {
  TNX_CHECK_ARG(A && prev && prev_out && prev != prev_out, "gauge_left: bad pointers");
  TNX_CHECK_ARG(chil > 0 && d > 0 && chir > 0 && prev_rows > 0, "gauge_left: bad dims");
  const int m = d * chir, n = chil;
  TNX_CHECK_ARG(m >= n, "gauge_left: d*chir=%d < chil=%d (bond would shrink)", m, n);
  TNX_CHECK_ARG(ws && ws_bytes >= gauge_ws_bytes(chil, d, chir), "gauge_left: workspace too small");
  char* p = (char*)(((uintptr_t)ws + 255) & ~(uintptr_t)255);
  double* At = (double*)p; p += al((size_t)m * n * 8);
  double* R = (double*)p; p += al((size_t)n * n * 8);
  // A (chil x d*chir) -> At (d*chir x chil); At = Q R; A = Q^T; prev <- prev R^T
  auto carry = [&]() -> int {  // prev_out = prev R^T
    GemmDesc g{};
    g.M = prev_rows; g.N = n; g.K = n; g.batch = 1;
    g.A = prev; g.ta = DT::F64; g.lda = n; g.sA = 0; g.a_kcontig = true;
    g.B = R; g.tb = DT::F64; g.ldb = n; g.sB = 0; g.b_ncontig = false;
    g.C = prev_out; g.tc = DT::F64; g.ldc = n; g.sC = 0;
    g.alpha = 1.0; g.beta = 0.0; g.prec = Prec::F64;
    return gemm(g, s);
  };
  if (qr_chol_fits(m, n)) {
    TNX_TRY(qr_chol(A, m, n, 1, R, 1, s));
    return carry();
  }
  TNX_TRY(transpose_f64(A, At, n, m, s));
  return qr_then(At, m, n, R, p, qr_ws_bytes(m, n), s, QrUse::GaugeLeft, [&]() -> int {
    TNX_TRY(transpose_f64(At, A, m, n, s));
    return carry();
  });
}

size_t gauge_b_ws_bytes(int chil, int d, int chir, int batch) {
  const size_t n = (size_t)std::max(chil, chir);
  return al(n * n * 8 * (size_t)batch) + 256;
}

int gauge_right_b(double* A, const double* next, double* next_out, int chil, int d, int chir,
                  int next_cols, int batch, void* ws, size_t ws_bytes, hipStream_t s) {
  TNX_CHECK_ARG(A && next && next_out && next != next_out, "gauge_right_batched: bad pointers");
  TNX_CHECK_ARG(chil > 0 && d > 0 && chir > 0 && next_cols > 0 && batch > 0,
                "gauge_right_batched: bad dims");
  const int m = chil * d, n = chir;
  TNX_CHECK_ARG(m >= n, "gauge_right_batched: chil*d=%d < chir=%d", m, n);
  TNX_CHECK_ARG(ws && ws_bytes >= gauge_b_ws_bytes(chil, d, chir, batch),
                "gauge_right_batched: workspace too small");
  double* R = (double*)(((uintptr_t)ws + 255) & ~(uintptr_t)255);
  TNX_TRY(qr_small_b(A, m, n, 0, R, batch, s));
  GemmDesc g{};
  g.M = n; g.N = next_cols; g.K = n; g.batch = batch;
  g.A = R; g.ta = DT::F64; g.lda = n; g.sA = (int64_t)n * n; g.a_kcontig = true;
  g.B = next; g.tb = DT::F64; g.ldb = next_cols; g.sB = (int64_t)n * next_cols; g.b_ncontig = true;
  g.C = next_out; g.tc = DT::F64; g.ldc = next_cols; g.sC = (int64_t)n * next_cols;
  g.alpha = 1.0; g.beta = 0.0; g.prec = Prec::F64;
  return gemm(g, s);
}

int gauge_left_b(double* A, const double* prev, double* prev_out, int chil, int d, int chir,
                 int prev_rows, int batch, void* ws, size_t ws_bytes, hipStream_t s) {
  TNX_CHECK_ARG(A && prev && prev_out && prev != prev_out, "gauge_left_batched: bad pointers");
  TNX_CHECK_ARG(chil > 0 && d > 0 && chir > 0 && prev_rows > 0 && batch > 0,
                "gauge_left_batched: bad dims");
  const int m = d * chir, n = chil;
  TNX_CHECK_ARG(m >= n, "gauge_left_batched: d*chir=%d < chil=%d", m, n);
  TNX_CHECK_ARG(ws && ws_bytes >= gauge_b_ws_bytes(chil, d, chir, batch),
                "gauge_left_batched: workspace too small");
  double* R = (double*)(((uintptr_t)ws + 255) & ~(uintptr_t)255);
  TNX_TRY(qr_small_b(A, m, n, 1, R, batch, s));
  // prev <- prev R^T
  GemmDesc g{};
  g.M = prev_rows; g.N = n; g.K = n; g.batch = batch;
  g.A = prev; g.ta = DT::F64; g.lda = n; g.sA = (int64_t)prev_rows * n; g.a_kcontig = true;
  g.B = R; g.tb = DT::F64; g.ldb = n; g.sB = (int64_t)n * n; g.b_ncontig = false;
  g.C = prev_out; g.tc = DT::F64; g.ldc = n; g.sC = (int64_t)prev_rows * n;
  g.alpha = 1.0; g.beta = 0.0; g.prec = Prec::F64;
  return gemm(g, s);
}

}  // namespace tnx

extern "C" {

size_t tnx_qr_workspace_bytes(int m, int n) { return tnx::qr_ws_bytes(m, n); }

int tnx_qr(double* A, int m, int n, double* R, void* ws, size_t ws_bytes, tnx_stream_t stream) {
  return tnx::qr(A, m, n, R, ws, ws_bytes, (hipStream_t)stream, tnx::QrUse::Plain);
}

size_t tnx_gauge_workspace_bytes(int chil, int d, int chir) {
  return tnx::gauge_ws_bytes(chil, d, chir);
}

int tnx_gauge_right(double* A, const double* next, double* next_out, int chil, int d, int chir,
                    int next_cols, void* ws, size_t ws_bytes, tnx_stream_t stream) {
  return tnx::gauge_right(A, next, next_out, chil, d, chir, next_cols, ws, ws_bytes,
                          (hipStream_t)stream);
}

int tnx_gauge_left(double* A, const double* prev, double* prev_out, int chil, int d, int chir,
                   int prev_rows, void* ws, size_t ws_bytes, tnx_stream_t stream) {
  return tnx::gauge_left(A, prev, prev_out, chil, d, chir, prev_rows, ws, ws_bytes,
                         (hipStream_t)stream);
}

size_t tnx_gauge_batched_workspace_bytes(int chil, int d, int chir, int batch) {
  return tnx::gauge_b_ws_bytes(chil, d, chir, batch);
}

int tnx_gauge_right_batched(double* A, const double* next, double* next_out,
                            int chil, int d, int chir, int next_cols, int batch,
                            void* ws, size_t ws_bytes, tnx_stream_t stream) {
  return tnx::gauge_right_b(A, next, next_out, chil, d, chir, next_cols, batch, ws, ws_bytes,
                            (hipStream_t)stream);
}

int tnx_gauge_left_batched(double* A, const double* prev, double* prev_out,
                           int chil, int d, int chir, int prev_rows, int batch,
                           void* ws, size_t ws_bytes, tnx_stream_t stream) {
  return tnx::gauge_left_b(A, prev, prev_out, chil, d, chir, prev_rows, batch, ws, ws_bytes,
                           (hipStream_t)stream);
}

}  // extern "C"
