// Lowest eigenpair of the one-site effective Hamiltonian on the device, and
// the small dense symmetric eigensolver.
//
// Replaces primme.eigsh(which='SA', k=1) (tnpy/linalg.py:64-87, called at
// tnpy/finite_dmrg.py:111) and np.linalg.eigh below exact_solver_dim
// (tnpy/linalg.py:42-61, tnpy/finite_dmrg.py:108-110).
//
// Krylov method: Lanczos with full reorthogonalisation (classical
// Gram-Schmidt, two passes) and thick restart keeping `keep` Ritz vectors. The
// projected matrix stays tridiagonal; its lowest pair is found by one
// wavefront (64-way multisection on Sturm counts around predicted roots, then
// a twisted factorisation).
// All Krylov scalars live in device memory; the host reads one small status
// block per iteration to decide convergence / restart.
//
// Mixed precision: the Krylov matvecs run in FP32 or BF16x3; every cycle
// starts from an FP64 matvec on the current Ritz vector (Rayleigh quotient
// and residual in FP64), and the next cycle's basis is [y, r/|r|]. The
// returned eigenvalue, residual and H*y are FP64.
//
// Vector kernels are HBM bound: a CGS pass over J basis vectors of length N
// reads (J+1)*N*8 bytes (+N*8 written when it updates w).
#include "tnx_common.h"

#include <algorithm>
#include <cmath>
#include <mutex>
#include <type_traits>
#include <utility>
#include <vector>

namespace tnx {

int heff1_matvec(const double* L, const double* W, const double* R, const double* x,
                 double* y, int chil, int Dl, int Dr, int d, int chir, int prec,
                 void* ws, size_t ws_bytes, hipStream_t s);
size_t heff1_ws_bytes(int chil, int Dl, int Dr, int d, int chir);
int heff2_matvec(const double* L, const double* W1, const double* W2, const double* R,
                 const void* x, int x_f32, double* y, int chil, int Dl, int Dm, int Dr, int d,
                 int chir, int prec, void* ws, size_t ws_bytes, hipStream_t s);
int heff1_matvec_b(const void* L, const double* W, const void* R, const void* x, int x_f32,
                   double* y, int chil, int Dl, int Dr, int d, int chir, int prec, int batch,
                   int count, const int* bidx, int64_t sx, int64_t sy, void* ws, size_t ws_bytes,
                   hipStream_t s, int env_f32);
size_t heff2_ws_bytes(int chil, int Dl, int Dm, int Dr, int d, int chir);

// Lane i's value of a wave-distributed double, as a wave-uniform scalar
// (v_readlane: no LDS round trip). i must be wave-uniform.
__device__ __forceinline__ double lane_val(double v, int i) {
  const long long u = __double_as_longlong(v);
  const unsigned lo = __builtin_amdgcn_readlane((int)(u & 0xffffffffll), i);
  const unsigned hi = __builtin_amdgcn_readlane((int)(u >> 32), i);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// The value of the lane that a DPP control selects, `none` where there is
// none. Reductions and scans over a wave go through these and lane reads: a
// step costs a few cycles, where a shuffle waits for an LDS round trip.
template <int CTRL>
__device__ __forceinline__ double dpp(double x, double none = 0.0) {
  const long long u = __double_as_longlong(x), w = __double_as_longlong(none);
  const unsigned lo = __builtin_amdgcn_update_dpp((int)w, (int)u, CTRL, 0xf, 0xf, false);
  const unsigned hi = __builtin_amdgcn_update_dpp((int)(w >> 32), (int)(u >> 32), CTRL, 0xf, 0xf, false);
  return __longlong_as_double((long long)((unsigned long long)hi << 32 | lo));
}

// op over each 16 lanes, in all of them: neighbours, pairs, then the mirrored
// halves; over the wave, the four groups by lane reads.
template <typename OP>
__device__ __forceinline__ double reduce16(double x, OP op) {
  x = op(x, dpp<0xB1>(x));     // quad_perm 1 0 3 2
  x = op(x, dpp<0x4E>(x));     // quad_perm 2 3 0 1
  x = op(x, dpp<0x141>(x));    // row_half_mirror
  return op(x, dpp<0x140>(x));  // row_mirror
}

template <typename OP>
__device__ __forceinline__ double wave_reduce(double x, OP op) {
  x = reduce16(x, op);
  return op(op(lane_val(x, 0), lane_val(x, 16)), op(lane_val(x, 32), lane_val(x, 48)));
}

__device__ __forceinline__ double sum16(double x) {
  return reduce16(x, [](double a, double b) { return a + b; });
}
__device__ __forceinline__ double sum64(double x) {
  return wave_reduce(x, [](double a, double b) { return a + b; });
}
__device__ __forceinline__ double wave_min(double x) {
  return wave_reduce(x, [](double a, double b) { return fmin(a, b); });
}
__device__ __forceinline__ double wave_max(double x) {
  return wave_reduce(x, [](double a, double b) { return fmax(a, b); });
}

// x of the lower half of the wave beside y of the upper (HALF 32), or of the
// even and odd rows of 16 (HALF 16), plus what each gets from the other:
// lanes of the first kind return x + the partner's x, the others y + its y.
template <int HALF>
__device__ __forceinline__ double swap_add(double x, double y) {
  const long long a = __double_as_longlong(x), b = __double_as_longlong(y);
  double r[2];
  if constexpr (HALF == 32) {
    const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)a, (unsigned)b, false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)(a >> 32), (unsigned)(b >> 32), false, false);
    for (int q = 0; q < 2; ++q) r[q] = __longlong_as_double((long long)((unsigned long long)hi[q] << 32 | lo[q]));
  } else {
    const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)a, (unsigned)b, false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)(a >> 32), (unsigned)(b >> 32), false, false);
    for (int q = 0; q < 2; ++q) r[q] = __longlong_as_double((long long)((unsigned long long)hi[q] << 32 | lo[q]));
  }
  return r[0] + r[1];
}

// Sum over the wave in all lanes, as the tree of lane ^ 32, ^ 16, ... ^ 1 (once
// the sums repeat every 8 or 4 lanes, a rotation reaches the same partner).
__device__ __forceinline__ double wave_sum(double x) {
  x = swap_add<32>(x, x);
  x = swap_add<16>(x, x);
  x += dpp<0x128>(x);  // row_ror 8, 4
  x += dpp<0x124>(x);
  x += dpp<0x4E>(x);  // quad_perm 2 3 0 1, 1 0 3 2
  return x + dpp<0xB1>(x);
}

// Problem map of a batched launch: launched problem i = blockIdx.y works on
// logical problem idx[i] (or i when idx is null), whose work arrays sit at
// +problem * sp doubles from the base pointers. One problem: idx null, sp 0.
struct PMap {
  const int* idx;
  int64_t sp;
  __device__ __forceinline__ int pid() const { return idx ? idx[blockIdx.y] : (int)blockIdx.y; }
  __device__ __forceinline__ int64_t off() const { return (int64_t)pid() * sp; }
};
static const PMap kOne{nullptr, 0};

constexpr int kMaxBasis = 64;        // Lanczos vectors kept before restart
constexpr int kPartStride = kMaxBasis + 2;
constexpr int kCgsBlocks = 512;      // blocks of a CGS pass (partials rows)

// One classical Gram-Schmidt pass over basis V[0..J-1] (row stride ldv):
//   if hsub:  w -= sum_j V[j] * hsub[j]               (in place)
//   partial[blk][j] = sum_i V[j][i] w[i]   (j < J, if DOTS)
//   partial[blk][JMAX... stored at index J] = sum_i w[i]^2
template <int JMAX, bool DOTS, typename VT>
__global__ __launch_bounds__(256) void cgs_pass_kernel(const VT* __restrict__ V,
                                                       int64_t ldv, int J,
                                                       double* __restrict__ w,
                                                       const double* __restrict__ hsub,
                                                       double* __restrict__ partials,
                                                       int64_t N, PMap pm) {
  {
    const int64_t o = pm.off();
    V += o; w += o; partials += o;
    if (hsub) hsub += o;
  }
  __shared__ double hs[JMAX];
  __shared__ double red[4][JMAX + 1];
  if (threadIdx.x < JMAX) hs[threadIdx.x] = (hsub && (int)threadIdx.x < J) ? hsub[threadIdx.x] : 0.0;
  __syncthreads();
  double acc[JMAX];
#pragma unroll
  for (int j = 0; j < JMAX; ++j) acc[j] = 0.0;
  double nrm = 0.0;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  if constexpr (std::is_same<VT, double>::value) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < N; i += stride) {
      double vv[JMAX];
#pragma unroll
      for (int j = 0; j < JMAX; ++j) vv[j] = (j < J) ? V[(int64_t)j * ldv + i] : 0.0;
      double wi = w[i];
      if (hsub) {
#pragma unroll
        for (int j = 0; j < JMAX; ++j) wi -= vv[j] * hs[j];
        w[i] = wi;
      }
      if (DOTS) {
#pragma unroll
        for (int j = 0; j < JMAX; ++j) acc[j] += vv[j] * wi;
      }
      nrm += wi * wi;
    }
  } else {
    // FP32 basis: unconditional loads (rows past J re-read row J-1, a cache
    // hit) and the widening after all of them. A guarded load with its
    // conversion in the same branch waits for its data before the next
    // load issues.
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < N; i += stride) {
      float raw[JMAX];
#pragma unroll
      for (int j = 0; j < JMAX; ++j) raw[j] = V[(int64_t)(j < J ? j : J - 1) * ldv + i];
      double vv[JMAX];
#pragma unroll
      for (int j = 0; j < JMAX; ++j) vv[j] = (j < J) ? (double)raw[j] : 0.0;
      double wi = w[i];
      if (hsub) {
#pragma unroll
        for (int j = 0; j < JMAX; ++j) wi -= vv[j] * hs[j];
        w[i] = wi;
      }
      if (DOTS) {
#pragma unroll
        for (int j = 0; j < JMAX; ++j) acc[j] += vv[j] * wi;
      }
      nrm += wi * wi;
    }
  }
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  if (DOTS) {
#pragma unroll
    for (int j = 0; j < JMAX; ++j) {
      const double t = wave_sum(acc[j]);
      if (lane == 0) red[wv][j] = t;
    }
  }
  {
    const double t = wave_sum(nrm);
    if (lane == 0) red[wv][JMAX] = t;
  }
  __syncthreads();
  double* out = partials + (int64_t)blockIdx.x * kPartStride;
  if ((int)threadIdx.x < J && DOTS)
    out[threadIdx.x] = red[0][threadIdx.x] + red[1][threadIdx.x] + red[2][threadIdx.x] + red[3][threadIdx.x];
  if (threadIdx.x == 0) out[J] = red[0][JMAX] + red[1][JMAX] + red[2][JMAX] + red[3][JMAX];
}

// The same pass with R lanes per group of E elements (FP64 basis: R = 2,
// E = 2; FP32: R = 4, E = 4; one 16-byte load per basis row): lane
// h = lane % R of a group reads basis rows [h*JMAX/R, (h+1)*JMAX/R) of its
// group; the subtraction's partial sums are combined across the group by
// shuffles, and each lane accumulates dot products for its own rows
// (reduced over the lanes with its h). Every load moves 16 bytes and a lane
// holds 1/R of the rows, against 4- or 8-byte loads of all rows for one
// lane per element. Needs N and ldv multiples of E and V, w 16-byte aligned
// (cgs_pass checks).
__device__ __forceinline__ double vcomp(const double2& v, int q) { return q == 0 ? v.x : v.y; }
__device__ __forceinline__ double vcomp(const float4& v, int q) {
  return q == 0 ? v.x : (q == 1 ? v.y : (q == 2 ? v.z : v.w));
}

template <int JMAX, bool DOTS, typename VT>
__global__ __launch_bounds__(256) void cgs_pair_kernel(const VT* __restrict__ V, int64_t ldv,
                                                       int J, double* __restrict__ w,
                                                       const double* __restrict__ hsub,
                                                       double* __restrict__ partials, int64_t N,
                                                       PMap pm) {
  using PV = typename std::conditional<std::is_same<VT, float>::value, float4, double2>::type;
  constexpr int E = 16 / sizeof(VT);
  constexpr int R = E;
  constexpr int JH = JMAX / R;
  {
    const int64_t o = pm.off();
    V += o; w += o; partials += o;
    if (hsub) hsub += o;
  }
  __shared__ double hs[JMAX];
  __shared__ double red[4][JMAX + 1];
  if (threadIdx.x < JMAX) hs[threadIdx.x] = (hsub && (int)threadIdx.x < J) ? hsub[threadIdx.x] : 0.0;
  __syncthreads();
  const int h = threadIdx.x & (R - 1);
  const int r0 = h * JH;
  double acc[JH];
#pragma unroll
  for (int j = 0; j < JH; ++j) acc[j] = 0.0;
  double nrm = 0.0;
  const PV* Vp = reinterpret_cast<const PV*>(V);
  double2* w2 = reinterpret_cast<double2*>(w);
  const int64_t NE = N / E, ldE = ldv / E;
  const int64_t stride = ((int64_t)gridDim.x * blockDim.x) / R;
  for (int64_t e = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / R; e < NE; e += stride) {
    PV raw[JH];
#pragma unroll
    for (int jj = 0; jj < JH; ++jj) {
      const int j = r0 + jj;
      raw[jj] = Vp[(int64_t)(j < J ? j : J - 1) * ldE + e];
    }
    double wv[E];
#pragma unroll
    for (int q = 0; q < E / 2; ++q) {
      const double2 t = w2[e * (E / 2) + q];
      wv[2 * q] = t.x;
      wv[2 * q + 1] = t.y;
    }
    if (hsub) {
      double sm[E];
#pragma unroll
      for (int q = 0; q < E; ++q) sm[q] = 0.0;
#pragma unroll
      for (int jj = 0; jj < JH; ++jj) {
        const double hj = hs[r0 + jj];
#pragma unroll
        for (int q = 0; q < E; ++q) sm[q] += vcomp(raw[jj], q) * hj;
      }
#pragma unroll
      for (int o = 1; o < R; o <<= 1)
#pragma unroll
        for (int q = 0; q < E; ++q) sm[q] += __shfl_xor(sm[q], o, 64);
#pragma unroll
      for (int q = 0; q < E; ++q) wv[q] -= sm[q];
      if (h == 0) {
#pragma unroll
        for (int q = 0; q < E / 2; ++q) w2[e * (E / 2) + q] = make_double2(wv[2 * q], wv[2 * q + 1]);
      }
    }
    if (DOTS) {
#pragma unroll
      for (int jj = 0; jj < JH; ++jj) {
        double t = 0.0;
#pragma unroll
        for (int q = 0; q < E; ++q) t += vcomp(raw[jj], q) * wv[q];
        acc[jj] += t;
      }
    }
    if (h == 0) {
#pragma unroll
      for (int q = 0; q < E; ++q) nrm += wv[q] * wv[q];
    }
  }
  const int lane = threadIdx.x & 63, wv_ = threadIdx.x >> 6;
  if (DOTS) {
#pragma unroll
    for (int jj = 0; jj < JH; ++jj) {
      double t = acc[jj];
#pragma unroll
      for (int o = 32; o >= R; o >>= 1) t += __shfl_xor(t, o, 64);  // lanes with one h
      if (lane < R) red[wv_][lane * JH + jj] = t;
    }
  }
  {
    const double t = wave_sum(nrm);
    if (lane == 0) red[wv_][JMAX] = t;
  }
  __syncthreads();
  double* out = partials + (int64_t)blockIdx.x * kPartStride;
  if ((int)threadIdx.x < J && DOTS)
    out[threadIdx.x] = red[0][threadIdx.x] + red[1][threadIdx.x] + red[2][threadIdx.x] + red[3][threadIdx.x];
  if (threadIdx.x == 0) out[J] = red[0][JMAX] + red[1][JMAX] + red[2][JMAX] + red[3][JMAX];
}

// out[j] = sum over blocks of partials[blk][j], j <= J. One workgroup per
// j; a fixed strided split and a fixed tree, so the sum is deterministic.
__global__ __launch_bounds__(256) void reduce_partials_kernel(const double* partials, int nblk,
                                                              int J, double* out, PMap pm) {
  {
    const int64_t o = pm.off();
    partials += o; out += o;
  }
  __shared__ double red[4];
  const int j = blockIdx.x;
  double s = 0.0;
  for (int b = threadIdx.x; b < nblk; b += blockDim.x) s += partials[(int64_t)b * kPartStride + j];
  s = wave_sum(s);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) out[j] = (red[0] + red[1]) + (red[2] + red[3]);
}

// One CGS pass over a basis stored in VT (double, or float for the basis of
// a low-precision Krylov cycle); w and all sums are FP64.
template <typename VT>
static int cgs_pass(const VT* V, int64_t ldv, int J, double* w, const double* hsub,
                    bool dots, double* partials, double* out, int64_t N, hipStream_t s,
                    PMap pm = kOne, int count = 1) {
  const int nblk = (int)std::min<int64_t>(count > 1 ? std::max(kCgsBlocks / count, 8) : kCgsBlocks,
                                          (N + 255) / 256);
  // Passes with dot products take the pair kernel (measured faster); the
  // subtract-and-norm pass keeps one lane per element (the pair form is
  // slower there). The pair kernel needs lengths in whole 16-byte groups and
  // 16-byte aligned pointers (offsets of batched problems are multiples of
  // 256 bytes).
  constexpr int E = 16 / sizeof(VT);
  const bool pair = dots && J >= 2 && N % E == 0 && ldv % E == 0 && ((uintptr_t)V % 16) == 0 &&
                    ((uintptr_t)w % 16) == 0;
  auto go = [&](auto jtag, auto dtag) {
    constexpr int JM = decltype(jtag)::value;
    constexpr bool DT_ = decltype(dtag)::value;
    if (pair)
      hipLaunchKernelGGL((cgs_pair_kernel<JM, DT_, VT>), dim3(nblk, count), dim3(256), 0, s, V,
                         ldv, J, w, hsub, partials, N, pm);
    else
      hipLaunchKernelGGL((cgs_pass_kernel<JM, DT_, VT>), dim3(nblk, count), dim3(256), 0, s, V, ldv,
                         J, w, hsub, partials, N, pm);
  };
  using T8 = std::integral_constant<int, 8>;
  using T16 = std::integral_constant<int, 16>;
  using T32 = std::integral_constant<int, 32>;
  using T64 = std::integral_constant<int, 64>;
  using BT = std::integral_constant<bool, true>;
  using BF = std::integral_constant<bool, false>;
  TNX_CHECK_ARG(J >= 0 && J <= kMaxBasis, "cgs_pass: J=%d out of range", J);
  if (J <= 8) { if (dots) go(T8{}, BT{}); else go(T8{}, BF{}); }
  else if (J <= 16) { if (dots) go(T16{}, BT{}); else go(T16{}, BF{}); }
  else if (J <= 32) { if (dots) go(T32{}, BT{}); else go(T32{}, BF{}); }
  else { if (dots) go(T64{}, BT{}); else go(T64{}, BF{}); }
  TNX_LAUNCH_CHECK();
  hipLaunchKernelGGL(reduce_partials_kernel, dim3(J + 1, count), dim3(256), 0, s, partials, nblk,
                     J, out, pm);
  TNX_LAUNCH_CHECK();
  return TNX_OK;
}

// ---- the orthogonalisation of a Lanczos step at small and middle lengths ----
// CGS2 as four launches, with no reduction launches between them: dots |
// subtract + dots | subtract + norm | normalise. Each kernel starts by
// summing the partials of the one before it (every workgroup the same sums
// in the same order, from L2) instead of waiting for a kernel that does.
// What bounds these lengths is latency and how many CUs share the basis: a
// workgroup takes 128 elements at a time, its four waves a quarter of the
// basis rows each (JW rows, two elements per lane), so N = 7200 runs on 57
// CUs with 16 loads in flight per lane, and a wave's JW dot products are
// summed over its lanes together (halving exchanges, 17 for 16 rows against 6 per row). With one 256-element workgroup per launch partial and three
// reduction kernels a step at N = 7200, J = 64 took 44 us for the three
// passes and the normalisation; this form 15.
constexpr int kRowsBlocks = 160;  // partial rows of one pass; three passes fit the kCgsBlocks rows
constexpr int kRowsElems = 128;

typedef double kr_f64x2 __attribute__((ext_vector_type(2), aligned(8)));
typedef float kr_f32x2 __attribute__((ext_vector_type(2), aligned(4)));

// Sum of partials[b][c], b < nb <= kRowsBlocks, c < cnt <= 64, into out
// (LDS), by 256 threads: four partial sums over b = p, p + 4, .. combined in
// fixed order. In two halves, so that a caller can issue its own loads
// between them: the first kPartFetch values of a thread are loaded by
// fetch_partials (before anything slower in the same queue), the rest by
// sum_partials.
constexpr int kPartFetch = 16;
__device__ __forceinline__ void fetch_partials(const double* __restrict__ partials, int nb, int cnt,
                                               double (&v)[kPartFetch]) {
  const int c = threadIdx.x & 63, part = threadIdx.x >> 6;
#pragma unroll
  for (int u = 0; u < kPartFetch; ++u) {
    const int b = part + 4 * u;
    v[u] = c < cnt && b < nb ? partials[(int64_t)b * kPartStride + c] : 0.0;
  }
}

__device__ __forceinline__ void sum_partials(const double* __restrict__ partials, int nb, int cnt,
                                             const double (&first)[kPartFetch], double* out, double (*red)[64]) {
  const int c = threadIdx.x & 63, part = threadIdx.x >> 6;
  double acc = 0.0;
#pragma unroll
  for (int u = 0; u < kPartFetch; ++u) acc += first[u];
  if (c < cnt)
    for (int b = part + 4 * kPartFetch; b < nb; b += 32) {
      double v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = b + 4 * u < nb ? partials[(int64_t)(b + 4 * u) * kPartStride + c] : 0.0;
#pragma unroll
      for (int u = 0; u < 8; ++u) acc += v[u];
    }
  red[part][c] = acc;
  __syncthreads();
  if (threadIdx.x < 64) out[c] = (red[0][c] + red[1][c]) + (red[2][c] + red[3][c]);
  __syncthreads();
}

// Sum over the 64 lanes of each of JW values per lane; on return lane l's
// v[0] is the total of row cgs_row_of<JW>(l) of the wave's rows.
template <int JW>
__device__ __forceinline__ double lane_totals(double (&v)[JW]) {
  // halves of the wave, then rows of 16, by swaps; inside a row by DPP
  const int lane = threadIdx.x & 63;
  static_assert(JW == 4 || JW == 8 || JW == 16, "two swapped levels, the rest inside a row");
  auto other = [&](double x, int o) {  // of lane ^ o
    if (o == 8) return dpp<0x128>(x);
    if (o == 4) {
      const double before = dpp<0x124>(x), behind = dpp<0x12C>(x);
      return lane & 4 ? before : behind;
    }
    return o == 2 ? dpp<0x4E>(x) : dpp<0xB1>(x);
  };
  int o = 32;
#pragma unroll
  for (int c = JW / 2; c >= 1; c >>= 1) {
    const bool up = lane & o;
#pragma unroll
    for (int k = 0; k < c; ++k) {
      if (o == 32) {
        v[k] = swap_add<32>(v[k], v[c + k]);
      } else if (o == 16) {
        v[k] = swap_add<16>(v[k], v[c + k]);
      } else {
        const double keep = up ? v[c + k] : v[k], send = up ? v[k] : v[c + k];
        v[k] = keep + other(send, o);
      }
    }
    o >>= 1;
  }
  double t = v[0];
#pragma unroll
  for (; o > 0; o >>= 1) t += other(t, o);
  return t;
}

template <int JW>
__device__ __forceinline__ int cgs_row_of(int lane) {
  int row = 0, o = 32;
#pragma unroll
  for (int c = JW / 2; c >= 1; c >>= 1) {
    if (lane & o) row += c;
    o >>= 1;
  }
  return row;
}

// PASS 0: partials pout[b][j] of V[j] . w. PASS 1: h1 from pin, w -= V h1,
// partials of V[j] . w. PASS 2: h2 from pin, w -= V h2, partials pout[b][0] of
// w . w. h (global): the sums of this pass's start, written by workgroup 0.
// N even; V's rows at stride ldv.
template <int JW, int PASS, typename VT>
__global__ __launch_bounds__(256) void cgs_rows_kernel(const VT* __restrict__ V, int64_t ldv, int J,
                                                       double* __restrict__ w,
                                                       const double* __restrict__ pin, int nin,
                                                       double* __restrict__ h, double* __restrict__ pout,
                                                       int64_t N, PMap pm) {
  using V2 = typename std::conditional<sizeof(VT) == 8, kr_f64x2, kr_f32x2>::type;
  {
    const int64_t o = pm.off();
    V += o; w += o; pout += o;
    if (PASS > 0) { pin += o; h += o; }
  }
  __shared__ double hs[64];
  __shared__ double red[4][64];
  __shared__ kr_f64x2 sub[4][64];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int j0 = wv * JW;
  const int64_t step = (int64_t)gridDim.x * kRowsElems;
  int64_t i = (int64_t)blockIdx.x * kRowsElems + 2 * lane;
  // rows past J - 1 re-read row J - 1 (a cache hit) with a zero coefficient
  V2 raw[JW];
  kr_f64x2 wi = {0.0, 0.0};
  auto fetch = [&](int64_t at) {
    const int64_t q = at < N ? at : 0;
#pragma unroll
    for (int k = 0; k < JW; ++k)
      raw[k] = *reinterpret_cast<const V2*>(V + (int64_t)min(j0 + k, J - 1) * ldv + q);
    // where w is updated, its one writer (the first wave) is its one reader
    if (PASS == 0 || wv == 0) wi = *reinterpret_cast<const kr_f64x2*>(w + q);
  };
  double part[kPartFetch];
  if (PASS > 0) fetch_partials(pin, nin, J, part);
  fetch(i);  // in flight under the partial sums
  if (PASS > 0) {
    sum_partials(pin, nin, J, part, hs, red);
    if (blockIdx.x == 0 && (int)threadIdx.x < J) h[threadIdx.x] = hs[threadIdx.x];
  }
  double hj[JW], acc[JW];
#pragma unroll
  for (int k = 0; k < JW; ++k) {
    hj[k] = PASS > 0 && j0 + k < J ? hs[j0 + k] : 0.0;
    acc[k] = 0.0;
  }
  double nrm = 0.0;
  const int64_t end = (N + kRowsElems - 1) / kRowsElems * kRowsElems;  // whole workgroup steps
  for (int64_t base = (int64_t)blockIdx.x * kRowsElems; base < end; base += step, i += step) {
    const bool on = i < N;
    if (base != (int64_t)blockIdx.x * kRowsElems) fetch(i);
    double w0 = on ? wi[0] : 0.0, w1 = on ? wi[1] : 0.0;
    if (PASS > 0) {
      // the first wave contributes w minus its rows' share, the others minus
      // theirs
      double s0 = w0, s1 = w1;
#pragma unroll
      for (int k = 0; k < JW; ++k) {
        s0 = fma(-(double)raw[k][0], hj[k], s0);
        s1 = fma(-(double)raw[k][1], hj[k], s1);
      }
      sub[wv][lane] = kr_f64x2{s0, s1};
      __syncthreads();
      const kr_f64x2 t0 = sub[0][lane], t1 = sub[1][lane], t2 = sub[2][lane], t3 = sub[3][lane];
      __syncthreads();
      w0 = on ? t0[0] + (t1[0] + (t2[0] + t3[0])) : 0.0;
      w1 = on ? t0[1] + (t1[1] + (t2[1] + t3[1])) : 0.0;
      if (on && wv == 0) *reinterpret_cast<kr_f64x2*>(w + i) = kr_f64x2{w0, w1};
    }
    if (PASS < 2) {
#pragma unroll
      for (int k = 0; k < JW; ++k)
        acc[k] = fma((double)raw[k][0], w0, fma((double)raw[k][1], w1, acc[k]));
    } else {
      nrm = fma(w0, w0, fma(w1, w1, nrm));
    }
  }
  double* out = pout + (int64_t)blockIdx.x * kPartStride;
  if (PASS < 2) {
    const double t = lane_totals<JW>(acc);
    const int j = j0 + cgs_row_of<JW>(lane);
    if ((lane & (64 / JW - 1)) == 0 && j < J) out[j] = t;
  } else if (wv == 0) {
    const double t = wave_sum(nrm);
    if (lane == 0) out[0] = t;
  }
}

// Workgroups of one rows pass.
static int rows_blocks(int64_t N, int count) {
  const int cap = count > 1 ? std::max(2048 / count, 16) : kRowsBlocks;
  return (int)std::min<int64_t>(std::min(cap, kRowsBlocks), (N + kRowsElems - 1) / kRowsElems);
}

// The rows form takes even lengths up to 2^17 (every workgroup sums all
// partials, and a lane's loads are one element pair at a time: past that the
// streaming kernels above, with their reductions, are faster).
static bool rows_form(int64_t N) { return N % 2 == 0 && N >= 2 && N <= ((int64_t)1 << 17); }

// w orthogonalised twice against V[0..J-1] by the rows form: h1 and h2 hold
// the two passes' sums on return; |w|^2 stays in the third pass's partials,
// for finish_step.
template <typename VT>
static int cgs2_rows(const VT* V, int64_t ldv, int J, double* w, double* partials, double* h1, double* h2,
                     int64_t N, hipStream_t s, PMap pm = kOne, int count = 1) {
  TNX_CHECK_ARG(J >= 1 && J <= kMaxBasis, "cgs2_rows: J=%d out of range", J);
  const int nb = rows_blocks(N, count);
  double* p0 = partials;
  double* p1 = p0 + (size_t)kRowsBlocks * kPartStride;
  double* p2 = p1 + (size_t)kRowsBlocks * kPartStride;
  const dim3 grid(nb, count), block(256);
  auto go = [&](auto jt) {
    constexpr int JW = decltype(jt)::value;
    hipLaunchKernelGGL((cgs_rows_kernel<JW, 0, VT>), grid, block, 0, s, V, ldv, J, w, (const double*)nullptr, 0,
                       (double*)nullptr, p0, N, pm);
    hipLaunchKernelGGL((cgs_rows_kernel<JW, 1, VT>), grid, block, 0, s, V, ldv, J, w, (const double*)p0, nb, h1, p1,
                       N, pm);
    hipLaunchKernelGGL((cgs_rows_kernel<JW, 2, VT>), grid, block, 0, s, V, ldv, J, w, (const double*)p1, nb, h2, p2,
                       N, pm);
  };
  if (J <= 16) go(std::integral_constant<int, 4>{});
  else if (J <= 32) go(std::integral_constant<int, 8>{});
  else go(std::integral_constant<int, 16>{});
  TNX_LAUNCH_CHECK();
  return TNX_OK;
}

// out[i] = sum_j c[j] V[j][i]   (Ritz vector from the basis)
template <typename VT>
__global__ void vcomb_kernel(const VT* __restrict__ V, int64_t ldv, int J,
                             const double* __restrict__ c, double* __restrict__ out, int64_t N,
                             PMap pm) {
  {
    const int64_t o = pm.off();
    V += o; c += o; out += o;
  }
  __shared__ double cs[kMaxBasis + 1];
  if ((int)threadIdx.x < J) cs[threadIdx.x] = c[threadIdx.x];
  __syncthreads();
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < N;
       i += (int64_t)gridDim.x * blockDim.x) {
    double acc = 0.0;
    for (int j = 0; j < J; ++j) acc += cs[j] * (double)V[(int64_t)j * ldv + i];
    out[i] = acc;
  }
}

// out = x / sqrt(*nrm2)  (unit vector; zero if the norm underflows)
template <typename OT>
__global__ void normalize_kernel(const double* __restrict__ x, const double* __restrict__ nrm2,
                                 OT* __restrict__ out, int64_t N, PMap pm) {
  {
    const int64_t o = pm.off();
    x += o; nrm2 += o; out += o;
  }
  const double n2 = *nrm2;
  const double inv = n2 > 0.0 ? 1.0 / sqrt(n2) : 0.0;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < N;
       i += (int64_t)gridDim.x * blockDim.x)
    out[i] = (OT)(x[i] * inv);
}

// out = (double)x
__global__ void to_f64_kernel(const float* __restrict__ x, double* __restrict__ out, int64_t N) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < N;
       i += (int64_t)gridDim.x * blockDim.x)
    out[i] = (double)x[i];
}

// out = (float)x (the first vector of a low-precision Krylov basis)
__global__ void to_f32_kernel(const double* __restrict__ x, float* __restrict__ out, int64_t N) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < N;
       i += (int64_t)gridDim.x * blockDim.x)
    out[i] = (float)x[i];
}

// out = (*a) * x + (*b) * z, scalars read from device memory. Batched:
// a, x, b, z move with the problem map, out by so doubles per problem.
__global__ void axpbz_dev_kernel(const double* __restrict__ a, const double* __restrict__ x,
                                 const double* __restrict__ b, const double* __restrict__ z,
                                 double* __restrict__ out, int64_t N, PMap pm, int64_t so) {
  {
    const int64_t o = pm.off();
    a += o; x += o;
    if (b) b += o;
    if (z) z += o;
    out += (int64_t)pm.pid() * so;
  }
  const double av = *a, bv = b ? *b : 0.0;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < N;
       i += (int64_t)gridDim.x * blockDim.x)
    out[i] = av * x[i] + (z ? bv * z[i] : 0.0);
}

__global__ void axpy_kernel(int64_t n, double a, const double* __restrict__ x, double* __restrict__ y) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    y[i] += a * x[i];
}
__global__ void scal_kernel(int64_t n, double a, double* __restrict__ x) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    x[i] *= a;
}

static int vec_blocks(int64_t N, int count = 1) {
  return (int)std::min<int64_t>((N + 255) / 256, count > 1 ? std::max(4096 / count, 8) : 4096);
}

// A Lanczos step's orthogonalisation: w against V[0..J-1], twice; then
// finish_step makes V[J] = w / |w|. Sums in h1, h2, and |w|^2 in h3[J] (by
// finish_step where the rows form runs).
template <typename VT>
static int cgs_step(const VT* V, int64_t N, int J, double* w, double* partials, double* h1, double* h2,
                    double* h3, hipStream_t s, PMap pm = kOne, int count = 1) {
  if (rows_form(N)) return cgs2_rows(V, N, J, w, partials, h1, h2, N, s, pm, count);
  TNX_TRY(cgs_pass(V, N, J, w, nullptr, true, partials, h1, N, s, pm, count));
  TNX_TRY(cgs_pass(V, N, J, w, h1, true, partials, h2, N, s, pm, count));
  return cgs_pass(V, N, J, w, h2, false, partials, h3, N, s, pm, count);
}

// out_p = in_p for the mapped problems: in moves with the map (sp), out by so.
__global__ void copy_map_kernel(const double* __restrict__ in, double* __restrict__ out,
                                int64_t N, PMap pm, int64_t sin_, int64_t so) {
  const int64_t p = pm.pid();
  in += p * sin_;
  out += p * so;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < N;
       i += (int64_t)gridDim.x * blockDim.x)
    out[i] = in[i];
}

// ---------------------------------------------------------------------------
// Symmetric tridiagonal lowest eigenpair, one wavefront.
// diag a[0..n-1], off-diagonal b[0..n-2]. Writes the unit eigenvector to
// s[0..n-1] and status: st[0] = theta, st[1] = |bres * s[n-1]| (Lanczos
// residual estimate, bres read from *bres if given), st[2] = max row sum
// (estimate of ||T||, a lower bound of ||H||).
// ---------------------------------------------------------------------------
constexpr int kTriMax = 256;

// Orders one wave's LDS writes before its later reads of other lanes'
// values (LDS serves a wave's instructions in order; this keeps the compiler
// from moving them).
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The rows of T in LDS, {a_k, b_{k-1}^2}, padded by a zero row so that loads
// may run past the end; and the minors of the twisted factorisation.
struct TriLds {
  double2 row[kTriMax + 16];
  double2 q[2][kTriMax];
};

// One evaluation of the characteristic polynomial at x (a point per lane):
// `cnt` = number of eigenvalues below x, from the sign changes of the leading
// principal minors p_k = det(T_k - x I) (p_0 = 1), and `g` = -p'/p = sum_i
// 1 / (lambda_i - x). Three-term recurrences without divisions; every 4 rows
// the carried minors and derivatives are rescaled by a power of two so they
// neither overflow nor underflow. An exact zero minor takes the sign opposite
// to its predecessor (the pivot convention q = -0). The rows come from LDS as
// broadcasts, four in flight ahead of their use.
__device__ __forceinline__ void char_poly(const double2* row, int n, double x, int& cnt, double& g) {
  double pm = 0.0, p = 1.0, dm = 0.0, d = 0.0;
  bool neg_prev = false;
  int c = 0;
  auto step = [&](const double2& r) {
    const double t = r.x - x;
    const double pn = fma(t, p, -r.y * pm);
    const double dn = fma(t, d, fma(-r.y, dm, -p));
    pm = p; dm = d;
    p = pn; d = dn;
    const bool neg = (p < 0.0) | ((p == 0.0) & !neg_prev);
    c += (int)(neg ^ neg_prev);
    neg_prev = neg;
  };
  auto rescale = [&]() {
    const int e = __builtin_amdgcn_frexp_exp(p == 0.0 ? pm : p);
    p = ldexp(p, -e);
    pm = ldexp(pm, -e);
    d = ldexp(d, -e);
    dm = ldexp(dm, -e);
  };
  double2 cur[4], nxt[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) cur[u] = row[u];
  int i = 0;
  for (; i + 4 <= n; i += 4) {
#pragma unroll
    for (int u = 0; u < 4; ++u) nxt[u] = row[i + 4 + u];
#pragma unroll
    for (int u = 0; u < 4; ++u) step(cur[u]);
    rescale();
#pragma unroll
    for (int u = 0; u < 4; ++u) cur[u] = nxt[u];
  }
#pragma unroll
  for (int u = 0; u < 3; ++u)
    if (i + u < n) step(cur[u]);
  cnt = c;
  g = -d / p;
}

// Pivots of T - x I from both ends: lanes 0..31 run down the leading minors,
// 32..63 up the trailing ones; q[0][k] = {p_{k+1}, p_k}, whose ratio is the
// pivot of row k, q[1][k] the same from below.
__device__ __forceinline__ void twisted_minors(TriLds& t, int n, double x) {
  const int lane = threadIdx.x;
  const bool up = lane >= 32, wr = (lane & 31) == 0;
  const double2* ra = up ? t.row + (n - 1) : t.row;  // a of this direction's row i at ra[i * dir]
  const double2* rb = up ? t.row + n : t.row;        // its coupling to row i - 1 (row n is zero)
  double2* qo = up ? t.q[1] + (n - 1) : t.q[0];
  const int dir = up ? -1 : 1;
  double pm = 0.0, p = 1.0;
  auto rescale = [&]() {
    const int e = __builtin_amdgcn_frexp_exp(p == 0.0 ? pm : p);
    p = ldexp(p, -e);
    pm = ldexp(pm, -e);
  };
  auto step = [&](double av, double bv, int i) {
    const double pn = fma(av - x, p, -bv * pm);
    if (wr) qo[i * dir] = make_double2(pn, p);
    pm = p;
    p = pn;
  };
  int i = 0;
  for (; i + 4 <= n; i += 4) {
    double av[4], bv[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      av[u] = ra[(i + u) * dir].x;
      bv[u] = rb[(i + u) * dir].y;
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) step(av[u], bv[u], i + u);
    rescale();
  }
  for (; i < n; ++i) step(ra[i * dir].x, rb[i * dir].y, i);
}

// The same pivots by their own recurrence q_k = a_k - x - b_{k-1}^2 / q_{k-1},
// {q_k, 1}, where one below `tiny` is replaced by it before the next is formed.
// A minor that is zero, or a rounding error, leaves a finite pivot behind it
// that belongs to a matrix within `tiny` of T. A reciprocal a row instead of
// two products (80 cycles against 16).
__device__ __forceinline__ void twisted_pivots(TriLds& t, int n, double x, double tiny) {
  const int lane = threadIdx.x;
  const bool up = lane >= 32, wr = (lane & 31) == 0;
  const double2* ra = up ? t.row + (n - 1) : t.row;
  const double2* rb = up ? t.row + n : t.row;
  double2* qo = up ? t.q[1] + (n - 1) : t.q[0];
  const int dir = up ? -1 : 1;
  double q = 0.0;
  for (int i = 0; i < n; ++i) {
    const double c = i > 0 ? rb[i * dir].y * rcp_nr(q) : 0.0;
    q = ra[i * dir].x - x - c;
    if (!(fabs(q) >= tiny)) q = tiny;
    if (wr) qo[i * dir] = make_double2(q, 1.0);
  }
}

// The lowest eigenpair for n <= 64 NC (NC = 1: every Lanczos projection), by
// one wave; row k = 64 c + lane in register c of its lane.
//
// What bounds it is the length of the serial chains: n dependent rows per
// evaluation of the polynomial. Evenly spaced 64-point rounds gain 6 bits
// each, about nine evaluations; here a round's points crowd around a
// prediction of the root instead (two or three evaluations), and the
// eigenvector comes from a twisted factorisation (Parlett and Dhillon,
// "Fernando's solution to Wilkinson's problem", 1997): both ends' pivots in
// one pass, then products of ratios, which are scans over the lanes, in
// place of a pivoted LU and four triangular solves. Measured over a solve
// (n = 2..64): 25 -> 9.5 us; at n = 64 alone 36 -> 15.
template <int NC>
__device__ __forceinline__ void tridiag_lowest_wave(TriLds& t, const double* __restrict__ ad, const double* __restrict__ bd,
                                    int n, bool has_bres, double bres_v, bool fin, double a_last,
                                    double* __restrict__ s, double* st, int hinted) {
  const int lane = threadIdx.x;
  // the previous call's theta (st[0]), read before this call overwrites it
  double hint_in = hinted ? st[0] : 0.0;
  double ar[NC], bl[NC], bn[NC];  // a_k, b_{k-1}, b_k
  double lo = 1e308, hi = 1e308, tnorm = 0.0;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int k = 64 * c + lane;
    ar[c] = k < n ? ((fin && k == n - 1) ? a_last : ad[k]) : 0.0;
    bn[c] = k < n - 1 ? bd[k] : 0.0;
    bl[c] = k > 0 && k < n ? bd[k - 1] : 0.0;
    t.row[k] = make_double2(ar[c], bl[c] * bl[c]);
    // Gershgorin bounds and ||T|| estimate
    const double r = fabs(bl[c]) + fabs(bn[c]);
    if (k < n) {
      lo = fmin(lo, ar[c] - r);
      hi = fmin(hi, ar[c]);
      tnorm = fmax(tnorm, fabs(ar[c]) + r);
    }
  }
  if (lane < 16) t.row[64 * NC + lane] = make_double2(0.0, 0.0);
  wave_lds_fence();
  lo = wave_min(lo);
  hi = wave_min(hi);
  tnorm = wave_max(tnorm);
  // far from 1 the products of rows would leave the range: by a power of two
  int ex = __builtin_amdgcn_frexp_exp(tnorm);
  if (ex < -64 || ex > 64) {
    lo = ldexp(lo, -ex);
    hi = ldexp(hi, -ex);
    tnorm = ldexp(tnorm, -ex);
    hint_in = ldexp(hint_in, -ex);
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      ar[c] = ldexp(ar[c], -ex);
      bn[c] = ldexp(bn[c], -ex);
      bl[c] = ldexp(bl[c], -ex);
      t.row[64 * c + lane] = make_double2(ar[c], bl[c] * bl[c]);
    }
    wave_lds_fence();
  } else {
    ex = 0;
  }
  const double pivmin = fmax(tnorm, 1e-300) * 1e-300 + 1e-300;
  const double eps = 2.220446049250313e-16;
  // d0 times 2^(e k), k this lane's place: a geometric spacing
  auto spaced = [&](double d0, float e, int k) {
    const float x = e * (float)k, fl = floorf(x);
    return d0 * ldexp((double)exp2f(x - fl), (int)fl);
  };
  auto log2_ratio = [](double a, double b) {  // at least log2(a / b), a >= b > 0
    return (float)(__builtin_amdgcn_frexp_exp(a) - __builtin_amdgcn_frexp_exp(b) + 1);
  };
  // Multisection. The 64 points of a round may be any non-decreasing sequence
  // in [lo, hi]: the first with a count >= 1 and its predecessor bracket the
  // lowest eigenvalue whatever the points are. First round: spaced
  // geometrically below a hint h (the lowest Ritz value of the previous
  // Lanczos step, an upper bound of this one by interlacing, usually just
  // above it) with one point above it, or evenly without a hint. Later
  // rounds: geometrically to both sides of a prediction. With u = lambda - x2
  // and two points x1 < x2 = x1 + h left of the root, g(x2) - g(x1) = 1/u -
  // 1/(u + h) up to the change of the other eigenvalues' share over h, a
  // quadratic in u; the bracket then shrinks to the prediction's error. A
  // round that does not shrink the bracket 16-fold (a bad hint or
  // prediction) is followed by an even one, so it costs one round, never the
  // result.
  double h = hint_in;
  if (!(h > lo && h <= hi)) h = hi;
  const double dmin = 2.0 * eps * fabs(h) + pivmin;
  bool below = hinted && (h - lo) > 4.0 * dmin;  // first round: below the hint
  bool around = false;                           // around the prediction `ctr`
  double ctr = 0.0;
  for (int it = 0; it < 24; ++it) {
    if (hi - lo <= 4.0 * eps * fmax(fabs(lo), fabs(hi)) + pivmin) break;
    const double width = hi - lo;
    double x;
    if (below) {
      // lanes 0..62 from far below up to h - dmin, lane 63 just above h: a
      // Ritz value that has converged is bracketed at once
      x = lane < 63 ? h - spaced(dmin, log2_ratio(h - lo, dmin) / 62.0f, 62 - lane) : h + dmin;
      x = fmin(fmax(x, lo), hi);
    } else if (around) {
      // lanes 0..31: ctr - delta, largest first; 32..63: ctr + delta
      const double d0 = 1.5 * eps * fmax(fabs(lo), fabs(hi)) + pivmin;
      const double dl = spaced(d0, log2_ratio(fmax(width, 2.0 * d0), d0) / 31.0f, lane < 32 ? 31 - lane : lane - 32);
      x = lane < 32 ? ctr - dl : ctr + dl;
      x = fmin(fmax(x, lo), hi);
    } else {
      x = lo + width * (double)(lane + 1) / 65.0;
    }
    int cnt;
    double g;
    char_poly(t.row, n, x, cnt, g);
    const unsigned long long mask = __ballot(cnt >= 1);
    const int f = mask == 0ull ? 64 : __ffsll((long long)mask) - 1;
    const double xl = lane_val(x, f > 0 ? f - 1 : 0);
    if (f < 64) hi = lane_val(x, f);
    if (f > 0) lo = xl;
    // predict from the two points left of the root
    const bool was_even = !(below || around);
    below = false;
    around = false;
    if (f >= 2 && (was_even || (hi - lo) * 16.0 <= width)) {
      const double x1 = lane_val(x, f - 2), gd = lane_val(g, f - 1) - lane_val(g, f - 2);
      const double hh = xl - x1;
      if (hh > 0.0 && gd > 0.0) {
        const double q = 4.0 * hh / gd;
        ctr = xl + 0.5 * q / (hh + sqrt(fma(hh, hh, q)));
        around = ctr > lo && ctr < hi;
      }
    }
  }
  const double theta = 0.5 * (lo + hi);
  // Eigenvector: pivots q+ from above and q- from below; row r where
  // gamma = q+ + q- - (a - theta) is smallest is where the two meet, and
  // z_r = 1, z_k = -b_k / q+_k z_{k+1} above it, -b_{k-1} / q-_k z_{k-1}
  // below. The pivots come from ratios of minors, which lose them where the
  // lowest level is degenerate: a level that two uncoupled blocks share makes
  // the minors from both ends zero, and 0 / 0 says nothing of r; blocks coupled
  // at rounding level give two nearly singular pivots that cancel (residuals up
  // to 1e-11 |T|). So the residual is looked at, and a vector beyond 6 eps |T|
  // (the others stay below 5.5) is formed again from the guarded recurrence,
  // whose residuals stay below that on such matrices too.
  const double tiny = fmax(eps * tnorm, 1e-290);
  double z[NC], nn = 0.0, mx = 0.0;
  auto twisted = [&]() {
    double up[NC], dn[NC], gam[NC], gmin = 1e308;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int k = 64 * c + lane;
      up[c] = dn[c] = 1.0;
      gam[c] = 1e308;
      if (k < n) {
        const double2 a = t.q[0][k], b = t.q[1][k];
        double qp = a.x / a.y, qm = b.x / b.y;
        const double gm = fabs(qp + qm - (ar[c] - theta));
        if (gm < 1e308) gam[c] = gm;  // not for a NaN or an infinity
        if (!(fabs(qp) >= tiny)) qp = tiny;
        if (!(fabs(qm) >= tiny)) qm = tiny;
        up[c] = -bn[c] / qp;
        dn[c] = -bl[c] / qm;
      }
      gmin = fmin(gmin, gam[c]);
    }
    gmin = wave_min(gmin);
    int r = -1;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const unsigned long long at = __ballot(gam[c] == gmin && 64 * c + lane < n);
      if (r < 0 && at != 0ull) r = 64 * c + __ffsll((long long)at) - 1;
    }
    double carry = 1.0;
    // below r: running products downwards
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int k = 64 * c + lane;
      double f = k > r && k < n ? dn[c] : 1.0;
      for (int o = 1; o < 64; o <<= 1) {
        const double v = __shfl_up(f, o, 64);
        if (lane >= o) f *= v;
      }
      z[c] = f * carry;
      if (NC > 1) carry = lane_val(z[c], 63);
    }
    // above r: running products upwards
    carry = 1.0;
#pragma unroll
    for (int c = NC - 1; c >= 0; --c) {
      const int k = 64 * c + lane;
      double f = k < r ? up[c] : 1.0;
      for (int o = 1; o < 64; o <<= 1) {
        const double v = __shfl_down(f, o, 64);
        if (lane + o < 64) f *= v;
      }
      f *= carry;
      if (NC > 1) carry = lane_val(f, 0);
      z[c] = k < n ? z[c] * f : 0.0;
    }
    nn = 0.0;
    mx = 0.0;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      nn += z[c] * z[c];
      mx = fmax(mx, fabs(z[c]));
    }
    nn = wave_sum(nn);
    mx = wave_max(mx);
  };
  twisted_minors(t, n, theta);
  wave_lds_fence();
  twisted();
  double rm = 0.0;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    double zu = dpp<0x138>(z[c]), zd = dpp<0x130>(z[c]);  // wave_shr 1, wave_shl 1
    if (c > 0 && lane == 0) zu = lane_val(z[c > 0 ? c - 1 : 0], 63);
    if (c + 1 < NC && lane == 63) zd = lane_val(z[c + 1 < NC ? c + 1 : c], 0);
    const double rk = fabs(fma(ar[c] - theta, z[c], fma(bl[c], zu, bn[c] * zd)));
    rm = fmax(rm, 64 * c + lane < n ? (rk <= 1e300 ? rk : 1e308) : 0.0);  // a NaN counts
  }
  rm = wave_max(rm);
  const double lim = 6.0 * eps * tnorm;
  if (!(rm * rm <= lim * lim * nn && nn < 1e200)) {
    wave_lds_fence();
    twisted_pivots(t, n, theta, tiny);
    wave_lds_fence();
    twisted();
  }
  // unit length; sign: largest |component| positive, the first such index on
  // ties
  double sg = 1.0 / sqrt(nn), zl = 0.0;
  bool found = false;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const unsigned long long at = __ballot(64 * c + lane < n && fabs(z[c]) == mx);
    if (!found && at != 0ull) {
      if (lane_val(z[c], __ffsll((long long)at) - 1) < 0.0) sg = -sg;
      found = true;
    }
    if ((n - 1) / 64 == c) zl = lane_val(z[c], (n - 1) % 64);
  }
  if (lane == 0) {
    st[0] = ldexp(theta, ex);
    st[1] = has_bres ? fabs(bres_v * zl * sg) : 0.0;
    st[2] = ldexp(tnorm, ex);
  }
#pragma unroll
  for (int c = 0; c < NC; ++c)
    if (64 * c + lane < n) s[64 * c + lane] = sg * z[c];
}

// The end of a Lanczos step, folded into the solve that follows it: from
// the step's CGS sums, alpha[j] = h1[j] + h2[j] and beta[j] = |w|
// (j = n - 1, the new row; beta[j] is also the residual coupling), written to
// alpha, beta and the dense T. h1 == nullptr: no step to finish.
struct TriFinish {
  const double* h1; const double* h2;
  double* alpha; double* beta; double* T;
};

// hinted: st[0] holds the lowest eigenvalue of the previous, one row
// smaller projection of the same Lanczos run (a search hint only).
// With a step to finish (f.h1), ad is f.alpha, the new row's alpha and the
// coupling come from the sums directly (|w|^2 = n2; every lane computes them;
// lane 0 stores them for the later users), never through memory in this
// kernel.
// Device-decided convergence for a batched run that reads the statuses only
// every few steps (ctol >= 0; negative switches it off): st[12] keeps the running ||T|| estimate (the
// criterion's anorm); once est <= ctol * anorm, st[10] = 1 and st[11] = n,
// and the problem's later calls return at once, leaving its Ritz pair
// (st[0..2], s) and the basis rows up to n as they were at convergence.
__device__ __forceinline__ void chunk_mark(double* st, int n, double ctol) {
  if (ctol >= 0.0 && threadIdx.x == 0) {
    const double an = fmax(st[12], st[2]);
    st[12] = an;
    if (st[1] <= ctol * an) {
      st[10] = 1.0;
      st[11] = (double)n;
    }
  }
}

// One wave (threads 0..63); the pointers are the problem's own.
template <int NC>
__device__ __forceinline__ void tridiag_lowest_problem(TriLds& t, const double* ad, const double* bd, int n,
                                                       double* s, double* st, int hinted, const TriFinish& f,
                                                       double n2, double ctol) {
  if (ctol >= 0.0 && st[10] != 0.0) return;
  const bool fin = f.h1 != nullptr;
  double a_last = 0.0, b_new = 0.0;
  if (fin) {
    const int j = n - 1;
    a_last = f.h1[j] + f.h2[j];
    b_new = sqrt(fmax(n2, 0.0));
    if (threadIdx.x == 0) {
      f.alpha[j] = a_last;
      f.beta[j] = b_new;
      f.T[j * kMaxBasis + j] = a_last;
      if (j + 1 < kMaxBasis) {
        f.T[j * kMaxBasis + j + 1] = b_new;
        f.T[(j + 1) * kMaxBasis + j] = b_new;
      }
    }
  }
  if (n == 1) {
    if (threadIdx.x == 0) {
      const double a0 = fin ? a_last : ad[0];
      s[0] = 1.0;
      st[0] = a0;
      st[1] = fin ? fabs(b_new) : 0.0;
      st[2] = fabs(a0);
    }
  } else if (NC == 1 || n <= 64) {
    tridiag_lowest_wave<1>(t, ad, bd, n, fin, b_new, fin, a_last, s, st, hinted);
  } else {
    tridiag_lowest_wave<NC>(t, ad, bd, n, fin, b_new, fin, a_last, s, st, hinted);
  }
  chunk_mark(st, n, ctol);
}

// The dense eigensolver's projected problem (n <= kTriMax).
__global__ __launch_bounds__(64) void tridiag_lowest_kernel(const double* __restrict__ ad,
                                                            const double* __restrict__ bd, int n,
                                                            double* __restrict__ s, double* st, PMap pm) {
  __shared__ TriLds t;
  const int64_t o = pm.off();
  tridiag_lowest_problem<4>(t, ad + o, bd + o, n, s + o, st + o, 0, TriFinish{}, 0.0, -1.0);
}

// The end of Lanczos step J - 1 in one launch: workgroup 0 solves the
// projected problem (n = J rows; alpha, beta and T get the new row), the
// others write V[J] = w / |w| (a zero norm gives a zero vector). |w|^2: with
// the rows form's partials `pin`, summed by every workgroup and stored to
// h3[J]; else (pin null) read from h3[J]. host_st (a pinned host block, or
// null) receives st[0..2], which saves a copy between the solve and the
// host's wait.
// Bound by the one wave's serial chain (9 us at n = 45, against 3 for the
// vector), so the vector is free; as two launches 13 us.
template <typename VT>
__global__ __launch_bounds__(256, 4) void finish_step_kernel(const double* __restrict__ w, VT* __restrict__ V,
                                                          int64_t N, int J, const double* __restrict__ pin,
                                                          int nin, double* __restrict__ h3, double* s,
                                                          double* st, TriFinish f, double ctol,
                                                          double* __restrict__ host_st, PMap pm) {
  __shared__ TriLds t;
  __shared__ double red[4];
  const int64_t o = pm.off();
  const int lane = threadIdx.x & 63;
  h3 += o;
  double n2;
  if (pin) {
    pin += o;
    double a[3];  // nin <= 3 * 64, in the same order in every workgroup
#pragma unroll
    for (int q = 0; q < 3; ++q) a[q] = 64 * q + lane < nin ? pin[(int64_t)(64 * q + lane) * kPartStride] : 0.0;
    if (blockIdx.x == 0) {
      if (threadIdx.x >= 64) return;
      n2 = (wave_sum(a[0]) + wave_sum(a[1])) + wave_sum(a[2]);
      if (threadIdx.x == 0) h3[J] = n2;
    } else {
      const int wv = threadIdx.x >> 6;
      if (wv < 3) {
        const double v = wave_sum(wv == 0 ? a[0] : (wv == 1 ? a[1] : a[2]));
        if (lane == 0) red[wv] = v;
      }
      __syncthreads();
      n2 = (red[0] + red[1]) + red[2];
    }
  } else {
    if (blockIdx.x == 0 && threadIdx.x >= 64) return;
    n2 = h3[J];
  }
  if (blockIdx.x == 0) {
    f.h1 += o; f.h2 += o; f.alpha += o; f.beta += o; f.T += o;
    s += o; st += o;
    tridiag_lowest_problem<1>(t, f.alpha, f.beta, J, s, st, 1, f, n2, ctol);
    if (host_st && threadIdx.x == 0)
      for (int q = 0; q < 3; ++q) host_st[q] = st[q];
    return;
  }
  w += o;
  VT* v = V + o + (int64_t)J * N;
  const double inv = n2 > 0.0 ? 1.0 / sqrt(n2) : 0.0;
  for (int64_t i = (int64_t)(blockIdx.x - 1) * blockDim.x + threadIdx.x; i < N;
       i += (int64_t)(gridDim.x - 1) * blockDim.x)
    v[i] = (VT)(w[i] * inv);
}

// nin: the partial rows that the step's cgs_step wrote, rows_blocks of the
// count it was launched with (fewer problems may be left by now).
template <typename VT>
static int finish_step(VT* V, int64_t N, int J, const double* w, const double* partials, int nin, double* h3,
                       double* sv, double* st, const TriFinish& f, double ctol, double* host_st, hipStream_t s,
                       PMap pm = kOne, int count = 1) {
  const bool rows = rows_form(N);
  // at N = 2^21 a lane writes 8 elements
  const int nb = std::min(vec_blocks(N, count), rows ? 256 : 1024);
  hipLaunchKernelGGL(finish_step_kernel<VT>, dim3(nb + 1, count), dim3(256), 0, s, w, V, N, J,
                     rows ? partials + (size_t)2 * kRowsBlocks * kPartStride : nullptr, nin, h3, sv, st, f, ctol, host_st,
                     pm);
  TNX_LAUNCH_CHECK();
  return TNX_OK;
}

// ---------------------------------------------------------------------------
// Dense symmetric tridiagonalisation (one workgroup) and back-transform.
// Householder reflectors H_k = I - tau_k v_k v_k^T act on indices k+1..n-1.
// ---------------------------------------------------------------------------
// Tridiagonalisation with the matrix in registers: 16 lanes hold R rows, C
// elements of each (in pairs of columns), so a step is two barriers: the
// product p = tau A v with v from LDS (sums inside the 16 lanes), and the
// rank-2 update with w = p - (tau p.v / 2) v, after which the 16 lanes of the
// next row form the next reflector alone. M (stride sM between problems) is
// read once and left as it is. Bound by the latency of those steps: at n = 64 and
// 128 64 and 205 us, where a thread per row, its row read from L2, took 620 and
// 2490; at n = 192 1860 against 6000.
template <int R, int C, int NG>
__global__ __launch_bounds__(16 * NG) void sytrd_reg_kernel(const double* __restrict__ M, int64_t sM, int n,
                                                            double* __restrict__ Vst, double* __restrict__ tau,
                                                            double* __restrict__ dg, double* __restrict__ eg,
                                                            PMap pm) {
  {
    const int64_t o = pm.off();
    Vst += o; tau += o; dg += o; eg += o;
    M += (int64_t)pm.pid() * sM;
  }
  constexpr int NR = 16 * C;
  static_assert(R * NG == NR && NG <= 64 && C % 2 == 0, "square, one partial per lane, columns in pairs");
  __shared__ __attribute__((aligned(16))) double v[NR], p[NR];
  __shared__ double part[NG], tks;
  const int t = threadIdx.x, lane = t & 63, s = t & 15, g = t >> 4;
  auto col = [&](int c) { return 2 * (s + 16 * (c >> 1)) + (c & 1); };
  double a[R][C];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const int i = R * g + r, j = col(c);
      a[r][c] = i < n && j < n ? M[(int64_t)i * n + j] : 0.0;
    }
  // the reflector of row k, by the 16 lanes that hold it
  auto reflect = [&](int k) {
    double x[C], sig = 0.0, al = 0.0;
    const int rk = k % R;
#pragma unroll
    for (int c = 0; c < C; ++c) {
      x[c] = a[0][c];
#pragma unroll
      for (int r = 1; r < R; ++r) x[c] = rk == r ? a[r][c] : x[c];
      const int j = col(c);
      sig = fma(j > k + 1 ? x[c] : 0.0, x[c], sig);
      al += j == k + 1 ? x[c] : 0.0;
    }
    sig = sum16(sig);
    al = sum16(al);
    double tk = 0.0, beta = al, sc = 0.0;
    if (sig != 0.0) {
      const double n2 = fma(al, al, sig), rs = rsqrt_nr(n2), nrm = n2 * rs;
      beta = al >= 0.0 ? -nrm : nrm;
      tk = fma(fabs(al), rs, 1.0);  // (beta - al) / beta
      sc = rcp_nr(al - beta);
    }
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const int j = col(c);
      const double y = j <= k ? 0.0 : (j == k + 1 ? 1.0 : x[c] * sc);
      v[j] = y;
      if (j > k && j < n) Vst[(int64_t)k * n + j - k - 1] = y;
    }
    if (s == 0) {
      tau[k] = tk;
      eg[k] = beta;
      tks = tk;
    }
  };
  for (int i = t; i < NR; i += 16 * NG) v[i] = 0.0;
  __syncthreads();
  if (g == 0 && n > 2) reflect(0);
  __syncthreads();
  for (int k = 0; k + 2 < n; ++k) {
    const double tk = tks;
    double vj[C], vi[R], pi[R], pv = 0.0;
#pragma unroll
    for (int c = 0; c < C; ++c) vj[c] = v[col(c)];
#pragma unroll
    for (int r = 0; r < R; ++r) vi[r] = v[R * g + r];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      double e = 0.0, f = 0.0;
#pragma unroll
      for (int c = 0; c < C; c += 2) {
        e = fma(a[r][c], vj[c], e);
        f = fma(a[r][c + 1], vj[c + 1], f);
      }
      pi[r] = e + f;
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
      pi[r] = R * g + r > k ? tk * sum16(pi[r]) : 0.0;
      pv = fma(pi[r], vi[r], pv);
    }
    if (s == 0) {
#pragma unroll
      for (int r = 0; r < R; ++r) p[R * g + r] = pi[r];
      part[g] = pv;
    }
    __syncthreads();
    const double K = 0.5 * tk * sum64(lane < NG ? part[lane] : 0.0);
    double wj[C];
#pragma unroll
    for (int c = 0; c < C; ++c) wj[c] = fma(-K, vj[c], p[col(c)]);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const double wi = fma(-K, vi[r], pi[r]);
#pragma unroll
      for (int c = 0; c < C; ++c) a[r][c] = fma(-vi[r], wj[c], fma(-wi, vj[c], a[r][c]));
    }
    if (k + 3 < n && g == (k + 1) / R) reflect(k + 1);
    __syncthreads();
  }
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const int i = R * g + r, j = col(c);
      if (i == j && i < n) dg[i] = a[r][c];
      if (i == n - 1 && j == n - 2) eg[n - 2] = a[r][c];
    }
}

// The same for 192 < n <= 256: A (n x n, global, overwritten) does not fit in
// one workgroup's registers.
__device__ double block_sum(double v, double* red) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  v = wave_sum(v);
  __syncthreads();
  if (lane == 0) red[wv] = v;
  __syncthreads();
  double t = 0.0;
  const int nw = (blockDim.x + 63) >> 6;
  for (int i = 0; i < nw; ++i) t += red[i];
  return t;
}

__global__ __launch_bounds__(256) void sytrd_kernel(double* __restrict__ A, int n,
                                                   double* __restrict__ Vst,
                                                   double* __restrict__ tau,
                                                   double* __restrict__ dg,
                                                   double* __restrict__ eg, PMap pm) {
  {
    const int64_t o = pm.off();
    A += o; Vst += o; tau += o; dg += o; eg += o;
  }
  __shared__ double v[kTriMax], p[kTriMax];
  __shared__ double red[8];
  const int t = threadIdx.x;
  for (int k = 0; k + 2 < n; ++k) {
    const int m = n - k - 1;
    const double alpha = A[(int64_t)(k + 1) * n + k];
    double part = 0.0;
    for (int i = 1 + t; i < m; i += blockDim.x) {
      const double x = A[(int64_t)(k + 1 + i) * n + k];
      part += x * x;
    }
    const double sigma = block_sum(part, red);
    double tk, beta;
    if (sigma == 0.0) {
      tk = 0.0; beta = alpha;
      for (int i = t; i < m; i += blockDim.x) v[i] = (i == 0) ? 1.0 : 0.0;
    } else {
      const double nrm = sqrt(alpha * alpha + sigma);
      beta = alpha >= 0.0 ? -nrm : nrm;
      tk = (beta - alpha) / beta;
      const double sc = 1.0 / (alpha - beta);
      for (int i = t; i < m; i += blockDim.x) v[i] = (i == 0) ? 1.0 : A[(int64_t)(k + 1 + i) * n + k] * sc;
    }
    __syncthreads();
    for (int i = t; i < m; i += blockDim.x) Vst[(int64_t)k * n + i] = v[i];
    if (t == 0) { tau[k] = tk; eg[k] = beta; }
    if (tk != 0.0) {
      // p = tau * A22 v
      for (int i = t; i < m; i += blockDim.x) {
        const double* row = A + (int64_t)(k + 1 + i) * n + (k + 1);
        double acc = 0.0;
        for (int j = 0; j < m; ++j) acc += row[j] * v[j];
        p[i] = tk * acc;
      }
      __syncthreads();
      double pv = 0.0;
      for (int i = t; i < m; i += blockDim.x) pv += p[i] * v[i];
      const double K = 0.5 * tk * block_sum(pv, red);
      for (int i = t; i < m; i += blockDim.x) p[i] -= K * v[i];  // p <- w
      __syncthreads();
      for (int i = t; i < m; i += blockDim.x) {
        double* row = A + (int64_t)(k + 1 + i) * n + (k + 1);
        const double vi = v[i], wi = p[i];
        for (int j = 0; j < m; ++j) row[j] -= vi * p[j] + wi * v[j];
      }
    }
    __syncthreads();
  }
  for (int i = t; i < n; i += blockDim.x) dg[i] = A[(int64_t)i * n + i];
  if (t == 0 && n >= 2) eg[n - 2] = A[(int64_t)(n - 1) * n + (n - 2)];
}

// x = H_0 H_1 ... H_(n-3) z by one wave, Q elements per lane; the reflectors
// are read four steps ahead (n = 64, 128: 53, 105 us with two block sums a step,
// 12, 27 so).
template <int Q>
__global__ __launch_bounds__(64) void ormtr_kernel(const double* __restrict__ Vst, const double* __restrict__ tau,
                                                   int n, const double* __restrict__ zin, double* __restrict__ x,
                                                   PMap pm, int64_t so) {
  {
    const int64_t o = pm.off();
    Vst += o; tau += o; zin += o;
    x += (int64_t)pm.pid() * so;
  }
  const int t = threadIdx.x;
  double xs[Q];
#pragma unroll
  for (int q = 0; q < Q; ++q) xs[q] = t + 64 * q < n ? zin[t + 64 * q] : 0.0;
  double v[4][Q], tk[4];
  auto load = [&](int k0) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int k = k0 - u;
      tk[u] = k >= 0 ? tau[k] : 0.0;
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        const int i = t + 64 * q;
        v[u][q] = k >= 0 && i > k && i < n ? Vst[(int64_t)k * n + i - k - 1] : 0.0;
      }
    }
  };
  load(n - 3);
  for (int k = n - 3; k >= 0; k -= 4) {
    double w[4][Q], f[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      f[u] = tk[u];
#pragma unroll
      for (int q = 0; q < Q; ++q) w[u][q] = v[u][q];
    }
    load(k - 4);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      double d = 0.0;
#pragma unroll
      for (int q = 0; q < Q; ++q) d = fma(w[u][q], xs[q], d);
      d = -f[u] * sum64(d);
#pragma unroll
      for (int q = 0; q < Q; ++q) xs[q] = fma(d, w[u][q], xs[q]);
    }
  }
#pragma unroll
  for (int q = 0; q < Q; ++q)
    if (t + 64 * q < n) x[t + 64 * q] = xs[q];
}

// Tridiagonal form of `batch` matrices M (stride sM between them) by the form
// that holds them in registers; A is workspace for those that do not fit.
static int sytrd(const double* M, int64_t sM, int n, double* A, double* Vst, double* tau, double* dg, double* eg,
                 int batch, PMap pm, hipStream_t s) {
#define TNX_SYTRD(R_, C_, NG_)                                                                                     \
  hipLaunchKernelGGL((sytrd_reg_kernel<R_, C_, NG_>), dim3(1, batch), dim3(16 * NG_), 0, s, M, sM, n, Vst, tau, dg, \
                     eg, pm)
  if (n <= 32) {
    TNX_SYTRD(2, 2, 16);
  } else if (n <= 64) {
    TNX_SYTRD(2, 4, 32);
  } else if (n <= 128) {
    TNX_SYTRD(2, 8, 64);
  } else if (n <= 192) {
    TNX_SYTRD(6, 12, 32);
  } else {
    const int64_t nn = (int64_t)n * n;
    hipLaunchKernelGGL(copy_map_kernel, dim3(vec_blocks(nn, batch), batch), dim3(256), 0, s, M, A, nn, pm, sM,
                       pm.sp);
    TNX_LAUNCH_CHECK();
    hipLaunchKernelGGL(sytrd_kernel, dim3(1, batch), dim3(256), 0, s, A, n, Vst, tau, dg, eg, pm);
  }
#undef TNX_SYTRD
  TNX_LAUNCH_CHECK();
  return TNX_OK;
}

static int ormtr(const double* Vst, const double* tau, int n, const double* z, double* x, int batch, PMap pm,
                 int64_t so, hipStream_t s) {
  if (n <= 64)
    hipLaunchKernelGGL(ormtr_kernel<1>, dim3(1, batch), dim3(64), 0, s, Vst, tau, n, z, x, pm, so);
  else if (n <= 128)
    hipLaunchKernelGGL(ormtr_kernel<2>, dim3(1, batch), dim3(64), 0, s, Vst, tau, n, z, x, pm, so);
  else
    hipLaunchKernelGGL(ormtr_kernel<4>, dim3(1, batch), dim3(64), 0, s, Vst, tau, n, z, x, pm, so);
  TNX_LAUNCH_CHECK();
  return TNX_OK;
}

size_t syev_ws_bytes(int n) {
  const size_t nn = (size_t)n * n;
  return (2 * nn + 6 * (size_t)n + 16) * 8 + 256;
}

// Lowest eigenpair of a dense symmetric n x n matrix (device). eval written
// to *eval_dev (device) or copied to host if eval_host is given.
int syev_lowest(const double* M, int n, double* evec, double* eval_host, void* ws,
                size_t ws_bytes, hipStream_t s) {
  TNX_CHECK_ARG(n >= 1 && n <= kTriMax, "syev_lowest: n=%d outside [1, %d]", n, kTriMax);
  TNX_CHECK_ARG(M && evec, "syev_lowest: null pointer");
  TNX_CHECK_ARG(ws && ws_bytes >= syev_ws_bytes(n), "syev_lowest: workspace too small");
  double* A = (double*)ws;
  double* Vst = A + (size_t)n * n;
  double* tau = Vst + (size_t)n * n;
  double* dg = tau + n;
  double* eg = dg + n;
  double* z = eg + n;
  double* st = z + n + 8;
  if (n == 1) {
    TNX_TRY(fill_f64(evec, 1, 1.0, s));
    if (eval_host) {
      TNX_HIP(hipMemcpyAsync(eval_host, M, sizeof(double), hipMemcpyDeviceToHost, s));
      TNX_HIP(hipStreamSynchronize(s));
    }
    return TNX_OK;
  }
  TNX_TRY(sytrd(M, 0, n, A, Vst, tau, dg, eg, 1, kOne, s));
  hipLaunchKernelGGL(tridiag_lowest_kernel, dim3(1), dim3(64), 0, s, dg, eg, n, z, st, kOne);
  TNX_LAUNCH_CHECK();
  TNX_TRY(ormtr(Vst, tau, n, z, evec, 1, kOne, 0, s));
  if (eval_host) {
    TNX_HIP(hipMemcpyAsync(eval_host, st, sizeof(double), hipMemcpyDeviceToHost, s));
    TNX_HIP(hipStreamSynchronize(s));
  }
  return TNX_OK;
}

// ---------------------------------------------------------------------------
// All eigenpairs of a symmetric tridiagonal matrix (n <= 64): eigenvalues
// ascending to w, eigenvectors as columns of S (row stride ldS). Used at thick
// restarts, where the projected matrix is tridiagonal.
//
// Implicit QL is one chain of about 1.7 n^2 / 2 rotations, 1 ms at n = 64.
// Instead lane j finds eigenvalue j by sections, four points a round (one per
// wave, 24 rounds of 1.5 us), and its eigenvector from the twisted
// factorisation at that value; the vectors, orthonormal to rounding over the
// relative gap, are then orthonormalised symmetrically (Z <- Z (I - E / 2), E
// = Z^T Z - I, which converges quadratically and moves each vector least).
// Mixing two vectors by eps ||T|| / gap changes a residual by eps ||T||, so
// this is as accurate as QL while E starts small; clusters so tight that it
// does not (E above 1e-6) take QL.
// ---------------------------------------------------------------------------
constexpr int kAllLd = 65;
typedef double tri_f64x4 __attribute__((ext_vector_type(4)));

// Implicit QL by one wave (threads 0..63); Z: 64 rows of stride kAllLd, dsh: 64.
__device__ void tridiag_ql_wave(const double* __restrict__ ad, const double* __restrict__ bd, int n,
                                double* __restrict__ w, double* __restrict__ S, int ldS, double* Z, double* dsh) {
  // Implicit QL with eigenvectors (n <= 64). d[i], e[i] live in lane i's
  // registers: the rotation chain runs on all lanes as wave-uniform scalars,
  // reading a row with v_readlane and writing lane i's value with a lane
  // select, so no step waits on LDS. Row k of the eigenvector matrix Z is
  // private to lane k (in LDS); within a sweep the lane carries the freshly
  // rotated element Z[k][i] in a register to the next step, so its LDS row
  // sees only reads of untouched columns and stores nobody waits for.
  const int k = threadIdx.x;
  double dr = k < n ? ad[k] : 0.0;
  double er = k < n - 1 ? bd[k] : 0.0;
  if (k < n)
    for (int c = 0; c < n; ++c) Z[k * kAllLd + c] = (k == c) ? 1.0 : 0.0;
  const double eps = 2.220446049250313e-16;
  for (int l = 0; l < n; ++l) {
    for (int iter = 0; iter < 60; ++iter) {
      // m = first index >= l with a negligible e[m] (n - 1 if none)
      const double dnext = __shfl_down(dr, 1, 64);  // every lane takes part
      const bool negl = k >= l && k < n - 1 && fabs(er) <= eps * (fabs(dr) + fabs(dnext));
      const unsigned long long mk = __ballot(negl);
      const int m = mk ? __ffsll((long long)mk) - 1 : n - 1;
      if (m == l) break;
      const double el = lane_val(er, l), dl = lane_val(dr, l);
      double g = (lane_val(dr, l + 1) - dl) / (2.0 * el);
      double r = hypot(g, 1.0);
      g = lane_val(dr, m) - dl + el / (g + (g >= 0.0 ? fabs(r) : -fabs(r)));
      double sn = 1.0, cs = 1.0, p = 0.0;
      bool early = false;
      double zc = 0.0;  // rotated Z[k][hidx], not yet stored
      int hidx = -1;    // -1: nothing held
      for (int i = m - 1; i >= l; --i) {
        const double ei = lane_val(er, i);
        double f = sn * ei;
        const double b = cs * ei;
        // |f|, |g| <= ||T||: no scaling needed for the rotation length; its
        // reciprocal root is the only long operation of the chain (a square
        // root and a division before: n = 64 took 860 us, now 750)
        const double r2 = fma(f, f, g * g);
        const double ir = rsqrt_nr(r2);
        r = r2 == 0.0 ? 0.0 : r2 * ir;
        if (k == i + 1) er = r;
        if (r == 0.0) {
          if (k == i + 1) dr -= p;
          if (k == m) er = 0.0;
          early = true;
          break;
        }
        sn = f * ir;
        cs = g * ir;
        g = lane_val(dr, i + 1) - p;
        r = (lane_val(dr, i) - g) * sn + 2.0 * cs * b;
        p = sn * r;
        if (k == i + 1) dr = g + p;
        g = cs * r - b;
        if (k < n) {
          const double zi1 = hidx == i + 1 ? zc : Z[k * kAllLd + i + 1];
          const double zi = Z[k * kAllLd + i];
          Z[k * kAllLd + i + 1] = sn * zi + cs * zi1;
          zc = cs * zi - sn * zi1;
        }
        hidx = i;
      }
      // store the held element: Z[k][l] after a full sweep, Z[k][i+1] when
      // the sweep stopped at step i
      if (k < n && hidx >= 0) Z[k * kAllLd + hidx] = zc;
      if (early) continue;
      if (k == l) { dr -= p; er = g; }
      if (k == m) er = 0.0;
    }
  }
  if (k < n) dsh[k] = dr;
  wave_lds_fence();
  if (k < n) {
    const double dk = dr;
    int rank = 0;
    for (int j = 0; j < n; ++j) rank += (dsh[j] < dk) || (dsh[j] == dk && j < k);
    w[rank] = dk;
    for (int row = 0; row < n; ++row) S[row * ldS + rank] = Z[row * kAllLd + k];
  }
}

__global__ __launch_bounds__(256) void tridiag_all_kernel(const double* __restrict__ ad,
                                                          const double* __restrict__ bd, int n,
                                                          double* __restrict__ w, double* __restrict__ S, int ldS,
                                                          PMap pm) {
  {
    const int64_t o = pm.off();
    ad += o; bd += o; w += o; S += o;
  }
  __shared__ double2 row[kMaxBasis + 16];  // {a_k, b_{k-1}^2}
  __shared__ double bb[kMaxBasis];         // b_k
  __shared__ double Z[64 * kAllLd], U[64 * kAllLd], D[64 * kAllLd];
  __shared__ int cnt[2][4][64];
  __shared__ double part[2][64], red[4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, lr = lane & 15, lk = lane >> 4;
  // ---- the matrix, by a power of two near 1 where its norm is far from it
  double a = lane < n ? ad[lane] : 0.0, b = lane < n - 1 ? bd[lane] : 0.0;
  double bl = lane > 0 && lane < n ? bd[lane - 1] : 0.0;
  double r0 = fabs(b) + fabs(bl), tn = lane < n ? fabs(a) + r0 : 0.0;
  tn = wave_max(tn);
  int ex = __builtin_amdgcn_frexp_exp(tn);
  if (ex >= -64 && ex <= 64) ex = 0;
  a = ldexp(a, -ex);
  b = ldexp(b, -ex);
  bl = ldexp(bl, -ex);
  r0 = ldexp(r0, -ex);
  tn = ldexp(tn, -ex);
  const double eps = 2.220446049250313e-16;
  double lo = lane < n ? a - r0 : 1e308, hi = lane < n ? a + r0 : -1e308;
  lo = wave_min(lo);
  hi = wave_max(hi);
  lo -= 4.0 * eps * tn + 1e-300;
  hi += 4.0 * eps * tn + 1e-300;
  if (wave == 0) {
    row[lane] = make_double2(a, bl * bl);
    bb[lane] = b;
    if (lane < 16) row[kMaxBasis + lane] = make_double2(0.0, 0.0);
  }
  __syncthreads();
  // ---- eigenvalue `lane`: at most `lane` of them below lo, more below hi;
  // each round keeps a fifth (5^-24 of the Gershgorin range in the end)
  const int j = min(lane, n - 1);
  for (int it = 0; it < 24; ++it) {
    const double h = 0.2 * (hi - lo), x0 = lo;
    int c;
    double g;
    char_poly(row, n, fma(h, (double)(wave + 1), x0), c, g);
    cnt[it & 1][wave][lane] = c;
    __syncthreads();
    bool found = false;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const double x = fma(h, (double)(s + 1), x0);
      const bool above = cnt[it & 1][s][lane] > j;
      if (!found) {
        if (above) hi = x;
        else lo = x;
      }
      found = found || above;
    }
  }
  const double lam = 0.5 * (lo + hi);
  // ---- twisted factorisation: pivots and their ratios from above (wave 0)
  // and from below (wave 1)
  const double tiny = 0.25 * eps * tn + 1e-290;
  if (wave == 0) {
    double q = row[0].x - lam;
    for (int k = 0; k < n; ++k) {
      if (!(fabs(q) >= tiny)) q = tiny;
      const double rq = rcp_nr(q);
      Z[k * kAllLd + lane] = q;
      U[k * kAllLd + lane] = -bb[k] * rq;
      q = row[k + 1].x - lam - row[k + 1].y * rq;
    }
  } else if (wave == 1) {
    double q = row[n - 1].x - lam;
    for (int k = n - 1; k >= 0; --k) {
      if (!(fabs(q) >= tiny)) q = tiny;
      const double rq = rcp_nr(q), bk = k > 0 ? bb[k - 1] : 0.0;
      D[k * kAllLd + lane] = -bk * rq;
      q = (k > 0 ? row[k - 1].x : 0.0) - lam - bk * bk * rq;
    }
  }
  __syncthreads();
  // where they meet: the smallest gamma_k = q+_k + b_k D_{k+1}
  int r = 0;
  if (wave < 2) {
    double best = 1e308;
    for (int k = 0; k < n; ++k) {
      const double dn = k + 1 < n ? D[(k + 1) * kAllLd + lane] : 0.0;
      const double gm = fabs(fma(bb[k], dn, Z[k * kAllLd + lane]));
      r = gm < best ? k : r;
      best = fmin(best, gm);
    }
  }
  __syncthreads();
  if (wave < 2) {
    // z_r = 1, products of ratios upwards (wave 0) and downwards (wave 1)
    double z = 1.0, nn = 0.0;
    if (wave == 0) {
      for (int k = n - 1; k >= 0; --k) {
        if (k > r) continue;
        if (k < r) z *= U[k * kAllLd + lane];
        Z[k * kAllLd + lane] = z;
        nn = fma(z, z, nn);
      }
    } else {
      for (int k = 1; k < n; ++k) {
        if (k <= r) continue;
        z *= D[k * kAllLd + lane];
        Z[k * kAllLd + lane] = z;
        nn = fma(z, z, nn);
      }
    }
    part[wave][lane] = nn;
  }
  __syncthreads();
  {
    const double f = rsqrt_nr(part[0][lane] + part[1][lane]);
    for (int k = wave; k < 64; k += 4) {
      const double z = k < n ? Z[k * kAllLd + lane] : 0.0;
      Z[k * kAllLd + lane] = k < n && lane < n ? z * f : 0.0;
    }
  }
  __syncthreads();
  // ---- symmetric orthonormalisation on 16 x 16 matrix tiles; wave w takes
  // block column w
  bool ql = false;
  for (int it = 0; it < 4; ++it) {
    double mx = 0.0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      tri_f64x4 e = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int k = 0; k < 64; k += 4)
        e = __builtin_amdgcn_mfma_f64_16x16x4f64(Z[(k + lk) * kAllLd + 16 * i + lr],
                                                 Z[(k + lk) * kAllLd + 16 * wave + lr], e, 0, 0, 0);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int p = 16 * i + lk + 4 * v, q = 16 * wave + lr;
        const double x = p < n && q < n ? e[v] - (p == q ? 1.0 : 0.0) : 0.0;
        U[p * kAllLd + q] = x;
        mx = fmax(mx, fabs(x) <= 1e300 ? fabs(x) : 1e308);  // a NaN counts
      }
    }
    mx = wave_max(mx);
    if (lane == 0) red[wave] = mx;
    __syncthreads();
    mx = fmax(fmax(red[0], red[1]), fmax(red[2], red[3]));
    ql = it == 0 && mx > 1e-6;
    if (ql || mx <= 1e-15) break;
    tri_f64x4 z[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      tri_f64x4 c = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int k = 0; k < 64; k += 4)
        c = __builtin_amdgcn_mfma_f64_16x16x4f64(Z[(16 * i + lr) * kAllLd + k + lk],
                                                 U[(k + lk) * kAllLd + 16 * wave + lr], c, 0, 0, 0);
#pragma unroll
      for (int v = 0; v < 4; ++v) z[i][v] = fma(-0.5, c[v], Z[(16 * i + lk + 4 * v) * kAllLd + 16 * wave + lr]);
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int v = 0; v < 4; ++v) Z[(16 * i + lk + 4 * v) * kAllLd + 16 * wave + lr] = z[i][v];
    __syncthreads();
  }
  if (ql) {
    __syncthreads();
    if (wave == 0) tridiag_ql_wave(ad, bd, n, w, S, ldS, Z, part[0]);
    return;
  }
  if (wave == 0 && lane < n) w[lane] = ldexp(lam, ex);
  for (int k = wave; k < n; k += 4)
    if (lane < n) S[k * ldS + lane] = Z[k * kAllLd + lane];
}

// ---------------------------------------------------------------------------
// Lanczos driver
// ---------------------------------------------------------------------------
struct KWork {
  double* V;      // (m+1) x N basis
  double* Y;      // keep x N restart vectors
  double* w;      // N
  double* y;      // N
  void* mv;       // matvec workspace
  size_t mv_bytes;
  double* partials;
  double* h1; double* h2; double* h3;  // reductions (kPartStride each)
  double* alpha; double* beta;         // tridiagonal part, kMaxBasis + 2 each
  double* T;                           // dense projected matrix, kMaxBasis^2
  double* S;                           // its eigenvectors, kMaxBasis^2
  double* Cm;                          // restart combination, kMaxBasis^2
  double* theta;                       // its eigenvalues, kMaxBasis
  double* s;                           // Ritz coefficients of the lowest pair
  double* st;                          // status (16)
  double* scal;                        // scratch scalars (16)
};

static size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

static int keep_of(int m, int keep) {
  int k = keep > 0 ? keep : m / 4 + 2;
  return std::max(1, std::min(k, m - 2));
}

static size_t eigsh_ws_bytes_n(size_t N, size_t mvb, int max_basis) {
  const int m = std::max(3, std::min(max_basis, kMaxBasis));
  size_t b = 0;
  b += align256((size_t)(m + 1) * N * 8);
  b += align256((size_t)(m - 2) * N * 8);
  b += 2 * align256(N * 8);
  b += align256(mvb);
  b += align256((size_t)kCgsBlocks * kPartStride * 8);
  b += 3 * align256(kPartStride * 8);
  b += 3 * align256((kMaxBasis + 2) * 8);
  b += 3 * align256((size_t)kMaxBasis * kMaxBasis * 8);
  b += align256((kMaxBasis + 2) * 8);
  b += 2 * align256(16 * 8);
  return b + 256;
}

// Single-problem solver: the Lanczos block plus the FP64 correction block
// of the mixed-precision path (W = H V for up to m vectors, and the small
// arrays of its dense Rayleigh-Ritz).
static size_t gd_ws_bytes(size_t N, int m) {
  return align256((size_t)m * N * 8) + align256((size_t)8 * (kMaxBasis + 8) * 8);
}

static size_t eigsh_single_ws_bytes(size_t N, size_t mvb, int max_basis, size_t env32_bytes = 0) {
  const int m = std::max(3, std::min(max_basis, kMaxBasis));
  return eigsh_ws_bytes_n(N, mvb, max_basis) + gd_ws_bytes(N, m) + align256(env32_bytes);
}

// FP32 copies of L and R for the low-precision cycles of a one-site solve
static size_t env32_bytes_of(int chil, int Dl, int Dr, int chir) {
  return align256((size_t)chil * Dl * chil * 4) + align256((size_t)chir * Dr * chir * 4);
}

size_t eigsh_ws_bytes(int chil, int Dl, int Dr, int d, int chir, int max_basis) {
  return eigsh_single_ws_bytes((size_t)chil * d * chir, heff1_ws_bytes(chil, Dl, Dr, d, chir),
                               max_basis, env32_bytes_of(chil, Dl, Dr, chir));
}

size_t eigsh2_ws_bytes(int chil, int Dl, int Dm, int Dr, int d, int chir, int max_basis) {
  return eigsh_single_ws_bytes((size_t)chil * d * d * chir,
                               heff2_ws_bytes(chil, Dl, Dm, Dr, d, chir), max_basis);
}

static void carve(KWork& k, void* ws, int m, size_t N, size_t mvb) {
  char* p = (char*)(((uintptr_t)ws + 255) & ~(uintptr_t)255);
  auto take = [&](size_t bytes) { char* r = p; p += align256(bytes); return r; };
  k.V = (double*)take((size_t)(m + 1) * N * 8);
  k.Y = (double*)take((size_t)(m - 2) * N * 8);
  k.w = (double*)take(N * 8);
  k.y = (double*)take(N * 8);
  k.mv = take(mvb); k.mv_bytes = mvb;
  k.partials = (double*)take((size_t)kCgsBlocks * kPartStride * 8);
  k.h1 = (double*)take(kPartStride * 8);
  k.h2 = (double*)take(kPartStride * 8);
  k.h3 = (double*)take(kPartStride * 8);
  k.alpha = (double*)take((kMaxBasis + 2) * 8);
  k.beta = (double*)take((kMaxBasis + 2) * 8);
  k.s = (double*)take((kMaxBasis + 2) * 8);
  k.T = (double*)take((size_t)kMaxBasis * kMaxBasis * 8);
  k.S = (double*)take((size_t)kMaxBasis * kMaxBasis * 8);
  k.Cm = (double*)take((size_t)kMaxBasis * kMaxBasis * 8);
  k.theta = (double*)take((kMaxBasis + 2) * 8);
  k.st = (double*)take(16 * 8);
  k.scal = (double*)take(16 * 8);
}

// H y = theta y + (beta_j s_j) V[j+1] for the lowest Ritz pair:
// scal[0] = theta, scal[1] = beta_j * s_j
__global__ void ritz_scalars_kernel(const double* st, const double* s, const double* beta, int j,
                                    double* scal, PMap pm) {
  {
    const int64_t o = pm.off();
    st += o; s += o; beta += o; scal += o;
  }
  if (threadIdx.x == 0 && blockIdx.x == 0) {
    scal[0] = st[0];
    scal[1] = beta[j] * s[j];
  }
}

// Thick restart that keeps the projected matrix tridiagonal. The kept Ritz
// pairs (theta_i, Y_i = V S[:, i]), i < k, satisfy H Y_i = theta_i Y_i +
// c_i v_next with c_i = beta_j S[j][i]. A Lanczos run on diag(theta) started
// from c / |c| gives an orthonormal Q (k x k') in which diag(theta) is
// tridiagonal and only its first vector couples to v_next (with |c|). The new
// basis is the reversed Q columns, so the coupling sits on the last kept
// vector and the Lanczos recurrence continues from V[k'] = v_next.
// Writes C (J x k', ld kMaxBasis) with V_new = V_old C, the new alpha/beta
// (beta[k'-1] = |c|), the dense T, and k' to *kp_out. One wavefront.
__global__ __launch_bounds__(64) void tr_restart_kernel(const double* __restrict__ theta,
                                                        const double* __restrict__ S,
                                                        const double* __restrict__ beta_in, int j,
                                                        int k, int J, double* __restrict__ Cm,
                                                        double* __restrict__ alpha,
                                                        double* __restrict__ beta,
                                                        double* __restrict__ T, int* kp_out,
                                                        PMap pm) {
  {
    const int64_t o = pm.off();
    theta += o; S += o; beta_in += o; Cm += o; alpha += o; beta += o; T += o;
    kp_out = reinterpret_cast<int*>(reinterpret_cast<double*>(kp_out) + o);
  }
  __shared__ double q[kMaxBasis][kMaxBasis];
  __shared__ double a[kMaxBasis], b[kMaxBasis];
  const int l = threadIdx.x;  // component index of the k-vectors
  const double bj = beta_in[j];
  const double cl = (l < k) ? bj * S[j * kMaxBasis + l] : 0.0;
  const double th = (l < k) ? theta[l] : 0.0;
  double tmax = fabs(th);
  tmax = wave_max(tmax);
  const double cn = sqrt(wave_sum(cl * cl));
  double qi = (cn > 0.0) ? cl / cn : (l == 0 ? 1.0 : 0.0);
  if (l < kMaxBasis) q[0][l] = (l < k) ? qi : 0.0;
  int kp = 1;
  double qprev = 0.0, bprev = 0.0;
  for (int i = 0; i < k; ++i) {
    double w = th * qi;
    const double ai = wave_sum(qi * w);
    w -= ai * qi + bprev * qprev;
    for (int pass = 0; pass < 2; ++pass)
      for (int t = 0; t <= i; ++t) {
        const double h = wave_sum(q[t][l] * w);
        w -= h * q[t][l];
      }
    if (l < k) {} else w = 0.0;
    if (l == 0) a[i] = ai;
    const double bn = sqrt(wave_sum(w * w));
    kp = i + 1;
    if (i == k - 1) break;
    if (bn > 1e-13 * fmax(tmax, 1e-300)) {
      if (l == 0) b[i] = bn;
      qprev = qi;
      bprev = bn;
      qi = w / bn;
    } else {
      // span(q[0..i]) is invariant under diag(theta): continue in its
      // complement from the unit vector e_t with the largest component
      // there (zero coupling b[i]), so exactly k vectors are kept.
      double best = -1.0, qb = 0.0;
      for (int t = 0; t < k; ++t) {
        double u = (l == t) ? 1.0 : 0.0;
        for (int pass = 0; pass < 2; ++pass)
          for (int r = 0; r <= i; ++r) {
            const double h = wave_sum(q[r][l] * u);
            u -= h * q[r][l];
          }
        if (l >= k) u = 0.0;
        const double un = sqrt(wave_sum(u * u));
        if (un > best) { best = un; qb = u / un; }
      }
      if (l == 0) b[i] = 0.0;
      qprev = 0.0;
      bprev = 0.0;
      qi = qb;
    }
    q[i + 1][l] = qi;
  }
  __syncthreads();
  // reversed order: new index r holds q[kp-1-r]
  for (int r = 0; r < kp; ++r) {
    const int i = kp - 1 - r;
    for (int row = l; row < J; row += 64) {
      double acc = 0.0;
      for (int t = 0; t < k; ++t) acc += S[row * kMaxBasis + t] * q[i][t];
      Cm[row * kMaxBasis + r] = acc;
    }
  }
  for (int e = l; e < kMaxBasis * kMaxBasis; e += 64) T[e] = 0.0;
  __syncthreads();
  if (l == 0) {
    for (int r = 0; r < kp; ++r) {
      const int i = kp - 1 - r;
      alpha[r] = a[i];
      T[r * kMaxBasis + r] = a[i];
      const double br = (r < kp - 1) ? b[i - 1] : cn;
      beta[r] = br;
      T[r * kMaxBasis + r + 1] = br;
      T[(r + 1) * kMaxBasis + r] = br;
    }
    *kp_out = kp;
  }
}

// Outer (FP64) step scalars: theta = y.(Hy) = h1[0] + h2[0] (both CGS
// passes), rho^2 = h3[1] (norm of r). Resets the projected matrix to the
// two-vector basis [y, r/rho].
__global__ void outer_scalars_kernel(const double* h1, const double* h2, const double* h3,
                                     double* alpha, double* beta, double* scal, double* st,
                                     double* T, PMap pm) {
  {
    const int64_t o = pm.off();
    h1 += o; h2 += o; h3 += o; alpha += o; beta += o; scal += o; st += o; T += o;
  }
  const double th = h1[0] + h2[0];
  const double rho = sqrt(fmax(h3[1], 0.0));
  for (int e = threadIdx.x; e < kMaxBasis * kMaxBasis; e += blockDim.x) {
    const int i = e / kMaxBasis, c = e % kMaxBasis;
    T[e] = (i == 0 && c == 0) ? th : ((i + c == 1) ? rho : 0.0);
  }
  if (threadIdx.x == 0) {
    alpha[0] = th; beta[0] = rho;
    scal[0] = th; scal[2] = -th; scal[3] = 1.0;
    st[4] = th; st[5] = rho;
  }
}

// The operator of one eigensolve: the one-site H_eff (W2 == nullptr) or
// the two-site H_eff (W, W2 with middle MPO bond Dm).
struct EigCtx {
  const double *L, *W, *R;
  const double* W2 = nullptr;
  int chil, Dl, Dm = 0, Dr, d, chir;
  int64_t N;
  hipStream_t s;
  KWork k;
  int matvecs = 0, matvecs64 = 0;
  double* Wd = nullptr;   // FP64 correction: H V (m x N)
  double* gsm = nullptr;  // its small arrays (8 x (kMaxBasis + 8))
  // one-site problems: L and R rounded to FP32 at most once per solve (at
  // its first low-precision cycle), read by the low-precision matvecs (the
  // same values their tile staging would round to, half the bytes, no
  // conversion per matvec); null until converted and for FP64 solves
  const float* L32 = nullptr;
  const float* R32 = nullptr;
  float* L32_buf = nullptr;  // their workspace (set for low-precision solves)
  float* R32_buf = nullptr;
  size_t env32_bytes = 0;  // workspace reserved for them
};

static int apply_h(EigCtx& c, const void* x, int x_f32, double* y, int prec) {
  c.matvecs++;
  if (prec == TNX_F64) c.matvecs64++;
  if (c.W2)
    return heff2_matvec(c.L, c.W, c.W2, c.R, x, x_f32, y, c.chil, c.Dl, c.Dm, c.Dr, c.d, c.chir,
                        prec, c.k.mv, c.k.mv_bytes, c.s);
  if (prec != TNX_F64 && c.L32)
    return heff1_matvec_b(c.L32, c.W, c.R32, x, x_f32, y, c.chil, c.Dl, c.Dr, c.d, c.chir, prec, 1,
                          1, nullptr, c.N, c.N, c.k.mv, c.k.mv_bytes, c.s, 1);
  return heff1_matvec_b(c.L, c.W, c.R, x, x_f32, y, c.chil, c.Dl, c.Dr, c.d, c.chir, prec, 1, 1,
                        nullptr, c.N, c.N, c.k.mv, c.k.mv_bytes, c.s, 0);
}

static int read_status(EigCtx& c, double* host, int n) {
  TNX_HIP(hipMemcpyAsync(host, c.k.st, sizeof(double) * n, hipMemcpyDeviceToHost, c.s));
  TNX_HIP(hipStreamSynchronize(c.s));
  return TNX_OK;
}

// FP64 outer step on the unit vector y (in k.y): w = H y, theta = y.w,
// r = w - theta y (in k.w), rho = |r|. Sets alpha[0] = theta, beta[0] = rho
// and T = [[theta, rho], [rho, .]]. Returns theta, rho on the host.
static int outer_step(EigCtx& c, double* theta, double* rho) {
  KWork& k = c.k;
  const int64_t N = c.N;
  TNX_TRY(apply_h(c, k.y, 0, k.w, TNX_F64));
  TNX_TRY(cgs_pass(k.y, N, 1, k.w, nullptr, true, k.partials, k.h1, N, c.s));
  TNX_TRY(cgs_pass(k.y, N, 1, k.w, k.h1, true, k.partials, k.h2, N, c.s));
  TNX_TRY(cgs_pass(k.y, N, 1, k.w, k.h2, false, k.partials, k.h3, N, c.s));
  hipLaunchKernelGGL(outer_scalars_kernel, dim3(1), dim3(256), 0, c.s, k.h1, k.h2, k.h3,
                     k.alpha, k.beta, k.scal, k.st, k.T, kOne);
  TNX_LAUNCH_CHECK();
  double h[8];
  TNX_TRY(read_status(c, h, 8));
  *theta = h[4];
  *rho = h[5];
  return TNX_OK;
}

static int eigsh_run(EigCtx& c, const double* v0, double* vec, double* hvec,
                     const tnx_eigsh_opts_t* opts, tnx_eigsh_info_t* info, void* ws,
                     size_t ws_bytes, size_t mvb);

// ---------------------------------------------------------------------------
// FP64 correction after a low-precision Lanczos cycle (mixed precision).
// A cycle that has reached its arithmetic's floor holds, in its kept Ritz
// vectors, the cluster of low eigenvalues its Krylov space has resolved. A
// fresh FP64 Lanczos from [y, r] would have to resolve that cluster again.
// Instead: take the `keep` lowest Ritz vectors of the cycle, orthonormalise
// them in FP64, apply H to each in FP64 (W = H V), and run a subspace
// expansion with an exact dense projection G = V^T H V: each step takes
// the lowest Ritz pair of G, its FP64 residual r = W s - theta V s (exact,
// no recurrence estimate), stops when |r| <= tol ||H||_est, else adds
// r (orthogonalised) to V and H r to W. (Without a preconditioner this
// spans the same space as Lanczos from the kept block, but keeps the block
// exact in FP64.)
// ---------------------------------------------------------------------------

// z = V s, hz = W s, r = hz - theta z (theta = *st), J vectors each
__global__ void gd_residual_kernel(const double* __restrict__ V, const double* __restrict__ Wm,
                                   int64_t ld, int J, const double* __restrict__ sv,
                                   const double* __restrict__ st, double* __restrict__ z,
                                   double* __restrict__ hz, double* __restrict__ r, int64_t N) {
  __shared__ double cs[kMaxBasis + 1];
  if ((int)threadIdx.x < J) cs[threadIdx.x] = sv[threadIdx.x];
  __syncthreads();
  const double th = st[0];
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < N;
       i += (int64_t)gridDim.x * blockDim.x) {
    double a = 0.0, b = 0.0;
    for (int j = 0; j < J; ++j) {
      a += cs[j] * V[(int64_t)j * ld + i];
      b += cs[j] * Wm[(int64_t)j * ld + i];
    }
    z[i] = a;
    hz[i] = b;
    r[i] = b - th * a;
  }
}

// column and row J of the dense projected matrix: G[i][J] = G[J][i] = h[i]
__global__ void gd_gcol_kernel(const double* __restrict__ h, int J, double* __restrict__ G) {
  const int i = threadIdx.x;
  if (i <= J) {
    G[i * kMaxBasis + J] = h[i];
    G[J * kMaxBasis + i] = h[i];
  }
}

// compact symmetric copy A[J][J] of G (row stride kMaxBasis)
__global__ void gd_compact_kernel(const double* __restrict__ G, int J, double* __restrict__ A) {
  for (int e = threadIdx.x; e < J * J; e += blockDim.x) {
    const int i = e / J, j = e % J;
    A[e] = 0.5 * (G[i * kMaxBasis + j] + G[j * kMaxBasis + i]);
  }
}

// Returns TNX_OK; *done says whether the criterion was met (then k.y = z,
// hvec = H z, *theta and *rho set). If not, k.y holds the best Ritz vector
// and the caller continues with FP64 Lanczos from it.
static int gd_correction(EigCtx& c, const float* V32, int J32, int keep, int m, double tol,
                         double* anorm, int max_mv, double* hvec, double* theta, double* rho,
                         bool* done) {
  KWork& k = c.k;
  hipStream_t s = c.s;
  const int64_t N = c.N;
  const int nb = vec_blocks(N);
  *done = false;
  // kept Ritz values of the cycle (ascending); the block is the cluster
  // within 0.1% of ||H||_est of the lowest (at least 2, at most `keep`): a
  // gapped spectrum needs a couple of FP64 matvecs here, a clustered one
  // keeps the whole cluster
  hipLaunchKernelGGL(tridiag_all_kernel, dim3(1), dim3(256), 0, s, k.alpha, k.beta, J32, k.theta,
                     k.S, kMaxBasis, kOne);
  TNX_LAUNCH_CHECK();
  std::vector<double> th(J32);
  TNX_HIP(hipMemcpyAsync(th.data(), k.theta, sizeof(double) * J32, hipMemcpyDeviceToHost, s));
  TNX_HIP(hipStreamSynchronize(s));
  int kk = 1;
  while (kk < std::min(keep, J32) && th[kk] - th[0] <= 1e-3 * *anorm) ++kk;
  kk = std::min(std::max(kk, 2), std::min(keep, J32));
  double* A = k.S;        // compact copy of G for the dense solve
  double* Vst = k.Cm;     // its Householder vectors
  double* tau = c.gsm;
  double* dg = tau + (kMaxBasis + 8);
  double* eg = dg + (kMaxBasis + 8);
  double* zt = eg + (kMaxBasis + 8);
  double* stg = zt + (kMaxBasis + 8);
  double* G = k.T;
  // kept Ritz vectors of the low-precision cycle, in FP64: Y = V32 S[:, :kk]
  {
    GemmDesc g{};
    g.M = kk; g.N = (int)N; g.K = J32; g.batch = 1;
    g.A = k.S; g.ta = DT::F64; g.lda = kMaxBasis; g.sA = 0; g.a_kcontig = false;
    g.B = V32; g.tb = DT::F32; g.ldb = N; g.sB = 0; g.b_ncontig = true;
    g.C = k.Y; g.tc = DT::F64; g.ldc = N; g.sC = 0;
    g.alpha = 1.0; g.beta = 0.0; g.prec = Prec::F64;
    TNX_TRY(gemm(g, s));
  }
  double* V = k.V;  // the FP64 basis of the correction (V32 is no longer needed)
  TNX_HIP(hipMemcpyAsync(V, k.Y, sizeof(double) * kk * N, hipMemcpyDeviceToDevice, s));
  // orthonormalise (CGS2) and apply H in FP64, building G column by column
  for (int i = 0; i < kk; ++i) {
    double* vi = V + (int64_t)i * N;
    if (i > 0) {
      TNX_TRY(cgs_pass(V, N, i, vi, nullptr, true, k.partials, k.h1, N, s));
      TNX_TRY(cgs_pass(V, N, i, vi, k.h1, true, k.partials, k.h2, N, s));
    }
    TNX_TRY(cgs_pass(V, N, i, vi, i > 0 ? k.h2 : nullptr, false, k.partials, k.h3, N, s));
    hipLaunchKernelGGL(normalize_kernel<double>, dim3(nb), dim3(256), 0, s, vi, k.h3 + i, vi, N,
                       kOne);
    TNX_LAUNCH_CHECK();
    double* wi = c.Wd + (int64_t)i * N;
    TNX_TRY(apply_h(c, vi, 0, wi, TNX_F64));
    TNX_TRY(cgs_pass(V, N, i + 1, wi, nullptr, true, k.partials, k.h1, N, s));
    hipLaunchKernelGGL(gd_gcol_kernel, dim3(1), dim3(kMaxBasis + 1), 0, s, k.h1, i, G);
    TNX_LAUNCH_CHECK();
  }
  int J = kk;
  while (true) {
    // lowest Ritz pair of G (J x J): Householder tridiagonalisation,
    // multisection + twisted factorisation, back-transform into k.s
    hipLaunchKernelGGL(gd_compact_kernel, dim3(1), dim3(256), 0, s, G, J, A);
    TNX_LAUNCH_CHECK();
    if (J == 1) {
      TNX_TRY(fill_f64(k.s, 1, 1.0, s));
      TNX_HIP(hipMemcpyAsync(stg, A, sizeof(double), hipMemcpyDeviceToDevice, s));
    } else {
      TNX_TRY(sytrd(A, 0, J, nullptr, Vst, tau, dg, eg, 1, kOne, s));  // J <= 64
      hipLaunchKernelGGL(tridiag_lowest_kernel, dim3(1), dim3(64), 0, s, dg, eg, J, zt, stg, kOne);
      TNX_LAUNCH_CHECK();
      TNX_TRY(ormtr(Vst, tau, J, zt, k.s, 1, kOne, 0, s));
    }
    // z = V s -> k.y, H z = W s -> k.w, r -> V[J] (the next basis slot)
    double* r = V + (int64_t)J * N;
    hipLaunchKernelGGL(gd_residual_kernel, dim3(nb), dim3(256), 0, s, V, c.Wd, N, J, k.s, stg,
                       k.y, k.w, r, N);
    TNX_LAUNCH_CHECK();
    TNX_TRY(cgs_pass(r, N, 0, r, nullptr, false, k.partials, k.h3, N, s));
    double h[2];
    TNX_HIP(hipMemcpyAsync(&h[0], stg, sizeof(double), hipMemcpyDeviceToHost, s));
    TNX_HIP(hipMemcpyAsync(&h[1], k.h3, sizeof(double), hipMemcpyDeviceToHost, s));
    TNX_HIP(hipStreamSynchronize(s));
    *theta = h[0];
    *rho = std::sqrt(std::max(h[1], 0.0));
    *anorm = std::max(*anorm, std::fabs(h[0]));
    if (*rho <= tol * *anorm || *rho == 0.0) {
      if (hvec) TNX_TRY(copy_f64(k.w, hvec, N, s));
      *done = true;
      return TNX_OK;
    }
    if (J >= m || c.matvecs >= max_mv) return TNX_OK;
    // expand: r orthogonalised against V, normalised, and H r
    TNX_TRY(cgs_pass(V, N, J, r, nullptr, true, k.partials, k.h1, N, s));
    TNX_TRY(cgs_pass(V, N, J, r, k.h1, true, k.partials, k.h2, N, s));
    TNX_TRY(cgs_pass(V, N, J, r, k.h2, false, k.partials, k.h3, N, s));
    hipLaunchKernelGGL(normalize_kernel<double>, dim3(nb), dim3(256), 0, s, r, k.h3 + J, r, N,
                       kOne);
    TNX_LAUNCH_CHECK();
    double* wj = c.Wd + (int64_t)J * N;
    TNX_TRY(apply_h(c, r, 0, wj, TNX_F64));
    TNX_TRY(cgs_pass(V, N, J + 1, wj, nullptr, true, k.partials, k.h1, N, s));
    hipLaunchKernelGGL(gd_gcol_kernel, dim3(1), dim3(kMaxBasis + 1), 0, s, k.h1, J, G);
    TNX_LAUNCH_CHECK();
    ++J;
  }
}

int eigsh_heff1(const double* L, const double* W, const double* R, const double* v0,
                double* vec, double* hvec, int chil, int Dl, int Dr, int d, int chir,
                const tnx_eigsh_opts_t* opts, tnx_eigsh_info_t* info, void* ws,
                size_t ws_bytes, hipStream_t s) {
  TNX_CHECK_ARG(opts && info, "eigsh: null opts/info");
  TNX_CHECK_ARG(L && W && R && v0 && vec, "eigsh: null pointer");
  TNX_CHECK_ARG(chil > 0 && Dl > 0 && Dr > 0 && d > 0 && chir > 0, "eigsh: bad dims");
  EigCtx c;
  c.L = L; c.W = W; c.R = R;
  c.chil = chil; c.Dl = Dl; c.Dr = Dr; c.d = d; c.chir = chir;
  c.N = (int64_t)chil * d * chir;
  c.s = s;
  c.env32_bytes = env32_bytes_of(chil, Dl, Dr, chir);
  return eigsh_run(c, v0, vec, hvec, opts, info, ws, ws_bytes, heff1_ws_bytes(chil, Dl, Dr, d, chir));
}

int eigsh_heff2(const double* L, const double* W1, const double* W2, const double* R,
                const double* v0, double* vec, double* hvec, int chil, int Dl, int Dm, int Dr,
                int d, int chir, const tnx_eigsh_opts_t* opts, tnx_eigsh_info_t* info, void* ws,
                size_t ws_bytes, hipStream_t s) {
  TNX_CHECK_ARG(opts && info, "eigsh2: null opts/info");
  TNX_CHECK_ARG(L && W1 && W2 && R && v0 && vec, "eigsh2: null pointer");
  TNX_CHECK_ARG(chil > 0 && Dl > 0 && Dm > 0 && Dr > 0 && d > 0 && chir > 0, "eigsh2: bad dims");
  EigCtx c;
  c.L = L; c.W = W1; c.W2 = W2; c.R = R;
  c.chil = chil; c.Dl = Dl; c.Dm = Dm; c.Dr = Dr; c.d = d; c.chir = chir;
  c.N = (int64_t)chil * d * d * chir;
  c.s = s;
  return eigsh_run(c, v0, vec, hvec, opts, info, ws, ws_bytes,
                   heff2_ws_bytes(chil, Dl, Dm, Dr, d, chir));
}

static int eigsh_run(EigCtx& c, const double* v0, double* vec, double* hvec,
                     const tnx_eigsh_opts_t* opts, tnx_eigsh_info_t* info, void* ws,
                     size_t ws_bytes, size_t mvb) {
  TNX_CHECK_ARG(opts->precision >= TNX_F64 && opts->precision <= TNX_BF16X3, "eigsh: bad precision");
  TNX_CHECK_ARG(opts->tol >= 0.0, "eigsh: negative tol");
  const int m = std::max(3, std::min(opts->max_basis, kMaxBasis));
  TNX_CHECK_ARG(ws && ws_bytes >= eigsh_single_ws_bytes((size_t)c.N, mvb, m, c.env32_bytes),
                "eigsh: workspace too small");
  hipStream_t s = c.s;
  carve(c.k, ws, m, (size_t)c.N, mvb);
  {
    // the correction block follows the Lanczos block
    char* gp = (char*)(((uintptr_t)ws + 255) & ~(uintptr_t)255) +
               (eigsh_ws_bytes_n((size_t)c.N, mvb, m) - 256);
    c.Wd = (double*)gp;
    c.gsm = (double*)(gp + align256((size_t)m * c.N * 8));
    if (c.env32_bytes && !c.W2 && opts->precision != TNX_F64) {
      // converted at the first low-precision cycle (a solve that converges
      // on its first FP64 step never reads them)
      c.L32_buf = (float*)(gp + gd_ws_bytes((size_t)c.N, m));
      c.R32_buf = (float*)((char*)c.L32_buf + align256((size_t)c.chil * c.Dl * c.chil * 4));
    }
  }
  auto env_to_f32 = [&]() -> int {
    if (c.L32 || !c.L32_buf) return TNX_OK;
    const int64_t nl = (int64_t)c.chil * c.Dl * c.chil, nr = (int64_t)c.chir * c.Dr * c.chir;
    hipLaunchKernelGGL(to_f32_kernel, dim3(vec_blocks(nl)), dim3(256), 0, s, c.L, c.L32_buf, nl);
    TNX_LAUNCH_CHECK();
    hipLaunchKernelGGL(to_f32_kernel, dim3(vec_blocks(nr)), dim3(256), 0, s, c.R, c.R32_buf, nr);
    TNX_LAUNCH_CHECK();
    c.L32 = c.L32_buf;
    c.R32 = c.R32_buf;
    return TNX_OK;
  };
  KWork& k = c.k;
  const int64_t N = c.N;
  const int prec = opts->precision;
  const int max_mv = opts->max_matvecs > 0 ? opts->max_matvecs : 10000;
  const double tol = opts->tol;
  const int nb = vec_blocks(N);
  // Basis size cannot exceed the dimension (Krylov space exhausts at N).
  const int mb = (int)std::min<int64_t>(m, std::max<int64_t>(N, 1));
  const int keep = keep_of(mb, opts->keep);

  // y = v0 / |v0|
  TNX_TRY(cgs_pass(v0, N, 0, const_cast<double*>(v0), nullptr, false, k.partials, k.h3, N, s));
  hipLaunchKernelGGL(normalize_kernel<double>, dim3(nb), dim3(256), 0, s, v0, k.h3, k.y, N, kOne);
  TNX_LAUNCH_CHECK();

  double theta = 0.0, rho = 0.0, anorm = 0.0;
  int restarts = 0;
  bool converged = false;
  bool have_hy = false;  // k.w holds r = H y - theta y for the final y
  // Krylov matvec precision of the current cycle: starts at `prec`, and
  // escalates to FP64 when an FP64-corrected cycle fails to cut the true
  // residual by 4x (the low-precision operator cannot resolve the local
  // spectrum, e.g. clusters narrower than its rounding).
  int cprec = prec;
  double rho_prev = 0.0;
  bool first_cycle = true;
  // Step pipelining: the next step's matvec and CGS passes (they need only
  // V[j+1]) are queued before the host reads step j's status, so the GPU
  // works while the host decides. When step j ends the cycle, that queued
  // step is discarded (its buffers are rewritten before any later use) and
  // not counted.
  StepEvent sev;
  PinnedLease pin_lease(64);
  double* pin = pin_lease.get();
  const bool pipelined = sev.e != nullptr && pin != nullptr;

  while (true) {
    TNX_TRY(outer_step(c, &theta, &rho));
    have_hy = true;
    anorm = std::max(anorm, std::fabs(theta));
    if (cprec != TNX_F64 && rho_prev > 0.0 && rho > 0.25 * rho_prev) cprec = TNX_F64;
    // After the first low-precision cycle (run to its arithmetic's floor), a
    // tolerance below that floor is reached in FP64: a further low-precision
    // cycle would restart the Krylov space for a target it cannot resolve.
    if (cprec != TNX_F64 && !first_cycle && tol < 8.0 * (cprec == TNX_F32 ? 5.96e-8 : 3.9e-6))
      cprec = TNX_F64;
    rho_prev = rho;
    const bool mixed = cprec != TNX_F64;
    if (rho <= tol * anorm || rho == 0.0 || N == 1) {
      converged = true;
      break;
    }
    if (c.matvecs >= max_mv) break;
    // Inner Lanczos cycle in `cprec`, from column j = 1 on V[0] = y,
    // V[1] = r / rho. Inner target. FP64: the final tolerance. Low
    // precision: the first cycle runs the full thick-restart Lanczos down to
    // the rounding floor of its arithmetic (it keeps its restart subspace
    // the whole way); later cycles start from [y, r/|r|] and only need to
    // cut the FP64 residual. A low-precision cycle keeps its basis in FP32:
    // it resolves nothing below FP32 rounding, and the CGS passes and the
    // matvec read half the bytes.
    const double rho_outer = rho;
    const double unit_lp = cprec == TNX_F32 ? 5.96e-8 : 3.9e-6;
    // A first low-precision cycle whose target is below its arithmetic's
    // floor runs on its own (low-precision operator) residual estimate down
    // to tol: the residual it reaches against H stays at the floor, but its
    // Krylov space keeps growing into the low spectrum (near-degenerate
    // states below the first converged Ritz value appear late), and its kept
    // block then goes to the FP64 correction.
    const bool gd_after = mixed && first_cycle && tol < 8.0 * unit_lp;
    const double inner_tol =
        !mixed ? tol * anorm
               : (first_cycle ? (gd_after ? tol : std::max(tol, 4.0 * unit_lp)) * anorm
                              : std::max(tol * anorm, std::min(1e-3 * rho_outer, 0.5 * rho_outer)));
    first_cycle = false;
    have_hy = false;  // the inner cycle reuses k.w
    int last_J = 0;   // Lanczos basis size when the cycle stopped
    auto cycle = [&](auto* V, auto* Yb) -> int {
      using VT = std::remove_pointer_t<decltype(V)>;
      constexpr bool f32 = std::is_same<VT, float>::value;
      if constexpr (f32) {
        hipLaunchKernelGGL(to_f32_kernel, dim3(nb), dim3(256), 0, s, k.y, V, N);
      } else {
        TNX_TRY(copy_f64(k.y, V, N, s));
      }
      hipLaunchKernelGGL(normalize_kernel<VT>, dim3(nb), dim3(256), 0, s, k.w, k.h3 + 1, V + N, N,
                         kOne);
      TNX_LAUNCH_CHECK();
      // Step jj's matvec and CGS passes: w = H V[jj] orthogonalised against
      // V[0..jj] (sums in h1, h2, h3).
      auto front = [&](int jj) -> int {
        if constexpr (f32) {
          if (c.L32) {
            // FP32 basis row and FP32 environments
            TNX_TRY(apply_h(c, V + (int64_t)jj * N, 1, k.w, cprec));
          } else {
            // FP64 environments: widen V[jj] into k.y (free until the
            // cycle's Ritz vector is formed), so both operands have one type
            // (the BF16X3 tile table's shapes do; the FP32 products take any
            // pair and round the widened values back to the same floats)
            hipLaunchKernelGGL(to_f64_kernel, dim3(nb), dim3(256), 0, s, V + (int64_t)jj * N, k.y, N);
            TNX_LAUNCH_CHECK();
            TNX_TRY(apply_h(c, k.y, 0, k.w, cprec));
          }
        } else {
          TNX_TRY(apply_h(c, V + (int64_t)jj * N, 0, k.w, cprec));
        }
        return cgs_step(V, N, jj + 1, k.w, k.partials, k.h1, k.h2, k.h3, s);
      };
      int j = 1;
      bool queued = false;  // step j's front already launched
      while (true) {
        const int J = j + 1;
        if (!queued) TNX_TRY(front(j));
        const int mv_now = c.matvecs, mv64_now = c.matvecs64;
        // the next step goes ahead only where this one, not ending the
        // cycle, would be followed by it (no restart, not exhausted)
        const bool ahead = pipelined && J < mb && J < N && mv_now < max_mv;
        // V[j+1] = w / |w| and the projected problem
        TNX_TRY(finish_step(V, N, J, k.w, k.partials, rows_blocks(N, 1), k.h3, k.s, k.st,
                            TriFinish{k.h1, k.h2, k.alpha, k.beta, k.T}, -1.0, ahead ? pin : nullptr, s));
        double h[4];
        if (ahead) {
          TNX_HIP(hipEventRecord(sev.e, s));
          TNX_TRY(front(j + 1));
          TNX_HIP(hipEventSynchronize(sev.e));
          for (int q = 0; q < 3; ++q) h[q] = pin[q];
        } else {
          TNX_TRY(read_status(c, h, 3));
        }
        const double theta_in = h[0];
        const double est = h[1];
        anorm = std::max(anorm, h[2]);
        const bool exhausted = (J >= N);
        // FP64 cycles test against the current ||H|| estimate (it grows with
        // the Ritz values seen); low-precision cycles against their fixed target
        const double itol = mixed ? inner_tol : tol * anorm;
        if (est <= itol || exhausted || mv_now >= max_mv) {
          if (ahead) {  // the queued step is not used
            c.matvecs = mv_now;
            c.matvecs64 = mv64_now;
          }
          last_J = J;
          // Ritz vector y = V[0..j] s
          hipLaunchKernelGGL(vcomb_kernel<VT>, dim3(nb), dim3(256), 0, s, V, N, J, k.s, k.y, N,
                             kOne);
          TNX_LAUNCH_CHECK();
          if constexpr (f32) {
            // an FP32 basis is orthonormal only to FP32 rounding: renormalise
            // y in FP64 before the FP64 step takes its Rayleigh quotient
            TNX_TRY(cgs_pass(k.y, N, 0, k.y, nullptr, false, k.partials, k.h3, N, s));
            hipLaunchKernelGGL(normalize_kernel<double>, dim3(nb), dim3(256), 0, s, k.y, k.h3, k.y,
                               N, kOne);
            TNX_LAUNCH_CHECK();
          }
          if constexpr (!f32) {
            if (!mixed && (est <= tol * anorm || exhausted)) {
              // FP64 Lanczos: H y = theta y + beta_j s_j V[j+1]
              hipLaunchKernelGGL(ritz_scalars_kernel, dim3(1), dim3(1), 0, s, k.st, k.s, k.beta, j,
                                 k.scal, kOne);
              TNX_LAUNCH_CHECK();
              if (hvec) {
                hipLaunchKernelGGL(axpbz_dev_kernel, dim3(nb), dim3(256), 0, s, k.scal, k.y,
                                   exhausted ? nullptr : k.scal + 1, V + (int64_t)(j + 1) * N,
                                   hvec, N, kOne, (int64_t)0);
                TNX_LAUNCH_CHECK();
              }
              theta = theta_in;
              rho = est;
              converged = true;
            }
          }
          return TNX_OK;
        }
        if (J >= mb) {
          // Thick restart keeping the `keep` lowest Ritz pairs in a basis
          // where the projected matrix stays tridiagonal.
          hipLaunchKernelGGL(tridiag_all_kernel, dim3(1), dim3(256), 0, s, k.alpha, k.beta, J,
                             k.theta, k.S, kMaxBasis, kOne);
          TNX_LAUNCH_CHECK();
          int* kp_dev = reinterpret_cast<int*>(k.st + 8);
          hipLaunchKernelGGL(tr_restart_kernel, dim3(1), dim3(64), 0, s, k.theta, k.S, k.beta, j,
                             keep, J, k.Cm, k.alpha, k.beta, k.T, kp_dev, kOne);
          TNX_LAUNCH_CHECK();
          int kp = 0;
          TNX_HIP(hipMemcpyAsync(&kp, kp_dev, sizeof(int), hipMemcpyDeviceToHost, s));
          TNX_HIP(hipStreamSynchronize(s));
          TNX_CHECK_ARG(kp == keep, "eigsh: restart kept %d of %d vectors", kp, keep);
          const DT vt = f32 ? DT::F32 : DT::F64;
          GemmDesc g{};
          g.M = kp; g.N = (int)N; g.K = J; g.batch = 1;
          g.A = k.Cm; g.ta = DT::F64; g.lda = kMaxBasis; g.sA = 0; g.a_kcontig = false;
          g.B = V; g.tb = vt; g.ldb = N; g.sB = 0; g.b_ncontig = true;
          g.C = Yb; g.tc = vt; g.ldc = N; g.sC = 0;
          g.alpha = 1.0; g.beta = 0.0; g.prec = Prec::F64;
          TNX_TRY(gemm(g, s));
          TNX_HIP(hipMemcpyAsync(V, Yb, sizeof(VT) * kp * N, hipMemcpyDeviceToDevice, s));
          TNX_HIP(hipMemcpyAsync(V + (int64_t)kp * N, V + (int64_t)(j + 1) * N, sizeof(VT) * N,
                                 hipMemcpyDeviceToDevice, s));
          restarts++;
          j = kp;
          queued = false;
        } else {
          j++;
          queued = ahead;
        }
      }
    };
    if (mixed && N % 2 == 0) {
      TNX_TRY(env_to_f32());
      TNX_TRY(cycle(reinterpret_cast<float*>(k.V), reinterpret_cast<float*>(k.Y)));
    } else {
      TNX_TRY(cycle(k.V, k.Y));
    }
    if (gd_after && N % 2 == 0 && last_J > 0 && c.matvecs < max_mv) {
      bool done = false;
      TNX_TRY(gd_correction(c, reinterpret_cast<const float*>(k.V), last_J, keep, mb, tol, &anorm,
                            max_mv, hvec, &theta, &rho, &done));
      if (done) {
        converged = true;
        have_hy = false;  // outputs: k.y, and hvec written by the correction
        break;
      }
      cprec = TNX_F64;  // continue with FP64 Lanczos from the best vector
    }
    if (converged) break;
    if (c.matvecs >= max_mv) break;
    // loop: next outer step re-evaluates y in FP64 (mixed precision, or
    // FP64 when the matvec limit cut the cycle short)
  }

  // Outputs. After an outer step k.w holds r = H y - theta y.
  if (have_hy) {
    TNX_TRY(copy_f64(k.y, vec, N, s));
    if (hvec) {
      // H y = r + theta y  (scal[3] = 1, scal[0] = theta)
      hipLaunchKernelGGL(axpbz_dev_kernel, dim3(nb), dim3(256), 0, s, k.scal + 3, k.w, k.scal,
                         k.y, hvec, N, kOne, (int64_t)0);
      TNX_LAUNCH_CHECK();
    }
  } else {
    // FP64 Lanczos exit: hvec was written from the Lanczos relation.
    TNX_TRY(copy_f64(k.y, vec, N, s));
  }
  TNX_HIP(hipStreamSynchronize(s));
  info->eval = theta;
  info->resnorm = rho;
  info->anorm = anorm;
  info->matvecs = c.matvecs;
  info->matvecs_f64 = c.matvecs64;
  info->restarts = restarts;
  info->converged = converged ? 1 : 0;
  return converged ? TNX_OK : TNX_ERR_NOCONV;
}

// ---------------------------------------------------------------------------
// Batched eigensolves: `batch` independent one-site problems of one shape
// (stacks of L, W, R, v0; outputs vec, hvec stacked). FP64 thick-restart
// Lanczos in lockstep: every problem is at the same Lanczos step (restarts
// keep exactly `keep` vectors), each problem's Krylov scalars are its own,
// and a problem leaves the launched set (device index list) once its
// residual estimate meets tol * ||H||_est. One launch per kernel per step
// covers all problems still iterating.
// ---------------------------------------------------------------------------
size_t heff1_ws_bytes_b(int chil, int Dl, int Dr, int d, int chir, int batch);

// out[i * nst + t] = st[first + t] of launched problem i
__global__ void gather_status_kernel(const double* __restrict__ st, int first, int nst,
                                     double* __restrict__ out, PMap pm) {
  const int t = threadIdx.x;
  if (t < nst) out[(int64_t)blockIdx.y * nst + t] = st[pm.off() + first + t];
}

// Device-decided convergence (see chunk_mark): clear the flags and start
// the running ||T|| estimate at |theta| of the start vector (st[4]).
__global__ void chunk_init_kernel(double* st, PMap pm) {
  st += pm.off();
  if (threadIdx.x == 0) {
    st[10] = 0.0;
    st[11] = 0.0;
    st[12] = fabs(st[4]);
  }
}

// Results of the problems that finished within a run of steps: with Jc
// the problem's row count at convergence (st[11]; Jl for one that did not
// converge), vec = y = V[0..Jc) s and hvec = theta y + beta[Jc-1] s[Jc-1]
// V[Jc] (the beta term dropped for a problem stopped by an exhausted
// space). vec/hvec of logical problem p at p * N.
__global__ void chunk_finalize_kernel(const double* __restrict__ V, int64_t N,
                                      const double* __restrict__ s, const double* __restrict__ st,
                                      const double* __restrict__ beta, int Jl, int exhausted,
                                      double* __restrict__ vec, double* __restrict__ hvec, PMap pm) {
  const int64_t o = pm.off();
  V += o; s += o; st += o; beta += o;
  const int64_t po = (int64_t)pm.pid() * N;
  __shared__ double cs[kMaxBasis + 1];
  const bool done = st[10] != 0.0;
  const int Jc = done ? (int)st[11] : Jl;
  if ((int)threadIdx.x < Jc) cs[threadIdx.x] = s[threadIdx.x];
  __syncthreads();
  const double th = st[0];
  const double c = (!done && exhausted) ? 0.0 : beta[Jc - 1] * s[Jc - 1];
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < N;
       i += (int64_t)gridDim.x * blockDim.x) {
    double acc = 0.0;
    for (int t = 0; t < Jc; ++t) acc += cs[t] * V[(int64_t)t * N + i];
    vec[po + i] = acc;
    if (hvec) hvec[po + i] = th * acc + c * V[(int64_t)Jc * N + i];
  }
}

static size_t eigsh_b_problem_bytes(size_t N, int m) { return align256(eigsh_ws_bytes_n(N, 0, m)); }

size_t eigsh_b_ws_bytes(int chil, int Dl, int Dr, int d, int chir, int max_basis, int batch) {
  const int m = std::max(3, std::min(max_basis, kMaxBasis));
  const size_t N = (size_t)chil * d * chir;
  return align256(heff1_ws_bytes_b(chil, Dl, Dr, d, chir, batch)) +
         2 * align256((size_t)batch * sizeof(int)) + align256((size_t)batch * 16 * 8) +
         eigsh_b_problem_bytes(N, m) * (size_t)batch + 256;
}

int eigsh_heff1_b(const double* L, const double* W, const double* R, const double* v0,
                  double* vec, double* hvec, int chil, int Dl, int Dr, int d, int chir,
                  int batch, const tnx_eigsh_opts_t* opts, tnx_eigsh_info_t* info, void* ws,
                  size_t ws_bytes, hipStream_t s) {
  TNX_CHECK_ARG(opts && info, "eigsh_batched: null opts/info");
  TNX_CHECK_ARG(L && W && R && v0 && vec && hvec, "eigsh_batched: null pointer");
  TNX_CHECK_ARG(chil > 0 && Dl > 0 && Dr > 0 && d > 0 && chir > 0, "eigsh_batched: bad dims");
  TNX_CHECK_ARG(batch >= 1 && batch <= 65535, "eigsh_batched: bad batch %d", batch);
  TNX_CHECK_ARG(opts->tol >= 0.0, "eigsh_batched: negative tol");
  if (opts->precision != TNX_F64) {
    set_error("eigsh_batched: only FP64 (precision 0) is supported, got %d", opts->precision);
    return TNX_ERR_UNSUPPORTED;
  }
  const int m = std::max(3, std::min(opts->max_basis, kMaxBasis));
  const int64_t N = (int64_t)chil * d * chir;
  TNX_CHECK_ARG(ws && ws_bytes >= eigsh_b_ws_bytes(chil, Dl, Dr, d, chir, m, batch),
                "eigsh_batched: workspace too small");
  const int max_mv = opts->max_matvecs > 0 ? opts->max_matvecs : 10000;
  const double tol = opts->tol;
  const int mb = (int)std::min<int64_t>(m, std::max<int64_t>(N, 1));
  const int keep = keep_of(mb, opts->keep);

  char* p = (char*)(((uintptr_t)ws + 255) & ~(uintptr_t)255);
  void* mv = p;
  const size_t mvb = heff1_ws_bytes_b(chil, Dl, Dr, d, chir, batch);
  p += align256(mvb);
  int* idx = (int*)p; p += align256((size_t)batch * sizeof(int));
  int* fidx = (int*)p; p += align256((size_t)batch * sizeof(int));
  double* stat = (double*)p; p += align256((size_t)batch * 16 * 8);
  const size_t P = eigsh_b_problem_bytes((size_t)N, m);
  const int64_t sp = (int64_t)(P / 8);
  KWork k;
  carve(k, p, m, (size_t)N, 0);  // problem 0; problem q at + q * sp doubles

  std::vector<int> act(batch), fin;
  for (int b = 0; b < batch; ++b) act[b] = b;
  std::vector<double> anorm(batch, 0.0), hs((size_t)batch * 16);
  for (int b = 0; b < batch; ++b) info[b] = tnx_eigsh_info_t{0.0, 0.0, 0.0, 0, 0, 0, 0};
  int matvecs = 0, restarts = 0;
  bool any_fail = false;

  auto upload = [&](int* dst, const std::vector<int>& v) -> int {
    TNX_HIP(hipMemcpyAsync(dst, v.data(), v.size() * sizeof(int), hipMemcpyHostToDevice, s));
    return TNX_OK;
  };
  auto status = [&](int first, int nst, int cnt) -> int {
    hipLaunchKernelGGL(gather_status_kernel, dim3(1, cnt), dim3(64), 0, s, k.st, first, nst, stat,
                       PMap{idx, sp});
    TNX_LAUNCH_CHECK();
    TNX_HIP(hipMemcpyAsync(hs.data(), stat, sizeof(double) * nst * cnt, hipMemcpyDeviceToHost, s));
    TNX_HIP(hipStreamSynchronize(s));
    return TNX_OK;
  };
  auto matvec = [&](const double* x, double* y, int cnt) -> int {
    matvecs++;
    return heff1_matvec_b(L, W, R, x, 0, y, chil, Dl, Dr, d, chir, TNX_F64, batch, cnt, idx, sp,
                          sp, mv, mvb, s, 0);
  };

  TNX_TRY(upload(idx, act));
  int cnt = batch;
  PMap pm{idx, sp};
  // y = v0 / |v0|
  hipLaunchKernelGGL(copy_map_kernel, dim3(vec_blocks(N, cnt), cnt), dim3(256), 0, s, v0, k.y, N,
                     pm, N, sp);
  TNX_LAUNCH_CHECK();
  TNX_TRY(cgs_pass(k.y, N, 0, k.y, nullptr, false, k.partials, k.h3, N, s, pm, cnt));
  hipLaunchKernelGGL(normalize_kernel<double>, dim3(vec_blocks(N, cnt), cnt), dim3(256), 0, s, k.y, k.h3,
                     k.y, N, pm);
  TNX_LAUNCH_CHECK();
  // FP64 step on the start vectors: theta = y.Hy, r = Hy - theta y
  TNX_TRY(matvec(k.y, k.w, cnt));
  TNX_TRY(cgs_pass(k.y, N, 1, k.w, nullptr, true, k.partials, k.h1, N, s, pm, cnt));
  TNX_TRY(cgs_pass(k.y, N, 1, k.w, k.h1, true, k.partials, k.h2, N, s, pm, cnt));
  TNX_TRY(cgs_pass(k.y, N, 1, k.w, k.h2, false, k.partials, k.h3, N, s, pm, cnt));
  hipLaunchKernelGGL(outer_scalars_kernel, dim3(1, cnt), dim3(256), 0, s, k.h1, k.h2, k.h3,
                     k.alpha, k.beta, k.scal, k.st, k.T, pm);
  TNX_LAUNCH_CHECK();
  TNX_TRY(status(4, 2, cnt));
  {
    std::vector<int> rest;
    fin.clear();
    for (int i = 0; i < cnt; ++i) {
      const int b = act[i];
      const double th = hs[2 * i], rho = hs[2 * i + 1];
      anorm[b] = std::max(anorm[b], std::fabs(th));
      info[b].eval = th;
      info[b].resnorm = rho;
      info[b].matvecs = info[b].matvecs_f64 = matvecs;
      if (rho <= tol * anorm[b] || rho == 0.0 || N == 1) {
        fin.push_back(b);
        info[b].converged = 1;
      } else {
        rest.push_back(b);
      }
    }
    if (!fin.empty()) {
      // converged start vectors: vec = y, hvec = r + theta y
      TNX_TRY(upload(fidx, fin));
      const int fc = (int)fin.size();
      PMap pf{fidx, sp};
      hipLaunchKernelGGL(copy_map_kernel, dim3(vec_blocks(N, fc), fc), dim3(256), 0, s, k.y, vec,
                         N, pf, sp, N);
      TNX_LAUNCH_CHECK();
      hipLaunchKernelGGL(axpbz_dev_kernel, dim3(vec_blocks(N, fc), fc), dim3(256), 0, s,
                         k.scal + 3, k.w, k.scal, k.y, hvec, N, pf, N);
      TNX_LAUNCH_CHECK();
    }
    act.swap(rest);
  }
  cnt = (int)act.size();
  if (cnt > 0) {
    TNX_TRY(upload(idx, act));
    // V[0] = y, V[1] = r / rho
    hipLaunchKernelGGL(copy_map_kernel, dim3(vec_blocks(N, cnt), cnt), dim3(256), 0, s, k.y, k.V,
                       N, pm, sp, sp);
    TNX_LAUNCH_CHECK();
    hipLaunchKernelGGL(normalize_kernel<double>, dim3(vec_blocks(N, cnt), cnt), dim3(256), 0, s, k.w,
                       k.h3 + 1, k.V + N, N, pm);
    TNX_LAUNCH_CHECK();
  }
  // Step pipelining as in the single-problem solver: the next step's
  // matvec and CGS passes for every active problem are queued before the
  // host reads this step's statuses; problems that finish here drop theirs
  // (not counted), the others take it as their next step.
  StepEvent sev;
  PinnedLease pin_lease((size_t)3 * batch);
  double* pin = pin_lease.get();
  const bool pipelined = sev.e != nullptr && pin != nullptr;
  int prows = 0;  // partial rows of the last front
  auto front = [&](int jj) -> int {
    prows = rows_blocks(N, cnt);
    TNX_TRY(matvec(k.V + (int64_t)jj * N, k.w, cnt));
    return cgs_step(k.V, N, jj + 1, k.w, k.partials, k.h1, k.h2, k.h3, s, pm, cnt);
  };
  // Device-decided convergence: with steps_per_check K > 1 the host queues
  // up to K lockstep steps (bounded by the next restart, an exhausted space
  // and the matvec limit) without reading statuses. Each problem's
  // tridiagonal solve tests the criterion itself and freezes the problem's
  // Ritz pair when it is met (chunk_mark), so a finished problem keeps its
  // result while the others step on. One status read per run of steps then
  // retires the finished problems (their Ritz vectors from the basis rows up
  // to their own convergence) and restarts the rest when the basis is full.
  const int K = opts->steps_per_check > 1 ? std::min(opts->steps_per_check, kMaxBasis) : 1;
  if (K > 1 && cnt > 0) {
    hipLaunchKernelGGL(chunk_init_kernel, dim3(1, cnt), dim3(64), 0, s, k.st, pm);
    TNX_LAUNCH_CHECK();
    int jc = 1;
    while (cnt > 0) {
      const int nb = vec_blocks(N, cnt);
      const int mv0 = matvecs;
      int steps = std::min(K, mb - jc);
      steps = (int)std::min<int64_t>(steps, N - jc);
      steps = std::max(0, std::min(steps, max_mv - matvecs));
      for (int t = 0; t < steps; ++t) {
        const int jj = jc + t, JJ = jj + 1;
        TNX_TRY(front(jj));
        TNX_TRY(finish_step(k.V, N, JJ, k.w, k.partials, prows, k.h3, k.s, k.st,
                            TriFinish{k.h1, k.h2, k.alpha, k.beta, k.T}, tol, nullptr, s, pm, cnt));
      }
      const int Jl = jc + steps;  // basis rows after the last step
      TNX_TRY(status(0, 13, cnt));
      const bool exhausted = Jl >= N;
      const bool limit = matvecs >= max_mv;
      std::vector<int> rest;
      fin.clear();
      for (int i = 0; i < cnt; ++i) {
        const int b = act[i];
        const double* h = &hs[(size_t)13 * i];
        const bool done = h[10] != 0.0;
        anorm[b] = std::max(anorm[b], h[12]);
        if (done || exhausted || limit) {
          const int Jc = done ? (int)h[11] : Jl;
          fin.push_back(b);
          info[b].eval = h[0];
          info[b].resnorm = h[1];
          info[b].matvecs = info[b].matvecs_f64 = mv0 + (Jc - jc);
          info[b].restarts = restarts;
          info[b].converged = (done || exhausted) ? 1 : 0;
          any_fail |= !(done || exhausted);
        } else {
          rest.push_back(b);
        }
      }
      if (!fin.empty()) {
        TNX_TRY(upload(fidx, fin));
        const int fc = (int)fin.size();
        hipLaunchKernelGGL(chunk_finalize_kernel, dim3(vec_blocks(N, fc), fc), dim3(256), 0, s,
                           k.V, N, k.s, k.st, k.beta, Jl, exhausted ? 1 : 0, vec, hvec,
                           PMap{fidx, sp});
        TNX_LAUNCH_CHECK();
        act.swap(rest);
        cnt = (int)act.size();
        if (cnt == 0) break;
        TNX_TRY(upload(idx, act));
      }
      if (Jl >= mb) {
        const int jl = Jl - 1;
        hipLaunchKernelGGL(tridiag_all_kernel, dim3(1, cnt), dim3(256), 0, s, k.alpha, k.beta, Jl,
                           k.theta, k.S, kMaxBasis, pm);
        TNX_LAUNCH_CHECK();
        hipLaunchKernelGGL(tr_restart_kernel, dim3(1, cnt), dim3(64), 0, s, k.theta, k.S, k.beta, jl,
                           keep, Jl, k.Cm, k.alpha, k.beta, k.T,
                           reinterpret_cast<int*>(k.st + 8), pm);
        TNX_LAUNCH_CHECK();
        GemmDesc g{};
        g.M = keep; g.N = (int)N; g.K = Jl; g.batch = cnt; g.bidx = idx;
        g.A = k.Cm; g.ta = DT::F64; g.lda = kMaxBasis; g.sA = sp; g.a_kcontig = false;
        g.B = k.V; g.tb = DT::F64; g.ldb = N; g.sB = sp; g.b_ncontig = true;
        g.C = k.Y; g.tc = DT::F64; g.ldc = N; g.sC = sp;
        g.alpha = 1.0; g.beta = 0.0; g.prec = Prec::F64;
        TNX_TRY(gemm(g, s));
        hipLaunchKernelGGL(copy_map_kernel, dim3(vec_blocks((int64_t)keep * N, cnt), cnt),
                           dim3(256), 0, s, k.Y, k.V, (int64_t)keep * N, pm, sp, sp);
        TNX_LAUNCH_CHECK();
        hipLaunchKernelGGL(copy_map_kernel, dim3(vec_blocks(N, cnt), cnt), dim3(256), 0, s,
                           k.V + (int64_t)Jl * N, k.V + (int64_t)keep * N, N, pm, sp, sp);
        TNX_LAUNCH_CHECK();
        restarts++;
        jc = keep;
      } else {
        jc = Jl;
      }
    }
    TNX_HIP(hipStreamSynchronize(s));
    for (int b = 0; b < batch; ++b) info[b].anorm = anorm[b];
    if (any_fail) {
      set_error("eigsh_batched: matvec limit %d reached before convergence", max_mv);
      return TNX_ERR_NOCONV;
    }
    return TNX_OK;
  }
  int j = 1;
  bool queued = false;  // step j's front already launched for the active set
  while (cnt > 0) {
    const int nb = vec_blocks(N, cnt);
    const int J = j + 1;
    if (!queued) TNX_TRY(front(j));
    const int mv_now = matvecs;
    TNX_TRY(finish_step(k.V, N, J, k.w, k.partials, prows, k.h3, k.s, k.st,
                        TriFinish{k.h1, k.h2, k.alpha, k.beta, k.T}, -1.0, nullptr, s, pm, cnt));
    const bool ahead = pipelined && J < mb && J < N && mv_now < max_mv;
    if (ahead) {
      hipLaunchKernelGGL(gather_status_kernel, dim3(1, cnt), dim3(64), 0, s, k.st, 0, 3, stat, pm);
      TNX_LAUNCH_CHECK();
      TNX_HIP(hipMemcpyAsync(pin, stat, sizeof(double) * 3 * cnt, hipMemcpyDeviceToHost, s));
      TNX_HIP(hipEventRecord(sev.e, s));
      TNX_TRY(front(j + 1));
      TNX_HIP(hipEventSynchronize(sev.e));
      std::copy(pin, pin + (size_t)3 * cnt, hs.begin());
    } else {
      TNX_TRY(status(0, 3, cnt));
    }
    const bool exhausted = (J >= N);
    const bool limit = mv_now >= max_mv;
    std::vector<int> rest;
    fin.clear();
    for (int i = 0; i < cnt; ++i) {
      const int b = act[i];
      const double th = hs[3 * i], est = hs[3 * i + 1];
      anorm[b] = std::max(anorm[b], hs[3 * i + 2]);
      const bool conv = est <= tol * anorm[b] || exhausted;
      if (conv || limit) {
        fin.push_back(b);
        info[b].eval = th;
        info[b].resnorm = est;
        info[b].matvecs = info[b].matvecs_f64 = mv_now;
        info[b].restarts = restarts;
        info[b].converged = conv ? 1 : 0;
        any_fail |= !conv;
      } else {
        rest.push_back(b);
      }
    }
    if (!fin.empty()) {
      // Ritz vector y = V s; H y = theta y + beta_j s_j V[j+1]
      TNX_TRY(upload(fidx, fin));
      const int fc = (int)fin.size();
      const int nf = vec_blocks(N, fc);
      PMap pf{fidx, sp};
      hipLaunchKernelGGL(vcomb_kernel<double>, dim3(nf, fc), dim3(256), 0, s, k.V, N, J, k.s, k.y, N, pf);
      TNX_LAUNCH_CHECK();
      hipLaunchKernelGGL(ritz_scalars_kernel, dim3(1, fc), dim3(1), 0, s, k.st, k.s, k.beta, j,
                         k.scal, pf);
      TNX_LAUNCH_CHECK();
      hipLaunchKernelGGL(axpbz_dev_kernel, dim3(nf, fc), dim3(256), 0, s, k.scal, k.y,
                         exhausted ? nullptr : k.scal + 1, k.V + (int64_t)(j + 1) * N, hvec, N,
                         pf, N);
      TNX_LAUNCH_CHECK();
      hipLaunchKernelGGL(copy_map_kernel, dim3(nf, fc), dim3(256), 0, s, k.y, vec, N, pf, sp, N);
      TNX_LAUNCH_CHECK();
      act.swap(rest);
      cnt = (int)act.size();
      if (cnt == 0) break;
      TNX_TRY(upload(idx, act));
    }
    if (J >= mb) {
      hipLaunchKernelGGL(tridiag_all_kernel, dim3(1, cnt), dim3(256), 0, s, k.alpha, k.beta, J,
                         k.theta, k.S, kMaxBasis, pm);
      TNX_LAUNCH_CHECK();
      hipLaunchKernelGGL(tr_restart_kernel, dim3(1, cnt), dim3(64), 0, s, k.theta, k.S, k.beta, j,
                         keep, J, k.Cm, k.alpha, k.beta, k.T,
                         reinterpret_cast<int*>(k.st + 8), pm);
      TNX_LAUNCH_CHECK();
      // Y = C^T V (keep x N per problem), then V[0..keep) = Y, V[keep] = V[j+1]
      GemmDesc g{};
      g.M = keep; g.N = (int)N; g.K = J; g.batch = cnt; g.bidx = idx;
      g.A = k.Cm; g.ta = DT::F64; g.lda = kMaxBasis; g.sA = sp; g.a_kcontig = false;
      g.B = k.V; g.tb = DT::F64; g.ldb = N; g.sB = sp; g.b_ncontig = true;
      g.C = k.Y; g.tc = DT::F64; g.ldc = N; g.sC = sp;
      g.alpha = 1.0; g.beta = 0.0; g.prec = Prec::F64;
      TNX_TRY(gemm(g, s));
      hipLaunchKernelGGL(copy_map_kernel, dim3(vec_blocks((int64_t)keep * N, cnt), cnt),
                         dim3(256), 0, s, k.Y, k.V, (int64_t)keep * N, pm, sp, sp);
      TNX_LAUNCH_CHECK();
      hipLaunchKernelGGL(copy_map_kernel, dim3(nb, cnt), dim3(256), 0, s,
                         k.V + (int64_t)(j + 1) * N, k.V + (int64_t)keep * N, N, pm, sp, sp);
      TNX_LAUNCH_CHECK();
      restarts++;
      j = keep;
      queued = false;
    } else {
      j++;
      queued = ahead;
    }
  }
  TNX_HIP(hipStreamSynchronize(s));
  for (int b = 0; b < batch; ++b) info[b].anorm = anorm[b];
  if (any_fail) {
    set_error("eigsh_batched: matvec limit %d reached before convergence", max_mv);
    return TNX_ERR_NOCONV;
  }
  return TNX_OK;
}

// Lowest eigenpairs of `batch` dense symmetric n x n matrices (stacked).
size_t syev_b_ws_bytes(int n, int batch) {
  return align256((size_t)batch * 8) + align256(syev_ws_bytes(n)) * (size_t)batch + 256;
}

int syev_lowest_b(const double* M, int n, int batch, double* evec, double* eval_host, void* ws,
                  size_t ws_bytes, hipStream_t s) {
  TNX_CHECK_ARG(n >= 1 && n <= kTriMax, "syev_batched: n=%d outside [1, %d]", n, kTriMax);
  TNX_CHECK_ARG(batch >= 1 && batch <= 65535, "syev_batched: bad batch %d", batch);
  TNX_CHECK_ARG(M && evec && eval_host, "syev_batched: null pointer");
  TNX_CHECK_ARG(ws && ws_bytes >= syev_b_ws_bytes(n, batch), "syev_batched: workspace too small");
  char* p = (char*)(((uintptr_t)ws + 255) & ~(uintptr_t)255);
  double* ev = (double*)p; p += align256((size_t)batch * 8);
  const int64_t nn = (int64_t)n * n;
  if (n == 1) {
    TNX_TRY(fill_f64(evec, batch, 1.0, s));
    TNX_HIP(hipMemcpyAsync(eval_host, M, sizeof(double) * batch, hipMemcpyDeviceToHost, s));
    TNX_HIP(hipStreamSynchronize(s));
    return TNX_OK;
  }
  const int64_t sp = (int64_t)(align256(syev_ws_bytes(n)) / 8);
  double* A = (double*)p;
  double* Vst = A + nn;
  double* tau = Vst + nn;
  double* dg = tau + n;
  double* eg = dg + n;
  double* z = eg + n;
  double* st = z + n + 8;
  const PMap pm{nullptr, sp};
  TNX_TRY(sytrd(M, nn, n, A, Vst, tau, dg, eg, batch, pm, s));
  hipLaunchKernelGGL(tridiag_lowest_kernel, dim3(1, batch), dim3(64), 0, s, dg, eg, n, z, st, pm);
  TNX_LAUNCH_CHECK();
  TNX_TRY(ormtr(Vst, tau, n, z, evec, batch, pm, n, s));
  hipLaunchKernelGGL(gather_status_kernel, dim3(1, batch), dim3(64), 0, s, st, 0, 1, ev, pm);
  TNX_LAUNCH_CHECK();
  TNX_HIP(hipMemcpyAsync(eval_host, ev, sizeof(double) * batch, hipMemcpyDeviceToHost, s));
  TNX_HIP(hipStreamSynchronize(s));
  return TNX_OK;
}

}  // namespace tnx

// ---- C-ABI -----------------------------------------------------------------
extern "C" {

size_t tnx_syev_lowest_workspace_bytes(int n) { return tnx::syev_ws_bytes(n); }

int tnx_syev_lowest(const double* M, int n, double* evec, double* eval_host, void* ws,
                    size_t ws_bytes, tnx_stream_t stream) {
  TNX_CHECK_ARG(eval_host, "tnx_syev_lowest: null eval_host");
  return tnx::syev_lowest(M, n, evec, eval_host, ws, ws_bytes, (hipStream_t)stream);
}

size_t tnx_eigsh_heff1_workspace_bytes(int chil, int Dl, int Dr, int d, int chir,
                                       int max_basis) {
  return tnx::eigsh_ws_bytes(chil, Dl, Dr, d, chir, max_basis);
}

size_t tnx_eigsh_heff2_workspace_bytes(int chil, int Dl, int Dm, int Dr, int d, int chir,
                                       int max_basis) {
  return tnx::eigsh2_ws_bytes(chil, Dl, Dm, Dr, d, chir, max_basis);
}

int tnx_eigsh_heff2(const double* L, const double* W1, const double* W2, const double* R,
                    const double* v0, double* vec, double* hvec, int chil, int Dl, int Dm,
                    int Dr, int d, int chir, const tnx_eigsh_opts_t* opts,
                    tnx_eigsh_info_t* info, void* ws, size_t ws_bytes, tnx_stream_t stream) {
  return tnx::eigsh_heff2(L, W1, W2, R, v0, vec, hvec, chil, Dl, Dm, Dr, d, chir, opts, info,
                          ws, ws_bytes, (hipStream_t)stream);
}

int tnx_eigsh_heff1(const double* L, const double* W, const double* R, const double* v0,
                    double* vec, double* hvec, int chil, int Dl, int Dr, int d, int chir,
                    const tnx_eigsh_opts_t* opts, tnx_eigsh_info_t* info, void* ws,
                    size_t ws_bytes, tnx_stream_t stream) {
  return tnx::eigsh_heff1(L, W, R, v0, vec, hvec, chil, Dl, Dr, d, chir, opts, info, ws,
                          ws_bytes, (hipStream_t)stream);
}

int tnx_axpy(int64_t n, double alpha, const double* x, double* y, tnx_stream_t stream) {
  using namespace tnx;
  TNX_CHECK_ARG(n >= 0, "tnx_axpy: negative n");
  if (n == 0) return TNX_OK;
  TNX_CHECK_ARG(x && y, "tnx_axpy: null pointer");
  hipLaunchKernelGGL(axpy_kernel, dim3(vec_blocks(n)), dim3(256), 0, (hipStream_t)stream, n,
                     alpha, x, y);
  TNX_LAUNCH_CHECK();
  return TNX_OK;
}

int tnx_scal(int64_t n, double alpha, double* x, tnx_stream_t stream) {
  using namespace tnx;
  TNX_CHECK_ARG(n >= 0, "tnx_scal: negative n");
  if (n == 0) return TNX_OK;
  TNX_CHECK_ARG(x, "tnx_scal: null pointer");
  hipLaunchKernelGGL(scal_kernel, dim3(vec_blocks(n)), dim3(256), 0, (hipStream_t)stream, n,
                     alpha, x);
  TNX_LAUNCH_CHECK();
  return TNX_OK;
}

size_t tnx_dot_workspace_bytes(int64_t n) {
  (void)n;
  return (size_t)(tnx::kCgsBlocks + 2) * tnx::kPartStride * 8 + 256;
}

int tnx_dot(int64_t n, const double* x, const double* y, double* out_host, void* ws,
            size_t ws_bytes, tnx_stream_t stream) {
  using namespace tnx;
  TNX_CHECK_ARG(n >= 1 && x && y && out_host, "tnx_dot: bad arguments");
  TNX_CHECK_ARG(ws && ws_bytes >= tnx_dot_workspace_bytes(n), "tnx_dot: workspace too small");
  hipStream_t s = (hipStream_t)stream;
  double* partials = (double*)(((uintptr_t)ws + 255) & ~(uintptr_t)255);
  double* out = partials + (size_t)kCgsBlocks * kPartStride;
  // one pass with V = x (J = 1), w = y: out[0] = x.y
  TNX_TRY(cgs_pass(x, n, 1, const_cast<double*>(y), nullptr, true, partials, out, n, s));
  TNX_HIP(hipMemcpyAsync(out_host, out, sizeof(double), hipMemcpyDeviceToHost, s));
  TNX_HIP(hipStreamSynchronize(s));
  return TNX_OK;
}

size_t tnx_syev_lowest_batched_workspace_bytes(int n, int batch) {
  return tnx::syev_b_ws_bytes(n, batch);
}

int tnx_syev_lowest_batched(const double* M, int n, int batch, double* evec,
                            double* eval_host, void* ws, size_t ws_bytes,
                            tnx_stream_t stream) {
  return tnx::syev_lowest_b(M, n, batch, evec, eval_host, ws, ws_bytes, (hipStream_t)stream);
}

size_t tnx_eigsh_heff1_batched_workspace_bytes(int chil, int Dl, int Dr, int d, int chir,
                                               int max_basis, int batch) {
  return tnx::eigsh_b_ws_bytes(chil, Dl, Dr, d, chir, max_basis, batch);
}

int tnx_eigsh_heff1_batched(const double* L, const double* W, const double* R,
                            const double* v0, double* vec, double* hvec, int chil,
                            int Dl, int Dr, int d, int chir, int batch,
                            const tnx_eigsh_opts_t* opts, tnx_eigsh_info_t* info,
                            void* ws, size_t ws_bytes, tnx_stream_t stream) {
  return tnx::eigsh_heff1_b(L, W, R, v0, vec, hvec, chil, Dl, Dr, d, chir, batch, opts, info, ws,
                            ws_bytes, (hipStream_t)stream);
}

}  // extern "C"
