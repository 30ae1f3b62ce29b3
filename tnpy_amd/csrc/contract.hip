// One-site effective-Hamiltonian matvec, environment updates and the dense
// effective matrix.
//
// Each contraction is GEMM -> W-apply -> GEMM:
//   matvec  (tnpy/matrix_product_state.py:411-440)
//     T1[a,k,v,s] = sum_r   x[a,k,r] R[r,v,s]            GEMM, K = chir
//     T2[a,w,c,s] = sum_k,v W[w,v,k,c] T1[a,k,v,s]        W-apply
//     y[b,c,s]    = sum_a,w L[a,w,b] T2[a,w,c,s]          GEMM, K = chil*Dl
//   left env  (tnpy/matrix_product_state.py:296-315)
//     T1[w,b,k,r] = sum_a   L[a,w,b] A[a,k,r]            GEMM, K = chil
//     T2[v,b,c,r] = sum_w,k W[w,v,k,c] T1[w,b,k,r]        W-apply
//     L'[r,v,s]   = sum_b,c T2[v,b,c,r] A[b,c,s]          Dr batched GEMMs
//   right env (tnpy/matrix_product_state.py:317-336)
//     T1[a,k,v,s] = sum_r   A[a,k,r] R[r,v,s]            GEMM
//     T2[a,w,c,s] = sum_k,v W[w,v,k,c] T1[a,k,v,s]        W-apply
//     R'[a,w,b]   = sum_c,s T2[a,w,c,s] A[b,c,s]          GEMM (B k-contiguous)
// The GEMMs carry 2*D*d*chi^3 flops each; the W-apply is a D*d-wide local
// map on the matrix cores, bound by HBM (each (outer, inner) pair reads d*Dr
// values and writes Dl*d values, coalesced along the inner bond index).
#include "tnx_common.h"

#include <type_traits>

namespace tnx {

// out[o][p][q][i] = sum_{x,y} C(p,q,x,y) in[o][x][y][i], C from W by a
// permutation selected by `mode`:
//   mode 0 (matvec / right env): p=w, q=c, x=k, y=v : C = W[w][v][k][c]
//   mode 1 (left env)          : p=v, q=c, x=w, y=k : C = W[w][v][k][c]
struct WApply {
  const void* in; void* out; const double* W;
  int in_f32;  // in and out are float (else double)
  int64_t n_outer, n_inner;
  int64_t in_so, in_sx, in_sy;     // strides of o, x, y in `in`
  int64_t out_so, out_sp, out_sq;  // strides of o, p, q in `out`
  int NX, NY, NP, NQ;
  int Dl, Dr, d, mode;
  // batch of independent problems (grid.y): strides of in, out and W
  int batch = 1;
  int64_t in_sb = 0, out_sb = 0, W_sb = 0;
  const int* bidx = nullptr;  // launched -> logical problem, or null
};

// The local map on the FP64 matrix cores: out = C in, C (outputs x inputs,
// at most 64 x 64) in registers as the A operand, the inputs of 32 points as
// the B operand. A matrix of D d rows per point is far below the matrix
// cores' rate, so the kernel is left bound by HBM (each value written once and
// read once per 16 outputs, a grid slice each: one reading at D d <= 16, four
// at D d = 50) or, at small bonds, by one round of loads. The form before
// (one point per thread, C in LDS, D d dot products of D d terms each on the
// VALU) measured 51 us at chi = 1024, D = 5 (168 MB), 12 us at chi = 32 and
// 137 us at chi = 200 with D = 25; this one 27 (6.1 TB/s), 3.9 and 20 us.
//
// A wave takes 16 pairs of neighbouring points at a time: lane (i = lane %
// 16, g = lane / 16) loads input rows t = 4 ks + g of pair i (two points,
// one 16-byte load of doubles) and feeds the pair's points to two MFMA
// columns, so an output row is stored as pairs too. Pairs lie along the
// inner index and are numbered through all outer ones, so short inner
// extents still fill the wave; the last pair of an odd extent is loaded one
// point back. PAIR = false (inner extent 1): one point per lane. Inputs past
// the last row are zero and never loaded from outside.
typedef double wa_f64x2 __attribute__((ext_vector_type(2), aligned(8)));
typedef float wa_f32x2 __attribute__((ext_vector_type(2), aligned(4)));
typedef double wa_f64x4 __attribute__((ext_vector_type(4)));

template <int KS, bool PAIR, typename T>
__global__ __launch_bounds__(256) void wapply_kernel(WApply a) {
  using T2 = typename std::conditional<sizeof(T) == 8, wa_f64x2, wa_f32x2>::type;
  const int nin = a.NX * a.NY, nout = a.NP * a.NQ;
  const int lane = threadIdx.x & 63, li = lane & 15, lg = lane >> 4;
  const int b = a.bidx ? a.bidx[blockIdx.y] : (int)blockIdx.y;
  const T* in = (const T*)a.in + (int64_t)b * a.in_sb;
  T* out = (T*)a.out + (int64_t)b * a.out_sb;
  const double* W = a.W + (int64_t)b * a.W_sb;
  // C's fragments: row r0 + li, column 4 ks + lg
  const int r0 = 16 * blockIdx.z;
  double c[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    const int r = r0 + li, t = 4 * ks + lg;
    c[ks] = 0.0;
    if (r < nout && t < nin) {
      const int p = r / a.NQ, q = r % a.NQ, x = t / a.NY, y = t % a.NY;
      const int w = a.mode == 0 ? p : x, v = a.mode == 0 ? y : p, k = a.mode == 0 ? x : y;
      c[ks] = W[((w * a.Dr + v) * a.d + k) * a.d + q];
    }
  }
  int64_t irow[KS];  // offset of input row 4 ks + lg (row 0 past the last)
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    const int t = 4 * ks + lg;
    irow[ks] = t < nin ? (t / a.NY) * a.in_sx + (t % a.NY) * a.in_sy : 0;
  }
  int64_t orow[4];  // offset of output row r0 + lg + 4 v
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const int r = r0 + lg + 4 * v;
    orow[v] = (r / a.NQ) * a.out_sp + (r % a.NQ) * a.out_sq;
  }
  const unsigned inner = (unsigned)a.n_inner;
  const unsigned per = PAIR ? (inner + 1) / 2 : inner;  // columns per outer index
  const int64_t total = (int64_t)a.n_outer * per;
  const int64_t wave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const int64_t waves = ((int64_t)gridDim.x * blockDim.x) >> 6;
  for (int64_t c0 = wave * 16; c0 < total; c0 += waves * 16) {
    const int64_t col = c0 + li;
    const bool on = col < total;
    const unsigned pc = (unsigned)(on ? col : 0);
    const unsigned o = pc / per;
    const unsigned i = (pc - o * per) * (PAIR ? 2 : 1);
    const bool half = PAIR && i + 1 == inner;  // odd extent: one point left
    const T* src = in + (int64_t)o * a.in_so + (half ? i - 1 : i);
    double x0[KS], x1[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const bool in_k = 4 * ks + lg < nin;
      if constexpr (PAIR) {
        const T2 v = *reinterpret_cast<const T2*>(src + irow[ks]);
        x0[ks] = in_k ? (double)(half ? v[1] : v[0]) : 0.0;
        x1[ks] = in_k ? (double)v[1] : 0.0;
      } else {
        x0[ks] = in_k ? (double)src[irow[ks]] : 0.0;
      }
    }
    wa_f64x4 y0 = {0.0, 0.0, 0.0, 0.0}, y1 = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      y0 = __builtin_amdgcn_mfma_f64_16x16x4f64(c[ks], x0[ks], y0, 0, 0, 0);
      if constexpr (PAIR) y1 = __builtin_amdgcn_mfma_f64_16x16x4f64(c[ks], x1[ks], y1, 0, 0, 0);
    }
    // element v sits at row lg + 4 v, column li
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      if (!on || r0 + lg + 4 * v >= nout) continue;
      T* dst = out + (int64_t)o * a.out_so + orow[v] + i;
      if (PAIR && !half) *reinterpret_cast<T2*>(dst) = T2{(T)y0[v], (T)y1[v]};
      else *dst = (T)y0[v];
    }
  }
}

// At most kWaColumns columns a launch, which the kernel counts in 32 bits.
constexpr int64_t kWaColumns = ((int64_t)1 << 31) - 1;

static int launch_wapply(const WApply& a, hipStream_t s) {
  const int nin = a.NX * a.NY, nout = a.NP * a.NQ;
  TNX_CHECK_ARG(nout <= 64 && nin <= 64,
                "W-apply: D*d = %d / %d exceeds 64", nout, nin);
  if (a.n_outer * a.n_inner == 0) return TNX_OK;
  TNX_CHECK_ARG(a.batch >= 1 && a.batch <= 65535, "W-apply: bad batch %d", a.batch);
  const bool pair = a.n_inner >= 2;
  const int64_t per = pair ? (a.n_inner + 1) / 2 : a.n_inner, most = std::max<int64_t>(kWaColumns / per, 1);
  if (a.n_outer > most) {
    const int64_t es = a.in_f32 ? 4 : 8;
    for (int64_t o = 0; o < a.n_outer; o += most) {
      WApply part = a;
      part.in = (const char*)a.in + o * a.in_so * es;
      part.out = (char*)a.out + o * a.out_so * es;
      part.n_outer = std::min(most, a.n_outer - o);
      TNX_TRY(launch_wapply(part, s));
    }
    return TNX_OK;
  }
  const int64_t cols = a.n_outer * per;
  // one 16-column step per wave up to the 8192 waves that the chip holds;
  // one-wave blocks while those do not reach every CU
  const int64_t steps = (cols + 15) / 16;
  const int row_tiles = (nout + 15) / 16;
  const int nt = steps * a.batch * row_tiles <= 1024 ? 64 : 256;
  const int64_t blocks =
      std::min<int64_t>((steps * 64 + nt - 1) / nt, std::max<int64_t>(2048 / ((int64_t)a.batch * row_tiles), 8));
  const dim3 grid((int)blocks, a.batch, row_tiles), block(nt);
  auto go = [&](auto ks, auto pr) {
    constexpr int KS = decltype(ks)::value;
    constexpr bool PR = decltype(pr)::value;
    if (a.in_f32) hipLaunchKernelGGL((wapply_kernel<KS, PR, float>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((wapply_kernel<KS, PR, double>), grid, block, 0, s, a);
  };
  auto pick = [&](auto pr) {
    if (nin <= 12) go(std::integral_constant<int, 3>{}, pr);  // D = 5, 6
    else if (nin <= 16) go(std::integral_constant<int, 4>{}, pr);
    else if (nin <= 32) go(std::integral_constant<int, 8>{}, pr);
    else if (nin <= 52) go(std::integral_constant<int, 13>{}, pr);  // D = 25
    else go(std::integral_constant<int, 16>{}, pr);
  };
  if (pair) pick(std::true_type{});
  else pick(std::false_type{});
  TNX_LAUNCH_CHECK();
  return TNX_OK;
}

__global__ void to_f32_cvt_kernel(const double* __restrict__ x, float* __restrict__ y, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    y[i] = (float)x[i];
}

static bool valid_dims(int chil, int Dl, int Dr, int d, int chir) {
  return chil > 0 && Dl > 0 && Dr > 0 && d > 0 && chir > 0;
}

// Element size of the intermediates for a given precision.
static size_t inter_bytes(int prec) { return prec == TNX_F64 ? 8 : 4; }

// Workspace: T1, T2, and FP64 split-K partials for the last GEMM in BF16X3
// (its output, chil x d*chir, has few tiles at chil = chir and K = chil*Dl is
// long; the split rule in gemm.hip decides how many are used; FP64 and FP32
// sum parts of K inside a workgroup, but for one-column outputs):
// partial sums of up to 4 K-splits of an output of out_elems doubles
static size_t splitk_bytes(int64_t out_elems) { return (size_t)out_elems * 4 * 8; }

size_t heff1_ws_bytes_b(int chil, int Dl, int Dr, int d, int chir, int batch) {
  const size_t t1 = (size_t)chil * d * Dr * chir;
  const size_t t2 = (size_t)chil * Dl * d * chir;
  return ((t1 + t2) * 8 + splitk_bytes((int64_t)chil * d * chir)) * (size_t)batch + 512;
}

size_t heff1_ws_bytes(int chil, int Dl, int Dr, int d, int chir) {
  return heff1_ws_bytes_b(chil, Dl, Dr, d, chir, 1);
}

// y_p = H_eff(L_p, W_p, R_p) x_p for the problems p of a stack of `batch`:
// all of them (bidx null) or the `count` listed in bidx. L, W, R are
// contiguous stacks; x_p = x + p*sx, y_p = y + p*sy (sx = sy = chil*d*chir
// for contiguous stacks). One problem: batch = count = 1. x is FP64, or
// FP32 when x_f32 (a low-precision Krylov basis); y is FP64.
int heff1_matvec_b(const void* L, const double* W, const void* R, const void* x, int x_f32,
                   double* y, int chil, int Dl, int Dr, int d, int chir, int prec, int batch,
                   int count, const int* bidx, int64_t sx, int64_t sy, void* ws, size_t ws_bytes,
                   hipStream_t s, int env_f32) {
  TNX_CHECK_ARG(valid_dims(chil, Dl, Dr, d, chir), "heff1_matvec: bad dims");
  TNX_CHECK_ARG(batch >= 1 && batch <= 65535, "heff1_matvec: bad batch %d", batch);
  TNX_CHECK_ARG(count >= 1 && count <= batch && (bidx || count == batch),
                "heff1_matvec: bad count %d", count);
  TNX_CHECK_ARG(L && W && R && x && y, "heff1_matvec: null pointer");
  TNX_CHECK_ARG(prec >= TNX_F64 && prec <= TNX_BF16X3, "heff1_matvec: bad precision");
  TNX_CHECK_ARG(!env_f32 || prec != TNX_F64, "heff1_matvec: FP32 environments need a low-precision arithmetic");
  TNX_CHECK_ARG(ws && ws_bytes >= heff1_ws_bytes_b(chil, Dl, Dr, d, chir, batch),
                "heff1_matvec: workspace too small");
  const size_t eb = inter_bytes(prec);
  const DT it = prec == TNX_F64 ? DT::F64 : DT::F32;
  const int64_t nx = (int64_t)chil * d * chir;
  const int64_t nt1 = (int64_t)chil * d * Dr * chir, nt2 = (int64_t)chil * Dl * d * chir;
  char* T1 = (char*)ws;
  char* T2 = T1 + (((size_t)nt1 * batch * eb + 255) & ~(size_t)255);
  char* P = T2 + (((size_t)nt2 * batch * eb + 255) & ~(size_t)255);
  // T1[(a,k),(v,s)] = X[(a,k), r] R[r, (v,s)]
  GemmDesc g1{};
  g1.M = chil * d; g1.N = Dr * chir; g1.K = chir; g1.batch = count; g1.bidx = bidx;
  g1.A = x; g1.ta = x_f32 ? DT::F32 : DT::F64; g1.lda = chir; g1.sA = sx; g1.a_kcontig = true;
  g1.B = R; g1.tb = env_f32 ? DT::F32 : DT::F64; g1.ldb = (int64_t)Dr * chir; g1.sB = (int64_t)chir * Dr * chir; g1.b_ncontig = true;
  g1.C = T1; g1.tc = it; g1.ldc = (int64_t)Dr * chir; g1.sC = nt1;
  g1.alpha = 1.0; g1.beta = 0.0; g1.prec = (Prec)prec;
  TNX_TRY(gemm(g1, s));
  WApply wa{};
  wa.in = T1; wa.out = T2; wa.W = W; wa.in_f32 = (prec != TNX_F64);
  wa.n_outer = chil; wa.n_inner = chir;
  wa.in_so = (int64_t)d * Dr * chir; wa.in_sx = (int64_t)Dr * chir; wa.in_sy = chir;
  wa.out_so = (int64_t)Dl * d * chir; wa.out_sp = (int64_t)d * chir; wa.out_sq = chir;
  wa.NX = d; wa.NY = Dr; wa.NP = Dl; wa.NQ = d;
  wa.Dl = Dl; wa.Dr = Dr; wa.d = d; wa.mode = 0;
  wa.batch = count; wa.bidx = bidx;
  wa.in_sb = nt1; wa.out_sb = nt2; wa.W_sb = (int64_t)Dl * Dr * d * d;
  TNX_TRY(launch_wapply(wa, s));
  // y[b, (c,s)] = sum_{(a,w)} L[(a,w), b] T2[(a,w), (c,s)]
  GemmDesc g3{};
  g3.M = chil; g3.N = d * chir; g3.K = chil * Dl; g3.batch = count; g3.bidx = bidx;
  g3.A = L; g3.ta = env_f32 ? DT::F32 : DT::F64; g3.lda = chil; g3.sA = (int64_t)chil * Dl * chil; g3.a_kcontig = false;
  g3.B = T2; g3.tb = it; g3.ldb = (int64_t)d * chir; g3.sB = nt2; g3.b_ncontig = true;
  g3.C = y; g3.tc = DT::F64; g3.ldc = (int64_t)d * chir; g3.sC = sy;
  g3.alpha = 1.0; g3.beta = 0.0; g3.prec = (Prec)prec;
  g3.splitk_ws = reinterpret_cast<double*>(P);
  g3.splitk_ws_bytes = splitk_bytes(nx) * batch;
  return gemm(g3, s);
}

int heff1_matvec(const double* L, const double* W, const double* R,
                 const double* x, double* y, int chil, int Dl, int Dr, int d,
                 int chir, int prec, void* ws, size_t ws_bytes, hipStream_t s) {
  const int64_t nx = (int64_t)chil * d * chir;
  return heff1_matvec_b(L, W, R, x, 0, y, chil, Dl, Dr, d, chir, prec, 1, 1, nullptr, nx, nx, ws,
                        ws_bytes, s, 0);
}

// Two-site effective Hamiltonian (no reference function: the two-site
// solver is a stub at tnpy/finite_dmrg.py:113-114):
//   y[l',c1,c2,r'] = sum L[l,w,l'] W1[w,u,k1,c1] W2[u,v,k2,c2] R[r,v,r'] x[l,k1,k2,r]
//   T1[(l,k1,k2),(v,r')] = X[(l,k1,k2), r] R[r,(v,r')]          GEMM, K = chir
//   T2[l,k1,u,c2,r']     = sum_k2,v W2[u,v,k2,c2] T1[l,k1,k2,v,r']   W-apply
//   T3[l,w,c1,c2,r']     = sum_k1,u W1[w,u,k1,c1] T2[l,k1,u,c2,r']   W-apply
//   y[l',(c1,c2,r')]     = sum_(l,w) L[(l,w),l'] T3[(l,w),(c1,c2,r')]  GEMM, K = chil*Dl
// T3 reuses T1's memory.
size_t heff2_ws_bytes(int chil, int Dl, int Dm, int Dr, int d, int chir) {
  const size_t t1 = (size_t)chil * d * d * Dr * chir;
  const size_t t3 = (size_t)chil * Dl * d * d * chir;
  const size_t t2 = (size_t)chil * d * Dm * d * chir;
  return (std::max(t1, t3) + t2) * 8 + 256;
}

int heff2_matvec(const double* L, const double* W1, const double* W2, const double* R,
                 const void* x, int x_f32, double* y, int chil, int Dl, int Dm, int Dr, int d,
                 int chir, int prec, void* ws, size_t ws_bytes, hipStream_t s) {
  TNX_CHECK_ARG(chil > 0 && Dl > 0 && Dm > 0 && Dr > 0 && d > 0 && chir > 0, "heff2_matvec: bad dims");
  TNX_CHECK_ARG(L && W1 && W2 && R && x && y, "heff2_matvec: null pointer");
  TNX_CHECK_ARG(prec >= TNX_F64 && prec <= TNX_BF16X3, "heff2_matvec: bad precision");
  TNX_CHECK_ARG(ws && ws_bytes >= heff2_ws_bytes(chil, Dl, Dm, Dr, d, chir),
                "heff2_matvec: workspace too small");
  const size_t eb = inter_bytes(prec);
  const DT it = prec == TNX_F64 ? DT::F64 : DT::F32;
  const size_t t1 = (size_t)chil * d * d * Dr * chir;
  const size_t t3 = (size_t)chil * Dl * d * d * chir;
  char* T1 = (char*)ws;
  char* T2 = T1 + ((std::max(t1, t3) * eb + 255) & ~(size_t)255);
  char* T3 = T1;
  GemmDesc g1{};
  g1.M = chil * d * d; g1.N = Dr * chir; g1.K = chir; g1.batch = 1;
  g1.A = x; g1.ta = x_f32 ? DT::F32 : DT::F64; g1.lda = chir; g1.sA = 0; g1.a_kcontig = true;
  g1.B = R; g1.tb = DT::F64; g1.ldb = (int64_t)Dr * chir; g1.sB = 0; g1.b_ncontig = true;
  g1.C = T1; g1.tc = it; g1.ldc = (int64_t)Dr * chir; g1.sC = 0;
  g1.alpha = 1.0; g1.beta = 0.0; g1.prec = (Prec)prec;
  TNX_TRY(gemm(g1, s));
  WApply a2{};  // W2 over (k2, v) -> (u, c2), outer (l,k1), inner r'
  a2.in = T1; a2.out = T2; a2.W = W2; a2.in_f32 = (prec != TNX_F64);
  a2.n_outer = (int64_t)chil * d; a2.n_inner = chir;
  a2.in_so = (int64_t)d * Dr * chir; a2.in_sx = (int64_t)Dr * chir; a2.in_sy = chir;
  a2.out_so = (int64_t)Dm * d * chir; a2.out_sp = (int64_t)d * chir; a2.out_sq = chir;
  a2.NX = d; a2.NY = Dr; a2.NP = Dm; a2.NQ = d;
  a2.Dl = Dm; a2.Dr = Dr; a2.d = d; a2.mode = 0;
  TNX_TRY(launch_wapply(a2, s));
  WApply a1{};  // W1 over (k1, u) -> (w, c1), outer l, inner (c2, r')
  a1.in = T2; a1.out = T3; a1.W = W1; a1.in_f32 = (prec != TNX_F64);
  a1.n_outer = chil; a1.n_inner = (int64_t)d * chir;
  a1.in_so = (int64_t)d * Dm * d * chir; a1.in_sx = (int64_t)Dm * d * chir; a1.in_sy = (int64_t)d * chir;
  a1.out_so = (int64_t)Dl * d * d * chir; a1.out_sp = (int64_t)d * d * chir; a1.out_sq = (int64_t)d * chir;
  a1.NX = d; a1.NY = Dm; a1.NP = Dl; a1.NQ = d;
  a1.Dl = Dl; a1.Dr = Dm; a1.d = d; a1.mode = 0;
  TNX_TRY(launch_wapply(a1, s));
  GemmDesc g3{};
  g3.M = chil; g3.N = d * d * chir; g3.K = chil * Dl; g3.batch = 1;
  g3.A = L; g3.ta = DT::F64; g3.lda = chil; g3.sA = 0; g3.a_kcontig = false;
  g3.B = T3; g3.tb = it; g3.ldb = (int64_t)d * d * chir; g3.sB = 0; g3.b_ncontig = true;
  g3.C = y; g3.tc = DT::F64; g3.ldc = (int64_t)d * d * chir; g3.sC = 0;
  g3.alpha = 1.0; g3.beta = 0.0; g3.prec = (Prec)prec;
  return gemm(g3, s);
}

size_t env_ws_bytes_b(int chil, int Dl, int Dr, int d, int chir, int batch) {
  return (size_t)chil * d * chir * (Dl + Dr) * 8 * (size_t)batch + 512;
}

size_t env_ws_bytes(int chil, int Dl, int Dr, int d, int chir) {
  return env_ws_bytes_b(chil, Dl, Dr, d, chir, 1);
}

// Left environment update for a contiguous stack of `batch` problems
// (L, A, W, Lout each a stack of per-problem blocks).
int env_left_b(const double* L, const double* A, const double* W, double* Lout,
               int chil, int Dl, int Dr, int d, int chir, int prec, int batch, void* ws,
               size_t ws_bytes, hipStream_t s) {
  TNX_CHECK_ARG(valid_dims(chil, Dl, Dr, d, chir), "env_left: bad dims");
  TNX_CHECK_ARG(batch >= 1 && (int64_t)batch * Dr <= 65535, "env_left: bad batch %d", batch);
  TNX_CHECK_ARG(L && A && W && Lout, "env_left: null pointer");
  TNX_CHECK_ARG(prec >= TNX_F64 && prec <= TNX_BF16X3, "env_left: bad precision");
  TNX_CHECK_ARG(ws && ws_bytes >= env_ws_bytes_b(chil, Dl, Dr, d, chir, batch),
                "env_left: workspace too small");
  const size_t eb = inter_bytes(prec);
  const DT it = prec == TNX_F64 ? DT::F64 : DT::F32;
  const int64_t nA = (int64_t)chil * d * chir;
  const int64_t nT1 = (int64_t)Dl * nA, nT2 = (int64_t)Dr * nA;
  char* T1 = (char*)ws;
  char* T2 = T1 + (((size_t)nT1 * batch * eb + 255) & ~(size_t)255);
  // T1[(w,b),(k,r)] = sum_a L[a,(w,b)] A[a,(k,r)]
  GemmDesc g1{};
  g1.M = Dl * chil; g1.N = d * chir; g1.K = chil; g1.batch = batch;
  g1.A = L; g1.ta = DT::F64; g1.lda = (int64_t)Dl * chil; g1.sA = (int64_t)chil * Dl * chil; g1.a_kcontig = false;
  g1.B = A; g1.tb = DT::F64; g1.ldb = (int64_t)d * chir; g1.sB = nA; g1.b_ncontig = true;
  g1.C = T1; g1.tc = it; g1.ldc = (int64_t)d * chir; g1.sC = nT1;
  g1.alpha = 1.0; g1.beta = 0.0; g1.prec = (Prec)prec;
  TNX_TRY(gemm(g1, s));
  WApply wa{};
  wa.in = T1; wa.out = T2; wa.W = W; wa.in_f32 = (prec != TNX_F64);
  wa.n_outer = chil; wa.n_inner = chir;
  wa.in_so = (int64_t)d * chir; wa.in_sx = nA; wa.in_sy = chir;
  wa.out_so = (int64_t)d * chir; wa.out_sp = nA; wa.out_sq = chir;
  wa.NX = Dl; wa.NY = d; wa.NP = Dr; wa.NQ = d;
  wa.Dl = Dl; wa.Dr = Dr; wa.d = d; wa.mode = 1;
  wa.batch = batch; wa.in_sb = nT1; wa.out_sb = nT2; wa.W_sb = (int64_t)Dl * Dr * d * d;
  TNX_TRY(launch_wapply(wa, s));
  // L'[r, v, s] = sum_{(b,c)} T2[v][(b,c)][r] A[(b,c)][s], batched over
  // (problem, v)
  GemmDesc g3{};
  g3.M = chir; g3.N = chir; g3.K = chil * d; g3.batch = batch * Dr; g3.nb2 = Dr;
  g3.A = T2; g3.ta = it; g3.lda = chir; g3.sA = nT2; g3.sA2 = nA; g3.a_kcontig = false;
  g3.B = A; g3.tb = DT::F64; g3.ldb = chir; g3.sB = nA; g3.sB2 = 0; g3.b_ncontig = true;
  g3.C = Lout; g3.tc = DT::F64; g3.ldc = (int64_t)Dr * chir; g3.sC = (int64_t)chir * Dr * chir;
  g3.sC2 = chir;
  g3.alpha = 1.0; g3.beta = 0.0; g3.prec = (Prec)prec;
  return gemm(g3, s);
}

int env_left(const double* L, const double* A, const double* W, double* Lout,
             int chil, int Dl, int Dr, int d, int chir, int prec, void* ws,
             size_t ws_bytes, hipStream_t s) {
  return env_left_b(L, A, W, Lout, chil, Dl, Dr, d, chir, prec, 1, ws, ws_bytes, s);
}

// Right environment update for a contiguous stack of `batch` problems.
int env_right_b(const double* R, const double* A, const double* W, double* Rout,
                int chil, int Dl, int Dr, int d, int chir, int prec, int batch, void* ws,
                size_t ws_bytes, hipStream_t s) {
  TNX_CHECK_ARG(valid_dims(chil, Dl, Dr, d, chir), "env_right: bad dims");
  TNX_CHECK_ARG(batch >= 1 && batch <= 65535, "env_right: bad batch %d", batch);
  TNX_CHECK_ARG(R && A && W && Rout, "env_right: null pointer");
  TNX_CHECK_ARG(prec >= TNX_F64 && prec <= TNX_BF16X3, "env_right: bad precision");
  TNX_CHECK_ARG(ws && ws_bytes >= env_ws_bytes_b(chil, Dl, Dr, d, chir, batch),
                "env_right: workspace too small");
  const size_t eb = inter_bytes(prec);
  const DT it = prec == TNX_F64 ? DT::F64 : DT::F32;
  const int64_t nA = (int64_t)chil * d * chir;
  const int64_t nT1 = (int64_t)Dr * nA, nT2 = (int64_t)Dl * nA;
  char* T1 = (char*)ws;
  char* T2 = T1 + (((size_t)nT1 * batch * eb + 255) & ~(size_t)255);
  GemmDesc g1{};
  g1.M = chil * d; g1.N = Dr * chir; g1.K = chir; g1.batch = batch;
  g1.A = A; g1.ta = DT::F64; g1.lda = chir; g1.sA = nA; g1.a_kcontig = true;
  g1.B = R; g1.tb = DT::F64; g1.ldb = (int64_t)Dr * chir; g1.sB = (int64_t)chir * Dr * chir; g1.b_ncontig = true;
  g1.C = T1; g1.tc = it; g1.ldc = (int64_t)Dr * chir; g1.sC = nT1;
  g1.alpha = 1.0; g1.beta = 0.0; g1.prec = (Prec)prec;
  TNX_TRY(gemm(g1, s));
  WApply wa{};
  wa.in = T1; wa.out = T2; wa.W = W; wa.in_f32 = (prec != TNX_F64);
  wa.n_outer = chil; wa.n_inner = chir;
  wa.in_so = (int64_t)d * Dr * chir; wa.in_sx = (int64_t)Dr * chir; wa.in_sy = chir;
  wa.out_so = (int64_t)Dl * d * chir; wa.out_sp = (int64_t)d * chir; wa.out_sq = chir;
  wa.NX = d; wa.NY = Dr; wa.NP = Dl; wa.NQ = d;
  wa.Dl = Dl; wa.Dr = Dr; wa.d = d; wa.mode = 0;
  wa.batch = batch; wa.in_sb = nT1; wa.out_sb = nT2; wa.W_sb = (int64_t)Dl * Dr * d * d;
  TNX_TRY(launch_wapply(wa, s));
  // R'[(a,w), b] = sum_{(c,s)} T2[(a,w),(c,s)] A[b,(c,s)]
  GemmDesc g3{};
  g3.M = chil * Dl; g3.N = chil; g3.K = d * chir; g3.batch = batch;
  g3.A = T2; g3.ta = it; g3.lda = (int64_t)d * chir; g3.sA = nT2; g3.a_kcontig = true;
  g3.B = A; g3.tb = DT::F64; g3.ldb = (int64_t)d * chir; g3.sB = nA; g3.b_ncontig = false;
  g3.C = Rout; g3.tc = DT::F64; g3.ldc = chil; g3.sC = (int64_t)chil * Dl * chil;
  g3.alpha = 1.0; g3.beta = 0.0; g3.prec = (Prec)prec;
  return gemm(g3, s);
}

int env_right(const double* R, const double* A, const double* W, double* Rout,
              int chil, int Dl, int Dr, int d, int chir, int prec, void* ws,
              size_t ws_bytes, hipStream_t s) {
  return env_right_b(R, A, W, Rout, chil, Dl, Dr, d, chir, prec, 1, ws, ws_bytes, s);
}

// M[(a,k,r),(b,c,s)] = sum_{w,v} L[a,w,b] W[w,v,k,c] R[r,v,s]
// Stacks over blockIdx.y: problem p reads L, W, R, M + p * (their sizes).
__global__ void heff_dense_kernel(const double* L, const double* W, const double* R,
                                  double* M, int chil, int Dl, int Dr, int d, int chir) {
  const int64_t N = (int64_t)chil * d * chir;
  {
    const int64_t p = blockIdx.y;
    L += p * chil * Dl * chil;
    W += p * Dl * Dr * d * d;
    R += p * chir * Dr * chir;
    M += p * N * N;
  }
  for (int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; g < N * N;
       g += (int64_t)gridDim.x * blockDim.x) {
    const int64_t row = g / N, col = g % N;
    const int a = (int)(row / ((int64_t)d * chir)), k = (int)((row / chir) % d), r = (int)(row % chir);
    const int b = (int)(col / ((int64_t)d * chir)), c = (int)((col / chir) % d), s = (int)(col % chir);
    double acc = 0.0;
    for (int w = 0; w < Dl; ++w) {
      const double l = L[((int64_t)a * Dl + w) * chil + b];
      if (l == 0.0) continue;
      for (int v = 0; v < Dr; ++v)
        acc += l * W[((w * Dr + v) * d + k) * d + c] * R[((int64_t)r * Dr + v) * chir + s];
    }
    M[g] = acc;
  }
}

int heff1_dense_b(const double* L, const double* W, const double* R, double* M,
                  int chil, int Dl, int Dr, int d, int chir, int batch, hipStream_t s) {
  TNX_CHECK_ARG(valid_dims(chil, Dl, Dr, d, chir), "heff1_dense: bad dims");
  TNX_CHECK_ARG(batch >= 1 && batch <= 65535, "heff1_dense: bad batch %d", batch);
  TNX_CHECK_ARG(L && W && R && M, "heff1_dense: null pointer");
  const int64_t N = (int64_t)chil * d * chir;
  TNX_CHECK_ARG(N <= 8192, "heff1_dense: dimension %lld too large for a dense H_eff", (long long)N);
  const int blocks = (int)std::min<int64_t>((N * N + 255) / 256, std::max(4096 / batch, 16));
  hipLaunchKernelGGL(heff_dense_kernel, dim3(blocks, batch), dim3(256), 0, s, L, W, R, M, chil,
                     Dl, Dr, d, chir);
  TNX_LAUNCH_CHECK();
  return TNX_OK;
}

int heff1_dense(const double* L, const double* W, const double* R, double* M,
                int chil, int Dl, int Dr, int d, int chir, hipStream_t s) {
  return heff1_dense_b(L, W, R, M, chil, Dl, Dr, d, chir, 1, s);
}

// ---- elementwise helpers ---------------------------------------------------
__global__ void transpose_kernel(const double* in, double* out, int rows, int cols) {
  __shared__ double tile[32][33];
  const int bx = blockIdx.x * 32, by = blockIdx.y * 32;
  for (int j = threadIdx.y; j < 32; j += 8) {
    const int r = by + j, c = bx + threadIdx.x;
    if (r < rows && c < cols) tile[j][threadIdx.x] = in[(int64_t)r * cols + c];
  }
  __syncthreads();
  for (int j = threadIdx.y; j < 32; j += 8) {
    const int c = bx + j, r = by + threadIdx.x;
    if (r < rows && c < cols) out[(int64_t)c * rows + r] = tile[threadIdx.x][j];
  }
}

int transpose_f64(const double* in, double* out, int rows, int cols, hipStream_t s) {
  if (rows == 0 || cols == 0) return TNX_OK;
  TNX_CHECK_ARG(in && out && in != out, "transpose: bad pointers");
  TNX_CHECK_ARG(ceil_div(rows, 32) <= 65535, "transpose: too many rows");
  dim3 grid(ceil_div(cols, 32), ceil_div(rows, 32));
  hipLaunchKernelGGL(transpose_kernel, grid, dim3(32, 8), 0, s, in, out, rows, cols);
  TNX_LAUNCH_CHECK();
  return TNX_OK;
}

__global__ void copy_kernel(const double* in, double* out, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    out[i] = in[i];
}
__global__ void fill_kernel(double* out, int64_t n, double v) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    out[i] = v;
}

int copy_f64(const double* in, double* out, int64_t n, hipStream_t s) {
  if (n <= 0) return TNX_OK;
  const int blocks = (int)std::min<int64_t>((n + 255) / 256, 8192);
  hipLaunchKernelGGL(copy_kernel, dim3(blocks), dim3(256), 0, s, in, out, n);
  TNX_LAUNCH_CHECK();
  return TNX_OK;
}

int fill_f64(double* out, int64_t n, double v, hipStream_t s) {
  if (n <= 0) return TNX_OK;
  const int blocks = (int)std::min<int64_t>((n + 255) / 256, 8192);
  hipLaunchKernelGGL(fill_kernel, dim3(blocks), dim3(256), 0, s, out, n, v);
  TNX_LAUNCH_CHECK();
  return TNX_OK;
}

}  // namespace tnx

// ---- C-ABI -----------------------------------------------------------------
extern "C" {

size_t tnx_heff1_workspace_bytes(int chil, int Dl, int Dr, int d, int chir) {
  return tnx::heff1_ws_bytes(chil, Dl, Dr, d, chir);
}

int tnx_heff1_matvec(const double* L, const double* W, const double* R,
                     const double* x, double* y, int chil, int Dl, int Dr,
                     int d, int chir, int precision, void* ws, size_t ws_bytes,
                     tnx_stream_t stream) {
  return tnx::heff1_matvec(L, W, R, x, y, chil, Dl, Dr, d, chir, precision, ws,
                           ws_bytes, (hipStream_t)stream);
}

int tnx_heff1_dense(const double* L, const double* W, const double* R,
                    double* M, int chil, int Dl, int Dr, int d, int chir,
                    tnx_stream_t stream) {
  return tnx::heff1_dense(L, W, R, M, chil, Dl, Dr, d, chir, (hipStream_t)stream);
}

size_t tnx_env_workspace_bytes(int chil, int Dl, int Dr, int d, int chir) {
  return tnx::env_ws_bytes(chil, Dl, Dr, d, chir);
}

size_t tnx_heff2_workspace_bytes(int chil, int Dl, int Dm, int Dr, int d, int chir) {
  return tnx::heff2_ws_bytes(chil, Dl, Dm, Dr, d, chir);
}

int tnx_heff2_matvec(const double* L, const double* W1, const double* W2, const double* R,
                     const double* x, double* y, int chil, int Dl, int Dm, int Dr, int d,
                     int chir, int precision, void* ws, size_t ws_bytes, tnx_stream_t stream) {
  return tnx::heff2_matvec(L, W1, W2, R, x, 0, y, chil, Dl, Dm, Dr, d, chir, precision, ws,
                           ws_bytes, (hipStream_t)stream);
}

int tnx_env_left(const double* L, const double* A, const double* W,
                 double* Lout, int chil, int Dl, int Dr, int d, int chir,
                 int precision, void* ws, size_t ws_bytes, tnx_stream_t stream) {
  return tnx::env_left(L, A, W, Lout, chil, Dl, Dr, d, chir, precision, ws,
                       ws_bytes, (hipStream_t)stream);
}

int tnx_env_right(const double* R, const double* A, const double* W,
                  double* Rout, int chil, int Dl, int Dr, int d, int chir,
                  int precision, void* ws, size_t ws_bytes, tnx_stream_t stream) {
  return tnx::env_right(R, A, W, Rout, chil, Dl, Dr, d, chir, precision, ws,
                        ws_bytes, (hipStream_t)stream);
}

size_t tnx_heff1_batched_workspace_bytes(int chil, int Dl, int Dr, int d, int chir, int batch) {
  return tnx::heff1_ws_bytes_b(chil, Dl, Dr, d, chir, batch);
}

int tnx_heff1_matvec_ex(const void* L, const double* W, const void* R, const void* x, double* y,
                        int chil, int Dl, int Dr, int d, int chir, int env_f32, int x_f32,
                        int precision, void* ws, size_t ws_bytes, tnx_stream_t stream) {
  const int64_t nx = (int64_t)chil * d * chir;
  return tnx::heff1_matvec_b(L, W, R, x, x_f32, y, chil, Dl, Dr, d, chir, precision, 1, 1, nullptr,
                             nx, nx, ws, ws_bytes, (hipStream_t)stream, env_f32);
}

int tnx_to_f32(const double* x, float* y, int64_t n, tnx_stream_t stream) {
  TNX_CHECK_ARG(x && y && n >= 0, "tnx_to_f32: bad arguments");
  if (n == 0) return TNX_OK;
  const int nb = (int)std::min<int64_t>((n + 255) / 256, 8192);
  hipLaunchKernelGGL(tnx::to_f32_cvt_kernel, dim3(nb), dim3(256), 0, (hipStream_t)stream, x, y, n);
  TNX_LAUNCH_CHECK();
  return TNX_OK;
}

int tnx_heff1_matvec_batched(const double* L, const double* W, const double* R,
                             const double* x, double* y, int chil, int Dl, int Dr,
                             int d, int chir, int batch, int precision, void* ws,
                             size_t ws_bytes, tnx_stream_t stream) {
  const int64_t nx = (int64_t)chil * d * chir;
  return tnx::heff1_matvec_b(L, W, R, x, 0, y, chil, Dl, Dr, d, chir, precision, batch, batch,
                             nullptr, nx, nx, ws, ws_bytes, (hipStream_t)stream, 0);
}

int tnx_heff1_dense_batched(const double* L, const double* W, const double* R,
                            double* M, int chil, int Dl, int Dr, int d, int chir,
                            int batch, tnx_stream_t stream) {
  return tnx::heff1_dense_b(L, W, R, M, chil, Dl, Dr, d, chir, batch, (hipStream_t)stream);
}

size_t tnx_env_batched_workspace_bytes(int chil, int Dl, int Dr, int d, int chir, int batch) {
  return tnx::env_ws_bytes_b(chil, Dl, Dr, d, chir, batch);
}

int tnx_env_left_batched(const double* L, const double* A, const double* W,
                         double* Lout, int chil, int Dl, int Dr, int d, int chir,
                         int batch, int precision, void* ws, size_t ws_bytes,
                         tnx_stream_t stream) {
  return tnx::env_left_b(L, A, W, Lout, chil, Dl, Dr, d, chir, precision, batch, ws, ws_bytes,
                         (hipStream_t)stream);
}

int tnx_env_right_batched(const double* R, const double* A, const double* W,
                          double* Rout, int chil, int Dl, int Dr, int d, int chir,
                          int batch, int precision, void* ws, size_t ws_bytes,
                          tnx_stream_t stream) {
  return tnx::env_right_b(R, A, W, Rout, chil, Dl, Dr, d, chir, precision, batch, ws, ws_bytes,
                          (hipStream_t)stream);
}

}  // extern "C"
