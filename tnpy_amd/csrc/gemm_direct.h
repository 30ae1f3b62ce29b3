// Strided, batched GEMM for the FP64 and FP32 arithmetics: every wave loads
// its MFMA operands from memory straight into registers and runs on its own
// (no LDS tiles, no barriers in the k loop).
//
// Why no LDS. The FP64 (FP32) matrix instruction v_mfma_*_16x16x4 keeps a
// SIMD busy for 64 (32) cycles per 16 x 16 x 4 product, so a wave with a
// 64 x 80 tile asks for 144 values per 4 k's in 1280 (640) cycles: about
// 14 B/clk per CU, far below what the L1 and L2 deliver. What bounded the
// LDS form was the k-tile boundary, where all waves of a CU converted,
// stored and met at a barrier (MFMA busy 64..76 %), and at small sizes the
// same boundary's exposed load latency. Here the loads of the next groups of
// 8 k's are in flight under the MFMAs of the current one (PD groups ahead)
// and the waves drift freely. Measured on MI355X, LDS form -> this one:
// 2048 x 5120 x 1024 FP64 330 -> 296 us (72.5 TF/s, 0.92 of peak), FP32 with
// float operands 192 -> 169 us (127 TF/s); 1024 x 2048 x 5120 FP64 379 ->
// 300 us; 600 x 1536 x 256 35 -> 14 us, 60 x 120 x 300 12.8 -> 4.2 us.
//
// Tiles. A wave owns TM x TN accumulator tiles of 16 x 16; a block is
// WM x WN of them times WK parts of K. WK > 1 cuts K over waves of one
// block and sums the parts in LDS at the end (recursive halving, so every
// wave finishes and stores a quarter of the tile): an output with few tiles
// and a long K fills the chip without partial sums in memory.
//
// Operand order. In a group of 8 k's lane (i = lane % 16, g = lane / 16)
// feeds k = 2 g + s to MFMA step s = 0, 1 (any order of k will do that both
// operands share), and an even number of 16-wide fragments is taken in
// interleaved pairs, index 32 p + 2 i + f for fragment 2 p + f. So every
// load is a pair of neighbours along the operand's contiguous dimension
// (16 bytes of doubles, 8 of floats), whichever dimension that is, and the
// output is stored as pairs too. Pairs need only the element's own alignment
// (dword-aligned multi-dword accesses), so odd leading dimensions and bases
// take the same path.
//
// Edges. Indices past the matrix are clamped to its last element (their
// output rows and columns are not stored); the k's of a last partial group
// past the end are zero in both operands, so no value outside the matrix is
// ever multiplied into the result.
#pragma once

#include "gemm_kernel.h"

namespace tnx {

typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
// pair stores at the element's own alignment
typedef double f64x2_u __attribute__((ext_vector_type(2), aligned(8)));
typedef float f32x2_u __attribute__((ext_vector_type(2), aligned(4)));

// Two neighbouring elements, and one, as the raw registers of a load.
template <typename E> struct Raw2;
template <> struct Raw2<double> { using pair = u32x4; using one = u32x2; };
template <> struct Raw2<float> { using pair = u32x2; using one = unsigned; };

template <typename E>
__device__ __forceinline__ typename Raw2<E>::pair load_pair(__amdgpu_buffer_rsrc_t r, unsigned off, int so) {
  if constexpr (sizeof(E) == 8) return __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, so, 0);
  else return __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, so, 0);
}

template <typename E>
__device__ __forceinline__ typename Raw2<E>::one load_one(__amdgpu_buffer_rsrc_t r, unsigned off, int so) {
  if constexpr (sizeof(E) == 8) return __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, so, 0);
  else return __builtin_amdgcn_raw_buffer_load_b32(r, (int)off, so, 0);
}

template <typename E>
__device__ __forceinline__ E pair_elem(const typename Raw2<E>::pair& v, int j) {
  if constexpr (sizeof(E) == 8) {
    const unsigned long long lo = v[2 * j], hi = v[2 * j + 1];
    return __longlong_as_double((long long)((hi << 32) | lo));
  } else {
    return __uint_as_float(v[j]);
  }
}

template <typename E>
__device__ __forceinline__ E one_elem(const typename Raw2<E>::one& v) {
  if constexpr (sizeof(E) == 8) {
    const unsigned long long lo = v[0], hi = v[1];
    return __longlong_as_double((long long)((hi << 32) | lo));
  } else {
    return __uint_as_float(v);
  }
}

template <typename E>
__device__ __forceinline__ typename Raw2<E>::pair make_pair_raw(E x, E y) {
  if constexpr (sizeof(E) == 8) {
    const unsigned long long a = (unsigned long long)__double_as_longlong(x);
    const unsigned long long b = (unsigned long long)__double_as_longlong(y);
    return u32x4{(unsigned)a, (unsigned)(a >> 32), (unsigned)b, (unsigned)(b >> 32)};
  } else {
    return u32x2{__float_as_uint(x), __float_as_uint(y)};
  }
}

// A wave-uniform pointer, made so for the compiler: a buffer base that it
// keeps in vector registers turns each load into a loop over lanes.
__device__ __forceinline__ const char* uniform_ptr(const char* p) {
  const unsigned long long u = (unsigned long long)p;
  const unsigned lo = __builtin_amdgcn_readfirstlane((int)(u & 0xffffffffull));
  const unsigned hi = __builtin_amdgcn_readfirstlane((int)(u >> 32));
  return (const char*)(((unsigned long long)hi << 32) | lo);
}

// Index of fragment t, lane index i, inside a wave's T fragments.
template <int T>
__device__ __forceinline__ int frag_index(int t, int i) {
  return t < 2 * (T / 2) ? 32 * (t >> 1) + 2 * i + (t & 1) : 16 * t + i;
}

// T fragments of one operand along its row (A) or column (B) dimension.
// KC: the k dimension is the contiguous one (a pair is k, k + 1 of one
// index); else the row / column dimension is (a pair is two indices of one
// k; an odd last fragment is loaded singly).
template <int T, bool KC, typename E>
struct GemmOperand {
  static constexpr int NP = T / 2;
  static constexpr bool ODD = (T & 1) != 0;
  struct Group {
    typename Raw2<E>::pair p[KC ? T : (NP ? 2 * NP : 1)];
    typename Raw2<E>::one o[(!KC && ODD) ? 2 : 1];
  };
  unsigned off[KC ? T : NP + 1];  // byte offsets from `base`
  bool last[NP + 1];              // !KC: this pair was moved back by one, its index is the second value
  const char* base;               // the group's k 0, advanced by `adv` bytes per group
  int64_t adv;
  int krow;  // !KC: bytes from one k to the next

  // x0: the wave's first index, X: the dimension's extent (x0 < X; !KC: X >=
  // 2), k0: the first k of the wave's part, (i, g): the lane.
  __device__ __forceinline__ void init(const char* P, int64_t ld, int x0, int X, int k0, int i, int g) {
    constexpr int64_t es = sizeof(E);
    if constexpr (KC) {
      base = uniform_ptr(P + ((int64_t)x0 * ld + k0) * es);
      adv = 8 * es;
      krow = 0;
#pragma unroll
      for (int t = 0; t < T; ++t) {
        const int x = min(frag_index<T>(t, i), X - 1 - x0);
        off[t] = (unsigned)(((int64_t)x * ld + 2 * g) * es);
      }
    } else {
      const int xb = min(x0, X - 2);
      base = uniform_ptr(P + ((int64_t)k0 * ld + xb) * es);
      adv = 8 * ld * es;
      krow = (int)(ld * es);
#pragma unroll
      for (int p = 0; p < NP; ++p) {
        const int x = x0 + 32 * p + 2 * i;
        last[p] = x == X - 1;
        off[p] = (unsigned)((2 * (int64_t)g * ld + (min(x, X - 2) - xb)) * es);
      }
      const int x = x0 + 16 * (T - 1) + i;
      off[NP] = (unsigned)((2 * (int64_t)g * ld + (min(x, X - 1) - xb)) * es);
    }
  }

  __device__ __forceinline__ void load(Group& r, const char* at) const {
    const __amdgpu_buffer_rsrc_t rs = gemm_rsrc(at);
    if constexpr (KC) {
#pragma unroll
      for (int t = 0; t < T; ++t) r.p[t] = load_pair<E>(rs, off[t], 0);
    } else {
#pragma unroll
      for (int s = 0; s < 2; ++s) {
#pragma unroll
        for (int p = 0; p < NP; ++p) r.p[s * NP + p] = load_pair<E>(rs, off[p], s * krow);
        if constexpr (ODD) r.o[s] = load_one<E>(rs, off[NP], s * krow);
      }
    }
  }

  // The last, partial group: `left` (1..7) k's remain; klim: K minus the
  // group's first k, with K >= 2 when KC.
  __device__ __forceinline__ void load_tail(Group& r, const char* at, int left, int klim, int g) const {
    constexpr int es = sizeof(E);
    if constexpr (KC) {
      // one k left of K >= 2: the group starts past k = 0, so a pair can
      // start one k before it
      const int back = klim < 2 ? 1 : 0;
      const __amdgpu_buffer_rsrc_t rs = gemm_rsrc(at - back * es);
      const int k = 2 * g;
      const int d = (min(k, klim - 2) + back - k) * es;
#pragma unroll
      for (int t = 0; t < T; ++t) {
        const typename Raw2<E>::pair v = load_pair<E>(rs, off[t] + (unsigned)d, 0);
        E x = pair_elem<E>(v, 0), y = pair_elem<E>(v, 1);
        if (k == klim - 1) x = y;
        if (k >= left) x = 0;
        if (k + 1 >= left) y = 0;
        r.p[t] = make_pair_raw<E>(x, y);
      }
    } else {
      const __amdgpu_buffer_rsrc_t rs = gemm_rsrc(at);
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        // a lane whose k is past the end re-reads the group's first k
        const bool in = 2 * g + s < left;
        const unsigned d = (unsigned)(in ? s * krow : -2 * g * krow);
#pragma unroll
        for (int p = 0; p < NP; ++p) {
          const typename Raw2<E>::pair v = load_pair<E>(rs, off[p] + d, 0);
          r.p[s * NP + p] = in ? v : typename Raw2<E>::pair{};
        }
        if constexpr (ODD) {
          const typename Raw2<E>::one v = load_one<E>(rs, off[NP] + d, 0);
          r.o[s] = in ? v : typename Raw2<E>::one{};
        }
      }
    }
  }

  template <typename CT>
  __device__ __forceinline__ CT value(const Group& r, int t, int s) const {
    if constexpr (KC) {
      return (CT)pair_elem<E>(r.p[t], s);
    } else {
      if (t >= 2 * NP) return (CT)one_elem<E>(r.o[s]);
      const E y = pair_elem<E>(r.p[s * NP + t / 2], 1);
      if (t & 1) return (CT)y;
      const E x = pair_elem<E>(r.p[s * NP + t / 2], 0);
      return (CT)(last[t / 2] ? y : x);
    }
  }
};

template <int PREC, int TM, int TN, int WM, int WN, int WK, int PD, int OCC, bool A_K, bool B_N,
          typename TA, typename TB>
__global__ __launch_bounds__(64 * WM * WN * WK, OCC) void gemm_direct_kernel(GemmArgs g) {
  if (g.gate && *g.gate == 0) return;
  using acc_t = typename PT<PREC>::acc_t;
  using CT = typename PT<PREC>::lds_t;
  using OA = GemmOperand<TM, A_K, TA>;
  using OB = GemmOperand<TN, !B_N, TB>;
  static_assert(WK == 1 || (WK == 4 && (TN % 2 == 0 || TM * TN == 1)), "K parts: 1 or 4, an even split of the units");
  constexpr int RING = PD + 1;
  // units of the finished tile: (i, column pair, v, f), or v for one tile
  constexpr int NU = TM * TN * 4;
  constexpr int MU = WK == 1 ? NU : NU / 4;  // units a wave stores
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15, lg = lane >> 4;
  const int wn = wave % WN, wm = (wave / WN) % WM, wk = wave / (WN * WM);

  const int bat = g.bidx ? g.bidx[blockIdx.y] : (int)blockIdx.y;
  const int tile = gemm_tile_of(g);
  const int m0 = (tile / g.tiles_n) * (16 * TM * WM) + wm * (16 * TM);
  const int n0 = (tile % g.tiles_n) * (16 * TN * WN) + wn * (16 * TN);
  const int kc = WK > 1 ? ((g.K + WK - 1) / WK + 7) / 8 * 8 : g.K;
  const int k0 = min(wk * kc, g.K), k1 = min(g.K, k0 + kc);
  const int b1 = bat / g.nb2, b2 = bat % g.nb2;
  const char* Ab = (const char*)g.A + ((int64_t)b1 * g.sA + (int64_t)b2 * g.sA2) * (int64_t)sizeof(TA);
  const char* Bb = (const char*)g.B + ((int64_t)b1 * g.sB + (int64_t)b2 * g.sB2) * (int64_t)sizeof(TB);
  char* Cb = (char*)g.C + ((int64_t)b1 * g.sC + (int64_t)b2 * g.sC2) * (g.tc == 0 ? 8 : 4);
  const bool live = m0 < g.M && n0 < g.N;

  // rows and columns of the accumulators: element v of MFMA tile (i, j)
  // sits at MFMA row lg + 4 v (FP64) or 4 lg + v (FP32), column li
  auto row_of = [&](int i, int v) { return m0 + frag_index<TM>(i, PREC == 0 ? lg + 4 * v : lg * 4 + v); };
  auto load_c = [&](int m, int n) -> double {
    if (!(m < g.M && n < g.N)) return 0.0;
    const int64_t o = (int64_t)m * g.ldc + n;
    return g.tc == 0 ? reinterpret_cast<const double*>(Cb)[o] : (double)reinterpret_cast<const float*>(Cb)[o];
  };
  // unit u -> (tile row i, tile column j, element v): per tile row first the
  // column pairs as (pair, v, f), then an odd last column as (v)
  constexpr int PU = 8 * (TN / 2);
  auto unit_i = [](int u) { return u / (4 * TN); };
  auto unit_j = [](int u) {
    const int e = u % (4 * TN);
    return e < PU ? 2 * (e / 8) + (e & 1) : TN - 1;
  };
  auto unit_v = [](int u) {
    const int e = u % (4 * TN);
    return e < PU ? (e / 2) & 3 : e - PU;
  };
  auto unit_paired = [](int u) { return u % (4 * TN) < PU; };
  // Few units per wave: their old C values are loaded before the k loop, so
  // with beta != 0 the two reads overlap (the rank-32 and rank-128 updates
  // of the blocked QR have only a few groups of k).
  constexpr bool PRE_C = MU <= 16;
  const bool pre_c = PRE_C && g.beta != 0.0 && live;
  double cpre[PRE_C ? MU : 1];
  auto with_part = [&](auto f) {
    if constexpr (WK == 1) {
      f(std::integral_constant<int, 0>{});
    } else {
      if (wk == 0) f(std::integral_constant<int, 0>{});
      else if (wk == 1) f(std::integral_constant<int, 1>{});
      else if (wk == 2) f(std::integral_constant<int, 2>{});
      else f(std::integral_constant<int, 3>{});
    }
  };
  if constexpr (PRE_C) {
    if (pre_c) {
      with_part([&](auto part) {
        constexpr int U0 = decltype(part)::value * MU;
#pragma unroll
        for (int q = 0; q < MU; ++q)
          cpre[q] = load_c(row_of(unit_i(U0 + q), unit_v(U0 + q)), n0 + frag_index<TN>(unit_j(U0 + q), li));
      });
    }
  }

  acc_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = acc_t{0, 0, 0, 0};

  if (live && k0 < k1) {
    OA oa;
    OB ob;
    oa.init(Ab, g.lda, m0, g.M, k0, li, lg);
    ob.init(Bb, g.ldb, n0, g.N, k0, li, lg);
    const int ng = (k1 - k0) / 8, left = (k1 - k0) % 8;
    auto compute = [&](const typename OA::Group& ra, const typename OB::Group& rb) {
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        CT a[TM], b[TN];
#pragma unroll
        for (int i = 0; i < TM; ++i) a[i] = oa.template value<CT>(ra, i, s);
#pragma unroll
        for (int j = 0; j < TN; ++j) b[j] = ob.template value<CT>(rb, j, s);
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j) {
            if constexpr (PREC == 0)
              acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i], b[j], acc[i][j], 0, 0, 0);
            else
              acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], b[j], acc[i][j], 0, 0, 0);
          }
      }
    };
    if (ng > 0) {
      // ring of PD groups in flight and one in use; past the last group the
      // loads repeat it (unused), so the loop has no branches
      typename OA::Group ra[RING];
      typename OB::Group rb[RING];
      const char* pa = oa.base;
      const char* pb = ob.base;
      int at = 0;
      auto next = [&](int slot) {
        oa.load(ra[slot], pa);
        ob.load(rb[slot], pb);
        if (at + 1 < ng) {
          ++at;
          pa += oa.adv;
          pb += ob.adv;
        }
      };
#pragma unroll
      for (int u = 0; u < PD; ++u) next(u);
      int it = 0;
      for (; it + RING <= ng; it += RING) {
#pragma unroll
        for (int u = 0; u < RING; ++u) {
          next((u + PD) % RING);
          compute(ra[u], rb[u]);
        }
      }
      // fewer than RING groups remain, loaded into slots 0, 1, ..
#pragma unroll
      for (int u = 0; u < PD; ++u)
        if (it + u < ng) compute(ra[u], rb[u]);
    }
    if (left) {
      typename OA::Group ta;
      typename OB::Group tb;
      const int klim = g.K - (k0 + ng * 8);
      oa.load_tail(ta, oa.base + (int64_t)ng * oa.adv, left, klim, lg);
      ob.load_tail(tb, ob.base + (int64_t)ng * ob.adv, left, klim, lg);
      compute(ta, tb);
    }
  }

  auto unit = [&](int u) -> double { return (double)acc[unit_i(u)][unit_j(u)][unit_v(u)]; };
  double val[MU];
  if constexpr (WK == 1) {
#pragma unroll
    for (int u = 0; u < NU; ++u) val[u] = unit(u);
  } else {
    // Sum of the four K parts by recursive halving: parts 2 apart exchange
    // halves of the units, then neighbours exchange quarters. FP32 parts are
    // summed in FP64.
    constexpr int HU = NU / 2;
    __shared__ CT xh[WM * WN * 4 * HU * 64];
    __shared__ double xq[PREC == 0 ? 1 : WM * WN * 4 * MU * 64];
    double half[HU];
    const int wt = wm * WN + wn;
    CT* mine = xh + (size_t)(wt * 4 + wk) * HU * 64 + lane;
    const CT* other = xh + (size_t)(wt * 4 + (wk ^ 2)) * HU * 64 + lane;
    // keep the upper half of the units (parts 2, 3) or the lower (0, 1)
    auto send_half = [&](auto hi) {
      constexpr int SEND = HU - decltype(hi)::value * HU;
#pragma unroll
      for (int u = 0; u < HU; ++u) mine[u * 64] = acc[unit_i(SEND + u)][unit_j(SEND + u)][unit_v(SEND + u)];
    };
    auto take_half = [&](auto hi) {
      constexpr int KEEP = decltype(hi)::value * HU;
#pragma unroll
      for (int u = 0; u < HU; ++u) half[u] = unit(KEEP + u) + (double)other[u * 64];
    };
    using Lo = std::integral_constant<int, 0>;
    using Hi = std::integral_constant<int, 1>;
    if (wk & 2) send_half(Hi{}); else send_half(Lo{});
    __syncthreads();
    if (wk & 2) take_half(Hi{}); else take_half(Lo{});
    // FP64 reuses the first exchange's LDS, once every wave has read it
    double* mq;
    const double* oq;
    if constexpr (PREC == 0) {
      __syncthreads();
      mq = xh + (size_t)(wt * 4 + wk) * MU * 64 + lane;
      oq = xh + (size_t)(wt * 4 + (wk ^ 1)) * MU * 64 + lane;
    } else {
      mq = xq + (size_t)(wt * 4 + wk) * MU * 64 + lane;
      oq = xq + (size_t)(wt * 4 + (wk ^ 1)) * MU * 64 + lane;
    }
    // (values, not elements, in the selects: a select between array elements
    // would put the array in scratch memory)
    const bool hi = wk & 1;
#pragma unroll
    for (int u = 0; u < MU; ++u) {
      const double a = half[u], b = half[MU + u];
      mq[u * 64] = hi ? a : b;
      val[u] = hi ? b : a;
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < MU; ++u) val[u] += oq[u * 64];
  }
  if (!live) return;

  with_part([&](auto part) {
    constexpr int U0 = decltype(part)::value * MU;
    // 16 units at a time: with beta != 0 their old C values (unless loaded
    // before) all come before their stores
    constexpr int CH = MU < 16 ? MU : (MU % 16 == 0 ? 16 : 20);
#pragma unroll
    for (int c0 = 0; c0 < MU; c0 += CH) {
      double out[CH];
#pragma unroll
      for (int q = 0; q < CH; ++q) {
        const int u = U0 + c0 + q;
        out[q] = g.alpha * val[c0 + q];
        if (g.beta != 0.0) {
          double old;
          if constexpr (PRE_C) old = cpre[c0 + q];
          else old = load_c(row_of(unit_i(u), unit_v(u)), n0 + frag_index<TN>(unit_j(u), li));
          out[q] += g.beta * old;
        }
      }
#pragma unroll
      for (int q = 0; q < CH; ++q) {
        const int u = U0 + c0 + q;
        if (unit_paired(u) && (u & 1)) continue;  // stored with its first
        const int m = row_of(unit_i(u), unit_v(u)), n = n0 + frag_index<TN>(unit_j(u), li);
        if (m >= g.M || n >= g.N) continue;
        const bool two = unit_paired(u) && n + 1 < g.N;
        const int64_t o = (int64_t)m * g.ldc + n;
        const double x0 = out[q], x1 = out[q + 1 < CH ? q + 1 : q];
        if (g.tc == 0) {
          double* c = reinterpret_cast<double*>(Cb) + o;
          if (two) *reinterpret_cast<f64x2_u*>(c) = f64x2_u{x0, x1};
          else *c = x0;
        } else {
          float* c = reinterpret_cast<float*>(Cb) + o;
          if (two) *reinterpret_cast<f32x2_u*>(c) = f32x2_u{(float)x0, (float)x1};
          else *c = (float)x0;
        }
      }
    }
  });
}

// ---------------------------------------------------------------------------
// Wave-tile configurations and the rule that picks one.
// ---------------------------------------------------------------------------
struct DirectCfg { int tm, tn, wm, wn, wk, pd, occ; };

template <int PREC> struct DirectCfgs;
template <> struct DirectCfgs<0> {
  static constexpr int n = 8;
  static constexpr DirectCfg c[n] = {{4, 5, 4, 1, 1, 1, 2}, {2, 4, 2, 2, 1, 2, 2}, {4, 4, 1, 1, 4, 1, 2},
                                     {2, 4, 1, 1, 4, 2, 2}, {2, 2, 2, 2, 1, 3, 2}, {2, 2, 1, 1, 4, 3, 2},
                                     {1, 1, 1, 1, 4, 4, 2}, {1, 1, 2, 2, 1, 4, 2}};
};
template <> struct DirectCfgs<1> {
  static constexpr int n = 8;
  static constexpr DirectCfg c[n] = {{4, 5, 4, 1, 1, 2, 2}, {8, 5, 2, 2, 1, 1, 1}, {4, 4, 1, 1, 4, 2, 2},
                                     {2, 4, 1, 1, 4, 3, 2}, {2, 2, 2, 2, 1, 4, 2}, {2, 2, 1, 1, 4, 4, 2},
                                     {1, 1, 1, 1, 4, 4, 2}, {1, 1, 2, 2, 1, 4, 2}};
};

// True where the kernel applies: FP64 or FP32 arithmetic, a pair to load
// along each operand's contiguous dimension, and offsets inside a wave's tile
// within a buffer's 2 GiB range.
bool gemm_direct_ok(const GemmDesc& d);

void gemm_direct_f64(const GemmDesc& d, const GemmArgs& g, hipStream_t s);
void gemm_direct_f32(const GemmDesc& d, const GemmArgs& g, hipStream_t s);

// The rule: the configuration with the least modelled time in cycles of the
// busiest CU. Per group of 8 k's a wave needs 2 TM TN matrix instructions
// (64 or 32 cycles each) and (TM + TN) operand loads per lane, which the CU's
// four SIMDs share; below that lies a latency per group, hidden by the PD
// groups in flight; then the epilogue, the K-part sum and a start-up cost per
// block. The constants were fitted to launches of 112 (FP64) and 80 (FP32)
// shapes of the contractions here at bond dimensions 16..1024, batches of
// chains and QR / SVD block products among them; the picked configuration is
// within 2.5 % of the best one measured on the mean, 25 % at worst.
template <int PREC>
inline int gemm_direct_pick(const GemmDesc& d) {
  using L = DirectCfgs<PREC>;
  constexpr double mfma = PREC == 0 ? 64.0 : 32.0;
  constexpr double ld = PREC == 0 ? 48.0 : 24.5;
  constexpr double lat = PREC == 0 ? 630.0 : 2930.0;
  constexpr double epi = PREC == 0 ? 290.0 : 23.0;
  constexpr double red = PREC == 0 ? 800.0 : 400.0;
  constexpr double blk = PREC == 0 ? 320.0 : 177.0;
  int best = 0;
  double best_t = 1e300;
  for (int i = 0; i < L::n; ++i) {
    const DirectCfg& c = L::c[i];
    // one wave per SIMD (8 x 5): considered after the rule, below
    if (c.occ == 1) continue;
    const double blocks = std::ceil((double)d.M / (16 * c.tm * c.wm)) *
                          std::ceil((double)d.N / (16 * c.tn * c.wn)) * (double)d.batch;
    const double per_cu = std::ceil(blocks / 256.0);
    const double waves = std::ceil(per_cu * c.wm * c.wn * c.wk / 4.0);  // per SIMD
    const double groups = std::ceil(std::ceil((double)d.K / c.wk) / 8.0);
    const double work = waves * groups * std::max(2.0 * c.tm * c.tn * mfma, 4.0 * (c.tm + c.tn) * ld);
    // the FP64 fit hides a group's latency per wave, the FP32 one per pair
    const double wait = groups * lat / c.pd * (PREC == 0 ? waves : std::max(1.0, waves / 2.0));
    const double t = std::max(work, wait) + lat + epi * c.tm * c.tn * waves +
                     (c.wk > 1 ? red * c.tm * c.tn : 0.0) + blk * per_cu;
    if (t < best_t) { best_t = t; best = i; }
  }
  if (PREC == 1 && best == 0 && d.ta == DT::F32 && d.tb == DT::F32) {
    // 8 x 5 tiles (one wave per SIMD, 30 % fewer operand bytes per product)
    // where they take no more rounds than the 4 x 5 ones: 190 -> 169 us at
    // 2048 x 5120 x 1024. With operands in FP64 the conversions of a lone
    // wave are exposed (388 -> 567 us at 4096 x 5120 x 1024).
    auto rounds = [&](const DirectCfg& c) {
      return std::ceil(std::ceil((double)d.M / (16 * c.tm * c.wm)) * std::ceil((double)d.N / (16 * c.tn * c.wn)) *
                       (double)d.batch / 256.0) * c.tm * c.tn * c.wm * c.wn;
    };
    if (rounds(L::c[1]) <= rounds(L::c[0])) best = 1;
  }
  return best;
}

template <int PREC, int I, typename TA, typename TB>
static void gemm_direct_launch(const GemmDesc& d, const GemmArgs& g0, hipStream_t s) {
  constexpr DirectCfg c = DirectCfgs<PREC>::c[I];
  GemmArgs g = g0;
  constexpr int BM = 16 * c.tm * c.wm, BN = 16 * c.tn * c.wn;
  g.tiles_n = ceil_div(d.N, BN);
  const int tiles_m = ceil_div(d.M, BM);
  g.group_m = gemm_group_m(tiles_m, g.tiles_n, BM, BN, d.batch);
  const dim3 grid(tiles_m * g.tiles_n, d.batch), block(64 * c.wm * c.wn * c.wk);
#define TNX_DIRECT(AK, BN_)                                                                     \
  hipLaunchKernelGGL((gemm_direct_kernel<PREC, c.tm, c.tn, c.wm, c.wn, c.wk, c.pd, c.occ, AK,   \
                                         BN_, TA, TB>), grid, block, 0, s, g)
  if (d.a_kcontig && d.b_ncontig) TNX_DIRECT(true, true);
  else if (d.a_kcontig) TNX_DIRECT(true, false);
  else if (d.b_ncontig) TNX_DIRECT(false, true);
  else TNX_DIRECT(false, false);
#undef TNX_DIRECT
}

template <int PREC, typename TA, typename TB>
static void gemm_direct_run(const GemmDesc& d, const GemmArgs& g, hipStream_t s) {
  switch (gemm_direct_pick<PREC>(d)) {
    case 0: return gemm_direct_launch<PREC, 0, TA, TB>(d, g, s);
    case 1: return gemm_direct_launch<PREC, 1, TA, TB>(d, g, s);
    case 2: return gemm_direct_launch<PREC, 2, TA, TB>(d, g, s);
    case 3: return gemm_direct_launch<PREC, 3, TA, TB>(d, g, s);
    case 4: return gemm_direct_launch<PREC, 4, TA, TB>(d, g, s);
    case 5: return gemm_direct_launch<PREC, 5, TA, TB>(d, g, s);
    case 6: return gemm_direct_launch<PREC, 6, TA, TB>(d, g, s);
    default: return gemm_direct_launch<PREC, 7, TA, TB>(d, g, s);
  }
}

}  // namespace tnx
