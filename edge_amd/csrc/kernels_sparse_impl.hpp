// Element kernels that walk the non-zeros of the reference-element matrices
// on the vector ALU (elastic, geometry-built solvers).
//
// In the hierarchical orthogonal basis 82 % of the stiffness and 58 % of the
// flux matrices' entries are zero, and which ones is known when the kernels
// are compiled.  A lane holds one column, one (element, run) pair, and a
// workgroup of W waves works on 64 columns (64 / R elements).  Each wave owns
// a share of the modes of every quantity (Deal): it keeps their DOFs in
// registers, so everything that mixes quantities at one mode is lane-local,
// and it computes the outputs of its modes of every matrix product.  The
// inputs of a product pass through LDS: the owners publish a column
// [mode][64] and every wave reads the modes its outputs need.  Each non-zero
// is one fused multiply-add with the entry as a literal (FP64: from two scalar
// moves that serve two columns): no operand loads, no padding, no work on
// zeros.  The waves run different code (their own
// non-zeros), the partition of the modes balances it.
//
// Instead of the 9 x 9 star matrices and flux solvers the kernels use what
// they are made of (phys): with G_ki the gradient d v_i / d x_k, the stresses
// change by -(lambda tr G delta + mu (G + G^T)), and the velocities by
// -1 / rho times the stress divergence.  A face's flux depends on each side
// only through the vector w of its waves travelling towards the face,
//   w = (zs v - T) / (zs1 + zs2) + n [(zp v_n - T_n) / (zp1 + zp2) -
//       (zs v_n - T_n) / (zs1 + zs2)],   T = sigma n, n outward,
// and seen from its own side that is the same vector for the element's own
// flux and for its neighbour's (the normal and the traction both change
// sign), so one projection per face serves the local and the neighbour step
// (on a free surface the mirrored state gives the element's own w again).
// The neighbour takes it to its own face coordinates with the orientation
// map R_v (ec64_pack.hpp).
//
// What bounds it: vector-ALU issue (about 40,000 instructions per tile and
// 64 columns at order 5 against 131,000 cycles of padded MFMA tiles; the
// vector ALUs are busy 55 % of the time) and the memory latency that two (order
// 5) or three workgroups per CU leave exposed.  A load behind output stores waits
// for all of them, so constants come first, the projections leave last and
// tInt is written while they are formed.
// Eight waves of half the modes (128 registers) took 10.9 ms per order-5 step
// against 7.7 for four.
// Measured against the kernels that did the same before (ms per step): order
// 5, 196,608 tets, 16 runs with sources and receivers 8.60 -> 6.4 (MFMA, runs
// on N); one run 1.19 -> 0.53 (MFMA, 16 elements on N); order 5, 36,720 tets,
// 8 runs 6.81 -> 0.69 (generic); order 4 with a fault, 331,776 tets, 16 runs
// 10.3 -> 5.1; FP64 order 4, 12,870 tets, 16 runs 5.66 -> 0.64
// (generic); order 5, 10,368 tets, 8 runs 5.85 -> 0.73 (generic).
//
// Operations (src/impl/seismic/solvers/AderDg.hpp:362-533, :553-722):
//   local: CK time prediction (TimePredVanilla.hpp:200-306), volume integral
//          (VolIntVanilla.hpp:189-241), local surface integral
//          (SurfIntVanilla.hpp:212-262);
//   neigh: neighbouring surface integral (SurfIntVanilla.hpp:274-357).
#pragma once

#include <hip/hip_runtime.h>

#include <utility>

#include "dg_masks.hpp"
#include "kernels_sparse.hpp"

#pragma clang fp contract(off)

namespace edge {
namespace {

// Lambdas over register arrays: inlined before anything else happens to them,
// so that the arrays stay registers whatever branch they are passed into.
#define EDGE_INLINE __attribute__((always_inline))

constexpr int kCols = 64;  // columns (lanes) per workgroup tile
// Waves per workgroup: four, in FP64 at orders 4 and 5 eight (the DOFs, the
// time integral and the update of a quarter of the modes need more than the
// 256 registers that two waves per SIMD leave a lane).
#ifndef EDGE_SP_WAVES
#define EDGE_SP_WAVES 4
#endif
constexpr int kWaves = EDGE_SP_WAVES;
// The order of a product's sums over the input modes: in FP32 the high ones
// first.  A smooth column's are small, so the partial sums and their roundings
// stay small until the low modes come (error against 64 bits after 4 steps of
// smooth waves, 3,024 tets, order 5, 16 runs: 4.16e-7 -> 3.45e-7).  FP64 keeps
// the low ones first: its error is the same either way (order 4: 5.88e-15).
#ifndef EDGE_SP_LOW_FIRST
#define EDGE_SP_LOW_FIRST 0
#endif
constexpr bool kLowFirst = EDGE_SP_LOW_FIRST;
constexpr int nth(int i, int n) { return kLowFirst ? i : n - 1 - i; }

// The order in which the modes and face modes are dealt to the waves: wave w
// of W owns the modes at positions j W + w, and a column's LDS row is the
// position.  Found by balancing the waves' non-zeros per product; the modes
// of every lower order come first (a derivative's outputs are a prefix).
template <int O>
struct Deal;
template <>
struct Deal<2> {
  static constexpr int mode[4] = {0, 2, 1, 3};
  static constexpr int face[3] = {0, 2, 1};
};
template <>
struct Deal<3> {
  static constexpr int mode[10] = {0, 1, 3, 2, 6, 5, 9, 8, 4, 7};
  static constexpr int face[6] = {2, 3, 0, 1, 5, 4};
};
#if EDGE_SP_WAVES == 8
template <>
struct Deal<4> {
  static constexpr int mode[20] = {0, 2, 3, 1, 4, 5, 6, 8, 9, 7, 12, 17, 19, 16, 18, 13, 10, 15, 14, 11};
  static constexpr int face[10] = {6, 9, 4, 5, 1, 0, 2, 3, 7, 8};
};
template <>
struct Deal<5> {
  static constexpr int mode[35] = {0,  2,  3,  1,  5,  7,  6,  4,  9,  8,  14, 17, 11, 12, 13, 16, 19, 15,
                                   10, 18, 24, 34, 26, 31, 21, 25, 28, 32, 33, 23, 27, 22, 20, 30, 29};
  static constexpr int face[15] = {10, 0, 6, 8, 12, 11, 1, 3, 2, 14, 9, 7, 5, 4, 13};
};
#else
template <>
struct Deal<4> {
  static constexpr int mode[20] = {0, 3, 2, 1, 9, 4, 5, 6, 8, 7, 19, 12, 11, 16, 14, 17, 10, 15, 13, 18};
  static constexpr int face[10] = {7, 8, 0, 2, 9, 6, 5, 3, 1, 4};
};
template <>
struct Deal<5> {
  static constexpr int mode[35] = {0,  3,  2,  1,  8,  4,  5,  7,  9,  6,  14, 19, 13, 15, 11, 10, 16, 18,
                                   17, 12, 30, 34, 29, 33, 21, 25, 32, 31, 20, 23, 27, 24, 28, 26, 22};
  static constexpr int face[15] = {5, 8, 4, 9, 12, 13, 14, 0, 11, 7, 10, 2, 1, 6, 3};
};
#endif

template <int O>
struct Dim {
  static constexpr int N = n_modes(O), NF = n_face_modes(O);
  static constexpr int W = kWaves;
  static constexpr int own(int nn) { return (nn + W - 1) / W; }  // most modes below nn of a wave
  static constexpr int M = own(N), MF = own(NF);
  // mode / face mode at position j of wave w, -1: none
  static constexpr int mode(int w, int j) { return j * W + w < N ? Deal<O>::mode[j * W + w] : -1; }
  static constexpr int face(int w, int j) { return j * W + w < NF ? Deal<O>::face[j * W + w] : -1; }
  static constexpr int row(int k) {
    for (int p = 0; p < N; p++)
      if (Deal<O>::mode[p] == k) return p;
    return -1;
  }
  static constexpr int face_row(int k) {
    for (int p = 0; p < NF; p++)
      if (Deal<O>::face[p] == k) return p;
    return -1;
  }
  static constexpr int WROWS = 12 * NF;    // all four faces' w
  static constexpr int CROWS = 4 * N;      // four columns of the CK's first stage
  static constexpr int LROWS = 2 * CROWS > WROWS + 3 * N ? 2 * CROWS : WROWS + 3 * N;
};

template <int V>
using Int = std::integral_constant<int, V>;

template <typename F, int... I>
__device__ __forceinline__ void each(F f, std::integer_sequence<int, I...>) {
  (f(Int<I>{}), ...);
}

// The matrices: Out[n] += at(k, n) In[k].
template <int O, int D>
struct Ck {
  static constexpr double at(int k, int n) { return -masks::Mats<O>::stiffT[(D * n_modes(O) + k) * n_modes(O) + n]; }
};
template <int O, int D>
struct Vol {
  static constexpr double at(int k, int n) { return masks::Mats<O>::stiffV[(D * n_modes(O) + k) * n_modes(O) + n]; }
};
template <int O, int F>
struct Prj {
  static constexpr double at(int k, int f) {
    return masks::Mats<O>::fluxL[(F * n_modes(O) + k) * n_face_modes(O) + f];
  }
};
template <int O, int F>
struct Lift {
  static constexpr double at(int f, int n) {
    return masks::Mats<O>::fluxT[(F * n_face_modes(O) + f) * n_modes(O) + n];
  }
};

// Every sum is spelled out (no contraction chosen per context), so that the
// kernels that share this code agree bit for bit.
__device__ __forceinline__ float fma_(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double fma_(double a, double b, double c) { return __builtin_fma(a, b, c); }
template <typename T>
__device__ __forceinline__ T dot3(T a0, T b0, T a1, T b1, T a2, T b2) {
  return fma_(a2, b2, fma_(a1, b1, a0 * b0));
}

// No input of output N that comes before K in the order of the sums (below NK)
// has a non-zero entry.
template <typename Mat, int K, int N, int NK>
constexpr bool starts() {
  for (int k = kLowFirst ? 0 : K + 1; N >= 0 && k < (kLowFirst ? K : NK); k++)
    if (Mat::at(k, N) != 0.0) return false;
  return true;
}

// A matrix entry as an operand: a literal in FP32; in FP64 a pair of scalar
// registers written where it is used (left to the compiler, hundreds of them
// stay live across a product and spill).
template <typename T>
__device__ __forceinline__ T entry(double v) {
  if constexpr (sizeof(T) == 8) {
    const long long b = __builtin_bit_cast(long long, v);
    int lo, hi;
    asm volatile("s_mov_b32 %0, %1" : "=s"(lo) : "i"((int)b));
    asm volatile("s_mov_b32 %0, %1" : "=s"(hi) : "i"((int)(b >> 32)));
    return __builtin_bit_cast(double, (long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
  } else {
    return T(v);
  }
}

// out[j] += M[k][n_j] x over wave W's outputs n_j < nn with a non-zero entry
// (out[j] = for the first one).
template <typename Mat, int K, int N, bool FIRST, typename T>
__device__ __forceinline__ void term(T x, T& out) {
  if constexpr (N >= 0) {
    constexpr double v = Mat::at(K, N);
    if constexpr (v != 0.0) {
      const T c = entry<T>(v);
      out = FIRST ? c * x : fma_(c, x, out);
    }
  }
}
template <int O, int NN, int W, int J>
constexpr int mode_of() {
  return Dim<O>::mode(W, J) < NN ? Dim<O>::mode(W, J) : -1;
}
template <int O, int NN, int W, typename Mat, int K, int NK, typename T, int... J>
__device__ __forceinline__ void terms(T x, T* out, std::integer_sequence<int, J...>) {
  (term<Mat, K, mode_of<O, NN, W, J>(), starts<Mat, K, mode_of<O, NN, W, J>(), NK>()>(x, out[J]), ...);
}
template <int O, int W, typename Mat, int K, int NK, typename T, int... J>
__device__ __forceinline__ void face_terms(T x, T* out, std::integer_sequence<int, J...>) {
  (term<Mat, K, Dim<O>::face(W, J), starts<Mat, K, Dim<O>::face(W, J), NK>()>(x, out[J]), ...);
}
// Input K of two columns with matrix D of three: p += M x and, summed over
// the matrices, v += M y, each entry used for both.
template <int O, int NN, int W, typename M0, typename M1, typename M2, int K, int NK, int D, int J, typename T>
__device__ __forceinline__ void pair_term(T x, T y, T& p, T& v) {
  constexpr int N = mode_of<O, NN, W, J>();
  if constexpr (N >= 0) {
    using M = std::conditional_t<D == 0, M0, std::conditional_t<D == 1, M1, M2>>;
    constexpr double m = M::at(K, N);
    if constexpr (m != 0.0) {
      constexpr bool s = starts<M0, K, N, NK>() && starts<M1, K, N, NK>() && starts<M2, K, N, NK>();
      constexpr bool n0 = M0::at(K, N) != 0.0, n1 = M1::at(K, N) != 0.0;
      constexpr bool first = s && (D < 1 || !n0) && (D < 2 || !n1);
      const T c = entry<T>(m);
      p = starts<M, K, N, NK>() ? c * x : fma_(c, x, p);
      v = first ? c * y : fma_(c, y, v);
    }
  }
}
template <int O, int NN, int W, typename M0, typename M1, typename M2, int K, int NK, int D, typename T, int... J>
__device__ __forceinline__ void pair_terms(T x, T y, T* p, T* v, std::integer_sequence<int, J...>) {
  (pair_term<O, NN, W, M0, M1, M2, K, NK, D, J>(x, y, p[J], v[J]), ...);
}

template <int O, bool CK, int D>
using Stiff = std::conditional_t<CK, Ck<O, D>, Vol<O, D>>;

// The LDS reads of a product in the order of its sums, each with the columns
// and inputs it feeds.  A wave takes them in groups of G: the next group is
// requested before the present one's multiply-adds, which keeps the LDS
// latency behind 15 to 30 of them (left to itself the compiler reads just
// ahead of each use).
struct Read {
  int col, k;
};
template <int MAX>
struct Reads {
  int n = 0;
  Read r[MAX] = {};
  constexpr void add(int col, int k) {
    r[n].col = col;
    r[n].k = k;
    n++;
  }
};

// One published component: column 0 (the raw velocity) times all three
// stiffness matrices into p[d], columns 1 + d times matrix d, summed, into v;
// outputs of wave V below NN, inputs below NK.
template <int O, bool CK, int NK, int NN, int V>
struct StiffReads {
  // (order 5, FP32: groups of 8 instead of 16, order 5, 16 runs, 24,576 tets, 4 steps 3.03 -> 2.96 ms)
  static constexpr int J = Dim<O>::own(NN), G = O == 5 ? 8 : 64 / kWaves, ROWS = NK;
  template <int D>
  static constexpr bool feeds(int k) {
    for (int j = 0; j < J; j++) {
      const int n = Dim<O>::mode(V, j);
      if (n >= 0 && n < NN && Stiff<O, CK, D>::at(k, n) != 0.0) return true;
    }
    return false;
  }
  // per input the four columns, one after the other
  static constexpr Reads<4 * NK> list() {
    Reads<4 * NK> l;
    for (int i = 0; i < NK; i++) {
      const int k = nth(i, NK);
      if (feeds<0>(k) || feeds<1>(k) || feeds<2>(k))
        for (int c = 0; c < 4; c++) l.add(c, k);
    }
    return l;
  }
  static constexpr int row(int k) { return Dim<O>::row(k); }
  template <int COL, int K, typename T>
  static __device__ __forceinline__ void use(const T* x, T (&p)[3][J], T (&v)[J]) {
    if constexpr (COL == 0) {
      using M0 = Stiff<O, CK, 0>;
      using M1 = Stiff<O, CK, 1>;
      using M2 = Stiff<O, CK, 2>;
      using JS = std::make_integer_sequence<int, J>;
      pair_terms<O, NN, V, M0, M1, M2, K, NK, 0>(x[0], x[1], p[0], v, JS{});
      pair_terms<O, NN, V, M0, M1, M2, K, NK, 1>(x[0], x[2], p[1], v, JS{});
      pair_terms<O, NN, V, M0, M1, M2, K, NK, 2>(x[0], x[3], p[2], v, JS{});
    }
  }
};

// One column of a face's w in the element's modes to the wave's face modes.
template <int O, int F, int V>
struct ProjectReads {
  static constexpr int N = Dim<O>::N, J = Dim<O>::MF, G = 48 / kWaves, ROWS = 0;
  static constexpr Reads<N> list() {
    Reads<N> l;
    for (int i = 0; i < N; i++) {
      const int k = nth(i, N);
      bool on = false;
      for (int j = 0; j < J; j++) {
        const int n = Dim<O>::face(V, j);
        on = on || (n >= 0 && Prj<O, F>::at(k, n) != 0.0);
      }
      if (on) l.add(0, k);
    }
    return l;
  }
  static constexpr int row(int k) { return Dim<O>::row(k); }
  template <int COL, int K, typename T>
  static __device__ __forceinline__ void use(const T* x, T (&u)[J]) {
    face_terms<O, V, Prj<O, F>, K, N>(x[0], u, std::make_integer_sequence<int, J>{});
  }
};

// One face column to the wave's modes.
template <int O, int F, int V>
struct LiftReads {
  static constexpr int NF = Dim<O>::NF, J = Dim<O>::M, G = 64 / kWaves, ROWS = 0;
  static constexpr Reads<NF> list() {
    Reads<NF> l;
    for (int i = 0; i < NF; i++) {
      const int k = nth(i, NF);
      bool on = false;
      for (int j = 0; j < J; j++) {
        const int n = Dim<O>::mode(V, j);
        on = on || (n >= 0 && Lift<O, F>::at(k, n) != 0.0);
      }
      if (on) l.add(0, k);
    }
    return l;
  }
  static constexpr int row(int k) { return Dim<O>::face_row(k); }
  template <int COL, int K, typename T>
  static __device__ __forceinline__ void use(const T* x, T (&u)[J]) {
    terms<O, Dim<O>::N, V, Lift<O, F>, K, NF>(x[0], u, std::make_integer_sequence<int, J>{});
  }
};

// Group C of the reads of S into x / its multiply-adds.
template <typename S, int C, typename T, int... I>
__device__ __forceinline__ void fetch(const T* l, T (&x)[S::G], std::integer_sequence<int, I...>) {
  constexpr auto list = S::list();
  (
      [&]() EDGE_INLINE {
        constexpr int at = C * S::G + I;
        if constexpr (at < list.n) {
          constexpr int off = (list.r[at].col * S::ROWS + S::row(list.r[at].k)) * kCols;
          x[I] = l[off];
        }
      }(),
      ...);
}
template <typename S, int C, typename T, int... I, typename... Out>
__device__ __forceinline__ void consume(const T (&x)[S::G], std::integer_sequence<int, I...>, Out&... out) {
  constexpr auto list = S::list();
  (
      [&]() EDGE_INLINE {
        constexpr int at = C * S::G + I;
        if constexpr (at < list.n) {
          constexpr int col = list.r[at].col, k = list.r[at].k;
          S::template use<col, k>(x + I, out...);
        }
      }(),
      ...);
}
template <typename S, int C, typename T, typename... Out>
__device__ __forceinline__ void stream(const T* l, const T (&x)[S::G], Out&... out) {
  constexpr int n = S::list().n;
  using GS = std::make_integer_sequence<int, S::G>;
  T next[S::G];
  if constexpr ((C + 1) * S::G < n) fetch<S, C + 1>(l, next, GS{});
  __builtin_amdgcn_sched_barrier(0);
  consume<S, C>(x, GS{}, out...);
  __builtin_amdgcn_sched_barrier(0);
  if constexpr ((C + 1) * S::G < n) stream<S, C + 1>(l, next, out...);
}
// out += S (columns at the lane's first row l)
template <typename S, typename T, typename... Out>
__device__ __forceinline__ void product(const T* l, Out&... out) {
  if constexpr (S::list().n > 0) {
    T x[S::G];
    fetch<S, 0>(l, x, std::make_integer_sequence<int, S::G>{});
    stream<S, 0>(l, x, out...);
  }
}

// The calling wave's code (w is uniform across the wave).  The (empty, but
// different) last statements keep the branches from being merged over the
// registers they update, which would put those into memory.
template <int W, int I = 0, typename F>
__device__ __forceinline__ void by_wave(int w, F f) {
  if constexpr (I + 1 < W) {
    if (w == I) {
      f(Int<I>{});
      asm volatile("; wave %0" ::"n"(I));
    } else {
      by_wave<W, I + 1>(w, f);
    }
  } else {
    f(Int<I>{});
    asm volatile("; wave %0" ::"n"(I));
  }
}
template <typename F>
__device__ __forceinline__ void by_axis(int i, F f) {
  if (i == 0) {
    f(Int<0>{});
    asm volatile("; axis 0");
  } else if (i == 1) {
    f(Int<1>{});
    asm volatile("; axis 1");
  } else {
    f(Int<2>{});
    asm volatile("; axis 2");
  }
}

// Stress component (i, k) of the symmetric tensor in the DOFs' order
// (sxx, syy, szz, sxy, syz, sxz).
__host__ __device__ constexpr int voigt(int i, int k) { return i == k ? i : (i + k == 1 ? 3 : i + k == 3 ? 4 : 5); }

// Buffer access: a wave-uniform base and offset (scalar registers) plus the
// lane's byte offset (one vector register for all of a tile's accesses; plain
// pointers had the compiler keep dozens of 64-bit addresses live).  Lanes at
// kSkip or past the buffer read zeros and store nothing.
constexpr unsigned kSkip = 0x80000000u;
typedef uint32_t u2 __attribute__((ext_vector_type(2)));
template <typename T>
struct Buf {
  __amdgpu_buffer_rsrc_t r;
  __device__ __forceinline__ Buf(const T* base, unsigned values)
      : r(__builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(base), 0, values * sizeof(T), 0x00027000)) {}
  __device__ __forceinline__ T load(unsigned lane, unsigned uniform) const {
    if constexpr (sizeof(T) == 4)
      return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(r, lane, uniform, 0));
    else
      return __builtin_bit_cast(T, (u2)__builtin_amdgcn_raw_buffer_load_b64(r, lane, uniform, 0));
  }
  __device__ __forceinline__ void store(T v, unsigned lane, unsigned uniform) const {
    if constexpr (sizeof(T) == 4)
      __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), r, lane, uniform, 0);
    else
      __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u2, v), r, lane, uniform, 0);
  }
};

template <typename T>
struct Mat4 {  // -(lambda + 2 mu), -lambda, -mu, -1 / rho
  T lam2, lam, mu, irho;
};

// y_sigma += -(lambda G_ii delta + mu (G_ki + G_ik)) for the gradients
// G_k = G_ki of the velocity component i, over m modes.
template <int I, int M, int MY, typename T>
__device__ __forceinline__ void add_stress(T (&y)[9][MY], const T (&g)[3][M], const Mat4<T>& c) {
#pragma unroll
  for (int k = 0; k < 3; k++)
#pragma unroll
    for (int j = 0; j < M; j++) {
      if (k == I) {
        y[0][j] = fma_(I == 0 ? c.lam2 : c.lam, g[k][j], y[0][j]);
        y[1][j] = fma_(I == 1 ? c.lam2 : c.lam, g[k][j], y[1][j]);
        y[2][j] = fma_(I == 2 ? c.lam2 : c.lam, g[k][j], y[2][j]);
      } else {
        y[voigt(I, k)][j] = fma_(c.mu, g[k][j], y[voigt(I, k)][j]);
      }
    }
}

// One tile of 64 columns, as seen by a lane of wave w.
template <typename T, int O, int R>
struct Tile {
  using D = Dim<O>;
  static constexpr int N = D::N, SZ = 9 * N * R, M = D::M, W = D::W;
  T* lds;
  int w, lane;
  int64_t el;      // the lane's element (the last one's for lanes past the range)
  int64_t first;   // first element of the tile
  int n_el;        // elements of the tile inside the range
  bool valid;
  const T* cst;    // the element's constants: in LDS (fused runs) ...
  Buf<T> ph;       // ... or in memory
  unsigned ph_off;
  // The inverse Jacobian and the material: in registers, at order 5 with
  // fused runs read from LDS where they are used (the registers are full).
  static constexpr bool HELD = R == 1 || O < 5 || sizeof(T) == 8;
  T ji1[3][3];
  Mat4<T> mat1;
  // FP32: where registers hold it, what a step adds to the DOFs is summed first,
  // so that fewer roundings are of the DOFs' size:
  //   SUM: all of a side's update (with several runs it takes a wave per SIMD:
  //   order 3, 16 runs, 48,000 tets, 4 steps 1172 -> 1274 us);
  //   VEL: the velocities that a component lifts, one rounding instead of four
  //   (all components' in the neighbour step: order 5, 16 runs, 24,576 tets, 4
  //   steps 2.96 -> 3.17 ms).
  // Error against 64 bits after 4 steps of smooth waves, 3,024 tets, without
  // and with: order 3, one run 1.9e-7 -> 1.5e-7, order 4, one run 2.6e-7 ->
  // 2.3e-7.
  static constexpr bool F32 = sizeof(T) == 4, SUM = F32 && R == 1 && O <= 3;
  static constexpr bool VEL = F32 && !SUM && (O <= 3 || (O == 4 && R == 1));
  // The time step is multiplied into what the volume integral and the
  // projections take and give, or (SCALED) into their constants, whose
  // rounding then is the same in every mode.  Order 4, 16 runs, 24,576 tets, 4
  // steps: 1.42 ms with scaled constants, 1.30 without, error 2.9e-7 -> 2.7e-7;
  // order 5, 16 runs: 2.99 and 3.09 ms, 3.45e-7 and 3.30e-7; FP64, order 4, 16
  // runs, 12,870 tets, 2 steps: 1.27 and 1.28 ms, the same error.
  static constexpr bool SCALED = R > 1 && (O == 5 || !F32);

  static constexpr int PB = phys::block(R);
  __device__ __forceinline__ Tile(const T* phys_el, int64_t first_)
      : first(first_), ph(phys_el + first_ / PB * (phys::kSize * PB), R == 1 ? 2 * phys::kSize * PB : 0) {}
  // With fused runs the few elements' constants are copied to LDS before
  // anything else: a load of them between the output stores would wait for
  // the stores (the counter runs in order; it took half of the time).
  __device__ __forceinline__ T c(int k) const {
    if constexpr (R == 1)
      return ph.load(ph_off, k * PB * (unsigned)sizeof(T));
    else
      return cst[k];
  }
  __device__ __forceinline__ T jinv(int k, int d) const {
    if constexpr (HELD)
      return ji1[k][d];
    else
      return cst[phys::kJinv + 3 * k + d];
  }
  __device__ __forceinline__ Mat4<T> mat() const {
    if constexpr (HELD)
      return mat1;
    else
      return {cst[phys::kLam2], cst[phys::kLam], cst[phys::kMu], cst[phys::kIrho]};
  }
  // byte offset of the lane's column in a DOF array of the tile
  __device__ __forceinline__ unsigned column() const {
    return (unsigned)((el - first) * SZ + lane % R) * (unsigned)sizeof(T);
  }
  __device__ __forceinline__ T face(int f, int k) const { return c(phys::kFace + phys::kPerFace * f + k); }
  // the wave's modes, six bits each (where it has fewer than M, its first
  // mode again: those registers hold copies that nothing reads)
  uint64_t modes;
  static constexpr uint64_t pack(int v) {
    uint64_t b = 0;
    for (int j = 0; j < M; j++) b |= (uint64_t)D::mode(v, D::mode(v, j) < 0 ? 0 : j) << (6 * j);
    return b;
  }
  __device__ __forceinline__ int mode(int j) const { return (int)(modes >> (6 * j)) & 63; }
  // position j of the wave is below nn (known at compile time but for the last)
  __device__ __forceinline__ bool has(int j, int nn) const { return (j + 1) * W <= nn || j * W + w < nn; }

  // the wave's modes of a DOF array (zeros past the last one)
  __device__ __forceinline__ void load(const T* __restrict__ a, T (&x)[9][M]) {
    if constexpr (R == 1) {
      // one element is contiguous: three quantities of the 64 elements at a
      // time pass through LDS (rows of 65 columns: no bank conflicts); every
      // load is requested before the first is waited for
      constexpr int PER = (kCols * 3 * N + 64 * W - 1) / (64 * W);
      T v[3][PER];
      const Buf<T> src(a + first * SZ, n_el * SZ);
#pragma unroll
      for (int qb = 0; qb < 3; qb++)
#pragma unroll
        for (int i = 0; i < PER; i++) {
          const unsigned k = threadIdx.x + i * 64 * W;
          v[qb][i] = src.load((k / (3 * N) * SZ + k % (3 * N)) * (unsigned)sizeof(T), qb * 3 * N * (unsigned)sizeof(T));
        }
#pragma unroll
      for (int qb = 0; qb < 3; qb++) {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < PER; i++) {
          const unsigned k = threadIdx.x + i * 64 * W;
          if (k < kCols * 3 * N) lds[k % (3 * N) * (kCols + 1) + k / (3 * N)] = v[qb][i];
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 3; q++)
#pragma unroll
          for (int j = 0; j < M; j++) x[3 * qb + q][j] = lds[(q * N + mode(j)) * (kCols + 1) + lane];
      }
      __syncthreads();
    } else {
      const Buf<T> src(a + first * SZ, n_el * SZ);
      const unsigned off = column();
#pragma unroll
      for (int j = 0; j < M; j++)
#pragma unroll
        for (int q = 0; q < 9; q++) x[q][j] = src.load(off, (unsigned)((mode(j) + q * N) * R * (int)sizeof(T)));
    }
  }

  // stores the wave's modes (fused runs: of the lanes with `on`), SC: times sca
  template <bool SC = false>
  __device__ __forceinline__ void store(T* __restrict__ a, const T (&x)[9][M], bool on, T sca = T(1)) {
    if constexpr (R == 1) {
#pragma unroll
      for (int qb = 0; qb < 9; qb += 3) {
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 3; q++)
#pragma unroll
          for (int j = 0; j < M; j++) {
            if (has(j, N)) lds[(q * N + mode(j)) * (kCols + 1) + lane] = SC ? sca * x[qb + q][j] : x[qb + q][j];
          }
        constexpr int PER = (kCols * 3 * N + 64 * W - 1) / (64 * W);
        const Buf<T> dst(a + first * SZ, n_el * SZ);
        __syncthreads();
#pragma unroll
        for (int i = 0; i < PER; i++) {
          const unsigned k = threadIdx.x + i * 64 * W;
          const bool in = k < kCols * 3 * N;
          dst.store(in ? lds[k % (3 * N) * (kCols + 1) + k / (3 * N)] : T(0),
                    in ? (k / (3 * N) * SZ + k % (3 * N)) * (unsigned)sizeof(T) : kSkip, qb * N * (unsigned)sizeof(T));
        }
      }
    } else {
      const Buf<T> dst(a + first * SZ, n_el * SZ);
      const unsigned off = on ? column() : kSkip;
#pragma unroll
      for (int j = 0; j < M; j++) {
        if (!has(j, N)) continue;
#pragma unroll
        for (int q = 0; q < 9; q++)
          dst.store(SC ? sca * x[q][j] : x[q][j], off, (unsigned)((mode(j) + q * N) * R * (int)sizeof(T)));
      }
    }
  }

  // Publishes velocity component I and the three star-combined rows
  // sum_k j[k][d] sigma_Ik of the modes below NK.
  template <int I, int NK, int MK>
  __device__ __forceinline__ void publish(T* l, const T (&x)[9][MK], const T (&j3)[3][3], Int<I>) const {
#pragma unroll
    for (int j = 0; j < MK; j++) {
      if (!has(j, NK)) continue;
      T* o = l + j * W * kCols;
      o[0] = x[6 + I][j];
#pragma unroll
      for (int d = 0; d < 3; d++)
        o[(d + 1) * NK * kCols] =
            dot3(j3[0][d], x[voigt(I, 0)][j], j3[1][d], x[voigt(I, 1)][j], j3[2][d], x[voigt(I, 2)][j]);
    }
  }

  // Component i of S (stiffness products of x), x on the modes below NK,
  // outputs below NN: the gradients g of velocity component i and the stress
  // divergence v of its row; buf holds the published columns.
  template <bool CK, int NK, int NN, bool SC = false, int MK, int MN>
  __device__ __forceinline__ void component(int i, const T (&x)[9][MK], T* buf, T (&g)[3][MN], T (&v)[MN],
                                            T sca = T(1)) {
    // (opaque to the optimiser: the combined rows of every component would
    // otherwise be formed ahead of the loop and spilled)
    T j3[3][3];
    auto load_j = [&]() EDGE_INLINE {
#pragma unroll
    for (int k = 0; k < 3; k++)
#pragma unroll
      for (int d = 0; d < 3; d++) {
        j3[k][d] = SC ? sca * jinv(k, d) : jinv(k, d);
        asm volatile("" : "+v"(j3[k][d]));
      }
    };
    load_j();
    by_axis(i, [&](auto I) EDGE_INLINE { publish<decltype(I)::value, NK>(buf + w * kCols + lane, x, j3, I); });
    __syncthreads();
    T p[3][MN];
#pragma unroll
    for (int j = 0; j < MN; j++) p[0][j] = p[1][j] = p[2][j] = v[j] = T(0);
    by_wave<W>(w, [&](auto V) EDGE_INLINE {
      product<StiffReads<O, CK, NK, NN, decltype(V)::value>>(buf + lane, p, v);
    });
    if constexpr (!HELD) load_j();
#pragma unroll
    for (int j = 0; j < MN; j++)
#pragma unroll
      for (int k = 0; k < 3; k++) g[k][j] = dot3(j3[k][0], p[0][j], j3[k][1], p[1][j], j3[k][2], p[2][j]);
  }

  // y += S (stiffness products of x): per velocity component one published
  // set of columns; buffers alternate (step counts them), so one barrier per
  // component is enough.
  template <int NK, int NN, int MX, int MN>
  __device__ __forceinline__ void stiffness(const T (&x)[9][MX], T (&y)[9][MN], int& step) {
    constexpr int MK = D::own(NK);
    T xk[9][MK];
#pragma unroll
    for (int q = 0; q < 9; q++)
#pragma unroll
      for (int j = 0; j < MK; j++) xk[q][j] = x[q][j];
#pragma unroll 1
    for (int i = 0; i < 3; i++) {
      T g[3][MN], v[MN];
      component<true, NK, NN>(i, xk, lds + (step & 1) * D::CROWS * kCols, g, v);
      step++;
      const Mat4<T> m = mat();
      by_axis(i, [&](auto I) EDGE_INLINE {
        add_stress<decltype(I)::value>(y, g, m);
#pragma unroll
        for (int j = 0; j < MN; j++) y[6 + decltype(I)::value][j] = fma_(m.irho, v[j], y[6 + decltype(I)::value][j]);
      });
    }
  }

  // CK stages DE .. O - 1: x the derivative DE - 1 (modes below n_modes(O - DE + 1)),
  // t += sum_de dt^de / (de + 1)! der_de
  template <int DE, int MX>
  __device__ __forceinline__ void ck(const T (&x)[9][MX], T (&t)[9][M], T dt, T sca, int& step) {
    if constexpr (DE < O) {
      constexpr int NK = n_modes(O - DE + 1), NN = n_modes(O - DE), MN = D::own(NN);
      T y[9][MN];
#pragma unroll
      for (int q = 0; q < 9; q++)
#pragma unroll
        for (int j = 0; j < MN; j++) y[q][j] = T(0);
      stiffness<NK, NN>(x, y, step);
      sca *= dt / T(DE + 1);
#pragma unroll
      for (int q = 0; q < 9; q++)
#pragma unroll
        for (int j = 0; j < MN; j++) t[q][j] = fma_(sca, y[q][j], t[q][j]);
      ck<DE + 1>(y, t, dt, sca, step);
    }
  }

  // Component i of the faces' lifted flux, the w of all faces in the first
  // WROWS rows of LDS: velocities into vel (VEL) or acc, gradients into g; KC:
  // phys::kOwn (the element's side) or phys::kOth (the other side)
  template <int KC>
  __device__ __forceinline__ void lift(int i, T (&acc)[9][M], T (&vel)[3][M], T (&g)[3][M]) {
    const T* li = lds + i * D::NF * kCols + lane;
    each(
        [&](auto F) EDGE_INLINE {
          constexpr int f = decltype(F)::value;
          T u[M], n[3], sn[3], e[3];
#pragma unroll
          for (int k = 0; k < 3; k++) n[k] = face(f, phys::kNrm + k);
#pragma unroll
          for (int k = 0; k < 3; k++) sn[k] = face(f, phys::kScN + k);
          const T c1 = face(f, KC + 1), c0 = face(f, KC);
#pragma unroll
          for (int j = 0; j < M; j++) u[j] = T(0);
          by_wave<W>(w, [&](auto V) EDGE_INLINE {
            product<LiftReads<O, f, decltype(V)::value>>(li + 3 * f * D::NF * kCols, u);
          });
          const T ni = c1 * (i == 0 ? n[0] : i == 1 ? n[1] : n[2]);
#pragma unroll
          for (int k = 0; k < 3; k++) e[k] = fma_(ni, n[k], k == i ? c0 : T(0));
#pragma unroll
          for (int k = 0; k < 3; k++)
#pragma unroll
            for (int j = 0; j < M; j++) {
              g[k][j] = fma_(sn[k], u[j], g[k][j]);
              T& v = VEL ? vel[k][j] : acc[6 + k][j];
              v = fma_(e[k], u[j], v);
            }
        },
        std::make_integer_sequence<int, 4>{});
  }

  // acc += what f adds to its argument (SUM: to zeros)
  template <typename F>
  static __device__ __forceinline__ void add(T (&acc)[9][M], F f) {
    if constexpr (SUM) {
      T d[9][M];
#pragma unroll
      for (int q = 0; q < 9; q++) zero(d[q]);
      f(d);
#pragma unroll
      for (int q = 0; q < 9; q++)
#pragma unroll
        for (int j = 0; j < M; j++) acc[q][j] += d[q][j];
    } else {
      f(acc);
    }
  }
  static __device__ __forceinline__ void zero(T (&x)[M]) {
#pragma unroll
    for (int j = 0; j < M; j++) x[j] = T(0);
  }
  // VEL: acc += the summed velocities
  static __device__ __forceinline__ void add_velocities(T (&acc)[9][M], const T (&vel)[3][M]) {
    if constexpr (VEL)
#pragma unroll
      for (int k = 0; k < 3; k++)
#pragma unroll
        for (int j = 0; j < M; j++) acc[6 + k][j] += vel[k][j];
  }

  // acc += the neighbours' side of the faces' flux
  __device__ __forceinline__ void neigh(T (&acc)[9][M]) {
    add(acc, [&](T(&a)[9][M]) EDGE_INLINE {
#pragma unroll 1
      for (int i = 0; i < 3; i++) {
        T g[3][M], vel[3][M];
#pragma unroll
        for (int k = 0; k < 3; k++) zero(g[k]);
#pragma unroll
        for (int k = 0; k < 3; k++) zero(vel[k]);
        lift<phys::kOth>(i, a, vel, g);
        add_velocities(a, vel);
        const Mat4<T> m = mat();
        by_axis(i, [&](auto I) EDGE_INLINE { add_stress<decltype(I)::value>(a, g, m); });
      }
    });
  }

  // acc += volume integral and the element's side of the faces' flux, one
  // velocity component of both at a time (t: tInt / dt)
  __device__ __forceinline__ void space(const T (&t)[9][M], T (&acc)[9][M], T dt) {

    constexpr int NK = n_modes(O - 1), MK = D::own(NK);
    T* buf = lds + D::WROWS * kCols;
    T xk[9][MK];
#pragma unroll
    for (int q = 0; q < 9; q++)
#pragma unroll
      for (int j = 0; j < MK; j++) xk[q][j] = SCALED ? t[q][j] : dt * t[q][j];
    add(acc, [&](T(&a)[9][M]) EDGE_INLINE {
#pragma unroll 1
      for (int i = 0; i < 3; i++) {
        T g[3][M], v[M];
        __syncthreads();  // the previous columns have been read
        component<false, NK, D::N, SCALED>(i, xk, buf, g, v, dt);
        const T irho = mat().irho;
        by_axis(i, [&](auto I) EDGE_INLINE {
#pragma unroll
          for (int j = 0; j < M; j++) a[6 + decltype(I)::value][j] = fma_(irho, v[j], a[6 + decltype(I)::value][j]);
        });
        T vel[3][M];
#pragma unroll
        for (int k = 0; k < 3; k++) zero(vel[k]);
        lift<phys::kOwn>(i, a, vel, g);
        add_velocities(a, vel);
        const Mat4<T> m = mat();
        by_axis(i, [&](auto I) EDGE_INLINE { add_stress<decltype(I)::value>(a, g, m); });
      }
    });
  }

  // w of every face in the element's face coordinates, to LDS rows [f][i][NF]
  // (t: tInt / dt)
  __device__ __forceinline__ void project(const T (&t)[9][M], T dt) {
    T* cols = lds + D::WROWS * kCols;
    T* own = cols + w * kCols + lane;
    T next[7];  // the next face's normal and factors, a face ahead
#pragma unroll
    for (int k = 0; k < 7; k++) next[k] = face(0, k);
#pragma unroll 1
    for (int f = 0; f < 4; f++) {
      T n[3], a[4];
#pragma unroll
      for (int k = 0; k < 3; k++) n[k] = next[phys::kNrm + k];
#pragma unroll
      for (int k = 0; k < 4; k++) a[k] = SCALED ? dt * next[phys::kPrj + k] : next[phys::kPrj + k];
#pragma unroll
      for (int k = 0; k < 7; k++) next[k] = face(f < 3 ? f + 1 : 3, k);
      __syncthreads();  // the previous columns have been read
#pragma unroll
      for (int j = 0; j < M; j++) {
        if (!has(j, N)) continue;
        T tr[3];
#pragma unroll
        for (int k = 0; k < 3; k++)
          tr[k] = dot3(n[0], t[voigt(k, 0)][j], n[1], t[voigt(k, 1)][j], n[2], t[voigt(k, 2)][j]);
        const T vn = dot3(n[0], t[6][j], n[1], t[7][j], n[2], t[8][j]);
        const T tn = dot3(n[0], tr[0], n[1], tr[1], n[2], tr[2]);
        const T b = fma_(a[2], vn, -(a[3] * tn));
#pragma unroll
        for (int k = 0; k < 3; k++) {
          const T wk = fma_(n[k], b, fma_(a[0], t[6 + k][j], -(a[1] * tr[k])));
          own[(k * N + j * W) * kCols] = SCALED ? wk : dt * wk;
        }
      }
      __syncthreads();
#pragma unroll 1
      for (int i = 0; i < 3; i++) {
        T u[D::MF];
#pragma unroll
        for (int j = 0; j < D::MF; j++) u[j] = T(0);
        const T* li = cols + i * N * kCols + lane;
        by_wave<W>(w, [&](auto V) EDGE_INLINE {
          constexpr int wv = decltype(V)::value;
          if (f == 0)
            product<ProjectReads<O, 0, wv>>(li, u);
          else if (f == 1)
            product<ProjectReads<O, 1, wv>>(li, u);
          else if (f == 2)
            product<ProjectReads<O, 2, wv>>(li, u);
          else
            product<ProjectReads<O, 3, wv>>(li, u);
        });
        T* o = lds + ((f * 3 + i) * D::NF + w) * kCols + lane;
#pragma unroll
        for (int j = 0; j < D::MF; j++)
          if (has(j, D::NF)) o[j * W * kCols] = u[j];
      }
    }
  }

  // the faces' w from LDS to the projections of the tile's elements, four
  // values per store: vector v of 4 NV goes to wave v % W
  typedef T vec4 __attribute__((ext_vector_type(4)));
  static constexpr int NV = sp_proj_vectors(O);
  __device__ __forceinline__ void send(T* __restrict__ proj) const {
    if (!valid) return;
    vec4* o = reinterpret_cast<vec4*>(proj) + el * 4 * NV * R + lane % R;
#pragma unroll
    for (int f = 0; f < 4; f++)
#pragma unroll
      for (int v = 0; v < (NV + W - 1) / W; v++) {
        const int k = v * W + w;
        if (k >= NV) continue;
        vec4 x;
#pragma unroll
        for (int j = 0; j < 4; j++) x[j] = lds[(f * 3 * D::NF + (4 * k + j < 3 * D::NF ? 4 * k + j : 0)) * kCols + lane];
        o[(f * NV + k) * R] = x;
      }
  }

  // the neighbours' w (projections p), taken to the element's face
  // coordinates, to LDS rows [f][i][NF]: wave w takes face w % 4 (slot, fm:
  // its projection slot and flux matrix); of eight waves the first four take
  // the first two components
  __device__ __forceinline__ void receive(int32_t slot, int fm, const T* __restrict__ rot, const T* __restrict__ p,
                                          T (&u)[4 * NV], T (&r)[phys::kRotPad]) const {
    const vec4* src = reinterpret_cast<const vec4*>(p) + (int64_t)(slot < 0 ? 0 : slot) * NV * R + lane % R;
    const vec4* rv = reinterpret_cast<const vec4*>(rot) + (fm < 4 ? 0 : 1 + (fm - 4) / 4) * (phys::kRotPad / 4);
#pragma unroll
    for (int v = 0; v < NV; v++) {
      if (W == 8 && (w < 4 ? 4 * v >= 2 * D::NF : 4 * v + 3 < 2 * D::NF)) continue;
      const vec4 x = src[v * R];
#pragma unroll
      for (int j = 0; j < 4; j++) u[4 * v + j] = x[j];
    }
#pragma unroll
    for (int v = 0; v < (phys::rot_off(O) + 3) / 4; v++) {
      const vec4 x = rv[v];
#pragma unroll
      for (int j = 0; j < 4; j++) r[4 * v + j] = x[j];
    }
  }
  __device__ __forceinline__ void rotate(int32_t slot, const T (&u)[4 * NV], const T (&r)[phys::kRotPad]) {
    T* dst = lds + (w % 4) * 3 * D::NF * kCols + lane;
#pragma unroll
    for (int i = 0; i < 3; i++) {
      if (W == 8 && (w < 4) != (i < 2)) continue;
      each(
          [&](auto P) EDGE_INLINE {
            constexpr int p0 = decltype(P)::value, lo = p0 * (p0 + 1) / 2;
            each(
                [&](auto Mo) EDGE_INLINE {
                  constexpr int m = decltype(Mo)::value;
                  T v = T(0);
                  each(
                      [&](auto K) EDGE_INLINE {
                        constexpr int k = decltype(K)::value;
                        v = fma_(r[phys::rot_off(p0) + k * (p0 + 1) + m], u[i * D::NF + D::face_row(lo + k)], v);
                      },
                      std::make_integer_sequence<int, p0 + 1>{});
                  // (no slot: an outflow, fault or time-step interface face gives nothing)
                  dst[(i * D::NF + D::face_row(lo + m)) * kCols] = slot < 0 ? T(0) : v;
                },
                std::make_integer_sequence<int, p0 + 1>{});
          },
          std::make_integer_sequence<int, O>{});
    }
  }
};

// blockIdx -> tile: contiguous tile ranges per XCD, or in order.
__device__ __forceinline__ int64_t tile_index(int64_t n, bool xcd) {
  const int64_t b = blockIdx.x, chunk = (n + 7) / 8;
  return xcd ? (b & 7) * chunk + (b >> 3) : b;
}

// Waves per SIMD the registers are limited for: what the tiles' LDS allows
// (order 4 with three: 6.44 against 6.69 ms per step with two).
constexpr int waves_per_simd(int order, int bytes) { return order == 5 || bytes == 8 ? 2 : 3; }

// NB: the neighbouring surface integral from the projections proj_in; LOC:
// the local step (projections to x.proj, of a local step alone: unless null).  Both: the neighbour step of the
// previous time step first (its DOFs also go to s.tap for the elements
// s.tap_on marks).
template <typename T, int O, int R, bool NB, bool LOC>
__global__ __launch_bounds__(64 * kWaves, waves_per_simd(O, sizeof(T))) void k_sparse(SolverDev<T> s, SpDev<T> x, int64_t first, int64_t n, T dt, T* __restrict__ dofs, T* __restrict__ t_int,
              const T* __restrict__ proj_in) {
  using D = Dim<O>;
  constexpr int M = D::M, W = D::W, E = kCols / R;
  constexpr int STAGE = R == 1 ? (3 * D::N * (kCols + 1) + kCols - 1) / kCols : 0;
  constexpr int ROWS = !LOC ? D::WROWS : D::LROWS;
  __shared__ T lds[(ROWS > STAGE ? ROWS : STAGE) * kCols + (R == 1 ? 0 : E * phys::kSize)];
  const int64_t nt = (n + E - 1) / E, tile = tile_index(nt, s.xcd_map);
  if (tile >= nt) return;
  Tile<T, O, R> b(x.phys, first + tile * E);
  b.lds = lds;
  b.w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  b.lane = threadIdx.x & 63;
  by_wave<W>(b.w, [&](auto V) EDGE_INLINE {
    constexpr uint64_t m = Tile<T, O, R>::pack(decltype(V)::value);
    b.modes = m;
  });
  const int64_t left = n - tile * E;
  b.n_el = left < E ? (int)left : E;
  const int e = b.lane / R;
  b.valid = e < b.n_el;
  b.el = b.first + (b.valid ? e : b.n_el - 1);
  // the neighbours first (their projections are the longest chain of loads)
  int32_t slot = -1;
  int fm = 0;
  if constexpr (NB) {
    slot = s.rcv[b.el * 4 + b.w % 4];
    fm = s.nb.fmat[b.el * 4 + b.w % 4];
  }
  if constexpr (R == 1) {
    constexpr int PB = phys::block(R);
    b.ph_off = (unsigned)((b.el / PB - b.first / PB) * (phys::kSize * PB) + b.el % PB) * (unsigned)sizeof(T);
  } else {
    constexpr int C0 = (ROWS > STAGE ? ROWS : STAGE) * kCols;
    for (int i = threadIdx.x; i < b.n_el * phys::kSize; i += 64 * W)
      lds[C0 + i] = x.phys[b.first * phys::kSize + i];
    b.cst = lds + C0 + (int)(b.el - b.first) * phys::kSize;
  }
  T acc[9][M];
  auto constants = [&]() EDGE_INLINE {
    if constexpr (Tile<T, O, R>::HELD) {
      b.mat1 = {b.c(phys::kLam2), b.c(phys::kLam), b.c(phys::kMu), b.c(phys::kIrho)};
#pragma unroll
      for (int k = 0; k < 3; k++)
#pragma unroll
        for (int d = 0; d < 3; d++) b.ji1[k][d] = b.c(phys::kJinv + 3 * k + d);
    }
  };
  if constexpr (NB) {
    T u[4 * Tile<T, O, R>::NV], r[phys::kRotPad];
    b.receive(slot, fm, x.rot, proj_in, u, r);
    b.load(dofs, acc);
    b.rotate(slot, u, r);
    __syncthreads();
    constants();
    b.neigh(acc);
    if constexpr (LOC) {
      if (R > 1 && s.tap) b.store(s.tap, acc, b.valid && s.tap_on[b.el]);
      __syncthreads();
    } else {
      b.store(dofs, acc, b.valid);
    }
  }
  if constexpr (LOC) {
    // t = Q, then the time-integrated DOFs over dt.  The CK leaves the
    // highest modes as they are, so a copy of the others keeps Q in registers
    // until the volume integral (reading it again, and with NB writing it
    // first, was a third of the memory traffic).
    constexpr int NL = n_modes(O - 1), ML = D::own(NL);
    T t[9][M], low[9][ML];
    if constexpr (NB) {
#pragma unroll
      for (int q = 0; q < 9; q++)
#pragma unroll
        for (int j = 0; j < M; j++) t[q][j] = acc[q][j];
    } else {
      b.load(dofs, t);
      if constexpr (R > 1) __syncthreads();  // the constants are in LDS
      constants();
    }
#pragma unroll
    for (int q = 0; q < 9; q++)
#pragma unroll
      for (int j = 0; j < ML; j++) low[q][j] = t[q][j];
    int step = 0;
    b.template ck<1>(t, t, dt, T(1), step);
    // tInt: all of it, or of the elements in x.need; the projections (which
    // load nothing) run while it is written
    const bool on = b.valid && (x.tint || (x.need && x.need[b.el]));
    if constexpr (R > 1)
      if (__any(on)) b.template store<true>(t_int, t, on, dt);
    b.project(t, dt);
#pragma unroll
    for (int q = 0; q < 9; q++)
#pragma unroll
      for (int j = 0; j < M; j++) acc[q][j] = j < ML ? low[q][j < ML ? j : 0] : t[q][j];
    b.space(t, acc, dt);
    // (one run and FP32 with 16: always, their neighbour steps read nothing else)
    constexpr bool ALWAYS = NB || R == 1 || (R == 16 && sizeof(T) == 4);
    if (ALWAYS || x.proj) b.send(x.proj);
    if constexpr (R == 1) {
      if (x.tint || x.need) b.template store<true>(t_int, t, on, dt);
      __syncthreads();
    }
    b.store(dofs, acc, b.valid);
  }
}

template <typename T, int O, int R, bool NB, bool LOC>
int launch(const SolverDev<T>& s, const SpDev<T>& x, int64_t first, int64_t n, T dt, T* dofs, T* t_int,
           const T* proj_in, hipStream_t st) {
  const int64_t nt = (n + kCols / R - 1) / (kCols / R);
  const int64_t grid = s.xcd_map ? 8 * ((nt + 7) / 8) : nt;
  hipLaunchKernelGGL((k_sparse<T, O, R, NB, LOC>), dim3((unsigned)grid), dim3(64 * kWaves), 0, st, s, x, first, n, dt,
                     dofs, t_int, proj_in);
  EDGE_HIP_TRY(hipGetLastError());
  return EDGE_OK;
}

template <typename T, int O, int R>
int by_op(int op, const SolverDev<T>& s, const SpDev<T>& x, int64_t first, int64_t n, T dt, T* dofs, T* t_int,
          const T* proj_in, hipStream_t st) {
  if (op == kSpLocal) return launch<T, O, R, false, true>(s, x, first, n, dt, dofs, t_int, proj_in, st);
  if (op == kSpNeigh) return launch<T, O, R, true, false>(s, x, first, n, dt, dofs, t_int, proj_in, st);
  return launch<T, O, R, true, true>(s, x, first, n, dt, dofs, t_int, proj_in, st);
}

}  // namespace

template <typename T, int O>
int launch_sp(int op, const SolverDev<T>& s, const SpDev<T>& x, int64_t first, int64_t n, T dt, T* dofs, T* t_int,
              const T* proj_in, hipStream_t st) {
  if (n <= 0) return EDGE_OK;
  switch (s.n_runs) {
    case 1:
      if constexpr (sizeof(T) == 4 || O < 5) return by_op<T, O, 1>(op, s, x, first, n, dt, dofs, t_int, proj_in, st);
      break;
    case 8: return by_op<T, O, 8>(op, s, x, first, n, dt, dofs, t_int, proj_in, st);
    case 16:
      if constexpr (sizeof(T) == 4 || O < 5) return by_op<T, O, 16>(op, s, x, first, n, dt, dofs, t_int, proj_in, st);
      break;
  }
  return fail(EDGE_ERR_UNSUPPORTED, "runs");
}

}  // namespace edge
