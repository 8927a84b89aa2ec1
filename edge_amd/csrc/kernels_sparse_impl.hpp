// Element kernels that walk the non-zeros of the reference-element matrices
// on the vector ALU (elastic, geometry-built solvers).
//
// In the hierarchical orthogonal basis 82 % of the stiffness and 58 % of the
// flux matrices' entries are zero, and which ones is known when the kernels
// are compiled.  A lane holds one column, one (element, run) pair, and a
// workgroup of four waves works on 64 columns (64 / R elements).  Wave w owns
// a quarter of the modes of every quantity (Own): it keeps their DOFs in
// registers, so everything that mixes quantities at one mode is lane-local,
// and it computes the outputs of its modes of every matrix product.  The
// inputs of a product pass through LDS: the owners publish a column
// [mode][64] and every wave reads the modes its outputs need.  Each non-zero
// is one v_fmac_f32 with the entry as a literal: no operand loads, no
// padding, no work on zeros.  The four waves run different code (their own
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
// 64 columns at order 5 against 131,000 cycles of padded MFMA tiles) and, with
// two workgroups per CU, the LDS and memory latency they leave exposed.
// Measured against the kernels that did the same before (ms per step): order
// 5, 196,608 tets, 16 runs 8.59 -> 7.70 (MFMA, runs on N); one run 1.19 ->
// 1.01 (MFMA, 16 elements on N); order 5, 36,720 tets, 8 runs 6.81 -> 0.87
// (generic); order 4 with a fault, 331,776 tets, 16 runs 10.3 -> 6.69.
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
constexpr int kWaves = 4;

// Modes and face modes of each wave: found by balancing the waves' non-zeros
// per product, with the modes of every lower order spread evenly as well (a
// derivative's outputs are a prefix of each list).  -1: none.
template <int O>
struct Own;
template <>
struct Own<2> {
  static constexpr int mode[4][1] = {{0}, {1}, {2}, {3}};
  static constexpr int face[4][1] = {{0}, {1}, {2}, {-1}};
};
template <>
struct Own<3> {
  static constexpr int mode[4][3] = {{0, 6, -1}, {1, 5, 7}, {3, 4, 9}, {2, 8, -1}};
  static constexpr int face[4][2] = {{3, 4}, {2, 5}, {1, -1}, {0, -1}};
};
template <>
struct Own<4> {
  static constexpr int mode[4][5] = {{0, 8, 10, 12, 16}, {1, 7, 11, 15, 17}, {2, 5, 9, 13, 18}, {3, 4, 6, 14, 19}};
  static constexpr int face[4][3] = {{4, 6, 8}, {1, 7, 9}, {0, 5, -1}, {2, 3, -1}};
};
template <>
struct Own<5> {
  static constexpr int mode[4][9] = {{0, 6, 11, 13, 19, 22, 27, 33, -1},
                                     {1, 7, 10, 16, 18, 25, 26, 29, 30},
                                     {2, 5, 9, 14, 15, 20, 24, 28, 31},
                                     {3, 4, 8, 12, 17, 21, 23, 32, 34}};
  static constexpr int face[4][4] = {{2, 5, 10, 12}, {6, 7, 8, 13}, {1, 4, 11, 14}, {0, 3, 9, -1}};
};

template <int O>
struct Dim {
  static constexpr int N = n_modes(O), NF = n_face_modes(O);
  static constexpr int M = (N + 3) / 4, MF = (NF + 3) / 4;  // most modes / face modes of a wave
  // most of the modes below nn that a wave owns: a column of nn modes takes
  // 4 own(nn) LDS rows, mode Own[w][j] in row 4 j + w
  static constexpr int own(int nn) {
    int most = 0;
    for (int w = 0; w < 4; w++) {
      int c = 0;
      for (int j = 0; j < M; j++) c += Own<O>::mode[w][j] >= 0 && Own<O>::mode[w][j] < nn;
      most = c > most ? c : most;
    }
    return most;
  }
  static constexpr int row(int k) {
    for (int w = 0; w < 4; w++)
      for (int j = 0; j < M; j++)
        if (Own<O>::mode[w][j] == k) return 4 * j + w;
    return -1;
  }
  static constexpr int face_row(int k) {
    for (int w = 0; w < 4; w++)
      for (int j = 0; j < MF; j++)
        if (Own<O>::face[w][j] == k) return 4 * j + w;
    return -1;
  }
  static constexpr int FR = 4 * MF;                 // rows of a face column
  static constexpr int WROWS = 12 * FR;             // all four faces' w
  static constexpr int CROWS = 4 * 4 * own(N);      // four columns of the CK's first stage
  static constexpr int LROWS = 2 * CROWS > WROWS + 3 * 4 * M ? 2 * CROWS : WROWS + 3 * 4 * M;
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

// Output N's first non-zero among the inputs below K.
template <typename Mat, int K, int N>
constexpr bool starts() {
  for (int k = 0; N >= 0 && k < K; k++)
    if (Mat::at(k, N) != 0.0) return false;
  return true;
}

// out[j] += M[k][n_j] x over wave W's outputs n_j < nn with a non-zero entry
// (out[j] = for the first one).
template <typename Mat, int K, int N, bool FIRST, typename T>
__device__ __forceinline__ void term(T x, T& out) {
  if constexpr (N >= 0) {
    constexpr double v = Mat::at(K, N);
    if constexpr (v != 0.0) out = FIRST ? T(v) * x : fma_(T(v), x, out);
  }
}
template <int O, int NN, int W, int J>
constexpr int mode_of() {
  return Own<O>::mode[W][J] < NN ? Own<O>::mode[W][J] : -1;
}
template <int O, int NN, int W, typename Mat, int K, typename T, int... J>
__device__ __forceinline__ void terms(T x, T* out, std::integer_sequence<int, J...>) {
  (term<Mat, K, mode_of<O, NN, W, J>(), starts<Mat, K, mode_of<O, NN, W, J>()>()>(x, out[J]), ...);
}
template <int O, int W, typename Mat, int K, typename T, int... J>
__device__ __forceinline__ void face_terms(T x, T* out, std::integer_sequence<int, J...>) {
  (term<Mat, K, Own<O>::face[W][J], starts<Mat, K, Own<O>::face[W][J]>()>(x, out[J]), ...);
}
// The same with the sum running over three matrices per input.
template <int O, int NN, int W, typename M0, typename M1, typename M2, int K, typename T, int J>
__device__ __forceinline__ void term3(T x0, T x1, T x2, T& out) {
  constexpr int N = mode_of<O, NN, W, J>();
  if constexpr (N >= 0) {
    constexpr bool s = starts<M0, K, N>() && starts<M1, K, N>() && starts<M2, K, N>();
    constexpr bool n0 = M0::at(K, N) != 0.0, n1 = M1::at(K, N) != 0.0;
    term<M0, K, N, s>(x0, out);
    term<M1, K, N, s && !n0>(x1, out);
    term<M2, K, N, s && !n0 && !n1>(x2, out);
  }
}
template <int O, int NN, int W, typename M0, typename M1, typename M2, int K, typename T, int... J>
__device__ __forceinline__ void terms3(T x0, T x1, T x2, T* out, std::integer_sequence<int, J...>) {
  (term3<O, NN, W, M0, M1, M2, K, T, J>(x0, x1, x2, out[J]), ...);
}

template <int O, bool CK, int D>
using Stiff = std::conditional_t<CK, Ck<O, D>, Vol<O, D>>;

// One published component: column 0 (the raw velocity) times all three
// stiffness matrices into p[d], columns 1 + d times matrix d, summed, into v;
// outputs of wave W below NN, inputs below NK.  l: the lane's first row;
// RK: rows per column.
template <int O, bool CK, int NK, int NN, int W, typename T, int... K>
__device__ __forceinline__ void stiff_mul(const T* l, T (&p)[3][Dim<O>::own(NN)], T (&v)[Dim<O>::own(NN)],
                                          std::integer_sequence<int, K...>) {
  constexpr int RK = 4 * Dim<O>::own(NK) * kCols;
  using J = std::make_integer_sequence<int, Dim<O>::own(NN)>;
  (
      [&]() EDGE_INLINE {
        const T x = l[Dim<O>::row(K) * kCols];
        terms<O, NN, W, Stiff<O, CK, 0>, K>(x, p[0], J{});
        terms<O, NN, W, Stiff<O, CK, 1>, K>(x, p[1], J{});
        terms<O, NN, W, Stiff<O, CK, 2>, K>(x, p[2], J{});
      }(),
      ...);
  (
      [&]() EDGE_INLINE {
        terms3<O, NN, W, Stiff<O, CK, 0>, Stiff<O, CK, 1>, Stiff<O, CK, 2>, K>(
            l[RK + Dim<O>::row(K) * kCols], l[2 * RK + Dim<O>::row(K) * kCols], l[3 * RK + Dim<O>::row(K) * kCols], v,
            J{});
      }(),
      ...);
}

// One column of a face's w in the element's modes to the wave's face modes.
template <int O, int F, int W, typename T, int... K>
__device__ __forceinline__ void project_mul(const T* l, T (&u)[Dim<O>::MF], std::integer_sequence<int, K...>) {
  (face_terms<O, W, Prj<O, F>, K>(l[Dim<O>::row(K) * kCols], u, std::make_integer_sequence<int, Dim<O>::MF>{}), ...);
}

// One face column to the wave's modes.
template <int O, int F, int W, typename T, int... K>
__device__ __forceinline__ void lift_mul(const T* l, T (&u)[Dim<O>::M], std::integer_sequence<int, K...>) {
  (terms<O, Dim<O>::N, W, Lift<O, F>, K>(l[Dim<O>::face_row(K) * kCols], u,
                                         std::make_integer_sequence<int, Dim<O>::M>{}),
   ...);
}

// The calling wave's code (w is uniform across the wave).  The (empty, but
// different) last statements keep the branches from being merged over the
// registers they update, which would put those into memory.
template <typename F>
__device__ __forceinline__ void by_wave(int w, F f) {
  if (w == 0) {
    f(Int<0>{});
    asm volatile("; wave 0");
  } else if (w == 1) {
    f(Int<1>{});
    asm volatile("; wave 1");
  } else if (w == 2) {
    f(Int<2>{});
    asm volatile("; wave 2");
  } else {
    f(Int<3>{});
    asm volatile("; wave 3");
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
  static constexpr int N = D::N, SZ = 9 * N * R, M = D::M;
  T* lds;
  int w, lane;
  int64_t el;      // the lane's element (the last one's for lanes past the range)
  int64_t first;   // first element of the tile
  int n_el;        // elements of the tile inside the range
  bool valid;
  Buf<T> ph;       // constants of the tile's elements
  unsigned ph_off;
  T ji[3][3];
  Mat4<T> mat;

  __device__ __forceinline__ Tile(const T* phys_el, int64_t first_)
      : first(first_), ph(phys_el + first_ / phys::kBlock * (phys::kSize * phys::kBlock), 2 * phys::kSize * phys::kBlock) {}
  __device__ __forceinline__ T c(int k) const { return ph.load(ph_off, k * phys::kBlock * (unsigned)sizeof(T)); }
  // byte offset of the lane's column in a DOF array of the tile
  __device__ __forceinline__ unsigned column() const {
    return (unsigned)((el - first) * SZ + lane % R) * (unsigned)sizeof(T);
  }
  __device__ __forceinline__ T face(int f, int k) const { return c(phys::kFace + phys::kPerFace * f + k); }
  // the wave's modes, six bits each (where it has fewer than M, its first
  // mode again: those registers hold copies that nothing reads)
  uint64_t modes;
  static constexpr uint64_t pack(int w) {
    uint64_t b = 0;
    for (int j = 0; j < M; j++)
      b |= (uint64_t)(Own<O>::mode[w][j] < 0 ? Own<O>::mode[w][0] : Own<O>::mode[w][j]) << (6 * j);
    return b;
  }
  __device__ __forceinline__ int mode(int j) const { return (int)(modes >> (6 * j)) & 63; }
  static constexpr bool every(int j) {  // every wave has a j-th mode
    for (int w = 0; w < 4; w++)
      if (Own<O>::mode[w][j] < 0) return false;
    return true;
  }
  __device__ __forceinline__ bool has(int j) const { return every(j) || j == 0 || mode(j) != mode(0); }

  // the wave's modes of a DOF array (zeros past the last one)
  __device__ __forceinline__ void load(const T* __restrict__ a, T (&x)[9][M]) {
    if constexpr (R == 1) {
      // one element is contiguous: three quantities of the 64 elements at a
      // time pass through LDS (rows of 65 columns: no bank conflicts)
#pragma unroll
      for (int qb = 0; qb < 9; qb += 3) {
        __syncthreads();
        const T* src = a + first * SZ + qb * N;
#pragma unroll 4
        for (int i = threadIdx.x; i < kCols * 3 * N; i += 64 * kWaves) {
          const int e = i / (3 * N), v = i % (3 * N);
          lds[v * (kCols + 1) + e] = src[(e < n_el ? e : n_el - 1) * SZ + v];
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 3; q++)
#pragma unroll
          for (int j = 0; j < M; j++) {
            x[qb + q][j] = lds[(q * N + mode(j)) * (kCols + 1) + lane];
          }
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

  // stores the wave's modes (fused runs: of the lanes with `on`); ADD: adds
  // them to the array (one run only)
  template <bool ADD = false>
  __device__ __forceinline__ void store(T* __restrict__ a, const T (&x)[9][M], bool on) {
    if constexpr (R == 1) {
#pragma unroll
      for (int qb = 0; qb < 9; qb += 3) {
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 3; q++)
#pragma unroll
          for (int j = 0; j < M; j++) {
            if (has(j)) lds[(q * N + mode(j)) * (kCols + 1) + lane] = x[qb + q][j];
          }
        __syncthreads();
        T* dst = a + first * SZ + qb * N;
#pragma unroll 4
        for (int i = threadIdx.x; i < n_el * 3 * N; i += 64 * kWaves) {
          const int e = i / (3 * N), v = i % (3 * N);
          const T y = lds[v * (kCols + 1) + e];
          dst[e * SZ + v] = ADD ? dst[e * SZ + v] + y : y;
        }
      }
    } else {
      static_assert(!ADD || R == 1, "fused runs start from the DOFs");
      const Buf<T> dst(a + first * SZ, n_el * SZ);
      const unsigned off = on ? column() : kSkip;
#pragma unroll
      for (int j = 0; j < M; j++) {
        if (!has(j)) continue;
#pragma unroll
        for (int q = 0; q < 9; q++) dst.store(x[q][j], off, (unsigned)((mode(j) + q * N) * R * (int)sizeof(T)));
      }
    }
  }

  // Publishes velocity component I and the three star-combined rows
  // sum_k j[k][d] sigma_Ik of the modes below NK.
  template <int I, int MK>
  __device__ __forceinline__ void publish(T* l, const T (&x)[9][MK], const T (&j3)[3][3], Int<I>) const {
    constexpr int RK = 4 * MK * kCols;
#pragma unroll
    for (int j = 0; j < MK; j++) {
      T* o = l + 4 * j * kCols;
      o[0] = x[6 + I][j];
#pragma unroll
      for (int d = 0; d < 3; d++)
        o[(d + 1) * RK] = dot3(j3[0][d], x[voigt(I, 0)][j], j3[1][d], x[voigt(I, 1)][j], j3[2][d], x[voigt(I, 2)][j]);
    }
  }

  // y += S (stiffness products of x), x on the modes below NK, y below NN:
  // per velocity component i one published set of columns; buffers alternate
  // (step counts them), so one barrier per component is enough.
  template <bool CK, int NK, int NN, int MX, int MY>
  __device__ __forceinline__ void stiffness(const T (&x)[9][MX], T (&y)[9][MY], int& step) {
    constexpr int MK = D::own(NK), MN = D::own(NN);
    static_assert(MX >= MK && MY >= MN, "registers of the wave's modes");
    T xk[9][MK];
#pragma unroll
    for (int q = 0; q < 9; q++)
#pragma unroll
      for (int j = 0; j < MK; j++) xk[q][j] = x[q][j];
#pragma unroll 1
    for (int i = 0; i < 3; i++) {
      T* buf = lds + (step & 1) * D::CROWS * kCols;
      step++;
      // (opaque to the optimiser: the combined rows of every component would
      // otherwise be formed ahead of the loop and spilled)
      T j3[3][3];
#pragma unroll
      for (int k = 0; k < 3; k++)
#pragma unroll
        for (int d = 0; d < 3; d++) {
          j3[k][d] = ji[k][d];
          asm volatile("" : "+v"(j3[k][d]));
        }
      by_axis(i, [&](auto I) EDGE_INLINE { publish(buf + w * kCols + lane, xk, j3, I); });
      __syncthreads();
      T p[3][MN], v[MN];
#pragma unroll
      for (int j = 0; j < MN; j++) p[0][j] = p[1][j] = p[2][j] = v[j] = T(0);
      by_wave(w, [&](auto W) EDGE_INLINE {
        stiff_mul<O, CK, NK, NN, decltype(W)::value>(buf + lane, p, v, std::make_integer_sequence<int, NK>{});
      });
      T g[3][MN];
#pragma unroll
      for (int k = 0; k < 3; k++)
#pragma unroll
        for (int j = 0; j < MN; j++) g[k][j] = dot3(ji[k][0], p[0][j], ji[k][1], p[1][j], ji[k][2], p[2][j]);
      by_axis(i, [&](auto I) EDGE_INLINE {
        add_stress<decltype(I)::value>(y, g, mat);
#pragma unroll
        for (int j = 0; j < MN; j++) y[6 + decltype(I)::value][j] = fma_(mat.irho, v[j], y[6 + decltype(I)::value][j]);
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
      stiffness<true, NK, NN>(x, y, step);
      sca *= dt / T(DE + 1);
#pragma unroll
      for (int q = 0; q < 9; q++)
#pragma unroll
        for (int j = 0; j < MN; j++) t[q][j] = fma_(sca, y[q][j], t[q][j]);
      ck<DE + 1>(y, t, dt, sca, step);
    }
  }

  // acc += the lifted flux of the w of all faces in the first WROWS rows of
  // LDS; KC: phys::kOwn (the element's side) or phys::kOth (the other side)
  template <int KC>
  __device__ __forceinline__ void lifts(T (&acc)[9][M]) {
#pragma unroll 1
    for (int i = 0; i < 3; i++) {
      T g[3][M];
#pragma unroll
      for (int j = 0; j < M; j++) g[0][j] = g[1][j] = g[2][j] = T(0);
      const T* li = lds + i * D::FR * kCols + lane;
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
            by_wave(w, [&](auto W) EDGE_INLINE {
              lift_mul<O, f, decltype(W)::value>(li + 3 * f * D::FR * kCols, u,
                                                 std::make_integer_sequence<int, D::NF>{});
            });
            const T ni = c1 * (i == 0 ? n[0] : i == 1 ? n[1] : n[2]);
#pragma unroll
            for (int k = 0; k < 3; k++) e[k] = fma_(ni, n[k], k == i ? c0 : T(0));
#pragma unroll
            for (int k = 0; k < 3; k++) {
              const T m = sn[k];
#pragma unroll
              for (int j = 0; j < M; j++) {
                g[k][j] = fma_(m, u[j], g[k][j]);
                acc[6 + k][j] = fma_(e[k], u[j], acc[6 + k][j]);
              }
            }
          },
          std::make_integer_sequence<int, 4>{});
      by_axis(i, [&](auto I) EDGE_INLINE { add_stress<decltype(I)::value>(acc, g, mat); });
    }
  }

  // w of every face in the element's face coordinates: to LDS rows
  // [f][i][FR] and to the projections proj
  __device__ __forceinline__ void project(const T (&t)[9][M], T* __restrict__ proj) {
    T* cols = lds + D::WROWS * kCols;
    T* own = cols + w * kCols + lane;
#pragma unroll 1
    for (int f = 0; f < 4; f++) {
      T n[3], a[4];
#pragma unroll
      for (int k = 0; k < 3; k++) n[k] = face(f, phys::kNrm + k);
#pragma unroll
      for (int k = 0; k < 4; k++) a[k] = face(f, phys::kPrj + k);
      __syncthreads();  // the previous columns have been read
#pragma unroll
      for (int j = 0; j < M; j++) {
        T tr[3];
#pragma unroll
        for (int k = 0; k < 3; k++)
          tr[k] = dot3(n[0], t[voigt(k, 0)][j], n[1], t[voigt(k, 1)][j], n[2], t[voigt(k, 2)][j]);
        const T vn = dot3(n[0], t[6][j], n[1], t[7][j], n[2], t[8][j]);
        const T tn = dot3(n[0], tr[0], n[1], tr[1], n[2], tr[2]);
        const T b = fma_(a[2], vn, -(a[3] * tn));
#pragma unroll
        for (int k = 0; k < 3; k++) own[(k * 4 * M + 4 * j) * kCols] = fma_(n[k], b, fma_(a[0], t[6 + k][j], -(a[1] * tr[k])));
      }
      __syncthreads();
#pragma unroll 1
      for (int i = 0; i < 3; i++) {
        T u[D::MF];
#pragma unroll
        for (int j = 0; j < D::MF; j++) u[j] = T(0);
        const T* li = cols + i * 4 * M * kCols + lane;
        by_wave(w, [&](auto W) EDGE_INLINE {
          constexpr int wv = decltype(W)::value;
          using K = std::make_integer_sequence<int, N>;
          if (f == 0)
            project_mul<O, 0, wv>(li, u, K{});
          else if (f == 1)
            project_mul<O, 1, wv>(li, u, K{});
          else if (f == 2)
            project_mul<O, 2, wv>(li, u, K{});
          else
            project_mul<O, 3, wv>(li, u, K{});
        });
        T* o = lds + ((f * 3 + i) * D::FR + w) * kCols + lane;
#pragma unroll
        for (int j = 0; j < D::MF; j++) o[4 * j * kCols] = u[j];
        if (valid) {
          T* g = proj + ((((el * 4 + f) * 12 + i * 4 + w) * R) + lane % R) * D::MF;
#pragma unroll
          for (int j = 0; j < D::MF; j++) g[j] = u[j];
        }
      }
    }
  }

  // the neighbours' w (projections p), taken to the element's face
  // coordinates, to LDS rows [f][i][FR]: wave w takes face w
  __device__ __forceinline__ void receive(const SolverDev<T>& s, const T* __restrict__ rot, const T* __restrict__ p) {
    const int32_t slot = s.rcv[el * 4 + w];
    const int fm = s.nb.fmat[el * 4 + w];
    const T* rv = rot + (fm < 4 ? 0 : 1 + (fm - 4) / 4) * phys::kRotPad;
    const T* src = p + (((int64_t)(slot < 0 ? 0 : slot) * 12 * R) + lane % R) * D::MF;
    T* dst = lds + w * 3 * D::FR * kCols + lane;
    T u[3][D::FR];
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
      for (int o = 0; o < 4; o++)
#pragma unroll
        for (int j = 0; j < D::MF; j++) u[i][4 * j + o] = src[((i * 4 + o) * R) * D::MF + j];
    if (slot < 0) {  // outflow, fault and time-step interfaces: nothing
#pragma unroll
      for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < D::FR; j++) u[i][j] = T(0);
    }
    each(
        [&](auto P) EDGE_INLINE {
          constexpr int p0 = decltype(P)::value, lo = p0 * (p0 + 1) / 2;
          T r[p0 + 1][p0 + 1];
#pragma unroll
          for (int k = 0; k <= p0; k++)
#pragma unroll
            for (int m = 0; m <= p0; m++) r[k][m] = rv[phys::rot_off(p0) + k * (p0 + 1) + m];
          each(
              [&](auto Mo) EDGE_INLINE {
                constexpr int m = decltype(Mo)::value;
#pragma unroll
                for (int i = 0; i < 3; i++) {
                  T v = T(0);
                  each([&](auto K) EDGE_INLINE { v = fma_(r[decltype(K)::value][m], u[i][D::face_row(lo + decltype(K)::value)], v); },
                       std::make_integer_sequence<int, p0 + 1>{});
                  dst[(i * D::FR + D::face_row(lo + m)) * kCols] = v;
                }
              },
              std::make_integer_sequence<int, p0 + 1>{});
        },
        std::make_integer_sequence<int, O>{});
  }
};

// blockIdx -> tile: contiguous tile ranges per XCD, or in order.
__device__ __forceinline__ int64_t tile_index(int64_t n, bool xcd) {
  const int64_t b = blockIdx.x, chunk = (n + 7) / 8;
  return xcd ? (b & 7) * chunk + (b >> 3) : b;
}

// NB: the neighbouring surface integral from the projections proj_in; LOC:
// the local step (projections to x.proj).  Both: the neighbour step of the
// previous time step first, its DOFs go back to global memory (and to s.tap
// for the elements s.tap_on marks) and are read again for the output.
template <typename T, int O, int R, bool NB, bool LOC>
__global__ __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(2)))
void k_sparse(SolverDev<T> s, SpDev<T> x, int64_t first, int64_t n, T dt, T* __restrict__ dofs, T* __restrict__ t_int,
              const T* __restrict__ proj_in) {
  using D = Dim<O>;
  constexpr int M = D::M, E = kCols / R;
  constexpr int STAGE = R == 1 ? (3 * D::N * (kCols + 1) + kCols - 1) / kCols : 0;
  constexpr int ROWS = !LOC ? D::WROWS : D::LROWS;
  __shared__ T lds[(ROWS > STAGE ? ROWS : STAGE) * kCols];
  const int64_t nt = (n + E - 1) / E, tile = tile_index(nt, s.xcd_map);
  if (tile >= nt) return;
  Tile<T, O, R> b(x.phys, first + tile * E);
  b.lds = lds;
  b.w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  b.lane = threadIdx.x & 63;
  {
    using Ti = Tile<T, O, R>;
    constexpr uint64_t m0 = Ti::pack(0), m1 = Ti::pack(1), m2 = Ti::pack(2), m3 = Ti::pack(3);
    b.modes = b.w == 0 ? m0 : b.w == 1 ? m1 : b.w == 2 ? m2 : m3;
  }
  const int64_t left = n - tile * E;
  b.n_el = left < E ? (int)left : E;
  const int e = b.lane / R;
  b.valid = e < b.n_el;
  b.el = b.first + (b.valid ? e : b.n_el - 1);
  b.ph_off = (unsigned)((b.el / phys::kBlock - b.first / phys::kBlock) * (phys::kSize * phys::kBlock) +
                        b.el % phys::kBlock) * (unsigned)sizeof(T);
  b.mat = {b.c(phys::kLam2), b.c(phys::kLam), b.c(phys::kMu), b.c(phys::kIrho)};
  T acc[9][M];
  auto start = [&]() EDGE_INLINE {  // one run: the DOFs are added where the update is stored
    if constexpr (R == 1) {
#pragma unroll
      for (int q = 0; q < 9; q++)
#pragma unroll
        for (int j = 0; j < M; j++) acc[q][j] = T(0);
    } else {
      b.load(dofs, acc);
    }
  };
  if constexpr (NB) {
    start();
    b.receive(s, x.rot, proj_in);
    __syncthreads();
    b.template lifts<phys::kOth>(acc);
    b.template store<R == 1>(dofs, acc, b.valid);
    if constexpr (LOC) {
      if (s.tap) b.store(s.tap, acc, b.valid && s.tap_on[b.el]);
      __syncthreads();
    }
  }
  if constexpr (LOC) {
#pragma unroll
    for (int k = 0; k < 3; k++)
#pragma unroll
      for (int d = 0; d < 3; d++) b.ji[k][d] = b.c(phys::kJinv + 3 * k + d);
    T t[9][M];
    if constexpr (NB) {
#pragma unroll
      for (int q = 0; q < 9; q++)
#pragma unroll
        for (int j = 0; j < M; j++) t[q][j] = acc[q][j];
    } else {
      b.load(dofs, t);
    }
    int step = 0;
    b.template ck<1>(t, t, dt, T(1), step);
#pragma unroll
    for (int q = 0; q < 9; q++)
#pragma unroll
      for (int j = 0; j < M; j++) t[q][j] *= dt;
    if constexpr (R == 1) __syncthreads();  // (the staging buffer is the products' buffer)
    b.store(t_int, t, b.valid);
    if constexpr (R == 1) __syncthreads();
    start();
    b.template stiffness<false, n_modes(O - 1), D::N>(t, acc, step);
    b.project(t, x.proj);
    __syncthreads();
    b.template lifts<phys::kOwn>(acc);
    b.template store<R == 1>(dofs, acc, b.valid);
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
  if constexpr (R > 1) return launch<T, O, R, true, true>(s, x, first, n, dt, dofs, t_int, proj_in, st);
  return fail(EDGE_ERR_UNSUPPORTED, "fused sparse step: 8 or 16 runs");
}

}  // namespace

template <typename T, int O>
int launch_sp(int op, const SolverDev<T>& s, const SpDev<T>& x, int64_t first, int64_t n, T dt, T* dofs, T* t_int,
              const T* proj_in, hipStream_t st) {
  if (n <= 0) return EDGE_OK;
  switch (s.n_runs) {
    case 1: return by_op<T, O, 1>(op, s, x, first, n, dt, dofs, t_int, proj_in, st);
    case 8: return by_op<T, O, 8>(op, s, x, first, n, dt, dofs, t_int, proj_in, st);
    case 16: return by_op<T, O, 16>(op, s, x, first, n, dt, dofs, t_int, proj_in, st);
  }
  return fail(EDGE_ERR_UNSUPPORTED, "runs");
}

}  // namespace edge
