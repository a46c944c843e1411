// Batched dense complex linear algebra for the Beyn contour loop:
// blocked LU with partial pivoting (replaces lu!(T; check=false), i.e.
// LAPACK zgetrf, beyn.jl:270-277), the two triangular solves with the row
// permutation (ldiv!, zgetrs, beyn.jl:281), the FP64 residual of the
// mixed-precision refinement, and the moment sums (axpy!, beyn.jl:282-283).
//
// Every routine works on a batch of matrices with a fixed stride (one matrix
// per contour node), so one launch covers all nodes of a window.  Matrices
// are column-major, complex interleaved.  T = cf (complex64) or cd
// (complex128).
//
// Structure (right-looking, panel width NB = qb_lu_nb(n), 256 or 512):
//   panel (recursive, leaf width 32: single-workgroup column elimination)
//   -> row swaps on the other columns -> unit-lower TRSM of the block row
//   -> trailing update C -= A*B on MFMA.
// The trailing update and every GEMM inside the recursions run in
// k_gemm_sub, which splits complex operands into real/imaginary planes in
// LDS and issues 4 real 16x16x4 MFMAs per complex product block
// (v_mfma_f32_16x16x4_f32 for complex64, v_mfma_f64_16x16x4_f64 for
// complex128) with accumulation in the operand precision.
#include <stdlib.h>

#include <type_traits>
#include <vector>

#include "qb_internal.h"
#include "qb_linalg.h"

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef double doublex4 __attribute__((ext_vector_type(4)));

template <typename T>
struct Scal;
template <>
struct Scal<cf> {
  typedef float S;
  typedef floatx4 V4;
};
template <>
struct Scal<cd> {
  typedef double S;
  typedef doublex4 V4;
};

__device__ __forceinline__ floatx4 mfma16(float a, float b, floatx4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ doublex4 mfma16(double a, double b, doublex4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// Tile of this workgroup of a (gx, gy, batch) grid.  Workgroups are dispatched
// round-robin over the 8 XCDs (each with its own L2): those of one L mod 8 of a
// matrix run on one XCD and take a contiguous range of tile ids, which walk groups
// of `grp` m-tiles sweeping n, so that the workgroups resident on an XCD share A and B
// panels in its L2.  Ranges differ by one tile where the count is no multiple of 8.
__device__ __forceinline__ void xcd_tile(unsigned grp, int* mt, int* nt) {
  const unsigned gx = gridDim.x, gy = gridDim.y, n = gx * gy;
  const unsigned L = blockIdx.x + gx * blockIdx.y, x = L & 7u, rem = n & 7u;
  const unsigned t = x * (n >> 3) + (x < rem ? x : rem) + (L >> 3);
  const unsigned first = t / (grp * gy) * grp;
  const unsigned gm = gx - first < grp ? gx - first : grp;
  const unsigned loc = t - first * gy;
  *mt = (int)(first + loc % gm);
  *nt = (int)(loc / gm);
}

// ---------------------------------------------------------------------------
// GEMM: C[b] -= A[b] * B[b]  (A: M x K, B: K x N, C: M x N)
// ---------------------------------------------------------------------------
// Workgroup tile BM x BN, k-tile BK, 4 waves arranged WGM x WGN; each wave
// computes a (BM/WGM) x (BN/WGN) tile of 16 x 16 MFMA blocks, one
// accumulator block for the real and one for the imaginary part.  MFMA
// 16x16x4 operand layout (one value per lane): A[i][k] with i = lane % 16,
// k = lane / 16; B[k][j] with j = lane % 16, k = lane / 16.  Result
// register v of a lane holds D[4*(lane/16) + v][lane % 16] for the f32
// instruction and D[4*v + lane/16][lane % 16] for the f64 one (checked on
// gfx950).
//
// Pipeline: the next k-tile is loaded from global memory into registers
// while the current one is multiplied out of LDS; the two LDS buffers
// alternate, so each k-tile costs one barrier.  A is stored k-major
// ([k][m], row pad of 16 words puts the four k rows a wave reads in
// different bank quarters), B n-major ([n][k], row stride below) so that
// both the coalesced global loads and the fragment reads are conflict-free.  A is
// negated when it is written to LDS, so the accumulators hold -A*B and the
// epilogue adds them to C.
template <typename T, int BM, int BN, int BK, int WGM, int WGN, bool XCD, bool G3, int PF,
          int OCC>
__global__ void __launch_bounds__(256, OCC) k_gemm_sub(int M, int N, int K, const T* __restrict__ A,
                                                  int64_t lda, int64_t sA,
                                                  const T* __restrict__ B, int64_t ldb,
                                                  int64_t sB, T* __restrict__ C, int64_t ldc,
                                                  int64_t sC, const int* __restrict__ bix) {
  typedef typename Scal<T>::S S;
  typedef typename Scal<T>::V4 V4;
  static_assert(WGM * WGN == 4, "4 waves");
  constexpr int WM = BM / WGM, WN = BN / WGN;
  constexpr int FM = WM / 16, FN = WN / 16;
  constexpr int APAD = (sizeof(S) == 4) ? 16 : 8;
  constexpr int AST = BM + APAD;       // A row stride (elements)
  // B row stride: the f32 fragment read (li * BST + lk, li < 16, lk < 4)
  // maps the 64 lanes of a wave onto 64 distinct 4-byte banks when BST is 4
  // times an odd number (BK + 4 for BK = 16, 32); BK + 1 wraps lane 15 onto
  // lane 0.
  constexpr int BST = (sizeof(S) == 4) ? BK + 4 : BK + 1;
  constexpr int NA = BM * BK / 256;    // complex elements of A per thread per tile
  constexpr int NB = BN * BK / 256;
  static_assert(NA * 256 == BM * BK && NB * 256 == BN * BK, "tile/thread mismatch");
  __shared__ S As[2][2][BK * AST];     // [buf][re/im]
  __shared__ S Bs[2][2][BN * BST];

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int wm0 = (wave % WGM) * WM, wn0 = (wave / WGM) * WN;
  int mt = blockIdx.x, ntile = blockIdx.y;
  if constexpr (XCD) {
    xcd_tile(8, &mt, &ntile);
  }
  const int m0 = mt * BM, n0 = ntile * BN;
  const int64_t b = bix ? bix[blockIdx.z] : blockIdx.z;
  A += b * sA;
  B += b * sB;
  C += b * sC;
  const int li = lane & 15, lk = lane >> 4;

  // acc_re / acc_im hold -Re(AB) / -Im(AB); with G3 (Gauss's three-product
  // form) they hold P1 = (-Ar) Br and P2 = (-Ai) Bi, and acc_s holds
  // P3 = -(Ar + Ai)(Br + Bi): -Re = P1 - P2, -Im = P3 - P1 - P2.
  V4 acc_re[FM][FN], acc_im[FM][FN], acc_s[G3 ? FM : 1][G3 ? FN : 1];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      acc_re[i][j] = V4{0, 0, 0, 0};
      acc_im[i][j] = V4{0, 0, 0, 0};
      if constexpr (G3) acc_s[i][j] = V4{0, 0, 0, 0};
    }

  // PF register slots stage k-tiles on their way from global memory to LDS:
  // with PF = 2 the loads of k-tile t+2 are issued while k-tile t is
  // multiplied, so they have two k-tiles of MFMA work to arrive in.
  T ra[PF][NA], rb[PF][NB];
  // tiles fully inside M x N (all but the edge tiles) load k-tiles that are
  // fully inside K without per-element bounds checks
  const bool full_mn = (m0 + BM <= M) && (n0 + BN <= N);
  auto gload = [&](auto slot, int k0) {
    constexpr int sl = decltype(slot)::value;
    if (full_mn && k0 + BK <= K) {
#pragma unroll
      for (int p = 0; p < NA; ++p) {
        int e = tid + 256 * p;
        int m = e % BM, kk = e / BM;
        ra[sl][p] = A[(m0 + m) + (int64_t)(k0 + kk) * lda];
      }
#pragma unroll
      for (int p = 0; p < NB; ++p) {
        int e = tid + 256 * p;
        int kk = e % BK, n = e / BK;
        rb[sl][p] = B[(k0 + kk) + (int64_t)(n0 + n) * ldb];
      }
      return;
    }
#pragma unroll
    for (int p = 0; p < NA; ++p) {
      int e = tid + 256 * p;
      int m = e % BM, kk = e / BM;
      int gm = m0 + m, gk = k0 + kk;
      ra[sl][p] = (gm < M && gk < K) ? A[gm + (int64_t)gk * lda] : T{0, 0};
    }
#pragma unroll
    for (int p = 0; p < NB; ++p) {
      int e = tid + 256 * p;
      int kk = e % BK, n = e / BK;
      int gn = n0 + n, gk = k0 + kk;
      rb[sl][p] = (gn < N && gk < K) ? B[gk + (int64_t)gn * ldb] : T{0, 0};
    }
  };
  auto sstore = [&](auto slot, int buf) {
    constexpr int sl = decltype(slot)::value;
#pragma unroll
    for (int p = 0; p < NA; ++p) {
      int e = tid + 256 * p;
      int m = e % BM, kk = e / BM;
      As[buf][0][kk * AST + m] = -ra[sl][p].re;
      As[buf][1][kk * AST + m] = -ra[sl][p].im;
    }
#pragma unroll
    for (int p = 0; p < NB; ++p) {
      int e = tid + 256 * p;
      int kk = e % BK, n = e / BK;
      Bs[buf][0][n * BST + kk] = rb[sl][p].re;
      Bs[buf][1][n * BST + kk] = rb[sl][p].im;
    }
  };
  using S0 = std::integral_constant<int, 0>;
  using S1 = std::integral_constant<int, PF - 1>;

  auto compute = [&](int buf) {
    const S* Ar = As[buf][0];
    const S* Ai = As[buf][1];
    const S* Br = Bs[buf][0];
    const S* Bi = Bs[buf][1];
#pragma unroll
    for (int k4 = 0; k4 < BK; k4 += 4) {
      S ar[FM], ai[FM], nai[FM], br[FN], bi[FN];
#pragma unroll
      for (int i = 0; i < FM; ++i) {
        int off = (k4 + lk) * AST + wm0 + i * 16 + li;
        ar[i] = Ar[off];
        ai[i] = Ai[off];
        nai[i] = -ai[i];
      }
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        int off = (wn0 + j * 16 + li) * BST + k4 + lk;
        br[j] = Br[off];
        bi[j] = Bi[off];
      }
      if constexpr (G3) {
        S as[FM], bs[FN];
#pragma unroll
        for (int i = 0; i < FM; ++i) as[i] = ar[i] + ai[i];
#pragma unroll
        for (int j = 0; j < FN; ++j) bs[j] = br[j] + bi[j];
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j) {
            acc_re[i][j] = mfma16(ar[i], br[j], acc_re[i][j]);
            acc_im[i][j] = mfma16(ai[i], bi[j], acc_im[i][j]);
            acc_s[i][j] = mfma16(as[i], bs[j], acc_s[i][j]);
          }
      } else {
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j) {
            acc_re[i][j] = mfma16(ar[i], br[j], acc_re[i][j]);
            acc_re[i][j] = mfma16(nai[i], bi[j], acc_re[i][j]);
            acc_im[i][j] = mfma16(ar[i], bi[j], acc_im[i][j]);
            acc_im[i][j] = mfma16(ai[i], br[j], acc_im[i][j]);
          }
      }
    }
  };

  constexpr bool CAHEAD = PF == 1 && FM * FN == 1;
  T cv[FN][4];
  auto load_c = [&](int i) {
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const int gn = n0 + wn0 + j * 16 + li;
      const T* Cj = C + (int64_t)(gn < N ? gn : N - 1) * ldc;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int gm = m0 + wm0 + i * 16 + (sizeof(S) == 8 ? 4 * v + lk : lk * 4 + v);
        const T* p = Cj + (gm < M ? gm : M - 1);
        cv[j][v].re = p->re;
        cv[j][v].im = p->im;
      }
    }
  };
  const int nt = (K + BK - 1) / BK;
  if constexpr (PF == 1) {
    gload(S0{}, 0);
    if constexpr (CAHEAD) load_c(0);
    sstore(S0{}, 0);
    __syncthreads();
    for (int t = 0; t < nt; ++t) {
      const int buf = t & 1;
      if (t + 1 < nt) gload(S0{}, (t + 1) * BK);
      compute(buf);
      if (t + 1 < nt) sstore(S0{}, buf ^ 1);
      __syncthreads();
    }
  } else {
    // k-tile t sits in LDS buffer t & 1 and came through slot t & 1; when it
    // is multiplied, slot t & 1 is free for k-tile t+2 and slot (t+1) & 1
    // holds k-tile t+1, stored to the other buffer at the end of the step.
    gload(S0{}, 0);
    if (nt > 1) gload(S1{}, BK);
    sstore(S0{}, 0);
    __syncthreads();
    auto step = [&](auto P, int t) {
      constexpr int p = decltype(P)::value;
      if (t + 2 < nt) gload(std::integral_constant<int, p>{}, (t + 2) * BK);
      compute(p);
      if (t + 1 < nt) sstore(std::integral_constant<int, 1 - p>{}, 1 - p);
      __syncthreads();
    };
    for (int t = 0; t < nt; t += 2) {
      step(S0{}, t);
      if (t + 1 < nt) step(S1{}, t + 1);
    }
  }
  // C a block row at a time: its loads (at clamped addresses) before its stores,
  // and with one block per wave before the products (32 x 32 tile in an N = 530
  // window: 10.9 -> 9.9 us per launch)
#pragma unroll
  for (int i = 0; i < FM; ++i) {
    if constexpr (!CAHEAD) load_c(i);
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const int gn = n0 + wn0 + j * 16 + li;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int gm = m0 + wm0 + i * 16 + (sizeof(S) == 8 ? 4 * v + lk : lk * 4 + v);
        T c = cv[j][v];
        if constexpr (G3) {
          const S p1 = acc_re[i][j][v], p2 = acc_im[i][j][v];
          c.re += p1 - p2;
          c.im += acc_s[i][j][v] - p1 - p2;
        } else {
          c.re += acc_re[i][j][v];
          c.im += acc_im[i][j][v];
        }
        if (gn < N && gm < M) {
          T* p = C + gm + (int64_t)gn * ldc;
          p->re = c.re;
          p->im = c.im;
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------
// C[b] -= A[b] * B[b] (complex128 on FP64 MFMA, complex64 on FP32 MFMA) with
// the operands streamed from global memory straight into the MFMA operand
// registers: no LDS and no barrier.  Each wave owns a WM x WN tile of C
// (WGM x WGN waves per workgroup share their A rows and B columns through
// L1) and keeps the fragments of the next D k-steps (4-deep each) in flight
// in a register ring.  Lane l holds A[m0 + 16i + l % 16][k + l / 16] and
// B[k + l / 16][n0 + 16j + l % 16]: 16 lanes read one contiguous run of an A
// column, 4 lanes one of a B column.  Gauss's three products as in
// k_gemm_sub (P1 = Ar Br, P2 = Ai Bi, P3 = (Ar + Ai)(Br + Bi)), accumulated
// as +AB and subtracted in the epilogue, the same k order and MFMA as
// k_gemm_sub, so the two give the same bits.  XCD: the tile order of
// k_gemm_sub, with GRP m-tiles per group (2-4 keep the in-flight A and B
// panels of an XCD within its L2).
// ---------------------------------------------------------------------------
template <int I, int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    static_for<I + 1, N>(f);
  }
}

typedef double qb_d2 __attribute__((ext_vector_type(2)));
typedef float qb_f2 __attribute__((ext_vector_type(2)));
template <typename T>
struct RegVec;
template <>
struct RegVec<cd> {
  typedef qb_d2 V2;
};
template <>
struct RegVec<cf> {
  typedef qb_f2 V2;
};

template <typename T, int WM, int WN, int WGM, int WGN, int D, int OCC, bool XCD, int GRP = 8>
__global__ void __launch_bounds__(64 * WGM * WGN, OCC)
    k_gemm_reg(int M, int N, int K, const T* __restrict__ A, int64_t lda, int64_t sA,
               const T* __restrict__ B, int64_t ldb, int64_t sB, T* __restrict__ C,
               int64_t ldc, int64_t sC, const int* __restrict__ bix) {
  typedef typename Scal<T>::S S;
  typedef typename Scal<T>::V4 V4;
  typedef typename RegVec<T>::V2 V2;
  constexpr int FM = WM / 16, FN = WN / 16;
  constexpr int BM = WM * WGM, BN = WN * WGN;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int li = lane & 15, lk = lane >> 4;
  int mt = blockIdx.x, ntile = blockIdx.y;
  if constexpr (XCD) {
    // the XCD-aware tile order of k_gemm_sub, in groups of GRP m-tiles
    xcd_tile(GRP, &mt, &ntile);
  }
  const int m0 = mt * BM + (wave % WGM) * WM, n0 = ntile * BN + (wave / WGM) * WN;
  if (m0 >= M || n0 >= N) return;  // the wave has no rows or columns (no barrier follows)
  const int64_t b = bix ? bix[blockIdx.z] : blockIdx.z;
  A += b * sA;
  B += b * sB;
  C += b * sC;
  // rows, columns and k outside the operands are read at a clamped address
  // (so every load is in bounds and unconditional) and zeroed when used
  const T* Ap[FM];
  const T* Bp[FN];
  bool aok[FM], bok[FN];
#pragma unroll
  for (int i = 0; i < FM; ++i) {
    const int row = m0 + 16 * i + li;
    aok[i] = row < M;
    Ap[i] = A + (aok[i] ? row : M - 1);
  }
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    const int col = n0 + 16 * j + li;
    bok[j] = col < N;
    Bp[j] = B + (int64_t)(bok[j] ? col : N - 1) * ldb;
  }
  const int ns = (K + 3) >> 2;  // k-steps of 4
  V2 ra[D][FM], rb[D][FN];  // (re, im) of the lane's A and B elements, as loaded
  auto load = [&](auto slot, int s) {
    constexpr int d = decltype(slot)::value;
    const int k = 4 * s + lk < K ? 4 * s + lk : K - 1;
#pragma unroll
    for (int i = 0; i < FM; ++i) ra[d][i] = *(const V2*)(Ap[i] + (int64_t)k * lda);
#pragma unroll
    for (int j = 0; j < FN; ++j) rb[d][j] = *(const V2*)(Bp[j] + k);
  };
  V4 p1[FM][FN], p2[FM][FN], p3[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      p1[i][j] = V4{0, 0, 0, 0};
      p2[i][j] = V4{0, 0, 0, 0};
      p3[i][j] = V4{0, 0, 0, 0};
    }
  // k-step s: multiply ring slot s % D, masking rows, columns and k outside
  // the operands
  // (MASK: rows, columns or k of the wave's tile fall outside the operands;
  // interior tiles with K a multiple of 4 multiply the loads as they are)
  auto mult = [&](auto slot, int s, auto mask) {
    constexpr int d = decltype(slot)::value;
    constexpr bool MASK = decltype(mask)::value;
    const bool kok = 4 * s + lk < K;
    S xr[FM], xi[FM], yr[FN], yi[FN], as[FM], bs[FN];
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      const bool ok = !MASK || (aok[i] && kok);
      xr[i] = ok ? ra[d][i].x : S(0);
      xi[i] = ok ? ra[d][i].y : S(0);
      as[i] = xr[i] + xi[i];
    }
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const bool ok = !MASK || (bok[j] && kok);
      yr[j] = ok ? rb[d][j].x : S(0);
      yi[j] = ok ? rb[d][j].y : S(0);
      bs[j] = yr[j] + yi[j];
    }
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        p1[i][j] = mfma16(xr[i], yr[j], p1[i][j]);
        p2[i][j] = mfma16(xi[i], yi[j], p2[i][j]);
        p3[i][j] = mfma16(as[i], bs[j], p3[i][j]);
      }
  };
  // the ring is refilled without conditions (clamped addresses are always
  // valid), so the loop body is straight-line code and the compiler waits
  // only for the slot it is about to multiply
  static_for<0, D>([&](auto slot) { load(slot, decltype(slot)::value); });
  int s0 = 0;
  auto rounds = [&](auto mask) {
    for (; s0 + D <= ns; s0 += D) {
      static_for<0, D>([&](auto slot) {
        mult(slot, s0 + decltype(slot)::value, mask);
        load(slot, s0 + decltype(slot)::value + D);
      });
    }
  };
  const bool interior = m0 + WM <= M && n0 + WN <= N && (K & 3) == 0;  // uniform per wave
  if (interior)
    rounds(std::false_type{});
  else
    rounds(std::true_type{});
  static_for<0, D>([&](auto slot) {
    if (s0 + decltype(slot)::value < ns) mult(slot, s0 + decltype(slot)::value, std::true_type{});
  });
  // C: every load (at clamped addresses) before the first store.  Element by
  // element, behind its bounds, a wave waited sixteen times in a row here: 37.3 ->
  // 34.2 us per launch of an N = 530 window (large updates, where other waves
  // multiply meanwhile, are unchanged).
  V2 cv[FM][FN][4];
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    const int gn = n0 + 16 * j + li;
    const T* Cj = C + (int64_t)(gn < N ? gn : N - 1) * ldc;
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        // result register v of a lane: row 4v + lane/16 (f64), 4(lane/16) + v (f32)
        const int gm = m0 + 16 * i + (sizeof(S) == 8 ? 4 * v + lk : 4 * lk + v);
        cv[i][j][v] = *(const V2*)(Cj + (gm < M ? gm : M - 1));
      }
  }
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    const int gn = n0 + 16 * j + li;
    T* Cj = C + (int64_t)gn * ldc;
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int gm = m0 + 16 * i + (sizeof(S) == 8 ? 4 * v + lk : 4 * lk + v);
        const S q1 = p1[i][j][v], q2 = p2[i][j][v];
        V2 c = cv[i][j][v];
        c.x -= q1 - q2;
        c.y -= p3[i][j][v] - q1 - q2;
        if (gn < N && gm < M) *(V2*)(Cj + gm) = c;
      }
  }
}

template <int WM, int WN, int WGM, int WGN, int D, int OCC, bool XCD, int GRP = 8, typename T = cd>
static void launch_gemm_reg(qb_ctx* ctx, int M, int N, int K, const T* A, int64_t lda,
                            int64_t sA, const T* B, int64_t ldb, int64_t sB, T* C,
                            int64_t ldc, int64_t sC, int batch) {
  constexpr int BM = WM * WGM, BN = WN * WGN;
  dim3 g((M + BM - 1) / BM, (N + BN - 1) / BN, batch);
  hipLaunchKernelGGL((k_gemm_reg<T, WM, WN, WGM, WGN, D, OCC, XCD, GRP>), g, dim3(64 * WGM * WGN), 0,
                     ctx->stream, M, N, K, A, lda, sA, B, ldb, sB, C, ldc, sC, ctx->bix);
}

// OCC: waves per SIMD the register allocation must allow (__launch_bounds__).
template <typename T, int BM, int BN, int BK, int WGM, int WGN, bool XCD = false,
          bool G3 = false, int PF = 1, int OCC = (PF == 2 ? 2 : 1)>
static void launch_gemm(qb_ctx* ctx, int M, int N, int K, const T* A, int64_t lda, int64_t sA,
                        const T* B, int64_t ldb, int64_t sB, T* C, int64_t ldc, int64_t sC,
                        int batch) {
  dim3 g((M + BM - 1) / BM, (N + BN - 1) / BN, batch);
  hipLaunchKernelGGL((k_gemm_sub<T, BM, BN, BK, WGM, WGN, XCD, G3, PF, OCC>), g, dim3(256), 0,
                     ctx->stream, M, N, K, A, lda, sA, B, ldb, sB, C, ldc, sC, ctx->bix);
}

// ---------------------------------------------------------------------------
// complex64 C[b] -= A[b] * B[b] on the bf16 matrix cores
// ---------------------------------------------------------------------------
// Each FP32 operand x is split into three bf16 parts, x = h + m + l with
// h = bf16(x), m = bf16(x - h), l = bf16(x - h - m) (round to nearest; both
// differences are exact in FP32), which keeps 24 significant bits.  A real
// product a b is then the six products h h + h m + m h + h l + m m + l h with
// FP32 accumulation (the dropped m l, l m, l l are below 2^-24 |a b|): the
// accuracy of an FP32 product at 6 bf16 MFMAs (2.5 PFLOP/s dense) instead of
// one FP32 one (157.3 TFLOP/s), i.e. up to 2.7x the FP32 rate.  A complex
// block product is 4 real ones (Re = Ar Br + Ai (-Bi), Im = Ar Bi + Ai Br):
// 24 v_mfma_f32_16x16x32_bf16 per 16 x 16 block and 32-deep k-tile.
//
// Tiles: workgroup BM x BN, k-tile 32, 4 waves WGM x WGN; operands staged in
// LDS as FP32 planes [row][k] (k contiguous, row stride 36 floats: the
// 32-byte fragment reads of 16 lanes cover the 64 banks once) and split into
// bf16 in registers when the fragments are read.  Operand lanes: row / column
// lane % 16, k = 8 (lane / 16) + 0..7 on both sides; result register v of a
// lane holds D[4 (lane / 16) + v][lane % 16].
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ void split3_bf16(const float* x, bf16x8& h, bf16x8& m, bf16x8& l) {
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const __bf16 a = (__bf16)x[e];
    const float r1 = x[e] - (float)a;
    const __bf16 b = (__bf16)r1;
    const float r2 = r1 - (float)b;
    h[e] = a;
    m[e] = b;
    l[e] = (__bf16)r2;
  }
}

__device__ __forceinline__ bf16x8 neg_bf16(bf16x8 v) {
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = -v[e];
  return v;
}

__device__ __forceinline__ floatx4 mfma_bf6(const bf16x8* a, const bf16x8* b, floatx4 c) {
  // a[0..2], b[0..2] = h, m, l: the six products down to 2^-24 (small ones first)
  c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[2], b[0], c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[1], b[1], c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[0], b[2], c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[1], b[0], c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[0], b[1], c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[0], b[0], c, 0, 0, 0);
  return c;
}

template <int BM, int BN, int WGM, int WGN, bool XCD>
__global__ void __launch_bounds__(256, 1) k_gemm_bf6(int M, int N, int K, const cf* __restrict__ A,
                                                     int64_t lda, int64_t sA,
                                                     const cf* __restrict__ B, int64_t ldb,
                                                     int64_t sB, cf* __restrict__ C, int64_t ldc,
                                                     int64_t sC, const int* __restrict__ bix) {
  static_assert(WGM * WGN == 4, "4 waves");
  constexpr int BK = 32, ST = BK + 4;
  constexpr int WM = BM / WGM, WN = BN / WGN;
  constexpr int FM = WM / 16, FN = WN / 16;
  constexpr int NA = BM * BK / 256, NB = BN * BK / 256;
  __shared__ __align__(16) float As[2][2][BM * ST];  // [buf][re/im][m][k]
  __shared__ __align__(16) float Bs[2][2][BN * ST];  // [buf][re/im][n][k]
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm0 = (wave % WGM) * WM, wn0 = (wave / WGM) * WN;
  int mt = blockIdx.x, ntile = blockIdx.y;
  if constexpr (XCD) {
    // the XCD-aware tile order of k_gemm_sub
    xcd_tile(8, &mt, &ntile);
  }
  const int m0 = mt * BM, n0 = ntile * BN;
  const int64_t b = bix ? bix[blockIdx.z] : blockIdx.z;
  A += b * sA;
  B += b * sB;
  C += b * sC;
  const int li = lane & 15, lg = lane >> 4;
  floatx4 acc_re[FM][FN], acc_im[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      acc_re[i][j] = floatx4{0, 0, 0, 0};
      acc_im[i][j] = floatx4{0, 0, 0, 0};
    }
  cf ra[NA], rb[NB];
  const bool full_mn = (m0 + BM <= M) && (n0 + BN <= N);
  auto gload = [&](int k0) {
    if (full_mn && k0 + BK <= K) {
#pragma unroll
      for (int p = 0; p < NA; ++p) {
        const int e = tid + 256 * p, m = e % BM, kk = e / BM;
        ra[p] = A[(m0 + m) + (int64_t)(k0 + kk) * lda];
      }
#pragma unroll
      for (int p = 0; p < NB; ++p) {
        const int e = tid + 256 * p, kk = e % BK, n = e / BK;
        rb[p] = B[(k0 + kk) + (int64_t)(n0 + n) * ldb];
      }
      return;
    }
#pragma unroll
    for (int p = 0; p < NA; ++p) {
      const int e = tid + 256 * p, m = e % BM, kk = e / BM;
      const int gm = m0 + m, gk = k0 + kk;
      ra[p] = (gm < M && gk < K) ? A[gm + (int64_t)gk * lda] : cf{0, 0};
    }
#pragma unroll
    for (int p = 0; p < NB; ++p) {
      const int e = tid + 256 * p, kk = e % BK, n = e / BK;
      const int gn = n0 + n, gk = k0 + kk;
      rb[p] = (gn < N && gk < K) ? B[gk + (int64_t)gn * ldb] : cf{0, 0};
    }
  };
  auto sstore = [&](int buf) {
#pragma unroll
    for (int p = 0; p < NA; ++p) {
      const int e = tid + 256 * p, m = e % BM, kk = e / BM;
      As[buf][0][m * ST + kk] = ra[p].re;
      As[buf][1][m * ST + kk] = ra[p].im;
    }
#pragma unroll
    for (int p = 0; p < NB; ++p) {
      const int e = tid + 256 * p, kk = e % BK, n = e / BK;
      Bs[buf][0][n * ST + kk] = rb[p].re;
      Bs[buf][1][n * ST + kk] = rb[p].im;
    }
  };
  auto compute = [&](int buf) {
    bf16x8 ar[FM][3], ai[FM][3];
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      const int off = (wm0 + 16 * i + li) * ST + 8 * lg;
      float xr[8], xi[8];
      *(float4*)&xr[0] = *(const float4*)&As[buf][0][off];
      *(float4*)&xr[4] = *(const float4*)&As[buf][0][off + 4];
      *(float4*)&xi[0] = *(const float4*)&As[buf][1][off];
      *(float4*)&xi[4] = *(const float4*)&As[buf][1][off + 4];
      split3_bf16(xr, ar[i][0], ar[i][1], ar[i][2]);
      split3_bf16(xi, ai[i][0], ai[i][1], ai[i][2]);
    }
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const int off = (wn0 + 16 * j + li) * ST + 8 * lg;
      float yr[8], yi[8];
      *(float4*)&yr[0] = *(const float4*)&Bs[buf][0][off];
      *(float4*)&yr[4] = *(const float4*)&Bs[buf][0][off + 4];
      *(float4*)&yi[0] = *(const float4*)&Bs[buf][1][off];
      *(float4*)&yi[4] = *(const float4*)&Bs[buf][1][off + 4];
      bf16x8 br[3], bi[3], nbi[3];
      split3_bf16(yr, br[0], br[1], br[2]);
      split3_bf16(yi, bi[0], bi[1], bi[2]);
#pragma unroll
      for (int s = 0; s < 3; ++s) nbi[s] = neg_bf16(bi[s]);
#pragma unroll
      for (int i = 0; i < FM; ++i) {
        acc_re[i][j] = mfma_bf6(ar[i], br, acc_re[i][j]);
        acc_re[i][j] = mfma_bf6(ai[i], nbi, acc_re[i][j]);
        acc_im[i][j] = mfma_bf6(ar[i], bi, acc_im[i][j]);
        acc_im[i][j] = mfma_bf6(ai[i], br, acc_im[i][j]);
      }
    }
  };
  const int nt = (K + BK - 1) / BK;
  gload(0);
  sstore(0);
  __syncthreads();
  for (int t = 0; t < nt; ++t) {
    const int buf = t & 1;
    if (t + 1 < nt) gload((t + 1) * BK);
    compute(buf);
    if (t + 1 < nt) sstore(buf ^ 1);
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const int gn = n0 + wn0 + j * 16 + li;
      if (gn >= N) continue;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int gm = m0 + wm0 + i * 16 + lg * 4 + v;
        if (gm < M) {
          cf* p = C + gm + (int64_t)gn * ldc;
          cf c = *p;
          c.re -= acc_re[i][j][v];
          c.im -= acc_im[i][j][v];
          *p = c;
        }
      }
    }
}

template <int BM, int BN, int WGM, int WGN, bool XCD = false>
static void launch_gemm_bf6(qb_ctx* ctx, int M, int N, int K, const cf* A, int64_t lda,
                            int64_t sA, const cf* B, int64_t ldb, int64_t sB, cf* C, int64_t ldc,
                            int64_t sC, int batch) {
  dim3 g((M + BM - 1) / BM, (N + BN - 1) / BN, batch);
  hipLaunchKernelGGL((k_gemm_bf6<BM, BN, WGM, WGN, XCD>), g, dim3(256), 0, ctx->stream, M, N, K,
                     A, lda, sA, B, ldb, sB, C, ldc, sC, ctx->bix);
}

// Tile variants and the per-context choice.  Variant 0/1 are the defaults
// (wide / narrow N); the autotuner (qb_gemm_tune) may pick another per shape
// class, measured on the device.
typedef void (*gemm_fn_c64)(qb_ctx*, int, int, int, const cf*, int64_t, int64_t, const cf*,
                            int64_t, int64_t, cf*, int64_t, int64_t, int);
typedef void (*gemm_fn_c128)(qb_ctx*, int, int, int, const cd*, int64_t, int64_t, const cd*,
                             int64_t, int64_t, cd*, int64_t, int64_t, int);
static const gemm_fn_c64 kGemmC64[QB_GEMM_VARIANTS] = {
    launch_gemm<cf, 128, 128, 16, 2, 2>,      launch_gemm<cf, 256, 64, 16, 4, 1>,
    launch_gemm<cf, 64, 256, 16, 1, 4>,       launch_gemm<cf, 128, 64, 16, 2, 2>,
    launch_gemm<cf, 128, 128, 32, 2, 2>,      launch_gemm<cf, 128, 64, 16, 2, 2, true>,
    launch_gemm<cf, 128, 128, 16, 2, 2, true>, launch_gemm<cf, 128, 64, 16, 2, 2, false, true>,
    launch_gemm<cf, 128, 128, 16, 2, 2, false, true>, launch_gemm<cf, 128, 64, 16, 2, 2, true, true>,
    launch_gemm<cf, 64, 64, 16, 2, 2, false, true>, launch_gemm<cf, 64, 64, 16, 2, 2, true, true>,
    launch_gemm<cf, 64, 64, 16, 2, 2>,         launch_gemm_bf6<128, 128, 2, 2>,
    launch_gemm_bf6<128, 128, 2, 2, true>,     launch_gemm_bf6<128, 64, 2, 2>,
    launch_gemm_bf6<64, 64, 2, 2>,
    // 17-22: operands streamed into registers, no LDS (k_gemm_reg)
    launch_gemm_reg<32, 32, 4, 1, 8, 2, true, 2, cf>, launch_gemm_reg<32, 64, 2, 2, 6, 2, true, 2, cf>,
    launch_gemm_reg<32, 32, 2, 2, 8, 2, true, 2, cf>, launch_gemm_reg<64, 32, 2, 2, 6, 2, true, 2, cf>,
    launch_gemm_reg<32, 32, 4, 1, 8, 3, true, 2, cf>, launch_gemm_reg<32, 32, 4, 1, 12, 2, true, 2, cf>};
static const gemm_fn_c128 kGemmC128[QB_GEMM_VARIANTS] = {
    launch_gemm<cd, 128, 64, 16, 2, 2>,       launch_gemm<cd, 128, 32, 16, 4, 1>,
    launch_gemm<cd, 64, 64, 16, 2, 2>,        launch_gemm<cd, 64, 128, 16, 2, 2>,
    launch_gemm<cd, 256, 32, 16, 4, 1>,       launch_gemm<cd, 64, 64, 16, 2, 2, true>,
    launch_gemm<cd, 128, 64, 16, 2, 2, true>, launch_gemm<cd, 64, 64, 16, 2, 2, false, true>,
    launch_gemm<cd, 64, 32, 16, 2, 2, false, true>, launch_gemm<cd, 64, 64, 16, 2, 2, true, false, 2>,
    launch_gemm<cd, 64, 32, 16, 2, 2, false, true, 2>, launch_gemm<cd, 64, 64, 16, 2, 2, false, true, 1, 2>,
    launch_gemm<cd, 64, 64, 16, 2, 2, true, true, 2, 2>,
    // 13: the lean tile of the LU panel beside the trailing update (19 KB of
    // LDS; always taken through qb_ctx::panel_lean, and open to the tuner).  No bf16-split
    // counterpart for complex128: the other slots repeat the default and the
    // tuner skips them (kGemmAvail)
    launch_gemm<cd, 32, 32, 8, 2, 2, false, true>, launch_gemm<cd, 64, 64, 8, 2, 2, true, true, 2, 3>,
    launch_gemm<cd, 64, 64, 8, 2, 2, true, true, 1, 4>, launch_gemm<cd, 64, 64, 8, 2, 2, true, true, 1, 3>,
    // 17-20: operands streamed into registers, no LDS (k_gemm_reg).  Wave
    // tiles of 32 x 64 and 64 x 32 at one wave per SIMD were slower: the
    // compiler shuttles their accumulators between AGPRs and VGPRs
    launch_gemm_reg<32, 32, 4, 1, 7, 2, true>, launch_gemm_reg<32, 32, 4, 1, 8, 2, true>,
    launch_gemm_reg<32, 32, 2, 2, 6, 2, true>,
    // 20: 32 x 128 workgroup tile for updates of few rows (the block-row TRSM)
    launch_gemm_reg<32, 32, 1, 4, 7, 2, true>,
    // 21, 22: the 128 x 32 tile in XCD groups of 2 and 4 m-tiles (less of A in L2)
    launch_gemm_reg<32, 32, 4, 1, 7, 2, true, 2>, launch_gemm_reg<32, 32, 4, 1, 7, 2, true, 4>};
static_assert(QB_GEMM_LEAN_C128 == 13, "the lean complex128 tile is variant 13");
static const char* kGemmNames[2][QB_GEMM_VARIANTS] = {
    {"128x128x16", "256x64x16", "64x256x16", "128x64x16", "128x128x32", "128x64x16/xcd",
     "128x128x16/xcd", "128x64x16/3m", "128x128x16/3m", "128x64x16/3m/xcd", "64x64x16/3m", "64x64x16/3m/xcd", "64x64x16",
     "128x128x32/bf16x6", "128x128x32/bf16x6/xcd", "128x64x32/bf16x6", "64x64x32/bf16x6",
     "128x32x4/3m/xcd2/reg/d8", "64x128x4/3m/xcd2/reg/d6", "64x64x4/3m/xcd2/reg/d8",
     "128x64x4/3m/xcd2/reg/d6", "128x32x4/3m/xcd2/reg/d8/occ3", "128x32x4/3m/xcd2/reg/d12"},
    {"128x64x16", "128x32x16", "64x64x16", "64x128x16", "256x32x16", "64x64x16/xcd",
     "128x64x16/xcd", "64x64x16/3m", "64x32x16/3m", "64x64x16/xcd/pf2", "64x32x16/3m/pf2", "64x64x16/3m/o2",
     "64x64x16/3m/xcd/pf2", "32x32x8/3m/lean", "64x64x8/3m/xcd/pf2/occ3", "64x64x8/3m/xcd/occ4",
     "64x64x8/3m/xcd/occ3", "128x32x4/3m/xcd/reg/d7", "128x32x4/3m/xcd/reg/d8",
     "64x64x4/3m/xcd/reg/d6", "32x128x4/3m/xcd/reg/d7", "128x32x4/3m/xcd2/reg/d7",
     "128x32x4/3m/xcd4/reg/d7"}};
// Variants that exist for the type (the tuner times only these).
static const bool kGemmAvail[2][QB_GEMM_VARIANTS] = {
    {true, true, true, true, true, true, true, true, true, true, true, true, true, true, true, true,
     true, true, true, true, true, true, true},
    {true, true, true, true, true, true, true, true, true, true, true, true, true, true, true,
     true, true, true, true, true, true, true, true}};
// Variants on the bf16 matrix cores (three-way bf16 splits of FP32 operands).
static const bool kGemmBf6[2][QB_GEMM_VARIANTS] = {
    {false, false, false, false, false, false, false, false, false, false, false, false, false,
     true, true, true, true, false, false, false, false, false, false},
    {false}};

// Variants built on Gauss's three-product form (3 real MFMA products per
// complex block product instead of 4).
static const bool kGemmG3[2][QB_GEMM_VARIANTS] = {
    {false, false, false, false, false, false, false, true, true, true, true, true, false, false,
     false, false, false, true, true, true, true, true, true},
    {false, false, false, false, false, false, false, true, true, false, true, true, true, true,
     true, true, true, true, true, true, true, true, true}};

// Register-streamed variants (k_gemm_reg: no LDS, no barriers).
static const bool kGemmReg[2][QB_GEMM_VARIANTS] = {
    {false, false, false, false, false, false, false, false, false, false, false, false, false,
     false, false, false, false, true, true, true, true, true, true},
    {false, false, false, false, false, false, false, false, false, false, false, false, false,
     false, false, false, false, true, true, true, true, true, true}};

// Variants that pack 3-4 waves per SIMD (small tiles or k-tiles, low
// register and LDS use): fastest alone, but they leave a concurrently
// running kernel (the lookahead panel) no room on a CU, so gemm_pick_conc
// excludes them.
static const bool kGemmPacks[2][QB_GEMM_VARIANTS] = {
    {false, false, false, false, false, false, false, false, false, false, true, true, true, false,
     false, false, false, false, false, false, false, true, false},
    {false, false, false, false, false, false, false, false, false, false, false, false, false,
     false, true, true, true, false, false, false, false, false, false}};

int qb_gemm_class(int M, int N, int K) {
  int cm = M < 1024 ? 0 : (M < 4096 ? 1 : 2);
  int cn = N <= 32 ? 0 : N <= 64 ? 1 : N <= 256 ? 2 : N <= 1024 ? 3 : 4;
  int ck = K <= 64 ? 0 : K <= 256 ? 1 : 2;
  return (cm * 5 + cn) * 3 + ck;
}

template <typename T>
static int gemm_default(int M, int N, int K, bool conc = false) {
  // the tile a shape gets when the autotuner has not timed its class (the
  // serving loop's windows of many sizes): for complex128 the autotuner's
  // usual picks; complex64 keeps four-product tiles (the three-product form
  // loses about a bit more of FP32 accuracy, which the refinement pays for).
  // Of these the 64 x 64 one, with four workgroups per CU, is the fastest for every
  // shape of a window (32 matrices, 8 M N K per second against the 128 x 128 or
  // 256 x 64 tile): 2816 x 2816 x 256 112 against 85 TFLOP/s, 1536 x 352 x 1536 105
  // against 80, 64 x 352 x 64 28 against 10, 2048 x 32 x 32 25 against 20.  The
  // bits are the same: every tile sums in the order of k.  Beside the lookahead
  // panel (conc) four workgroups leave its leaves no place (610 against 320 us per
  // leaf of N = 3072): there the 128 x 64 tile, 102 TFLOP/s.  A mixed window of 3072,
  // 32 nodes: 140 ms with the 128 x 128 tile, 113 with 64 x 64 everywhere, 104 with both
  // (and with faster norms, 5 ms of the difference).
  (void)M;
  if constexpr (sizeof(T) == sizeof(cf))
    return conc ? 3 : 12;
  else
    return (N <= 32 || K <= 32) ? QB_GEMM_LEAN_C128 : K <= 64 ? 16 : 21;  // 128x32 register tile
}

template <typename T>
static void gemm_launch_variant(qb_ctx* ctx, int v, int M, int N, int K, const T* A, int64_t lda,
                                int64_t sA, const T* B, int64_t ldb, int64_t sB, T* C,
                                int64_t ldc, int64_t sC, int batch) {
  if constexpr (sizeof(T) == sizeof(cf))
    kGemmC64[v](ctx, M, N, K, A, lda, sA, B, ldb, sB, C, ldc, sC, batch);
  else
    kGemmC128[v](ctx, M, N, K, A, lda, sA, B, ldb, sB, C, ldc, sC, batch);
}

template <typename T>
int gemm_sub(qb_ctx* ctx, int M, int N, int K, const T* A, int64_t lda, int64_t sA, const T* B,
             int64_t ldb, int64_t sB, T* C, int64_t ldc, int64_t sC, int batch) {
  if (M <= 0 || N <= 0 || K <= 0 || batch <= 0) return QB_OK;
  const int ty = sizeof(T) == sizeof(cf) ? 0 : 1;
  int v = (ctx->gemm_conc ? ctx->gemm_pick_conc : ctx->gemm_pick)[ty][qb_gemm_class(M, N, K)];
  if (v < 0) v = gemm_default<T>(M, N, K, ctx->gemm_conc);
  if (ty == 1 && ctx->panel_lean) v = QB_GEMM_LEAN_C128;
  return gemm_sub_v<T>(ctx, v, M, N, K, A, lda, sA, B, ldb, sB, C, ldc, sC, batch);
}

template <typename T>
int gemm_sub_v(qb_ctx* ctx, int v, int M, int N, int K, const T* A, int64_t lda, int64_t sA,
               const T* B, int64_t ldb, int64_t sB, T* C, int64_t ldc, int64_t sC, int batch) {
  if (M <= 0 || N <= 0 || K <= 0 || batch <= 0) return QB_OK;
  const int ty = sizeof(T) == sizeof(cf) ? 0 : 1;
  if (v < 0 || v >= QB_GEMM_VARIANTS || !kGemmAvail[ty][v]) v = gemm_default<T>(M, N, K);
  const int kind = ty == 0 ? (kGemmBf6[ty][v] ? QB_K_GEMM_C64_BF16 : QB_K_GEMM_C64) : QB_K_GEMM_C128;
  int slot = qb_prof_begin(ctx, kind, 8.0 * M * N * K * (double)batch,
                           (double)sizeof(T) * ((double)M * K + (double)K * N + 2.0 * M * N) * batch);
  if (ctx->prof)
    ctx->prof_issued[kind] +=
        (kGemmBf6[ty][v] ? 48.0 : kGemmG3[ty][v] ? 6.0 : 8.0) * M * N * K * (double)batch;
  gemm_launch_variant<T>(ctx, v, M, N, K, A, lda, sA, B, ldb, sB, C, ldc, sC, batch);
  qb_prof_end(ctx, slot);
  QB_HIP(ctx, hipGetLastError());
  return QB_OK;
}

// Autotuner: time every variant on synthetic operands of the given shape
// (batch capped so the operands stay below ~1.5 GiB) and keep the fastest
// for the shape's class.  Returns the chosen variant.
__global__ void k_fill_bits(double* p, int64_t n) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 1e-3 * (double)((i * 2654435761ull) % 997) / 997.0;
}

template <typename T>
int qb_gemm_tune(qb_ctx* ctx, int M, int N, int K, int batch, double* best_tflops) {
  const int ty = sizeof(T) == sizeof(cf) ? 0 : 1;
  size_t per = ((size_t)M * K + (size_t)K * N + (size_t)M * N) * sizeof(T);
  int b = batch;
  while (b > 1 && per * b > ((size_t)3 << 29)) --b;
  T *A = nullptr, *B = nullptr, *C = nullptr;
  int rc = qb_dev_alloc(ctx, (void**)&A, (size_t)M * K * b * sizeof(T));
  if (!rc) rc = qb_dev_alloc(ctx, (void**)&B, (size_t)K * N * b * sizeof(T));
  if (!rc) rc = qb_dev_alloc(ctx, (void**)&C, (size_t)M * N * b * sizeof(T));
  int best = gemm_default<T>(M, N, K), best_conc = best;
  double best_ms = 1e300, best_conc_ms = 1e300;
  if (!rc) {
    int64_t na = (int64_t)M * K * b * sizeof(T) / 8, nb = (int64_t)K * N * b * sizeof(T) / 8,
            nc = (int64_t)M * N * b * sizeof(T) / 8;
    hipLaunchKernelGGL(k_fill_bits, dim3((na + 255) / 256), dim3(256), 0, ctx->stream, (double*)A, na);
    hipLaunchKernelGGL(k_fill_bits, dim3((nb + 255) / 256), dim3(256), 0, ctx->stream, (double*)B, nb);
    hipLaunchKernelGGL(k_fill_bits, dim3((nc + 255) / 256), dim3(256), 0, ctx->stream, (double*)C, nc);
    hipEvent_t e0 = nullptr, e1 = nullptr;
    (void)hipEventCreate(&e0);
    (void)hipEventCreate(&e1);
    // QB_TUNE_SKIP (both operand types), QB_TUNE_SKIP_C64, QB_TUNE_SKIP_C128:
    // comma-separated variant indices the tuner leaves out (a diagnostic for
    // comparing tile families in whole windows)
    std::vector<char> skip(QB_GEMM_VARIANTS, 0);
    for (const char* env : {"QB_TUNE_SKIP", ty == 0 ? "QB_TUNE_SKIP_C64" : "QB_TUNE_SKIP_C128"}) {
      const char* sk = getenv(env);
      for (const char* c = sk; c && *c;) {
        char* end = nullptr;
        const long v = strtol(c, &end, 10);
        if (end == c) {
          ++c;
          continue;
        }
        if (v >= 0 && v < QB_GEMM_VARIANTS) skip[v] = 1;
        c = end;
      }
    }
    for (int v = 0; v < QB_GEMM_VARIANTS; ++v) {
      if (skip[v] || !kGemmAvail[ty][v]) continue;
      gemm_launch_variant<T>(ctx, v, M, N, K, A, M, (int64_t)M * K, B, K, (int64_t)K * N, C, M,
                             (int64_t)M * N, b);
      (void)hipEventRecord(e0, ctx->stream);
      for (int it = 0; it < 3; ++it)
        gemm_launch_variant<T>(ctx, v, M, N, K, A, M, (int64_t)M * K, B, K, (int64_t)K * N, C, M,
                               (int64_t)M * N, b);
      (void)hipEventRecord(e1, ctx->stream);
      (void)hipEventSynchronize(e1);
      float ms = 0.f;
      if (hipGetLastError() == hipSuccess && hipEventElapsedTime(&ms, e0, e1) == hipSuccess &&
          ms > 0.f) {
        if (ms < best_ms) {
          best_ms = ms;
          best = v;
        }
        if (!kGemmPacks[ty][v] && ms < best_conc_ms) {
          best_conc_ms = ms;
          best_conc = v;
        }
      }
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    const int cls = qb_gemm_class(M, N, K);
    if (ctx->gemm_pick[ty][cls] != best || ctx->gemm_pick_conc[ty][cls] != best_conc)
      ++ctx->gemm_epoch;
    ctx->gemm_pick[ty][cls] = best;
    ctx->gemm_pick_conc[ty][cls] = best_conc;
  }
  (void)hipStreamSynchronize(ctx->stream);
  qb_dev_free(ctx, A, (size_t)M * K * b * sizeof(T));
  qb_dev_free(ctx, B, (size_t)K * N * b * sizeof(T));
  qb_dev_free(ctx, C, (size_t)M * N * b * sizeof(T));
  if (best_tflops) *best_tflops = best_ms < 1e299 ? 8.0 * M * N * (double)K * b * 3 / (best_ms * 1e-3) / 1e12 : 0;
  return rc ? rc : best;
}

const char* qb_gemm_variant_name(int ty, int v) {
  return (ty >= 0 && ty < 2 && v >= 0 && v < QB_GEMM_VARIANTS) ? kGemmNames[ty][v] : "?";
}

__device__ __forceinline__ double fma_(double a, double b, double c) {
  return __builtin_fma(a, b, c);
}
__device__ __forceinline__ float fma_(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
// Explicit fused operations: every kernel that forms these rounds alike.
template <typename T>
__device__ __forceinline__ T cmul_(T a, T b) {
  return T{fma_(a.re, b.re, -(a.im * b.im)), fma_(a.re, b.im, a.im * b.re)};
}
// conj(a) / |a|^2
template <typename T>
__device__ __forceinline__ T cinv_(T a) {
  const auto den = fma_(a.re, a.re, a.im * a.im);
  return T{a.re / den, -a.im / den};
}
// x -= a y: the product first, so that a term rounds the running value once.  Four
// multiply-adds into x would round it twice: rms backward error of a 32-row solve
// 0.089 against 0.076 u |L||U||x|, of a 32-column LU 5.2 against 4.7 u.
template <typename T>
__device__ __forceinline__ void cnma_(T& x, const T& a, const T& y) {
  const T p = cmul_(a, y);
  x.re -= p.re;
  x.im -= p.im;
}
// x -= sum a[u] y[u] of U terms, summed first: x rounds once for all of them, and the
// terms take 4 U + 2 operations instead of 6 U (0.070 and 4.6 u where the leaves use it;
// windows of 530 to 1792 nodes 1 to 2 % faster than with every term by itself).
template <int U, typename T>
__device__ __forceinline__ void cnma_sum_(T& x, const T* a, const T* y) {
  T p = cmul_(a[0], y[0]);
#pragma unroll
  for (int u = 1; u < U; ++u) {
    p.re = fma_(-a[u].im, y[u].im, fma_(a[u].re, y[u].re, p.re));
    p.im = fma_(a[u].im, y[u].re, fma_(a[u].re, y[u].im, p.im));
  }
  x.re -= p.re;
  x.im -= p.im;
}

// A[i] when ok, else 0, loaded component by component (a conditional
// aggregate load can leave a per-thread temporary in memory, which the
// compiler then places in LDS, 16 bytes per thread of the workgroup).
template <typename T>
__device__ __forceinline__ T ld_or0(const T* p, bool ok) {
  T v{0, 0};
  if (ok) {
    v.re = p->re;
    v.im = p->im;
  }
  return v;
}

// Workgroup barrier that orders LDS only: outstanding global loads and stores
// stay in flight across it.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// One step of a wave maximum: max(x, x of the lane that the DPP control names),
// x itself where there is none.
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_max(double x) {
  const int lo = __double2loint(x), hi = __double2hiint(x);
  const int l2 = __builtin_amdgcn_update_dpp(lo, lo, CTRL, ROWS, 0xf, false);
  const int h2 = __builtin_amdgcn_update_dpp(hi, hi, CTRL, ROWS, 0xf, false);
  return __builtin_fmax(x, __hiloint2double(h2, l2));
}
template <int CTRL, int ROWS>
__device__ __forceinline__ float dpp_max(float x) {
  const int i = __float_as_int(x);
  const int o = __builtin_amdgcn_update_dpp(i, i, CTRL, ROWS, 0xf, false);
  return __builtin_fmaxf(x, __int_as_float(o));
}
__device__ __forceinline__ double lane_value(double x, int l) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(x), l),
                          __builtin_amdgcn_readlane(__double2loint(x), l));
}
__device__ __forceinline__ float lane_value(float x, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), l));
}
// Maximum over the wave's 64 lanes (x holds no NaN): row shifts by 1, 2, 4 and
// 8, then the row broadcasts; lane 63 holds the result.
template <typename S>
__device__ __forceinline__ S wave_max(S x) {
  x = dpp_max<0x111, 0xf>(x);
  x = dpp_max<0x112, 0xf>(x);
  x = dpp_max<0x114, 0xf>(x);
  x = dpp_max<0x118, 0xf>(x);
  x = dpp_max<0x142, 0xa>(x);
  x = dpp_max<0x143, 0xc>(x);
  return lane_value(x, 63);
}

// The row whose content stands in row x after the interchanges (k0 + k, p[k]),
// k = kb .. np-1, applied in order: x traced back through them.
__device__ __forceinline__ int swap_source(int x, int k0, const int* p, int kb, int np) {
  for (int k = np - 1; k >= kb; --k) {
    const int pk = p[k], ck = k0 + k;
    x = x == pk ? ck : (x == ck ? pk : x);
  }
  return x;
}

// ---------------------------------------------------------------------------
// Leaf panel factorisation: columns [c0, c0+w) of rows [c0, n), w <= 32, one
// workgroup of NT threads per matrix.  The columns are taken W at a time and
// held in registers, RPT rows per thread (RPT * NT >= n - c0, RPT * W = 32
// for complex128, 64 for complex64: 128 VGPRs), so a column step touches no
// global memory on its critical path: the pivot search on max |re|+|im|
// (LAPACK's izamax measure, first row of the maximum) is a DPP maximum per
// wave and one LDS candidate per wave (its row with it), and
// the rank-1 update stays in registers (shifting the columns left by one, so
// that the current column is always the first).  Finished columns of L and
// rows of U are stored as they come.  The interchanges of the W steps reach
// the other columns of the leaf at the end of the sub-block, all at once: each
// affected row is traced back to its source (swap_source), loaded, and stored
// after a barrier.  Before its steps a sub-block takes the update with the s
// columns of L before it (each read once per sub-block).  A zero pivot leaves
// the column unscaled and counts in info, the behaviour of zgetf2 behind
// lu!(check=false).
//
// What bounds it: the latency of 32 column steps (one LDS barrier each) and of
// 32/W changes of sub-block, and with many rows the L2 bandwidth of one CU, which
// reads 32/W * 16 columns.  Four waves of 256 VGPRs (half a CU) find room beside
// a trailing-update workgroup that ends; eight wait for both of a CU's, unless the
// update leaves places often (qb_panel_leaf_form).  Per leaf of N = 530 and N = 1792
// windows (32 matrices), on average: 91 and 94 us (up to 512 rows), 107 (1024) and 179
// (2048); with the columns in global memory (k_getf2_long's order) 172 and 254 us.
// ---------------------------------------------------------------------------
template <typename T, int NT, int RPT, int W>
__global__ void __launch_bounds__(NT) k_getf2(T* __restrict__ A, int64_t lda, int64_t sA, int n,
                                               int c0, int w, int* __restrict__ ipiv, int64_t sP,
                                               int* __restrict__ info) {
  typedef typename Scal<T>::S S;
  constexpr int NWV = NT / 64;
  constexpr int PH = W >= 16 ? 8 : (W == 8 ? 4 : W);  // steps per phase: the columns still live
  __shared__ T Lt[32][33];   // Lt[i][k] = L(c0 + i, c0 + k), k < i
  __shared__ T Us[32][W];    // U(c0 + i, c0 + s + k)
  // of alternate steps: each wave's candidate (value, row, the row itself) and
  // the row that the pivot row replaces
  __shared__ T cand[2][NWV][W], crow[2][W];
  __shared__ S red_v[2][NWV];
  __shared__ int red_i[2][NWV];
  __shared__ int piv[32];
  const int64_t b = blockIdx.x;
  A += b * sA + (int64_t)c0 * lda;  // column cc of the leaf at A + cc * lda
  ipiv += b * sP;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  for (int s = 0; s < w; s += W) {
    const int nw = w - s < W ? w - s : W;
    const int r0 = c0 + s + tid;  // own rows r0 + q * NT
    unsigned ro[RPT];             // clamped to the last row: loads are unconditional
#pragma unroll
    for (int q = 0; q < RPT; ++q) ro[q] = r0 + q * NT < n ? r0 + q * NT : n - 1;
    T a[RPT][W];
#pragma unroll
    for (int k = 0; k < W; ++k)
#pragma unroll
      for (int q = 0; q < RPT; ++q) {
        a[q][k] = T{0, 0};
        if (k < nw) {
          const T* p = A + (int64_t)(s + k) * lda + ro[q];
          a[q][k].re = p->re;
          a[q][k].im = p->im;
        }
      }
    if (W < 32 && s > 0) {
      // U part of the sub-block's columns: one wave per column, a row per lane
      for (int k = wv; k < W; k += NWV) {
        T* Ac = A + c0 + (int64_t)(s + k) * lda;
        T x = ld_or0(Ac + lane, lane < s && k < nw);
        for (int i = 0; i + 1 < s; ++i) {
          const T xi = T{lane_value(x.re, i), lane_value(x.im, i)};
          if (lane > i && lane < s) {
            const T l = Lt[lane][i];
            cnma_(x, l, xi);
          }
        }
        if (lane < s) {
          Us[lane][k] = x;
          if (k < nw) Ac[lane] = x;
        }
      }
      lds_barrier();
      // rows below: a -= L(:, 0..s-1) U
      // UN terms summed before they reach a, QC rows at a time: as many as registers allow
      constexpr int UN = W >= 8 || (W == 4 && NT == 256) ? 4 : 2;
      constexpr int QC = W >= 8 && sizeof(S) == 8 ? 2 : RPT < 4 ? RPT : 4;
#pragma unroll
      for (int q0 = 0; q0 < RPT; q0 += QC) {
        int i = 0;
        for (; i + UN <= s; i += UN) {
          T l[QC][UN];
#pragma unroll
          for (int u = 0; u < UN; ++u)
#pragma unroll
            for (int q = 0; q < QC; ++q) {
              const T* p = A + (int64_t)(i + u) * lda + ro[q0 + q];
              l[q][u].re = p->re;
              l[q][u].im = p->im;
            }
#pragma unroll
          for (int k = 0; k < W; ++k) {
            // U read a column at a time: few registers
            if (k * UN % 4 == 0) asm volatile("" ::: "memory");
            T uk[UN];
#pragma unroll
            for (int u = 0; u < UN; ++u) uk[u] = Us[i + u][k];
#pragma unroll
            for (int q = 0; q < QC; ++q) cnma_sum_<UN>(a[q0 + q][k], l[q], uk);
          }
        }
        for (; i < s; ++i)
#pragma unroll
          for (int q = 0; q < QC; ++q) {
            const T* p = A + (int64_t)i * lda + ro[q0 + q];
            const T lq = T{p->re, p->im};
#pragma unroll
            for (int k = 0; k < W; ++k) cnma_(a[q0 + q][k], lq, Us[i][k]);
          }
      }
    }
    // the column steps; phase p works on the LIVE columns that may be left
    static_for<0, W / PH>([&](auto phase) {
      constexpr int P = decltype(phase)::value, LIVE = W - P * PH;
      for (int j = P * PH; j < (P + 1) * PH && j < nw; ++j) {
        const int c = s + j, row = c0 + c;
        S best = -1;
        int bi = n;
#pragma unroll
        for (int q = 0; q < RPT; ++q) {
          const int r = r0 + q * NT;
          const S v = fabs(a[q][0].re) + fabs(a[q][0].im);
          if (r >= row && r < n && v > best) {
            best = v;
            bi = r;
          }
        }
        const S wm = wave_max(best);
        unsigned long long at = __ballot(best == wm);
        int wi = __builtin_amdgcn_readlane(bi, __ffsll(at) - 1);
        for (at &= at - 1; at; at &= at - 1) {  // ties: the smallest row
          const int o = __builtin_amdgcn_readlane(bi, __ffsll(at) - 1);
          wi = o < wi ? o : wi;
        }
        const int par = j & 1;
        if (lane == 0) {
          red_v[par][wv] = wm;
          red_i[par][wv] = wi;
        }
        if (tid == j) {
#pragma unroll
          for (int k = 0; k < LIVE; ++k) crow[par][k] = a[0][k];
        }
#pragma unroll
        for (int q = 0; q < RPT; ++q)
          if (r0 + q * NT == wi) {
#pragma unroll
            for (int k = 0; k < LIVE; ++k) cand[par][wv][k] = a[q][k];
          }
        lds_barrier();
        S bv = red_v[par][0];
        int p = red_i[par][0], pw = 0;
#pragma unroll
        for (int q = 1; q < NWV; ++q) {
          const S v = red_v[par][q];
          const int i = red_i[par][q];
          if (v > bv || (v == bv && i < p)) {
            bv = v;
            p = i;
            pw = q;
          }
        }
        pw = __builtin_amdgcn_readfirstlane(pw);
        // no candidate (a column of NaN): the row stays
        const T* prow = p < n ? cand[par][pw] : crow[par];
        if (p >= n) p = row;
        if (tid == 0) {
          ipiv[row] = p;
          piv[c] = p;
        }
        if (p != row) {
#pragma unroll
          for (int q = 0; q < RPT; ++q)
            if (r0 + q * NT == p) {
#pragma unroll
              for (int k = 0; k < LIVE; ++k) a[q][k] = crow[par][k];
            }
        }
        if (tid < nw - j) A[row + (int64_t)(c + tid) * lda] = prow[tid];
        const T pv = prow[0];
        const bool nz = pv.re != 0 || pv.im != 0;
        if (!nz && tid == 0 && info) atomicCAS(info + b, 0, row + 1);
        const T inv = cinv_(pv);
        T l[RPT];
#pragma unroll
        for (int q = 0; q < RPT; ++q) {
          l[q] = nz ? cmul_(a[q][0], inv) : a[q][0];
          const int r = r0 + q * NT;
          if (r > row && r < n) {
            T* d = A + (int64_t)c * lda + (unsigned)r;
            d->re = l[q].re;
            d->im = l[q].im;
          }
        }
#pragma unroll
        for (int k = 1; k < LIVE; ++k) {
          const T u = prow[k];
#pragma unroll
          for (int q = 0; q < RPT; ++q) {
            T x = a[q][k];
            cnma_(x, l[q], u);
            a[q][k - 1] = x;
          }
        }
      }
    });
    // the sub-block's interchanges in the other columns of the leaf, and in its
    // own finished columns from the step after each
    __syncthreads();
    constexpr int NI = 64 * W > NT ? 64 * W / NT : 1;
    T v[NI];
    int64_t dst[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int e = tid + i * NT, t = e % (2 * W), cc = e / (2 * W);
      const int k = t < W ? t : t - W;
      dst[i] = -1;
      if (cc < w && k < nw) {
        const int x = t < W ? c0 + s + k : piv[s + k];
        const int kb = cc >= s && cc < s + nw ? cc - s + 1 : 0;
        const int y = swap_source(x, c0 + s, piv + s, kb, nw);
        if (y != x) {
          dst[i] = x + (int64_t)cc * lda;
          const T* p = A + y + (int64_t)cc * lda;
          v[i].re = p->re;
          v[i].im = p->im;
        }
      }
    }
    __builtin_amdgcn_s_waitcnt(0);  // every load has returned before the first store
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NI; ++i)
      if (dst[i] >= 0) {
        A[dst[i]].re = v[i].re;
        A[dst[i]].im = v[i].im;
      }
    __syncthreads();
    if (W < 32 && s + W < w) {
      for (int e = tid; e < W * 32; e += NT) {
        const int i = s + e / 32, k = e % 32;
        if (k < i) Lt[i][k] = A[c0 + i + (int64_t)k * lda];
      }
      __syncthreads();
    }
  }
}

template <typename T, int NT, int RPT, int W>
static void launch_getf2(qb_ctx* ctx, T* A, int64_t lda, int64_t sA, int n, int c0, int w,
                         int* ipiv, int64_t sP, int* info, int batch) {
  hipLaunchKernelGGL((k_getf2<T, NT, RPT, W>), dim3(batch), dim3(NT), 0, ctx->stream, A, lda, sA, n,
                     c0, w, ipiv, sP, info);
}

// The same leaf for columns too long for registers: left-looking (Crout) order with
// the columns in global memory.  Step c forms the U part of column c by forward
// substitution with the unit-lower top block kept in LDS, updates the rest of
// column c with all previous L columns at once, picks the pivot, swaps the pivot row
// into place across the w columns and scales the column.
template <typename T>
__global__ void __launch_bounds__(512) k_getf2_long(T* __restrict__ A, int64_t lda, int64_t sA,
                                                    int n, int c0, int w, int* __restrict__ ipiv,
                                                    int64_t sP, int* __restrict__ info) {
  typedef typename Scal<T>::S S;
  __shared__ T Lt[32][33];  // Lt[j][k] = L(c0 + j, c0 + k), k < j
  __shared__ T u[32];       // U(c0 + k, col), k < c
  __shared__ T prow[32];
  __shared__ S red_v[16];
  __shared__ int red_i[16];
  __shared__ int s_piv;
  const int64_t b = blockIdx.x;
  A += b * sA;
  ipiv += b * sP;
  const int tid = threadIdx.x, nt = blockDim.x;
  const int lane = tid & 63, wv = tid >> 6;
  const T* L0 = A + (int64_t)c0 * lda;  // first panel column
  for (int c = 0; c < w; ++c) {
    const int col = c0 + c;
    T* Ac = A + (int64_t)col * lda;
    // (1) U(c0 + k, col) = L11^{-1} A(c0.., col), k < c, on wave 0
    if (wv == 0) {
      T a = ld_or0(Ac + c0 + lane, lane < c);
      for (int k = 0; k < c; ++k) {
        T uk = T{__shfl(a.re, k), __shfl(a.im, k)};
        if (lane > k && lane < c) {
          T l = Lt[lane][k];
          a.re -= l.re * uk.re - l.im * uk.im;
          a.im -= l.re * uk.im + l.im * uk.re;
        }
      }
      if (lane < c) {
        u[lane] = a;
        Ac[c0 + lane] = a;
      }
    }
    __syncthreads();
    // (2) rows col..n-1: A(r, col) -= sum_k L(r, c0 + k) U(c0 + k, col); pivot search
    S best = -1;
    int bi = n;
    for (int r = col + tid; r < n; r += 2 * nt) {
      const int r2 = r + nt;
      const bool two = r2 < n;
      T a0 = Ac[r];
      T a1 = ld_or0(Ac + r2, two);
      const T* Lr0 = L0 + r;
      int k = 0;
      for (; k + 4 <= c; k += 4) {
        T l[4], m[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          l[q] = Lr0[(int64_t)(k + q) * lda];
          m[q] = ld_or0(Lr0 + (int64_t)(k + q) * lda + nt, two);
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          T uk = u[k + q];
          a0.re -= l[q].re * uk.re - l[q].im * uk.im;
          a0.im -= l[q].re * uk.im + l[q].im * uk.re;
          a1.re -= m[q].re * uk.re - m[q].im * uk.im;
          a1.im -= m[q].re * uk.im + m[q].im * uk.re;
        }
      }
      for (; k < c; ++k) {
        T uk = u[k];
        T l = Lr0[(int64_t)k * lda];
        T m = ld_or0(Lr0 + (int64_t)k * lda + nt, two);
        a0.re -= l.re * uk.re - l.im * uk.im;
        a0.im -= l.re * uk.im + l.im * uk.re;
        a1.re -= m.re * uk.re - m.im * uk.im;
        a1.im -= m.re * uk.im + m.im * uk.re;
      }
      Ac[r] = a0;
      S v0 = fabs(a0.re) + fabs(a0.im);
      if (v0 > best) {
        best = v0;
        bi = r;
      }
      if (two) {
        Ac[r2] = a1;
        S v1 = fabs(a1.re) + fabs(a1.im);
        if (v1 > best) {
          best = v1;
          bi = r2;
        }
      }
    }
    for (int off = 32; off >= 1; off >>= 1) {
      S ob = __shfl_xor(best, off);
      int oi = __shfl_xor(bi, off);
      if (ob > best || (ob == best && oi < bi)) {
        best = ob;
        bi = oi;
      }
    }
    if (lane == 0) {
      red_v[wv] = best;
      red_i[wv] = bi;
    }
    __syncthreads();
    if (tid == 0) {
      S bv = red_v[0];
      int bix = red_i[0];
      for (int q = 1; q < (nt + 63) / 64; ++q)
        if (red_v[q] > bv || (red_v[q] == bv && red_i[q] < bix)) {
          bv = red_v[q];
          bix = red_i[q];
        }
      if (bix >= n) bix = col;
      s_piv = bix;
      ipiv[col] = bix;
    }
    __syncthreads();
    const int piv = s_piv;
    // (3) swap rows col and piv across the w panel columns; the pivot row's
    // L part becomes row c of the top block
    for (int cc = tid; cc < w; cc += nt) {
      T* Acc = A + (int64_t)(c0 + cc) * lda;
      // component by component: a struct copy here keeps x in memory (16
      // bytes of LDS per thread once the compiler promotes it)
      T x;
      x.re = Acc[piv].re;
      x.im = Acc[piv].im;
      if (piv != col) {
        const auto yr = Acc[col].re, yi = Acc[col].im;
        Acc[piv].re = yr;
        Acc[piv].im = yi;
        Acc[col].re = x.re;
        Acc[col].im = x.im;
      }
      prow[cc] = x;
      if (cc < c) Lt[c][cc] = x;
    }
    __syncthreads();
    // (4) scale the column below the pivot
    const T p = prow[c];
    const bool nz = (p.re != 0 || p.im != 0);
    if (!nz && tid == 0 && info) atomicCAS(info + b, 0, col + 1);
    if (nz) {
      S den = p.re * p.re + p.im * p.im;
      T inv = T{p.re / den, -p.im / den};
      for (int r = col + 1 + tid; r < n; r += nt) Ac[r] = cmul_(Ac[r], inv);
    }
    __syncthreads();
  }
}

// Row interchanges ipiv[k0..k0+np) applied in order to columns [cb, ce)
// (LAPACK zlaswp).  Every workgroup first turns them into the list of rows
// that change and their sources: each affected row (the np rows from k0 on and
// the pivot rows below them) is traced back through the interchanges by a
// thread of its own.  It then moves its cpw columns, up to eight rows per
// thread at a time: load all, barrier, store all.  P2 lanes (the next power of
// two of the list's length, at most 256) take one column.  What bounds it: for
// few interchanges the latency of one load and one store, where the kernel it
// replaces (one lane per column, swap after swap) paid a round trip per
// interchange; for many, the memory lines of the pivot rows, of which each
// column uses 16 bytes.  Measured, per launch of an N = 530, 1792 and 8192 window
// on average: 5.7, 12 and 19 us against 9.2, 25 and 68 us.
template <typename T>
__global__ void __launch_bounds__(256) k_laswp(T* __restrict__ A, int64_t lda, int64_t sA, int cb,
                                               int ce, int k0, int np,
                                               const int* __restrict__ ipiv, int64_t sP,
                                               int cpw) {
  extern __shared__ int sm_swap[];
  int* ip = sm_swap;         // [np]
  int* rdst = ip + np;       // [2 np]
  int* rsrc = rdst + 2 * np;  // [2 np]
  __shared__ int s_nm;
  const int64_t b = blockIdx.y;
  const int tid = threadIdx.x;
  A += b * sA;
  ipiv += b * sP;
  if (tid == 0) s_nm = 0;
  for (int i = tid; i < np; i += 256) ip[i] = ipiv[k0 + i];
  __syncthreads();
  for (int t = tid; t < 2 * np; t += 256) {
    const int x = t < np ? k0 + t : ip[t - np];
    if (t >= np && x < k0 + np) continue;  // listed among the first np
    const int y = swap_source(x, k0, ip, 0, np);
    if (y != x) {
      const int at = atomicAdd(&s_nm, 1);
      rdst[at] = x;
      rsrc[at] = y;
    }
  }
  __syncthreads();
  const int nm = s_nm;
  if (nm == 0) return;  // uniform: no row changes
  int p2 = 16;
  while (p2 < nm && p2 < 256) p2 <<= 1;
  int nr = 1;  // rounds of 256 rows per column, a power of two (8 from 1025 rows on)
  while (nr < 8 && nr * p2 < nm) nr <<= 1;
  const int cols = 256 / p2, sub = tid / p2, l0 = tid & (p2 - 1), ng = 8 / nr;
  const int c_end = min(ce, cb + ((int)blockIdx.x + 1) * cpw);
  for (int c0 = cb + blockIdx.x * cpw; c0 < c_end; c0 += cols * ng) {
    T v[8];
    int64_t dst[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int idx = (u & (nr - 1)) * p2 + l0, c = c0 + (u / nr) * cols + sub;
      dst[u] = -1;
      if (idx < nm && c < c_end) {
        const T* p = A + rsrc[idx] + (int64_t)c * lda;
        v[u].re = p->re;
        v[u].im = p->im;
        dst[u] = rdst[idx] + (int64_t)c * lda;
      }
    }
    __builtin_amdgcn_s_waitcnt(0);  // every load has returned before the first store
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (dst[u] >= 0) {
        A[dst[u]].re = v[u].re;
        A[dst[u]].im = v[u].im;
      }
  }
}

// Broadcast of lane G (0..3) of each group of four lanes.
template <int G>
__device__ __forceinline__ int quad_bcast(int x) {
  return __builtin_amdgcn_update_dpp(0, x, G * 0x55, 0xf, 0xf, true);
}
template <int G>
__device__ __forceinline__ double quad_bcast(double x) {
  return __hiloint2double(quad_bcast<G>(__double2hiint(x)), quad_bcast<G>(__double2loint(x)));
}
template <int G>
__device__ __forceinline__ float quad_bcast(float x) {
  return __int_as_float(quad_bcast<G>(__float_as_int(x)));
}

// ---------------------------------------------------------------------------
// Triangular-solve leaf, n <= 32 rows: X = L^{-1} B (unit lower) or X = U^{-1} B
// (upper).  Four lanes per column (64 columns per workgroup of 256 threads): lane g
// holds the rows 4 s + g, s < 8, in registers, a solved row reaches the other three by
// a DPP quad broadcast, and the triangle stands in LDS (17 KB).  All loads of a lane
// are issued before the first is used.  What bounds it is latency: one load, the chain
// of 32 rows, one store: 6.2 us for the 32 x 64 leaves of an N = 530 window's solves, 8
// us for the upper ones (a lane per column, staged through LDS: 28 us).  With thousands
// of right-hand sides (the LU's block rows) it beats a whole column per lane as well
// (LU of 240 matrices of 1640: 113.3 against 115.6 ms per window, of 48 of 8192: 1.228
// against 1.238 s).
// ---------------------------------------------------------------------------
template <typename T, bool UNIT_LOWER>
__global__ void __launch_bounds__(256, 4) k_trsm_leaf(int n, int nrhs, const T* __restrict__ L,
                                                   int64_t ldl, int64_t sL, T* __restrict__ B,
                                                   int64_t ldb, int64_t sB,
                                                   const int* __restrict__ bix) {
  __shared__ T Ls[32][33];
  const int64_t b = bix ? bix[blockIdx.y] : blockIdx.y;
  const int tid = threadIdx.x, g = tid & 3, col = blockIdx.x * 64 + (tid >> 2);
  L += b * sL;
  B += b * sB + (int64_t)(col < nrhs ? col : nrhs - 1) * ldb;
  T v[8], l[4];
#pragma unroll
  for (int s = 0; s < 8; ++s) v[s] = ld_or0(B + 4 * s + g, 4 * s + g < n);
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const int i = (tid + 256 * t) & 31, j = (tid + 256 * t) >> 5;
    l[t] = ld_or0(L + i + (int64_t)j * ldl, i < n && j < n);
  }
#pragma unroll
  for (int t = 0; t < 4; ++t) Ls[(tid + 256 * t) & 31][(tid + 256 * t) >> 5] = l[t];
  __syncthreads();
  if (UNIT_LOWER) {
    // four rows at a time: among themselves, then in the rows below at once
    static_for<0, 8>([&](auto ss) {
      constexpr int s0 = decltype(ss)::value;
      T x[4];
      static_for<0, 4>([&](auto oo) {
        constexpr int o = decltype(oo)::value;
        x[o] = T{quad_bcast<o>(v[s0].re), quad_bcast<o>(v[s0].im)};
        if constexpr (o < 3) {
          T t = v[s0];  // selected, not branched over: the updates stay in one block
          cnma_(t, Ls[4 * s0 + g][4 * s0 + o], x[o]);
          v[s0].re = g > o ? t.re : v[s0].re;
          v[s0].im = g > o ? t.im : v[s0].im;
        }
      });
#pragma unroll
      for (int s = s0 + 1; s < 8; ++s) {
        const T l[4] = {Ls[4 * s + g][4 * s0], Ls[4 * s + g][4 * s0 + 1], Ls[4 * s + g][4 * s0 + 2],
                        Ls[4 * s + g][4 * s0 + 3]};
        cnma_sum_<4>(v[s], l, x);
        if (s & 1) asm volatile("" ::: "memory");  // LDS reads of two slots at a time
      }
    });
  } else {
    if (tid < 32) {
      const T d = tid < n ? Ls[tid][tid] : T{1, 0};
      Ls[tid][tid] = cinv_(d);
    }
    __syncthreads();
    // blocks of 8 rows from the bottom: first the solved rows below the block
    // in ascending order, then the block's own rows
    static_for<0, 4>([&](auto bb) {
      constexpr int ib = 24 - 8 * decltype(bb)::value, s0 = ib >> 2;
      static_for<s0 + 2, 8>([&](auto ss) {
        constexpr int s = decltype(ss)::value;
        const T x[4] = {T{quad_bcast<0>(v[s].re), quad_bcast<0>(v[s].im)},
                        T{quad_bcast<1>(v[s].re), quad_bcast<1>(v[s].im)},
                        T{quad_bcast<2>(v[s].re), quad_bcast<2>(v[s].im)},
                        T{quad_bcast<3>(v[s].re), quad_bcast<3>(v[s].im)}};
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const T* u = &Ls[ib + 4 * h + g][4 * s];
          const T l[4] = {u[0], u[1], u[2], u[3]};
          cnma_sum_<4>(v[s0 + h], l, x);
        }
        // the next solved rows are broadcast after this point, not all at the start
        if constexpr (s < 7) asm volatile("" : "+v"(v[s + 1].re), "+v"(v[s + 1].im)::"memory");
      });
      static_for<0, 8>([&](auto aa) {
        constexpr int a = 7 - decltype(aa)::value, sa = s0 + (a >> 2);
        T x = v[sa];
        if constexpr (a < 7) {  // the row solved last comes last
          T l[7 - a], xs[7 - a];
          static_for<0, 7 - a>([&](auto uu) {
            constexpr int u = decltype(uu)::value, c = 7 - u, sc = s0 + (c >> 2);
            l[u] = Ls[ib + a][ib + c];
            xs[u] = T{quad_bcast<(c & 3)>(v[sc].re), quad_bcast<(c & 3)>(v[sc].im)};
          });
          cnma_sum_<7 - a>(x, l, xs);
        }
        const T d = Ls[ib + a][ib + a];
        x = cmul_(x, d);
        v[sa].re = g == (a & 3) ? x.re : v[sa].re;
        v[sa].im = g == (a & 3) ? x.im : v[sa].im;
        asm volatile("" ::: "memory");
      });
    });
  }
  if (col < nrhs) {
#pragma unroll
    for (int s = 0; s < 8; ++s)
      if (4 * s + g < n) {
        B[4 * s + g].re = v[s].re;
        B[4 * s + g].im = v[s].im;
      }
  }
}

// ---------------------------------------------------------------------------
// Host orchestration
// ---------------------------------------------------------------------------
template <typename T>
static int laswp(qb_ctx* ctx, T* A, int64_t lda, int64_t sA, int cb, int ce, int k0, int k1,
                 const int* ipiv, int64_t sP, int batch) {
  if (ce <= cb || k1 <= k0) return QB_OK;
  const int np = k1 - k0, cpw = np <= 64 ? 16 : 64;
  dim3 g((ce - cb + cpw - 1) / cpw, batch);
  hipLaunchKernelGGL(k_laswp<T>, g, dim3(256), 5 * (size_t)np * sizeof(int), ctx->stream, A, lda,
                     sA, cb, ce, k0, np, ipiv, sP, cpw);
  QB_HIP(ctx, hipGetLastError());
  return QB_OK;
}

static int split32(int n) {
  int h = (n / 2 + 31) / 32 * 32;
  return h >= n ? n / 2 : h;
}

// There is one leaf kernel: every mode selects it.
void qb_set_trsm_leaf_lds(int) {}

template <typename T, bool LOWER>
static int trsm_leaf(qb_ctx* ctx, int n, int nrhs, const T* L, int64_t ldl, int64_t sL, T* B,
                     int64_t ldb, int64_t sB, int batch) {
  int slot = qb_prof_begin(ctx, QB_K_TRSM, 4.0 * n * n * (double)nrhs * batch, 0);
  hipLaunchKernelGGL((k_trsm_leaf<T, LOWER>), dim3((nrhs + 63) / 64, batch), dim3(256), 0,
                     ctx->stream, n, nrhs, L, ldl, sL, B, ldb, sB, ctx->bix);
  qb_prof_end(ctx, slot);
  QB_HIP(ctx, hipGetLastError());
  return QB_OK;
}

// X = L^{-1} B with L the unit-lower n x n block at L (ld ldl).
template <typename T>
static int trsm_lower(qb_ctx* ctx, int n, int nrhs, const T* L, int64_t ldl, int64_t sL, T* B,
                      int64_t ldb, int64_t sB, int batch) {
  if (n <= 0 || nrhs <= 0) return QB_OK;
  if (n <= 32) return trsm_leaf<T, true>(ctx, n, nrhs, L, ldl, sL, B, ldb, sB, batch);
  int n1 = split32(n);
  int rc = trsm_lower(ctx, n1, nrhs, L, ldl, sL, B, ldb, sB, batch);
  if (rc) return rc;
  rc = gemm_sub<T>(ctx, n - n1, nrhs, n1, L + n1, ldl, sL, B, ldb, sB, B + n1, ldb, sB, batch);
  if (rc) return rc;
  return trsm_lower(ctx, n - n1, nrhs, L + n1 + (int64_t)n1 * ldl, ldl, sL, B + n1, ldb, sB,
                    batch);
}

// X = U^{-1} B with U the upper n x n block.
template <typename T>
static int trsm_upper(qb_ctx* ctx, int n, int nrhs, const T* U, int64_t ldu, int64_t sU, T* B,
                      int64_t ldb, int64_t sB, int batch) {
  if (n <= 0 || nrhs <= 0) return QB_OK;
  if (n <= 32) return trsm_leaf<T, false>(ctx, n, nrhs, U, ldu, sU, B, ldb, sB, batch);
  int n1 = split32(n);
  int rc = trsm_upper(ctx, n - n1, nrhs, U + n1 + (int64_t)n1 * ldu, ldu, sU, B + n1, ldb, sB,
                      batch);
  if (rc) return rc;
  rc = gemm_sub<T>(ctx, n1, nrhs, n - n1, U + (int64_t)n1 * ldu, ldu, sU, B + n1, ldb, sB, B,
                   ldb, sB, batch);
  if (rc) return rc;
  return trsm_upper(ctx, n1, nrhs, U, ldu, sU, B, ldb, sB, batch);
}

// The lean kernels for a complex128 panel beside the trailing update
// (qb_ctx::panel_lean).  They leave LDS to the trailing tile, which pays only
// when that tile holds LDS: beside a register-streamed tile (no LDS) the
// ordinary panel kernels are faster (1009 ms against 1022 ms of LU on the
// 48 matrices of N = 8192).  QB_PANEL_LEAN (read once): 0 never, 1 always,
// unset: when the trailing update of the step takes an LDS tile.
static int panel_lean_mode() {
  static const int mode = [] {
    const char* e = getenv("QB_PANEL_LEAN");
    return !e || !e[0] ? -1 : e[0] == '0' ? 0 : 1;
  }();
  return mode;
}

template <typename T>
static bool panel_lean_beside(const qb_ctx* ctx, int M, int N, int K) {
  if (sizeof(T) != sizeof(cd)) return false;
  const int mode = panel_lean_mode();
  if (mode >= 0) return mode == 1;
  int v = ctx->gemm_pick_conc[1][qb_gemm_class(M, N, K)];
  if (v < 0 || v >= QB_GEMM_VARIANTS || !kGemmAvail[1][v]) v = gemm_default<T>(M, N, K);
  return !kGemmReg[1][v];
}

// The complex128 trailing updates that run on the int8 matrix cores (qb_rns.hip):
// steps of the full panel width of 512 with at least kRnsMin rows left.  An
// update takes 33 to 36 ps per entry there against 48.8 ps, and its slices 12.5
// ps for each of 512 (M + N) elements: at 1024 rows the two meet.  They come with
// the panels of 512 columns (qb_lu_nb), whose line lies at 4096 rows.  Windows of 32
// matrices with panels of 512 and residues against panels of 256: 1536, 1792 and 2100
// rows 3 % slower, 2600, 3100, 3600 and 4095 rows 2, 4, 6 and 10 % faster, 4096 10 %: a
// line of its own at about 2400 rows would be the better one for complex128.
static const int kRnsMin = 1024;
static bool lu_rns(int n) { return qb_lu_nb(n) == 512 && n - 512 >= kRnsMin; }

// The form of a leaf of m rows of an n x n matrix: threads, rows per thread and columns
// held at a time of k_getf2 (rows x columns per thread: 32 for complex128, 64 for
// complex64, at most the leaf's 32 columns), or zeros for k_getf2_long.  beside_fp64:
// the panel runs beside an FP64 trailing update.
//   complex128 with 512-wide panels, 1025 to 4096 rows: eight waves, twice the columns
//   at a time and half the reads of L.  Per leaf of N = 4100 (32 matrices) beside the
//   residue updates, 2049 to 4096 rows: 333 us; 1025 to 2048: 158 (with four waves half
//   as much again and a fifth more; up to 1024 100 either way).  Beside FP64 updates a
//   window of 4100 takes 155 ms, with four waves 161.
//   complex128, 4097 to 8192 rows: 0.95 ms per leaf beside the residue updates (N =
//   8192, 48 matrices), k_getf2_long 2.56; beside FP64 updates k_getf2_long, whose
//   registers leave room for their waves: windows of 6000 and 8192 394 ms and 1.245 s,
//   against 417 ms and 1.30 s.
//   complex64 above 4096 rows: k_getf2_long, beside the FP32 tiles.
QbLeaf qb_panel_leaf_form(bool c128, int n, int m, bool beside_fp64) {
  const int x = c128 ? 1 : 2;
  if (c128 && lu_rns(n) && m > 1024 && m <= 4096)
    return m <= 2048 ? QbLeaf{512, 4, 8} : QbLeaf{512, 8, 4};
  if (m <= 512) return {256, 2, 16};
  if (m <= 1024) return {256, 4, 8 * x};
  if (m <= 2048) return {256, 8, 4 * x};
  if (m <= 4096) return {256, 16, 2 * x};
  if (c128 && m <= 8192 && !beside_fp64) return {512, 16, 2};
  return {0, 0, 0};
}

template <typename T>
static void panel_leaf(qb_ctx* ctx, T* A, int64_t lda, int64_t sA, int n, int c0, int w,
                       int* ipiv, int64_t sP, int* info, int batch, bool beside_fp64) {
  constexpr bool C128 = sizeof(T) == sizeof(cd);
  constexpr int X = C128 ? 1 : 2;
  const QbLeaf f = qb_panel_leaf_form(C128, n, n - c0, beside_fp64);
  if (f.threads == 0) {
    hipLaunchKernelGGL(k_getf2_long<T>, dim3(batch), dim3(512), 0, ctx->stream, A, lda, sA, n, c0,
                       w, ipiv, sP, info);
  } else if (f.threads == 256) {
    auto* k = f.rows == 2   ? &launch_getf2<T, 256, 2, 16>
              : f.rows == 4 ? &launch_getf2<T, 256, 4, 8 * X>
              : f.rows == 8 ? &launch_getf2<T, 256, 8, 4 * X>
                            : &launch_getf2<T, 256, 16, 2 * X>;
    k(ctx, A, lda, sA, n, c0, w, ipiv, sP, info, batch);
  } else if constexpr (C128) {
    auto* k = f.rows == 4   ? &launch_getf2<T, 512, 4, 8>
              : f.rows == 8 ? &launch_getf2<T, 512, 8, 4>
                            : &launch_getf2<T, 512, 16, 2>;
    k(ctx, A, lda, sA, n, c0, w, ipiv, sP, info, batch);
  }
}

// Recursive panel: factor columns [c0, c0+w) (rows c0..n-1) of every matrix.
template <typename T>
static int panel_rec(qb_ctx* ctx, T* A, int64_t lda, int64_t sA, int n, int c0, int w, int* ipiv,
                     int64_t sP, int* info, int batch, bool beside_fp64) {
  if (w <= 32) {
    int slot = qb_prof_begin(ctx, QB_K_PANEL, 8.0 * (double)(n - c0) * w * w / 2 * batch, 0);
    panel_leaf<T>(ctx, A, lda, sA, n, c0, w, ipiv, sP, info, batch, beside_fp64);
    qb_prof_end(ctx, slot);
    QB_HIP(ctx, hipGetLastError());
    return QB_OK;
  }
  int w1 = split32(w);
  int rc = panel_rec(ctx, A, lda, sA, n, c0, w1, ipiv, sP, info, batch, beside_fp64);
  if (rc) return rc;
  rc = laswp(ctx, A, lda, sA, c0 + w1, c0 + w, c0, c0 + w1, ipiv, sP, batch);
  if (rc) return rc;
  T* A11 = A + c0 + (int64_t)c0 * lda;
  rc = trsm_lower(ctx, w1, w - w1, A11, lda, sA, A + c0 + (int64_t)(c0 + w1) * lda, lda, sA,
                  batch);
  if (rc) return rc;
  rc = gemm_sub<T>(ctx, n - c0 - w1, w - w1, w1, A + c0 + w1 + (int64_t)c0 * lda, lda, sA,
                   A + c0 + (int64_t)(c0 + w1) * lda, lda, sA,
                   A + c0 + w1 + (int64_t)(c0 + w1) * lda, lda, sA, batch);
  if (rc) return rc;
  rc = panel_rec(ctx, A, lda, sA, n, c0 + w1, w - w1, ipiv, sP, info, batch,
                 beside_fp64);
  if (rc) return rc;
  return laswp(ctx, A, lda, sA, c0, c0 + w1, c0 + w1, c0 + w, ipiv, sP, batch);
}

// Panel width of the blocked LU of n x n matrices: 512 from n = 4096 (the
// trailing updates then read and write the trailing matrix half as often;
// measured at n = 8192, 48 matrices: complex64 LU 677 ms at 512 against 713
// at 256, complex128 window 1.94 s against 2.00), 256 below, where the
// factorisation is panel-bound.  QB_LU_NB (a multiple of 32 in [64, 1024],
// read once) overrides it.
int qb_lu_nb(int n) {
  static const int env = [] {
    const char* e = getenv("QB_LU_NB");
    long v = e ? strtol(e, nullptr, 10) : 0;
    return (v >= 64 && v <= 1024 && v % 32 == 0) ? (int)v : 0;
  }();
  if (env) return env;
  return n >= 4096 ? 512 : 256;
}

// QB_LASWP_AUX=0 (read once) keeps every row interchange on the main stream.
static bool laswp_left_aux() {
  static const bool on = [] {
    const char* e = getenv("QB_LASWP_AUX");
    return !(e && e[0] == '0');
  }();
  return on;
}

template <typename T>
int qb_getrf_first_panel(qb_ctx* ctx, T* A, int n, int64_t lda, int64_t sA, int* ipiv,
                         int64_t sP, int* info, int batch) {
  const int NB = qb_lu_nb(n);
  hipStream_t main = ctx->stream, aux = ctx->stream_aux;
  QB_HIP(ctx, hipEventRecord(ctx->ev_main, main));
  QB_HIP(ctx, hipStreamWaitEvent(aux, ctx->ev_main, 0));
  ctx->stream = aux;
  const int rc = panel_rec(ctx, A, lda, sA, n, 0, n < NB ? n : NB, ipiv, sP, info, batch, false);
  ctx->stream = main;
  if (rc) return rc;
  QB_HIP(ctx, hipEventRecord(ctx->ev_first, aux));
  return QB_OK;
}

int64_t qb_getrf_rns_bytes(int64_t n, int batch) {
  return lu_rns((int)n) ? qb_rns_bytes(n - 512, n - 512, batch) : 0;
}

template <typename T>
int qb_getrf_batched(qb_ctx* ctx, T* A, int n, int64_t lda, int64_t sA, int* ipiv, int64_t sP,
                     int* info, int batch, bool first_done) {
  // Lookahead: after the block row of step s is solved, the columns of panel
  // s+1 are updated first; panel s+1 is then factored on the auxiliary
  // stream while the rest of the trailing update runs on the main stream.
  // The two touch disjoint columns; the main stream waits for the panel
  // before the row swaps of step s+1.
  const int NB = qb_lu_nb(n);
  hipStream_t main = ctx->stream, aux = ctx->stream_aux;
  auto on_aux = [&](auto&& f) -> int {
    ctx->stream = aux;
    int rc = f();
    ctx->stream = main;
    return rc;
  };
  int rc = QB_OK;
  if (first_done)
    QB_HIP(ctx, hipStreamWaitEvent(main, ctx->ev_first, 0));
  else
    rc = panel_rec(ctx, A, lda, sA, n, 0, n < NB ? n : NB, ipiv, sP, info, batch, false);
  if (rc) return rc;
  // Residue buffers of the complex128 trailing updates; without room for them,
  // and under capture (no allocation there), every update takes the FP64 tiles.
  QbRns rns;
  bool use_rns = false;
  if constexpr (sizeof(T) == sizeof(cd))
    use_rns = lu_rns(n) && ctx->residues && !ctx->graphs &&
              qb_rns_open(ctx, &rns, n - NB, n - NB, batch) == QB_OK;
  struct Close {  // on every way out
    qb_ctx* ctx;
    QbRns* h;
    ~Close() { qb_rns_close(ctx, h); }
  } close_rns{ctx, &rns};
  // The interchanges of step s in the columns left of its panel (the L part
  // of earlier panels) run on the auxiliary stream, ahead of the next panel:
  // nothing on the main stream touches those columns any more once the
  // previous trailing update (which reads the last panel's L) is done.
  const bool left_aux = laswp_left_aux();
  for (int k0 = 0; k0 < n; k0 += NB) {
    int kb = n - k0 < NB ? n - k0 : NB;
    if (left_aux && k0 > 0) {
      QB_HIP(ctx, hipEventRecord(ctx->ev_main, main));
      QB_HIP(ctx, hipStreamWaitEvent(aux, ctx->ev_main, 0));
      rc = on_aux([&] {
        return laswp(ctx, A, lda, sA, 0, k0, k0, k0 + kb, ipiv, sP, batch);
      });
    } else {
      rc = laswp(ctx, A, lda, sA, 0, k0, k0, k0 + kb, ipiv, sP, batch);
    }
    if (rc) return rc;
    rc = laswp(ctx, A, lda, sA, k0 + kb, n, k0, k0 + kb, ipiv, sP, batch);
    if (rc) return rc;
    if (k0 + kb >= n) break;
    const int k1 = k0 + kb, m = n - k1;
    const int kb1 = m < NB ? m : NB;
    T* A11 = A + k0 + (int64_t)k0 * lda;
    T* A12 = A + k0 + (int64_t)k1 * lda;
    T* A21 = A + k1 + (int64_t)k0 * lda;
    rc = trsm_lower(ctx, kb, m, A11, lda, sA, A12, lda, sA, batch);
    if (rc) return rc;
    // next panel's columns first
    const bool rns_step = use_rns && kb == NB && m >= kRnsMin;
    if constexpr (sizeof(T) == sizeof(cd)) {
      if (rns_step) {
        rc = qb_rns_set_a(ctx, &rns, m, A21, lda, sA);
        if (!rc)
          rc = qb_rns_sub(ctx, &rns, kb1, A12, lda, sA, A + k1 + (int64_t)k1 * lda, lda, sA);
      }
    }
    if (!rns_step)
      rc = gemm_sub<T>(ctx, m, kb1, kb, A21, lda, sA, A12, lda, sA, A + k1 + (int64_t)k1 * lda,
                       lda, sA, batch);
    if (rc) return rc;
    QB_HIP(ctx, hipEventRecord(ctx->ev_main, main));
    QB_HIP(ctx, hipStreamWaitEvent(aux, ctx->ev_main, 0));
    rc = on_aux([&] {
      ctx->panel_lean = m > kb1 && panel_lean_beside<T>(ctx, m, m - kb1, kb);
      const int r = panel_rec(ctx, A, lda, sA, n, k1, kb1, ipiv, sP, info, batch,
                              m > kb1 && !rns_step);
      ctx->panel_lean = false;
      return r;
    });
    if (rc) return rc;
    QB_HIP(ctx, hipEventRecord(ctx->ev_aux, aux));
    if (m > kb1) {
      ctx->gemm_conc = true;  // beside the panel on the second stream
      if constexpr (sizeof(T) == sizeof(cd)) {
        if (rns_step)
          rc = qb_rns_sub(ctx, &rns, m - kb1, A12 + (int64_t)kb1 * lda, lda, sA,
                          A + k1 + (int64_t)(k1 + kb1) * lda, lda, sA);
      }
      if (!rns_step)
        rc = gemm_sub<T>(ctx, m, m - kb1, kb, A21, lda, sA, A12 + (int64_t)kb1 * lda, lda, sA,
                         A + k1 + (int64_t)(k1 + kb1) * lda, lda, sA, batch);
      ctx->gemm_conc = false;
      if (rc) return rc;
    }
    QB_HIP(ctx, hipStreamWaitEvent(main, ctx->ev_aux, 0));
  }
  if (left_aux && n > NB) {  // the last step's interchanges
    QB_HIP(ctx, hipEventRecord(ctx->ev_aux, aux));
    QB_HIP(ctx, hipStreamWaitEvent(main, ctx->ev_aux, 0));
  }
  return QB_OK;
}

void qb_graphs_clear(qb_ctx* ctx) {
  for (auto& g : ctx->graph_cache) (void)hipGraphExecDestroy(g.exec);
  ctx->graph_cache.clear();
}

template <typename T>
int qb_getrf_graph(qb_ctx* ctx, T* A, int n, int64_t lda, int64_t sA, int* ipiv, int64_t sP,
                   int* info, int batch, bool first_done) {
  if (!ctx->graphs || ctx->prof || ctx->bix || first_done)
    return qb_getrf_batched<T>(ctx, A, n, lda, sA, ipiv, sP, info, batch, first_done);
  const int ty = sizeof(T) == sizeof(cf) ? 0 : 1;
  for (auto& g : ctx->graph_cache)
    if (g.ty == ty && g.A == (const void*)A && g.n == n && g.lda == lda && g.sA == sA &&
        g.ipiv == ipiv && g.sP == sP && g.info == info && g.batch == batch &&
        g.epoch == ctx->gemm_epoch) {
      QB_HIP(ctx, hipGraphLaunch(g.exec, ctx->stream));
      return QB_OK;
    }
  QB_HIP(ctx, hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal));
  int rc = qb_getrf_batched<T>(ctx, A, n, lda, sA, ipiv, sP, info, batch);
  hipGraph_t graph = nullptr;
  hipError_t e = hipStreamEndCapture(ctx->stream, &graph);
  if (rc || e != hipSuccess || !graph) {
    if (graph) (void)hipGraphDestroy(graph);
    if (!rc) rc = qb_fail(ctx, QB_E_HIP, "LU graph capture failed");
    return rc;
  }
  hipGraphExec_t exec = nullptr;
  e = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
  (void)hipGraphDestroy(graph);
  if (e != hipSuccess) return qb_fail(ctx, QB_E_HIP, hipGetErrorString(e));
  if (ctx->graph_cache.size() >= 16) {
    (void)hipGraphExecDestroy(ctx->graph_cache.front().exec);
    ctx->graph_cache.erase(ctx->graph_cache.begin());
  }
  ctx->graph_cache.push_back({ty, A, n, lda, sA, ipiv, sP, info, batch, ctx->gemm_epoch, exec});
  QB_HIP(ctx, hipGraphLaunch(exec, ctx->stream));
  return QB_OK;
}

// B <- U^{-1} L^{-1} B with the factors of qb_getrf_batched; the row
// permutation of zgetrs is applied by the caller (fused into a gather).
template <typename T>
int qb_trsm_lu_batched(qb_ctx* ctx, const T* LU, int n, int64_t lda, int64_t sA, T* B, int nrhs,
                       int64_t ldb, int64_t sB, int batch) {
  int rc = trsm_lower(ctx, n, nrhs, LU, lda, sA, B, ldb, sB, batch);
  if (rc) return rc;
  return trsm_upper(ctx, n, nrhs, LU, lda, sA, B, ldb, sB, batch);
}

// perm[b][i]: the row of the original right-hand side that lands in row i
// after the interchanges ipiv[b][0..n) are applied in order.
__global__ void k_perm_from_ipiv(const int* __restrict__ ipiv, int* __restrict__ perm, int n,
                                 int batch) {
  int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= batch) return;
  const int* ip = ipiv + (int64_t)b * n;
  int* pm = perm + (int64_t)b * n;
  for (int i = 0; i < n; ++i) pm[i] = i;
  for (int s = 0; s < n; ++s) {
    int p = ip[s];
    if (p != s) {
      int t = pm[s];
      pm[s] = pm[p];
      pm[p] = t;
    }
  }
}

// The same with one workgroup per matrix and both arrays in LDS (8 n bytes):
// the interchanges stay sequential, but on LDS instead of global memory.
__global__ void __launch_bounds__(256) k_perm_from_ipiv_lds(const int* __restrict__ ipiv,
                                                            int* __restrict__ perm, int n) {
  extern __shared__ int sm_perm[];
  int* pm = sm_perm;
  int* ip = sm_perm + n;
  const int64_t b = blockIdx.x;
  for (int i = threadIdx.x; i < n; i += 256) {
    pm[i] = i;
    ip[i] = ipiv[b * n + i];
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int s = 0; s < n; ++s) {
      const int p = ip[s];
      if (p != s) {
        const int t = pm[s];
        pm[s] = pm[p];
        pm[p] = t;
      }
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < n; i += 256) perm[b * n + i] = pm[i];
}

int qb_perm_from_ipiv(qb_ctx* ctx, const int* ipiv, int* perm, int n, int batch) {
  const size_t lds = (size_t)8 * n;
  if (n > 0 && lds <= (size_t)96 * 1024) {
    if (lds > (size_t)64 * 1024)
      (void)hipFuncSetAttribute((const void*)k_perm_from_ipiv_lds,
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    hipLaunchKernelGGL(k_perm_from_ipiv_lds, dim3(batch), dim3(256), lds, ctx->stream, ipiv, perm,
                       n);
  } else {
    hipLaunchKernelGGL(k_perm_from_ipiv, dim3((batch + 63) / 64), dim3(64), 0, ctx->stream, ipiv,
                       perm, n, batch);
  }
  QB_HIP(ctx, hipGetLastError());
  return QB_OK;
}

template <typename TO>
__global__ void k_gather_rows(const cd* __restrict__ src, int64_t s_src,
                              const int* __restrict__ perm, TO* __restrict__ dst, int n, int nrhs,
                              const int* __restrict__ bix) {
  const int64_t b = bix ? bix[blockIdx.z] : blockIdx.z;
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  int c = blockIdx.y;
  if (i >= n) return;
  int pi = perm[b * (int64_t)n + i];
  cd v = src[b * s_src + pi + (int64_t)c * n];
  TO* d = dst + b * (int64_t)n * nrhs + i + (int64_t)c * n;
  if constexpr (sizeof(TO) == sizeof(cf))
    *d = to_cf(v);
  else
    *d = v;
}

int qb_gather_rows_cd(qb_ctx* ctx, const cd* src, int64_t s_src, const int* perm, cd* dst, int n,
                      int nrhs, int batch) {
  dim3 g((n + 255) / 256, nrhs, batch);
  hipLaunchKernelGGL(k_gather_rows<cd>, g, dim3(256), 0, ctx->stream, src, s_src, perm, dst, n,
                     nrhs, ctx->bix);
  QB_HIP(ctx, hipGetLastError());
  return QB_OK;
}
int qb_gather_rows_cd2cf(qb_ctx* ctx, const cd* src, int64_t s_src, const int* perm, cf* dst,
                         int n, int nrhs, int batch) {
  dim3 g((n + 255) / 256, nrhs, batch);
  hipLaunchKernelGGL(k_gather_rows<cf>, g, dim3(256), 0, ctx->stream, src, s_src, perm, dst, n,
                     nrhs, ctx->bix);
  QB_HIP(ctx, hipGetLastError());
  return QB_OK;
}

// ---------------------------------------------------------------------------
// Elementwise helpers
// ---------------------------------------------------------------------------
__global__ void k_cd_to_cf(const cd* __restrict__ x, cf* __restrict__ y, int64_t n) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int64_t st = (int64_t)gridDim.x * blockDim.x;
  for (; i < n; i += st) y[i] = to_cf(x[i]);
}
__global__ void k_add_cf_to_cd(const cf* __restrict__ d, cd* __restrict__ x, int64_t n) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int64_t st = (int64_t)gridDim.x * blockDim.x;
  for (; i < n; i += st) {
    cd v = x[i];
    cf e = d[i];
    v.re += (double)e.re;
    v.im += (double)e.im;
    x[i] = v;
  }
}
// X_b += D_b for the nodes of the batch (slot stride ns).
__global__ void k_add_cf_to_cd_nodes(const cf* __restrict__ d, cd* __restrict__ x, int64_t n,
                                     int64_t ns, const int* __restrict__ bix) {
  const int64_t b = bix ? bix[blockIdx.y] : blockIdx.y;
  d += b * ns;
  x += b * ns;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    cd v = x[i];
    cf e = d[i];
    v.re += (double)e.re;
    v.im += (double)e.im;
    x[i] = v;
  }
}
// Copy the first nv entries of V into every node's slot of R (slot stride ns).
__global__ void k_bcast(const cd* __restrict__ V, cd* __restrict__ R, int64_t nv, int64_t ns,
                        int nb, const int* __restrict__ bix) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int64_t st = (int64_t)gridDim.x * blockDim.x;
  for (; i < nv * nb; i += st) {
    int64_t z = i / nv, e = i - z * nv;
    int64_t b = bix ? bix[z] : z;
    R[b * ns + e] = V[e];
  }
}
// A0 = sum_j w_j X_j, A1 = sum_j w_j z_j X_j over nq nodes (beyn.jl:282-283).
__global__ void k_moments(const cd* __restrict__ X, int64_t nv, int nq, const cd* __restrict__ w,
                          const cd* __restrict__ wz, cd* __restrict__ A0, cd* __restrict__ A1) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nv) return;
  cd a0 = mk(0, 0), a1 = mk(0, 0);
  for (int j = 0; j < nq; ++j) {
    cd x = X[(int64_t)j * nv + i];
    a0 = a0 + w[j] * x;
    a1 = a1 + wz[j] * x;
  }
  A0[i] = a0;
  A1[i] = a1;
}
// Per-node max |.|_inf of n_per entries (|re|+|im| bound not used: true modulus).
// 64 workgroups of 256 per node, each with one atomic: with 1024 of them and one per
// wave the atomics to a node's address took the time (32 nodes of 3072 x 352:
// 844 -> 86 us).
__global__ void k_node_maxabs(const cd* __restrict__ X, int64_t n_per, int64_t stride,
                              double* __restrict__ out, const int* __restrict__ bix) {
  const int64_t b = bix ? bix[blockIdx.y] : blockIdx.y;
  X += b * stride;
  double m = 0;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n_per;
       i += (int64_t)gridDim.x * blockDim.x)
    m = fmax(m, cabsd(X[i]));
  for (int off = 32; off >= 1; off >>= 1) m = fmax(m, __shfl_xor(m, off));
  __shared__ double red[4];
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    m = fmax(fmax(red[0], red[1]), fmax(red[2], red[3]));
    atomicMax((unsigned long long*)(out + b), (unsigned long long)__double_as_longlong(m));
  }
}
__global__ void k_node_maxabs32(const cf* __restrict__ X, int64_t n_per, double* __restrict__ out) {
  const int64_t b = blockIdx.y;
  X += b * n_per;
  double m = 0;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n_per;
       i += (int64_t)gridDim.x * blockDim.x)
    m = fmax(m, (double)hypotf(X[i].re, X[i].im));
  for (int off = 32; off >= 1; off >>= 1) m = fmax(m, __shfl_xor(m, off));
  if ((threadIdx.x & 63) == 0)
    atomicMax((unsigned long long*)(out + b), (unsigned long long)__double_as_longlong(m));
}
// Per-node infinity norm of the matrix: max_i sum_j |A_ij|.  A workgroup takes 64
// rows, each of its four waves every fourth group of four columns (one thread per row left
// half the places of the chip empty; 32 matrices of 3072: 2.0 -> 0.95 ms, 5.1 TB/s).
__global__ void __launch_bounds__(256) k_node_rownorm(const cd* __restrict__ A, int64_t n,
                                                      int64_t sA, double* __restrict__ out) {
  __shared__ double red[4][64];
  const int64_t b = blockIdx.y;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int64_t i = (int64_t)blockIdx.x * 64 + lane;
  const cd* a = A + b * sA + (i < n ? i : n - 1);
  double s = 0;
  int64_t j = 4 * w;
  for (; j + 4 <= n; j += 16) {
    cd v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) v[u] = a[(j + u) * n];
#pragma unroll
    for (int u = 0; u < 4; ++u) s += cabsd(v[u]);
  }
  for (; j < n && j % 16 < 4 * w + 4; ++j) s += cabsd(a[j * n]);
  red[w][lane] = s;
  __syncthreads();
  if (w) return;
  s = i < n ? (red[0][lane] + red[1][lane]) + (red[2][lane] + red[3][lane]) : 0.0;
  for (int off = 32; off >= 1; off >>= 1) s = fmax(s, __shfl_xor(s, off));
  if (lane == 0)
    atomicMax((unsigned long long*)(out + b), (unsigned long long)__double_as_longlong(s));
}

static unsigned grid1(int64_t n) {
  int64_t g = (n + 255) / 256;
  return (unsigned)(g > 65536 ? 65536 : (g < 1 ? 1 : g));
}

int qb_cd_to_cf(qb_ctx* ctx, const cd* x, cf* y, int64_t n) {
  hipLaunchKernelGGL(k_cd_to_cf, dim3(grid1(n)), dim3(256), 0, ctx->stream, x, y, n);
  QB_HIP(ctx, hipGetLastError());
  return QB_OK;
}
int qb_add_cf_to_cd(qb_ctx* ctx, const cf* d, cd* x, int64_t n) {
  hipLaunchKernelGGL(k_add_cf_to_cd, dim3(grid1(n)), dim3(256), 0, ctx->stream, d, x, n);
  QB_HIP(ctx, hipGetLastError());
  return QB_OK;
}
int qb_add_cf_to_cd_nodes(qb_ctx* ctx, const cf* d, cd* x, int64_t n, int64_t ns, int nb) {
  int64_t g = (n + 255) / 256;
  dim3 grid((unsigned)(g > 4096 ? 4096 : g), nb);
  hipLaunchKernelGGL(k_add_cf_to_cd_nodes, grid, dim3(256), 0, ctx->stream, d, x, n, ns, ctx->bix);
  QB_HIP(ctx, hipGetLastError());
  return QB_OK;
}
int qb_bcast(qb_ctx* ctx, const cd* V, cd* R, int64_t nv, int64_t ns, int nb) {
  hipLaunchKernelGGL(k_bcast, dim3(grid1(nv * nb)), dim3(256), 0, ctx->stream, V, R, nv, ns, nb,
                     ctx->bix);
  QB_HIP(ctx, hipGetLastError());
  return QB_OK;
}
int qb_moments(qb_ctx* ctx, const cd* X, int64_t nv, int nq, const cd* w, const cd* wz, cd* A0,
               cd* A1) {
  hipLaunchKernelGGL(k_moments, dim3((unsigned)((nv + 255) / 256)), dim3(256), 0, ctx->stream, X,
                     nv, nq, w, wz, A0, A1);
  QB_HIP(ctx, hipGetLastError());
  return QB_OK;
}
int qb_node_maxabs(qb_ctx* ctx, const cd* X, int64_t n_per, int64_t stride, int nb,
                   double* out_dev, int n_out) {
  // out_dev[b] for the physical node b of every batch entry; all n_out
  // entries are cleared first
  QB_HIP(ctx, hipMemsetAsync(out_dev, 0, (n_out > nb ? n_out : nb) * sizeof(double), ctx->stream));
  int64_t g = (n_per + 255) / 256;
  dim3 grid((unsigned)(g > 64 ? 64 : g), nb);
  hipLaunchKernelGGL(k_node_maxabs, grid, dim3(256), 0, ctx->stream, X, n_per, stride, out_dev,
                     ctx->bix);
  QB_HIP(ctx, hipGetLastError());
  return QB_OK;
}
int qb_node_maxabs32(qb_ctx* ctx, const cf* X, int64_t n_per, int nb, double* out_dev) {
  QB_HIP(ctx, hipMemsetAsync(out_dev, 0, nb * sizeof(double), ctx->stream));
  int64_t g = (n_per + 255) / 256;
  dim3 grid((unsigned)(g > 1024 ? 1024 : g), nb);
  hipLaunchKernelGGL(k_node_maxabs32, grid, dim3(256), 0, ctx->stream, X, n_per, out_dev);
  QB_HIP(ctx, hipGetLastError());
  return QB_OK;
}
int qb_node_rownorm(qb_ctx* ctx, const cd* A, int64_t n, int nb, double* out_dev) {
  QB_HIP(ctx, hipMemsetAsync(out_dev, 0, nb * sizeof(double), ctx->stream));
  dim3 grid((unsigned)((n + 63) / 64), nb);
  hipLaunchKernelGGL(k_node_rownorm, grid, dim3(256), 0, ctx->stream, A, n, n * n, out_dev);
  QB_HIP(ctx, hipGetLastError());
  return QB_OK;
}

// explicit instantiations
template int qb_getrf_batched<cf>(qb_ctx*, cf*, int, int64_t, int64_t, int*, int64_t, int*, int,
                                  bool);
template int qb_getrf_batched<cd>(qb_ctx*, cd*, int, int64_t, int64_t, int*, int64_t, int*, int,
                                  bool);
template int qb_getrf_first_panel<cf>(qb_ctx*, cf*, int, int64_t, int64_t, int*, int64_t, int*,
                                      int);
template int qb_getrf_first_panel<cd>(qb_ctx*, cd*, int, int64_t, int64_t, int*, int64_t, int*,
                                      int);
template int qb_getrf_graph<cf>(qb_ctx*, cf*, int, int64_t, int64_t, int*, int64_t, int*, int,
                                bool);
template int qb_getrf_graph<cd>(qb_ctx*, cd*, int, int64_t, int64_t, int*, int64_t, int*, int,
                                bool);
template int qb_trsm_lu_batched<cf>(qb_ctx*, const cf*, int, int64_t, int64_t, cf*, int, int64_t,
                                    int64_t, int);
template int qb_trsm_lu_batched<cd>(qb_ctx*, const cd*, int, int64_t, int64_t, cd*, int, int64_t,
                                    int64_t, int);
template int qb_gemm_tune<cf>(qb_ctx*, int, int, int, int, double*);
template int qb_gemm_tune<cd>(qb_ctx*, int, int, int, int, double*);
template int gemm_sub<cf>(qb_ctx*, int, int, int, const cf*, int64_t, int64_t, const cf*, int64_t,
                          int64_t, cf*, int64_t, int64_t, int);
template int gemm_sub<cd>(qb_ctx*, int, int, int, const cd*, int64_t, int64_t, const cd*, int64_t,
                          int64_t, cd*, int64_t, int64_t, int);
template int gemm_sub_v<cd>(qb_ctx*, int, int, int, int, const cd*, int64_t, int64_t, const cd*, int64_t,
                          int64_t, cd*, int64_t, int64_t, int);
