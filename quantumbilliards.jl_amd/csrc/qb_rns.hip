// complex128 C -= A B on the int8 matrix cores, through residues.
//
// MI355X multiplies int8 at 4.6 PO/s (measured; FP64 MFMA: 75 TF/s), and an
// integer product modulo small moduli is exact.  Row i of A is scaled by a
// power of two so that its largest component lies in [2^52, 2^53) and rounded
// to integers, column j of B likewise; the product of the integers is formed
// exactly modulo M = prod m_l (117.7 bits) by the Chinese remainder theorem
// (the scheme of Ozaki, Uchino and Imamura, "Ozaki scheme II"), scaled back and
// subtracted.
//
// Accuracy.  An operand's entry keeps 53 bits below the largest component of its row
// (A) or column (B), m_i = max_k |a_ik|, n_j = max_k |b_kj|, and the product itself is
// exact to about u m_i n_j (u = 2^-53), so that
//   |error_ij| <= 2 u (m_i sum_k |b_kj| + n_j sum_k |a_ik|) + 16 u m_i n_j
// and a rounding of C.  An FP64 sum errs by multiples of u sum_k |a_ik| |b_kj|: this is
// less unless entries grow along k in A and fall in B alike (rows of very unequal
// scales, before the LU).  With products of equal size, graded by 2^10 / 2^20 / 2^40
// along k, the residues err by 9e-15 / 6e-12 / 4e-6 of sum |a||b|, an FP64 sum by 1e-16.
// The factors of this library's operators are not graded so (row maximum 1.4 to 2.5
// times the median): there the error is 1/15 to 1/150 of that of the three-product FP64
// tiles, and no more with growths e^(|Im k| r) of 1e18 across a matrix.
//
// Every modulus is a product of primes = 1 mod 4, so -1 has a square root j_l
// modulo m_l, and a + b i -> (a + j_l b, a - j_l b) maps the complex numbers
// modulo m_l onto two independent residues: a complex product costs two int8
// products per modulus, 32 in all, instead of three or four.  |residue| <= 121
// and K = 512 keep the int32 sums below 2^23.
//
// k_rns_slice  residues of one operand, in the lane order of the MFMA operands
// k_rns_gemm   the products, the reconstruction and the update of C
#include "qb_internal.h"
#include "qb_linalg.h"

#define RNS_L 16   // moduli
#define RNS_K 512  // inner dimension of the products

namespace {

constexpr int kMod[RNS_L] = {241, 233, 229, 221, 205, 197, 193, 181,
                             173, 157, 149, 137, 113, 109, 101, 97};

struct RnsSlice {  // per modulus, for k_rns_slice
  double m, inv;
  float mf, invf;
  float sa, ja;  // A: (M / m)^-1 / 2 mod m, and j times that
  float jb;      // B: j
  float pad;
};
struct RnsRecon {  // per modulus, for k_rns_gemm
  float inv;
  int nm, bias;      // -m; the accumulators start at a multiple of m near 2^23
  int re[3], im[3];  // 1/m and j/m as 32 + 20 + 20 fraction bits, balanced
  int pad[7];
};
struct RnsTables {
  RnsSlice s[RNS_L];
  RnsRecon r[RNS_L];
  double mscale;  // M 2^-52 2^-106 (fraction bits, operand bits) 4 (scales are 2^(e-1))
};

constexpr int mulmod(int a, int b, int m) { return (int)((long long)a * b % m); }
constexpr int invmod(int a, int m) {
  for (int x = 1; x < m; ++x)
    if (mulmod(a, x, m) == 1) return x;
  return 0;
}
constexpr int sqrt_minus1(int m) {
  for (int x = 1; x < m; ++x)
    if (mulmod(x, x, m) == m - 1) return x;
  return 0;
}
constexpr int balanced(int a, int m) { return a > m / 2 ? a - m : a; }

// a / m (|a| < m) as t 2^-32 + u 2^-52 + v 2^-72, u and v in [-2^19, 2^19]
constexpr void fraction(long long a, int m, int* f) {
  auto round_div = [](long long x, long long y) {  // y > 0, to nearest
    long long q = x / y, r = x - q * y;
    if (r < 0) {
      r += y;
      --q;
    }
    return 2 * r >= y ? q + 1 : q;
  };
  const long long t = round_div(a * (1ll << 32), m);
  const long long r1 = a * (1ll << 32) - t * m;
  const long long u = round_div(r1 * (1ll << 20), m);
  const long long r2 = r1 * (1ll << 20) - u * m;
  f[0] = (int)t;
  f[1] = (int)u;
  f[2] = (int)round_div(r2 * (1ll << 20), m);
}

constexpr RnsTables make_tables() {
  RnsTables T{};
  double M = 1.0;  // rounds at the last few factors: 1 ulp of the result's scale
  for (int l = 0; l < RNS_L; ++l) {
    const int m = kMod[l], j = sqrt_minus1(m);
    int cof = 1;
    for (int k = 0; k < RNS_L; ++k)
      if (k != l) cof = mulmod(cof, kMod[k] % m, m);
    const int s = mulmod(invmod(cof, m), (m + 1) / 2, m);
    T.s[l].m = m;
    T.s[l].inv = 1.0 / m;
    T.s[l].mf = (float)m;
    T.s[l].invf = 1.0f / (float)m;
    T.s[l].sa = (float)balanced(s, m);
    T.s[l].ja = (float)balanced(mulmod(s, j, m), m);
    T.s[l].jb = (float)balanced(j, m);
    T.r[l].inv = 1.0f / (float)m;
    T.r[l].nm = -m;
    T.r[l].bias = (1 << 23) / m * m;
    fraction(1, m, T.r[l].re);
    fraction(balanced(j, m), m, T.r[l].im);
    M *= m;
  }
  for (int i = 0; i < 156; ++i) M *= 0.5;
  T.mscale = M;
  return T;
}

__constant__ RnsTables kRns = make_tables();

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

// t mod m in [-m/2, m/2] as the low byte of the result (|t| < 2^22, exact)
__device__ __forceinline__ int mod_byte(float t, float m, float inv) {
  const float q = __builtin_rintf(t * inv);
  return __float_as_int(__builtin_fmaf(-q, m, t + 12582912.0f));
}
// low bytes of four words
__device__ __forceinline__ int pack4(int a, int b, int c, int d) {
  const int lo = __builtin_amdgcn_perm(b, a, 0x0c0c0400);
  const int hi = __builtin_amdgcn_perm(d, c, 0x04000c0c);
  return lo | hi;
}

// ---------------------------------------------------------------------------
// Residues of an operand: R rows (A, elements src[i + k ld]) or columns (B,
// src[k + i ld]) of length 512, a workgroup of 16 waves per 32 of them.
// Lane = (k / 16 % 2, i % 32) of its wave's 32 k holds 16 elements and writes
// 16 bytes per plane: the 1 KB of a (plane, k / 32) is what a wave's MFMA
// 32x32x32 operand takes, lane by lane.  The planes of 32 rows stand together,
// [i / 32][plane][k / 32], so that a tile of the product reads a few megabytes
// in one piece (plane by plane over all rows, every plane is another page).
// scale[i] = 2^(e-1) with e the exponent of the largest component (NaN when the
// row holds an infinity or NaN, which makes every result of the row NaN).
// What bounds it: about 290 FP64 / FP32 operations per element for its 32
// bytes of residues.  12.5 ps per element (7680 x 512 rows of 48 matrices),
// 3.8 TB/s of reads and writes; an update of 7680 x 7680 spends 4.5 % of its
// time here.
// ---------------------------------------------------------------------------
template <bool ISA>
__global__ void __launch_bounds__(1024) k_rns_slice(int R, const cd* __restrict__ src,
                                                    int64_t ld, int64_t stride,
                                                    const int* __restrict__ bix, int b0,
                                                    signed char* __restrict__ out, int64_t ostride,
                                                    double* __restrict__ scale,
                                                    int64_t sstride) {
  __shared__ unsigned smax[16][32];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  constexpr int nw = RNS_K / 32;
  const int ii = lane & 31, i = blockIdx.x * 32 + ii, k0 = 32 * w + 16 * (lane >> 5);
  const int64_t b = bix ? bix[b0 + blockIdx.y] : b0 + blockIdx.y;
  src += b * stride;
  const int ic = i < R ? i : R - 1;  // rows past the end repeat the last one, unused
  double xr[16], xi[16];
  unsigned mx = 0;
#pragma unroll
  for (int t = 0; t < 16; ++t) {
    const cd* p = ISA ? src + ic + (int64_t)(k0 + t) * ld : src + (k0 + t) + (int64_t)ic * ld;
    xr[t] = p->re;
    xi[t] = p->im;
  }
#pragma unroll
  for (int t = 0; t < 16; ++t) {
    const unsigned hr = __double2hiint(xr[t]) & 0x7fffffff, hi = __double2hiint(xi[t]) & 0x7fffffff;
    mx = hr > mx ? hr : mx;
    mx = hi > mx ? hi : mx;
  }
  const unsigned other = __shfl_xor((int)mx, 32);
  mx = other > mx ? other : mx;
  if (lane < 32) smax[w][lane] = mx;
  __syncthreads();
  for (int q = 0; q < nw; ++q) mx = smax[q][ii] > mx ? smax[q][ii] : mx;
  const bool fin = mx < 0x7ff00000u;
  const int e = mx >= 0x00100000u ? (int)(mx >> 20) : 1;  // biased exponent of the largest component
  if (w == 0 && lane < 32 && i < R)
    scale[(int64_t)blockIdx.y * sstride + i] =
        fin ? __builtin_ldexp(1.0, e - 1023) : __longlong_as_double(0x7ff8000000000000ll);
#pragma unroll
  for (int t = 0; t < 16; ++t) {
    xr[t] = fin ? __builtin_rint(__builtin_ldexp(xr[t], 1075 - e)) : 0.0;
    xi[t] = fin ? __builtin_rint(__builtin_ldexp(xi[t], 1075 - e)) : 0.0;
  }
  constexpr int plane = nw * 1024;
  signed char* o = out + (int64_t)blockIdx.y * ostride + (int64_t)blockIdx.x * 2 * RNS_L * plane +
                   w * 1024 + lane * 16;
#pragma unroll 1
  for (int l = 0; l < RNS_L; ++l) {
    const RnsSlice c = kRns.s[l];
    int p[4], n[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      int bp[4], bn[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const double x = xr[4 * g + t], y = xi[4 * g + t];
        const float rr = (float)__builtin_fma(-__builtin_rint(x * c.inv), c.m, x);
        const float ri = (float)__builtin_fma(-__builtin_rint(y * c.inv), c.m, y);
        const float u = ISA ? rr * c.sa : rr, jv = ISA ? c.ja : c.jb;
        bp[t] = mod_byte(__builtin_fmaf(ri, jv, u), c.mf, c.invf);
        bn[t] = mod_byte(__builtin_fmaf(-ri, jv, u), c.mf, c.invf);
      }
      p[g] = pack4(bp[0], bp[1], bp[2], bp[3]);
      n[g] = pack4(bn[0], bn[1], bn[2], bn[3]);
    }
    *(v4i*)(o + (2 * l) * plane) = v4i{p[0], p[1], p[2], p[3]};
    *(v4i*)(o + (2 * l + 1) * plane) = v4i{n[0], n[1], n[2], n[3]};
  }
}

// ---------------------------------------------------------------------------
// C -= A B from the residue planes.
//
// A workgroup of 8 waves owns a 128 x 64 tile of C, each wave 32 x 32 of it
// (16 complex entries per lane).  It runs through the 32 planes one after the
// other; plane (l, +) and (l, -) are two int8 products with their own 16
// accumulators, reduced modulo m_l in registers and added into three 32-bit
// words of the fraction x / M per component (the top word wraps, which is the
// reduction modulo M): 96 VGPRs per lane, so that nothing but C leaves the CU.
// The operands come through a ring of S stages of 128 k (24 KB each) filled by
// global-to-LDS loads of whole MFMA operands, S - 1 stages ahead, one barrier
// per stage; the ring runs on across planes.  The B fragment is the first MFMA
// operand, so that a lane's results stand in one row of C and 32 lanes cover 32
// rows: C moves in whole lines.
//
// Workgroups are dispatched round-robin over the 8 XCDs: 4 x 8 tiles (512 x
// 512 entries) run on the 32 CUs of one XCD at a time, which share their planes
// through its L2.  What bounds it: the L2-to-LDS rate (24 KB per stage at 50
// bytes per clock and CU: 44 of the 74 us of a tile with nothing else in the
// loop), and the LDS reads and the additions, which the barriers keep from
// hiding behind it entirely (matrix instructions alone: 24 us).  33 to 36 ps per
// entry of C, 122 TFLOP/s counted as 8 M N K; the FP64 tiles take 48.8 ps (84
// TFLOP/s counted so, at 6 M N K of the 78.6 TFLOP/s FP64 matrix peak).
// With K = 256 a tile's prologue and its pass over C double against the
// products and the FP64 tiles are as fast, so there is no such form.
// ---------------------------------------------------------------------------
constexpr int RNS_S = 6;             // stages in the ring
constexpr int RNS_STAGE = 24 * 1024;  // bytes of one: 16 blocks of A, 8 of B

__global__ void __launch_bounds__(512, 2)
    k_rns_gemm(int M, int N, const signed char* __restrict__ Ap, int64_t strideA,
               const double* __restrict__ scA, int64_t sstrideA, const signed char* __restrict__ Bp,
               int64_t strideB, const double* __restrict__ scB, int64_t sstrideB,
               cd* __restrict__ C, int64_t ldc, int64_t sC, const int* __restrict__ bix, int b0,
               int nmat, int mt_n, int nt_n, int sm_n, unsigned sb_n) {
  __shared__ __align__(1024) signed char ring[RNS_S * RNS_STAGE];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // block id -> tile: superblocks of 4 x 8 tiles (of every matrix in turn), one
  // per XCD
  const unsigned id = blockIdx.x, xcd = id & 7, slot = id >> 3;
  const unsigned gsb = (slot >> 5) * 8 + xcd, in = slot & 31;
  const unsigned y = gsb / sb_n, sb = gsb - y * sb_n;
  if ((int)y >= nmat) return;
  const int mt = (int)(sb % sm_n) * 4 + (int)(in & 3), nt = (int)(sb / sm_n) * 8 + (int)(in >> 2);
  if (mt >= mt_n || nt >= nt_n) return;
  const int64_t b = bix ? bix[b0 + y] : b0 + y;
  C += b * sC;
  constexpr int KS = RNS_K / 128;  // stages per plane
  constexpr int KB = 4 * KS;       // blocks of 32 k
  // this wave's three blocks of a stage: 3 w .. 3 w + 2 of 16 of A and 8 of B
  const signed char* src[3];
#pragma unroll
  for (int u = 0; u < 3; ++u) {
    const int i = 3 * w + u;
    const int64_t rows = i < 16 ? mt * 4 + i / 4 : nt * 2 + (i - 16) / 4;
    src[u] = (i < 16 ? Ap + y * strideA : Bp + y * strideB) + (rows * 2 * RNS_L * KB + i % 4) * 1024;
  }
  const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) signed char*)ring;
  const unsigned voff = lane * 16;
  unsigned ld_off = 0;     // its place in the ring
  auto load_stage = [&] {
#pragma unroll
    for (int u = 0; u < 3; ++u) {
      // m0 holds the LDS address (an operand: the compiler sets it); one wait state
      asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                   :
                   : "v"(voff), "s"(src[u]), "{m0}"(lds0 + ld_off + (3 * w + u) * 1024)
                   : "memory");
      src[u] += 4096;
    }
    ld_off = ld_off == (RNS_S - 1) * RNS_STAGE ? 0 : ld_off + RNS_STAGE;
  };
  const int wm = w & 3, wn = w >> 2;
  const signed char* fa = ring + wm * 4096 + lane * 16;
  const signed char* fb = ring + 16384 + wn * 4096 + lane * 16;
  unsigned rd_off = 0;
  unsigned top[2][16];
  int mid[2][16], low[2][16];
#pragma unroll
  for (int e = 0; e < 16; ++e)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      top[h][e] = 0;
      mid[h][e] = 0;
      low[h][e] = 0;
    }
  auto mul_lo = [](int x, int f) {  // (a fused 64-bit multiply-add would pair registers)
    int r;
    asm("v_mul_lo_u32 %0, %1, %2" : "=v"(r) : "v"(x), "s"(f));
    return (unsigned)r;
  };
  // A biased sum's residue: the quotient stands in the low bits of 2^23 + q.
  auto residue = [&](const RnsRecon& c, int P) {
    return __mul24(__float_as_int(__builtin_fmaf((float)P, c.inv, 8388608.0f)), c.nm) + P;
  };
  // Entry e of a finished modulus: residue rp of its first plane, sum Q of its
  // second.
  auto add_entry = [&](const RnsRecon& c, int e, int rp, int Q) {
    const int rm = residue(c, Q), u = rp + rm, v = rm - rp;
    top[0][e] += mul_lo(u, c.re[0]);
    mid[0][e] += __mul24(u, c.re[1]);
    low[0][e] += __mul24(u, c.re[2]);
    top[1][e] += mul_lo(v, c.im[0]);
    mid[1][e] += __mul24(v, c.im[1]);
    low[1][e] += __mul24(v, c.im[2]);
  };
  auto start = [&](int l) {
    v16i a;
    const int bias = kRns.r[l].bias;
#pragma unroll
    for (int e = 0; e < 16; ++e) a[e] = bias;
    return a;
  };
  // Operands of two stages: x of a pair's first, yv of its second.  One is on
  // its way from LDS (eight reads per wave: half as many keep LDS at half its
  // rate) while the other is multiplied.
  v4i x[8], yv[8];
  auto read_stage = [&](v4i* r) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      r[q] = *(const v4i*)(fa + rd_off + q * 1024);
      r[4 + q] = *(const v4i*)(fb + rd_off + q * 1024);
    }
    rd_off = rd_off == (RNS_S - 1) * RNS_STAGE ? 0 : rd_off + RNS_STAGE;
  };
  auto multiply = [&](v16i& acc, const v4i* r) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
      acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(r[4 + q], r[q], acc, 0, 0, 0);
  };
  // Two stages begin when their own loads have landed (all but the newer ones
  // are done), then everybody's have, and nobody reads the two before them.
#define RNS_WAIT(n) asm volatile("s_waitcnt vmcnt(" #n ") lgkmcnt(0)\n\ts_barrier" ::: "memory")
#pragma unroll 1
  for (int t = 0; t < 4; ++t) load_stage();
  constexpr int EP = 32 / KS;  // entries reduced or added per pair
  v16i P, Q;
  int rp[16];
#pragma unroll
  for (int e = 0; e < 16; ++e) {
    Q[e] = 0;
    rp[e] = 0;
  }
#pragma unroll
  for (int q = 0; q < 8; ++q) yv[q] = v4i{0, 0, 0, 0};
  // C by 32-bit offsets from the wave's corner; past the edges they repeat the
  // last row or column, which is not stored
  const int row0 = mt * 128 + wm * 32 < M ? mt * 128 + wm * 32 : M - 1;
  const int col0 = nt * 64 + wn * 32 < N ? nt * 64 + wn * 32 : N - 1;
  const int rl = lane & 31, cl = 4 * (lane >> 5);
  cd* Cw = C + row0 + (int64_t)col0 * ldc;
  const int rc = rl < M - row0 ? rl : M - 1 - row0;
  auto at = [&](int e, unsigned ld) {
    const int c = cl + 8 * (e / 4) + e % 4;
    return (unsigned)rc + (unsigned)(c < N - col0 ? c : N - 1 - col0) * ld;
  };
  auto own_ld = [&] {  // opaque: the offsets are formed where they are used, not kept
    unsigned ld = (unsigned)ldc;
    asm volatile("" : "+s"(ld));
    return ld;
  };
  const double* scol = scB + y * sstrideB + col0;
  double2 cv[2][8];  // eight entries at a time: few registers
  auto load_c = [&](int g) {
    const unsigned ld = own_ld();
#pragma unroll
    for (int e = 0; e < 8; ++e) cv[g][e] = *(const double2*)(Cw + at(8 * g + e, ld));
    asm volatile("" ::: "memory");
  };
  int left = KS * RNS_L;  // pairs of stages from this one on
#pragma unroll 1
  for (int l = 0; l < RNS_L; ++l) {
    // the second plane of the modulus before is added under the first of this
    // one, whose sums are reduced under the second (l = 0: the sums are zero)
    const RnsRecon c = kRns.r[l], c1 = kRns.r[l ? l - 1 : 0];
    P = start(l);
#pragma unroll
    for (int p = 0; p < KS; ++p) {
      if (left > 2) {  // a pair is 6 loads of the wave
        RNS_WAIT(6);
        load_stage();
        load_stage();
      } else if (left == 2) {
        RNS_WAIT(6);
      } else {
        RNS_WAIT(0);
      }
      --left;
      read_stage(x);
      if (p == 0)
        multiply(Q, yv);
      else if (p <= KS / 2)
        multiply(P, yv);
      else
        multiply(Q, yv);
      if (p == KS / 2) Q = start(l);
      read_stage(yv);
      if (p < KS / 2)
        multiply(P, x);
      else
        multiply(Q, x);
#pragma unroll
      for (int e = 0; e < EP; ++e) {
        if (p < KS / 2) {
          add_entry(c1, p * EP + e, rp[p * EP + e], Q[p * EP + e]);
        } else {
          const int i = (p - KS / 2) * EP + e;
          rp[i] = residue(c, P[i]);
        }
      }
    }
  }
  multiply(Q, yv);
  load_c(0);
#undef RNS_WAIT
  {
    const RnsRecon c = kRns.r[RNS_L - 1];
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      add_entry(c, e, rp[e], Q[e]);
      // formed here, not where they are used: fewer registers
      asm volatile("" : "+v"(top[0][e]), "+v"(mid[0][e]), "+v"(low[0][e]), "+v"(top[1][e]),
                   "+v"(mid[1][e]), "+v"(low[1][e]));
    }
  }
  const unsigned ld = own_ld();
  const bool rok = mt * 128 + wm * 32 + rl < M;
  const double sa = scA[y * sstrideA + row0 + rc] * kRns.mscale;
#pragma unroll
  for (int g = 0; g < 2; ++g) {
    asm volatile("" ::: "memory");
    double sc[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int cc = cl + 8 * (2 * g + e / 4) + e % 4;
      sc[e] = scol[cc < N - col0 ? cc : N - 1 - col0];
    }
    if (g == 0) load_c(1);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int i = 8 * g + e;
      // x / M in units of 2^-52
      const double fr = __builtin_fma((double)(int)top[0][i], 1048576.0,
                                      __builtin_fma((double)low[0][i], 0x1p-20, (double)mid[0][i]));
      const double fi = __builtin_fma((double)(int)top[1][i], 1048576.0,
                                      __builtin_fma((double)low[1][i], 0x1p-20, (double)mid[1][i]));
      const double s = sa * sc[e];
      const double2 r = {__builtin_fma(-fr, s, cv[g][e].x), __builtin_fma(-fi, s, cv[g][e].y)};
      if (rok && nt * 64 + wn * 32 + cl + 8 * (i / 4) + i % 4 < N) *(double2*)(Cw + at(i, ld)) = r;
    }
  }
}

}  // namespace

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------
static int64_t rns_blocks(int64_t n, int mult) { return (n + 32 * mult - 1) / (32 * mult) * mult; }
static int64_t rns_plane_bytes(int64_t nblk) { return 2 * RNS_L * nblk * 32 * RNS_K; }

// B is sliced for as many nodes at a time as fit in this many bytes.
static const int64_t kRnsBBytes = (int64_t)1 << 30;
static int rns_b_nodes(int64_t strideB, int batch) {
  const int64_t n = kRnsBBytes / strideB;
  return (int)(n < 1 ? 1 : n < batch ? n : batch);
}

int64_t qb_rns_bytes(int64_t M, int64_t N, int batch) {
  const int64_t a = rns_plane_bytes(rns_blocks(M, 4)), b = rns_plane_bytes(rns_blocks(N, 2));
  return batch * (a + M * 8) + (int64_t)rns_b_nodes(b, batch) * (b + N * 8);
}

int qb_rns_open(qb_ctx* ctx, QbRns* h, int64_t M, int64_t N, int batch) {
  h->maxM = M;
  h->maxN = N;
  h->batch = batch;
  h->strideA = rns_plane_bytes(rns_blocks(M, 4));
  h->strideB = rns_plane_bytes(rns_blocks(N, 2));
  h->nb = rns_b_nodes(h->strideB, batch);
  h->bytes = (size_t)qb_rns_bytes(M, N, batch);
  h->mem = (signed char*)qb_block_take(ctx, h->bytes);
  h->own = h->mem == nullptr;
  if (h->own) {
    const std::string err = ctx->err;
    const int rc = qb_dev_alloc(ctx, (void**)&h->mem, h->bytes);
    if (rc) {  // no room: the caller takes its FP64 kernels
      ctx->err = err;
      h->mem = nullptr;
      return rc;
    }
  }
  h->A = h->mem;
  h->B = h->A + batch * h->strideA;
  h->scA = (double*)(h->B + h->nb * h->strideB);
  h->scB = h->scA + batch * M;
  return QB_OK;
}

void qb_rns_close(qb_ctx* ctx, QbRns* h) {
  if (!h->mem) return;
  if (h->own)
    qb_dev_free(ctx, h->mem, h->bytes);
  else
    qb_block_put(ctx);
  h->mem = nullptr;
}

int qb_rns_set_a(qb_ctx* ctx, QbRns* h, int M, const cd* A, int64_t lda, int64_t sA) {
  h->M = M;
  int slot = qb_prof_begin(ctx, QB_K_OTHER, 0, 0);
  hipLaunchKernelGGL(k_rns_slice<true>, dim3((M + 31) / 32, h->batch), dim3(2 * RNS_K), 0,
                     ctx->stream, M, A, lda, sA, ctx->bix, 0, h->A, h->strideA,
                     h->scA, h->maxM);
  qb_prof_end(ctx, slot);
  QB_HIP(ctx, hipGetLastError());
  return QB_OK;
}

int qb_rns_sub(qb_ctx* ctx, QbRns* h, int N, const cd* B, int64_t ldb, int64_t sB, cd* C,
               int64_t ldc, int64_t sC) {
  if (h->M <= 0 || N <= 0) return QB_OK;
  const int M = h->M;
  const int mt = (M + 127) / 128, nt = (N + 63) / 64, sm = (mt + 3) / 4, sn = (nt + 7) / 8;
  for (int b0 = 0; b0 < h->batch; b0 += h->nb) {
    const int n = h->batch - b0 < h->nb ? h->batch - b0 : h->nb;
    int slot = qb_prof_begin(ctx, QB_K_OTHER, 0, 0);
    hipLaunchKernelGGL(k_rns_slice<false>, dim3((N + 31) / 32, n), dim3(2 * RNS_K), 0, ctx->stream,
                       N, B, ldb, sB, ctx->bix, b0, h->B, h->strideB, h->scB, h->maxN);
    qb_prof_end(ctx, slot);
    QB_HIP(ctx, hipGetLastError());
    slot = qb_prof_begin(ctx, QB_K_GEMM_C128_I8, 8.0 * M * N * RNS_K * (double)n,
                         16.0 * ((double)M * RNS_K + (double)RNS_K * N + 2.0 * M * N) * n);
    if (ctx->prof) ctx->prof_issued[QB_K_GEMM_C128_I8] += 64.0 * M * N * RNS_K * (double)n;
    const unsigned grid = (unsigned)(((int64_t)sm * sn * n + 7) / 8 * 256);
    hipLaunchKernelGGL(k_rns_gemm, dim3(grid), dim3(512), 0, ctx->stream, M, N,
                       h->A + b0 * h->strideA, h->strideA, h->scA + b0 * h->maxM, h->maxM, h->B,
                       h->strideB, h->scB, h->maxN, C, ldc, sC, ctx->bix, b0, n, mt, nt, sm,
                       (unsigned)(sm * sn));
    qb_prof_end(ctx, slot);
    QB_HIP(ctx, hipGetLastError());
  }
  return QB_OK;
}
