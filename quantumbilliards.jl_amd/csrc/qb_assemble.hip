// K1 / K2: batched CFIE-Kress and DLP-Kress assembly of T(z) = I - K(z).
//
// Entry formulas follow _all_k_nosymm_CFIE_chebyshev!
// (src/chebyshev/chebyshev_euclidian_helmholtz_cfie_kress.jl:543-665) and
// _construct_dlp_kress_matrices_chebyshev! + the I - D pass
// (chebyshev_euclidian_helmholtz_dlp_kress.jl:702-769, :1086-1095).
//
// Layout: out[q*N*N + i + j*N] (column-major per wavenumber, Julia's layout).
// The geometry of a pair (distance, 1/r, the DLP numerator, the circulant
// Kress R and log term) is computed in registers instead of being read from
// N x N caches as the reference does.  As in the reference, the specials of a
// distance are evaluated once for the pair (i, j), (j, i).
#include "qb_bessel.h"
#include "qb_cheb.h"
#include "qb_internal.h"
#include <functional>

#define QB_INV_TWO_PI 0.15915494309189533577
#define QB_EULER_OVER_PI (QB_EULER_GAMMA / QB_PI)

struct TabView {
  const cd* H;  // this wavenumber's Hankel table
  const cd* J;  // this wavenumber's J table
  int np_h, M_h, np_j, M_j;
  double rmin_h, rmax;
};

// H0, H1 (and J0, J1) below |z| = 0.2: qb_hankel1_01's series alone, without the
// code and the registers of its other regions.
__device__ __forceinline__ void hank_series(cd z, cd* h0, cd* h1, cd* j0, cd* j1) {
  cd y0, y1;
  qb_bessel_series(z, true, j0, j1, &y0, &y1);
  *h0 = *j0 + mk(-y0.im, y0.re);
  *h1 = *j1 + mk(-y1.im, y1.re);
}

template <int MH, int MJ>
__device__ __forceinline__ void hank(const TabView& tv, double r, cd k, bool cutoff, cd* h0,
                                     cd* h1) {
  // h0_h1_multi_ks_at_r! (bessels:1190-1206): |kr| < 0.2 evaluates directly
  // (the |kr| < 1e-3 series is the same expansion), else interpolates.
  cd z = mk(k.re * r, k.im * r);
  if (cutoff && cabsd(z) < 0.2) {
    qb_hankel1_01(z, h0, h1);
    return;
  }
  int p;
  double t;
  qb_panel(r, tv.rmin_h, tv.rmax, tv.np_h, &p, &t);
  const cd* c = tv.H + (int64_t)p * (2 * (tv.M_h + 1));
  if (MH > 0)
    qb_clenshaw2<MH>(c, t, h0, h1);
  else
    qb_clenshaw2_dyn(c, tv.M_h, t, h0, h1);
}

template <int MH, int MJ>
__device__ __forceinline__ void bessj(const TabView& tv, double r, cd* j0, cd* j1) {
  int p;
  double t;
  qb_panel(r, 0.0, tv.rmax, tv.np_j, &p, &t);
  const cd* c = tv.J + (int64_t)p * (2 * (tv.M_j + 1));
  if (MJ > 0)
    qb_clenshaw2<MJ>(c, t, j0, j1);
  else
    qb_clenshaw2_dyn(c, tv.M_j, t, j0, j1);
}

// Special functions of one distance r at one wavenumber: H0, H1 (Hankel
// table, or the direct evaluation below |kr| = 0.2 for CFIE), J0, J1 (J table,
// only needed inside one component).
struct Spec {
  cd h0, h1, j0, j1;
};

template <int OP, int MH, int MJ>
__device__ __forceinline__ Spec specials(const TabView& tv, double r, cd k, bool same) {
  Spec s;
  hank<MH, MJ>(tv, r, k, OP == QB_CFIE_KRESS, &s.h0, &s.h1);
  if (same) {
    bessj<MH, MJ>(tv, r, &s.j0, &s.j1);
  } else {
    s.j0 = mk(0, 0);
    s.j1 = mk(0, 0);
  }
  return s;
}

// Off-diagonal entry A(z)[i,j] (target i, source j) from the shared
// specials of r = |x_i - x_j| (cheb-CFIE :594-612 and :636-646;
// cheb-DLP :737-765 with F = I - D).
template <int OP>
__device__ __forceinline__ cd offdiag_entry(const DevGeom& g, int64_t i, int64_t j, double dx,
                                            double dy, double invr, bool same, double Rij,
                                            double lt, cd k, const Spec& sp) {
  const cd ik = mk(-k.im, k.re);
  const cd aL2 = mk(-0.5 * k.im, 0.5 * k.re);  // i k / 2
  const cd aM2 = mk(0.0, 0.5);
  const cd aL1 = mk(-k.re * QB_INV_TWO_PI, -k.im * QB_INV_TWO_PI);
  const double aM1 = -QB_INV_TWO_PI;
  double wj = g.ws[j];
  double inn = g.dy[j] * dx - g.dx[j] * dy;  // t_j x (x_i - x_j)
  if (OP == QB_DLP_KRESS) {
    double cD = inn * invr;
    double c1 = Rij * cD, c2 = wj * cD, c3 = wj * lt * cD;
    cd l1 = aL1 * sp.j1, ht = aL2 * sp.h1;
    return -(c1 * l1 + c2 * ht - c3 * l1);
  }
  double sj = g.speed[j];
  if (!same) {
    double cD = wj * inn * invr;
    double cS = wj * sj;
    cd v = cD * (aL2 * sp.h1) + ik * (cS * (aM2 * sp.h0));
    return -v;
  }
  cd L1 = aL1 * sp.j1, L2 = aL2 * sp.h1;
  cd M1 = aM1 * sp.j0, M2 = aM2 * sp.h0;
  double cD1 = Rij * inn * invr, cD2 = wj * inn * invr, cD3 = wj * lt * inn * invr;
  double cS1 = Rij * sj, cS2 = wj * sj, cS3 = wj * sj * lt;
  cd dval = cD1 * L1 + cD2 * L2 - cD3 * L1;
  cd sval = cS1 * M1 + cS2 * M2 - cS3 * M1;
  return -(dval + ik * sval);
}

// Diagonal entry (cheb-CFIE :585-591; cheb-DLP :729-733 with F = I - D).
template <int OP>
__device__ __forceinline__ cd diag_entry(const DevGeom& g, int64_t j, cd k) {
  double wj = g.ws[j];
  if (OP == QB_DLP_KRESS) return mk(1.0 - wj * g.kappa[j], 0.0);
  const cd ik = mk(-k.im, k.re);
  double sj = g.speed[j];
  double rjj = g.rk[g.off[g.comp[j]]];
  cd dval = mk(wj * g.kappa[j], 0.0);
  double m1 = -QB_INV_TWO_PI * sj;
  cd k2 = k * k;
  cd lg = clog(mk(0.25 * k2.re * (sj * sj), 0.25 * k2.im * (sj * sj)));
  cd m2 = mk(-QB_EULER_OVER_PI - QB_INV_TWO_PI * lg.re, 0.5 - QB_INV_TWO_PI * lg.im) * sj;
  cd sval = mk(rjj * m1, 0.0) + wj * m2;
  cd v = dval + ik * sval;
  return mk(1.0 - v.re, -v.im);
}

// Tile-pair assembly.  Block b of grid.x is the pair of 64 x 64 tiles (I, J)
// and (J, I), I >= J, enumerated diagonal by diagonal (d = I - J), so the
// workgroups resident together work on similar distances and read nearby
// table panels.  Each thread computes the specials of 16 distances once and
// produces both A[i,j] (stored directly: a wave writes 64 consecutive rows)
// and A[j,i] (staged in LDS, then written column by column of the mirror
// tile).  grid.z walks the wavenumbers.
template <int OP, int MH, int MJ>
__global__ void __launch_bounds__(256) k_assemble(DevGeom g, const cd* __restrict__ zk,
                                                  const cd* __restrict__ H,
                                                  const cd* __restrict__ J, int np_h, int M_h,
                                                  int np_j, int M_j, double rmin_h, double rmax,
                                                  int64_t q0, int T, cd* __restrict__ out64,
                                                  cf* __restrict__ out32) {
  __shared__ cd mir[64][65];  // mir[i_local][j_local] = A[j, i]
  const int64_t N = g.N;
  const int64_t q = q0 + blockIdx.z;
  // pair index -> (d, J): diagonal d has T - d pairs
  int64_t p = blockIdx.x;
  int d = 0;
  while (p >= T - d) {
    p -= T - d;
    ++d;
  }
  const int Jt = (int)p, It = Jt + d;
  TabView tv;
  tv.H = H + q * (int64_t)np_h * (2 * (M_h + 1));
  tv.J = J + q * (int64_t)np_j * (2 * (M_j + 1));
  tv.np_h = np_h;
  tv.M_h = M_h;
  tv.np_j = np_j;
  tv.M_j = M_j;
  tv.rmin_h = rmin_h;
  tv.rmax = rmax;
  const cd k = zk[q];
  const int il = threadIdx.x & 63, jl0 = threadIdx.x >> 6;
  const int64_t i = (int64_t)It * 64 + il;
  const int64_t base = (q - q0) * N * N;
  const bool diag_tile = (It == Jt);
  const bool iok = i < N;
  double xi = 0, yi = 0;
  int ci = 0;
  if (iok) {
    xi = g.x[i];
    yi = g.y[i];
    ci = g.comp[i];
  }
#pragma unroll 1
  for (int c = 0; c < 16; ++c) {
    const int jl = jl0 + 4 * c;
    const int64_t j = (int64_t)Jt * 64 + jl;
    if (!iok || j >= N) continue;
    cd vij, vji = mk(0, 0);
    if (i == j) {
      vij = diag_entry<OP>(g, j, k);
    } else {
      double dx = xi - g.x[j], dy = yi - g.y[j];
      double r = hypot(dx, dy);
      double invr = 1.0 / r;
      int cj = g.comp[j];
      bool same = (ci == cj);
      double Rij = 0, lt = 0;
      if (same) {
        int64_t o = g.off[ci];
        int64_t nc = g.off[ci + 1] - o;
        int64_t dd = i - j;  // both in [o, o + nc)
        if (dd < 0) dd += nc;
        Rij = g.rk[o + dd];
        lt = g.lt[o + dd];  // both circulant columns are even in (i - j)
      }
      Spec sp = specials<OP, MH, MJ>(tv, r, k, same || OP == QB_DLP_KRESS);
      vij = offdiag_entry<OP>(g, i, j, dx, dy, invr, same, Rij, lt, k, sp);
      if (!diag_tile) vji = offdiag_entry<OP>(g, j, i, -dx, -dy, invr, same, Rij, lt, k, sp);
    }
    int64_t idx = base + i + j * N;
    if (out64) out64[idx] = vij;
    if (out32) out32[idx] = to_cf(vij);
    if (!diag_tile) mir[il][jl] = vji;
  }
  if (diag_tile) return;
  __syncthreads();
  // mirror tile: column i (64 of them), rows j = Jt*64 + 0..63 contiguous
#pragma unroll 1
  for (int c = 0; c < 16; ++c) {
    const int il2 = jl0 + 4 * c;             // which column of the mirror tile
    const int jl2 = threadIdx.x & 63;        // row inside it
    const int64_t ii = (int64_t)It * 64 + il2, jj = (int64_t)Jt * 64 + jl2;
    if (ii >= N || jj >= N) continue;
    cd v = mir[il2][jl2];
    int64_t idx = base + jj + ii * N;
    if (out64) out64[idx] = v;
    if (out32) out32[idx] = to_cf(v);
  }
}

template <int OP, int MH, int MJ>
static void launch_asm(qb_ctx* ctx, const qb_geom* g, const cd* z, int64_t q0, int64_t nzc,
                       const DevTables& t, cd* o64, cf* o32) {
  int64_t N = g->d.N;
  int T = (int)((N + 63) / 64);
  int64_t pairs = (int64_t)T * (T + 1) / 2;
  dim3 grid((unsigned)pairs, 1, (unsigned)nzc);
  double ent = (double)N * N * nzc;
  int slot = qb_prof_begin(ctx, QB_K_ASSEMBLE, 0.0,
                           ent * ((o64 ? sizeof(cd) : 0) + (o32 ? sizeof(cf) : 0)));
  hipLaunchKernelGGL((k_assemble<OP, MH, MJ>), grid, dim3(256), 0, ctx->stream, g->d, z, t.H,
                     t.J, t.np_h, t.M_h, t.np_j, t.M_j, t.rmin_h, t.rmax, q0, T, o64, o32);
  qb_prof_end(ctx, slot);
}

// Conjugate-pair assembly for contours symmetric about the real axis (the
// Beyn windows with real k0): nodes a and b with k_b = conj(k_a) share the
// panel of every distance, and
//   J_n(k_a r) = (H_n(k_a r) + conj(H_n(k_b r))) / 2,  J_n(k_b r) = conj(J_n(k_a r))
// (H^(2)(z) = conj(H^(1)(conj z)) for real order), so one block assembles both
// matrices from the two nodes' Hankel panels alone: per entry pair and node,
// one panel gather instead of the H and J gathers of k_assemble.  A
// self-conjugate node (real k, a == b) gives J = Re H.  The mirror entries
// (j, i) of both nodes are staged in LDS 32 rows at a time and written as
// columns of the mirror tiles.  pairs[blockIdx.z] = (a, b); outputs indexed
// by node from out64 / out32.
template <int OP, int MH>
__global__ void __launch_bounds__(256)
k_assemble_conj(DevGeom g, const cd* __restrict__ zk, const cd* __restrict__ H, int np_h,
                double rmin_h, double rmax, const int* __restrict__ pairs, int T,
                cd* __restrict__ out64, cf* __restrict__ out32) {
  __shared__ cd mir[2][64][33];  // [node][i_local][j_local - 32 h] = A[j, i], half h
  constexpr int PH = 2 * (MH + 1);
  const int64_t N = g.N;
  const int qa = pairs[2 * blockIdx.z], qb = pairs[2 * blockIdx.z + 1];
  const bool two = qa != qb;
  int64_t p = blockIdx.x;
  int d = 0;
  while (p >= T - d) {
    p -= T - d;
    ++d;
  }
  const int Jt = (int)p, It = Jt + d;
  const cd* Ha = H + (int64_t)qa * np_h * PH;
  const cd* Hb = H + (int64_t)qb * np_h * PH;
  const cd ka = zk[qa], kb = zk[qb];
  const int il = threadIdx.x & 63, jl0 = threadIdx.x >> 6;
  const int64_t i = (int64_t)It * 64 + il;
  const bool iok = i < N;
  const int64_t ba = (int64_t)qa * N * N, bb = (int64_t)qb * N * N;
  const bool diag_tile = (It == Jt);
  const int64_t ic = iok ? i : N - 1;
  const double xi = g.x[ic], yi = g.y[ic];
  const int ci = g.comp[ic];
#pragma unroll 1
  for (int h = 0; h < 2; ++h) {
#pragma unroll 1
    for (int c = 8 * h; c < 8 * h + 8; ++c) {
      const int jl = jl0 + 4 * c;
      const int64_t j = (int64_t)Jt * 64 + jl;
      if (!iok || j >= N) continue;
      cd va, vb, wa = mk(0, 0), wb = mk(0, 0);  // (i, j) and (j, i) of nodes a and b
      if (i == j) {
        va = diag_entry<OP>(g, j, ka);
        vb = two ? diag_entry<OP>(g, j, kb) : va;
      } else {
        const double dx = xi - g.x[j], dy = yi - g.y[j];
        const double r = hypot(dx, dy);
        const double invr = 1.0 / r;
        const bool same = (ci == g.comp[j]);
        double Rij = 0, lt = 0;
        if (same) {
          const int64_t o = g.off[ci];
          const int64_t nc = g.off[ci + 1] - o;
          int64_t dd = i - j;  // both in [o, o + nc)
          if (dd < 0) dd += nc;
          Rij = g.rk[o + dd];
          lt = g.lt[o + dd];  // both circulant columns are even in (i - j)
        }
        int pp;
        double t;
        qb_panel(r, rmin_h, rmax, np_h, &pp, &t);
        Spec sa, sb;
        qb_clenshaw2<MH>(Ha + (int64_t)pp * PH, t, &sa.h0, &sa.h1);
        if (two)
          qb_clenshaw2<MH>(Hb + (int64_t)pp * PH, t, &sb.h0, &sb.h1);
        else
          sb = sa;
        if (OP == QB_CFIE_KRESS) {
          // h0_h1_multi_ks_at_r! (bessels:1190-1206): |kr| < 0.2 directly
          const cd z = mk(ka.re * r, ka.im * r);
          if (cabsd(z) < 0.2) {
            qb_hankel1_01(z, &sa.h0, &sa.h1);
            if (two)
              qb_hankel1_01(mk(kb.re * r, kb.im * r), &sb.h0, &sb.h1);
            else
              sb = sa;
          }
        }
        if (same || OP == QB_DLP_KRESS) {
          sa.j0 = 0.5 * (sa.h0 + cconj(sb.h0));
          sa.j1 = 0.5 * (sa.h1 + cconj(sb.h1));
        } else {
          sa.j0 = mk(0, 0);
          sa.j1 = mk(0, 0);
        }
        sb.j0 = cconj(sa.j0);
        sb.j1 = cconj(sa.j1);
        va = offdiag_entry<OP>(g, i, j, dx, dy, invr, same, Rij, lt, ka, sa);
        vb = two ? offdiag_entry<OP>(g, i, j, dx, dy, invr, same, Rij, lt, kb, sb) : va;
        if (!diag_tile) {
          wa = offdiag_entry<OP>(g, j, i, -dx, -dy, invr, same, Rij, lt, ka, sa);
          wb = two ? offdiag_entry<OP>(g, j, i, -dx, -dy, invr, same, Rij, lt, kb, sb) : wa;
        }
      }
      const int64_t e1 = i + j * N;
      if (out64) {
        out64[ba + e1] = va;
        if (two) out64[bb + e1] = vb;
      }
      if (out32) {
        out32[ba + e1] = to_cf(va);
        if (two) out32[bb + e1] = to_cf(vb);
      }
      if (!diag_tile) {
        mir[0][il][jl - 32 * h] = wa;
        mir[1][il][jl - 32 * h] = wb;
      }
    }
    if (diag_tile) continue;  // uniform over the block
    __syncthreads();
    // mirror rows j = Jt*64 + 32h + 0..31 of the 64 columns i: lanes 0..31
    // write one column's 32 contiguous rows, lanes 32..63 the next column
#pragma unroll 1
    for (int c = 0; c < 8; ++c) {
      const int il2 = 2 * (jl0 + 4 * c) + (threadIdx.x >> 5 & 1);
      const int jl2 = threadIdx.x & 31;
      const int64_t ii = (int64_t)It * 64 + il2, jj = (int64_t)Jt * 64 + 32 * h + jl2;
      if (ii >= N || jj >= N) continue;
      const int64_t e2 = jj + ii * N;
      const cd xa = mir[0][il2][jl2];
      if (out64) out64[ba + e2] = xa;
      if (out32) out32[ba + e2] = to_cf(xa);
      if (two) {
        const cd xb = mir[1][il2][jl2];
        if (out64) out64[bb + e2] = xb;
        if (out32) out32[bb + e2] = to_cf(xb);
      }
    }
    __syncthreads();
  }
}

// One-to-one pairing of the wavenumbers with their conjugates (several
// disks of one window can share a real node): a real node pairs with itself,
// any other node with an unused conjugate.  False when some node has none.
bool qb_conj_pairs(const cd* z_host, int64_t nz, std::vector<int>* pr) {
  pr->clear();
  std::vector<char> used(nz, 0);
  for (int64_t a = 0; a < nz; ++a) {
    if (used[a]) continue;
    const cd za = z_host[a];
    const double sc = fabs(za.re) + fabs(za.im);
    int64_t b = -1;
    if (fabs(za.im) <= 1e-14 * sc) {
      b = a;
    } else {
      for (int64_t c = a + 1; c < nz; ++c) {
        const cd zc = z_host[c];
        if (!used[c] && fabs(zc.re - za.re) <= 1e-14 * sc && fabs(zc.im + za.im) <= 1e-14 * sc) {
          b = c;
          break;
        }
      }
    }
    if (b < 0) return false;
    used[a] = used[b] = 1;
    pr->push_back((int)a);
    pr->push_back((int)b);
  }
  const int64_t npair = (int64_t)pr->size() / 2;
  return npair >= 1 && npair <= 65535;
}

int qb_assemble_conj_dev(qb_ctx* ctx, const qb_geom* g, int op, const cd* z_host,
                         const cd* z_dev, int64_t nz, const DevTables& t, cd* out64,
                         cf* out32) {
  // usable: plain geometry, tables of static degree 5 or 7, and every node's
  // conjugate among the nodes (to rounding); returns 1 when not usable
  if (g->sym.m > 0 || t.M_h != t.M_j || (t.M_h != 5 && t.M_h != 7)) return 1;
  if (op != QB_CFIE_KRESS && op != QB_DLP_KRESS) return 1;
  if (op == QB_DLP_KRESS && g->d.ncomp != 1) return 1;
  std::vector<int> pr;
  if (!qb_conj_pairs(z_host, nz, &pr)) return 1;
  int npair = (int)pr.size() / 2;
  int* pd = nullptr;
  int rc = qb_dev_alloc(ctx, (void**)&pd, pr.size() * sizeof(int));
  if (rc) return rc;
  if (hipMemcpyAsync(pd, pr.data(), pr.size() * sizeof(int), hipMemcpyHostToDevice,
                     ctx->stream) != hipSuccess) {
    qb_dev_free(ctx, pd, pr.size() * sizeof(int));
    return qb_fail(ctx, QB_E_HIP, "pair upload failed");
  }
  const int64_t N = g->d.N;
  const int T = (int)((N + 63) / 64);
  const int64_t tpairs = (int64_t)T * (T + 1) / 2;
  const double ent = (double)N * N * nz;
  int slot = qb_prof_begin(ctx, QB_K_ASSEMBLE, 0.0,
                           ent * ((out64 ? sizeof(cd) : 0) + (out32 ? sizeof(cf) : 0)));
  const dim3 grid((unsigned)tpairs, 1, (unsigned)npair);
  if (op == QB_CFIE_KRESS) {
    if (t.M_h == 5)
      hipLaunchKernelGGL((k_assemble_conj<QB_CFIE_KRESS, 5>), grid, dim3(256), 0, ctx->stream,
                         g->d, z_dev, t.H, t.np_h, t.rmin_h, t.rmax, pd, T, out64, out32);
    else
      hipLaunchKernelGGL((k_assemble_conj<QB_CFIE_KRESS, 7>), grid, dim3(256), 0, ctx->stream,
                         g->d, z_dev, t.H, t.np_h, t.rmin_h, t.rmax, pd, T, out64, out32);
  } else {
    if (t.M_h == 5)
      hipLaunchKernelGGL((k_assemble_conj<QB_DLP_KRESS, 5>), grid, dim3(256), 0, ctx->stream,
                         g->d, z_dev, t.H, t.np_h, t.rmin_h, t.rmax, pd, T, out64, out32);
    else
      hipLaunchKernelGGL((k_assemble_conj<QB_DLP_KRESS, 7>), grid, dim3(256), 0, ctx->stream,
                         g->d, z_dev, t.H, t.np_h, t.rmin_h, t.rmax, pd, T, out64, out32);
  }
  qb_prof_end(ctx, slot);
  hipError_t e = hipGetLastError();
  // the pair list must outlive the launch: wait before handing it back
  if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
  qb_dev_free(ctx, pd, pr.size() * sizeof(int));
  if (e != hipSuccess) return qb_fail(ctx, QB_E_HIP, hipGetErrorString(e));
  return QB_OK;
}

// ---------------------------------------------------------------------------
// Conjugate-pair assembly from envelope tables (the kernel of Beyn windows
// with real k0)
// ---------------------------------------------------------------------------
// H_n^(1)(z) = e^{iz} E_n(z) with E_n smooth and non-oscillatory (~ (2 / pi
// z)^{1/2} (1 + O(1/z)) for large z; the log / pole of H_n at z = 0 for
// small z).  At fixed wavenumber k the envelope E_n(k r) is a Chebyshev
// series of low degree on geometric panels: quarter octaves
// [2^o (1 + q/4), 2^o (1 + (q+1)/4)], degree 12, about 1e-15 relative on
// every panel (E_n is analytic in the Bernstein ellipse of a quarter octave,
// whose nearest singularity, r = 0, lies 9 half-widths from its centre).
// From rmin ~ 1e-3 to rmax ~ 2.6 that is 52 panels and 21 KB per wavenumber
// for E_0 and E_1, against the ~1.2e5 panels of the uniform tables of H_n
// itself (their oscillation e^{ikr} at k = 800 needs them), so both nodes'
// tables of a conjugate pair sit in LDS.  Per distance: the panel from the
// exponent and the top mantissa bits of r (exact), one Clenshaw sweep per
// node, one sincos(Re k r) and one exp(Im k r) shared by the pair
// (e^{i conj(k) r} = e^{i Re k r} e^{Im k r}).  H comes out to ~1e-14
// relative, at least as accurate as the reference's uniform tables at their
// 1e-12 tolerance; J, the |k r| < 0.2 direct branch and the entry formulas
// are those of k_assemble_conj.
#define QB_ENV_M 12
#define QB_ENV_NC (QB_ENV_M + 1)
#define QB_ENV_PMAX 128  // 32 octaves

struct EnvLob {
  double t[QB_ENV_NC];  // cospi(j / M)
};

// Quarter-octave panel p (0-based from octave o0) and local coordinate t of r.
__device__ __forceinline__ void env_panel(double r, int o0, int P, int* p, double* t) {
  const int e = ilogb(r);
  const double m = ldexp(r, -e);  // [1, 2)
  int q = (int)((m - 1.0) * 4.0);
  q = q > 3 ? 3 : q;
  int pp = 4 * (e - o0) + q;
  pp = pp < 0 ? 0 : (pp > P - 1 ? P - 1 : pp);
  *p = pp;
  *t = 8.0 * m - (9.0 + 2.0 * q);
}

// Envelope tables: coefficients of the interpolant at the M+1 Lobatto points
// (DCT-I with c_0 and c_M halved), E_0 and E_1 interleaved:
// env[((q P + p) (M+1) + m) 2 + {0, 1}].  A lane evaluates one point, a wave
// four panels, and turns from its point to its coefficient through LDS.  What
// bounds it: one evaluation's serial arithmetic; one thread per panel did 13 in
// a row (ellipse of 530 nodes, 32 wavenumbers: 355 -> 23 us).
#define QB_ENV_PPW (64 / QB_ENV_NC)  // panels per wave

__global__ __launch_bounds__(64) void k_env_tables(const cd* __restrict__ zk, int64_t nz, int o0,
                                                   int P, EnvLob lc, cd* __restrict__ env) {
  __shared__ cd f0[64], f1[64];
  __shared__ double ct[QB_ENV_NC];
  const int lane = threadIdx.x, pl = lane / QB_ENV_NC, j = lane - pl * QB_ENV_NC;
  const int64_t gid = (int64_t)blockIdx.x * QB_ENV_PPW + pl;
  const bool on = pl < QB_ENV_PPW && gid < nz * (int64_t)P;
  if (lane < QB_ENV_NC) ct[lane] = lc.t[lane];
  __syncthreads();
  if (on) {
    const int64_t q = gid / P;
    const int p = (int)(gid - q * P);
    const int oct = o0 + p / 4, qq = p % 4;
    const double a = ldexp(1.0 + 0.25 * qq, oct), b = ldexp(1.25 + 0.25 * qq, oct);
    const double c = 0.5 * (a + b), h = 0.5 * (b - a);
    const double r = fma(h, ct[j], c);
    const cd k = zk[q];
    const cd z = mk(k.re * r, k.im * r);
    cd h0, h1;
    qb_hankel1_01(z, &h0, &h1);
    double sn, cs;
    sincos(z.re, &sn, &cs);
    const double g = exp(z.im);
    const cd e = mk(cs * g, -sn * g);  // e^{-i z}
    f0[lane] = h0 * e;
    f1[lane] = h1 * e;
  }
  __syncthreads();
  if (!on) return;
  const int m = j, base = pl * QB_ENV_NC;
  const double sg = (m & 1) ? -1.0 : 1.0;
  cd s0 = 0.5 * f0[base] + 0.5 * (sg * f0[base + QB_ENV_M]);
  cd s1 = 0.5 * f1[base] + 0.5 * (sg * f1[base + QB_ENV_M]);
#pragma unroll
  for (int i = 1; i < QB_ENV_M; ++i) {
    int x = (i * m) % (2 * QB_ENV_M);  // cospi(i m / M) from the nodes
    x = x > QB_ENV_M ? 2 * QB_ENV_M - x : x;
    s0 = s0 + f0[base + i] * ct[x];
    s1 = s1 + f1[base + i] * ct[x];
  }
  const double s2 = 2.0 / QB_ENV_M;
  const double w = (m == 0 || m == QB_ENV_M) ? 0.5 * s2 : s2;
  cd* o = env + gid * (int64_t)(2 * QB_ENV_NC);
  o[2 * m] = w * s0;
  o[2 * m + 1] = w * s1;
}

// MW: columns of the mirror tile staged through LDS at a time (16, or 4 for
// the variant that fits three workgroups per CU: 2 x 64 x 5 instead of
// 2 x 64 x 17 entries); OCC: waves per SIMD the registers must allow.
template <int OP, int MW, int OCC>
__global__ void __launch_bounds__(256, OCC)
k_assemble_env(DevGeom g, const cd* __restrict__ zk, const cd* __restrict__ env, int o0, int P,
               const int* __restrict__ pairs, int nout, int T, int J0, int first,
               cd* __restrict__ out64, cf* __restrict__ out32) {
  static_assert(MW == 4 || MW == 8 || MW == 16, "mirror width");
  extern __shared__ __align__(16) cd smem[];
  const int tsz = P * 2 * QB_ENV_NC;  // complex coefficients per node
  cd* Ta = smem;
  cd* Tb = smem + tsz;
  cd (*mir)[64][MW + 1] = (cd (*)[64][MW + 1])(smem + 2 * tsz);  // [node][i_local][j_local - MW h]
  const int64_t N = g.N;
  const int qa = pairs[2 * blockIdx.z], qb = pairs[2 * blockIdx.z + 1];
  const bool two = qa != qb;
  const bool both = two && qb < nout;  // node b is an output too
  for (int e = threadIdx.x; e < tsz; e += 256) {
    Ta[e] = env[(int64_t)qa * tsz + e];
    Tb[e] = env[(int64_t)qb * tsz + e];
  }
  // tile pair (It, Jt), It >= Jt: first = 1 walks the pairs with Jt < J0
  // column by column (the first J0 tile columns, and by the mirror the first
  // J0 tile rows, complete); first = 0 the pairs with Jt >= J0 diagonal by
  // diagonal (J0 = 0: every pair)
  int64_t p = blockIdx.x;
  int It, Jt;
  if (first) {
    int j = 0;
    while (p >= T - j) {
      p -= T - j;
      ++j;
    }
    Jt = j;
    It = j + (int)p;
  } else {
    const int Tr = T - J0;
    int d = 0;
    while (p >= Tr - d) {
      p -= Tr - d;
      ++d;
    }
    Jt = J0 + (int)p;
    It = Jt + d;
  }
  const cd ka = zk[qa], kb = zk[qb];
  const int il = threadIdx.x & 63, jl0 = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t i = (int64_t)It * 64 + il;
  const bool iok = i < N;
  const int64_t ba = (int64_t)qa * N * N, bb = (int64_t)qb * N * N;
  const bool diag_tile = (It == Jt);
  const int64_t ic = iok ? i : N - 1;
  const double xi = g.x[ic], yi = g.y[ic];
  const int ci = g.comp[ic];
  __syncthreads();
  constexpr int CPS = MW / 4;  // column groups (4 columns each) per mirror stage
#pragma unroll 1
  for (int h = blockIdx.y; h < 64 / MW; h += gridDim.y) {
#pragma unroll 1
    for (int c = CPS * h; c < CPS * h + CPS; ++c) {
      const int jl = jl0 + 4 * c;
      const int64_t j = (int64_t)Jt * 64 + jl;
      if (!iok || j >= N) continue;
      cd va, vb, wa = mk(0, 0), wb = mk(0, 0);  // (i, j) and (j, i) of nodes a and b
      if (i == j) {
        va = diag_entry<OP>(g, j, ka);
        vb = both ? diag_entry<OP>(g, j, kb) : va;
      } else {
        const double dx = xi - g.x[j], dy = yi - g.y[j];
        const double r = hypot(dx, dy);
        const double invr = 1.0 / r;
        const bool same = (ci == g.comp[j]);
        double Rij = 0, lt = 0;
        if (same) {
          const int64_t o = g.off[ci];
          const int64_t nc = g.off[ci + 1] - o;
          int64_t dd = i - j;  // both in [o, o + nc)
          if (dd < 0) dd += nc;
          Rij = g.rk[o + dd];
          lt = g.lt[o + dd];  // both circulant columns are even in (i - j)
        }
        Spec sa, sb;
        const cd za = mk(ka.re * r, ka.im * r);
        if (OP == QB_CFIE_KRESS && cabsd(za) < 0.2) {
          // h0_h1_multi_ks_at_r! (bessels:1190-1206): |kr| < 0.2 directly
          cd j0, j1;  // formed below, as elsewhere
          hank_series(za, &sa.h0, &sa.h1, &j0, &j1);
          if (two)
            hank_series(mk(kb.re * r, kb.im * r), &sb.h0, &sb.h1, &j0, &j1);
          else
            sb = sa;
        } else {
          int pp;
          double t;
          env_panel(r, o0, P, &pp, &t);
          double sn, cs;
          sincos(za.re, &sn, &cs);
          const double ga = exp(-za.im);  // |e^{i k_a r}|; node b has k_b = conj(k_a)
          cd e0, e1;
          qb_clenshaw2<QB_ENV_M>(Ta + pp * (2 * QB_ENV_NC), t, &e0, &e1);
          const cd ea = mk(cs * ga, sn * ga);
          sa.h0 = e0 * ea;
          sa.h1 = e1 * ea;
          if (two) {
            qb_clenshaw2<QB_ENV_M>(Tb + pp * (2 * QB_ENV_NC), t, &e0, &e1);
            const double gb = 1.0 / ga;
            const cd eb = mk(cs * gb, sn * gb);
            sb.h0 = e0 * eb;
            sb.h1 = e1 * eb;
          } else {
            sb = sa;
          }
        }
        if (same || OP == QB_DLP_KRESS) {
          sa.j0 = 0.5 * (sa.h0 + cconj(sb.h0));
          sa.j1 = 0.5 * (sa.h1 + cconj(sb.h1));
        } else {
          sa.j0 = mk(0, 0);
          sa.j1 = mk(0, 0);
        }
        sb.j0 = cconj(sa.j0);
        sb.j1 = cconj(sa.j1);
        va = offdiag_entry<OP>(g, i, j, dx, dy, invr, same, Rij, lt, ka, sa);
        vb = both ? offdiag_entry<OP>(g, i, j, dx, dy, invr, same, Rij, lt, kb, sb) : va;
        if (!diag_tile) {
          wa = offdiag_entry<OP>(g, j, i, -dx, -dy, invr, same, Rij, lt, ka, sa);
          wb = both ? offdiag_entry<OP>(g, j, i, -dx, -dy, invr, same, Rij, lt, kb, sb) : wa;
        }
      }
      const int64_t e1 = i + j * N;
      if (out64) {
        out64[ba + e1] = va;
        if (both) out64[bb + e1] = vb;
      }
      if (out32) {
        out32[ba + e1] = to_cf(va);
        if (both) out32[bb + e1] = to_cf(vb);
      }
      if (!diag_tile) {
        mir[0][il][jl - MW * h] = wa;
        if (both) mir[1][il][jl - MW * h] = wb;
      }
    }
    if (diag_tile) continue;  // uniform over the block
    __syncthreads();
    // mirror rows j = Jt*64 + MW h + 0..MW-1 of the 64 columns i: each group
    // of MW lanes writes one column's MW contiguous rows
#pragma unroll 1
    for (int c = 0; c < MW / 4; ++c) {
      const int il2 = (int)(threadIdx.x / MW) + (256 / MW) * c;
      const int jl2 = (int)(threadIdx.x % MW);
      const int64_t ii = (int64_t)It * 64 + il2, jj = (int64_t)Jt * 64 + MW * h + jl2;
      if (ii >= N || jj >= N) continue;
      const int64_t e2 = jj + ii * N;
      const cd xa = mir[0][il2][jl2];
      if (out64) out64[ba + e2] = xa;
      if (out32) out32[ba + e2] = to_cf(xa);
      if (both) {
        const cd xb = mir[1][il2][jl2];
        if (out64) out64[bb + e2] = xb;
        if (out32) out32[bb + e2] = to_cf(xb);
      }
    }
    __syncthreads();
  }
}

// Default variant of the envelope assembly per operator, chosen by measurement
// (three workgroups per CU for DLP, whose registers fit without spilling).
static bool env_occ3_default(int op) { return op == QB_DLP_KRESS; }

// Panels of the envelope tables for distances in [rmin, rmax]: the first octave
// and the panel count, or false when there are too many.
static bool env_range(double rmin, double rmax, int* o0, int* P) {
  if (!(rmin > 0.0) || !(rmax > rmin)) return false;
  *o0 = ilogb(rmin);
  *P = 4 * (ilogb(rmax) - *o0 + 1);
  return *P <= QB_ENV_PMAX;
}
static size_t env_bytes(int64_t nz, int P) { return (size_t)nz * P * 2 * QB_ENV_NC * sizeof(cd); }
static void env_launch_tables(qb_ctx* ctx, const cd* z_dev, int64_t nz, int o0, int P, cd* env) {
  EnvLob lc;
  qb_lobatto_host(QB_ENV_M, lc.t);
  const int64_t nt = nz * (int64_t)P;
  int slot = qb_prof_begin(ctx, QB_K_TABLES, 0.0, (double)env_bytes(nz, P));
  hipLaunchKernelGGL(k_env_tables, dim3((unsigned)((nt + QB_ENV_PPW - 1) / QB_ENV_PPW)),
                     dim3(64), 0, ctx->stream, z_dev, nz, o0, P, lc, env);
  qb_prof_end(ctx, slot);
}

// Workgroups that share the column stages of a tile pair when the tile pairs alone
// are fewer than two rounds of the chip's 512 places (one matrix of N = 128, three
// tile pairs: 53 -> 18 us).
static unsigned env_split(int64_t tiles, unsigned stages) {
  unsigned n = 1;
  while (n < stages && tiles * n < 1024) n *= 2;
  return n;
}

static int assemble_env_pairs(qb_ctx* ctx, const qb_geom* g, int op, const cd* z_dev, int64_t nz,
                              int64_t nout, const std::vector<int>& pr, int o0, int P, cd* out64,
                              cf* out32, int cols_first, const std::function<int()>& between,
                              void* mem = nullptr);

int qb_assemble_env_dev(qb_ctx* ctx, const qb_geom* g, int op, const cd* z_host,
                        const cd* z_dev, int64_t nz, double rmin, double rmax, cd* out64,
                        cf* out32, int cols_first, const std::function<int()>& between) {
  // usable: plain geometry and every node's conjugate among the nodes;
  // returns 1 when not usable
  if (g->sym.m > 0) return 1;
  if (op != QB_CFIE_KRESS && op != QB_DLP_KRESS) return 1;
  if (op == QB_DLP_KRESS && g->d.ncomp != 1) return 1;
  std::vector<int> pr;
  int o0, P;
  if (!env_range(rmin, rmax, &o0, &P) || !qb_conj_pairs(z_host, nz, &pr)) return 1;
  return assemble_env_pairs(ctx, g, op, z_dev, nz, nz, pr, o0, P, out64, out32, cols_first,
                            between);
}

// The pairs `pr` of the nz nodes z_dev; only nodes below nout have a matrix.  mem:
// the caller's device memory for the tables and the pairs, or null.
static int assemble_env_pairs(qb_ctx* ctx, const qb_geom* g, int op, const cd* z_dev, int64_t nz,
                              int64_t nout, const std::vector<int>& pr, int o0, int P, cd* out64,
                              cf* out32, int cols_first, const std::function<int()>& between,
                              void* mem) {
  const int npair = (int)pr.size() / 2;
  const size_t ebytes = env_bytes(nz, P);
  cd* env = (cd*)mem;
  int* pd = mem ? (int*)((char*)mem + ebytes) : nullptr;
  if (!mem) {
    int rc = qb_dev_alloc(ctx, (void**)&env, ebytes);
    if (!rc) rc = qb_dev_alloc(ctx, (void**)&pd, pr.size() * sizeof(int));
    if (rc) {
      qb_dev_free(ctx, env, ebytes);
      return rc;
    }
  }
  auto release = [&] {
    if (mem) return;
    qb_dev_free(ctx, pd, pr.size() * sizeof(int));
    qb_dev_free(ctx, env, ebytes);
  };
  env_launch_tables(ctx, z_dev, nz, o0, P, env);
  int slot;
  hipError_t e = hipGetLastError();
  if (e == hipSuccess)
    e = hipMemcpyAsync(pd, pr.data(), pr.size() * sizeof(int), hipMemcpyHostToDevice,
                       ctx->stream);
  if (e == hipSuccess) {
    const int64_t N = g->d.N;
    const int T = (int)((N + 63) / 64);
    const int64_t tpairs = (int64_t)T * (T + 1) / 2;
    // the first cols_first columns (whole 64-column tiles) in a launch of
    // their own, then `between` (enqueued while the rest assembles)
    const int J0 = between && cols_first > 0 && cols_first % 64 == 0 && cols_first / 64 < T
                       ? cols_first / 64
                       : 0;
    const int64_t pairs_first = (int64_t)J0 * T - (int64_t)J0 * (J0 - 1) / 2;
    // the three-workgroups-per-CU variant (4-column mirror stages) where its
    // LDS fits three times in a CU (QB_ASM_ENV_OCC=2 or 3 forces a variant)
    const size_t tab = (size_t)2 * P * 2 * QB_ENV_NC * sizeof(cd);
    const size_t lds16 = tab + 2 * 64 * 17 * sizeof(cd), lds4 = tab + 2 * 64 * 5 * sizeof(cd);
    bool occ3 = lds4 <= (size_t)(160 * 1024) / 3 && env_occ3_default(op);
    if (const char* e = getenv("QB_ASM_ENV_OCC"))
      occ3 = e[0] == '3' && lds4 <= (size_t)(160 * 1024) / 3;
    const size_t lds = occ3 ? lds4 : lds16;
    const double ent = (double)N * N * nout;
    slot = qb_prof_begin(ctx, QB_K_ASSEMBLE, 0.0,
                         ent * ((out64 ? sizeof(cd) : 0) + (out32 ? sizeof(cf) : 0)));
    auto launch = [&](auto kern, int64_t npairs, int first) {
      (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)lds);
      hipLaunchKernelGGL(kern, dim3((unsigned)npairs, env_split(npairs * npair, occ3 ? 16 : 4),
                                    (unsigned)npair),
                         dim3(256), lds, ctx->stream, g->d, z_dev, env, o0, P, pd, (int)nout, T, J0,
                         first, out64, out32);
    };
    auto launch_all = [&](int64_t npairs, int first) {
      if (op == QB_CFIE_KRESS) {
        if (occ3)
          launch(k_assemble_env<QB_CFIE_KRESS, 4, 3>, npairs, first);
        else
          launch(k_assemble_env<QB_CFIE_KRESS, 16, 1>, npairs, first);
      } else {
        if (occ3)
          launch(k_assemble_env<QB_DLP_KRESS, 4, 3>, npairs, first);
        else
          launch(k_assemble_env<QB_DLP_KRESS, 16, 1>, npairs, first);
      }
    };
    int brc = 0;
    if (J0 > 0) {
      launch_all(pairs_first, 1);
      e = hipGetLastError();
      if (e == hipSuccess) brc = between();
      if (e == hipSuccess && brc == 0) launch_all(tpairs - pairs_first, 0);
    } else {
      launch_all(tpairs, 0);
    }
    qb_prof_end(ctx, slot);
    if (e == hipSuccess) e = hipGetLastError();
    if (e == hipSuccess && brc != 0) {
      (void)hipStreamSynchronize(ctx->stream);
      release();
      return brc;
    }
  }
  // the tables and the pair list must outlive the launch
  if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
  else (void)hipStreamSynchronize(ctx->stream);
  release();
  if (e != hipSuccess) return qb_fail(ctx, QB_E_HIP, hipGetErrorString(e));
  return QB_OK;
}

// Whether uniform tables of the sizes cp would give the Hankel and Bessel values at the
// wavenumber z so exactly (tables tuned to an absolute error of 1e-12) that the envelope
// tables may stand in for them: they are within 1e-14 of the functions, built in 25 us
// and read from LDS.  Coarser tables are interpolated as the caller asked.  Each
// wavenumber of a call is judged by itself, so a matrix does not change with the others.
// The error of a panel of half-width d is about its last coefficient (entering whole,
// as in the reference): for the pole of H_1, at the first distance that the operator
// reads from the table, 2 rho^-M / (s^2 - 1)^(1/2) with s the pole's distance in
// half-widths, for e^{ikr} 2 (|k| d / 2)^M / M!.  Against the actual errors of tables of
// 500 to 75000 panels the estimate is 1.5 to 10 times them, hence the bound 1.2e-11.
// Both routes, tables included: 16 DLP matrices of N = 4096 6.55 (uniform) and 1.45 ms,
// 24 CFIE ones of 1562 1.34 and 0.51 ms, 32 near-real ones of 2050 6.15 and 2.05 ms, one
// of 128 98 and 38 us, six of 1500 with both derivatives 0.74 and 0.37 ms: what bounds
// the uniform route is the L1 request per lane and coefficient.
bool qb_env_stands_in(bool direct, cd z, double rmin, double rmax, const qb_cheb_params& cp) {
  int o0, P;
  if (getenv("QB_ASM_TABLES") || !env_range(rmin, rmax, &o0, &P)) return false;
  const double dh = (rmax - rmin) / (2.0 * cp.n_panels_h), dj = rmax / (2.0 * cp.n_panels_j);
  auto osc = [](double q, int M) {  // 2 q^M / M!, geometric tail
    double v = 2.0;
    for (int n = 1; n <= M; ++n) v *= q / n;
    return q < 0.5 * (M + 1) ? v / (1.0 - q / (M + 1)) : INFINITY;
  };
  const double ak = hypot(z.re, z.im);
  if (!(z.re > 0.0) || !(fabs(z.im) * rmax < 50.0) || !(ak < 1e12)) return false;
  const double grow = exp(fabs(z.im) * rmax);
  const double r1 = direct && 0.2 / ak > rmin ? 0.2 / ak : rmin;  // first distance read
  const double c = fmax(rmin + dh, r1 - dh), s = c / dh;
  if (!(s > 1.0)) return false;
  const double w = sqrt(s * s - 1.0), rho = s + w;
  const double pole = 2.0 * s / w * pow(rho, -cp.M_h) * rho / (rho - 1.0);
  const double amp = 2.0 / (QB_PI * ak * c) + sqrt(2.0 / (QB_PI * ak * c));
  const double eh = grow * amp * (pole + osc(0.5 * ak * dh, cp.M_h));
  const double ej = grow * osc(0.5 * ak * dj, cp.M_j);
  return eh < 1.2e-11 && ej < 1.2e-11;
}

static int env_upload_z(qb_ctx* ctx, const std::vector<cd>& zs, cd* zd) {
  if (hipMemcpyAsync(zd, zs.data(), zs.size() * sizeof(cd), hipMemcpyHostToDevice, ctx->stream) !=
      hipSuccess)
    return qb_fail(ctx, QB_E_HIP, "wavenumber upload failed");
  return QB_OK;
}

// Matrices of any wavenumbers (Re z > 0) of a plain geometry from envelope tables.  A
// wavenumber whose conjugate is in the list to rounding (equal real parts, imaginary
// parts within u |k| of opposite: less than the rounding of k r moves the argument at
// every r) is assembled with it, which may change its last bit; for the others the
// conjugate's table is built beside their own (J_n = (H_n(k r) + conj H_n(conj(k) r)) / 2)
// and only their matrix is written.
// mem: mem_bytes of device memory to work in, or null; 1 when too few.
int qb_assemble_env_list(qb_ctx* ctx, const qb_geom* g, int op, const cd* z_host, int64_t nz,
                         double rmin, double rmax, cd* out64, void* mem, size_t mem_bytes) {
  int o0, P;
  if (!env_range(rmin, rmax, &o0, &P)) return qb_fail(ctx, QB_E_ARG, "distance range");
  // a wavenumber and its partner take a node's tables, z and two pair indices each
  const size_t most = (size_t)(nz < 1024 ? nz : 1024) * 2 * (env_bytes(1, P) + sizeof(cd) + 8);
  if (mem && most > mem_bytes) return 1;
  const int64_t N = g->d.N;
  for (int64_t q0 = 0; q0 < nz; q0 += 1024) {
    const int64_t n = nz - q0 < 1024 ? nz - q0 : 1024;
    std::vector<cd> zs(z_host + q0, z_host + q0 + n);
    std::vector<int> pr;
    std::vector<char> used(n, 0);
    for (int64_t a = 0; a < n; ++a) {
      if (used[a]) continue;
      const double eps = 1.1e-16 * zs[a].re;
      int64_t b = fabs(zs[a].im) <= eps ? a : -1;
      for (int64_t c = a + 1; b < 0 && c < n; ++c)
        if (!used[c] && zs[c].re == zs[a].re && fabs(zs[c].im + zs[a].im) <= eps) b = c;
      if (b < 0) {
        b = (int64_t)zs.size();
        zs.push_back(mk(zs[a].re, -zs[a].im));
      } else {
        used[b] = 1;
      }
      pr.push_back((int)a);
      pr.push_back((int)b);
    }
    const size_t zb = zs.size() * sizeof(cd);
    cd* zd = (cd*)mem;
    int rc = mem ? QB_OK : qb_dev_alloc(ctx, (void**)&zd, zb);
    if (!rc) rc = env_upload_z(ctx, zs, zd);
    if (!rc)
      rc = assemble_env_pairs(ctx, g, op, zd, (int64_t)zs.size(), n, pr, o0, P,
                              out64 + q0 * N * N, nullptr, 0, std::function<int()>(),
                              mem ? (char*)mem + zb : nullptr);
    if (!mem) qb_dev_free(ctx, zd, zb);
    if (rc) return rc;
  }
  return QB_OK;
}

int qb_assemble_dev(qb_ctx* ctx, const qb_geom* g, int op, const cd* z_dev, int64_t nz,
                    const DevTables& t, cd* out64, cf* out32) {
  if (op != QB_CFIE_KRESS && op != QB_DLP_KRESS)
    return qb_fail(ctx, QB_E_ARG, "unknown operator");
  if (op == QB_DLP_KRESS && g->d.ncomp != 1)
    return qb_fail(ctx, QB_E_ARG, "DLP_kress expects one boundary component");
  if (g->sym.m > 0) return qb_assemble_red_dev(ctx, g, op, z_dev, nz, t, out64, out32);
  int64_t N = g->d.N;
  // grid.x = number of 64 x 64 tile pairs (2^31 - 1 limit: N < 2.9e6)
  // grid.z is limited to 65535; chunk the wavenumbers
  for (int64_t q0 = 0; q0 < nz; q0 += 1024) {
    int64_t nzc = nz - q0 < 1024 ? nz - q0 : 1024;
    cd* o64 = out64 ? out64 + q0 * N * N : nullptr;
    cf* o32 = out32 ? out32 + q0 * N * N : nullptr;
    // the kernel indexes its output from the chunk start; pass q0 for tables
    const int mh = t.M_h, mj = t.M_j;
    if (op == QB_CFIE_KRESS) {
      if (mh == 5 && mj == 5)
        launch_asm<QB_CFIE_KRESS, 5, 5>(ctx, g, z_dev, q0, nzc, t, o64, o32);
      else if (mh == 7 && mj == 7)
        launch_asm<QB_CFIE_KRESS, 7, 7>(ctx, g, z_dev, q0, nzc, t, o64, o32);
      else
        launch_asm<QB_CFIE_KRESS, 0, 0>(ctx, g, z_dev, q0, nzc, t, o64, o32);
    } else {
      if (mh == 5 && mj == 5)
        launch_asm<QB_DLP_KRESS, 5, 5>(ctx, g, z_dev, q0, nzc, t, o64, o32);
      else if (mh == 7 && mj == 7)
        launch_asm<QB_DLP_KRESS, 7, 7>(ctx, g, z_dev, q0, nzc, t, o64, o32);
      else
        launch_asm<QB_DLP_KRESS, 0, 0>(ctx, g, z_dev, q0, nzc, t, o64, o32);
    }
    QB_HIP(ctx, hipGetLastError());
  }
  return QB_OK;
}

// One wavenumber's envelope tables in LDS: its own (Ta) and its conjugate's (Tb).
struct EnvView {
  const cd *Ta, *Tb;
  int o0, P;
};
// Tables of a launch: the uniform ones (t), or the envelope tables env
// [2 nz][P][13][2] (the conjugates' from nz on) for the kernels with MH = -1.
struct AsmTabs {
  DevTables t;
  const cd* env;
  int o0, P;
  int64_t nz;
};
// The view of wavenumber q.  Envelope tables are copied to `smem` by the whole
// workgroup (a barrier follows).
template <int MH>
__device__ __forceinline__ auto tab_view(const AsmTabs& tb, int64_t q, cd* smem) {
  if constexpr (MH < 0) {
    const int tsz = tb.P * 2 * QB_ENV_NC;
    for (int e = threadIdx.x; e < tsz; e += blockDim.x) {
      smem[e] = tb.env[q * tsz + e];
      smem[tsz + e] = tb.env[(tb.nz + q) * tsz + e];
    }
    __syncthreads();
    return EnvView{smem, smem + tsz, tb.o0, tb.P};
  } else {
    TabView tv;
    tv.H = tb.t.H + q * (int64_t)tb.t.np_h * (2 * (tb.t.M_h + 1));
    tv.J = tb.t.J ? tb.t.J + q * (int64_t)tb.t.np_j * (2 * (tb.t.M_j + 1)) : nullptr;
    tv.np_h = tb.t.np_h;
    tv.M_h = tb.t.M_h;
    tv.np_j = tb.t.np_j;
    tv.M_j = tb.t.M_j;
    tv.rmin_h = tb.t.rmin_h;
    tv.rmax = tb.t.rmax;
    return tv;
  }
}

// The specials from envelope tables: H_n(k r) = E_n e^{ikr} with the node's own
// table, J_n = (H_n(k r) + conj H_n(conj(k) r)) / 2 with the conjugate's; one
// sincos and one exp serve both.  Below |k r| = 0.2 (direct) the functions
// themselves.
__device__ __forceinline__ Spec specials_env(const EnvView& ev, double r, cd k, bool direct,
                                             bool want_j) {
  Spec s;
  s.j0 = mk(0, 0);
  s.j1 = mk(0, 0);
  const cd z = mk(k.re * r, k.im * r);
  if (direct && cabsd(z) < 0.2) {
    hank_series(z, &s.h0, &s.h1, &s.j0, &s.j1);
    return s;
  }
  int pp;
  double t, sn, cs;
  env_panel(r, ev.o0, ev.P, &pp, &t);
  sincos(z.re, &sn, &cs);
  const double ga = exp(-z.im);
  cd e0, e1;
  qb_clenshaw2<QB_ENV_M>(ev.Ta + pp * (2 * QB_ENV_NC), t, &e0, &e1);
  const cd ea = mk(cs * ga, sn * ga);
  s.h0 = e0 * ea;
  s.h1 = e1 * ea;
  if (want_j) {
    qb_clenshaw2<QB_ENV_M>(ev.Tb + pp * (2 * QB_ENV_NC), t, &e0, &e1);
    const double gb = 1.0 / ga;
    const cd eb = mk(cs * gb, sn * gb);
    const cd g0 = e0 * eb, g1 = e1 * eb;
    s.j0 = 0.5 * (s.h0 + cconj(g0));
    s.j1 = 0.5 * (s.h1 + cconj(g1));
  }
  return s;
}
template <int OP, int MH, int MJ>
__device__ __forceinline__ Spec specials(const EnvView& ev, double r, cd k, bool same) {
  return specials_env(ev, r, k, OP == QB_CFIE_KRESS, same);
}

// ---------------------------------------------------------------------------
// Assembly with the first and second wavenumber derivatives, T, dT/dk and
// d2T/dk2, for the expanded boundary integral method:
//   CFIE: _all_k_nosymm_CFIE_chebyshev_deriv! (cheb-CFIE:881-1059) behind
//         construct_boundary_matrices_with_derivatives! (cheb-CFIE:1507-1530);
//   DLP:  _construct_dlp_kress_matrices_derivatives_chebyshev! and the sign
//         flip + identity of its caller (cheb-DLP:881-952, :1097-1108), behind
//         construct_boundary_matrices_with_derivatives! (cheb-DLP:1126-1144).
// Both read H0, H1, J0, J1 with the |kr| < 0.2 direct branch
// (h0_h1_j0_j1_multi_ks_at_r!; the plain DLP path has no such branch).
// ---------------------------------------------------------------------------
struct D3 {
  cd a, a1, a2;
};

template <int MH, int MJ>
__device__ __forceinline__ Spec specials_all(const TabView& tv, double r, cd k, bool want_j) {
  Spec s;
  hank<MH, MJ>(tv, r, k, true, &s.h0, &s.h1);
  if (want_j) {
    bessj<MH, MJ>(tv, r, &s.j0, &s.j1);
  } else {
    s.j0 = mk(0, 0);
    s.j1 = mk(0, 0);
  }
  return s;
}

template <int MH, int MJ>
__device__ __forceinline__ Spec specials_all(const EnvView& ev, double r, cd k, bool want_j) {
  return specials_env(ev, r, k, true, want_j);
}

// Off-diagonal entry (target i, source j) of T, T', T''.
// Between components the derivative of the double-layer term
// w_j (inn/r)(i k/2) H1(kr) is +(i/2) w_j inn k H0 (and its k-derivative);
// the reference writes both with a minus sign (cheb-CFIE:1031-1032).
// off_sign = -1 reproduces that, +1 (the default) is the derivative.
template <int OP>
__device__ __forceinline__ D3 offdiag_deriv(const DevGeom& g, int64_t j, double dx, double dy,
                                            double r, double invr, bool same, double Rij,
                                            double lt, cd k, const Spec& sp, double off_sign) {
  const cd ik = mk(-k.im, k.re);
  const cd I = mk(0.0, 1.0);
  const cd aL1 = mk(-k.re * QB_INV_TWO_PI, -k.im * QB_INV_TWO_PI);
  const cd aL2 = mk(-0.5 * k.im, 0.5 * k.re);
  const cd aM2 = mk(0.0, 0.5);
  const double aM1 = -QB_INV_TWO_PI;
  const double wj = g.ws[j];
  const double inn = g.dy[j] * dx - g.dx[j] * dy;
  const cd kr = k * r;
  D3 o;
  if (OP == QB_DLP_KRESS) {
    const double cD = inn * invr;
    const double c1 = Rij * cD, c2 = wj * cD, c3 = wj * lt * cD;
    const cd l1 = aL1 * sp.j1;
    const cd D = c1 * l1 + c2 * (aL2 * sp.h1) - c3 * l1;
    const cd kc = k * QB_INV_TWO_PI;
    const cd D1 = kc * ((-Rij * inn) * sp.j0 + wj * ((lt * inn) * sp.j0 + (QB_PI * inn) * (I * sp.h0)));
    const cd u = sp.j0 - kr * sp.j1, v = sp.h0 - kr * sp.h1;
    const cd D2 = (inn * QB_INV_TWO_PI) * ((-Rij) * u + wj * (lt * u + QB_PI * (I * v)));
    o.a = -D;
    o.a1 = -D1;
    o.a2 = -D2;
    return o;
  }
  const double sj = g.speed[j];
  const cd mh = mk(0.0, -0.5), ph = mk(0.0, 0.5);
  if (!same) {
    const double cD = wj * inn * invr, cD1 = wj * inn, cS = wj * sj;
    const cd dval = cD * (aL2 * sp.h1);
    const cd dval1 = off_sign * (ph * (cD1 * (k * sp.h0)));
    const cd dval2 = off_sign * (ph * (cD1 * (sp.h0 - kr * sp.h1)));
    const cd sval = cS * (aM2 * sp.h0);
    const cd sval1 = mh * ((cS * r) * sp.h1);
    const cd sval2 = ph * ((cS * r) * cdiv(sp.h1 - kr * sp.h0, k));
    o.a = -(dval + ik * sval);
    o.a1 = -(dval1 + I * sval + ik * sval1);
    o.a2 = -(dval2 + 2.0 * (I * sval1) + ik * sval2);
    return o;
  }
  const cd L1 = aL1 * sp.j1, L2 = aL2 * sp.h1;
  const cd M1 = aM1 * sp.j0, M2 = aM2 * sp.h0;
  const double cDR = Rij * inn * invr, cDW = wj * inn * invr, cDL = wj * lt * inn * invr;
  const double cR = Rij * inn * QB_INV_TWO_PI, cW = wj * inn * QB_INV_TWO_PI;
  const double cSR = Rij * sj, cS = wj * sj;
  const cd dval = cDR * L1 + cDW * L2 - cDL * L1;
  const cd dval1 = -(cR * (k * sp.j0)) + cW * (k * (lt * sp.j0 + QB_PI * (I * sp.h0)));
  const cd dval2 = cR * (kr * sp.j1 - sp.j0) +
                   cW * (lt * (sp.j0 - kr * sp.j1) + QB_PI * (I * (sp.h0 - kr * sp.h1)));
  const cd sval = cSR * M1 + cS * M2 - (cS * lt) * M1;
  const cd sval1 = (r * sj * QB_INV_TWO_PI) * (Rij * sp.j1 - wj * (lt * sp.j1 + QB_PI * (I * sp.h1)));
  const cd sval2 = (r * sj * QB_INV_TWO_PI) *
                   cdiv(Rij * (kr * sp.j0 - sp.j1) +
                            wj * (lt * (sp.j1 - kr * sp.j0) + QB_PI * (I * (sp.h1 - kr * sp.h0))),
                        k);
  o.a = -(dval + ik * sval);
  o.a1 = -(dval1 + I * sval + ik * sval1);
  o.a2 = -(dval2 + 2.0 * (I * sval1) + ik * sval2);
  return o;
}

// Diagonal entries (cheb-CFIE:922-941; cheb-DLP: D_ii = w_i kappa_i, no
// derivative terms, then F = I - D).
template <int OP>
__device__ __forceinline__ D3 diag_deriv(const DevGeom& g, int64_t j, cd k) {
  D3 o;
  const double wj = g.ws[j];
  if (OP == QB_DLP_KRESS) {
    o.a = mk(1.0 - wj * g.kappa[j], 0.0);
    o.a1 = mk(0, 0);
    o.a2 = mk(0, 0);
    return o;
  }
  const cd I = mk(0.0, 1.0);
  const cd ik = mk(-k.im, k.re);
  const double sj = g.speed[j];
  const double rjj = g.rk[g.off[g.comp[j]]];
  const cd dval = mk(wj * g.kappa[j], 0.0);
  const double m1 = -QB_INV_TWO_PI * sj;
  const cd k2 = k * k;
  const cd lg = clog(mk(0.25 * k2.re * (sj * sj), 0.25 * k2.im * (sj * sj)));
  const cd m2 = mk(-QB_EULER_OVER_PI - QB_INV_TWO_PI * lg.re, 0.5 - QB_INV_TWO_PI * lg.im) * sj;
  const cd sval = mk(rjj * m1, 0.0) + wj * m2;
  const cd sval1 = (-wj * sj / QB_PI) * crecip(k);
  const cd sval2 = (wj * sj / QB_PI) * crecip(k2);
  const cd v = dval + ik * sval;
  o.a = mk(1.0 - v.re, -v.im);
  o.a1 = -(I * sval + ik * sval1);
  o.a2 = -(2.0 * (I * sval1) + ik * sval2);
  return o;
}

// Tile pairs as in k_assemble; the mirrored tile of each of the three
// outputs is staged in LDS CW source columns at a time (3 x 16 x 65 complex
// = 50 KB; 8 beside envelope tables, so that two workgroups fit in a CU) and
// written CW contiguous rows per column.
template <int OP, int MH, int MJ>
__global__ void __launch_bounds__(256, MH < 0 ? 2 : 1)
k_assemble_deriv(DevGeom g, const cd* __restrict__ zk, AsmTabs tb, int64_t q0, int T,
                 cd* __restrict__ o0, cd* __restrict__ o1, cd* __restrict__ o2, double off_sign) {
  constexpr int CW = MH < 0 ? 8 : 16;
  __shared__ cd mir[3][CW][65];  // mir[out][j_local - CW ch][i_local] = A[j, i]
  extern __shared__ __align__(16) cd smem[];
  const int64_t N = g.N;
  const int64_t q = q0 + blockIdx.z;
  int64_t p = blockIdx.x;
  int d = 0;
  while (p >= T - d) {
    p -= T - d;
    ++d;
  }
  const int Jt = (int)p, It = Jt + d;
  const auto tv = tab_view<MH>(tb, q, smem);
  const cd k = zk[q];
  const int il = threadIdx.x & 63, jl0 = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t i = (int64_t)It * 64 + il;
  const int64_t base = (q - q0) * N * N;
  const bool diag_tile = (It == Jt);
  const bool iok = i < N;
  double xi = 0, yi = 0;
  int ci = 0;
  if (iok) {
    xi = g.x[i];
    yi = g.y[i];
    ci = g.comp[i];
  }
#pragma unroll 1
  for (int ch = blockIdx.y; ch < 64 / CW; ch += gridDim.y) {
#pragma unroll 1
    for (int c = 0; c < CW / 4; ++c) {
      const int jc = jl0 + 4 * c;  // 0..CW-1 inside the chunk
      const int64_t j = (int64_t)Jt * 64 + CW * ch + jc;
      if (!iok || j >= N) continue;
      D3 vij, vji;
      if (i == j) {
        vij = diag_deriv<OP>(g, j, k);
      } else {
        const double dx = xi - g.x[j], dy = yi - g.y[j];
        const double r = hypot(dx, dy);
        const double invr = 1.0 / r;
        const int cj = g.comp[j];
        const bool same = (ci == cj);
        double Rij = 0, lt = 0;
        if (same) {
          const int64_t o = g.off[ci];
          const int64_t nc = g.off[ci + 1] - o;
          int64_t dd = i - j;  // both in [o, o + nc)
          if (dd < 0) dd += nc;
          Rij = g.rk[o + dd];
          lt = g.lt[o + dd];
        }
        const Spec sp = specials_all<MH, MJ>(tv, r, k, same);
        vij = offdiag_deriv<OP>(g, j, dx, dy, r, invr, same, Rij, lt, k, sp, off_sign);
        if (!diag_tile)
          vji = offdiag_deriv<OP>(g, i, -dx, -dy, r, invr, same, Rij, lt, k, sp, off_sign);
      }
      const int64_t idx = base + i + j * N;
      o0[idx] = vij.a;
      o1[idx] = vij.a1;
      o2[idx] = vij.a2;
      if (!diag_tile) {
        mir[0][jc][il] = vji.a;
        mir[1][jc][il] = vji.a1;
        mir[2][jc][il] = vji.a2;
      }
    }
    if (diag_tile) continue;  // uniform over the workgroup
    __syncthreads();
    for (int e = threadIdx.x; e < CW * 64; e += 256) {
      const int jr = e % CW, il2 = e / CW;
      const int64_t ii = (int64_t)It * 64 + il2, jj = (int64_t)Jt * 64 + CW * ch + jr;
      if (ii >= N || jj >= N) continue;
      const int64_t idx = base + jj + ii * N;
      o0[idx] = mir[0][jr][il2];
      o1[idx] = mir[1][jr][il2];
      o2[idx] = mir[2][jr][il2];
    }
    __syncthreads();
  }
}

template <int OP, int MH, int MJ>
static void launch_asm_deriv(qb_ctx* ctx, const qb_geom* g, const cd* z, int64_t q0, int64_t nzc,
                             const AsmTabs& tb, cd* o0, cd* o1, cd* o2, double off_sign) {
  int64_t N = g->d.N;
  int T = (int)((N + 63) / 64);
  int64_t pairs = (int64_t)T * (T + 1) / 2;
  dim3 grid((unsigned)pairs, env_split(pairs * nzc, MH < 0 ? 8 : 4), (unsigned)nzc);
  int slot = qb_prof_begin(ctx, QB_K_ASSEMBLE, 0.0, 3.0 * (double)N * N * nzc * sizeof(cd));
  const size_t lds = MH < 0 ? 2 * env_bytes(1, tb.P) : 0;
  if (MH < 0)
    (void)hipFuncSetAttribute((const void*)k_assemble_deriv<OP, MH, MJ>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  hipLaunchKernelGGL((k_assemble_deriv<OP, MH, MJ>), grid, dim3(256), lds, ctx->stream, g->d, z,
                     tb, q0, T, o0, o1, o2, off_sign);
  qb_prof_end(ctx, slot);
}

int qb_assemble_deriv_dev(qb_ctx* ctx, const qb_geom* g, int op, const cd* z_dev, int64_t nz,
                          const DevTables& t, cd* out, cd* dout, cd* ddout, bool ref_sign) {
  const double off_sign = ref_sign ? -1.0 : 1.0;
  if (op != QB_CFIE_KRESS && op != QB_DLP_KRESS)
    return qb_fail(ctx, QB_E_ARG, "unknown operator");
  if (op == QB_DLP_KRESS && g->d.ncomp != 1)
    return qb_fail(ctx, QB_E_ARG, "DLP_kress expects one boundary component");
  if (!t.J) return qb_fail(ctx, QB_E_ARG, "derivative assembly needs the J tables");
  if (g->sym.m > 0 && g->sym.nirr != 1)
    return qb_fail(ctx, QB_E_ARG, "derivative assembly takes one irrep");
  if (g->sym.m > 0)
    return qb_assemble_red_deriv_dev(ctx, g, op, z_dev, nz, t, out, dout, ddout, off_sign);
  int64_t N = g->d.N;
  const AsmTabs tb{t, nullptr, 0, 0, nz};
  for (int64_t q0 = 0; q0 < nz; q0 += 1024) {
    int64_t nzc = nz - q0 < 1024 ? nz - q0 : 1024;
    const int64_t o = q0 * N * N;
    const int mh = t.M_h, mj = t.M_j;
    if (op == QB_CFIE_KRESS) {
      if (mh == 7 && mj == 7)
        launch_asm_deriv<QB_CFIE_KRESS, 7, 7>(ctx, g, z_dev, q0, nzc, tb, out + o, dout + o,
                                              ddout + o, off_sign);
      else
        launch_asm_deriv<QB_CFIE_KRESS, 0, 0>(ctx, g, z_dev, q0, nzc, tb, out + o, dout + o,
                                              ddout + o, off_sign);
    } else {
      if (mh == 7 && mj == 7)
        launch_asm_deriv<QB_DLP_KRESS, 7, 7>(ctx, g, z_dev, q0, nzc, tb, out + o, dout + o,
                                             ddout + o, off_sign);
      else
        launch_asm_deriv<QB_DLP_KRESS, 0, 0>(ctx, g, z_dev, q0, nzc, tb, out + o, dout + o,
                                             ddout + o, off_sign);
    }
    QB_HIP(ctx, hipGetLastError());
  }
  return QB_OK;
}

// Envelope tables of the wavenumbers zs and then of their conjugates, in memory
// for env_free.
struct EnvTabs {
  cd *z = nullptr, *env = nullptr;
  size_t zb = 0, eb = 0;
};
static void env_free(qb_ctx* ctx, EnvTabs* e) {
  qb_dev_free(ctx, e->env, e->eb);
  qb_dev_free(ctx, e->z, e->zb);
  *e = EnvTabs();
}
static int env_build(qb_ctx* ctx, const cd* z_host, int64_t nz, double rmin, double rmax,
                     EnvTabs* e, AsmTabs* tb) {
  tb->nz = nz;
  if (!env_range(rmin, rmax, &tb->o0, &tb->P)) return qb_fail(ctx, QB_E_ARG, "distance range");
  std::vector<cd> zs(z_host, z_host + nz);
  for (int64_t i = 0; i < nz; ++i) zs.push_back(mk(z_host[i].re, -z_host[i].im));
  e->zb = zs.size() * sizeof(cd);
  e->eb = env_bytes(2 * nz, tb->P);
  int rc = qb_dev_alloc(ctx, (void**)&e->z, e->zb);
  if (!rc) rc = qb_dev_alloc(ctx, (void**)&e->env, e->eb);
  if (!rc) rc = env_upload_z(ctx, zs, e->z);
  if (!rc) {
    env_launch_tables(ctx, e->z, 2 * nz, tb->o0, tb->P, e->env);
    if (hipGetLastError() != hipSuccess) rc = qb_fail(ctx, QB_E_HIP, "table launch failed");
  }
  // the host copies are read before the call returns
  if (hipStreamSynchronize(ctx->stream) != hipSuccess && !rc)
    rc = qb_fail(ctx, QB_E_HIP, "tables failed");
  tb->env = e->env;
  if (rc) env_free(ctx, e);
  return rc;
}

// T, T', T'' of a plain geometry from envelope tables (qb_env_stands_in).
int qb_assemble_deriv_env(qb_ctx* ctx, const qb_geom* g, int op, const cd* z_host, int64_t nz,
                          double rmin, double rmax, cd* out, cd* dout, cd* ddout, bool ref_sign) {
  const double off_sign = ref_sign ? -1.0 : 1.0;
  const int64_t N = g->d.N;
  for (int64_t q0 = 0; q0 < nz; q0 += 1024) {
    const int64_t nzc = nz - q0 < 1024 ? nz - q0 : 1024, o = q0 * N * N;
    EnvTabs e;
    AsmTabs tb{};
    int rc = env_build(ctx, z_host + q0, nzc, rmin, rmax, &e, &tb);
    if (rc) return rc;
    if (op == QB_CFIE_KRESS)
      launch_asm_deriv<QB_CFIE_KRESS, -1, -1>(ctx, g, e.z, 0, nzc, tb, out + o, dout + o, ddout + o,
                                              off_sign);
    else
      launch_asm_deriv<QB_DLP_KRESS, -1, -1>(ctx, g, e.z, 0, nzc, tb, out + o, dout + o, ddout + o,
                                             off_sign);
    const hipError_t le = hipGetLastError(), se = hipStreamSynchronize(ctx->stream);
    env_free(ctx, &e);
    if (le != hipSuccess) return qb_fail(ctx, QB_E_HIP, hipGetErrorString(le));
    if (se != hipSuccess) return qb_fail(ctx, QB_E_HIP, hipGetErrorString(se));
  }
  return QB_OK;
}

// ---------------------------------------------------------------------------
// Symmetry-reduced assembly (geometry with orbits, qb_geom_set_orbits):
//   CFIE: _all_k_symm_CFIE_chebyshev! (cheb-CFIE:698-824) and its derivative
//         twin _all_k_symm_CFIE_chebyshev_deriv! (cheb-CFIE:1087-1243);
//   DLP:  the reduced _construct_dlp_kress_matrices_chebyshev! (cheb-DLP:771-880)
//         and its derivative twin (cheb-DLP:955-1050), then F = I - D.
// Entry (a, b) of the m x m reduced matrix is
//   sum_l scale[b, l] * A(rep_a, img[b, l]),
// A the full operator entry computed exactly as k_assemble / k_assemble_deriv
// compute it (same specials, same Kress terms, identity on the diagonal).
// One thread per reduced entry and wavenumber: a wave holds 64 consecutive
// rows a of one column b, so the images of b are wave-uniform and the stores
// are coalesced.  The workgroup covers a 64 x 64 tile; grid.z walks the
// wavenumbers.
// ---------------------------------------------------------------------------
struct PairGeo {
  double dx, dy, r, invr, Rij, lt;
  bool same;
};

__device__ __forceinline__ PairGeo pair_geo(const DevGeom& g, int64_t i, int64_t j, double xi,
                                            double yi, int ci) {
  PairGeo p;
  p.dx = xi - g.x[j];
  p.dy = yi - g.y[j];
  p.r = hypot(p.dx, p.dy);
  p.invr = 1.0 / p.r;
  p.same = (ci == g.comp[j]);
  p.Rij = 0;
  p.lt = 0;
  if (p.same) {
    const int64_t o = g.off[ci];
    const int64_t nc = g.off[ci + 1] - o;
    int64_t dd = i - j;  // both in [o, o + nc)
    if (dd < 0) dd += nc;
    p.Rij = g.rk[o + dd];
    p.lt = g.lt[o + dd];
  }
  return p;
}

__device__ __forceinline__ TabView tab_view(const cd* H, const cd* J, int64_t q, int np_h,
                                            int M_h, int np_j, int M_j, double rmin_h,
                                            double rmax) {
  TabView tv;
  tv.H = H + q * (int64_t)np_h * (2 * (M_h + 1));
  tv.J = J ? J + q * (int64_t)np_j * (2 * (M_j + 1)) : nullptr;
  tv.np_h = np_h;
  tv.M_h = M_h;
  tv.np_j = np_j;
  tv.M_j = M_j;
  tv.rmin_h = rmin_h;
  tv.rmax = rmax;
  return tv;
}

// One thread per reduced entry (a, b); with several irreps (s.nirr, at most
// MAXI) every image term is evaluated once and summed into the entry of each
// irrep with that irrep's weight.  Output matrix e * nz + q (irrep-major).
template <int OP, int MH, int MJ, int MAXI>
__global__ void __launch_bounds__(256) k_assemble_red(DevGeom g, DevSym s, const cd* __restrict__ zk,
                                                      const cd* __restrict__ H,
                                                      const cd* __restrict__ J, int np_h, int M_h,
                                                      int np_j, int M_j, double rmin_h,
                                                      double rmax, int64_t q0, int64_t nz,
                                                      cd* __restrict__ out64,
                                                      cf* __restrict__ out32) {
  const int64_t m = s.m;
  const int G = s.G;
  const int nirr = s.nirr;
  const int64_t q = q0 + blockIdx.z;
  const TabView tv = tab_view(H, J, q, np_h, M_h, np_j, M_j, rmin_h, rmax);
  const cd k = zk[q];
  const int il = threadIdx.x & 63, jl0 = threadIdx.x >> 6;
  const int64_t a = (int64_t)blockIdx.x * 64 + il;
  if (a >= m) return;  // no barrier in this kernel
  const int64_t i = s.img[a * G];
  const double xi = g.x[i], yi = g.y[i];
  const int ci = g.comp[i];
#pragma unroll 1
  for (int c = 0; c < 16; ++c) {
    const int64_t b = (int64_t)blockIdx.y * 64 + jl0 + 4 * c;
    if (b >= m) break;
    cd acc[MAXI];
#pragma unroll
    for (int e = 0; e < MAXI; ++e) acc[e] = mk(0, 0);
#pragma unroll 1
    for (int l = 0; l < G; ++l) {
      const int64_t j = s.img[b * G + l];
      cd v;
      if (i == j) {
        v = diag_entry<OP>(g, j, k);
      } else {
        const PairGeo p = pair_geo(g, i, j, xi, yi, ci);
        const Spec sp = specials<OP, MH, MJ>(tv, p.r, k, p.same || OP == QB_DLP_KRESS);
        v = offdiag_entry<OP>(g, i, j, p.dx, p.dy, p.invr, p.same, p.Rij, p.lt, k, sp);
      }
#pragma unroll
      for (int e = 0; e < MAXI; ++e)
        if (e < nirr) acc[e] = acc[e] + s.scale[((int64_t)e * m + b) * G + l] * v;
    }
#pragma unroll
    for (int e = 0; e < MAXI; ++e) {
      if (e >= nirr) break;
      const int64_t idx = ((int64_t)e * nz + q) * m * m + a + b * m;
      if (out64) out64[idx] = acc[e];
      if (out32) out32[idx] = to_cf(acc[e]);
    }
  }
}

// Pair-shared reduced assembly (geometry with verified isometric orbits,
// DevSym::pair).  Workgroups walk 64 x 64 tile pairs (I, J), I >= J, as
// k_assemble does.  Off the diagonal a thread evaluates the specials of
// r = |x_{rep_a} - x_{img[b,l]}| once per l and uses them for the image term
// of entry (a, b) and for the image term inv[l] of entry (b, a), whose
// distance |x_{rep_b} - x_{img[a,inv[l]]}| is the same; every other factor
// (direction, tangent, component, Kress R and log term) is computed for each
// entry from its own nodes.  Entry (b, a) is staged in LDS and written as
// columns of the mirror tile.  Diagonal tiles are assembled entry by entry.
template <int OP, int MH, int MJ>
__global__ void __launch_bounds__(256) k_assemble_red_pair(DevGeom g, DevSym s,
                                                           const cd* __restrict__ zk,
                                                           const cd* __restrict__ H,
                                                           const cd* __restrict__ J, int np_h,
                                                           int M_h, int np_j, int M_j,
                                                           double rmin_h, double rmax, int64_t q0,
                                                           int T, cd* __restrict__ out64,
                                                           cf* __restrict__ out32) {
  __shared__ cd mir[64][65];  // mir[a_local][b_local] = A_red[b, a]
  const int64_t m = s.m;
  const int G = s.G;
  const int64_t q = q0 + blockIdx.z;
  int64_t p = blockIdx.x;
  int d = 0;
  while (p >= T - d) {
    p -= T - d;
    ++d;
  }
  const int Jt = (int)p, It = Jt + d;
  const TabView tv = tab_view(H, J, q, np_h, M_h, np_j, M_j, rmin_h, rmax);
  const cd k = zk[q];
  const int il = threadIdx.x & 63, jl0 = threadIdx.x >> 6;
  const int64_t a = (int64_t)It * 64 + il;
  const bool aok = a < m;
  const bool diag_tile = (It == Jt);
  const int64_t base = (q - q0) * m * m;
  int64_t i = 0;
  double xi = 0, yi = 0;
  int ci = 0;
  if (aok) {
    i = s.img[a * G];
    xi = g.x[i];
    yi = g.y[i];
    ci = g.comp[i];
  }
#pragma unroll 1
  for (int c = 0; c < 16; ++c) {
    const int jl = jl0 + 4 * c;
    const int64_t b = (int64_t)Jt * 64 + jl;
    if (!aok || b >= m) continue;
    cd acc = mk(0, 0), accm = mk(0, 0);
    if (diag_tile) {
#pragma unroll 1
      for (int l = 0; l < G; ++l) {
        const int64_t j = s.img[b * G + l];
        cd v;
        if (i == j) {
          v = diag_entry<OP>(g, j, k);
        } else {
          const PairGeo pg = pair_geo(g, i, j, xi, yi, ci);
          const Spec sp = specials<OP, MH, MJ>(tv, pg.r, k, pg.same || OP == QB_DLP_KRESS);
          v = offdiag_entry<OP>(g, i, j, pg.dx, pg.dy, pg.invr, pg.same, pg.Rij, pg.lt, k, sp);
        }
        acc = acc + s.scale[b * G + l] * v;
      }
    } else {
      const int64_t ib = s.img[b * G];
      const double xb = g.x[ib], yb = g.y[ib];
      const int cb = g.comp[ib];
#pragma unroll 1
      for (int l = 0; l < G; ++l) {
        const int64_t j = s.img[b * G + l];
        const int ls = s.inv[l];
        const int64_t jm = s.img[a * G + ls];
        const PairGeo p1 = pair_geo(g, i, j, xi, yi, ci);
        const PairGeo p2 = pair_geo(g, ib, jm, xb, yb, cb);  // its r equals p1.r
        const Spec sp = specials<OP, MH, MJ>(tv, p1.r, k,
                                             p1.same || p2.same || OP == QB_DLP_KRESS);
        const cd v1 = offdiag_entry<OP>(g, i, j, p1.dx, p1.dy, p1.invr, p1.same, p1.Rij, p1.lt,
                                        k, sp);
        const cd v2 = offdiag_entry<OP>(g, ib, jm, p2.dx, p2.dy, p1.invr, p2.same, p2.Rij,
                                        p2.lt, k, sp);
        acc = acc + s.scale[b * G + l] * v1;
        accm = accm + s.scale[a * G + ls] * v2;
      }
      mir[il][jl] = accm;
    }
    const int64_t idx = base + a + b * m;
    if (out64) out64[idx] = acc;
    if (out32) out32[idx] = to_cf(acc);
  }
  if (diag_tile) return;  // uniform over the workgroup
  __syncthreads();
#pragma unroll 1
  for (int c = 0; c < 16; ++c) {
    const int il2 = jl0 + 4 * c;       // column a of the mirror tile
    const int jl2 = threadIdx.x & 63;  // row b inside it
    const int64_t aa = (int64_t)It * 64 + il2, bb = (int64_t)Jt * 64 + jl2;
    if (aa >= m || bb >= m) continue;
    const cd v = mir[il2][jl2];
    const int64_t idx = base + bb + aa * m;
    if (out64) out64[idx] = v;
    if (out32) out32[idx] = to_cf(v);
  }
}

// Largest mismatch | |x_{rep_a} - x_{img[b,l]}| - |x_{rep_b} - x_{img[a,inv[l]]}| |
// / (1e-13 r + floor_abs) over one 64 x 64 tile of (a, b) and all l, one value
// per workgroup (<= 1: the distances mirror).  floor_abs is a few ulps of the
// coordinate scale, the rounding every distance carries from its nodes.
__global__ void __launch_bounds__(256) k_orbit_check(DevGeom g, DevSym s, double floor_abs,
                                                     double* out) {
  __shared__ double red[256];
  const int64_t m = s.m;
  const int G = s.G;
  const int il = threadIdx.x & 63, jl0 = threadIdx.x >> 6;
  const int64_t a = (int64_t)blockIdx.x * 64 + il;
  double worst = 0.0;
  if (a < m) {
    const int64_t i = s.img[a * G];
    for (int c = 0; c < 16; ++c) {
      const int64_t b = (int64_t)blockIdx.y * 64 + jl0 + 4 * c;
      if (b >= m) break;
      const int64_t ib = s.img[b * G];
      for (int l = 0; l < G; ++l) {
        const int64_t j = s.img[b * G + l];
        const int64_t jm = s.img[a * G + s.inv[l]];
        const double r1 = hypot(g.x[i] - g.x[j], g.y[i] - g.y[j]);
        const double r2 = hypot(g.x[ib] - g.x[jm], g.y[ib] - g.y[jm]);
        const double dd = fabs(r1 - r2) / (1e-13 * r1 + floor_abs);
        worst = fmax(worst, (i == j) != (ib == jm) ? 1e300 : dd);
      }
    }
  }
  red[threadIdx.x] = worst;
  __syncthreads();
  for (int w = 128; w >= 1; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] = fmax(red[threadIdx.x], red[threadIdx.x + w]);
    __syncthreads();
  }
  if (threadIdx.x == 0) out[(int64_t)blockIdx.y * gridDim.x + blockIdx.x] = red[0];
}

int qb_orbit_pairs_ok(qb_ctx* ctx, const DevGeom& g, const DevSym& s, double floor_abs, int* ok) {
  *ok = 0;
  const unsigned Tm = (unsigned)((s.m + 63) / 64);
  const size_t nb = (size_t)Tm * Tm;
  double* d = nullptr;
  int rc = qb_dev_alloc(ctx, (void**)&d, nb * sizeof(double));
  if (rc) return rc;
  hipLaunchKernelGGL(k_orbit_check, dim3(Tm, Tm), dim3(256), 0, ctx->stream, g, s, floor_abs, d);
  std::vector<double> h(nb);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess)
    e = hipMemcpyAsync(h.data(), d, nb * sizeof(double), hipMemcpyDeviceToHost, ctx->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
  qb_dev_free(ctx, d, nb * sizeof(double));
  if (e != hipSuccess) return qb_fail(ctx, QB_E_HIP, std::string("orbit check: ") + hipGetErrorString(e));
  double worst = 0.0;
  for (double v : h) worst = v > worst ? v : worst;
  *ok = worst <= 1.0 ? 1 : 0;
  return QB_OK;
}

template <int OP, int MH, int MJ>
__global__ void __launch_bounds__(256) k_assemble_red_deriv(
    DevGeom g, DevSym s, const cd* __restrict__ zk, const cd* __restrict__ H,
    const cd* __restrict__ J, int np_h, int M_h, int np_j, int M_j, double rmin_h, double rmax,
    int64_t q0, cd* __restrict__ o0, cd* __restrict__ o1, cd* __restrict__ o2, double off_sign) {
  const int64_t m = s.m;
  const int G = s.G;
  const int64_t q = q0 + blockIdx.z;
  const TabView tv = tab_view(H, J, q, np_h, M_h, np_j, M_j, rmin_h, rmax);
  const cd k = zk[q];
  const int il = threadIdx.x & 63, jl0 = threadIdx.x >> 6;
  const int64_t a = (int64_t)blockIdx.x * 64 + il;
  if (a >= m) return;
  const int64_t i = s.img[a * G];
  const double xi = g.x[i], yi = g.y[i];
  const int ci = g.comp[i];
  const int64_t base = (q - q0) * m * m;
#pragma unroll 1
  for (int c = 0; c < 16; ++c) {
    const int64_t b = (int64_t)blockIdx.y * 64 + jl0 + 4 * c;
    if (b >= m) break;
    cd a0 = mk(0, 0), a1 = mk(0, 0), a2 = mk(0, 0);
#pragma unroll 1
    for (int l = 0; l < G; ++l) {
      const int64_t j = s.img[b * G + l];
      const cd sc = s.scale[b * G + l];
      D3 v;
      if (i == j) {
        v = diag_deriv<OP>(g, j, k);
      } else {
        const PairGeo p = pair_geo(g, i, j, xi, yi, ci);
        const Spec sp = specials_all<MH, MJ>(tv, p.r, k, p.same);
        v = offdiag_deriv<OP>(g, j, p.dx, p.dy, p.r, p.invr, p.same, p.Rij, p.lt, k, sp,
                              off_sign);
      }
      a0 = a0 + sc * v.a;
      a1 = a1 + sc * v.a1;
      a2 = a2 + sc * v.a2;
    }
    const int64_t idx = base + a + b * m;
    o0[idx] = a0;
    o1[idx] = a1;
    o2[idx] = a2;
  }
}

// Multi-irrep twin of k_assemble_red_pair: one specials evaluation per image
// term serves entry (a, b) and entry (b, a) of all nirr irreps at once.  The
// nirr mirror values of a thread are summed in LDS four columns at a time (24
// registers fewer) and written as four contiguous rows.  What bounds it is
// the registers: with envelope tables, five irreps of 1640 and 48 nodes took 30 ms
// while 85 of them were spilled, 17.4 ms with 30.  Diagonal tiles are assembled entry by entry.
// Outputs indexed as in k_assemble_red (matrix e * nz + q from the base).
template <int OP, int MH, int MJ, int MAXI>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2)))
k_assemble_red_pair_multi(DevGeom g, DevSym s, const cd* __restrict__ zk,
                          AsmTabs tb, int64_t q0, int64_t nz,
                          int T, cd* __restrict__ out64, cf* __restrict__ out32) {
  extern __shared__ __align__(16) cd smem[];
  const int64_t m = s.m;
  const int G = s.G;
  const int nirr = s.nirr;
  const int64_t q = q0 + blockIdx.z;
  int64_t p = blockIdx.x;
  int d = 0;
  while (p >= T - d) {
    p -= T - d;
    ++d;
  }
  const int Jt = (int)p, It = Jt + d;
  const auto tv = tab_view<MH>(tb, q, smem);
  const cd k = zk[q];
  const int il = threadIdx.x & 63;
  // the wave's column: uniform, so its node, images and weights are scalar loads
  const int jl0 = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t a = (int64_t)It * 64 + il;
  __shared__ cd mir[MAXI][64][5];  // mir[e][a_local][b_local % 4] = A_red[b, a]
  const bool aok = a < m;
  const bool diag_tile = (It == Jt);
  const int64_t mm = m * m;
  const int64_t i = s.img[(aok ? a : m - 1) * G];
  const double xi = g.x[i], yi = g.y[i];
  const int ci = g.comp[i];
#pragma unroll 1
  for (int c = 0; c < 16; ++c) {
    const int64_t b = (int64_t)Jt * 64 + jl0 + 4 * c;
    const bool ok = aok && b < m;
    cd acc[MAXI];
#pragma unroll
    for (int e = 0; e < MAXI; ++e) acc[e] = mir[e][il][jl0] = mk(0, 0);
    if (!ok) {
    } else if (diag_tile) {
#pragma unroll 1
      for (int l = 0; l < G; ++l) {
        const int64_t j = s.img[b * G + l];
        cd v;
        if (i == j) {
          v = diag_entry<OP>(g, j, k);
        } else {
          const PairGeo pg = pair_geo(g, i, j, xi, yi, ci);
          const Spec sp = specials<OP, MH, MJ>(tv, pg.r, k, pg.same || OP == QB_DLP_KRESS);
          v = offdiag_entry<OP>(g, i, j, pg.dx, pg.dy, pg.invr, pg.same, pg.Rij, pg.lt, k, sp);
        }
#pragma unroll
        for (int e = 0; e < MAXI; ++e)
          acc[e] = acc[e] + s.scale[((int64_t)(e < nirr ? e : 0) * m + b) * G + l] * v;
      }
    } else {
      const int64_t ib = s.img[b * G];
      const double xb = g.x[ib], yb = g.y[ib];
      const int cb = g.comp[ib];
#pragma unroll 1
      for (int l = 0; l < G; ++l) {
        const int64_t j = s.img[b * G + l];
        const int ls = s.inv[l];
        const int64_t jm = s.img[a * G + ls];
        const PairGeo p1 = pair_geo(g, i, j, xi, yi, ci);
        const PairGeo p2 = pair_geo(g, ib, jm, xb, yb, cb);  // its r equals p1.r
        const Spec sp = specials<OP, MH, MJ>(tv, p1.r, k,
                                             p1.same || p2.same || OP == QB_DLP_KRESS);
        const cd v1 = offdiag_entry<OP>(g, i, j, p1.dx, p1.dy, p1.invr, p1.same, p1.Rij, p1.lt,
                                        k, sp);
        const cd v2 = offdiag_entry<OP>(g, ib, jm, p2.dx, p2.dy, p1.invr, p2.same, p2.Rij,
                                        p2.lt, k, sp);
        // weights without a condition: behind branches on nirr their loads stood in
        // a row, ten waits per image
#pragma unroll
        for (int e = 0; e < MAXI; ++e) {
          const int64_t em = (int64_t)(e < nirr ? e : 0) * m;
          acc[e] = acc[e] + s.scale[(em + b) * G + l] * v1;
          mir[e][il][jl0] = mir[e][il][jl0] + s.scale[(em + a) * G + ls] * v2;
        }
      }
    }
#pragma unroll
    for (int e = 0; e < MAXI; ++e) {
      if (e >= nirr || !ok) break;
      const int64_t idx = ((int64_t)e * nz + q) * mm + a + b * m;
      if (out64) out64[idx] = acc[e];
      if (out32) out32[idx] = to_cf(acc[e]);
    }
    if (diag_tile) continue;  // uniform over the workgroup
    __syncthreads();
    {
      const int il2 = threadIdx.x >> 2, jr = threadIdx.x & 3;
      const int64_t a2 = (int64_t)It * 64 + il2, b2 = (int64_t)Jt * 64 + 4 * c + jr;
      if (a2 < m && b2 < m)
        for (int e = 0; e < nirr; ++e) {
          const int64_t idt = ((int64_t)e * nz + q) * mm + b2 + a2 * m;
          const cd v = mir[e][il2][jr];
          if (out64) out64[idt] = v;
          if (out32) out32[idt] = to_cf(v);
        }
    }
    __syncthreads();
  }
}

// o64 / o32: the output base (matrix 0); the kernels index matrix e * nz + q.
template <int OP, int MH, int MJ>
static void launch_red(qb_ctx* ctx, const qb_geom* g, const cd* z, int64_t q0, int64_t nzc,
                       int64_t nz, const DevTables& t, cd* o64, cf* o32) {
  const int64_t m = g->sym.m;
  const int nirr = g->sym.nirr;
  const unsigned Tm = (unsigned)((m + 63) / 64);
  const double ent = (double)m * m * nzc * nirr;
  int slot = qb_prof_begin(ctx, QB_K_ASSEMBLE, 0.0,
                           ent * ((o64 ? sizeof(cd) : 0) + (o32 ? sizeof(cf) : 0)));
  const dim3 grid(Tm, Tm, (unsigned)nzc);
  if (g->sym.pair && nirr == 1) {
    const int64_t pairs = (int64_t)Tm * (Tm + 1) / 2;
    hipLaunchKernelGGL((k_assemble_red_pair<OP, MH, MJ>), dim3((unsigned)pairs, 1, (unsigned)nzc),
                       dim3(256), 0, ctx->stream, g->d, g->sym, z, t.H, t.J, t.np_h, t.M_h,
                       t.np_j, t.M_j, t.rmin_h, t.rmax, q0, (int)Tm,
                       o64 ? o64 + q0 * m * m : nullptr, o32 ? o32 + q0 * m * m : nullptr);
  } else if (nirr == 1) {
    hipLaunchKernelGGL((k_assemble_red<OP, MH, MJ, 1>), grid, dim3(256), 0, ctx->stream, g->d,
                       g->sym, z, t.H, t.J, t.np_h, t.M_h, t.np_j, t.M_j, t.rmin_h, t.rmax, q0,
                       nz, o64, o32);
  } else if (g->sym.pair && nirr <= 8) {
    const int64_t pairs = (int64_t)Tm * (Tm + 1) / 2;
    hipLaunchKernelGGL((k_assemble_red_pair_multi<OP, MH, MJ, 8>),
                       dim3((unsigned)pairs, 1, (unsigned)nzc), dim3(256), 0, ctx->stream, g->d,
                       g->sym, z, AsmTabs{t, nullptr, 0, 0, nz}, q0, nz, (int)Tm, o64, o32);
  } else if (nirr <= 8) {
    hipLaunchKernelGGL((k_assemble_red<OP, MH, MJ, 8>), grid, dim3(256), 0, ctx->stream, g->d,
                       g->sym, z, t.H, t.J, t.np_h, t.M_h, t.np_j, t.M_j, t.rmin_h, t.rmax, q0,
                       nz, o64, o32);
  } else {
    hipLaunchKernelGGL((k_assemble_red<OP, MH, MJ, QB_MAX_IRREPS>), grid, dim3(256), 0,
                       ctx->stream, g->d, g->sym, z, t.H, t.J, t.np_h, t.M_h, t.np_j, t.M_j,
                       t.rmin_h, t.rmax, q0, nz, o64, o32);
  }
  qb_prof_end(ctx, slot);
}

template <int OP, int MH, int MJ>
static void launch_red_deriv(qb_ctx* ctx, const qb_geom* g, const cd* z, int64_t q0,
                             int64_t nzc, const DevTables& t, cd* o0, cd* o1, cd* o2,
                             double off_sign) {
  const int64_t m = g->sym.m;
  const unsigned Tm = (unsigned)((m + 63) / 64);
  int slot = qb_prof_begin(ctx, QB_K_ASSEMBLE, 0.0, 3.0 * (double)m * m * nzc * sizeof(cd));
  hipLaunchKernelGGL((k_assemble_red_deriv<OP, MH, MJ>), dim3(Tm, Tm, (unsigned)nzc), dim3(256),
                     0, ctx->stream, g->d, g->sym, z, t.H, t.J, t.np_h, t.M_h, t.np_j, t.M_j,
                     t.rmin_h, t.rmax, q0, o0, o1, o2, off_sign);
  qb_prof_end(ctx, slot);
}

template <int OP>
struct RedPairMulti {
  template <int MAXI>
  auto operator()() const {
    return k_assemble_red_pair_multi<OP, -1, -1, MAXI>;
  }
};

// Reduced matrices of 2 to 8 irreps with pair sharing, from envelope tables;
// other geometries return 1.  nz_out: wavenumbers of the whole output (irrep e's
// matrices start at e * nz_out).
int qb_assemble_red_env(qb_ctx* ctx, const qb_geom* g, int op, const cd* z_host, int64_t nz,
                        int64_t nz_out, double rmin, double rmax, cd* out64, cf* out32) {
  const int64_t m = g->sym.m;
  const int nirr = g->sym.nirr;
  if (m <= 0 || !g->sym.pair || nirr < 2 || nirr > 8 || nz > 1024) return 1;
  EnvTabs e;
  AsmTabs tb{};
  int rc = env_build(ctx, z_host, nz, rmin, rmax, &e, &tb);
  if (rc) return rc;
  const unsigned Tm = (unsigned)((m + 63) / 64);
  const double ent = (double)m * m * nz * nirr;
  const size_t lds = 2 * env_bytes(1, tb.P);
  int slot = qb_prof_begin(ctx, QB_K_ASSEMBLE, 0.0,
                           ent * ((out64 ? sizeof(cd) : 0) + (out32 ? sizeof(cf) : 0)));
  auto launch = [&](auto k) {
    // accumulators for the number of irreps: with room for eight the kernel spills
    auto kern = nirr <= 4 ? k.template operator()<4>() : nirr <= 6 ? k.template operator()<6>()
                                                                   : k.template operator()<8>();
    (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)lds);
    hipLaunchKernelGGL(kern, dim3(Tm * (Tm + 1) / 2, 1, (unsigned)nz), dim3(256), lds, ctx->stream,
                       g->d, g->sym, e.z, tb, (int64_t)0, nz_out, (int)Tm, out64, out32);
  };
  if (op == QB_CFIE_KRESS)
    launch(RedPairMulti<QB_CFIE_KRESS>());
  else
    launch(RedPairMulti<QB_DLP_KRESS>());
  qb_prof_end(ctx, slot);
  const hipError_t le = hipGetLastError(), se = hipStreamSynchronize(ctx->stream);
  env_free(ctx, &e);
  if (le != hipSuccess) return qb_fail(ctx, QB_E_HIP, hipGetErrorString(le));
  if (se != hipSuccess) return qb_fail(ctx, QB_E_HIP, hipGetErrorString(se));
  return QB_OK;
}

int qb_assemble_red_dev(qb_ctx* ctx, const qb_geom* g, int op, const cd* z_dev, int64_t nz,
                        const DevTables& t, cd* out64, cf* out32, int64_t nz_out) {
  if (nz_out == 0) nz_out = nz;
  for (int64_t q0 = 0; q0 < nz; q0 += 1024) {
    const int64_t nzc = nz - q0 < 1024 ? nz - q0 : 1024;
    const int mh = t.M_h, mj = t.M_j;
    if (op == QB_CFIE_KRESS) {
      if (mh == 7 && mj == 7)
        launch_red<QB_CFIE_KRESS, 7, 7>(ctx, g, z_dev, q0, nzc, nz_out, t, out64, out32);
      else if (mh == 5 && mj == 5)
        launch_red<QB_CFIE_KRESS, 5, 5>(ctx, g, z_dev, q0, nzc, nz_out, t, out64, out32);
      else
        launch_red<QB_CFIE_KRESS, 0, 0>(ctx, g, z_dev, q0, nzc, nz_out, t, out64, out32);
    } else {
      if (mh == 7 && mj == 7)
        launch_red<QB_DLP_KRESS, 7, 7>(ctx, g, z_dev, q0, nzc, nz_out, t, out64, out32);
      else if (mh == 5 && mj == 5)
        launch_red<QB_DLP_KRESS, 5, 5>(ctx, g, z_dev, q0, nzc, nz_out, t, out64, out32);
      else
        launch_red<QB_DLP_KRESS, 0, 0>(ctx, g, z_dev, q0, nzc, nz_out, t, out64, out32);
    }
    QB_HIP(ctx, hipGetLastError());
  }
  return QB_OK;
}

int qb_assemble_red_deriv_dev(qb_ctx* ctx, const qb_geom* g, int op, const cd* z_dev,
                              int64_t nz, const DevTables& t, cd* out, cd* dout, cd* ddout,
                              double off_sign) {
  const int64_t m = g->sym.m;
  for (int64_t q0 = 0; q0 < nz; q0 += 1024) {
    const int64_t nzc = nz - q0 < 1024 ? nz - q0 : 1024;
    const int64_t o = q0 * m * m;
    const int mh = t.M_h, mj = t.M_j;
    if (op == QB_CFIE_KRESS) {
      if (mh == 7 && mj == 7)
        launch_red_deriv<QB_CFIE_KRESS, 7, 7>(ctx, g, z_dev, q0, nzc, t, out + o, dout + o,
                                              ddout + o, off_sign);
      else
        launch_red_deriv<QB_CFIE_KRESS, 0, 0>(ctx, g, z_dev, q0, nzc, t, out + o, dout + o,
                                              ddout + o, off_sign);
    } else {
      if (mh == 7 && mj == 7)
        launch_red_deriv<QB_DLP_KRESS, 7, 7>(ctx, g, z_dev, q0, nzc, t, out + o, dout + o,
                                             ddout + o, off_sign);
      else
        launch_red_deriv<QB_DLP_KRESS, 0, 0>(ctx, g, z_dev, q0, nzc, t, out + o, dout + o,
                                             ddout + o, off_sign);
    }
    QB_HIP(ctx, hipGetLastError());
  }
  return QB_OK;
}
