// Cell arithmetic of the training kernels (D2Q9 and D3Q27): the learned
// collision around its MLP and the adjoint of it, the layouts of the parameter
// vector and of the per-cell record.  The formulas stand in lbm_train.hip.
#pragma once

#include "lbm_step_impl.h"

namespace lbm {

constexpr int HID = LBM_LEARNED_HIDDEN;
constexpr int NPARAM = HID * 6 + HID + HID * HID + HID + 3 * HID + 3;  // 1379
constexpr int NREC = 6 + HID + HID + HID + HID + 3;                    // 137

// offsets of the parameter vector [W1 (32x6), b1, W2 (32x32), b2, W3 (3x32), b3]
constexpr int P_W1 = 0, P_B1 = P_W1 + HID * 6, P_W2 = P_B1 + HID, P_B2 = P_W2 + HID * HID,
              P_W3 = P_B2 + HID, P_B3 = P_W3 + 3 * HID;
// offsets of the per-cell record [x (6), a1, a2, dz1, dz2, do (3)]
constexpr int R_X = 0, R_A1 = 6, R_A2 = R_A1 + HID, R_DZ1 = R_A2 + HID, R_DZ2 = R_DZ1 + HID,
              R_DO = R_DZ2 + HID;
static_assert(P_B3 + 3 == NPARAM, "parameter count");
static_assert(R_DO + 3 == NREC, "record size");

struct TrainArgs {
  const void* params;  // NPARAM values of the arithmetic type
  double in_scale, rate_lo, rate_hi;
};

// D2Q9 raw moment rows T, N, Pxy, xxy, xyy, xxyy (as 9-vectors)
__device__ constexpr int MROW[6][9] = {
    {0, 1, 1, 1, 1, 2, 2, 2, 2},    {0, 1, -1, 1, -1, 0, 0, 0, 0},
    {0, 0, 0, 0, 0, 1, -1, 1, -1},  {0, 0, 0, 0, 0, 1, 1, -1, -1},
    {0, 0, 0, 0, 0, 1, -1, -1, 1},  {0, 0, 0, 0, 0, 1, 1, 1, 1}};
__device__ constexpr double PHI_D[3][9] = {
    {0., 0., -0.5, 0., 0.5, 0.25, 0.25, -0.25, -0.25},
    {0., -0.5, 0., 0.5, 0., 0.25, -0.25, -0.25, 0.25},
    {1., -0.5, -0.5, -0.5, -0.5, 0.25, 0.25, 0.25, 0.25}};

// ---------------------------------------------------------------------------
// D3Q27 raw moments.  t[a][b][c] is the moment x^a y^b z^c (a, b, c <= 2);
// population q sits at t[e_x + 1][e_y + 1][e_z + 1] before the transform.
// The basis is the tensor product of the 1D moments (1, x, x^2) at
// x in {-1, 0, 1}, so M, M^-1 and their transposes are one 3-point map
// along each of the three axes.
// ---------------------------------------------------------------------------
template <int AXIS, class C, class F>
__device__ __forceinline__ void map_axis(C (&t)[3][3][3], const F& A) {
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      if constexpr (AXIS == 0) A(t[0][i][j], t[1][i][j], t[2][i][j]);
      else if constexpr (AXIS == 1) A(t[i][0][j], t[i][1][j], t[i][2][j]);
      else A(t[i][j][0], t[i][j][1], t[i][j][2]);
    }
}
template <class C, class F>
__device__ __forceinline__ void map_all(C (&t)[3][3][3], const F& A) {
  map_axis<0>(t, A);
  map_axis<1>(t, A);
  map_axis<2>(t, A);
}

// t <- M v
template <class C>
__device__ __forceinline__ void m27_moments(const C (&v)[27], C (&t)[3][3][3]) {
  using S = D3Q27;
#pragma unroll
  for (int q = 0; q < 27; ++q) t[S::e[q][0] + 1][S::e[q][1] + 1][S::e[q][2] + 1] = v[q];
  map_all(t, [](C& a, C& b, C& c) {  // (v-, v0, v+) -> (v- + v0 + v+, v+ - v-, v+ + v-)
    const C m0 = a + b + c, m1 = c - a, m2 = c + a;
    a = m0, b = m1, c = m2;
  });
}

// v <- v + sign * (M^-1 t); t is overwritten
template <class C>
__device__ __forceinline__ void m27_add_inverse(C (&t)[3][3][3], C sign, C (&v)[27]) {
  using S = D3Q27;
  map_all(t, [](C& a, C& b, C& c) {  // (m0, m1, m2) -> ((m2 - m1)/2, m0 - m2, (m1 + m2)/2)
    const C vm = C(0.5) * (c - b), v0 = a - c, vp = C(0.5) * (b + c);
    a = vm, b = v0, c = vp;
  });
#pragma unroll
  for (int q = 0; q < 27; ++q) v[q] += sign * t[S::e[q][0] + 1][S::e[q][1] + 1][S::e[q][2] + 1];
}

// nu <- (M^-1)^T lam
template <class C>
__device__ __forceinline__ void m27_inverse_transposed(const C (&lam)[27], C (&nu)[3][3][3]) {
  using S = D3Q27;
#pragma unroll
  for (int q = 0; q < 27; ++q) nu[S::e[q][0] + 1][S::e[q][1] + 1][S::e[q][2] + 1] = lam[q];
  map_all(nu, [](C& a, C& b, C& c) {  // (l-, l0, l+) -> (l0, (l+ - l-)/2, (l- + l+)/2 - l0)
    const C n0 = b, n1 = C(0.5) * (c - a), n2 = C(0.5) * (a + c) - b;
    a = n0, b = n1, c = n2;
  });
}

// v <- v + M^T g; g is overwritten
template <class C>
__device__ __forceinline__ void m27_add_transposed(C (&g)[3][3][3], C (&v)[27]) {
  using S = D3Q27;
  map_all(g, [](C& a, C& b, C& c) {  // (g0, g1, g2) -> (g0 - g1 + g2, g0, g0 + g1 + g2)
    const C vm = a - b + c, v0 = a, vp = a + b + c;
    a = vm, b = v0, c = vp;
  });
#pragma unroll
  for (int q = 0; q < 27; ++q) v[q] += g[S::e[q][0] + 1][S::e[q][1] + 1][S::e[q][2] + 1];
}

// 1D moments sum_x W(x) x^p of W(0) = 2/3, W(+-1) = 1/6, whose products are
// the D3Q27 weights, and their products P3(a, b, c) = raw moment abc of w
__host__ __device__ constexpr double mu1d(int p) {
  return p == 0 ? 1.0 : (p % 2 ? 0.0 : 1.0 / 3.0);
}
__host__ __device__ constexpr double p3(int a, int b, int c) { return mu1d(a) * mu1d(b) * mu1d(c); }

// raw moment abc of feq(rho, u) / rho for the quadratic equilibrium
// feq = w rho (1 + 3 e.u + 4.5 (e.u)^2 - 1.5 u.u), and its derivatives in u
template <class C>
__device__ __forceinline__ C meq_unit(int a, int b, int c, const C (&u)[3], C (&du)[3]) {
  const C uu = u[0] * u[0] + u[1] * u[1] + u[2] * u[2];
  const int ex[3][3] = {{1, 0, 0}, {0, 1, 0}, {0, 0, 1}};
  C m = (C)p3(a, b, c) * (C(1) - C(1.5) * uu);
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const C pd = (C)p3(a + ex[d][0], b + ex[d][1], c + ex[d][2]);
    m += C(3) * u[d] * pd;
    du[d] = C(-3) * u[d] * (C)p3(a, b, c) + C(3) * pd;
#pragma unroll
    for (int e = 0; e < 3; ++e) {
      const C pde = (C)p3(a + ex[d][0] + ex[e][0], b + ex[d][1] + ex[e][1], c + ex[d][2] + ex[e][2]);
      m += C(4.5) * u[d] * u[e] * pde;
      du[d] += C(9) * u[e] * pde;
    }
  }
  return m;
}

// relaxation weight of moment abc: 1/tau on order 2, r_0 / r_1 / r_2 on
// orders 3 / 4 / 5-6, 0 on orders 0 and 1; g = the rate group (-1: none)
__device__ __forceinline__ int m27_group(int a, int b, int c) {
  const int o = a + b + c;
  return o <= 2 ? -1 : (o == 3 ? 0 : (o == 4 ? 1 : 2));
}


// ---------------------------------------------------------------------------
// One cell's collision around the MLP: features() takes the pulled
// populations to the MLP's inputs F.x, update() applies the clamped rates r;
// adjoint_rates() gives dL/dr (q) for the output adjoint lam, and adjoint()
// the input adjoint mu once dL/dx (gx) is known.
// ---------------------------------------------------------------------------
template <class C>
struct CellFwd27 {
  C rho, ri, u[3], t[3][3][3], x[6];
};
// what adjoint_rates leaves for adjoint
template <class C>
struct CellAdj27 {
  C nu[3][3][3];
};

template <class C>
__device__ __forceinline__ void features(const C (&g)[27], C s, CellFwd27<C>& F) {
  m27_moments(g, F.t);
  F.rho = F.t[0][0][0];
  F.ri = C(1) / F.rho;
  F.u[0] = F.t[1][0][0] * F.ri;
  F.u[1] = F.t[0][1][0] * F.ri;
  F.u[2] = F.t[0][0][1] * F.ri;
#pragma unroll
  for (int a = 0; a < 3; ++a)
#pragma unroll
    for (int b = 0; b < 3; ++b)
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        if (a + b + c <= 1) continue;
        C du[3];
        F.t[a][b][c] -= F.rho * meq_unit(a, b, c, F.u, du);
      }
  const C xx = F.t[2][0][0], yy = F.t[0][2][0], zz = F.t[0][0][2];
  const C sc = s * F.ri;
  F.x[0] = (xx + yy + zz) * sc;
  F.x[1] = (xx - zz) * sc;
  F.x[2] = (yy - zz) * sc;
  F.x[3] = F.t[1][1][0] * sc;
  F.x[4] = F.t[1][0][1] * sc;
  F.x[5] = F.t[0][1][1] * sc;
}

template <class C>
__device__ __forceinline__ void update(const C (&g)[27], const CellFwd27<C>& F, const C (&r)[3],
                                       C tau_inv, C (&out)[27]) {
  C y[3][3][3];
#pragma unroll
  for (int a = 0; a < 3; ++a)
#pragma unroll
    for (int b = 0; b < 3; ++b)
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const int o = a + b + c, grp = m27_group(a, b, c);
        y[a][b][c] = o <= 1 ? C(0) : (grp < 0 ? tau_inv : r[grp]) * F.t[a][b][c];
      }
#pragma unroll
  for (int q = 0; q < 27; ++q) out[q] = g[q];
  m27_add_inverse(y, C(-1), out);
}

template <class C>
__device__ __forceinline__ void adjoint_rates(const C (&lam)[27], const CellFwd27<C>& F,
                                              CellAdj27<C>& A, C (&q)[3]) {
  // out = g - Phi y, y = w . t: dL/dy = -Phi^T lam
  m27_inverse_transposed(lam, A.nu);
  q[0] = q[1] = q[2] = 0;
#pragma unroll
  for (int a = 0; a < 3; ++a)
#pragma unroll
    for (int b = 0; b < 3; ++b)
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const int grp = m27_group(a, b, c);
        if (grp >= 0) q[grp] += F.t[a][b][c] * -A.nu[a][b][c];
      }
}

template <class C>
__device__ __forceinline__ void adjoint(const C (&lam)[27], const CellFwd27<C>& F,
                                        const CellAdj27<C>& A, const C (&r)[3], const C (&gx)[6],
                                        C tau_inv, C s, C (&mu)[27]) {
  C gt[3][3][3];
#pragma unroll
  for (int a = 0; a < 3; ++a)
#pragma unroll
    for (int b = 0; b < 3; ++b)
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const int o = a + b + c, grp = m27_group(a, b, c);
        gt[a][b][c] = o <= 1 ? C(0) : (grp < 0 ? tau_inv : r[grp]) * -A.nu[a][b][c];
      }
  // x = s / rho (T, Nxz, Nyz, Pxy, Pxz, Pyz) of t
  const C sc = s * F.ri;
  C grho = 0;
#pragma unroll
  for (int k = 0; k < 6; ++k) grho -= gx[k] * F.x[k] * F.ri;
  gt[2][0][0] += sc * (gx[0] + gx[1]);
  gt[0][2][0] += sc * (gx[0] + gx[2]);
  gt[0][0][2] += sc * (gx[0] - gx[1] - gx[2]);
  gt[1][1][0] += sc * gx[3];
  gt[1][0][1] += sc * gx[4];
  gt[0][1][1] += sc * gx[5];
  // t = M g - rho meq_unit(u) on orders >= 2
  C gu[3] = {0, 0, 0};
#pragma unroll
  for (int a = 0; a < 3; ++a)
#pragma unroll
    for (int b = 0; b < 3; ++b)
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        if (a + b + c <= 1) continue;
        C du[3];
        const C m = meq_unit(a, b, c, F.u, du);
        grho -= gt[a][b][c] * m;
#pragma unroll
        for (int d = 0; d < 3; ++d) gu[d] -= gt[a][b][c] * F.rho * du[d];
      }
  // u = j / rho, rho = (M g)_000, j = (M g)_100, _010, _001
  gt[0][0][0] = grho;
  gt[1][0][0] = gu[0] * F.ri;
  gt[0][1][0] = gu[1] * F.ri;
  gt[0][0][1] = gu[2] * F.ri;
  gt[0][0][0] -= (gu[0] * F.u[0] + gu[1] * F.u[1] + gu[2] * F.u[2]) * F.ri;
#pragma unroll
  for (int q = 0; q < 27; ++q) mu[q] = lam[q];
  m27_add_transposed(gt, mu);
}

template <class C>
struct CellFwd9 {
  C rho, ri, u[3], fe[9], ds[9], x[6], mg[3];
};
template <class C>
struct CellAdj9 {
  C lp[3];
};

template <class C>
__device__ __forceinline__ void features(const C (&g)[9], C s, CellFwd9<C>& F) {
  using S = D2Q9;
  moments<S, C>(g, F.rho, F.u);
  F.ri = C(1) / F.rho;
  equilibrium<S, C>(F.rho, F.u, F.fe);
  C df[9];
#pragma unroll
  for (int q = 0; q < 9; ++q) df[q] = g[q] - F.fe[q];
  kbc_shear<S, C>(df, F.ds);
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    C m = 0;
#pragma unroll
    for (int q = 0; q < 9; ++q)
      if (MROW[k][q]) m += MROW[k][q] * df[q];
    F.x[k] = s * F.ri * m;
  }
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    C m = 0;
#pragma unroll
    for (int q = 0; q < 9; ++q)
      if (MROW[3 + k][q]) m += MROW[3 + k][q] * (df[q] - F.ds[q]);
    F.mg[k] = m;
  }
}

template <class C>
__device__ __forceinline__ void update(const C (&g)[9], const CellFwd9<C>& F, const C (&r)[3],
                                       C tau_inv, C (&out)[9]) {
#pragma unroll
  for (int q = 0; q < 9; ++q) {
    C upd = 0;
#pragma unroll
    for (int k = 0; k < 3; ++k) upd += r[k] * F.mg[k] * (C)PHI_D[k][q];
    out[q] = g[q] - F.ds[q] * tau_inv - upd;
  }
}

template <class C>
__device__ __forceinline__ void adjoint_rates(const C (&lam)[9], const CellFwd9<C>& F, CellAdj9<C>& A,
                                              C (&q)[3]) {
  // out = g - ds tau_inv - sum_k r_k mg_k phi_k
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    C lp = 0;
#pragma unroll
    for (int i = 0; i < 9; ++i) lp += lam[i] * (C)PHI_D[k][i];
    A.lp[k] = lp;
    q[k] = -F.mg[k] * lp;
  }
}

template <class C>
__device__ __forceinline__ void adjoint(const C (&lam)[9], const CellFwd9<C>& F, const CellAdj9<C>& A,
                                        const C (&r)[3], const C (&gx)[6], C tau_inv, C s,
                                        C (&mu)[9]) {
  using S = D2Q9;
  C gmg[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) gmg[k] = -r[k] * A.lp[k];
  // mg = rows of dh, dh = df - ds
  C gds[9], gdf[9];
#pragma unroll
  for (int q = 0; q < 9; ++q) {
    C v = 0;
#pragma unroll
    for (int k = 0; k < 3; ++k)
      if (MROW[3 + k][q]) v += MROW[3 + k][q] * gmg[k];
    gds[q] = -lam[q] * tau_inv - v;
    gdf[q] = v;
  }
  // ds from (T, N, Pxy): ds0 = -T, ds1 = ds3 = (T+N)/4, ds2 = ds4 = (T-N)/4,
  // ds5 = ds7 = Pxy/4, ds6 = ds8 = -Pxy/4
  const C gT = -gds[0] + C(0.25) * (gds[1] + gds[3] + gds[2] + gds[4]);
  const C gN = C(0.25) * (gds[1] + gds[3] - gds[2] - gds[4]);
  const C gP = C(0.25) * (gds[5] + gds[7] - gds[6] - gds[8]);
  // T = xx + yy, N = xx - yy; xx, yy, Pxy are rows of df
  const C gxx = gT + gN, gyy = gT - gN;
#pragma unroll
  for (int q = 1; q < 9; ++q) {
    const int ex = S::e[q][0], ey = S::e[q][1];
    if (ex != 0) gdf[q] += gxx;
    if (ey != 0) gdf[q] += gyy;
    if (ex * ey != 0) gdf[q] += (ex * ey > 0) ? gP : -gP;
  }
  // x_k = s / rho * M_k df
  C grho = 0;
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    grho -= gx[k] * F.x[k] * F.ri;
#pragma unroll
    for (int q = 0; q < 9; ++q)
      if (MROW[k][q]) gdf[q] += s * F.ri * gx[k] * MROW[k][q];
  }
  // df = g - feq(rho, u), feq = w rho (1 + 3 eu - 3/2 uu + 9/2 eu^2)
  C gu[2] = {0, 0};
#pragma unroll
  for (int q = 0; q < 9; ++q) {
    const C gfe = -gdf[q];
    grho += gfe * F.fe[q] * F.ri;
    const C eu = S::e[q][0] * F.u[0] + S::e[q][1] * F.u[1];
    const C c = gfe * (C)S::w[q] * F.rho;
#pragma unroll
    for (int d = 0; d < 2; ++d)
      gu[d] += c * (C(3) * S::e[q][d] - C(3) * F.u[d] + C(9) * eu * S::e[q][d]);
  }
  // u = j / rho
  C gj[2];
#pragma unroll
  for (int d = 0; d < 2; ++d) {
    gj[d] = gu[d] * F.ri;
    grho -= gu[d] * F.u[d] * F.ri;
  }
#pragma unroll
  for (int q = 0; q < 9; ++q)
    mu[q] = lam[q] + gdf[q] + grho + gj[0] * S::e[q][0] + gj[1] * S::e[q][1];
}

template <class S, class C>
using CellFwd = std::conditional_t<S::Q == 9, CellFwd9<C>, CellFwd27<C>>;
template <class S, class C>
using CellAdj = std::conditional_t<S::Q == 9, CellAdj9<C>, CellAdj27<C>>;

// cell index c -> (i0, i1, i2) and the periodic neighbour tables
__device__ __forceinline__ void cell_tables(const KParams& p, int64_t c, int (&a0)[3], int (&a1)[3],
                                            int (&a2)[3]) {
  const int i2 = (int)(c % p.n2);
  const int64_t r = c / p.n2;
  const int i1 = (int)(r % p.n1), i0 = (int)(r / p.n1);
  axis_offsets(i0, p.n0, (int)p.s0, a0);  // fewer than 2^31 populations
  axis_offsets(i1, p.n1, p.s1, a1);
  axis_offsets(i2, p.n2, 1, a2);
}

}  // namespace lbm
