/*
 * k_adjoint.hip -- discrete adjoint of the RK4 volume update (interior
 * stencil, CFS-PML, free surface); the fault part is in k_adj_fault.hip.
 *
 * One forward stage computes, at every physical point p,
 *   h(p) = H(p) . [D_d f(p)],  D_d f(p) = sum_t c_t f(p + (o_d + t) e_d)
 * (the 5-point one-sided operators of fd_t.cu:85-109 along each axis d,
 * o_d = -1 forward / -3 backward), where H(p) forms the physical gradients
 * g(f,a) = sum_d M[d][a] D_d f with the metric rows M[d] = (xi, eta, zeta)_{x,y,z}
 * and then momentum and Hooke's law (sv_curv_col_el_iso_gpu.cu:349-386).
 * Its transpose applied to an adjoint rhs c is
 *   lambda_f(q) = sum_d sum_t c_t kappa(f,d)(q - (o_d + t) e_d),
 *   kappa(f,d)(p) = sum_a M[d][a](p) gamma(f,a)(p),
 * where gamma are the adjoints of the physical gradients, formed pointwise
 * from c(p) and the media at p:
 *   stress fields: gamma from S = (1/rho) c_V (3 values),
 *   velocity fields: gamma(V,a) from the stress adjoints through Hooke's law
 *   (9 values G).
 * So each reverse stage is two kernels: k_adj_prep writes S and G at the
 * physical points (ghost entries stay zero: the forward never uses h at a
 * ghost), and k_adj_stage gathers the transposed operators with the metric
 * at each tap and does the pointwise RK-adjoint accumulations.
 *
 * CFS-PML (sv_curv_col_el_iso_gpu.cu:916-1288): at a point of face (d, side)
 * the forward adds (B-1) r_d - B a to the rhs and advances the auxiliary a
 * with rhs D r_d - A a, r_d being the part of the rhs from the derivatives
 * along d. Its transpose: the adjoint of r_d gains (B-1) c + D c_a, kept per
 * face as extra S and G (added by the gather at taps inside the face), and
 * the auxiliary's stage adjoint is -B c - A c_a, pointwise, with the same
 * reverse RK structure as the wavefield (c_a: the auxiliary rhs adjoint).
 *
 * Free surface (sv_curv_col_el_iso_gpu.cu:398-747, top four layers): the
 * forward replaces the velocity rhs by the traction-image form (timg) and
 * the stress rhs by Hooke's law on the reduced-order velocity gradient
 * (vlow), and the x/y PML faces add a term through the free-surface
 * matrices at the surface. Transposed: the prep leaves out the base S / G of
 * what was replaced and writes, for the points of the top four planes, the
 * adjoints of timg's momentum sums and of vlow's differences (12 values, the
 * surface PML term among them); the gather of the top five planes adds their
 * taps. A scatter of the same sums by atomic adds, one kernel more, took 26
 * of a stage's 52 us at 50 x 71 x 40: device-scope atomics leave the XCD's L2.
 *
 * Fault columns of split nodes (their rhs comes from the fault kernels) get
 * no S and G here and no top-layer sums; k_adj_fault.hip transposes them.
 *
 * RK4 (drv_rk_curv_col.cu:329-568) with a = {1/2, 1/2, 1}, b = {1/6, 1/3,
 * 1/3, 1/6}, ca = a dt, cb = b dt, reversed (E = adjoint of the step's
 * output, P = adjoint of its input):
 *   stage 3: A  = L3^T (cb3 E)
 *   stage 2: B  = L2^T (ca2 A + cb2 E),  P  = E + A
 *   stage 1: A  = L1^T (ca1 B + cb1 E),  P += B
 *   stage 0: P += A + L0^T (ca0 A + cb0 E)
 */
#include "cgfd_dev.h"
#include "cgfd_kernels.h"
#include "k_vol_common.h"

namespace cgfd {

/* S (3) and the 6 distinct entries of G of an adjoint rhs c with the media
   at the point: G is symmetric (gamma(Vx, y) = gamma(Vy, x) = mu c_xy and
   so on), so a point stores 9 values, not 12 */
constexpr int kSG = 9;
DEVI void sg_of(const float *c, float l, float m, float s, float *o) {
  const float l2m = l + 2.0f * m;
  o[0] = s * c[VX];
  o[1] = s * c[VY];
  o[2] = s * c[VZ];
  o[3] = l2m * c[TXX] + l * c[TYY] + l * c[TZZ];  /* gamma(Vx, x) */
  o[4] = l * c[TXX] + l2m * c[TYY] + l * c[TZZ];  /* gamma(Vy, y) */
  o[5] = l * c[TXX] + l * c[TYY] + l2m * c[TZZ];  /* gamma(Vz, z) */
  o[6] = m * c[TXY];                              /* gamma(Vx, y) = gamma(Vy, x) */
  o[7] = m * c[TXZ];                              /* gamma(Vx, z) = gamma(Vz, x) */
  o[8] = m * c[TYZ];                              /* gamma(Vy, z) = gamma(Vz, y) */
}

DEVI bool in_face(const AdjFace &F, int i, int j, int k) {
  return F.on && i >= F.i1 && i <= F.i2 && j >= F.j1 && j <= F.j2 && k >= F.k1 && k <= F.k2;
}
DEVI long face_idx(const AdjFace &F, int i, int j, int k) {
  return (long)(k - F.k1) * ((long)F.bn * F.an) + (long)(j - F.j1) * F.an + (i - F.ax0);
}

/* Tiles of the three kernels start at ghost-inclusive column 0, as the
   forward kernels' do: a 64-lane row of any array is then two whole 128-byte
   lines instead of parts of three, and one more tile for the last columns
   when ni mod 64 is 0, 62 or 63 moves no more lines than the row did before.
   160x240x100: k_adj_prep 200 -> 175 us, k_adj_stage 325 -> 258 us. */
constexpr int kTileW = 64;
static unsigned tiles_x(const Grid &g) { return (unsigned)((g.ni + 3 + kTileW - 1) / kTileW); }

/* entry e of the top-layer sums, plane nk2 - kk */
DEVI long top_idx(const Grid &g, int e, int kk, int i, int j) { return (long)(e * 4 + kk) * g.siz + i + (long)j * g.siy; }

/* Adjoints of the free-surface replacements' own sums at a point of the top
   four planes, from its rhs adjoint c: entries 0-2 of timg's sums (the taps'
   coef J xi_d times these), 3-5, 6-8, 9-11 of vlow's D_x, D_y, D_z of V (z:
   mac22 / mac24; at the surface D_z is a matrix of D_x and D_y). ax, ay: the
   surface PML term. */
DEVI void top_source(const Grid &g, const AdjTop &top, int i, int j, int k, long p, const float *c, float l, float m,
                     float s, const float *ax, const float *ay, int kdir) {
  const int kk = g.nk2 - k;
  const long sc = g.sicmp;
  float w[3] = {0.0f, 0.0f, 0.0f}, dl[3][3] = {};
  if (kk <= (kdir ? 3 : 1)) {
    const float sj = s / top.met[p];
#pragma unroll
    for (int cc = 0; cc < 3; cc++) w[cc] = c[cc] * sj;
  }
  if (kk <= 2) {
    const float l2m = (float)(l + 2.0 * m);
    float gm[3][3];  /* adjoint of the physical gradient dV_c/dx_a */
    gm[0][0] = l2m * c[TXX] + l * c[TYY] + l * c[TZZ];
    gm[1][1] = l * c[TXX] + l2m * c[TYY] + l * c[TZZ];
    gm[2][2] = l * c[TXX] + l * c[TYY] + l2m * c[TZZ];
    gm[0][1] = gm[1][0] = m * c[TXY];
    gm[0][2] = gm[2][0] = m * c[TXZ];
    gm[1][2] = gm[2][1] = m * c[TYZ];
#pragma unroll
    for (int d = 0; d < 3; d++) {
      const float e0 = top.met[(1 + 3 * d) * sc + p], e1 = top.met[(2 + 3 * d) * sc + p],
                  e2 = top.met[(3 + 3 * d) * sc + p];
#pragma unroll
      for (int cc = 0; cc < 3; cc++) dl[d][cc] = e0 * gm[cc][0] + e1 * gm[cc][1] + e2 * gm[cc][2];
    }
    if (kk == 0) {
      const long ij = ((long)i + (long)j * g.siy) * 9;
#pragma unroll
      for (int cc = 0; cc < 3; cc++) {
        float bx = ax[cc], by = ay[cc];
#pragma unroll
        for (int r = 0; r < 3; r++) {
          bx += top.mx[ij + 3 * r + cc] * dl[2][r];
          by += top.my[ij + 3 * r + cc] * dl[2][r];
        }
        dl[0][cc] += bx;
        dl[1][cc] += by;
      }
    }
  }
#pragma unroll
  for (int cc = 0; cc < 3; cc++) {
    top.src[top_idx(g, cc, kk, i, j)] = w[cc];
#pragma unroll
    for (int d = 0; d < 3; d++) top.src[top_idx(g, 3 + 3 * d + cc, kk, i, j)] = dl[d][cc];
  }
}

/* S and G from c = alpha X + beta E at physical points (X may be null);
   at CFS-PML points also the per-face extra S and G and the auxiliaries'
   reverse stage (MODE as k_adj_stage) */
template <int MODE>
__global__ void __launch_bounds__(256) k_adj_prep(Grid g, const float *__restrict__ lam, const float *__restrict__ mu,
                                                  const float *__restrict__ slw, const float *__restrict__ X,
                                                  float alpha, const float *__restrict__ E, float beta,
                                                  float *__restrict__ SG, AdjPml pm, AdjTop top, int kdir) {
  const int i = blockIdx.x * kTileW + (int)threadIdx.x, j = blockIdx.y * 4 + (int)threadIdx.y + 3;
  const int k = (int)blockIdx.z + 3;
  if (i < 3 || i >= g.ni + 3 || j >= g.nj + 3) return;
  const long sc = g.sicmp;
  const long p = i + j * g.siy + (long)k * g.siz;
  if (pm.fs.nfault > 0 && fault_column(pm.fs, i, j + (long)k * g.ny)) {
#pragma unroll
    for (int q = 0; q < kSG; q++) SG[q * sc + p] = 0.0f;
    if (top.src && g.nk2 - k < 4)
#pragma unroll
      for (int q = 0; q < 12; q++) top.src[top_idx(g, q, g.nk2 - k, i, j)] = 0.0f;
    return;
  }
  float c[9];
#pragma unroll
  for (int f = 0; f < 9; f++) c[f] = beta * E[f * sc + p] + (X ? alpha * X[f * sc + p] : 0.0f);
  const float l = lam[p], m = mu[p], s = slw[p];
  float o[kSG];
  sg_of(c, l, m, s, o);
  if (top.src) {
    /* what timg (velocity rhs) and vlow (stress rhs) replace at the top */
    if (k >= g.nk2 - (kdir ? 3 : 1)) o[0] = o[1] = o[2] = 0.0f;
    if (k >= g.nk2 - 2)
#pragma unroll
      for (int q = 3; q < kSG; q++) o[q] = 0.0f;
  }
#pragma unroll
  for (int q = 0; q < kSG; q++) SG[q * sc + p] = o[q];
  float ax[3] = {0.0f, 0.0f, 0.0f}, ay[3] = {0.0f, 0.0f, 0.0f};  /* surface PML term: adjoints of D_x V, D_y V */
#pragma unroll 1
  for (int fc = 0; pm.on && fc < 6; fc++) {
    const AdjFace &F = pm.f[fc];
    if (!in_face(F, i, j, k)) continue;
    const long ia = face_idx(F, i, j, k), n = F.n;
    const int ic = F.dim == 0 ? i - F.i1 : (F.dim == 1 ? j - F.j1 : k - F.k1);
    const float cA = F.A[ic], cB = F.B[ic], cD = F.D[ic];
    const float *Ea = F.lev + (long)pm.le * 9 * n, *Aa = F.lev + 9 * n, *Ba = F.lev + 18 * n;
    float *Pa = F.lev + (long)pm.lp * 9 * n;
    float *Aw = F.lev + 9 * n, *Bw = F.lev + 18 * n;
    const float *Xa = MODE == 3 ? nullptr : (MODE == 1 ? Ba : Aa);
    /* loads before stores, which may alias them for all the compiler knows: one
       wait per face instead of one per component */
    float dc[9], ev[9], xv[9], av[9], pv[9];
#pragma unroll
    for (int f = 0; f < 9; f++) {
      const long o2 = f * n + ia;
      ev[f] = Ea[o2];
      xv[f] = Xa ? Xa[o2] : 0.0f;
      av[f] = MODE == 2 || MODE == 0 ? Aa[o2] : (MODE == 1 ? Ba[o2] : 0.0f);
      pv[f] = MODE < 2 ? Pa[o2] : 0.0f;
    }
#pragma unroll
    for (int f = 0; f < 9; f++) {
      const long o2 = f * n + ia;
      const float ca_ = beta * ev[f] + (Xa ? alpha * xv[f] : 0.0f);  /* auxiliary rhs adjoint */
      dc[f] = (cB - 1.0f) * c[f] + cD * ca_;
      const float la = -cB * c[f] - cA * ca_;                          /* auxiliary stage adjoint */
      if (MODE == 3) Aw[o2] = la;
      else if (MODE == 2) { Bw[o2] = la; Pa[o2] = ev[f] + av[f]; }
      else if (MODE == 1) { Aw[o2] = la; Pa[o2] = pv[f] + av[f]; }
      else Pa[o2] = pv[f] + (av[f] + la);
    }
    sg_of(dc, l, m, s, o);
#pragma unroll
    for (int q = 0; q < kSG; q++) F.dsg[q * n + ia] = o[q];
    if (top.src && k == g.nk2 && fc < 4) {
      /* the free-surface term of the x/y PML faces: qT from D_dim V through
         the matrices, added to the stress rhs with (B-1) and to the auxiliary
         rhs with D (sv_curv_col_el_iso_gpu.cu:1000-1060, :1146-1205) */
      const float l2m = l + 2.0f * m;
      const float zx = top.met[7 * sc + p], zy = top.met[8 * sc + p], zz = top.met[9 * sc + p];
      const float q0 = l2m * zx * dc[TXX] + l * zx * dc[TYY] + l * zx * dc[TZZ] + m * zy * dc[TXY] + m * zz * dc[TXZ];
      const float q1 = l * zy * dc[TXX] + l2m * zy * dc[TYY] + l * zy * dc[TZZ] + m * zx * dc[TXY] + m * zz * dc[TYZ];
      const float q2 = l * zz * dc[TXX] + l * zz * dc[TYY] + l2m * zz * dc[TZZ] + m * zx * dc[TXZ] + m * zy * dc[TYZ];
      const float *X = (F.dim == 0 ? top.mx : top.my) + ((long)i + (long)j * g.siy) * 9;
#pragma unroll
      for (int cc = 0; cc < 3; cc++) {
        const float v = X[cc] * q0 + X[3 + cc] * q1 + X[6 + cc] * q2;
        if (F.dim == 0) ax[cc] += v;
        else ay[cc] += v;
      }
    }
  }
  if (top.src && g.nk2 - k < 4) top_source(g, top, i, j, k, p, c, l, m, s, ax, ay, kdir);
}

template <int DIR>
DEVI float tap_coef(int t) {
  return DIR ? (t == 0 ? CGFD_CF0 : t == 1 ? CGFD_CF1 : t == 2 ? CGFD_CF2 : t == 3 ? CGFD_CF3 : CGFD_CF4)
             : (t == 0 ? CGFD_CB0 : t == 1 ? CGFD_CB1 : t == 2 ? CGFD_CB2 : t == 3 ? CGFD_CB3 : CGFD_CB4);
}

/* S and G (and nothing else) of one tap; the entries the direction's metric
   row multiplies. AX = 0 or 1: only M[AX] is nonzero (the xi and eta rows on a
   grid of vertical columns, see acc_core); AX = -1: the full row */
template <int AX>
DEVI void load_sg(float *g, const float *__restrict__ SG, long sc, long p) {
#pragma unroll
  for (int q = 0; q < kSG; q++)
    if (AX == -1 || q < 3 || (AX == 0 && (q == 3 || q == 6 || q == 7)) || (AX == 1 && (q == 4 || q == 6 || q == 8)))
      g[q] = SG[q * sc + p];
}
/* add w * kappa(., d) for all nine fields from a tap's S and G (g) and metric
   row (M) */
template <int AX>
DEVI void add_kappa(float *lm, float w, const float *g, const float *M) {
  if (AX == 0) {
    const float u = w * M[0];
    lm[VX] += u * g[3];
    lm[VY] += u * g[6];
    lm[VZ] += u * g[7];
    lm[TXX] += u * g[0];
    lm[TXY] += u * g[1];
    lm[TXZ] += u * g[2];
  } else if (AX == 1) {
    const float u = w * M[1];
    lm[VX] += u * g[6];
    lm[VY] += u * g[4];
    lm[VZ] += u * g[8];
    lm[TYY] += u * g[1];
    lm[TXY] += u * g[0];
    lm[TYZ] += u * g[2];
  } else {
    lm[VX] += w * (M[0] * g[3] + M[1] * g[6] + M[2] * g[7]);
    lm[VY] += w * (M[0] * g[6] + M[1] * g[4] + M[2] * g[8]);
    lm[VZ] += w * (M[0] * g[7] + M[1] * g[8] + M[2] * g[5]);
    lm[TXX] += w * (M[0] * g[0]);
    lm[TYY] += w * (M[1] * g[1]);
    lm[TZZ] += w * (M[2] * g[2]);
    lm[TXY] += w * (M[0] * g[1] + M[1] * g[0]);
    lm[TXZ] += w * (M[0] * g[2] + M[2] * g[0]);
    lm[TYZ] += w * (M[1] * g[2] + M[2] * g[1]);
  }
}

/* the transposed operator along D (operator direction FW): the five taps'
   metric rows and S, G are loaded together, and only then, where a tap lies
   in a CFS-PML face of this direction, the faces' extra S and G, again
   together. (With the faces tested tap by tap the kernel waited for memory
   at every tap.) */
template <int D, int FW, int AX>
DEVI void gather_dir(float *lm, const Grid &g, const float *__restrict__ met, const float *__restrict__ SG,
                     const AdjPml &pm, int i, int j, int k, long q) {
  constexpr int o0 = FW ? -1 : -3;
  const long sc = g.sicmp, st = D == 0 ? 1 : (D == 1 ? g.siy : g.siz);
  float M[5][3], s[5][kSG];
#pragma unroll
  for (int t = 0; t < 5; t++) {
    const long p = q - (o0 + t) * st;
#pragma unroll
    for (int c = 0; c < 3; c++) M[t][c] = AX == -1 || AX == c ? met[(1 + 3 * D + c) * sc + p] : 0.0f;
    load_sg<AX>(s[t], SG, sc, p);
  }
#pragma unroll
  for (int t = 0; t < 5; t++) add_kappa<AX>(lm, tap_coef<FW>(t), s[t], M[t]);
  if (!pm.on) return;
  const int x = D == 0 ? i : (D == 1 ? j : k);
#pragma unroll 1
  for (int side = 0; side < 2; side++) {
    const AdjFace &F = pm.f[2 * D + side];
    if (!F.on) continue;
    const int lo = D == 0 ? F.i1 : (D == 1 ? F.j1 : F.k1), hi = D == 0 ? F.i2 : (D == 1 ? F.j2 : F.k2);
    /* some tap x - o0 - t, t = 0..4, in [lo, hi], and the other coordinates in the face */
    const bool near = x - o0 >= lo && x - o0 - 4 <= hi && (D == 0 || (i >= F.i1 && i <= F.i2)) &&
                      (D == 1 || (j >= F.j1 && j <= F.j2)) && (D == 2 || (k >= F.k1 && k <= F.k2));
    if (!near) continue;
    const long fs = D == 0 ? 1 : (D == 1 ? (long)F.an : (long)F.bn * F.an), f0 = face_idx(F, i, j, k);
#pragma unroll
    for (int t = 0; t < 5; t++) {
      const int tx = x - (o0 + t);
      const bool in = tx >= lo && tx <= hi;
#pragma unroll
      for (int e = 0; e < kSG; e++) s[t][e] = 0.0f;
      if (in) load_sg<AX>(s[t], F.dsg, F.n, f0 - (o0 + t) * fs);
    }
#pragma unroll
    for (int t = 0; t < 5; t++) add_kappa<AX>(lm, tap_coef<FW>(t), s[t], M[t]);
  }
}

/* the top-layer sums (top_source) gathered at a point of the top five planes:
   the transposes of timg, vlow and the surface PML term, added to lm. Points
   off the grid hold zeros. */
template <int ID, int JD, int KD>
DEVI void gather_top(float *lm, const Grid &g, const float *__restrict__ met, const float *__restrict__ src, int i,
                     int j, int k, long q) {
  const long sc = g.sicmp, sy = g.siy;
  const int kt = g.nk2 - k;
  constexpr int ox = ID ? -1 : -3, oy = JD ? -1 : -3, oz = KD ? -1 : -3;
  float M[10];
#pragma unroll
  for (int e = 0; e < 10; e++) M[e] = met[e * sc + q];
  float sx[3] = {0.0f, 0.0f, 0.0f}, sy_[3] = {0.0f, 0.0f, 0.0f}, sz_[3] = {0.0f, 0.0f, 0.0f};
  if (kt <= oz + 4) {
#pragma unroll
    for (int cc = 0; cc < 3; cc++)
#pragma unroll
      for (int t = 0; t < 5; t++) {
        sx[cc] += tap_coef<ID>(t) * src[top_idx(g, cc, kt, i, j) - (ox + t)];
        sy_[cc] += tap_coef<JD>(t) * src[top_idx(g, cc, kt, i, j) - (oy + t) * sy];
      }
  }
  if (kt <= 2) {
#pragma unroll
    for (int cc = 0; cc < 3; cc++)
#pragma unroll
      for (int t = 0; t < 5; t++)
        lm[cc] += tap_coef<ID>(t) * src[top_idx(g, 3 + cc, kt, i, j) - (ox + t)] +
                  tap_coef<JD>(t) * src[top_idx(g, 6 + cc, kt, i, j) - (oy + t) * sy];
  }
  if (kt > 0) {
    /* a tap of plane ks (nk2 - ks) on this plane, and the one above the
       surface whose odd image this plane is */
#pragma unroll
    for (int ks = 0; ks <= oz + 4; ks++) {
      const int n1 = ks - kt - oz, n2 = ks + kt - oz;
      float w = 0.0f;
#pragma unroll
      for (int t = 0; t < 5; t++) w += (n1 == t ? tap_coef<KD>(t) : 0.0f) - (n2 == t ? tap_coef<KD>(t) : 0.0f);
#pragma unroll
      for (int cc = 0; cc < 3; cc++) sz_[cc] += tap_mul(w, src[top_idx(g, cc, ks, i, j)]);
    }
  }
  {
    /* mac22 of plane 1 and mac24 of plane 2 */
    const float b1 = (float)kB1, b2 = (float)kB2, b3 = (float)kB3;
    const float w1 = KD ? (kt == 0 ? 1.0f : (kt == 1 ? -1.0f : 0.0f)) : (kt == 1 ? 1.0f : (kt == 2 ? -1.0f : 0.0f));
    const float w2 = KD ? (kt == 0 ? b3 : (kt == 1 ? b2 : (kt == 2 ? b1 : 0.0f)))
                        : (kt == 2 ? -b1 : (kt == 3 ? -b2 : (kt == 4 ? -b3 : 0.0f)));
#pragma unroll
    for (int cc = 0; cc < 3; cc++)
      lm[cc] += tap_mul(w1, src[top_idx(g, 9 + cc, 1, i, j)]) + tap_mul(w2, src[top_idx(g, 9 + cc, 2, i, j)]);
  }
  float t[3][3];
#pragma unroll
  for (int cc = 0; cc < 3; cc++)
#pragma unroll
    for (int a = 0; a < 3; a++) t[cc][a] = M[0] * (M[1 + a] * sx[cc] + M[4 + a] * sy_[cc] + M[7 + a] * sz_[cc]);
  lm[TXX] += t[0][0];
  lm[TYY] += t[1][1];
  lm[TZZ] += t[2][2];
  lm[TXY] += t[0][1] + t[1][0];
  lm[TXZ] += t[0][2] + t[2][0];
  lm[TYZ] += t[1][2] + t[2][1];
}

/* MODE 3: A = L^T;  2: B = L^T, P = E + A;  1: A = L^T, P += B;  0: P += A + L^T.
   VC: vertical columns (xi_y, xi_z, eta_x, eta_z left out, as the forward
   box split does).
   Bound by the L1 misses a CU can have in flight, so the 2 x 2 rows of a
   block share taps both ways: 160x240x100 258 us as 4 x 1 rows, 250 as 2 x 2;
   50x71x40 16.0, 14.5; 80x128x48 30.6, 31.7. */
template <int ID, int JD, int KD, int MODE, bool VC>
__global__ void __launch_bounds__(256, 4) k_adj_stage(Grid g, const float *__restrict__ met,
                                                   const float *__restrict__ SG, const float *__restrict__ E,
                                                   float *A, float *B, float *P, AdjPml pm, const float *__restrict__ src) {
  const int i = blockIdx.x * kTileW + (int)threadIdx.x, j = blockIdx.y * 2 + (int)threadIdx.y + 3;
  const int k = (int)(blockIdx.z * 2 + threadIdx.z) + 3;
  if (i < 3 || i >= g.ni + 3 || j >= g.nj + 3 || k > g.nk2) return;
  const long sc = g.sicmp, sy = g.siy, sz = g.siz;
  const long q = i + j * sy + (long)k * sz;
  float lm[9];
#pragma unroll
  for (int f = 0; f < 9; f++) lm[f] = 0.0f;
  gather_dir<0, ID, VC ? 0 : -1>(lm, g, met, SG, pm, i, j, k, q);
  __asm__ volatile("" : "+v"(lm[0]), "+v"(lm[1]), "+v"(lm[2]), "+v"(lm[3]), "+v"(lm[4]), "+v"(lm[5]),
                   "+v"(lm[6]), "+v"(lm[7]), "+v"(lm[8]) : : "memory");
  gather_dir<1, JD, VC ? 1 : -1>(lm, g, met, SG, pm, i, j, k, q);
  __asm__ volatile("" : "+v"(lm[0]), "+v"(lm[1]), "+v"(lm[2]), "+v"(lm[3]), "+v"(lm[4]), "+v"(lm[5]),
                   "+v"(lm[6]), "+v"(lm[7]), "+v"(lm[8]) : : "memory");
  gather_dir<2, KD, -1>(lm, g, met, SG, pm, i, j, k, q);
  if (src && g.nk2 - k <= 4) gather_top<ID, JD, KD>(lm, g, met, src, i, j, k, q);
  /* loads before stores */
  float av[9], pv[9];
#pragma unroll
  for (int f = 0; f < 9; f++) {
    const long o = f * sc + q;
    av[f] = MODE == 2 || MODE == 0 ? A[o] : (MODE == 1 ? B[o] : 0.0f);
    pv[f] = MODE == 2 ? E[o] : (MODE < 2 ? P[o] : 0.0f);
  }
#pragma unroll
  for (int f = 0; f < 9; f++) {
    const long o = f * sc + q;
    if (MODE == 3) A[o] = lm[f];
    else if (MODE == 2) { B[o] = lm[f]; P[o] = pv[f] + av[f]; }
    else if (MODE == 1) { A[o] = lm[f]; P[o] = pv[f] + av[f]; }
    else P[o] = pv[f] + (av[f] + lm[f]);
  }
}

/* P += residual row n at the stations (all nine components), the transpose
   of the recording: each term's node takes the residual times the term's
   weight fx fy fz (a station on a node: one term of weight 1) */
__global__ void k_adj_inject(const long *__restrict__ term, const float *__restrict__ fac, int nterm, int nsta,
                             const float *__restrict__ res, int nt, int n, long sicmp, float *P) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= nsta * 9 * nterm) return;
  const int u = t % nterm, sc = t / nterm;
  const int s = sc / 9, c = sc % 9;
  const float *f = fac + ((long)s * nterm + u) * 3;
  const float w = (f[0] * f[1]) * f[2];
  if (w == 0.0f) return;
  atomicAdd(P + c * sicmp + term[(long)s * nterm + u], res[((long)s * nt + n) * 9 + c] * w);
}

void launch_adj_prep(int mode, const Grid &g, const float *lam, const float *mu, const float *slw, const float *X,
                     float alpha, const float *E, float beta, float *SG, const AdjPml &pm, const AdjTop &top, int kdir,
                     hipStream_t st) {
  dim3 blk(kTileW, 4, 1), grd(tiles_x(g), (g.nj + 3) / 4, g.nk);
  switch (mode) {
    case 3:
      hipLaunchKernelGGL(k_adj_prep<3>, grd, blk, 0, st, g, lam, mu, slw, X, alpha, E, beta, SG, pm, top, kdir);
      break;
    case 2:
      hipLaunchKernelGGL(k_adj_prep<2>, grd, blk, 0, st, g, lam, mu, slw, X, alpha, E, beta, SG, pm, top, kdir);
      break;
    case 1:
      hipLaunchKernelGGL(k_adj_prep<1>, grd, blk, 0, st, g, lam, mu, slw, X, alpha, E, beta, SG, pm, top, kdir);
      break;
    default:
      hipLaunchKernelGGL(k_adj_prep<0>, grd, blk, 0, st, g, lam, mu, slw, X, alpha, E, beta, SG, pm, top, kdir);
      break;
  }
}

template <int ID, int JD, int KD, bool VC>
static void adj_stage_dir(int mode, const Grid &g, const float *met, const float *SG, const float *E, float *A,
                          float *B, float *P, const AdjPml &pm, const float *src, hipStream_t st) {
  dim3 blk(kTileW, 2, 2), grd(tiles_x(g), (g.nj + 1) / 2, (g.nk + 1) / 2);
  switch (mode) {
    case 3: hipLaunchKernelGGL((k_adj_stage<ID, JD, KD, 3, VC>), grd, blk, 0, st, g, met, SG, E, A, B, P, pm, src); break;
    case 2: hipLaunchKernelGGL((k_adj_stage<ID, JD, KD, 2, VC>), grd, blk, 0, st, g, met, SG, E, A, B, P, pm, src); break;
    case 1: hipLaunchKernelGGL((k_adj_stage<ID, JD, KD, 1, VC>), grd, blk, 0, st, g, met, SG, E, A, B, P, pm, src); break;
    default: hipLaunchKernelGGL((k_adj_stage<ID, JD, KD, 0, VC>), grd, blk, 0, st, g, met, SG, E, A, B, P, pm, src); break;
  }
}

template <bool VC>
static void adj_stage_vc(int mode, int idir, int jdir, int kdir, const Grid &g, const float *met, const float *SG,
                         const float *E, float *A, float *B, float *P, const AdjPml &pm, const float *src,
                         hipStream_t st) {
  switch (idir * 4 + jdir * 2 + kdir) {
    case 0: adj_stage_dir<0, 0, 0, VC>(mode, g, met, SG, E, A, B, P, pm, src, st); break;
    case 1: adj_stage_dir<0, 0, 1, VC>(mode, g, met, SG, E, A, B, P, pm, src, st); break;
    case 2: adj_stage_dir<0, 1, 0, VC>(mode, g, met, SG, E, A, B, P, pm, src, st); break;
    case 3: adj_stage_dir<0, 1, 1, VC>(mode, g, met, SG, E, A, B, P, pm, src, st); break;
    case 4: adj_stage_dir<1, 0, 0, VC>(mode, g, met, SG, E, A, B, P, pm, src, st); break;
    case 5: adj_stage_dir<1, 0, 1, VC>(mode, g, met, SG, E, A, B, P, pm, src, st); break;
    case 6: adj_stage_dir<1, 1, 0, VC>(mode, g, met, SG, E, A, B, P, pm, src, st); break;
    default: adj_stage_dir<1, 1, 1, VC>(mode, g, met, SG, E, A, B, P, pm, src, st); break;
  }
}

void launch_adj_stage(int mode, int idir, int jdir, int kdir, const Grid &g, const float *met, const float *SG,
                      const float *E, float *A, float *B, float *P, const AdjPml &pm, const float *src, int vcol,
                      hipStream_t st) {
  if (vcol) adj_stage_vc<true>(mode, idir, jdir, kdir, g, met, SG, E, A, B, P, pm, src, st);
  else adj_stage_vc<false>(mode, idir, jdir, kdir, g, met, SG, E, A, B, P, pm, src, st);
}

void launch_adj_inject(const long *term, const float *fac, int nterm, int nsta, const float *res, int nt, int n,
                       long sicmp, float *P, hipStream_t st) {
  const int nthr = nsta * 9 * nterm;
  if (nthr <= 0) return;
  hipLaunchKernelGGL(k_adj_inject, dim3((nthr + 255) / 256), dim3(256), 0, st, term, fac, nterm, nsta, res, nt, n,
                     sicmp, P);
}

}  // namespace cgfd
