/*
 * k_vol_common.h -- per-point pieces shared by the volume kernels: interior
 * rhs, CFS-PML correction + auxiliary update, fault-column ownership test and
 * the RK stage update.
 */
#ifndef CGFD_K_VOL_COMMON_H
#define CGFD_K_VOL_COMMON_H

#include "cgfd_dev.h"

namespace cgfd {

/* component order Vx,Vy,Vz,Txx,Tyy,Tzz,Tyz,Txz,Txy (wav_t.cu:56-106) */
enum { VX = 0, VY, VZ, TXX, TYY, TZZ, TYZ, TXZ, TXY };

/* interior rhs at a point (sv_curv_col_el_iso_gpu.cu:349-386) */
DEVI void rhs_interior(const float *Dx, const float *Dy, const float *Dz, float xx, float xy, float xz, float ex,
                       float ey, float ez, float zx, float zy, float zz, float l, float m, float s, float *h) {
  float l2m = l + 2.0f * m;
  h[VX] = s * (xx * Dx[TXX] + xy * Dx[TXY] + xz * Dx[TXZ] + ex * Dy[TXX] + ey * Dy[TXY] + ez * Dy[TXZ] + zx * Dz[TXX] + zy * Dz[TXY] + zz * Dz[TXZ]);
  h[VY] = s * (xx * Dx[TXY] + xy * Dx[TYY] + xz * Dx[TYZ] + ex * Dy[TXY] + ey * Dy[TYY] + ez * Dy[TYZ] + zx * Dz[TXY] + zy * Dz[TYY] + zz * Dz[TYZ]);
  h[VZ] = s * (xx * Dx[TXZ] + xy * Dx[TYZ] + xz * Dx[TZZ] + ex * Dy[TXZ] + ey * Dy[TYZ] + ez * Dy[TZZ] + zx * Dz[TXZ] + zy * Dz[TYZ] + zz * Dz[TZZ]);
  h[TXX] = l2m * (xx * Dx[VX] + ex * Dy[VX] + zx * Dz[VX]) + l * (xy * Dx[VY] + ey * Dy[VY] + zy * Dz[VY] + xz * Dx[VZ] + ez * Dy[VZ] + zz * Dz[VZ]);
  h[TYY] = l2m * (xy * Dx[VY] + ey * Dy[VY] + zy * Dz[VY]) + l * (xx * Dx[VX] + ex * Dy[VX] + zx * Dz[VX] + xz * Dx[VZ] + ez * Dy[VZ] + zz * Dz[VZ]);
  h[TZZ] = l2m * (xz * Dx[VZ] + ez * Dy[VZ] + zz * Dz[VZ]) + l * (xx * Dx[VX] + ex * Dy[VX] + zx * Dz[VX] + xy * Dx[VY] + ey * Dy[VY] + zy * Dz[VY]);
  h[TXY] = m * (xy * Dx[VX] + xx * Dx[VY] + ey * Dy[VX] + ex * Dy[VY] + zy * Dz[VX] + zx * Dz[VY]);
  h[TXZ] = m * (xz * Dx[VX] + xx * Dx[VZ] + ez * Dy[VX] + ex * Dy[VZ] + zz * Dz[VX] + zx * Dz[VZ]);
  h[TYZ] = m * (xz * Dx[VY] + xy * Dx[VZ] + ez * Dy[VY] + ey * Dy[VZ] + zz * Dz[VY] + zy * Dz[VZ]);
}


/* The auxiliary variables of a CFS-PML face follow the wavefield's RK
   bookkeeping (rk_point): stage s reads level pre, la, lb or lc and writes
   the next one; stage 3 writes t_{n+1} over la. */
DEVI const float *aux_input(const PmlFace &f, int istage) {
  return istage == 0 ? f.pre : (istage == 1 ? f.la : (istage == 2 ? f.lb : f.lc));
}

/* byte offset of (i, j, k) in one component of the face's arrays, which are
   smaller than a field */
DEVI unsigned face_off(const PmlFace &f, int i, int j, int k) {
  return (unsigned)(((k - f.k1) * f.bn + (j - f.j1)) * f.an + (i - f.ax0)) * 4u;
}

/* components C0 .. C0+NC-1 at byte offset oa; av: the stage input's values
   there (already read), ar: the auxiliary rhs */
template <int C0, int NC>
DEVI void aux_update(const PmlFace &f, const VolArgs &a, long poff, unsigned oa, const float *av, const float *ar) {
  poff += C0 * f.n;
  const float *pre = f.pre + poff;
  float pv[NC];
  if (a.istage < 3) {
    float *out = (a.istage == 0 ? f.la : (a.istage == 1 ? f.lb : f.lc)) + poff;
#pragma unroll
    for (int c = 0; c < NC; c++) pv[c] = a.istage == 0 ? av[c] : ld32(pre + c * f.n, oa);
#pragma unroll
    for (int c = 0; c < NC; c++) st32(out + c * f.n, oa, pv[c] + a.ca * ar[c]);
  } else {
    float *la = f.la + poff;
    const float *lb = f.lb + poff;
    float ev[NC], bv[NC];
#pragma unroll
    for (int c = 0; c < NC; c++) {
      pv[c] = ld32(pre + c * f.n, oa);
      ev[c] = ld32(la + c * f.n, oa);
      bv[c] = ld32(lb + c * f.n, oa);
    }
#pragma unroll
    for (int c = 0; c < NC; c++) st32(la + c * f.n, oa, rk_end(pv[c], ev[c], bv[c], av[c], a.cb * ar[c]));
  }
}

/* CFS-PML correction of every face containing (i,j,k) plus the auxiliary
   RK update (sv_curv_col_el_iso_gpu.cu:916-1288, drv_rk_curv_col.cu:368-567) */
DEVI void pml_point(const VolArgs &a, int i, int j, int k, long p, const float *Dx, const float *Dy, const float *Dz,
                    float l, float m, float s, float *h, long poff = 0) {
  const long sc = a.g.sicmp;
#pragma unroll 1
  for (int dim = 0; dim < 3; dim++) {
#pragma unroll 1
    for (int side = 0; side < 2; side++) {
      const PmlFace &f = a.pml[dim][side];
      if (!f.on) continue;
      if (i < f.i1 || i > f.i2 || j < f.j1 || j > f.j2 || k < f.k1 || k > f.k2) continue;
      const unsigned oa = face_off(f, i, j, k);
      int ic = dim == 0 ? i - f.i1 : (dim == 1 ? j - f.j1 : k - f.k1);
      float cD = f.D[ic], cA = f.A[ic], cB = f.B[ic];
      float cB1 = cB - 1.0f;
      const float *D = dim == 0 ? Dx : (dim == 1 ? Dy : Dz);
      const float *mr = a.met + (long)(1 + 3 * dim) * sc;
      float e1 = mr[p], e2 = mr[p + sc], e3 = mr[p + 2 * sc];
      float l2m = l + 2.0f * m;
      float r[9];
      r[VX] = s * (e1 * D[TXX] + e2 * D[TXY] + e3 * D[TXZ]);
      r[VY] = s * (e1 * D[TXY] + e2 * D[TYY] + e3 * D[TYZ]);
      r[VZ] = s * (e1 * D[TXZ] + e2 * D[TYZ] + e3 * D[TZZ]);
      r[TXX] = l2m * e1 * D[VX] + l * e2 * D[VY] + l * e3 * D[VZ];
      r[TYY] = l * e1 * D[VX] + l2m * e2 * D[VY] + l * e3 * D[VZ];
      r[TZZ] = l * e1 * D[VX] + l * e2 * D[VY] + l2m * e3 * D[VZ];
      r[TXY] = m * (e2 * D[VX] + e1 * D[VY]);
      r[TXZ] = m * (e3 * D[VX] + e1 * D[VZ]);
      r[TYZ] = m * (e3 * D[VY] + e2 * D[VZ]);
      const float *auxc = aux_input(f, a.istage) + poff;
      float av[9], ar[9];
#pragma unroll
      for (int c = 0; c < 9; c++) av[c] = ld32(auxc + c * f.n, oa);
#pragma unroll
      for (int c = 0; c < 9; c++) {
        h[c] += cB1 * r[c] - cB * av[c];
        ar[c] = cD * r[c] - cA * av[c];
      }
      if (dim < 2 && a.isfree && k == a.g.nk2) {
        /* free-surface contribution on x/y faces (:1000-1060, :1146-1205) */
        long ij = ((long)i + (long)j * a.g.siy) * 9;
        const float *X = (dim == 0 ? a.matVx2Vz : a.matVy2Vz) + ij;
        float q0 = X[0] * D[VX] + X[1] * D[VY] + X[2] * D[VZ];
        float q1 = X[3] * D[VX] + X[4] * D[VY] + X[5] * D[VZ];
        float q2 = X[6] * D[VX] + X[7] * D[VY] + X[8] * D[VZ];
        float zx = a.met[7 * sc + p], zy = a.met[8 * sc + p], zz = a.met[9 * sc + p];
        float qT[9];
        qT[TXX] = l2m * (zx * q0) + l * (zy * q1 + zz * q2);
        qT[TYY] = l2m * (zy * q1) + l * (zx * q0 + zz * q2);
        qT[TZZ] = l2m * (zz * q2) + l * (zx * q0 + zy * q1);
        qT[TXY] = m * (zy * q0 + zx * q1);
        qT[TXZ] = m * (zz * q0 + zx * q2);
        qT[TYZ] = m * (zz * q1 + zy * q2);
#pragma unroll
        for (int c = 3; c < 9; c++) {
          h[c] = (float)(h[c] + (cB - 1.0) * qT[c]);
          ar[c] += cD * qT[c];
        }
      }
      /* auxiliary RK update; the slab point is owned by this thread only */
      aux_update<0, 9>(f, a, poff, oa, av, ar);
    }
  }
}

DEVI bool fault_column(const FaultSkip &fs, int i, long pf) {
#pragma unroll 1
  for (int q = 0; q < fs.nfault; q++) {
    int d = i - fs.i0[q];
    if (d >= -3 && d <= 3 && fs.united[q][pf] == 0) return true;
  }
  return false;
}

/* RK stage update of the nine wavefield components at p: stages 0..2 write
   the next stage input pre + a_s dt h (wav_update, wav_t.cu:218-226),
   stage 3 the level at t_{n+1} over level A (rk_end). Every load stands
   before the first store: the compiler may not move a load over a store that
   could alias it, and a load, store, load, ... sequence waits for memory once
   per component (grouped, the top-layer kernel takes 0.034 ms per stage
   instead of 0.047 at 160 x 240 x 100) */
DEVI void rk_point(const VolArgs &a, long p, const float *h, long woff = 0) {
  const long sc = a.g.sicmp;
  p += woff;
  if (a.istage < 3) {
    float pv[9];
#pragma unroll
    for (int c = 0; c < 9; c++) pv[c] = a.pre[c * sc + p];
#pragma unroll
    for (int c = 0; c < 9; c++) a.tnew[c * sc + p] = pv[c] + a.ca * h[c];
  } else {
    float pv[9], ev[9], bv[9], cv[9];
#pragma unroll
    for (int c = 0; c < 9; c++) {
      pv[c] = a.pre[c * sc + p];
      ev[c] = a.end[c * sc + p];
      bv[c] = a.lb[c * sc + p];
      cv[c] = a.cur[c * sc + p];
    }
#pragma unroll
    for (int c = 0; c < 9; c++) a.end[c * sc + p] = rk_end(pv[c], ev[c], bv[c], cv[c], a.cb * h[c]);
  }
}

/* rk_point with 32-bit byte offsets (o = 4 p) from the scenario's levels,
   for components C0 .. C0+NC-1; the stage input's own value at stage 3 comes
   from the cache (the stencil has just read it). Loads first, as in
   rk_point. */
template <int C0, int NC>
DEVI void rk_part32(const VolArgs &a, unsigned o, const float *h, long woff) {
  const long sc = a.g.sicmp;
  woff += C0 * sc;
  const float *pre = a.pre + woff;
  float pv[NC];
#pragma unroll
  for (int c = 0; c < NC; c++) pv[c] = ld32nt(pre + c * sc, o);
  if (a.istage < 3) {
    float *tnew = a.tnew + woff;
#pragma unroll
    for (int c = 0; c < NC; c++) st32nt(tnew + c * sc, o, pv[c] + a.ca * h[c]);
  } else {
    float *end = a.end + woff;
    const float *lb = a.lb + woff, *cur = a.cur + woff;
    float ev[NC], bv[NC], cv[NC];
#pragma unroll
    for (int c = 0; c < NC; c++) {
      ev[c] = ld32nt(end + c * sc, o);
      bv[c] = ld32nt(lb + c * sc, o);
      cv[c] = ld32(cur + c * sc, o);
    }
#pragma unroll
    for (int c = 0; c < NC; c++) st32nt(end + c * sc, o, rk_end(pv[c], ev[c], bv[c], cv[c], a.cb * h[c]));
  }
}
/* in groups of three components: with all nine in flight the interior kernel
   takes 61 VGPRs instead of 43 and 1% longer at 400 x 800 x 266, one by one
   it is 1% faster there and 10-15% slower up to 160 x 240 x 100 (0.094 ->
   0.086 ms per stage) */
DEVI void rk_point32(const VolArgs &a, unsigned o, const float *h, long woff = 0) {
  rk_part32<0, 3>(a, o, h, woff);
  rk_part32<3, 3>(a, o, h + 3, woff);
  rk_part32<6, 3>(a, o, h + 6, woff);
}

}  // namespace cgfd

#endif
