/*
 * k_adj_fault.hip -- discrete adjoint of the fault part of one RK stage
 * (split-node slip-weakening fault, k_fault.hip) and of the per-step fault
 * accumulators, for the reverse sweep of k_adjoint.hip.
 *
 * Forward stage (k_fault.hip, drv_rk_curv_col.cu:215-568):
 *   1 wave2fault   welded nodes copy the stage input onto both split nodes
 *   2 trial_t1     traction columns T1 slots 0-2, 4-6 from the stress
 *   3 trial        trial traction, friction -> T1 slot 3; split-node average
 *                  written onto the stage input at the plane (fault2wave)
 *   4 volume/top   every point but the fault columns of split nodes
 *   5 fault_cols   the six columns next to the plane
 *   6 fault_nodes  split-node rates and RK, fault2wave onto the stage output;
 *                  at the last stage Slip += |V_s| dt, hT1, mT1
 * Everything but the friction law (trial_slipweakening.cu:296-364) and the
 * slip-rate magnitude (fault_wav_t.cu:219-262) is linear with coefficients
 * fixed at setup, so the reverse sweep needs no recomputed forward state:
 * the forward kernels record a tape per step and node (the trial traction of
 * each stage, Slip at the step start, the split-node velocity jump of the
 * last stage), from which the friction branch and its derivatives follow.
 *
 * The value fault2wave writes onto the stage output at the plane is
 * overwritten by the next stage's trial before anything reads it; only the
 * last stage's (the step's end level) is seen, by the station records and
 * the surface maxima at the next step start. The value the trial writes
 * onto the stage input is what the neighbours' stencils read.
 *
 * Reverse of one stage (the node kernels are the scatter transposes of their
 * forward gathers, same lanes and addresses, with atomic adds where lanes
 * share a target; k_adjf_cols, with by far the most taps, is a gather):
 *   k_adjf_lev   RK structure of the split-node levels (as the wavefield's)
 *   [wave prep / stage, fault columns left out]
 *   k_adjf_cols  5^T into the wavefield adjoint, T1 slot 3, split velocity
 *   k_adjf_nodes 6^T into T1, neighbouring split-node state, hT1
 *   k_adjf_trial 3^T (fault2wave, friction on the taped branch, trial) and
 *                2^T; parameter gradients
 *   k_adjf_w2f   1^T at welded nodes
 * and once per step, before the last stage: k_adjf_begin (accumulators
 * and the end-level fault2wave).
 */
#include "cgfd_dev.h"
#include "cgfd_kernels.h"

namespace cgfd {

enum { VX = 0, VY, VZ, TXX, TYY, TZZ, TYZ, TXZ, TXY };

DEVI long fidx(int c, int m, long ss) { return (long)(2 * c + m) * ss; }

/* per-fault adjoint block, offsets in units of sslice */
constexpr int kOffT1 = 72, kOffHT1 = 93, kOffMT1 = 96, kOffSlip = 99, kOffGrad = 100, kOffSlip12 = 107,
              kOffVsr = 109;

DEVI void aadd(float *p, float v) { atomicAdd(p, v); }
/* transposes of the fd_t.h difference macros: add a * d(op)/d(tap) */
DEVI void t_mac22(float *p, long s, int f, float a) {
  if (f == 1) { aadd(p + s, a); aadd(p, -a); }
  else { aadd(p, a); aadd(p - s, -a); }
}
DEVI void t_mac24(float *p, long s, int f, float a) {
  const float b1 = (float)kB1, b2 = (float)kB2, b3 = (float)kB3;
  if (f == 1) { aadd(p, b1 * a); aadd(p + s, b2 * a); aadd(p + 2 * s, b3 * a); }
  else { aadd(p, -b1 * a); aadd(p - s, -b2 * a); aadd(p - 2 * s, -b3 * a); }
}
DEVI void t_macdrp(float *p, long s, int f, float a) {
  const float c1 = (float)kC1, c2 = (float)kC2, c3 = (float)kC3, c4 = (float)kC4, c5 = (float)kC5;
  if (f == 1) {
    aadd(p - s, c1 * a); aadd(p, c2 * a); aadd(p + s, c3 * a); aadd(p + 2 * s, c4 * a); aadd(p + 3 * s, c5 * a);
  } else {
    aadd(p + s, -c1 * a); aadd(p, -c2 * a); aadd(p - s, -c3 * a); aadd(p - 2 * s, -c4 * a); aadd(p - 3 * s, -c5 * a);
  }
}
/* coefficient of tap o (-3..3) in vecc(c, f) */
DEVI float vecc_coef(int o, int f) {
  if (f == 1)
    return o == -1 ? (float)kC1 : o == 0 ? (float)kC2 : o == 1 ? (float)kC3 : o == 2 ? (float)kC4 : o == 3 ? (float)kC5 : 0.0f;
  return o == 1 ? -(float)kC1 : o == 0 ? -(float)kC2 : o == -1 ? -(float)kC3 : o == -2 ? -(float)kC4
                                                                    : o == -3 ? -(float)kC5 : 0.0f;
}
/* odd image across the free surface on a 7-point column (entries above the
   surface replaced), transposed in place on the tap adjoints v */
DEVI void t_free_image(float *v, int n_free) {
  for (int l = 6; l > n_free; l--) {
    v[2 * n_free - l] -= v[l];
    v[l] = 0.0f;
  }
  v[n_free] = 0.0f;
}
/* the free-surface image t_free (k_fault.hip) transposed onto the column at col */
DEVI void t_dz_free_image(float *col, long ny, int n_free, int kdir, float a) {
  float v[7];
#pragma unroll
  for (int l = 0; l < 7; l++) v[l] = tap_val(vecc_coef(l - 3, kdir), a) * vecc_coef(l - 3, kdir);
  t_free_image(v, n_free);
#pragma unroll
  for (int l = 0; l < 7; l++)
    if (v[l] != 0.0f) aadd(col + (l - 3) * ny, v[l]);
}
/* x += M^T y for M stored SoA (element e at M[e*stride], row-major) */
DEVI void mv3t_add(const float *__restrict__ M, long stride, const float *y, float *x, float sign = 1.0f) {
#pragma unroll
  for (int j = 0; j < 3; j++)
    x[j] += sign * (M[j * stride] * y[0] + M[(3 + j) * stride] * y[1] + M[(6 + j) * stride] * y[2]);
}

DEVI void metric_cols(const float *met, long sc, long p, float M[3][3]) {
  M[0][0] = met[sc + p];     M[0][1] = met[4 * sc + p]; M[0][2] = met[7 * sc + p];
  M[1][0] = met[2 * sc + p]; M[1][1] = met[5 * sc + p]; M[1][2] = met[8 * sc + p];
  M[2][0] = met[3 * sc + p]; M[2][1] = met[6 * sc + p]; M[2][2] = met[9 * sc + p];
}

/* jac and the nine metric entries of a point, metric_cols' order */
DEVI void load_met(const float *met, long sc, long p, float &jac, float M[3][3]) {
  jac = met[p];
  metric_cols(met, sc, p, M);
}

/* fault2wave_node (k_fault.hip, transform.cu:331-372) transposed: from the
   adjoint aw of the nine wavefield values written at the plane, t[c] for T1
   slot 3 (t[c][0]) and the split-node tractions 2 and 3 (half of t[c][1] and
   t[c][2] to each side). M: metric_cols of the point (inverted in place) */
DEVI void f2w_adj(const AdjFaultArgs &a, float jac, float M[3][3], const float *aw, float t[3][3]) {
  const float rj = (float)(1.0 / jac);
  inv3(M);
  float aS[3][3];
  aS[0][0] = aw[TXX];
  aS[1][1] = aw[TYY];
  aS[2][2] = aw[TZZ];
  aS[0][1] = aS[1][0] = 0.5f * aw[TXY];
  const float axz = aw[a.fix_q1 ? TXZ : TYZ], ayz = aw[a.fix_q1 ? TYZ : TXZ];
  aS[0][2] = aS[2][0] = 0.5f * axz;
  aS[1][2] = aS[2][1] = 0.5f * ayz;
#pragma unroll
  for (int c = 0; c < 3; c++)
#pragma unroll
    for (int k = 0; k < 3; k++) t[c][k] = rj * (aS[c][0] * M[k][0] + aS[c][1] * M[k][1] + aS[c][2] * M[k][2]);
}
/* its split-node state adjoints (own node; atomic) */
DEVI void f2w_scatter(const float t[3][3], const float *aw, float *af, long ss, long pf) {
#pragma unroll
  for (int c = 0; c < 3; c++)
#pragma unroll
    for (int m = 0; m < 2; m++) {
      aadd(af + fidx(3 + c, m, ss) + pf, 0.5f * t[c][1]);
      aadd(af + fidx(6 + c, m, ss) + pf, 0.5f * t[c][2]);
      aadd(af + fidx(c, m, ss) + pf, 0.5f * aw[c]);
    }
}

DEVI float *adj_block(const AdjFaultArgs &a, int id) { return a.adjf + (long)id * kAdjFaultFloats * a.g.sslice; }
DEVI float *adj_lev(const AdjFaultArgs &a, float *blk, int l) { return l < 0 ? nullptr : blk + (long)l * 18 * a.g.sslice; }

/* The node kernels: one lane per node, a block of one wavefront (a fault plane
   is 100 to 3000 wavefronts on 256 CUs, so nothing hides a wait), and every
   load ahead of the first store or atomic: the vector memory counter is in
   order, so a load issued after an atomic waits for it as well. Measured at
   48 x 128 nodes (240 x 100): trial 29.6 -> 11.9 us (44 -> 21), nodes 28.8 ->
   25.5 (41 -> 38), w2f 11.9 -> 5.0 (21 -> 9.7), lev 6.7 -> 4.8 (8.8 -> 5.3),
   begin 14.2 -> 6.0 (19 -> 16). */
constexpr int kNodeLanes = 64;

/* ---------------------------------------------------------------------- */
/* Once per reverse step, before its last stage: the split-node P level is
   cleared (it accumulates over the step); the last stage's hT1/mT1 update,
   Slip += |V_s| dt and the fault2wave onto the end level are transposed. */
__global__ void __launch_bounds__(kNodeLanes) k_adjf_begin(AdjFaultArgs a) {
  const int iy = blockIdx.x * kNodeLanes + threadIdx.x, iz = blockIdx.y;
  if (iy >= a.g.nj) return;
  const int id = blockIdx.z;
  const FaultDev &F = a.ftab[id];
  const long ss = a.g.sslice, sc = a.g.sicmp;
  const long pf = (iy + 3) + (long)(iz + 3) * a.g.ny;
  float *blk = adj_block(a, id);
  float *fP = adj_lev(a, blk, a.lp), *fE = adj_lev(a, blk, a.le);
  if (F.united[pf] != 0) {
#pragma unroll
    for (int q = 0; q < 18; q++) fP[q * ss + pf] = 0.0f;
    return;
  }
  float *aT1 = blk + kOffT1 * ss, *aH = blk + kOffHT1 * ss, *aM = blk + kOffMT1 * ss;
  const float dt = a.dt;
  const long p0 = F.i0 + (long)(iy + 3) * a.g.siy + (long)(iz + 3) * a.g.siz;
  const float *tp = a.tape + ((long)id * a.tape_nt + a.n) * kTapeFloats * ss + pf;
  float *vr = blk + kOffVsr * ss + pf;
  /* loads */
  float h[3], m1[3], t3[3], dV[3], s1[3], s2[3], aw[9], jac, M[3][3];
#pragma unroll
  for (int c = 0; c < 3; c++) {
    h[c] = aH[c * ss + pf];
    m1[c] = aM[c * ss + pf];
    t3[c] = aT1[(long)(7 * c + 3) * ss + pf];
    dV[c] = tp[(13 + c) * ss];
    s1[c] = F.vs[c * ss + pf];
    s2[c] = F.vs[(3 + c) * ss + pf];
  }
  const float vr0 = vr[0], vr1 = vr[ss], vr2 = vr[2 * ss];
  const float as0 = blk[kOffSlip * ss + pf], as1 = blk[kOffSlip12 * ss + pf], as2 = blk[(kOffSlip12 + 1) * ss + pf];
#pragma unroll
  for (int f = 0; f < 9; f++) aw[f] = a.wE[f * sc + p0];
  load_met(a.met, sc, p0, jac, M);

  /* Vs1, Vs2 = projections of the velocity jump, Vs = |(Vs1, Vs2)|;
     Slip += Vs dt, Slip1 += Vs1 dt, Slip2 += Vs2 dt; plus the receiver
     residuals of Vs, Vs1, Vs2 of this step */
  const float Vs1 = dV[0] * s1[0] + dV[1] * s1[1] + dV[2] * s1[2];
  const float Vs2 = dV[0] * s2[0] + dV[1] * s2[1] + dV[2] * s2[2];
  const float Vs = sqrtf(Vs2 * Vs2 + Vs1 * Vs1);
  const float aVs = vr0 + as0 * dt;
  float aV1 = vr1 + as1 * dt;
  float aV2 = vr2 + as2 * dt;
  if (Vs > 0.0f) {
    aV1 += aVs * Vs1 / Vs;
    aV2 += aVs * Vs2 / Vs;
  }
  /* fault2wave onto the end level */
  float t[3][3];
  f2w_adj(a, jac, M, aw, t);

#pragma unroll
  for (int q = 0; q < 18; q++) fP[q * ss + pf] = 0.0f;
  vr[0] = vr[ss] = vr[2 * ss] = 0.0f;
#pragma unroll
  for (int c = 0; c < 3; c++) {
    const float hd = h[c] / dt;
    aT1[(long)(7 * c + 3) * ss + pf] = t3[c] + (hd + m1[c]) + t[c][0];
    aM[c * ss + pf] = -hd;
    aH[c * ss + pf] = 0.0f;
  }
#pragma unroll
  for (int f = 0; f < 9; f++) a.wE[f * sc + p0] = 0.0f;
#pragma unroll
  for (int c = 0; c < 3; c++) {
    const float g = aV1 * s1[c] + aV2 * s2[c];
    aadd(fE + fidx(c, 1, ss) + pf, g);
    aadd(fE + fidx(c, 0, ss) + pf, -g);
  }
  f2w_scatter(t, aw, fE, ss, pf);
}

/* fault-receiver residuals of one sample (the outputs after the step being
   reversed): Slip, Slip1, Slip2 into their running adjoints, Vs, Vs1, Vs2
   into this step's; welded nodes output nothing */
__global__ void k_adjf_receivers(AdjFaultArgs a, const int *rec, const float *fac, int nterm, int nrec,
                                 const float *res, int nt, int sample) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= nrec * nterm) return;
  const int r = t / nterm;
  const int id = rec[2 * t];
  const long pf = rec[2 * t + 1], ss = a.g.sslice;
  const float w = fac[2 * t] * fac[2 * t + 1];
  if (w == 0.0f || a.ftab[id].united[pf] != 0) return;
  float *blk = adj_block(a, id);
  const float *q = res + ((long)r * nt + sample) * 9;
  aadd(blk + kOffVsr * ss + pf, q[3] * w);
  aadd(blk + (kOffVsr + 1) * ss + pf, q[4] * w);
  aadd(blk + (kOffVsr + 2) * ss + pf, q[5] * w);
  aadd(blk + kOffSlip * ss + pf, q[6] * w);
  aadd(blk + kOffSlip12 * ss + pf, q[7] * w);
  aadd(blk + (kOffSlip12 + 1) * ss + pf, q[8] * w);
}

/* RK structure of the split-node levels at reverse stage MODE (the
   wavefield's, k_adjoint.hip): the stage input's adjoint level starts from
   zero (stage 0: P accumulates) */
template <int MODE>
__global__ void __launch_bounds__(kNodeLanes) k_adjf_lev(AdjFaultArgs a) {
  const int iy = blockIdx.x * kNodeLanes + threadIdx.x, iz = blockIdx.y;
  if (iy >= a.g.nj) return;
  const long ss = a.g.sslice;
  const long pf = (iy + 3) + (long)(iz + 3) * a.g.ny;
  float *blk = adj_block(a, blockIdx.z);
  const float *E = adj_lev(a, blk, a.le);
  float *A = adj_lev(a, blk, 1), *B = adj_lev(a, blk, 2), *P = adj_lev(a, blk, a.lp);
  float pv[18];
  if (MODE != 3) {
#pragma unroll
    for (int q = 0; q < 18; q++) {
      const long o = q * ss + pf;
      pv[q] = P[o] + (MODE == 2 ? E[o] + A[o] : (MODE == 1 ? B[o] : A[o]));
    }
  }
#pragma unroll
  for (int q = 0; q < 18; q++) {
    const long o = q * ss + pf;
    if (MODE != 3) P[o] = pv[q];
    if (MODE == 3 || MODE == 1) A[o] = 0.0f;
    if (MODE == 2) B[o] = 0.0f;
  }
}

/* ---------------------------------------------------------------------- */
/* fault_cols (k_fault.hip) transposed, as a gather. A block owns the targets
   of kColNodes x kColRows nodes (ghost rows and planes included): the twelve
   wavefield columns the forward stencils of these rows read, and the plane.
   Phase 1 forms, for the six column points of every node whose taps reach the
   tile (the tile and three nodes to each side: a cross), the adjoints of the
   traction sums and of the velocity differences; phase 2 sums each target's
   taps from LDS and adds them to what the stage wrote, one lane to a target.
   A scatter with atomic adds (500 to a node, and device-scope atomics leave
   the XCD's L2) took 121 us at 240 x 100 nodes and 36.7 at 128 x 48; this
   takes 56 and 20, with three times the loads for the cross. */
constexpr int kColNodes = 10, kColRows = 4, kColLanes = 384;
constexpr int kColY = (kColNodes + 6) * kColRows;            /* the tile's rows with their y halo */
constexpr int kColSrc = kColY + kColNodes * 6;               /* and the z halo */
DEVI void col_src(int m, int &jn, int &kr) {
  if (m < kColY) {
    jn = m % (kColNodes + 6) - 3;
    kr = m / (kColNodes + 6);
  } else {
    jn = (m - kColY) % kColNodes;
    kr = (m - kColY) / kColNodes;
    kr = kr < 3 ? kr - 3 : kr - 3 + kColRows;
  }
}
DEVI int col_src_z(int jn, int kr) {  /* source of tile row kr in [-3, kColRows + 3) at the tile's jn */
  return kr >= 0 && kr < kColRows ? jn + 3 + (kColNodes + 6) * kr
                                  : kColY + jn + kColNodes * (kr < 0 ? kr + 3 : kr + 3 - kColRows);
}

template <int IDIR>
__global__ void __launch_bounds__(kColLanes) k_adjf_cols(AdjFaultArgs a) {
  __shared__ float sg[12][6 * kColSrc]; /* traction sums, D_x V, D_y V, D_z V (three components each) */
  /* x stencils over the columns i0 - 6 .. i0 + 6 (6: the plane): cxv weights
     D_x V; cxt[.][.][l] how often the product of tap l counts, images beyond
     the plane included (a sum of products, not a product with a sum: far from
     the receivers the traction sums are denormal, where products round
     coarsely and sums are exact) */
  __shared__ float cxt[6][13][7], cxv[6][13];
  const int id = blockIdx.z;
  const FaultDev &F = a.ftab[id];
  const long ss = a.g.sslice, sc = a.g.sicmp, sy = a.g.siy, sz = a.g.siz;
  const int i0 = F.i0;
  const int j0 = (int)blockIdx.x * kColNodes - 3, k0 = (int)blockIdx.y * kColRows - 3;
  const int tid = threadIdx.x;
  const bool surf = a.isfree == 1;
  const float *met = a.met;
  constexpr int kIt = (6 * kColSrc + kColLanes - 1) / kColLanes;
  bool mine[kIt], any = false;
#pragma unroll
  for (int it = 0; it < kIt; it++) {
    const int v = tid + it * kColLanes;
    int jn, kr;
    col_src(v / 6, jn, kr);
    const int iy = j0 + jn, iz = k0 + kr;
    mine[it] = v < 6 * kColSrc && iy >= 0 && iy < a.g.nj && iz >= 0 && iz < a.g.nk &&
               F.united[(iy + 3) + (long)(iz + 3) * a.g.ny] == 0;
    any |= mine[it];
  }
  if (!__syncthreads_or(any)) return;  /* no split node reaches the tile */

  if (tid < 6) {
    const int mm = tid < 3 ? tid - 3 : tid - 2, n = -mm;
    float *cv = cxv[tid];
#pragma unroll
    for (int x = 0; x < 13; x++) cv[x] = 0.0f;
    for (int x = 0; x < 13; x++)
#pragma unroll
      for (int l = 0; l < 7; l++) cxt[tid][x][l] = 0.0f;
    float(*au)[7] = cxt[tid] + (mm + 3);  /* au[t]: what tap t of this column holds */
#pragma unroll
    for (int l = 0; l < 7; l++) au[l][l] = 1.0f;
    /* images beyond the plane: from tap f, twice to tap g and minus once to tap h */
    auto image = [&](int f, int g, int h) {
#pragma unroll
      for (int l = 0; l < 7; l++) {
        au[g][l] += 2.0f * au[f][l];
        au[h][l] -= au[f][l];
        au[f][l] = 0.0f;
      }
    };
    if (n == 2) image(6, 5, 4);
    if (n == 1) { image(6, 4, 2); image(5, 4, 3); }
    if (n == -1) { image(1, 2, 3); image(0, 2, 4); }
    if (n == -2) image(0, 1, 2);
    /* reduced differences towards the plane, whose split side is the tap at 6 */
    const float b1 = (float)kB1, b2 = (float)kB2, b3 = (float)kB3;
    const float c1 = (float)kC1, c2 = (float)kC2, c3 = (float)kC3, c4 = (float)kC4, c5 = (float)kC5;
    float *q = cv + 6;
    if (IDIR == 1) {
      if (mm == -1) { q[0] = 1.0f; q[-1] = -1.0f; }
      else if (mm == -2) { q[-2] = b1; q[-1] = b2; q[0] = b3; }
      else if (mm == 1) { q[2] = 1.0f; q[1] = -1.0f; }
      else if (mm == 2) { q[2] = b1; q[3] = b2; q[4] = b3; }
      else { q[mm - 1] = c1; q[mm] = c2; q[mm + 1] = c3; q[mm + 2] = c4; q[mm + 3] = c5; }
    } else {
      if (mm == 1) { q[1] = 1.0f; q[0] = -1.0f; }
      else if (mm == 2) { q[0] = -b3; q[1] = -b2; q[2] = -b1; }
      else if (mm == -1) { q[-1] = 1.0f; q[-2] = -1.0f; }
      else if (mm == -2) { q[-2] = -b1; q[-3] = -b2; q[-4] = -b3; }
      else { q[mm + 1] = -c1; q[mm] = -c2; q[mm - 1] = -c3; q[mm - 2] = -c4; q[mm - 3] = -c5; }
    }
  }

  /* phase 1 */
#pragma unroll
  for (int it = 0; it < kIt; it++) {
    const int v = tid + it * kColLanes;
    if (v >= 6 * kColSrc) continue;
    float o[12];
#pragma unroll
    for (int e = 0; e < 12; e++) o[e] = 0.0f;
    if (mine[it]) {
      int jn, kr;
      col_src(v / 6, jn, kr);
      const int cl = v % 6, iy = j0 + jn, iz = k0 + kr;
      const int i = i0 + (cl < 3 ? cl - 3 : cl - 2);
      const long p = i + (long)(iy + 3) * sy + (long)(iz + 3) * sz;
      float hh[9], mt[9];
#pragma unroll
      for (int f = 0; f < 9; f++) hh[f] = a.cb * a.wE[f * sc + p] + (a.wX ? a.ca * a.wX[f * sc + p] : 0.0f);
#pragma unroll
      for (int f = 0; f < 9; f++) mt[f] = met[(1 + f) * sc + p];
      const float l = a.lam[p], m = a.mu[p], l2m = (float)(l + 2.0 * m);
      /* velocity rhs: (dvx + dvy + dvz) slw / J over the traction vectors at
         the taps */
      const float rrhojac = a.slw[p] / met[p];
#pragma unroll
      for (int c = 0; c < 3; c++) o[c] = hh[c] * rrhojac;
      /* stress rhs: Hooke's law on the velocity differences */
      float aG[3][3];
      aG[0][0] = l2m * hh[TXX] + l * hh[TYY] + l * hh[TZZ];
      aG[1][1] = l * hh[TXX] + l2m * hh[TYY] + l * hh[TZZ];
      aG[2][2] = l * hh[TXX] + l * hh[TYY] + l2m * hh[TZZ];
      aG[0][1] = aG[1][0] = m * hh[TXY];
      aG[0][2] = aG[2][0] = m * hh[TXZ];
      aG[1][2] = aG[2][1] = m * hh[TYZ];
#pragma unroll
      for (int d = 0; d < 3; d++)
#pragma unroll
        for (int c = 0; c < 3; c++)
          o[3 + 3 * d + c] = mt[3 * d] * aG[c][0] + mt[3 * d + 1] * aG[c][1] + mt[3 * d + 2] * aG[c][2];
      if (surf && iz == a.g.nk - 1) {
        const long ij = ((long)i + (long)(iy + 3) * sy) * 9;
        const float *X = a.matVx2Vz + ij, *Y = a.matVy2Vz + ij;
#pragma unroll
        for (int c = 0; c < 3; c++) {
          o[3 + c] += X[c] * o[9] + X[3 + c] * o[10] + X[6 + c] * o[11];
          o[6 + c] += Y[c] * o[9] + Y[3 + c] * o[10] + Y[6 + c] * o[11];
        }
        o[9] = o[10] = o[11] = 0.0f;
      }
    }
#pragma unroll
    for (int e = 0; e < 12; e++) sg[e][v] = o[e];
  }
  __syncthreads();

  /* phase 2 */
  float *T = a.wT;
  float *blk = adj_block(a, id);
  float *aT1 = blk + kOffT1 * ss, *aV = adj_lev(a, blk, a.lc) + fidx(0, IDIR == 1 ? 0 : 1, ss);
  const bool alone = a.nfault == 1;  /* another fault's columns may be the same points */
#pragma unroll 1
  for (int u = tid; u < 13 * kColNodes * kColRows; u += kColLanes) {
    const int xi = u % 13, nd = u / 13, jn = nd % kColNodes, kr = nd / kColNodes;
    const int x = i0 - 6 + xi, jg = j0 + jn + 3, kg = k0 + kr + 3;
    if (x < 0 || x >= a.g.nx || jg < 0 || jg >= a.g.ny || kg < 0 || kg >= a.g.nz) continue;
    float vel[3] = {0.0f, 0.0f, 0.0f}, tx[3] = {0.0f, 0.0f, 0.0f};
    const int m0 = 6 * (jn + 3 + (kColNodes + 6) * kr);
#pragma unroll
    for (int cl = 0; cl < 6; cl++) {
      const float wv = cxv[cl][xi];
#pragma unroll
      for (int c = 0; c < 3; c++) {
        const float g = sg[c][m0 + cl];
#pragma unroll
        for (int l = 0; l < 7; l++)
          if (vecc_coef(l - 3, IDIR) != 0.0f) {
            const float w = cxt[cl][xi][l];
            tx[c] += w * tap_val(w, __fmul_rn(g, vecc_coef(l - 3, IDIR)));
          }
        vel[c] += tap_mul(wv, sg[3 + c][m0 + cl]);
      }
    }
    if (xi == 6) {  /* the plane: the fault traction and the split side's velocity */
      const bool node = jg >= 3 && jg < a.g.nj + 3 && kg >= 3 && kg < a.g.nk + 3;
      const long pf = jg + (long)kg * a.g.ny;
      if (node && F.united[pf] == 0) {
        float t3[3], v3[3];
#pragma unroll
        for (int c = 0; c < 3; c++) {
          t3[c] = aT1[(long)(7 * c + 3) * ss + pf];
          v3[c] = aV[2 * c * ss + pf];
        }
#pragma unroll
        for (int c = 0; c < 3; c++) {
          aT1[(long)(7 * c + 3) * ss + pf] = t3[c] + tx[c];
          aV[2 * c * ss + pf] = v3[c] + vel[c];
        }
      }
      continue;
    }
    const long q = x + (long)jg * sy + (long)kg * sz;
    const bool near = xi >= 3 && xi <= 9;
    float w[9], M[10];
#pragma unroll
    for (int f = 0; f < 9; f++) w[f] = alone ? T[f * sc + q] : 0.0f;
#pragma unroll
    for (int e = 0; e < 10; e++) M[e] = e < 4 || near ? met[e * sc + q] : 0.0f;
    float ty[3] = {0.0f, 0.0f, 0.0f}, tz[3] = {0.0f, 0.0f, 0.0f};
    if (near) {
      const int cl = xi < 6 ? xi - 3 : xi - 4;
#pragma unroll
      for (int o = -3; o <= 3; o++) {
        /* the source whose tap o this is */
        const float wy = vecc_coef(o, a.jdir);
        const int my = 6 * (jn - o + 3 + (kColNodes + 6) * kr) + cl;
        const int mz = 6 * col_src_z(jn, kr - o) + cl;
        const int km = a.g.nk - (kg - 3 - o + 1);
        float wt = vecc_coef(o, a.kdir), wi = 0.0f, wv = wt;
        if (surf && km <= 3) {
          /* odd traction image about plane km above the source (t_free_image) */
          const int im = 2 * km - o;
          if (o >= km) wt = 0.0f;
          else
#pragma unroll
            for (int t = -3; t <= 3; t++)
              if (im == t) wi = vecc_coef(t, a.kdir);
          /* mac22, mac24 */
          if (km == 1) wv = a.kdir == 1 ? (o == 1 ? 1.0f : o == 0 ? -1.0f : 0.0f) : (o == 0 ? 1.0f : o == -1 ? -1.0f : 0.0f);
          if (km == 2) {
            const int so = a.kdir == 1 ? o : -o;
            const float b = so == 0 ? (float)kB1 : so == 1 ? (float)kB2 : so == 2 ? (float)kB3 : 0.0f;
            wv = a.kdir == 1 ? b : -b;
          }
        }
#pragma unroll
        for (int c = 0; c < 3; c++) {
          const float gy = sg[c][my], gz = sg[c][mz];
          ty[c] = __fadd_rn(ty[c], __fmul_rn(wy, tap_val(wy, gy)));
          tz[c] = __fadd_rn(tz[c], __fsub_rn(__fmul_rn(wt, tap_val(wt, gz)), __fmul_rn(wi, tap_val(wi, gz))));
          vel[c] += tap_mul(wy, sg[6 + c][my]) + tap_mul(wv, sg[9 + c][mz]);
        }
      }
    }
    /* stress adjoints of the traction vectors: tv_c = J (a1 s_c0 + a2 s_c1 + a3 s_c2);
       J first: the sums carry 1 / J and far from the receivers are denormal */
    float t[3][3];
#pragma unroll
    for (int c = 0; c < 3; c++) {
      tx[c] *= M[0];
      ty[c] *= M[0];
      tz[c] *= M[0];
#pragma unroll
      for (int e = 0; e < 3; e++) t[c][e] = M[1 + e] * tx[c] + M[4 + e] * ty[c] + M[7 + e] * tz[c];
    }
    const float add[9] = {vel[0], vel[1], vel[2], t[0][0], t[1][1], t[2][2],
                          t[1][2] + t[2][1], t[0][2] + t[2][0], t[0][1] + t[1][0]};  /* by field: V, TXX .. TXY */
    if (alone) {
#pragma unroll
      for (int f = 0; f < 9; f++) T[f * sc + q] = w[f] + add[f];
    } else {
#pragma unroll
      for (int f = 0; f < 9; f++)
        if (add[f] != 0.0f) aadd(T + f * sc + q, add[f]);
    }
  }
}

/* ---------------------------------------------------------------------- */
/* fault_nodes (k_fault.hip) transposed: one lane per node */
template <int IDIR>
__global__ void __launch_bounds__(kNodeLanes) k_adjf_nodes(AdjFaultArgs a) {
  const int iy = blockIdx.x * kNodeLanes + threadIdx.x, iz = blockIdx.y;
  if (iy >= a.g.nj) return;
  const int id = blockIdx.z;
  const FaultDev &F = a.ftab[id];
  const long ss = a.g.sslice, sc = a.g.sicmp, ny = a.g.ny, sy = a.g.siy, sz = a.g.siz;
  const long pf = (iy + 3) + (long)(iz + 3) * ny;
  if (F.united[pf] != 0) return;
  const int jdir = a.jdir, kdir = a.kdir, i0 = F.i0;
  const long row = (long)(iy + 3) * sy + (long)(iz + 3) * sz;
  const long p0 = i0 + row;
  const int km = a.g.nk - (iz + 1), n_free = km + 3;
  const bool surf = a.isfree == 1;
  const int ry = F.rupy[pf], rz = F.rupz[pf];
  float *blk = adj_block(a, id);
  float *aT1 = blk + kOffT1 * ss, *aC = adj_lev(a, blk, a.lc);
  const float *aE = adj_lev(a, blk, a.le), *aX = adj_lev(a, blk, a.lx);
  float r[2][9];
#pragma unroll
  for (int mside = 0; mside < 2; mside++)
#pragma unroll
    for (int c = 0; c < 9; c++) {
      const long o = fidx(c, mside, ss) + pf;
      r[mside][c] = a.cb * aE[o] + (aX ? a.ca * aX[o] : 0.0f);
    }
  const float *met = a.met;
  float *aH = blk + kOffHT1 * ss;
  const float jac = met[p0], rho[2] = {F.rho_f[pf], F.rho_f[ss + pf]};
  const bool fgrid = F.faultgrid[pf] == 1;
  float T1[3][7], h1[3];
#pragma unroll
  for (int c = 0; c < 3; c++) {
    h1[c] = aH[c * ss + pf];
#pragma unroll
    for (int t = 0; t < 7; t++) T1[c][t] = aT1[(long)(7 * c + t) * ss + pf];
  }
  const long ms = ss, mq = 9 * ss;
  /* traction rates fhT2/fhT3 = D (DxV, DyV, DzV) */
  float aDx[2][3] = {}, aDy[2][3] = {}, aDz[2][3] = {};
#pragma unroll
  for (int mside = 0; mside < 2; mside++) {
    const float *Db = F.D + (long)(mside * 6) * mq + pf;
    mv3t_add(Db + 0 * mq, ms, r[mside] + 3, aDx[mside]);
    mv3t_add(Db + 1 * mq, ms, r[mside] + 3, aDy[mside]);
    mv3t_add(Db + 2 * mq, ms, r[mside] + 3, aDz[mside]);
    mv3t_add(Db + 3 * mq, ms, r[mside] + 6, aDx[mside]);
    mv3t_add(Db + 4 * mq, ms, r[mside] + 6, aDy[mside]);
    mv3t_add(Db + 5 * mq, ms, r[mside] + 6, aDz[mside]);
  }
  constexpr int S_ = IDIR == 1 ? 1 : 0, O_ = 1 - S_;
  const float *Ms = (IDIR == 1 ? F.P2M : F.M2P) + pf;
  const float *M2 = F.M2 + pf;
  float aDt[3] = {0.0f, 0.0f, 0.0f};
  auto method1_t = [&]() {
    mv3t_add(Ms + 0 * mq, ms, aDx[O_], aDx[S_]);
    mv3t_add(Ms + 1 * mq, ms, aDx[O_], aDy[S_]);
    mv3t_add(Ms + 2 * mq, ms, aDx[O_], aDz[S_]);
    mv3t_add(Ms + 3 * mq, ms, aDx[O_], aDy[O_], -1.0f);
    mv3t_add(Ms + 4 * mq, ms, aDx[O_], aDz[O_], -1.0f);
#pragma unroll
    for (int c = 0; c < 3; c++) aDx[O_][c] = 0.0f;
  };
  auto method2_t = [&]() {
    mv3t_add(M2 + 3 * mq, ms, aDx[1], aDt);
    mv3t_add(M2 + 4 * mq, ms, aDx[1], aDy[1], -1.0f);
    mv3t_add(M2 + 5 * mq, ms, aDx[1], aDz[1], -1.0f);
    mv3t_add(M2 + 0 * mq, ms, aDx[0], aDt);
    mv3t_add(M2 + 1 * mq, ms, aDx[0], aDy[0], -1.0f);
    mv3t_add(M2 + 2 * mq, ms, aDx[0], aDz[0], -1.0f);
#pragma unroll
    for (int c = 0; c < 3; c++) aDx[0][c] = aDx[1][c] = 0.0f;
  };
  /* the one-sided x difference of method 1 (own split node and the first
     wavefield column on side S) */
  auto diff_t = [&]() {
#pragma unroll
    for (int c = 0; c < 3; c++) {
      const float g = aDx[S_][c];
      if (IDIR == 1) { aadd(a.wT + c * sc + (i0 + 1) + row, g); aadd(aC + fidx(c, 1, ss) + pf, -g); }
      else { aadd(aC + fidx(c, 0, ss) + pf, g); aadd(a.wT + c * sc + (i0 - 1) + row, -g); }
      aDx[S_][c] = 0.0f;
    }
  };
  const float *fV[3] = {aC + fidx(0, 0, ss), aC + fidx(1, 0, ss), aC + fidx(2, 0, ss)};
  if (surf && km == 0) {
    const float *Fm = F.Fm + (iy + 3);
    const long fs_ = ny, fq = 9 * ny;
    mv3t_add(Fm + 2 * fq, fs_, aDz[1], aDx[1]);
    mv3t_add(Fm + 3 * fq, fs_, aDz[1], aDy[1]);
    mv3t_add(Fm + 0 * fq, fs_, aDz[0], aDx[0]);
    mv3t_add(Fm + 1 * fq, fs_, aDz[0], aDy[0]);
#pragma unroll
    for (int c = 0; c < 3; c++) aDz[0][c] = aDz[1][c] = 0.0f;
    if (a.imethod == 1) {
      const float *Mf = Fm + (IDIR == 1 ? 4 : 7) * fq;
      mv3t_add(Mf, fs_, aDx[O_], aDx[S_]);
      mv3t_add(Mf + fq, fs_, aDx[O_], aDy[S_]);
      mv3t_add(Mf + 2 * fq, fs_, aDx[O_], aDy[O_], -1.0f);
#pragma unroll
      for (int c = 0; c < 3; c++) aDx[O_][c] = 0.0f;
      diff_t();
    } else {
      mv3t_add(Fm + 12 * fq, fs_, aDx[1], aDt);
      mv3t_add(Fm + 13 * fq, fs_, aDx[1], aDy[1], -1.0f);
      mv3t_add(Fm + 10 * fq, fs_, aDx[0], aDt);
      mv3t_add(Fm + 11 * fq, fs_, aDx[0], aDy[0], -1.0f);
    }
  } else {
    if (a.imethod == 1) { method1_t(); diff_t(); }
    else method2_t();
#pragma unroll
    for (int c = 0; c < 3; c++)
#pragma unroll
      for (int mside = 0; mside < 2; mside++) {
        float *q = (float *)fV[c] + (mside ? ss : 0) + pf;
        const float g = aDz[mside][c];
        if (surf && km == 1) t_mac22(q, ny, kdir, g);
        else if (surf && km == 2) t_mac24(q, ny, kdir, g);
        else if (rz == 1) t_mac22(q, ny, kdir, g);
        else t_macdrp(q, ny, kdir, g);
      }
  }
#pragma unroll
  for (int c = 0; c < 3; c++)
#pragma unroll
    for (int mside = 0; mside < 2; mside++) {
      float *q = (float *)fV[c] + (mside ? ss : 0) + pf;
      if (ry == 1) t_mac22(q, 1, jdir, aDy[mside][c]);
      else t_macdrp(q, 1, jdir, aDy[mside][c]);
    }
  if (fgrid)
#pragma unroll
    for (int c = 0; c < 3; c++) aH[c * ss + pf] = h1[c] + aDt[c];
  /* split-node velocity rates from T1 and the traction differences */
#pragma unroll
  for (int mside = 0; mside < 2; mside++) {
    const float rrhojac = (float)(1.0 / (rho[mside] * jac));
#pragma unroll
    for (int c = 0; c < 3; c++) {
      const float g = r[mside][c] * rrhojac;
      float *t = T1[c];
      if (mside == 0) {
        t[3] += (float)kA0 * g; t[2] -= (float)kA1 * g; t[1] -= (float)kA2 * g; t[0] -= (float)kA3 * g;
      } else {
        t[3] -= (float)kA0 * g; t[4] += (float)kA1 * g; t[5] += (float)kA2 * g; t[6] += (float)kA3 * g;
      }
      float *p2 = aC + fidx(3 + c, mside, ss) + pf, *p3 = aC + fidx(6 + c, mside, ss) + pf;
      if (ry == 1) t_mac22(p2, 1, jdir, g);
      else if (ry == 0) t_macdrp(p2, 1, jdir, g);
      if (surf && km <= 3) t_dz_free_image(p3, ny, n_free, kdir, g);
      else if (rz == 1) t_mac22(p3, ny, kdir, g);
      else if (rz == 0) t_macdrp(p3, ny, kdir, g);
    }
  }
#pragma unroll
  for (int c = 0; c < 3; c++)
#pragma unroll
    for (int t = 0; t < 7; t++) aT1[(long)(7 * c + t) * ss + pf] = T1[c][t];
}

/* ---------------------------------------------------------------------- */
/* trial (k_fault.hip, trial_slipweakening.cu:91-388) and trial_t1
   transposed, with the parameter gradients; one lane per split node */
__global__ void __launch_bounds__(kNodeLanes) k_adjf_trial(AdjFaultArgs a) {
  const int iy = blockIdx.x * kNodeLanes + threadIdx.x, iz = blockIdx.y;
  if (iy >= a.g.nj) return;
  const int id = blockIdx.z;
  const FaultDev &F = a.ftab[id];
  const long ss = a.g.sslice, sc = a.g.sicmp, ny = a.g.ny;
  const long pf = (iy + 3) + (long)(iz + 3) * ny;
  if (F.united[pf] != 0) return;
  const int jdir = a.jdir, kdir = a.kdir;
  const float *met = a.met;
  const long row = (long)(iy + 3) * a.g.siy + (long)(iz + 3) * a.g.siz;
  const long p0 = F.i0 + row;
  const int km = a.g.nk - (iz + 1), n_free = km + 3;
  const int ry = F.rupy[pf], rz = F.rupz[pf];
  float *blk = adj_block(a, id);
  float *aT1 = blk + kOffT1 * ss, *aC = adj_lev(a, blk, a.lc), *aP = adj_lev(a, blk, a.lp);
  float *gr = blk + kOffGrad * ss;
  float *W = a.wT;

  /* loads: the plane and its metric, T1, the tape and parameters, and the
     three stress columns on either side with their metric rows */
  float aw[9], jac0, M[3][3], T1[3][7], w6[6][6], m4[6][4], g7[7];
#pragma unroll
  for (int f = 0; f < 9; f++) aw[f] = W[f * sc + p0];
  load_met(met, sc, p0, jac0, M);
#pragma unroll
  for (int c = 0; c < 3; c++)
#pragma unroll
    for (int t = 0; t < 7; t++) T1[c][t] = aT1[(long)(7 * c + t) * ss + pf];
  const float *tp = a.tape + ((long)id * a.tape_nt + a.n) * kTapeFloats * ss + pf;
  const float Trial[3] = {tp[(3 * a.istage) * ss], tp[(3 * a.istage + 1) * ss], tp[(3 * a.istage + 2) * ss]};
  const float Slip = tp[12 * ss];
  const float T0[3] = {F.T0[pf], F.T0[ss + pf], F.T0[2 * ss + pf]};
  const float mus = F.fric[pf], mud = F.fric[ss + pf], Dc = F.fric[2 * ss + pf], C0 = F.fric[3 * ss + pf];
  const float rho0 = F.rho_f[pf], rho1 = F.rho_f[ss + pf];
#pragma unroll
  for (int q = 0; q < 7; q++) g7[q] = gr[q * ss + pf];
  const float aSlip = blk[kOffSlip * ss + pf];
#pragma unroll
  for (int l = 0; l < 6; l++) {
    const long q = p0 + (l < 3 ? l - 3 : l - 2);
#pragma unroll
    for (int f = 0; f < 6; f++) w6[l][f] = W[(TXX + f) * sc + q];
#pragma unroll
    for (int f = 0; f < 4; f++) m4[l][f] = met[f * sc + q];
  }

  float vn[3] = {M[0][0], M[1][0], M[2][0]};
  /* fault2wave onto the stage input at the plane */
  float tw[3][3];
  f2w_adj(a, jac0, M, aw, tw);

  /* friction on the taped branch */
  float at[3];
#pragma unroll
  for (int c = 0; c < 3; c++) at[c] = T1[c][3] + tw[c][0];
  const float vn0 = norm3(vn);
  const float jacvec = jac0 * vn0;
#pragma unroll
  for (int c = 0; c < 3; c++) vn[c] /= vn0;
  float TL[3], Ts[3];
#pragma unroll
  for (int c = 0; c < 3; c++) TL[c] = Trial[c] / jacvec + T0[c];
  const float Tn0 = dot3(TL, vn);
#pragma unroll
  for (int c = 0; c < 3; c++) Ts[c] = TL[c] - vn[c] * Tn0;
  const float Ts0 = norm3(Ts);
  const bool open = Tn0 >= 0.0f;
  const float Tau_n = open ? 0.0f : Tn0;
  const bool weak = Slip <= Dc;
  const float fr = weak ? mus - (mus - mud) * Slip / Dc : mud;
  const float Tau_c = -fr * Tau_n + C0;
  const bool capped = Ts0 >= Tau_c;
  const bool ifchange = open || capped;
  float aTrial[3];
  if (!ifchange) {
#pragma unroll
    for (int c = 0; c < 3; c++) aTrial[c] = at[c];
  } else {
    /* T1_3 = (Tau - T0) jacvec, Tau = Tau_n vn + (Tau_s / Ts0) Ts */
    float aTau[3], aTL[3] = {0.0f, 0.0f, 0.0f}, aT0[3];
#pragma unroll
    for (int c = 0; c < 3; c++) {
      aTau[c] = at[c] * jacvec;
      aT0[c] = -aTau[c];
    }
    float aTau_n = dot3(aTau, vn), aTs0 = 0.0f, aTau_s = 0.0f;
    float aTs[3] = {0.0f, 0.0f, 0.0f};
    const float Tau_s = capped ? Tau_c : Ts0;
    if (!(fabsf(Ts0) < 1e-1f)) {
      const float kap = Tau_s / Ts0;
      const float akap = dot3(aTau, Ts);
#pragma unroll
      for (int c = 0; c < 3; c++) aTs[c] = kap * aTau[c];
      aTau_s = akap / Ts0;
      aTs0 = -akap * Tau_s / (Ts0 * Ts0);
    }
    float aTau_c = 0.0f;
    if (capped) aTau_c = aTau_s;
    else aTs0 += aTau_s;
    /* Tau_c = -fr Tau_n + C0 */
    const float afr = -aTau_c * Tau_n;
    aTau_n += -fr * aTau_c;
    gr[3 * ss + pf] = g7[3] + aTau_c;
    if (weak) {
      gr[pf] = g7[0] + afr * (1.0f - Slip / Dc);
      gr[ss + pf] = g7[1] + afr * (Slip / Dc);
      gr[2 * ss + pf] = g7[2] + afr * (mus - mud) * Slip / (Dc * Dc);
      blk[kOffSlip * ss + pf] = aSlip - afr * (mus - mud) / Dc;
    } else {
      gr[ss + pf] = g7[1] + afr;
    }
    float aTn0 = open ? 0.0f : aTau_n;
    if (Ts0 > 0.0f)
#pragma unroll
      for (int c = 0; c < 3; c++) aTs[c] += aTs0 * Ts[c] / Ts0;
#pragma unroll
    for (int c = 0; c < 3; c++) aTL[c] += aTs[c];
    aTn0 -= dot3(aTs, vn);
#pragma unroll
    for (int c = 0; c < 3; c++) aTL[c] += aTn0 * vn[c];
#pragma unroll
    for (int c = 0; c < 3; c++) {
      aTrial[c] = aTL[c] / jacvec;
      gr[(4 + c) * ss + pf] = g7[4 + c] + (aTL[c] + aT0[c]);
    }
  }

  /* Trial = 2 (M0 M1 dV / dt + M0 R1 - M1 R0) / (a0 (M0 + M1)) */
  const float M0 = (float)(0.5 * jac0 * rho0), M1 = (float)(0.5 * jac0 * rho1);
  const float den = (float)(2.0 / (kA0 * (M0 + M1)));
  float ad[2][3], adv[3];
#pragma unroll
  for (int c = 0; c < 3; c++) {
    const float g = aTrial[c] * den;
    adv[c] = g * M0 * M1 / a.dt;
#pragma unroll
    for (int mside = 0; mside < 2; mside++) {
      const int sd = 2 * mside - 1;
      const float aR = mside ? g * M0 : -g * M1;
      const float ar = 0.5f * (float)sd * aR;
      ad[mside][c] = 0.5f * aR;
      T1[c][3 + sd] += (float)kA1 * ar;
      T1[c][3 + 2 * sd] += (float)kA2 * ar;
      T1[c][3 + 3 * sd] += (float)kA3 * ar;
    }
  }

  /* traction columns T1 slots 0-2 / 4-6 from the stress (trial_t1) */
#pragma unroll
  for (int l = 0; l < 6; l++) {
    const int slot = l < 3 ? l : l + 1;
    const long q = p0 + (slot - 3);
    const float jl = m4[l][0], x1 = m4[l][1], x2 = m4[l][2], x3 = m4[l][3];
    const float a0 = jl * T1[0][slot], a1 = jl * T1[1][slot], a2 = jl * T1[2][slot];
    const float *w = w6[l];
    W[TXX * sc + q] = w[TXX - TXX] + x1 * a0;
    W[TXY * sc + q] = w[TXY - TXX] + (x2 * a0 + x1 * a1);
    W[TXZ * sc + q] = w[TXZ - TXX] + (x3 * a0 + x1 * a2);
    W[TYY * sc + q] = w[TYY - TXX] + x2 * a1;
    W[TYZ * sc + q] = w[TYZ - TXX] + (x3 * a1 + x2 * a2);
    W[TZZ * sc + q] = w[TZZ - TXX] + x3 * a2;
  }
#pragma unroll
  for (int f = 0; f < 9; f++) W[f * sc + p0] = 0.0f;
#pragma unroll
  for (int c = 0; c < 3; c++)
#pragma unroll
    for (int t = 0; t < 7; t++) aT1[(long)(7 * c + t) * ss + pf] = 0.0f;

  f2w_scatter(tw, aw, aC, ss, pf);
#pragma unroll
  for (int c = 0; c < 3; c++) {
    aadd(aP + fidx(c, 1, ss) + pf, adv[c]);
    aadd(aP + fidx(c, 0, ss) + pf, -adv[c]);
#pragma unroll
    for (int mside = 0; mside < 2; mside++) {
      float *p2 = aC + fidx(3 + c, mside, ss) + pf, *p3 = aC + fidx(6 + c, mside, ss) + pf;
      const float g = ad[mside][c];
      if (ry == 1) t_mac22(p2, 1, jdir, g);
      else if (ry == 0) t_macdrp(p2, 1, jdir, g);
      if (a.isfree == 1 && km <= 3) t_dz_free_image(p3, ny, n_free, kdir, g);
      else if (rz == 1) t_mac22(p3, ny, kdir, g);
      else if (rz == 0) t_macdrp(p3, ny, kdir, g);
    }
  }
}

/* wave2fault (k_fault.hip, transform.cu:100-212) transposed at welded nodes */
__global__ void __launch_bounds__(kNodeLanes) k_adjf_w2f(AdjFaultArgs a) {
  const int iy = blockIdx.x * kNodeLanes + threadIdx.x, iz = blockIdx.y;
  if (iy >= a.g.nj) return;
  const int id = blockIdx.z;
  const FaultDev &F = a.ftab[id];
  const long ss = a.g.sslice, sc = a.g.sicmp;
  const long pf = (iy + 3) + (long)(iz + 3) * a.g.ny;
  if (F.united[pf] != 1) return;
  const long p = F.i0 + (long)(iy + 3) * a.g.siy + (long)(iz + 3) * a.g.siz;
  float *blk = adj_block(a, id);
  float *aT1 = blk + kOffT1 * ss, *aC = adj_lev(a, blk, a.lc);
  float *W = a.wT;
  float aTr[3][3], aV[3], w[9], jac, M[3][3];
#pragma unroll
  for (int c = 0; c < 3; c++) {
    aTr[c][0] = aT1[(long)(7 * c + 3) * ss + pf];
    aTr[c][1] = aTr[c][2] = aV[c] = 0.0f;
#pragma unroll
    for (int m = 0; m < 2; m++) {
      aV[c] += aC[fidx(c, m, ss) + pf];
      aTr[c][1] += aC[fidx(3 + c, m, ss) + pf];
      aTr[c][2] += aC[fidx(6 + c, m, ss) + pf];
    }
  }
  load_met(a.met, sc, p, jac, M);
#pragma unroll
  for (int f = 0; f < 9; f++) w[f] = W[f * sc + p];
  float aS[3][3];
#pragma unroll
  for (int r = 0; r < 3; r++)
#pragma unroll
    for (int k = 0; k < 3; k++) aS[r][k] = jac * (aTr[r][0] * M[k][0] + aTr[r][1] * M[k][1] + aTr[r][2] * M[k][2]);
#pragma unroll
  for (int c = 0; c < 3; c++) {
    aT1[(long)(7 * c + 3) * ss + pf] = 0.0f;
    W[c * sc + p] = w[c] + aV[c];
  }
#pragma unroll
  for (int q = 0; q < 18; q++) aC[q * ss + pf] = 0.0f;
  W[TXX * sc + p] = w[TXX] + aS[0][0];
  W[TYY * sc + p] = w[TYY] + aS[1][1];
  W[TZZ * sc + p] = w[TZZ] + aS[2][2];
  W[TXY * sc + p] = w[TXY] + (aS[0][1] + aS[1][0]);
  W[TXZ * sc + p] = w[TXZ] + (aS[0][2] + aS[2][0]);
  W[TYZ * sc + p] = w[TYZ] + (aS[1][2] + aS[2][1]);
}

/* ---------------------------------------------------------------------- */
static dim3 node_grid(const AdjFaultArgs &a) { return dim3((a.g.nj + kNodeLanes - 1) / kNodeLanes, a.g.nk, a.nfault); }

void launch_adjf_begin(const AdjFaultArgs &a, hipStream_t st) {
  if (a.nfault <= 0) return;
  hipLaunchKernelGGL(k_adjf_begin, node_grid(a), dim3(kNodeLanes), 0, st, a);
}

void launch_adjf_receivers(const AdjFaultArgs &a, const int *rec, const float *fac, int nterm, int nrec,
                           const float *res, int nt, int sample, hipStream_t st) {
  if (a.nfault <= 0 || nrec <= 0 || !res) return;
  hipLaunchKernelGGL(k_adjf_receivers, dim3((nrec * nterm + 63) / 64), dim3(64), 0, st, a, rec, fac, nterm, nrec, res,
                     nt, sample);
}

void launch_adjf_stage_pre(const AdjFaultArgs &a, hipStream_t st) {
  if (a.nfault <= 0) return;
  const dim3 g = node_grid(a), b(kNodeLanes);
  switch (a.istage) {
    case 3: hipLaunchKernelGGL(k_adjf_lev<3>, g, b, 0, st, a); break;
    case 2: hipLaunchKernelGGL(k_adjf_lev<2>, g, b, 0, st, a); break;
    case 1: hipLaunchKernelGGL(k_adjf_lev<1>, g, b, 0, st, a); break;
    default: hipLaunchKernelGGL(k_adjf_lev<0>, g, b, 0, st, a); break;
  }
}

void launch_adjf_stage_post(const AdjFaultArgs &a, hipStream_t st) {
  if (a.nfault <= 0) return;
  /* tiles from ghost row and plane 0 */
  const dim3 cg((a.g.nj + 6 + kColNodes - 1) / kColNodes, (a.g.nk + 6 + kColRows - 1) / kColRows, a.nfault);
  if (a.idir == 1) {
    hipLaunchKernelGGL(k_adjf_cols<1>, cg, dim3(kColLanes), 0, st, a);
    hipLaunchKernelGGL(k_adjf_nodes<1>, node_grid(a), dim3(kNodeLanes), 0, st, a);
  } else {
    hipLaunchKernelGGL(k_adjf_cols<0>, cg, dim3(kColLanes), 0, st, a);
    hipLaunchKernelGGL(k_adjf_nodes<0>, node_grid(a), dim3(kNodeLanes), 0, st, a);
  }
  hipLaunchKernelGGL(k_adjf_trial, node_grid(a), dim3(kNodeLanes), 0, st, a);
  hipLaunchKernelGGL(k_adjf_w2f, node_grid(a), dim3(kNodeLanes), 0, st, a);
}

}  // namespace cgfd
