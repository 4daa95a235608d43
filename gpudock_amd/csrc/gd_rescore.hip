/*
 * gd_rescore.hip -- FP64 energies of given poses on gfx950.
 *
 * The reference formulas (calcenergy_d.cu:69-309) in double.  A workgroup
 * takes a task: one or two poses on one protein conformer, `split` = 8 or 4
 * wavefronts each.  It stages the conformer's pocket points and the pair
 * table in LDS, places the poses' atoms there in double, and every
 * wavefront then sums its slices of the pose: slice i holds ligand atoms
 * i, i + 8, ..., KDE rounds and position restraints of the same indices.
 * Every slice is summed on its own and the eight sums are added in order,
 * so a pose's energies have the same bits however many wavefronts share it.
 *
 * What bounds it: FP64 VALU issue (a wavefront instruction takes four
 * cycles of its SIMD; about 105 a 64-pair chunk now, 70 % of the issue slots).
 * One pair needs d, 1/d^6, 1/d^9, two quotients and an exponential: from one
 * v_rsq_f64 and one v_rcp_f64, each refined by one third-order step, and a
 * degree-11 exponential, in place of a library sqrt, five divisions and exp.
 * Two atoms of a slice run through the point loop together: they share the
 * point's LDS reads and conversions and the loop's branches, and each hides
 * the other's latency.  One wavefront per pose with library math and the
 * tables read through the caches | this split, an atom at a time between the
 * branches, literal coefficients | as it is: 16,384 poses of 48 atoms x 800
 * points 6.12 | 2.07 | 1.96 ms, 4,096 of them - | 674 | 621 us, 4,096 of 128 x
 * 4,000 18.8 | 7.71 | 6.89 ms, 592 of 61 x 1,037 662 | 166 | 155 us, one pose of
 * 24 x 300 114 | 18 | 18 us.  The error against 80-bit arithmetic is as before
 * or smaller (1e-16 of the energies' norm).
 */
#include <hip/hip_runtime.h>
#include "gd_device.h"
#include "gd_launch.h"

#define GD_R64_WAVES 8                 /* wavefronts of a workgroup */
#define GD_R64_SLICES 8

typedef __attribute__((address_space(3))) double gd_lds_f64;

/* ------------------------------------------------------------------------ */
/* FP64 building blocks                                                      */
/* ------------------------------------------------------------------------ */
/* 1/sqrt(x), x positive and finite: the hardware estimate (relative error e
 * below 2^-22) and one third-order step, error e^3. */
__device__ __forceinline__ double gd_rsqrt64(double x)
{
  const double y = __builtin_amdgcn_rsq(x);
  const double e = __builtin_fma(-(x * y), y, 1.0);
  return __builtin_fma(y * e, __builtin_fma(0.375, e, 0.5), y);
}

/* 1/x, x finite and non-zero: estimate and one third-order step. */
__device__ __forceinline__ double gd_rcp64(double x)
{
  const double y = __builtin_amdgcn_rcp(x);
  const double e = __builtin_fma(-x, y, 1.0);
  return __builtin_fma(y, __builtin_fma(e, e, e), y);
}

/* e^x for x <= 709: n = round(x / ln2) by adding 1.5 * 2^52 (its integer
 * is then the low word), r = x - n ln2 in two steps, e^r = 1 + r + r^2 q(r)
 * with q of degree 9 interpolated here at the Chebyshev nodes of
 * |r| <= ln2 / 2 (truncation below 1e-17), scaled by v_ldexp_f64.  Clamped at
 * -700 (1e-304: no sum can tell it from 0) by a compare, which leaves a NaN a
 * NaN where a maximum would drop it.  The coefficients of r^11 .. r^3
 * come in scalar registers (gd_exp64_coeffs): as literals each is copied into
 * the accumulator of its fma first, a fifth of the pair loop's instructions. */
struct gd_exp64_c {
  double c[9];
};

__device__ __forceinline__ gd_exp64_c gd_exp64_coeffs()
{
  gd_exp64_c K = {{0x1.af389ecfc4b9cp-26, 0x1.28917c89a43a7p-22, 0x1.71de0db2f6b19p-19,
                   0x1.a019b9149a41cp-16, 0x1.a01a01a7c2efep-13, 0x1.6c16c17889ef1p-10,
                   0x1.11111111109b5p-7, 0x1.5555555553d68p-5, 0x1.5555555555556p-3}};
#pragma unroll
  for (int k = 0; k < 9; ++k)
    asm volatile("" : "+s"(K.c[k]));
  return K;
}

__device__ __forceinline__ double gd_exp64(double x, const gd_exp64_c &K)
{
  const double xc = x < -700.0 ? -700.0 : x;
  const double t = __builtin_fma(xc, 0x1.71547652b82fep+0, 0x1.8p+52);
  const double n = t - 0x1.8p+52;
  double r = __builtin_fma(-n, 0x1.62e42fefa39efp-1, xc);
  r = __builtin_fma(-n, 0x1.abc9e3b39803fp-56, r);
  double p = K.c[0];
#pragma unroll
  for (int k = 1; k < 9; ++k)
    p = __builtin_fma(p, r, K.c[k]);
  p = __builtin_fma(p, r, 0.5);
  p = __builtin_fma(p, r, 1.0);
  p = __builtin_fma(p, r, 1.0);
  return __builtin_amdgcn_ldexp(p, __double2loint(t));
}

template <int CTRL>
__device__ __forceinline__ double gd_dpp64(double v)
{
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xF, 0xF, false);
  return __hiloint2double(hi, lo);
}

/* Lane `lane`'s value, uniform. */
__device__ __forceinline__ double gd_bcast64(double v, int lane)
{
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                          __builtin_amdgcn_readlane(__double2loint(v), lane));
}

/* Sum over the 64 lanes, uniform: pairs of lanes by DPP within a row of 16,
 * then row 0 into row 1 and row 2 into row 3 (row_bcast:15), and row 1 into
 * row 3 (row_bcast:31), read from lane 63. */
__device__ __forceinline__ double gd_wave_sum64(double v)
{
  v += gd_dpp64<0xB1>(v);
  v += gd_dpp64<0x4E>(v);
  v += gd_dpp64<0x141>(v);
  v += gd_dpp64<0x140>(v);
  v += gd_dpp64<0x142>(v);
  v += gd_dpp64<0x143>(v);
  return gd_bcast64(v, 63);
}

/* ------------------------------------------------------------------------ */
/* The Bayesian total in FP64: the same fitted pdfs and the same floor (1e-8 */
/* for a zero or non-finite pdf or an exponential factor below e^-86).       */
/* ------------------------------------------------------------------------ */
__device__ double gd_pdf64(int family, double x, double loc, double scale)
{
  const double pi = 3.14159265358979323846;
  double v, arg = 0.0;
  if (family == 0) {
    const double d = x - loc;
    arg = -d * d / (2.0 * scale * scale);
    v = exp(arg) / (scale * sqrt(2.0 * pi));
  } else if (family == 1) {
    const double t = (x - loc) / scale;
    v = 1.0 / (pi * scale * (1.0 + t * t));
  } else if (family == 2) {
    arg = -fabs((x - loc) / scale);
    const double e = exp(arg);
    v = e / ((1.0 + e) * (1.0 + e)) / scale;
  } else {
    const double nx = (x - loc) / scale;
    if (!(nx > 0.0))
      return 1e-8;
    arg = -(nx - 1.0) * (nx - 1.0) / (2.0 * nx);
    v = exp(arg) / (sqrt(2.0 * pi * nx * nx * nx) * scale);
  }
  return (v > 0.0 && v < HUGE_VAL && arg >= -86.0) ? v : 1e-8;
}

__device__ double gd_bayes_total64(const double nf[9])
{
  const float hi[9][2] = GD_BAYES_HIGH_INIT;
  const float lo[9][2] = GD_BAYES_LOW_INIT;
  const int fam[9] = GD_BAYES_FAMILY_INIT;
  double ph = 0.0, pl = 0.0;
  for (int k = 0; k < 9; ++k) {
    ph += log10(gd_pdf64(fam[k], nf[k], hi[k][0], hi[k][1]));
    pl += log10(gd_pdf64(fam[k], nf[k], lo[k][0], lo[k][1]));
  }
  return pl - ph;
}

/* ------------------------------------------------------------------------ */
/* Pair loop                                                                 */
/* ------------------------------------------------------------------------ */
/* What every pair needs, uniform. */
struct gd_r64_consts {
  double lj0, lj01;            /* soft-LJ: p4 = 1 + p1 (lj0 + lj0 lj1 d^2) */
  double el0, a1, b1, el1;     /* g(s) = el0 + a1 s^2 + b1 s^3 below s = el1 d = 1 */
  double inv_el1;
  unsigned near_hi, far_hi;    /* high words of dcut^2 (just above) and of infinity */
  gd_exp64_c K;
};

struct gd_r64_acc {
  double vdw, ele, pmf, psp, hdb;
};

/* The pairs of M ligand atoms with every pocket point: lane partials into
 * acc, and hacc[i] = twice atom i's hydrophobic sum.  ele: sum of
 * ele_point g per atom times its charge. */
template <int M>
__device__ __forceinline__ void gd_r64_atoms(const gd_pack &P, const char *smem, int prt,
                                             bool pocket_lds, int off_tab,
                                             const gd_r64_consts &C, const double (*xyz)[3],
                                             const gd_atom_rec *ar, gd_r64_acc &acc,
                                             double *hacc)
{
  const int lane = threadIdx.x & (GD_WAVE - 1);
  const int nchunk = P.pnp_pad / GD_WAVE;
  const int kp = __builtin_amdgcn_readfirstlane(P.chunk_bounds[2 * prt + 1]);
  const float4 *g_pos = P.pt_pos + (size_t) prt * P.pnp_pad;
  const float2 *g_eh = P.pt_eh + (size_t) prt * P.pnp_pad;
  const float *g_psp = P.psp_pt + (size_t) prt * P.n_rows * P.pnp_pad;
  double ele[M];
  int any_hdb = 0;
#pragma unroll
  for (int i = 0; i < M; ++i) {
    ele[i] = 0.0;
    hacc[i] = 0.0;
    any_hdb |= ar[i].hdb;
  }
  any_hdb = __builtin_amdgcn_readfirstlane(any_hdb);
  for (int k = 0; k < nchunk; ++k) {
    float4 q;
    float2 eh;
    if (pocket_lds) {
      const float2 *c = (const float2 *) (smem + k * GD_LDS_CHUNK_BYTES) + lane;
      const float2 xy = c[0], zw = c[GD_WAVE];
      q = make_float4(xy.x, xy.y, zw.x, zw.y);
      eh = c[2 * GD_WAVE];
    } else {
      q = g_pos[k * GD_WAVE + lane];
      eh = g_eh[k * GD_WAVE + lane];
    }
    const bool lead = k < kp;   /* chunks with hydrophobic or class-2 points */
    float pv[M];
#pragma unroll
    for (int i = 0; i < M; ++i)
      pv[i] = lead ? g_psp[(size_t) ar[i].row * P.pnp_pad + k * GD_WAVE + lane] : 0.0f;
    const double qx = q.x, qy = q.y, qz = q.z, qe = eh.x, qh = eh.y;
    const unsigned bits = __float_as_uint(q.w);
    /* the atoms side by side, branches shared: the one's chain of dependent
     * operations fills the other's waits */
    const char *row[M];
    float4 tp[M];
    double d2[M], r1[M], d[M], dl[M], g[M], dm[M];
    bool out = false;
#pragma unroll
    for (int i = 0; i < M; ++i) {
      row[i] = smem + off_tab + ar[i].row * (GD_ROW_STRIDE * (int) sizeof(gd_pair_param)) + bits;
      tp[i] = *(const float4 *) row[i];   /* p1a p2a pmf0 pmf1 */
      const double dx = xyz[i][0] - qx, dy = xyz[i][1] - qy, dz = xyz[i][2] - qz;
      d2[i] = __builtin_fma(dz, dz, __builtin_fma(dy, dy, dx * dx));
      r1[i] = gd_rsqrt64(d2[i]);
      d[i] = d2[i] * r1[i];
      dl[i] = d2[i];                      /* d^2 of the soft-LJ denominator */
      g[i] = r1[i] * C.inv_el1;
      out |= (unsigned) __double2hiint(d2[i]) - C.near_hi >= C.far_hi - C.near_hi;
    }
    /* pairs inside the short range, and the degenerate distances 0 and
     * infinity, in a branch that a wavefront seldom takes (one unsigned
     * compare of the high word finds both) */
    if (__ballot(out)) {
      asm volatile("");
#pragma unroll
      for (int i = 0; i < M; ++i) {
        if (d2[i] == 0.0 || d2[i] == HUGE_VAL) {
          /* the soft-LJ quotient is inf - inf or 0 inf there; the others
           * are finite */
          r1[i] = 0.0;
          d[i] = d2[i];
          dl[i] = 0.0;
          g[i] = 0.0;
          acc.vdw += __builtin_nan("");
        }
        const double s = C.el1 * d[i];
        if (s < 1.0)
          g[i] = __builtin_fma(s * s, __builtin_fma(C.b1, s, C.a1), C.el0);
      }
    }
#pragma unroll
    for (int i = 0; i < M; ++i) {
      const double r2 = r1[i] * r1[i];
      const double r3 = r2 * r1[i];
      const double r6 = r3 * r3;
      const double p1 = (double) tp[i].x * (r6 * r3);
      const double p2 = (double) tp[i].y * r6;
      const double p4 = __builtin_fma(p1, __builtin_fma(C.lj01, dl[i], C.lj0), 1.0);
      ele[i] = __builtin_fma(qe, g[i], ele[i]);
      dm[i] = d[i] - (double) tp[i].z;
      const double q1 = 1.0 + gd_exp64(__builtin_fma(-0.5, d[i], 6.0) * dm[i], C.K);
      const double rr = gd_rcp64(p4 * q1);   /* serves both quotients */
      acc.vdw = __builtin_fma((p1 - p2) * q1, rr, acc.vdw);
      acc.pmf = __builtin_fma((double) tp[i].w * p4, rr, acc.pmf);
    }
    if (lead) {
#pragma unroll
      for (int i = 0; i < M; ++i) {
        acc.psp += dm[i] <= 0.0 ? (double) pv[i] : 0.0;
        /* (1 - u)^3 (1 - u/2) = w^3 (1 + w) / 2, u = d^2 / 81, w = 1 - u */
        const double w = __builtin_fmax(__builtin_fma(d2[i], -1.0 / 81.0, 1.0), 0.0);
        hacc[i] = __builtin_fma((w * w) * w, __builtin_fma(w, qh, qh), hacc[i]);
      }
    }
    if (any_hdb) {
      float2 hb[M];
      bool on = false;
#pragma unroll
      for (int i = 0; i < M; ++i) {
        hb[i] = *(const float2 *) (row[i] + 16);   /* hdb0 hdb1 */
        on |= hb[i].x > 0.1f;
      }
      if (on) {
#pragma unroll
        for (int i = 0; i < M; ++i) {
          const double h = (d[i] - (double) hb[i].x) * (double) hb[i].y;
          const double v = __builtin_fma((double) hb[i].y, gd_exp64((-0.5 * h) * h, C.K), acc.hdb);
          acc.hdb = hb[i].x > 0.1f ? v : acc.hdb;
        }
      }
    }
  }
#pragma unroll
  for (int i = 0; i < M; ++i)
    acc.ele = __builtin_fma((double) ar[i].q, ele[i], acc.ele);
}

/* ------------------------------------------------------------------------ */
/* The kernel.  items: tasks of up to 8 / split poses.  Poses come from      */
/* order[] (pose ids into lig_conf and move, energies at row id) or, with    */
/* order null, are the best poses of replicas begin .. begin + count - 1 of  */
/* the task's complex, energies from row `out` on.                           */
/* ------------------------------------------------------------------------ */
__global__ void __launch_bounds__(GD_WAVE *GD_R64_WAVES) __attribute__((amdgpu_waves_per_eu(4, 8)))
gd_rescore64_kernel(const gd_pack *__restrict__ packs, const gd_r64_task *__restrict__ tasks,
                    int split, int max_lna, int lds_bytes, const int *__restrict__ order,
                    const int *__restrict__ lig_conf, const float *__restrict__ move,
                    double *__restrict__ energy)
{
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const gd_r64_task task = tasks[blockIdx.x];
  const gd_pack &P = packs[task.cx];
  const int lane = threadIdx.x & (GD_WAVE - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / GD_WAVE);
  const int G = GD_R64_WAVES / split;
  const int slot = wave / split, part = wave - slot * split;
  const int lna = P.lna, prt = task.prt;

  /* LDS: the poses' areas at the end, the pocket (when it fits) and the
   * pair table before them */
  const int area = gd_r64_area_bytes(max_lna);
  const int tab_bytes = P.n_rows * GD_ROW_STRIDE * (int) sizeof(gd_pair_param);
  const int pocket_bytes = P.pnp_pad / GD_WAVE * GD_LDS_CHUNK_BYTES;
  const bool pocket_lds = pocket_bytes + tab_bytes + G * area <= lds_bytes;
  const int off_tab = pocket_lds ? pocket_bytes : 0;
  gd_lds_f64 *A = (gd_lds_f64 *) (smem + lds_bytes - (G - slot) * area);
  gd_lds_f64 *ax = A, *ay = A + max_lna, *az = A + 2 * max_lna, *aw = A + 3 * max_lna;
  gd_lds_f64 *S = A + 4 * max_lna;   /* [slice][term] */

  if (pocket_lds) {
    const float4 *g_pos = P.pt_pos + (size_t) prt * P.pnp_pad;
    const float2 *g_eh = P.pt_eh + (size_t) prt * P.pnp_pad;
    for (int i = threadIdx.x; i < P.pnp_pad; i += blockDim.x) {
      const float4 q = g_pos[i];
      float2 *c = (float2 *) (smem + (i / GD_WAVE) * GD_LDS_CHUNK_BYTES) + (i & (GD_WAVE - 1));
      c[0] = make_float2(q.x, q.y);
      c[GD_WAVE] = make_float2(q.z, q.w);
      c[2 * GD_WAVE] = g_eh[i];
    }
  }
  {
    float4 *s_tab = (float4 *) (smem + off_tab);
    const float4 *g_tab = (const float4 *) P.tab;
    for (int i = threadIdx.x; i < P.n_rows * GD_ROW_STRIDE * 2; i += blockDim.x)
      s_tab[i] = g_tab[i];
  }

  const bool active = slot < task.count;
  int id = 0, lconf = 0;
  const float *mv = nullptr;
  double *out = nullptr;
  double cen[3] = {0.0, 0.0, 0.0};
  if (active) {
    if (order) {
      id = order[task.begin + slot];
      lconf = lig_conf[id];
      mv = move + (size_t) id * 6;
      out = energy + (size_t) id * 10;
    } else {
      id = task.begin + slot;
      lconf = P.rep_lig[id];
      mv = P.S.mv_best + (size_t) id * 8;
      out = energy + ((size_t) task.out + slot) * 10;
    }
    for (int k = 0; k < 3; ++k)
      cen[k] = (double) P.center[k] + (double) mv[k];
  }
  if (active && part == 0) {
    /* the three angles in lanes 0-2 of every group of four */
    const double ang = (double) mv[3 + ((lane & 3) < 3 ? (lane & 3) : 2)];
    const double sn = sin(ang), cs = cos(ang);
    const double s1 = gd_bcast64(sn, 0), s2 = gd_bcast64(sn, 1), s3 = gd_bcast64(sn, 2);
    const double c1 = gd_bcast64(cs, 0), c2 = gd_bcast64(cs, 1), c3 = gd_bcast64(cs, 2);
    const double R[9] = {c1 * c2, c1 * s2 * s3 - c3 * s1, s1 * s3 + c1 * c3 * s2,
                         c2 * s1, c1 * c3 + s1 * s2 * s3, c3 * s1 * s2 - c1 * s3,
                         -s2,     c2 * s3,                c2 * c3};
    for (int l = lane; l < lna; l += GD_WAVE) {
      const float4 o = P.lig_xyz[(size_t) lconf * lna + l];
      ax[l] = R[0] * o.x + R[1] * o.y + R[2] * o.z + cen[0];
      ay[l] = R[3] * o.x + R[4] * o.y + R[5] * o.z + cen[1];
      az[l] = R[6] * o.x + R[7] * o.y + R[8] * o.z + cen[2];
      const int row = P.lig_row[l];
      const int n = P.kde_seg[2 * row + 1] - P.kde_seg[2 * row];
      aw[l] = n > 0 ? 1.0 / (double) n : 0.0;
    }
  }
  __syncthreads();

  if (active) {
    gd_r64_consts C;
    C.K = gd_exp64_coeffs();
    {
      const double lj0 = P.sc.lj0, el0 = P.sc.el0, el1 = P.sc.el1;
      C.lj0 = lj0;
      C.lj01 = lj0 * (double) P.sc.lj1;
      C.el0 = el0;
      C.el1 = el1;
      C.a1 = 4.0 - 3.0 * el0;
      C.b1 = 2.0 * el0 - 3.0;
      C.inv_el1 = 1.0 / el1;
      C.far_hi = 0x7ff00000u;
      C.near_hi = el1 > 0.0 ? (unsigned) __double2hiint(C.inv_el1 * C.inv_el1) + 1u : C.far_hi;
      if (C.near_hi > C.far_hi)
        C.near_hi = C.far_hi;   /* every pair inside: the branch is always taken */
    }
    const int r_lo = (P.kde_n_lo + GD_WAVE - 1) / GD_WAVE;
    const int n_rounds = r_lo + (P.kde_n_hi + GD_WAVE - 1) / GD_WAVE;
    for (int sl = part; sl < GD_R64_SLICES; sl += split) {
      gd_r64_acc acc = {0.0, 0.0, 0.0, 0.0, 0.0};
      double hpc = 0.0;
      /* the restraint on an atom's hydrophobic sum (calcenergy_d.cu:142-149) */
      auto restrain = [&](int l, double h2) {
        const int t = P.lig_type[l];
        const double z = (0.5 * gd_wave_sum64(h2) - (double) P.hpl0[t]) / (double) P.hpl1[t];
        hpc += 0.5 * z * z - (double) P.hpl2[t];
      };
      int l = sl;
      for (; l + GD_R64_SLICES < lna; l += 2 * GD_R64_SLICES) {
        const int m = l + GD_R64_SLICES;
        const double xyz[2][3] = {{ax[l], ay[l], az[l]}, {ax[m], ay[m], az[m]}};
        const gd_atom_rec ar[2] = {P.atom[l], P.atom[m]};
        double h2[2];
        gd_r64_atoms<2>(P, smem, prt, pocket_lds, off_tab, C, xyz, ar, acc, h2);
        restrain(l, h2[0]);
        restrain(m, h2[1]);
      }
      if (l < lna) {
        const double xyz[1][3] = {{ax[l], ay[l], az[l]}};
        const gd_atom_rec ar[1] = {P.atom[l]};
        double h2[1];
        gd_r64_atoms<1>(P, smem, prt, pocket_lds, off_tab, C, xyz, ar, acc, h2);
        restrain(l, h2[0]);
      }
      double kde = 0.0;
      for (int r = sl; r < n_rounds; r += GD_R64_SLICES) {
        const unsigned e = P.kde_pairs[r * GD_WAVE + lane];
        const int a = (int) ((e & 0xffu) >> 2) + (r >= r_lo ? GD_WAVE : 0);
        const float4 q = P.kde[e >> 16];
        const double ex = ax[a] - q.x, ey = ay[a] - q.y, ez = az[a] - q.z;
        const double d2 = __builtin_fma(ez, ez, __builtin_fma(ey, ey, ex * ex));
        /* the pairs that pad a round name a point of weight 0 */
        kde += q.w != 0.0f ? aw[a] * gd_exp64((double) P.kde2 * d2, C.K) : 0.0;
      }
      double lhm = 0.0;
      for (int mm = sl; mm < P.pos; mm += GD_R64_SLICES) {
        double s = 0.0;
        int c = 0;
        for (int b = 0; b < lna; b += GD_WAVE) {
          const int a = b + lane;
          bool have = false;
          if (a < lna) {
            const float4 t = P.mcs[(size_t) mm * lna + a];
            have = t.w != 0.0f;
            if (have) {
              const double ex = ax[a] - t.x, ey = ay[a] - t.y, ez = az[a] - t.z;
              s += ex * ex + ey * ey + ez * ez;
            }
          }
          c += __popcll(__ballot(have));
        }
        s = gd_wave_sum64(s);
        if (c > 0)
          lhm += (double) P.mcs_tcc[mm] * sqrt(s / (double) c);
      }
      const double v[8] = {gd_wave_sum64(acc.vdw), gd_wave_sum64(acc.ele),
                           gd_wave_sum64(acc.pmf), hpc,
                           gd_wave_sum64(acc.hdb), gd_wave_sum64(acc.psp),
                           gd_wave_sum64(kde), lhm};
      if (lane == 0) {
#pragma unroll
        for (int k = 0; k < 8; ++k)
          S[sl * 8 + k] = v[k];
      }
    }
  }
  __syncthreads();

  if (active && part == 0) {
    /* one term per lane: lane f < 9 forms file-order term f (vdw ele pmf hpc
     * hdb dst psp kde lhm) */
    const int f = lane < GD_F_NTERM ? lane : 0;
    const int col = f < GD_F_DST ? f : f - 1;   /* its column in S */
    double x = 0.0;
    for (int sl = 0; sl < GD_R64_SLICES; ++sl)
      x += S[sl * 8 + (f == GD_F_DST ? 0 : col)];
    double y = x;
    if (f == GD_F_KDE)
      y = y / (double) P.kde3;
    y = y / (double) lna;
    if (f == GD_F_HDB)
      y = -y / sqrt(2.0 * 3.14159265358979323846);
    if (f == GD_F_DST) {
      const double dx = cen[0] - P.pocket_center[0], dy = cen[1] - P.pocket_center[1],
                   dz = cen[2] - P.pocket_center[2];
      y = sqrt(dx * dx + dy * dy + dz * dz);
    }
    if (f == GD_F_LHM)
      y = P.pos > 0 ? log(x / (double) P.pos) : 0.0;
    const int f2s[GD_F_NTERM] = GD_FILE_TO_SLOT_INIT;
    int my_slot = 0;
#pragma unroll
    for (int k = 0; k < GD_F_NTERM; ++k)
      my_slot = f == k ? f2s[k] : my_slot;
    /* parameters by file-order term, or by slot */
    const int par = P.term_order == 0 ? f : my_slot;
    const double v = (double) P.a_para[par] * y + (double) P.b_para[par];
    double total = 0.0, nf[GD_F_NTERM];
#pragma unroll
    for (int k = 0; k < GD_F_NTERM; ++k)
      nf[k] = gd_bcast64(v, k);
    if (P.combine == 1) {
      total = gd_bayes_total64(nf);
    } else {
      /* w x value in parameter order */
#pragma unroll
      for (int k = 0; k < GD_F_NTERM; ++k) {
        double u = nf[k];
        if (P.term_order != 0) {
#pragma unroll
          for (int j = 0; j < GD_F_NTERM; ++j)
            u = f2s[j] == k ? nf[j] : u;
        }
        total += (double) P.w[k] * u;
      }
    }
    if (lane < GD_F_NTERM)
      out[my_slot] = v;
    if (lane == GD_F_NTERM)
      out[GD_E_TOTAL] = total;
  }
}

/* ------------------------------------------------------------------------ */
/* launch                                                                    */
/* ------------------------------------------------------------------------ */
/* Wavefronts per pose: all eight of a workgroup up to four poses a CU, four
 * beyond.  Few poses leave the device idle and a pose's time is its own
 * latency: 256 poses of 48 atoms x 800 points take 62 us with eight, 104
 * with four, 359 with one; with 1,024 poses eight and four are level (152
 * and 161 us; 128 atoms x 4,000 points 1,988 and 1,975), and from 2,048 on
 * four is ahead by 1-2 % where one wavefront per pose is 30 % behind (367
 * against 284 us) and catches up only at 8,192. */
int gd_rescore64_split(long long n_pose, int n_cu) { return n_pose <= 4LL * n_cu ? 8 : 4; }

int gd_rescore64_lds(const gd_pack &P, int split, int max_lna, int max_lds)
{
  const int tab = P.n_rows * GD_ROW_STRIDE * (int) sizeof(gd_pair_param);
  const int pocket = P.pnp_pad / GD_WAVE * GD_LDS_CHUNK_BYTES;
  const int areas = GD_R64_WAVES / split * gd_r64_area_bytes(max_lna);
  return pocket + tab + areas <= max_lds ? pocket + tab + areas : tab + areas;
}

hipError_t gd_launch_rescore64(const gd_pack *packs, const gd_r64_task *tasks, int n_tasks,
                               int split, int max_lna, int lds_bytes, int max_lds,
                               const int *order, const int *lig_conf, const float *move,
                               double *energy, hipStream_t st)
{
  if (n_tasks <= 0)
    return hipSuccess;
  if ((split != 4 && split != 8) || max_lna < 1 ||
      lds_bytes > max_lds)
    return hipErrorInvalidValue;
  /* the device's limit, whatever this launch needs: launches of other
   * threads set the same value */
  hipError_t e = hipFuncSetAttribute((const void *) gd_rescore64_kernel,
                                     hipFuncAttributeMaxDynamicSharedMemorySize, max_lds);
  if (e != hipSuccess)
    return e;
  hipLaunchKernelGGL(gd_rescore64_kernel, dim3(n_tasks), dim3(GD_WAVE * GD_R64_WAVES), lds_bytes,
                     st, packs, tasks, split, max_lna, lds_bytes, order, lig_conf, move, energy);
  return hipGetLastError();
}
