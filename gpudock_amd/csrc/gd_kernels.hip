/*
 * gd_kernels.hip -- CDNA4 (gfx950) kernels of the REMC docking core.
 *
 *   gd_mc_kernel       fused Move + CalcEnergy + Accept for one cycle of MC
 *                      steps of every replica of every resident complex
 *                      (montecarlo_d.cu:59-106 with move_d.cu:73-134,
 *                      calcenergy_d.cu:22-374, accept_d.cu:12-52), or the
 *                      initial energies (MonteCarlo_Init_d, :12-55).
 *   gd_mc_split_kernel the same cycle with one to four replicas split over
 *                      a workgroup's wavefronts (launches with few replicas).
 *   gd_exchange1_kernel / gd_exchange_kernel temperature swaps, one
 *                      wavefront per chain, one lane per temperature pair
 *                      (exchangereplicas_d.cu:7-136), then the advance.
 *   gd_advance_kernel  advances each complex's device step counter after a
 *                      cycle and re-arms the work queue.
 *   gd_score_kernel    energies of caller-given poses (FP32).
 *   gd_pose_split_kernel the same and the initial energies, each pose split
 *                      over a workgroup's wavefronts (few poses).
 * (FP64 energies: gd_rescore.hip.)
 *
 * Execution model: a workgroup takes a task -- up to WPG replicas of one
 * protein conformer of one complex -- either by its block index or, in the
 * persistent form, from a device work queue (an atomic counter over a task
 * list sorted by cost).  It stages that conformer's pocket points, the
 * pair-parameter rows of the ligand's atom types and (when it fits) the
 * type-grouped KDE points in LDS, restaging only when the next task needs
 * another conformer; each wavefront then owns one replica for the whole
 * cycle.  Lanes run over pocket points (over KDE points / ligand atoms in
 * the smaller loops); the ligand atom of the outer loop is broadcast from
 * the lane that holds it with v_readlane, so it sits in scalar registers.
 * The replica's uniform state (movematrices, energies) lives in a per-wave
 * LDS slot, not in vector registers; read-only uniform data (the task, pack
 * fields, each atom's table row, type and charge) is read through the
 * scalar unit, and the per-atom PSP rows and HBM-resident KDE points through
 * raw buffer resources with a fixed lane offset and a scalar chunk offset.  Per-term sums are per-lane FP32
 * accumulators combined with the near-first pairing tree the CPU replay
 * reproduces bit for bit.  The step index of each complex lives in device
 * memory, so the three launches of a cycle (MC, exchange, advance) replay
 * unchanged from a captured hipGraph.
 */
#include <hip/hip_runtime.h>
#include <mutex>
#include "gd_device.h"
#include "gd_launch.h"

/* Word 3 of a raw buffer resource on gfx9-family GPUs (32-bit data
 * format, no swizzle): reads past num_records return 0. */
#define GD_BUFFER_DWORD3 0x00020000

typedef float gd_f4 __attribute__((ext_vector_type(4)));
typedef float gd_f2 __attribute__((ext_vector_type(2)));

template <bool B>
struct gd_bool {
  static constexpr bool value = B;
};

/* The wave's slot in LDS, addressed as LDS (not through flat accesses). */
typedef __attribute__((address_space(3))) float gd_lds_f32;

/* A read of read-only, wave-uniform data through the scalar unit. */
template <typename T>
__device__ __forceinline__ T gd_uload(const T *p)
{
  return *(const __attribute__((address_space(4))) T *) p;
}

/* One atom record through the scalar unit (a single 32-byte load). */
typedef int gd_i8 __attribute__((ext_vector_type(8)));
__device__ __forceinline__ gd_atom_rec gd_load_atom(const gd_atom_rec *p)
{
  return __builtin_bit_cast(gd_atom_rec, *(const __attribute__((address_space(4))) gd_i8 *) p);
}

__device__ __forceinline__ float gd_bcast(float v, int lane)
{
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

template <int CTRL>
__device__ __forceinline__ float gd_dpp(float v)
{
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF,
                                                    false));
}

/* Sum over the 64 lanes with the pairing tree of an xor butterfly taken
 * near-first (lane pairs j^1, then j^2, j^4, j^8, j^16, j^32): DPP
 * quad_perm [1,0,3,2] and [2,3,0,1], row_half_mirror (pairs the two quads
 * of a half-row), row_mirror (pairs the two halves of a row) leave every
 * lane of row i with the row sum r_i; row_bcast:15 adds r0 to row 1 and r2
 * to row 3, row_bcast:31 adds row 1's (r0 + r1) to row 3's (r2 + r3), read
 * from lane 63 (what the other rows receive is not read).  Every partial is the same float addition
 * as in that butterfly (addition commutes), so the result is bit-identical
 * to it; it is returned uniform. */
__device__ __forceinline__ float gd_wave_sum(float v)
{
  v += gd_dpp<0xB1>(v);
  v += gd_dpp<0x4E>(v);
  v += gd_dpp<0x141>(v);
  v += gd_dpp<0x140>(v);
  v += gd_dpp<0x142>(v);   /* rows 1 and 3 are the ones read */
  v += gd_dpp<0x143>(v);   /* row 3 is the one read */
  return gd_bcast(v, 63);
}

/* ------------------------------------------------------------------------ */
/* Workgroup staging                                                         */
/* ------------------------------------------------------------------------ */
__device__ __forceinline__ void gd_stage(const gd_pack &P, int prt, char *smem)
{
  float4 *s_tab = (float4 *) (smem + P.off_tab);
  const int pnp_pad = P.pnp_pad;
  const float4 *g_pos = P.pt_pos + (size_t) prt * pnp_pad;
  const float2 *g_eh = P.pt_eh + (size_t) prt * pnp_pad;
  /* chunk c of 64 points: {x, y} of its points, then {z, type}, then
   * {ele, hpp}, 512 B each */
  if (P.pocket_in_lds)
    for (int i = threadIdx.x; i < pnp_pad; i += blockDim.x) {
      const float4 q = g_pos[i];
      float2 *c = (float2 *) (smem + (i / GD_WAVE) * GD_LDS_CHUNK_BYTES) + (i & (GD_WAVE - 1));
      c[0] = make_float2(q.x, q.y);
      c[GD_WAVE] = make_float2(q.z, q.w);
      c[2 * GD_WAVE] = g_eh[i];
    }
  const float4 *g_tab = (const float4 *) P.tab;
  const int ntab4 = P.n_rows * GD_ROW_STRIDE * 2;
  for (int i = threadIdx.x; i < ntab4; i += blockDim.x)
    s_tab[i] = g_tab[i];
  if (P.kde_in_lds) {
    float4 *s_kde = (float4 *) (smem + P.off_kde);
    const int n_kde = P.pnk + 1;   /* with the zero-weight padding point */
    for (int i = threadIdx.x; i < n_kde; i += blockDim.x)
      s_kde[i] = P.kde[i];
  }
}

/* ------------------------------------------------------------------------ */
/* Energy of one pose (calcenergy_d.cu:22-374), in summation blocks          */
/* (gd_block_size in gd_canon.h): atom blocks of the pair loop, blocks of    */
/* KDE rounds, one item per position restraint.  Lane j holds ligand atoms   */
/* j and j + 64 in (ax0..az0) and (ax1..az1).  prt = the protein conformer   */
/* staged in smem.                                                           */
/* ------------------------------------------------------------------------ */
/* What the energy loops need of a complex and a protein conformer.  The split
 * steps read it once per cycle and keep it, in scalar registers as far as they
 * go and in lanes of vector registers beyond: read where it is used instead,
 * the loads are repeated after every barrier and atomic, six of them one behind
 * the other (some 2,000 cycles) before an atom block's first pair.  One
 * wavefront per replica has no barriers and hides such loads behind the other
 * replicas of its SIMD, so there it is read where it is used: kept over the
 * cycle instead, it spilled 153 scalar registers for 126 (146 for 123 at 6
 * waves a SIMD, where 16,384 replicas of 48 x 800 took 8.30 ms a cycle for
 * 8.19; no difference at the other budgets). */
struct gd_hot {
  int lna, nchunk, pnp_pad;
  int kp;                           /* chunks that hold a class-2 point */
  int off_tab, off_kde, pocket_in_lds, kde_in_lds;
  int pnk, rounds_lo, n_rounds;     /* KDE rounds of atoms < 64, in all */
  float kde2, ea1, eb1, lj0, lj01, el01, dcut2;
  const gd_atom_rec *atom;
  const float *psp;
  const float4 *pos;
  const float2 *eh;
  const unsigned long long *mref;   /* null: no MCC */
  const uint32_t *kde_pairs;
  const float4 *kde;
  const float4 *mcs;
  const float *mcs_tcc;
};

__device__ __forceinline__ gd_hot gd_hot_of(const gd_pack &P, int prt)
{
  gd_hot H;
  H.lna = P.lna;
  H.pnp_pad = P.pnp_pad;
  H.nchunk = P.pnp_pad / GD_WAVE;   /* padding points add exact zeros */
  H.kp = gd_uload(P.chunk_bounds + 2 * prt + 1);
  H.off_tab = P.off_tab;
  H.off_kde = P.off_kde;
  H.pocket_in_lds = P.pocket_in_lds;
  H.kde_in_lds = P.kde_in_lds;
  H.pnk = P.pnk;
  H.rounds_lo = (P.kde_n_lo + GD_WAVE - 1) / GD_WAVE;
  H.n_rounds = H.rounds_lo + (P.kde_n_hi + GD_WAVE - 1) / GD_WAVE;
  H.kde2 = P.kde2;
  H.ea1 = P.sc.ea1;
  H.eb1 = P.sc.eb1;
  H.lj0 = P.sc.lj0;
  H.lj01 = P.sc.lj01;
  H.el01 = P.sc.el01;
  H.dcut2 = P.sc.dcut2;
  H.atom = P.atom;
  H.psp = P.psp_pt + (size_t) prt * P.n_rows * P.pnp_pad;
  H.pos = P.pt_pos + (size_t) prt * P.pnp_pad;
  H.eh = P.pt_eh + (size_t) prt * P.pnp_pad;
  H.mref = P.mcc_ref ? P.mcc_ref + (size_t) prt * P.lna * H.nchunk : nullptr;
  H.kde_pairs = P.kde_pairs;
  H.kde = P.kde;
  H.mcs = P.mcs;
  H.mcs_tcc = P.mcs_tcc;
  return H;
}

/* Lane partials of the directly summed terms over one atom block. */
struct gd_blk {
  float vdw, pmf, psp, hdb, ele;
};

/* Fewest chunks of a pocket that a split replica takes two at a time. */
#define GD_PAIR_CHUNKS 12

/* Two consecutive chunks of one ligand atom at once: per pair the operations
 * of gd_pair_terms, the sums in chunk order, so the same bits as two calls.
 * One pair is a chain of about 40 dependent operations among 54; the two
 * chains are written side by side so that each fills the other's waits. */
__device__ __forceinline__ void gd_pair_terms2(const float (&d2)[2], const float (&ele)[2],
                                               const gd_pair_param (&pp)[2],
                                               const gd_pair_scalars &sc, bool is_c2,
                                               const float (&psp)[2], bool hdb_row,
                                               int near_any, gd_pair_acc &acc,
                                               int (&contact)[2])
{
  float r1[2], d[2], p1[2], p2[2], p4[2], q1[2], rr[2], dm[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    r1[i] = gd_rsqrt(d2[i]);
    d[i] = d2[i] * r1[i];
    const float r2 = r1[i] * r1[i];
    const float r3 = r2 * r1[i];
    const float r6 = r3 * r3;
    const float r9 = r6 * r3;
    p1[i] = pp[i].p1a * r9;
    p2[i] = pp[i].p2a * r6;
    p4[i] = gd_fma(p1[i], gd_fma(sc.lj01, d2[i], sc.lj0), 1.0f);
  }
  if (near_any) {
    GD_KEEP_BRANCH();
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const float gn = gd_fma(d2[i], gd_fma(d[i], sc.eb1, sc.ea1), sc.el01);
      acc.ele = gd_fma(ele[i], d2[i] < sc.dcut2 ? gn : r1[i], acc.ele);
    }
  } else {
#pragma unroll
    for (int i = 0; i < 2; ++i)
      acc.ele = gd_fma(ele[i], r1[i], acc.ele);
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    dm[i] = d[i] - pp[i].pmf0;
    float es;
    const float ep = gd_exp_hot_split(gd_fma(-0.5f, d[i], 6.0f) * dm[i], &es);
    q1[i] = gd_fma(ep, es, 1.0f);
    rr[i] = gd_rcp(p4[i] * q1[i]);
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    acc.vdw = gd_fma((p1[i] - p2[i]) * q1[i], rr[i], acc.vdw);
    acc.pmf = gd_fma(pp[i].pmf1 * p4[i], rr[i], acc.pmf);
    if (is_c2)
      acc.psp += (dm[i] <= 0.0f) ? psp[i] : 0.0f;
    contact[i] = dm[i] <= 0.0f;
  }
  if (hdb_row && (pp[0].hdb0 > 0.1f || pp[1].hdb0 > 0.1f)) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const float h = (d[i] - pp[i].hdb0) * pp[i].hdb1;
      const float v = gd_fma(pp[i].hdb1, gd_exp_hot((-0.5f * h) * h), acc.hdb);
      acc.hdb = pp[i].hdb0 > 0.1f ? v : acc.hdb;
    }
  }
}

/* Pair loop + hydrophobic restraint (calcenergy_d.cu:56-149) over ligand
 * atoms [l0, l1): lane partials from +0 into blk, the block's restraint sum
 * (uniform) into *ehpc_b, MCC confusion counts (uniform) added to tp/fp/fn.
 * The PSP rows come from HBM, the pocket from LDS or HBM as staged. */
template <bool PAIRED>
__device__ __forceinline__ void gd_atoms_block(
    const gd_hot &H, const char *smem, float ax0, float ay0, float az0, float ax1,
    float ay1, float az1, int l0, int l1, gd_blk &blk, float *ehpc_b, int &tp, int &fp,
    int &fn)
{
  const gd_pair_param *__restrict__ s_tab = (const gd_pair_param *) (smem + H.off_tab);
  const int lane = threadIdx.x & (GD_WAVE - 1);
  const int nchunk = H.nchunk;
  /* the near-field coefficients and lj0 sit beside other scalars in one
   * fma (one scalar operand per instruction): held in vector registers, the
   * loop needs no copy per pair */
  gd_pair_scalars sc_v;
  sc_v.ea1 = H.ea1;
  sc_v.eb1 = H.eb1;
  sc_v.lj0 = H.lj0;
  sc_v.lj01 = H.lj01;
  sc_v.el01 = H.el01;
  sc_v.dcut2 = H.dcut2;
  asm volatile("" : "+v"(sc_v.ea1), "+v"(sc_v.eb1), "+v"(sc_v.lj0));
  /* no load may be in flight when the loops begin: the wait for one that an
   * earlier item left unread (the KDE rounds' last prefetch) would stand
   * inside the pair loop and catch its own PSP reads */
  __builtin_amdgcn_s_waitcnt(0x0f70);   /* vmcnt(0) */

  gd_pair_acc acc;
  acc.vdw = 0.0f; acc.ele = 0.0f; acc.pmf = 0.0f; acc.psp = 0.0f; acc.hdb = 0.0f;
  float eele = 0.0f;
  float ehpc = 0.0f;
  /* MCC confusion counts (wave-uniform): contacts now vs reference, from one
   * ballot per chunk against the reference mask, read through scalar loads */
  typedef const __attribute__((address_space(4))) unsigned long long *mask_ptr;
  const mask_ptr mref = (mask_ptr) H.mref;
  typedef const __attribute__((address_space(1))) float *gfloat_ptr;
  const gfloat_ptr psp_prt = (gfloat_ptr) H.psp;
  /* Two chunks at a time from GD_PAIR_CHUNKS chunks on: a cycle of 592
   * replicas of 61 atoms x 17 chunks 757 -> 698 us, of 4,096 of 128 x 63 26.6
   * -> 25.0 ms; of 128 of 32 x 10 107 -> 108 us, of 64 of 24 x 5 64.7 -> 67.9:
   * few chunks leave a rest as long as the pairs. */
  const bool pairs = PAIRED && nchunk >= GD_PAIR_CHUNKS;
  int kp = H.kp;
  if (pairs)   /* whole pairs: the chunk past the bound adds exact zeros */
    kp = min((kp + 1) & ~1, nchunk);
  const unsigned ulane = (unsigned) lane;
  const int pocket_lds = H.pocket_in_lds;
  const __amdgpu_buffer_rsrc_t pos_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      (void *) H.pos, 0, H.pnp_pad * 16, GD_BUFFER_DWORD3);
  const __amdgpu_buffer_rsrc_t eh_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      (void *) H.eh, 0, H.pnp_pad * 8, GD_BUFFER_DWORD3);

  /* the atom loops, for one way of reading the pocket: the choice is made
   * once per call, not per atom */
  auto atoms = [&](auto read) {
    /* atoms l < 64 sit in lane l of (ax0, ay0, az0), atoms l >= 64 in lane
     * l - 64 of (ax1, ay1, az1): one pass per register set, so an atom's
     * coordinates are three readlanes */
#pragma unroll 1
    for (int g = l0 / GD_WAVE; g * GD_WAVE < l1; ++g) {
      const float gx = g ? ax1 : ax0, gy = g ? ay1 : ay0, gz = g ? az1 : az0;
      const int la = l0 > g * GD_WAVE ? l0 : g * GD_WAVE;
      const int lb = l1 < (g + 1) * GD_WAVE ? l1 : (g + 1) * GD_WAVE;
      for (int l = la; l < lb; ++l) {
        const int src = l & (GD_WAVE - 1);
        const float lx = gd_bcast(gx, src);
        const float ly = gd_bcast(gy, src);
        const float lz = gd_bcast(gz, src);
        const gd_atom_rec ar = gd_load_atom(H.atom + l);
        const int row = ar.row;
        const float lq = ar.q;
        const gd_pair_param *trow = s_tab + row * GD_ROW_STRIDE;
        /* the PSP row as a buffer: lane offset fixed, chunk offset scalar */
        const __amdgpu_buffer_rsrc_t psp_rsrc = __builtin_amdgcn_make_buffer_rsrc(
            (void *) (psp_prt + (size_t) row * H.pnp_pad), 0, H.pnp_pad * 4, GD_BUFFER_DWORD3);
        float hacc = 0.0f;
        acc.ele = 0.0f;
        /* chunks [0, kh) hold the hydrophobic-class points (the canonical order
         * puts them first) and [0, kp) the class-2 points, kp >= kh; beyond kp
         * every hydrophobic weight and every PSP value is 0, whose terms would
         * add exact zeros, so that loop leaves the terms (and the PSP read) out */
        auto chunks = [&](auto read, auto hpc_tag, auto hdb_tag, auto psp_tag, int k0, int k1) {
          int k = k0;
          if (PAIRED)
            for (; pairs && k + 1 < k1; k += 2) {
              float4 q[2];
              float2 eh[2];
              float pv[2] = {0.0f, 0.0f}, d2[2];
              gd_pair_param pp[2];
#pragma unroll
              for (int i = 0; i < 2; ++i) {
                read(k + i, q[i], eh[i]);
                if (decltype(psp_tag)::value)
                  pv[i] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
                      psp_rsrc, ulane * 4u, (k + i) * GD_WAVE * 4, 0));
              }
#pragma unroll
              for (int i = 0; i < 2; ++i) {
                pp[i] = *(const gd_pair_param *) ((const char *) trow + __float_as_uint(q[i].w));
                d2[i] = gd_dist2(lx - q[i].x, ly - q[i].y, lz - q[i].z);
                if (decltype(hpc_tag)::value)
                  hacc = gd_hpc_acc2(d2[i], eh[i].y, hacc);
              }
              const int near_any = __ballot(fminf(d2[0], d2[1]) < sc_v.dcut2) != 0;
              const float ele[2] = {eh[0].x, eh[1].x};
              int contact[2];
              gd_pair_terms2(d2, ele, pp, sc_v, decltype(psp_tag)::value, pv,
                             decltype(hdb_tag)::value, near_any, acc, contact);
              if (mref)
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                  const unsigned long long now = __ballot(contact[i]);
                  const unsigned long long ref = mref[(size_t) l * nchunk + k + i];
                  tp += __popcll(now & ref);
                  fp += __popcll(now & ~ref);
                  fn += __popcll(~now & ref);
                }
            }
          for (; k < k1; ++k) {
            float4 q;
            float2 eh;
            read(k, q, eh);
            const uint32_t bits = __float_as_uint(q.w);
            /* the PSP read (chunk base uniform, lane offset fixed) is consumed
             * at the end of the pair; points outside class 2 hold PSP 0 */
            float pv = 0.0f;
            if (decltype(psp_tag)::value)
              pv = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
                  psp_rsrc, ulane * 4u, k * GD_WAVE * 4, 0));
            const float d2 = gd_dist2(lx - q.x, ly - q.y, lz - q.z);
            if (decltype(hpc_tag)::value)
              hacc = gd_hpc_acc2(d2, eh.y, hacc);
            const gd_pair_param pp =
                *(const gd_pair_param *) ((const char *) trow + bits);
            const int near_any = __ballot(d2 < sc_v.dcut2) != 0;
            const int contact = gd_pair_terms(d2, eh.x, &pp, &sc_v, decltype(psp_tag)::value,
                                              pv, decltype(hdb_tag)::value, near_any, &acc);
            if (mref) {
              const unsigned long long now = __ballot(contact);
              const unsigned long long ref = mref[(size_t) l * nchunk + k];
              tp += __popcll(now & ref);
              fp += __popcll(now & ~ref);
              fn += __popcll(~now & ref);
            }
          }
        };
        /* rows of ligand types without any H-bond pair leave that test out;
         * the chunks [kh, kp) (none in what the loaders build) run with the
         * hydrophobic term, whose points there hold hpp = 0 and add exact
         * zeros, so an atom needs two loops, not three */
        auto rows = [&](auto read) {
          const gd_bool<true> on;
          const gd_bool<false> off;
          if (ar.hdb) {
            chunks(read, on, on, on, 0, kp);
            chunks(read, off, on, off, kp, nchunk);
          } else {
            chunks(read, on, off, on, 0, kp);
            chunks(read, off, off, off, kp, nchunk);
          }
        };
        rows(read);
        eele = gd_fma(lq, acc.ele, eele);
        const float hs = 0.5f * gd_wave_sum(hacc);   /* the pairs added twice the kernel */
        const float z = (hs - ar.hpl0) * ar.inv_hpl1;
        ehpc += 0.5f * z * z - ar.hpl2;
      }
    }
  };
  if (pocket_lds) {
    atoms([&](int k, float4 &q, float2 &eh) {
      const float2 *__restrict__ c = (const float2 *) (smem + k * GD_LDS_CHUNK_BYTES) + lane;
      const float2 xy = c[0], zw = c[GD_WAVE];
      q = make_float4(xy.x, xy.y, zw.x, zw.y);
      eh = c[2 * GD_WAVE];
    });
  } else {
    /* whole-protein pockets: the conformer's points as raw buffers, lane
     * offset fixed, chunk offset scalar */
    atoms([&](int k, float4 &q, float2 &eh) {
      const gd_f4 v = __builtin_bit_cast(gd_f4, __builtin_amdgcn_raw_buffer_load_b128(
                                                    pos_rsrc, ulane * 16u, k * GD_WAVE * 16, 0));
      const gd_f2 w = __builtin_bit_cast(gd_f2, __builtin_amdgcn_raw_buffer_load_b64(
                                                    eh_rsrc, ulane * 8u, k * GD_WAVE * 8, 0));
      q = make_float4(v.x, v.y, v.z, v.w);
      eh = make_float2(w.x, w.y);
    });
  }
  blk.vdw = acc.vdw;
  blk.pmf = acc.pmf;
  blk.psp = acc.psp;
  blk.hdb = acc.hdb;
  blk.ele = eele;
  *ehpc_b = ehpc;
}

/* KDE rounds (calcenergy_d.cu:175-213): the pose's (atom, KDE point) pairs as
 * one list, 64 to a round -- atoms < 64 first, then atoms >= 64, each group
 * padded to whole rounds -- so that no lane idles at the end of an atom's
 * short segment.  Lane j of round r takes pair 64 r + j: its atom's
 * coordinates come from the lane that holds the atom, the point carries the
 * pair's weight 1 / (segment length) in .w; the padding pairs name a point
 * of weight 0 after the segments, so they add exact zeros (the sums are
 * never -0) and every lane keeps its sum.  Returns this lane's sum over
 * rounds [r0, r1) from +0. */
__device__ __forceinline__ float gd_kde_rounds(const gd_hot &H, const char *smem, float ax0,
                                               float ay0, float az0, float ax1, float ay1,
                                               float az1, int r0, int r1)
{
  const unsigned ulane = threadIdx.x & (GD_WAVE - 1);
  const float kde2 = H.kde2;
  const int rounds_lo = H.rounds_lo;
  const __amdgpu_buffer_rsrc_t pairs_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      (void *) H.kde_pairs, 0, H.n_rounds * GD_WAVE * 4, GD_BUFFER_DWORD3);
  float lane_sum = 0.0f;
  auto rounds = [&](auto read) {
    /* rounds [ra, rb) of one group, whose atoms lanes hold in (gx, gy, gz);
     * padding entries name lane 0 and the zero-weight point */
    auto entry = [&](int r) -> uint32_t {
      return __builtin_amdgcn_raw_buffer_load_b32(pairs_rsrc, ulane * 4u, r * GD_WAVE * 4, 0);
    };
    auto group = [&](int ra, int rb, float gx, float gy, float gz) {
      if (ra >= rb)
        return;
      /* each round's entries are loaded one round ahead (the last round
       * loads its own again), so the point read does not wait for them */
      uint32_t e_next = entry(ra);
      for (int r = ra; r < rb; ++r) {
        const uint32_t e = e_next;
        e_next = entry(r + 1 < rb ? r + 1 : r);
        const int src = (int) (e & 0xffu);
        const float lx = __int_as_float(__builtin_amdgcn_ds_bpermute(src, __float_as_int(gx)));
        const float ly = __int_as_float(__builtin_amdgcn_ds_bpermute(src, __float_as_int(gy)));
        const float lz = __int_as_float(__builtin_amdgcn_ds_bpermute(src, __float_as_int(gz)));
        const gd_f4 q = read(e >> 12);   /* byte offset of the point */
        const float d2 = gd_dist2(lx - q.x, ly - q.y, lz - q.z);
        float es;
        const float ep = gd_exp_hot_split(kde2 * d2, &es);
        lane_sum = gd_fma(ep * es, q.w, lane_sum);   /* ep * 2^n is exact */
      }
    };
    group(r0, r1 < rounds_lo ? r1 : rounds_lo, ax0, ay0, az0);
    group(r0 > rounds_lo ? r0 : rounds_lo, r1, ax1, ay1, az1);
  };
  if (H.kde_in_lds) {
    const __attribute__((address_space(3))) char *pts =
        (const __attribute__((address_space(3))) char *) (smem + H.off_kde);
    rounds([&](uint32_t off) {
      return *(const __attribute__((address_space(3))) gd_f4 *) (pts + off);
    });
  } else {
    /* from HBM as a raw buffer */
    const __amdgpu_buffer_rsrc_t kde_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        (void *) H.kde, 0, (H.pnk + 1) * 16, GD_BUFFER_DWORD3);
    rounds([&](uint32_t off) {
      return __builtin_bit_cast(gd_f4, __builtin_amdgcn_raw_buffer_load_b128(kde_rsrc, off, 0,
                                                                             0));
    });
  }
  return lane_sum;
}

/* Position restraint m (calcenergy_d.cu:240-258): tcc_m sqrt(mean squared
 * distance of the atoms it names), 0 when it names none (uniform). */
__device__ __forceinline__ float gd_lhm_one(const gd_hot &H, float ax0, float ay0, float az0,
                                            float ax1, float ay1, float az1, int m)
{
  const int lane = threadIdx.x & (GD_WAVE - 1);
  const int lna = H.lna;
  float s = 0.0f;
  int c = 0;   /* atoms it names */
  const float4 *tm = H.mcs + (size_t) m * lna;
  float4 t0 = make_float4(0.0f, 0.0f, 0.0f, 0.0f), t1 = t0;
  if (lane < lna)
    t0 = tm[lane];
  if (lane + GD_WAVE < lna)
    t1 = tm[lane + GD_WAVE];
  if (t0.w != 0.0f)
    s += gd_dist2(ax0 - t0.x, ay0 - t0.y, az0 - t0.z);
  if (t1.w != 0.0f)
    s += gd_dist2(ax1 - t1.x, ay1 - t1.y, az1 - t1.z);
  c = __popcll(__ballot(t0.w != 0.0f)) + __popcll(__ballot(t1.w != 0.0f));
  s = gd_wave_sum(s);
  return c > 0 ? gd_uload(H.mcs_tcc + m) * gd_sqrt(s / (float) c) : 0.0f;
}

/* distance of the placed centre to the pocket centre (calcenergy_d.cu:276-283) */
__device__ __forceinline__ float gd_edst(const float pc[3], const float cen[3])
{
  return gd_sqrt(gd_dist2(cen[0] - pc[0], cen[1] - pc[1], cen[2] - pc[2]));
}

/* From the lane totals to the energies: wave sums, KDE normalisation, the
 * restraint log, the distance term, averaging, normalisation and total
 * (calcenergy_d.cu:276-371); out[] (slot order) and *cmcc uniform. */
__device__ __forceinline__ void gd_energy_tail(const gd_pack &P, const gd_blk &tot,
                                               float ehpc, float kde_lane, float elhm_sum,
                                               int tp, int fp, int fn, const float cen[3],
                                               float out[GD_E_N], float *cmcc)
{
  const int pos = P.pos;
  float sums[GD_F_NTERM];
  sums[GD_F_VDW] = gd_wave_sum(tot.vdw);
  sums[GD_F_ELE] = gd_wave_sum(tot.ele) * P.sc.inv_el1;   /* the pair loop sums el1 g */
  sums[GD_F_PMF] = gd_wave_sum(tot.pmf);
  sums[GD_F_HPC] = ehpc;
  sums[GD_F_HDB] = gd_wave_sum(tot.hdb);
  sums[GD_F_DST] = gd_edst(P.pocket_center, cen);
  sums[GD_F_PSP] = gd_wave_sum(tot.psp);
  sums[GD_F_KDE] = gd_wave_sum(kde_lane) / P.kde3;
  sums[GD_F_LHM] = (pos > 0) ? gd_log(elhm_sum / (float) pos) : 0.0f;
  gd_finalize(sums, (float) P.lna, P.a_para, P.b_para, P.w, P.term_order, P.combine, out);
  *cmcc = 0.0f;
  if (P.mcc_ref) {
    const int tn = P.lna * P.pnp - tp - fp - fn;   /* padding points are never contacts */
    *cmcc = gd_mcc((float) tp, (float) fn, (float) fp, (float) tn);
  }
}

/* One wavefront evaluates every block in order.  On return out[] (slot
 * order) and *cmcc (MCC against the reference contacts, CalcMcc_d
 * calcmcc_d.cu:148-213, or 0) are identical in every lane. */
__device__ __forceinline__ void gd_energy_wave(
    const gd_pack &P, const char *smem, int prt, float ax0, float ay0, float az0, float ax1,
    float ay1, float az1, const float cen[3], float out[GD_E_N], float *cmcc)
{
  gd_blk tot;
  tot.vdw = 0.0f; tot.pmf = 0.0f; tot.psp = 0.0f; tot.hdb = 0.0f; tot.ele = 0.0f;
  float ehpc = 0.0f;
  int tp = 0, fp = 0, fn = 0;
  const int lna = P.lna;
  const int bs = gd_block_size(lna);
  for (int l0 = 0; l0 < lna; l0 += bs) {
    gd_blk blk;
    float eb;
    gd_atoms_block<false>(gd_hot_of(P, prt), smem, ax0, ay0, az0, ax1, ay1, az1, l0,
                          min(l0 + bs, lna), blk, &eb, tp, fp, fn);
    tot.vdw += blk.vdw;
    tot.pmf += blk.pmf;
    tot.psp += blk.psp;
    tot.hdb += blk.hdb;
    tot.ele += blk.ele;
    ehpc += eb;
  }
  const int n_rounds = gd_hot_of(P, prt).n_rounds;
  const int kbs = gd_block_size(n_rounds > 0 ? n_rounds : 1);
  float kde_lane = 0.0f;
  for (int r0 = 0; r0 < n_rounds; r0 += kbs)
    kde_lane += gd_kde_rounds(gd_hot_of(P, prt), smem, ax0, ay0, az0, ax1, ay1, az1, r0,
                              min(r0 + kbs, n_rounds));
  float elhm = 0.0f;
  for (int m = 0; m < P.pos; ++m)
    elhm += gd_lhm_one(gd_hot_of(P, prt), ax0, ay0, az0, ax1, ay1, az1, m);
  gd_energy_tail(P, tot, ehpc, kde_lane, elhm, tp, fp, fn, cen, out, cmcc);
}

/* Move the conformer held by this lane (move_d.cu:86-132). */
__device__ __forceinline__ void gd_place(const gd_pack &P, const float m[6],
                                         float bx0, float by0, float bz0,
                                         float bx1, float by1, float bz1,
                                         float *ax0, float *ay0, float *az0,
                                         float *ax1, float *ay1, float *az1,
                                         float cen[3])
{
  float rot[9];
  gd_rotation(m, rot);
  const float c[3] = {P.center[0], P.center[1], P.center[2]};
  gd_transform(rot, m, c, bx0, by0, bz0, ax0, ay0, az0);
  gd_transform(rot, m, c, bx1, by1, bz1, ax1, ay1, az1);
  cen[0] = c[0] + m[0];
  cen[1] = c[1] + m[1];
  cen[2] = c[2] + m[2];
}

/* Centroid-relative conformer coordinates, two atoms per lane. */
__device__ __forceinline__ void gd_load_conformer_at(const float4 *cx, int lna, float *bx0,
                                                     float *by0, float *bz0, float *bx1,
                                                     float *by1, float *bz1)
{
  const int lane = threadIdx.x & (GD_WAVE - 1);
  *bx0 = *by0 = *bz0 = *bx1 = *by1 = *bz1 = 0.0f;
  if (lane < lna) {
    const float4 v = cx[lane];
    *bx0 = v.x; *by0 = v.y; *bz0 = v.z;
  }
  if (lane + GD_WAVE < lna) {
    const float4 v = cx[lane + GD_WAVE];
    *bx1 = v.x; *by1 = v.y; *bz1 = v.z;
  }
}

__device__ __forceinline__ void gd_load_conformer(const gd_pack &P, int conf, float *bx0,
                                                  float *by0, float *bz0, float *bx1,
                                                  float *by1, float *bz1)
{
  gd_load_conformer_at(P.lig_xyz + (size_t) conf * P.lna, P.lna, bx0, by0, bz0, bx1, by1, bz1);
}

/* Steps of a launch of n_cyc cycles for a complex: spe a cycle while steps
 * are left (steps_run is a whole number of cycles). */
__device__ __forceinline__ int gd_launch_steps(const gd_pack &P, int s0, int n_cyc)
{
  const int left = P.steps_run - s0, want = P.spe * n_cyc;
  return left < want ? left : want;
}

/* ------------------------------------------------------------------------ */
/* One replica, one wavefront.                                               */
/* ------------------------------------------------------------------------ */
__device__ __forceinline__ void gd_replica_init(const gd_pack &P, const char *smem, int r,
                                                int prt)
{
  const int lane = threadIdx.x & (GD_WAVE - 1);
  const gd_state S = P.S;
  float bx0, by0, bz0, bx1, by1, bz1;
  gd_load_conformer(P, P.rep_lig[r], &bx0, &by0, &bz0, &bx1, &by1, &bz1);
  float m[6];
#pragma unroll
  for (int k = 0; k < 6; ++k)
    m[k] = S.mv[r * 8 + k];
  if (P.away) {
#pragma unroll
    for (int k = 0; k < 6; ++k)
      m[k] = P.move_scale[k] * 44.5f + m[k];
  }
  float ax0, ay0, az0, ax1, ay1, az1, cen[3], e[GD_E_N], cm;
  gd_place(P, m, bx0, by0, bz0, bx1, by1, bz1, &ax0, &ay0, &az0, &ax1, &ay1, &az1, cen);
  gd_energy_wave(P, smem, prt, ax0, ay0, az0, ax1, ay1, az1, cen, e, &cm);
  if (lane == 0) {
    S.cmcc[r] = cm;
    S.cmcc_best[r] = cm;
#pragma unroll
    for (int k = 0; k < 6; ++k) {
      S.mv[r * 8 + k] = m[k];
      S.mv_best[r * 8 + k] = m[k];
    }
#pragma unroll
    for (int i = 0; i < GD_E_N; ++i) {
      S.e[r * 10 + i] = e[i];
      S.e_best[r * 10 + i] = e[i];
    }
    S.step_best[r] = -1;
  }
}

/* ------------------------------------------------------------------------ */
/* Replicas split over the wavefronts of a workgroup.  Each replica has an   */
/* area in LDS (GD_SA_ offsets).  The wavefronts take items -- atom blocks,  */
/* blocks of KDE rounds, position restraints, of any of the workgroup's      */
/* replicas -- from one counter until none is left, so one that finishes     */
/* early takes more.  Each item writes its own slots and the sums read them  */
/* in block order -- the order one wavefront keeps alone -- so the energies  */
/* have the same bits whichever wavefront evaluated which item.              */
/* ------------------------------------------------------------------------ */
typedef __attribute__((address_space(3))) int gd_lds_i32;

/* What the steps need besides, read once per cycle as well: lane k < 10 holds
 * a_para[k] and b_para[k]. */
struct gd_split_consts {
  gd_hot H;
  int bs, nb;               /* atom block size and count */
  int kbs, nbk;             /* KDE rounds per block, blocks */
  int pos;
  int share, share_inv;     /* replicas of the workgroup; 65536 / share, rounded up */
  int term_order, combine, fixed_draws, reverse, mcc_pairs;
  float a_l, b_l;
  float lna_f, inv_el1, kde3;
  float center[3], pocket_center[3];
};

__device__ __forceinline__ gd_split_consts gd_split_consts_of(const gd_pack &P, int prt,
                                                              int share)
{
  const int lane = threadIdx.x & (GD_WAVE - 1);
  gd_split_consts z;
  z.H = gd_hot_of(P, prt);
  z.bs = gd_block_size(z.H.lna);
  z.nb = (z.H.lna + z.bs - 1) / z.bs;
  z.kbs = gd_block_size(z.H.n_rounds > 0 ? z.H.n_rounds : 1);
  z.nbk = (z.H.n_rounds + z.kbs - 1) / z.kbs;
  z.pos = P.pos;
  z.share = share;
  z.share_inv = (65535 + share) / share;
  z.term_order = P.term_order;
  z.combine = P.combine;
  z.fixed_draws = P.fixed_draws;
  z.reverse = P.reverse;
  z.mcc_pairs = z.H.lna * P.pnp;   /* padding points are never contacts */
  z.a_l = lane < 10 ? P.a_para[lane] : 0.0f;
  z.b_l = lane < 10 ? P.b_para[lane] : 0.0f;
  z.lna_f = (float) z.H.lna;
  z.inv_el1 = P.sc.inv_el1;
  z.kde3 = P.kde3;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    z.center[k] = P.center[k];
    z.pocket_center[k] = P.pocket_center[k];
  }
  return z;
}

/* Takes items until none is left: `item` first, then by the counter.  Lane j
 * of sel_l names the pose buffer of replica j.  Item i: block i / share of
 * replica i % share, so that every replica's atom blocks (the longest items)
 * come first.  place() runs once: before the first item is worked on, or with
 * place_late before the second, at the latest when no item is left. */
template <class F>
__device__ __forceinline__ void gd_split_items(const char *smem, gd_lds_f32 *areas,
                                               gd_lds_i32 *ctr, const gd_split_consts &Z,
                                               int sel_l, int item, bool place_late,
                                               F place)
{
  const int lane = threadIdx.x & (GD_WAVE - 1);
  const int lna = Z.H.lna;
  const int n_items = (Z.nb + Z.nbk + Z.pos) * Z.share;
  int j_held = -1;
  float xyz[6];
#pragma unroll
  for (int k = 0; k < 6; ++k)
    xyz[k] = 0.0f;
  bool placed = false;
  for (bool first = true;; first = false) {
    if (item < 0) {
      /* every lane adds 1 (one LDS atomic of 64 for the wavefront) and the
       * first lane's old value / 64 is the item: no lane-divergent branch
       * feeds the loop */
      const int got = __hip_atomic_fetch_add(ctr, 1, __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_WORKGROUP);
      item = __builtin_amdgcn_readfirstlane(got) >> 6;
    }
    if (!placed && (!first || !place_late || item >= n_items)) {
      place();
      placed = true;
    }
    if (item >= n_items)
      break;
    /* exact: item < 4 (16 + 16 + 64), share <= 4 */
    const int i = (item * Z.share_inv) >> 16;
    const int j = item - i * Z.share;
    gd_lds_f32 *A = areas + j * GD_SA_FLOATS;
    if (j != j_held) {
      const gd_lds_f32 *pb =
          A + GD_SA_POSE + __builtin_amdgcn_readlane(sel_l, j) * GD_PB_FLOATS + lane;
#pragma unroll
      for (int k = 0; k < 6; ++k)
        xyz[k] = pb[k * GD_WAVE];
      j_held = j;
    }
    if (i < Z.nb) {
      gd_blk blk;
      float eb;
      int tp = 0, fp = 0, fn = 0;
      gd_atoms_block<true>(Z.H, smem, xyz[0], xyz[1], xyz[2], xyz[3], xyz[4], xyz[5],
                           i * Z.bs, min(i * Z.bs + Z.bs, lna), blk, &eb, tp, fp, fn);
      gd_lds_f32 *pb = A + GD_SA_PART + i * 5 * GD_WAVE + lane;
      pb[0 * GD_WAVE] = blk.vdw;
      pb[1 * GD_WAVE] = blk.pmf;
      pb[2 * GD_WAVE] = blk.psp;
      pb[3 * GD_WAVE] = blk.hdb;
      pb[4 * GD_WAVE] = blk.ele;
      if (lane == 0) {
        A[GD_SA_EHPC + i] = eb;
        A[GD_SA_MCC + 3 * i + 0] = __int_as_float(tp);
        A[GD_SA_MCC + 3 * i + 1] = __int_as_float(fp);
        A[GD_SA_MCC + 3 * i + 2] = __int_as_float(fn);
      }
    } else if (i < Z.nb + Z.nbk) {
      const int kb = i - Z.nb;
      A[GD_SA_KPART + kb * GD_WAVE + lane] =
          gd_kde_rounds(Z.H, smem, xyz[0], xyz[1], xyz[2], xyz[3], xyz[4], xyz[5], kb * Z.kbs,
                        min(kb * Z.kbs + Z.kbs, Z.H.n_rounds));
    } else {
      const int m = i - Z.nb - Z.nbk;
      const float v = gd_lhm_one(Z.H, xyz[0], xyz[1], xyz[2], xyz[3], xyz[4], xyz[5], m);
      if (lane == 0)
        A[GD_SA_LHM + m] = v;
    }
    item = -1;
  }
}

/* src[0] + src[stride] + ... over the GD_MAX_BLOCKS slots, in order.  Slots
 * past the last block hold +0, which leaves the sum's bits unchanged (a sum
 * that starts at +0 is never -0), so no test stands between the adds. */
__device__ __forceinline__ float gd_ordered_sum(const gd_lds_f32 *src, int stride)
{
  float v[GD_MAX_BLOCKS];
#pragma unroll
  for (int b = 0; b < GD_MAX_BLOCKS; ++b)
    v[b] = src[b * stride];
  float t = 0.0f;
#pragma unroll
  for (int b = 0; b < GD_MAX_BLOCKS; ++b)
    t += v[b];
  return t;
}

/* file-order term <-> slot, 4 bits each: slot i holds file term s2f[i] */
#define GD_S2F 0x587346210ull
#define GD_F2S 0x763845210ull

/* Normalised value of file-order term f (raw: the term as gd_finalize takes
 * it) into the terms of one step, by the index of the parameter that applies
 * to it: gd_finalize's operations. */
__device__ __forceinline__ void gd_term_put(const gd_split_consts &Z,
                                            gd_lds_f32 *term, int f, float raw)
{
  const int lane = threadIdx.x & (GD_WAVE - 1);
  const int k = Z.term_order ? (int) ((GD_F2S >> (4 * f)) & 0xfu) : f;
  const float v = gd_fma(gd_bcast(Z.a_l, k), raw, gd_bcast(Z.b_l, k));
  if (lane == 0)
    term[k] = v;
}

/* After the items: the partials added in block order and reduced, each term
 * normalised, spread over the wavefronts -- job q of a replica: 0-4 the vdw,
 * pmf, psp, hdb, ele lane totals over the atom blocks and their wave sums, 5
 * the KDE lane total and its wave sum, 6 the restraint sum and the MCC
 * counts, 7 the position-restraint sum.  The divisions and the logarithm are done here, by eight
 * wavefronts at once, not by the one that decides. */
__device__ __forceinline__ void gd_split_sums(gd_lds_f32 *areas, int role, int split,
                                              const gd_split_consts &Z)
{
  const int lane = threadIdx.x & (GD_WAVE - 1);
  const int nb = Z.nb;
  const float lna_f = Z.lna_f;
  for (int job = role; job < 8 * Z.share; job += split) {
    const int q = job & 7;
    gd_lds_f32 *A = areas + (job >> 3) * GD_SA_FLOATS;
    gd_lds_f32 *term = A + GD_SA_TERM;
    if (q < 6) {
      float x = gd_wave_sum(
          q < 5 ? gd_ordered_sum(A + GD_SA_PART + q * GD_WAVE + lane, 5 * GD_WAVE)
                : gd_ordered_sum(A + GD_SA_KPART + lane, GD_WAVE));
      /* file-order term of each job */
      const int f = (int) ((0x714620u >> (4 * q)) & 0xfu);
      if (f == GD_F_ELE)
        x = x * Z.inv_el1;   /* the pair loop sums el1 g */
      if (f == GD_F_KDE)
        x = x / Z.kde3;
      float y = x / lna_f;
      if (f == GD_F_HDB) {
        GD_KEEP_BRANCH();
        y = y / 0x1.40d932p+1f * -1.0f;   /* sqrt(2 pi) */
      }
      gd_term_put(Z, term, f, y);
    } else if (q == 6) {
      gd_term_put(Z, term, GD_F_HPC, gd_ordered_sum(A + GD_SA_EHPC, 1) / lna_f);
      /* the MCC counts are integers: any order */
      if (Z.H.mref) {
        const bool in_b = lane < nb;
        int tp = in_b ? __float_as_int(A[GD_SA_MCC + 3 * lane + 0]) : 0;
        int fp = in_b ? __float_as_int(A[GD_SA_MCC + 3 * lane + 1]) : 0;
        int fn = in_b ? __float_as_int(A[GD_SA_MCC + 3 * lane + 2]) : 0;
#pragma unroll
        for (int off = 1; off < GD_MAX_BLOCKS; off <<= 1) {
          tp += __shfl_xor(tp, off, GD_WAVE);
          fp += __shfl_xor(fp, off, GD_WAVE);
          fn += __shfl_xor(fn, off, GD_WAVE);
        }
        if (lane == 0) {
          A[GD_SA_CNT + 0] = __int_as_float(tp);
          A[GD_SA_CNT + 1] = __int_as_float(fp);
          A[GD_SA_CNT + 2] = __int_as_float(fn);
        }
      }
    } else {
      /* position restraints in order; the slots past the last hold +0 */
      const int pos = Z.pos;
      float elhm = 0.0f;
      if (pos > 0) {
        for (int m0 = 0; m0 < pos; m0 += 8) {
          float v[8];
#pragma unroll
          for (int m = 0; m < 8; ++m)
            v[m] = A[GD_SA_LHM + m0 + m];
#pragma unroll
          for (int m = 0; m < 8; ++m)
            elhm += v[m];
        }
        elhm = gd_log(elhm / (float) pos);
      }
      gd_term_put(Z, term, GD_F_LHM, elhm);
    }
  }
}

/* The Bayesian total of the terms of one step (uniform). */
__device__ __forceinline__ float gd_split_bayes(const gd_split_consts &Z, const gd_lds_f32 *term)
{
  float nf[GD_F_NTERM];
#pragma unroll
  for (int f = 0; f < GD_F_NTERM; ++f)
    nf[f] = term[Z.term_order ? (int) ((GD_F2S >> (4 * f)) & 0xfu) : f];
  return gd_bayes_total(nf);
}

/* The weighted sum of the terms of one step, in parameter order. */
__device__ __forceinline__ float gd_split_total(const gd_lds_f32 *term, const float *w)
{
  float total = 0.0f;
#pragma unroll
  for (int k = 0; k < GD_F_NTERM; ++k)
    total = gd_fma(w[k], term[k], total);
  return total;
}

/* Lane i < GD_E_N: the energy of slot i. */
__device__ __forceinline__ float gd_split_energy(const gd_split_consts &Z, const gd_lds_f32 *term,
                                                 float total)
{
  const int lane = threadIdx.x & (GD_WAVE - 1);
  const int i = lane < GD_F_NTERM ? lane : 0;
  const int k = Z.term_order ? i : (int) ((GD_S2F >> (4 * i)) & 0xfu);
  const float v = term[k];
  return lane == GD_E_TOTAL ? total : v;
}

/* gd_exp without a branch: the general form at the clamped argument, then the
 * special cases selected.  The same bits; three branches on a vector compare
 * cost the deciding wavefront, which all others wait for, more than they save. */
__device__ __forceinline__ float gd_exp_select(float x)
{
  const float xc = __builtin_fminf(__builtin_fmaxf(x, -86.0f), 88.0f);
  const float n = gd_rint(xc * 0x1.715476p+0f);
  float r = gd_fma(-n, 0x1.62e430p-1f, xc);
  r = gd_fma(-n, -0x1.05c610p-29f, r);
  float p = 0x1.a01a02p-13f;
  p = gd_fma(p, r, 0x1.6c16c2p-10f);
  p = gd_fma(p, r, 0x1.111112p-7f);
  p = gd_fma(p, r, 0x1.555556p-5f);
  p = gd_fma(p, r, 0x1.555556p-3f);
  p = gd_fma(p, r, 0.5f);
  p = gd_fma(p, r, 1.0f);
  p = gd_fma(p, r, 1.0f);
  float v = p * gd_as_float((uint32_t) ((int) n + 127) << 23);
  v = x > 88.0f ? gd_as_float(GD_INF_BITS) : v;
  v = x < -86.0f ? 0.0f : v;
  return x != x ? x : v;
}

/* gd_metropolis with it. */
__device__ __forceinline__ int gd_split_decide(float e_new, float e_old, float mb, float u,
                                               float u2, int fixed_draws, int reverse)
{
  const float d = e_new - e_old;
  const float p = gd_exp_select((reverse ? -d : d) * mb);
  return fixed_draws || (reverse ? u2 : u) < p;
}

/* MCC from the counts of the step's sums (uniform; 0 without MCC). */
__device__ __forceinline__ float gd_split_mcc(const gd_split_consts &Z, const gd_lds_f32 *A)
{
  if (!Z.H.mref)
    return 0.0f;
  const int tp = __float_as_int(A[GD_SA_CNT + 0]), fp = __float_as_int(A[GD_SA_CNT + 1]);
  const int fn = __float_as_int(A[GD_SA_CNT + 2]);
  const int tn = Z.mcc_pairs - tp - fp - fn;
  return gd_mcc((float) tp, (float) fn, (float) fp, (float) tn);
}

/* The draws of step s of replica r (move_d.cu:73-84, accept_d.cu:20-27): the
 * movematrix displacement d[6] and the two acceptance draws (the second only
 * for the reversed test). */
__device__ __forceinline__ void gd_draws(const gd_pack &P, int r, int s, uint32_t seed,
                                         uint32_t cid, float d[6], float u_acc[2])
{
  const gd_u32x4 ra = gd_philox4x32_10((uint32_t) r, (uint32_t) s, GD_CTR_MOVE_A, 0u, seed, cid);
  const gd_u32x4 rb = gd_philox4x32_10((uint32_t) r, (uint32_t) s, GD_CTR_MOVE_B, 0u, seed, cid);
  const int fx = P.fixed_draws;
  d[0] = P.move_scale[0] * gd_perturbation(fx, ra.v[0]);
  d[1] = P.move_scale[1] * gd_perturbation(fx, ra.v[1]);
  d[2] = P.move_scale[2] * gd_perturbation(fx, ra.v[2]);
  d[3] = P.move_scale[3] * gd_perturbation(fx, ra.v[3]);
  d[4] = P.move_scale[4] * gd_perturbation(fx, rb.v[0]);
  d[5] = P.move_scale[5] * gd_perturbation(fx, rb.v[1]);
  u_acc[0] = gd_u01(rb.v[2]);
  u_acc[1] = gd_u01(rb.v[3]);
}

/* RecordLigand_d (util_d.cu:72-94): the state before step s, one word per
 * lane. */
__device__ __forceinline__ void gd_record(const gd_pack &P, const gd_lds_f32 *ws, int r,
                                          int itmp, int s)
{
  const int lane = threadIdx.x & (GD_WAVE - 1);
  uint32_t *rec = P.rec + ((size_t) r * P.rec_per_window +
                           (s % P.rec_window) / P.rec_stride) * GD_REC_WORDS;
  float fv = 0.0f;
  if (lane >= 4 && lane < 14)
    fv = ws[GD_WS_EOLD + lane - 4];
  else if (lane == 14)
    fv = ws[GD_WS_CMCC];
  else if (lane >= 15 && lane < 21)
    fv = ws[GD_WS_MOLD + lane - 15];
  uint32_t v = __float_as_uint(fv);
  if (lane == 0) v = (uint32_t) r;
  if (lane == 1) v = (uint32_t) P.rep_prt[r];
  if (lane == 2) v = (uint32_t) itmp;
  if (lane == 3) v = (uint32_t) P.rep_lig[r];
  if (lane == 21) v = (uint32_t) s;
  if (lane < GD_REC_WORDS)
    rec[lane] = v;
}

/* Metropolis (accept_d.cu:12-52) on wavefront-uniform energies: the state
 * in the slot, the best pose in HBM; returns 1 if the move was taken. */
__device__ __forceinline__ int gd_accept(const gd_pack &P, gd_lds_f32 *ws, int r, int s,
                                         const float u_acc[2], float mb,
                                         const float e_new[GD_E_N], float cm_new,
                                         float *e_old_total, float *best_total)
{
  const int lane = threadIdx.x & (GD_WAVE - 1);
  const gd_state S = P.S;
  if (!gd_metropolis(e_new[GD_E_TOTAL], *e_old_total, mb, u_acc[0], u_acc[1], P.fixed_draws,
                     P.reverse))
    return 0;
  *e_old_total = e_new[GD_E_TOTAL];
  if (lane == 0) {
#pragma unroll
    for (int i = 0; i < GD_E_N; ++i)
      ws[GD_WS_EOLD + i] = e_new[i];
#pragma unroll
    for (int k = 0; k < 6; ++k)
      ws[GD_WS_MOLD + k] = ws[GD_WS_MNEW + k];
    ws[GD_WS_CMCC] = cm_new;
  }
  if (e_new[GD_E_TOTAL] < *best_total) {
    *best_total = e_new[GD_E_TOTAL];
    if (lane == 0) {
#pragma unroll
      for (int k = 0; k < 6; ++k)
        S.mv_best[r * 8 + k] = ws[GD_WS_MNEW + k];
#pragma unroll
      for (int i = 0; i < GD_E_N; ++i)
        S.e_best[r * 10 + i] = e_new[i];
      S.cmcc_best[r] = cm_new;
      S.step_best[r] = s;
    }
  }
  return 1;
}

/* The slot from the replica's state in HBM (wavefront 0 of the replica). */
__device__ __forceinline__ void gd_slot_load(const gd_pack &P, gd_lds_f32 *ws, int r)
{
  const int lane = threadIdx.x & (GD_WAVE - 1);
  const gd_state S = P.S;
  if (lane < 6)
    ws[GD_WS_MOLD + lane] = S.mv[r * 8 + lane];
  if (lane < GD_E_N)
    ws[GD_WS_EOLD + lane] = S.e[r * 10 + lane];
  if (lane == 0)
    ws[GD_WS_CMCC] = S.cmcc[r];
}

/* The replica's state in HBM from the slot, and the cycle's accept count. */
__device__ __forceinline__ void gd_slot_store(const gd_pack &P, const gd_lds_f32 *ws, int r,
                                              int acs)
{
  const int lane = threadIdx.x & (GD_WAVE - 1);
  const gd_state S = P.S;
  if (lane < 6)
    S.mv[r * 8 + lane] = ws[GD_WS_MOLD + lane];
  if (lane < GD_E_N)
    S.e[r * 10 + lane] = ws[GD_WS_EOLD + lane];
  if (lane == 0) {
    S.acs_mc[r] += acs;
    S.cmcc[r] = ws[GD_WS_CMCC];
  }
}

/* n_steps MC steps from step s0 of replica r on one wavefront.  The
 * movematrices and energies live in the replica's LDS slot
 * ws[GD_WSLOT_FLOATS]; only totals stay in registers. */
__device__ __forceinline__ void gd_replica_cycle(const gd_pack &P, const char *smem,
                                                 gd_lds_f32 *ws, int r, int prt, int s0,
                                                 int n_steps)
{
  const int lane = threadIdx.x & (GD_WAVE - 1);
  const gd_state S = P.S;
  const int lconf = gd_uload(P.rep_lig + r);
  gd_slot_load(P, ws, r);
  __builtin_amdgcn_wave_barrier();
  float e_old_total = S.e[r * 10 + GD_E_TOTAL];
  float best_total = S.e_best[r * 10 + GD_E_TOTAL];
  const int itmp = S.idx_tmp[r];
  const float mb = P.minus_beta[itmp];
  const uint32_t seed = P.seed, cid = P.cid;
  int acs = 0;

  for (int s = s0; s < s0 + n_steps; ++s) {
    if (P.rec != nullptr && s % P.rec_stride == 0)
      gd_record(P, ws, r, itmp, s);
    float d[6], u_acc[2];
    gd_draws(P, r, s, seed, cid, d, u_acc);
    float m_new[6];
#pragma unroll
    for (int k = 0; k < 6; ++k)
      m_new[k] = d[k] + ws[GD_WS_MOLD + k];

    /* the conformer is re-read every step (an L1 hit) rather than held in
     * registers across the energy evaluation */
    float bx0, by0, bz0, bx1, by1, bz1;
    gd_load_conformer(P, lconf, &bx0, &by0, &bz0, &bx1, &by1, &bz1);
    float ax0, ay0, az0, ax1, ay1, az1, cen[3], e_new[GD_E_N], cm_new;
    gd_place(P, m_new, bx0, by0, bz0, bx1, by1, bz1, &ax0, &ay0, &az0, &ax1, &ay1,
             &az1, cen);
    if (lane == 0) {
#pragma unroll
      for (int k = 0; k < 6; ++k)
        ws[GD_WS_MNEW + k] = m_new[k];
    }
    gd_energy_wave(P, smem, prt, ax0, ay0, az0, ax1, ay1, az1, cen, e_new, &cm_new);
    acs += gd_accept(P, ws, r, s, u_acc, mb, e_new, cm_new, &e_old_total, &best_total);
    __builtin_amdgcn_wave_barrier();
  }
  gd_slot_store(P, ws, r, acs);
}

/* Pose buffer pb from the movematrix that lanes 0-5 hold (m_l) and ligand
 * conformer conf: one sine-cosine sequence serves the three angles. */
__device__ __forceinline__ void gd_pose_put(const gd_split_consts &Z, gd_lds_f32 *pb,
                                            float m_l, const float4 *conf)
{
  const int lane = threadIdx.x & (GD_WAVE - 1);
  float bx0, by0, bz0, bx1, by1, bz1;
  gd_load_conformer_at(conf, Z.H.lna, &bx0, &by0, &bz0, &bx1, &by1, &bz1);
  float s_l, c_l;
  gd_sincos(m_l, &s_l, &c_l);
  float rot[9];
  gd_rotation_sc(gd_bcast(s_l, 3), gd_bcast(c_l, 3), gd_bcast(s_l, 4), gd_bcast(c_l, 4),
                 gd_bcast(s_l, 5), gd_bcast(c_l, 5), rot);
  const float m[6] = {gd_bcast(m_l, 0), gd_bcast(m_l, 1), gd_bcast(m_l, 2), 0.0f, 0.0f, 0.0f};
  const float c[3] = {Z.center[0], Z.center[1], Z.center[2]};
  float ax0, ay0, az0, ax1, ay1, az1;
  gd_transform(rot, m, c, bx0, by0, bz0, &ax0, &ay0, &az0);
  gd_transform(rot, m, c, bx1, by1, bz1, &ax1, &ay1, &az1);
  pb[0 * GD_WAVE + lane] = ax0;
  pb[1 * GD_WAVE + lane] = ay0;
  pb[2 * GD_WAVE + lane] = az0;
  pb[3 * GD_WAVE + lane] = ax1;
  pb[4 * GD_WAVE + lane] = ay1;
  pb[5 * GD_WAVE + lane] = az1;
  if (lane < 6)
    pb[GD_PB_M + lane] = m_l;
  if (lane == 0) {
#pragma unroll
    for (int k = 0; k < 3; ++k)
      pb[GD_PB_CEN + k] = c[k] + m[k];
  }
}

/* The distance term of the pose in buffer pb. */
__device__ __forceinline__ float gd_pose_edst(const gd_split_consts &Z, const gd_lds_f32 *pb)
{
  const float cen[3] = {pb[GD_PB_CEN + 0], pb[GD_PB_CEN + 1], pb[GD_PB_CEN + 2]};
  return gd_edst(Z.pocket_center, cen);
}

/* The draws of n <= GD_SPLIT_DRAWS steps from step s0 of replica r (gd_draws),
 * one Philox sequence for all: lane 2 i + h takes call h of step s0 + i. */
__device__ __forceinline__ void gd_split_draws(const gd_pack &P, gd_lds_f32 *out, int r, int s0)
{
  const int lane = threadIdx.x & (GD_WAVE - 1);
  const int h = lane & 1;
  const gd_u32x4 u = gd_philox4x32_10((uint32_t) r, (uint32_t) (s0 + (lane >> 1)),
                                      h ? GD_CTR_MOVE_B : GD_CTR_MOVE_A, 0u, P.seed, P.cid);
  const int fx = P.fixed_draws;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const float sc = h ? P.move_scale[k < 2 ? 4 + k : 0] : P.move_scale[k];
    const float d = sc * gd_perturbation(fx, u.v[k]);
    out[lane * 4 + k] = h && k >= 2 ? gd_u01(u.v[k]) : d;
  }
}
static_assert(GD_SPLIT_DRAWS * 2 == GD_WAVE, "one lane per draw call");

/* n_steps MC steps from step s0 of the Z.share replicas r0, r0 + 1, .. on the
 * SPLIT wavefronts of the workgroup, `role` = this wavefront's index.
 * Two wavefronts lead replica j, and the first of them keeps its state.  Per
 * step: the wavefronts take items; barrier; the sums; barrier; the keepers take
 * the decisions; barrier.  The move of step s + 1 never waits for the decision:
 * among their items the two leaders place both poses that step may start from,
 * in the replica's two other buffers (the move from the
 * current pose if this one is rejected, from the proposed one if it is
 * accepted: the same draws and arithmetic as placing it after the decision),
 * and the decision only selects the buffer; the state, the best pose and the
 * records follow behind the barrier, while the others already take items. */
template <int SPLIT>
__device__ __forceinline__ void gd_replica_cycle_split(const gd_pack &P, const char *smem,
                                                       gd_lds_f32 *areas, gd_lds_i32 *ctr,
                                                       int role, int r0, int s0, int n_steps,
                                                       const gd_split_consts &Z)
{
  const int lane = threadIdx.x & (GD_WAVE - 1);
  const gd_state S = P.S;
  const int share = Z.share;
  /* Each wavefront begins with the item of its own index, unasked.  Where the
   * others cover the atom blocks, the leaders place their poses first and are
   * the last wavefronts, since a SIMD issues its oldest first and the blocks
   * last longest; else they are the oldest, take a block like the others and
   * place the poses behind it.  Workgroups of 4 or 8 always place first: with
   * one or two wavefronts a SIMD the rounds are many and the placing fits
   * beside them (64 replicas of 24 x 300, eight to a replica, behind a block 94
   * us a cycle, first 88). */
  const bool place_late = SPLIT == 16 && Z.nb * share > SPLIT - 2 * share;
  const int q = place_late ? role : SPLIT - 1 - role;
  const int j_lead = q >> 1;
  const bool lead = j_lead < share;
  const bool keeper = lead && (q & 1) == 0;
  const int n_first = place_late ? SPLIT : SPLIT - 2 * share;
  gd_lds_f32 *A = areas + (lead ? j_lead : 0) * GD_SA_FLOATS;
  gd_lds_f32 *ws = A;
  gd_lds_f32 *pose = A + GD_SA_POSE;
  const int r = r0 + (lead ? j_lead : 0);
  const float4 *conf = P.lig_xyz + (size_t) gd_uload(P.rep_lig + r) * Z.H.lna;
  float e_old = 0.0f, best_total = 0.0f, mb = 0.0f;
  int acs = 0, itmp = 0;
  float w[GD_F_NTERM];
#pragma unroll
  for (int k = 0; k < GD_F_NTERM; ++k)
    w[k] = P.w[k];
  if (keeper) {
    gd_slot_load(P, ws, r);
    e_old = S.e[r * 10 + GD_E_TOTAL];
    best_total = S.e_best[r * 10 + GD_E_TOTAL];
    itmp = S.idx_tmp[r];
    mb = P.minus_beta[itmp];
  }
  /* slots that no item writes count as +0 in the sums */
  for (int j = 0; j < share; ++j)
    for (int i = GD_SA_PART + (int) threadIdx.x; i < GD_SA_POSE; i += GD_WAVE * SPLIT)
      areas[j * GD_SA_FLOATS + i] = 0.0f;

  for (int c0 = s0; c0 < s0 + n_steps; c0 += GD_SPLIT_DRAWS) {
    const int c1 = min(c0 + GD_SPLIT_DRAWS, s0 + n_steps);
    /* the draws of these steps and the pose of the first, in buffer 0 */
    if (keeper) {
      gd_split_draws(P, A + GD_SA_DRAW, r, c0);
      __builtin_amdgcn_wave_barrier();
      const int k = lane < 6 ? lane : 0;
      gd_pose_put(Z, pose, A[GD_SA_DRAW + k] + ws[GD_WS_MOLD + k], conf);
    }
    if (role == 0 && lane == 0) {
      ctr[0] = n_first * GD_WAVE;
      ctr[1] = n_first * GD_WAVE;
    }
    int sel_l = 0;   /* lane j: the pose buffer of replica j */
    __syncthreads();

    for (int s = c0; s < c1; ++s) {
      const int par = (s - c0) & 1;
      const int k = lane < 6 ? lane : 0;
      const int sel = __builtin_amdgcn_readlane(sel_l, lead ? j_lead : 0);
      const gd_lds_f32 *pc = pose + sel * GD_PB_FLOATS;
      float m_l = 0.0f;   /* keeper: the movematrix being evaluated */
      gd_split_items(smem, areas, ctr + par, Z, sel_l, lead && !place_late ? -1 : role,
                     place_late, [&]() {
                       if (!lead)
                         return;
                       const int ia = sel == 2 ? 0 : sel + 1;
                       const int ib = ia == 2 ? 0 : ia + 1;
                       m_l = pc[GD_PB_M + k];
                       if (keeper) {
                         if (P.rec != nullptr && s % P.rec_stride == 0)
                           gd_record(P, ws, r, itmp, s);
                         gd_term_put(Z, A + GD_SA_TERM, GD_F_DST, gd_pose_edst(Z, pc));
                       }
                       if (s + 1 < c1)
                         gd_pose_put(Z, pose + (keeper ? ia : ib) * GD_PB_FLOATS,
                                     A[GD_SA_DRAW + (s + 1 - c0) * 8 + k] +
                                         (keeper ? ws[GD_WS_MOLD + k] : m_l),
                                     conf);
                     });
      __syncthreads();
      gd_split_sums(areas, role, SPLIT, Z);
      if (role == 0 && lane == 0)
        ctr[par ^ 1] = n_first * GD_WAVE;   /* last used before the barrier above */
      __syncthreads();
      int took = 0;
      float total = 0.0f;
      if (keeper) {
        const gd_lds_f32 *term = A + GD_SA_TERM;
        const gd_lds_f32 *u = A + GD_SA_DRAW + (s - c0) * 8 + 6;
        total = Z.combine ? gd_split_bayes(Z, term) : gd_split_total(term, w);
        took = gd_split_decide(total, e_old, mb, u[0], u[1], Z.fixed_draws, Z.reverse);
        int next = sel + (took ? 2 : 1);
        next = next >= 3 ? next - 3 : next;
        *(gd_lds_i32 *) (A + GD_SA_SEL) = next;
      }
      __syncthreads();
      sel_l = *(const gd_lds_i32 *) (areas + (lane < share ? lane : 0) * GD_SA_FLOATS +
                                     GD_SA_SEL);
      if (took) {   /* (the terms and counts are next written behind two barriers
                       that this wavefront takes part in) */
        ++acs;
        e_old = total;
        const float e_l = gd_split_energy(Z, A + GD_SA_TERM, total);
        const float cm = gd_split_mcc(Z, A);
        if (lane < GD_E_N)
          ws[GD_WS_EOLD + lane] = e_l;
        if (lane < 6)
          ws[GD_WS_MOLD + lane] = m_l;
        if (lane == 0)
          ws[GD_WS_CMCC] = cm;
        if (total < best_total) {
          best_total = total;
          if (lane < 6)
            S.mv_best[r * 8 + lane] = m_l;
          if (lane < GD_E_N)
            S.e_best[r * 10 + lane] = e_l;
          if (lane == 0) {
            S.cmcc_best[r] = cm;
            S.step_best[r] = s;
          }
        }
        __builtin_amdgcn_wave_barrier();
      }
    }
  }
  if (keeper)
    gd_slot_store(P, ws, r, acs);
}

/* ------------------------------------------------------------------------ */
/* Temperature exchange (exchangereplicas_d.cu:28-78), one wavefront per     */
/* chain.  The pairs of one sweep are disjoint in temperature, so each       */
/* pair's decision reads only the two slots it may swap: lane j decides pair */
/* j, with the draws and arithmetic of the serial walk, and writes the two   */
/* slots' new temperature indices and acceptance counts.  Then the step      */
/* counters advance and the work queues are re-armed: by the one workgroup   */
/* of a launch over few chains, else by the last workgroup to finish.        */
/* ------------------------------------------------------------------------ */
#define GD_MAXTMP_DEV 64
#define GD_XWAVES 4        /* wavefronts per workgroup, many-chain form */
#define GD_X1_WAVES 16     /* wavefronts of the one-workgroup form */
#define GD_X1_MAX_CHAINS 32
/* LDS words one exchanging wavefront uses */
#define GD_X_WORDS (2 * GD_MAXTMP_DEV)

__device__ __forceinline__ void gd_advance_all(const gd_pack *__restrict__ packs, int n_cx,
                                               int *queue, int n_queue, int n_cyc)
{
  const int n = n_cx > n_queue ? n_cx : n_queue;
  for (int i = threadIdx.x; i < n; i += blockDim.x) {
    if (i < n_queue)
      queue[i] = 0;
    if (i < n_cx) {
      const gd_pack &P = packs[i];
      const int s0 = P.step[0];
      const int k = gd_launch_steps(P, s0, n_cyc);
      if (k > 0) {
        P.step[0] = s0 + k;
        P.step[1] = P.step[1] + k / P.spe;
      }
    }
  }
}

/* Chain g (none if g >= n_chain) by this wavefront, LDS scratch sx of
 * GD_X_WORDS words; every wavefront of the workgroup calls it (it holds two
 * workgroup barriers). */
__device__ __forceinline__ void gd_exchange_wave(const gd_pack *__restrict__ packs,
                                                 const gd_chain *__restrict__ chains,
                                                 int n_chain, int g, int *sx)
{
  int *s_orders = sx;                                 /* temperature -> slot */
  float *s_ener = (float *) (sx + GD_MAXTMP_DEV);     /* slot -> total energy */
  const int lane = threadIdx.x & (GD_WAVE - 1);
  int active = 0, n_tmp = 0, n_lig = 0, base = 0, x = 0, c = 0;
  const gd_pack *P = nullptr;
  if (g < n_chain) {
    const gd_chain ch = chains[g];
    P = &packs[ch.cx];
    n_tmp = P->n_tmp;
    active = P->exchange && n_tmp >= 2 && gd_launch_steps(*P, P->step[0], 1) > 0;
    if (active) {
      x = P->step[1];
      c = ch.c;
      n_lig = P->n_lig;
      const int p = c / n_lig;
      base = n_tmp * n_lig * p + (c - p * n_lig);
      if (lane < n_tmp) {
        const int a = base + n_lig * lane;
        s_ener[lane] = P->S.e[a * 10 + GD_E_TOTAL];
        s_orders[P->S.idx_tmp[a]] = lane;
      }
    }
  }
  __syncthreads();
  if (active) {
    /* cycle x is launch x % lpw of its steps_per_dump window; the mode
     * alternates from 0 in every window (gpusingle.cu:14-18) */
    const int mode = (x % P->lpw) & 1;
    const int maxpair = n_tmp / 2 - ((n_tmp % 2 == 0) && mode == 1 ? 1 : 0);
    const int j = lane;
    if (j < maxpair) {
      const gd_u32x4 u4 = gd_philox4x32_10((uint32_t) c, (uint32_t) x, GD_CTR_EXCHANGE,
                                           (uint32_t) (j >> 2), P->seed, P->cid);
      const int q = j & 3;
      const uint32_t uw = q == 0 ? u4.v[0] : q == 1 ? u4.v[1] : q == 2 ? u4.v[2] : u4.v[3];
      const float u = gd_exchange_draw(P->fixed_draws, uw);
      const int i1 = 2 * j + mode;
      const int i2 = i1 + 1;
      const int o1 = s_orders[i1];
      const int o2 = s_orders[i2];
      const float delta = (P->minus_beta[i1] - P->minus_beta[i2]) * (s_ener[o2] - s_ener[o1]);
      if (gd_exp(delta) > u) {
        const gd_state S = P->S;
        const int a1 = base + n_lig * o1;
        const int a2 = base + n_lig * o2;
        S.idx_tmp[a1] = i2;
        S.idx_tmp[a2] = i1;
        S.acs_x[a1] += 1;
        S.acs_x[a2] += 1;
      }
    }
  }
  __syncthreads();
}

/* Exchange of at most GD_X1_MAX_CHAINS chains by one workgroup, its
 * wavefronts taking chains in turn, then the advance. */
__global__ void __launch_bounds__(GD_WAVE * GD_X1_WAVES)
gd_exchange1_kernel(const gd_pack *__restrict__ packs, const gd_chain *__restrict__ chains,
                    int n_chain, int n_cx, int *queue, int n_queue)
{
  __shared__ int s_x[GD_X1_WAVES * GD_X_WORDS];
  const int nw = (int) (blockDim.x / GD_WAVE);
  const int wv = threadIdx.x / GD_WAVE;
  for (int g0 = 0; g0 < n_chain; g0 += nw)
    gd_exchange_wave(packs, chains, n_chain, g0 + wv, s_x + wv * GD_X_WORDS);
  gd_advance_all(packs, n_cx, queue, n_queue, 1);
}

/* Exchange of chains GD_XWAVES per workgroup; the last workgroup to finish
 * advances.  Its count orders only the other workgroups' reads of the step
 * counters (all consumed before they count) before the advance's writes:
 * nothing else written here is read here, so no fence is taken. */
__global__ void __launch_bounds__(GD_WAVE * GD_XWAVES)
gd_exchange_kernel(const gd_pack *__restrict__ packs, const gd_chain *__restrict__ chains,
                   int n_chain, int n_cx, int *queue, int n_queue, int *done)
{
  __shared__ int s_x[GD_XWAVES * GD_X_WORDS];
  __shared__ int s_last;
  const int wv = threadIdx.x / GD_WAVE;
  gd_exchange_wave(packs, chains, n_chain, blockIdx.x * GD_XWAVES + wv, s_x + wv * GD_X_WORDS);
  if (threadIdx.x == 0)
    s_last = atomicAdd(done, 1) == (int) gridDim.x - 1;
  __syncthreads();
  if (s_last) {
    gd_advance_all(packs, n_cx, queue, n_queue, 1);
    if (threadIdx.x == 0)
      atomicExch(done, 0);
  }
}

/* After MC (no temperature chains to exchange): step[0] += steps of the
 * launch, step[1] += its cycles; threads 0 .. n_queue-1 re-arm the persistent work
 * queues. */
__global__ void __launch_bounds__(256)
gd_advance_kernel(const gd_pack *__restrict__ packs, int n_cx, int *queue, int n_queue,
                  int n_cyc)
{
  if (blockIdx.x == 0)
    gd_advance_all(packs, n_cx, queue, n_queue, n_cyc);
}

/* Issue priority of this wavefront in its SIMD (s_setprio takes an
 * immediate): with launches of several streams sharing the device, the
 * higher one issues first whenever both have an instruction ready.  It
 * changes no result. */
__device__ __forceinline__ void gd_set_prio(int p)
{
  if (p == 1)
    __builtin_amdgcn_s_setprio(1);
  else if (p == 2)
    __builtin_amdgcn_s_setprio(2);
  else if (p >= 3)
    __builtin_amdgcn_s_setprio(3);
}

/* ------------------------------------------------------------------------ */
/* MC kernel                                                                 */
/* mode 0: n_cyc cycles (steps from each complex's device counter)           */
/* mode 1: initial energies (44.5 * move_scale displacement if P.away)       */
/* queue != nullptr: persistent -- tasks are taken from *queue until it      */
/* passes n_tasks (every workgroup exits once the list is drained).          */
/* ------------------------------------------------------------------------ */
/* WPG: waves (replicas) per workgroup.  MINW: waves per SIMD the register
 * allocation must allow (1 = the compiler's choice, about 90 VGPRs, 5 waves;
 * 6 = 80 VGPRs; 8 = 64 VGPRs with a few spill slots) -- the launch shape
 * and this are picked by timing. */
template <int WPG, int MINW>
__global__ void __launch_bounds__(GD_WAVE *WPG) __attribute__((amdgpu_waves_per_eu(MINW, 8)))
gd_mc_kernel(const gd_pack *__restrict__ packs, const gd_task *__restrict__ tasks,
             int n_tasks, int *queue, int mode, int n_cyc, int wslot_off, int prio)
{
  extern __shared__ __attribute__((aligned(16))) char smem[];
  gd_set_prio(prio);
  __shared__ int s_task;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / GD_WAVE);
  gd_lds_f32 *ws = (gd_lds_f32 *) (smem + wslot_off) + w * GD_WSLOT_FLOATS;
  int staged_cx = -1, staged_prt = -1;
  int t = queue ? -1 : (int) blockIdx.x;

  for (;;) {
    if (queue) {
      if (threadIdx.x == 0)
        s_task = atomicAdd(queue, 1);
      __syncthreads();
      /* the task index is workgroup-uniform: keep it (and every pack field
       * read through it) in scalar registers */
      t = __builtin_amdgcn_readfirstlane(s_task);
      __syncthreads();
    } else if (t != (int) blockIdx.x) {
      break;  /* grid form: one task per workgroup */
    }
    if (t >= n_tasks)
      break;
    const gd_task task = tasks[t];
    const gd_pack &P = packs[task.cx];
    int s0 = 0, n_steps = 0;
    if (mode == 0) {
      s0 = __builtin_amdgcn_readfirstlane(P.step[0]);
      n_steps = gd_launch_steps(P, s0, n_cyc);
    }
    if (mode != 0 || n_steps > 0) {
      if (task.cx != staged_cx || task.prt != staged_prt) {
        __syncthreads();
        gd_stage(P, task.prt, smem);
        __syncthreads();
        staged_cx = task.cx;
        staged_prt = task.prt;
      }
      if (w < task.r_count) {
        const int r = task.r_begin + w;
        if (mode == 0)
          gd_replica_cycle(P, smem, ws, r, task.prt, s0, n_steps);
        else
          gd_replica_init(P, smem, r, task.prt);
      }
    }
    if (!queue)
      t = -2;
  }
}

/* MC cycle with SPLIT wavefronts per workgroup and the task's one to four
 * replicas sharing them, grid form or persistent as gd_mc_kernel: for launches
 * with too few replicas to give every SIMD several, where one wavefront per
 * replica leaves most of the device idle and every step waits on its own
 * latency.  Workgroups of 4 and 8 have one replica each (the engine's rule),
 * known to the compiler, and registers for four wavefronts a SIMD, so that two
 * workgroups of 8 fit a CU. */
template <int SPLIT>
__global__ void __launch_bounds__(GD_WAVE *SPLIT) __attribute__((amdgpu_waves_per_eu(4, 8)))
gd_mc_split_kernel(const gd_pack *__restrict__ packs, const gd_task *__restrict__ tasks,
                   int n_tasks, int *queue, int n_cyc, int area_off, int prio)
{
  extern __shared__ __attribute__((aligned(16))) char smem[];
  gd_set_prio(prio);
  __shared__ int s_task;
  __shared__ int s_ctr[2];
  const int role = __builtin_amdgcn_readfirstlane(threadIdx.x / GD_WAVE);
  gd_lds_f32 *areas = (gd_lds_f32 *) (smem + area_off);
  int staged_cx = -1, staged_prt = -1;
  int t = queue ? -1 : (int) blockIdx.x;

  for (;;) {
    if (queue) {
      if (threadIdx.x == 0)
        s_task = atomicAdd(queue, 1);
      __syncthreads();
      t = __builtin_amdgcn_readfirstlane(s_task);
      __syncthreads();
    } else if (t != (int) blockIdx.x) {
      break;
    }
    if (t >= n_tasks)
      break;
    const gd_task task = tasks[t];
    const gd_pack &P = packs[task.cx];
    const int s0 = __builtin_amdgcn_readfirstlane(P.step[0]);
    const int n_steps = gd_launch_steps(P, s0, n_cyc);
    if (n_steps > 0) {
      if (task.cx != staged_cx || task.prt != staged_prt) {
        __syncthreads();
        gd_stage(P, task.prt, smem);
        staged_cx = task.cx;
        staged_prt = task.prt;
      }
      /* (the cycle's first barrier covers the staging) */
      gd_replica_cycle_split<SPLIT>(P, smem, areas, (gd_lds_i32 *) s_ctr, role, task.r_begin,
                                    s0, n_steps,
                                    gd_split_consts_of(P, task.prt, SPLIT < 16 ? 1 : task.r_count));
    }
    if (!queue)
      t = -2;
  }
}


/* ------------------------------------------------------------------------ */
/* Energies of given poses (FP32).                                           */
/* ------------------------------------------------------------------------ */
__global__ void __launch_bounds__(GD_WAVE * 8)
gd_score_kernel(const gd_pack *__restrict__ packs, const gd_task *__restrict__ tasks,
                const int *__restrict__ pose_ids, const int *__restrict__ lig_conf,
                const float *__restrict__ move, float *__restrict__ energy)
{
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const gd_task task = tasks[blockIdx.x];
  const gd_pack &P = packs[task.cx];
  gd_stage(P, task.prt, smem);
  __syncthreads();
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / GD_WAVE);
  if (w >= task.r_count)
    return;
  const int lane = threadIdx.x & (GD_WAVE - 1);
  const int i = pose_ids[task.r_begin + w];
  float bx0, by0, bz0, bx1, by1, bz1;
  gd_load_conformer(P, lig_conf[i], &bx0, &by0, &bz0, &bx1, &by1, &bz1);
  float m[6];
#pragma unroll
  for (int k = 0; k < 6; ++k)
    m[k] = move[i * 6 + k];
  float ax0, ay0, az0, ax1, ay1, az1, cen[3], e[GD_E_N];
  gd_place(P, m, bx0, by0, bz0, bx1, by1, bz1, &ax0, &ay0, &az0, &ax1, &ay1, &az1, cen);
  float cm;
  gd_energy_wave(P, smem, task.prt, ax0, ay0, az0, ax1, ay1, az1, cen, e, &cm);
  if (lane == 0) {
#pragma unroll
    for (int k = 0; k < GD_E_N; ++k)
      energy[i * GD_E_N + k] = e[k];
  }
}

/* The energies of one to four poses a workgroup, each split over its 16
 * wavefronts as the MC steps are: with energy, of the given poses of the task
 * (as gd_score_kernel); else the initial energies of its replicas (as
 * gd_mc_kernel's mode 1).  A wavefront alone waits on its own latency: one
 * pose of 24 atoms x 300 points 60 us whole | 14 split, 189 of 34 x 344
 * 99 | 18, 592 replicas of 61 x 1,037 352 | 79. */
__global__ void __launch_bounds__(GD_WAVE *GD_POSE_SPLIT)
gd_pose_split_kernel(const gd_pack *__restrict__ packs, const gd_task *__restrict__ tasks,
                     const int *__restrict__ pose_ids, const int *__restrict__ lig_conf,
                     const float *__restrict__ move, float *__restrict__ energy, int area_off)
{
  extern __shared__ __attribute__((aligned(16))) char smem[];
  __shared__ int s_ctr;
  const gd_task task = tasks[blockIdx.x];
  const gd_pack &P = packs[task.cx];
  const int role = __builtin_amdgcn_readfirstlane(threadIdx.x / GD_WAVE);
  const int lane = threadIdx.x & (GD_WAVE - 1);
  gd_lds_f32 *areas = (gd_lds_f32 *) (smem + area_off);
  const gd_split_consts Z = gd_split_consts_of(P, task.prt, task.r_count);
  gd_stage(P, task.prt, smem);
  /* slots that no item writes count as +0 in the sums */
  for (int j = 0; j < Z.share; ++j)
    for (int i = GD_SA_PART + (int) threadIdx.x; i < GD_SA_POSE; i += GD_WAVE * GD_POSE_SPLIT)
      areas[j * GD_SA_FLOATS + i] = 0.0f;
  if (threadIdx.x == 0)
    s_ctr = GD_POSE_SPLIT * GD_WAVE;   /* every wavefront begins with its own item */

  /* wavefront j: pose j of the task */
  const bool lead = role < Z.share;
  gd_lds_f32 *A = areas + (lead ? role : 0) * GD_SA_FLOATS;
  const int at = task.r_begin + (lead ? role : 0);
  const int i = energy ? gd_uload(pose_ids + at) : at;
  const int k = lane < 6 ? lane : 0;
  float m_l = 0.0f;
  if (lead) {
    if (energy) {
      m_l = move[i * 6 + k];
    } else {
      m_l = P.S.mv[i * 8 + k];
      if (P.away)
        m_l = P.move_scale[k] * 44.5f + m_l;
    }
    const int conf = gd_uload((energy ? lig_conf : P.rep_lig) + i);
    gd_pose_put(Z, A + GD_SA_POSE, m_l, P.lig_xyz + (size_t) conf * Z.H.lna);
    __builtin_amdgcn_wave_barrier();
    gd_term_put(Z, A + GD_SA_TERM, GD_F_DST, gd_pose_edst(Z, A + GD_SA_POSE));
  }
  __syncthreads();
  gd_split_items(smem, areas, (gd_lds_i32 *) &s_ctr, Z, 0, role, false, []() {});
  __syncthreads();
  gd_split_sums(areas, role, GD_POSE_SPLIT, Z);
  __syncthreads();
  if (!lead)
    return;
  float w[GD_F_NTERM];
#pragma unroll
  for (int t = 0; t < GD_F_NTERM; ++t)
    w[t] = P.w[t];
  const gd_lds_f32 *term = A + GD_SA_TERM;
  const float total = Z.combine ? gd_split_bayes(Z, term) : gd_split_total(term, w);
  const float e_l = gd_split_energy(Z, term, total);
  if (energy) {
    if (lane < GD_E_N)
      energy[i * GD_E_N + lane] = e_l;
    return;
  }
  const gd_state S = P.S;
  const float cm = gd_split_mcc(Z, A);
  if (lane < 6) {
    S.mv[i * 8 + lane] = m_l;
    S.mv_best[i * 8 + lane] = m_l;
  }
  if (lane < GD_E_N) {
    S.e[i * 10 + lane] = e_l;
    S.e_best[i * 10 + lane] = e_l;
  }
  if (lane == 0) {
    S.cmcc[i] = cm;
    S.cmcc_best[i] = cm;
    S.step_best[i] = -1;
  }
}

/* ------------------------------------------------------------------------ */
/* host-callable launch wrappers                                             */
/* ------------------------------------------------------------------------ */
template <int WPG, int MINW>
static hipError_t launch_mc_var(const gd_pack *packs, const gd_task *tasks, int n_tasks,
                                int *queue, int grid, int mode, int n_cyc, int stage_bytes,
                                int prio, hipStream_t st)
{
  const int lds = stage_bytes + WPG * GD_WSLOT_FLOATS * 4;
  hipLaunchKernelGGL((gd_mc_kernel<WPG, MINW>), dim3(grid), dim3(GD_WAVE * WPG), lds, st,
                     packs, tasks, n_tasks, queue, mode, n_cyc, stage_bytes, prio);
  return hipGetLastError();
}

template <int WPG>
static hipError_t launch_mc_wpg(const gd_launch_cfg &C, const gd_pack *packs,
                                const gd_task *tasks, int n_tasks, int *queue, int grid,
                                int mode, int n_cyc, hipStream_t st)
{
  switch (C.occ) {
  case 6:
    return launch_mc_var<WPG, 6>(packs, tasks, n_tasks, queue, grid, mode, n_cyc,
                                 C.stage_bytes, C.prio, st);
  case 8:
    return launch_mc_var<WPG, 8>(packs, tasks, n_tasks, queue, grid, mode, n_cyc,
                                 C.stage_bytes, C.prio, st);
  default:
    return launch_mc_var<WPG, 1>(packs, tasks, n_tasks, queue, grid, mode, n_cyc,
                                 C.stage_bytes, C.prio, st);
  }
}

template <int SPLIT>
static hipError_t launch_split(const gd_launch_cfg &C, const gd_pack *packs,
                               const gd_task *tasks, int n_tasks, int *queue, int grid,
                               int n_cyc, hipStream_t st)
{
  const int lds = C.stage_bytes + GD_SPLIT_LDS_BYTES(C.share) - GD_SPLIT_ROOM;
  hipLaunchKernelGGL(gd_mc_split_kernel<SPLIT>, dim3(grid), dim3(GD_WAVE * SPLIT), lds, st,
                     packs, tasks, n_tasks, queue, n_cyc, C.stage_bytes, C.prio);
  return hipGetLastError();
}

static hipError_t launch_pose_split(const gd_pack *packs, const gd_task *tasks, int n_tasks,
                                    const int *pose_ids, const int *lig_conf,
                                    const float *move, int stage_bytes, int share,
                                    float *energy, hipStream_t st)
{
  if (n_tasks <= 0)
    return hipSuccess;
  hipLaunchKernelGGL(gd_pose_split_kernel, dim3(n_tasks), dim3(GD_WAVE * GD_POSE_SPLIT),
                     stage_bytes + GD_SPLIT_LDS_BYTES(share) - GD_SPLIT_ROOM, st, packs, tasks,
                     pose_ids, lig_conf, move, energy, stage_bytes);
  return hipGetLastError();
}

hipError_t gd_launch_mc(const gd_launch_cfg &C, const gd_pack *packs, const gd_task *tasks,
                        int n_tasks, int *queue, int grid, int mode, int n_cyc, hipStream_t st)
{
  if (n_tasks <= 0 || grid <= 0)
    return hipSuccess;
  if (mode == 0 && C.split > 1) {
    switch (C.split) {
    case 4: return launch_split<4>(C, packs, tasks, n_tasks, queue, grid, n_cyc, st);
    case 8: return launch_split<8>(C, packs, tasks, n_tasks, queue, grid, n_cyc, st);
    case 16: return launch_split<16>(C, packs, tasks, n_tasks, queue, grid, n_cyc, st);
    default: return hipErrorInvalidValue;
    }
  }
  switch (C.wpg) {
  case 4: return launch_mc_wpg<4>(C, packs, tasks, n_tasks, queue, grid, mode, n_cyc, st);
  case 16: return launch_mc_wpg<16>(C, packs, tasks, n_tasks, queue, grid, mode, n_cyc, st);
  default: return launch_mc_wpg<8>(C, packs, tasks, n_tasks, queue, grid, mode, n_cyc, st);
  }
}

hipError_t gd_launch_exchange(const gd_pack *packs, const gd_chain *chains, int n_chain,
                              int n_cx, int *queue, int n_queue, int *done, hipStream_t st)
{
  if (n_chain <= 0)
    return gd_launch_advance(packs, n_cx, queue, n_queue, 1, st);
  if (n_chain <= GD_X1_MAX_CHAINS) {
    const int nw = n_chain < GD_X1_WAVES ? n_chain : GD_X1_WAVES;
    hipLaunchKernelGGL(gd_exchange1_kernel, dim3(1), dim3(GD_WAVE * nw), 0, st, packs, chains,
                       n_chain, n_cx, queue, n_queue);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(gd_exchange_kernel, dim3((n_chain + GD_XWAVES - 1) / GD_XWAVES),
                     dim3(GD_WAVE * GD_XWAVES), 0, st, packs, chains, n_chain, n_cx, queue,
                     n_queue, done);
  return hipGetLastError();
}

hipError_t gd_launch_advance(const gd_pack *packs, int n_cx, int *queue, int n_queue,
                             int n_cyc, hipStream_t st)
{
  hipLaunchKernelGGL(gd_advance_kernel, dim3(1), dim3(256), 0, st, packs, n_cx, queue,
                     n_queue, n_cyc);
  return hipGetLastError();
}

hipError_t gd_launch_score(const gd_pack *packs, const gd_task *tasks, int n_tasks,
                           const int *pose_ids, const int *lig_conf, const float *move,
                           int stage_bytes, int share, float *energy, hipStream_t st)
{
  if (n_tasks <= 0)
    return hipSuccess;
  if (share > 0)
    return launch_pose_split(packs, tasks, n_tasks, pose_ids, lig_conf, move, stage_bytes,
                             share, energy, st);
  hipLaunchKernelGGL(gd_score_kernel, dim3(n_tasks), dim3(GD_WAVE * 8), stage_bytes, st,
                     packs, tasks, pose_ids, lig_conf, move, energy);
  return hipGetLastError();
}

hipError_t gd_launch_init_split(const gd_pack *packs, const gd_task *tasks, int n_tasks,
                                int stage_bytes, int share, hipStream_t st)
{
  return launch_pose_split(packs, tasks, n_tasks, nullptr, nullptr, nullptr, stage_bytes,
                           share, nullptr, st);
}

/* The dynamic LDS limit of every MC and scoring kernel: the device's LDS less
 * the room for static LDS, whatever a launch needs.  The limit belongs to the
 * process, so launches of other threads and engines must set the same value;
 * one that set its own smaller need would lower it between another's setting
 * and launch.  (No complex runs that needs more: the image and the engine
 * check the same sums.) */
hipError_t gd_set_kernel_attrs()
{
  int dev = 0, max_lds = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e == hipSuccess)
    e = hipDeviceGetAttribute(&max_lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev);
  const void *kernels[] = {
      (const void *) gd_pose_split_kernel,   (const void *) gd_mc_split_kernel<4>,
      (const void *) gd_mc_split_kernel<8>,  (const void *) gd_mc_split_kernel<16>,
      (const void *) gd_mc_kernel<4, 1>,     (const void *) gd_mc_kernel<4, 6>,
      (const void *) gd_mc_kernel<4, 8>,     (const void *) gd_mc_kernel<8, 1>,
      (const void *) gd_mc_kernel<8, 6>,     (const void *) gd_mc_kernel<8, 8>,
      (const void *) gd_mc_kernel<16, 1>,    (const void *) gd_mc_kernel<16, 6>,
      (const void *) gd_mc_kernel<16, 8>,    (const void *) gd_score_kernel};
  for (const void *k : kernels)
    if (e == hipSuccess)
      e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize,
                              max_lds - GD_SPLIT_ROOM);
  return e;
}

template <int WPG, int MINW>
static hipError_t occ_var(int stage_bytes, int *blocks)
{
  return hipOccupancyMaxActiveBlocksPerMultiprocessor(
      blocks, gd_mc_kernel<WPG, MINW>, GD_WAVE * WPG, stage_bytes + WPG * GD_WSLOT_FLOATS * 4);
}

template <int WPG>
static hipError_t occ_wpg(int occ, int stage_bytes, int *blocks)
{
  switch (occ) {
  case 6: return occ_var<WPG, 6>(stage_bytes, blocks);
  case 8: return occ_var<WPG, 8>(stage_bytes, blocks);
  default: return occ_var<WPG, 1>(stage_bytes, blocks);
  }
}

template <int SPLIT>
static hipError_t occ_split(int share, int stage_bytes, int *blocks)
{
  return hipOccupancyMaxActiveBlocksPerMultiprocessor(
      blocks, gd_mc_split_kernel<SPLIT>, GD_WAVE * SPLIT,
      stage_bytes + GD_SPLIT_LDS_BYTES(share) - GD_SPLIT_ROOM);
}

hipError_t gd_mc_occupancy(const gd_launch_cfg &C, int stage_bytes, int *blocks_per_cu)
{
  switch (C.split) {
  case 4: return occ_split<4>(C.share, stage_bytes, blocks_per_cu);
  case 8: return occ_split<8>(C.share, stage_bytes, blocks_per_cu);
  case 16: return occ_split<16>(C.share, stage_bytes, blocks_per_cu);
  default: break;
  }
  switch (C.wpg) {
  case 4: return occ_wpg<4>(C.occ, stage_bytes, blocks_per_cu);
  case 16: return occ_wpg<16>(C.occ, stage_bytes, blocks_per_cu);
  default: return occ_wpg<8>(C.occ, stage_bytes, blocks_per_cu);
  }
}

/* ------------------------------------------------------------------------ */
/* Static device workspace of the allocation-free pose scoring entry point:  */
/* one array per GPU, for the whole process.  Host code never uses the      */
/* array's name as an address: gd_scratch_region resolves each device's     */
/* own copy once, with that device current, and hands out that address.     */
/* ------------------------------------------------------------------------ */
static __device__ __align__(256) char scratch[GD_SCRATCH_BYTES + GD_SCRATCH_SLACK];

#define GD_SCRATCH_MAX_DEVICES 64

hipError_t gd_scratch_region(int device, char **ptr)
{
  static std::mutex mu;
  static char *dev_ptr[GD_SCRATCH_MAX_DEVICES] = {};
  if (device < 0 || device >= GD_SCRATCH_MAX_DEVICES)
    return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lk(mu);
  if (!dev_ptr[device]) {
    int cur = -1;
    hipError_t e = hipGetDevice(&cur);
    if (e != hipSuccess)
      return e;
    if (cur != device)
      return hipErrorInvalidDevice;   /* the caller makes `device` current */
    void *p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess)
      return e;
    if (!p)
      return hipErrorInvalidSymbol;
    dev_ptr[device] = (char *) p;
  }
  *ptr = dev_ptr[device];
  return hipSuccess;
}

/* ------------------------------------------------------------------------ */
/* VALU issue-rate probe: eight independent FMA chains per lane, every       */
/* operand in a vector register (v_fmac_f32_e32), 16 x iters rounds; one     */
/* store per lane keeps the chains live.  Calibrates the FP32 VALU ceiling   */
/* that the MC kernel's instruction rate is read against.                    */
/* ------------------------------------------------------------------------ */
__global__ void __launch_bounds__(256) gd_valu_probe_kernel(float *out, int iters)
{
  const float a = 0.999f + (float) threadIdx.x * 1e-7f;
  const float b = 1e-3f + (float) threadIdx.x * 1e-7f;
  float x[8];
#pragma unroll
  for (int c = 0; c < 8; ++c)
    x[c] = (float) threadIdx.x * 1e-3f + (float) c;
  for (int i = 0; i < iters; ++i) {
#pragma unroll
    for (int k = 0; k < 16; ++k) {
#pragma unroll
      for (int c = 0; c < 8; ++c)
        x[c] = gd_fma(a, b, x[c]);
    }
  }
  float s = 0.0f;
#pragma unroll
  for (int c = 0; c < 8; ++c)
    s += x[c];
  out[blockIdx.x * blockDim.x + threadIdx.x] = s;
}

hipError_t gd_launch_valu_probe(float *out, int blocks, int iters, hipStream_t st)
{
  hipLaunchKernelGGL(gd_valu_probe_kernel, dim3(blocks), dim3(256), 0, st, out, iters);
  return hipGetLastError();
}

/* Issue rate of one VALU instruction kind: eight independent register
 * chains per lane, 16 rounds of them per loop iteration, nothing but
 * registers inside the loop and one store per lane at the end.  The kinds
 * are the ones the energy loops are made of (gd_valu_kind_names). */
#define GD_K8(...)                                                              \
  do {                                                                          \
    _Pragma("unroll") for (int k_ = 0; k_ < 16; ++k_) {                        \
      GD_K1(x0, __VA_ARGS__); GD_K1(x1, __VA_ARGS__); GD_K1(x2, __VA_ARGS__);  \
      GD_K1(x3, __VA_ARGS__); GD_K1(x4, __VA_ARGS__); GD_K1(x5, __VA_ARGS__);  \
      GD_K1(x6, __VA_ARGS__); GD_K1(x7, __VA_ARGS__);                          \
    }                                                                           \
  } while (0)
template <int KIND>
__global__ void __launch_bounds__(256)
    gd_valu_kind_kernel(float *out, int iters, unsigned long long mask, float sv)
{
  float x0 = (float) threadIdx.x * 1e-3f, x1 = x0 + 1.0f, x2 = x0 + 2.0f, x3 = x0 + 3.0f;
  float x4 = x0 + 4.0f, x5 = x0 + 5.0f, x6 = x0 + 6.0f, x7 = x0 + 7.0f;
  const float a = 0.999f, b = 1e-3f;
  int sink = 0;
  for (int i = 0; i < iters; ++i) {
    if (KIND == 0) {
#define GD_K1(x, ...) asm volatile("v_fmac_f32 %0, %1, %2" : "+v"(x) : "v"(a), "v"(b))
      GD_K8(0);
#undef GD_K1
    } else if (KIND == 1) {
#define GD_K1(x, ...) asm volatile("v_fma_f32 %0, %1, %2, %0" : "+v"(x) : "s"(sv), "v"(b))
      GD_K8(0);
#undef GD_K1
    } else if (KIND == 2) {
#define GD_K1(x, ...) asm volatile("v_mul_f32 %0, %0, %1" : "+v"(x) : "v"(a))
      GD_K8(0);
#undef GD_K1
    } else if (KIND == 3) {
#define GD_K1(x, ...) asm volatile("v_max_f32 %0, %0, %1" : "+v"(x) : "v"(b))
      GD_K8(0);
#undef GD_K1
    } else if (KIND == 4) {
#define GD_K1(x, ...) asm volatile("v_cndmask_b32_e64 %0, %0, %1, %2" : "+v"(x) : "v"(a), "s"(mask))
      GD_K8(0);
#undef GD_K1
    } else if (KIND == 5) {
#define GD_K1(x, ...) asm volatile("v_lshl_add_u32 %0, %0, 1, %1" : "+v"(x) : "v"(b))
      GD_K8(0);
#undef GD_K1
    } else if (KIND == 6) {
#define GD_K1(x, ...) asm volatile("v_cmp_gt_f32 vcc, %0, %1" : : "v"(x), "v"(a) : "vcc")
      GD_K8(0);
#undef GD_K1
    } else if (KIND == 7) {
#define GD_K1(x, ...) \
  asm volatile("v_add_f32_dpp %0, %0, %0 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf" : "+v"(x))
      GD_K8(0);
#undef GD_K1
    } else if (KIND == 8) {
#define GD_K1(x, ...)                                                    \
  do {                                                                   \
    int s_;                                                              \
    asm volatile("v_readlane_b32 %0, %1, 5" : "=s"(s_) : "v"(x));        \
    sink ^= s_;                                                          \
  } while (0)
      GD_K8(0);
#undef GD_K1
    } else {
      /* FMA and max alternating: how much of a slower kind hides behind
       * the full-rate one */
#define GD_K1(x, ...) asm volatile("v_fmac_f32 %0, %1, %2\n\tv_max_f32 %0, %0, %1" : "+v"(x) : "v"(a), "v"(b))
      GD_K8(0);
#undef GD_K1
    }
  }
  out[blockIdx.x * blockDim.x + threadIdx.x] =
      ((x0 + x1) + (x2 + x3)) + ((x4 + x5) + (x6 + x7)) + (float) sink;
}
#undef GD_K8

hipError_t gd_launch_valu_kind(int kind, float *out, int blocks, int iters, hipStream_t st)
{
  const unsigned long long m = 0x5555555555555555ull;
  switch (kind) {
  case 0: hipLaunchKernelGGL(gd_valu_kind_kernel<0>, dim3(blocks), dim3(256), 0, st, out, iters, m, 1.0f); break;
  case 1: hipLaunchKernelGGL(gd_valu_kind_kernel<1>, dim3(blocks), dim3(256), 0, st, out, iters, m, 1.0f); break;
  case 2: hipLaunchKernelGGL(gd_valu_kind_kernel<2>, dim3(blocks), dim3(256), 0, st, out, iters, m, 1.0f); break;
  case 3: hipLaunchKernelGGL(gd_valu_kind_kernel<3>, dim3(blocks), dim3(256), 0, st, out, iters, m, 1.0f); break;
  case 4: hipLaunchKernelGGL(gd_valu_kind_kernel<4>, dim3(blocks), dim3(256), 0, st, out, iters, m, 1.0f); break;
  case 5: hipLaunchKernelGGL(gd_valu_kind_kernel<5>, dim3(blocks), dim3(256), 0, st, out, iters, m, 1.0f); break;
  case 6: hipLaunchKernelGGL(gd_valu_kind_kernel<6>, dim3(blocks), dim3(256), 0, st, out, iters, m, 1.0f); break;
  case 7: hipLaunchKernelGGL(gd_valu_kind_kernel<7>, dim3(blocks), dim3(256), 0, st, out, iters, m, 1.0f); break;
  case 8: hipLaunchKernelGGL(gd_valu_kind_kernel<8>, dim3(blocks), dim3(256), 0, st, out, iters, m, 1.0f); break;
  default: hipLaunchKernelGGL(gd_valu_kind_kernel<9>, dim3(blocks), dim3(256), 0, st, out, iters, m, 1.0f); break;
  }
  return hipGetLastError();
}
