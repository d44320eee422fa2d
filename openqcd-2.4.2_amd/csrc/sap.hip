// sap.hip -- Schwarz alternating procedure (SAP) on gfx950.
//
// Replaces sap/sap.c:592-790 (sap, update_flds0/1/2), sap/blk_solv.c:1117-1186
// (blk_mres, blk_eo_mres), dirac/Dw.c:1475-1907 (the block operators),
// dirac/Dw_bnd.c:801-1011 with sap/sap_com.c:465-501 (block boundary update)
// and the SAP_BLOCKS parts of block/blk_grid.c, map_u2blk.c, map_sw2blk.c and
// map_s2blk.c.
//
// Blocks of 4^4 points are held in the registers of a work-group (k_sap_reg),
// larger ones of multiples of 4 in those of several (k_sap_cluster), other
// blocks of up to 1365 points in the registers and LDS of one (k_sap_lds).  For
// the rest and in FP64 (k_sap_blocks) one work-group handles one block of the
// current colour, and the block's three
// fields (solution s0, residual s1, work s2) are kept block-compact in a
// scratch area (site-block layout over the block-local point index, even
// points first, as the reference's block geometry, lattice/blk_geometry.c);
// links and SW matrices are read from the global single-precision fields
// through the block's embedding table imb.  All nmr minimal-residual steps of
// a block run inside the work-group: the block Dirac operator with Dirichlet
// exterior, the two block reductions (LDS tree in double precision, rounded
// to float as salg.c does) and the two vector updates, separated by
// work-group barriers.
//
// The reference computes the hopping terms from each block across its faces
// (Dw_bnd) and subtracts them from the residual of the neighbouring blocks
// after all blocks of the colour are done (sap_com).  k_sap_reg and
// k_sap_cluster write these terms as Weyl fields on the faces of their blocks and
// add those of the other colour at the start of a solve.  k_sap_lds and
// k_sap_blocks write the block corrections s0 to a global field and a second
// kernel gathers, for every face point of the blocks of the other colour, the
// hopping terms from its neighbours in other blocks, so that no point is updated
// by two work-items.
#include <cfloat>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <array>
#include <vector>

#include <hip/hip_fp16.h>

#include "dirac_dev.h"

namespace oqh {

constexpr int SWG = 256;      // work-group size of the block kernels
constexpr int SWG_MAX = 1024; // work-group size of the generic FP32 block solver
constexpr int NBF = 4;    // block fields of the API per block: s[0..2] + the Dwhat_blk intermediate
#ifndef OQH_SAP_REG
#define OQH_SAP_REG 1
#endif

struct SapGrid
{
   bool ready = false;
   int bs[4] = {0, 0, 0, 0};
   int nb = 0, nbh = 0, bvol = 0, bh = 0;
   size_t Ub = 0;                        // units per block field
   int *d_imb = nullptr;                 // [nb][bvol]
   int *d_bnb = nullptr;                 // [8][bvol], bvol = outside
   int *d_face[2] = {nullptr, nullptr};  // face points of colour-c blocks
   unsigned char *d_fmask[2] = {nullptr, nullptr};
   int nface[2] = {0, 0};
   float2 *d_swb = nullptr;              // FP32 SW field of the block solver
   int swb_set = -1;                     // ptset_t used for the inversion, -1 none
   int swb_epoch = -1;                   // SW field version it was made from
   float2 *d_scr = nullptr;              // [nbh][3][Ub]
   float2 *d_s0g = nullptr;              // global field of block corrections
   float2 *d_bs = nullptr;               // block fields of the API, [nb][3][Ub]
   double2 *d_bsd = nullptr;             // FP64 block fields of the API, [nb][NBF][Ub]
   bool need64 = false;                  // FP64 block operators in use: keep d_swb64
   __half2 *d_u16 = nullptr;             // FP16 links (FP16 variant of the solver)
   __half2 *d_swb16 = nullptr;           // FP16 block SW field
   float2 *d_wf = nullptr;               // face fields of the register kernel (one source)
   float2 *d_wfm = nullptr;              // those of several sources
   int wfm_n = 0;                        // number of sources in d_wfm
   int *d_nbn = nullptr;                 // neighbouring blocks [nb][8] (4^4 blocks)
   int ns = 0;                           // 4^4 sub-blocks per block (k_sap_cluster) or 0
   std::vector<int> imb4;                // points of the sub-blocks [nb][ns][256]
   int *d_imb4 = nullptr, *d_nbs = nullptr;
   unsigned *d_count = nullptr;          // ticket and arrival counters
   unsigned long long *d_x = nullptr;    // exchange buffers, sums
   int *h_dead = nullptr;                // host flag of k_sap_cluster
   double2 *d_swb64 = nullptr;           // FP64 block SW field (FP64 variant)
   int swb64_version = -1;
   double2 *d_h64[3] = {nullptr, nullptr, nullptr};  // FP64 psi, rho, s0g
   double2 *d_scr64 = nullptr;           // FP64 block fields [nbh][3][Ub]
   __half2 *d_h16[2] = {nullptr, nullptr};  // FP16 psi, rho
   float *d_hsc[2] = {nullptr, nullptr};    // their per-site scales
   int u16_epoch = -1, swb16_epoch = -1; // versions they were made from
   int swb_version = 0;                  // incremented by every assign_swb
   std::vector<int> imb;                 // host copy
   std::vector<int> bo;                  // [nb][4]
   int *d_ipp = nullptr;                 // face points of a block, faces 0..7 in turn
   int fofs[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};  // offsets of the faces in d_ipp
   float2 *d_bw = nullptr;               // Weyl fields of Dw_bnd, [nb][fofs[8]][6]
};

static SapGrid G;

template <typename C> struct SArgsT
{
   const C *u, *sw;
   const int *imb, *bnb, *nbr;
   const unsigned char *bnd;
   int V, h, bvol, bh, masked, eoflg, nmr;
   decltype(C::x) mu, muo;
   size_t Ub;
   C *psi, *rho, *s0g, *scr;
   int n0;             // first block of the colour
   // register kernel: face fields of the block corrections and neighbour
   // blocks ([nb][8])
   C *wf;
   const int *nbn;
   // FP16 variant: psi and rho as FP16 spinors with per-site scales
   __half2 *psi16, *rho16;
   float *psc, *rsc;
   int pz;             // psi is zero on entry (not read)
   int pull;           // add the terms of the other colour's face fields first
   // several right-hand sides in one launch (FP32): nsrc > 0 replaces psi,
   // rho, wf by the fields of source blockIdx % nsrc
   int nsrc;
   C *pl[16], *rl[16], *wl[16];
};
typedef SArgsT<float2> SArgs;   // FP32 and FP16 variants
typedef SArgsT<double2> SArgsD; // FP64 variant

// FP16 spinor with per-site scale: the 12 colour components of site x are
// stored as v / m in FP16 (same unit layout as the FP32 fields), m = the
// largest modulus of a real component of the spinor at x
__device__ inline void load_h16(const __half2 *h, const float *sc, int x, float2 *v)
{
   const float m = sc[x];
   const __half2 *p = h + (size_t)(x >> 6) * (12 * SB) + (x & (SB - 1));
#pragma unroll
   for (int c = 0; c < 12; c++)
   {
      float2 f = __half22float2(p[c * SB]);
      v[c] = make_float2(f.x * m, f.y * m);
   }
}

__device__ inline void store_h16(__half2 *h, float *sc, int x, const float2 *v)
{
   float m = 0.0f;
#pragma unroll
   for (int c = 0; c < 12; c++) m = fmaxf(m, fmaxf(fabsf(v[c].x), fabsf(v[c].y)));
   const float r = m > 0.0f ? 1.0f / m : 0.0f;
   sc[x] = m;
   __half2 *p = h + (size_t)(x >> 6) * (12 * SB) + (x & (SB - 1));
#pragma unroll
   for (int c = 0; c < 12; c++) p[c * SB] = __float22half2_rn(make_float2(v[c].x * r, v[c].y * r));
}

// link of direction mu, forward (x->x+mu) or backward (x-mu->x), seen from
// global point gx with global neighbour gy
template <typename C>
__device__ inline const C *blk_link(const SArgsT<C> &a, int gx, int gy, int mu, bool fwd)
{
   if (gx >= a.h) return link_ptr(a.u, gx - a.h, fwd ? 2 * mu : 2 * mu + 1);
   return link_ptr(a.u, gy - a.h, fwd ? 2 * mu + 1 : 2 * mu);
}

// acc += hopping terms from the in-block neighbours of block point i;
// neighbours on the global boundary (open bc) contribute nothing
template <int MU, typename C>
__device__ inline void blk_hop_mu(const SArgsT<C> &a, const int *imb, const C *S, int i, int gx, C *acc)
{
   C sp[12];
   int j = a.bnb[(2 * MU) * a.bvol + i];
   if (j < a.bvol)
   {
      int gy = imb[j];
      if (!(a.masked && a.bnd[gy]))
      {
         load_spinor(S, j, sp);
         hop_one<C, MU, true>(sp, blk_link(a, gx, gy, MU, true), acc);
      }
   }
   j = a.bnb[(2 * MU + 1) * a.bvol + i];
   if (j < a.bvol)
   {
      int gy = imb[j];
      if (!(a.masked && a.bnd[gy]))
      {
         load_spinor(S, j, sp);
         hop_one<C, MU, false>(sp, blk_link(a, gx, gy, MU, false), acc);
      }
   }
}

template <typename C>
__device__ inline void blk_hop(const SArgsT<C> &a, const int *imb, const C *S, int i, int gx, C *acc)
{
   blk_hop_mu<0>(a, imb, S, i, gx, acc);
   blk_hop_mu<1>(a, imb, S, i, gx, acc);
   blk_hop_mu<2>(a, imb, S, i, gx, acc);
   blk_hop_mu<3>(a, imb, S, i, gx, acc);
}

template <typename C> __device__ inline void zero12(C *v)
{
#pragma unroll
   for (int c = 0; c < 12; c++) v[c] = cmk<C>(0, 0);
}

// work-group sum of two doubles, broadcast to all threads
__device__ inline void wg_sum2(double &x, double &y, int nt)
{
   __shared__ double sh[2][SWG_MAX / 64];
#pragma unroll
   for (int m = 32; m >= 1; m >>= 1)
   {
      x += __shfl_xor(x, m);
      y += __shfl_xor(y, m);
   }
   int w = threadIdx.x >> 6;
   if ((threadIdx.x & 63) == 0)
   {
      sh[0][w] = x;
      sh[1][w] = y;
   }
   __syncthreads();
   x = 0.0;
   y = 0.0;
   for (int k = 0; k < (nt >> 6); k++)
   {
      x += sh[0][k];
      y += sh[1][k];
   }
   __syncthreads();
}

__device__ inline void wg_sum3(double &x, double &y, double &z, int nt)
{
   __shared__ double sh[3][SWG_MAX / 64];
#pragma unroll
   for (int m = 32; m >= 1; m >>= 1)
   {
      x += __shfl_xor(x, m);
      y += __shfl_xor(y, m);
      z += __shfl_xor(z, m);
   }
   int w = threadIdx.x >> 6;
   if ((threadIdx.x & 63) == 0)
   {
      sh[0][w] = x;
      sh[1][w] = y;
      sh[2][w] = z;
   }
   __syncthreads();
   x = y = z = 0.0;
   for (int k = 0; k < (nt >> 6); k++)
   {
      x += sh[0][k];
      y += sh[1][k];
      z += sh[2][k];
   }
   __syncthreads();
}

// S2 = Dw_blk S1 on the points [i0, i1) of the block (Dw.c:1475)
template <typename C>
__device__ void blk_dw(const SArgsT<C> &a, const int *imb, C *S1, C *S2, int i0, int i1, decltype(C::x) mu_e, int nt)
{
   typedef decltype(C::x) R;
   for (int i = i0 + threadIdx.x; i < i1; i += nt)
   {
      int gx = imb[i];
      C o[12];
      if (a.masked && a.bnd[gx])
      {
         zero12(o);
         store_spinor(S2, i, o);
         continue;
      }
      C acc[12], v[12];
      zero12(acc);
      blk_hop(a, imb, S1, i, gx, acc);
      load_spinor((const C *)S1, i, v);
      pauli_site(a.sw, gx, i < a.bh ? mu_e : a.muo, v, o);
#pragma unroll
      for (int c = 0; c < 12; c++) o[c] = cadd(o[c], cscale(acc[c], (R)-0.5));
      store_spinor(S2, i, o);
   }
}

// even points: S2_e = Dwhat_blk S1 (Dw.c:1828); the odd half of T holds the
// intermediate A_oo^-1 D_oe S1 (T = S2 inside the Schwarz cycles, a separate
// field for the block API, which leaves the odd half of S2 unchanged)
template <typename C>
__device__ void blk_dwhat(const SArgsT<C> &a, const int *imb, C *S1, C *S2, C *T, decltype(C::x) mu, int nt)
{
   typedef decltype(C::x) R;
   for (int i = a.bh + threadIdx.x; i < a.bvol; i += nt)
   {
      int gx = imb[i];
      C o[12];
      if (a.masked && a.bnd[gx])
      {
         zero12(o);
         store_spinor(T, i, o);
         continue;
      }
      C acc[12];
      zero12(acc);
      blk_hop(a, imb, S1, i, gx, acc);
#pragma unroll
      for (int c = 0; c < 12; c++) acc[c] = cscale(acc[c], (R)-0.5);
      pauli_site(a.sw, gx, (R)0, acc, o);
      store_spinor(T, i, o);
   }
   __syncthreads();
   for (int i = threadIdx.x; i < a.bh; i += nt)
   {
      int gx = imb[i];
      C o[12];
      if (a.masked && a.bnd[gx])
      {
         zero12(o);
         store_spinor(S2, i, o);
         continue;
      }
      C acc[12], v[12];
      zero12(acc);
      blk_hop(a, imb, T, i, gx, acc);
      load_spinor((const C *)S1, i, v);
      pauli_site(a.sw, gx, mu, v, o);
#pragma unroll
      for (int c = 0; c < 12; c++) o[c] = cadd(o[c], cscale(acc[c], (R)0.5));
      store_spinor(S2, i, o);
   }
}

// minimal residual steps on points [0, nv) (blk_solv.c:1117-1186); T: odd
// intermediate of Dwhat_blk (EO)
template <bool EO, typename C>
__device__ void blk_mres_dev(const SArgsT<C> &a, const int *imb, C *S0, C *S1, C *S2, C *T, decltype(C::x) mu, int nt)
{
   typedef decltype(C::x) R;
   const R rmin = sizeof(R) == 4 ? (R)FLT_MIN : (R)DBL_MIN;
   int nv = EO ? a.bh : a.bvol;
   for (int i = threadIdx.x; i < nv; i += nt) zero_spinor(S0, i);
   __syncthreads();
   for (int imr = 0; imr < a.nmr; imr++)
   {
      if (EO)
         blk_dwhat(a, imb, S1, S2, T, mu, nt);
      else
         blk_dw(a, imb, S1, S2, 0, a.bvol, mu, nt);
      __syncthreads();
      double rr = 0.0, zr = 0.0, zi = 0.0;
      for (int i = threadIdx.x; i < nv; i += nt)
      {
         const C *p2 = S2 + (size_t)(i >> 6) * (12 * SB) + (i & (SB - 1));
         const C *p1 = S1 + (size_t)(i >> 6) * (12 * SB) + (i & (SB - 1));
#pragma unroll
         for (int k = 0; k < 4; k++)
         {
            R nr = 0, pr = 0, pi = 0;
#pragma unroll
            for (int c = 0; c < 3; c++)
            {
               C u = p2[(3 * k + c) * SB], v = p1[(3 * k + c) * SB];
               nr += u.x * u.x + u.y * u.y;
               pr += u.x * v.x + u.y * v.y;
               pi += u.x * v.y - u.y * v.x;
            }
            rr += (double)nr;
            zr += (double)pr;
            zi += (double)pi;
         }
      }
      wg_sum3(rr, zr, zi, nt);
      R r = (R)rr;
      if (r < (R)2 * rmin) break;
      r = (R)1 / r;
      C z = cmk<C>((R)zr * r, (R)zi * r);
      for (int i = threadIdx.x; i < nv; i += nt)
      {
         C *p0 = S0 + (size_t)(i >> 6) * (12 * SB) + (i & (SB - 1));
         C *p1 = S1 + (size_t)(i >> 6) * (12 * SB) + (i & (SB - 1));
         const C *p2 = S2 + (size_t)(i >> 6) * (12 * SB) + (i & (SB - 1));
#pragma unroll
         for (int c = 0; c < 12; c++)
         {
            C s1 = p1[c * SB], s2 = p2[c * SB], s0 = p0[c * SB];
            p0[c * SB] = cmk<C>(s0.x + (z.x * s1.x - z.y * s1.y), s0.y + (z.x * s1.y + z.y * s1.x));
            p1[c * SB] = cmk<C>(s1.x - (z.x * s2.x - z.y * s2.y), s1.y - (z.x * s2.y + z.y * s2.x));
         }
      }
      __syncthreads();
   }
}

// isolv=1 preparation: S1_o = A_oo^-1 S1_o, then S1_e -= D_eo S1_o
// (Dwoo_blk, Dweo_blk of sap.c:759-761)
template <typename C> __device__ void blk_eo_prepare(const SArgsT<C> &a, const int *imb, C *S1, int nt)
{
   typedef decltype(C::x) R;
   for (int i = a.bh + threadIdx.x; i < a.bvol; i += nt)
   {
      int gx = imb[i];
      C v[12], o[12];
      if (a.masked && a.bnd[gx])
         zero12(o);
      else
      {
         load_spinor((const C *)S1, i, v);
         pauli_site(a.sw, gx, (R)0, v, o);
      }
      store_spinor(S1, i, o);
   }
   __syncthreads();
   for (int i = threadIdx.x; i < a.bh; i += nt)
   {
      int gx = imb[i];
      C o[12];
      if (a.masked && a.bnd[gx])
         zero12(o);
      else
      {
         C acc[12];
         zero12(acc);
         blk_hop(a, imb, S1, i, gx, acc);
         load_spinor((const C *)S1, i, o);
#pragma unroll
         for (int c = 0; c < 12; c++) o[c] = cadd(o[c], cscale(acc[c], (R)0.5));
      }
      store_spinor(S1, i, o);
   }
   __syncthreads();
}

// isolv=1 completion: odd solution (Dwoe_blk, Dwoo_blk; update_flds1/2)
template <typename C> __device__ void blk_eo_finish(const SArgsT<C> &a, const int *imb, C *S0, C *S1, int nt)
{
   typedef decltype(C::x) R;
   for (int i = a.bh + threadIdx.x; i < a.bvol; i += nt)
   {
      int gx = imb[i];
      C o[12];
      if (a.masked && a.bnd[gx])
         zero12(o);
      else
      {
         C acc[12];
         zero12(acc);
         blk_hop(a, imb, S0, i, gx, acc);
#pragma unroll
         for (int c = 0; c < 12; c++) acc[c] = cscale(acc[c], (R)-0.5);
         pauli_site(a.sw, gx, (R)0, acc, o);
      }
      // s0_o = s1_o - A_oo^-1 D_oe s0_e
      C r1[12];
      load_spinor((const C *)S1, i, r1);
#pragma unroll
      for (int c = 0; c < 12; c++) o[c] = csub(r1[c], o[c]);
      store_spinor(S0, i, o);
   }
}

// ---------------------------------------------------------------------------
// the Schwarz sweep over the blocks of one colour
// ---------------------------------------------------------------------------

template <int ISOLV, typename C, int TPB = SWG>
__global__ __launch_bounds__(TPB) void k_sap_blocks(SArgsT<C> a)
{
   typedef decltype(C::x) R;
   int n = a.n0 + blockIdx.x;
   const int *imb = a.imb + (size_t)n * a.bvol;
   C *S0 = a.scr + (size_t)blockIdx.x * 3 * a.Ub;
   C *S1 = S0 + a.Ub, *S2 = S1 + a.Ub;

   for (int i = threadIdx.x; i < a.bvol; i += TPB)
   {
      int gx = imb[i];
      C v[12];
      if (!ISOLV && a.masked && a.bnd[gx])
         zero12(v);
      else
         load_spinor((const C *)a.rho, gx, v);
      store_spinor(S1, i, v);
   }
   __syncthreads();

   if (ISOLV)
   {
      blk_eo_prepare(a, imb, S1, TPB);
      blk_mres_dev<true>(a, imb, S0, S1, S2, S2, a.mu, TPB);
      blk_eo_finish(a, imb, S0, S1, TPB);
      __syncthreads();
   }
   else
      blk_mres_dev<false>(a, imb, S0, S1, S2, S2, a.mu, TPB);

   for (int i = threadIdx.x; i < a.bvol; i += TPB)
   {
      int gx = imb[i];
      C s0[12], s1[12], p[12];
      load_spinor((const C *)S0, i, s0);
      load_spinor((const C *)S1, i, s1);
      load_spinor((const C *)a.psi, gx, p);
#pragma unroll
      for (int c = 0; c < 12; c++) p[c] = cadd(p[c], s0[c]);
      store_spinor(a.psi, gx, p);
      if (ISOLV && i >= a.bh)
      {
         // odd residual -i mu gamma5 s0 (update_flds1) or 0 (eoflg, update_flds2)
         R m = a.eoflg ? (R)0 : a.mu;
#pragma unroll
         for (int c = 0; c < 12; c++)
         {
            R cm = (c < 6) ? -m : m;
            s1[c] = cmk<C>(-cm * s0[c].y, cm * s0[c].x);
         }
      }
      store_spinor(a.rho, gx, s1);
      store_spinor(a.s0g, gx, s0);
   }
}

// ---------------------------------------------------------------------------
// the Schwarz sweep with the block held in registers (blocks of 4^4 points)
//
// Lane x of the work-group owns block point x: its Pauli pair, its forward
// links U(x,mu) and the values of the block fields at x stay in registers
// for the whole block solve, so the global memory is read once (links, SW,
// residual) and written once per block.  A hopping pass of one parity
// exchanges only spinors: the lanes of the other parity (separate wavefronts)
// put their values into LDS (F) and pass the backward terms, formed with
// their own links, through LDS (X, two colour vectors after the spin
// projection); the output lanes add the forward terms from F and the
// backward terms from X.
//
// The hopping terms into the blocks of the other colour (Dw_bnd, sap_com of
// the reference) leave the block solve as Weyl fields on the eight faces:
// through a forward face the finished term U(x,mu)^+ (1+gamma_mu) s0(x),
// through a backward face (1-gamma_mu) s0(x), which the receiving point
// multiplies with its own forward link.  The next block solve of the
// receiving block adds them to its residual, so that neither the corrections
// nor the faces' links are gathered point by point.
// ---------------------------------------------------------------------------

constexpr int RBV = 256;
constexpr int FPT = 64;              // points of a face
constexpr int FUN = 8 * 6 * FPT;     // units of the face fields of a block

// complex multiply-accumulate as FMA chains: acc + a b, acc + conj(a) b
__device__ inline float2 cmac(float2 acc, float2 a, float2 b)
{
   return make_float2(fmaf(a.x, b.x, fmaf(-a.y, b.y, acc.x)), fmaf(a.x, b.y, fmaf(a.y, b.x, acc.y)));
}
__device__ inline float2 cmacc(float2 acc, float2 a, float2 b)
{
   return make_float2(fmaf(a.x, b.x, fmaf(a.y, b.y, acc.x)), fmaf(a.x, b.y, fmaf(-a.y, b.x, acc.y)));
}

// c = U h or U^dag h (U in registers) with FMA chains
template <bool DAG> __device__ inline void su3_mul_f(const float2 *u, const float2 *h, float2 *c)
{
#pragma unroll
   for (int i = 0; i < 3; i++)
   {
      if (!DAG)
         c[i] = cmac(cmac(cmul(u[3 * i], h[0]), u[3 * i + 1], h[1]), u[3 * i + 2], h[2]);
      else
         c[i] = cmacc(cmacc(cmulc(u[i], h[0]), u[3 + i], h[1]), u[6 + i], h[2]);
   }
}

// storage of links and SW matrices in the block solver: float2, or __half2
// in the FP16 variant (arithmetic in FP32 either way)
__device__ inline float2 to_f2(float2 v) { return v; }
__device__ inline float2 to_f2(__half2 v) { return __half22float2(v); }
template <typename S> __device__ inline S from_f2(float2 v);
template <> __device__ inline float2 from_f2<float2>(float2 v) { return v; }
template <> __device__ inline __half2 from_f2<__half2>(float2 v) { return __float22half2_rn(v); }

// Block point of a lane.  The order of the points of a 4^4 block is
// lexicographic within each parity, even points first: lane x < 128 is the
// even point, x >= 128 the odd point of pair i = x % 128, with
// i = lex / 2, so the forward neighbour of a point has the pair index
// i + 32, i + 8, i + 2 or i + (x3 odd) among the points of the other parity.
template <typename S> struct RegBlock
{
   S u[4][9];  // U(x,mu)
   int lex;    // t, x1, x2, x3 in two bits each, from the top
   bool odd;
   bool bp;    // open-bc boundary point
   __device__ int coord(int mu) const { return (lex >> (6 - 2 * mu)) & 3; }
   __device__ int pair() const { return lex >> 1; }
   __device__ int fwd(int mu) const  // pair index of x + mu (if it is in the block)
   {
      return pair() + (mu == 0 ? 32 : (mu == 1 ? 8 : (mu == 2 ? 2 : (lex & 1))));
   }
   // index of the point on a face orthogonal to mu as its sender has it: the
   // transverse coordinates in pairs, the points of even senders first
   __device__ int face_point(int mu, bool sender_odd) const
   {
      const int hi = lex >> (8 - 2 * mu), lo = lex & ((1 << (6 - 2 * mu)) - 1);
      return (((hi << (6 - 2 * mu)) | lo) >> 1) + (sender_odd ? 32 : 0);
   }
};

// o = (A + i mu) w (ADD: added to o) on one Weyl half (pauli_half), the 18
// units of A in q.
// LAST: the diagonal term, by far the largest, comes last, for each term of a
// chain of fused operations is rounded at the size of the sum so far.  Five cycles
// of 8^4 blocks on 16^4, isolv = 1, against FP64: 1.15e-7 (solution) and 3.2e-7
// (residual), with the diagonal first 1.47e-7 and 3.9e-7, with the separate
// products of k_sap_blocks 1.21e-7 and 3.4e-7; the time is the same.  With FP16
// storage (errors of 1e-4) the diagonal comes first, which takes 1.5 us less of a
// cycle of 82 at 16^4 (isolv = 0).
template <bool ADD = false, bool LAST = true>
__device__ inline void pauli_half_reg(const float2 *q, float mu, const float2 *w, float2 *o)
{
   static_assert(LAST || !ADD, "the diagonal starts the sum");
   float d[6] = {q[0].x, q[0].y, q[1].x, q[1].y, q[2].x, q[2].y};
   if (!LAST)
   {
#pragma unroll
      for (int i = 0; i < 6; i++) o[i] = make_float2(d[i] * w[i].x - mu * w[i].y, d[i] * w[i].y + mu * w[i].x);
   }
   constexpr bool FRESH = LAST && !ADD;
   int p = 3;
#pragma unroll
   for (int i = 0; i < 6; i++)
#pragma unroll
      for (int j = i + 1; j < 6; j++)
      {
         o[i] = (FRESH && i == 0 && j == 1) ? cmul(q[p], w[j]) : cmac(o[i], q[p], w[j]);
         o[j] = (FRESH && i == 0) ? cmulc(q[p], w[i]) : cmacc(o[j], q[p], w[i]);
         p++;
      }
   if (!LAST) return;
#pragma unroll
   for (int i = 0; i < 6; i++)
      o[i] = make_float2(fmaf(d[i], w[i].x, fmaf(-mu, w[i].y, o[i].x)), fmaf(d[i], w[i].y, fmaf(mu, w[i].x, o[i].y)));
}

// both Weyl halves; the half hh = 0 of A is read at m0 with stride st0, the
// half hh = 1 at m1 with stride st1 (registers or LDS)
template <bool ADD = false, typename S>
__device__ inline void pauli_reg2(const S *m0, int st0, const S *m1, int st1, float mu, const float2 *v, float2 *out)
{
#pragma unroll
   for (int hh = 0; hh < 2; hh++)
   {
      float2 q[18];
      const S *m = hh ? m1 : m0;
      const int stride = hh ? st1 : st0;
#pragma unroll
      for (int k = 0; k < 18; k++) q[k] = to_f2(m[k * stride]);
      pauli_half_reg<ADD, sizeof(S) == sizeof(float2)>(q, hh ? -mu : mu, v + 6 * hh, out + 6 * hh);
   }
}

template <int MU, bool FWD> __device__ inline void weyl_project(const float2 *sp, float2 *h)
{
   spin_project<float2, MU, FWD>(sp, h, h + 3);
}

// hopping pass into the points of parity OUT: the hopping terms from the
// in-block neighbours (src of the lanes of the other parity, zero on the
// boundary points of open bc) are added to w of the lanes of parity OUT,
// forward terms of mu = 0..3, then backward terms.  src and w may be the same
// registers.  lb: LDS of 18 * RBV float2.  hook.put() and hook.sent() are called
// by the source lanes once their values are in LDS and once they have formed
// their terms, hook.take() by the output lanes at the end.
struct NoHook
{
   __device__ void put() const {}
   __device__ void sent() const {}
   __device__ void take() const {}
};
template <int OUT, typename S, typename HOOK = NoHook>
__device__ inline void rb_hop(const RegBlock<S> &b, const float2 *src, float2 *w, float2 *lb, const HOOK &hook = HOOK())
{
   constexpr int RBH = RBV / 2;
   float2(*F)[RBH] = (float2(*)[RBH])lb;
   float2(*X)[6][RBH] = (float2(*)[6][RBH])(lb + 12 * RBH);
   const bool own = (OUT == (int)b.odd);
   const int i = b.pair();
   if (!own)
   {
#pragma unroll
      for (int c = 0; c < 12; c++) F[c][i] = src[c];
   }
   __syncthreads();
   if (!own) hook.put();
#pragma unroll
   for (int mu = 0; mu < 4; mu++)
   {
      const int y = b.fwd(mu);
      if (b.coord(mu) < 3)
      {
         float2 h[6], c[6], u[9];
#pragma unroll
         for (int k = 0; k < 9; k++) u[k] = to_f2(b.u[mu][k]);
         if (own)
         {
            float2 sp[12];
#pragma unroll
            for (int k = 0; k < 12; k++) sp[k] = F[k][y];
            if (mu == 0) weyl_project<0, true>(sp, h);
            if (mu == 1) weyl_project<1, true>(sp, h);
            if (mu == 2) weyl_project<2, true>(sp, h);
            if (mu == 3) weyl_project<3, true>(sp, h);
            su3_mul_f<false>(u, h, c);
            su3_mul_f<false>(u, h + 3, c + 3);
            if (mu == 0) spin_expand_add<float2, 0, true>(c, c + 3, w);
            if (mu == 1) spin_expand_add<float2, 1, true>(c, c + 3, w);
            if (mu == 2) spin_expand_add<float2, 2, true>(c, c + 3, w);
            if (mu == 3) spin_expand_add<float2, 3, true>(c, c + 3, w);
         }
         else
         {
            if (mu == 0) weyl_project<0, false>(src, h);
            if (mu == 1) weyl_project<1, false>(src, h);
            if (mu == 2) weyl_project<2, false>(src, h);
            if (mu == 3) weyl_project<3, false>(src, h);
            su3_mul_f<true>(u, h, c);
            su3_mul_f<true>(u, h + 3, c + 3);
#pragma unroll
            for (int k = 0; k < 6; k++) X[mu][k][y] = c[k];
         }
      }
   }
   if (!own) hook.sent();
   __syncthreads();
   if (own)
   {
#pragma unroll
      for (int mu = 0; mu < 4; mu++)
      {
         if (b.coord(mu) > 0)
         {
            float2 c[6];
#pragma unroll
            for (int k = 0; k < 6; k++) c[k] = X[mu][k][i];
            if (mu == 0) spin_expand_add<float2, 0, false>(c, c + 3, w);
            if (mu == 1) spin_expand_add<float2, 1, false>(c, c + 3, w);
            if (mu == 2) spin_expand_add<float2, 2, false>(c, c + 3, w);
            if (mu == 3) spin_expand_add<float2, 3, false>(c, c + 3, w);
         }
      }
      hook.take();
   }
}

// sum over the 64 lanes of a wavefront, complete in lane 63 (row operations
// in the vector unit instead of LDS permutes)
template <int CTRL, int ROWS> __device__ inline double dpp_add(double x)
{
   const long long v = __double_as_longlong(x);
   const int lo = __builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xf, false);
   const int hi = __builtin_amdgcn_update_dpp(0, (int)(v >> 32), CTRL, ROWS, 0xf, false);
   return x + __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

__device__ inline double wave_sum63(double x)
{
   x = dpp_add<0xb1, 0xf>(x);   // quad_perm [1,0,3,2]
   x = dpp_add<0x4e, 0xf>(x);   // quad_perm [2,3,0,1]
   x = dpp_add<0x141, 0xf>(x);  // row_half_mirror
   x = dpp_add<0x140, 0xf>(x);  // row_mirror: every lane has its row's sum
   x = dpp_add<0x142, 0xa>(x);  // row_bcast15: rows 1 and 3 add rows 0 and 2
   x = dpp_add<0x143, 0xc>(x);  // row_bcast31: rows 2 and 3 add row 1
   return x;
}

// block sums of |s2|^2 and (s2, s1) as in blk_mres_dev over the lanes with
// act (whole wavefronts).  sh may be written again only after another
// barrier has been passed.
__device__ inline void rb_sums(bool act, const float2 *s2, const float2 *s1, double (*sh)[4], double &rr, double &zr,
                               double &zi)
{
   const int wv = threadIdx.x >> 6;
   rr = zr = zi = 0.0;
   if (act)
   {
#pragma unroll
      for (int k = 0; k < 4; k++)
      {
         float nr = 0.0f, pr = 0.0f, pi = 0.0f;
#pragma unroll
         for (int c = 0; c < 3; c++)
         {
            float2 u = s2[3 * k + c], v = s1[3 * k + c];
            nr += u.x * u.x + u.y * u.y;
            pr += u.x * v.x + u.y * v.y;
            pi += u.x * v.y - u.y * v.x;
         }
         rr += (double)nr;
         zr += (double)pr;
         zi += (double)pi;
      }
      rr = wave_sum63(rr);
      zr = wave_sum63(zr);
      zi = wave_sum63(zi);
   }
   if ((threadIdx.x & 63) == 63)
   {
      sh[0][wv] = rr;
      sh[1][wv] = zr;
      sh[2][wv] = zi;
   }
   __syncthreads();
   rr = (sh[0][0] + sh[0][1]) + (sh[0][2] + sh[0][3]);
   zr = (sh[1][0] + sh[1][1]) + (sh[1][2] + sh[1][3]);
   zi = (sh[2][0] + sh[2][1]) + (sh[2][2] + sh[2][3]);
}

// face fields: unit c of point p on face f of block n at
// ((8 n + f) 6 + c) 64 + p; f = 2 mu the forward, 2 mu + 1 the backward face
__device__ inline size_t face_unit(int n, int f) { return ((size_t)n * 8 + f) * (6 * FPT); }

// acc += hopping terms into the point from outside the block, from the face
// fields of the neighbouring blocks nbn[0..7] (forward neighbours 2 mu,
// backward neighbours 2 mu + 1; SUB: a sub-block, negative where the face lies
// inside the block)
template <bool SUB = false, typename S>
__device__ inline void rb_pull(const RegBlock<S> &b, const float2 *W, const int *nbn, float2 *acc)
{
   // all loads first: a point lies on at most one of the faces of a
   // direction
   float2 h[4][6];
#pragma unroll
   for (int mu = 0; mu < 4; mu++)
   {
      const int x = b.coord(mu);
      if ((x == 3 && !(SUB && nbn[2 * mu] < 0)) || (x == 0 && !(SUB && nbn[2 * mu + 1] < 0)))
      {
         const size_t f = (x == 3) ? face_unit(nbn[2 * mu], 2 * mu + 1) : face_unit(nbn[2 * mu + 1], 2 * mu);
         const float2 *p = W + f + b.face_point(mu, !b.odd);
#pragma unroll
         for (int c = 0; c < 6; c++) h[mu][c] = p[c * FPT];
      }
   }
#pragma unroll
   for (int mu = 0; mu < 4; mu++)
   {
      const int x = b.coord(mu);
      if (x == 3 && !(SUB && nbn[2 * mu] < 0))
      {
         float2 c[6], u[9];
#pragma unroll
         for (int k = 0; k < 9; k++) u[k] = to_f2(b.u[mu][k]);
         su3_mul_f<false>(u, h[mu], c);
         su3_mul_f<false>(u, h[mu] + 3, c + 3);
         if (mu == 0) spin_expand_add<float2, 0, true>(c, c + 3, acc);
         if (mu == 1) spin_expand_add<float2, 1, true>(c, c + 3, acc);
         if (mu == 2) spin_expand_add<float2, 2, true>(c, c + 3, acc);
         if (mu == 3) spin_expand_add<float2, 3, true>(c, c + 3, acc);
      }
      else if (x == 0 && !(SUB && nbn[2 * mu + 1] < 0))
      {
         if (mu == 0) spin_expand_add<float2, 0, false>(h[mu], h[mu] + 3, acc);
         if (mu == 1) spin_expand_add<float2, 1, false>(h[mu], h[mu] + 3, acc);
         if (mu == 2) spin_expand_add<float2, 2, false>(h[mu], h[mu] + 3, acc);
         if (mu == 3) spin_expand_add<float2, 3, false>(h[mu], h[mu] + 3, acc);
      }
   }
}

// the block's face fields from its correction s0, towards the neighbours nbn
template <bool SUB = false, typename S>
__device__ inline void rb_push(const RegBlock<S> &b, const float2 *s0, float2 *W, int n, const int *nbn)
{
#pragma unroll
   for (int mu = 0; mu < 4; mu++)
   {
      const int x = b.coord(mu);
      if (x == 3 && !(SUB && nbn[2 * mu] < 0))
      {
         float2 h[6], c[6], u[9];
#pragma unroll
         for (int k = 0; k < 9; k++) u[k] = to_f2(b.u[mu][k]);
         if (mu == 0) weyl_project<0, false>(s0, h);
         if (mu == 1) weyl_project<1, false>(s0, h);
         if (mu == 2) weyl_project<2, false>(s0, h);
         if (mu == 3) weyl_project<3, false>(s0, h);
         su3_mul_f<true>(u, h, c);
         su3_mul_f<true>(u, h + 3, c + 3);
         float2 *p = W + face_unit(n, 2 * mu) + b.face_point(mu, b.odd);
#pragma unroll
         for (int k = 0; k < 6; k++) p[k * FPT] = c[k];
      }
      else if (x == 0 && !(SUB && nbn[2 * mu + 1] < 0))
      {
         float2 h[6];
         if (mu == 0) weyl_project<0, true>(s0, h);
         if (mu == 1) weyl_project<1, true>(s0, h);
         if (mu == 2) weyl_project<2, true>(s0, h);
         if (mu == 3) weyl_project<3, true>(s0, h);
         float2 *p = W + face_unit(n, 2 * mu + 1) + b.face_point(mu, b.odd);
#pragma unroll
         for (int k = 0; k < 6; k++) p[k * FPT] = h[k];
      }
   }
}

// point, links (S: FP32 or FP16) and boundary flag of the lane with point x;
// OUTER: only the links that leave the block
template <typename S, bool MASKED, bool OUTER = false>
__device__ inline void rb_load(const SArgs &a, const S *ub, int x, int gx, RegBlock<S> &b)
{
   const int i = x & (RBV / 2 - 1);
   b.odd = x >= RBV / 2;
   // the parity of t + x1 + x2 + x3 fixes the last bit of the point
   b.lex = 2 * i + (((i >> 5) ^ (i >> 3) ^ (i >> 1) ^ (int)b.odd) & 1);
   b.bp = MASKED && a.bnd[gx];
#pragma unroll
   for (int mu = 0; mu < 4; mu++)
   {
      if (OUTER && b.coord(mu) < 3) continue;
      const int J = b.odd ? gx - a.h : (a.nbr[(size_t)(2 * mu) * a.V + gx] & 0x7fffffff) - a.h;
      const S *up = ub + (size_t)(J >> 6) * (72 * SB) + (J & (SB - 1)) + (size_t)(9 * (b.odd ? 2 * mu : 2 * mu + 1)) * SB;
#pragma unroll
      for (int k = 0; k < 9; k++) b.u[mu][k] = up[k * SB];
   }
}

#ifndef OQH_SAP_WAVES16
#define OQH_SAP_WAVES16 2
#endif
#ifndef OQH_SAP_WAVES32
#define OQH_SAP_WAVES32 2
#endif
#ifndef OQH_SAP_MHALF
#define OQH_SAP_MHALF 1
#endif

// Two wavefronts per SIMD (256 registers per lane and at most 80 KiB of LDS
// per work-group): the FP16 variant keeps its links in FP16 registers and
// its Pauli matrices in LDS; the FP32 variant keeps the first Pauli matrix
// of each point in LDS and the second in registers (OQH_SAP_MHALF; with
// both in registers it needs 310 registers and runs one wavefront per SIMD,
// 1.50 against 0.82 ms per colour at 48^4).
// With isolv = 1 the two parities work at the same time on A_oo^-1 of the odd
// and A_ee of the even points, and one set of registers holds the value a
// point sends or the sum it receives.  A colour at 48^4 takes 0.86 ms and a
// cycle 2.0 ms; with a gather kernel for the faces (0.39 ms) and the two
// Pauli products one after the other it was 0.82 and 2.45 ms (FP16 storage at
// 32^3x64: 0.34 against 0.38 ms per colour).  Bound by both sides: 8200
// vector instructions per wave take 0.55 ms of issue, the 1150 bytes per
// point 0.55 ms, and two work-groups per CU overlap them only in part (0.1 ms
// per further MinRes step).  Swapping the parities' waves in every other
// work-group, delaying the second work-group of a CU and s_setprio changed
// nothing.
// MASKED: open-bc boundary points exist (bc != 3); without them the masking
// of boundary values is compiled out
template <int ISOLV, typename S, bool MASKED>
__global__ __launch_bounds__(RBV)
__attribute__((amdgpu_waves_per_eu(sizeof(S) == 4 ? OQH_SAP_WAVES16 : OQH_SAP_WAVES32)))
void k_sap_reg(SArgs a0, const S *u16, const S *sw16)
{
   __shared__ float2 LB[18 * RBV];  // hopping exchange (rb_hop)
   __shared__ double sh[3][4];      // block sums
   // FP16 variant: the Pauli matrices of the block live in LDS, and psi and
   // rho are FP16 spinors with per-site scales; FP32 variant with
   // OQH_SAP_MHALF: the first Pauli matrix of each point in LDS, the second
   // in registers
   constexpr bool MLDS = sizeof(S) == 4;
   constexpr bool MHALF = !MLDS && OQH_SAP_MHALF;
   constexpr int ML = MLDS ? 36 : (MHALF ? 18 : 0);  // units in LDS
   __shared__ S MS[ML ? ML : 1][RBV];
   // several sources: consecutive work-groups take the same block for
   // different sources, so its links and SW matrices come from the cache
   const int src = a0.nsrc ? (int)(blockIdx.x % a0.nsrc) : 0;
   const int bi = a0.nsrc ? (int)(blockIdx.x / a0.nsrc) : (int)blockIdx.x;
   SArgs a = a0;
   if (a0.nsrc)
   {
      a.psi = a0.pl[src];
      a.rho = a0.rl[src];
      a.wf = a0.wl[src];
   }
   const int x = threadIdx.x;
   const int n = a.n0 + bi;
   const int gx = a.imb[(size_t)n * RBV + x];
   const bool even = x < RBV / 2;
   // links and SW matrices: the FP32 fields, or their FP16 copies
   const S *ub = sizeof(S) == sizeof(float2) ? (const S *)a.u : u16;
   const S *swb = sizeof(S) == sizeof(float2) ? (const S *)a.sw : sw16;
   RegBlock<S> b;
   rb_load<S, MASKED>(a, ub, x, gx, b);
   S mreg[ML == 36 ? 1 : 36 - ML];
   {
      const S *m = swb + (size_t)(gx >> 6) * (36 * SB) + (gx & (SB - 1));
#pragma unroll
      for (int k = 0; k < 36; k++)
      {
         if (k < ML)
            MS[k][x] = m[k * SB];
         else
            mreg[k - ML] = m[k * SB];
      }
   }
   const S *mp0 = ML ? &MS[0][x] : mreg;
   const int mst0 = ML ? RBV : 1;
   const S *mp1 = ML == 36 ? &MS[18 % (ML ? ML : 1)][x] : mreg + (18 - ML);
   const int mst1 = ML == 36 ? RBV : 1;
   const float2 zero = make_float2(0.0f, 0.0f);
   float2 s0[12], s1[12], w[12];
   if (MLDS)
      load_h16(a.rho16, a.rsc, gx, s1);
   else
      load_spinor((const float2 *)a.rho, gx, s1);
   if (a.pull)
   {
      zero12(w);
      rb_pull(b, a.wf, a.nbn + 8 * (size_t)n, w);
#pragma unroll
      for (int c = 0; c < 12; c++) s1[c] = cadd(s1[c], cscale(w[c], 0.5f));
   }
#pragma unroll
   for (int c = 0; c < 12; c++)
   {
      s0[c] = zero;
      if (!ISOLV && b.bp) s1[c] = zero;
   }

   if (ISOLV)
   {
      // odd points: s1 = A_oo^-1 s1, then even points: s1 += 1/2 hops
      // (Dwoo_blk, Dweo_blk of sap.c:759-761)
      zero12(w);
      if (!even)
      {
         pauli_reg2(mp0, mst0, mp1, mst1, 0.0f, s1, w);
#pragma unroll
         for (int c = 0; c < 12; c++)
         {
            if (b.bp) w[c] = zero;
            s1[c] = w[c];
         }
      }
      rb_hop<0>(b, w, w, LB);
      if (even)
      {
#pragma unroll
         for (int c = 0; c < 12; c++) s1[c] = b.bp ? zero : cadd(s1[c], cscale(w[c], 0.5f));
      }
   }

   // minimal residual steps (blk_solv.c:1117-1186): w = D s1
   for (int imr = 0; imr < a.nmr; imr++)
   {
      if (ISOLV)
      {
         // odd: v = -1/2 hops of s1_e, even: v = s1; w = A_oo^-1 v and
         // A_ee v at once; even: w += 1/2 hops of w_o
         zero12(w);
         rb_hop<1>(b, s1, w, LB);
         float2 o[12];
#pragma unroll
         for (int c = 0; c < 12; c++) w[c] = even ? s1[c] : cscale(w[c], -0.5f);
         pauli_reg2(mp0, mst0, mp1, mst1, even ? a.mu : 0.0f, w, o);
         const float f = even ? 2.0f : 1.0f;
#pragma unroll
         for (int c = 0; c < 12; c++) w[c] = (b.bp && !even) ? zero : cscale(o[c], f);
         rb_hop<0>(b, w, w, LB);
#pragma unroll
         for (int c = 0; c < 12; c++) w[c] = (b.bp && even) ? zero : cscale(w[c], 0.5f);
      }
      else
      {
         float2 o[12];
         pauli_reg2(mp0, mst0, mp1, mst1, even ? a.mu : a.muo, s1, o);
         // the accumulators start from -2 A s1, so that w = -1/2 their sum
#pragma unroll
         for (int c = 0; c < 12; c++) w[c] = cscale(o[c], -2.0f);
         rb_hop<1>(b, s1, w, LB);
         rb_hop<0>(b, s1, w, LB);
#pragma unroll
         for (int c = 0; c < 12; c++) w[c] = b.bp ? zero : cscale(w[c], -0.5f);
      }
      double rr, zr, zi;
      rb_sums(ISOLV ? even : true, w, s1, sh, rr, zr, zi);
      float r = (float)rr;
      if (r < 2.0f * FLT_MIN) break;
      r = 1.0f / r;
      float2 z = make_float2((float)zr * r, (float)zi * r), mz = make_float2(-z.x, -z.y);
      if (!ISOLV || even)
      {
#pragma unroll
         for (int c = 0; c < 12; c++)
         {
            s0[c] = cmac(s0[c], z, s1[c]);
            s1[c] = cmac(s1[c], mz, w[c]);
         }
      }
   }

   if (ISOLV)
   {
      // odd solution s0_o = s1_o - A_oo^-1 (-1/2 hops of s0_e) (Dwoe_blk, Dwoo_blk)
      zero12(w);
      rb_hop<1>(b, s0, w, LB);
      if (!even)
      {
         float2 o[12];
#pragma unroll
         for (int c = 0; c < 12; c++) w[c] = cscale(w[c], -0.5f);
         pauli_reg2(mp0, mst0, mp1, mst1, 0.0f, w, o);
#pragma unroll
         for (int c = 0; c < 12; c++)
         {
            if (b.bp) o[c] = zero;
            s0[c] = csub(s1[c], o[c]);
         }
      }
   }

   rb_push(b, s0, a.wf, n, a.nbn + 8 * (size_t)n);
   if (a.pz)
   {
#pragma unroll
      for (int c = 0; c < 12; c++) w[c] = s0[c];
   }
   else
   {
      if (MLDS)
         load_h16(a.psi16, a.psc, gx, w);
      else
         load_spinor((const float2 *)a.psi, gx, w);
#pragma unroll
      for (int c = 0; c < 12; c++) w[c] = cadd(w[c], s0[c]);
   }
   if (MLDS)
      store_h16(a.psi16, a.psc, gx, w);
   else
      store_spinor(a.psi, gx, w);
   if (ISOLV && !even)
   {
      // odd residual -i mu gamma5 s0 (update_flds1) or 0 (eoflg, update_flds2)
      float m = a.eoflg ? 0.0f : a.mu;
#pragma unroll
      for (int c = 0; c < 12; c++)
      {
         float cm = (c < 6) ? -m : m;
         s1[c] = make_float2(-cm * s0[c].y, cm * s0[c].x);
      }
   }
   if (MLDS)
      store_h16(a.rho16, a.rsc, gx, s1);
   else
      store_spinor(a.rho, gx, s1);
}

// rho += hopping terms from the face fields of the neighbouring blocks for
// the 4^4 blocks or sub-blocks (points imb) from n0 on: completes the residual
// after the last block solves
template <typename S>
__global__ __launch_bounds__(RBV) void k_sap_complete(SArgs a0, const int *imb, const S *u16)
{
   constexpr bool H = sizeof(S) == 4;
   const int src = a0.nsrc ? (int)(blockIdx.x % a0.nsrc) : 0;
   const int bi = a0.nsrc ? (int)(blockIdx.x / a0.nsrc) : (int)blockIdx.x;
   SArgs a = a0;
   if (a0.nsrc)
   {
      a.rho = a0.rl[src];
      a.wf = a0.wl[src];
   }
   const int n = a.n0 + bi;
   const int gx = imb[(size_t)n * RBV + threadIdx.x];
   RegBlock<S> b;
   rb_load<S, false, true>(a, H ? u16 : (const S *)a.u, threadIdx.x, gx, b);
   float2 r[12], acc[12];
   if (H)
      load_h16(a.rho16, a.rsc, gx, r);
   else
      load_spinor((const float2 *)a.rho, gx, r);
   zero12(acc);
   rb_pull<true>(b, a.wf, a.nbn + 8 * (size_t)n, acc);
#pragma unroll
   for (int c = 0; c < 12; c++) r[c] = cadd(r[c], cscale(acc[c], 0.5f));
   if (H)
      store_h16(a.rho16, a.rsc, gx, r);
   else
      store_spinor(a.rho, gx, r);
}

#ifndef OQH_FACE_GROUP
#define OQH_FACE_GROUP 4
#endif

// ---------------------------------------------------------------------------
// the Schwarz sweep with a block shared by several work-groups (block sizes
// that are multiples of 4, FP32)
//
// The block is cut into sub-blocks of 4^4 points, each held in the registers of
// one work-group as in k_sap_reg.  In every hopping pass the work-groups of a
// block pass the Weyl fields on their common faces (those of rb_push, the
// points of one parity) through global memory, and for every MinRes step
// their shares of the block sums.
//
// Which sub-block a work-group takes is decided by a ticket drawn when it
// starts to run, block by block, so at any time all but the last block begun
// have all their work-groups running and can finish; the last one gets its
// missing work-groups as the others end.  A block needs only as many
// work-groups running at once as it has sub-blocks (at most CLMAX, far fewer
// than the device holds), and no wait depends on the order in which
// work-groups are started.  Waits are bounded all the same: a wavefront that
// has polled Lib::sap_polls times gives up waiting for good, the kernel ends
// with incomplete sums and faces, and the call that launched it reports the
// error once it has waited for the stream (sap_gave_up).
//
// The exchanged values are written and read with relaxed atomics of device
// scope; a work-group counts itself in after its writes have completed.  Two
// exchange buffers alternate: who writes the one of pass k + 2 has seen
// everybody arrive in pass k + 1, that is, done with reading pass k.
//
// Per cycle (us, isolv = 1, nmr = 4; k_sap_cluster / k_sap_lds or, for 8^4,
// k_sap_blocks): 8^4 blocks on 16^4 213 / 1436, on 32^4 1090 / 2605, on 32^3x64
// 2150 / 3700; 16x8^3 on 32x16^3 251 / 3050; 8x4^3 on 16x8^3 132 / 146, on 32^3x16
// 384 / 446; 8^2x4^2 on 16^2x8^2 153 / 203, on 32^3x16 430 / 463 (a call of sap()
// takes 8 more, for its wait).  Bound by the 14 exchanges of a block solve, about
// 3.5 us each (write, count, poll, read).  With the counters of all blocks in
// one line they took 20 us (8^4 on 32^4: 3400).
// ---------------------------------------------------------------------------

// psi += s0 (or = s0 for pz), rho = s1, correction s0 (if asked for) of one point
template <bool COR> __device__ inline void lds_store(const SArgs &a, int gx, const float2 *s0, const float2 *s1)
{
   float2 p[12];
   if (a.pz)
   {
#pragma unroll
      for (int c = 0; c < 12; c++) p[c] = s0[c];
   }
   else
   {
      load_spinor((const float2 *)a.psi, gx, p);
#pragma unroll
      for (int c = 0; c < 12; c++) p[c] = cadd(p[c], s0[c]);
   }
   store_spinor(a.psi, gx, p);
   store_spinor(a.rho, gx, s1);
   if (COR) store_spinor(a.s0g, gx, s0);
}

constexpr int CLMAX = 64;         // sub-blocks of a block
constexpr int CLPAD = 64;         // distance of the counters: a line each
constexpr int CLSLEEP = 8;        // pause between polls, 64 clocks each

struct ClArgs
{
   int ns;                     // sub-blocks per block
   const int *imb4;            // [nb][ns][RBV] points of the sub-blocks
   const int *nbs;             // [ns][8] neighbouring sub-block in the block or -1
   unsigned *ticket, *count;   // [CLPAD], [nbh][CLPAD]: zero at the start
   unsigned long long *x;      // [2][nbh][ns] face fields
   unsigned long long *sums;   // [nbh][ns][4]
   size_t xlen;                // length of one of the two
   int polls;                  // polls of a wait
   int *dead;                  // set if a wait was given up (host memory)
};

__device__ inline void cl_store(unsigned long long *p, unsigned long long v)
{
   __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline unsigned long long cl_load(const unsigned long long *p)
{
   return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline unsigned long long cl_bits(float2 v)
{
   return ((unsigned long long)__float_as_uint(v.y) << 32) | __float_as_uint(v.x);
}
__device__ inline float2 cl_value(unsigned long long b)
{
   return make_float2(__uint_as_float((unsigned)b), __uint_as_float((unsigned)(b >> 32)));
}

struct ClState
{
   int bi, sub;       // block of the colour, sub-block
   unsigned phase;    // arrivals so far
   int buf;           // exchange buffer of the next pass
   bool gone;         // a wait was given up
};

// Arrivals are counted in wavefronts, two per work-group and phase: in a hopping
// pass those of the source points, for the sums twice the first.

// the wavefront's writes and reads are done: count it in n times
__device__ inline void cl_arrive(const ClArgs &q, const ClState &st, unsigned n)
{
   asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
   if ((threadIdx.x & 63) == 0)
      __hip_atomic_fetch_add(q.count + (size_t)st.bi * CLPAD, n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// until all work-groups of the block have arrived (the wavefront as a whole)
__device__ inline void cl_wait(const ClArgs &q, ClState &st)
{
   const unsigned want = 2u * st.phase * (unsigned)q.ns;
   int k = 0;
   while (!st.gone && __hip_atomic_load(q.count + (size_t)st.bi * CLPAD, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < want)
   {
      if (++k >= q.polls)
      {
         st.gone = true;
         __hip_atomic_store(q.dead, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      }
      __builtin_amdgcn_s_sleep(CLSLEEP);
   }
   asm volatile("" ::: "memory");
}

// the face values of the lane (a source) for the neighbouring sub-blocks nb
template <typename S>
__device__ inline void cl_push(const ClArgs &q, const ClState &st, const RegBlock<S> &b, const int *nb, const float2 *s)
{
   unsigned long long *X = q.x + st.buf * q.xlen;
   const int n = st.bi * q.ns + st.sub;
#pragma unroll
   for (int mu = 0; mu < 4; mu++)
   {
      const int x = b.coord(mu);
      if (x == 3 && nb[2 * mu] >= 0)
      {
         float2 h[6], c[6], u[9];
#pragma unroll
         for (int k = 0; k < 9; k++) u[k] = to_f2(b.u[mu][k]);
         if (mu == 0) weyl_project<0, false>(s, h);
         if (mu == 1) weyl_project<1, false>(s, h);
         if (mu == 2) weyl_project<2, false>(s, h);
         if (mu == 3) weyl_project<3, false>(s, h);
         su3_mul_f<true>(u, h, c);
         su3_mul_f<true>(u, h + 3, c + 3);
         unsigned long long *p = X + face_unit(n, 2 * mu) + b.face_point(mu, b.odd);
#pragma unroll
         for (int k = 0; k < 6; k++) cl_store(p + k * FPT, cl_bits(c[k]));
      }
      else if (x == 0 && nb[2 * mu + 1] >= 0)
      {
         float2 h[6];
         if (mu == 0) weyl_project<0, true>(s, h);
         if (mu == 1) weyl_project<1, true>(s, h);
         if (mu == 2) weyl_project<2, true>(s, h);
         if (mu == 3) weyl_project<3, true>(s, h);
         unsigned long long *p = X + face_unit(n, 2 * mu + 1) + b.face_point(mu, b.odd);
#pragma unroll
         for (int k = 0; k < 6; k++) cl_store(p + k * FPT, cl_bits(h[k]));
      }
   }
}

// w += the terms from the neighbouring sub-blocks
template <typename S>
__device__ inline void cl_pull(const ClArgs &q, const ClState &st, const RegBlock<S> &b, const int *nb, float2 *w)
{
   const unsigned long long *X = q.x + st.buf * q.xlen;
#pragma unroll
   for (int mu = 0; mu < 4; mu++)
   {
      const int x = b.coord(mu);
      const bool fw = x == 3 && nb[2 * mu] >= 0, bw = x == 0 && nb[2 * mu + 1] >= 0;
      if (fw || bw)
      {
         const size_t f = fw ? face_unit(st.bi * q.ns + nb[2 * mu], 2 * mu + 1)
                             : face_unit(st.bi * q.ns + nb[2 * mu + 1], 2 * mu);
         const unsigned long long *p = X + f + b.face_point(mu, !b.odd);
         float2 h[6];
#pragma unroll
         for (int c = 0; c < 6; c++) h[c] = cl_value(cl_load(p + c * FPT));
         if (fw)
         {
            float2 c[6], u[9];
#pragma unroll
            for (int k = 0; k < 9; k++) u[k] = to_f2(b.u[mu][k]);
            su3_mul_f<false>(u, h, c);
            su3_mul_f<false>(u, h + 3, c + 3);
            if (mu == 0) spin_expand_add<float2, 0, true>(c, c + 3, w);
            if (mu == 1) spin_expand_add<float2, 1, true>(c, c + 3, w);
            if (mu == 2) spin_expand_add<float2, 2, true>(c, c + 3, w);
            if (mu == 3) spin_expand_add<float2, 3, true>(c, c + 3, w);
         }
         else
         {
            if (mu == 0) spin_expand_add<float2, 0, false>(h, h + 3, w);
            if (mu == 1) spin_expand_add<float2, 1, false>(h, h + 3, w);
            if (mu == 2) spin_expand_add<float2, 2, false>(h, h + 3, w);
            if (mu == 3) spin_expand_add<float2, 3, false>(h, h + 3, w);
         }
      }
   }
}

// hopping pass over the whole block: the terms across the sub-blocks' faces
// travel while the work-group forms its own
template <typename S> struct ClHook
{
   const ClArgs &q;
   ClState &st;
   const RegBlock<S> &b;
   const int *nb;
   const float2 *src;
   float2 *w;
   __device__ void put() const { cl_push(q, st, b, nb, src); }
   __device__ void sent() const { cl_arrive(q, st, 1); }
   __device__ void take() const
   {
      cl_wait(q, st);
      cl_pull(q, st, b, nb, w);
   }
};

template <int OUT, typename S>
__device__ inline void cl_hop(const ClArgs &q, ClState &st, const RegBlock<S> &b, const int *nb, const float2 *src,
                              float2 *w, float2 *lb)
{
   st.phase++;
   rb_hop<OUT>(b, src, w, lb, ClHook<S>{q, st, b, nb, src, w});
   st.buf ^= 1;
}

// sums over the block from the work-groups' shares
// (sh may be written again only after another barrier has been passed)
__device__ inline void cl_sums(const ClArgs &q, ClState &st, double *sh, double &rr, double &zr, double &zi)
{
   unsigned long long *p = q.sums + (size_t)st.bi * q.ns * 4;
   st.phase++;
   if (threadIdx.x < 64)
   {
      const int l = threadIdx.x;
      if (l == 0)
      {
         cl_store(p + 4 * st.sub, (unsigned long long)__double_as_longlong(rr));
         cl_store(p + 4 * st.sub + 1, (unsigned long long)__double_as_longlong(zr));
         cl_store(p + 4 * st.sub + 2, (unsigned long long)__double_as_longlong(zi));
      }
      cl_arrive(q, st, 2);
      cl_wait(q, st);
      double v[3] = {0.0, 0.0, 0.0};
      if (l < q.ns)
      {
#pragma unroll
         for (int k = 0; k < 3; k++) v[k] = __longlong_as_double((long long)cl_load(p + 4 * l + k));
      }
#pragma unroll
      for (int k = 0; k < 3; k++) v[k] = wave_sum63(v[k]);
      if (l == 63)
      {
         sh[0] = v[0];
         sh[1] = v[1];
         sh[2] = v[2];
      }
   }
   __syncthreads();
   rr = sh[0];
   zr = sh[1];
   zi = sh[2];
}

__global__ void k_cl_reset(unsigned *p, int n)
{
   const int k = blockIdx.x * 256 + threadIdx.x;
   if (k < n) p[(size_t)k * CLPAD] = 0;
}

template <int ISOLV, bool MASKED>
__global__ __launch_bounds__(RBV) __attribute__((amdgpu_waves_per_eu(2))) void k_sap_cluster(SArgs a, ClArgs q)
{
   __shared__ float2 LB[18 * RBV];  // hopping exchange (rb_hop)
   __shared__ float2 MS[18][RBV];   // first Pauli matrix of each point
   __shared__ double sh[3][4], shc[3];
   __shared__ int tk, nb[8];
   const int x = threadIdx.x;
   if (x == 0) tk = (int)__hip_atomic_fetch_add(q.ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
   __syncthreads();
   ClState st;
   st.bi = tk / q.ns;
   st.sub = tk % q.ns;
   st.phase = 0;
   st.buf = 0;
   st.gone = false;
   if (x < 8) nb[x] = q.nbs[8 * st.sub + x];
   const int gx = q.imb4[((size_t)(a.n0 + st.bi) * q.ns + st.sub) * RBV + x];
   const bool even = x < RBV / 2;
   RegBlock<float2> b;
   rb_load<float2, MASKED>(a, a.u, x, gx, b);
   float2 mreg[18];
   {
      const float2 *m = a.sw + (size_t)(gx >> 6) * (36 * SB) + (gx & (SB - 1));
#pragma unroll
      for (int k = 0; k < 18; k++)
      {
         MS[k][x] = m[k * SB];
         mreg[k] = m[(18 + k) * SB];
      }
   }
   const float2 zero = make_float2(0.0f, 0.0f);
   float2 s0[12], s1[12], w[12], o[12];
   load_spinor((const float2 *)a.rho, gx, s1);
   const int sb = (a.n0 + st.bi) * q.ns + st.sub;  // number of the sub-block
   if (a.pull)
   {
      zero12(w);
      rb_pull<true>(b, a.wf, a.nbn + 8 * (size_t)sb, w);
#pragma unroll
      for (int c = 0; c < 12; c++) s1[c] = cadd(s1[c], cscale(w[c], 0.5f));
   }
#pragma unroll
   for (int c = 0; c < 12; c++)
   {
      s0[c] = zero;
      if (!ISOLV && b.bp) s1[c] = zero;
   }
   __syncthreads();

   if (ISOLV)
   {
      // odd points: s1 = A_oo^-1 s1, then even points: s1 += 1/2 hops
      zero12(w);
      if (!even)
      {
         pauli_reg2(&MS[0][x], RBV, mreg, 1, 0.0f, s1, w);
#pragma unroll
         for (int c = 0; c < 12; c++)
         {
            if (b.bp) w[c] = zero;
            s1[c] = w[c];
         }
      }
      cl_hop<0>(q, st, b, nb, w, w, LB);
      if (even)
      {
#pragma unroll
         for (int c = 0; c < 12; c++) s1[c] = b.bp ? zero : cadd(s1[c], cscale(w[c], 0.5f));
      }
   }

   // minimal residual steps: w = D s1 (k_sap_reg)
   for (int imr = 0; imr < a.nmr; imr++)
   {
      if (ISOLV)
      {
         zero12(w);
         cl_hop<1>(q, st, b, nb, s1, w, LB);
#pragma unroll
         for (int c = 0; c < 12; c++) w[c] = even ? s1[c] : cscale(w[c], -0.5f);
         pauli_reg2(&MS[0][x], RBV, mreg, 1, even ? a.mu : 0.0f, w, o);
         const float f = even ? 2.0f : 1.0f;
#pragma unroll
         for (int c = 0; c < 12; c++) w[c] = (b.bp && !even) ? zero : cscale(o[c], f);
         cl_hop<0>(q, st, b, nb, w, w, LB);
#pragma unroll
         for (int c = 0; c < 12; c++) w[c] = (b.bp && even) ? zero : cscale(w[c], 0.5f);
      }
      else
      {
         // unlike in k_sap_reg the hops are summed by themselves, which is more
         // precise than k_sap_blocks was (five cycles of 8^4 blocks on 16^4
         // against FP64: 1.09e-7 for 1.16e-7; started from -2 A s1 1.20e-7) and
         // costs 3 % of a cycle
         zero12(w);
         cl_hop<1>(q, st, b, nb, s1, w, LB);
         cl_hop<0>(q, st, b, nb, s1, w, LB);
#pragma unroll
         for (int c = 0; c < 12; c++) w[c] = cscale(w[c], -0.5f);
         pauli_reg2<true>(&MS[0][x], RBV, mreg, 1, even ? a.mu : a.muo, s1, w);
         if (b.bp) zero12(w);
      }
      double rr, zr, zi;
      rb_sums(ISOLV ? even : true, w, s1, sh, rr, zr, zi);
      cl_sums(q, st, shc, rr, zr, zi);
      float r = (float)rr;
      if (r < 2.0f * FLT_MIN) break;
      r = 1.0f / r;
      const float2 z = make_float2((float)zr * r, (float)zi * r), mz = make_float2(-z.x, -z.y);
      if (!ISOLV || even)
      {
#pragma unroll
         for (int c = 0; c < 12; c++)
         {
            s0[c] = cmac(s0[c], z, s1[c]);
            s1[c] = cmac(s1[c], mz, w[c]);
         }
      }
   }

   if (ISOLV)
   {
      // odd solution s0_o = s1_o - A_oo^-1 (-1/2 hops of s0_e)
      zero12(w);
      cl_hop<1>(q, st, b, nb, s0, w, LB);
      if (!even)
      {
#pragma unroll
         for (int c = 0; c < 12; c++) w[c] = cscale(w[c], -0.5f);
         pauli_reg2(&MS[0][x], RBV, mreg, 1, 0.0f, w, o);
         const float m = a.eoflg ? 0.0f : a.mu;
#pragma unroll
         for (int c = 0; c < 12; c++)
         {
            if (b.bp) o[c] = zero;
            s0[c] = csub(s1[c], o[c]);
            // odd residual -i mu gamma5 s0 (update_flds1) or 0 (eoflg, update_flds2)
            const float cm = (c < 6) ? -m : m;
            s1[c] = make_float2(-cm * s0[c].y, cm * s0[c].x);
         }
      }
   }
   rb_push<true>(b, s0, a.wf, sb, a.nbn + 8 * (size_t)sb);
   lds_store<false>(a, gx, s0, s1);
}

// ---------------------------------------------------------------------------
// the Schwarz sweep with the block's spinors on the chip (blocks of up to
// 1365 points whose sizes are not all multiples of 4, FP32)
//
// Lane i of the work-group owns the even point i and the odd point bh + i of
// the block.  The block fields s0, s1 stay in its registers; the source of a
// hopping pass, one parity, lies in LDS (96 bytes per point), where the output
// lanes gather all eight neighbours.  Links and SW matrices are too many for
// the chip (600 bytes per point) and are streamed, each once per pass and
// parity: 864 bytes per point and MinRes step, against 1350 and more of
// k_sap_blocks, whose fields also pass through global memory.
// Per cycle (us, k_sap_lds / k_sap_blocks, nmr = 4): 4x6^3 blocks on 8x12^3
// 229 / 445, on 16x24^3 348 / 675; 6^4 on 12^4 351 / 622, on 36^2x24^2 1359 /
// 2119 (12 wavefronts, 168 registers, 21 spilled).
// ---------------------------------------------------------------------------

constexpr int BLV_MAX = 1365;  // points of a block, two per lane: 64 KiB of LDS

// acc += hopping terms into block point i (global point gx) of parity ODD
// from the values F of the other parity
template <int MU, bool FWD, bool ODD>
__device__ inline void lds_hop_one(const SArgs &a, const int *imb, const float2 *F, int i, int gx, float2 *acc)
{
   const int j = a.bnb[(2 * MU + (FWD ? 0 : 1)) * a.bvol + i];
   if (j >= a.bvol) return;
   const float2 *up = ODD ? link_ptr(a.u, gx - a.h, FWD ? 2 * MU : 2 * MU + 1)
                          : link_ptr(a.u, imb[j] - a.h, FWD ? 2 * MU + 1 : 2 * MU);
   float2 u[9], sp[12], h[6], c[6];
#pragma unroll
   for (int k = 0; k < 9; k++) u[k] = up[k * SB];
   const float2 *f = F + (ODD ? j : j - a.bh);
#pragma unroll
   for (int k = 0; k < 12; k++) sp[k] = f[k * a.bh];
   spin_project<float2, MU, FWD>(sp, h, h + 3);
   su3_mul_f<!FWD>(u, h, c);
   su3_mul_f<!FWD>(u, h + 3, c + 3);
   spin_expand_add<float2, MU, FWD>(c, c + 3, acc);
}

// the loads of a direction stay within it: the compiler would otherwise move
// those of all eight ahead and spill the block fields
template <bool ODD, bool WIDE>
__device__ inline void lds_hop(const SArgs &a, const int *imb, const float2 *F, int i, int gx, float2 *acc)
{
   zero12(acc);
#define OQH_LDS_HOP(MU)                                                \
   lds_hop_one<MU, true, ODD>(a, imb, F, i, gx, acc);                  \
   if (!WIDE) __builtin_amdgcn_sched_barrier(0);                       \
   lds_hop_one<MU, false, ODD>(a, imb, F, i, gx, acc);                 \
   __builtin_amdgcn_sched_barrier(0);
   OQH_LDS_HOP(0)
   OQH_LDS_HOP(1)
   OQH_LDS_HOP(2)
   OQH_LDS_HOP(3)
#undef OQH_LDS_HOP
}

__device__ inline void lds_put(float2 *F, int bh, int i, const float2 *v)
{
#pragma unroll
   for (int c = 0; c < 12; c++) F[c * bh + i] = v[c];
}

// o = (A + i mu gamma5) v at global point gx, one Weyl half after the other
__device__ inline void lds_pauli(const SArgs &a, int gx, float mu, const float2 *v, float2 *o)
{
   const float2 *m = a.sw + (size_t)(gx >> 6) * (36 * SB) + (gx & (SB - 1));
#pragma unroll
   for (int hh = 0; hh < 2; hh++)
   {
      float2 q[18];
#pragma unroll
      for (int k = 0; k < 18; k++) q[k] = m[(18 * hh + k) * SB];
      pauli_half_reg(q, hh ? -mu : mu, v + 6 * hh, o + 6 * hh);
      __builtin_amdgcn_sched_barrier(0);
   }
}

// |s2|^2 and (s2, s1) of a point, added as in blk_mres_dev
__device__ inline void point_sums(const float2 *s2, const float2 *s1, double &rr, double &zr, double &zi)
{
#pragma unroll
   for (int k = 0; k < 4; k++)
   {
      float nr = 0.0f, pr = 0.0f, pi = 0.0f;
#pragma unroll
      for (int c = 0; c < 3; c++)
      {
         float2 u = s2[3 * k + c], v = s1[3 * k + c];
         nr += u.x * u.x + u.y * u.y;
         pr += u.x * v.x + u.y * v.y;
         pi += u.x * v.y - u.y * v.x;
      }
      rr += (double)nr;
      zr += (double)pr;
      zi += (double)pi;
   }
}

template <int ISOLV, int TPB, bool MASKED>
__global__ __launch_bounds__(TPB) __attribute__((amdgpu_waves_per_eu(TPB <= 512 ? 2 : 3))) void k_sap_lds(SArgs a)
{
   extern __shared__ float2 F[];  // [12][bh]
   constexpr bool WIDE = TPB <= 512 && ISOLV;
   const int n = a.n0 + blockIdx.x, bh = a.bh, i = threadIdx.x;
   const int *imb = a.imb + (size_t)n * a.bvol;
   const bool own = i < bh;  // lanes without points take part in the barriers
   int ge = imb[own ? i : 0], go = imb[own ? bh + i : bh];
   const bool be = MASKED && a.bnd[ge], bo = MASKED && a.bnd[go];
   const float2 zero = make_float2(0.0f, 0.0f);
   float2 s0[12], s1[12], w[12];
   // ISOLV = 0: the odd point's fields
   float2 t0[ISOLV ? 1 : 12], t1[ISOLV ? 1 : 12], tw[ISOLV ? 1 : 12];
   zero12(s0);
   zero12(s1);
   if (ISOLV)
   {
      // odd points: A_oo^-1 rho, then even points: s1 = rho + 1/2 hops
      if (own)
      {
         float2 o[12];
         load_spinor((const float2 *)a.rho, go, w);
         lds_pauli(a, go, 0.0f, w, o);
#pragma unroll
         for (int c = 0; c < 12; c++) w[c] = bo ? zero : o[c];
         lds_put(F, bh, i, w);
         load_spinor((const float2 *)a.rho, ge, s1);
      }
      __syncthreads();
      if (own)
      {
         lds_hop<false, WIDE>(a, imb, F, i, ge, w);
#pragma unroll
         for (int c = 0; c < 12; c++) s1[c] = be ? zero : cadd(s1[c], cscale(w[c], 0.5f));
      }
      __syncthreads();
   }
   else if (own)
   {
      load_spinor((const float2 *)a.rho, ge, s1);
      load_spinor((const float2 *)a.rho, go, t1);
      zero12(t0);
#pragma unroll
      for (int c = 0; c < 12; c++)
      {
         if (be) s1[c] = zero;
         if (bo) t1[c] = zero;
      }
   }

   // minimal residual steps (blk_solv.c:1117-1186): w = D s1
   for (int imr = 0; imr < a.nmr; imr++)
   {
      double rr = 0.0, zr = 0.0, zi = 0.0;
      // links and matrices are read again in every step: without this the
      // compiler loads them once, before the loop, and spills them
      asm volatile("" : "+v"(ge), "+v"(go), "+s"(a.bnb));
      if (own) lds_put(F, bh, i, s1);
      __syncthreads();
      if (ISOLV)
      {
         float2 o[12];
         if (own)
         {
            lds_hop<true, WIDE>(a, imb, F, bh + i, go, w);
#pragma unroll
            for (int c = 0; c < 12; c++) w[c] = cscale(w[c], -0.5f);
            lds_pauli(a, go, 0.0f, w, o);
#pragma unroll
            for (int c = 0; c < 12; c++) o[c] = bo ? zero : o[c];
         }
         __syncthreads();
         if (own) lds_put(F, bh, i, o);
         __syncthreads();
         if (own)
         {
            lds_hop<false, WIDE>(a, imb, F, i, ge, w);
            lds_pauli(a, ge, a.mu, s1, o);
#pragma unroll
            for (int c = 0; c < 12; c++) w[c] = be ? zero : cadd(o[c], cscale(w[c], 0.5f));
            point_sums(w, s1, rr, zr, zi);
         }
      }
      else
      {
         float2 o[12];
         if (own)
         {
            lds_hop<true, WIDE>(a, imb, F, bh + i, go, tw);
            lds_pauli(a, go, a.muo, t1, o);
#pragma unroll
            for (int c = 0; c < 12; c++) tw[c] = bo ? zero : cadd(o[c], cscale(tw[c], -0.5f));
            point_sums(tw, t1, rr, zr, zi);
         }
         __syncthreads();
         if (own) lds_put(F, bh, i, t1);
         __syncthreads();
         if (own)
         {
            lds_hop<false, WIDE>(a, imb, F, i, ge, w);
            lds_pauli(a, ge, a.mu, s1, o);
#pragma unroll
            for (int c = 0; c < 12; c++) w[c] = be ? zero : cadd(o[c], cscale(w[c], -0.5f));
            point_sums(w, s1, rr, zr, zi);
         }
      }
      wg_sum3(rr, zr, zi, TPB);
      float r = (float)rr;
      if (r < 2.0f * FLT_MIN) break;
      r = 1.0f / r;
      const float2 z = make_float2((float)zr * r, (float)zi * r), mz = make_float2(-z.x, -z.y);
      if (own)
      {
#pragma unroll
         for (int c = 0; c < 12; c++)
         {
            s0[c] = cmac(s0[c], z, s1[c]);
            s1[c] = cmac(s1[c], mz, w[c]);
            if (!ISOLV)
            {
               t0[c] = cmac(t0[c], z, t1[c]);
               t1[c] = cmac(t1[c], mz, tw[c]);
            }
         }
      }
   }

   if (ISOLV)
   {
      // odd solution A_oo^-1 (rho_o + 1/2 hops of s0_e), odd residual
      // -i mu gamma5 s0 (update_flds1) or 0 (eoflg, update_flds2)
      __syncthreads();
      if (own) lds_put(F, bh, i, s0);
      __syncthreads();
      if (!own) return;
      lds_store<true>(a, ge, s0, s1);
      float2 v[12], o[12];
      lds_hop<true, WIDE>(a, imb, F, bh + i, go, w);
      load_spinor((const float2 *)a.rho, go, v);
#pragma unroll
      for (int c = 0; c < 12; c++) v[c] = cadd(v[c], cscale(w[c], 0.5f));
      lds_pauli(a, go, 0.0f, v, o);
      const float m = a.eoflg ? 0.0f : a.mu;
#pragma unroll
      for (int c = 0; c < 12; c++)
      {
         if (bo) o[c] = zero;
         const float cm = (c < 6) ? -m : m;
         v[c] = make_float2(-cm * o[c].y, cm * o[c].x);
      }
      lds_store<true>(a, go, o, v);
   }
   else if (own)
   {
      lds_store<true>(a, ge, s0, s1);
      lds_store<true>(a, go, t0, t1);
   }
}

// rho(y) -= hopping terms into y from the block corrections of the
// neighbouring blocks, for the face points y of the blocks of one colour
// (the blocks of k_sap_lds and k_sap_blocks)
__global__ __launch_bounds__(256) void k_sap_faces(SArgs a, const int *face, const unsigned char *fmask, int nf)
{
   int k = blockIdx.x * 256 + threadIdx.x;
   if (k >= nf) return;
   int y = face[k];
   int m = fmask[k];
   float2 acc[12], h0[3], h1[3], c0[3], c1[3];
   zero12(acc);
   int odd = y >= a.h;
   // a point of a block of width >= 2 lies on at most one of the faces -mu,
   // +mu: the loads of each direction are issued for all lanes at once (one
   // neighbour and one link per direction and lane), OQH_FACE_GROUP
   // directions ahead of the arithmetic, which adds the terms in the order
   // mu = 0..3 (forward before backward)
   constexpr int FG = OQH_FACE_GROUP;
   for (int m0 = 0; m0 < 4; m0 += FG)
   {
      float2 sp[FG][12], u[FG][9];
#pragma unroll
      for (int j = 0; j < FG; j++)
      {
         const int MU = m0 + j;
         const bool fw = m & (1 << (2 * MU)), bw = m & (2 << (2 * MU));
         if (fw || bw)
         {
            const int dir = fw ? 2 * MU : 2 * MU + 1;
            const int x = a.nbr[(size_t)dir * a.V + y] & 0x7fffffff;
            load_spinor((const float2 *)a.s0g, x, sp[j]);
            // forward: U(y, mu) (odd y) or U(x, mu) stored at the odd x
            const int J = odd ? y - a.h : x - a.h;
            const int l = (odd == fw) ? 2 * MU : 2 * MU + 1;
            const float2 *up = link_ptr(a.u, J, l);
#pragma unroll
            for (int q = 0; q < 9; q++) u[j][q] = up[q * SB];
         }
      }
#pragma unroll
      for (int j = 0; j < FG; j++)
      {
         const int MU = m0 + j;
         const bool fw = m & (1 << (2 * MU)), bw = m & (2 << (2 * MU));
#define OQH_FACE_TERM(M)                                                               \
   if (MU == M)                                                                       \
   {                                                                                  \
      if (fw)                                                                         \
      {                                                                               \
         spin_project<float2, M, true>(sp[j], h0, h1);                                \
         su3_mul_f<false>(u[j], h0, c0);                                              \
         su3_mul_f<false>(u[j], h1, c1);                                              \
         spin_expand_add<float2, M, true>(c0, c1, acc);                               \
      }                                                                               \
      else if (bw)                                                                    \
      {                                                                               \
         spin_project<float2, M, false>(sp[j], h0, h1);                               \
         su3_mul_f<true>(u[j], h0, c0);                                               \
         su3_mul_f<true>(u[j], h1, c1);                                               \
         spin_expand_add<float2, M, false>(c0, c1, acc);                              \
      }                                                                               \
   }
         OQH_FACE_TERM(0)
         OQH_FACE_TERM(1)
         OQH_FACE_TERM(2)
         OQH_FACE_TERM(3)
#undef OQH_FACE_TERM
      }
   }
   float2 r[12];
   load_spinor((const float2 *)a.rho, y, r);
#pragma unroll
   for (int c = 0; c < 12; c++) r[c] = cadd(r[c], cscale(acc[c], 0.5f));
   store_spinor(a.rho, y, r);
}

// ---------------------------------------------------------------------------
// block operators on the block fields of the API (one work-group per call)
// ---------------------------------------------------------------------------

enum BlkOp { BOP_DW = 0, BOP_DWHAT, BOP_MRES, BOP_EO_MRES, BOP_DWEE, BOP_DWOO, BOP_DWOE, BOP_DWEO };

template <typename C>
__global__ __launch_bounds__(SWG) void k_blk_op(SArgsT<C> a, int n, int op, int k, int l, decltype(C::x) mu)
{
   typedef decltype(C::x) R;
   const int *imb = a.imb + (size_t)n * a.bvol;
   C *F = a.scr + (size_t)n * NBF * a.Ub;  // the block's fields 0,1,2
   C *Sk = F + (size_t)k * a.Ub, *Sl = F + (size_t)l * a.Ub;
   C *T = F + 3 * a.Ub;  // odd intermediate of Dwhat_blk
   // open bc: the operators zero their input on the boundary points (all of
   // them for Dw_blk, the even ones for Dwhat_blk, Dwee_blk and Dwoe_blk,
   // the odd ones for Dwoo_blk and Dweo_blk); in the MinRes solvers the
   // input is field 1
   if (a.masked)
   {
      const bool even = (op == BOP_DWHAT || op == BOP_EO_MRES || op == BOP_DWEE || op == BOP_DWOE);
      const bool odd = (op == BOP_DWOO || op == BOP_DWEO);
      C *In = (op == BOP_MRES || op == BOP_EO_MRES) ? F + a.Ub : Sk;
      for (int i = threadIdx.x; i < a.bvol; i += SWG)
         if (a.bnd[imb[i]] && (!even || i < a.bh) && (!odd || i >= a.bh)) zero_spinor(In, i);
      __syncthreads();
   }
   if (op == BOP_DW)
      blk_dw(a, imb, Sk, Sl, 0, a.bvol, mu, SWG);
   else if (op == BOP_DWHAT)
   {
      // Dwhat_blk leaves the odd half of the output unchanged
      blk_dwhat(a, imb, Sk, Sl, T, mu, SWG);
   }
   else if (op == BOP_DWEE || op == BOP_DWOO)
   {
      // (A + i mu gamma5) on one parity (Dw.c:1584-1694); the fields may coincide
      const bool ee = op == BOP_DWEE;
      const R m = ee ? mu : a.muo;
      for (int i = (ee ? 0 : a.bh) + threadIdx.x; i < (ee ? a.bh : a.bvol); i += SWG)
      {
         const int gx = imb[i];
         C v[12], o[12];
         if (a.masked && a.bnd[gx])
            zero12(o);
         else
         {
            load_spinor((const C *)Sk, i, v);
            pauli_site(a.sw, gx, m, v, o);
         }
         store_spinor(Sl, i, o);
      }
   }
   else if (op == BOP_DWOE || op == BOP_DWEO)
   {
      // hopping terms between the parities with zero exterior (Dw.c:1696-1826):
      // Dwoe_blk assigns D_oe s to the odd points, Dweo_blk subtracts D_eo s
      // from the even points; the output parity is never read
      const bool oe = op == BOP_DWOE;
      for (int i = (oe ? a.bh : 0) + threadIdx.x; i < (oe ? a.bvol : a.bh); i += SWG)
      {
         const int gx = imb[i];
         C acc[12], o[12];
         zero12(acc);
         if (a.masked && a.bnd[gx])
            zero12(o);
         else
         {
            blk_hop(a, imb, (const C *)Sk, i, gx, acc);
            if (oe)
            {
#pragma unroll
               for (int c = 0; c < 12; c++) o[c] = cscale(acc[c], (R)-0.5);
            }
            else
            {
               load_spinor((const C *)Sl, i, o);
#pragma unroll
               for (int c = 0; c < 12; c++) o[c] = cadd(o[c], cscale(acc[c], (R)0.5));
            }
         }
         store_spinor(Sl, i, o);
      }
   }
   else if (op == BOP_MRES)
      blk_mres_dev<false>(a, imb, F, F + a.Ub, F + 2 * a.Ub, T, mu, SWG);
   else
      blk_mres_dev<true>(a, imb, F, F + a.Ub, F + 2 * a.Ub, T, mu, SWG);
}

// Dw_bnd (dirac/Dw_bnd.c:801-1011): for the face points x of block n the
// Weyl field w = -1/2 U chi of the hopping term into the exterior neighbour
// y, chi the upper components of (1 -+ gamma_mu) s(x): faces -mu (y = x - mu)
// use U(y,mu), faces +mu (y = x + mu) U(x,mu)^+.  Faces on the open time
// boundary give zero and zero s at their points.  One work-group per call.
struct FaceOfs
{
   int o[9];
};

__global__ __launch_bounds__(SWG) void k_dw_bnd(SArgs a, int n, int k, const int *ipp, FaceOfs fo, float2 *W)
{
   const int *imb = a.imb + (size_t)n * a.bvol;
   float2 *S = a.scr + ((size_t)n * NBF + k) * a.Ub;
   float2 *Wn = W + (size_t)n * fo.o[8] * 6;
   for (int ifc = 0; ifc < 8; ifc++)
   {
      const int mu = ifc >> 1;
      const bool up = ifc & 1;
      for (int j = fo.o[ifc] + threadIdx.x; j < fo.o[ifc + 1]; j += SWG)
      {
         const int x = ipp[j], gx = imb[x];
         float2 w[6];
         if (mu == 0 && a.masked && a.bnd[gx])
         {
#pragma unroll
            for (int c = 0; c < 6; c++) w[c] = make_float2(0.0f, 0.0f);
            zero_spinor(S, x);
         }
         else
         {
            float2 sp[12], h[6], u[9];
            load_spinor((const float2 *)S, x, sp);
            // chi (spin components 1, 2) per face, from Dw_bnd.c:825-1009
#pragma unroll
            for (int c = 0; c < 3; c++)
            {
               const float2 s1 = sp[c], s2 = sp[3 + c], s3 = sp[6 + c], s4 = sp[9 + c];
               float2 a1, a2;
               if (mu == 0)
               {
                  a1 = up ? csub(s1, s3) : cadd(s1, s3);
                  a2 = up ? csub(s2, s4) : cadd(s2, s4);
               }
               else if (mu == 1)
               {
                  a1 = up ? csubi(s1, s4) : caddi(s1, s4);
                  a2 = up ? csubi(s2, s3) : caddi(s2, s3);
               }
               else if (mu == 2)
               {
                  a1 = up ? csub(s1, s4) : cadd(s1, s4);
                  a2 = up ? cadd(s2, s3) : csub(s2, s3);
               }
               else
               {
                  a1 = up ? csubi(s1, s3) : caddi(s1, s3);
                  a2 = up ? caddi(s2, s4) : csubi(s2, s4);
               }
               h[c] = cscale(a1, -0.5f);
               h[3 + c] = cscale(a2, -0.5f);
            }
            const int gy = a.nbr[(size_t)(up ? 2 * mu : 2 * mu + 1) * a.V + gx] & 0x7fffffff;
            const float2 *lp = blk_link(a, gx, gy, mu, up);
#pragma unroll
            for (int q = 0; q < 9; q++) u[q] = lp[q * SB];
            if (up)
            {
               su3_mul<float2, true>(u, h, w);
               su3_mul<float2, true>(u, h + 3, w + 3);
            }
            else
            {
               su3_mul<float2, false>(u, h, w);
               su3_mul<float2, false>(u, h + 3, w + 3);
            }
         }
#pragma unroll
         for (int c = 0; c < 6; c++) Wn[(size_t)j * 6 + c] = w[c];
      }
      // the time faces zero s on the open boundary before the other faces
      // read it (the faces are processed in the order -0, +0, ..., +3)
      if (ifc < 2) __syncthreads();
   }
}

template <typename C> __global__ void k_blk_copy(C *glob, C *blk, const int *imb, int i0, int i1, int to_blk)
{
   int i = i0 + blockIdx.x * 256 + threadIdx.x;
   if (i >= i1) return;
   int gx = imb[i];
   C v[12];
   if (to_blk)
   {
      load_spinor((const C *)glob, gx, v);
      store_spinor(blk, i, v);
   }
   else
   {
      load_spinor((const C *)blk, i, v);
      store_spinor(glob, gx, v);
   }
}

// ---------------------------------------------------------------------------
// host side: block grid
// ---------------------------------------------------------------------------

static int lexb(const int *bs, const int *y) { return y[3] + bs[3] * (y[2] + bs[2] * (y[1] + bs[1] * y[0])); }

static void drop_sap_graph();

static void free_grid()
{
   drop_sap_graph();
   dev_free(G.d_imb); dev_free(G.d_bnb);
   for (int c = 0; c < 2; c++) { dev_free(G.d_face[c]); dev_free(G.d_fmask[c]); G.d_face[c] = nullptr; G.d_fmask[c] = nullptr; }
   dev_free(G.d_swb); dev_free(G.d_scr); dev_free(G.d_s0g); dev_free(G.d_bs);
   dev_free(G.d_u16); dev_free(G.d_swb16);
   for (int k = 0; k < 2; k++) { dev_free(G.d_h16[k]); dev_free(G.d_hsc[k]); }
   for (int k = 0; k < 3; k++) dev_free(G.d_h64[k]);
   dev_free(G.d_swb64); dev_free(G.d_scr64); dev_free(G.d_bsd);
   dev_free(G.d_wf); dev_free(G.d_wfm); dev_free(G.d_nbn);
   dev_free(G.d_imb4); dev_free(G.d_nbs); dev_free(G.d_count); dev_free(G.d_x);
   if (G.h_dead) HIP_OK(hipHostFree(G.h_dead));
   dev_free(G.d_ipp); dev_free(G.d_bw);
   G = SapGrid();
}

static bool reg_kernel() { return OQH_SAP_REG && G.bvol == RBV; }

// tables and buffers of k_sap_cluster; false if the block size does not allow
// it (bipt: block point of a position in the block)
static bool build_cluster(const int *bs, const std::vector<int> &bipt)
{
   int ns = 1, nd[4];
   for (int mu = 0; mu < 4; mu++)
   {
      if (bs[mu] % 4) return false;
      nd[mu] = bs[mu] / 4;
      ns *= nd[mu];
   }
   if (ns < 2 || ns > CLMAX) return false;
   std::vector<int> &imb4 = G.imb4, nbs(8 * (size_t)ns), loc(G.bvol);
   imb4.assign((size_t)G.nb * G.bvol, 0);
   int m[4], y[4], x[4];
   for (int k = 0; k < ns; k++)
   {
      int r = k;
      for (int mu = 3; mu >= 0; mu--)
      {
         m[mu] = r % nd[mu];
         r /= nd[mu];
      }
      for (int mu = 0; mu < 4; mu++)
         for (int s = 0; s < 2; s++)
         {
            const int c = m[mu] + (s ? -1 : 1);
            int z[4] = {m[0], m[1], m[2], m[3]};
            z[mu] = c;
            nbs[8 * (size_t)k + 2 * mu + s] =
               (c < 0 || c >= nd[mu]) ? -1 : z[3] + nd[3] * (z[2] + nd[2] * (z[1] + nd[1] * z[0]));
         }
      int ofs[2] = {0, RBV / 2};
      for (x[0] = 0; x[0] < 4; x[0]++)
      for (x[1] = 0; x[1] < 4; x[1]++)
      for (x[2] = 0; x[2] < 4; x[2]++)
      for (x[3] = 0; x[3] < 4; x[3]++)
      {
         for (int mu = 0; mu < 4; mu++) y[mu] = 4 * m[mu] + x[mu];
         loc[(size_t)k * RBV + ofs[(x[0] + x[1] + x[2] + x[3]) & 1]++] = bipt[lexb(bs, y)];
      }
   }
   for (int n = 0; n < G.nb; n++)
      for (int i = 0; i < G.bvol; i++) imb4[(size_t)n * G.bvol + i] = G.imb[(size_t)n * G.bvol + loc[i]];
   const size_t nx = (size_t)G.nbh * ns * FUN;
   G.d_imb4 = (int *)dev_alloc(sizeof(int) * imb4.size());
   G.d_nbs = (int *)dev_alloc(sizeof(int) * nbs.size());
   G.d_count = (unsigned *)dev_alloc(sizeof(unsigned) * CLPAD * ((size_t)G.nbh + 1));
   G.d_x = (unsigned long long *)dev_alloc(sizeof(unsigned long long) * (2 * nx + (size_t)G.nbh * ns * 4));
   if (hipHostMalloc((void **)&G.h_dead, sizeof(int), 0) != hipSuccess) G.h_dead = nullptr;
   if (!G.d_imb4 || !G.d_nbs || !G.d_count || !G.d_x || !G.h_dead) return false;
   *G.h_dead = 0;
   HIP_OK(hipMemcpy(G.d_imb4, imb4.data(), sizeof(int) * imb4.size(), hipMemcpyHostToDevice));
   HIP_OK(hipMemcpy(G.d_nbs, nbs.data(), sizeof(int) * nbs.size(), hipMemcpyHostToDevice));
   G.ns = ns;
   return true;
}

static bool build_grid(const char *where)
{
   Lib &L = lib();
   if (!require_geometry(where)) return false;
   if (L.sap_ncy == 0)
   {
      fail(where, "SAP parameters are not set");
      return false;
   }
   if (G.ready && memcmp(G.bs, L.sap_bs, sizeof(G.bs)) == 0) return true;
   if (G.ready) free_grid();
   const int *bs = L.sap_bs;
   int nbl[4], cb[4], nbs[4];
   for (int mu = 0; mu < 4; mu++) nbl[mu] = L.g.L[mu] / bs[mu];
   memcpy(G.bs, bs, sizeof(G.bs));
   G.nb = nbl[0] * nbl[1] * nbl[2] * nbl[3];
   G.nbh = G.nb / 2;
   G.bvol = bs[0] * bs[1] * bs[2] * bs[3];
   G.bh = G.bvol / 2;
   G.Ub = units_for(G.bvol, 12);

   // block-local point order (blk_geometry.c:56-128): cache blocks, even first
   std::vector<int> bipt(G.bvol);
   cb[0] = bs[0];
   for (int mu = 1; mu < 4; mu++) cb[mu] = (bs[mu] % 4 == 0) ? 4 : ((bs[mu] % 3 == 0) ? 3 : 2);
   for (int mu = 0; mu < 4; mu++) nbs[mu] = bs[mu] / cb[mu];
   {
      int ofs[2] = {0, G.bh}, j[4], x[4], y[4];
      for (j[0] = 0; j[0] < nbs[0]; j[0]++)
      for (j[1] = 0; j[1] < nbs[1]; j[1]++)
      for (j[2] = 0; j[2] < nbs[2]; j[2]++)
      for (j[3] = 0; j[3] < nbs[3]; j[3]++)
         for (x[0] = 0; x[0] < cb[0]; x[0]++)
         for (x[1] = 0; x[1] < cb[1]; x[1]++)
         for (x[2] = 0; x[2] < cb[2]; x[2]++)
         for (x[3] = 0; x[3] < cb[3]; x[3]++)
         {
            for (int mu = 0; mu < 4; mu++) y[mu] = j[mu] * cb[mu] + x[mu];
            bipt[lexb(bs, y)] = ofs[(y[0] + y[1] + y[2] + y[3]) & 1]++;
         }
   }
   std::vector<int> bnb(8 * (size_t)G.bvol), bcoord(4 * (size_t)G.bvol);
   {
      int y[4];
      for (y[0] = 0; y[0] < bs[0]; y[0]++)
      for (y[1] = 0; y[1] < bs[1]; y[1]++)
      for (y[2] = 0; y[2] < bs[2]; y[2]++)
      for (y[3] = 0; y[3] < bs[3]; y[3]++)
      {
         int i = bipt[lexb(bs, y)];
         for (int mu = 0; mu < 4; mu++) bcoord[4 * (size_t)i + mu] = y[mu];
         for (int mu = 0; mu < 4; mu++)
         {
            int z[4];
            memcpy(z, y, sizeof(z));
            z[mu] = y[mu] + 1;
            bnb[(size_t)(2 * mu) * G.bvol + i] = (z[mu] < bs[mu]) ? bipt[lexb(bs, z)] : G.bvol;
            z[mu] = y[mu] - 1;
            bnb[(size_t)(2 * mu + 1) * G.bvol + i] = (z[mu] >= 0) ? bipt[lexb(bs, z)] : G.bvol;
         }
      }
   }
   // blocks: colour-0 blocks first, lexicographic (blk_grid.c:63-113)
   G.imb.assign((size_t)G.nb * G.bvol, 0);
   G.bo.assign(4 * (size_t)G.nb, 0);
   std::vector<int> colour_of_site(L.g.V, 0), inface(L.g.V, 0);
   std::vector<unsigned char> fm(L.g.V, 0);
   int ib = 0, m[4];
   for (int col = 0; col < 2; col++)
      for (m[0] = 0; m[0] < nbl[0]; m[0]++)
      for (m[1] = 0; m[1] < nbl[1]; m[1]++)
      for (m[2] = 0; m[2] < nbl[2]; m[2]++)
      for (m[3] = 0; m[3] < nbl[3]; m[3]++)
      {
         if (((m[0] + m[1] + m[2] + m[3]) & 1) != col) continue;
         for (int mu = 0; mu < 4; mu++) G.bo[4 * (size_t)ib + mu] = m[mu] * bs[mu];
         for (int i = 0; i < G.bvol; i++)
         {
            int g[4];
            for (int mu = 0; mu < 4; mu++) g[mu] = m[mu] * bs[mu] + bcoord[4 * (size_t)i + mu];
            int gx = L.g.ipt[g[3] + L.g.L[3] * (g[2] + L.g.L[2] * (g[1] + L.g.L[1] * g[0]))];
            G.imb[(size_t)ib * G.bvol + i] = gx;
            colour_of_site[gx] = col;
            unsigned char mk = 0;
            for (int mu = 0; mu < 4; mu++)
            {
               if (bnb[(size_t)(2 * mu) * G.bvol + i] == G.bvol) mk |= (unsigned char)(1 << (2 * mu));
               if (bnb[(size_t)(2 * mu + 1) * G.bvol + i] == G.bvol) mk |= (unsigned char)(2 << (2 * mu));
            }
            fm[gx] = mk;
         }
         ib++;
      }
   std::vector<int> face[2];
   std::vector<unsigned char> fmask[2];
   for (int ix = 0; ix < L.g.V; ix++)
      if (fm[ix])
      {
         face[colour_of_site[ix]].push_back(ix);
         fmask[colour_of_site[ix]].push_back(fm[ix]);
      }
   G.d_imb = (int *)dev_alloc(sizeof(int) * G.imb.size());
   // face points of the block boundaries in the order of bnd_geometry
   // (lattice/blk_geometry.c:241-313): odd points first, then even, each
   // point entered on the faces -mu/+mu whose neighbour lies outside
   {
      std::vector<int> fl[8];
      for (int ix = 0; ix < G.bvol; ix++)
      {
         const int iy = ix < G.bh ? ix + G.bh : ix - G.bh;
         for (int mu = 0; mu < 4; mu++)
         {
            if (bnb[(size_t)(2 * mu) * G.bvol + iy] == G.bvol) fl[2 * mu + 1].push_back(iy);
            if (bnb[(size_t)(2 * mu + 1) * G.bvol + iy] == G.bvol) fl[2 * mu].push_back(iy);
         }
      }
      std::vector<int> ipp;
      for (int ifc = 0; ifc < 8; ifc++)
      {
         G.fofs[ifc] = (int)ipp.size();
         ipp.insert(ipp.end(), fl[ifc].begin(), fl[ifc].end());
      }
      G.fofs[8] = (int)ipp.size();
      G.d_ipp = (int *)dev_alloc(sizeof(int) * ipp.size());
      HIP_OK(hipMemcpy(G.d_ipp, ipp.data(), sizeof(int) * ipp.size(), hipMemcpyHostToDevice));
   }
   G.d_bnb = (int *)dev_alloc(sizeof(int) * bnb.size());
   HIP_OK(hipMemcpy(G.d_imb, G.imb.data(), sizeof(int) * G.imb.size(), hipMemcpyHostToDevice));
   HIP_OK(hipMemcpy(G.d_bnb, bnb.data(), sizeof(int) * bnb.size(), hipMemcpyHostToDevice));
   for (int c = 0; c < 2; c++)
   {
      G.nface[c] = (int)face[c].size();
      G.d_face[c] = (int *)dev_alloc(sizeof(int) * (face[c].size() + 1));
      G.d_fmask[c] = (unsigned char *)dev_alloc(fmask[c].size() + 1);
      if (G.nface[c])
      {
         HIP_OK(hipMemcpy(G.d_face[c], face[c].data(), sizeof(int) * face[c].size(), hipMemcpyHostToDevice));
         HIP_OK(hipMemcpy(G.d_fmask[c], fmask[c].data(), fmask[c].size(), hipMemcpyHostToDevice));
      }
   }
   G.d_swb = (float2 *)dev_alloc(units_for(L.g.V, 36) * sizeof(float2));
   if (reg_kernel() || build_cluster(bs, bipt))
   {
      // neighbouring 4^4 (sub-)blocks across the block's faces: that of a
      // point one step outside, -1 inside the block
      const int ns = std::max(G.ns, 1);
      const std::vector<int> &im = G.ns ? G.imb4 : G.imb;
      std::vector<int> sub(L.g.V), nbn(8 * (size_t)G.nb * ns, -1);
      for (size_t k = 0; k < im.size(); k++) sub[im[k]] = (int)(k / RBV);
      for (size_t k = 0; k < im.size(); k++)
         for (int mu = 0; mu < 4; mu++)
         {
            const size_t gx = im[k];
            const int n = (int)(k / RBV), up = sub[L.g.iup[4 * gx + mu]], dn = sub[L.g.idn[4 * gx + mu]];
            if (fm[gx] & (1 << (2 * mu))) nbn[8 * (size_t)n + 2 * mu] = up;
            if (fm[gx] & (2 << (2 * mu))) nbn[8 * (size_t)n + 2 * mu + 1] = dn;
         }
      G.d_nbn = (int *)dev_alloc(sizeof(int) * nbn.size());
      HIP_OK(hipMemcpy(G.d_nbn, nbn.data(), sizeof(int) * nbn.size(), hipMemcpyHostToDevice));
      G.d_wf = (float2 *)dev_alloc((size_t)G.nb * ns * FUN * sizeof(float2));
   }
   else
   {
      G.d_scr = (float2 *)dev_alloc((size_t)G.nbh * 3 * G.Ub * sizeof(float2));
      G.d_s0g = (float2 *)dev_alloc(units_for(L.g.V, 12) * sizeof(float2));
      HIP_OK(hipMemset(G.d_s0g, 0, units_for(L.g.V, 12) * sizeof(float2)));
   }
   G.swb_set = -1;
   G.ready = true;
   return true;
}

// FP32 SW field of the block solver: single-precision copy of swd with the
// points of the set inverted in double precision first (map_sw2blk.c:53-100)
static int assign_swb(int set)
{
   Lib &L = lib();
   ensure_swd(0, 0);  // as sap_gcr.c:181-197: the SW field must not be inverted
   int h = L.g.V / 2, ifail = 0;
   size_t nun = units_for(L.g.V, 36);
   double2 *tmp = (double2 *)tmp_buffer(nun * sizeof(double2));
   HIP_OK(hipMemcpyAsync(tmp, L.d_swd, nun * sizeof(double2), hipMemcpyDeviceToDevice, L.stream));
   if (set == ALL_PTS || set == EVEN_PTS) ifail |= invert_pauli(tmp, tmp, 0, h, 0.0);
   if (set == ALL_PTS || set == ODD_PTS) ifail |= invert_pauli(tmp, tmp, h, h, 0.0);
   convert_f64_to_f32(tmp, G.d_swb, nun, L.stream);
   G.swb_version++;
   if (L.sap_prec == 2 || G.need64)
   {
      if (!G.d_swb64) G.d_swb64 = (double2 *)dev_alloc(nun * sizeof(double2));
      if (G.d_swb64)
      {
         HIP_OK(hipMemcpyAsync(G.d_swb64, tmp, nun * sizeof(double2), hipMemcpyDeviceToDevice, L.stream));
         G.swb64_version = G.swb_version;
      }
   }
   HIP_OK(hipStreamSynchronize(L.stream));
   G.swb_set = set;
   G.swb_epoch = L.swd_epoch;
   return ifail;
}

static SArgs sargs(float mu, int nmr)
{
   Lib &L = lib();
   SArgs a;
   memset(&a, 0, sizeof(a));  // compared bytewise by the graph cache
   a.u = L.d_u;
   a.sw = G.d_swb;
   a.imb = G.d_imb;
   a.bnb = G.d_bnb;
   a.nbr = L.d_nbr;
   a.bnd = L.d_bnd;
   a.V = L.g.V;
   a.h = L.g.V / 2;
   a.bvol = G.bvol;
   a.bh = G.bh;
   a.masked = (L.bc != 3);
   a.eoflg = L.eoflg;
   a.nmr = nmr;
   a.mu = mu;
   a.muo = L.eoflg ? 0.0f : mu;
   a.Ub = G.Ub;
   a.psi = a.rho = nullptr;
   a.s0g = G.d_s0g;
   a.scr = G.d_scr;
   a.n0 = 0;
   a.psi16 = G.d_h16[0];
   a.rho16 = G.d_h16[1];
   a.psc = G.d_hsc[0];
   a.rsc = G.d_hsc[1];
   a.wf = G.d_wf;
   a.nbn = G.d_nbn;
   a.pz = 0;
   return a;
}

static bool half_variant()
{
   return OQH_SAP_REG && G.bvol == RBV && lib().sap_prec == 1 && G.d_h16[0] && G.d_h16[1] && G.d_u16 &&
          G.d_swb16;
}

// the block's spinors fit on the chip (k_sap_lds)
static bool lds_kernel() { return G.bvol != RBV && !G.ns && G.bvol <= BLV_MAX; }

template <int TPB> static void launch_lds(const SArgs &a, int isolv, unsigned nb)
{
   hipStream_t st = lib().stream;
   const size_t lds = (size_t)12 * G.bh * sizeof(float2);
   if (isolv && a.masked)
      k_sap_lds<1, TPB, true><<<nb, TPB, lds, st>>>(a);
   else if (isolv)
      k_sap_lds<1, TPB, false><<<nb, TPB, lds, st>>>(a);
   else if (a.masked)
      k_sap_lds<0, TPB, true><<<nb, TPB, lds, st>>>(a);
   else
      k_sap_lds<0, TPB, false><<<nb, TPB, lds, st>>>(a);
}

// a block shared by several work-groups (k_sap_cluster)
static void launch_cluster(const SArgs &a, int isolv)
{
   hipStream_t st = lib().stream;
   ClArgs q;
   q.ns = G.ns;
   q.imb4 = G.d_imb4;
   q.nbs = G.d_nbs;
   q.ticket = G.d_count;
   q.count = G.d_count + CLPAD;
   q.x = G.d_x;
   q.xlen = (size_t)G.nbh * G.ns * FUN;
   q.sums = G.d_x + 2 * q.xlen;
   q.polls = lib().sap_polls;
   q.dead = G.h_dead;
   const unsigned nb = (unsigned)(G.nbh * G.ns);
   k_cl_reset<<<(G.nbh + 256) / 256, 256, 0, st>>>(G.d_count, G.nbh + 1);
   if (isolv && a.masked)
      k_sap_cluster<1, true><<<nb, RBV, 0, st>>>(a, q);
   else if (isolv)
      k_sap_cluster<1, false><<<nb, RBV, 0, st>>>(a, q);
   else if (a.masked)
      k_sap_cluster<0, true><<<nb, RBV, 0, st>>>(a, q);
   else
      k_sap_cluster<0, false><<<nb, RBV, 0, st>>>(a, q);
}

// block solves of the blocks of colour ic; the register kernel first adds
// the terms of the other colour's face fields if pull is set
static void sap_blocks(const SArgs &a0, int ic, int isolv, int pull)
{
   Lib &L = lib();
   SArgs a = a0;
   a.n0 = ic ? G.nbh : 0;
   a.pull = pull;
   const unsigned nb = (unsigned)(G.nbh * std::max(a.nsrc, 1));
   if (half_variant() && !a.nsrc)
   {
      if (isolv && a.masked)
         k_sap_reg<1, __half2, true><<<nb, RBV, 0, L.stream>>>(a, G.d_u16, G.d_swb16);
      else if (isolv)
         k_sap_reg<1, __half2, false><<<nb, RBV, 0, L.stream>>>(a, G.d_u16, G.d_swb16);
      else if (a.masked)
         k_sap_reg<0, __half2, true><<<nb, RBV, 0, L.stream>>>(a, G.d_u16, G.d_swb16);
      else
         k_sap_reg<0, __half2, false><<<nb, RBV, 0, L.stream>>>(a, G.d_u16, G.d_swb16);
   }
   else if (reg_kernel())
   {
      if (isolv && a.masked)
         k_sap_reg<1, float2, true><<<nb, RBV, 0, L.stream>>>(a, nullptr, nullptr);
      else if (isolv)
         k_sap_reg<1, float2, false><<<nb, RBV, 0, L.stream>>>(a, nullptr, nullptr);
      else if (a.masked)
         k_sap_reg<0, float2, true><<<nb, RBV, 0, L.stream>>>(a, nullptr, nullptr);
      else
         k_sap_reg<0, float2, false><<<nb, RBV, 0, L.stream>>>(a, nullptr, nullptr);
   }
   else if (G.ns)
      launch_cluster(a, isolv);
   else if (lds_kernel())
   {
      if (G.bh <= 256)
         launch_lds<256>(a, isolv, nb);
      else if (G.bh <= 512)
         launch_lds<512>(a, isolv, nb);
      else
         launch_lds<768>(a, isolv, nb);
   }
   else if (isolv)
      // 1024 threads per block: the few blocks of a lattice would otherwise
      // leave most of the chip idle
      k_sap_blocks<1, float2, SWG_MAX><<<nb, SWG_MAX, 0, L.stream>>>(a);
   else
      k_sap_blocks<0, float2, SWG_MAX><<<nb, SWG_MAX, 0, L.stream>>>(a);
}

// face terms from the corrections of the colour-(1-c) blocks into rho on
// the faces of the colour-c blocks (those of k_sap_lds and k_sap_blocks)
static void sap_push_faces(const SArgs &a, int c)
{
   if (!G.nface[c]) return;
   k_sap_faces<<<(G.nface[c] + 255) / 256, 256, 0, lib().stream>>>(a, G.d_face[c], G.d_fmask[c], G.nface[c]);
}

// one Schwarz cycle (sap.c:720-790): colour 0, faces of colour 1, colour 1,
// faces of colour 0.  With the 4^4 (sub-)block kernels the face terms into a colour
// are added by its next block solve; first: rho is complete on entry (none
// for colour 0); finish: complete rho at the end (faces of colour 0).
static void sap_cycle(const SArgs &a, int isolv, bool first, bool finish)
{
   if (reg_kernel() || G.ns)
   {
      sap_blocks(a, 0, isolv, !first);
      sap_blocks(a, 1, isolv, 1);
      if (!finish) return;
      SArgs c = a;
      c.n0 = 0;
      const unsigned nb = (unsigned)(G.nbh * std::max(G.ns, 1) * std::max(a.nsrc, 1));
      if (half_variant() && !a.nsrc)
         k_sap_complete<__half2><<<nb, RBV, 0, lib().stream>>>(c, G.d_imb, G.d_u16);
      else
         k_sap_complete<float2><<<nb, RBV, 0, lib().stream>>>(c, G.ns ? G.d_imb4 : G.d_imb, nullptr);
   }
   else
   {
      sap_blocks(a, 0, isolv, 0);
      sap_push_faces(a, 1);
      sap_blocks(a, 1, isolv, 0);
      sap_push_faces(a, 0);
   }
}

// FP32 field <-> FP16 field with per-site scales
__global__ void k_s32_to_h16(const float2 *__restrict__ f, __half2 *h, float *sc, int V)
{
   int x = blockIdx.x * 256 + threadIdx.x;
   if (x >= V) return;
   float2 v[12];
   load_spinor(f, x, v);
   store_h16(h, sc, x, v);
}

__global__ void k_h16_to_s32(const __half2 *h, const float *sc, float2 *__restrict__ f, int V)
{
   int x = blockIdx.x * 256 + threadIdx.x;
   if (x >= V) return;
   float2 v[12];
   load_h16(h, sc, x, v);
   store_spinor(f, x, v);
}

// ---------------------------------------------------------------------------
// FP64 variant: the generic block solver on double fields, FP64 links and
// the FP64 block SW field
// ---------------------------------------------------------------------------

__global__ __launch_bounds__(256) void k_sap_faces64(SArgsD a, const int *face, const unsigned char *fmask, int nf)
{
   int k = blockIdx.x * 256 + threadIdx.x;
   if (k >= nf) return;
   int y = face[k];
   int m = fmask[k];
   double2 acc[12], sp[12];
   zero12(acc);
   int odd = y >= a.h;
#define OQH_FACE64(MU)                                                                 \
   if (m & (1 << (2 * MU)))                                                           \
   {                                                                                  \
      int x = a.nbr[(size_t)(2 * MU) * a.V + y] & 0x7fffffff;                         \
      load_spinor((const double2 *)a.s0g, x, sp);                                     \
      const double2 *up = odd ? link_ptr(a.u, y - a.h, 2 * MU) : link_ptr(a.u, x - a.h, 2 * MU + 1); \
      hop_one<double2, MU, true>(sp, up, acc);                                        \
   }                                                                                  \
   if (m & (2 << (2 * MU)))                                                           \
   {                                                                                  \
      int x = a.nbr[(size_t)(2 * MU + 1) * a.V + y] & 0x7fffffff;                     \
      load_spinor((const double2 *)a.s0g, x, sp);                                     \
      const double2 *up = odd ? link_ptr(a.u, y - a.h, 2 * MU + 1) : link_ptr(a.u, x - a.h, 2 * MU); \
      hop_one<double2, MU, false>(sp, up, acc);                                       \
   }
   OQH_FACE64(0)
   OQH_FACE64(1)
   OQH_FACE64(2)
   OQH_FACE64(3)
#undef OQH_FACE64
   double2 r[12];
   load_spinor((const double2 *)a.rho, y, r);
#pragma unroll
   for (int c = 0; c < 12; c++) r[c] = cadd(r[c], cscale(acc[c], 0.5));
   store_spinor(a.rho, y, r);
}

__global__ void k_s32_to_s64(const float2 *__restrict__ a, double2 *__restrict__ b, size_t n)
{
   size_t k = (size_t)blockIdx.x * 256 + threadIdx.x;
   if (k < n) b[k] = make_double2(a[k].x, a[k].y);
}

// phi = psi, chi = rho_in - rho (FP64 fields rounded to FP32)
__global__ void k_mop64_out(const double2 *__restrict__ psi, const double2 *__restrict__ rho,
                            const float2 *__restrict__ rin, float2 *__restrict__ phi, float2 *__restrict__ chi, size_t n)
{
   size_t k = (size_t)blockIdx.x * 256 + threadIdx.x;
   if (k >= n) return;
   phi[k] = make_float2((float)psi[k].x, (float)psi[k].y);
   chi[k] = make_float2((float)((double)rin[k].x - rho[k].x), (float)((double)rin[k].y - rho[k].y));
}

static SArgsD sargs64(double mu, int nmr)
{
   Lib &L = lib();
   SArgsD a;
   memset(&a, 0, sizeof(a));
   a.u = L.d_ud;
   a.sw = G.d_swb64;
   a.imb = G.d_imb;
   a.bnb = G.d_bnb;
   a.nbr = L.d_nbr;
   a.bnd = L.d_bnd;
   a.V = L.g.V;
   a.h = L.g.V / 2;
   a.bvol = G.bvol;
   a.bh = G.bh;
   a.masked = (L.bc != 3);
   a.eoflg = L.eoflg;
   a.nmr = nmr;
   a.mu = mu;
   a.muo = L.eoflg ? 0.0 : mu;
   a.Ub = G.Ub;
   a.psi = G.d_h64[0];
   a.rho = G.d_h64[1];
   a.s0g = G.d_h64[2];
   a.scr = G.d_scr64;
   return a;
}

static bool f64_variant() { return lib().sap_prec == 2 && G.d_h64[0] && G.d_scr64 && G.d_swb64; }

// one Schwarz cycle on the FP64 fields psi64, rho64
static void sap_cycle64(const SArgsD &a0, int isolv)
{
   Lib &L = lib();
   SArgsD a = a0;
   for (int ic = 0; ic < 2; ic++)
   {
      a.n0 = ic ? G.nbh : 0;
      if (isolv)
         k_sap_blocks<1><<<G.nbh, SWG, 0, L.stream>>>(a);
      else
         k_sap_blocks<0><<<G.nbh, SWG, 0, L.stream>>>(a);
      int c = 1 - ic;
      if (G.nface[c])
         k_sap_faces64<<<(G.nface[c] + 255) / 256, 256, 0, L.stream>>>(a, G.d_face[c], G.d_fmask[c], G.nface[c]);
   }
}

// the SAP preconditioner of sap_gcr in the FP64 variant: ncy cycles on FP64
// fields from psi = 0, rho = rho_in; phi = psi, chi = rho_in - rho
bool sap_mop64(double mu, int isolv, int nmr, int ncy, const float2 *rho, float2 *phi, float2 *chi)
{
   if (!f64_variant()) return false;
   Lib &L = lib();
   const size_t nu = units_for(L.g.V, 12);
   const unsigned nbk = (unsigned)((nu + 255) / 256);
   SArgsD a = sargs64(mu, nmr);
   HIP_OK(hipMemsetAsync(G.d_h64[0], 0, nu * sizeof(double2), L.stream));
   k_s32_to_s64<<<nbk, 256, 0, L.stream>>>(rho, G.d_h64[1], nu);
   for (int n = 0; n < ncy; n++) sap_cycle64(a, isolv);
   k_mop64_out<<<nbk, 256, 0, L.stream>>>(G.d_h64[0], G.d_h64[1], rho, phi, chi, nu);
   return true;
}

// ncy SAP cycles on device fields (no synchronisation); the FP16 variant
// converts psi and rho to FP16 spinors and back.  zero: the cycles start
// from psi = 0 (psi need not be set); want_res: rho is needed on return.
void sap_cycles(float mu, int isolv, int nmr, int ncy, float2 *psi, float2 *rho, bool zero, bool want_res)
{
   Lib &L = lib();
   const size_t nu = units_for(L.g.V, 12);
   const unsigned nbu = (unsigned)((nu + 255) / 256);
   if (f64_variant())
   {
      if (zero) HIP_OK(hipMemsetAsync(psi, 0, nu * sizeof(float2), L.stream));
      k_s32_to_s64<<<nbu, 256, 0, L.stream>>>(psi, G.d_h64[0], nu);
      k_s32_to_s64<<<nbu, 256, 0, L.stream>>>(rho, G.d_h64[1], nu);
      for (int n = 0; n < ncy; n++) sap_cycle64(sargs64(mu, nmr), isolv);
      convert_f64_to_f32(G.d_h64[0], psi, nu, L.stream);
      convert_f64_to_f32(G.d_h64[1], rho, nu, L.stream);
      return;
   }
   SArgs a = sargs(mu, nmr);
   a.psi = psi;
   a.rho = rho;
   const int V = L.g.V;
   const unsigned nbk = (V + 255) / 256;
   const bool pz = zero && (reg_kernel() || lds_kernel() || G.ns);
   if (zero && !pz) HIP_OK(hipMemsetAsync(psi, 0, nu * sizeof(float2), L.stream));
   if (half_variant())
   {
      if (!pz) k_s32_to_h16<<<nbk, 256, 0, L.stream>>>(psi, G.d_h16[0], G.d_hsc[0], V);
      k_s32_to_h16<<<nbk, 256, 0, L.stream>>>(rho, G.d_h16[1], G.d_hsc[1], V);
   }
   for (int n = 0; n < ncy; n++)
   {
      // the blocks of both colours see psi = 0 in the first cycle
      a.pz = (n == 0 && pz);
      sap_cycle(a, isolv, n == 0, n == ncy - 1 && want_res);
   }
   if (half_variant())
   {
      k_h16_to_s32<<<nbk, 256, 0, L.stream>>>(G.d_h16[0], G.d_hsc[0], psi, V);
      if (want_res) k_h16_to_s32<<<nbk, 256, 0, L.stream>>>(G.d_h16[1], G.d_hsc[1], rho, V);
   }
}

// ncy Schwarz cycles (FP32) from psi = 0 on n sources at once (n <= 16):
// psi[k] and rho[k] are full FP32 device fields; each launch takes all
// sources.  False, with nothing done, if the face fields cannot be had.
bool sap_multi_device(float mu, int isolv, int nmr, int ncy, int n, float2 *const *psi, float2 *const *rho)
{
   if (n < 1 || n > 16 || !reg_kernel()) return false;
   const size_t nw = (size_t)G.nb * FUN;
   if (n > G.wfm_n)
   {
      HIP_OK(hipStreamSynchronize(lib().stream));
      dev_free(G.d_wfm);
      G.d_wfm = (float2 *)dev_try_alloc(n * nw * sizeof(float2));
      G.wfm_n = G.d_wfm ? n : 0;
      if (!G.d_wfm) return false;
   }
   SArgs a = sargs(mu, nmr);
   a.nsrc = n;
   for (int k = 0; k < n; k++)
   {
      a.pl[k] = psi[k];
      a.rl[k] = rho[k];
      a.wl[k] = G.d_wfm + (size_t)k * nw;
   }
   for (int c = 0; c < ncy; c++)
   {
      a.pz = (c == 0);
      sap_cycle(a, isolv, c == 0, c == ncy - 1);
   }
   return true;
}

// the FP16 residual of the last Schwarz cycles as an FP32 field
void sap_mixed_residual(float2 *r)
{
   Lib &L = lib();
   const int V = L.g.V;
   k_h16_to_s32<<<(V + 255) / 256, 256, 0, L.stream>>>(G.d_h16[1], G.d_hsc[1], r, V);
}

#ifndef OQH_SAP_GRAPH
#define OQH_SAP_GRAPH 1
#endif

// the Schwarz cycles of the FP16 preconditioner as one HIP graph: its kernel
// arguments depend only on rho (fixed within fgcr), the SAP parameters and
// the grid, so the graph is made when the same arguments come a second time
// in a row and replayed for every further Krylov vector; calls with
// changing arguments (the fields of dfl_modes) run eagerly
struct SapCall
{
   SArgs a;
   const float2 *rho = nullptr;
   int isolv = -1, ncy = -1, want_res = -1;
   bool same(const SapCall &o) const
   {
      return rho && rho == o.rho && isolv == o.isolv && ncy == o.ncy && want_res == o.want_res &&
             memcmp(&a, &o.a, sizeof(a)) == 0;
   }
};
static struct
{
   hipGraphExec_t exec = nullptr;
   SapCall made;  // the arguments of exec
   SapCall last;  // the arguments of the last eager call
} SG;

static void drop_sap_graph()
{
   if (SG.exec)
   {
      // a launch of the graph may still be running on the library stream
      HIP_OK(hipStreamSynchronize(lib().stream));
      HIP_OK(hipGraphExecDestroy(SG.exec));
   }
   SG.exec = nullptr;
   SG.made = SapCall();
   SG.last = SapCall();
}

// rho -> FP16, then ncy cycles from psi = 0 (enqueued on the library stream);
// the final face terms only if the residual is wanted
static void enqueue_mixed_cycles(const SArgs &a0, int isolv, int ncy, const float2 *rho, bool want_res)
{
   Lib &L = lib();
   const int V = L.g.V;
   SArgs a = a0;
   k_s32_to_h16<<<(V + 255) / 256, 256, 0, L.stream>>>(rho, G.d_h16[1], G.d_hsc[1], V);
   for (int n = 0; n < ncy; n++)
   {
      // the blocks of both colours see psi = 0 in the first cycle
      a.pz = (n == 0);
      sap_cycle(a, isolv, n == 0, n == ncy - 1 && want_res);
   }
}

// the SAP preconditioner of sap_gcr in the FP16 variant: ncy cycles on FP16
// fields starting from psi = 0, rho = rho_in, then phi = psi (sap_gcr.c:99-117
// with the fields kept in FP16).  The residual carried in FP16 no longer
// equals rho_in - D psi to FP32 accuracy, so the caller computes chi = D phi
// with the FP32 operator instead of taking rho_in - rho.
bool sap_mixed_mop(float mu, int isolv, int nmr, int ncy, const float2 *rho, float2 *phi, bool want_res)
{
   if (!half_variant()) return false;
   Lib &L = lib();
   const int V = L.g.V;
   SArgs a = sargs(mu, nmr);
   SapCall c;
   memset(&c.a, 0, sizeof(c.a));  // padding included, for the byte comparison
   c.a = a;
   c.rho = rho;
   c.isolv = isolv;
   c.ncy = ncy;
   c.want_res = (int)want_res;
   if (OQH_SAP_GRAPH && L.sap_graph && SG.exec && SG.made.same(c))
      HIP_OK(hipGraphLaunch(SG.exec, L.stream));
   else if (OQH_SAP_GRAPH && L.sap_graph && SG.last.same(c))
   {
      drop_sap_graph();
      hipGraph_t g;
      HIP_OK(hipStreamBeginCapture(L.stream, hipStreamCaptureModeThreadLocal));
      enqueue_mixed_cycles(a, isolv, ncy, rho, want_res);
      HIP_OK(hipStreamEndCapture(L.stream, &g));
      HIP_OK(hipGraphInstantiate(&SG.exec, g, nullptr, nullptr, 0));
      HIP_OK(hipGraphDestroy(g));
      SG.made = c;
      HIP_OK(hipGraphLaunch(SG.exec, L.stream));
   }
   else
   {
      enqueue_mixed_cycles(a, isolv, ncy, rho, want_res);
      SG.last = c;
   }
   k_h16_to_s32<<<(V + 255) / 256, 256, 0, L.stream>>>(G.d_h16[0], G.d_hsc[0], phi, V);
   return true;
}

__global__ void k_f32_to_f16(const float2 *__restrict__ a, __half2 *__restrict__ b, size_t n)
{
   size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
   if (i < n) b[i] = __float22half2_rn(a[i]);
}

// FP16 copies of the links and of the block SW field (FP16 variant)
static void ensure_half_fields()
{
   Lib &L = lib();
   size_t nu = units_for(L.g.V / 2, 72), ns = units_for(L.g.V, 36);
   if (!G.d_u16) G.d_u16 = (__half2 *)dev_alloc(nu * sizeof(__half2));
   if (!G.d_swb16) G.d_swb16 = (__half2 *)dev_alloc(ns * sizeof(__half2));
   for (int k = 0; k < 2; k++)
   {
      if (!G.d_h16[k]) G.d_h16[k] = (__half2 *)dev_alloc(units_for(L.g.V, 12) * sizeof(__half2));
      if (!G.d_hsc[k]) G.d_hsc[k] = (float *)dev_alloc((size_t)L.g.V * sizeof(float));
      if (!G.d_h16[k] || !G.d_hsc[k]) return;
   }
   if (!G.d_u16 || !G.d_swb16) return;
   if (G.u16_epoch != L.u_epoch)
   {
      k_f32_to_f16<<<(unsigned)((nu + 255) / 256), 256, 0, L.stream>>>(L.d_u, G.d_u16, nu);
      G.u16_epoch = L.u_epoch;
   }
   if (G.swb16_epoch != G.swb_version)
   {
      k_f32_to_f16<<<(unsigned)((ns + 255) / 256), 256, 0, L.stream>>>(G.d_swb, G.d_swb16, ns);
      G.swb16_epoch = G.swb_version;
   }
}

// grid, single-precision links and block SW field for the solver; returns
// false if the odd-point inversion is unsafe (reported as ifail=-3 by
// sap_gcr, as an error by sap)
bool sap_prepare(int isolv, const char *where, bool quiet)
{
   Lib &L = lib();
   if (!build_grid(where)) return false;
   if (!L.ud_set)
   {
      fail(where, "gauge field is not set");
      return false;
   }
   ensure_u();
   int want = isolv ? ODD_PTS : NO_PTS;
   if (!L.swd_valid || L.swd_inv[0] || L.swd_inv[1]) ensure_swd(0, 0);
   if (G.swb_set != want || G.swb_epoch != L.swd_epoch || (L.sap_prec == 2 && G.swb64_version != G.swb_version))
   {
      if (assign_swb(want))
      {
         G.swb_set = -1;
         if (!quiet) fail(where, "The inversion of the SW term was not safe");
         return false;
      }
   }
   if (L.sap_prec == 1 && G.bvol == RBV) ensure_half_fields();
   if (L.sap_prec == 2)
   {
      for (int k = 0; k < 3; k++)
         if (!G.d_h64[k]) G.d_h64[k] = (double2 *)dev_alloc(units_for(L.g.V, 12) * sizeof(double2));
      if (!G.d_scr64) G.d_scr64 = (double2 *)dev_alloc((size_t)G.nbh * 3 * G.Ub * sizeof(double2));
      if (!G.d_h64[0] || !G.d_h64[1] || !G.d_h64[2] || !G.d_scr64 || !G.d_swb64) return false;
   }
   return true;
}

// true if a wait in the Schwarz cycles since the last call was given up, so
// that what they left is wrong: an error at where (none for a null pointer).
// The caller has waited for the stream.
bool sap_gave_up(const char *where)
{
   if (!G.h_dead || !*(volatile int *)G.h_dead) return false;
   *G.h_dead = 0;
   if (where) fail(where, "a work-group of a Schwarz block did not get its neighbours' values");
   return true;
}

int sap_grid_nblocks() { return G.ready ? G.nb : 0; }

// the grid belongs to the geometry: released with it
void sap_release()
{
   drop_sap_graph();
   if (G.ready || G.d_bs || G.d_bsd) free_grid();
}

}  // namespace oqh

using namespace oqh;

extern "C" void sap(float mu, int isolv, int nmr, spinor *psi, spinor *eta)
{
   Lib &L = lib();
   if (!sap_prepare(isolv, "sap [sap.c]", false)) return;
   int V = L.g.V;
   Res p = resolve(psi, F32, V, 0, true);
   Res r = resolve(eta, F32, V, 1, true);
   if (!p.dev || !r.dev) return;
   if (p.off || r.off)
   {
      fail("sap [sap.c]", "the fields must be full fields");
      return;
   }
   sap_cycles(mu, isolv, nmr, 1, (float2 *)p.dev, (float2 *)r.dev, false, true);
   if (G.ns)
   {
      HIP_OK(hipStreamSynchronize(L.stream));
      if (sap_gave_up("sap [sap.c]")) return;
   }
   finish(p, F32, V, true);
   finish(r, F32, V, true);
}

// ---------------------------------------------------------------------------
// block-size autotuner (no counterpart in the reference)
// ---------------------------------------------------------------------------

// reproducible test field: uniform values in [-1, 1) from a hash of the index
__global__ void k_hash_fill(float2 *f, size_t n, unsigned long long seed)
{
   size_t k = (size_t)blockIdx.x * 256 + threadIdx.x;
   if (k >= n) return;
   unsigned long long z = seed + 0x9E3779B97F4A7C15ull * (k + 1);
   z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
   z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
   z ^= z >> 31;
   const float a = (float)(z & 0xffffff) * (1.0f / 8388608.0f) - 1.0f;
   const float b = (float)((z >> 24) & 0xffffff) * (1.0f / 8388608.0f) - 1.0f;
   f[k] = make_float2(a, b);
}

__global__ void k_sq_partial(const float2 *f, size_t n, double *part)
{
   __shared__ double sh[256];
   double s = 0.0;
   for (size_t k = (size_t)blockIdx.x * 256 + threadIdx.x; k < n; k += (size_t)gridDim.x * 256)
      s += (double)f[k].x * f[k].x + (double)f[k].y * f[k].y;
   sh[threadIdx.x] = s;
   __syncthreads();
   for (int m = 128; m > 0; m >>= 1)
   {
      if (threadIdx.x < m) sh[threadIdx.x] += sh[threadIdx.x + m];
      __syncthreads();
   }
   if (threadIdx.x == 0) part[blockIdx.x] = sh[0];
}

static double field_norm(const float2 *f, size_t n, double *d_part, double *h_part)
{
   Lib &L = lib();
   k_sq_partial<<<256, 256, 0, L.stream>>>(f, n, d_part);
   HIP_OK(hipMemcpyAsync(h_part, d_part, 256 * sizeof(double), hipMemcpyDeviceToHost, L.stream));
   HIP_OK(hipStreamSynchronize(L.stream));
   double s = 0.0;
   for (int b = 0; b < 256; b++) s += h_part[b];
   return sqrt(s);
}

// legal block sizes (sap_parms.c / README.block: even, >= 4, dividing the
// lattice with an even number of blocks per axis), spatially isotropic, at
// most maxvol points
static std::vector<std::array<int, 4>> block_candidates(const int *Lx, int maxvol)
{
   std::vector<std::array<int, 4>> out;
   auto legal = [](int l, int b) { return b >= 4 && b % 2 == 0 && l % b == 0 && (l / b) % 2 == 0; };
   for (int b0 = 4; b0 <= Lx[0]; b0 += 2)
      for (int bs = 4; bs <= std::min(Lx[1], std::min(Lx[2], Lx[3])); bs += 2)
      {
         if (!legal(Lx[0], b0) || !legal(Lx[1], bs) || !legal(Lx[2], bs) || !legal(Lx[3], bs)) continue;
         if ((long)b0 * bs * bs * bs > maxvol) continue;
         out.push_back({b0, bs, bs, bs});
      }
   return out;
}

extern "C" void oqh_set_sap_graph(int on)
{
   if (on != 0 && on != 1)
   {
      fail("oqh_set_sap_graph", "the argument must be 0 or 1");
      return;
   }
   lib().sap_graph = on;
}

extern "C" void oqh_set_sap_polls(int n)
{
   if (n < 1)
   {
      fail("oqh_set_sap_polls", "the number of polls must be positive");
      return;
   }
   lib().sap_polls = n;
}

extern "C" void oqh_set_sap_prec(int prec)
{
   if (prec != 0 && prec != 1 && prec != 2)
   {
      fail("oqh_set_sap_prec", "the precision must be 0 (FP32), 1 (FP16 storage) or 2 (FP64)");
      return;
   }
   lib().sap_prec = prec;
}

extern "C" void alloc_bgr(blk_grid_t grid)
{
   if (grid != SAP_BLOCKS)
   {
      fail("alloc_bgr [blk_grid.c]", "only the SAP_BLOCKS grid is provided");
      return;
   }
   build_grid("alloc_bgr [blk_grid.c]");
}

extern "C" void assign_ud2ubgr(blk_grid_t grid)
{
   (void)grid;
   Lib &L = lib();
   if (!require_geometry("assign_ud2ubgr [map_u2blk.c]")) return;
   L.u_valid = false;
   ensure_u();
}

extern "C" int assign_swd2swbgr(blk_grid_t grid, ptset_t set)
{
   if (grid != SAP_BLOCKS || !build_grid("assign_swd2swbgr [map_sw2blk.c]")) return 1;
   return assign_swb((int)set);
}

static bool blk_check(int n, int k, const char *where)
{
   if (!build_grid(where)) return false;
   if (n < 0 || n >= G.nb || k < 0 || k > 2)
   {
      fail(where, "Block number or field index is out of range");
      return false;
   }
   if (!G.d_bs) G.d_bs = (float2 *)dev_alloc((size_t)G.nb * NBF * G.Ub * sizeof(float2));
   return true;
}

static void blk_copy(int n, ptset_t set, int k, spinor *s, int to_blk, const char *where)
{
   Lib &L = lib();
   if (!blk_check(n, k, where)) return;
   Res r = resolve(s, F32, L.g.V, 0, true);
   if (!r.dev) return;
   int i0 = (set == ODD_PTS) ? G.bh : 0, i1 = (set == EVEN_PTS) ? G.bh : G.bvol;
   if (set == NO_PTS) i1 = i0;
   float2 *blk = G.d_bs + ((size_t)n * NBF + k) * G.Ub;
   if (i1 > i0)
      k_blk_copy<<<(i1 - i0 + 255) / 256, 256, 0, L.stream>>>((float2 *)r.dev, blk, G.d_imb + (size_t)n * G.bvol,
                                                              i0, i1, to_blk);
   finish(r, F32, L.g.V, !to_blk);
}

extern "C" void assign_s2sblk(blk_grid_t grid, int n, ptset_t set, spinor *s, int k)
{
   (void)grid;
   blk_copy(n, set, k, s, 1, "assign_s2sblk [map_s2blk.c]");
}

extern "C" void assign_sblk2s(blk_grid_t grid, int n, ptset_t set, int k, spinor *s)
{
   (void)grid;
   blk_copy(n, set, k, s, 0, "assign_sblk2s [map_s2blk.c]");
}

static void blk_op(int n, int op, int k, int l, float mu, int nmr, const char *where)
{
   Lib &L = lib();
   if (!blk_check(n, k, where) || !blk_check(n, l, where)) return;
   if (!L.ud_set)
   {
      fail(where, "gauge field is not set");
      return;
   }
   ensure_u();
   // the block SW field follows the SW term of the current gauge field and
   // parameters: it is (re)made with the last assigned point set (or the one
   // of the SAP parameters) when it is missing or older than the SW field
   if (G.swb_set < 0 || !L.swd_valid || G.swb_epoch != L.swd_epoch)
   {
      int set = (G.swb_set >= 0) ? G.swb_set : (L.sap_isolv ? ODD_PTS : NO_PTS);
      if (assign_swb(set))
      {
         G.swb_set = -1;
         fail(where, "The inversion of the SW term was not safe");
         return;
      }
   }
   SArgs a = sargs(mu, nmr);
   a.scr = G.d_bs;
   k_blk_op<<<1, SWG, 0, L.stream>>>(a, n, op, k, l, mu);
   HIP_OK(hipStreamSynchronize(L.stream));
}

extern "C" void Dw_blk(blk_grid_t grid, int n, float mu, int k, int l)
{
   (void)grid;
   if (k == l)
   {
      fail("Dw_blk [Dw.c]", "Input and output fields must be different");
      return;
   }
   blk_op(n, BOP_DW, k, l, mu, 0, "Dw_blk [Dw.c]");
}

extern "C" void Dwhat_blk(blk_grid_t grid, int n, float mu, int k, int l)
{
   (void)grid;
   if (k == l)
   {
      fail("Dwhat_blk [Dw.c]", "Input and output fields must be different");
      return;
   }
   blk_op(n, BOP_DWHAT, k, l, mu, 0, "Dwhat_blk [Dw.c]");
}

extern "C" void Dwee_blk(blk_grid_t grid, int n, float mu, int k, int l)
{
   (void)grid;
   blk_op(n, BOP_DWEE, k, l, mu, 0, "Dwee_blk [Dw.c]");
}

extern "C" void Dwoo_blk(blk_grid_t grid, int n, float mu, int k, int l)
{
   (void)grid;
   blk_op(n, BOP_DWOO, k, l, mu, 0, "Dwoo_blk [Dw.c]");
}

extern "C" void Dwoe_blk(blk_grid_t grid, int n, int k, int l)
{
   (void)grid;
   blk_op(n, BOP_DWOE, k, l, 0.0f, 0, "Dwoe_blk [Dw.c]");
}

extern "C" void Dweo_blk(blk_grid_t grid, int n, int k, int l)
{
   (void)grid;
   blk_op(n, BOP_DWEO, k, l, 0.0f, 0, "Dweo_blk [Dw.c]");
}

// ---------------------------------------------------------------------------
// double-precision block fields and operators (block/map_s2blk.c:
// assign_sd2sdblk, assign_sdblk2sd; dirac/Dw_dble.c:1891-2290): the same
// block kernels on FP64 block fields with the FP64 links and the FP64 block
// SW field (inverted on the point set of the single-precision one)
// ---------------------------------------------------------------------------

static bool blk_check64(int n, int k, const char *where)
{
   if (!blk_check(n, k, where)) return false;
   if (!G.d_bsd) G.d_bsd = (double2 *)dev_alloc((size_t)G.nb * NBF * G.Ub * sizeof(double2));
   if (!G.d_bsd) return false;
   return true;
}

static void blk_copy64(int n, ptset_t set, int k, spinor_dble *sd, int to_blk, const char *where)
{
   Lib &L = lib();
   if (!blk_check64(n, k, where)) return;
   Res r = resolve(sd, F64, L.g.V, 0, true);
   if (!r.dev) return;
   int i0 = (set == ODD_PTS) ? G.bh : 0, i1 = (set == EVEN_PTS) ? G.bh : G.bvol;
   if (set == NO_PTS) i1 = i0;
   double2 *blk = G.d_bsd + ((size_t)n * NBF + k) * G.Ub;
   if (i1 > i0)
      k_blk_copy<<<(i1 - i0 + 255) / 256, 256, 0, L.stream>>>((double2 *)r.dev, blk, G.d_imb + (size_t)n * G.bvol,
                                                              i0, i1, to_blk);
   finish(r, F64, L.g.V, !to_blk);
}

extern "C" void assign_sd2sdblk(blk_grid_t grid, int n, ptset_t set, spinor_dble *sd, int k)
{
   (void)grid;
   blk_copy64(n, set, k, sd, 1, "assign_sd2sdblk [map_s2blk.c]");
}

extern "C" void assign_sdblk2sd(blk_grid_t grid, int n, ptset_t set, int k, spinor_dble *sd)
{
   (void)grid;
   blk_copy64(n, set, k, sd, 0, "assign_sdblk2sd [map_s2blk.c]");
}

static void blk_op64(int n, int op, int k, int l, double mu, const char *where)
{
   Lib &L = lib();
   if (!blk_check64(n, k, where) || !blk_check64(n, l, where)) return;
   if (!L.ud_set)
   {
      fail(where, "gauge field is not set");
      return;
   }
   ensure_u();
   G.need64 = true;
   if (G.swb_set < 0 || !L.swd_valid || G.swb_epoch != L.swd_epoch || !G.d_swb64 ||
       G.swb64_version != G.swb_version)
   {
      int set = (G.swb_set >= 0) ? G.swb_set : (L.sap_isolv ? ODD_PTS : NO_PTS);
      if (assign_swb(set) || !G.d_swb64)
      {
         G.swb_set = -1;
         fail(where, "The inversion of the SW term was not safe");
         return;
      }
   }
   SArgsD a = sargs64(mu, 0);
   a.scr = G.d_bsd;
   k_blk_op<<<1, SWG, 0, L.stream>>>(a, n, op, k, l, mu);
   HIP_OK(hipStreamSynchronize(L.stream));
}

extern "C" void Dw_blk_dble(blk_grid_t grid, int n, double mu, int k, int l)
{
   (void)grid;
   if (k == l)
   {
      fail("Dw_blk_dble [Dw_dble.c]", "Input and output fields must be different");
      return;
   }
   blk_op64(n, BOP_DW, k, l, mu, "Dw_blk_dble [Dw_dble.c]");
}

extern "C" void Dwhat_blk_dble(blk_grid_t grid, int n, double mu, int k, int l)
{
   (void)grid;
   if (k == l)
   {
      fail("Dwhat_blk_dble [Dw_dble.c]", "Input and output fields must be different");
      return;
   }
   blk_op64(n, BOP_DWHAT, k, l, mu, "Dwhat_blk_dble [Dw_dble.c]");
}

extern "C" void Dwee_blk_dble(blk_grid_t grid, int n, double mu, int k, int l)
{
   (void)grid;
   blk_op64(n, BOP_DWEE, k, l, mu, "Dwee_blk_dble [Dw_dble.c]");
}

extern "C" void Dwoo_blk_dble(blk_grid_t grid, int n, double mu, int k, int l)
{
   (void)grid;
   blk_op64(n, BOP_DWOO, k, l, mu, "Dwoo_blk_dble [Dw_dble.c]");
}

extern "C" void Dwoe_blk_dble(blk_grid_t grid, int n, int k, int l)
{
   (void)grid;
   blk_op64(n, BOP_DWOE, k, l, 0.0, "Dwoe_blk_dble [Dw_dble.c]");
}

extern "C" void Dweo_blk_dble(blk_grid_t grid, int n, int k, int l)
{
   (void)grid;
   blk_op64(n, BOP_DWEO, k, l, 0.0, "Dweo_blk_dble [Dw_dble.c]");
}

// FP64 block field k of block n as a host array in block order (test access)
extern "C" void oqh_export_sdblk(int n, int k, spinor_dble *host)
{
   Lib &L = lib();
   if (!blk_check64(n, k, "oqh_export_sdblk")) return;
   size_t bytes = (size_t)G.bvol * sizeof(spinor_dble);
   void *aos = tmp_buffer(bytes);
   blocks_to_aos_f64(G.d_bsd + ((size_t)n * NBF + k) * G.Ub, (double2 *)aos, G.bvol, 12, L.stream);
   HIP_OK(hipMemcpyAsync(host, aos, bytes, hipMemcpyDeviceToHost, L.stream));
   HIP_OK(hipStreamSynchronize(L.stream));
}

extern "C" void Dw_bnd(blk_grid_t grid, int n, int k, int l)
{
   Lib &L = lib();
   const char *where = "Dw_bnd [Dw_bnd.c]";
   (void)grid;
   if (!blk_check(n, k, where)) return;
   if (l != 0)
   {
      fail(where, "Parameters are out of range");
      return;
   }
   if (!L.ud_set)
   {
      fail(where, "gauge field is not set");
      return;
   }
   ensure_u();
   if (!G.d_bw)
   {
      G.d_bw = (float2 *)dev_alloc(sizeof(float2) * 6 * (size_t)G.nb * G.fofs[8]);
      if (!G.d_bw) return;
   }
   SArgs a = sargs(0.0f, 0);
   a.scr = G.d_bs;
   FaceOfs fo;
   memcpy(fo.o, G.fofs, sizeof(fo.o));
   k_dw_bnd<<<1, SWG, 0, L.stream>>>(a, n, k, G.d_ipp, fo, G.d_bw);
   HIP_OK(hipStreamSynchronize(L.stream));
}

extern "C" void oqh_export_bnd(int n, int ifc, int l, weyl *w)
{
   Lib &L = lib();
   const char *where = "oqh_export_bnd";
   if (!blk_check(n, 0, where)) return;
   if (ifc < 0 || ifc > 7 || l != 0 || !G.d_bw)
   {
      fail(where, "no such boundary field (Dw_bnd has not been called or parameters out of range)");
      return;
   }
   const size_t off = ((size_t)n * G.fofs[8] + G.fofs[ifc]) * 6;
   const size_t cnt = (size_t)(G.fofs[ifc + 1] - G.fofs[ifc]) * 6;
   HIP_OK(hipMemcpyAsync(w, G.d_bw + off, cnt * sizeof(float2), hipMemcpyDeviceToHost, L.stream));
   HIP_OK(hipStreamSynchronize(L.stream));
}

extern "C" void blk_mres(int n, float mu, int nmr)
{
   blk_op(n, BOP_MRES, 0, 2, mu, nmr, "blk_mres [blk_solv.c]");
}

extern "C" void blk_eo_mres(int n, float mu, int nmr)
{
   blk_op(n, BOP_EO_MRES, 0, 2, mu, nmr, "blk_eo_mres [blk_solv.c]");
}

extern "C" void oqh_export_sblk(int n, int k, spinor *host)
{
   Lib &L = lib();
   if (!blk_check(n, k, "oqh_export_sblk")) return;
   size_t bytes = (size_t)G.bvol * sizeof(spinor);
   void *aos = tmp_buffer(bytes);
   blocks_to_aos_f32(G.d_bs + ((size_t)n * NBF + k) * G.Ub, (float2 *)aos, G.bvol, 12, L.stream);
   HIP_OK(hipMemcpyAsync(host, aos, bytes, hipMemcpyDeviceToHost, L.stream));
   HIP_OK(hipStreamSynchronize(L.stream));
}

extern "C" void oqh_get_imb(int n, int *imb)
{
   if (!build_grid("oqh_get_imb")) return;
   memcpy(imb, G.imb.data() + (size_t)n * G.bvol, sizeof(int) * G.bvol);
}

// Chooses the SAP block size with the least time per e-fold of residual
// reduction: for every candidate, ncy Schwarz cycles with the given isolv and
// nmr (current precision variant) on a reproducible test residual, timed
// with HIP events after one warm-up cycle.  On success only the block size of
// the SAP parameters changes (isolv, nmr and ncy keep their values; if no SAP
// parameters were set, they become the given ones); on failure nothing
// changes.  Returns the best time per e-fold in seconds (0 on failure).
extern "C" double oqh_sap_autotune(int isolv, int nmr, int ncy, int maxvol, int *bs_out)
{
   const char *where = "oqh_sap_autotune";
   Lib &L = lib();
   if (!require_geometry(where)) return 0.0;
   if (!L.ud_set)
   {
      fail(where, "gauge field is not set");
      return 0.0;
   }
   if (maxvol <= 0) maxvol = 4096;
   auto cand = block_candidates(L.g.L, maxvol);
   if (cand.empty())
   {
      fail(where, "no legal block size");
      return 0.0;
   }
   const size_t nu = units_for(L.g.V, 12);
   float2 *psi = (float2 *)dev_alloc(nu * sizeof(float2));
   float2 *rho = (float2 *)dev_alloc(nu * sizeof(float2));
   double *d_part = (double *)dev_alloc(256 * sizeof(double));
   double *h_part = nullptr;
   HIP_OK(hipHostMalloc((void **)&h_part, 256 * sizeof(double), 0));
   hipEvent_t e0, e1;
   HIP_OK(hipEventCreate(&e0));
   HIP_OK(hipEventCreate(&e1));
   double best = 0.0;
   std::array<int, 4> bbest = cand[0];
   const int keep[4] = {L.sap_bs[0], L.sap_bs[1], L.sap_bs[2], L.sap_bs[3]};
   const int keep_isolv = L.sap_isolv, keep_nmr = L.sap_nmr, keep_ncy = L.sap_ncy;
   for (const auto &bs : cand)
   {
      memcpy(L.sap_bs, bs.data(), sizeof(L.sap_bs));
      L.sap_isolv = isolv;
      L.sap_nmr = nmr;
      L.sap_ncy = ncy;
      if (!psi || !rho || !sap_prepare(isolv, where, true)) continue;
      const unsigned nbk = (unsigned)((nu + 255) / 256);
      // warm-up cycle
      HIP_OK(hipMemsetAsync(psi, 0, nu * sizeof(float2), L.stream));
      k_hash_fill<<<nbk, 256, 0, L.stream>>>(rho, nu, 12345);
      sap_cycles(0.0f, isolv, nmr, 1, psi, rho, false, true);
      HIP_OK(hipMemsetAsync(psi, 0, nu * sizeof(float2), L.stream));
      k_hash_fill<<<nbk, 256, 0, L.stream>>>(rho, nu, 12345);
      const double r0 = field_norm(rho, nu, d_part, h_part);
      HIP_OK(hipEventRecord(e0, L.stream));
      sap_cycles(0.0f, isolv, nmr, ncy, psi, rho, false, true);
      HIP_OK(hipEventRecord(e1, L.stream));
      HIP_OK(hipEventSynchronize(e1));
      float ms = 0.0f;
      HIP_OK(hipEventElapsedTime(&ms, e0, e1));
      const double r1 = field_norm(rho, nu, d_part, h_part);
      if (sap_gave_up(nullptr) || !(r1 > 0.0) || r1 >= r0) continue;
      const double score = 1e-3 * ms / log(r0 / r1);
      if (best == 0.0 || score < best)
      {
         best = score;
         bbest = bs;
      }
   }
   HIP_OK(hipEventDestroy(e0));
   HIP_OK(hipEventDestroy(e1));
   HIP_OK(hipHostFree(h_part));
   dev_free(psi);
   dev_free(rho);
   dev_free(d_part);
   if (keep_ncy != 0 || best == 0.0)
   {
      // SAP parameters set before keep isolv, nmr and ncy
      L.sap_isolv = keep_isolv;
      L.sap_nmr = keep_nmr;
      L.sap_ncy = keep_ncy;
   }
   if (best == 0.0)
   {
      memcpy(L.sap_bs, keep, sizeof(L.sap_bs));
      fail(where, "no block size reduced the residual");
      return 0.0;
   }
   memcpy(L.sap_bs, bbest.data(), sizeof(L.sap_bs));
   for (int mu = 0; mu < 4; mu++) bs_out[mu] = bbest[mu];
   return best;
}

