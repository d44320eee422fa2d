// ptc.hip -- gauge-equivariant network used as a learned preconditioner of
// sap_gcr (no counterpart in the reference).
//
// A field with C channels holds C colour vectors per point in the unit
// layout of the spinor fields (unit 3 i + a of point x is channel i, colour
// a; a spinor is the field with its 4 spin components as channels).  One
// layer maps C_in to C_out channels through the parallel-transport stencil
//
//    out(x)[o] = sum_{p=0..8} sum_i W[p][o][i] (T_p in)(x)[i],
//    T_0 = 1,  T_{2mu+1} in(x) = U(x,mu) in(x+mu),
//    T_{2mu+2} in(x) = U(x-mu,mu)^+ in(x-mu),
//
// with complex weights acting on the channel index only (the layer commutes
// with gauge transformations).  The network is linear: a learned
// approximation of D^-1 applied to the residual that the Schwarz cycles
// leave.
//
// k_ptc: a work-group takes 128 points.  For two directions p at a time its
// threads transport the input channels of the neighbours with the links (FP32
// in training, an FP16 copy in the preconditioner, where the links are most
// of the bytes a layer reads) and store them as BF16 in LDS (a K x N matrix, K = real and imaginary
// parts of the C_in channels, N = 3 colours x 128 points); the channel
// mixing is then a real GEMM [2 C_out x K] x [K x N] on the matrix cores
// (v_mfma_f32_32x32x16_bf16, FP32 accumulation over the 9 directions), the
// weights in the real form [[Re W, -Im W], [Im W, Re W]] as BF16.  The
// input gradient of a layer is the same kernel with the weights
// W'[p] = W[pbar]^+ (T_p^+ = T_pbar); the weight gradient
// dW[p][o][i] = sum_{x,a} g(x)[o][a] conj((T_p in)(x)[i][a]) is formed per
// 128 points by FP32 matrix instructions and summed in double.
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "dirac_dev.h"
#include "oqh_internal.h"

namespace oqh {

constexpr int NDIR = 9;
constexpr int PNS = 128;  // points per work-group
constexpr int PWG = 256;  // threads per work-group
constexpr int NLMAX = 8;  // layers
constexpr int CMAX = 16;  // channels
constexpr int NBMAX = 16; // pairs of a training batch per launch

// inputs and outputs of the samples of a launch (blockIdx.y)
struct Batch
{
   const void *in[NBMAX];
   void *out[NBMAX];
};

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// K of one direction (2 C reals) rounded up to the MFMA depth 16
__host__ __device__ constexpr int kpad(int c) { return ((2 * c + 15) / 16) * 16; }

__device__ inline int pbar_of(int p) { return p == 0 ? 0 : ((p & 1) ? p + 1 : p - 1); }

// address of the link of the transport T_p at point x (neighbour y), and
// whether it enters daggered
template <typename UL>
__device__ inline const UL *ptc_link(const UL *u, int x, int y, int p, int h, bool &dag)
{
   const int mu = (p - 1) >> 1;
   const bool fwd = p & 1;
   dag = !fwd;
   if (fwd) return (x >= h) ? link_ptr(u, x - h, 2 * mu) : link_ptr(u, y - h, 2 * mu + 1);
   return (x >= h) ? link_ptr(u, x - h, 2 * mu + 1) : link_ptr(u, y - h, 2 * mu);
}

__device__ inline int ptc_nbr(const int *nbr, int V, int x, int p)
{
   if (p == 0) return x;
   const int mu = (p - 1) >> 1;
   return nbr[(size_t)((p & 1) ? 2 * mu : 2 * mu + 1) * V + x] & 0x7fffffff;
}

// activations: FP32 complex numbers (training, the network's input and
// output), or BF16 pairs between the layers of the preconditioner
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

__device__ inline float2 ld_act(const float2 *p, size_t i) { return p[i]; }
__device__ inline float2 ld_act(const bf16x2 *p, size_t i)
{
   const bf16x2 b = p[i];
   return make_float2((float)b.x, (float)b.y);
}
__device__ inline void st_act(float2 *p, size_t i, float2 v) { p[i] = v; }
__device__ inline void st_act(bf16x2 *p, size_t i, float2 v)
{
   bf16x2 b;
   b.x = (__bf16)v.x;
   b.y = (__bf16)v.y;
   p[i] = b;
}

// links: FP32, or the FP16 copy that the preconditioner reads
__device__ inline float2 lnk(float2 v) { return v; }
__device__ inline float2 lnk(__half2 v) { return __half22float2(v); }

// out (+)= layer(in); wp: packed BF16 weights [9][32][kpad(CI)].  Two
// directions per phase (five phases): the two halves of the work-group
// transport all input channels of their point for direction 2q and 2q+1,
// so every link is loaded once, and one barrier pair serves two directions.
// accum (out += ...) only with FP32 output.
template <int CI, int CO, typename TI = float2, typename TO = float2, typename UL = float2>
__global__ __launch_bounds__(PWG) void k_ptc(Batch bt, const __bf16 *__restrict__ wp, const UL *__restrict__ u,
                                             const int *__restrict__ nbr, int V, int accum)
{
   const TI *__restrict__ in = (const TI *)bt.in[blockIdx.y];
   TO *__restrict__ out = (TO *)bt.out[blockIdx.y];
   constexpr int KP = kpad(CI);
   constexpr int LD = 2 * KP + 8;  // LDS row stride (bf16): two direction blocks
   static_assert(2 * CO <= 32 && CI % 2 == 0, "channel counts");
   __shared__ __attribute__((aligned(16))) __bf16 Bt[3 * PNS * LD];
   const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
   const int x0 = blockIdx.x * PNS, h = V / 2;
   for (int q = t; q < 3 * PNS; q += PWG)
      for (int k = 2 * CI; k < KP; k++) Bt[q * LD + k] = Bt[q * LD + KP + k] = (__bf16)0.0f;
   f32x16 acc[3];
#pragma unroll
   for (int tt = 0; tt < 3; tt++)
#pragma unroll
      for (int j = 0; j < 16; j++) acc[tt][j] = 0.0f;
   const int s = t & (PNS - 1), hh = t >> 7;
   const int x = x0 + s;
   for (int ph = 0; ph < (NDIR + 1) / 2; ph++)
   {
      const int p = 2 * ph + hh;
      __bf16 *brow = Bt + s * LD + hh * KP;
      if (x < V && p < NDIR)
      {
         const int y = ptc_nbr(nbr, V, x, p);
         float2 um[9];
         bool dag = false;
         if (p > 0)
         {
            const UL *up = ptc_link(u, x, y, p, h, dag);
#pragma unroll
            for (int k = 0; k < 9; k++) um[k] = lnk(up[k * SB]);
         }
         // all loads first (independent), then the products
         float2 v[CI][3];
#pragma unroll
         for (int i = 0; i < CI; i++)
#pragma unroll
            for (int a = 0; a < 3; a++) v[i][a] = ld_act(in, unit_index(y, 3 * i + a, 3 * CI));
#pragma unroll
         for (int i = 0; i < CI; i++)
         {
            float2 w[3];
            if (p == 0)
            {
#pragma unroll
               for (int a = 0; a < 3; a++) w[a] = v[i][a];
            }
            else if (dag)
               su3_mul<float2, true>(um, v[i], w);
            else
               su3_mul<float2, false>(um, v[i], w);
#pragma unroll
            for (int a = 0; a < 3; a++)
            {
               bf16x2 b;
               b.x = (__bf16)w[a].x;
               b.y = (__bf16)w[a].y;
               *(bf16x2 *)(brow + a * PNS * LD + 2 * i) = b;
            }
         }
      }
      else
      {
         bf16x2 z;
         z.x = z.y = (__bf16)0.0f;
#pragma unroll
         for (int i = 0; i < CI; i++)
#pragma unroll
            for (int a = 0; a < 3; a++) *(bf16x2 *)(brow + a * PNS * LD + 2 * i) = z;
      }
      __syncthreads();
#pragma unroll
      for (int tt = 0; tt < 3; tt++)
      {
         const int n = (wv + 4 * tt) * 32 + (lane & 31);
#pragma unroll
         for (int d = 0; d < 2; d++)
         {
            const int pd = 2 * ph + d;
            if (pd >= NDIR) break;
#pragma unroll
            for (int k0 = 0; k0 < KP; k0 += 16)
            {
               const bf16x8 a = *(const bf16x8 *)(wp + (size_t)(pd * 32 + (lane & 31)) * KP + k0 + 8 * (lane >> 5));
               const bf16x8 b = *(const bf16x8 *)(Bt + n * LD + d * KP + k0 + 8 * (lane >> 5));
               acc[tt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc[tt], 0, 0, 0);
            }
         }
      }
      __syncthreads();
   }
   // D[m][n]: lane holds n = lane % 32 and rows 8 (j/4) + 4 (lane/32) + j%4;
   // rows 2o, 2o+1 are Re and Im of channel o
#pragma unroll
   for (int tt = 0; tt < 3; tt++)
   {
      const int n = (wv + 4 * tt) * 32 + (lane & 31);
      const int a = n / PNS, xo = x0 + n % PNS;
      if (xo >= V) continue;
#pragma unroll
      for (int j = 0; j < 16; j += 2)
      {
         const int m = 8 * (j >> 2) + 4 * (lane >> 5) + (j & 3);
         const int o = m >> 1;
         if (o < CO)
         {
            float2 v = make_float2(acc[tt][j], acc[tt][j + 1]);
            const size_t id = unit_index(xo, 3 * o + a, 3 * CO);
            if (accum)
            {
               float2 w = ld_act(out, id);
               v.x += w.x;
               v.y += w.y;
            }
            st_act(out, id, v);
         }
      }
   }
}

// packed BF16 weights of a layer with ci inputs and co outputs from the
// complex weights w[9][co][ci]; adj: the adjoint layer (co inputs, ci
// outputs) with W'[p] = W[pbar]^+
__global__ void k_ptc_pack(const float2 *w, int ci, int co, int adj, __bf16 *wp)
{
   const int p = blockIdx.x;
   const int cin = adj ? co : ci, cout = adj ? ci : co;
   const int KP = kpad(cin);
   for (int e = threadIdx.x; e < 32 * KP; e += blockDim.x)
   {
      const int m = e / KP, k = e % KP;
      const int o = m >> 1, r = m & 1, i = k >> 1, q = k & 1;
      float val = 0.0f;
      if (o < cout && i < cin)
      {
         float2 z;
         if (!adj)
            z = w[((size_t)p * co + o) * ci + i];
         else
         {
            float2 y = w[((size_t)pbar_of(p) * co + i) * ci + o];
            z = make_float2(y.x, -y.y);
         }
         // [[Re, -Im], [Im, Re]]
         val = (r == q) ? z.x : (r == 0 ? -z.y : z.y);
      }
      wp[((size_t)p * 32 + m) * KP + k] = (__bf16)val;
   }
}

// Partial weight gradients: part[b][p][o][i] for the point sets b; nothing is
// taken from a sample without target (sums, k_ptc_loss_sum).
//
// With real and imaginary parts as rows the products sum_x g(x) conj(t(x))^T
// are real GEMMs [2 C_out x K] x [K x 2 C_in], K = 3 colours x 128 points, on
// the FP32 matrix instructions (v_mfma_f32_16x16x4_f32: FP32 products and
// sums, as the fused multiply-adds they replace).  The transported channels
// go to LDS as [K][2 C_in]; each wave owns one 16 x 16 tile of the result (or,
// with fewer than four tiles, a share of K) and keeps its rows of g, which
// are the same for all nine directions, in registers.  Two wavefronts per SIMD
// (with one, 255 + 4 registers, a layer of 8 samples took 0.84 ms): the loads
// of one work-group overlap the 96 matrix instructions per direction of the
// other.  The gradient of 8 pairs at 16^4 (4-12-16-12-4) takes 4.0 ms against
// 13.0 ms with scalar products of the LDS rows and a sum over the
// work-groups by one thread per element.
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int WG_TILES(int ci, int co) { return ((2 * co + 15) / 16) * ((2 * ci + 15) / 16); }
constexpr int WG_KSPLIT(int ci, int co) { return 4 / WG_TILES(ci, co); }  // point sets per work-group

template <int CI, int CO>
__global__ __launch_bounds__(PWG) __attribute__((amdgpu_waves_per_eu(2))) void k_ptc_wgrad(Batch bt, const float2 *__restrict__ u,
                                                   const int *__restrict__ nbr, int V, const double *__restrict__ sums,
                                                   float2 *part)
{
   const float2 *__restrict__ in = (const float2 *)bt.in[blockIdx.y];
   const float2 *__restrict__ g = (const float2 *)bt.out[blockIdx.y];  // output gradients
   constexpr int NT = (2 * CI + 15) / 16, TILES = WG_TILES(CI, CO), KS = WG_KSPLIT(CI, CO);
   constexpr int CM = CI > CO ? CI : CO;
   // rows of 16-column tiles, padded by one pair against bank conflicts
   constexpr int LD = ((2 * CM + 15) / 16) * 16 + 2;
   constexpr int STEPS = 3 * PNS / 4 / KS;  // matrix instructions per wave, tile and direction
   __shared__ float T[3 * PNS][LD];
   const int t = threadIdx.x, x0 = blockIdx.x * PNS, h = V / 2;
   const int lane = t & 63, w = t >> 6;
   const int tile = w % TILES, ks = w / TILES;
   const int mt = tile / NT, nt = tile % NT;
   const int row = lane & 15, kk = lane >> 4;
   const int s = t & (PNS - 1), hh = t >> 7;
   const int x = x0 + s;
   const bool live = x < V && sums[2 * blockIdx.y] != 0.0;
   for (int e = t; e < 3 * PNS * LD; e += PWG) (&T[0][0])[e] = 0.0f;
   __syncthreads();
   if (live)
      for (int c = hh; c < 3 * CO; c += 2)
      {
         const float2 v = g[unit_index(x, c, 3 * CO)];
         *(float2 *)&T[(c % 3) * PNS + s][2 * (c / 3)] = v;
      }
   __syncthreads();
   float A[STEPS];
#pragma unroll
   for (int k = 0; k < STEPS; k++) A[k] = T[(ks * STEPS + k) * 4 + kk][16 * mt + row];
   __syncthreads();
   // the columns beyond C_in must be zero where g had values
   if (CI < CO)
   {
      for (int e = t; e < 3 * PNS * LD; e += PWG) (&T[0][0])[e] = 0.0f;
      __syncthreads();
   }
   constexpr int CH = CI / 2;
   int yn = x;  // neighbour of the next direction, one step ahead
   for (int p = 0; p < NDIR; p++)
   {
      if (live)
      {
         const int y = yn;
         if (p + 1 < NDIR) yn = ptc_nbr(nbr, V, x, p + 1);
         float2 um[9];
         bool dag = false;
         if (p > 0)
         {
            const float2 *up = ptc_link(u, x, y, p, h, dag);
#pragma unroll
            for (int k = 0; k < 9; k++) um[k] = up[k * SB];
         }
         float2 v[CH][3];
#pragma unroll
         for (int c = 0; c < CH; c++)
#pragma unroll
            for (int a = 0; a < 3; a++) v[c][a] = in[unit_index(y, 3 * (hh * CH + c) + a, 3 * CI)];
#pragma unroll
         for (int c = 0; c < CH; c++)
         {
            float2 z[3];
            if (p == 0)
            {
#pragma unroll
               for (int a = 0; a < 3; a++) z[a] = v[c][a];
            }
            else if (dag)
               su3_mul<float2, true>(um, v[c], z);
            else
               su3_mul<float2, false>(um, v[c], z);
#pragma unroll
            for (int a = 0; a < 3; a++) *(float2 *)&T[a * PNS + s][2 * (hh * CH + c)] = z[a];
         }
      }
      else
      {
         for (int c = 0; c < CH; c++)
            for (int a = 0; a < 3; a++) *(float2 *)&T[a * PNS + s][2 * (hh * CH + c)] = make_float2(0.0f, 0.0f);
      }
      __syncthreads();
      f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int k = 0; k < STEPS; k++)
      {
         const float b = T[(ks * STEPS + k) * 4 + kk][16 * nt + row];
         acc = __builtin_amdgcn_mfma_f32_16x16x4f32(A[k], b, acc, 0, 0, 0);
      }
      // lane: column n = 16 nt + lane % 16, rows m = 16 mt + 4 (lane / 16) + r;
      // (2o, 2o+1) and (2i, 2i+1) are real and imaginary parts
#pragma unroll
      for (int r = 0; r < 4; r += 2)
      {
         const float re1 = __shfl_xor(acc[r + 1], 1), im1 = __shfl_xor(acc[r], 1);
         const int o = 8 * mt + 2 * kk + (r >> 1), i = 8 * nt + (row >> 1);
         if (!(row & 1) && o < CO && i < CI)
            part[((((size_t)blockIdx.y * gridDim.x + blockIdx.x) * KS + ks) * NDIR + p) * CO * CI + o * CI + i] =
                make_float2(acc[r] + re1, acc[r + 1] - im1);
      }
      __syncthreads();
   }
}

// grad[e] += sum over the point sets b < nb of part[b][e] (double, fixed
// order): 64 elements per work-group, each of the 16 waves takes every 16th
// set
constexpr int WSW = 16;

__global__ __launch_bounds__(64 * WSW) void k_ptc_wgrad_sum(const float2 *part, int nb, int n, float2 *grad)
{
   __shared__ double2 sh[WSW][64];
   const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, e = blockIdx.x * 64 + lane;
   double zr = 0.0, zi = 0.0;
   if (e < n)
      for (int b = w; b < nb; b += WSW)
      {
         const float2 v = part[(size_t)b * n + e];
         zr += v.x;
         zi += v.y;
      }
   sh[w][lane] = make_double2(zr, zi);
   __syncthreads();
   if (w || e >= n) return;
   for (int k = 1; k < WSW; k++)
   {
      zr += sh[k][lane].x;
      zi += sh[k][lane].y;
   }
   grad[e].x += (float)zr;
   grad[e].y += (float)zi;
}

// whether unit k of a spinor field belongs to a point: the last storage block
// may have more than the lattice
__device__ inline bool unit_used(int k, int V)
{
   return V % SB == 0 || k / (12 * SB) * SB + (k & (SB - 1)) < V;
}

// loss terms of a sample (blockIdx.y): partial sums of |e|^2 and |out - e|^2
__global__ void k_ptc_loss(Batch bt, int V, int n, double *part)
{
   const float2 *out = (const float2 *)bt.out[blockIdx.y], *e = (const float2 *)bt.in[blockIdx.y];
   __shared__ double sh[2][256];
   double se = 0.0, sd = 0.0;
   auto add = [&](int k)
   {
      float2 a = out[k], b = e[k];
      double dx = (double)a.x - b.x, dy = (double)a.y - b.y;
      se += (double)b.x * b.x + (double)b.y * b.y;
      sd += dx * dx + dy * dy;
   };
   const int full = V / SB * (12 * SB);  // units of full storage blocks
   int k = blockIdx.x * 256 + threadIdx.x;
   for (; k < full; k += gridDim.x * 256) add(k);
   for (; k < n; k += gridDim.x * 256)
      if (unit_used(k, V)) add(k);
   sh[0][threadIdx.x] = se;
   sh[1][threadIdx.x] = sd;
   __syncthreads();
   for (int m = 128; m > 0; m >>= 1)
   {
      if (threadIdx.x < m)
      {
         sh[0][threadIdx.x] += sh[0][threadIdx.x + m];
         sh[1][threadIdx.x] += sh[1][threadIdx.x + m];
      }
      __syncthreads();
   }
   if (threadIdx.x == 0)
   {
      double *p = part + 2 * ((size_t)blockIdx.y * gridDim.x + blockIdx.x);
      p[0] = sh[0][0];
      p[1] = sh[1][0];
   }
}

// |e|^2 and |out - e|^2 of a sample (one wave each, fixed order)
__global__ __launch_bounds__(64) void k_ptc_loss_sum(const double *part, int nb, double *sums)
{
   double se = 0.0, sd = 0.0;
   const double *p = part + 2 * (size_t)blockIdx.x * nb;
   for (int b = threadIdx.x; b < nb; b += 64)
   {
      se += p[2 * b];
      sd += p[2 * b + 1];
   }
   for (int m = 32; m >= 1; m >>= 1)
   {
      se += __shfl_xor(se, m);
      sd += __shfl_xor(sd, m);
   }
   if (threadIdx.x == 0)
   {
      sums[2 * blockIdx.x] = se;
      sums[2 * blockIdx.x + 1] = sd;
   }
}

// output gradient of the mean loss over npair pairs, g = 2 (out - e) /
// (npair |e|^2) in place of out (0 for a pair without target)
__global__ void k_ptc_lgrad(Batch bt, const double *sums, int npair, int V, int n)
{
   const float2 *e = (const float2 *)bt.in[blockIdx.y];
   float2 *g = (float2 *)bt.out[blockIdx.y];
   const double se = sums[2 * blockIdx.y];
   const float c = (float)(2.0 / (se * npair));
   const int k = blockIdx.x * 256 + threadIdx.x;
   if (k >= n || !unit_used(k, V)) return;
   g[k] = se != 0.0 ? make_float2(c * (g[k].x - e[k].x), c * (g[k].y - e[k].y)) : make_float2(0.0f, 0.0f);
}

// Adam step on n reals
__global__ void k_adam(float *w, const float *g, float *m, float *v, int n, float lr, float b1, float b2, float eps,
                       float c1, float c2)
{
   const int k = blockIdx.x * 256 + threadIdx.x;
   if (k >= n) return;
   const float gk = g[k];
   m[k] = b1 * m[k] + (1.0f - b1) * gk;
   v[k] = b2 * v[k] + (1.0f - b2) * gk * gk;
   w[k] -= lr * (m[k] * c1) / (sqrtf(v[k] * c2) + eps);
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------

__global__ void k_ptc_link16(const float2 *a, __half2 *b, size_t n)
{
   const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
   if (i < n) b[i] = __float22half2_rn(a[i]);
}

namespace {

struct Net
{
   int nl = 0;
   int w[NLMAX + 1] = {};
   size_t off[NLMAX + 1] = {};           // offsets of the layers in the weight array
   float2 *d_w = nullptr, *d_g = nullptr;  // complex weights and gradients
   float *d_m = nullptr, *d_v = nullptr;   // Adam moments
   __bf16 *d_pf[NLMAX] = {}, *d_pa[NLMAX] = {};
   bool packed = false;
   int adam_t = 0;
   int V = 0;
   int nbatch = 0;                 // samples the following fields hold
   int cap = NBMAX;                // samples there was memory for
   float2 *d_act[NLMAX + 1] = {};  // activations of the last forward
   float2 *d_gb[2] = {};           // outputs, then the gradients of the layers (ping-pong)
   float2 *d_part = nullptr;       // weight-gradient partials
   double *d_lpart = nullptr, *d_lsum = nullptr, *h_lsum = nullptr;  // loss terms
   float2 *d_tmp = nullptr;         // spinor work field of the preconditioner
   bf16x2 *d_inf[2] = {};           // BF16 activations of the preconditioner (ping-pong)
   __half2 *d_u16 = nullptr;        // FP16 links of the preconditioner
   int u16_epoch = -1;              // link epoch of d_u16
};

Net N;

bool valid_width(int c) { return c == 4 || c == 8 || c == 12 || c == 16; }

void free_net()
{
   dev_free(N.d_w); dev_free(N.d_g); dev_free(N.d_m); dev_free(N.d_v);
   for (int l = 0; l < NLMAX; l++) { dev_free(N.d_pf[l]); dev_free(N.d_pa[l]); }
   for (int l = 0; l <= NLMAX; l++) dev_free(N.d_act[l]);
   dev_free(N.d_gb[0]); dev_free(N.d_gb[1]); dev_free(N.d_part); dev_free(N.d_lpart); dev_free(N.d_lsum); dev_free(N.d_tmp);
   dev_free(N.d_inf[0]); dev_free(N.d_inf[1]); dev_free(N.d_u16);
   if (N.h_lsum) HIP_OK(hipHostFree(N.h_lsum));
   N = Net();
}

size_t nweights() { return N.off[N.nl]; }

void pack()
{
   if (N.packed) return;
   Lib &L = lib();
   for (int l = 0; l < N.nl; l++)
   {
      k_ptc_pack<<<NDIR, 256, 0, L.stream>>>(N.d_w + N.off[l], N.w[l], N.w[l + 1], 0, N.d_pf[l]);
      k_ptc_pack<<<NDIR, 256, 0, L.stream>>>(N.d_w + N.off[l], N.w[l], N.w[l + 1], 1, N.d_pa[l]);
   }
   N.packed = true;
}

// samples that are worked on together: as many as 2 GiB of activations,
// gradients and weight-gradient shares allow (a batch of 16 at 16^4; one at
// 32^3x64, whose layers fill the device by themselves), and no more than could
// be allocated before (N.cap)
int batch_size(int n)
{
   const size_t V = lib().g.V;
   size_t units = 0;
   int wmax = 4;
   for (int l = 1; l < N.nl; l++)
   {
      units += 3 * N.w[l];
      wmax = std::max(wmax, N.w[l]);
   }
   units += 2 * 3 * wmax;
   const size_t bytes = V * (units + NDIR * CMAX * CMAX / PNS) * sizeof(float2);
   return (int)std::max<size_t>(1, std::min<size_t>(std::min(n, N.cap), ((size_t)2 << 30) / bytes));
}

// activations of nb samples for the current lattice; the fields of several
// samples are given up without an error if they cannot be had
bool ensure_fields(int nb = 1)
{
   Lib &L = lib();
   if (N.V == L.g.V && N.nbatch >= nb) return true;
   auto alloc = [nb](size_t bytes) { return nb > 1 ? dev_try_alloc(bytes) : dev_alloc(bytes); };
   HIP_OK(hipStreamSynchronize(L.stream));
   for (int l = 0; l <= NLMAX; l++) { dev_free(N.d_act[l]); N.d_act[l] = nullptr; }
   for (int k = 0; k < 2; k++) { dev_free(N.d_gb[k]); N.d_gb[k] = nullptr; }
   dev_free(N.d_part);
   N.d_part = nullptr;
   N.nbatch = 0;
   const size_t V64 = units_for(L.g.V, 1);
   int wmax = 4;
   bool ok = true;
   for (int l = 1; l < N.nl; l++)
   {
      N.d_act[l] = (float2 *)alloc(nb * V64 * 3 * N.w[l] * sizeof(float2));
      wmax = std::max(wmax, N.w[l]);
      ok = ok && N.d_act[l];
   }
   for (int k = 0; k < 2; k++) N.d_gb[k] = (float2 *)alloc(nb * V64 * 3 * wmax * sizeof(float2));
   const int np = (L.g.V + PNS - 1) / PNS;
   N.d_part = (float2 *)alloc((size_t)nb * np * NDIR * CMAX * CMAX * sizeof(float2));
   ok = ok && N.d_gb[0] && N.d_gb[1] && N.d_part;
   if (N.V != L.g.V)
   {
      for (int k = 0; k < 2; k++) { dev_free(N.d_inf[k]); N.d_inf[k] = nullptr; }
      dev_free(N.d_tmp); dev_free(N.d_u16);
      N.u16_epoch = -1;
      N.V = L.g.V;
      N.d_tmp = (float2 *)dev_alloc(units_for(N.V, 12) * sizeof(float2));
      for (int k = 0; k < 2; k++) N.d_inf[k] = (bf16x2 *)dev_alloc(units_for(N.V, 3 * CMAX) * sizeof(bf16x2));
      N.d_u16 = (__half2 *)dev_alloc(units_for(N.V / 2, 72) * sizeof(__half2));
   }
   ok = ok && N.d_tmp && N.d_inf[0] && N.d_inf[1] && N.d_u16;
   if (ok) N.nbatch = nb;
   return ok;
}

// activations of as many of n samples as there is memory for; their number, 0
// (an error) if there is none for one
int ensure_batch(int n)
{
   int B = batch_size(n);
   while (!ensure_fields(B))
   {
      if (B == 1) return 0;
      B /= 2;
      N.cap = B;
   }
   return B;
}

template <int CI, int CO> void launch_layer(const Batch &bt, int n, const __bf16 *wp)
{
   Lib &L = lib();
   const int V = L.g.V;
   k_ptc<CI, CO><<<dim3((V + PNS - 1) / PNS, n), PWG, 0, L.stream>>>(bt, wp, L.d_u, L.d_nbr, V, 0);
}

// one layer of the preconditioner: mode 0 FP32 -> BF16, 1 BF16 -> BF16,
// 2 BF16 -> FP32 added to out, 3 FP32 -> FP32 added to out
template <int CI, int CO> void launch_inf(const void *in, void *out, const __bf16 *wp, int mode)
{
   Lib &L = lib();
   const int V = L.g.V;
   const unsigned nb = (V + PNS - 1) / PNS;
   const __half2 *u = N.d_u16;
   Batch bt = {};
   bt.in[0] = in;
   bt.out[0] = out;
   if (mode == 0)
      k_ptc<CI, CO, float2, bf16x2, __half2><<<nb, PWG, 0, L.stream>>>(bt, wp, u, L.d_nbr, V, 0);
   else if (mode == 1)
      k_ptc<CI, CO, bf16x2, bf16x2, __half2><<<nb, PWG, 0, L.stream>>>(bt, wp, u, L.d_nbr, V, 0);
   else if (mode == 2)
      k_ptc<CI, CO, bf16x2, float2, __half2><<<nb, PWG, 0, L.stream>>>(bt, wp, u, L.d_nbr, V, 1);
   else
      k_ptc<CI, CO, float2, float2, __half2><<<nb, PWG, 0, L.stream>>>(bt, wp, u, L.d_nbr, V, 1);
}

template <int CI, int CO> void launch_wgrad(const Batch &bt, int n)
{
   Lib &L = lib();
   const int V = L.g.V, nb = (V + PNS - 1) / PNS;
   k_ptc_wgrad<CI, CO><<<dim3(nb, n), PWG, 0, L.stream>>>(bt, L.d_u, L.d_nbr, V, N.d_lsum, N.d_part);
}

#define OQH_PTC_DISPATCH(F, ci, co, ...)                                             \
   do                                                                               \
   {                                                                                \
      const int ci_ = (ci), co_ = (co);                                             \
      bool done_ = false;                                                           \
      OQH_PTC_CASE(F, 4, 4, __VA_ARGS__) OQH_PTC_CASE(F, 4, 8, __VA_ARGS__)           \
      OQH_PTC_CASE(F, 4, 12, __VA_ARGS__) OQH_PTC_CASE(F, 4, 16, __VA_ARGS__)         \
      OQH_PTC_CASE(F, 8, 4, __VA_ARGS__) OQH_PTC_CASE(F, 8, 8, __VA_ARGS__)           \
      OQH_PTC_CASE(F, 8, 12, __VA_ARGS__) OQH_PTC_CASE(F, 8, 16, __VA_ARGS__)         \
      OQH_PTC_CASE(F, 12, 4, __VA_ARGS__) OQH_PTC_CASE(F, 12, 8, __VA_ARGS__)         \
      OQH_PTC_CASE(F, 12, 12, __VA_ARGS__) OQH_PTC_CASE(F, 12, 16, __VA_ARGS__)       \
      OQH_PTC_CASE(F, 16, 4, __VA_ARGS__) OQH_PTC_CASE(F, 16, 8, __VA_ARGS__)         \
      OQH_PTC_CASE(F, 16, 12, __VA_ARGS__) OQH_PTC_CASE(F, 16, 16, __VA_ARGS__)       \
      if (!done_) fail("ptc", "unsupported channel counts");                        \
   } while (0)
#define OQH_PTC_CASE(F, A, B, ...)                                                   \
   if (!done_ && ci_ == A && co_ == B)                                              \
   {                                                                                \
      F<A, B>(__VA_ARGS__);                                                         \
      done_ = true;                                                                 \
   }

// sample k of a workspace of n samples with nc units per point
float2 *sample(float2 *f, int k, int nc) { return f + (size_t)k * units_for(lib().g.V, nc); }

// forward pass of n samples; keeps the activations of the hidden layers
void forward(int n, const float2 *const *in, float2 *const *out)
{
   pack();
   Batch bt = {};
   for (int k = 0; k < n; k++) bt.in[k] = in[k];
   for (int l = 0; l < N.nl; l++)
   {
      for (int k = 0; k < n; k++) bt.out[k] = (l == N.nl - 1) ? out[k] : sample(N.d_act[l + 1], k, 3 * N.w[l + 1]);
      OQH_PTC_DISPATCH(launch_layer, N.w[l], N.w[l + 1], bt, n, N.d_pf[l]);
      for (int k = 0; k < n; k++) bt.in[k] = bt.out[k];
   }
}

// gradients of the weights (added to d_g) for the output gradients g of the
// last forward pass with inputs in
void backward(int n, const float2 *const *in, float2 *const *g)
{
   Lib &L = lib();
   const int nb = (L.g.V + PNS - 1) / PNS;
   Batch bt = {}, bg = {};  // layer inputs and output gradients; the layer's adjoint
   for (int k = 0; k < n; k++) bt.out[k] = g[k];
   for (int l = N.nl - 1; l >= 0; l--)
   {
      for (int k = 0; k < n; k++) bt.in[k] = l ? sample(N.d_act[l], k, 3 * N.w[l]) : in[k];
      OQH_PTC_DISPATCH(launch_wgrad, N.w[l], N.w[l + 1], bt, n);
      const int nw = NDIR * N.w[l] * N.w[l + 1];
      k_ptc_wgrad_sum<<<(nw + 63) / 64, 64 * WSW, 0, L.stream>>>(N.d_part, n * nb * WG_KSPLIT(N.w[l], N.w[l + 1]), nw,
                                                                 N.d_g + N.off[l]);
      if (l > 0)
      {
         for (int k = 0; k < n; k++)
         {
            bg.in[k] = bt.out[k];
            bt.out[k] = bg.out[k] = sample(N.d_gb[l & 1], k, 3 * N.w[l]);
         }
         OQH_PTC_DISPATCH(launch_layer, N.w[l + 1], N.w[l], bg, n, N.d_pa[l]);
      }
   }
}

constexpr int LNB = 256;  // work-groups of a sample's loss

// mean loss over the samples; gradients of the mean loss in d_g; false if
// there is no memory for the activations
bool loss_and_grad(int n, float2 *const *r, float2 *const *e, double &loss)
{
   Lib &L = lib();
   const int nu = (int)units_for(L.g.V, 12);
   const int B = ensure_batch(n);
   loss = 0.0;
   if (!B) return false;
   HIP_OK(hipMemsetAsync(N.d_g, 0, nweights() * sizeof(float2), L.stream));
   float2 *out[NBMAX];
   // the buffer that the first backward step does not write
   for (int k = 0; k < B; k++) out[k] = sample(N.d_gb[N.nl & 1], k, 12);
   for (int k0 = 0; k0 < n; k0 += B)
   {
      const int m = std::min(B, n - k0);
      forward(m, r + k0, out);
      Batch bt = {};
      for (int k = 0; k < m; k++)
      {
         bt.in[k] = e[k0 + k];
         bt.out[k] = out[k];
      }
      k_ptc_loss<<<dim3(LNB, m), 256, 0, L.stream>>>(bt, L.g.V, nu, N.d_lpart);
      k_ptc_loss_sum<<<m, 64, 0, L.stream>>>(N.d_lpart, LNB, N.d_lsum);
      k_ptc_lgrad<<<dim3((nu + 255) / 256, m), 256, 0, L.stream>>>(bt, N.d_lsum, n, L.g.V, nu);
      backward(m, r + k0, out);
      HIP_OK(hipMemcpyAsync(N.h_lsum, N.d_lsum, 2 * m * sizeof(double), hipMemcpyDeviceToHost, L.stream));
      HIP_OK(hipStreamSynchronize(L.stream));
      for (int k = 0; k < m; k++)
         if (N.h_lsum[2 * k] != 0.0) loss += N.h_lsum[2 * k + 1] / N.h_lsum[2 * k] / n;
   }
   return true;
}

bool require_net(const char *where)
{
   if (!N.nl)
   {
      fail(where, "the network is not created");
      return false;
   }
   if (!require_geometry(where) || !lib().ud_set)
   {
      if (lib().g.V) fail(where, "gauge field is not set");
      return false;
   }
   ensure_u();
   return ensure_fields();
}

// device fields of n spinors, all registered full fields
bool fields_of(int n, spinor **s, std::vector<float2 *> &out, const char *where)
{
   out.resize(n);
   for (int k = 0; k < n; k++)
   {
      int off = 0;
      out[k] = (float2 *)device_field(s[k], F32, &off);
      if (!out[k] || off)
      {
         fail(where, "the fields must be full single-precision device fields");
         return false;
      }
   }
   return true;
}

}  // namespace

bool nn_ready() { return N.nl > 0 && lib().nn_prec; }

// phi += NN(r) for the preconditioner (device fields of the lattice): the
// activations between the layers are kept in BF16, the values the channel
// mixing rounds them to anyway, and the last layer adds its output to phi
bool nn_correct(const float2 *r, float2 *phi)
{
   if (!N.nl || !ensure_fields()) return false;
   pack();
   Lib &L = lib();
   if (N.u16_epoch != L.u_epoch)
   {
      // the transports of the preconditioner read the links in FP16 (half
      // the bytes of the layer's dominant stream; the BF16 channel mixing
      // rounds more coarsely)
      const size_t nu = units_for(L.g.V / 2, 72);
      k_ptc_link16<<<(unsigned)((nu + 255) / 256), 256, 0, L.stream>>>(L.d_u, N.d_u16, nu);
      N.u16_epoch = L.u_epoch;
   }
   const void *x = r;
   for (int l = 0; l < N.nl; l++)
   {
      const bool first = l == 0, last = l == N.nl - 1;
      const int mode = last ? (first ? 3 : 2) : (first ? 0 : 1);
      void *y = last ? (void *)phi : (void *)N.d_inf[l & 1];
      OQH_PTC_DISPATCH(launch_inf, N.w[l], N.w[l + 1], x, y, N.d_pf[l], mode);
      x = y;
   }
   return true;
}

float2 *nn_work() { return ensure_fields() ? N.d_tmp : nullptr; }

void release_nn() { free_net(); }

}  // namespace oqh

using namespace oqh;

extern "C" int oqh_nn_create(int nlayer, const int *widths)
{
   free_net();
   if (nlayer < 1 || nlayer > NLMAX || widths[0] != 4 || widths[nlayer] != 4)
   {
      fail("oqh_nn_create", "1 to 8 layers with 4 input and 4 output channels are supported");
      return 1;
   }
   for (int l = 0; l <= nlayer; l++)
      if (!valid_width(widths[l]))
      {
         fail("oqh_nn_create", "channel counts must be 4, 8, 12 or 16");
         return 1;
      }
   N.nl = nlayer;
   for (int l = 0; l <= nlayer; l++) N.w[l] = widths[l];
   for (int l = 0; l < nlayer; l++) N.off[l + 1] = N.off[l] + (size_t)NDIR * N.w[l] * N.w[l + 1];
   size_t nw = nweights();
   N.d_w = (float2 *)dev_alloc(nw * sizeof(float2));
   N.d_g = (float2 *)dev_alloc(nw * sizeof(float2));
   N.d_m = (float *)dev_alloc(2 * nw * sizeof(float));
   N.d_v = (float *)dev_alloc(2 * nw * sizeof(float));
   for (int l = 0; l < nlayer; l++)
   {
      N.d_pf[l] = (__bf16 *)dev_alloc((size_t)NDIR * 32 * kpad(N.w[l]) * sizeof(__bf16));
      N.d_pa[l] = (__bf16 *)dev_alloc((size_t)NDIR * 32 * kpad(N.w[l + 1]) * sizeof(__bf16));
   }
   N.d_lpart = (double *)dev_alloc(2 * NBMAX * LNB * sizeof(double));
   N.d_lsum = (double *)dev_alloc(2 * NBMAX * sizeof(double));
   if (hipHostMalloc((void **)&N.h_lsum, 2 * NBMAX * sizeof(double), 0) != hipSuccess) N.h_lsum = nullptr;
   bool ok = N.d_w && N.d_g && N.d_m && N.d_v && N.d_lpart && N.d_lsum && N.h_lsum;
   for (int l = 0; l < nlayer; l++) ok = ok && N.d_pf[l] && N.d_pa[l];
   if (!ok)
   {
      free_net();
      fail("oqh_nn_create", "no memory for the network");
      return 1;
   }
   HIP_OK(hipMemset(N.d_w, 0, nw * sizeof(float2)));
   HIP_OK(hipMemset(N.d_m, 0, 2 * nw * sizeof(float)));
   HIP_OK(hipMemset(N.d_v, 0, 2 * nw * sizeof(float)));
   return 0;
}

extern "C" int oqh_nn_nweights() { return (int)nweights(); }

extern "C" void oqh_nn_set_weights(const double *w)
{
   if (!N.nl)
   {
      fail("oqh_nn_set_weights", "the network is not created");
      return;
   }
   size_t nw = nweights();
   std::vector<float2> h(nw);
   for (size_t k = 0; k < nw; k++) h[k] = make_float2((float)w[2 * k], (float)w[2 * k + 1]);
   HIP_OK(hipMemcpy(N.d_w, h.data(), nw * sizeof(float2), hipMemcpyHostToDevice));
   HIP_OK(hipMemset(N.d_m, 0, 2 * nw * sizeof(float)));
   HIP_OK(hipMemset(N.d_v, 0, 2 * nw * sizeof(float)));
   N.adam_t = 0;
   N.packed = false;
}

extern "C" void oqh_nn_get_weights(double *w)
{
   if (!N.nl)
   {
      fail("oqh_nn_get_weights", "the network is not created");
      return;
   }
   size_t nw = nweights();
   std::vector<float2> h(nw);
   HIP_OK(hipStreamSynchronize(lib().stream));
   HIP_OK(hipMemcpy(h.data(), N.d_w, nw * sizeof(float2), hipMemcpyDeviceToHost));
   for (size_t k = 0; k < nw; k++)
   {
      w[2 * k] = h[k].x;
      w[2 * k + 1] = h[k].y;
   }
}

extern "C" void oqh_nn_apply(spinor *in, spinor *out)
{
   const char *where = "oqh_nn_apply";
   if (!require_net(where)) return;
   Lib &L = lib();
   int V = L.g.V;
   Res a = resolve(in, F32, V, 0, true);
   Res b = resolve(out, F32, V, 1, false);
   if (!a.dev || !b.dev) return;
   if (a.off || b.off || a.dev == b.dev)
   {
      fail(where, "the fields must be distinct full fields");
      return;
   }
   const float2 *fi = (const float2 *)a.dev;
   float2 *fo = (float2 *)b.dev;
   forward(1, &fi, &fo);
   finish(a, F32, V, false);
   finish(b, F32, V, true);
}

// phi += NN(r) as the preconditioner applies it (BF16 activations between
// the layers); full single-precision device fields
extern "C" void oqh_nn_correct(spinor *r, spinor *phi)
{
   const char *where = "oqh_nn_correct";
   if (!require_net(where)) return;
   int o0 = 0, o1 = 0;
   float2 *a = (float2 *)device_field(r, F32, &o0), *b = (float2 *)device_field(phi, F32, &o1);
   if (!a || !b || o0 || o1 || a == b)
   {
      fail(where, "the fields must be distinct full single-precision device fields");
      return;
   }
   nn_correct(a, b);
   HIP_OK(hipStreamSynchronize(lib().stream));
}

extern "C" double oqh_nn_grad(int n, spinor **r, spinor **e, double *dw)
{
   const char *where = "oqh_nn_grad";
   if (!require_net(where)) return 0.0;
   std::vector<float2 *> rr, ee;
   if (!fields_of(n, r, rr, where) || !fields_of(n, e, ee, where)) return 0.0;
   double loss;
   if (!loss_and_grad(n, rr.data(), ee.data(), loss)) return 0.0;
   size_t nw = nweights();
   std::vector<float2> h(nw);
   HIP_OK(hipStreamSynchronize(lib().stream));
   HIP_OK(hipMemcpy(h.data(), N.d_g, nw * sizeof(float2), hipMemcpyDeviceToHost));
   for (size_t k = 0; k < nw; k++)
   {
      dw[2 * k] = h[k].x;
      dw[2 * k + 1] = h[k].y;
   }
   return loss;
}

extern "C" double oqh_nn_train_step(int n, spinor **r, spinor **e, double lr)
{
   const char *where = "oqh_nn_train_step";
   if (!require_net(where)) return 0.0;
   std::vector<float2 *> rr, ee;
   if (!fields_of(n, r, rr, where) || !fields_of(n, e, ee, where)) return 0.0;
   Lib &L = lib();
   double loss;
   if (!loss_and_grad(n, rr.data(), ee.data(), loss)) return 0.0;
   const float b1 = 0.9f, b2 = 0.999f;
   N.adam_t++;
   const float c1 = 1.0f / (1.0f - powf(b1, (float)N.adam_t)), c2 = 1.0f / (1.0f - powf(b2, (float)N.adam_t));
   const int nr = (int)(2 * nweights());
   k_adam<<<(nr + 255) / 256, 256, 0, L.stream>>>((float *)N.d_w, (const float *)N.d_g, N.d_m, N.d_v, nr, (float)lr, b1,
                                                  b2, 1e-8f, c1, c2);
   N.packed = false;
   HIP_OK(hipStreamSynchronize(L.stream));
   return loss;
}

extern "C" void oqh_set_nn_prec(int on)
{
   if (on != 0 && on != 1)
   {
      fail("oqh_set_nn_prec", "the argument must be 0 or 1");
      return;
   }
   if (on && !N.nl)
   {
      fail("oqh_set_nn_prec", "the network is not created");
      return;
   }
   lib().nn_prec = on;
}

extern "C" void oqh_nn_free() { free_net(); lib().nn_prec = 0; }
