// Setup kernels: collocation integrals, point kernels, small batched GEMMs
// and the pivoted modified Gram-Schmidt that builds the sampled bases.
// All of it runs in FP64.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <mutex>
#include <stdexcept>
#include <vector>

#include "device.h"
#include "geometry.h"
#include "integrals.h"
#include "op.h"

namespace fsvd {

// One workgroup per IntBlock; threads stride over the (point, panel) pairs.
__global__ void __launch_bounds__(256) k_integral_blocks(const IntBlock* __restrict__ blocks,
                                                         const double* __restrict__ bpts,
                                                         const int* __restrict__ bpan,
                                                         const PanelGeom* __restrict__ panels, int kernel,
                                                         double kappa, double* __restrict__ out) {
   const IntBlock b = blocks[blockIdx.x];
   const int total = b.npt * b.npan;
   for (int e = threadIdx.x; e < total; e += blockDim.x) {
      int i = e / b.npan;
      int j = e - i * b.npan;
      const double* x = bpts + 3 * (size_t)(b.pt_off + i);
      const PanelGeom& P = panels[bpan[b.pan_off + j]];
      double s, d;
      panel_integrals(kernel, kappa, x, P, s, d);
      long long o = b.out_off + (long long)i * b.ld_pt + (long long)j * b.ld_pan;
      if (b.layer_stride >= 0) {
         out[o] = s;
         out[o + b.layer_stride] = d;
      } else {
         out[o] = d;   // double layer only
      }
   }
}

__global__ void __launch_bounds__(256) k_green_blocks(const GreenBlock* __restrict__ blocks,
                                                      const double* __restrict__ dest,
                                                      const double* __restrict__ src, int kernel, double kappa,
                                                      double* __restrict__ out) {
   const GreenBlock b = blocks[blockIdx.x];
   const int total = b.ndest * b.nsrc;
   for (int e = threadIdx.x; e < total; e += blockDim.x) {
      int i = e / b.nsrc;
      int j = e - i * b.nsrc;
      double g = green(kernel, kappa, dest + 3 * (size_t)(b.dest_off + i), src + 3 * (size_t)(b.src_off + j));
      out[b.out_off + (long long)i * b.ld_dest + (long long)j * b.ld_src] = g;
   }
}

// C = A*B with arbitrary element strides, one descriptor per grid.y.
// 32x32 output tiles (grid.x strides over a problem's tiles), K staged in
// LDS chunks of 32; each thread owns a 2x2 block of the tile.  Each output
// is summed over k in increasing order.  Tile loads read along whichever
// operand dimension has unit stride.
__global__ void __launch_bounds__(256) k_gemm_batched(const GemmDesc* __restrict__ descs) {
   const GemmDesc d = descs[blockIdx.y];
   __shared__ double As[32][33], Bs[32][33];   // As[i][k], Bs[k][j]
   const int tm = (d.M + 31) / 32, tn = (d.N + 31) / 32;
   const int tid = threadIdx.x, tx = tid & 15, ty = tid >> 4;
   for (int tile = blockIdx.x; tile < tm * tn; tile += gridDim.x) {
      const int i0 = (tile / tn) * 32, j0 = (tile % tn) * 32;
      double c00 = 0.0, c01 = 0.0, c10 = 0.0, c11 = 0.0;
      for (int k0 = 0; k0 < d.K; k0 += 32) {
         for (int e = tid; e < 1024; e += 256) {
            int ii, kk;
            if (d.a_cs == 1) {
               ii = e >> 5;
               kk = e & 31;
            } else {
               kk = e >> 5;
               ii = e & 31;
            }
            const int gi = i0 + ii, gk = k0 + kk;
            As[ii][kk] = (gi < d.M && gk < d.K) ? d.A[(long long)gi * d.a_rs + (long long)gk * d.a_cs] : 0.0;
            int jj;
            if (d.b_rs == 1) {
               jj = e >> 5;
               kk = e & 31;
            } else {
               kk = e >> 5;
               jj = e & 31;
            }
            const int gj = j0 + jj, gk2 = k0 + kk;
            Bs[kk][jj] = (gj < d.N && gk2 < d.K) ? d.B[(long long)gk2 * d.b_rs + (long long)gj * d.b_cs] : 0.0;
         }
         __syncthreads();
#pragma unroll 8
         for (int kk = 0; kk < 32; kk++) {
            const double a0 = As[2 * ty][kk], a1 = As[2 * ty + 1][kk];
            const double b0 = Bs[kk][2 * tx], b1 = Bs[kk][2 * tx + 1];
            c00 += a0 * b0;
            c01 += a0 * b1;
            c10 += a1 * b0;
            c11 += a1 * b1;
         }
         __syncthreads();
      }
      const int i = i0 + 2 * ty, j = j0 + 2 * tx;
      if (i < d.M && j < d.N) d.C[(long long)i * d.c_rs + (long long)j * d.c_cs] = c00;
      if (i < d.M && j + 1 < d.N) d.C[(long long)i * d.c_rs + (long long)(j + 1) * d.c_cs] = c01;
      if (i + 1 < d.M && j < d.N) d.C[(long long)(i + 1) * d.c_rs + (long long)j * d.c_cs] = c10;
      if (i + 1 < d.M && j + 1 < d.N) d.C[(long long)(i + 1) * d.c_rs + (long long)(j + 1) * d.c_cs] = c11;
   }
}

// ---------------------------------------------------------------------------
// Column bases by pivoted MGS with the rank cut ||col|| < eps*||A||_F
// (reference Matrix_columnbasis_pivotedmgs, Matrix.c:215-307): at step k the
// remaining column of largest norm (ties to the lowest current position,
// positions k and the pivot's exchanged, as the reference exchanges columns)
// becomes q_k and is projected out of the rest.  One workgroup runs one
// problem from its first to its last step, so a batch is a launch or two
// instead of a pair of launches per step:
//   k_mgs_reg  the matrix in registers (at most 16 rows x 64 lanes by 2 x
//              1024/lanes columns: the leaf cubes and most of the next level)
//   k_mgs_blk  larger matrices, read from L2 once per step and written once
//              per block of steps
// Kernel time of one operator pair's bases (MI355X), against one launch per
// pivot step with the matrices read and written in each: 31 000 panels
// 61 -> 37 ms in 60 launches instead of 1700, 100 000 panels 228 -> 81 ms.

// Value of another lane of the row by DPP (quad permutations, half-row and
// row mirrors): VALU moves, without the LDS round trip of a shuffle.
template <int CTRL>
__device__ __forceinline__ int dpp_i(int v) {
   return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xf, 0xf, true);
}
template <int CTRL>
__device__ __forceinline__ double dpp_d(double v) {
   return __hiloint2double(dpp_i<CTRL>(__double2hiint(v)), dpp_i<CTRL>(__double2loint(v)));
}
constexpr int DPP_XOR1 = 0xB1, DPP_XOR2 = 0x4E, DPP_HALF_MIRROR = 0x141, DPP_MIRROR = 0x140;

// Sum over the S lanes (a power of two) of the lane's aligned segment, the
// same in all of them.  The mirrors pair lanes whose quads (half rows)
// already hold equal sums, so they act as exchanges with the lane 4 (8) away.
__device__ __forceinline__ double seg_sum(double v, int S) {
   if (S > 1) v += dpp_d<DPP_XOR1>(v);
   if (S > 2) v += dpp_d<DPP_XOR2>(v);
   if (S > 4) v += dpp_d<DPP_HALF_MIRROR>(v);
   if (S > 8) v += dpp_d<DPP_MIRROR>(v);
   if (S > 16) v += __shfl_xor(v, 16, 64);
   if (S > 32) v += __shfl_xor(v, 32, 64);
   return v;
}
// Largest value over the wave (NaN ignored) and, among the lanes that hold
// it, the lowest position.
__device__ __forceinline__ double wave_max(double v) {
   v = fmax(v, dpp_d<DPP_XOR1>(v));
   v = fmax(v, dpp_d<DPP_XOR2>(v));
   v = fmax(v, dpp_d<DPP_HALF_MIRROR>(v));
   v = fmax(v, dpp_d<DPP_MIRROR>(v));
   v = fmax(v, __shfl_xor(v, 16, 64));
   return fmax(v, __shfl_xor(v, 32, 64));
}
__device__ __forceinline__ int wave_min(int v) {
   v = min(v, dpp_i<DPP_XOR1>(v));
   v = min(v, dpp_i<DPP_XOR2>(v));
   v = min(v, dpp_i<DPP_HALF_MIRROR>(v));
   v = min(v, dpp_i<DPP_MIRROR>(v));
   v = min(v, __shfl_xor(v, 16, 64));
   return min(v, __shfl_xor(v, 32, 64));
}

// Sum over the block, the same in every thread; red holds one value per
// wave.  A barrier separates consecutive uses of red.
__device__ __forceinline__ double block_total(double v, double* red, int nw) {
   v = seg_sum(v, 64);
   if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
   __syncthreads();
   double t = 0.0;
   for (int w = 0; w < nw; w++) t += red[w];
   __syncthreads();
   return t;
}

// Register kernel.  S = seg lanes share two columns (j = g and g + NT/S of
// lane group g), 16 rows of each per lane: row pairs 2 (sl + S u), u < 8, so
// that the pivot vector is read from LDS in conflict-free 16-byte pieces,
// once per step, into registers.  Each step makes the two projections
// a -= (q . a) q of the reference's re-orthogonalising MGS and the fresh
// squared norm.  FP64 rate and the two barriers of a step bound it; the
// matrix is read from HBM once.  (The 16 300 leaf problems of a 100 000-panel
// tree took 10 ms with the matrix in LDS, a thread per column: 96 KB of LDS
// left one workgroup per CU.)
constexpr int MGS_NR = 16;
template <int NT>
__global__ void __launch_bounds__(NT) k_mgs_reg(const MgsDesc* __restrict__ descs, const int* __restrict__ list,
                                                const double* __restrict__ Abuf, double* __restrict__ Qbuf,
                                                int* __restrict__ ranks, double eps) {
   constexpr int NW = NT / 64, NP = MGS_NR / 2;
   __shared__ __align__(16) double qs[MGS_NR * 64];
   __shared__ double wv[NW];
   __shared__ int wp[NW];
   const MgsDesc d = descs[list[blockIdx.x]];
   const int rows = d.rows, cols = d.cols, S = d.seg, tid = threadIdx.x, wave = tid >> 6;
   const int g = tid / S, sl = tid - g * S, G = NT / S;
   double v[2][MGS_NR];
   double n2[2];
   int pos[2];   // the column's current position; INT_MAX: none, -1: taken
#pragma unroll
   for (int c = 0; c < 2; c++) {
      const int j = g + c * G;
      const double* a = Abuf + d.a_off + (long long)(j < cols ? j : 0) * d.lda;
      pos[c] = j < cols ? j : 0x7fffffff;
      double s = 0.0;
#pragma unroll
      for (int u = 0; u < NP; u++) {
         const int i = 2 * (sl + S * u);
         // the even column stride makes row i + 1 readable whenever row i is
         const double2 x = *(const double2*)(a + (i < rows ? i : 0));
         v[c][2 * u] = j < cols && i < rows ? x.x : 0.0;
         v[c][2 * u + 1] = j < cols && i + 1 < rows ? x.y : 0.0;
      }
#pragma unroll
      for (int t = 0; t < MGS_NR; t++) s = fma(v[c][t], v[c][t], s);
      n2[c] = seg_sum(s, S);
   }
   const double fro = sqrt(block_total(sl == 0 ? n2[0] + n2[1] : 0.0, wv, NW));
   const int kmax = min(rows, cols);
   int k = 0;
   for (; k < kmax; k++) {
      double bv = 0.0;
      int bp = 0x7fffffff;
#pragma unroll
      for (int c = 0; c < 2; c++)
         if (pos[c] >= k && pos[c] != 0x7fffffff && (n2[c] > bv || (n2[c] == bv && pos[c] < bp))) {
            bv = n2[c];
            bp = pos[c];
         }
      double mx = wave_max(bv);
      int best = wave_min(bv == mx ? bp : 0x7fffffff);
      if constexpr (NW > 1) {
         if ((tid & 63) == 0) {
            wv[wave] = mx;
            wp[wave] = best;
         }
         __syncthreads();
         mx = wv[0];
         best = wp[0];
#pragma unroll
         for (int w = 1; w < NW; w++) {
            const double ov = wv[w];
            const int op = wp[w];
            if (ov > mx || (ov == mx && op < best)) {
               mx = ov;
               best = op;
            }
         }
      }
      if (!(mx > 0.0)) best = k;
      const double nrm = sqrt(mx);
      if (k >= 1 && nrm < eps * fro) break;
      double* q = Qbuf + d.q_off + (long long)k * rows;
#pragma unroll
      for (int c = 0; c < 2; c++) {
         if (pos[c] == best) {
#pragma unroll
            for (int u = 0; u < NP; u++) {
               const int i = 2 * (sl + S * u);
               const double x = v[c][2 * u] / nrm, y = v[c][2 * u + 1] / nrm;
               *(double2*)(qs + i) = make_double2(x, y);
               if (i < rows) q[i] = x;
               if (i + 1 < rows) q[i + 1] = y;
            }
            pos[c] = -1;
         } else if (pos[c] == k) {
            pos[c] = best;
         }
      }
      __syncthreads();
      double p[MGS_NR];
#pragma unroll
      for (int u = 0; u < NP; u++) {
         const double2 x = *(const double2*)(qs + 2 * (sl + S * u));
         p[2 * u] = x.x;
         p[2 * u + 1] = x.y;
      }
#pragma unroll
      for (int c = 0; c < 2; c++) {
#pragma unroll
         for (int pass = 0; pass < 2; pass++) {
            double r0 = 0.0, r1 = 0.0;
#pragma unroll
            for (int t = 0; t < MGS_NR; t += 2) {
               r0 = fma(p[t], v[c][t], r0);
               r1 = fma(p[t + 1], v[c][t + 1], r1);
            }
            const double r = seg_sum(r0 + r1, S);
#pragma unroll
            for (int t = 0; t < MGS_NR; t++) v[c][t] = fma(-p[t], r, v[c][t]);
         }
         double s0 = 0.0, s1 = 0.0;
#pragma unroll
         for (int t = 0; t < MGS_NR; t += 2) {
            s0 = fma(v[c][t], v[c][t], s0);
            s1 = fma(v[c][t + 1], v[c][t + 1], s1);
         }
         n2[c] = seg_sum(s0 + s1, S);
      }
      // qs is rewritten after the next step's barrier (with one wave, by
      // program order)
   }
   if (tid == 0) ranks[d.rank_slot] = k;
}

// Blocked kernel.  The columns stay as they were at the start of a block of
// up to nb steps; a step reads them once for the products r_j = q_k . a_j,
// kept in R, and takes r_j^2 off the squared norms; the block's end takes
// the block's directions out of the columns and forms their squared norms
// afresh.  A block also ends when the largest norm^2 has fallen by 1e-4, so
// the running norms carry errors below 1e-12 relative to the largest, the
// size of the columns' own rounding errors.  The pivot's vector takes the
// block's products off its column and is then orthogonalised once more
// against every earlier q (the reference re-orthogonalises against each q in
// turn).  Columns whose norm^2 is below a quarter of the squared cut can
// never be pivots and are no longer read.  The reads of the columns, from L2
// and the Infinity Cache, and the latency of the step's phases bound it
// (2986 x 160 at rank 70: 80 us a step), so 16 waves share a problem.
// Arrays (LDS, or global scratch when GLB): v[rows rounded up to even],
// R[nb * cols], n2[cols], h[min(rows, cols)], order[cols], act[cols].
constexpr int MGS_BT = 1024;
__host__ __device__ inline size_t mgs_blk_bytes(int rows, int cols, int nb) {
   const int kmax = rows < cols ? rows : cols;
   return sizeof(double) * ((size_t)cols * (nb + 1) + kmax + (rows + 1) / 2 * 2) + sizeof(int) * 2 * (size_t)cols + 16;
}
template <bool GLB>
__global__ void __launch_bounds__(MGS_BT) k_mgs_blk(const MgsDesc* __restrict__ descs, const int* __restrict__ list,
                                                    double* __restrict__ Abuf, double* __restrict__ Qbuf,
                                                    int* __restrict__ ranks, double eps,
                                                    unsigned char* __restrict__ scratch) {
   extern __shared__ __align__(16) unsigned char sm[];
   __shared__ double red[MGS_BT / 64];
   __shared__ int redi[MGS_BT / 64];
   __shared__ int s_nact;
   constexpr int NW = MGS_BT / 64, U = 8;
   const MgsDesc d = descs[list[blockIdx.x]];
   const int m = d.rows, K = d.cols, NB = d.nb, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
   const int kmax = min(m, K), mpad = (m + 1) / 2 * 2;
   const long long lda = d.lda;
   double* A = Abuf + d.a_off;
   double* Q = Qbuf + d.q_off;
   double* v = (double*)(GLB ? scratch + d.ws_off : sm);   // first: 16-byte aligned
   double* R = v + mpad;
   double* n2 = R + (size_t)NB * K;
   double* h = n2 + K;
   int* order = (int*)(h + kmax);
   int* act = order + K;
   // lanes per column: whole waves for long columns, parts of one for short
   const int S = m > 256 ? 64 : (m > 128 ? 32 : 16);
   const int sub = lane / S, sl = lane - sub * S, CPW = 64 / S;
   double part = 0.0;
   for (int j0 = wave * CPW; j0 < K; j0 += NW * CPW) {
      const int j = j0 + sub;
      const double* a = A + (long long)(j < K ? j : 0) * lda;
      double s = 0.0;
      for (int i0 = 0; i0 < m; i0 += 2 * S * U) {
         double2 x[U];
#pragma unroll
         for (int u = 0; u < U; u++) {
            const int i = i0 + 2 * (sl + S * u);
            x[u] = *(const double2*)(a + (i < m ? i : 0));
         }
#pragma unroll
         for (int u = 0; u < U; u++) {
            const int i = i0 + 2 * (sl + S * u);
            const double p = i < m ? x[u].x : 0.0, q = i + 1 < m ? x[u].y : 0.0;
            s = fma(p, p, s);
            s = fma(q, q, s);
         }
      }
      s = seg_sum(s, S);
      if (j < K && sl == 0) {
         n2[j] = s;
         order[j] = j;
         act[j] = j;
         part += s;
      }
   }
   const double fro = sqrt(block_total(part, red, NW));
   const double cut = eps * fro, lim = 0.25 * cut * cut;
   int k = 0, b = 0, nact = K;
   double mx0 = 0.0;
   while (k < kmax) {
      // the pivot among the positions k..K-1
      double bv = 0.0;
      int bp = 0x7fffffff;
      for (int p = k + tid; p < K; p += MGS_BT) {
         const double x = n2[order[p]];
         if (x > bv || (x == bv && p < bp)) {
            bv = x;
            bp = p;
         }
      }
      double mx = wave_max(bv);
      int best = wave_min(bv == mx ? bp : 0x7fffffff);
      if (lane == 0) {
         red[wave] = mx;
         redi[wave] = best;
      }
      __syncthreads();
      mx = red[0];
      best = redi[0];
      for (int w = 1; w < NW; w++)
         if (red[w] > mx || (red[w] == mx && redi[w] < best)) {
            mx = red[w];
            best = redi[w];
         }
      if (!(mx > 0.0)) best = k;
      const bool fresh = b == 0;
      if (fresh) mx0 = mx;
      const bool fell = !fresh && mx < 1e-4 * mx0;
      if (k >= 1 && !fell && sqrt(mx) < cut) break;   // uniform over the block
      if (fell || b == NB) {
         // end of the block: its directions out of the active columns, four
         // columns per wave part, norms afresh
         for (int a0 = wave * CPW * 4; a0 < nact; a0 += NW * CPW * 4) {
            int j[4];
            double s[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int c = 0; c < 4; c++) {
               const int ai = a0 + sub * 4 + c;
               j[c] = ai < nact ? act[ai] : -1;
            }
            for (int i = 2 * sl; i < m; i += 2 * S) {
               double2 x[4];
#pragma unroll
               for (int c = 0; c < 4; c++) x[c] = *(const double2*)(A + (long long)max(j[c], 0) * lda + i);
               for (int t = 0; t < b; t++) {
                  // q columns are rows apart: not 16-byte aligned for odd rows
                  const double* q = Q + (long long)(k - b + t) * m + i;
                  const double q0 = q[0], q1 = i + 1 < m ? q[1] : 0.0;
#pragma unroll
                  for (int c = 0; c < 4; c++) {
                     const double r = R[(size_t)t * K + max(j[c], 0)];
                     x[c].x = fma(-r, q0, x[c].x);
                     x[c].y = fma(-r, q1, x[c].y);
                  }
               }
#pragma unroll
               for (int c = 0; c < 4; c++) {
                  if (i + 1 >= m) x[c].y = 0.0;
                  if (j[c] >= 0) *(double2*)(A + (long long)j[c] * lda + i) = x[c];
                  s[c] = fma(x[c].x, x[c].x, s[c]);
                  s[c] = fma(x[c].y, x[c].y, s[c]);
               }
            }
#pragma unroll
            for (int c = 0; c < 4; c++) {
               const double t = seg_sum(s[c], S);
               if (j[c] >= 0 && sl == 0) n2[j[c]] = t;
            }
         }
         __syncthreads();
         // positions k.. above the limit stay active
         if (wave == 0) {
            int cnt = 0;
            for (int p0 = k; p0 < K; p0 += 64) {
               const int p = p0 + lane, j = p < K ? order[p] : 0;
               const bool on = p < K && !(n2[j] < lim);
               const unsigned long long mask = __ballot(on);
               if (on) act[cnt + __popcll(mask & ((1ull << lane) - 1ull))] = j;
               cnt += __popcll(mask);
            }
            if (lane == 0) s_nact = cnt;
         }
         __syncthreads();
         nact = s_nact;
         b = 0;
         continue;
      }
      const int pj = order[best];
      const double* ap = A + (long long)pj * lda;
      // the pivot's residual
      for (int i = tid; i < m; i += MGS_BT) {
         double x = ap[i];
         const double* q = Q + (long long)(k - b) * m + i;
         const double* r = R + pj;
#pragma unroll 4
         for (int t = 0; t < b; t++) {
            x = fma(-*r, *q, x);
            q += m;
            r += K;
         }
         v[i] = x;
      }
      if (tid == 0 && mpad > m) v[m] = 0.0;
      __syncthreads();
      if (tid == 0) {
         order[best] = order[k];
         order[k] = pj;
      }
      // once more against every earlier direction, eight loads in flight
      for (int t0 = wave; t0 < k; t0 += NW) {
         const double* q = Q + (long long)t0 * m;
         double s0 = 0.0, s1 = 0.0;
         for (int i0 = 0; i0 < m; i0 += 64 * U) {
            double x[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
               const int i = i0 + lane + 64 * u;
               x[u] = q[i < m ? i : 0];
            }
#pragma unroll
            for (int u = 0; u < U; u += 2) {
               const int i = i0 + lane + 64 * u;
               s0 = fma(i < m ? x[u] : 0.0, v[i < m ? i : 0], s0);
               s1 = fma(i + 64 < m ? x[u + 1] : 0.0, v[i + 64 < m ? i + 64 : 0], s1);
            }
         }
         const double s = seg_sum(s0 + s1, 64);
         if (lane == 0) h[t0] = s;
      }
      __syncthreads();
      double nn = 0.0;
      for (int i = tid; i < m; i += MGS_BT) {
         double x = v[i];
         const double* q = Q + i;
         int t = 0;
         for (; t + 7 < k; t += 8, q += 8 * m) {
            double qv[8];
#pragma unroll
            for (int u = 0; u < 8; u++) qv[u] = q[(long long)u * m];
#pragma unroll
            for (int u = 0; u < 8; u++) x = fma(-h[t + u], qv[u], x);
         }
#pragma unroll 4
         for (; t < k; t++, q += m) x = fma(-h[t], *q, x);
         v[i] = x;
         nn = fma(x, x, nn);
      }
      const double nrm = sqrt(block_total(nn, red, NW));
      for (int i = tid; i < m; i += MGS_BT) {
         const double x = v[i] / nrm;
         v[i] = x;
         Q[(long long)k * m + i] = x;
      }
      if (tid == 0) n2[pj] = -1.0;
      __syncthreads();
      // products of the active columns with q_k
      for (int a0 = wave * CPW; a0 < nact; a0 += NW * CPW) {
         const int ai = a0 + sub, j = act[ai < nact ? ai : 0];
         const double* a = A + (long long)j * lda;
         double r0 = 0.0, r1 = 0.0;
         for (int i0 = 0; i0 < m; i0 += 2 * S * U) {
            double2 x[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
               const int i = i0 + 2 * (sl + S * u);
               x[u] = *(const double2*)(a + (i < m ? i : 0));
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
               const int i = i0 + 2 * (sl + S * u);
               const double2 q = *(const double2*)(v + (i < m ? i : 0));
               r0 = fma(i < m ? x[u].x : 0.0, q.x, r0);
               r1 = fma(i + 1 < m ? x[u].y : 0.0, q.y, r1);
            }
         }
         const double r = seg_sum(r0 + r1, S);
         if (ai < nact && sl == 0) {
            R[(size_t)b * K + j] = r;
            if (n2[j] >= 0.0) n2[j] = fma(-r, r, n2[j]);
         }
      }
      __syncthreads();
      b++;
      k++;
   }
   if (tid == 0) ranks[d.rank_slot] = k;
}

__global__ void k_f64_to_f32(const double* __restrict__ a, float* __restrict__ b, long long n) {
   for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
      b[i] = (float)a[i];
}

}  // namespace fsvd

namespace fsvd {

void launch_integral_blocks(int nblk, const IntBlock* blocks, const double* bpts, const int* bpan,
                            const PanelGeom* panels, int kernel, double kappa, double* out, hipStream_t s) {
   if (nblk > 0)
      hipLaunchKernelGGL(k_integral_blocks, dim3(nblk), dim3(256), 0, s, blocks, bpts, bpan, panels, kernel, kappa, out);
}

void launch_green_blocks(int nblk, const GreenBlock* blocks, const double* dest, const double* src, int kernel,
                         double kappa, double* out, hipStream_t s) {
   if (nblk > 0)
      hipLaunchKernelGGL(k_green_blocks, dim3(nblk), dim3(256), 0, s, blocks, dest, src, kernel, kappa, out);
}

void launch_gemm_batched(int nbatch, int maxtiles, const GemmDesc* descs, hipStream_t s) {
   if (nbatch > 0)
      hipLaunchKernelGGL(k_gemm_batched, dim3(maxtiles, nbatch), dim3(256), 0, s, descs);
}

// The register kernel takes every problem of up to 16 x 64 rows whose column
// pairs fit its 1024 threads, in launches by the threads they need (small
// workgroups share a CU); the others go to the blocked kernel, the largest
// first, its arrays in LDS or, past the LDS, in global scratch.
void run_mgs(std::vector<MgsDesc>& descs, double* A, double* Q, std::vector<int>& ranks, double eps,
             hipStream_t s) {
   constexpr size_t LDS_MAX = 158 * 1024;
   const int nprob = (int)descs.size();
   ranks.assign(nprob, 0);
   if (nprob == 0) return;
   constexpr int NC = 5;   // register kernel: 64, 128, 256, 512, 1024 threads
   std::vector<int> list[NC + 2];
   size_t lds = 0, ws = 0;
   for (int p = 0; p < nprob; p++) {
      MgsDesc& d = descs[p];
      if ((d.lda & 1) || (d.a_off & 1) || d.lda < d.rows) throw std::runtime_error("sampled matrix not 16-byte aligned");
      int S = 1;
      while (S < 64 && d.rows > MGS_NR * S) S <<= 1;
      d.seg = S;
      const long long threads = (long long)S * ((d.cols + 1) / 2);
      if (d.rows <= MGS_NR * S && threads <= 1024) {
         int c = 0;
         while ((64 << c) < threads) c++;
         list[c].push_back(p);
         continue;
      }
      d.nb = 8;
      while (d.nb > 2 && mgs_blk_bytes(d.rows, d.cols, d.nb) > LDS_MAX) d.nb >>= 1;
      const size_t need = mgs_blk_bytes(d.rows, d.cols, d.nb);
      if (need > LDS_MAX) {
         d.nb = 8;
         d.ws_off = (long long)ws;
         ws += (mgs_blk_bytes(d.rows, d.cols, d.nb) + 15) / 16 * 16;
         list[NC + 1].push_back(p);
      } else {
         lds = std::max(lds, need);
         list[NC].push_back(p);
      }
   }
   for (int c = NC; c < NC + 2; c++)
      std::stable_sort(list[c].begin(), list[c].end(), [&](int x, int y) {
         return (long long)descs[x].lda * descs[x].cols > (long long)descs[y].lda * descs[y].cols;
      });
   std::vector<int> all;
   size_t at[NC + 3];
   for (int c = 0; c < NC + 2; c++) {
      at[c] = all.size();
      all.insert(all.end(), list[c].begin(), list[c].end());
   }
   at[NC + 2] = all.size();
   DBuf<MgsDesc> dd;
   DBuf<int> dl, dr;
   DBuf<unsigned char> dws;
   dd.upload(descs, s);
   dl.upload(all, s);
   dr.alloc(nprob);
   if (ws) dws.alloc(ws);
   static std::once_flag attr;
   std::call_once(attr, [] {
      FSVD_CHECK(hipFuncSetAttribute((const void*)k_mgs_blk<false>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                     (int)LDS_MAX));
   });
   // the blocked problems first: they run longest
   for (int c = NC + 1; c >= 0; c--) {
      const unsigned n = (unsigned)(at[c + 1] - at[c]);
      const int* l = dl.p + at[c];
      if (!n) continue;
      switch (c) {
         case 0: hipLaunchKernelGGL(k_mgs_reg<64>, dim3(n), dim3(64), 0, s, dd.p, l, A, Q, dr.p, eps); break;
         case 1: hipLaunchKernelGGL(k_mgs_reg<128>, dim3(n), dim3(128), 0, s, dd.p, l, A, Q, dr.p, eps); break;
         case 2: hipLaunchKernelGGL(k_mgs_reg<256>, dim3(n), dim3(256), 0, s, dd.p, l, A, Q, dr.p, eps); break;
         case 3: hipLaunchKernelGGL(k_mgs_reg<512>, dim3(n), dim3(512), 0, s, dd.p, l, A, Q, dr.p, eps); break;
         case 4: hipLaunchKernelGGL(k_mgs_reg<1024>, dim3(n), dim3(1024), 0, s, dd.p, l, A, Q, dr.p, eps); break;
         case 5:
            hipLaunchKernelGGL(k_mgs_blk<false>, dim3(n), dim3(MGS_BT), lds, s, dd.p, l, A, Q, dr.p, eps, nullptr);
            break;
         default:
            hipLaunchKernelGGL(k_mgs_blk<true>, dim3(n), dim3(MGS_BT), 0, s, dd.p, l, A, Q, dr.p, eps, dws.p);
            break;
      }
   }
   FSVD_CHECK(hipGetLastError());
   std::vector<int> h(nprob);
   FSVD_CHECK(hipMemcpyAsync(h.data(), dr.p, sizeof(int) * nprob, hipMemcpyDeviceToHost, s));
   FSVD_CHECK(hipStreamSynchronize(s));
   for (int i = 0; i < nprob; i++) ranks[descs[i].rank_slot] = h[descs[i].rank_slot];
   if (const char* e = std::getenv("FFTSVD_TIMING"); e && e[0] == '1') {
      std::fprintf(stderr, "[fftsvd mgs] %d problems: in registers", nprob);
      for (int c = 0; c < NC; c++) std::fprintf(stderr, " %zu", list[c].size());
      std::fprintf(stderr, " (64..1024 threads), blocked %zu + %zu\n", list[NC].size(),
                   list[NC + 1].size());
   }
}

void launch_f64_to_f32(const double* a, float* b, long long n, hipStream_t s) {
   if (n <= 0) return;
   int blocks = (int)std::min<long long>((n + 255) / 256, 8192);
   hipLaunchKernelGGL(k_f64_to_f32, dim3(blocks), dim3(256), 0, s, a, b, n);
}

}  // namespace fsvd

namespace fsvd {
struct CopyDesc {
   const double* src;
   double* dst;
   long long n;
};
__global__ void k_batched_copy(const CopyDesc* __restrict__ d) {
   const CopyDesc c = d[blockIdx.x];
   for (long long i = threadIdx.x; i < c.n; i += blockDim.x) c.dst[i] = c.src[i];
}
void launch_batched_copy(int n, const void* descs, hipStream_t s) {
   if (n > 0) hipLaunchKernelGGL(k_batched_copy, dim3(n), dim3(256), 0, s, (const CopyDesc*)descs);
}
}  // namespace fsvd

namespace fsvd {
// Panel geometry records on the device (FlatPanel_allocate +
// FlatPanel_moments, FlatPanel.c:5-179,210-298) with the host's arithmetic,
// so every field equals the host record's bit for bit: record k is that of
// panel ids[k] (panel k without ids) of the 9-double vertex records verts9.
__global__ void __launch_bounds__(64) k_panel_records(const double* __restrict__ verts9, const int* __restrict__ ids,
                                                      int n, PanelGeom* __restrict__ out) {
   const int k = blockIdx.x * blockDim.x + threadIdx.x;
   if (k >= n) return;
   const double* v = verts9 + 9 * (long long)(ids ? ids[k] : k);
   double v0[3], v1[3], v2[3];
   for (int d = 0; d < 3; d++) {
      v0[d] = v[d];
      v1[d] = v[3 + d];
      v2[d] = v[6 + d];
   }
   PanelGeom g;
   geom::panel_geometry_hd(v0, v1, v2, &g);
   const double* src = reinterpret_cast<const double*>(&g);
   double* dst = reinterpret_cast<double*>(out + k);
   for (int q = 0; q < (int)(sizeof(PanelGeom) / sizeof(double)); q++) dst[q] = src[q];
}
void launch_panel_records(const double* verts9, const int* ids, int n, PanelGeom* out, hipStream_t s) {
   if (n > 0) hipLaunchKernelGGL(k_panel_records, dim3((n + 63) / 64), dim3(64), 0, s, verts9, ids, n, out);
}
}  // namespace fsvd
