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
// Column bases by pivoted MGS with two re-orthogonalisations and the rank cut
// ||col|| < eps*||A||_F (reference Matrix_columnbasis_pivotedmgs,
// Matrix.c:215-307): at step k the remaining column of largest norm (ties to
// the lowest current position, positions k and the pivot's exchanged, as the
// reference exchanges columns) becomes q_k = a / |a|, and the others have it
// taken out twice, a -= (q . a) q, and their norms formed afresh.
//
// The order of every sum is fixed by rows and cols alone (mgs_sum_lanes), so
// that a basis does not depend on the kernel that makes it: one lane, first
// row to last, where the matrix fits 96 KB; else the rows sl, sl + S, sl + 2S,
// ... per lane sl of S, the lanes' sums then added pairwise, lanes S/2 apart
// first.  Bases of the same span with other rounding move an FP64 product by
// up to 1e-13 of its norm: directions that the steps leave small are their
// rounding errors' size.
//
// One workgroup runs a problem from its first to its last step, so a batch is
// a few launches:
//   k_mgs_cols  one lane per column, columns in registers and LDS
//   k_mgs_reg   S lanes per two columns, all in registers
//   k_mgs_blk   larger ones, read from L2 once per step
//   k_mgs_long  the rest (more than 6144 rows)
// Against two launches per step over all problems, each reading and writing
// every matrix: one operator pair's bases take 111 ms of kernel time instead of
// 212 at 100 000 panels (55 launches instead of 2180), 39 instead of 59 at
// 31 000; the operators are there after 125 and 57 ms instead of 206 and 105,
// with the kept device memory.

// Value of another lane of the row by DPP (quad permutations, half-row mirror,
// row rotation): VALU moves, without the LDS round trip of a shuffle.
template <int CTRL>
__device__ __forceinline__ int dpp_i(int v) {
   return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xf, 0xf, true);
}
template <int CTRL>
__device__ __forceinline__ double dpp_d(double v) {
   return __hiloint2double(dpp_i<CTRL>(__double2hiint(v)), dpp_i<CTRL>(__double2loint(v)));
}
constexpr int DPP_XOR1 = 0xB1, DPP_XOR2 = 0x4E, DPP_XOR3 = 0x1B, DPP_XOR7 = 0x141, DPP_XOR8 = 0x128;

// Sum over the S lanes (a power of two) of the lane's aligned segment, lanes
// S/2 apart first; the same in all of them.
__device__ __forceinline__ double seg_sum(double v, int S) {
   if (S > 32) v += __shfl_xor(v, 32, 64);
   if (S > 16) v += __shfl_xor(v, 16, 64);
   if (S > 8) v += dpp_d<DPP_XOR8>(v);
   if (S > 4) v += dpp_d<DPP_XOR3>(dpp_d<DPP_XOR7>(v));
   if (S > 2) v += dpp_d<DPP_XOR2>(v);
   if (S > 1) v += dpp_d<DPP_XOR1>(v);
   return v;
}
// Largest value over the wave (NaN ignored) and, among the lanes that hold
// it, the lowest position.
__device__ __forceinline__ double wave_max(double v) {
   v = fmax(v, dpp_d<DPP_XOR1>(v));
   v = fmax(v, dpp_d<DPP_XOR2>(v));
   v = fmax(v, dpp_d<DPP_XOR7>(v));
   v = fmax(v, dpp_d<DPP_XOR8>(v));
   v = fmax(v, __shfl_xor(v, 16, 64));
   return fmax(v, __shfl_xor(v, 32, 64));
}
__device__ __forceinline__ int wave_min(int v) {
   v = min(v, dpp_i<DPP_XOR1>(v));
   v = min(v, dpp_i<DPP_XOR2>(v));
   v = min(v, dpp_i<DPP_XOR7>(v));
   v = min(v, dpp_i<DPP_XOR8>(v));
   v = min(v, __shfl_xor(v, 16, 64));
   return min(v, __shfl_xor(v, 32, 64));
}

// The pivot of a step: largest norm (0 if none is above it) and its position
// over the block, from each thread's candidate.  wv, wp: a value per wave,
// free for reuse after the caller's next barrier.
__device__ __forceinline__ void block_pivot(double bv, int bp, int nw, double* wv, int* wp, double& mx, int& best) {
   mx = wave_max(bv);
   best = wave_min(bv == mx ? bp : 0x7fffffff);
   if ((threadIdx.x & 63) == 0) {
      wv[threadIdx.x >> 6] = mx;
      wp[threadIdx.x >> 6] = best;
   }
   __syncthreads();
   mx = wv[0];
   best = wp[0];
   for (int w = 1; w < nw; w++) {
      const double ov = wv[w];
      const int op = wp[w];
      if (ov > mx || (ov == mx && op < best)) {
         mx = ov;
         best = op;
      }
   }
}

// Frobenius norm from the squared column norms n2 (LDS), in every lane: 256
// sums over the columns 256 apart, added pairwise, 128 apart first.
__device__ __forceinline__ double mgs_frobenius(const double* n2, int cols) {
   double p[4];
#pragma unroll
   for (int q = 0; q < 4; q++) {
      p[q] = 0.0;
      for (int j = (threadIdx.x & 63) + 64 * q; j < cols; j += 256) p[q] += n2[j];
   }
   return sqrt(seg_sum((p[0] + p[2]) + (p[1] + p[3]), 64));
}

// One lane per column: rows 0 .. NR - 1 in registers, the others in LDS (rem,
// row-major).  Bound by the FP64 rate, the latency of the sums' chains where
// few waves share a CU, and three barriers a step.
constexpr int mgs_cols_threads(int NR) { return NR == 32 ? 1024 : (NR == 64 ? 512 : 256); }
__host__ __device__ inline size_t mgs_cols_bytes(int rows, int cols, int NR) {
   return sizeof(double) * ((size_t)(rows > NR ? rows : NR) + (size_t)cols * (rows > NR ? rows - NR : 0));
}
template <int NR>
__global__ void __launch_bounds__(mgs_cols_threads(NR))
    k_mgs_cols(const MgsDesc* __restrict__ descs, const int* __restrict__ list, const double* __restrict__ Abuf,
               double* __restrict__ Qbuf, int* __restrict__ ranks, double eps) {
   constexpr int NT = mgs_cols_threads(NR), G = 8;
   extern __shared__ __align__(16) unsigned char sm[];
   __shared__ double n2[NT];
   __shared__ double wv[NT / 64];
   __shared__ int wp[NT / 64];
   const MgsDesc d = descs[list[blockIdx.x]];
   const int rows = d.rows, cols = d.cols, tid = threadIdx.x, nw = (int)blockDim.x >> 6;
   double* qs = (double*)sm;                      // rows, zeros up to NR
   double* rem = qs + max(rows, NR) + tid;        // (rows - NR) x cols
   const bool mine = tid < cols, busy = (tid & ~63) < cols;   // busy: a wave with columns
   const double* a = Abuf + d.a_off + (long long)(mine ? tid : 0) * rows;
   double v[NR];
   double sq = 0.0;
#pragma unroll
   for (int t = 0; t < NR; t++) v[t] = t < rows && mine ? a[t < rows ? t : 0] : 0.0;
#pragma unroll
   for (int t = 0; t < NR; t++) sq = fma(v[t], v[t], sq);
   if (mine)
      for (int t = NR; t < rows; t++) {
         const double x = a[t];
         rem[(size_t)(t - NR) * cols] = x;
         sq = fma(x, x, sq);
      }
   n2[tid] = sq;
   for (int t = rows + tid; t < NR; t += (int)blockDim.x) qs[t] = 0.0;
   __syncthreads();
   const double cut = eps * mgs_frobenius(n2, cols);
   double nrm = sqrt(sq);
   int pos = mine ? tid : -1;   // the column's current position; -1: taken or none
   const int kmax = min(rows, cols);
   int k = 0;
   for (; k < kmax; k++) {
      double mx;
      int best;
      const bool on = pos >= k && nrm >= 0.0;
      block_pivot(on ? nrm : 0.0, on ? pos : 0x7fffffff, nw, wv, wp, mx, best);
      if (!(mx > 0.0)) best = k;
      if (k >= 1 && mx < cut) break;   // uniform over the block
      if (pos == best) {
#pragma unroll
         for (int t = 0; t < NR; t++)
            if (t < rows) qs[t] = v[t];
         for (int t = NR; t < rows; t++) qs[t] = rem[(size_t)(t - NR) * cols];
         pos = -1;
      } else if (pos == k) {
         pos = best;
      }
      __syncthreads();
      for (int t = tid; t < rows; t += (int)blockDim.x) {
         const double x = qs[t] / mx;
         qs[t] = x;
         Qbuf[d.q_off + (long long)k * rows + t] = x;
      }
      __syncthreads();
      if (busy) {
         // r1 = q.a; a -= r1 q, r2 = q.a; a -= r2 q, |a|^2
         double r1 = 0.0, r2 = 0.0;
         sq = 0.0;
#pragma unroll
         for (int g = 0; g < NR; g += G)
            if (g < rows)
#pragma unroll
               for (int t = g; t < g + G; t++) r1 = fma(qs[t], v[t], r1);
         if (mine)
            for (int t = NR; t < rows; t++) r1 = fma(qs[t], rem[(size_t)(t - NR) * cols], r1);
#pragma unroll
         for (int g = 0; g < NR; g += G)
            if (g < rows)
#pragma unroll
               for (int t = g; t < g + G; t++) {
                  const double q = qs[t];
                  v[t] = fma(-q, r1, v[t]);
                  r2 = fma(q, v[t], r2);
               }
         if (mine)
            for (int t = NR; t < rows; t++) {
               const double q = qs[t], x = fma(-q, r1, rem[(size_t)(t - NR) * cols]);
               rem[(size_t)(t - NR) * cols] = x;
               r2 = fma(q, x, r2);
            }
#pragma unroll
         for (int g = 0; g < NR; g += G)
            if (g < rows)
#pragma unroll
               for (int t = g; t < g + G; t++) {
                  v[t] = fma(-qs[t], r2, v[t]);
                  sq = fma(v[t], v[t], sq);
               }
         if (mine)
            for (int t = NR; t < rows; t++) {
               const double x = fma(-qs[t], r2, rem[(size_t)(t - NR) * cols]);
               rem[(size_t)(t - NR) * cols] = x;
               sq = fma(x, x, sq);
            }
         nrm = sqrt(sq);
      }
   }
   if (tid == 0) ranks[d.rank_slot] = k;
}

// The lane's rows i = sl, sl + S, ... of a column, at most NR: four at a time
// while there are any (what they read past the column's end, of the next
// columns or the MGS_SLACK values after the last, mgs_mask makes zeros), the
// others zero.  One lane offset for all rows, so that their addresses cost no
// registers.
template <int NR>
__device__ __forceinline__ void mgs_load(double (&x)[NR], const double* A, unsigned at, int rows, int S) {
#pragma unroll
   for (int t0 = 0; t0 < NR; t0 += 4)
      if (S * t0 < rows) {
#pragma unroll
         for (int t = t0; t < t0 + 4; t++) x[t] = (A + S * t)[at];
      } else {
#pragma unroll
         for (int t = t0; t < t0 + 4; t++) x[t] = 0.0;
      }
}
template <int NR>
__device__ __forceinline__ void mgs_mask(double (&x)[NR], int rows, int S, int sl) {
#pragma unroll
   for (int t0 = 0; t0 < NR; t0 += 4)
      if (S * t0 < rows && S * (t0 + 4) > rows)
#pragma unroll
         for (int t = t0; t < t0 + 4; t++) x[t] = sl < rows - S * t ? x[t] : 0.0;
}

// S lanes per two columns (j = g and g + NT/S of lane group g), at most 16
// rows of each per lane.  Bound by the FP64 rate and three barriers a step;
// the matrix is read from HBM once.
constexpr int MGS_NR = 16;
template <int NT>
__global__ void __launch_bounds__(NT) k_mgs_reg(const MgsDesc* __restrict__ descs, const int* __restrict__ list,
                                                const double* __restrict__ Abuf, double* __restrict__ Qbuf,
                                                int* __restrict__ ranks, double eps) {
   __shared__ double qs[MGS_NR * 64];
   __shared__ double n2[NT / 2];   // S >= 4
   __shared__ double wv[NT / 64];
   __shared__ int wp[NT / 64];
   const MgsDesc d = descs[list[blockIdx.x]];
   const int rows = d.rows, cols = d.cols, S = d.seg, tid = threadIdx.x;
   const int g = tid / S, sl = tid - g * S, G = NT / S;
   double v[2][MGS_NR];
   double nrm[2];
   int pos[2];   // the column's current position; -1: taken or none
#pragma unroll
   for (int c = 0; c < 2; c++) {
      const int j = g + c * G;
      pos[c] = j < cols ? j : -1;
      double s = 0.0;
      mgs_load(v[c], Abuf + d.a_off, (unsigned)((j < cols ? j : 0) * rows + sl), rows, S);
      mgs_mask(v[c], rows, S, sl);
#pragma unroll
      for (int t = 0; t < MGS_NR; t++) v[c][t] = j < cols ? v[c][t] : 0.0;
#pragma unroll
      for (int t = 0; t < MGS_NR; t++) s = fma(v[c][t], v[c][t], s);
      s = seg_sum(s, S);
      if (sl == 0) n2[j] = s;
      nrm[c] = sqrt(s);
   }
   for (int i = rows + tid; i < MGS_NR * S; i += NT) qs[i] = 0.0;   // past the last row
   __syncthreads();
   const double cut = eps * mgs_frobenius(n2, cols);
   const int kmax = min(rows, cols);
   int k = 0;
   for (; k < kmax; k++) {
      double bv = 0.0, mx;
      int bp = 0x7fffffff, best;
#pragma unroll
      for (int c = 0; c < 2; c++)
         if (pos[c] >= k && (nrm[c] > bv || (nrm[c] == bv && pos[c] < bp))) {
            bv = nrm[c];
            bp = pos[c];
         }
      block_pivot(bv, bp, NT / 64, wv, wp, mx, best);
      if (!(mx > 0.0)) best = k;
      if (k >= 1 && mx < cut) break;   // uniform over the block
#pragma unroll
      for (int c = 0; c < 2; c++) {
         if (pos[c] == best) {
#pragma unroll
            for (int t = 0; t < MGS_NR; t++)
               if (sl + S * t < rows) qs[sl + S * t] = v[c][t];
            pos[c] = -1;
         } else if (pos[c] == k) {
            pos[c] = best;
         }
      }
      __syncthreads();
      for (int i = tid; i < rows; i += NT) {
         const double x = qs[i] / mx;
         qs[i] = x;
         Qbuf[d.q_off + (long long)k * rows + i] = x;
      }
      __syncthreads();
      double q[MGS_NR];
#pragma unroll
      for (int t = 0; t < MGS_NR; t++) q[t] = qs[sl + S * t];
#pragma unroll
      for (int c = 0; c < 2; c++) {
         double r1 = 0.0, r2 = 0.0, s = 0.0;
#pragma unroll
         for (int t = 0; t < MGS_NR; t++) r1 = fma(q[t], v[c][t], r1);
         r1 = seg_sum(r1, S);
#pragma unroll
         for (int t = 0; t < MGS_NR; t++) {
            v[c][t] = fma(-q[t], r1, v[c][t]);
            r2 = fma(q[t], v[c][t], r2);
         }
         r2 = seg_sum(r2, S);
#pragma unroll
         for (int t = 0; t < MGS_NR; t++) {
            v[c][t] = fma(-q[t], r2, v[c][t]);
            s = fma(v[c][t], v[c][t], s);
         }
         nrm[c] = sqrt(seg_sum(s, S));
      }
   }
   if (tid == 0) ranks[d.rank_slot] = k;
}

// Larger matrices.  A stays in memory as it was at the start of a block of nb
// steps; a step reads each column once, takes the block's earlier directions
// out of it with the coefficients kept in R (the same operations on the same
// values, so the same bits as a column written back every step), then does its
// own two projections and the norm, all in registers; the block's last step
// writes the columns back.  Up to NR rows a lane, 64 / S columns per wave.
// Columns whose norm is below half of the cut can never be pivots and are no
// longer read.  Bound by what one CU reads from L2 (about 60 GB/s) for long
// columns, where few waves fit the registers, and by latency for short ones:
// with PRE the next column is loaded during the work on one, the first of a
// step during the choice of its pivot.  2986 x 160: 78 us a step; 3658 x 176:
// 128; 662 of 316 x 176: 57 (nb = 2 or 4 the same; the registers that hold q
// from one sum to the next cost more than its reads from LDS).
// LDS: qs[nb * NR * S], R[nb * cols], n2[cols], order[cols], act[cols].
__host__ __device__ inline size_t mgs_blk_bytes(int NRS, int cols, int nb) {
   return sizeof(double) * (size_t)nb * NRS + sizeof(double2) * (size_t)nb * cols +
          (sizeof(double) + 2 * sizeof(int)) * (size_t)cols;
}
template <int NR, int S, int NT, bool PRE>
__device__ __forceinline__ void mgs_blk(const MgsDesc& d, double* __restrict__ Abuf, double* __restrict__ Qbuf,
                                        int* __restrict__ ranks, double eps, unsigned char* sm, double* wv,
                                        int* wp, int& s_nact) {
   constexpr int NW = NT / 64, G = NR > 32 ? 16 : 4;   // G: reads of q in flight, for few waves more
   constexpr int ldq = NR * S;
   const int m = d.rows, K = d.cols, NB = d.nb;
   const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
   const int sub = lane / S, sl = lane - sub * S;
   constexpr int CPW = 64 / S;   // columns per wave at a time
   const int kmax = min(m, K);
   double* A = Abuf + d.a_off;
   double* Q = Qbuf + d.q_off;
   double* qs = (double*)sm;
   double2* R = (double2*)(qs + NB * ldq);
   double* n2 = (double*)(R + NB * K);
   int* order = (int*)(n2 + K);
   int* act = order + K;
   for (int a0 = wave * CPW; a0 < K; a0 += NW * CPW) {
      const int j = a0 + sub;
      double s = 0.0, x[NR];
      mgs_load(x, A, (unsigned)((j < K ? j : 0) * m + sl), m, S);
      mgs_mask(x, m, S, sl);
#pragma unroll
      for (int t = 0; t < NR; t++) s = fma(x[t], x[t], s);
      s = seg_sum(s, S);
      if (j < K && sl == 0) {
         n2[j] = s;
         order[j] = j;
         act[j] = j;
      }
   }
   for (int u = 0; u < NB; u++)
      for (int i = m + tid; i < ldq; i += NT) qs[u * ldq + i] = 0.0;   // past the last row
   __syncthreads();
   const double cut = eps * mgs_frobenius(n2, K), lim = 0.25 * cut * cut;
   int k = 0, b = 0, nact = K;
   for (; k < kmax; k++) {
      double y[NR];
      int jy = 0;
      auto load = [&](int a0) {
         jy = act[min(a0 + sub, nact - 1)];
         mgs_load(y, A, (unsigned)(jy * m + sl), m, S);
      };
      if (PRE && nact) load(wave * CPW);
      // the pivot among the positions k .. K - 1
      double bv = 0.0, mx;
      int bp = 0x7fffffff, best;
      for (int p = k + tid; p < K; p += NT) {
         const double x = sqrt(n2[order[p]]);
         if (x > bv || (x == bv && p < bp)) {
            bv = x;
            bp = p;
         }
      }
      block_pivot(bv, bp, NW, wv, wp, mx, best);
      if (!(mx > 0.0)) best = k;
      if (k >= 1 && mx < cut) break;   // uniform over the block
      const int pj = order[best];
      for (int i = tid; i < m; i += NT) {
         double x = A[(unsigned)(pj * m + i)];
         for (int u = 0; u < b; u++) {
            const double q = qs[u * ldq + i];
            const double2 r = R[u * K + pj];
            x = fma(-q, r.y, fma(-q, r.x, x));
         }
         x /= mx;
         qs[b * ldq + i] = x;
         Q[(long long)k * m + i] = x;
      }
      __syncthreads();
      if (tid == 0) {
         order[best] = order[k];
         order[k] = pj;
      }
      const bool last = b + 1 == NB;
      if (k + 1 < kmax) {
         // read anew for each sum: kept, they cost 2 NR registers
         auto q_row = [&]() {
            int at = b * ldq + sl;
            asm volatile("" : "+v"(at));
            return qs + at;
         };
         for (int a0 = wave * CPW; a0 < nact; a0 += NW * CPW) {
            int rows = __builtin_amdgcn_readfirstlane(m), row = sl;
            asm volatile("" : "+s"(rows), "+v"(row));   // the row tests stay in the loop: hoisted, they cost registers
            if (!PRE) load(a0);
            const int j = jy;
            double x[NR];
#pragma unroll
            for (int t = 0; t < NR; t++) x[t] = y[t];
            mgs_mask(x, rows, S, row);
            if (PRE && a0 + NW * CPW < nact) load(a0 + NW * CPW);
            for (int u = 0; u < b; u++) {
               const double2 r = R[u * K + j];
               const double* qu = qs + u * ldq + sl;
#pragma unroll
               for (int t0 = 0; t0 < NR; t0 += G)
                  if (t0 * S < rows)
#pragma unroll
                     for (int t = t0; t < t0 + G; t++) {
                        const double p = qu[S * t];
                        x[t] = fma(-p, r.y, fma(-p, r.x, x[t]));
                     }
            }
            double r1 = 0.0, r2 = 0.0, s = 0.0;
            const double* qa = q_row();
#pragma unroll
            for (int t0 = 0; t0 < NR; t0 += G)
               if (t0 * S < rows)
#pragma unroll
                  for (int t = t0; t < t0 + G; t++) r1 = fma(qa[S * t], x[t], r1);
            r1 = seg_sum(r1, S);
            const double* qc = q_row();
#pragma unroll
            for (int t0 = 0; t0 < NR; t0 += G)
               if (t0 * S < rows)
#pragma unroll
                  for (int t = t0; t < t0 + G; t++) {
                     const double q = qc[S * t];
                     x[t] = fma(-q, r1, x[t]);
                     r2 = fma(q, x[t], r2);
                  }
            r2 = seg_sum(r2, S);
            const double* qd = q_row();
#pragma unroll
            for (int t0 = 0; t0 < NR; t0 += G)
               if (t0 * S < rows)
#pragma unroll
                  for (int t = t0; t < t0 + G; t++) {
                     x[t] = fma(-qd[S * t], r2, x[t]);
                     s = fma(x[t], x[t], s);
                  }
            s = seg_sum(s, S);
            if (a0 + sub < nact) {
               if (sl == 0) {
                  R[b * K + j] = make_double2(r1, r2);
                  n2[j] = s;
               }
               if (last) {
#pragma unroll
                  for (int t = 0; t < NR; t++)
                     if (row < rows - S * t) (A + S * t)[(unsigned)(j * m + row)] = x[t];
               }
            }
         }
      }
      __syncthreads();
      b++;
      if (last) {
         // the columns at positions k + 1 .. that may still be pivots
         if (wave == 0) {
            int cnt = 0;
            for (int p0 = k + 1; p0 < K; p0 += 64) {
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
      }
   }
   if (tid == 0) ranks[d.rank_slot] = k;
}

// The rows a lane takes and the lanes per column are settled per problem; the
// problems of all of them share a launch (launches of a stream run one after
// the other, and a level's are short of problems: a launch per shape made the
// 31 000-panel operators 64 ms instead of 57): 12 waves with up to 48 rows a
// lane, 8 waves above, by the registers.
enum { MGS_16x4, MGS_16x8, MGS_16x16, MGS_16x32, MGS_16x64, MGS_32x64, MGS_48x64, MGS_64x64, MGS_96x64 };
template <int NT>
__global__ void __launch_bounds__(NT) k_mgs_blk(const MgsDesc* __restrict__ descs, const int* __restrict__ list,
                                                double* __restrict__ Abuf, double* __restrict__ Qbuf,
                                                int* __restrict__ ranks, double eps) {
   extern __shared__ __align__(16) unsigned char sm[];
   __shared__ double wv[NT / 64];
   __shared__ int wp[NT / 64];
   __shared__ int s_nact;
   const MgsDesc d = descs[list[blockIdx.x]];
   if constexpr (NT == 512) {
      if (d.shape == MGS_64x64)
         mgs_blk<64, 64, NT, false>(d, Abuf, Qbuf, ranks, eps, sm, wv, wp, s_nact);
      else
         mgs_blk<96, 64, NT, false>(d, Abuf, Qbuf, ranks, eps, sm, wv, wp, s_nact);
   } else {
      switch (d.shape) {
         case MGS_16x4: mgs_blk<16, 4, NT, true>(d, Abuf, Qbuf, ranks, eps, sm, wv, wp, s_nact); break;
         case MGS_16x8: mgs_blk<16, 8, NT, true>(d, Abuf, Qbuf, ranks, eps, sm, wv, wp, s_nact); break;
         case MGS_16x16: mgs_blk<16, 16, NT, true>(d, Abuf, Qbuf, ranks, eps, sm, wv, wp, s_nact); break;
         case MGS_16x32: mgs_blk<16, 32, NT, true>(d, Abuf, Qbuf, ranks, eps, sm, wv, wp, s_nact); break;
         case MGS_16x64: mgs_blk<16, 64, NT, true>(d, Abuf, Qbuf, ranks, eps, sm, wv, wp, s_nact); break;
         case MGS_32x64: mgs_blk<32, 64, NT, false>(d, Abuf, Qbuf, ranks, eps, sm, wv, wp, s_nact); break;
         default: mgs_blk<48, 64, NT, false>(d, Abuf, Qbuf, ranks, eps, sm, wv, wp, s_nact); break;
      }
   }
}

// Any other size: the columns read three times and written once a step, their
// squared norms and order in memory (n2, order: ws_off).
constexpr int MGS_LT = 1024;
__host__ __device__ inline size_t mgs_long_bytes(int cols) {
   return (sizeof(double) + sizeof(int)) * (size_t)(cols + 1) / 16 * 16 + 16;
}
__global__ void __launch_bounds__(MGS_LT) k_mgs_long(const MgsDesc* __restrict__ descs, const int* __restrict__ list,
                                                     double* __restrict__ Abuf, double* __restrict__ Qbuf,
                                                     int* __restrict__ ranks, double eps,
                                                     unsigned char* __restrict__ scratch) {
   __shared__ double wv[MGS_LT / 64];
   __shared__ int wp[MGS_LT / 64];
   constexpr int NW = MGS_LT / 64;
   const MgsDesc d = descs[list[blockIdx.x]];
   const int m = d.rows, K = d.cols, S = d.seg, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
   const int sub = lane / S, sl = lane - sub * S, CPW = 64 / S, kmax = min(m, K);
   double* n2 = (double*)(scratch + d.ws_off);
   int* order = (int*)(n2 + K);
   for (int a0 = wave * CPW; a0 < K; a0 += NW * CPW) {
      const int j = a0 + sub;
      const double* a = Abuf + d.a_off + (long long)(j < K ? j : 0) * m;
      double s = 0.0;
      for (int i = sl; i < m; i += S) s = fma(a[i], a[i], s);
      s = seg_sum(s, S);
      if (j < K && sl == 0) {
         n2[j] = s;
         order[j] = j;
      }
   }
   __syncthreads();
   const double cut = eps * mgs_frobenius(n2, K), lim = 0.25 * cut * cut;
   int k = 0;
   for (; k < kmax; k++) {
      double bv = 0.0, mx;
      int bp = 0x7fffffff, best;
      for (int p = k + tid; p < K; p += MGS_LT) {
         const double x = sqrt(n2[order[p]]);
         if (x > bv || (x == bv && p < bp)) {
            bv = x;
            bp = p;
         }
      }
      block_pivot(bv, bp, NW, wv, wp, mx, best);
      if (!(mx > 0.0)) best = k;
      if (k >= 1 && mx < cut) break;   // uniform over the block
      const int pj = order[best];
      double* q = Qbuf + d.q_off + (long long)k * m;
      for (int i = tid; i < m; i += MGS_LT) q[i] = Abuf[d.a_off + (long long)pj * m + i] / mx;
      __syncthreads();
      if (tid == 0) {
         order[best] = order[k];
         order[k] = pj;
         n2[pj] = -1.0;   // taken
      }
      for (int a0 = wave * CPW; a0 < K; a0 += NW * CPW) {
         const int j = a0 + sub;
         const bool on = j < K && j != pj && !(n2[j] < lim);
         if (!__any(on)) continue;
         double* a = Abuf + d.a_off + (long long)(on ? j : pj) * m;
         double r1 = 0.0, r2 = 0.0, s = 0.0;
#pragma unroll 4
         for (int i = sl; i < m; i += S) r1 = fma(q[i], a[i], r1);
         r1 = seg_sum(r1, S);
#pragma unroll 4
         for (int i = sl; i < m; i += S) r2 = fma(q[i], fma(-q[i], r1, a[i]), r2);
         r2 = seg_sum(r2, S);
#pragma unroll 4
         for (int i = sl; i < m; i += S) {
            const double x = fma(-q[i], r2, fma(-q[i], r1, a[i]));
            if (on) a[i] = x;
            s = fma(x, x, s);
         }
         s = seg_sum(s, S);
         if (on && sl == 0) n2[j] = s;
      }
      __syncthreads();
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
      hipLaunchKernelGGL(k_integral_blocks, dim3(nblk), dim3(256), 0, s, blocks, bpts, bpan, panels, kernel, kappa,
                         out);
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

// Lanes that share a column's sums (the sums' order: see k_mgs_cols above).
static int mgs_sum_lanes(int rows, int cols) {
   if (sizeof(double) * ((size_t)(rows | 1) + 1) * cols <= 96 * 1024) return 1;
   int S = 4;
   while (S < 64 && rows > MGS_NR * S) S <<= 1;
   return S;
}

// Which kernel takes a problem is settled by rows and cols alone: one lane per
// column by the rows in registers, two columns a lane group while they fit the
// threads of a block, else a block that reads the matrix at each step while a
// column fits a wave's registers.
void run_mgs(std::vector<MgsDesc>& descs, double* A, double* Q, std::vector<int>& ranks, double eps,
             hipStream_t s) {
   constexpr size_t LDS_MAX = 150 * 1024;   // beside at most 8.2 KB of static LDS
   const int nprob = (int)descs.size();
   ranks.assign(nprob, 0);
   if (nprob == 0) return;
   struct Class {
      std::vector<int> list;
      size_t lds = 0;
   };
   // blk: 8, 12 waves; reg: 1024, 512 threads; cols: by rows in registers, by threads
   Class large, blk[2], reg[2], cols[3][5];
   constexpr int cols_rows[3] = {32, 64, 96};
   size_t ws = 0;
   auto put = [](Class& c, int p, size_t lds) {
      c.list.push_back(p);
      c.lds = std::max(c.lds, lds);
   };
   auto cols_lds = [&](int p, int n) { return mgs_cols_bytes(descs[p].rows, descs[p].cols, cols_rows[n]); };
   for (int p = 0; p < nprob; p++) {
      MgsDesc& d = descs[p];
      const int S = mgs_sum_lanes(d.rows, d.cols);
      d.seg = S;
      const int n = d.rows <= 32 ? 0 : (d.rows <= 64 ? 1 : 2);
      if (S == 1 && d.cols <= 1024 && cols_lds(p, n) <= LDS_MAX) {
         int c = 0;
         while ((64 << c) < d.cols) c++;
         put(cols[n][c], p, cols_lds(p, n));
         continue;
      }
      const long long threads = (long long)S * ((d.cols + 1) / 2);
      if (S > 1 && d.rows <= MGS_NR * S && threads <= 1024) {
         put(reg[threads <= 512 ? 1 : 0], p, 0);
         continue;
      }
      d.shape = MGS_96x64;
      int rows_a_lane = 96;
      if (d.rows <= MGS_NR * S) {
         d.shape = S == 64 ? MGS_16x64 : (S == 32 ? MGS_16x32 : (S == 16 ? MGS_16x16 : (S == 8 ? MGS_16x8 : MGS_16x4)));
         rows_a_lane = MGS_NR;
      } else if (d.rows <= 64 * S) {
         d.shape = d.rows <= 32 * S ? MGS_32x64 : (d.rows <= 48 * S ? MGS_48x64 : MGS_64x64);
         rows_a_lane = d.rows <= 32 * S ? 32 : (d.rows <= 48 * S ? 48 : 64);
      }
      const int nrs = rows_a_lane * S;
      d.nb = 4;
      while (d.nb > 1 && mgs_blk_bytes(nrs, d.cols, d.nb) > LDS_MAX) d.nb >>= 1;
      // (the kernel's offsets into a matrix are 32 bits)
      if (S > 1 && d.rows <= nrs && mgs_blk_bytes(nrs, d.cols, d.nb) <= LDS_MAX) {
         put(blk[rows_a_lane <= 48 ? 1 : 0], p, mgs_blk_bytes(nrs, d.cols, d.nb));
         continue;
      }
      d.ws_off = (long long)ws;
      ws += mgs_long_bytes(d.cols);
      put(large, p, 0);
   }
   // Launches of one stream run one after the other: those that would not fill
   // the chip join the next larger ones, with a lane per column by threads first
   // (at most as many as the kernel takes), then by rows.
   if (reg[1].list.size() < 512 && !reg[0].list.empty()) {
      for (int p : reg[1].list) put(reg[0], p, 0);
      reg[1].list.clear();
   }
   for (int n = 0; n < 3; n++)
      for (int c = 0; c < 4; c++)
         if (!cols[n][c].list.empty() && cols[n][c].list.size() < 512 && (128 << c) <= mgs_cols_threads(cols_rows[n])) {
            bool larger = false;
            for (int k = c + 1; k < 5; k++) larger = larger || !cols[n][k].list.empty();
            if (!larger) break;
            for (int p : cols[n][c].list) put(cols[n][c + 1], p, cols_lds(p, n));
            cols[n][c].list.clear();
         }
   for (int n = 0; n < 2; n++)
      for (int c = 0; c < 5; c++)
         if (cols[n][c].list.size() < 512 && (64 << c) <= mgs_cols_threads(cols_rows[n + 1]) &&
             !cols[n + 1][c].list.empty()) {
            for (int p : cols[n][c].list) put(cols[n + 1][c], p, cols_lds(p, n + 1));
            cols[n][c].list.clear();
         }
   // the largest ahead: they run longest
   auto longest_first = [&](Class& c) {
      std::stable_sort(c.list.begin(), c.list.end(), [&](int x, int y) {
         return (long long)descs[x].rows * descs[x].cols > (long long)descs[y].rows * descs[y].cols;
      });
   };
   longest_first(large);
   for (Class& c : blk) longest_first(c);
   std::vector<int> all(large.list);
   for (const Class& c : blk) all.insert(all.end(), c.list.begin(), c.list.end());
   for (const Class& c : reg) all.insert(all.end(), c.list.begin(), c.list.end());
   for (const auto& n : cols)
      for (const Class& c : n) all.insert(all.end(), c.list.begin(), c.list.end());
   DBuf<MgsDesc> dd;
   DBuf<int> dl, dr;
   DBuf<unsigned char> dws;
   dd.upload(descs, s);
   dl.upload(all, s);
   dr.alloc(nprob);
   if (ws) dws.alloc(ws);
   static std::once_flag attr;
   std::call_once(attr, [] {
      for (const void* k : {(const void*)k_mgs_blk<512>, (const void*)k_mgs_blk<768>, (const void*)k_mgs_cols<32>,
                            (const void*)k_mgs_cols<64>, (const void*)k_mgs_cols<96>})
         FSVD_CHECK(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDS_MAX));
   });
   const int* l = dl.p;
   int launches = 0;
   if (!large.list.empty())
      hipLaunchKernelGGL(k_mgs_long, dim3((unsigned)large.list.size()), dim3(MGS_LT), 0, s, dd.p, l, A, Q, dr.p, eps,
                         dws.p);
   l += large.list.size();
   auto launch = [&](auto kernel, const Class& c, int threads) {
      const unsigned n = (unsigned)c.list.size();
      if (n) hipLaunchKernelGGL(kernel, dim3(n), dim3(threads), c.lds, s, dd.p, l, A, Q, dr.p, eps);
      l += n;
      launches += n > 0;
   };
   launch(k_mgs_blk<512>, blk[0], 512);
   launch(k_mgs_blk<768>, blk[1], 768);
   launch(k_mgs_reg<1024>, reg[0], 1024);
   launch(k_mgs_reg<512>, reg[1], 512);
   for (int c = 0; c < 5; c++) launch(k_mgs_cols<32>, cols[0][c], 64 << c);
   for (int c = 0; c < 5; c++) launch(k_mgs_cols<64>, cols[1][c], 64 << c);
   for (int c = 0; c < 5; c++) launch(k_mgs_cols<96>, cols[2][c], 64 << c);
   FSVD_CHECK(hipGetLastError());
   std::vector<int> h(nprob);
   FSVD_CHECK(hipMemcpyAsync(h.data(), dr.p, sizeof(int) * nprob, hipMemcpyDeviceToHost, s));
   FSVD_CHECK(hipStreamSynchronize(s));
   for (int i = 0; i < nprob; i++) ranks[descs[i].rank_slot] = h[descs[i].rank_slot];
   if (const char* e = std::getenv("FFTSVD_TIMING"); e && e[0] == '1')
      std::fprintf(stderr, "[fftsvd mgs] %d problems: %zu large, %zu + %zu blocked, %zu in registers, the others a "
                   "lane per column; %d launches\n", nprob, large.list.size(), blk[0].list.size(), blk[1].list.size(),
                   reg[0].list.size() + reg[1].list.size(), launches);
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
