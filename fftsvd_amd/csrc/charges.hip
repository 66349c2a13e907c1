// Sums over the pairs of point charges and panels, FP64: the charge
// right-hand sides, the reaction potentials at the charges, and both
// transposed.  nq charges, ne panels, ncol charge or solution columns.
//
// Bound by FP64 arithmetic (about 120 operations for a pair's moment
// expansion, 30 for 1/r), once a panel's 656-byte record is not read again for
// every pair.  Two forms:
//   - sums over panels (potentials, transposed right-hand side): a wave has 64
//     charges on its lanes and walks through panels, whose records it reads
//     as wave-uniform (scalar) loads; no sum crosses lanes.
//   - sums over charges (right-hand sides, transposed potentials): a wave has
//     64 panels on its lanes, the part of their records that the moment
//     expansion needs in registers, and walks through charges (scalar loads).
// The walked range is split over blocks until the chip is full; the parts' sums
// go to ws and a second launch adds them in order.  The split depends on nq and
// ne alone, so a column's result does not depend on the other columns.  Not
// split are the right-hand sides of the surface operator: each panel's charges
// are one chain, whose rounding a plain sum shares (4e-16 from it; in parts
// 8e-16, 30 000 panels and 500 charges), so a small surface fills few blocks
// (1280 panels: 5).  Kernel times before and after (one block per
// charge or 256 panels, the record read from memory for each pair, a division
// per column): potentials of 2000 charges and 100 000 panels 9.5 to 2.1 ms, of
// 500 and 30 000 with 64 columns 5.5 to 1.8 ms; right-hand sides for the latter
// 3.7 to 0.4 ms; transposed potentials of 500 and 30 000 0.39 to 0.14 ms and
// transposed right-hand side 0.097 to 0.036 ms.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "device.h"
#include "integrals.h"
#include "op.h"

namespace fsvd {

namespace {
constexpr int COL_CHUNK = 64;      // columns per launch (bounds ws)
constexpr int ROUND_BLOCKS = 1024; // 4 waves for each of 1024 SIMDs
}  // namespace

// --- sums over panels: charges on lanes -------------------------------------
// part[(sp * ncol + col) * nq + j], block (group of 64 charges, part sp)

// Potentials: sum_e (a_e slp - b_e dlp) - (self ? 4 pi b_e : 0) with Laplace
// integrals of panel pidx[e] at the charge (direct branch of
// SurfaceOperator_calculateReactionPotentials, SurfaceOperator.c:364-396).
// For own panels a = sol[dphi], b = sol[phi], self check on; for child
// panels a = -(eps_c/eps) sol[dphi_c], b = -sol[phi_c], self check off.
// coef: (a, b) per element, columns 2 ne apart.
template <int NC>
__global__ void __launch_bounds__(256) k_potentials(int ne, int nq, int ncol, int ng, int per,
                                                    const PanelGeom* __restrict__ panels,
                                                    const int* __restrict__ pidx, const double* __restrict__ coef,
                                                    const int* __restrict__ self_ok,
                                                    const double* __restrict__ qpos, double* __restrict__ part) {
   __shared__ double red[4][64];
   const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
   const int g = blockIdx.x % ng, sp = blockIdx.x / ng, col0 = blockIdx.y * NC;
   const int j = min(64 * g + lane, nq - 1);
   const double x[3] = {qpos[3 * (size_t)j], qpos[3 * (size_t)j + 1], qpos[3 * (size_t)j + 2]};
   double s[NC];
#pragma unroll
   for (int c = 0; c < NC; c++) s[c] = 0.0;
   const int e1 = min(ne, (sp + 1) * per);
   int e = sp * per + wave;
   int pn = e < e1 ? pidx[e] : 0;
   for (; e < e1; e += 4) {
      const PanelGeom& P = panels[pn];
      pn = pidx[min(e + 4, e1 - 1)];
      double sl, dl;
      laplace_integrals(x, P, sl, dl);
      const bool self = self_ok[e] && x[0] == P.c[0] && x[1] == P.c[1] && x[2] == P.c[2];
#pragma unroll
      for (int c = 0; c < NC; c++) {
         // a column past the last repeats it (sum unused)
         const double* cf = coef + (NC == 1 ? (size_t)col0 : (size_t)min(col0 + c, ncol - 1)) * 2 * ne;
         const double a = cf[2 * (size_t)e], b = cf[2 * (size_t)e + 1];
         double v = fma(a, sl, -(b * dl));
         if (self) v = fma(-4.0 * M_PI, b, v);
         s[c] += v;
      }
   }
#pragma unroll
   for (int c = 0; c < NC; c++) {
      __syncthreads();
      red[wave][lane] = s[c];
      __syncthreads();
      if (wave == 0 && 64 * g + lane < nq && col0 + c < ncol)
         part[((size_t)sp * ncol + col0 + c) * nq + j] = (red[0][lane] + red[1][lane]) + (red[2][lane] + red[3][lane]);
   }
}

// Transposed right-hand side: sum_e lam[out[e]] / |c_e - x_j|
__global__ void __launch_bounds__(256) k_rhs_t(int ne, int nq, int ng, int per, const double* __restrict__ cent,
                                               const int* __restrict__ out, const double* __restrict__ lam,
                                               const double* __restrict__ qpos, double* __restrict__ part) {
   __shared__ double red[4][64];
   const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
   const int g = blockIdx.x % ng, sp = blockIdx.x / ng;
   const int j = min(64 * g + lane, nq - 1);
   const double x0 = qpos[3 * (size_t)j], x1 = qpos[3 * (size_t)j + 1], x2 = qpos[3 * (size_t)j + 2];
   double s = 0.0;
   const int e1 = min(ne, (sp + 1) * per);
#pragma unroll 2
   for (int e = sp * per + wave; e < e1; e += 4) {
      const double d0 = x0 - cent[3 * (size_t)e], d1 = x1 - cent[3 * (size_t)e + 1], d2 = x2 - cent[3 * (size_t)e + 2];
      s += lam[out[e]] / sqrt(d0 * d0 + d1 * d1 + d2 * d2);
   }
   red[wave][lane] = s;
   __syncthreads();
   if (wave == 0 && 64 * g + lane < nq)
      part[(size_t)sp * nq + j] = (red[0][lane] + red[1][lane]) + (red[2][lane] + red[3][lane]);
}

// y[i] += sum over sp of part[sp * n + i], 64 i per block
__global__ void __launch_bounds__(256) k_add_parts(long long n, int ns, const double* __restrict__ part,
                                                   double* __restrict__ y) {
   __shared__ double red[4][64];
   const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
   const long long i = 64LL * blockIdx.x + lane;
   double s = 0.0;
   if (i < n) {
#pragma unroll 8
      for (int sp = wave; sp < ns; sp += 4) s += part[sp * n + i];
   }
   red[wave][lane] = s;
   __syncthreads();
   if (wave == 0 && i < n) y[i] += (red[0][lane] + red[1][lane]) + (red[2][lane] + red[3][lane]);
}

// --- sums over charges: panels on lanes -------------------------------------
// part[(sp * ncol + col) * ne + e], block (256 panels, part sp); with one part
// (ns = 1, always for SUM_RHS) the result itself.

enum { SUM_RHS, SUM_QUAL, SUM_COLLECT };

// RHS: rhs[out[e]] += sum_i q_i / |x_i - c_e|, zero charges skipped
//    (SurfaceOperator_makeRHS, SurfaceOperator.c:291-321)
// QUAL: rhs[e] = sum_j -dlp(charge j, panel e) q_j / fourpe
//    (Charge_makerhs_ecf_qual, Charge.c:129-142)
// COLLECT: y[e] = sum_j q_j slp(j, e), y2[e] = sum_j q_j dlp(j, e), with the
//    4 pi self term of k_potentials when the charge sits at the centroid
template <int MODE>
__device__ __forceinline__ void panel_result(int e, int col, double v, const int* out, double fourpe, long long ldr,
                                             double* y, double* y2) {
   if (MODE == SUM_RHS)
      y[col * ldr + out[e]] += v;
   else if (MODE == SUM_QUAL)
      y[col * ldr + e] = v / fourpe;
   else
      (col ? y2 : y)[e] = v;
}

// 1/sqrt(v) as two rounded operations: contracted, the compiler may make it
// one reciprocal root of 1 ulp.
__device__ __forceinline__ double inverse_root(double v) {
#pragma clang fp contract(off)
   const double r = sqrt(v);
   return 1.0 / r;
}

template <int MODE, int NC>
__global__ void __launch_bounds__(256) k_panel_sums(int ne, int nq, int ncol, int nb, int ns, int per,
                                                    const double* __restrict__ cent,
                                                    const PanelGeom* __restrict__ panels,
                                                    const int* __restrict__ idx, const int* __restrict__ self_ok,
                                                    const double* __restrict__ qpos, const double* __restrict__ q,
                                                    double fourpe, long long ldr, double* part, double* y,
                                                    double* y2) {
   constexpr int NS = MODE == SUM_COLLECT ? 2 : NC;
   const int b = blockIdx.x % nb, sp = blockIdx.x / nb, col0 = blockIdx.y * NC;
   const int e = min(256 * b + (int)threadIdx.x, ne - 1);
   double s[NS];
#pragma unroll
   for (int c = 0; c < NS; c++) s[c] = 0.0;
   const int j0 = sp * per, j1 = min(nq, j0 + per);
   if constexpr (MODE == SUM_RHS) {
      const double c0 = cent[3 * (size_t)e], c1 = cent[3 * (size_t)e + 1], c2 = cent[3 * (size_t)e + 2];
#pragma unroll 2
      for (int j = j0; j < j1; j++) {
         const double d0 = qpos[3 * (size_t)j] - c0, d1 = qpos[3 * (size_t)j + 1] - c1,
                      d2 = qpos[3 * (size_t)j + 2] - c2;
         const double w = inverse_root(d0 * d0 + d1 * d1 + d2 * d2);
         // a zero charge must not meet an infinite w
         const bool far = __all(w < HUGE_VAL);
#pragma unroll
         for (int c = 0; c < NS; c++) {
            const double qj = q[(NC == 1 ? (size_t)col0 : (size_t)min(col0 + c, ncol - 1)) * nq + j];
            if (far || qj != 0.0) s[c] = fma(qj, w, s[c]);   // uniform over the wave
         }
      }
   } else {
      const PanelGeom& P = panels[MODE == SUM_COLLECT ? idx[e] : e];
      PanelGeom F;   // the moment expansion's part, in registers
#pragma unroll
      for (int k = 0; k < 3; k++) F.c[k] = P.c[k];
#pragma unroll
      for (int k = 0; k < 9; k++) F.ax[k] = P.ax[k];
#pragma unroll
      for (int k = 0; k < 16; k++) F.mom[k] = P.mom[k];
      F.maxd = P.maxd;
      const bool self = MODE == SUM_COLLECT && self_ok[e];
      for (int j = j0; j < j1; j++) {
         const double x[3] = {qpos[3 * (size_t)j], qpos[3 * (size_t)j + 1], qpos[3 * (size_t)j + 2]};
         double xn, yn, zn, sl, dl;
         if (!laplace_far(x, F, xn, yn, zn, sl, dl)) laplace_near(x, P, xn, yn, zn, sl, dl);
         if constexpr (MODE == SUM_COLLECT) {
            if (self && x[0] == F.c[0] && x[1] == F.c[1] && x[2] == F.c[2]) dl += 4.0 * M_PI;
            s[0] = fma(q[j], sl, s[0]);
            s[1] = fma(q[j], dl, s[1]);
         } else {
#pragma unroll
            for (int c = 0; c < NS; c++)
               s[c] = fma(-dl, q[(NC == 1 ? (size_t)col0 : (size_t)min(col0 + c, ncol - 1)) * nq + j], s[c]);
         }
      }
   }
   if (256 * b + (int)threadIdx.x >= ne) return;
   const int nc = MODE == SUM_COLLECT ? 2 : ncol;
#pragma unroll
   for (int c = 0; c < NS; c++) {
      if (col0 + c >= nc) break;
      if (MODE == SUM_RHS || ns == 1)
         panel_result<MODE>(e, col0 + c, s[c], idx, fourpe, ldr, y, y2);
      else
         part[((size_t)sp * nc + col0 + c) * ne + e] = s[c];
   }
}

template <int MODE>
__global__ void __launch_bounds__(256) k_panel_parts(int ne, int nc, int ns, const double* __restrict__ part,
                                                     const int* __restrict__ idx, double fourpe, long long ldr,
                                                     double* y, double* y2) {
   const int e = blockIdx.x * 256 + threadIdx.x, col = blockIdx.y;
   if (e >= ne) return;
   double s = 0.0;
#pragma unroll 4
   for (int sp = 0; sp < ns; sp++) s += part[((size_t)sp * nc + col) * ne + e];
   panel_result<MODE>(e, col, s, idx, fourpe, ldr, y, y2);
}

// ---------------------------------------------------------------------------
namespace {
struct Split {
   int groups, parts, per;
};
// `groups` blocks side by side, the walk over n in parts of at least `least`
Split split_walk(int groups, int n, int least) {
   Split w;
   w.groups = groups;
   const int want = std::max(1, std::min(512, (ROUND_BLOCKS + groups - 1) / groups));
   w.per = std::max(least, (n + want - 1) / want);
   w.parts = std::max(1, (n + w.per - 1) / w.per);
   return w;
}
double* room(DBuf<double>& ws, size_t n) {
   if (n > ws.n) ws.alloc(n);
   return ws.p;
}

template <int MODE>
void panel_sums(int ne, int nq, int ncol, const double* cent, const PanelGeom* panels, const int* idx,
                const int* self_ok, const double* qpos, const double* q, double fourpe, long long ldr, double* y,
                double* y2, DBuf<double>* ws, hipStream_t s) {
   if (ne <= 0 || ncol <= 0) return;
   const Split w = split_walk((ne + 255) / 256, nq, MODE == SUM_RHS ? std::max(nq, 1) : 16);
   for (int c0 = 0; c0 < ncol; c0 += COL_CHUNK) {
      const int nc = std::min(COL_CHUNK, ncol - c0), np = MODE == SUM_COLLECT ? 2 : nc;
      double* part = MODE != SUM_RHS && w.parts > 1 ? room(*ws, (size_t)w.parts * np * ne) : nullptr;
      const double* qc = q + (size_t)c0 * nq;
      double* yc = y + (size_t)c0 * ldr;
      constexpr int NB = MODE == SUM_COLLECT ? 1 : 16;
      if (nc == 1 || NB == 1)
         hipLaunchKernelGGL((k_panel_sums<MODE, 1>), dim3(w.groups * w.parts), dim3(256), 0, s, ne, nq, nc, w.groups,
                            w.parts, w.per, cent, panels, idx, self_ok, qpos, qc, fourpe, ldr, part, yc, y2);
      else
         hipLaunchKernelGGL((k_panel_sums<MODE, NB>), dim3(w.groups * w.parts, (nc + NB - 1) / NB), dim3(256), 0, s,
                            ne, nq, nc, w.groups, w.parts, w.per, cent, panels, idx, self_ok, qpos, qc, fourpe, ldr,
                            part, yc, y2);
      if constexpr (MODE != SUM_RHS)
         if (w.parts > 1)
            hipLaunchKernelGGL((k_panel_parts<MODE>), dim3((ne + 255) / 256, np), dim3(256), 0, s, ne, np, w.parts,
                               part, idx, fourpe, ldr, yc, y2);
   }
}
}  // namespace

void launch_rhs(int ne, const double* cent, const int* out, int nq, int ncol, const double* qpos, const double* q,
                long long ldr, double* rhs, hipStream_t s) {
   panel_sums<SUM_RHS>(ne, nq, ncol, cent, nullptr, out, nullptr, qpos, q, 0.0, ldr, rhs, nullptr, nullptr, s);
}
void launch_qual_rhs(int n, const PanelGeom* panels, int nq, int ncol, const double* qpos, const double* q,
                     double fourpe, long long ldr, double* rhs, DBuf<double>& ws, hipStream_t s) {
   panel_sums<SUM_QUAL>(n, nq, ncol, nullptr, panels, nullptr, nullptr, qpos, q, fourpe, ldr, rhs, nullptr, &ws, s);
}
void launch_collect_t(int ne, const PanelGeom* panels, const int* pidx, const int* self_ok, int nq, const double* qpos,
                      const double* q, double* ssl, double* sdl, DBuf<double>& ws, hipStream_t s) {
   panel_sums<SUM_COLLECT>(ne, nq, 1, nullptr, panels, pidx, self_ok, qpos, q, 0.0, 0, ssl, sdl, &ws, s);
}

void launch_potentials(int nq, int ne, int ncol, const PanelGeom* panels, const int* pidx, const double* coef,
                       const int* self_ok, const double* qpos, double* phi, DBuf<double>& ws, hipStream_t s) {
   if (nq <= 0 || ne <= 0 || ncol <= 0) return;
   const Split w = split_walk((nq + 63) / 64, ne, 32);
   for (int c0 = 0; c0 < ncol; c0 += COL_CHUNK) {
      const int nc = std::min(COL_CHUNK, ncol - c0);
      double* part = room(ws, (size_t)w.parts * nc * nq);
      const double* cf = coef + (size_t)c0 * 2 * ne;
      const dim3 grid(w.groups * w.parts);
      if (nc == 1)
         hipLaunchKernelGGL((k_potentials<1>), grid, dim3(256), 0, s, ne, nq, nc, w.groups, w.per, panels, pidx, cf,
                            self_ok, qpos, part);
      else if (nc <= 8)
         hipLaunchKernelGGL((k_potentials<8>), grid, dim3(256), 0, s, ne, nq, nc, w.groups, w.per, panels, pidx, cf,
                            self_ok, qpos, part);
      else
         hipLaunchKernelGGL((k_potentials<32>), dim3(grid.x, (nc + 31) / 32), dim3(256), 0, s, ne, nq, nc, w.groups,
                            w.per, panels, pidx, cf, self_ok, qpos, part);
      const long long n = (long long)nc * nq;
      hipLaunchKernelGGL(k_add_parts, dim3((unsigned)((n + 63) / 64)), dim3(256), 0, s, n, w.parts, part,
                         phi + (size_t)c0 * nq);
   }
}
void launch_rhs_t(int nq, int ne, const double* cent, const int* out, const double* lam, const double* qpos, double* g,
                  DBuf<double>& ws, hipStream_t s) {
   if (nq <= 0 || ne <= 0) return;
   const Split w = split_walk((nq + 63) / 64, ne, 32);
   double* part = room(ws, (size_t)w.parts * nq);
   hipLaunchKernelGGL(k_rhs_t, dim3(w.groups * w.parts), dim3(256), 0, s, ne, nq, w.groups, w.per, cent, out, lam,
                      qpos, part);
   hipLaunchKernelGGL(k_add_parts, dim3((nq + 63) / 64), dim3(256), 0, s, (long long)nq, w.parts, part, g);
}

}  // namespace fsvd
