// Matrix-vector product of one compressed FFT-SVD operator on the GPU.
//
//   y = D_s xs + D_d xd  (near field, dense per-leaf blocks)
//     + U UTI IFFT( sum_c T[d-c] . FFT(PV_s VT xs_c + PV_d VT xd_c) )  (far field)
//
// Storage precision T is float (mixed mode) or double (FP64 mode); vectors
// enter and leave in FP64.  The forward apply is five launches per tree
// (k_project, k_source, k_translate, k_target, k_leaf; each covers every
// level).  The transposed operator runs the same stages with the roles of the
// two sides swapped and one input vector, and k_leaf_t for its output.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>
#include <stdexcept>
#include <type_traits>

#include "device.h"

namespace fsvd {

template <typename T>
struct Cplx;
template <>
struct Cplx<float> {
   using type = float2;
};
template <>
struct Cplx<double> {
   using type = double2;
};

template <typename T>
__device__ __forceinline__ T wave_sum(T v) {
#pragma unroll
   for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
   return v;
}

// Marks a loaded value as used here, so the compiler cannot sink its load
// into a later conditional block (where it would wait for it alone).
template <typename T>
__device__ __forceinline__ void keep(const T& v) {
   asm volatile("" ::"v"(v));
}

// Workgroups are dealt round-robin to the 8 XCDs.  Launches whose blocks
// share data across tree-order neighbours use a host-built block map
// (xcd_block_map): block b runs logical block map[b], and each XCD gets a
// contiguous tree-order range of about equal work, so neighbouring work
// shares one L2.  -1 marks padding blocks.
// The threads that share one cube's work: a whole block (__syncthreads
// between phases) or one wavefront.  A wavefront's LDS accesses are
// processed in issue order, so between its phases only the compiler's
// reordering has to be fenced.
struct BlockGroup {
   int tid, nt;
   __device__ void sync() const { __syncthreads(); }
};
struct WaveGroup {
   int tid;
   static constexpr int nt = 64;
   __device__ void sync() const {
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
   }
};
__device__ __forceinline__ BlockGroup block_group() { return BlockGroup{(int)threadIdx.x, (int)blockDim.x}; }

// e^{-2 pi i m / N} table
template <typename T, int N, typename G = BlockGroup>
__device__ __forceinline__ void twiddle_table(T* cs, T* sn, const G& gr = block_group()) {
   for (int m = gr.tid; m < N; m += gr.nt) {
      double s, c;
      sincospi(2.0 * m / N, &s, &c);
      cs[m] = (T)c;
      sn[m] = (T)s;
   }
}

// Forward transform of an n^3 grid zero-padded at offset n/2 into an
// N^3 box (N = 2n-1), real-to-complex with the half last dimension
// (reference FFT_forwardGridTransform, FFT.c:66-113).  g: n^3 in LDS,
// out: N*N*H complex in global memory.  Work arrays A (n*n*H) and
// B (n*N*H) in LDS.
template <int n, typename T, typename G = BlockGroup>
__device__ void grid_forward(const T* g, typename Cplx<T>::type* A, typename Cplx<T>::type* B,
                             typename Cplx<T>::type* out, const T* cs, const T* sn, const G& gr = block_group()) {
   constexpr int N = 2 * n - 1, H = N / 2 + 1, OFF = n / 2;
   const int tid = gr.tid, nt = gr.nt;
   // along k
   for (int e = tid; e < n * n * H; e += nt) {
      int c = e % H, ij = e / H;
      T re = 0, im = 0;
#pragma unroll
      for (int k = 0; k < n; k++) {
         int m = (c * (k + OFF)) % N;
         T v = g[ij * n + k];
         re += v * cs[m];
         im -= v * sn[m];
      }
      A[e].x = re;
      A[e].y = im;
   }
   gr.sync();
   // along j
   for (int e = tid; e < n * N * H; e += nt) {
      int c = e % H, b = (e / H) % N, i = e / (H * N);
      T re = 0, im = 0;
#pragma unroll
      for (int j = 0; j < n; j++) {
         int m = (b * (j + OFF)) % N;
         auto a = A[(i * n + j) * H + c];
         re += a.x * cs[m] + a.y * sn[m];
         im += a.y * cs[m] - a.x * sn[m];
      }
      B[e].x = re;
      B[e].y = im;
   }
   gr.sync();
   // along i
   for (int e = tid; e < N * N * H; e += nt) {
      int c = e % H, b = (e / H) % N, a = e / (H * N);
      T re = 0, im = 0;
#pragma unroll
      for (int i = 0; i < n; i++) {
         int m = (a * (i + OFF)) % N;
         auto v = B[(i * N + b) * H + c];
         re += v.x * cs[m] + v.y * sn[m];
         im += v.y * cs[m] - v.x * sn[m];
      }
      out[e].x = re;
      out[e].y = im;
   }
}

// Inverse transform of an N*N*H half spectrum, cropped back to the n^3
// grid at offset n/2 and scaled by 1/N^3 (reference
// FFT_backwardGridTransform, FFT.c:117-150).  S in LDS (N*N*H),
// C1 (n*N*H), C2 (n*n*H) in LDS, h (n^3) in LDS.
template <int n, typename T, typename G = BlockGroup>
__device__ void grid_backward(const typename Cplx<T>::type* S, typename Cplx<T>::type* C1,
                              typename Cplx<T>::type* C2, T* h, const T* cs, const T* sn,
                              const G& gr = block_group()) {
   constexpr int N = 2 * n - 1, H = N / 2 + 1, OFF = n / 2;
   const int tid = gr.tid, nt = gr.nt;
   for (int e = tid; e < n * N * H; e += nt) {
      int c = e % H, b = (e / H) % N, i = e / (H * N);
      T re = 0, im = 0;
#pragma unroll
      for (int a = 0; a < N; a++) {
         int m = (a * (i + OFF)) % N;
         auto v = S[(a * N + b) * H + c];
         re += v.x * cs[m] - v.y * sn[m];
         im += v.y * cs[m] + v.x * sn[m];
      }
      C1[e].x = re;
      C1[e].y = im;
   }
   gr.sync();
   for (int e = tid; e < n * n * H; e += nt) {
      int c = e % H, j = (e / H) % n, i = e / (H * n);
      T re = 0, im = 0;
#pragma unroll
      for (int b = 0; b < N; b++) {
         int m = (b * (j + OFF)) % N;
         auto v = C1[(i * N + b) * H + c];
         re += v.x * cs[m] - v.y * sn[m];
         im += v.y * cs[m] + v.x * sn[m];
      }
      C2[e].x = re;
      C2[e].y = im;
   }
   gr.sync();
   const T scale = (T)(1.0 / ((double)N * N * N));
   for (int e = tid; e < n * n * n; e += nt) {
      int k = e % n, ij = e / n;
      const auto* row = C2 + ij * H;
      T v = row[0].x;
#pragma unroll
      for (int c = 1; c < H; c++) {
         int m = (c * (k + OFF)) % N;
         v += (T)2 * (row[c].x * cs[m] - row[c].y * sn[m]);
      }
      h[e] = v * scale;
   }
}

template <int n>
struct FarSizes {
   static constexpr int N = 2 * n - 1, H = N / 2 + 1, PAD = N * N * H, GP3 = n * n * n;
};

// ---------------------------------------------------------------------------
// Forward apply, one launch per stage over all levels of a tree:
//   k_project    chunk of a source cube's panels: partial VT.xs, VT.xd
//   k_source     source cube: sum of chunk partials, PV interpolation onto
//                the n^3 grid, zero-padded r2c DFT -> spectrum
//   k_translate  tile of <= TR_TILE target cubes x a bin chunk: sum over each
//                interaction list of T . spectrum, from LDS
//   k_target     target cube: cropped c2r DFT, w = UTI h
//   k_leaf       leaf: near-field block apply plus U w of every target cube
//                containing the leaf, writes y
// Every sum runs in a fixed order: the result does not depend on scheduling.

// Operator entries read once per launch are loaded nontemporal (NT), so
// they do not evict reusable lines from L2.  The column-batched launches
// read each block once per column copy and load it normally, so that the
// copies after the first hit L2.
template <bool NT, typename T>
__device__ __forceinline__ T ld_op(const T* p) {
   if constexpr (NT)
      return __builtin_nontemporal_load(p);
   else
      return *p;
}

// Rows e of a column-major E x m block (column c at blk + c*E), streamed
// with unit stride by G = 256/Ec column groups per row chunk; returns the
// thread's partial sum for (row e, layer inputs x0/x1 selected by e >= split).
template <typename T, bool NT>
__device__ __forceinline__ T stream_rows(const T* __restrict__ colp, int E, int m, int g, int G, const T* xl) {
   // eight columns in flight per thread
   const long long step = (long long)G * E;
   T a0 = 0, a1 = 0, a2 = 0, a3 = 0;
   int c = g;
   for (; c + 7 * G < m; c += 8 * G) {
      const T* pc = colp + (long long)c * E;
      T d[8];
#pragma unroll
      for (int u = 0; u < 8; u++) d[u] = ld_op<NT>(pc + u * step);
      a0 += d[0] * xl[c];
      a1 += d[1] * xl[c + G];
      a2 += d[2] * xl[c + 2 * G];
      a3 += d[3] * xl[c + 3 * G];
      a0 += d[4] * xl[c + 4 * G];
      a1 += d[5] * xl[c + 5 * G];
      a2 += d[6] * xl[c + 6 * G];
      a3 += d[7] * xl[c + 7 * G];
   }
   if (c < m) {
      // the last partial batch, all of its loads in flight together
      const T* pc = colp + (long long)c * E;
      T d[7];
#pragma unroll
      for (int u = 0; u < 7; u++) d[u] = c + u * G < m ? ld_op<NT>(pc + u * step) : (T)0;
#pragma unroll
      for (int u = 0; u < 7; u++)
         if (c + u * G < m) a0 += d[u] * xl[c + u * G];
   }
   return (a0 + a1) + (a2 + a3);
}

// Projection: one chunk of a source cube's panels per wavefront (four per
// block), tpart[out_off + e] = sum_i VT[e, i] xs[i] and, with two layers (NL),
// tpart[out_off + r + e] = sum_i VT[e, i] xd[i] over the chunk's columns.
// Lane (g, e) owns row e and the columns g, g + G, ... (G = 64 / rows of the
// row chunk); the G partial sums of a row are added in group order.
template <typename T, bool NT, int NL>
__global__ void __launch_bounds__(256) k_project(const ProjChunk* __restrict__ chunks, int nchunk,
                                                 const T* __restrict__ VTc, const double* __restrict__ xs,
                                                 const double* __restrict__ xd, T* __restrict__ tpart, int wave_lds,
                                                 int ncol, long long cs_x, long long cs_tpart) {
   extern __shared__ __align__(16) unsigned char smem[];
   const ColBlk cb = col_block(ncol);
   const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, ci = cb.b * 4 + wave;
   if (ci >= nchunk) return;
   xs += cb.c * cs_x;
   if (NL == 2) xd += cb.c * cs_x;
   tpart += cb.c * cs_tpart;
   const WaveGroup gr{lane};
   const ProjChunk c = chunks[ci];
   const int m = c.ncol, E = c.r;
   T* part = (T*)(smem + (size_t)wave * wave_lds);   // NL*64
   T* xl = part + NL * 64;                            // NL*m
   // x staged four columns per lane at a time, loads before stores
   for (int i0 = lane; i0 < m; i0 += 256) {
      double a[4], b[4];
#pragma unroll
      for (int u = 0; u < 4; u++) {
         const int i = i0 + 64 * u;
         a[u] = i < m ? xs[c.p0 + i] : 0.0;
         b[u] = NL == 2 && i < m ? xd[c.p0 + i] : 0.0;
      }
#pragma unroll
      for (int u = 0; u < 4; u++) {
         const int i = i0 + 64 * u;
         if (i < m) {
            xl[i] = (T)a[u];
            if (NL == 2) xl[m + i] = (T)b[u];
         }
      }
   }
   gr.sync();
   const T* blk = VTc + c.vt_off;
   for (int e0 = 0; e0 < E; e0 += 64) {
      const int Ec = min(64, E - e0), G = 64 / Ec;
      const int g = lane / Ec, e = e0 + lane - g * Ec;
      T as = 0, ad = 0;
      if (g < G) {
         const T* colp = blk + e;
         const long long step = (long long)G * E;
         T s0 = 0, s1 = 0, d0 = 0, d1 = 0;
         int i = g;
         // eight columns in flight per lane
         for (; i + 7 * G < m; i += 8 * G) {
            T v[8];
#pragma unroll
            for (int u = 0; u < 8; u++) v[u] = ld_op<NT>(colp + (long long)i * E + u * step);
#pragma unroll
            for (int u = 0; u < 8; u += 2) {
               s0 += v[u] * xl[i + u * G];
               if (NL == 2) d0 += v[u] * xl[m + i + u * G];
               s1 += v[u + 1] * xl[i + (u + 1) * G];
               if (NL == 2) d1 += v[u + 1] * xl[m + i + (u + 1) * G];
            }
         }
         if (i < m) {
            // the last partial batch, all of its loads in flight together
            T v[7];
#pragma unroll
            for (int u = 0; u < 7; u++)
               v[u] = i + u * G < m ? ld_op<NT>(colp + (long long)i * E + u * step) : (T)0;
#pragma unroll
            for (int u = 0; u < 7; u++)
               if (i + u * G < m) {
                  s0 += v[u] * xl[i + u * G];
                  if (NL == 2) d0 += v[u] * xl[m + i + u * G];
               }
         }
         as = s0 + s1;
         ad = d0 + d1;
      }
      part[lane] = as;
      if (NL == 2) part[64 + lane] = ad;
      gr.sync();
      if (lane < Ec) {
         T ss = 0, sd = 0;
         for (int gg = 0; gg < G; gg++) {
            ss += part[gg * Ec + lane];
            if (NL == 2) sd += part[64 + gg * Ec + lane];
         }
         tpart[c.out_off + e0 + lane] = ss;
         if (NL == 2) tpart[c.out_off + E + e0 + lane] = sd;
      }
      gr.sync();
   }
}

// k_project for NC columns per wave (column-batched applies): each VT entry
// is loaded once and multiplied into the NC columns' accumulators, each in
// k_project's order (inputs interleaved, input i of column j at
// xl[i * NC + j]), so every column's partials are k_project's bit for bit.
// A partial last group repeats its last column and stores only its own.
// columns per wave: four FP32, two FP64 (whose four would take the whole
// LDS of a CU for the widest chunk)
template <typename T>
constexpr int proj_nc() { return sizeof(T) == 4 ? 4 : 2; }
template <typename T, int NC>
__global__ void __launch_bounds__(256) k_project_mc(const ProjChunk* __restrict__ chunks, int nchunk,
                                                    const T* __restrict__ VTc, const double* __restrict__ xs,
                                                    const double* __restrict__ xd, T* __restrict__ tpart,
                                                    int wave_lds, int ncol, long long cs_x, long long cs_tpart) {
   extern __shared__ __align__(16) unsigned char smem[];
   const int ngrp = (ncol + NC - 1) / NC;
   const ColBlk cb = col_block(ngrp);
   const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, ci = cb.b * 4 + wave;
   if (ci >= nchunk) return;
   const int c0 = cb.c * NC, nc = min(NC, ncol - c0);
   const WaveGroup gr{lane};
   const ProjChunk c = chunks[ci];
   const int m = c.ncol, E = c.r;
   T* part = (T*)(smem + (size_t)wave * wave_lds);   // 2 * 64 * NC
   T* xl = part + 128 * NC;                           // 2 * m * NC
   for (int i = lane; i < m; i += 64) {
#pragma unroll
      for (int j = 0; j < NC; j++) {
         const long long o = (long long)(c0 + min(j, nc - 1)) * cs_x + c.p0 + i;
         xl[(size_t)i * NC + j] = (T)xs[o];
         xl[(size_t)(m + i) * NC + j] = (T)xd[o];
      }
   }
   gr.sync();
   const T* blk = VTc + c.vt_off;
   for (int e0 = 0; e0 < E; e0 += 64) {
      const int Ec = min(64, E - e0), G = 64 / Ec;
      const int g = lane / Ec, e = e0 + lane - g * Ec;
      T as[NC], ad[NC];
#pragma unroll
      for (int j = 0; j < NC; j++) as[j] = ad[j] = 0;
      if (g < G) {
         const T* colp = blk + e;
         const long long step = (long long)G * E;
         T s0[NC], s1[NC], d0[NC], d1[NC];
#pragma unroll
         for (int j = 0; j < NC; j++) s0[j] = s1[j] = d0[j] = d1[j] = 0;
         int i = g;
         for (; i + 7 * G < m; i += 8 * G) {
            T v[8];
#pragma unroll
            for (int u = 0; u < 8; u++) v[u] = colp[(long long)i * E + u * step];
#pragma unroll
            for (int u = 0; u < 8; u += 2) {
               const T* xa = xl + (size_t)(i + u * G) * NC;
               const T* xb = xl + (size_t)(i + (u + 1) * G) * NC;
               const T* ya = xl + (size_t)(m + i + u * G) * NC;
               const T* yb = xl + (size_t)(m + i + (u + 1) * G) * NC;
#pragma unroll
               for (int j = 0; j < NC; j++) {
                  s0[j] += v[u] * xa[j];
                  d0[j] += v[u] * ya[j];
                  s1[j] += v[u + 1] * xb[j];
                  d1[j] += v[u + 1] * yb[j];
               }
            }
         }
         if (i < m) {
            T v[7];
#pragma unroll
            for (int u = 0; u < 7; u++) v[u] = i + u * G < m ? colp[(long long)i * E + u * step] : (T)0;
#pragma unroll
            for (int u = 0; u < 7; u++)
               if (i + u * G < m) {
                  const T* xa = xl + (size_t)(i + u * G) * NC;
                  const T* ya = xl + (size_t)(m + i + u * G) * NC;
#pragma unroll
                  for (int j = 0; j < NC; j++) {
                     s0[j] += v[u] * xa[j];
                     d0[j] += v[u] * ya[j];
                  }
               }
         }
#pragma unroll
         for (int j = 0; j < NC; j++) {
            as[j] = s0[j] + s1[j];
            ad[j] = d0[j] + d1[j];
         }
      }
#pragma unroll
      for (int j = 0; j < NC; j++) {
         part[(2 * j) * 64 + lane] = as[j];
         part[(2 * j + 1) * 64 + lane] = ad[j];
      }
      gr.sync();
      if (lane < Ec) {
         for (int j = 0; j < nc; j++) {
            T ss = 0, sd = 0;
            for (int gg = 0; gg < G; gg++) {
               ss += part[(2 * j) * 64 + gg * Ec + lane];
               sd += part[(2 * j + 1) * 64 + gg * Ec + lane];
            }
            T* tp = tpart + (long long)(c0 + j) * cs_tpart;
            tp[c.out_off + e0 + lane] = ss;
            tp[c.out_off + E + e0 + lane] = sd;
         }
      }
      gr.sync();
   }
}

template <int n, typename T, bool NT, int NL, typename G>
__device__ void source_body(const SrcPlan& d, const T* __restrict__ tpart, const T* __restrict__ PV,
                            typename Cplx<T>::type* __restrict__ spec, unsigned char* smem, const G& gr) {
   using C2 = typename Cplx<T>::type;
   constexpr int N = FarSizes<n>::N, H = FarSizes<n>::H, GP3 = FarSizes<n>::GP3;
   C2* A = (C2*)smem;            // n*n*H
   C2* B = A + n * n * H;        // n*N*H
   T* cs = (T*)(B + n * N * H);  // N
   T* sn = cs + N;               // N
   T* g = sn + N;                // GP3
   T* part = g + GP3;            // partial grid values (block groups)
   const int tid = gr.tid, nt = gr.nt, R2 = NL * d.r;
   T* t = part + (nt > GP3 ? nt : 0);   // NL*r: ts then td
   twiddle_table<T, N>(cs, sn, gr);
   // sum of the chunk partials in chunk order, eight loads in flight
   for (int k = tid; k < R2; k += nt) {
      const T* pp = tpart + d.part_off + k;
      T a = 0;
      int j = 0;
      for (; j + 7 < d.nchunk; j += 8) {
         T v[8];
#pragma unroll
         for (int u = 0; u < 8; u++) v[u] = pp[(long long)(j + u) * R2];
#pragma unroll
         for (int u = 0; u < 8; u++) a += v[u];
      }
      if (j < d.nchunk) {
         T v[7];
#pragma unroll
         for (int u = 0; u < 7; u++) v[u] = j + u < d.nchunk ? pp[(long long)(j + u) * R2] : (T)0;
#pragma unroll
         for (int u = 0; u < 7; u++)
            if (j + u < d.nchunk) a += v[u];
      }
      t[k] = a;
   }
   gr.sync();
   // g = PV t over the rows (PVs then PVd, k-major): thread (kg, q) sums
   // the rows k = kg, kg + KG, ... so every thread streams PV
   const T* pv = PV + d.pv_off;
   const int KG = nt >= GP3 ? nt / GP3 : 1, QW = nt / KG;
   for (int q0 = 0; q0 < GP3; q0 += QW) {
      const int kg = tid / QW, q = q0 + tid - kg * QW;
      T a0 = 0, a1 = 0, a2 = 0, a3 = 0;
      if (q < GP3) {
         // eight rows in flight per thread
         int k = kg;
         for (; k + 7 * KG < R2; k += 8 * KG) {
            T v[8];
#pragma unroll
            for (int u = 0; u < 8; u++) v[u] = ld_op<NT>(pv + (long long)(k + u * KG) * GP3 + q);
            a0 += v[0] * t[k];
            a1 += v[1] * t[k + KG];
            a2 += v[2] * t[k + 2 * KG];
            a3 += v[3] * t[k + 3 * KG];
            a0 += v[4] * t[k + 4 * KG];
            a1 += v[5] * t[k + 5 * KG];
            a2 += v[6] * t[k + 6 * KG];
            a3 += v[7] * t[k + 7 * KG];
         }
         if (k < R2) {
            // the last partial batch, all of its loads in flight together
            T v[7];
#pragma unroll
            for (int u = 0; u < 7; u++)
               v[u] = k + u * KG < R2 ? ld_op<NT>(pv + (long long)(k + u * KG) * GP3 + q) : (T)0;
#pragma unroll
            for (int u = 0; u < 7; u++)
               if (k + u * KG < R2) a0 += v[u] * t[k + u * KG];
         }
      }
      const T sum = (a0 + a1) + (a2 + a3);
      if (KG == 1) {
         if (q < GP3) g[q] = sum;
      } else {
         part[kg * QW + (q - q0)] = sum;
         gr.sync();
         if (tid < QW && q0 + tid < GP3) {
            T acc = 0;
            for (int gg = 0; gg < KG; gg++) acc += part[gg * QW + tid];
            g[q0 + tid] = acc;
         }
      }
      gr.sync();
   }
   grid_forward<n, T>(g, A, B, spec + d.spec_off, cs, sn, gr);
}

// ---------------------------------------------------------------------------
// Cubes of four grid points per side (N = 7, H = 4, 64 grid values), one per
// wavefront.  What bounds grid_forward and grid_backward here is the LDS: three
// reads per complex multiply-add (the value, the table's cosine and sine) and an
// integer remainder for the table's index.  In these forms a lane makes a whole
// line of the seven-point transform from values read once, with literal
// twiddles; the other two dimensions take their four twiddles per lane from a
// 7-entry table, once.  About 45 LDS operations per target cube instead of 160.
// P columns side by side where a line's 28 lanes leave room for two.
// Kernel times before and after: k_target 6.6 to 4.9 us (FP64, 1280 panels), 17.7
// to 15.2 us (FP32, 30 000 panels; the other cubes bound it now), 70 to 62 us
// (100 000; UTI from memory bounds it); 64 FP32 columns of 30 000 panels: target
// 917 to 465 us a tree, source 575 to 407, of which the other cubes take 208
// and 225.

// e^{-2 pi i m / 7} = C7[m] - i S7[m]
constexpr double C7[7] = {1.0,
                          0.62348980185873353053,
                          -0.22252093395631440429,
                          -0.90096886790241912624,
                          -0.90096886790241912624,
                          -0.22252093395631440429,
                          0.62348980185873353053};
constexpr double S7[7] = {0.0,
                          0.78183148246802980871,
                          0.97492791218182360702,
                          0.43388373911755812048,
                          -0.43388373911755812048,
                          -0.97492791218182360702,
                          -0.78183148246802980871};

template <typename T>
__device__ __forceinline__ void table7(typename Cplx<T>::type* tw, int lane) {
   T c = 1, sn = 0;
#pragma unroll
   for (int m = 1; m < 7; m++) {
      c = lane == m ? (T)C7[m] : c;
      sn = lane == m ? (T)S7[m] : sn;
   }
   if (lane < 7) {
      tw[lane].x = c;
      tw[lane].y = sn;
   }
}

// v from lane ^ X, X a power of two below 16
template <int CTRL>
__device__ __forceinline__ float dpp_move(float v) {
   return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}
template <int CTRL>
__device__ __forceinline__ double dpp_move(double v) {
   const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, false);
   const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, false);
   return __hiloint2double(hi, lo);
}
template <int X, typename T>
__device__ __forceinline__ T lane_xor(T v) {
   if constexpr (X == 8) return dpp_move<0x128>(v);                       // row rotate by 8
   if constexpr (X == 4) return dpp_move<0x1B>(dpp_move<0x141>(v));       // ^7, then ^3 within quads
   if constexpr (X == 2) return dpp_move<0x4E>(v);
   return dpp_move<0xB1>(v);
}

// Sums of NV values over the 16 lanes of a row, in the order of a butterfly
// over 8, 4, 2, 1; each step hands half of the values on while there are two or
// more, so v[0] ends as the sum of value `lane15 / (16 / NV)`.
template <int NV, int X, typename T>
__device__ __forceinline__ void row_sums(T* v, int lane15) {
   if constexpr (NV > 1) {
      const bool up = lane15 & X;
#pragma unroll
      for (int k = 0; k < NV / 2; k++) {
         const T give = up ? v[k] : v[k + NV / 2], mine = up ? v[k + NV / 2] : v[k];
         v[k] = mine + lane_xor<X>(give);
      }
   } else {
      v[0] += lane_xor<X>(v[0]);
   }
   if constexpr (X > 1) row_sums<(NV > 1 ? NV / 2 : 1), X / 2>(v, lane15);
}

// A source cube's spectra, columns 0 .. nc - 1 of the group: as source_body.
template <typename T, bool NT, int NL, int NC>
__device__ void source4(const SrcPlan& d, const T* __restrict__ tpart, long long cs_tpart, const T* __restrict__ PV,
                        typename Cplx<T>::type* __restrict__ spec, long long cs_spec, int nc, unsigned char* smem,
                        int lane) {
   using C2 = typename Cplx<T>::type;
   constexpr int P = NC > 1 ? 2 : 1;
   T* g = (T*)smem;              // 64
   C2* A = (C2*)(g + 64);        // 16 lines x 4
   C2* B = A + 64;               // P x 28 lines x 4
   C2* tw = B + 112 * P;         // 7
   T* t = (T*)(tw + 8);          // NC x NL r: ts then td
   const WaveGroup gr{lane};
   const int R2 = NL * d.r;
   // the first rows of PV travel while the chunk partials are summed
   const T* pv = PV + d.pv_off + lane;
   T v[8];
#pragma unroll
   for (int u = 0; u < 8; u++) v[u] = R2 ? ld_op<NT>(pv + (u < R2 ? u : 0) * 64) : (T)0;
   table7<T>(tw, lane);
#pragma unroll
   for (int j = 0; j < NC; j++) {
      if (j >= nc) break;
      for (int k = lane; k < R2; k += 64) {
         // in chunk order, eight loads in flight
         const T* pp = tpart + j * cs_tpart + d.part_off + k;
         T a = 0;
         int i = 0;
         for (; i + 7 < d.nchunk; i += 8) {
            T q[8];
#pragma unroll
            for (int u = 0; u < 8; u++) q[u] = pp[(long long)(i + u) * R2];
#pragma unroll
            for (int u = 0; u < 8; u++) a += q[u];
         }
         if (i < d.nchunk) {
            T q[7];
#pragma unroll
            for (int u = 0; u < 7; u++) q[u] = i + u < d.nchunk ? pp[(long long)(i + u) * R2] : (T)0;
#pragma unroll
            for (int u = 0; u < 7; u++)
               if (i + u < d.nchunk) a += q[u];
         }
         t[j * R2 + k] = a;
      }
   }
   gr.sync();
   T a[NC][4];
#pragma unroll
   for (int j = 0; j < NC; j++)
#pragma unroll
      for (int u = 0; u < 4; u++) a[j][u] = 0;
   int k = 0;
   for (; k + 8 <= R2; k += 8) {
      T x[8];
#pragma unroll
      for (int u = 0; u < 8; u++) x[u] = v[u];
      // the next rows (past the last: its row again, unused)
      if (k + 8 < R2)
#pragma unroll
         for (int u = 0; u < 8; u++) v[u] = ld_op<NT>(pv + (long long)min(k + 8 + u, R2 - 1) * 64);
#pragma unroll
      for (int j = 0; j < NC; j++) {
         const T* tj = t + (j < nc ? j : 0) * R2 + k;
#pragma unroll
         for (int u = 0; u < 8; u++) a[j][u & 3] = fma(x[u], tj[u], a[j][u & 3]);
      }
   }
   if (k < R2) {
#pragma unroll
      for (int j = 0; j < NC; j++) {
         const T* tj = t + (j < nc ? j : 0) * R2 + k;
#pragma unroll
         for (int u = 0; u < 7; u++)
            if (k + u < R2) a[j][u & 3] = fma(v[u], tj[u], a[j][u & 3]);
      }
   }
   // twiddles of the first dimension (lane & 3 = c) and, for b = lane & 3
   // and b + 4, of the second; all for points 2 .. 5 of the box
   const int c4 = lane & 3;
   C2 w0[4], w1[4];
#pragma unroll
   for (int k = 0; k < 4; k++) {
      w0[k] = tw[(c4 * (k + 2)) % 7];
      w1[k] = tw[((c4 + 4) * (k + 2)) % 7];
   }
#pragma unroll
   for (int j0 = 0; j0 < NC; j0 += P) {
      if (j0 >= nc) break;
#pragma unroll
      for (int p = 0; p < P; p++) {
         if (j0 + p >= nc) break;
         const int j = j0 + p;
         g[lane] = (a[j][0] + a[j][1]) + (a[j][2] + a[j][3]);
         gr.sync();
         {
            const T* row = g + (lane & ~3);
            T re = 0, im = 0;
#pragma unroll
            for (int k = 0; k < 4; k++) {
               re = fma(row[k], w0[k].x, re);
               im = fma(-row[k], w0[k].y, im);
            }
            A[lane].x = re;   // (i, j, c)
            A[lane].y = im;
         }
         gr.sync();
         {
            const int c = (lane >> 2) & 3, i = lane >> 4;
            T r0 = 0, m0 = 0, r1 = 0, m1 = 0;
#pragma unroll
            for (int k = 0; k < 4; k++) {
               const C2 z = A[(4 * i + k) * 4 + c];
               r0 = fma(z.y, w0[k].y, fma(z.x, w0[k].x, r0));
               m0 = fma(-z.x, w0[k].y, fma(z.y, w0[k].x, m0));
               r1 = fma(z.y, w1[k].y, fma(z.x, w1[k].x, r1));
               m1 = fma(-z.x, w1[k].y, fma(z.y, w1[k].x, m1));
            }
            C2* Bp = B + 112 * p + 28 * i + c;   // (i, b, c)
            Bp[4 * c4].x = r0;
            Bp[4 * c4].y = m0;
            if (c4 < 3) {
               Bp[4 * (c4 + 4)].x = r1;
               Bp[4 * (c4 + 4)].y = m1;
            }
         }
         gr.sync();
      }
      const int p = P > 1 && lane >= 28 ? 1 : 0, bc = lane - 28 * p;
      if (bc < 28 && j0 + p < nc) {
         C2 z[4];
#pragma unroll
         for (int i = 0; i < 4; i++) z[i] = B[112 * p + 28 * i + bc];
         C2* o = spec + (j0 + p) * cs_spec + d.spec_off + bc;
#pragma unroll
         for (int m = 0; m < 7; m++) {
            T re = 0, im = 0;
#pragma unroll
            for (int i = 0; i < 4; i++) {
               const T cs = (T)C7[(m * (i + 2)) % 7], sn = (T)S7[(m * (i + 2)) % 7];
               re = fma(z[i].y, sn, fma(z[i].x, cs, re));
               im = fma(-z[i].x, sn, fma(z[i].y, cs, im));
            }
            C2 y;
            y.x = re;
            y.y = im;
            o[28 * m] = y;
         }
      }
      gr.sync();
   }
}

template <typename T>
__host__ __device__ constexpr size_t source4_lds(int maxr, int NC) {
   return (sizeof(T) * (64 + 2 * (64 + 112 * (NC > 1 ? 2 : 1) + 8) + 2 * (size_t)maxr * NC) + 15) / 16 * 16;
}

// A target cube's w = UTI h, columns 0 .. nc - 1 of the group: as target_body,
// each spectrum transformed straight from memory, each UTI row read once.
template <typename T, int NC>
__device__ void target4(const TgtPlan& d, const T* __restrict__ UTI, const typename Cplx<T>::type* __restrict__ acc,
                        long long cs_acc, T* __restrict__ w, long long cs_w, int nc, unsigned char* smem, int lane) {
   using C2 = typename Cplx<T>::type;
   constexpr int P = NC > 1 ? 2 : 1, RU = NC > 1 ? 2 : 4, RP = 4 * RU, NV = NC * RU;
   T* h = (T*)smem;             // NC x 64
   C2* C1 = (C2*)(h + 64 * NC); // P x 28 lines x 4
   C2* Cc = C1 + 112 * P;       // 16 lines x 4
   C2* tw = Cc + 64;            // 7
   const WaveGroup gr{lane};
   const int kr = lane >> 4, ql = lane & 15;
   const T* uti = UTI + d.uti_off + ql;
   // RU rows per lane; of a single column the first ones travel during the
   // transform (of several they would cost registers that the sums need)
   T x[RU][4];
   auto load_rows = [&](int k) {
#pragma unroll
      for (int u = 0; u < RU; u++) {
         const T* row = uti + (long long)(k + 4 * u < d.r ? k + 4 * u : 0) * 64;
#pragma unroll
         for (int q = 0; q < 4; q++) x[u][q] = row[16 * q];
      }
   };
   const int p = P > 1 && lane >= 28 ? 1 : 0, bc = lane - 28 * p;
   C2 z[7];
   auto load_line = [&](int j0) {
      const C2* in = acc + (j0 + p < nc ? j0 + p : j0) * cs_acc + d.acc_off + (bc < 28 ? bc : 0);
#pragma unroll
      for (int m = 0; m < 7; m++) z[m] = in[28 * m];
   };
   load_line(0);
   if (NC == 1 && kr < d.r) load_rows(kr);
   table7<T>(tw, lane);
   gr.sync();
   // twiddles of point (lane & 3) + 2, for the second and third dimension
   C2 wl[7];
#pragma unroll
   for (int b = 1; b < 7; b++) wl[b] = tw[(b * ((lane & 3) + 2)) % 7];
#pragma unroll 1
   for (int j0 = 0; j0 < NC && j0 < nc; j0 += P) {
      if (bc < 28) {
         C2* o = C1 + 112 * p + bc;   // (i, b, c)
#pragma unroll
         for (int i = 0; i < 4; i++) {
            T re = 0, im = 0;
#pragma unroll
            for (int m = 0; m < 7; m++) {
               const T cs = (T)C7[(m * (i + 2)) % 7], sn = (T)S7[(m * (i + 2)) % 7];
               re = fma(-z[m].y, sn, fma(z[m].x, cs, re));
               im = fma(z[m].x, sn, fma(z[m].y, cs, im));
            }
            o[28 * i].x = re;
            o[28 * i].y = im;
         }
      }
      if (j0 + P < nc) load_line(j0 + P);
      gr.sync();
#pragma unroll
      for (int pp = 0; pp < P; pp++) {
         if (j0 + pp >= nc) break;
         {
            const int c = (lane >> 2) & 3, i = lane >> 4;
            const C2* in = C1 + 112 * pp + 28 * i + c;
            T re = in[0].x, im = in[0].y;
#pragma unroll
            for (int b = 1; b < 7; b++) {
               const C2 y = in[4 * b];
               re = fma(-y.y, wl[b].y, fma(y.x, wl[b].x, re));
               im = fma(y.x, wl[b].y, fma(y.y, wl[b].x, im));
            }
            C2 y;
            y.x = re;
            y.y = im;
            Cc[16 * i + 4 * (lane & 3) + c] = y;   // (i, j, c)
         }
         gr.sync();
         {
            const C2* row = Cc + (lane & ~3);
            T v = row[0].x;
#pragma unroll
            for (int c = 1; c < 4; c++) v = fma((T)2, fma(-row[c].y, wl[c].y, row[c].x * wl[c].x), v);
            h[64 * (j0 + pp) + lane] = v * (T)(1.0 / 343.0);
         }
         gr.sync();
      }
   }
   T hq[NC][4];
#pragma unroll
   for (int j = 0; j < NC; j++)
#pragma unroll
      for (int q = 0; q < 4; q++) hq[j][q] = h[64 * (j < nc ? j : 0) + 16 * q + ql];
   for (int k = kr; k < d.r; k += RP) {
      if (NC > 1) load_rows(k);
      T s[NV];
#pragma unroll
      for (int j = 0; j < NC; j++)
#pragma unroll
         for (int u = 0; u < RU; u++) {
            T a = x[u][0] * hq[j][0];
#pragma unroll
            for (int q = 1; q < 4; q++) a = fma(x[u][q], hq[j][q], a);
            s[RU * j + u] = a;
         }
      if (NC == 1 && k + RP < d.r) load_rows(k + RP);
      row_sums<NV, 8>(s, ql);
      const int idx = ql / (16 / NV), j = idx / RU, row = k + 4 * (idx % RU);
      if (ql % (16 / NV) == 0 && j < nc && row < d.r) w[j * cs_w + d.w_off + row] = s[0];
   }
}

template <typename T>
__host__ __device__ constexpr size_t target4_lds(int NC) {
   return (sizeof(T) * (64 * NC + 2 * (112 * (NC > 1 ? 2 : 1) + 64 + 8)) + 15) / 16 * 16;
}

// LDS of one source cube's work (block groups of nt threads)
template <typename T>
__host__ __device__ constexpr size_t source_cube_lds(int n, int maxr, int nt) {
   return sizeof(typename Cplx<T>::type) * (size_t)(n * n * ((2 * n - 1) / 2 + 1) + n * (2 * n - 1) * ((2 * n - 1) / 2 + 1)) +
          sizeof(T) * (size_t)(2 * (2 * n - 1) + n * n * n + (nt > n * n * n ? nt : 0) + 2 * maxr) + 64;
}

// Source cubes, one launch: the nbig cubes with other than four grid points
// per side first, one block of CUBE_NT threads each (these cubes are few,
// so each gets many loads in flight), then the cubes of four grid points
// per side (n^3 = 64, one per lane), one per wavefront, CUBE_NT/64 per
// block, each wave in its own LDS slice of wave_lds bytes.  The small cubes
// run while the large ones finish.
constexpr int CUBE_NT = 512;
template <typename T, bool NT, int NL>
__global__ void __launch_bounds__(CUBE_NT) k_source(const SrcPlan* __restrict__ src, int nbig, int nsrc,
                                                    const T* __restrict__ tpart, const T* __restrict__ PV,
                                                    typename Cplx<T>::type* __restrict__ spec, int wave_lds, int nb,
                                                    int ncol, long long cs_tpart, long long cs_spec) {
   extern __shared__ __align__(16) unsigned char smem[];
   const ColBlk cb = col_block(ncol);
   if (cb.b >= nb) return;
   tpart += cb.c * cs_tpart;
   spec += cb.c * cs_spec;
   if (cb.b < nbig) {
      const SrcPlan d = src[cb.b];
      const BlockGroup gr = block_group();
      switch (d.n) {
         case 3: source_body<3, T, NT, NL>(d, tpart, PV, spec, smem, gr); break;
         case 5: source_body<5, T, NT, NL>(d, tpart, PV, spec, smem, gr); break;
         case 6: source_body<6, T, NT, NL>(d, tpart, PV, spec, smem, gr); break;
         case 7: source_body<7, T, NT, NL>(d, tpart, PV, spec, smem, gr); break;
         case 8: source_body<8, T, NT, NL>(d, tpart, PV, spec, smem, gr); break;
         case 9: source_body<9, T, NT, NL>(d, tpart, PV, spec, smem, gr); break;
         default: break;
      }
      return;
   }
   const int wave = threadIdx.x >> 6, i = nbig + (cb.b - nbig) * (CUBE_NT / 64) + wave;
   if (i >= nsrc) return;
   const SrcPlan d = src[i];
   source4<T, NT, NL, 1>(d, tpart, 0, PV, spec, 0, 1, smem + (size_t)wave * wave_lds, threadIdx.x & 63);
}

// Source cubes of four grid points per side for SRC_NC columns per wavefront
// (LDS for two in FP64), which share each read of PV: read once per column from
// L2 it was the bound, 0.35 ms per tree for 64 columns of 30 000 panels, now 0.18.
template <typename T>
constexpr int SRC_NC = sizeof(T) == 4 ? 4 : 2;
template <typename T>
__global__ void __launch_bounds__(CUBE_NT) k_source_mc(const SrcPlan* __restrict__ src, int nsrc,
                                                       const T* __restrict__ tpart, const T* __restrict__ PV,
                                                       typename Cplx<T>::type* __restrict__ spec, int wave_lds, int nb,
                                                       int ncol, long long cs_tpart, long long cs_spec) {
   extern __shared__ __align__(16) unsigned char smem[];
   const ColBlk cb = col_block((ncol + SRC_NC<T> - 1) / SRC_NC<T>);
   const int wave = threadIdx.x >> 6, i = cb.b * (CUBE_NT / 64) + wave, c0 = cb.c * SRC_NC<T>;
   if (cb.b >= nb || i >= nsrc) return;
   const SrcPlan d = src[i];
   source4<T, false, 2, SRC_NC<T>>(d, tpart + c0 * cs_tpart, cs_tpart, PV, spec + c0 * cs_spec, cs_spec,
                                min(SRC_NC<T>, ncol - c0), smem + (size_t)wave * wave_lds, threadIdx.x & 63);
}

// FP64 translation by tiles: a block owns BC frequency bins (one TR_ROW-byte
// row per spectrum) of one tile (up to TR_TILE neighbouring target cubes of
// one level).  It stages the 343 T rows of those bins and the rows of every
// source spectrum the tile's targets interact with in LDS; LPT lanes share a
// target, each owning TR_ROW / LPT bytes of the row, and sum its interaction
// list from LDS in list order; the packed interaction word holds the two
// row byte offsets, so an address is one AND or shift away.
template <typename T, int LPT>
struct TrVec;
template <>
struct TrVec<double, 4> {
   using type = double2;  // bin l
   static constexpr int NB = 1;
};

template <typename T, int LPT>
__device__ __forceinline__ void tr_mac(const typename TrVec<T, LPT>::type& t, const typename TrVec<T, LPT>::type& v,
                                       T* re, T* im) {
   // (t * v) accumulated per bin as four FMAs
   re[0] = fma(t.x, v.x, re[0]);
   re[0] = fma(-t.y, v.y, re[0]);
   im[0] = fma(t.x, v.y, im[0]);
   im[0] = fma(t.y, v.x, im[0]);
   if constexpr (TrVec<T, LPT>::NB == 2) {
      re[1] = fma(t.z, v.z, re[1]);
      re[1] = fma(-t.w, v.w, re[1]);
      im[1] = fma(t.z, v.w, im[1]);
      im[1] = fma(t.w, v.z, im[1]);
   }
}

template <typename T, int BC, int LPT>
__global__ void __launch_bounds__(TR_TILE * LPT) k_translate(const int4* __restrict__ tasks,
                                                           const TrTile* __restrict__ tiles,
                                                           const GTgt* __restrict__ gtgt,
                                                           const int* __restrict__ gsrc, const int* __restrict__ gint,
                                                           const typename Cplx<T>::type* __restrict__ Tspec,
                                                           const typename Cplx<T>::type* __restrict__ spec,
                                                           typename Cplx<T>::type* __restrict__ acc, int nb, int ncol,
                                                           long long cs_spec, long long cs_acc) {
   using C2 = typename Cplx<T>::type;
   using V = typename TrVec<T, LPT>::type;
   constexpr int NB = TrVec<T, LPT>::NB;
   static_assert(BC * sizeof(C2) == TR_ROW && NB * sizeof(C2) * LPT == TR_ROW, "translation row layout");
   extern __shared__ __align__(16) unsigned char smem[];
   const ColBlk cb = col_block(ncol);
   if (cb.b >= nb) return;   // uniform over the block: no barrier is reached
   spec += cb.c * cs_spec;
   acc += cb.c * cs_acc;
   const int4 tk = tasks[cb.b];   // first tile, tile count, first bin
   const int b0 = tk.z, tid = threadIdx.x, nthr = TR_TILE * LPT;
   const int pad = tiles[tk.x].pad, pst = tiles[tk.x].pst;
   const long long t_off = tiles[tk.x].t_off;
   C2* Ts = (C2*)smem;        // 343 rows
   C2* Ss = Ts + 343 * BC;    // source rows
   // staging: eight loads in flight per thread before their LDS stores
   constexpr int U = 8;
   for (int i0 = tid; i0 < 343 * BC; i0 += U * nthr) {
      C2 v[U];
#pragma unroll
      for (int u = 0; u < U; u++) {
         const int i = i0 + u * nthr, c = i / BC, b = i - c * BC;
         v[u].x = 0;
         v[u].y = 0;
         if (i < 343 * BC && b0 + b < pad) v[u] = Tspec[t_off + (long long)c * pst + b0 + b];
      }
#pragma unroll
      for (int u = 0; u < U; u++)
         if (i0 + u * nthr < 343 * BC) Ts[i0 + u * nthr] = v[u];
   }
   const int j = tid / LPT, l = tid % LPT;
   const int bb = l * NB;   // lane's first bin in the row
   // lane's bytes of T row 0 and source row 0
   const unsigned char* Tl = smem + l * (TR_ROW / LPT);
   const unsigned char* Sl = Tl + 343 * TR_ROW;
   for (int ti = tk.x; ti < tk.x + tk.y; ti++) {
      const TrTile tl = tiles[ti];
      __syncthreads();   // the previous tile's sums are done with Ss
      const int ns = tl.nsrc * BC;
      for (int i0 = tid; i0 < ns; i0 += U * nthr) {
         int so[U];
#pragma unroll
         for (int u = 0; u < U; u++) {
            const int i = i0 + u * nthr;
            so[u] = i < ns ? gsrc[tl.src_off + i / BC] : 0;
         }
         C2 v[U];
#pragma unroll
         for (int u = 0; u < U; u++) {
            const int i = i0 + u * nthr, b = i - (i / BC) * BC;
            v[u].x = 0;
            v[u].y = 0;
            if (i < ns && b0 + b < pad) v[u] = spec[(long long)so[u] + b0 + b];
         }
#pragma unroll
         for (int u = 0; u < U; u++)
            if (i0 + u * nthr < ns) Ss[i0 + u * nthr] = v[u];
      }
      __syncthreads();
      if (j < tl.nt && b0 + bb < pad) {
         const GTgt tt = gtgt[tl.tgt0 + j];
         const int* it = gint + tt.int_off;
         T re0[NB] = {}, im0[NB] = {}, re1[NB] = {}, im1[NB] = {};
         int e = 0;
         // the next four interaction words load while the current four are
         // summed (a list is followed by at least four readable words)
         int4 q = *(const int4*)it;
         for (; e + 3 < tt.nint; e += 4) {
            int4 qn = *(const int4*)(it + e + 4);
            const unsigned u0 = (unsigned)q.x, u1 = (unsigned)q.y, u2 = (unsigned)q.z, u3 = (unsigned)q.w;
            const V t0 = *(const V*)(Tl + (u0 & 0xffffu)), s0 = *(const V*)(Sl + (u0 >> 16));
            const V t1 = *(const V*)(Tl + (u1 & 0xffffu)), s1 = *(const V*)(Sl + (u1 >> 16));
            const V t2 = *(const V*)(Tl + (u2 & 0xffffu)), s2 = *(const V*)(Sl + (u2 >> 16));
            const V t3 = *(const V*)(Tl + (u3 & 0xffffu)), s3 = *(const V*)(Sl + (u3 >> 16));
            tr_mac<T, LPT>(t0, s0, re0, im0);
            tr_mac<T, LPT>(t1, s1, re1, im1);
            tr_mac<T, LPT>(t2, s2, re0, im0);
            tr_mac<T, LPT>(t3, s3, re1, im1);
            // consumed here, after the sums: keeps the read-ahead load from
            // being moved to the top of the next iteration
            asm volatile("" : "+v"(qn.x), "+v"(qn.y), "+v"(qn.z), "+v"(qn.w));
            q = qn;
         }
         for (; e < tt.nint; e++) {
            const unsigned u0 = (unsigned)it[e];
            const V t0 = *(const V*)(Tl + (u0 & 0xffffu)), s0 = *(const V*)(Sl + (u0 >> 16));
            tr_mac<T, LPT>(t0, s0, re0, im0);
         }
#pragma unroll
         for (int k = 0; k < NB; k++) {
            if (b0 + bb + k < pad) {
               C2 out;
               out.x = re0[k] + re1[k];
               out.y = im0[k] + im1[k];
               acc[tt.acc_off + b0 + bb + k] = out;
            }
         }
      }
   }
}

// ---------------------------------------------------------------------------
// Pipelined FP32 translation.  See TpTile / TpOct in device.h for the layout.
// Producer waves stage task tk (tile tl, nsrc >= 1) into the LDS buffer
// buf: the tile's source rows, and the T rows of the task's level and chunk
// when stage_t.  The rows are 64 bytes (8 bins), moved in 16-byte pieces:
// producer lane pl takes pieces pl, pl + 64 TP_PW, ...  Loads are issued
// in batches before their stores (addresses clamped to valid pieces,
// stores only for real ones); the source row offsets are loaded first,
// the T rows moved last.
constexpr int TP_PL = 64 * TP_PW;                            // producer lanes
constexpr int TP_SPIECES = (TP_MAX_SRC * 4 + TP_PL - 1) / TP_PL;   // source pieces per lane
constexpr int TP_TPIECES = (343 * 4 + TP_PL - 1) / TP_PL;          // T pieces per lane
constexpr int TP_BATCH = 10;
__device__ __forceinline__ void tp_stage(const int4& tk, const TpTile& tl, bool stage_t, unsigned char* buf, int pl,
                                         const int* __restrict__ gsrc) {
   const int b0 = tk.y;
   const int npiece = tl.nsrc * 4;
   // byte offsets of the pieces in the spectrum array (below 4 GiB, checked
   // when the plan is built), so each load is one 32-bit register offset
   unsigned so[TP_SPIECES];
#pragma unroll
   for (int u = 0; u < TP_SPIECES; u++) {
      const int p = pl + TP_PL * u;
      so[u] = 8u * (unsigned)(gsrc[tl.src_off + min(p >> 2, tl.nsrc - 1)] + b0 + 2 * (p & 3));
   }
   unsigned char* sbuf = buf + TP_TROWS * 64;
#pragma unroll
   for (int u0 = 0; u0 < TP_SPIECES; u0 += TP_BATCH) {
      float4 v[TP_BATCH];
#pragma unroll
      for (int u = 0; u < TP_BATCH; u++)
         if (u0 + u < TP_SPIECES) v[u] = *(const float4*)((const char*)tl.spec + so[u0 + u]);
#pragma unroll
      for (int u = 0; u < TP_BATCH; u++) {
         const int p = pl + TP_PL * (u0 + u);
         if (u0 + u < TP_SPIECES && p < npiece) *(float4*)(sbuf + 16 * p) = v[u];
      }
      __builtin_amdgcn_sched_barrier(0);   // one batch of registers at a time
   }
   if (stage_t) {
      float4 v[TP_TPIECES];
#pragma unroll
      for (int u = 0; u < TP_TPIECES; u++) {
         const int p = min(pl + TP_PL * u, 343 * 4 - 1);
         v[u] = *(const float4*)(tl.T + (long long)(p >> 2) * tl.pst + b0 + 2 * (p & 3));
      }
#pragma unroll
      for (int u = 0; u < TP_TPIECES; u++)
         if (pl + TP_PL * u < 343 * 4) *(float4*)(buf + 16 * (pl + TP_PL * u)) = v[u];
   }
}

// The same staging by direct global->LDS transfers (16 bytes per lane, lane
// i of a transfer writes base + 16 i): no registers hold the rows.  The
// transfers are issued unconditionally, in straight-line code, so the
// compiler can keep them all in flight: source transfers cover all
// TP_MAX_SRC rows (rows past the tile's sources repeat its last one and are
// never read), T transfers 352 rows (rows past 342 repeat row 342), which
// leaves the zero row TP_ZERO_ROW untouched.
typedef __attribute__((address_space(3))) void* lds_ptr_t;
__device__ __forceinline__ void tp_dma16(const void* g, unsigned char* base) {
   __builtin_amdgcn_global_load_lds(g, (lds_ptr_t)base, 16, 0, 0);
}
__device__ __forceinline__ void tp_stage_dma(const int4& tk, const TpTile& tl, bool stage_t, unsigned char* buf,
                                             int pw, int lane, const int* __restrict__ gsrc) {
   constexpr int NS = TP_MAX_SRC * 4 / 64, NT = 352 * 4 / 64;   // transfers per buffer
   constexpr int MS = (NS + TP_PW - 1) / TP_PW, MT = (NT + TP_PW - 1) / TP_PW;
   const int b0 = tk.y, q2 = 2 * (lane & 3);
   int so[MS];
#pragma unroll
   for (int u = 0; u < MS; u++) {
      const int i = min(pw + u * TP_PW, NS - 1);
      so[u] = gsrc[tl.src_off + min(i * 16 + (lane >> 2), tl.nsrc - 1)];
   }
   unsigned char* sbuf = buf + TP_TROWS * 64;
#pragma unroll
   for (int u = 0; u < MS; u++) {
      const int i = min(pw + u * TP_PW, NS - 1);   // a repeated transfer rewrites the same rows
      tp_dma16(tl.spec + so[u] + b0 + q2, sbuf + i * 1024);
   }
   if (stage_t) {
#pragma unroll
      for (int u = 0; u < MT; u++) {
         const int i = min(pw + u * TP_PW, NT - 1);
         const int row = min(i * 16 + (lane >> 2), 342);
         tp_dma16(tl.T + (long long)row * tl.pst + b0 + q2, buf + i * 1024);
      }
   }
   __builtin_amdgcn_s_waitcnt(0);
}


// Word group i (steps 4i..4i+3) of target t of octet o; reads past the
// octet's last group are clamped to it.
__device__ __forceinline__ int4 tp_group(const int* __restrict__ gint, const TpOct& o, int i, int t) {
   const int last = max(o.nk / 4 - 1, 0);
   return *((const int4*)(gint + o.int_off) + 8 * min(i, last) + t);
}

// Two word groups (eight steps) of a lane: all sixteen LDS reads are issued
// before the first sum (a scheduling barrier keeps the compiler from
// interleaving them), then the sums, steps alternating over four
// accumulator pairs.
__device__ __forceinline__ void tp_groups2(const int4& x, const int4& y, const unsigned char* Tl,
                                           const unsigned char* Sl, float* re, float* im) {
   const unsigned u[8] = {(unsigned)x.x, (unsigned)x.y, (unsigned)x.z, (unsigned)x.w,
                          (unsigned)y.x, (unsigned)y.y, (unsigned)y.z, (unsigned)y.w};
   float2 t[8], v[8];
#pragma unroll
   for (int q = 0; q < 8; q++) {
      t[q] = *(const float2*)(Tl + (u[q] & 0xffffu));
      v[q] = *(const float2*)(Sl + (u[q] >> 16));
   }
   __builtin_amdgcn_sched_barrier(0);
#pragma unroll
   for (int q = 0; q < 8; q++) {
      float& r = re[q & 3];
      float& m = im[q & 3];
      r = fmaf(t[q].x, v[q].x, r);
      r = fmaf(-t[q].y, v[q].y, r);
      m = fmaf(t[q].x, v[q].y, m);
      m = fmaf(t[q].y, v[q].x, m);
   }
}

// Word-group pair p (steps 8p..8p+7) of target t of octet o (clamped to the
// last pair).
struct TpPair {
   int4 x, y;
};
__device__ __forceinline__ TpPair tp_pair(const int* __restrict__ gint, const TpOct& o, int p, int t) {
   return {tp_group(gint, o, 2 * p, t), tp_group(gint, o, 2 * p + 1, t)};
}

// The lane's steps of octet o (nk a multiple of 8, uniform over the wave),
// one word-group pair (eight steps, sixteen LDS reads) at a time; the
// words load two pairs ahead of their use, in three rotating register sets
// (no copies, so no wait on a load in flight).  A: pair 0, loaded; B: pair
// 1, issued by the caller.
__device__ __forceinline__ void tp_sum(const TpOct& o, int t, TpPair A, TpPair B, const int* __restrict__ gint,
                                       const unsigned char* Tl, const unsigned char* Sl, float* re, float* im) {
   const int np = o.nk / 8;
   for (int p = 0; p < np; p += 3) {
      const TpPair C = tp_pair(gint, o, p + 2, t);
      tp_groups2(A.x, A.y, Tl, Sl, re, im);
      if (p + 1 >= np) break;
      A = tp_pair(gint, o, p + 3, t);
      tp_groups2(B.x, B.y, Tl, Sl, re, im);
      if (p + 2 >= np) break;
      B = tp_pair(gint, o, p + 4, t);
      tp_groups2(C.x, C.y, Tl, Sl, re, im);
   }
}

// Producer waves: stage task 0, then task k+1 while the consumers sum task
// k; one barrier per task, as many as the consumers pass.
template <int MODE>
__device__ __forceinline__ void tp_producer(const int4* __restrict__ tasks, int n, const TpTile* __restrict__ tiles,
                                            const int* __restrict__ gsrc, unsigned char* smem, int* ctr, int pw,
                                            int lane, long long sdel) {
   long long key0, key1 = -1;   // the T rows (level and chunk) each buffer holds
   {
      const int4 t0 = tasks[0];
      TpTile tl = tiles[t0.x];
      tl.spec = (const float2*)((const char*)tl.spec + sdel);
      key0 = (long long)(tl.T + t0.y);
      if constexpr (MODE == 1)
         tp_stage_dma(t0, tl, true, smem, pw, lane, gsrc);
      else
         tp_stage(t0, tl, true, smem, 64 * pw + lane, gsrc);
   }
   __syncthreads();
   for (int k = 0; k < n; k++) {
      // task k+2's counter was task k-1's, done at the last barrier; it is
      // claimed from no earlier than the barrier that ends this iteration
      if (pw == 0 && lane == 0) ctr[(k + 2) % 3] = 0;
      if (k + 1 < n) {
         const int4 tn = tasks[k + 1];
         TpTile tl = tiles[tn.x];
         tl.spec = (const float2*)((const char*)tl.spec + sdel);
         const long long key = (long long)(tl.T + tn.y);
         const int nb = (k + 1) & 1;
         const bool st = (nb ? key1 : key0) != key;
         if (nb)
            key1 = key;
         else
            key0 = key;
         if constexpr (MODE == 1)
            tp_stage_dma(tn, tl, st, smem + nb * TP_BUF, pw, lane, gsrc);
         else
            tp_stage(tn, tl, st, smem + nb * TP_BUF, 64 * pw + lane, gsrc);
      }
      __syncthreads();
   }
}

// One claim on task k's octet counter (three counters in rotation, in LDS
// after the two buffers): the next unclaimed octet index of the task.  One
// lane of the wave adds, the wave reads its result.
__device__ __forceinline__ int tp_claim(int* ctr, int k, int lane) {
   int v = 0;
   if (lane == 0) v = atomicAdd(ctr + k % 3, 1);
   return __builtin_amdgcn_readfirstlane(v);
}

// Consumer waves claim the octets of task k one at a time, longest first
// (the plan sorts them), so the waves of a block finish a task together.
// While an octet is summed, the next is claimed and its first words load:
// the next octet of task k, or, when task k has none left, one of task k+1
// (its counter was cleared before the previous barrier).  One barrier per
// task.
__device__ __forceinline__ void tp_consumer(const int4* __restrict__ tasks, int n, const TpTile* __restrict__ tiles,
                                            const TpOct* __restrict__ octs, const long long* __restrict__ oacc,
                                            const int* __restrict__ gint, const unsigned char* smem, int* ctr,
                                            int lane, long long adel) {
   const int t = lane >> 3, b = lane & 7;
   int kc = -1, ic = 0;   // the claimed octet (task kc, index ic), none when kc < k
   TpOct o = {0, 0, 0, 0};
   TpPair A = {make_int4(0, 0, 0, 0), make_int4(0, 0, 0, 0)};
   long long ao = -1;
   __syncthreads();
   for (int k = 0; k < n; k++) {
      const int4 tk = tasks[k];
      const int pad = tiles[tk.x].pad;
      float2* __restrict__ acc = (float2*)((char*)tiles[tk.x].acc + adel);
      const unsigned char* Tl = smem + (k & 1) * TP_BUF + b * 8;
      const unsigned char* Sl = Tl + TP_TROWS * 64;
      if (kc < k) {
         ic = tp_claim(ctr, k, lane);
         if (ic < tk.w) {
            kc = k;
            o = octs[tk.z + ic];
            A = tp_pair(gint, o, 0, t);
            ao = oacc[o.acc_idx + t];
         }
      }
      while (kc == k) {
         int kn = k, jn = tp_claim(ctr, k, lane);
         if (jn >= tk.w) {
            kn = -1;
            if (k + 1 < n) {
               jn = tp_claim(ctr, k + 1, lane);
               if (jn < tasks[k + 1].w) kn = k + 1;
            }
         }
         // pair 1 of this octet, then the next octet's pair 0 (issued in
         // this order, so waiting for the former never waits for the latter)
         const TpPair B = tp_pair(gint, o, 1, t);
         TpOct on = {0, 0, 0, 0};
         TpPair An = {make_int4(0, 0, 0, 0), make_int4(0, 0, 0, 0)};
         long long aon = -1;
         if (kn >= 0) {
            on = octs[tasks[kn].z + jn];
            An = tp_pair(gint, on, 0, t);
            aon = oacc[on.acc_idx + t];
         }
         {
            float re[4] = {0.f, 0.f, 0.f, 0.f}, im[4] = {0.f, 0.f, 0.f, 0.f};
            tp_sum(o, t, A, B, gint, Tl, Sl, re, im);
            const float rs = (re[0] + re[1]) + (re[2] + re[3]), is = (im[0] + im[1]) + (im[2] + im[3]);
            if (ao >= 0 && tk.y + b < pad) acc[ao + tk.y + b] = make_float2(rs, is);
         }
         kc = kn;
         ic = jn;
         o = on;
         A = An;
         ao = aon;
      }
      __syncthreads();
   }
}

template <int MODE>
__global__ void __launch_bounds__(TP_NT) k_translate_pipe(const int2* __restrict__ ranges,
                                                          const int4* __restrict__ tasks_all,
                                                          const TpTile* __restrict__ tiles,
                                                          const TpOct* __restrict__ octs,
                                                          const long long* __restrict__ oacc,
                                                          const int* __restrict__ gsrc, const int* __restrict__ gint,
                                                          int nb, int ncol, long long sdel, long long adel,
                                                          long long scs, long long acs) {
   extern __shared__ __align__(16) unsigned char smem[];
   const ColBlk cb = col_block(ncol);
   if (cb.b >= nb) return;   // uniform over the block: no barrier is reached
   const int2 rg = ranges[cb.b];
   const int tid = threadIdx.x, lane = tid & 63;
   const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
   // the zero T row (padding words) of both buffers, which no transfer
   // writes, and the three octet counters
   int* ctr = (int*)(smem + 2 * TP_BUF);
   if (tid < 16) ((float2*)(smem + (tid >> 3) * TP_BUF + TP_ZERO_ROW * 64))[tid & 7] = make_float2(0.f, 0.f);
   if (tid < 3) ctr[tid] = 0;
   if (rg.y == 0) return;   // uniform over the block: no barrier is reached
   // both roles pass rg.y + 1 barriers
   if (wave >= TP_CW)
      tp_producer<MODE>(tasks_all + rg.x, rg.y, tiles, gsrc, smem, ctr, wave - TP_CW, lane, sdel + cb.c * scs);
   else
      tp_consumer(tasks_all + rg.x, rg.y, tiles, octs, oacc, gint, smem, ctr, lane, adel + cb.c * acs);
}

// ---------------------------------------------------------------------------
// The pipelined translation for two columns at once (column-batched
// applies): the same tiles, octets, interaction words and per-target
// summation order as k_translate_pipe, with 4-bin chunks.  A source row
// holds both columns' bins interleaved (bin j: column c0 then c1, 16
// bytes), a T row 4 bins (32 bytes); lane (target, bin j) reads its T bin
// once and both columns' source bins with one 16-byte read, so every T read
// serves two complex multiply-adds.  Each column's accumulators see the
// single-column sequence of operations, so both outputs equal
// k_translate_pipe's bit for bit.  A wave sums two octets (16 targets, 4
// lanes each); staging goes through registers (the interleave rules out
// direct transfers).
constexpr int TP2_BUF = TP_TROWS * 32 + TP_MAX_SRC * 64;
static_assert(2 * TP2_BUF + 16 <= 163840, "two pair buffers must fit the LDS of a CU");
constexpr int TP2_SPIECES = (TP_MAX_SRC * 2 + TP_PL - 1) / TP_PL;   // source half-rows per producer lane
constexpr int TP2_TPIECES = (343 * 2 + TP_PL - 1) / TP_PL;          // T half-rows per producer lane

__device__ __forceinline__ void tp_stage2(const int4& tk, const TpTile& tl, const float2* spec1, bool stage_t,
                                          unsigned char* buf, int pl, const int* __restrict__ gsrc) {
   const int b0 = tk.y;
   const int npiece = tl.nsrc * 2;
   unsigned so[TP2_SPIECES];
#pragma unroll
   for (int u = 0; u < TP2_SPIECES; u++) {
      const int p = pl + TP_PL * u;
      so[u] = 8u * (unsigned)(gsrc[tl.src_off + min(p >> 1, tl.nsrc - 1)] + b0 + 2 * (p & 1));
   }
   unsigned char* sbuf = buf + TP_TROWS * 32;
   constexpr int B = 6;
#pragma unroll
   for (int u0 = 0; u0 < TP2_SPIECES; u0 += B) {
      float4 a[B], b[B];
#pragma unroll
      for (int u = 0; u < B; u++)
         if (u0 + u < TP2_SPIECES) {
            a[u] = *(const float4*)((const char*)tl.spec + so[u0 + u]);
            b[u] = *(const float4*)((const char*)spec1 + so[u0 + u]);
         }
#pragma unroll
      for (int u = 0; u < B; u++) {
         const int p = pl + TP_PL * (u0 + u);
         if (u0 + u < TP2_SPIECES && p < npiece) {
            unsigned char* row = sbuf + 64 * (p >> 1) + 32 * (p & 1);
            *(float4*)row = make_float4(a[u].x, a[u].y, b[u].x, b[u].y);
            *(float4*)(row + 16) = make_float4(a[u].z, a[u].w, b[u].z, b[u].w);
         }
      }
      __builtin_amdgcn_sched_barrier(0);
   }
   if (stage_t) {
      float4 v[TP2_TPIECES];
#pragma unroll
      for (int u = 0; u < TP2_TPIECES; u++) {
         const int p = min(pl + TP_PL * u, 343 * 2 - 1);
         v[u] = *(const float4*)(tl.T + (long long)(p >> 1) * tl.pst + b0 + 2 * (p & 1));
      }
#pragma unroll
      for (int u = 0; u < TP2_TPIECES; u++)
         if (pl + TP_PL * u < 343 * 2) *(float4*)(buf + 16 * (pl + TP_PL * u)) = v[u];
   }
}

__device__ __forceinline__ void tp_producer2(const int4* __restrict__ tasks, int n, const TpTile* __restrict__ tiles,
                                             const int* __restrict__ gsrc, unsigned char* smem, int* ctr, int pl,
                                             long long sdel0, long long sdel1) {
   long long key0, key1 = -1;
   {
      const int4 t0 = tasks[0];
      TpTile tl = tiles[t0.x];
      const float2* s1 = (const float2*)((const char*)tl.spec + sdel1);
      tl.spec = (const float2*)((const char*)tl.spec + sdel0);
      key0 = (long long)(tl.T + t0.y);
      tp_stage2(t0, tl, s1, true, smem, pl, gsrc);
   }
   __syncthreads();
   for (int k = 0; k < n; k++) {
      if (pl == 0) ctr[(k + 2) % 3] = 0;
      if (k + 1 < n) {
         const int4 tn = tasks[k + 1];
         TpTile tl = tiles[tn.x];
         const float2* s1 = (const float2*)((const char*)tl.spec + sdel1);
         tl.spec = (const float2*)((const char*)tl.spec + sdel0);
         const long long key = (long long)(tl.T + tn.y);
         const int nb = (k + 1) & 1;
         const bool st = (nb ? key1 : key0) != key;
         if (nb)
            key1 = key;
         else
            key0 = key;
         tp_stage2(tn, tl, s1, st, smem + nb * TP2_BUF, pl, gsrc);
      }
      __syncthreads();
   }
}

// Words of group i (steps 4i..4i+3) of target t of octet o; null words past
// the octet's steps (the other octet of the wave may run longer).
__device__ __forceinline__ int4 tp_group2(const int* __restrict__ gint, const TpOct& o, int i, int t) {
   if (4 * i >= o.nk) return make_int4((int)TP_NULL_WORD, (int)TP_NULL_WORD, (int)TP_NULL_WORD, (int)TP_NULL_WORD);
   return *((const int4*)(gint + o.int_off) + 8 * i + t);
}

// Two word groups (eight steps) for both columns: all sixteen LDS reads
// issued before the first multiply-add, then the steps in list order, step
// q on accumulator q & 3, as the single-column sum.
__device__ __forceinline__ void tp_steps2(const int4& x, const int4& y, const unsigned char* Tl,
                                          const unsigned char* Sl, float* re0, float* im0, float* re1, float* im1) {
   const unsigned u[8] = {(unsigned)x.x, (unsigned)x.y, (unsigned)x.z, (unsigned)x.w,
                          (unsigned)y.x, (unsigned)y.y, (unsigned)y.z, (unsigned)y.w};
   float2 t[8];
   float4 v[8];
#pragma unroll
   for (int q = 0; q < 8; q++) {
      t[q] = *(const float2*)(Tl + ((u[q] & 0xffffu) >> 1));
      v[q] = *(const float4*)(Sl + (u[q] >> 16));
   }
   __builtin_amdgcn_sched_barrier(0);
#pragma unroll
   for (int q = 0; q < 8; q++) {
      float& r0 = re0[q & 3];
      float& m0 = im0[q & 3];
      float& r1 = re1[q & 3];
      float& m1 = im1[q & 3];
      r0 = fmaf(t[q].x, v[q].x, r0);
      r0 = fmaf(-t[q].y, v[q].y, r0);
      m0 = fmaf(t[q].x, v[q].y, m0);
      m0 = fmaf(t[q].y, v[q].x, m0);
      r1 = fmaf(t[q].x, v[q].z, r1);
      r1 = fmaf(-t[q].y, v[q].w, r1);
      m1 = fmaf(t[q].x, v[q].w, m1);
      m1 = fmaf(t[q].y, v[q].z, m1);
   }
}

__device__ __forceinline__ void tp_consumer2(const int4* __restrict__ tasks, int n, const TpTile* __restrict__ tiles,
                                             const TpOct* __restrict__ octs, const long long* __restrict__ oacc,
                                             const int* __restrict__ gint, const unsigned char* smem, int* ctr,
                                             int lane, long long adel0, long long adel1) {
   const int h = lane >> 5, t = (lane >> 2) & 7, j = lane & 3;
   __syncthreads();
   for (int k = 0; k < n; k++) {
      const int4 tk = tasks[k];
      const int pad = tiles[tk.x].pad;
      float2* acc0 = (float2*)((char*)tiles[tk.x].acc + adel0);
      float2* acc1 = (float2*)((char*)tiles[tk.x].acc + adel1);
      const unsigned char* Tl = smem + (k & 1) * TP2_BUF + j * 8;
      const unsigned char* Sl = smem + (k & 1) * TP2_BUF + TP_TROWS * 32 + j * 16;
      for (;;) {
         int ic = 0;
         if (lane == 0) ic = atomicAdd(ctr + k % 3, 2);
         ic = __builtin_amdgcn_readfirstlane(ic);
         if (ic >= tk.w) break;
         // octets ic (lanes 0-31) and ic + 1 (lanes 32-63, if any); the wave
         // runs the longer one's steps, the other half reads null words
         const TpOct oa = octs[tk.z + ic];
         const bool hb = ic + 1 < tk.w;
         const TpOct ob = hb ? octs[tk.z + ic + 1] : TpOct{0, 0, 0, 0};
         const TpOct o = h ? ob : oa;
         const int nkw = max(oa.nk, ob.nk);
         const long long ao = (h == 0 || hb) ? oacc[o.acc_idx + t] : -1;
         float re0[4] = {0.f, 0.f, 0.f, 0.f}, im0[4] = {0.f, 0.f, 0.f, 0.f};
         float re1[4] = {0.f, 0.f, 0.f, 0.f}, im1[4] = {0.f, 0.f, 0.f, 0.f};
         // word-group pairs, loaded two pairs ahead of their use in three
         // rotating register sets
         const int np = nkw / 8;
         TpPair A = {tp_group2(gint, o, 0, t), tp_group2(gint, o, 1, t)};
         TpPair B = {tp_group2(gint, o, 2, t), tp_group2(gint, o, 3, t)};
         for (int q = 0; q < np; q += 3) {
            const TpPair C = {tp_group2(gint, o, 2 * q + 4, t), tp_group2(gint, o, 2 * q + 5, t)};
            tp_steps2(A.x, A.y, Tl, Sl, re0, im0, re1, im1);
            if (q + 1 >= np) break;
            A = {tp_group2(gint, o, 2 * q + 6, t), tp_group2(gint, o, 2 * q + 7, t)};
            tp_steps2(B.x, B.y, Tl, Sl, re0, im0, re1, im1);
            if (q + 2 >= np) break;
            B = {tp_group2(gint, o, 2 * q + 8, t), tp_group2(gint, o, 2 * q + 9, t)};
            tp_steps2(C.x, C.y, Tl, Sl, re0, im0, re1, im1);
         }
         if (ao >= 0 && tk.y + j < pad) {
            acc0[ao + tk.y + j] = make_float2((re0[0] + re0[1]) + (re0[2] + re0[3]), (im0[0] + im0[1]) + (im0[2] + im0[3]));
            acc1[ao + tk.y + j] = make_float2((re1[0] + re1[1]) + (re1[2] + re1[3]), (im1[0] + im1[1]) + (im1[2] + im1[3]));
         }
      }
      __syncthreads();
   }
}

__global__ void __launch_bounds__(TP_NT) k_translate_pipe2(const int2* __restrict__ ranges,
                                                           const int4* __restrict__ tasks_all,
                                                           const TpTile* __restrict__ tiles,
                                                           const TpOct* __restrict__ octs,
                                                           const long long* __restrict__ oacc,
                                                           const int* __restrict__ gsrc, const int* __restrict__ gint,
                                                           int nb, int ncol, long long sdel, long long adel,
                                                           long long scs, long long acs) {
   extern __shared__ __align__(16) unsigned char smem[];
   const ColBlk cb = col_block_major(nb, (ncol + 1) / 2);
   if (cb.b >= nb) return;   // uniform over the block: no barrier is reached
   const int c0 = 2 * cb.c, c1 = min(c0 + 1, ncol - 1);
   const int2 rg = ranges[cb.b];
   const int tid = threadIdx.x, lane = tid & 63;
   const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
   // the zero T row of both buffers (4 bins) and the three octet counters
   int* ctr = (int*)(smem + 2 * TP2_BUF);
   if (tid < 8) ((float2*)(smem + (tid >> 2) * TP2_BUF + TP_ZERO_ROW * 32))[tid & 3] = make_float2(0.f, 0.f);
   if (tid < 3) ctr[tid] = 0;
   if (rg.y == 0) return;
   if (wave >= TP_CW)
      tp_producer2(tasks_all + rg.x, rg.y, tiles, gsrc, smem, ctr, 64 * (wave - TP_CW) + lane, sdel + c0 * scs,
                   sdel + c1 * scs);
   else
      tp_consumer2(tasks_all + rg.x, rg.y, tiles, octs, oacc, gint, smem, ctr, lane, adel + c0 * acs,
                   adel + c1 * acs);
}

void launch_translate_pipe2(int nblk, const int2* range, const int4* tasks, const TpTile* tiles, const TpOct* octs,
                            const long long* oacc, const int* gsrc, const int* gint, hipStream_t s, int ncol,
                            long long sdel, long long adel, long long scs, long long acs) {
   constexpr size_t lds = 2 * (size_t)TP2_BUF + 16;
   static std::once_flag attr;
   std::call_once(attr, [] {
      FSVD_CHECK(hipFuncSetAttribute((const void*)k_translate_pipe2, hipFuncAttributeMaxDynamicSharedMemorySize,
                                     (int)lds));
   });
   if (nblk <= 0) return;
   hipLaunchKernelGGL(k_translate_pipe2, dim3(col_grid(nblk, (ncol + 1) / 2)), dim3(TP_NT), lds, s, range, tasks,
                      tiles, octs, oacc, gsrc, gint, nblk, ncol, sdel, adel, scs, acs);
}

template <int n, typename T, typename G>
__device__ void target_body(const TgtPlan& d, const T* __restrict__ UTI,
                            const typename Cplx<T>::type* __restrict__ acc, T* __restrict__ w, unsigned char* smem,
                            const G& gr) {
   using C2 = typename Cplx<T>::type;
   constexpr int N = FarSizes<n>::N, H = FarSizes<n>::H, PAD = FarSizes<n>::PAD, GP3 = FarSizes<n>::GP3;
   C2* S = (C2*)smem;             // PAD
   C2* C1 = S + PAD;              // n*N*H
   C2* Cc = C1 + n * N * H;       // n*n*H
   T* cs = (T*)(Cc + n * n * H);  // N
   T* sn = cs + N;
   T* h = sn + N;                 // GP3
   const int tid = gr.tid, nt = gr.nt;
   twiddle_table<T, N>(cs, sn, gr);
   // four bins per thread at a time, loads before stores
   for (int b0 = tid; b0 < PAD; b0 += 4 * nt) {
      C2 v[4];
#pragma unroll
      for (int u = 0; u < 4; u++) {
         const int b = b0 + u * nt;
         v[u] = acc[d.acc_off + (b < PAD ? b : 0)];   // valid address, no branch
         keep(v[u].x);
         keep(v[u].y);
      }
#pragma unroll
      for (int u = 0; u < 4; u++) {
         const int b = b0 + u * nt;
         if (b < PAD) S[b] = v[u];
      }
   }
   gr.sync();
   grid_backward<n, T>(S, C1, Cc, h, cs, sn, gr);
   gr.sync();
   const T* uti = UTI + d.uti_off;
   // w = UTI h: 16 lanes per row, nt/16 rows per pass, four rows per lane in
   // flight (each row summed over q in order, then a fixed butterfly)
   const int kr = tid >> 4, ql = tid & 15, RP = nt >> 4;
   for (int k = kr; k < d.r; k += 4 * RP) {
      const T* row[4];
      bool ok[4];
#pragma unroll
      for (int u = 0; u < 4; u++) {
         ok[u] = k + u * RP < d.r;
         row[u] = uti + (long long)(ok[u] ? k + u * RP : k) * GP3;   // a valid row either way
      }
      T a[4] = {0, 0, 0, 0};
#pragma unroll
      for (int q0 = 0; q0 < GP3; q0 += 16) {
         // clamped column and selects: no branch around the loads
         const int q = q0 + ql < GP3 ? q0 + ql : 0;
         const bool okq = q0 + ql < GP3;
         T x[4];
#pragma unroll
         for (int u = 0; u < 4; u++) x[u] = row[u][q];
         const T hq = h[q];
#pragma unroll
         for (int u = 0; u < 4; u++) a[u] += okq && ok[u] ? x[u] * hq : (T)0;
      }
#pragma unroll
      for (int u = 0; u < 4; u++)
#pragma unroll
         for (int o = 8; o > 0; o >>= 1) a[u] += __shfl_xor(a[u], o, 64);
      if (ql == 0)
#pragma unroll
         for (int u = 0; u < 4; u++)
            if (ok[u]) w[d.w_off + k + u * RP] = a[u];
   }
}

// target_body for NC columns of a group (c0 .. c0 + nc - 1): each column's
// spectrum is transformed as target_body does (the LDS transform buffers
// reused column after column, grid values kept per column), then every UTI
// row is loaded once for all columns, each column's sums in target_body's
// order, so w equals the single-column result bit for bit.
template <int n, typename T, int NC, typename G>
__device__ void target_body_mc(const TgtPlan& d, const T* __restrict__ UTI,
                               const typename Cplx<T>::type* __restrict__ acc, long long cs_acc,
                               T* __restrict__ w, long long cs_w, int c0, int nc, unsigned char* smem, const G& gr) {
   using C2 = typename Cplx<T>::type;
   constexpr int N = FarSizes<n>::N, H = FarSizes<n>::H, PAD = FarSizes<n>::PAD, GP3 = FarSizes<n>::GP3;
   C2* S = (C2*)smem;             // PAD
   C2* C1 = S + PAD;              // n*N*H
   C2* Cc = C1 + n * N * H;       // n*n*H
   T* cs = (T*)(Cc + n * n * H);  // N
   T* sn = cs + N;
   T* h = sn + N;                 // NC x GP3
   const int tid = gr.tid, nt = gr.nt;
   twiddle_table<T, N>(cs, sn, gr);
   for (int j = 0; j < nc; j++) {
      const C2* accj = acc + (long long)(c0 + j) * cs_acc;
      for (int b0 = tid; b0 < PAD; b0 += 4 * nt) {
         C2 v[4];
#pragma unroll
         for (int u = 0; u < 4; u++) {
            const int b = b0 + u * nt;
            v[u] = accj[d.acc_off + (b < PAD ? b : 0)];
            keep(v[u].x);
            keep(v[u].y);
         }
#pragma unroll
         for (int u = 0; u < 4; u++) {
            const int b = b0 + u * nt;
            if (b < PAD) S[b] = v[u];
         }
      }
      gr.sync();
      grid_backward<n, T>(S, C1, Cc, h + j * GP3, cs, sn, gr);
      gr.sync();
   }
   const T* uti = UTI + d.uti_off;
   const int kr = tid >> 4, ql = tid & 15, RP = nt >> 4;
   for (int k = kr; k < d.r; k += 2 * RP) {
      const T* row0 = uti + (long long)k * GP3;
      const bool two = k + RP < d.r;
      const T* row1 = two ? row0 + (long long)RP * GP3 : row0;
      T a[NC], b[NC];
#pragma unroll
      for (int j = 0; j < NC; j++) a[j] = b[j] = 0;
#pragma unroll
      for (int q0 = 0; q0 < GP3; q0 += 16) {
         const int q = q0 + ql < GP3 ? q0 + ql : 0;
         const bool okq = q0 + ql < GP3;
         const T x0 = row0[q], x1 = row1[q];
#pragma unroll
         for (int j = 0; j < NC; j++) {
            const T hq = h[(j < nc ? j : 0) * GP3 + q];
            a[j] += okq ? x0 * hq : (T)0;
            b[j] += okq && two ? x1 * hq : (T)0;
         }
      }
#pragma unroll
      for (int j = 0; j < NC; j++)
#pragma unroll
         for (int o = 8; o > 0; o >>= 1) {
            a[j] += __shfl_xor(a[j], o, 64);
            b[j] += __shfl_xor(b[j], o, 64);
         }
      if (ql == 0)
         for (int j = 0; j < nc; j++) {
            T* wj = w + (long long)(c0 + j) * cs_w;
            wj[d.w_off + k] = a[j];
            if (two) wj[d.w_off + k + RP] = b[j];
         }
   }
}

// LDS of one target cube's work
template <typename T>
__host__ __device__ constexpr size_t target_cube_lds(int n) {
   return sizeof(typename Cplx<T>::type) *
              (size_t)((2 * n - 1) * (2 * n - 1) * ((2 * n - 1) / 2 + 1) + n * (2 * n - 1) * ((2 * n - 1) / 2 + 1) +
                       n * n * ((2 * n - 1) / 2 + 1)) +
          sizeof(T) * (size_t)(2 * (2 * n - 1) + n * n * n) + 64;
}

// Target cubes, one launch: the nbig cubes with other than four grid points
// per side first, one block of CUBE_NT threads each, then the cubes of four
// grid points per side, one per wavefront in its own LDS slice.
template <typename T>
__global__ void __launch_bounds__(CUBE_NT, sizeof(T) == 4 ? 6 : 2) k_target(const TgtPlan* __restrict__ tgt, int nbig, int ntgt,
                                                    const T* __restrict__ UTI,
                                                    const typename Cplx<T>::type* __restrict__ acc,
                                                    T* __restrict__ w, int wave_lds, int nb, int ncol,
                                                    long long cs_acc, long long cs_w) {
   extern __shared__ __align__(16) unsigned char smem[];
   const ColBlk cb = col_block(ncol);
   if (cb.b >= nb) return;
   acc += cb.c * cs_acc;
   w += cb.c * cs_w;
   if (cb.b < nbig) {
      const TgtPlan d = tgt[cb.b];
      const BlockGroup gr = block_group();
      switch (d.n) {
         case 3: target_body<3, T>(d, UTI, acc, w, smem, gr); break;
         case 5: target_body<5, T>(d, UTI, acc, w, smem, gr); break;
         case 6: target_body<6, T>(d, UTI, acc, w, smem, gr); break;
         case 7: target_body<7, T>(d, UTI, acc, w, smem, gr); break;
         case 8: target_body<8, T>(d, UTI, acc, w, smem, gr); break;
         case 9: target_body<9, T>(d, UTI, acc, w, smem, gr); break;
         default: break;
      }
      return;
   }
   const int wave = threadIdx.x >> 6, i = nbig + (cb.b - nbig) * (CUBE_NT / 64) + wave;
   if (i >= ntgt) return;
   const TgtPlan d = tgt[i];
   target4<T, 1>(d, UTI, acc, 0, w, 0, 1, smem + (size_t)wave * wave_lds, threadIdx.x & 63);
}

// Column batches: TGT_NC columns of a cube of four grid points per side per
// wavefront, which share each read of UTI.
constexpr int TGT_NC = 4;
template <typename T>
__global__ void __launch_bounds__(CUBE_NT, sizeof(T) == 4 ? 6 : 4)
    k_target4_mc(const TgtPlan* __restrict__ tgt, int ntgt, const T* __restrict__ UTI,
                 const typename Cplx<T>::type* __restrict__ acc, T* __restrict__ w, int wave_lds, int nb, int ncol,
                 long long cs_acc, long long cs_w) {
   extern __shared__ __align__(16) unsigned char smem[];
   const ColBlk cb = col_block((ncol + TGT_NC - 1) / TGT_NC);
   const int wave = threadIdx.x >> 6, i = cb.b * (CUBE_NT / 64) + wave, c0 = cb.c * TGT_NC;
   if (cb.b >= nb || i >= ntgt) return;
   const TgtPlan d = tgt[i];
   target4<T, TGT_NC>(d, UTI, acc + c0 * cs_acc, cs_acc, w + c0 * cs_w, cs_w, min(TGT_NC, ncol - c0),
                      smem + (size_t)wave * wave_lds, threadIdx.x & 63);
}

// The other cubes, one block each, TGT_NC columns per block (FP64), with the
// extra grid values of each column in LDS.
template <typename T>
__global__ void __launch_bounds__(CUBE_NT) k_target_mc(const TgtPlan* __restrict__ tgt, int ntgt,
                                                       const T* __restrict__ UTI,
                                                       const typename Cplx<T>::type* __restrict__ acc,
                                                       T* __restrict__ w, int ncol, long long cs_acc,
                                                       long long cs_w) {
   extern __shared__ __align__(16) unsigned char smem[];
   const ColBlk cb = col_block((ncol + TGT_NC - 1) / TGT_NC);
   if (cb.b >= ntgt) return;
   const int c0 = cb.c * TGT_NC, nc = min(TGT_NC, ncol - c0);
   const TgtPlan d = tgt[cb.b];
   const BlockGroup gr = block_group();
   switch (d.n) {
      case 3: target_body_mc<3, T, TGT_NC>(d, UTI, acc, cs_acc, w, cs_w, c0, nc, smem, gr); break;
      case 5: target_body_mc<5, T, TGT_NC>(d, UTI, acc, cs_acc, w, cs_w, c0, nc, smem, gr); break;
      case 6: target_body_mc<6, T, TGT_NC>(d, UTI, acc, cs_acc, w, cs_w, c0, nc, smem, gr); break;
      case 7: target_body_mc<7, T, TGT_NC>(d, UTI, acc, cs_acc, w, cs_w, c0, nc, smem, gr); break;
      case 8: target_body_mc<8, T, TGT_NC>(d, UTI, acc, cs_acc, w, cs_w, c0, nc, smem, gr); break;
      case 9: target_body_mc<9, T, TGT_NC>(d, UTI, acc, cs_acc, w, cs_w, c0, nc, smem, gr); break;
      default: break;
   }
}

// Leaf output: y = D_s xs + D_d xd (interleaved 2p x m block) + sum over the
// leaf's far-field blocks of U w.  Thread (g, e) owns block row e and the
// columns c = g, g+G, ...; the G partial sums of each row are added in group
// order, then the two layers and the far field.
template <typename T, bool NT>
__global__ void __launch_bounds__(256) k_leaf(const LeafDesc* __restrict__ leaves, const int* __restrict__ dcol,
                                              const T* __restrict__ D, const double* __restrict__ xs,
                                              const double* __restrict__ xd, const LeafU* __restrict__ ublk,
                                              const T* __restrict__ UT, const T* __restrict__ w,
                                              double* __restrict__ y, const int* __restrict__ bmap, int nb, int ncol,
                                              long long cs_x, long long cs_w, long long cs_y,
                                              const int* __restrict__ sp_out, const double* __restrict__ sp_corr,
                                              double* __restrict__ sp_y) {
   extern __shared__ __align__(16) unsigned char smem[];
   const ColBlk cb = col_block(ncol);
   if (cb.b >= nb) return;
   const int li = bmap[cb.b];
   if (li < 0) return;
   xs += cb.c * cs_x;
   xd += cb.c * cs_x;
   w += cb.c * cs_w;
   y += cb.c * cs_y;
   const LeafDesc L = leaves[li];
   const int E = 2 * L.p, m = L.m, p = L.p;
   T* xg = (T*)smem;       // 2*m
   T* part = xg + 2 * m;   // 256
   T* rows = part + 256;   // 2p near rows, then p far rows
   const int tid = threadIdx.x;
   for (int c = tid; c < m; c += 256) {
      int col = dcol[L.col_off + c];
      xg[c] = (T)xs[col];
      xg[m + c] = (T)xd[col];
   }
   __syncthreads();
   const T* blk = D + L.d_off;
   for (int e0 = 0; e0 < E; e0 += 256) {
      const int Ec = min(256, E - e0), G = 256 / Ec;
      const int g = tid / Ec, e = e0 + tid - g * Ec;
      T acc = 0;
      if (g < G) acc = stream_rows<T, NT>(blk + e, E, m, g, G, xg + (e >= p ? m : 0));
      part[tid] = acc;
      __syncthreads();
      if (tid < Ec) {
         T sum = 0;
         for (int gg = 0; gg < G; gg++) sum += part[gg * Ec + tid];
         rows[e0 + tid] = sum;
      }
      __syncthreads();
   }
   // far field: rows e < p of every block, the k index split over G groups
   for (int e0 = 0; e0 < p; e0 += 256) {
      const int Ec = min(256, p - e0), G = 256 / Ec;
      const int g = tid / Ec, e = e0 + tid - g * Ec;
      T acc = 0;
      if (g < G)
         for (int u = 0; u < L.nu; u++) {
            const LeafU b = ublk[L.u0 + u];
            const T* col = UT + b.u_off + e;
            const T* wb = w + b.w_off;
            // up to eight k in flight (a masked last batch)
            for (int k = g; k < b.r; k += 8 * G) {
               T cv[8], wv[8];
#pragma unroll
               for (int v = 0; v < 8; v++) {
                  const int kk = k + v * G;
                  cv[v] = kk < b.r ? col[(long long)kk * b.ld] : (T)0;
                  wv[v] = kk < b.r ? wb[kk] : (T)0;
               }
#pragma unroll
               for (int v = 0; v < 8; v++) acc += cv[v] * wv[v];
            }
         }
      part[tid] = acc;
      __syncthreads();
      if (tid < Ec) {
         T sum = 0;
         for (int gg = 0; gg < G; gg++) sum += part[gg * Ec + tid];
         rows[E + e0 + tid] = sum;
      }
      __syncthreads();
   }
   // with sp_y: the region split fused in (k_split's y[out] = yt + corr xd)
   for (int r = tid; r < p; r += 256) {
      const double v = (double)((rows[r] + rows[p + r]) + rows[E + r]);
      if (sp_y)
         sp_y[sp_out[L.q0 + r]] = v + sp_corr[L.q0 + r] * xd[L.q0 + r];
      else
         y[L.q0 + r] = v;
   }
}

// columns per block of the multi-column leaf kernel
constexpr int LEAF_NC = 4;

// stream_rows for NC columns at once: every entry of the block is loaded
// once and multiplied into each column's accumulators; xl holds the
// columns' inputs interleaved (input i of column j at xl[i * NC + j]).  Each
// column's accumulators see the single-column sequence of operations, so
// out[j] is stream_rows's result for column j bit for bit.
template <typename T, int NC>
__device__ __forceinline__ void stream_rows_mc(const T* __restrict__ colp, int E, int m, int g, int G,
                                               const T* xl, T* out) {
   const long long step = (long long)G * E;
   T a[4][NC];
#pragma unroll
   for (int q = 0; q < 4; q++)
#pragma unroll
      for (int j = 0; j < NC; j++) a[q][j] = 0;
   int c = g;
   for (; c + 7 * G < m; c += 8 * G) {
      const T* pc = colp + (long long)c * E;
      T d[8];
#pragma unroll
      for (int u = 0; u < 8; u++) d[u] = pc[u * step];
#pragma unroll
      for (int u = 0; u < 8; u++) {
         const T* xv = xl + (size_t)(c + u * G) * NC;
#pragma unroll
         for (int j = 0; j < NC; j++) a[u & 3][j] += d[u] * xv[j];
      }
   }
   if (c < m) {
      const T* pc = colp + (long long)c * E;
      T d[7];
#pragma unroll
      for (int u = 0; u < 7; u++) d[u] = c + u * G < m ? pc[u * step] : (T)0;
#pragma unroll
      for (int u = 0; u < 7; u++)
         if (c + u * G < m) {
            const T* xv = xl + (size_t)(c + u * G) * NC;
#pragma unroll
            for (int j = 0; j < NC; j++) a[0][j] += d[u] * xv[j];
         }
   }
#pragma unroll
   for (int j = 0; j < NC; j++) out[j] = (a[0][j] + a[1][j]) + (a[2][j] + a[3][j]);
}

// k_leaf for NC columns per block: the near-field block and the U rows are
// read once for the NC columns of the block's group (columns c0 .. c0+NC-1
// of ncol; a partial last group repeats its last column and stores only its
// own).  Per column the arithmetic is k_leaf's, so y equals the
// single-column result bit for bit.  Grid: col_grid(nb, number of groups).
template <typename T, int NC>
__global__ void __launch_bounds__(256) k_leaf_mc(const LeafDesc* __restrict__ leaves, const int* __restrict__ dcol,
                                                 const T* __restrict__ D, const double* __restrict__ xs,
                                                 const double* __restrict__ xd, const LeafU* __restrict__ ublk,
                                                 const T* __restrict__ UT, const T* __restrict__ w,
                                                 double* __restrict__ y, const int* __restrict__ bmap, int nb,
                                                 int ncol, long long cs_x, long long cs_w, long long cs_y) {
   extern __shared__ __align__(16) unsigned char smem[];
   const int ngrp = (ncol + NC - 1) / NC;
   const ColBlk cb = col_block(ngrp);
   if (cb.b >= nb) return;
   const int li = bmap[cb.b];
   if (li < 0) return;
   const int c0 = cb.c * NC, nc = min(NC, ncol - c0);
   const LeafDesc L = leaves[li];
   const int E = 2 * L.p, m = L.m, p = L.p;
   T* xg = (T*)smem;                 // 2m x NC
   T* part = xg + 2 * m * NC;        // NC x 256
   T* rows = part + 256 * NC;        // NC x (2p near rows, then p far rows)
   const int tid = threadIdx.x, R3 = 3 * p;
   for (int c = tid; c < m; c += 256) {
      const int col = dcol[L.col_off + c];
#pragma unroll
      for (int j = 0; j < NC; j++) {
         const long long o = (long long)(c0 + min(j, nc - 1)) * cs_x + col;
         xg[(size_t)c * NC + j] = (T)xs[o];
         xg[(size_t)(m + c) * NC + j] = (T)xd[o];
      }
   }
   __syncthreads();
   const T* blk = D + L.d_off;
   for (int e0 = 0; e0 < E; e0 += 256) {
      const int Ec = min(256, E - e0), G = 256 / Ec;
      const int g = tid / Ec, e = e0 + tid - g * Ec;
      T acc[NC];
#pragma unroll
      for (int j = 0; j < NC; j++) acc[j] = 0;
      if (g < G) stream_rows_mc<T, NC>(blk + e, E, m, g, G, xg + (e >= p ? (size_t)m * NC : 0), acc);
#pragma unroll
      for (int j = 0; j < NC; j++) part[j * 256 + tid] = acc[j];
      __syncthreads();
      if (tid < Ec) {
#pragma unroll
         for (int j = 0; j < NC; j++) {
            T sum = 0;
            for (int gg = 0; gg < G; gg++) sum += part[j * 256 + gg * Ec + tid];
            rows[j * R3 + e0 + tid] = sum;
         }
      }
      __syncthreads();
   }
   for (int e0 = 0; e0 < p; e0 += 256) {
      const int Ec = min(256, p - e0), G = 256 / Ec;
      const int g = tid / Ec, e = e0 + tid - g * Ec;
      T acc[NC];
#pragma unroll
      for (int j = 0; j < NC; j++) acc[j] = 0;
      if (g < G)
         for (int u = 0; u < L.nu; u++) {
            const LeafU b = ublk[L.u0 + u];
            const T* col = UT + b.u_off + e;
            for (int k = g; k < b.r; k += 8 * G) {
               T cv[8];
#pragma unroll
               for (int v = 0; v < 8; v++) {
                  const int kk = k + v * G;
                  cv[v] = kk < b.r ? col[(long long)kk * b.ld] : (T)0;
               }
#pragma unroll
               for (int j = 0; j < NC; j++) {
                  const T* wb = w + (long long)(c0 + min(j, nc - 1)) * cs_w + b.w_off;
                  T wv[8];
#pragma unroll
                  for (int v = 0; v < 8; v++) {
                     const int kk = k + v * G;
                     wv[v] = kk < b.r ? wb[kk] : (T)0;
                  }
#pragma unroll
                  for (int v = 0; v < 8; v++) acc[j] += cv[v] * wv[v];
               }
            }
         }
#pragma unroll
      for (int j = 0; j < NC; j++) part[j * 256 + tid] = acc[j];
      __syncthreads();
      if (tid < Ec) {
#pragma unroll
         for (int j = 0; j < NC; j++) {
            T sum = 0;
            for (int gg = 0; gg < G; gg++) sum += part[j * 256 + gg * Ec + tid];
            rows[j * R3 + E + e0 + tid] = sum;
         }
      }
      __syncthreads();
   }
   for (int j = 0; j < nc; j++) {
      const T* rj = rows + j * R3;
      double* yj = y + (long long)(c0 + j) * cs_y;
      for (int r = tid; r < p; r += 256) yj[L.q0 + r] = (double)((rj[r] + rj[p + r]) + rj[E + r]);
   }
}

// ---------------------------------------------------------------------------
// Output of the transposed apply (reference Tree_multiply_transpose,
// Tree.c:769-832), one block per leaf (up to LT_SLAB of its panels): for its panels i
//   ys[i] = sum of the single-layer column i of every near-field block that
//           holds it, times x, plus sum_k VT[k, i] ws[k] over the leaf's source
//           cubes; yd likewise for the double layer.
// Gathered per leaf, so each near-field entry is read once and no output is
// shared between blocks (one scatter per block with FP64 atomics took 87 us a
// tree at 31 000 panels, beside ~60 per-level launches for the far field).
// Bound by latency: short gathers (32 rows per neighbour block, 20-60 columns),
// 39 us a launch at 31 000 panels with 7 waves per SIMD.  It moves 279 MB (FP32)
// and 548 MB (FP64) a tree at 100 000 panels, the forward k_leaf 254 and 501.
// Transposed product of both trees, host to host: 31 000 panels 1.22 to 0.27 ms
// FP32, 1.49 to 0.38 FP64; 100 000 panels 2.38 to 0.63 and 2.89 to 1.00.  Near
// field: the rows of all blocks are listed in LDS (TILE at a time: entry offset,
// column stride, x), lanes take rows, waves four columns each with both layers
// of a column in flight; FP64 sums.  Far field: 16 lanes per panel over the rows
// of its panel-major basis, summed in T per source cube and in FP64 over the
// cubes.
constexpr int LT_TILE = 512;
template <typename T>
__global__ void __launch_bounds__(256, sizeof(T) == 4 ? 7 : 5) k_leaf_t(const LeafT* __restrict__ leaves, const NearT* __restrict__ nbr,
                                                const T* __restrict__ D, const double* __restrict__ x,
                                                const LeafU* __restrict__ ublk, const T* __restrict__ VTc,
                                                const T* __restrict__ w, double* __restrict__ ys,
                                                double* __restrict__ yd) {
   extern __shared__ __align__(16) unsigned char smem[];
   __shared__ double xr[LT_TILE];
   __shared__ long long base[LT_TILE];
   __shared__ int st[LT_TILE];
   constexpr int CW = 4, RU = 2;
   const LeafT L = leaves[blockIdx.x];   // in launch order; np = 0: idle
   if (L.np == 0) return;
   double* res = (double*)smem;   // near field: np single-layer, then np double-layer sums
   const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, grp = tid >> 4, gl = tid & 15;
   for (int cb = 0; cb < L.np; cb += 4 * CW) {
      const int c0 = cb + CW * wave;
      double as[CW], ad[CW];
#pragma unroll
      for (int c = 0; c < CW; c++) as[c] = ad[c] = 0.0;
      for (int t0 = 0; t0 < L.rows; t0 += LT_TILE) {
         const int tn = min(LT_TILE, L.rows - t0);
         // one tile holds the rows of most leaves: listed once
         if (cb == 0 || L.rows > LT_TILE) {
            __syncthreads();
            for (int j = grp; j < L.nn; j += 16) {
               const NearT e = nbr[L.nb0 + j];
               for (int r = gl; r < e.p; r += 16) {
                  const int i = e.row0 + r - t0;
                  if (i >= 0 && i < tn) {
                     xr[i] = x[e.q0 + r];
                     base[i] = e.d_off + r;
                     st[i] = 2 * e.p;
                  }
               }
            }
            __syncthreads();
         }
         if (c0 < L.np)
            for (int i0 = lane; i0 < tn; i0 += 64 * RU) {
               // RU rows per lane in flight; a row past the last repeats it
               // with x = 0, a column past the last repeats it (sum unused)
               T vs[RU][CW], vd[RU][CW];
               double xi[RU];
#pragma unroll
               for (int q = 0; q < RU; q++) {
                  const int i = min(i0 + 64 * q, tn - 1);
                  xi[q] = i0 + 64 * q < tn ? xr[i] : 0.0;
                  const int sc = st[i];
                  const T* p = D + base[i];
#pragma unroll
                  for (int c = 0; c < CW; c++) {
                     const T* pc = p + (long long)min(c0 + c, L.np - 1) * sc;
                     if (ys) vs[q][c] = pc[0];
                     if (yd) vd[q][c] = pc[sc >> 1];
                  }
               }
#pragma unroll
               for (int q = 0; q < RU; q++)
#pragma unroll
                  for (int c = 0; c < CW; c++) {
                     if (ys) as[c] = fma((double)vs[q][c], xi[q], as[c]);
                     if (yd) ad[c] = fma((double)vd[q][c], xi[q], ad[c]);
                  }
            }
      }
#pragma unroll
      for (int c = 0; c < CW; c++) {
         if (c0 + c < L.np) {   // uniform over the wave
            const double s = ys ? wave_sum(as[c]) : 0.0, d = yd ? wave_sum(ad[c]) : 0.0;
            if (lane == 0) {
               res[c0 + c] = s;
               res[L.np + c0 + c] = d;
            }
         }
      }
   }
   __syncthreads();
   for (int i0 = 0; i0 < L.np; i0 += 16) {
      const int i = i0 + grp, ic = min(i, L.np - 1);
      double as = 0.0, ad = 0.0;
      // four source cubes at a time, their loads in flight together
      for (int u0 = 0; u0 < L.nu; u0 += 4) {
         LeafU b[4];
#pragma unroll
         for (int u = 0; u < 4; u++) b[u] = ublk[L.u0 + min(u0 + u, L.nu - 1)];
         T a[4] = {0, 0, 0, 0}, d[4] = {0, 0, 0, 0};
         int rmax = 0;
#pragma unroll
         for (int u = 0; u < 4; u++) {
            if (u0 + u >= L.nu) b[u].r = 0;
            rmax = max(rmax, b[u].r);
         }
         for (int k0 = gl; k0 < rmax; k0 += 32) {
            T vv[4][2], sv[4][2], dv[4][2];
#pragma unroll
            for (int u = 0; u < 4; u++)
#pragma unroll
               for (int q = 0; q < 2; q++) {
                  // clamped index, selected sums: no branch around the loads
                  const int k = k0 + 16 * q < b[u].r ? k0 + 16 * q : 0;
                  vv[u][q] = VTc[b[u].u_off + (long long)ic * b[u].ld + k];
                  if (ys) sv[u][q] = w[b[u].w_off + k];
                  if (yd) dv[u][q] = w[b[u].w_off + b[u].ld + k];
               }
#pragma unroll
            for (int u = 0; u < 4; u++)
#pragma unroll
               for (int q = 0; q < 2; q++) {
                  const T m = k0 + 16 * q < b[u].r ? vv[u][q] : (T)0;
                  if (ys) a[u] += m * sv[u][q];
                  if (yd) d[u] += m * dv[u][q];
               }
         }
#pragma unroll
         for (int u = 0; u < 4; u++) {
            as += (double)a[u];
            ad += (double)d[u];
         }
      }
#pragma unroll
      for (int o = 8; o > 0; o >>= 1) {
         as += __shfl_xor(as, o, 64);
         ad += __shfl_xor(ad, o, 64);
      }
      if (gl == 0 && i < L.np) {
         if (ys) ys[L.p0 + i] = res[i] + as;
         if (yd) yd[L.p0 + i] = res[L.np + i] + ad;
      }
   }
}

// ---------------------------------------------------------------------------
// Explicit instantiations and launchers
// gfx950: 160 KiB of LDS per workgroup
static void check_lds(size_t lds) {
   if (lds > 163840) throw std::runtime_error("LDS request above 160 KiB per workgroup");
}

void launch_translate_pipe(int nblk, int mode, const int2* range, const int4* tasks, const TpTile* tiles,
                           const TpOct* octs, const long long* oacc, const int* gsrc, const int* gint, hipStream_t s,
                           int ncol, long long sdel, long long adel, long long scs, long long acs) {
   // two LDS buffers per persistent block, three counters
   constexpr size_t lds = 2 * (size_t)TP_BUF + 16;
   check_lds(lds);
   static std::once_flag attr;
   std::call_once(attr, [] {
      FSVD_CHECK(hipFuncSetAttribute((const void*)k_translate_pipe<0>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                     (int)lds));
      FSVD_CHECK(hipFuncSetAttribute((const void*)k_translate_pipe<1>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                     (int)lds));
   });
   if (nblk <= 0) return;
   const int g = col_grid(nblk, ncol);
   if (mode == 1)
      hipLaunchKernelGGL(k_translate_pipe<1>, dim3(g), dim3(TP_NT), lds, s, range, tasks, tiles, octs, oacc, gsrc,
                         gint, nblk, ncol, sdel, adel, scs, acs);
   else
      hipLaunchKernelGGL(k_translate_pipe<0>, dim3(g), dim3(TP_NT), lds, s, range, tasks, tiles, octs, oacc, gsrc,
                         gint, nblk, ncol, sdel, adel, scs, acs);
}

template <typename T>
void launch_apply_stage(int stage, const ApplyArgs& a, hipStream_t s) {
   using C2 = typename Cplx<T>::type;
   if (a.max_n > 9) throw std::runtime_error("grid points per side above 9");
   switch (stage) {
      case 0: {
         const int wl = (int)((sizeof(T) * (size_t)(2 * a.proj_maxcols + 128) + 15) / 16 * 16);
         check_lds(4 * (size_t)wl);
         if (a.nchunk && a.ncol == 1) {
            auto kern = a.layers == 1 ? k_project<T, true, 1> : k_project<T, true, 2>;
            hipLaunchKernelGGL(kern, dim3((a.nchunk + 3) / 4), dim3(256), 4 * (size_t)wl, s, a.chunks, a.nchunk,
                               (const T*)a.VTc, a.xs, a.xd, (T*)a.tpart, wl, 1, a.cs_x, a.cs_tpart);
         } else if (a.nchunk) {
            constexpr int NC = proj_nc<T>();
            const int wlm = (int)((sizeof(T) * (size_t)NC * (2 * a.proj_maxcols + 128) + 15) / 16 * 16);
            check_lds(4 * (size_t)wlm);
            static std::once_flag attr;
            std::call_once(attr, [] {
               FSVD_CHECK(hipFuncSetAttribute((const void*)k_project_mc<T, NC>,
                                              hipFuncAttributeMaxDynamicSharedMemorySize, 163840));
            });
            const int ngrp = (a.ncol + NC - 1) / NC;
            hipLaunchKernelGGL((k_project_mc<T, NC>), dim3(col_grid((a.nchunk + 3) / 4, ngrp)), dim3(256),
                               4 * (size_t)wlm, s, a.chunks, a.nchunk, (const T*)a.VTc, a.xs, a.xd, (T*)a.tpart,
                               wlm, a.ncol, a.cs_x, a.cs_tpart);
         }
         break;
      }
      case 1: {
         const int wl = (int)source4_lds<T>(a.maxr_src, 1);
         size_t lds = (size_t)(CUBE_NT / 64) * wl;
         for (int n = 3; n <= a.max_n; n++)
            if (n != 4) lds = std::max(lds, source_cube_lds<T>(n, a.maxr_src, CUBE_NT));
         check_lds(lds);
         static std::once_flag attr;   // large n needs more than the default dynamic LDS
         std::call_once(attr, [] {
            FSVD_CHECK(hipFuncSetAttribute((const void*)k_source<T, true, 2>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, 163840));
            FSVD_CHECK(hipFuncSetAttribute((const void*)k_source<T, false, 2>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, 163840));
            FSVD_CHECK(hipFuncSetAttribute((const void*)k_source<T, true, 1>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, 163840));
            FSVD_CHECK(hipFuncSetAttribute((const void*)k_source_mc<T>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                           163840));
         });
         // batches: the wavefronts' cubes by groups of columns, unless their
         // ranks are too large for the groups' LDS
         const size_t wlm = source4_lds<T>(a.maxr_src, SRC_NC<T>);
         const bool mc = a.ncol > 1 && (CUBE_NT / 64) * wlm <= 163840;
         const int nsrc = mc ? a.nsrc_big : a.nsrc;
         const int nb = a.nsrc_big + (nsrc - a.nsrc_big + CUBE_NT / 64 - 1) / (CUBE_NT / 64);
         if (nb) {
            auto kern = a.layers == 1 ? k_source<T, true, 1> : (a.ncol == 1 ? k_source<T, true, 2> : k_source<T, false, 2>);
            hipLaunchKernelGGL(kern, dim3(col_grid(nb, a.ncol)), dim3(CUBE_NT), lds, s, a.src, a.nsrc_big, nsrc,
                               (const T*)a.tpart, (const T*)a.PV, (C2*)a.spec, wl, nb, a.ncol, a.cs_tpart,
                               a.cs_spec);
         }
         if (mc && a.nsrc > a.nsrc_big) {
            const int n4 = a.nsrc - a.nsrc_big, nb4 = (n4 + CUBE_NT / 64 - 1) / (CUBE_NT / 64);
            hipLaunchKernelGGL((k_source_mc<T>), dim3(col_grid(nb4, (a.ncol + SRC_NC<T> - 1) / SRC_NC<T>)), dim3(CUBE_NT),
                               (CUBE_NT / 64) * wlm, s, a.src + a.nsrc_big, n4, (const T*)a.tpart, (const T*)a.PV,
                               (C2*)a.spec, (int)wlm, nb4, a.ncol, a.cs_tpart, a.cs_spec);
         }
         break;
      }
      case 2: {
         if constexpr (std::is_same<T, float>::value) {
            if (a.ncol >= 2 && a.nblk_p2 > 0)
               launch_translate_pipe2(a.nblk_p2, a.range_p2, a.task_p2, a.tiles_p2, a.oct_p2, a.oacc_p2, a.gsrc_p2,
                                      a.gint_p2, s, a.ncol, a.spec_delta, a.acc_delta,
                                      a.cs_spec * (long long)sizeof(C2), a.cs_acc * (long long)sizeof(C2));
            else
               launch_translate_pipe(a.nblk_p, a.mode_p, a.range_p, a.task_p, a.tiles_p, a.oct_p, a.oacc_p,
                                     a.gsrc_p, a.gint_p, s, a.ncol, a.spec_delta, a.acc_delta,
                                     a.cs_spec * (long long)sizeof(C2), a.cs_acc * (long long)sizeof(C2));
         } else {
            // LDS: T spectra and at most TR_MAX_SRC source spectra of BC bins
            constexpr int BC = TR_BINS_F64, LPT = TR_LPT_F64;
            const size_t lds_max = sizeof(C2) * (size_t)(343 + TR_MAX_SRC) * BC;
            const size_t lds = sizeof(C2) * (size_t)(343 + a.tr_max_src) * BC;
            check_lds(lds_max);
            if (a.tr_max_src > TR_MAX_SRC) throw std::runtime_error("translation tile above its LDS bound");
            static std::once_flag attr;
            std::call_once(attr, [lds_max] {
               FSVD_CHECK(hipFuncSetAttribute((const void*)k_translate<T, BC, LPT>,
                                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_max));
            });
            if (a.ntask_d)
               hipLaunchKernelGGL((k_translate<T, BC, LPT>), dim3(col_grid(a.ntask_d, a.ncol)), dim3(TR_TILE * LPT),
                                  lds, s, a.task_d, a.tiles, a.gtgt, a.gsrc, a.gint, (const C2*)a.Tsp,
                                  (const C2*)a.spec, (C2*)a.acc, a.ntask_d, a.ncol, a.cs_spec, a.cs_acc);
         }
         break;
      }
      case 3: {
         const int wl = (int)target4_lds<T>(1), wlm = (int)target4_lds<T>(TGT_NC);
         size_t lds = (size_t)(CUBE_NT / 64) * wl, lmc = 0;
         for (int n = 3; n <= a.max_n; n++)
            if (n != 4) {
               lds = std::max(lds, target_cube_lds<T>(n));
               lmc = std::max(lmc, target_cube_lds<T>(n) + sizeof(T) * (size_t)(TGT_NC - 1) * n * n * n);
            }
         check_lds(lds);
         static std::once_flag attr;   // large n needs more than the default dynamic LDS
         std::call_once(attr, [] {
            FSVD_CHECK(hipFuncSetAttribute((const void*)k_target<T>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                           163840));
            FSVD_CHECK(hipFuncSetAttribute((const void*)k_target4_mc<T>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                           163840));
            if (sizeof(T) == 8)
               FSVD_CHECK(hipFuncSetAttribute((const void*)k_target_mc<double>,
                                              hipFuncAttributeMaxDynamicSharedMemorySize, 163840));
         });
         // Batches: the wavefronts' cubes by groups of TGT_NC columns.  The
         // large cubes, with one block each: in groups for FP64 (0.052 against
         // 0.063 ms per column on the 100k-panel globule), a block per column
         // for FP32 (0.033 against 0.042).
         const bool mc = a.ncol > 1, bigmc = mc && sizeof(T) == 8;
         const int ngrp = (a.ncol + TGT_NC - 1) / TGT_NC, n4 = a.ntgt - a.ntgt_big;
         if constexpr (sizeof(T) == 8) {
            if (bigmc && a.ntgt_big) {
               check_lds(lmc);
               hipLaunchKernelGGL((k_target_mc<T>), dim3(col_grid(a.ntgt_big, ngrp)), dim3(CUBE_NT), lmc, s, a.tgt,
                                  a.ntgt_big, (const T*)a.UTI, (const C2*)a.acc, (T*)a.w, a.ncol, a.cs_acc, a.cs_w);
            }
         }
         const int nt = mc ? (bigmc ? 0 : a.ntgt_big) : a.ntgt;
         const int nb = nt ? a.ntgt_big + (nt - a.ntgt_big + CUBE_NT / 64 - 1) / (CUBE_NT / 64) : 0;
         if (nb)
            hipLaunchKernelGGL((k_target<T>), dim3(col_grid(nb, a.ncol)), dim3(CUBE_NT), lds, s, a.tgt, a.ntgt_big,
                               nt, (const T*)a.UTI, (const C2*)a.acc, (T*)a.w, wl, nb, a.ncol, a.cs_acc, a.cs_w);
         if (mc && n4 > 0) {
            const int nb4 = (n4 + CUBE_NT / 64 - 1) / (CUBE_NT / 64);
            hipLaunchKernelGGL((k_target4_mc<T>), dim3(col_grid(nb4, ngrp)), dim3(CUBE_NT), (CUBE_NT / 64) * wlm, s,
                               a.tgt + a.ntgt_big, n4, (const T*)a.UTI, (const C2*)a.acc, (T*)a.w, wlm, nb4, a.ncol,
                               a.cs_acc, a.cs_w);
         }
         break;
      }
      case 4: {
         size_t lds = sizeof(T) * (size_t)(2 * a.maxm + 256 + 3 * a.maxp) + 64;
         check_lds(lds);
         if (a.nleaf && a.ncol == 1) {
            hipLaunchKernelGGL((k_leaf<T, true>), dim3(a.nmap_leaf), dim3(256), lds, s, a.leaves, a.dcol,
                               (const T*)a.D, a.xs, a.xd, a.ublk, (const T*)a.UT, (const T*)a.w, a.y, a.map_leaf,
                               a.nmap_leaf, 1, a.cs_x, a.cs_w, a.cs_y, a.sp_out, a.sp_corr, a.sp_y);
         } else if (a.nleaf && sizeof(T) * (size_t)LEAF_NC * (2 * a.maxm + 256 + 3 * a.maxp) + 64 > 163840) {
            // leaves too wide for LEAF_NC columns in LDS: one block copy per column
            hipLaunchKernelGGL((k_leaf<T, false>), dim3(col_grid(a.nmap_leaf, a.ncol)), dim3(256), lds, s, a.leaves,
                               a.dcol, (const T*)a.D, a.xs, a.xd, a.ublk, (const T*)a.UT, (const T*)a.w, a.y,
                               a.map_leaf, a.nmap_leaf, a.ncol, a.cs_x, a.cs_w, a.cs_y, nullptr, nullptr, nullptr);
         } else if (a.nleaf) {
            // LEAF_NC columns per block
            const size_t lmc = sizeof(T) * (size_t)LEAF_NC * (2 * a.maxm + 256 + 3 * a.maxp) + 64;
            check_lds(lmc);
            static std::once_flag attr;
            std::call_once(attr, [] {
               FSVD_CHECK(hipFuncSetAttribute((const void*)k_leaf_mc<T, LEAF_NC>,
                                              hipFuncAttributeMaxDynamicSharedMemorySize, 163840));
            });
            const int ngrp = (a.ncol + LEAF_NC - 1) / LEAF_NC;
            hipLaunchKernelGGL((k_leaf_mc<T, LEAF_NC>), dim3(col_grid(a.nmap_leaf, ngrp)), dim3(256), lmc, s,
                               a.leaves, a.dcol, (const T*)a.D, a.xs, a.xd, a.ublk, (const T*)a.UT, (const T*)a.w,
                               a.y, a.map_leaf, a.nmap_leaf, a.ncol, a.cs_x, a.cs_w, a.cs_y);
         }
         break;
      }
      case 5: {
         const size_t lds = sizeof(double) * 2 * (size_t)std::max(a.maxnpT, 1);   // at most 16 LT_SLAB bytes
         if (a.nleafT)
            hipLaunchKernelGGL((k_leaf_t<T>), dim3(a.nleafT), dim3(256), lds, s, a.leavesT, a.nbrT, (const T*)a.D,
                               a.xs, a.ublk, (const T*)a.VTc, (const T*)a.w, a.y, a.y2);
         break;
      }
      default: break;
   }
}

template <typename T>
__global__ void k_transpose_batched(const TransDesc* __restrict__ d) {
   const TransDesc t = d[blockIdx.x];
   const T* src = (const T*)t.src;
   T* dst = (T*)t.dst;
   const int total = t.rows * t.cols;
   for (int e = threadIdx.x; e < total; e += blockDim.x) {
      int j = e / t.rows, i = e - j * t.rows;
      dst[e] = src[(long long)i * t.cols + j];
   }
}

template <typename T>
void launch_transpose_batched(int n, const TransDesc* d, hipStream_t s) {
   for (int b0 = 0; b0 < n; b0 += 65535)
      hipLaunchKernelGGL((k_transpose_batched<T>), dim3(std::min(65535, n - b0)), dim3(256), 0, s, d + b0);
}

#define FSVD_INST(T)                                                  \
   template void launch_apply_stage<T>(int, const ApplyArgs&, hipStream_t); \
   template void launch_transpose_batched<T>(int, const TransDesc*, hipStream_t);
FSVD_INST(float)
FSVD_INST(double)

}  // namespace fsvd
