// sbp_rows.h -- the six SBP boundary rows of h^2 L(u) next to a free surface
// (k = 1..6 at the top, nk..nk-5 at the bottom; rhs4sg_rev.C:349-863), for the
// FP64 and FP32 kernels that read the field their own way (Load) and use the
// rows their own way (Epi).
//
// Row space: plane q = 0..8 is grid plane kbase + sgn (q - 1); row kr lives on
// q = kr.  Grouped by the outer derivative a row is
//   r = pp + qq + D_x F + D_y G + sum_q bope(kr,q) T(q) + (SBP second
//       k-difference and its ghost term),
// with F, G, T the products of material and first derivatives at one point:
// each is formed once and its neighbours read it, as in the curvilinear march.
// A workgroup owns a 32 x 8 tile; each point of the tile with its halo has a
// thread (four waves of outputs, two of the j halo, one of the i halo and the
// corners) that loads its column of nine planes.  The planes go to LDS once;
// T of the eight planes stays in registers for all rows; per row the columns
// form F and G, one barrier, and the outputs are finished.  block.y takes the
// rows 1 + block.y, the next gridDim.y on (more workgroups on small grids).
// Bound by latency (2 waves/SIMD: the planes fill a CU's LDS in FP64).
// Predictor and corrector rows of the step, against rows evaluated one after
// the other by one wave per SIMD with all neighbours' derivatives formed
// again: 62 + 60 -> 9 + 9 us at 40 x 36 points, 157 + 181 -> 55 + 55 at
// 301 x 301; FP32 there 67 + 82 -> 25 + 58, the damping (10, a pass of its own)
// included.
#pragma once
#include "kernels_common.h"
#include "kernels_fast.h"

namespace sw4amd {

constexpr int RTX = 32, RTY = 8, RHX = RTX + 4, RHY = RTY + 4, RPL = RHX * RHY, RNT = 448;

// A thread's point of the tile with its halo, and its part: 0 output, 1 j
// halo, 2 i halo and corners (whole waves; the last 16 threads repeat a point).
__device__ __forceinline__ void rows_point(int tid, int& role, int& hx, int& hy)
{
   role = __builtin_amdgcn_readfirstlane(tid < 256 ? 0 : tid < 384 ? 1 : 2);
   if (tid < 256) {
      hx = 2 + tid % RTX;
      hy = 2 + tid / RTX;
   } else if (tid < 384) {
      const int r = (tid - 256) / RTX;
      hx = 2 + tid % RTX;
      hy = r < 2 ? r : r + RTY;
   } else {
      const int q = tid - 384, c = q % 4, r = q / 4;  // rows 0..7: the tile's, 8..11: the corners'
      hx = c < 2 ? c : c + RTX;
      hy = r < RTY ? 2 + r : r < RTY + 2 ? r - RTY : r < RTY + 4 ? r : 2;
   }
}

template <class R, class Load, class Epi>
__device__ __forceinline__ void sbp_rows_body(const Box& b, int top, int nk, int ntx,
                                              const SbpTablesT<R>* __restrict__ sbp, const R* __restrict__ mu,
                                              const R* __restrict__ la, const R* __restrict__ strx,
                                              const R* __restrict__ stry, Load ld, Epi epi)
{
   __shared__ R su[8 * 3 * RPL];             // planes q = 1..8
   __shared__ R sm[6 * RPL], sl[6 * RPL];    // mu, lambda of the rows' planes
   __shared__ R sf[2 * 3 * RHX * RTY];       // F over the tile's rows, i halo included
   __shared__ R sg[2 * 3 * RTX * RHY];       // G over the tile's columns, j halo included
   __shared__ R ssx[RHX], ssy[RHY];
   const int tix = blockIdx.x % ntx, tjy = blockIdx.x / ntx;
   const int tid = threadIdx.x;
   int role, hx, hy;
   rows_point(tid, role, hx, hy);
   const bool own = tid < RPL;  // the last 16 threads repeat a point and store nothing
   const bool ihalo = role == 2 && tid < 384 + 4 * RTY;
   const int ia = b.ib + tix * RTX, ja = b.jb + tjy * RTY;
   const bool active = role == 0 && ia + hx <= b.ie - 2 && ja + hy <= b.je - 2;
   // points off the box repeat its last row or column: read by inactive outputs only
   const int i = min(ia + hx, b.ie), j = min(ja + hy, b.je);
   const long nij = b.nij, col = (i - b.ib) + b.ni * (j - b.jb);
   const int kbase = top ? 1 : nk, sgn = top ? 1 : -1;
   const R sx = strx[i - b.ib], sy = stry[j - b.jb];
   const int o = hy * RHX + hx;
   const R i12 = R(1.0 / 12);
   auto d4c1 = [](const R* f, int st) { return f[-2 * st] - f[2 * st] + 8 * (f[st] - f[-st]); };

   R u[9][3], m[9], l[9];  // the column, row space
#pragma unroll
   for (int q = 0; q <= 8; q++) {
      const long p = col + nij * (kbase + sgn * (q - 1) - b.kb);
#pragma unroll
      for (int c = 0; c < 3; c++) u[q][c] = ld(c, p);
      m[q] = mu[p];
      l[q] = la[p];
   }
   if (own) {
#pragma unroll
      for (int q = 1; q <= 8; q++) {
#pragma unroll
         for (int c = 0; c < 3; c++) su[((q - 1) * 3 + c) * RPL + o] = u[q][c];
         if (q <= 6) {
            sm[(q - 1) * RPL + o] = m[q];
            sl[(q - 1) * RPL + o] = l[q];
         }
      }
   }
   if (tid < RHX) ssx[tid] = strx[min(ia + tid, b.ie) - b.ib];
   if (tid >= 64 && tid < 64 + RHY) ssy[tid - 64] = stry[min(ja + tid - 64, b.je) - b.jb];
   __syncthreads();
   // T of the eight planes: mu w_x, mu w_y, la (u_x + v_y)
   R T[9][3];
   if (role == 0) {
#pragma unroll
      for (int q = 1; q <= 8; q++) {
         const R* f = su + (q - 1) * 3 * RPL + o;
         T[q][0] = m[q] * (sx * (i12 * d4c1(f + 2 * RPL, 1)));
         T[q][1] = m[q] * (sy * (i12 * d4c1(f + 2 * RPL, RHX)));
         T[q][2] = l[q] * (sx * (i12 * d4c1(f, 1)) + sy * (i12 * d4c1(f + RPL, RHX)));
      }
   }
   int par = 0;
#pragma unroll 1
   for (int kr = 1 + (int)blockIdx.y; kr <= 6; kr += (int)gridDim.y) {
      const R* f = su + (kr - 1) * 3 * RPL + o;
      const R mk = sm[(kr - 1) * RPL + o], lk = sl[(kr - 1) * RPL + o];
      R dz[3] = {0, 0, 0}, z[3] = {0, 0, 0};
#pragma unroll
      for (int q = 1; q <= 8; q++) {
         const R bq = (R)sgn * sbp->bope[(kr - 1) + 6 * (q - 1)];
#pragma unroll
         for (int c = 0; c < 3; c++) dz[c] += bq * u[q][c];
         if (role == 0) {
#pragma unroll
            for (int c = 0; c < 3; c++) z[c] += bq * T[q][c];
         }
      }
      if (role == 0 || ihalo) {
         R* w = sf + par * 3 * RHX * RTY + (hy - 2) * RHX + hx;
         w[0] = lk * (sy * (i12 * d4c1(f + RPL, RHX)) + dz[2]);
         w[RHX * RTY] = mk * (sy * (i12 * d4c1(f, RHX)));
         w[2 * RHX * RTY] = mk * dz[0];
      }
      if (role != 2) {
         R* w = sg + par * 3 * RTX * RHY + hy * RTX + hx - 2;
         w[0] = mk * (sx * (i12 * d4c1(f + RPL, 1)));
         w[RTX * RHY] = lk * (sx * (i12 * d4c1(f, 1)) + dz[2]);
         w[2 * RTX * RHY] = mk * dz[1];
      }
      if (role == 0) {
         // SBP second difference along k with its ghost term
         const R gh = sbp->ghcof[kr - 1];
         z[0] += gh * m[1] * u[0][0];
         z[1] += gh * m[1] * u[0][1];
         z[2] += gh * (2 * m[1] + l[1]) * u[0][2];
#pragma unroll
         for (int q = 1; q <= 8; q++) {
            R cm = 0, ck = 0;
#pragma unroll
            for (int e = 1; e <= 8; e++) {
               const R a = sbp->acof[(kr - 1) + 6 * (q - 1) + 48 * (e - 1)];
               cm += a * m[e];
               ck += a * (2 * m[e] + l[e]);
            }
            z[0] += cm * u[q][0];
            z[1] += cm * u[q][1];
            z[2] += ck * u[q][2];
         }
      }
      __syncthreads();
      if (active) {
         R r[3];
         {
            R am[5], al[5], mx[4], my[4], cx[4], cy[4];
            const R *pm = sm + (kr - 1) * RPL + o, *pl = sl + (kr - 1) * RPL + o;
#pragma unroll
            for (int t = 0; t < 5; t++) {
               am[t] = pm[t - 2] * ssx[hx + t - 2];
               al[t] = pl[t - 2] * ssx[hx + t - 2];
            }
            varcoef4(am, mx);
            varcoef4(al, cx);
#pragma unroll
            for (int t = 0; t < 5; t++) {
               am[t] = pm[(t - 2) * RHX] * ssy[hy + t - 2];
               al[t] = pl[(t - 2) * RHX] * ssy[hy + t - 2];
            }
            varcoef4(am, my);
            varcoef4(al, cy);
#pragma unroll
            for (int t = 0; t < 4; t++) {
               cx[t] += 2 * mx[t];
               cy[t] += 2 * my[t];
            }
#pragma unroll
            for (int c = 0; c < 3; c++) {
               const R* g = f + c * RPL;
               R v[5];
#pragma unroll
               for (int t = 0; t < 5; t++) v[t] = g[t - 2];
               R acc = sx * varsum4(c == 0 ? cx : mx, v);
#pragma unroll
               for (int t = 0; t < 5; t++) v[t] = g[(t - 2) * RHX];
               acc += sy * varsum4(c == 1 ? cy : my, v);
               r[c] = acc * R(1.0 / 6);
            }
         }
         const R* wf = sf + par * 3 * RHX * RTY + (hy - 2) * RHX + hx;
         const R* wg = sg + par * 3 * RTX * RHY + hy * RTX + hx - 2;
#pragma unroll
         for (int c = 0; c < 3; c++)
            r[c] += z[c] + sx * (i12 * d4c1(wf + c * RHX * RTY, 1)) + sy * (i12 * d4c1(wg + c * RTX * RHY, RTX));
         const R uc[3] = {f[0], f[RPL], f[2 * RPL]};
         epi(i, j, kbase + sgn * (kr - 1), col + nij * (kbase + sgn * (kr - 1) - b.kb), r, uc);
      }
      par ^= 1;
   }
}

// Rows over block.y: where a grid's tiles leave workgroup slots idle
// (per_cu workgroups on each CU) the rows are spread over them.
inline int sbp_rows_spread(int tiles, int per_cu)
{
   const int slots = compute_units() * per_cu;
   return 6 * tiles <= slots ? 6 : 3 * tiles <= slots ? 3 : 2 * tiles <= slots ? 2 : 1;
}

}  // namespace sw4amd
