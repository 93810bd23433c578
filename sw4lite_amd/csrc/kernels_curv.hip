// kernels_curv.hip -- gfx950 kernels of the curvilinear (topography-following)
// grid, behind the reference's kernel-level entry points:
//   metric / metric_rev            curvilinear-c.C:53-172, :175-295
//   rhs4sgcurv / rhs4sgcurv_rev    rhs4sgcurv.C:34-1406, rhs4sgcurv_rev.C:34-1395
//   addsgd4cfort(_indrev)          ew-cfromfort.C:1160-1240, :1323-1404
//   freesurfcurvisg(_rev)          curvilinear-c.C:465-618, :621-764
// Both Sarray layouts through the CO template parameter; the metric is a
// 4-component array in the same layout as the displacement.
//
// The divergence of stress on the curvilinear grid, with M1..M4 the metric,
// K = 2mu + lambda, sx = strx(i), sy = stry(j), D_p, D_q centred 4th-order
// first differences along i and j and D_r the k-derivative of the row (SBP
// bope on the top six rows, centred inside), is L(u)_a = sx sy / jac * r_a,
//   r_a = pp + qq + rr + pq + qp + pr + qr + rp + rq,
//   pp = (1/6)(A u_a,p)_p / sy with A = (a==0 ? K : mu) M1^2 strx,
//   qq = (1/6)(B u_a,q)_q / sx with B = (a==1 ? K : mu) M1^2 stry,
//   rr = sum_b S_ab (R_ab u_b,r)_r, R the 3x3 coupling of mu, lambda and the
//        metric, S the stretching scalings; acof/ghcof SBP rows at the top,
//   pq, qp = centred mixed products in the plane (u and v equations),
//   pr, qr = D_r of T_a(D_p u, D_q u) on the neighbouring planes,
//   rp, rq = D_p of P_a(D_r u), D_q of Q_a(D_r u) on the neighbouring columns.
// The terms are those of the reference; the grouping of sums is this file's.
#include "kernels_common.h"
#include "kernels_curv.h"
#include "kernels_fast.h"
#include "sbp_rows.h"

namespace sw4amd {

namespace {
inline unsigned cdiv(long a, long b) { return (unsigned)((a + b - 1) / b); }
}  // namespace

constexpr double CC1 = 2.0 / 3, CC2 = -1.0 / 12;

template <int CO>
__device__ __forceinline__ long midx(const Box& b, int c, int i, int j, int k)
{
   const long p = sidx(b, i, j, k);
   return CO ? p + b.npts * c : 4 * p + c;
}

// ---------------------------------------------------------------------------
// Metric
// ---------------------------------------------------------------------------
// Derivative along a grid line of n points at position s (0-based): centred
// 4th order inside, 6-point one-sided closures on the first and last two
// points (curvilinear-c.C:78-146).
__device__ __forceinline__ double line_derivative(const double* __restrict__ f, long st, int s, int n)
{
#define F(t) f[(long)(t) * st]
   if (s >= 2 && s <= n - 3) return CC2 * (F(s + 2) - F(s - 2)) + CC1 * (F(s + 1) - F(s - 1));
   if (s == 0)
      return -2.25 * F(0) + (4 + 5.0 / 6) * F(1) - (14.0 / 3) * F(2) + 3 * F(3) - (1 + 1.0 / 12) * F(4) +
             (1.0 / 6) * F(5);
   if (s == 1)
      return -(1.0 / 6) * F(0) - 1.25 * F(1) + (1 + 4.0 / 3) * F(2) - (4.0 / 3) * F(3) + 0.5 * F(4) -
             (1.0 / 12) * F(5);
   if (s == n - 2)
      return (1.0 / 6) * F(n - 1) + 1.25 * F(n - 2) - (1 + 4.0 / 3) * F(n - 3) + (4.0 / 3) * F(n - 4) -
             0.5 * F(n - 5) + (1.0 / 12) * F(n - 6);
   return 2.25 * F(n - 1) - (4 + 5.0 / 6) * F(n - 2) + (14.0 / 3) * F(n - 3) - 3 * F(n - 4) +
          (1 + 1.0 / 12) * F(n - 5) - (1.0 / 6) * F(n - 6);
#undef F
}

template <int CO>
__global__ void __launch_bounds__(256)
k_metric(Box b, double h, const double* __restrict__ z, double* __restrict__ met, double* __restrict__ jac,
         int* __restrict__ bad)
{
   const long p = blockIdx.x * (long)blockDim.x + threadIdx.x;
   if (p >= b.npts) return;
   const int ni = (int)b.ni, nj = b.je - b.jb + 1, nk = b.ke - b.kb + 1;
   const int ii = (int)(p % ni);
   const long r = p / ni;
   const int jj = (int)(r % nj), kk = (int)(r / nj);
   const double zr = line_derivative(z + (p - b.nij * kk), b.nij, kk, nk);
   const double zq = line_derivative(z + (p - b.ni * jj), b.ni, jj, nj);
   const double zp = line_derivative(z + (p - ii), 1, ii, ni);
   if (!(zr > 0)) {
      bad[0] = 1;
      return;
   }
   const double sq = sqrt(zr);
   jac[p] = h * h * zr;
   const long m0 = CO ? p : 4 * p, ms = CO ? b.npts : 1;
   met[m0] = sq;
   met[m0 + ms] = -zp / sq;
   met[m0 + 2 * ms] = -zq / sq;
   met[m0 + 3 * ms] = h / sq;
}

// ---------------------------------------------------------------------------
// Divergence of stress
// ---------------------------------------------------------------------------
template <int CO>
struct CurvG {
   Box b;
   const double* __restrict__ u;
   const double* __restrict__ mu;
   const double* __restrict__ la;
   const double* __restrict__ met;
   const double* __restrict__ strx;
   const double* __restrict__ stry;
   __device__ __forceinline__ double U(int c, int i, int j, int k) const { return u[vidx<CO>(b, c, i, j, k)]; }
   __device__ __forceinline__ double M(int c, int i, int j, int k) const { return met[midx<CO>(b, c, i, j, k)]; }
   __device__ __forceinline__ double MU(int i, int j, int k) const { return mu[sidx(b, i, j, k)]; }
   __device__ __forceinline__ double LA(int i, int j, int k) const { return la[sidx(b, i, j, k)]; }
   __device__ __forceinline__ double SX(int i) const { return strx[i - b.ib]; }
   __device__ __forceinline__ double SY(int j) const { return stry[j - b.jb]; }
   __device__ __forceinline__ double Dp(int c, int i, int j, int k) const
   {
      return CC2 * (U(c, i + 2, j, k) - U(c, i - 2, j, k)) + CC1 * (U(c, i + 1, j, k) - U(c, i - 1, j, k));
   }
   __device__ __forceinline__ double Dq(int c, int i, int j, int k) const
   {
      return CC2 * (U(c, i, j + 2, k) - U(c, i, j - 2, k)) + CC1 * (U(c, i, j + 1, k) - U(c, i, j - 1, k));
   }
};

__device__ __forceinline__ void vc4(const double a[5], double m[4])
{
   m[0] = a[1] - 0.75 * (a[2] + a[0]);
   m[1] = a[0] + a[3] + 3 * (a[2] + a[1]);
   m[2] = a[1] + a[4] + 3 * (a[3] + a[2]);
   m[3] = a[3] - 0.75 * (a[2] + a[4]);
}
__device__ __forceinline__ double vs4(const double m[4], const double f[5])
{
   return m[0] * (f[0] - f[2]) + m[1] * (f[1] - f[2]) + m[2] * (f[3] - f[2]) + m[3] * (f[4] - f[2]);
}

// traction-like combination of in-plane derivatives on plane m, column (i,j):
// the pr/qr terms of the operator and the tangential part of the free-
// surface traction (curvilinear-c.C:520-578)
template <class S>
__device__ __forceinline__ void t_terms(const S& s, int i, int j, int m, double sx, double sy, double isx,
                                        double isy, double T[3])
{
   const double mu = s.MU(i, j, m), la = s.LA(i, j, m), K = 2 * mu + la;
   const double m1 = s.M(0, i, j, m), m2 = s.M(1, i, j, m), m3 = s.M(2, i, j, m), m4 = s.M(3, i, j, m);
   const double p0 = s.Dp(0, i, j, m), p1 = s.Dp(1, i, j, m), p2 = s.Dp(2, i, j, m);
   const double q0 = s.Dq(0, i, j, m), q1 = s.Dq(1, i, j, m), q2 = s.Dq(2, i, j, m);
   const double a2 = m2 * m1, a3 = m3 * m1, a4 = m4 * m1;
   T[0] = K * a2 * p0 * sx * isy + mu * a3 * p1 + mu * a4 * p2 * isy + mu * a3 * q0 * sy * isx + la * a2 * q1;
   T[1] = la * a3 * p0 + mu * a2 * p1 * sx * isy + mu * a2 * q0 + K * a3 * q1 * sy * isx + mu * a4 * q2 * isx;
   T[2] = la * a4 * p0 * isy + mu * a2 * p2 * sx * isy + mu * a3 * q2 * sy * isx + la * a4 * q1 * isx;
}

// The interior rows as a k-march with every first derivative formed once.
// Grouped by the outer derivative the operator is
//   r = pp + qq + rr + D_p F + D_q G + D_r T,
// F, G, T the products of material, metric and first derivatives at one
// point (the flux-like sums whose D_p, D_q, D_r are pq and rp, qp and rq, pr
// and qr), so a point forms its nine first derivatives and nine products
// once and its neighbours read the products, instead of every output forming
// them for its twelve neighbours (about 700 operations a point instead of
// 2126).  A workgroup owns a 32 x 8 tile; each of the 36 x 12 points of the
// tile with its halo has a thread (four waves of outputs, two of the j halo,
// one of the i halo and corners), which loads its point's nine values one
// plane ahead and keeps the column n-4..n of the material and the metric in
// registers (that of u in LDS).  Per plane n: u and
// (mu, lambda) M1^2 go to LDS, one barrier, the in-plane derivatives give
// pp + qq and T of plane n; plane n-2 gets F and G (to LDS, read after the
// next barrier) and rr + D_r T; plane n-3 is finished.  The rings have five
// slots and the plane loop is unrolled by five, so every index is a constant
// and nothing is moved between registers.
// Bound by latency and VALU issue at 2 waves/SIMD (one workgroup per CU, 234
// registers): 384x384x256 points 1.90 ms against 6.7 ms of a thread per point reading every
// neighbour through the caches (2126 operations, 256 registers).
// (the scheduler would otherwise hoist the shared-memory reads of a whole
// plane to its start and spill)
#define SW4_SCHED_FENCE __builtin_amdgcn_sched_barrier(0)
constexpr int MTX = RTX, MTY = RTY, MHX = RHX, MHY = RHY, MPL = RPL, MNT = RNT;  // the tile of sbp_rows.h (rows_point)

template <int CO>
__global__ void __launch_bounds__(MNT, 1)
k_rhs4curv_march(Box b, int ntx, int nty, int ntiles, int klo, int khi, int kc, CurvG<CO> s,
                 const double* __restrict__ jac, double* __restrict__ lu)
{
   __shared__ double su[5][3 * MPL];               // u of planes n-4..n
   __shared__ double se[2][2 * MPL];               // mu M1^2, lambda M1^2 of plane n
   __shared__ double sf[2][3 * MHX * MTY];         // F over the tile's rows, i halo included
   __shared__ double sg[2][3 * MTX * MHY];         // G over the tile's columns, j halo included
   __shared__ double ssx[MHX], ssy[MHY];
   // XCD-aware order: a contiguous run of tiles per XCD (blocks go to the 8 XCDs round-robin)
   const int per = (ntiles + 7) / 8;
   const int t = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
   if (t >= ntiles) return;
   const int tix = t % ntx, tr = t / ntx, tjy = tr % nty, tkz = tr / nty;
   const int k0 = klo + tkz * kc, k1 = min(khi, k0 + kc - 1);
   const int tid = threadIdx.x;
   int role, hx, hy;
   rows_point(tid, role, hx, hy);
   const bool own = tid < MPL;  // the last 16 threads repeat a point and store nothing
   const Box& b_ = b;
   const int ia = b_.ib + tix * MTX, ja = b_.jb + tjy * MTY;
   const bool active = role == 0 && ia + hx <= b_.ie - 2 && ja + hy <= b_.je - 2;
   // points off the box repeat its last row or column: read by inactive outputs only
   const int i = min(ia + hx, b_.ie), j = min(ja + hy, b_.je);
   const long nij = b_.nij, npts = b_.npts;
   const long col = (i - b_.ib) + b_.ni * (j - b_.jb);
   const double sx = s.SX(i), sy = s.SY(j), isx = 1 / sx, isy = 1 / sy;
   if (tid < MHX) ssx[tid] = s.SX(min(ia + tid, b_.ie));
   if (tid >= 64 && tid < 64 + MHY) ssy[tid - 64] = s.SY(min(ja + tid - 64, b_.je));
   const int o = hy * MHX + hx;

   double mu[5], la[5], m1[5], m2[5], m3[5], m4[5];  // column ring
   double pq[5][4];                                  // D_p u, D_p v, D_q u, D_q v
   // pp + qq + rr + D_r T, the terms of D_r T added as their planes come
   double acc[5][3] = {};
   double rp[3] = {0, 0, 0};                         // acc of the plane finished next
   double nu[3], nmu, nla, nm[4], njac = 1.0;                 // loaded one plane ahead
   auto load = [&](int kk) {
      const long p = col + nij * (kk - b_.kb);
#pragma unroll
      for (int c = 0; c < 3; c++) nu[c] = s.u[CO ? p + npts * c : 3 * p + c];
      nmu = s.mu[p];
      nla = s.la[p];
#pragma unroll
      for (int c = 0; c < 4; c++) nm[c] = s.met[CO ? p + npts * c : 4 * p + c];
   };
   auto D = [](double fm2, double fm1, double fp1, double fp2) { return CC2 * (fp2 - fm2) + CC1 * (fp1 - fm1); };
   load(k0 - 2);
   int par = 0;
   for (int n0 = k0 - 2; n0 <= k1 + 3; n0 += 5) {
#pragma unroll
      for (int ph = 0; ph < 5; ph++) {
         const int n = n0 + ph;
         if (n > k1 + 3) break;
         const int s0 = ph, s1 = (ph + 4) % 5, s2 = (ph + 3) % 5, s3 = (ph + 2) % 5, s4 = (ph + 1) % 5;  // n..n-4
         const double cjac = njac;
         if (n <= k1 + 2) {
            mu[s0] = nmu;
            la[s0] = nla;
            m1[s0] = nm[0];
            m2[s0] = nm[1];
            m3[s0] = nm[2];
            m4[s0] = nm[3];
            if (own) {
               const double q = m1[s0] * m1[s0];
#pragma unroll
               for (int c = 0; c < 3; c++) su[s0][c * MPL + o] = nu[c];
               se[par][o] = mu[s0] * q;
               se[par][MPL + o] = la[s0] * q;
            }
         }
         __syncthreads();  // plane n is in su, se, F and G of plane n-3 in sf, sg[par ^ 1]
         if (n < k1 + 2) load(n + 1);
         if (role == 0 && n >= k0 + 2) njac = jac[col + nij * (n - 2 - b_.kb)];
         if (role == 0 && n >= k0 + 3 && active) {  // finish plane n-3
            const double* f = &sf[par ^ 1][(hy - 2) * MHX + hx];
            const double* g = &sg[par ^ 1][hy * MTX + hx - 2];
            const double w = sx * sy / cjac;
            const long p = col + nij * (n - 3 - b_.kb);
#pragma unroll
            for (int c = 0; c < 3; c++) {
               const double* fc = f + c * MHX * MTY;
               const double* gc = g + c * MTX * MHY;
               const double r = rp[c] + D(fc[-2], fc[-1], fc[1], fc[2]) +
                                D(gc[-2 * MTX], gc[-MTX], gc[MTX], gc[2 * MTX]);
               lu[CO ? p + npts * c : 3 * p + c] = r * w;
            }
         }
         if (n > k1 + 2) break;
         SW4_SCHED_FENCE;
         // in-plane derivatives of plane n
         const double* pu = su[s0] + o;
         const double* pe = se[par] + o;
         if (role == 0) {
            // pp and qq coefficients: cx, cy for the component along the axis, mx, my for the others
            double mx[4], my[4], cx[4], cy[4], p[3], q[3];
            {
               double am[5], al[5];
#pragma unroll
               for (int e = 0; e < 5; e++) {
                  am[e] = pe[e - 2] * ssx[hx + e - 2];
                  al[e] = pe[MPL + e - 2] * ssx[hx + e - 2];
               }
               vc4(am, mx);
               vc4(al, cx);
#pragma unroll
               for (int e = 0; e < 5; e++) {
                  am[e] = pe[(e - 2) * MHX] * ssy[hy + e - 2];
                  al[e] = pe[MPL + (e - 2) * MHX] * ssy[hy + e - 2];
               }
               vc4(am, my);
               vc4(al, cy);
#pragma unroll
               for (int e = 0; e < 4; e++) {
                  cx[e] += 2 * mx[e];
                  cy[e] += 2 * my[e];
               }
            }
#pragma unroll
            for (int c = 0; c < 3; c++) {
               SW4_SCHED_FENCE;
               const double* f = pu + c * MPL;
               const double x0 = f[-2], x1 = f[-1], x3 = f[1], x4 = f[2];
               const double y0 = f[-2 * MHX], y1 = f[-MHX], y3 = f[MHX], y4 = f[2 * MHX], u0 = f[0];
               p[c] = D(x0, x1, x3, x4);
               q[c] = D(y0, y1, y3, y4);
               const double* wx = c == 0 ? cx : mx;
               const double* wy = c == 1 ? cy : my;
               const double ax = wx[0] * (x0 - u0) + wx[1] * (x1 - u0) + wx[2] * (x3 - u0) + wx[3] * (x4 - u0);
               const double ay = wy[0] * (y0 - u0) + wy[1] * (y1 - u0) + wy[2] * (y3 - u0) + wy[3] * (y4 - u0);
               acc[s0][c] += (1.0 / 6) * (ax * isy + ay * isx);
            }
            SW4_SCHED_FENCE;
            pq[s0][0] = p[0];
            pq[s0][1] = p[1];
            pq[s0][2] = q[0];
            pq[s0][3] = q[1];
            {
               const double a2 = m2[s0] * m1[s0], a3 = m3[s0] * m1[s0], a4 = m4[s0] * m1[s0];
               const double xy = sx * isy, yx = sy * isx, K = 2 * mu[s0] + la[s0];
               double T[3];
               T[0] = K * a2 * xy * p[0] + mu[s0] * (a3 * p[1] + a4 * isy * p[2] + a3 * yx * q[0]) + la[s0] * a2 * q[1];
               T[1] = la[s0] * a3 * p[0] + mu[s0] * (a2 * xy * p[1] + a2 * q[0] + a4 * isx * q[2]) + K * a3 * yx * q[1];
               T[2] = la[s0] * a4 * (isy * p[0] + isx * q[1]) + mu[s0] * (a2 * xy * p[2] + a3 * yx * q[2]);
#pragma unroll
               for (int c = 0; c < 3; c++) {  // D_r T of planes n-2, n-1, n+1 and (its first term) n+2
                  acc[s2][c] += CC2 * T[c];
                  acc[s1][c] += CC1 * T[c];
                  acc[s4][c] -= CC1 * T[c];
                  acc[s3][c] = -CC2 * T[c];
               }
            }
         } else if (role == 1) {
#pragma unroll
            for (int c = 0; c < 2; c++) {
               const double* f = pu + c * MPL;
               pq[s0][c] = D(f[-2], f[-1], f[1], f[2]);
            }
         } else if (tid < 384 + 4 * MTY) {
#pragma unroll
            for (int c = 0; c < 2; c++) {
               const double* f = pu + c * MPL;
               pq[s0][2 + c] = D(f[-2 * MHX], f[-MHX], f[MHX], f[2 * MHX]);
            }
         }
         SW4_SCHED_FENCE;
         // plane k = n-2: F, G and the terms along the column
         if (n >= k0 + 2) {
            double dz[3];
#pragma unroll
            for (int c = 0; c < 3; c++)
               dz[c] = D(su[s4][c * MPL + o], su[s3][c * MPL + o], su[s1][c * MPL + o], su[s0][c * MPL + o]);
            const double q = m1[s2] * m1[s2], a2 = m2[s2] * m1[s2], a3 = m3[s2] * m1[s2], a4 = m4[s2] * m1[s2];
            const double xy = sx * isy, yx = sy * isx, K = 2 * mu[s2] + la[s2];
            if (role != 1 && tid < 384 + 4 * MTY) {
               double* f = &sf[par][(hy - 2) * MHX + hx];
               f[0] = la[s2] * (q * pq[s2][3] + isy * (a3 * sy * dz[1] + a4 * dz[2])) + K * a2 * xy * dz[0];
               f[MHX * MTY] = mu[s2] * (q * pq[s2][2] + a3 * dz[0] + a2 * xy * dz[1]);
               f[2 * MHX * MTY] = mu[s2] * (a4 * dz[0] + a2 * sx * dz[2]) * isy;
            }
            if (role != 2) {
               double* g = &sg[par][hy * MTX + hx - 2];
               g[0] = mu[s2] * (q * pq[s2][1] + a3 * yx * dz[0] + a2 * dz[1]);
               g[MTX * MHY] = la[s2] * (q * pq[s2][0] + a2 * dz[0] + a4 * isx * dz[2]) + K * a3 * yx * dz[1];
               g[2 * MTX * MHY] = mu[s2] * (a3 * sy * dz[2] + a4 * dz[1]) * isx;
            }
            SW4_SCHED_FENCE;
            if (role == 0) {
               // rr_a = 1/(6 sx sy) sum_t [mu |m|^2 w_a + (mu + lambda) m_a (m . w)]_t with m = (M2 sx, M3 sy, M4)
               // and w_t the weights of plane t's coefficient (a combination of u(k+q) - u(k))
               double w[5][3], rr[3] = {0, 0, 0};
#pragma unroll
               for (int c = 0; c < 3; c++) {
                  const int q = c * MPL + o;
                  const double u0 = su[s2][q], d0 = su[s4][q] - u0, d1 = su[s3][q] - u0, d3 = su[s1][q] - u0,
                               d4 = su[s0][q] - u0;
                  w[0][c] = d1 - 0.75 * d0;
                  w[1][c] = d0 + 3 * d1 + d3;
                  w[2][c] = 3 * (d1 + d3) - 0.75 * (d0 + d4);
                  w[3][c] = d1 + 3 * d3 + d4;
                  w[4][c] = d3 - 0.75 * d4;
               }
#pragma unroll
               for (int e = 0; e < 5; e++) {
                  const int se = (s0 + 1 + e) % 5;  // plane k - 2 + e
                  const double x = m2[se] * sx, y = m3[se] * sy, z = m4[se];
                  const double mn = mu[se] * (x * x + y * y + z * z);
                  const double ml = (mu[se] + la[se]) * (x * w[e][0] + y * w[e][1] + z * w[e][2]);
                  rr[0] += mn * w[e][0] + ml * x;
                  rr[1] += mn * w[e][1] + ml * y;
                  rr[2] += mn * w[e][2] + ml * z;
               }
               const double i6xy = (1.0 / 6) * isx * isy;
#pragma unroll
               for (int c = 0; c < 3; c++)
                  rp[c] = acc[s2][c] + i6xy * rr[c];
            }
         }
         par ^= 1;
      }
   }
}

// The top six rows (k = 1..6, SBP closures along k) with the same grouping
// and the same threads as the march: the planes k = 1..8 go to LDS once, T of
// the eight planes and the material of the column's rr are kept for all rows
// (256 registers and 22-24 spilled); per row the columns form F and G, one barrier, and the outputs
// are finished.  With rr written as in the march,
//   rr = 1/(sx sy) sum_q [mu |m|^2 w_a + (mu + lambda) m_a (m . w)]_q,
//   w_b(k, q) = sum_t acof(k, t, q) u_b(t)  (and ghcof on the ghost plane).
// block.y takes the rows 1 + block.y, the next gridDim.y on.  Against a
// thread per point (6049 operations): 384 x 384 points 394 -> 127 us,
// 65 x 65 40 -> 17.
template <int CO>
__global__ void __launch_bounds__(MNT, 1)
k_rhs4curv_rows(Box b, int ntx, const SbpTables* __restrict__ sbp, CurvG<CO> s, const double* __restrict__ jac,
                double* __restrict__ lu)
{
   __shared__ double su[8 * 3 * MPL];          // u of planes 1..8
   __shared__ double se[6 * 2 * MPL];          // mu M1^2, lambda M1^2 of the rows' planes
   __shared__ double sf[2][3 * MHX * MTY];     // F over the tile's rows, i halo included
   __shared__ double sg[2][3 * MTX * MHY];     // G over the tile's columns, j halo included
   __shared__ double ssx[MHX], ssy[MHY];
   const int tix = blockIdx.x % ntx, tjy = blockIdx.x / ntx;
   const int tid = threadIdx.x;
   int role, hx, hy;
   rows_point(tid, role, hx, hy);
   const bool own = tid < MPL;
   const bool ihalo = role == 2 && tid < 384 + 4 * MTY;
   const int ia = b.ib + tix * MTX, ja = b.jb + tjy * MTY;
   const bool active = role == 0 && ia + hx <= b.ie - 2 && ja + hy <= b.je - 2;
   const int i = min(ia + hx, b.ie), j = min(ja + hy, b.je);
   const long nij = b.nij, npts = b.npts;
   const long col = (i - b.ib) + b.ni * (j - b.jb);
   const double sx = s.SX(i), sy = s.SY(j), isx = 1 / sx, isy = 1 / sy, xy = sx * isy, yx = sy * isx;
   if (tid < MHX) ssx[tid] = s.SX(min(ia + tid, b.ie));
   if (tid >= 64 && tid < 64 + MHY) ssy[tid - 64] = s.SY(min(ja + tid - 64, b.je));
   const int o = hy * MHX + hx;
   auto D = [](const double* f, int st) { return CC2 * (f[2 * st] - f[-2 * st]) + CC1 * (f[st] - f[-st]); };
   auto at = [=](int c, long p) { return CO ? p + npts * c : 3 * p + c; };
   auto met = [=](int c, long p) { return s.met[CO ? p + npts * c : 4 * p + c]; };

   double u[9][3];
#pragma unroll
   for (int q = 0; q <= 8; q++) {
      const long p = col + nij * (q - b.kb);
#pragma unroll
      for (int c = 0; c < 3; c++) u[q][c] = s.u[at(c, p)];
      if (own && q >= 1) {
#pragma unroll
         for (int c = 0; c < 3; c++) su[((q - 1) * 3 + c) * MPL + o] = u[q][c];
         if (q <= 6) {
            const double m1 = met(0, p);
            se[(2 * q - 2) * MPL + o] = s.mu[p] * m1 * m1;
            se[(2 * q - 1) * MPL + o] = s.la[p] * m1 * m1;
         }
      }
   }
   __syncthreads();
   // of the planes 1..8: T, and mu |m|^2, mu + lambda, m of rr
   double T[9][3], mn[9], ml[9], mx_[9], my_[9], mz_[9];
   if (role == 0) {
#pragma unroll
      for (int q = 1; q <= 8; q++) {
         SW4_SCHED_FENCE;
         const long pt = col + nij * (q - b.kb);
         const double mu = s.mu[pt], la = s.la[pt], m1 = met(0, pt), m2 = met(1, pt), m3 = met(2, pt), m4 = met(3, pt);
         const double* f = su + (q - 1) * 3 * MPL + o;
         const double p0 = D(f, 1), p1 = D(f + MPL, 1), p2 = D(f + 2 * MPL, 1);
         const double q0 = D(f, MHX), q1 = D(f + MPL, MHX), q2 = D(f + 2 * MPL, MHX);
         const double a2 = m2 * m1, a3 = m3 * m1, a4 = m4 * m1, K = 2 * mu + la;
         T[q][0] = K * a2 * xy * p0 + mu * (a3 * p1 + a4 * isy * p2 + a3 * yx * q0) + la * a2 * q1;
         T[q][1] = la * a3 * p0 + mu * (a2 * xy * p1 + a2 * q0 + a4 * isx * q2) + K * a3 * yx * q1;
         T[q][2] = la * a4 * (isy * p0 + isx * q1) + mu * (a2 * xy * p2 + a3 * yx * q2);
         mx_[q] = m2 * sx;
         my_[q] = m3 * sy;
         mz_[q] = m4;
         mn[q] = mu * (mx_[q] * mx_[q] + my_[q] * my_[q] + mz_[q] * mz_[q]);
         ml[q] = mu + la;
      }
   }
   int par = 0;
#pragma unroll 1
   for (int kr = 1 + (int)blockIdx.y; kr <= 6; kr += (int)gridDim.y) {
      const long pt = col + nij * (kr - b.kb);
      const double mu = s.mu[pt], la = s.la[pt], m1 = met(0, pt), m2 = met(1, pt), m3 = met(2, pt), m4 = met(3, pt);
      const double w = role == 0 ? sx * sy / jac[pt] : 0.0;
      const double* f = su + (kr - 1) * 3 * MPL + o;
      double dz[3] = {0, 0, 0}, z[3] = {0, 0, 0};
#pragma unroll
      for (int q = 1; q <= 8; q++) {
         const double bq = sbp->bope[(kr - 1) + 6 * (q - 1)];
#pragma unroll
         for (int c = 0; c < 3; c++) dz[c] += bq * u[q][c];
         if (role == 0) {
#pragma unroll
            for (int c = 0; c < 3; c++) z[c] += bq * T[q][c];
         }
      }
      {
         const double q = m1 * m1, a2 = m2 * m1, a3 = m3 * m1, a4 = m4 * m1, K = 2 * mu + la;
         if (role == 0 || ihalo) {
            double* v = &sf[par][(hy - 2) * MHX + hx];
            v[0] = la * (q * D(f + MPL, MHX) + isy * (a3 * sy * dz[1] + a4 * dz[2])) + K * a2 * xy * dz[0];
            v[MHX * MTY] = mu * (q * D(f, MHX) + a3 * dz[0] + a2 * xy * dz[1]);
            v[2 * MHX * MTY] = mu * (a4 * dz[0] + a2 * sx * dz[2]) * isy;
         }
         if (role != 2) {
            double* v = &sg[par][hy * MTX + hx - 2];
            v[0] = mu * (q * D(f + MPL, 1) + a3 * yx * dz[0] + a2 * dz[1]);
            v[MTX * MHY] = la * (q * D(f, 1) + a2 * dz[0] + a4 * isx * dz[2]) + K * a3 * yx * dz[1];
            v[2 * MTX * MHY] = mu * (a3 * sy * dz[2] + a4 * dz[1]) * isx;
         }
      }
      SW4_SCHED_FENCE;
      if (role == 0) {
         double rr[3] = {0, 0, 0};
#pragma unroll
         for (int q = 1; q <= 8; q++) {
            double v[3] = {0, 0, 0};
            if (q == 1) {  // the ghost plane's term carries plane 1's coefficients
               const double g = sbp->ghcof[kr - 1];
#pragma unroll
               for (int c = 0; c < 3; c++) v[c] = g * u[0][c];
            }
#pragma unroll
            for (int e = 1; e <= 8; e++) {
               const double a = sbp->acof[(kr - 1) + 6 * (e - 1) + 48 * (q - 1)];
#pragma unroll
               for (int c = 0; c < 3; c++) v[c] += a * u[e][c];
            }
            const double t = ml[q] * (mx_[q] * v[0] + my_[q] * v[1] + mz_[q] * v[2]);
            rr[0] += mn[q] * v[0] + t * mx_[q];
            rr[1] += mn[q] * v[1] + t * my_[q];
            rr[2] += mn[q] * v[2] + t * mz_[q];
         }
#pragma unroll
         for (int c = 0; c < 3; c++) z[c] += isx * isy * rr[c];
      }
      __syncthreads();
      if (active) {
         const double* pe = se + (2 * kr - 2) * MPL + o;
         double mx[4], my[4], cx[4], cy[4], am[5], al[5];
#pragma unroll
         for (int e = 0; e < 5; e++) {
            am[e] = pe[e - 2] * ssx[hx + e - 2];
            al[e] = pe[MPL + e - 2] * ssx[hx + e - 2];
         }
         vc4(am, mx);
         vc4(al, cx);
#pragma unroll
         for (int e = 0; e < 5; e++) {
            am[e] = pe[(e - 2) * MHX] * ssy[hy + e - 2];
            al[e] = pe[MPL + (e - 2) * MHX] * ssy[hy + e - 2];
         }
         vc4(am, my);
         vc4(al, cy);
#pragma unroll
         for (int e = 0; e < 4; e++) {
            cx[e] += 2 * mx[e];
            cy[e] += 2 * my[e];
         }
         const double* vf = &sf[par][(hy - 2) * MHX + hx];
         const double* vg = &sg[par][hy * MTX + hx - 2];
#pragma unroll
         for (int c = 0; c < 3; c++) {
            const double* g = f + c * MPL;
            const double x[5] = {g[-2], g[-1], g[0], g[1], g[2]};
            const double y[5] = {g[-2 * MHX], g[-MHX], g[0], g[MHX], g[2 * MHX]};
            const double r = z[c] + (1.0 / 6) * (isy * vs4(c == 0 ? cx : mx, x) + isx * vs4(c == 1 ? cy : my, y)) +
                             D(vf + c * MHX * MTY, 1) + D(vg + c * MTX * MHY, MTX);
            lu[at(c, pt)] = r * w;
         }
      }
      par ^= 1;
   }
}

// ---------------------------------------------------------------------------
// Supergrid damping in x and y with rho -> rho jac
// ---------------------------------------------------------------------------
template <int CO>
__global__ void __launch_bounds__(256)
k_addsgd4c(Box b, double* __restrict__ up, const double* __restrict__ u, const double* __restrict__ um,
           const double* __restrict__ rho, const double* __restrict__ jac, SgCoef sg, double beta)
{
   const int i = b.ib + 2 + blockIdx.x * blockDim.x + threadIdx.x;
   const int j = b.jb + 2 + blockIdx.y * blockDim.y + threadIdx.y;
   const int k = b.kb + 2 + blockIdx.z;
   if (i > b.ie - 2 || j > b.je - 2) return;
   const int ii = i - b.ib, jj = j - b.jb;
   // every term carries one of these damping coefficients: where all six
   // vanish (the columns away from the x and y supergrid layers) the update
   // subtracts zero, and the point is left as it is
   if (sg.dcx[ii - 1] == 0 && sg.dcx[ii] == 0 && sg.dcx[ii + 1] == 0 && sg.dcy[jj - 1] == 0 && sg.dcy[jj] == 0 &&
       sg.dcy[jj + 1] == 0)
      return;
   const long p = sidx(b, i, j, k);
   const double w = beta / (rho[p] * jac[p]);
   double rx[3], ry[3];
#pragma unroll
   for (int t = 0; t < 3; t++) {
      const long px = sidx(b, i + t - 1, j, k), py = sidx(b, i, j + t - 1, k);
      rx[t] = rho[px] * sg.dcx[ii + t - 1] * jac[px];
      ry[t] = rho[py] * sg.dcy[jj + t - 1] * jac[py];
   }
   const double wx = sg.strx[ii] * sg.coy[jj], wy = sg.stry[jj] * sg.cox[ii];
#pragma unroll
   for (int c = 0; c < 3; c++) {
      double dx[5], dy[5];
#pragma unroll
      for (int t = 0; t < 5; t++) {
         long q = vidx<CO>(b, c, i + t - 2, j, k);
         dx[t] = u[q] - um[q];
         q = vidx<CO>(b, c, i, j + t - 2, k);
         dy[t] = u[q] - um[q];
      }
      const double ax = rx[2] * (dx[4] - 2 * dx[3] + dx[2]) - 2 * rx[1] * (dx[3] - 2 * dx[2] + dx[1]) +
                        rx[0] * (dx[2] - 2 * dx[1] + dx[0]);
      const double ay = ry[2] * (dy[4] - 2 * dy[3] + dy[2]) - 2 * ry[1] * (dy[3] - 2 * dy[2] + dy[1]) +
                        ry[0] * (dy[2] - 2 * dy[1] + dy[0]);
      up[vidx<CO>(b, c, i, j, k)] -= w * (wx * ax + wy * ay);
   }
}

// ---------------------------------------------------------------------------
// The pointwise stages of the curvilinear step around the operator, in two
// passes (component-blocked): predictor and acceleration, and corrector with
// the supergrid damping.  Sources, which act on a few points, follow each.
// ---------------------------------------------------------------------------
// up = 2u - um + dt2/rho lu, acc = (up - 2u + um) dt2i on the whole box
__global__ void __launch_bounds__(256)
k_curv_pred(long npts, const double* __restrict__ lu, const double* __restrict__ u, const double* __restrict__ um,
            const double* __restrict__ rho, double* __restrict__ up, double* __restrict__ acc, double dt2, double dt2i)
{
   const long p = blockIdx.x * (long)blockDim.x + threadIdx.x;
   if (p >= npts) return;
   const double sc = dt2 / rho[p];
#pragma unroll
   for (int c = 0; c < 3; c++) {
      const long q = p + npts * c;
      const double uv = u[q], mv = um[q], v = 2 * uv - mv + sc * lu[q];
      up[q] = v;
      acc[q] = dt2i * (v - 2 * uv + mv);
   }
}

// up += c4/rho lu - damping(u - um) (addsgd4c) on the interior columns of a
// 32 x 8 tile, planes k0..k1.  Tiles that meet an x or y layer stage d = u - um
// and rho jac of a plane in LDS, loaded one plane ahead by a thread for each
// point of the tile and its halo (one barrier per plane); the others only add.
// Bound by memory.
__global__ void __launch_bounds__(MNT, 2)
k_curv_corr(Box b, int ntx, int nty, int ntiles, int klo, int khi, int kc, double* __restrict__ up,
            const double* __restrict__ lu, const double* __restrict__ u, const double* __restrict__ um,
            const double* __restrict__ rho, const double* __restrict__ jac, SgCoef sg, double c4, double beta)
{
   __shared__ double sd[2][3 * MPL];
   __shared__ double sr[2][MPL];
   const int per = (ntiles + 7) / 8;
   const int t = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
   if (t >= ntiles) return;
   const int tix = t % ntx, tr = t / ntx, tjy = tr % nty, tkz = tr / nty;
   const int k0 = klo + tkz * kc, k1 = min(khi, k0 + kc - 1);
   const int tid = threadIdx.x;
   int role, hx, hy;
   rows_point(tid, role, hx, hy);
   const int ia = b.ib + tix * MTX, ja = b.jb + tjy * MTY;
   const bool active = role == 0 && ia + hx <= b.ie - 2 && ja + hy <= b.je - 2;
   const int ii = min(ia + hx, b.ie) - b.ib, jj = min(ja + hy, b.je) - b.jb;
   const long nij = b.nij, npts = b.npts;
   const long col = ii + b.ni * jj;
   bool meets = false;  // dc of the tile's columns and of one more at each end
   if (beta != 0 && tid < MTX + 2)
      meets = sg.dcx[min(tix * MTX + 1 + tid, (int)b.ni - 1)] != 0;
   else if (beta != 0 && tid >= 64 && tid < 64 + MTY + 2)
      meets = sg.dcy[min(tjy * MTY + 1 + tid - 64, b.je - b.jb)] != 0;
   if (!__syncthreads_or(meets)) {
      if (!active) return;
      for (int k = k0; k <= k1; k++) {
         const long p = col + nij * (k - b.kb);
         const double sc = c4 / rho[p];
#pragma unroll
         for (int c = 0; c < 3; c++) up[p + npts * c] += sc * lu[p + npts * c];
      }
      return;
   }
   const int o = hy * MHX + hx;
   const bool own = tid < MPL;
   // of an output's column: dc at -1, 0, +1 and the weights
   double gx[3] = {0, 0, 0}, gy[3] = {0, 0, 0}, wx = 0, wy = 0;
   if (active) {
#pragma unroll
      for (int e = 0; e < 3; e++) {
         gx[e] = sg.dcx[ii + e - 1];
         gy[e] = sg.dcy[jj + e - 1];
      }
      wx = sg.strx[ii] * sg.coy[jj];
      wy = sg.stry[jj] * sg.cox[ii];
   }
   const bool damped = gx[0] != 0 || gx[1] != 0 || gx[2] != 0 || gy[0] != 0 || gy[1] != 0 || gy[2] != 0;
   double nu[3], nm[3], nr, nj, np[3] = {0, 0, 0}, nl[3] = {0, 0, 0};
   auto load = [&](int k) {
      const long p = col + nij * (k - b.kb);
#pragma unroll
      for (int c = 0; c < 3; c++) {
         nu[c] = u[p + npts * c];
         nm[c] = um[p + npts * c];
         if (role == 0) {
            np[c] = up[p + npts * c];
            nl[c] = lu[p + npts * c];
         }
      }
      nr = rho[p];
      nj = jac[p];
   };
   load(k0);
   int par = 0;
   for (int k = k0; k <= k1; k++) {
      double d[3], pv[3], lv[3];
#pragma unroll
      for (int c = 0; c < 3; c++) {
         d[c] = nu[c] - nm[c];
         pv[c] = np[c];
         lv[c] = nl[c];
      }
      const double r = nr, rj = nr * nj;
      if (own) {
#pragma unroll
         for (int c = 0; c < 3; c++) sd[par][c * MPL + o] = d[c];
         sr[par][o] = rj;
      }
      __syncthreads();  // plane k is staged; plane k-1 was read from the other half
      if (k < k1) load(k + 1);
      if (active) {
         const double* q = &sr[par][o];
         const double w = beta / rj, sc = c4 / r;
         const double x2 = q[1] * gx[2], x1 = rj * gx[1], x0 = q[-1] * gx[0];
         const double y2 = q[MHX] * gy[2], y1 = rj * gy[1], y0 = q[-MHX] * gy[0];
#pragma unroll
         for (int c = 0; c < 3; c++) {
            const double* e = &sd[par][c * MPL + o];
            const double ax = x2 * (e[2] - 2 * e[1] + d[c]) - 2 * x1 * (e[1] - 2 * d[c] + e[-1]) +
                              x0 * (d[c] - 2 * e[-1] + e[-2]);
            const double ay = y2 * (e[2 * MHX] - 2 * e[MHX] + d[c]) - 2 * y1 * (e[MHX] - 2 * d[c] + e[-MHX]) +
                              y0 * (d[c] - 2 * e[-MHX] + e[-2 * MHX]);
            const double v = pv[c] + sc * lv[c];
            up[col + nij * (k - b.kb) + npts * c] = damped ? v - w * (wx * ax + wy * ay) : v;
         }
      }
      par ^= 1;
   }
}

// ---------------------------------------------------------------------------
// Traction-free ghost points on the curved boundary plane
// ---------------------------------------------------------------------------
// The normal stress on the plane is N (D_r u) + g with N = mu ac I +
// (mu+lambda) v v^T, v = (sqrt(sx/sy) M2, sqrt(sy/sx) M3, M4/sqrt(sx sy)),
// ac = |v|^2, g the tangential part minus the forcing.  D_r u = s0 u_ghost +
// sum_w s_w u_w, so u_ghost = -(sum_w s_w u_w + N^-1 g)/s0 with
// N^-1 = I/(mu ac) - (mu+lambda)/((2mu+lambda) mu ac^2) v v^T.
template <int CO>
__global__ void __launch_bounds__(256)
k_freesurf_curv(Box b, int k, int kl, CurvG<CO> s, const SbpTables* __restrict__ sbp,
                const double* __restrict__ forcing, double* __restrict__ u)
{
   const int i = b.ib + 2 + blockIdx.x * blockDim.x + threadIdx.x;
   const int j = b.jb + 2 + blockIdx.y * blockDim.y + threadIdx.y;
   if (i > b.ie - 2 || j > b.je - 2) return;
   const double sx = s.SX(i), sy = s.SY(j), isx = 1 / sx, isy = 1 / sy;
   double g[3];
   t_terms(s, i, j, k, sx, sy, isx, isy, g);
   if (forcing) {
      const long f = 3 * ((i - b.ib) + b.ni * (j - b.jb));
#pragma unroll
      for (int c = 0; c < 3; c++) g[c] -= forcing[f + c];
   }
   const double m2 = s.M(1, i, j, k), m3 = s.M(2, i, j, k), m4 = s.M(3, i, j, k);
   const double mu = s.MU(i, j, k), la = s.LA(i, j, k);
   const double ac = sx * isy * m2 * m2 + sy * isx * m3 * m3 + m4 * m4 * isy * isx;
   const double bc = 1 / (mu * ac);
   const double cc = (mu + la) / (2 * mu + la) * bc / ac;
   const double xy = sqrt(sx * isy);
   const double v[3] = {xy * m2, m3 / xy, isx * xy * m4};
   const double dc = cc * (v[0] * g[0] + v[1] * g[1] + v[2] * g[2]);
#pragma unroll
   for (int c = 0; c < 3; c++) {
      double acc = 0;
#pragma unroll
      for (int w = 1; w <= 4; w++) acc += sbp->sbop[w] * s.U(c, i, j, k + kl * (w - 1));
      u[vidx<CO>(b, c, i, j, k - kl)] = -(acc + bc * g[c] - dc * v[c]) / sbp->sbop[0];
   }
}

// ---------------------------------------------------------------------------
// Time step of the curvilinear grid (EW::computeDT, EW.C:5063-5136)
// ---------------------------------------------------------------------------
// Per point the symmetric matrix A (EW.C:5089-5102) of the curvilinear
// operator's principal part; the time step follows from its most negative
// eigenvalue: max over points of -lambda_min(A)/(4 rho).  The reference calls
// LAPACK dspev; here the eigenvalue comes from the closed form for symmetric
// 3x3 matrices (O. K. Smith, "Eigenvalues of a symmetric 3x3 matrix",
// Comm. ACM 4(4):168, 1961).
constexpr int CRED = 256;

__device__ __forceinline__ double sym3_min_eig(double a11, double a12, double a13, double a22, double a23,
                                               double a33)
{
   const double p1 = a12 * a12 + a13 * a13 + a23 * a23;
   const double q = (a11 + a22 + a33) / 3;
   if (p1 == 0) return fmin(a11, fmin(a22, a33));
   const double b11 = a11 - q, b22 = a22 - q, b33 = a33 - q;
   const double p2 = b11 * b11 + b22 * b22 + b33 * b33 + 2 * p1;
   const double p = sqrt(p2 / 6);
   const double ip = 1 / p;
   // r = det(B)/2 with B = (A - qI)/p
   const double det = b11 * (b22 * b33 - a23 * a23) - a12 * (a12 * b33 - a23 * a13) + a13 * (a12 * a23 - b22 * a13);
   const double r = fmin(1.0, fmax(-1.0, det * ip * ip * ip / 2));
   const double phi = acos(r) / 3;
   // eigenvalues q + 2p cos(phi + 2 pi m / 3); the smallest is m = 1
   return q + 2 * p * cos(phi + 2.0943951023931954923);
}

template <int CO>
__global__ void __launch_bounds__(CRED)
k_maxeig_curv(Box b, const double* __restrict__ met, const double* __restrict__ jac, const double* __restrict__ mu,
              const double* __restrict__ la, const double* __restrict__ rho, double* __restrict__ partial)
{
   __shared__ double sh[CRED];
   double m = -1;
   for (long p = blockIdx.x * (long)CRED + threadIdx.x; p < b.npts; p += (long)gridDim.x * CRED) {
      const long m0 = CO ? p : 4 * p, ms = CO ? b.npts : 1;
      const double m1 = met[m0], m2 = met[m0 + ms], m3 = met[m0 + 2 * ms], m4 = met[m0 + 3 * ms];
      const double l = la[p], u = mu[p], l2 = l + 2 * u, ji = 1 / jac[p];
      const double s1 = m1 * m1, s2 = m2 * m2, s3 = m3 * m3, s4 = m4 * m4;
      const double a11 = -4 * (s1 * l2 + s1 * u + s2 * l2 + s3 * u + s4 * u) * ji;
      const double a12 = -4 * m2 * m3 * (u + l) * ji;
      const double a13 = -4 * m2 * m4 * (u + l) * ji;
      const double a22 = -4 * (s1 * u + s1 * l2 + s2 * u + s3 * l2 + s4 * u) * ji;
      const double a23 = -4 * m3 * m4 * (u + l) * ji;
      const double a33 = -4 * (s1 * u + s1 * u + s2 * u + s3 * u + s4 * l2) * ji;
      const double w0 = sym3_min_eig(a11, a12, a13, a22, a23, a33);
      m = fmax(m, -w0 / (4 * rho[p]));
   }
   sh[threadIdx.x] = m;
   __syncthreads();
   for (int o = CRED / 2; o > 0; o >>= 1) {
      if ((int)threadIdx.x < o) sh[threadIdx.x] = fmax(sh[threadIdx.x], sh[threadIdx.x + o]);
      __syncthreads();
   }
   if (threadIdx.x == 0) partial[blockIdx.x] = sh[0];
}

__global__ void __launch_bounds__(CRED) k_final_max_curv(int n, const double* __restrict__ partial,
                                                         double* __restrict__ out)
{
   __shared__ double sh[CRED];
   double m = -1;
   for (int q = threadIdx.x; q < n; q += CRED) m = fmax(m, partial[q]);
   sh[threadIdx.x] = m;
   __syncthreads();
   for (int o = CRED / 2; o > 0; o >>= 1) {
      if ((int)threadIdx.x < o) sh[threadIdx.x] = fmax(sh[threadIdx.x], sh[threadIdx.x + o]);
      __syncthreads();
   }
   if (threadIdx.x == 0) out[0] = sh[0];
}

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------
int launch_metric(int co, const Box& b, double h, const double* z, double* met, double* jac, int* bad,
                  hipStream_t s)
{
   const unsigned g = cdiv(b.npts, 256);
   if (co)
      k_metric<1><<<g, 256, 0, s>>>(b, h, z, met, jac, bad);
   else
      k_metric<0><<<g, 256, 0, s>>>(b, h, z, met, jac, bad);
   return check_hip(hipGetLastError(), "metric launch");
}

template <int CO>
static void rhs4curv_co(const Box& b, const int* onesided, const SbpTables* d_sbp, const CurvG<CO>& cg,
                        const double* jac, double* lu, hipStream_t s)
{
   const int ntx = (int)cdiv(b.ie - b.ib - 3, MTX), nty = (int)cdiv(b.je - b.jb - 3, MTY);
   const int top = onesided[4] == 1;
   const int k1 = top ? 7 : b.kb + 2, k2 = b.ke - 2;
   if (top)
      k_rhs4curv_rows<CO><<<dim3(ntx * nty, sbp_rows_spread(ntx * nty, 1)), MNT, 0, s>>>(b, ntx, d_sbp, cg, jac, lu);
   if (k2 >= k1) {
      const int kc = march_kchunk((long)ntx * nty, k2 - k1 + 1, 1);
      const int ntiles = ntx * nty * (int)cdiv(k2 - k1 + 1, kc);
      k_rhs4curv_march<CO><<<8 * cdiv(ntiles, 8), MNT, 0, s>>>(b, ntx, nty, ntiles, k1, k2, kc, cg, jac, lu);
   }
}

int launch_rhs4sgcurv(int co, const Box& b, const int* onesided, const SbpTables* d_sbp, const double* u,
                      const double* mu, const double* la, const double* met, const double* jac, const double* strx,
                      const double* stry, double* lu, hipStream_t s)
{
   if (co)
      rhs4curv_co<1>(b, onesided, d_sbp, CurvG<1>{b, u, mu, la, met, strx, stry}, jac, lu, s);
   else
      rhs4curv_co<0>(b, onesided, d_sbp, CurvG<0>{b, u, mu, la, met, strx, stry}, jac, lu, s);
   return check_hip(hipGetLastError(), "rhs4sgcurv launch");
}

int launch_addsgd4c(int co, const Box& b, double* up, const double* u, const double* um, const double* rho,
                    const double* jac, const SgCoef& sg, double beta, hipStream_t s)
{
   if (beta == 0) return OK;
   const int nii = b.ie - b.ib - 3, njj = b.je - b.jb - 3, nkk = b.ke - b.kb - 3;
   dim3 grd(cdiv(nii, 64), cdiv(njj, 4), nkk), blk(64, 4, 1);
   if (co)
      k_addsgd4c<1><<<grd, blk, 0, s>>>(b, up, u, um, rho, jac, sg, beta);
   else
      k_addsgd4c<0><<<grd, blk, 0, s>>>(b, up, u, um, rho, jac, sg, beta);
   return check_hip(hipGetLastError(), "addsgd4c launch");
}

int launch_curv_pred(const Box& b, const double* lu, const double* u, const double* um, const double* rho, double* up,
                     double* acc, double dt, hipStream_t s)
{
   k_curv_pred<<<cdiv(b.npts, 256), 256, 0, s>>>(b.npts, lu, u, um, rho, up, acc, dt * dt, 1.0 / (dt * dt));
   return check_hip(hipGetLastError(), "curvilinear predictor launch");
}

int launch_curv_corr(const Box& b, int k1, int k2, double* up, const double* lu, const double* u, const double* um,
                     const double* rho, const double* jac, const SgCoef& sg, double beta, double dt, hipStream_t s)
{
   if (k2 < k1) return OK;
   const int ntx = (int)cdiv(b.ie - b.ib - 3, MTX), nty = (int)cdiv(b.je - b.jb - 3, MTY);
   const int kc = march_kchunk((long)ntx * nty, k2 - k1 + 1, 2);
   const int ntiles = ntx * nty * (int)cdiv(k2 - k1 + 1, kc);
   k_curv_corr<<<8 * cdiv(ntiles, 8), MNT, 0, s>>>(b, ntx, nty, ntiles, k1, k2, kc, up, lu, u, um, rho, jac, sg,
                                                   dt * dt * dt * dt / 12, beta);
   return check_hip(hipGetLastError(), "curvilinear corrector launch");
}

int launch_freesurf_curv(int co, const Box& b, int nz, int side, double* u, const double* mu, const double* la,
                         const double* met, const SbpTables* d_sbp, const double* forcing, const double* strx,
                         const double* stry, hipStream_t s)
{
   const int k = side == 4 ? 1 : nz, kl = side == 4 ? 1 : -1;
   const int nii = b.ie - b.ib - 3, njj = b.je - b.jb - 3;
   dim3 grd(cdiv(nii, 64), cdiv(njj, 4), 1), blk(64, 4, 1);
   if (co)
      k_freesurf_curv<1><<<grd, blk, 0, s>>>(b, k, kl, CurvG<1>{b, u, mu, la, met, strx, stry}, d_sbp, forcing, u);
   else
      k_freesurf_curv<0><<<grd, blk, 0, s>>>(b, k, kl, CurvG<0>{b, u, mu, la, met, strx, stry}, d_sbp, forcing, u);
   return check_hip(hipGetLastError(), "curvilinear free-surface launch");
}

template <int CO>
__global__ void k_enforce_cart_topo(Box cart, double* __restrict__ ucart, Box curv, double* __restrict__ ucurv, int g)
{
   const int i = cart.ib + blockIdx.x * blockDim.x + threadIdx.x;
   const int j = cart.jb + blockIdx.y * blockDim.y + threadIdx.y;
   if (i > cart.ie || j > cart.je) return;
   const int kbc = cart.kb, kec = curv.ke;
   for (int c = 0; c < 3; c++) {
      for (int q = 0; q < g; q++) ucart[vidx<CO>(cart, c, i, j, kbc + q)] = ucurv[vidx<CO>(curv, c, i, j, kec - 2 * g + q)];
      for (int q = 0; q <= g; q++) ucurv[vidx<CO>(curv, c, i, j, kec - q)] = ucart[vidx<CO>(cart, c, i, j, kbc + 2 * g - q)];
   }
}

int launch_enforce_cart_topo(int co, const Box& cart, double* ucart, const Box& curv, double* ucurv, int g,
                             hipStream_t s)
{
   const dim3 blk(64, 4, 1), grd(cdiv(cart.ni, 64), cdiv(cart.je - cart.jb + 1, 4), 1);
   if (co)
      k_enforce_cart_topo<1><<<grd, blk, 0, s>>>(cart, ucart, curv, ucurv, g);
   else
      k_enforce_cart_topo<0><<<grd, blk, 0, s>>>(cart, ucart, curv, ucurv, g);
   return check_hip(hipGetLastError(), "grid interface launch");
}

int launch_maxeig_curv(int co, const Box& b, const double* met, const double* jac, const double* mu, const double* la,
                       const double* rho, double* partial, int npartial, double* out, hipStream_t s)
{
   if (co)
      k_maxeig_curv<1><<<npartial, CRED, 0, s>>>(b, met, jac, mu, la, rho, partial);
   else
      k_maxeig_curv<0><<<npartial, CRED, 0, s>>>(b, met, jac, mu, la, rho, partial);
   k_final_max_curv<<<1, CRED, 0, s>>>(npartial, partial, out);
   return check_hip(hipGetLastError(), "curvilinear maxeig launch");
}

}  // namespace sw4amd
