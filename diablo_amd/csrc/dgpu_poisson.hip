// dgpu_poisson.hip -- POISSON_P_CHAN (for/channel.f:1217-1453) on the device.
//
// CP from CU1-3 (and CTH): the right-hand side sum_ij (du_i/dx_j)(du_j/dx_i)
// in physical space from the velocity and its x and z gradients on pair planes
// (dgpu_pairs.hip; the y differences of the reference's spectral inputs are
// taken on the physical planes, which is the same by linearity), then one
// tridiagonal solve per (kx,kz) mode.  The reference transforms each of its
// six products back; here they are summed first and two planes' sums share one
// complex x transform: nine inverse real transforms and one forward a plane.
// 192x129x192: 1031 -> 404 us for the whole call, of which the solve 179 -> 48.
// The solve rows that are read (1..NY) carry the same matrix as REM_DIV_CHAN's
// (for/channel.f:1126-1143 vs 1399-1440, boundary rows for/mpi.f:1293-1369),
// so the context's precomputed Poisson factorisation is reused.
#include "dgpu_kernels.hpp"

namespace dgpu {

// pairs: 0 (U1, U2), 1 (U3, dU1/dx), 2 (dU2/dx, dU3/dx), 3 (dU1/dz, dU2/dz),
// 4 (dU3/dz, -).  out plane q: the right-hand sides of rows 2 + 2q and 3 + 2q
// (0 beyond NY), q = qlo..qhi-1.  A thread owns one position and a chunk of plane
// pairs; the planes it has read roll through its registers.
__global__ void __launch_bounds__(256) k_pp_rhs(Geo g, PairDst pr, cx<double> *__restrict__ out,
                                                const double *__restrict__ dyf, int qlo, int qhi, int chunk)
{
    const long n = (long)g.nx * g.nz;
    const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= n) return;
    const int NY = g.ny, q0 = qlo + blockIdx.y * chunk, q1 = min(q0 + chunk, qhi);
    auto at = [&](int q, int j) { return pr.p[q][(long)min(j, NY + 1) * n + e]; };
    const int j0 = 2 + 2 * q0;
    double um = at(0, j0 - 1).re, wm = at(1, j0 - 1).re;
    cx<double> a = at(0, j0), b = at(1, j0), c = at(2, j0), d = at(3, j0), f = at(4, j0);
    for (int q = q0; q < q1; ++q) {
        double r[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int j = 2 + 2 * q + h;
            const cx<double> ap = at(0, j + 1), bp = at(1, j + 1), cp = at(2, j + 1), dp = at(3, j + 1),
                             fp = at(4, j + 1);
            const double i1 = 1.0 / dyf[min(j, NY + 1)], i2 = 0.5 * i1;
            const double vy = (ap.im - a.im) * i1, uy = (ap.re - um) * i2, wy = (bp.re - wm) * i2;
            const double vx = 0.5 * (c.re + cp.re), vz = 0.5 * (d.im + dp.im);
            r[h] = j <= NY ? b.im * b.im + vy * vy + f.re * f.re + 2.0 * uy * vx + 2.0 * wy * vz + 2.0 * d.re * c.im
                           : 0.0;
            um = a.re;
            wm = b.re;
            a = ap; b = bp; c = cp; d = dp; f = fp;
        }
        out[(long)q * n + e] = make_cx(r[0], r[1]);
    }
}

void launch_pp_rhs(hipStream_t s, const Geo &g, const PairDst &pr, cx<double> *out, const double *dyf, int qlo,
                   int qhi)
{
    const long n = (long)g.nx * g.nz;
    const int chunk = 8;  // 16 planes: one in nine read twice
    hipLaunchKernelGGL(k_pp_rhs, dim3((unsigned)((n + 255) / 256), (qhi - qlo + chunk - 1) / chunk), dim3(256), 0, s, g,
                       pr, out, dyf, qlo, qhi, chunk);
}

// Buoyancy term, the tridiagonal solve and CP (for/channel.f:1373-1449).  The
// elimination is two linear recurrences over the rows, g(j) = r(j) + m(j)
// g(j-1) and phi(j) = (g(j) - U(j) phi(j+1)) / B(j); a column is cut into 16
// segments run side by side from zero and then again from their carries, which
// pass from segment to segment through LDS (one thread a column took 179 us at
// 192x129x192: 131 waves, 258 dependent rows).  16 modes (256 B of a row) x 16
// segments a block.
__global__ void __launch_bounds__(256) k_pp_solve(Geo g, const cx<double> *__restrict__ cs,
                                                  const cx<double> *__restrict__ cth, double ri,
                                                  const double *__restrict__ gyf, const double *__restrict__ pmult,
                                                  const double *__restrict__ pinv, const double *__restrict__ rd,
                                                  cx<double> *__restrict__ scr, cx<double> *__restrict__ cp)
{
    __shared__ cx<double> end[16][16];
    __shared__ double prod[16][16];
    const int lm = threadIdx.x & 15, seg = threadIdx.x >> 4;
    const long mode = (long)blockIdx.x * 16 + lm;
    const bool on = mode < g.ps;
    const long m = on ? mode : g.ps - 1;
    const bool is00 = m == 0;
    const int NY = g.ny, len = (NY + 15) / 16, a = 1 + seg * len, b = min(NY, a + len - 1);
    const long ps = g.ps;
    const cx<double> zero = make_cx(0.0, 0.0);
    auto row = [&](int j, cx<double> gp) {  // forward recurrence
        const long o = m + (long)j * ps;
        if (j == 1) return zero;
        cx<double> v = zero;
        if (j < NY) {
            cx<double> s = cs[o];
            if (cth && !is00) {
                const cx<double> d = cth[o + ps] - cth[o - ps];
                const double den = gyf[j + 1] - gyf[j - 1];
                s = s + make_cx((ri * d.re) / den, (ri * d.im) / den);
            }
            v = make_cx(-s.re, -s.im);
        }
        const double mu = pmult[o];
        return make_cx(v.re + mu * gp.re, v.im + mu * gp.im);
    };
    cx<double> x = zero;
    double pr = 1.0;
    for (int j = a; j <= b; ++j) {
        x = row(j, x);
        pr = j == 1 ? 0.0 : pr * pmult[m + (long)j * ps];
    }
    end[seg][lm] = x;
    prod[seg][lm] = pr;
    __syncthreads();
    x = zero;
    for (int s = 0; s < seg; ++s) {
        const cx<double> t = end[s][lm];
        const double p = prod[s][lm];
        x = make_cx(t.re + p * x.re, t.im + p * x.im);
    }
    for (int j = a; j <= b; ++j) {
        x = row(j, x);
        if (on) scr[m + (long)j * ps] = x;
    }
    __syncthreads();
    // back substitution; the last row takes no row above
    auto back = [&](int j, cx<double> xp, double &w) {
        const long o = m + (long)j * ps;
        const cx<double> gj = scr[o];
        const double ip = pinv[o], U = j == NY ? 0.0 : (j == 1 ? (is00 ? 0.0 : -1.0) : rd[(long)j * 4]);
        w = -U * ip;
        return make_cx((gj.re - U * xp.re) * ip, (gj.im - U * xp.im) * ip);
    };
    x = zero;
    pr = 1.0;
    for (int j = b; j >= a; --j) {
        double w;
        x = back(j, x, w);
        pr *= w;
    }
    end[seg][lm] = x;
    prod[seg][lm] = pr;
    __syncthreads();
    x = zero;
    for (int s = 15; s > seg; --s) {
        const cx<double> t = end[s][lm];
        const double p = prod[s][lm];
        x = make_cx(t.re + p * x.re, t.im + p * x.im);
    }
    for (int j = b; j >= a; --j) {
        double w;
        x = back(j, x, w);
        if (on) cp[m + (long)j * ps] = x;
    }
}

void launch_pp_solve(hipStream_t s, const Geo &g, const cx<double> *cs, const cx<double> *cth, double ri,
                     const double *gyf, const double *pmult, const double *pinv, const double *rd, cx<double> *scr,
                     cx<double> *cp)
{
    hipLaunchKernelGGL(k_pp_solve, dim3((unsigned)((g.ps + 15) / 16)), dim3(256), 0, s, g, cs, cth, ri, gyf, pmult,
                       pinv, rd, scr, cp);
}

}  // namespace dgpu
