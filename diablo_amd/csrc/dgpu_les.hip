// dgpu_les.hip -- les_chan's constant Smagorinsky model (for/les.f:1-331) and
// RK_CHAN_1's LES terms on the device, in FP64, on the pair planes of
// dgpu_pairs.hip (P[j][zp][slot], two real fields a pair):
//
//   pair 0 (U1, U2)            pair 3 (dU1/dz + dU3/dx, dU3/dz)
//   pair 1 (U3, TH)            pair 4 (dU2/dz, dTH/dx)
//   pair 2 (dU1/dx, dU2/dx)    pair 5 (dTH/dz, -)
//
//   k_les_bc       APPLY_BC_LES (for/les.f:805-864) on the kept modes
//   k_les_bc_rows  APPLY_BC_VEL_PHYS (for/channel.f:2495-2640) of the wall rows
//   k_les_prod     S_ij, |S| on GYF and GY, NU_T, tau_ij (for/les.f:107-301,
//                  526-571), the explicit cross terms (for/les.f:302-331), the
//                  scalar's eddy flux (for/channel.f:313-375) and the eleven
//                  products of RK_CHAN_1, summed before one x forward
//   k_les_cn       the Crank-Nicolson solves in physical space
//
// tau_ij, the cross terms and the eddy flux enter CF1-3 and CFTH through the
// same i kx, i kz and d/dy as the products they sit beside, so they are added
// to the products in physical space and cost no transforms of their own (the
// transforms are linear: the sum differs by round-off only).
#include "dgpu_hot.hpp"

#include <algorithm>
#include <cmath>

namespace dgpu {

namespace {

__device__ __forceinline__ double sq(double x) { return x * x; }

}  // namespace

__global__ void k_les_bc(Geo g, cx<double> *__restrict__ cu1, cx<double> *__restrict__ cu3, int u_min, int u_max,
                         int w_min, int w_max)
{
    const long m = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (m >= g.ps) return;
    const int NY = g.ny;
    const long ps = g.ps;
    auto top = [&](cx<double> *a) {
        a[m + (long)NY * ps] = a[m + (long)(NY - 1) * ps];
        a[m + (long)(NY + 1) * ps] = a[m + (long)NY * ps];
    };
    auto bottom = [&](cx<double> *a) {
        a[m + ps] = a[m + 2 * ps];
        a[m] = a[m + ps];
    };
    if (u_max == 1) top(cu1);
    if (w_max == 1) top(cu3);
    if (u_min == 1) bottom(cu1);
    if (w_min == 1) bottom(cu3);
}

// APPLY_BC_VEL_PHYS_LOWER / _UPPER (for/channel.f:2495-2640) stated on the
// kept modes: a value C in physical space is C on the (0,0) mode and 0 on
// the others, and the Neumann rows are linear in the field.
__global__ void k_les_bc_phys(Geo g, cx<double> *__restrict__ cu1, cx<double> *__restrict__ cu2,
                              cx<double> *__restrict__ cu3, LesBc b, const double *__restrict__ dy,
                              const double *__restrict__ dyf)
{
    const long m = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (m >= g.ps) return;
    const int NY = g.ny;
    const long ps = g.ps;
    const double on = (m == 0) ? 1.0 : 0.0;
    auto R = [&](cx<double> *a, int j) -> cx<double> & { return a[m + (long)j * ps]; };
    auto cst = [&](double c) { return make_cx<double>(on * c, 0.0); };
    auto plus = [&](cx<double> a, double c) { return make_cx<double>(a.re + on * c, a.im); };
    for (int q = 0; q < 2; ++q) {
        cx<double> *u = q == 0 ? cu1 : cu3;
        const int lo = q == 0 ? b.u_lo : b.w_lo, hi = q == 0 ? b.u_hi : b.w_hi;
        const double clo = q == 0 ? b.u_lo_c : b.w_lo_c, chi = q == 0 ? b.u_hi_c : b.w_hi_c;
        if (lo == 0) {
            R(u, 0) = cst(clo);
            R(u, 1) = cst(clo);
        } else {
            R(u, 1) = plus(R(u, 2), -dy[2] * clo);
            R(u, 0) = plus(R(u, 1), -dy[1] * clo);
        }
        if (hi == 0) {
            R(u, NY) = cst(chi);
            R(u, NY + 1) = cst(chi);
        } else {
            R(u, NY) = plus(R(u, NY - 1), dy[NY] * chi);
            R(u, NY + 1) = plus(R(u, NY), dy[NY] * chi);
        }
    }
    if (b.v_lo == 0) {
        const cx<double> u2 = R(cu2, 2);
        R(cu2, 1) = make_cx<double>(2.0 * on * b.v_lo_c - u2.re, -u2.im);
        R(cu2, 0) = R(cu2, 1);
    } else {
        R(cu2, 1) = plus(R(cu2, 2), -dyf[1] * b.v_lo_c);
        R(cu2, 0) = plus(R(cu2, 1), -dyf[1] * b.v_lo_c);
    }
    if (b.v_hi == 0) {
        const cx<double> u2 = R(cu2, NY);
        R(cu2, NY + 1) = make_cx<double>(2.0 * on * b.v_hi_c - u2.re, -u2.im);
    } else {
        R(cu2, NY + 1) = plus(R(cu2, NY), dy[NY] * b.v_hi_c);
    }
}

// Rows 0, 1, NY, NY+1 of pairs 0 and 1 after APPLY_BC_VEL_PHYS_LOWER / _UPPER
// (for/channel.f:2495-2640), into bc[pair][4][NZ*NX]; TH and U2(NY) unchanged.
__global__ void k_les_bc_rows(Geo g, const cx<double> *__restrict__ p0, const cx<double> *__restrict__ p1,
                              cx<double> *__restrict__ bc, LesBc b, const double *__restrict__ dy,
                              const double *__restrict__ dyf)
{
    const long n = (long)g.nx * g.nz;
    const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= n) return;
    const int NY = g.ny;
    auto A = [&](const cx<double> *p, int j) { return p[(long)j * n + e]; };
    const cx<double> r0[4] = {A(p0, 0), A(p0, 1), A(p0, NY), A(p0, NY + 1)};
    const cx<double> r1[4] = {A(p1, 0), A(p1, 1), A(p1, NY), A(p1, NY + 1)};
    const cx<double> a2 = A(p0, 2), an = A(p0, NY - 1), b2 = A(p1, 2), bn = A(p1, NY - 1);
    auto horiz = [&](int lo, int hi, double clo, double chi, double u2, double un, double *o) {
        o[1] = lo == 0 ? clo : u2 - dy[2] * clo;
        o[0] = lo == 0 ? clo : o[1] - dy[1] * clo;
        o[2] = hi == 0 ? chi : un + dy[NY] * chi;
        o[3] = hi == 0 ? chi : o[2] + dy[NY] * chi;
    };
    double u[4], w[4], v[4];
    horiz(b.u_lo, b.u_hi, b.u_lo_c, b.u_hi_c, a2.re, an.re, u);
    horiz(b.w_lo, b.w_hi, b.w_lo_c, b.w_hi_c, b2.re, bn.re, w);
    v[1] = b.v_lo == 0 ? 2.0 * b.v_lo_c - a2.im : a2.im - dyf[1] * b.v_lo_c;
    v[0] = b.v_lo == 0 ? v[1] : v[1] - dyf[1] * b.v_lo_c;
    v[2] = r0[2].im;
    v[3] = b.v_hi == 0 ? 2.0 * b.v_hi_c - v[2] : v[2] + dy[NY] * b.v_hi_c;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        bc[r * n + e] = make_cx(u[r], v[r]);
        bc[(4 + r) * n + e] = make_cx(w[r], r1[r].im);
    }
}

// The rows of k_les_bc_rows back into the pairs (the fields the solves take).
__global__ void k_les_bc_put(Geo g, cx<double> *__restrict__ p0, cx<double> *__restrict__ p1,
                             const cx<double> *__restrict__ bc)
{
    const long n = (long)g.nx * g.nz;
    const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= n) return;
    const int r = blockIdx.y & 3, j = r < 2 ? r : g.ny - 2 + r;
    cx<double> *p = blockIdx.y < 4 ? p0 : p1;
    p[(long)j * n + e] = bc[(long)blockIdx.y * n + e];
}

// -------------------------------------------------------------------------
// k_les_prod: zr z rows per block, planes ja..jb (a chunk of the sweep).  A
// thread owns NP positions of the rows for the whole sweep and keeps what the
// stencils need of the plane before in registers, so every pair value is read
// from HBM once; the products of plane j = m - 1 (m the newest plane) go to
// LDS and NPO rows of T threads run their x forward while the next plane's
// values are on their way.  tab[j*8 + {0..6}]: 1/DYF, 1/DY, 1/(2 DYF),
// DYF(j-1)/(2 DY), DYF(j)/(2 DY), -2 C^2 DELTA^2 on GYF, on GY.
// force: the SGS force alone (dgpu_les_chan), no products and no scalar.
// 384x257x384: 1.90-1.95 ms (counted 3.7 GB read, 1.9 written: six pairs in, NU_T
// and eight row fields out, 2.9 TB/s; three waves per SIMD; 2.29 ms with two
// positions a thread, 256 registers and 44 of them spilled); it replaces the x
// kernel (1.30 ms), nine plane transforms (2.9 ms) and seven pointwise kernels
// (2.9 ms) of the Fortran-layout form, a substep of 18.1 ms, now 8.1.
// -------------------------------------------------------------------------
constexpr int kStash = 8;
template <int E, int NTH, int PID, int LM, bool WIDE>
__global__ void __launch_bounds__(WIDE ? 768 : 384) __attribute__((amdgpu_waves_per_eu(3))) k_les_prod(IpLen frt, const cx<double> *__restrict__ twg, int mk_rt, int ld,
                                                  LesProd a)
{
    constexpr int npo = XCount<NTH>::npo, NP = (E + LM * npo - 1) / (LM * npo);
    const IpLen &fx = plan_ref<PID>(frt);
    extern __shared__ unsigned char smem_raw[];
    cx<double> *const fb = reinterpret_cast<cx<double> *>(smem_raw);
    const int nx = fx.n, TT = fx.t, S = fx.nstages, NY = a.ny;
    const int mk = PID != 0 ? nx / 3 + 1 : mk_rt;
    const int tid = threadIdx.x, nthr = blockDim.x, zr = a.zr;
    // the first zr * npo * T threads run the transforms
    const int pg = tid / TT, zs = pg / npo, p = pg - zs * npo;
    const bool tr = zs < zr;
    int th = tid - pg * TT;
    cx<double> *tw = fb + (long)zr * npo * nx;
    double *kxs = reinterpret_cast<double *>(tw + fx.twn);
    // row m's products and fluxes wait here for the next plane (kStash values a
    // position, each lane its own): in registers they spilled, 2.2 GB of scratch
    // traffic a launch
    double *stash = kxs + mk + tid;
    for (int e = tid; e < fx.twn; e += nthr) tw[e] = twg[e];
    for (int e = tid; e < mk; e += nthr) kxs[e] = a.kx[e];
    const int zi = blockIdx.x * zr + zs;
    const bool zvalid = zi < a.nz;
    const int ja = a.jlo + blockIdx.y * a.chunk, jb = min(a.jhi, ja + a.chunk - 1);
    const long pp = (long)a.nz * nx;
    // this thread's positions: offset in a pair plane, LDS slot of product row 0
    int off[NP], ls[NP];
    bool on[NP];
#pragma unroll
    for (int k = 0; k < NP; ++k) {
        const int e0 = tid + nthr * k;
        const bool in = e0 < zr * nx;
        const int e = in ? e0 : 0, zq = e / nx, slot = e - zq * nx, zp = blockIdx.x * zr + zq;
        on[k] = in && zp < a.nz;
        off[k] = min(zp, a.nz - 1) * nx + slot;
        const int R = fx.radix[S - 1], idx = slot / TT, u = idx / R;
        const int pos = (slot - idx * TT + TT * u) * R + (idx - u * R);
        ls[k] = in ? zq * npo * nx + ip_swz(fx, pos) : -1;
    }
    struct Keep {
        double pu, pv, pw, pt, su, sw, s11, s13, s33, s22, s12, s23, t12, t23;
    } K[NP];
    enum { Q_P3, Q_P4, Q_F1, Q_F3, Q_FT, Q_Q, Q_X8, Q_X9 };
    double own[WIDE ? NP : 1][kStash];  // rows of more than 384 threads have no LDS left for it
    auto Q = [&](int k, int q) -> double & {
        if constexpr (WIDE) return own[k][q];
        else return stash[(k * kStash + q) * nthr];
    };
    cx<double> c0[NP], c1[NP], c2[NP], c3[NP], c4[NP], c5[NP], n0[NP];
    auto load = [&](int plane) {
#pragma unroll
        for (int k = 0; k < NP; ++k) {
            const long o = plane * pp + off[k];
            c1[k] = a.pr[1][o];
            c2[k] = a.pr[2][o];
            c3[k] = a.pr[3][o];
            c4[k] = a.pr[4][o];
            if constexpr (NTH > 0) c5[k] = a.pr[5][o];
        }
    };
    auto load0 = [&](int plane) {
#pragma unroll
        for (int k = 0; k < NP; ++k) n0[k] = a.pr[0][min(plane, NY + 1) * pp + off[k]];
    };
    load0(ja - 1);
    load(ja - 1);
#pragma unroll
    for (int k = 0; k < NP; ++k) {
        c0[k] = n0[k];
        K[k] = Keep{};
        K[k].su = c0[k].re;
        K[k].sw = c1[k].re;
    }
    load0(ja);
    auto ub = [&](int j) { return a.cu1[(long)j * a.ps].re; };
    auto wb = [&](int j) { return a.cu3[(long)j * a.ps].re; };
    const bool wave_rows = (64 % TT) == 0;
    auto row_sync = [&]() {
        if (wave_rows) wave_lds_sync();
        else __syncthreads();
    };
    double dub_j = 0.0, dwb_j = 0.0;
    if (ja >= 2) {
        dub_j = 0.5 * (ub(ja - 1) - ub(ja - 2)) * a.tab[(ja - 1) * 8 + 1];
        dwb_j = 0.5 * (wb(ja - 1) - wb(ja - 2)) * a.tab[(ja - 1) * 8 + 1];
    }
    for (int m = ja - 1; m <= jb + 1; ++m) {
        const int j = m - 1;
        const bool out = j >= ja;
        const double *T = a.tab + m * 8, *Tj = a.tab + max(j, 0) * 8;
        const double rdy = T[1], w0 = T[3], w1 = T[4], dG = T[6];
        const bool gy = m >= 2 && m <= NY, has_nut = m >= 3 && m <= NY - 1;
        const bool stress = j >= 2 && j <= NY - 1;
        const int br = m <= 1 ? m : (m >= NY ? m - NY + 2 : -1);
        double dub = dub_j, dwb = dwb_j;  // m = ja - 1: kept above
        if (m >= ja && m >= 1) {
            dub = 0.5 * (ub(m) - ub(m - 1)) * rdy;
            dwb = 0.5 * (wb(m) - wb(m - 1)) * rdy;
        }
#pragma unroll
        for (int k = 0; k < NP; ++k) {
            Keep &P = K[k];
            const double Us = c0[k].re, Vs = c0[k].im, Ws = c1[k].re, th0 = c1[k].im;
            double u = Us, v = Vs, w = Ws, t = th0;
            if (br >= 0) {
                const cx<double> x = a.bc[br * pp + off[k]], y = a.bc[(4 + br) * pp + off[k]];
                u = x.re;
                v = x.im;
                w = y.re;
            }
            if (a.force) u = v = w = t = 0.0;
            const double s11 = c2[k].re, s33 = c3[k].im, s13 = 0.5 * c3[k].re;
            const double s22 = (n0[k].im - Vs) * T[0];
            const double dU = (Us - P.su) * rdy, dW = (Ws - P.sw) * rdy;
            const double s12 = 0.5 * (dU + c2[k].im), s23 = 0.5 * (c4[k].re + dW);
            double t12 = 0.0, t23 = 0.0, nut = 0.0;
            if (gy) {
                const double S = sqrt(2.0 * sq(s11 * w0 + P.s11 * w1) + 4.0 * sq(s12 - dub) +
                                      4.0 * sq(s13 * w0 + P.s13 * w1) + 2.0 * sq(s22 * w0 + P.s22 * w1) +
                                      4.0 * sq(s23 - dwb) + 2.0 * sq(s33 * w0 + P.s33 * w1));
                t12 = dG * (S * (s12 - 0.5 * dU));
                t23 = dG * (S * (s23 - 0.5 * dW));
                if (has_nut) nut = -0.5 * dG * S;
            }
            // at GY row m
            const double p3 = (w1 * u + w0 * P.pu) * v + t12 - nut * dU;
            const double p4 = (w1 * w + w0 * P.pw) * v + t23 - nut * dW;
            const double f1 = (u + P.pu) * v, f3 = (w + P.pw) * v, ft = (t + P.pt) * v;
            const double q = 0.25 * sq(v + P.pv);
            if (out) {  // the products of plane j
                double x1 = P.pu * P.pu, x0 = P.pw * P.pu, x2 = P.pw * P.pw;
                double x5 = (f1 - Q(k, Q_F1)) * Tj[2], x6 = (f3 - Q(k, Q_F3)) * Tj[2];
                if (stress) {
                    const double S = sqrt(2.0 * sq(P.s11) + 4.0 * sq(0.5 * (s12 + P.s12) - dub_j - dub) +
                                          4.0 * sq(P.s13) + 2.0 * sq(P.s22) +
                                          4.0 * sq(0.5 * (s23 + P.s23) - dwb_j - dwb) + 2.0 * sq(P.s33));
                    const double A = Tj[5] * S;
                    x1 += A * P.s11;
                    x0 += A * P.s13;
                    x2 += A * P.s33;
                    x5 += (t12 - P.t12) * Tj[0];
                    x6 += (t23 - P.t23) * Tj[0];
                }
                if (ls[k] >= 0) {
                    cx<double> *f = fb + ls[k];
                    f[0 * nx] = make_cx(x1, x5);
                    f[1 * nx] = make_cx(Q(k, Q_P3), (q - Q(k, Q_Q)) * Tj[1]);
                    f[2 * nx] = make_cx(x0, x6);
                    f[3 * nx] = make_cx(Q(k, Q_P4), x2);
                    if constexpr (NTH > 0) {
                        f[4 * nx] = make_cx(Q(k, Q_X8), (ft - Q(k, Q_FT)) * Tj[2]);
                        f[5 * nx] = make_cx(Q(k, Q_X9), 0.0);
                    }
                }
            }
            P.pu = u; P.pv = v; P.pw = w; P.pt = t;
            P.su = Us; P.sw = Ws;
            P.s11 = s11; P.s13 = s13; P.s33 = s33; P.s22 = s22; P.s12 = s12; P.s23 = s23;
            P.t12 = t12; P.t23 = t23;
            if (on[k] && m >= ja && m <= jb) a.nut[m * pp + off[k]] = nut;
            Q(k, Q_P3) = p3;
            Q(k, Q_P4) = p4;
            Q(k, Q_F1) = f1;
            Q(k, Q_F3) = f3;
            Q(k, Q_Q) = q;
            if constexpr (NTH > 0) {
                Q(k, Q_FT) = ft;
                Q(k, Q_X8) = t * u - nut * c4[k].im;
                Q(k, Q_X9) = t * w - nut * c5[k].re;
            }
        }
        dub_j = dub;
        dwb_j = dwb;
        __syncthreads();
        if (m <= jb) {
#pragma unroll
            for (int k = 0; k < NP; ++k) c0[k] = n0[k];
            load0(m + 2);
            load(m + 1);
        }
        if (out) {
            asm volatile("" : "+v"(th));  // keeps the stages' index arithmetic out of the sweep's registers
            __builtin_assume(th >= 0 && th < TT);
            cx<double> *row = fb + (tr ? (long)zs * npo + p : 0) * nx;
            stage_loop<PID != 0>(0, S - 1, [&](int s) {
                if (tr) ip_stage_row<double, E, -1, false, PID != 0>(row, fx, S - 1 - s, tw, th);
                row_sync();
            });
            cx<double> *o0 = a.wt + ((long)j * a.nz + min(zi, a.nz - 1)) * ld;
            const long wf = a.wt_fs;
            const double h = 0.5 / nx;
            if (tr && zvalid) x_split<double, E>(fx, row, tw, th, mk, [&](int kp, cx<double> Zk, cx<double> Zn) {
                const cx<double> Xa = make_cx((Zk.re + Zn.re) * h, (Zk.im - Zn.im) * h);
                const cx<double> Xb = make_cx((Zk.im + Zn.im) * h, -(Zk.re - Zn.re) * h);
                const double kx = kxs[kp];
                const cx<double> G = make_cx(kx * Xa.im - Xb.re, -kx * Xa.re - Xb.im);  // -(i kx Xa + Xb)
                const cx<double> nXa = make_cx(-Xa.re, -Xa.im), nXb = make_cx(-Xb.re, -Xb.im);
                switch (p) {  // the outputs of k_xfused_ip's product rows
                case 0: o0[0 * wf + kp] = G; break;
                case 1: o0[2 * wf + kp] = G; break;
                case 2: o0[4 * wf + kp] = G; o0[1 * wf + kp] = nXa; break;
                case 3: o0[3 * wf + kp] = nXa; o0[5 * wf + kp] = nXb; break;
                case 4: o0[6 * wf + kp] = G; break;
                default: o0[7 * wf + kp] = nXa; break;
                }
            });
        }
        __syncthreads();
    }
}

// pick: nothing is launched, *pick receives the rule's planes per block (the x
// kernel's, dgpu_hot_x.hip: this kernel's blocks run c + 2 iterations, and the
// rule's shape is within 4 % of the best of 1, 2, 3, 4, 5, 6, 8, 11, 16, 22, 32, 43,
// 64 and 129 planes, whole LES steps at eleven sizes from 32x33x32 to 384x257x384).
// LM: threads a position is shared out over, in units of the transforms' own
// (2: one position a thread up to 12 values a transform thread).  WIDE: rows of
// more than 384 threads (NX above 512 or so), one unit.
template <int E, int NTH, int PID, int LM = (E > XCount<NTH>::npo ? 2 : 1), bool WIDE = false>
static void les_prod_e(hipStream_t s, const Geo &g, const IpLen &fx, const cx<double> *tw, int ld, LesProd a,
                       int *pick)
{
    constexpr int npo = XCount<NTH>::npo;
    if constexpr (!WIDE && PID == 0)
        if (LM * npo * fx.t > 384) return les_prod_e<E, NTH, PID, 1, true>(s, g, fx, tw, ld, a, pick);
    // short rows are packed as in the fused x kernel
    const size_t stash =  // a z row's
        WIDE ? 0 : sizeof(double) * kStash * ((E + LM * npo - 1) / (LM * npo)) * LM * npo * fx.t;
    const size_t row = sizeof(cx<double>) * (size_t)fx.n * npo + stash;
    const size_t fixed = sizeof(cx<double>) * fx.twn + sizeof(double) * g.mk;
    a.zr = 1;
    while (2 * a.zr * LM * npo * fx.t <= 384 && 2 * a.zr <= g.nz && fixed + 2 * a.zr * row <= 64 * 1024) a.zr *= 2;
    const int threads = a.zr * LM * npo * fx.t;
    const size_t lds = fixed + a.zr * row;
    if (lds > 64 * 1024)
        (void)hipFuncSetAttribute(reinterpret_cast<const void *>(&k_les_prod<E, NTH, PID, LM, WIDE>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    const long rows = (g.nz + a.zr - 1) / a.zr;
    if (pick) {
        const int planes = a.jhi - a.jlo + 1;
        *pick = sweep_rule(rows, &planes, 1, kernel_slots(&k_les_prod<E, NTH, PID, LM, WIDE>, threads, lds));
        return;
    }
    const int nchunks = (a.jhi - a.jlo + a.chunk) / a.chunk;
    hipLaunchKernelGGL((k_les_prod<E, NTH, PID, LM, WIDE>), dim3((unsigned)rows, nchunks), dim3(threads), lds, s, fx, tw, g.mk,
                       ld, a);
}

static void les_prod_any(hipStream_t s, const Geo &g, const IpLen &fx, const cx<double> *tw, int ld,
                         const LesProd &a, int *pick)
{
    if (g.nth == 1 && with_pid(const_plan_id(fx), XPids64{}, [&](auto pc) {
            constexpr int P = decltype(pc)::value;
            les_prod_e<kConstPlanSpecs[P].e, 1, P>(s, g, fx, tw, ld, a, pick);
        }))
        return;
    if (g.nth == 0) {
        DGPU_DISPATCH_XE64(fx.e, (les_prod_e<EE, 0, 0>(s, g, fx, tw, ld, a, pick)));
    } else {
        DGPU_DISPATCH_XE64(fx.e, (les_prod_e<EE, 1, 0>(s, g, fx, tw, ld, a, pick)));
    }
}

void launch_les_prod(hipStream_t s, const Geo &g, const IpLen &fx, const cx<double> *tw, int ld, const LesProd &a)
{
    les_prod_any(s, g, fx, tw, ld, a, nullptr);
}

int les_prod_auto_chunk(const Geo &g, const IpLen &fx, int jlo, int jhi)
{
    LesProd a{};
    a.jlo = jlo;
    a.jhi = jhi;
    int c = 0;
    les_prod_any(nullptr, g, fx, nullptr, 0, a, &c);
    return c > 0 ? c : jhi - jlo + 1;
}

// CF1-3 (rows 2..NY) += the SGS force in the nonlinear-term slots x, y, z.
__global__ void k_les_addcf(Geo g, cx<double> *__restrict__ cf, const cx<double> *__restrict__ f)
{
    const long m = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (m >= g.ps) return;
    const long o = m + (long)(2 + blockIdx.y) * g.ps;
    const cx<double> a = cf[o], b = f[o];
    cf[o] = make_cx(a.re + b.re, a.im + b.im);
}

void launch_les_addcf(hipStream_t s, const Geo &g, cx<double> *cf, const cx<double> *f)
{
    hipLaunchKernelGGL(k_les_addcf, dim3((unsigned)((g.ps + 255) / 256), g.ny - 1), dim3(256), 0, s, g, cf, f);
}

// NU_T of pair planes as a Fortran-layout field, pads and rows outside 0..NX-1,
// 0..NZ-1 zero.  zpos, slot: pair_zpos and pair_slot of every z and x.
__global__ void k_les_nut_out(Geo g, const double *__restrict__ nut, const int *__restrict__ zpos,
                              const int *__restrict__ slot, double *__restrict__ fort)
{
    const long plane = (long)(g.nx + 2) * (g.nz + 2);
    const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= plane) return;
    const int k = (int)(e / (g.nx + 2)), i = (int)(e - (long)k * (g.nx + 2)), j = blockIdx.y;
    fort[j * plane + e] =
        (k < g.nz && i < g.nx) ? nut[((long)j * g.nz + zpos[k]) * g.nx + slot[i]] : 0.0;
}

void launch_les_nut_out(hipStream_t s, const Geo &g, const double *nut, const int *zpos, const int *slot, double *fort)
{
    const long plane = (long)(g.nx + 2) * (g.nz + 2);
    hipLaunchKernelGGL(k_les_nut_out, dim3((unsigned)((plane + 255) / 256), g.ny + 2), dim3(256), 0, s, g, nut, zpos,
                       slot, fort);
}

// One Crank-Nicolson row of one system (for/channel.f:762-1029 with the LES
// terms): rows jlo..jhi from the molecular and eddy parts, the boundary rows
// of APPLY_BC_*_LOWER/UPPER (for/channel.f:1660-2282).  n0, np, nm: NU_T at
// rows j, j+1, j-1; u0, up, um the field, whose explicit eddy-viscosity half
// temp2 d/dy(nut du/dy) (for/channel.f:628-659, 748-760) joins the right-hand
// side r: on GYF rows with NU_T on the faces (U1, U3, TH), or on GY rows with
// NU_T averaged onto the GYF faces (U2).
// w: the row's metric weights (launch_les_cn).
__device__ __forceinline__ void les_row(const LesCn &a, int j, const double *__restrict__ w,
                                        const double *__restrict__ dy, const double *__restrict__ dyf, double n0, double np, double nm, double u0,
                                        double up, double um, double r, double &L, double &D, double &U, double &V)
{
    const int NY = a.ny;
    L = 0.0; D = 1.0; U = 0.0; V = 0.0;
    if (j >= a.jlo && j <= a.jhi) {
        const double c = a.cmol, t2 = a.temp2;
        const bool v = a.sys == LES_SYS_U2;
        // metric weights, and the eddy weights of rows j-1 and j+1
        const double wm = v ? w[4 * j] : w[4 * j + 1], wp = v ? w[4 * j + 1] : w[4 * j + 2];
        const double em = t2 * (v ? 0.5 * (n0 + nm) : n0) * wm, ep = t2 * (v ? 0.5 * (n0 + np) : np) * wp;
        L = -(c * wm + em);
        U = -(c * wp + ep);
        D = 1.0 + (c * wp + ep) + (c * wm + em);
        V = r + (ep * (up - u0) - em * (u0 - um));
    }
    auto set = [&](double l, double d, double u, double v) { L = l; D = d; U = u; V = v; };
    if (a.sys == LES_SYS_U2) {
        if (j == 0) set(0., 1., 0., 0.);
        if (a.lo == 0) {
            if (j == 1 || j == 2) set(0., 1., 0., a.clo_c);
        } else if (j == 1) {
            set(0., -1., 1., dyf[1] * a.clo_c);
        }
        if (a.hi == 0) {
            if (j == NY || j == NY + 1) set(0., 1., 0., a.chi_c);
        } else if (j == NY + 1) {
            set(-1., 1., 0., dyf[NY] * a.chi_c);
        }
    } else {
        if (j == 0) set(0., 1., 0., 0.);
        if (j == 1) {
            if (a.lo == 0) set(0., 1., 0., a.clo_c);
            else set(0., -1., 1., dy[2] * a.clo_c);
        }
        if (j == NY + 1) set(0., 1., 0., 0.);
        if (j == NY) {
            if (a.hi == 0) set(0., 1., 0., a.chi_c);
            else set(-1., 1., 0., dy[NY] * a.chi_c);
        }
    }
}

// The solves in segments: a real column (a double column of a pair plane) is
// cut into 32 segments of RM rows or fewer.  A lane eliminates its segment's
// rows [a, b] downwards,
//   x(j) = g(j) - c(j) x(j+1) - f(j) x(a-1),
// and folds them upwards to the same form for x(a) in x(b+1) and x(a-1); the
// two equations of every segment form a block-tridiagonal system that one lane
// a column solves through LDS, and each lane back-substitutes its rows.  The
// matrix differs from column to column (NU_T), so nothing is precomputed; rows
// stay in registers: each value is read once and written once (56 B a point and
// pair against 120 B of the sweeps below, whose scratch makes a round trip).
// 16 columns (128 B of a row) x 32 segments a block.
// 384x257x384: 1.98 -> 1.46 ms; 96x81x108, where one thread a column filled
// 162 CUs: 89 -> 40 us.
template <int RM>
__global__ void __launch_bounds__(512) k_les_cn_seg(Geo g, LesCnSet set, const double *__restrict__ nut,
                                                    const double *__restrict__ w, const double *__restrict__ dy,
                                                    const double *__restrict__ dyf)
{
    constexpr int NS = 32, NC = 16;
    __shared__ double eq[NS][6][NC];  // x(a): G, C, F; x(b): g, c, f -- then x(b+1), x(a-1)
    const int col = threadIdx.x & (NC - 1), seg = threadIdx.x / NC;
    const long n = 2L * g.nx * g.nz;  // doubles a pair plane; the last block's columns beyond it are off
    const long e0 = (long)blockIdx.x * NC + col;
    const bool on = e0 < n;
    const long e = on ? e0 : n - 1;
    const LesCn a = set.a[blockIdx.y][e & 1];
    const bool live = on && a.sys >= 0;
    const double *__restrict__ rhs = reinterpret_cast<const double *>(set.rhs[blockIdx.y]) + e;
    double *__restrict__ out = reinterpret_cast<double *>(set.out[blockIdx.y]) + e;
    const double *__restrict__ nt = nut + (e >> 1);
    const long nn = n >> 1;
    const int NY = g.ny, R = (NY + 2 + NS - 1) / NS, ja = seg * R, jb = min(ja + R - 1, NY + 1);
    double G[RM], C[RM], F[RM];
    double ga = 0.0, ca = -1.0, fa = 0.0, gb = 0.0, cb = 0.0, fb = -1.0;  // a segment without rows passes both through
    if (live && ja <= jb) {
        double um = ja > 0 ? out[(ja - 1) * n] : 0.0, u0 = out[ja * n];
        double nm = ja > 0 ? nt[(ja - 1) * nn] : 0.0, n0 = nt[ja * nn];
#pragma unroll
        for (int r = 0; r < RM; ++r) {
            const int j = ja + r;
            if (j <= jb) {
                const int jn = min(j + 1, NY + 1);
                const double up = out[jn * n], np = nt[jn * nn];
                double L, D, U, V;
                les_row(a, j, w, dy, dyf, n0, np, nm, u0, up, um, rhs[j * n], L, D, U, V);
                if (r > 0) {
                    D = D - L * C[r - 1];
                    V = V - L * G[r - 1];
                }
                const double rd = D != 0.0 ? 1.0 / D : 0.0;
                C[r] = U * rd;
                G[r] = V * rd;
                F[r] = r > 0 ? -L * F[r - 1] * rd : L * rd;
                um = u0;
                u0 = up;
                nm = n0;
                n0 = np;
            }
        }
        bool first = true;
#pragma unroll
        for (int r = RM - 1; r >= 0; --r) {
            if (ja + r <= jb) {
                if (first) {
                    ga = gb = G[r];
                    ca = cb = C[r];
                    fa = fb = F[r];
                    first = false;
                } else {
                    ga = G[r] - C[r] * ga;
                    fa = F[r] - C[r] * fa;
                    ca = -C[r] * ca;
                }
            }
        }
    }
    eq[seg][0][col] = ga;
    eq[seg][1][col] = ca;
    eq[seg][2][col] = fa;
    eq[seg][3][col] = gb;
    eq[seg][4][col] = cb;
    eq[seg][5][col] = fb;
    __syncthreads();
    if (seg == 0) {
        // x(b) of the segment before = al - be x(a) of this one
        double al = 0.0, be = 0.0;
        for (int s = 0; s < NS; ++s) {
            const double Ga = eq[s][0][col], Ca = eq[s][1][col], Fa = eq[s][2][col];
            const double Gb = eq[s][3][col], Cb = eq[s][4][col], Fb = eq[s][5][col];
            const double rw = 1.0 / (1.0 - Fa * be);
            const double ga_ = (Ga - Fa * al) * rw, de = Ca * rw;  // x(a) = ga_ - de x(b+1)
            eq[s][0][col] = ga_;
            eq[s][1][col] = de;
            eq[s][2][col] = al;
            eq[s][3][col] = be;
            const double t = Fb * be;
            al = Gb - Fb * al + t * ga_;
            be = Cb + t * de;
        }
        double X = 0.0;
        for (int s = NS - 1; s >= 0; --s) {
            const double xa = eq[s][0][col] - eq[s][1][col] * X;
            const double Y = eq[s][2][col] - eq[s][3][col] * xa;
            eq[s][4][col] = X;
            eq[s][5][col] = Y;
            X = xa;
        }
    }
    __syncthreads();
    if (live && ja <= jb) {
        double x = eq[seg][4][col];
        const double y = eq[seg][5][col];
#pragma unroll
        for (int r = RM - 1; r >= 0; --r) {
            const int j = ja + r;
            if (j <= jb) {
                x = G[r] - C[r] * x - F[r] * y;
                if (j >= a.clo && j <= a.chi) out[j * n] = x;
            }
        }
    }
}

// Columns of more than 542 rows: THOMAS_REAL (for/mpi.f:630-809) down the
// columns of a pair plane, one thread a real column of one of the pair's two
// systems (grid.y: the pair).  The
// forward sweep leaves U/B and G/B of every row in the scratch planes; the
// back substitution reads only those.  Rows clo..chi of the field are
// overwritten.  A column is read and written by its own thread only, every
// read of the field before the first write.
__global__ void __launch_bounds__(256) k_les_cn(Geo g, LesCnSet set, const double *__restrict__ nut,
                                                const double *__restrict__ w, const double *__restrict__ dy,
                                                const double *__restrict__ dyf)
{
    const long n = 2L * g.nx * g.nz;  // doubles a pair plane
    const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= n) return;
    const LesCn a = set.a[blockIdx.y][e & 1];
    if (a.sys < 0) return;
    const double *__restrict__ rhs = reinterpret_cast<const double *>(set.rhs[blockIdx.y]) + e;
    double *__restrict__ cw = reinterpret_cast<double *>(set.cw[blockIdx.y]) + e;
    double *__restrict__ gw = reinterpret_cast<double *>(set.gw[blockIdx.y]) + e;
    double *__restrict__ out = reinterpret_cast<double *>(set.out[blockIdx.y]) + e;
    const double *__restrict__ nt = nut + (e >> 1);
    const long nn = n >> 1;
    const int NY = g.ny;
    double um = 0.0, u0 = out[0], up = out[n], nm = 0.0, n0 = nt[0], np = nt[nn];
    double bprev = 1.0, cprev = 0.0, gprev = 0.0;
    for (int j = 0; j <= NY + 1; ++j) {
        double L, D, U, V;
        les_row(a, j, w, dy, dyf, n0, np, nm, u0, up, um, rhs[j * n], L, D, U, V);
        if (j > 0) {
            const double m = -L / bprev;
            D = D + m * cprev;
            V = V + m * gprev;
        }
        const double rb = D != 0.0 ? 1.0 / D : 0.0;  // zero-pivot guard of the back substitution
        cw[j * n] = U * rb;
        gw[j * n] = V * rb;
        bprev = D;
        cprev = U;
        gprev = V;
        um = u0;
        u0 = up;
        nm = n0;
        n0 = np;
        const int jn = j + 2 <= NY + 1 ? j + 2 : NY + 1;
        up = out[jn * n];
        np = nt[jn * nn];
    }
    double xn = 0.0;
    for (int j = NY + 1; j >= 0; --j) {
        xn = gw[j * n] - cw[j * n] * xn;
        if (j >= a.clo && j <= a.chi) out[j * n] = xn;
    }
}

// Rows a segment: the fewest registers that hold a 32nd of the column.
void launch_les_cn(hipStream_t s, const Geo &g, const LesCnSet &set, const double *nut, const double *w,
                   const double *dy, const double *dyf)
{
    const long n = 2L * g.nx * g.nz;
    const int rows = (g.ny + 2 + 31) / 32;
    const dim3 grid((unsigned)((n + 15) / 16), 2);
    if (rows <= 3)
        hipLaunchKernelGGL((k_les_cn_seg<3>), grid, dim3(512), 0, s, g, set, nut, w, dy, dyf);
    else if (rows <= 5)
        hipLaunchKernelGGL((k_les_cn_seg<5>), grid, dim3(512), 0, s, g, set, nut, w, dy, dyf);
    else if (rows <= 9)
        hipLaunchKernelGGL((k_les_cn_seg<9>), grid, dim3(512), 0, s, g, set, nut, w, dy, dyf);
    else if (rows <= 17)
        hipLaunchKernelGGL((k_les_cn_seg<17>), grid, dim3(512), 0, s, g, set, nut, w, dy, dyf);
    else
        hipLaunchKernelGGL(k_les_cn, dim3((unsigned)((n + 255) / 256), 2), dim3(256), 0, s, g, set, nut, w, dy, dyf);
}

// Per-plane maxima of |U1|, |U2|, |U3| on physical planes 1..NY into
// out[q * NY + j - 1] (COURANT's input, for/courant.f:25-45)
__global__ void __launch_bounds__(256) k_les_vmax(Geo g, const cx<double> *__restrict__ p0,
                                                  const cx<double> *__restrict__ p1, double *__restrict__ out)
{
    __shared__ double red[3][256];
    const int j = 1 + blockIdx.x, tid = threadIdx.x;
    const long n = (long)g.nx * g.nz;
    double m[3] = {0.0, 0.0, 0.0};
    for (long e = tid; e < n; e += 256) {
        const cx<double> a = p0[j * n + e], b = p1[j * n + e];
        m[0] = fmax(m[0], fabs(a.re));
        m[1] = fmax(m[1], fabs(a.im));
        m[2] = fmax(m[2], fabs(b.re));
    }
    for (int q = 0; q < 3; ++q) red[q][tid] = m[q];
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if (tid < h)
            for (int q = 0; q < 3; ++q) red[q][tid] = fmax(red[q][tid], red[q][tid + h]);
        __syncthreads();
    }
    if (tid < 3) out[(long)tid * g.ny + (j - 1)] = red[tid][0];
}

void launch_les_vmax(hipStream_t s, const Geo &g, const cx<double> *p0, const cx<double> *p1, double *out)
{
    hipLaunchKernelGGL(k_les_vmax, dim3(g.ny), dim3(256), 0, s, g, p0, p1, out);
}

// The reference forms CF from the velocity before les_chan resets its
// boundary rows (for/channel.f:175-290 precede for/channel.f:303); the
// column kernel saw the reset rows.  On rows 1 and NY (pre: the saved rows
// of CU1 and CU3, plane 0 row 1, plane 1 row NY, then the same for CU3) the
// linear terms that read them are corrected: horizontal viscosity and
// Coriolis in CF1, CF3, the background-gradient terms in CFTH.
__global__ void k_les_cf_rows(Geo g, const cx<double> *__restrict__ pre, const cx<double> *__restrict__ cu1,
                              const cx<double> *__restrict__ cu3, cx<double> *__restrict__ cf1,
                              cx<double> *__restrict__ cf3, cx<double> *__restrict__ cfth,
                              const double *__restrict__ kx2, const double *__restrict__ kz2, LesCfFix f)
{
    const long m = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (m >= g.ps) return;
    const int K = (int)(m / g.mk), i = (int)(m - (long)K * g.mk);
    const long ps = g.ps;
    const double k2 = kx2[i] + kz2[K];
    const double visc = f.nu * ((f.beta == 1.0) ? k2 : pow(k2, f.beta));
    for (int r = 0; r < 2; ++r) {
        const int j = r == 0 ? 1 : g.ny;
        const long o = m + (long)j * ps;
        const cx<double> a = pre[m + (long)r * ps], b = pre[m + (long)(2 + r) * ps];
        const cx<double> d1 = make_cx<double>(a.re - cu1[o].re, a.im - cu1[o].im);
        const cx<double> d3 = make_cx<double>(b.re - cu3[o].re, b.im - cu3[o].im);
        if (j >= f.jstart && j <= f.jend) {
            cx<double> x = cf1[o], z = cf3[o];
            x = make_cx<double>(x.re - visc * d1.re + f.i_ro * d3.re, x.im - visc * d1.im + f.i_ro * d3.im);
            z = make_cx<double>(z.re - visc * d3.re - f.i_ro * d1.re, z.im - visc * d3.im - f.i_ro * d1.im);
            cf1[o] = x;
            cf3[o] = z;
        }
        if (cfth && j >= f.jstart_th && j <= f.jend_th) {
            cx<double> t = cfth[o];
            t = make_cx<double>(t.re - (d1.re * f.drhodx + d3.re * f.drhodz), t.im - (d1.im * f.drhodx + d3.im * f.drhodz));
            cfth[o] = t;
        }
    }
}

void launch_les_cf_rows(hipStream_t s, const Geo &g, const cx<double> *pre, const cx<double> *cu1,
                        const cx<double> *cu3, cx<double> *cf1, cx<double> *cf3, cx<double> *cfth, const double *kx2,
                        const double *kz2, const LesCfFix &f)
{
    hipLaunchKernelGGL(k_les_cf_rows, dim3((unsigned)((g.ps + 255) / 256)), dim3(256), 0, s, g, pre, cu1, cu3, cf1,
                       cf3, cfth, kx2, kz2, f);
}

// tkebudget_chan_les (for/save_stats.f:887-960): per plane j = 1..NY the sum
// over the physical points of u_i times its implicit eddy-viscosity term;
// out[j - 1].  Fixed-order reduction.
__global__ void __launch_bounds__(256) k_les_eps(Geo g, const cx<double> *__restrict__ p0,
                                                 const cx<double> *__restrict__ p1, const double *__restrict__ nut,
                                                 const double *__restrict__ dy, const double *__restrict__ dyf,
                                                 double *__restrict__ out)
{
    __shared__ double red[256];
    const int j = 1 + blockIdx.x, tid = threadIdx.x;
    const long n = (long)g.nx * g.nz;
    double acc = 0.0;
    for (long e = tid; e < n; e += 256) {
        const long x = j * n + e, xp = x + n, xm = x - n;
        const cx<double> a = p0[x], ap = p0[xp], am = p0[xm];
        const double w = p1[x].re, wp = p1[xp].re, wm = p1[xm].re, n0 = nut[x], np = nut[xp], nm = nut[xm];
        acc += a.re * ((np * (ap.re - a.re) / dy[j + 1] - n0 * (a.re - am.re) / dy[j]) / dyf[j]) +
               w * ((np * (wp - w) / dy[j + 1] - n0 * (w - wm) / dy[j]) / dyf[j]) +
               a.im * ((0.5 * (n0 + np) * (ap.im - a.im) / dyf[j] - 0.5 * (n0 + nm) * (a.im - am.im) / dyf[j - 1]) /
                       dy[j]);
    }
    red[tid] = acc;
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if (tid < h) red[tid] += red[tid + h];
        __syncthreads();
    }
    if (tid == 0) out[j - 1] = red[0];
}

void launch_les_eps(hipStream_t s, const Geo &g, const cx<double> *p0, const cx<double> *p1, const double *nut,
                    const double *dy, const double *dyf, double *out)
{
    hipLaunchKernelGGL(k_les_eps, dim3(g.ny), dim3(256), 0, s, g, p0, p1, nut, dy, dyf, out);
}

void launch_les_bc(hipStream_t s, const Geo &g, cx<double> *cu1, cx<double> *cu3, int u_min, int u_max, int w_min,
                   int w_max)
{
    hipLaunchKernelGGL(k_les_bc, dim3((unsigned)((g.ps + 255) / 256)), dim3(256), 0, s, g, cu1, cu3, u_min, u_max,
                       w_min, w_max);
}

void launch_les_bc_phys(hipStream_t s, const Geo &g, cx<double> *cu1, cx<double> *cu2, cx<double> *cu3,
                        const LesBc &b, const double *dy, const double *dyf)
{
    hipLaunchKernelGGL(k_les_bc_phys, dim3((unsigned)((g.ps + 255) / 256)), dim3(256), 0, s, g, cu1, cu2, cu3, b, dy,
                       dyf);
}

void launch_les_bc_rows(hipStream_t s, const Geo &g, const cx<double> *p0, const cx<double> *p1, cx<double> *bc,
                        const LesBc &b, const double *dy, const double *dyf)
{
    const long n = (long)g.nx * g.nz;
    hipLaunchKernelGGL(k_les_bc_rows, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, g, p0, p1, bc, b, dy, dyf);
}

void launch_les_bc_put(hipStream_t s, const Geo &g, cx<double> *p0, cx<double> *p1, const cx<double> *bc)
{
    const long n = (long)g.nx * g.nz;
    hipLaunchKernelGGL(k_les_bc_put, dim3((unsigned)((n + 255) / 256), 8), dim3(256), 0, s, g, p0, p1, bc);
}

}  // namespace dgpu
