// dgpu_pairs.hip -- kept modes to physical "pair" planes and back in FP64, on
// the in-place transforms of dgpu_fft.hpp, for the paths that need physical
// fields outside the fused x kernel: LES (dgpu_les.hip) and POISSON_P_CHAN
// (dgpu_poisson.hip).
//
//   k_pairs_inv   x backward of the z-backward rows Zt[f][j][zp][kx]: a row
//                 pair (A, B), each a field or its x derivative, becomes the complex
//                 row a + i b of physical values
//   k_pairs_fwd   x forward of such rows into Wt[f][j][zp][kx] (unnormalised
//                 in z, 1/NX applied)
//
// A pair plane is P[j][zp][slot], NX slots a row, NZ rows.  zp is the z
// position of the in-place z transforms (digit-reversed); slot = idx*T + th
// numbers the E values idx of the T threads th of the last backward stage, so
// that stage's stores and the first forward stage's loads are contiguous.
// Everything done on pair planes is pointwise in x and z, so the order never
// matters (pair_slot gives it where natural order is wanted).
//
// Both kernels move 16 B per pair point and 16 B per kept row value: 384x257x384,
// 6 pairs back in 1.23 ms (5.3 GB, 4.3 TB/s), 2 pairs forward in 0.43 (2.0 GB,
// 4.7 TB/s), near the rate of a copy; three waves per SIMD hide the loads (at two,
// before the dealiasing gap was known at compile time, 1.99 ms).  The standalone
// transforms they replace took 0.33 ms per field and direction (Fortran-layout
// planes, one real row per complex transform).
#include "dgpu_hot.hpp"

#include <algorithm>

namespace dgpu {

namespace {

// Rows (pair, plane, zp) are numbered row = (pair * nplanes + plane) * nz +
// zp; a block's rb row groups take rb rows at a time, `reps` times over.
struct RowOf {
    int pair, plane, zp;
    bool ok;
};
__device__ __forceinline__ RowOf row_of(long r, int nz, int nplanes, long nrows)
{
    RowOf o;
    o.ok = r < nrows;
    const long rr = o.ok ? r : nrows - 1;
    o.zp = (int)(rr % nz);
    const long q = rr / nz;
    o.plane = (int)(q % nplanes);
    o.pair = (int)(q / nplanes);
    return o;
}

}  // namespace

template <int E, int PID>
__global__ void __launch_bounds__(128) k_pairs_inv(IpLen frt, const cx<double> *__restrict__ twg, int mk_rt, int ld,
                                                    const cx<double> *__restrict__ zt, long zt_fs, PairSrc src,
                                                    PairDst dst, const double *__restrict__ kxv, int nz, int j0,
                                                    int nplanes, long nrows, int reps)
{
    constexpr int R0 = E / 2;
    const IpLen &fx = plan_ref<PID>(frt);
    extern __shared__ unsigned char smem_raw[];
    const int nx = fx.n, TT = fx.t, S = fx.nstages;
    // constant with a compile-time plan: what lies in the dealiasing gap is known
    const int mk = PID != 0 ? nx / 3 + 1 : mk_rt;
    const int tid = threadIdx.x, p = tid / TT, th = tid - p * TT, rb = blockDim.x / TT;
    __builtin_assume(th >= 0 && th < TT);
    cx<double> *row = reinterpret_cast<cx<double> *>(smem_raw) + p * nx;
    cx<double> *tw = reinterpret_cast<cx<double> *>(smem_raw) + rb * nx;
    double *kxs = reinterpret_cast<double *>(tw + fx.twn);
    for (int e = tid; e < fx.twn; e += blockDim.x) tw[e] = twg[e];
    for (int e = tid; e < mk; e += blockDim.x) kxs[e] = kxv[e];
    __syncthreads();
    const bool wave_rows = (64 % TT) == 0;
    auto row_sync = [&]() {
        if (wave_rows) wave_lds_sync();
        else __syncthreads();
    };
    for (int k = 0; k < reps; ++k) {
        const RowOf o = row_of(((long)blockIdx.x * reps + k) * rb + p, nz, nplanes, nrows);
        const long at = ((long)(j0 + o.plane) * nz + o.zp) * ld;
        const cx<double> *za = zt + src.a[o.pair] * zt_fs + at, *zb = zt + max(src.b[o.pair], 0) * zt_fs + at;
        const bool hasb = src.b[o.pair] >= 0, da = src.da[o.pair], db = src.db[o.pair];
        // stage 0: the spectrum of a + i b from the Hermitian halves of both
        // rows; C2R ignores Im of the DC term
        ip_stage<double, E, R0, +1, true>(
            fx, 0, tw, th,
            [&](int, int f) {
                const int kk = f < mk ? f : (f > nx - mk ? nx - f : -1), kc = max(kk, 0);
                cx<double> A = za[kc], B = hasb ? zb[kc] : make_cx(0.0, 0.0);
                const double kx = kxs[kc];
                if (da) A = make_cx(-kx * A.im, kx * A.re);
                if (db) B = make_cx(-kx * B.im, kx * B.re);
                if (kk < 0) A = B = make_cx(0.0, 0.0);
                if (f == 0) A.im = B.im = 0.0;
                if (f > nx - mk) {
                    A.im = -A.im;
                    B.im = -B.im;
                }
                return make_cx(A.re - B.im, A.im + B.re);
            },
            [&](int, int pos, cx<double> v) { row[ip_swz(fx, pos)] = v; });
        row_sync();
        stage_loop<PID != 0>(1, S - 1, [&](int s) {
            ip_stage_row<double, E, +1, true, PID != 0>(row, fx, s, tw, th);
            row_sync();
        });
        cx<double> *out = dst.p[o.pair] + ((long)(j0 + o.plane) * nz + o.zp) * nx + th;
        with_radix<E>(fx.radix[S - 1], [&](auto rc) {
            constexpr int R = decltype(rc)::value;
            ip_stage<double, E, R, +1, true>(
                fx, S - 1, tw, th, [&](int, int pos) { return row[ip_swz(fx, pos)]; },
                [&](int idx, int, cx<double> v) {
                    if (o.ok) out[idx * TT] = v;
                });
        });
        row_sync();
    }
}

template <int E, int PID>
__global__ void __launch_bounds__(128) k_pairs_fwd(IpLen frt, const cx<double> *__restrict__ twg, int mk_rt, int ld,
                                                    PairDst src, cx<double> *__restrict__ wt, long wt_fs, PairOut out,
                                                    int nz, int j0, int nplanes, long nrows, int reps)
{
    const IpLen &fx = plan_ref<PID>(frt);
    extern __shared__ unsigned char smem_raw[];
    const int nx = fx.n, TT = fx.t, S = fx.nstages;
    // constant with a compile-time plan: what lies in the dealiasing gap is known
    const int mk = PID != 0 ? nx / 3 + 1 : mk_rt;
    const int tid = threadIdx.x, p = tid / TT, th = tid - p * TT, rb = blockDim.x / TT;
    __builtin_assume(th >= 0 && th < TT);
    cx<double> *row = reinterpret_cast<cx<double> *>(smem_raw) + p * nx;
    cx<double> *tw = reinterpret_cast<cx<double> *>(smem_raw) + rb * nx;
    for (int e = tid; e < fx.twn; e += blockDim.x) tw[e] = twg[e];
    __syncthreads();
    const bool wave_rows = (64 % TT) == 0;
    auto row_sync = [&]() {
        if (wave_rows) wave_lds_sync();
        else __syncthreads();
    };
    for (int k = 0; k < reps; ++k) {
        const RowOf o = row_of(((long)blockIdx.x * reps + k) * rb + p, nz, nplanes, nrows);
        const cx<double> *in = src.p[o.pair] + ((long)(j0 + o.plane) * nz + o.zp) * nx + th;
        with_radix<E>(fx.radix[S - 1], [&](auto rc) {
            constexpr int R = decltype(rc)::value;
            ip_stage<double, E, R, -1, false>(
                fx, S - 1, tw, th, [&](int idx, int) { return in[idx * TT]; },
                [&](int, int pos, cx<double> v) { row[ip_swz(fx, pos)] = v; });
        });
        row_sync();
        stage_loop<PID != 0>(1, S - 1, [&](int s) {
            ip_stage_row<double, E, -1, false, PID != 0>(row, fx, S - 1 - s, tw, th);
            row_sync();
        });
        cx<double> *o0 = wt + ((long)(j0 + o.plane) * nz + o.zp) * ld;
        const int fa = out.a[o.pair], fb = out.b[o.pair];
        const double h = 0.5 / nx;
        x_split<double, E>(fx, row, tw, th, mk, [&](int kp, cx<double> Zk, cx<double> Zn) {
            if (!o.ok) return;
            if (fa >= 0) o0[fa * wt_fs + kp] = make_cx((Zk.re + Zn.re) * h, (Zk.im - Zn.im) * h);
            if (fb >= 0) o0[fb * wt_fs + kp] = make_cx((Zk.im + Zn.im) * h, -(Zk.re - Zn.re) * h);
        });
        row_sync();
    }
}

namespace {

// Rows per block and repetitions: about 128 threads a block (four rows at
// NX = 384: 31 KB of LDS, five blocks per CU), several row groups per block
// so that the twiddle copy is paid once, but no fewer than ~8 blocks per CU.
struct PairGrid {
    int rb, reps;
    long blocks;
    size_t lds;
};
PairGrid pair_grid(const IpLen &fx, int mk, long nrows)
{
    PairGrid q;
    q.rb = std::max(1, 128 / fx.t);
    const long groups = (nrows + q.rb - 1) / q.rb;
    q.reps = (int)std::min<long>(8, std::max<long>(1, groups / 2048));
    q.blocks = (groups + q.reps - 1) / q.reps;
    q.lds = sizeof(cx<double>) * ((size_t)q.rb * fx.n + fx.twn) + sizeof(double) * mk;
    return q;
}

}  // namespace

template <int E, int PID>
static void pairs_inv_e(hipStream_t s, const Geo &g, const IpLen &fx, const cx<double> *tw, int ld,
                        const cx<double> *zt, long zt_fs, const PairSrc &src, const PairDst &dst, const double *kx,
                        int j0, int nplanes)
{
    const long nrows = (long)src.n * nplanes * g.nz;
    const PairGrid q = pair_grid(fx, g.mk, nrows);
    hipLaunchKernelGGL((k_pairs_inv<E, PID>), dim3((unsigned)q.blocks), dim3(q.rb * fx.t), q.lds, s, fx, tw, g.mk, ld,
                       zt, zt_fs, src, dst, kx, g.nz, j0, nplanes, nrows, q.reps);
}

template <int E, int PID>
static void pairs_fwd_e(hipStream_t s, const Geo &g, const IpLen &fx, const cx<double> *tw, int ld,
                        const PairDst &src, cx<double> *wt, long wt_fs, const PairOut &out, int j0, int nplanes)
{
    const long nrows = (long)out.n * nplanes * g.nz;
    const PairGrid q = pair_grid(fx, g.mk, nrows);
    hipLaunchKernelGGL((k_pairs_fwd<E, PID>), dim3((unsigned)q.blocks), dim3(q.rb * fx.t), q.lds, s, fx, tw, g.mk, ld,
                       src, wt, wt_fs, out, g.nz, j0, nplanes, nrows, q.reps);
}

void launch_pairs_inv(hipStream_t s, const Geo &g, const IpLen &fx, const cx<double> *tw, int ld,
                      const cx<double> *zt, long zt_fs, const PairSrc &src, const PairDst &dst, const double *kx,
                      int j0, int nplanes)
{
    if (with_pid(const_plan_id(fx), XPids64{}, [&](auto pc) {
            constexpr int P = decltype(pc)::value;
            pairs_inv_e<kConstPlanSpecs[P].e, P>(s, g, fx, tw, ld, zt, zt_fs, src, dst, kx, j0, nplanes);
        }))
        return;
    DGPU_DISPATCH_XE64(fx.e, (pairs_inv_e<EE, 0>(s, g, fx, tw, ld, zt, zt_fs, src, dst, kx, j0, nplanes)));
}

void launch_pairs_fwd(hipStream_t s, const Geo &g, const IpLen &fx, const cx<double> *tw, int ld, const PairDst &src,
                      cx<double> *wt, long wt_fs, const PairOut &out, int j0, int nplanes)
{
    if (with_pid(const_plan_id(fx), XPids64{}, [&](auto pc) {
            constexpr int P = decltype(pc)::value;
            pairs_fwd_e<kConstPlanSpecs[P].e, P>(s, g, fx, tw, ld, src, wt, wt_fs, out, j0, nplanes);
        }))
        return;
    DGPU_DISPATCH_XE64(fx.e, (pairs_fwd_e<EE, 0>(s, g, fx, tw, ld, src, wt, wt_fs, out, j0, nplanes)));
}

int pair_slot(const IpLen &f, int i)
{
    // position of index i after the backward (DIF) stages: its digits i = q0 +
    // R0 (q1 + R1 (q2 + ...)) weighted by the spans
    int pos = 0, rest = i;
    for (int s = 0; s < f.nstages; ++s) {
        pos += (rest % f.radix[s]) * f.span[s];
        rest /= f.radix[s];
    }
    const int R = f.radix[f.nstages - 1], t = pos / R, q = pos % R;
    return ((t / f.t) * R + q) * f.t + t % f.t;
}

int pair_zpos(const IpLen &f, int k)
{
    int pos = 0, rest = k;
    for (int s = 0; s < f.nstages; ++s) {
        pos += (rest % f.radix[s]) * f.span[s];
        rest /= f.radix[s];
    }
    return pos;
}

}  // namespace dgpu
