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
// The two rows of a pair are transformed together, and the round-off of a
// complex transform is that of its larger half.  Halves whose magnitudes are
// more than 2^10 apart (U3 and a scalar in a unit of its own) are brought to
// 2^10 by a power of two, which is exact, and taken back where they come apart,
// so what one field adds to the other's round-off is bounded: beside a passive
// scalar of 1e6 the LES substep's CU3 was off by 1.3e-13 of its maximum, 3e-15
// for a scalar of 1.  Nearer halves stay as they are: bringing U2 up to U1, whose
// maximum is its mean, costs U1's fluctuations four times their round-off.
//
// Both kernels move 16 B per pair point and 16 B per kept row value: 384x257x384,
// 6 pairs back in 1.25-1.28 ms (counted 2.4 GB read, 3.7 written, 4.8 TB/s), 2 pairs
// forward in 0.43 (1.2 + 0.8 GB, 4.7 TB/s), near the rate of a copy.  k_pairs_inv
// holds both rows until their scale is known: 198 registers, two waves per SIMD
// (1.23 ms at three without it; 25 to 32 registers spill when held to three, and
// reading the rows twice, once for the scale, takes 1.77).  The standalone
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

// Largest magnitudes so far of the values of rows A and B, as the high words
// of the doubles (ordered as the values are; NaN and infinity above all).
struct PairMax {
    int a = 0, b = 0;
    __device__ __forceinline__ static int hi(double x) { return __double2hiint(x) & 0x7fffffff; }
    __device__ __forceinline__ void take_a(double x) { a = max(a, hi(x)); }
    __device__ __forceinline__ void take_b(double x) { b = max(b, hi(x)); }
};

// Row B goes in times `up`, the halves come out times a and b: `up` is the
// power of two that brings the larger of the rows' largest values down to 2^10
// times the other (1 where they are nearer, or one is not finite), and a row of
// zeros comes out as zeros.
struct PairScale {
    double up, a, b;
};
__device__ __forceinline__ double pow2(int k) { return __hiloint2double((k + 1023) << 20, 0); }

// From every thread of the row: TT lanes of a wave, or through the two words ex
// (zero on entry) of a row that does not divide one.
__device__ __forceinline__ PairScale pair_balance(PairMax m, int TT, bool wave_rows, int *ex)
{
    int ea = m.a >> 20, eb = m.b >> 20;
    if (wave_rows) {
        int e = (ea << 16) | eb;  // two halves of 11 bits
        for (int h = TT >> 1; h > 0; h >>= 1) {
            const int o = __shfl_xor(e, h);
            e = (max(e >> 16, o >> 16) << 16) | max(e & 0xffff, o & 0xffff);
        }
        ea = e >> 16;
        eb = e & 0xffff;
    } else {
        atomicMax(&ex[0], ea);
        atomicMax(&ex[1], eb);
        __syncthreads();
        ea = ex[0];
        eb = ex[1];
    }
    const bool scaled = ea != 0 && eb != 0 && ea != 0x7ff && eb != 0x7ff;
    const int d = scaled ? ea - eb : 0, k = max(-1000, min(1000, d - max(-10, min(10, d))));
    return {pow2(k), ea ? 1.0 : 0.0, eb ? pow2(-k) : 0.0};
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
    int *ex = reinterpret_cast<int *>(kxs + mk) + 2 * p;
    for (int e = tid; e < fx.twn; e += blockDim.x) tw[e] = twg[e];
    for (int e = tid; e < mk; e += blockDim.x) kxs[e] = kxv[e];
    if (th == 0) ex[0] = ex[1] = 0;
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
        // the Hermitian halves of both rows; C2R ignores Im of the DC term
        cx<double> A[E], B[E];
        PairMax m;
        ip_groups<E, R0>(fx, 0, th, [&](int u, int b0, int) {
#pragma unroll
            for (int q = 0; q < R0; ++q) {
                const int f = b0 + q * fx.span[0];
                const int kk = f < mk ? f : (f > nx - mk ? nx - f : -1), kc = max(kk, 0);
                cx<double> a = za[kc], b = hasb ? zb[kc] : make_cx(0.0, 0.0);
                const double kx = kxs[kc];
                if (da) a = make_cx(-kx * a.im, kx * a.re);
                if (db) b = make_cx(-kx * b.im, kx * b.re);
                if (kk < 0) a = b = make_cx(0.0, 0.0);
                if (f == 0) a.im = b.im = 0.0;
                if (f > nx - mk) {
                    a.im = -a.im;
                    b.im = -b.im;
                }
                m.take_a(a.re);
                m.take_a(a.im);
                m.take_b(b.re);
                m.take_b(b.im);
                A[u * R0 + q] = a;
                B[u * R0 + q] = b;
            }
        });
        const PairScale sc = pair_balance(m, TT, wave_rows, ex);
        // stage 0: the spectrum of a + i b
        ip_stage<double, E, R0, +1, true>(
            fx, 0, tw, th,
            [&](int idx, int) {
                return make_cx(A[idx].re - sc.up * B[idx].im, A[idx].im + sc.up * B[idx].re);
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
                    if (o.ok) out[idx * TT] = make_cx(v.re * sc.a, v.im * sc.b);
                });
        });
        if (!wave_rows && th == 0) ex[0] = ex[1] = 0;
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
    int *ex = reinterpret_cast<int *>(tw + fx.twn) + 2 * p;
    for (int e = tid; e < fx.twn; e += blockDim.x) tw[e] = twg[e];
    if (th == 0) ex[0] = ex[1] = 0;
    __syncthreads();
    const bool wave_rows = (64 % TT) == 0;
    auto row_sync = [&]() {
        if (wave_rows) wave_lds_sync();
        else __syncthreads();
    };
    for (int k = 0; k < reps; ++k) {
        const RowOf o = row_of(((long)blockIdx.x * reps + k) * rb + p, nz, nplanes, nrows);
        const cx<double> *in = src.p[o.pair] + ((long)(j0 + o.plane) * nz + o.zp) * nx + th;
        cx<double> v[E];
        PairMax m;
#pragma unroll
        for (int e = 0; e < E; ++e) v[e] = in[e * TT];
#pragma unroll
        for (int e = 0; e < E; ++e) {
            m.take_a(v[e].re);
            m.take_b(v[e].im);
        }
        const PairScale sc = pair_balance(m, TT, wave_rows, ex);
        with_radix<E>(fx.radix[S - 1], [&](auto rc) {
            constexpr int R = decltype(rc)::value;
            ip_stage<double, E, R, -1, false>(
                fx, S - 1, tw, th, [&](int idx, int) { return make_cx(v[idx].re, v[idx].im * sc.up); },
                [&](int, int pos, cx<double> v) { row[ip_swz(fx, pos)] = v; });
        });
        row_sync();
        stage_loop<PID != 0>(1, S - 1, [&](int s) {
            ip_stage_row<double, E, -1, false, PID != 0>(row, fx, S - 1 - s, tw, th);
            row_sync();
        });
        cx<double> *o0 = wt + ((long)(j0 + o.plane) * nz + o.zp) * ld;
        const int fa = out.a[o.pair], fb = out.b[o.pair];
        const double ha = 0.5 / nx * sc.a, hb = 0.5 / nx * sc.b;
        x_split<double, E>(fx, row, tw, th, mk, [&](int kp, cx<double> Zk, cx<double> Zn) {
            if (!o.ok) return;
            if (fa >= 0) o0[fa * wt_fs + kp] = make_cx((Zk.re + Zn.re) * ha, (Zk.im - Zn.im) * ha);
            if (fb >= 0) o0[fb * wt_fs + kp] = make_cx((Zk.im + Zn.im) * hb, -(Zk.re - Zn.re) * hb);
        });
        if (!wave_rows && th == 0) ex[0] = ex[1] = 0;
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
    q.lds = sizeof(cx<double>) * ((size_t)q.rb * fx.n + fx.twn) + sizeof(double) * mk + 2 * sizeof(int) * q.rb;
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
