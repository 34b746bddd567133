// dgpu_hot.hpp -- pieces shared by the transform kernels of one RK substep
// (dgpu_hot_z.hip: zinv, zfwd_nl; dgpu_hot_x.hip: xfused, vmax).
#pragma once

#include <cstdlib>
#include <cstring>
#include <type_traits>

#include "dgpu_kernels.hpp"

namespace dgpu {

namespace {

template <typename TO, typename FROM>
__device__ __forceinline__ cx<TO> cvt_(cx<FROM> a) { return make_cx<TO>(TO(a.re), TO(a.im)); }

// Kept slot of z frequency index f (0..NZ-1), or -1 in the dealiasing gap
// (slot K <= NKZ holds kz = K, slot K > NKZ holds kz = K - (TNKZ+1),
// for/mpi.f:1602-1606).
__device__ __forceinline__ int slot_of_freq(int f, int nz, int nkz, int tnkz)
{
    if (f <= nkz) return f;
    if (f >= nz - nkz) return f - nz + tnkz + 1;
    return -1;
}

template <int NTH>
struct XCount {
    static constexpr int nin = 3 + NTH;         // u1 u2 u3 th...
    static constexpr int npi = (nin + 1) / 2;   // backward pairs
    static constexpr int npo = (8 + 3 * NTH + 1) / 2;  // forward pairs of the products
};

}  // namespace

// The plans the kernels are also built for at compile time (PID > 0).
__device__ constexpr IpLen kDevConstPlans[] = {const_plan(0),  const_plan(1),  const_plan(2),  const_plan(3),
                                               const_plan(4),  const_plan(5),  const_plan(6),  const_plan(7),
                                               const_plan(8),  const_plan(9),  const_plan(10), const_plan(11),
                                               const_plan(12), const_plan(13), const_plan(14), const_plan(15),
                                               const_plan(16), const_plan(17), const_plan(18), const_plan(19)};
static_assert(sizeof(kDevConstPlans) / sizeof(IpLen) == (size_t)kNumConstPlans, "one entry per compile-time plan");

template <int PID>
__device__ __forceinline__ const IpLen &plan_ref(const IpLen &rt)
{
    if constexpr (PID == 0)
        return rt;
    else
        return kDevConstPlans[PID];
}

#define DGPU_DISPATCH_IPE(E_, CALL)                                \
    switch (E_) {                                                  \
    case 4: { constexpr int EE = 4; CALL; } break;                 \
    case 6: { constexpr int EE = 6; CALL; } break;                 \
    case 8: { constexpr int EE = 8; CALL; } break;                 \
    case 12: { constexpr int EE = 12; CALL; } break;               \
    case 16: { constexpr int EE = 16; CALL; } break;               \
    case 24: { constexpr int EE = 24; CALL; } break;               \
    default: break;                                                \
    }

// the x plans of FP64: at most 12 values per thread
#define DGPU_DISPATCH_XE64(E_, CALL)                               \
    switch (E_) {                                                  \
    case 4: { constexpr int EE = 4; CALL; } break;                 \
    case 6: { constexpr int EE = 6; CALL; } break;                 \
    case 8: { constexpr int EE = 8; CALL; } break;                 \
    case 12: { constexpr int EE = 12; CALL; } break;               \
    default: break;                                                \
    }

static inline int z_lw(int t)
{
    int lw = 0;
    while ((2 << lw) * t <= 256) ++lw;
    return lw;
}

// Compile-time plans each kernel family is built for, per precision (ids of
// kConstPlanSpecs): the x and z plans of 64, 96, 128, 192, 256 and 384 in both
// precisions.  On a run-time plan the stage loops do not unroll and every index
// is computed with run-time divisors: one RK3 step at 128x129x128 FP64 726 ->
// 667 us, 192x129x192 FP64 1833 -> 1713 and mixed 1055 -> 949 us with the x
// kernel on the compile-time plan.
template <int... P>
struct PidList {};
template <typename T>
using XPids = std::conditional_t<sizeof(T) == 4, PidList<2, 3, 5, 13, 14, 17>, PidList<1, 2, 4, 12, 18, 19>>;
// the FP64 pair transforms (dgpu_pairs.hip) and the LES products
using XPids64 = XPids<double>;
template <typename T>
using ZPids = PidList<6, 8, 9, 10, 15, 16>;

// Calls fn(std::integral_constant<int, P>) for the P of the list equal to
// pid; false when pid is not in the list.
template <class F, int... P>
static bool with_pid(int pid, PidList<P...>, F &&fn)
{
    bool done = false;
    ((!done && pid == P ? (fn(std::integral_constant<int, P>{}), done = true) : false), ...);
    return done;
}

// The last forward (DIT) stage of an x row holding the transform of a + i b
// (a plan with R_0 = E/2): thread th takes groups th and L0 - th (0 and L0/2
// for th = 0), so it holds Z(k) and Z(NX - k) of its frequencies, and calls
// emit(k, Z(k), Z(NX - k)) for the kept ones.
template <typename T, int E, class F>
__device__ __forceinline__ void x_split(const IpLen &fx, const cx<T> *row, const cx<T> *tw, int th, int mk, F &&emit)
{
    constexpr int R0 = E / 2;
    const int L0 = fx.span[0], TT = fx.t;
    const int ga = th, gb = th == 0 ? TT : L0 - th;
    cx<T> va[R0], vb[R0];
#pragma unroll
    for (int q = 0; q < R0; ++q) {
        va[q] = row[ip_swz(fx, ga + q * L0)];
        vb[q] = row[ip_swz(fx, gb + q * L0)];
    }
    ip_group<T, R0, -1, false>(va, tw + fx.twoff[0], ga);
    ip_group<T, R0, -1, false>(vb, tw + fx.twoff[0], gb);
#pragma unroll
    for (int q = 0; q < R0; ++q) {
        const int ka = ga + q * L0;
        if (ka < mk) emit(ka, va[q], ga == 0 ? va[(R0 - q) % R0] : vb[R0 - 1 - q]);
        const int kb = gb + q * L0;
        if (kb < mk) emit(kb, vb[q], th == 0 ? vb[R0 - 1 - q] : va[R0 - 1 - q]);
    }
}

// Id of the compile-time plan equal to f, or 0 (dgpu_hot_z.hip).
int const_plan_id(const IpLen &f);

// Planes per block of a sweeping kernel over `runs` fields of so many planes,
// alone on the device or among others (dgpu_hot_x.hip).
int sweep_rule(long rows, const int *planes, int runs, long slots, bool among = false);

// Blocks of a kernel that the whole device holds at once.
template <class K>
static long kernel_slots(K kernel, int threads, size_t lds)
{
    int per = 0, dev = 0, cus = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, kernel, threads, lds) != hipSuccess || per < 1) per = 1;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 1)
        cus = 256;
    (void)hipGetLastError();
    return (long)per * cus;
}

}  // namespace dgpu
