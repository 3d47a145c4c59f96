// Device-side pair arithmetic shared by the per-move kernels and the
// device-resident Metropolis kernels.  Formulas follow the reference's pair
// potentials (potentials.h:42-49 LJ, 151-160 WCA, 203-207 hard sphere, 472-476
// plain Coulomb, 591-598 CoulombGalore wrapper) and the orthogonal minimum image
// (geometry.h:429-485).
#pragma once
#include <hip/hip_runtime.h>

#include "engine.hpp"

namespace fmc {

struct Box {
    double L[3], half[3];
};

__device__ __forceinline__ double min_image(double d, double L, double half) {
    if (d > half) d -= L;
    else if (d < -half) d += L;
    return d;
}

__device__ __forceinline__ double dist2(const Box& b, double ax, double ay, double az, double bx, double by,
                                        double bz) {
    const double dx = min_image(ax - bx, b.L[0], b.half[0]);
    const double dy = min_image(ay - by, b.L[1], b.half[1]);
    const double dz = min_image(az - bz, b.L[2], b.half[2]);
    return dx * dx + dy * dy + dz * dz;
}

// Squared distance to the nearest image by rounding: at most that of dist2 (equal to it up
// to rounding for coordinates inside the box) in half its instructions, to tell far pairs
// from near ones before dist2 is taken.
__device__ __forceinline__ double near_dist2(const Box& b, const double inv[3], double ax, double ay, double az,
                                             double bx, double by, double bz) {
    double dx = ax - bx, dy = ay - by, dz = az - bz;
    dx = fma(-b.L[0], rint(dx * inv[0]), dx);
    dy = fma(-b.L[1], rint(dy * inv[1]), dy);
    dz = fma(-b.L[2], rint(dz * inv[2]), dz);
    return dx * dx + dy * dy + dz * dz;
}

// e^{2 pi i n x / L} with inv = 1 / L, the phase e^{i k r} of one axis.  The angle is formed
// in revolutions, so that its reduction is exact and short: 91 instructions against 200 of
// sincos(2 pi n / L x), whose argument has one rounding more.
__device__ __forceinline__ double2 axis_phase(int n, double x, double inv) {
    double sn, cs;
    sincospi(2.0 * (static_cast<double>(n) * (x * inv)), &sn, &cs);
    return make_double2(cs, sn);
}

// Value at x of an Andrea spline (tabulate.h:184-202: interval by lower_bound, Horner from
// the top coefficient) whose search window is the `steps` knots from `lo`, a knot before the
// first one of x's bucket.  Within the window lower_bound's index advances once per knot
// below x, and the knots are increasing, so they are read independently and counted.  The
// buckets are fine enough that four knots cover nearly every window; the interval's lower
// knot is then one of the four in registers.  A pair energy is bound by its LDS reads, since
// all waves of a workgroup share one LDS: 14 reads with this window, 22 with 32 buckets per
// table and eight knots of which one was read again (1728 FP64 waters: 3.61 -> 3.30 ms for 200
// moves; the split kernel's 20000 Na/Cl, with the shorter phases: 3.39 -> 3.23 us per move,
// about the scatter of two builds).
// `knots` is padded with the last knot; `coeff` is 16-byte aligned.
__device__ __forceinline__ double spline_window(const double* __restrict__ knots, const double* __restrict__ coeff, int n,
                                                int lo, int steps, double x) {
    double v[4];
    int below = 0;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        v[s] = knots[lo + s];
        below += (s < steps && lo + s < n && v[s] < x) ? 1 : 0;
    }
    double k = below <= 1 ? v[0] : (below == 2 ? v[1] : (below == 3 ? v[2] : v[3]));
    int pos = lo + below - 1;
    if (steps > 4) { // uniform over the wave for one table
        for (int s = 4; s < steps; ++s) pos += (lo + s < n && knots[lo + s] < x) ? 1 : 0;
        pos = pos < 0 ? 0 : pos;
        k = knots[pos];
    }
    // lo's knot lies below x unless it is the first one; past the last interval (x beyond the
    // last knot) the value is not used, only its address kept in range
    pos = pos < 0 ? 0 : (pos > n - 2 ? n - 2 : pos);
    const double2* c = reinterpret_cast<const double2*>(coeff + 6 * pos);
    const double2 c01 = c[0], c23 = c[1], c45 = c[2];
    const double z = x - k;
    double s = z * c45.y;
    s = z * (s + c45.x);
    s = z * (s + c23.y);
    s = z * (s + c23.x);
    s = z * (s + c01.y);
    return s + c01.x;
}

// The Coulomb short-range function's spline at q.
__device__ __forceinline__ double coulomb_spline(const DevCoulomb& c, double q) {
    int b = static_cast<int>(q * static_cast<double>(kSplineBuckets));
    b = b < 0 ? 0 : (b > kSplineBuckets - 1 ? kSplineBuckets - 1 : b);
    const int lo = static_cast<int>(c.bucket[b]) - 1;
    return spline_window(c.knots, c.coeff, c.nknots, lo < 0 ? 0 : lo, c.spline_steps, q);
}

// Coulomb short-range part of one pair (kT).
__device__ __forceinline__ double coulomb_pair(const DevCoulomb& c, double qa, double qb, double r2) {
    if (c.scheme == kCoulPM) return c.lB * qa * qb / sqrt(r2);
    const double r = sqrt(r2) + 2.220446049250313e-16;
    if (c.scheme == kCoulPlain) return c.lB * (qa * qb / r);
    if (!(r < c.rc)) return 0.0;
    const double q = r * c.rc_inv;
    double s;
    if (c.splined) s = coulomb_spline(c, q);
    else if (c.scheme == kCoulEwald) s = erfc(c.alpha * c.rc * q);
    else {
        const double q5 = q * q * q * q * q;
        s = 1.0 - 1.75 * q + 5.25 * q5 - 7.0 * q5 * q + 2.5 * q5 * q * q;
    }
    return c.lB * (qa * qb / r * s);
}

// Additive pair energy u = LJ + WCA + HS + Coulomb (absent terms have zero parameters).
__device__ __forceinline__ double pair_energy_exact(const DevPair& p, const DevCoulomb& c, double qa, double qb,
                                                    double r2) {
    double u = 0.0;
    if (p.lj_e4 != 0.0) {
        double x = p.lj_s2 / r2;
        x = x * x * x;
        u = u + p.lj_e4 * (x * x - x);
    }
    if (p.wca_e4 != 0.0 && !(r2 > p.wca_s2 * 1.2599210498948732)) {
        double x = p.wca_s2 / r2;
        x = x * x * x;
        u = u + p.wca_e4 * (x * x - x + 0.25);
    }
    if (r2 < p.hs_s2) u = u + __builtin_huge_val();
    if (p.coul != 0.0) u = u + coulomb_pair(c, qa, qb, r2);
    return u;
}

// Andrea spline of a nonbonded_splined table at r2 in (rmin2, rmax2).
__device__ __forceinline__ double spline_table_eval(const DevSplineTable& T, double r2) {
    int b = static_cast<int>((r2 - T.x0) * T.inv_w);
    b = b < 0 ? 0 : (b > kSplBuckets - 1 ? kSplBuckets - 1 : b);
    const int lo = static_cast<int>(T.bucket[b]) - 1;
    return spline_window(T.knots, T.coeff, T.n, lo < 0 ? 0 : lo, T.steps, r2);
}

// SplinedPotential::operator() (potentials.h:807-823): zero from rmax on, the spline
// above rmin, +inf below rmin with hard-sphere repulsion, else the exact energy.
// `below` is true when the exact energy is needed (r2 <= rmin2, no hard sphere).
__device__ __forceinline__ double splined_pair(const DevSplineTable& T, double r2, bool& below) {
    below = false;
    if (r2 >= T.rmax2) return 0.0;
    if (r2 > T.rmin2) return spline_table_eval(T, r2);
    if (T.hs) return __builtin_huge_val();
    below = true;
    return 0.0;
}

// splined_pair without branches, for several pairs evaluated side by side: the table is
// read for every lane (clamped to its range) and the result selected.
__device__ __forceinline__ double splined_pair_select(const DevSplineTable& T, double r2, bool& below) {
    const double lo = T.rmin2, hi = T.rmax2;
    const bool in = r2 > lo, out = r2 >= hi;
    const double u = spline_table_eval(T, out ? hi : (in ? r2 : lo));
    const bool hs = T.hs != 0;
    below = !in && !out && !hs;
    return out ? 0.0 : (in ? u : (hs ? __builtin_huge_val() : 0.0));
}

// The nonbonded term's pair energy: splined when the term is nonbonded_splined.
__device__ __forceinline__ double pair_energy(const DevPair& p, const DevCoulomb& c, double qa, double qb,
                                              double r2) {
    if (c.nspl > 0) {
        bool below;
        const double u = splined_pair(c.spl[p.spl], r2, below);
        if (!below) return u;
    }
    return pair_energy_exact(p, c, qa, qb, r2);
}

// Copy of a struct into LDS by all threads of the block, 16 bytes per thread and step.
template <class T>
__device__ __forceinline__ void lds_copy(T& dst, const T* __restrict__ src, int tid, int nthreads) {
    static_assert(sizeof(T) % 16 == 0 && alignof(T) >= 16, "16-byte granules");
    const uint4* s = reinterpret_cast<const uint4*>(src);
    uint4* d = reinterpret_cast<uint4*>(&dst);
    for (int i = tid; i < static_cast<int>(sizeof(T) / 16); i += nthreads) d[i] = s[i];
}

// Lane `lane` (uniform) of x, in every lane.
__device__ __forceinline__ double readlane_f64(double x, int lane) {
    const long long b = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_readlane(static_cast<int>(b), lane);
    const int hi = __builtin_amdgcn_readlane(static_cast<int>(b >> 32), lane);
    return __longlong_as_double((static_cast<long long>(hi) << 32) | static_cast<unsigned>(lo));
}

// Sum of x over the 64 lanes of a wave, the same value in every lane and the same order
// of additions on every call: DPP moves within rows of 16 lanes (pair and quad swaps,
// half-row and row mirrors; no LDS round trip), then the four row sums read from lanes
// 0, 16, 32 and 48.  Every lane of the wave must be active.
__device__ __forceinline__ double wave_sum(double x) {
    x += __builtin_amdgcn_update_dpp(0.0, x, 0xB1, 0xF, 0xF, false);  // quad_perm [1,0,3,2]
    x += __builtin_amdgcn_update_dpp(0.0, x, 0x4E, 0xF, 0xF, false);  // quad_perm [2,3,0,1]
    x += __builtin_amdgcn_update_dpp(0.0, x, 0x141, 0xF, 0xF, false); // row_half_mirror
    x += __builtin_amdgcn_update_dpp(0.0, x, 0x140, 0xF, 0xF, false); // row_mirror
    const double r0 = readlane_f64(x, 0), r1 = readlane_f64(x, 16);
    const double r2 = readlane_f64(x, 32), r3 = readlane_f64(x, 48);
    return (r0 + r1) + (r2 + r3);
}

// Barrier of the block that orders LDS only: global loads in flight stay in flight (the full
// barrier waits for them).
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Inclusive prefix sum of x over the 64 lanes of a wave (DPP row shifts, then the row and
// half-wave broadcasts; no LDS).  Every lane of the wave must be active.
__device__ __forceinline__ int wave_scan(int x) {
    x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xF, 0xF, false); // row_shr:1
    x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xF, 0xF, false); // row_shr:2
    x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xF, 0xF, false); // row_shr:4
    x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xF, 0xF, false); // row_shr:8
    x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xA, 0xF, false); // row_bcast:15
    x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xC, 0xF, false); // row_bcast:31
    return x;
}

// Wavefront (64 lanes) sum, then across the block's waves.
template <int kThreads>
__device__ __forceinline__ double block_sum(double v, double* lds) {
    v = wave_sum(v);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    __syncthreads();
    if (lane == 0) lds[wave] = v;
    __syncthreads();
    double s = 0.0;
    if (threadIdx.x == 0) {
        for (int w = 0; w < kThreads / 64; ++w) s += lds[w];
    }
    return s; // valid in thread 0
}

// Intra-molecular pair exclusion (MoleculeData::isPairExcluded) from per-particle
// sorted partner lists; no lists means no exclusions.
__device__ __forceinline__ bool pair_excluded(const int* __restrict__ off, const int* __restrict__ list, int a, int b) {
    if (off == nullptr) return false;
    int lo = off[a], hi = off[a + 1];
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        const int v = list[mid];
        if (v == b) return true;
        if (v < b) lo = mid + 1;
        else hi = mid;
    }
    return false;
}

// GroupCutoff::cut's squared cutoff (energy.h:761-768) for two groups' flag words
// (molecule type from bit 8) from the per-pair table of molecule types.
__device__ __forceinline__ double g2g_cutoff2(const double* __restrict__ table, int nmol, int flags_a, int flags_b) {
    return table[(flags_a >> 8) * nmol + (flags_b >> 8)];
}

__device__ __forceinline__ int unpack_n(int packed, int which) {
    return static_cast<int>(static_cast<signed char>((packed >> (8 * which)) & 0xff));
}

} // namespace fmc
