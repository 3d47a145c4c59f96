// Proposals of the general move set, shared by the kernels that draw them on the device:
// the part of a move that does not depend on the current coordinates.
#pragma once
#include <hip/hip_runtime.h>

#include <cfloat>
#include <cstdint>

#include "mc_batch.hpp"
#include "philox.hpp"

namespace fmc {
namespace {

constexpr int kMaxKinds = 8; // move kinds per replica

__device__ __forceinline__ int pick(uint32_t x, int n) {
    return static_cast<int>((static_cast<uint64_t>(x) * static_cast<uint64_t>(n)) >> 32);
}

// Isotropic unit vector from z = 2u-1 and phi = 2 pi u'.
__device__ __forceinline__ void unit_vector(uint32_t zw, uint32_t pw, double* v) {
    const double z = 2.0 * u01_from32(zw) - 1.0;
    const double phi = 6.283185307179586 * u01_from32(pw);
    const double s = sqrt(1.0 - z * z);
    v[0] = s * cos(phi);
    v[1] = s * sin(phi);
    v[2] = z;
}

// Rotation by `angle` about the unit vector u (Rodrigues' formula), row-major.
__device__ __forceinline__ void rotation_matrix_sc(const double* u, double s, double c, double* R) {
    const double sa0 = u[0] * s, sa1 = u[1] * s, sa2 = u[2] * s;
    const double ca0 = u[0] * (1.0 - c), ca1 = u[1] * (1.0 - c), ca2 = u[2] * (1.0 - c);
    R[0] = ca0 * u[0] + c;
    R[1] = ca0 * u[1] - sa2;
    R[2] = ca0 * u[2] + sa1;
    R[3] = ca0 * u[1] + sa2;
    R[4] = ca1 * u[1] + c;
    R[5] = ca1 * u[2] - sa0;
    R[6] = ca0 * u[2] - sa1;
    R[7] = ca1 * u[2] + sa0;
    R[8] = ca2 * u[2] + c;
}

__device__ __forceinline__ void rotation_matrix(const double* u, double angle, double* R) {
    rotation_matrix_sc(u, sin(angle), cos(angle), R);
}

// Random part of one proposal: everything that does not depend on the current
// coordinates (move kind, target group and atoms, displacement, rotation, acceptance
// deviate).  Drawn kDraw moves ahead, one lane of wave 0 per move, so that the
// Philox blocks, the transcendental functions and the table lookups of 64 proposals
// overlap instead of forming one serial chain per move.
constexpr int kDraw = 64;

struct MoveDraw {
    int kind;                // -1: nothing moves (m = 0)
    int group, mlo, mhi;
    int internal, flags;     // flags: 1 translate, 2 rotate (kind 1); 4 the moved atom has bonds (kind 0)
    int atom0, atom1;        // kind 2: pivot origin and the bond partner
    double accept_u, neg_log_u, scale;
    double dir[3];           // kind 0: unit direction (times scale at the trial); kind 1: displacement
    double R[9];             // kind 1 rotation; kind 2: R[0], R[1] = sin, cos of the angle
};

// move.cpp:225-345 (atoms), move.cpp:1618-1689 (molecules), chainmove.cpp:216-268 (pivot)
__device__ void draw_move(MoveDraw& D, unsigned long long mvi, uint32_t replica, unsigned long long seed,
                          const MoveKindDev* kinds, int nkinds, unsigned long long total_weight,
                          const int* __restrict__ kind_groups, const int* __restrict__ gbegin,
                          const int* __restrict__ gsize, const int2* __restrict__ pivot_bonds,
                          const uint32_t* __restrict__ meta, const double* dpa, const int* __restrict__ bond_off) {
    const uint32_t c0 = static_cast<uint32_t>(mvi), c1 = static_cast<uint32_t>(mvi >> 32);
    const uint32_t key0 = static_cast<uint32_t>(seed), key1 = static_cast<uint32_t>(seed >> 32);
    const Philox4 ra = philox4x32_10(c0, c1, replica, 0u, key0, key1);
    const Philox4 rb = philox4x32_10(c0, c1, replica, 1u, key0, key1);
    const Philox4 rc = philox4x32_10(c0, c1, replica, 2u, key0, key1);
    D.accept_u = (static_cast<double>(rb.v[0] >> 5) * 67108864.0 + static_cast<double>(rb.v[1] >> 6)) *
                 1.1102230246251565e-16;
    D.neg_log_u = -log(D.accept_u);
    D.kind = -1;
    D.group = -1;
    D.mlo = D.mhi = 0;
    D.internal = 0;
    D.flags = 0;
    D.atom0 = D.atom1 = 0;
    D.scale = 0.0;
    const uint64_t sel = (static_cast<uint64_t>(rb.v[2]) * total_weight) >> 32;
    int k = 0;
    while (k + 1 < nkinds && sel >= kinds[k].cum) ++k;
    const MoveKindDev K = kinds[k];
    if (K.kind == 0) {
        const int g = kind_groups[K.group_first + (K.group_count == 1 ? 0 : pick(rc.v[3], K.group_count))];
        D.group = g;
        const int size = gsize[g];
        if (size > 0) {
            const int i = gbegin[g] + pick(ra.v[0], size);
            const int ti = static_cast<int>(meta[i] & 0xffu);
            const double step = dpa[ti] >= 0.0 ? dpa[ti] : K.dp;
            if (step > 0.0) {
                unit_vector(ra.v[1], ra.v[2], D.dir);
                D.scale = step * (static_cast<double>(ra.v[3]) * 2.3283064365386963e-10);
                D.kind = 0;
                D.mlo = i;
                D.mhi = i + 1;
                D.internal = 1;
                if (bond_off != nullptr && bond_off[i + 1] > bond_off[i]) D.flags = 4;
            }
        }
    } else if (K.kind == 1) {
        const int g = kind_groups[K.group_first + pick(ra.v[0], K.group_count)];
        D.group = g;
        const int size = gsize[g];
        if (size > 0) {
            if (K.dp > 0.0) {
                unit_vector(ra.v[1], ra.v[2], D.dir);
                D.scale = K.dp * (static_cast<double>(ra.v[3]) * 2.3283064365386963e-10);
                D.dir[0] *= D.scale;
                D.dir[1] *= D.scale;
                D.dir[2] *= D.scale;
                D.flags |= 1;
            }
            if (K.dprot > DBL_EPSILON) {
                double axis[3];
                unit_vector(rc.v[0], rc.v[1], axis);
                rotation_matrix(axis, K.dprot * (u01_from32(rc.v[2]) - 0.5), D.R);
                D.flags |= 2;
            }
            if (D.flags) {
                D.kind = 1;
                D.mlo = gbegin[g];
                D.mhi = D.mlo + size;
            }
        }
    } else {
        const int g = kind_groups[K.group_first + pick(ra.v[0], K.group_count)];
        D.group = g;
        const int size = gsize[g], b0 = gbegin[g];
        if (size > 2 && K.bond_count > 0 && fabs(K.dprot) > 1e-9) {
            const int2 bd = pivot_bonds[K.bond_first + pick(rc.v[3], K.bond_count)];
            int atom0 = b0 + bd.x, atom1 = b0 + bd.y;
            int slo, shi;
            if (u01_from32(rb.v[3]) > 0.5) {
                slo = atom1 + 1;
                shi = b0 + size;
                const int tmp = atom0;
                atom0 = atom1;
                atom1 = tmp;
            } else {
                slo = b0;
                shi = atom0;
            }
            if (shi > slo) {
                const double angle = K.dprot * (u01_from32(rc.v[2]) - 0.5);
                D.R[0] = sin(angle);
                D.R[1] = cos(angle);
                D.atom0 = atom0;
                D.atom1 = atom1;
                D.kind = 2;
                D.mlo = slo;
                D.mhi = shi;
                D.internal = 1;
            }
        }
    }
}

} // namespace
} // namespace fmc
