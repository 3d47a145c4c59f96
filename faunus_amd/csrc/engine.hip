// GPU energy engine: kernels and host orchestration for the plain path
// (one trial move per launch) — the drop-in for the reference's
// Nonbonded::energy(Change) (energy.h:1561-1577) and Ewald::updateState/energy
// (energy.cpp:564-587).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstddef>
#include <cstring>
#include <numeric>
#include <stdexcept>
#include <string>

#include "device_math.hpp"
#include "engine.hpp"

namespace fmc {

void check_hip(hipError_t e, const char* what) {
    if (e != hipSuccess) throw std::runtime_error(std::string(what) + ": " + hipGetErrorString(e));
}

namespace {

struct GroupTable {
    const int* flags;     // bit0 molecular (not atomic), bit1 rigid, molecule type from bit 8
    const double* cm;     // 3 per group (accepted state)
    const double* g2g2;   // squared cutoff per pair of molecule types (null: none)
    int nmol;
    const int* excl_off;  // per-particle excluded partners (null: none)
    const int* excl;
};

struct CellArgs {
    const int* count;
    const int* members;
    int nc0, nc1, nc2, cap;
    double inv0, inv1, inv2;
};

__device__ __forceinline__ int cell_coord(double x, double half, double inv_cell, int nc) {
    int c = static_cast<int>(floor((x + half) * inv_cell));
    c %= nc;
    if (c < 0) c += nc;
    return c;
}

// The DevCoulomb header and the `nspl` tables in use, by all threads of the block (the whole
// struct is 22.7 KB, a system without tables needs 5.7).
__device__ __forceinline__ void copy_coulomb(DevCoulomb& dst, const DevCoulomb* __restrict__ src, int nspl, int tid,
                                             int nthreads) {
    static_assert(offsetof(DevCoulomb, spl) % 16 == 0 && sizeof(DevSplineTable) % 16 == 0, "16-byte granules");
    const uint4* s = reinterpret_cast<const uint4*>(src);
    uint4* d = reinterpret_cast<uint4*>(&dst);
    const int words = static_cast<int>((offsetof(DevCoulomb, spl) + static_cast<size_t>(nspl) * sizeof(DevSplineTable)) / 16);
    for (int i = tid; i < words; i += nthreads) d[i] = s[i];
}

// Position of particle j in the moved set (sorted by index), or -1.
__device__ __forceinline__ int moved_slot(const MovedParticle* mp, int m, int j) {
    int lo = 0, hi = m;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (mp[mid].idx < j) lo = mid + 1;
        else hi = mid;
    }
    return lo < m && mp[lo].idx == j ? lo : -1;
}

// How the pair blocks of delta_kernel share the work: without a cell list, block b takes
// every j_blocks-th run of 256 particles from run b mod j_blocks on, against the b div
// j_blocks-th run of a_run moved atoms; with one, `lanes` lanes walk each (moved atom,
// state, cell).  The Ewald blocks build phase tables of `chunk` moved particles at a time.
struct PairSplit {
    int blocks, j_blocks, a_run, lanes, nspl, chunk;
};

// ------------------------------------------------------------------------------
// Fused per-move kernel.  Blocks [0, split.blocks) sum the pair energies of the
// affected pairs in the new and old state; blocks [split.blocks, ewald_end) update the
// trial structure factors Q_trial(k) = Q_acc(k) + dQ(k) and sum A_k|Q|^2 for both
// states.  The last block to finish reduces all block partials in a fixed order
// and writes the results to host-visible memory.
// A launch is a few microseconds of latencies, so the kernel avoids what waits: partials and
// results travel as agent- and system-scope stores completed by a wait (a fence would write
// back the L2 of each block's XCD), the last block reads all partials at once (one thread
// read them one after the other: 88 of them at K = 17328), and the pairs are spread over as
// many lanes as there are.  Kernel time before -> now: 200 ions (cell list of 27 cells) 18.2 -> 8.8 us,
// 20000 Na/Cl 23.6 -> 8.3 us, 1000 waters with a group cutoff 43.9 -> 13.5 us.
// ------------------------------------------------------------------------------
template <bool kGroups, bool kCells>
__global__ __launch_bounds__(kBlock) void delta_kernel(
    const double4* __restrict__ pos, const uint32_t* __restrict__ meta, int n, const DevPair* __restrict__ pairs_g,
    int ntypes, const DevCoulomb* __restrict__ coul_g, Box box, GroupTable groups, CellArgs cells, MoveArgs mv,
    PairSplit split, const int* __restrict__ kn, const double* __restrict__ ak, const double2* __restrict__ q_acc,
    double2* __restrict__ q_trial, int nk, int ncut, double* __restrict__ partials, unsigned* __restrict__ ticket,
    DeltaResult* __restrict__ out, unsigned long long seq, double rec_prefactor, double cm_new_x, double cm_new_y,
    double cm_new_z, double cm_old_x, double cm_old_y, double cm_old_z, int ewald_end,
    const int* __restrict__ bond_off, const DevBond* __restrict__ bonds) {
    __shared__ DevPair s_pairs[kMaxTypes * kMaxTypes];
    __shared__ DevCoulomb s_coul;
    __shared__ MovedParticle s_moved[kPhaseTableMoved];
    __shared__ double s_red[6][kBlock / 64];
    __shared__ bool s_last;
    extern __shared__ double2 s_phase[]; // Ewald phase tables of up to kPhaseTableMoved moved particles

    const int tid = threadIdx.x;
    const int m = mv.m;
    const MovedParticle* moved = (m <= kMaxInlineMoved) ? mv.inl : mv.ext;
    const int m_lds = m < kPhaseTableMoved ? m : kPhaseTableMoved;
    for (int i = tid; i < m_lds; i += kBlock) s_moved[i] = moved[i];
    const MovedParticle* mp = (m <= kPhaseTableMoved) ? s_moved : moved;

    double acc_new = 0.0, acc_old = 0.0;
    const bool is_pair_block = static_cast<int>(blockIdx.x) < split.blocks;
    if (is_pair_block) {
        for (int i = tid; i < ntypes * ntypes; i += kBlock) s_pairs[i] = pairs_g[i];
        copy_coulomb(s_coul, coul_g, split.nspl, tid, kBlock);
        __syncthreads();
        const bool single = mv.change_group >= 0;
        // pair of a moved particle in group gi (the changed group when there is one) with a
        // static particle in group gj
        auto allowed = [&](int gi, int gj, bool new_state) -> bool {
            if (gi == gj) return single && mv.internal && (!kGroups || !(groups.flags[gi] & 2));
            if (!kGroups) return true;
            if (groups.g2g2 && (groups.flags[gi] & 1) && (groups.flags[gj] & 1)) { // GroupCutoff::cut (energy.h:761-768)
                const double* cj = groups.cm + 3 * gj;
                const double r2 = new_state ? dist2(box, cm_new_x, cm_new_y, cm_new_z, cj[0], cj[1], cj[2])
                                            : dist2(box, cm_old_x, cm_old_y, cm_old_z, cj[0], cj[1], cj[2]);
                return r2 < g2g_cutoff2(groups.g2g2, groups.nmol, groups.flags[gi], groups.flags[gj]);
            }
            return true;
        };
        // pair of two moved particles, each at its state's coordinates
        auto moved_pair = [&](const MovedParticle& A, const MovedParticle& B) {
            // several moved groups are atomic (molecular multi-group changes are rejected on the host)
            const bool ok = A.gid != B.gid || (single && mv.internal &&
                                               (!kGroups || (!(groups.flags[A.gid] & 2) &&
                                                             !pair_excluded(groups.excl_off, groups.excl, A.idx, B.idx))));
            if (!ok) return;
            const DevPair& p = s_pairs[A.type * ntypes + B.type];
            acc_new += pair_energy(p, s_coul, A.newp.w, B.newp.w,
                                   dist2(box, A.newp.x, A.newp.y, A.newp.z, B.newp.x, B.newp.y, B.newp.z));
            acc_old += pair_energy(p, s_coul, A.oldp.w, B.oldp.w,
                                   dist2(box, A.oldp.x, A.oldp.y, A.oldp.z, B.oldp.x, B.oldp.y, B.oldp.z));
        };
        if (!kCells) {
            const int a0 = static_cast<int>(blockIdx.x) / split.j_blocks * split.a_run, a1 = min(m, a0 + split.a_run);
            for (int j = (static_cast<int>(blockIdx.x) % split.j_blocks) * kBlock + tid; j < n; j += split.j_blocks * kBlock) {
                const double4 pj = pos[j];
                const uint32_t mj = meta[j];
                const int tj = static_cast<int>(mj & 0xffu), gj = static_cast<int>(mj >> 8);
                const int jm = moved_slot(mp, m, j);
                if (jm >= 0) {
                    for (int a = a0; a < min(a1, jm); ++a) moved_pair(mp[a], mp[jm]);
                    continue;
                }
                const bool ok_new = !single || allowed(mv.change_group, gj, true);
                const bool ok_old = !single || allowed(mv.change_group, gj, false);
                if (!ok_new && !ok_old) continue;
                for (int a = a0; a < a1; ++a) {
                    const MovedParticle& M = mp[a];
                    if (!single && M.gid == gj) continue;
                    if (kGroups && M.gid == gj && pair_excluded(groups.excl_off, groups.excl, M.idx, j)) continue;
                    const DevPair& p = s_pairs[M.type * ntypes + tj];
                    if (ok_new)
                        acc_new += pair_energy(p, s_coul, M.newp.w, pj.w,
                                               dist2(box, M.newp.x, M.newp.y, M.newp.z, pj.x, pj.y, pj.z));
                    if (ok_old)
                        acc_old += pair_energy(p, s_coul, M.oldp.w, pj.w,
                                               dist2(box, M.oldp.x, M.oldp.y, M.oldp.z, pj.x, pj.y, pj.z));
                }
            }
        } else {
            // Stencils of 27 cells around each moved particle's new and old position;
            // candidates are evaluated only for the state whose stencil holds them.
            const int first = (static_cast<int>(blockIdx.x) * kBlock + tid) / split.lanes;
            for (int job = first; job < m * 54; job += split.blocks * kBlock / split.lanes) {
                const int a = job / 54;
                const int s = (job / 27) & 1; // 0: new, 1: old
                const int c = job % 27;
                const MovedParticle& M = mp[a];
                const double4 P = s == 0 ? M.newp : M.oldp;
                const int cx = (cell_coord(P.x, box.half[0], cells.inv0, cells.nc0) + (c % 3) - 1 + cells.nc0) % cells.nc0;
                const int cy = (cell_coord(P.y, box.half[1], cells.inv1, cells.nc1) + ((c / 3) % 3) - 1 + cells.nc1) % cells.nc1;
                const int cz = (cell_coord(P.z, box.half[2], cells.inv2, cells.nc2) + (c / 9) - 1 + cells.nc2) % cells.nc2;
                const int cell = (cz * cells.nc1 + cy) * cells.nc0 + cx;
                const int cnt = cells.count[cell];
                for (int k = tid & (split.lanes - 1); k < cnt; k += split.lanes) {
                    const int j = cells.members[cell * cells.cap + k];
                    const double4 pj = pos[j];
                    const uint32_t mj = meta[j];
                    if (moved_slot(mp, m, j) >= 0) continue; // moved <-> moved handled below
                    const int tj = static_cast<int>(mj & 0xffu);
                    const int gj = static_cast<int>(mj >> 8);
                    if (!allowed(M.gid, gj, s == 0)) continue;
                    if (kGroups && M.gid == gj && pair_excluded(groups.excl_off, groups.excl, M.idx, j)) continue;
                    const DevPair& p = s_pairs[M.type * ntypes + tj];
                    const double u = pair_energy(p, s_coul, P.w, pj.w, dist2(box, P.x, P.y, P.z, pj.x, pj.y, pj.z));
                    if (s == 0) acc_new += u;
                    else acc_old += u;
                }
            }
            if (blockIdx.x == 0)
                for (int pairidx = tid; pairidx < m * m; pairidx += kBlock) {
                    const int a = pairidx / m, b = pairidx % m;
                    if (a < b) moved_pair(mp[a], mp[b]);
                }
        }
    } else if (static_cast<int>(blockIdx.x) >= ewald_end) {
        // Bonded::internalGroupEnergy (energy.cpp:1068-1088): bonds with at least one
        // moved atom, each counted once, in both states; only for internal changes.
        __syncthreads();
        if (mv.internal) {
            for (int a = tid; a < m; a += kBlock) {
                const MovedParticle& A = mp[a];
                for (int e = bond_off[A.idx]; e < bond_off[A.idx + 1]; ++e) {
                    const DevBond B = bonds[e];
                    const int om = moved_slot(mp, m, B.other);
                    if (om >= 0 && om < a) continue; // the pair is visited from the lower moved atom
                    const double4 on = om >= 0 ? mp[om].newp : pos[B.other];
                    const double4 oo = om >= 0 ? mp[om].oldp : on;
                    const double xn = B.req - sqrt(dist2(box, A.newp.x, A.newp.y, A.newp.z, on.x, on.y, on.z));
                    const double xo = B.req - sqrt(dist2(box, A.oldp.x, A.oldp.y, A.oldp.z, oo.x, oo.y, oo.z));
                    acc_new += B.half_k * xn * xn;
                    acc_old += B.half_k * xo * xo;
                }
            }
        }
    } else if (nk > 0) {
        // Ewald partial update (energy.cpp:219-247): dQ(k) = sum_i q_i (e^{ik.r_new} - e^{ik.r_old}),
        // with e^{i k_a(n) r_a}, n in [-ncut, ncut], per moved particle, state and axis in
        // LDS, split.chunk particles at a time; a thread holds two k-vectors
        const int eb = static_cast<int>(blockIdx.x) - split.blocks;
        const int e_blocks = ewald_end - split.blocks;
        const int width = 2 * ncut + 1;
        for (int k0 = eb * 2 * kBlock; k0 < nk; k0 += e_blocks * 2 * kBlock) {
            double dre[2] = {0.0, 0.0}, dim[2] = {0.0, 0.0};
            int packed[2];
            double2 qa[2];
            double A[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int k = min(k0 + i * kBlock + tid, nk - 1);
                packed[i] = kn[k];
                qa[i] = q_acc[k];
                A[i] = ak[k];
            }
            for (int c0 = 0; c0 < m; c0 += split.chunk) {
                const int cm = min(split.chunk, m - c0);
                __syncthreads(); // the moved particles, or the previous tables, are consumed
                for (int e = tid; e < cm * 6 * width; e += kBlock) {
                    const int nn = e % width - ncut;
                    const int axis = (e / width) % 3;
                    const int st = (e / (3 * width)) & 1;
                    const MovedParticle& M = mp[c0 + e / (6 * width)];
                    const double4 P = st == 0 ? M.newp : M.oldp;
                    s_phase[e] = axis_phase(nn, axis == 0 ? P.x : (axis == 1 ? P.y : P.z), 1.0 / box.L[axis]);
                }
                __syncthreads();
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const int nx = unpack_n(packed[i], 0) + ncut, ny = unpack_n(packed[i], 1) + ncut,
                              nz = unpack_n(packed[i], 2) + ncut;
                    for (int a = 0; a < cm; ++a) {
#pragma unroll
                        for (int st = 0; st < 2; ++st) {
                            const double2* t = s_phase + (a * 2 + st) * 3 * width;
                            const double2 ex = t[nx], ey = t[width + ny], ez = t[2 * width + nz];
                            const double re1 = ex.x * ey.x - ex.y * ey.y;
                            const double im1 = ex.x * ey.y + ex.y * ey.x;
                            const double q = st == 0 ? mp[c0 + a].newp.w : -mp[c0 + a].oldp.w;
                            dre[i] += q * (re1 * ez.x - im1 * ez.y);
                            dim[i] += q * (re1 * ez.y + im1 * ez.x);
                        }
                    }
                }
            }
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int k = k0 + i * kBlock + tid;
                if (k >= nk) continue;
                const double2 qt = make_double2(qa[i].x + dre[i], qa[i].y + dim[i]);
                q_trial[k] = qt;
                acc_new += A[i] * (qt.x * qt.x + qt.y * qt.y);
                acc_old += A[i] * (qa[i].x * qa[i].x + qa[i].y * qa[i].y);
            }
        }
    }

    // block partials: stored at agent scope, complete before the block's ticket
    const double bn = wave_sum(acc_new), bo = wave_sum(acc_old);
    if ((tid & 63) == 0) {
        s_red[0][tid >> 6] = bn;
        s_red[1][tid >> 6] = bo;
    }
    __syncthreads();
    if (tid == 0) {
        double v0 = 0.0, v1 = 0.0;
        for (int w = 0; w < kBlock / 64; ++w) {
            v0 += s_red[0][w];
            v1 += s_red[1][w];
        }
        __hip_atomic_store(partials + 2 * blockIdx.x, v0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(partials + 2 * blockIdx.x + 1, v1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        const unsigned t = __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        s_last = (t == gridDim.x - 1);
    }
    __syncthreads();
    if (!s_last) return;
    // last block: fixed-order reduction of the pair, Ewald and bond partials
    double v[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    for (int b = tid; b < static_cast<int>(gridDim.x); b += kBlock) {
        const double x = __hip_atomic_load(partials + 2 * b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const double y = __hip_atomic_load(partials + 2 * b + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const int r = b < split.blocks ? 0 : (b < ewald_end ? 2 : 4);
#pragma unroll
        for (int k = 0; k < 6; k += 2) {
            v[k] += r == k ? x : 0.0;
            v[k + 1] += r == k ? y : 0.0;
        }
    }
#pragma unroll
    for (int r = 0; r < 6; ++r) {
        const double x = wave_sum(v[r]);
        if ((tid & 63) == 0) s_red[r][tid >> 6] = x;
    }
    __syncthreads();
    if (tid < 6) {
        double x = 0.0;
        for (int w = 0; w < kBlock / 64; ++w) x += s_red[tid][w];
        if (tid == 2 || tid == 3) x *= rec_prefactor;
        // DeltaResult: pair, reciprocal and bond sums, each new and old
        __hip_atomic_store(&out->pair_new + tid, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        if (tid == 0) {
            *ticket = 0u;
            __hip_atomic_store(&out->seq, seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    }
}

// Accept: write the moved particles' trial coordinates into the accepted state, the moved
// group's mass centre (cm_group >= 0) and move the particles between cells of the cell list
// (one wave, in order; its lanes search a cell's members together).
__global__ __launch_bounds__(64) void commit_kernel(double4* pos, MoveArgs mv, CellArgs cells, int* cell_of, int* overflow,
                                                    Box box, int use_cells, double* gcm, int cm_group, double cx, double cy,
                                                    double cz) {
    const int lane = threadIdx.x;
    const MovedParticle* moved = (mv.m <= kMaxInlineMoved) ? mv.inl : mv.ext;
    if (lane < 3 && cm_group >= 0) gcm[3 * cm_group + lane] = lane == 0 ? cx : (lane == 1 ? cy : cz);
    for (int a = lane; a < mv.m; a += 64) pos[moved[a].idx] = moved[a].newp;
    if (!use_cells) return;
    int* cnt = const_cast<int*>(cells.count);
    int* mem = const_cast<int*>(cells.members);
    for (int a = 0; a < mv.m; ++a) {
        const MovedParticle& M = moved[a];
        const int x = cell_coord(M.newp.x, box.half[0], cells.inv0, cells.nc0);
        const int y = cell_coord(M.newp.y, box.half[1], cells.inv1, cells.nc1);
        const int z = cell_coord(M.newp.z, box.half[2], cells.inv2, cells.nc2);
        const int cnew = (z * cells.nc1 + y) * cells.nc0 + x;
        const int cold = cell_of[M.idx];
        if (cnew == cold) continue;
        const int nold = cnt[cold], nn = cnt[cnew];
        const int last = mem[cold * cells.cap + max(nold - 1, 0)];
        int slot = -1;
        for (int k = 0; k < nold && slot < 0; k += 64) {
            const unsigned long long found = __ballot(k + lane < nold && mem[cold * cells.cap + min(k + lane, nold - 1)] == M.idx);
            if (found) slot = k + __builtin_ctzll(found);
        }
        __syncthreads(); // every lane has read the lists
        if (lane == 0) {
            if (slot >= 0) mem[cold * cells.cap + slot] = last;
            cnt[cold] = nold - 1;
            if (nn >= cells.cap) *overflow = 1;
            else {
                mem[cnew * cells.cap + nn] = M.idx;
                cnt[cnew] = nn + 1;
                cell_of[M.idx] = cnew;
            }
        }
        __syncthreads(); // the next particle sees the changed lists
    }
}

// Full structure factors Q(k) = sum_j q_j e^{ik.r_j} (energy.cpp:191-206) as a matrix
// product.  A column is one (nx, ny); with B_j = q_j e^{i kx xj} e^{i ky yj} the row sums
//   R = sum_j Re(B_j) {cos, sin}(kz zj),  I = sum_j Im(B_j) {cos, sin}(kz zj)
// give Q at +nz and -nz, so the work is a real product of [2 x columns, particles] by
// [particles, 2 (ncut + 1)]: two multiply-adds per k-vector and particle, and 3 (ncut + 1)
// sincos per particle and block in place of one sincos per k-vector and particle.
// A block takes kQCols x kCT columns (16 per wave and tile) and a slice of the particles;
// per chunk it writes the particles' axis tables to LDS, from which each wave forms its A
// operands (lane: column l mod 16, particle l div 16) and reads its B operands.  Columns
// are sorted by their largest nz, so that a wave's tiles skip the nz no column of it has.
// The slices' partial Q(k) are added in slice order by sum_q_kernel.
// N = 20000, K = 17328: 4455 us with one thread per k-vector and a sincos per particle (68
// blocks, latency bound), now 95 + 7 us (the products and the tables' sincos);
// N = 12288, K = 1661: 2784 -> 20 + 12 us.
constexpr int kQThreads = 512;
constexpr int kQCols = 16 * kQThreads / 64; // columns per block and column tile
constexpr int kQTiles = 3;                  // 16-wide tiles of (cos, sin) x nz per wave
constexpr int kQChunk = 32;                 // particles per LDS chunk, at most

typedef double f64x4 __attribute__((ext_vector_type(4)));

template <int kCT>
__global__ __launch_bounds__(kQThreads) void full_q_kernel(const double4* __restrict__ pos, int n,
                                                           const QColumn* __restrict__ cols, int ncol, int ncut,
                                                           int chunk, int slice, int nk, Box box,
                                                           double2* __restrict__ partial) {
    extern __shared__ double2 s_tab[]; // [chunk][3][ncut + 1], the x table times the charge
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int w = ncut + 1, row = 3 * w;
    const double inv[3] = {1.0 / box.L[0], 1.0 / box.L[1], 1.0 / box.L[2]};
    const int c0 = kQTiles * 16 * static_cast<int>(blockIdx.z); // first (cos, sin) x nz entry of this block
    int nx[kCT], ny[kCT], tiles[kCT];
    double sy[kCT];
    f64x4 re[kCT][kQTiles], im[kCT][kQTiles];
    const int first = (static_cast<int>(blockIdx.x) * kCT * (kQThreads / 64) + wave * kCT) * 16;
#pragma unroll
    for (int ct = 0; ct < kCT; ++ct) {
        const int base = first + 16 * ct;
        const QColumn c = cols[min(base + (lane & 15), ncol - 1)];
        nx[ct] = c.nx;
        ny[ct] = c.ny < 0 ? -c.ny : c.ny;
        sy[ct] = c.ny < 0 ? -1.0 : 1.0;
        // the first column of a tile has its largest nz
        const int top = base < ncol ? 2 * (cols[base].nzmax + 1) - c0 : 0;
        tiles[ct] = __builtin_amdgcn_readfirstlane(top <= 0 ? 0 : min(kQTiles, (top + 15) / 16));
#pragma unroll
        for (int t = 0; t < kQTiles; ++t) re[ct][t] = im[ct][t] = f64x4{0.0, 0.0, 0.0, 0.0};
    }
    const int j1 = min(n, slice * (static_cast<int>(blockIdx.y) + 1));
    for (int base = slice * static_cast<int>(blockIdx.y); base < j1; base += chunk) {
        __syncthreads(); // the previous chunk's tables are consumed
        for (int e = tid; e < chunk * row; e += kQThreads) {
            const int j = e / row, r = e - j * row, axis = r / w;
            double2 v = make_double2(0.0, 0.0);
            if (base + j < j1) {
                const double4 p = pos[base + j];
                const double x = axis == 0 ? p.x : (axis == 1 ? p.y : p.z);
                v = axis_phase(r - axis * w, x, inv[axis]);
                if (axis == 0) v = make_double2(p.w * v.x, p.w * v.y);
            }
            s_tab[e] = v;
        }
        __syncthreads();
        for (int p = 0; p < chunk; p += 4) {
            const double2* tab = s_tab + (p + (lane >> 4)) * row;
            // entries past 2 (ncut + 1) belong to unused output columns: the next particle's
            // table, or the pad behind the last one
            const double* zt = reinterpret_cast<const double*>(tab + 2 * w) + c0 + (lane & 15);
            double bz[kQTiles];
#pragma unroll
            for (int t = 0; t < kQTiles; ++t) bz[t] = zt[16 * t];
#pragma unroll
            for (int ct = 0; ct < kCT; ++ct) {
                if (tiles[ct] == 0) continue;
                const double2 X = tab[nx[ct]], Y = tab[w + ny[ct]];
                const double yi = sy[ct] * Y.y;
                const double ar = X.x * Y.x - X.y * yi, ai = X.x * yi + X.y * Y.x;
#pragma unroll
                for (int t = 0; t < kQTiles; ++t)
                    if (t < tiles[ct]) {
                        re[ct][t] = __builtin_amdgcn_mfma_f64_16x16x4f64(ar, bz[t], re[ct][t], 0, 0, 0);
                        im[ct][t] = __builtin_amdgcn_mfma_f64_16x16x4f64(ai, bz[t], im[ct][t], 0, 0, 0);
                    }
            }
        }
    }
    // even lanes hold the cos sums of an nz and write Q(+nz), odd lanes its sin sums and
    // write Q(-nz); the partner's sums come by a pair swap.  Element r of lane l is column
    // 4 r + l div 16 of the tile, entry l mod 16.
    double2* out = partial + static_cast<size_t>(blockIdx.y) * static_cast<size_t>(nk);
#pragma unroll
    for (int ct = 0; ct < kCT; ++ct)
#pragma unroll
        for (int t = 0; t < kQTiles; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const double a = re[ct][t][r], b = im[ct][t][r];
                const double a2 = __builtin_amdgcn_update_dpp(0.0, a, 0xB1, 0xF, 0xF, false);
                const double b2 = __builtin_amdgcn_update_dpp(0.0, b, 0xB1, 0xF, 0xF, false);
                const int col = first + 16 * ct + 4 * r + (lane >> 4);
                const int nz = (c0 + 16 * t + (lane & 15)) >> 1;
                const bool odd = lane & 1;
                if (t >= tiles[ct] || col >= ncol || (odd && nz == 0)) continue;
                const QColumn c = cols[col];
                const int z = odd ? -nz : nz;
                const bool hole = c.nx == 0 && c.ny == 0; // k = 0 is left out
                if (z < c.nzmin || z > c.nzmax || (hole && z == 0)) continue;
                out[c.k0 + (z - c.nzmin) - (hole && z > 0 ? 1 : 0)] =
                    odd ? make_double2(a2 + b, b2 - a) : make_double2(a - b2, a2 + b);
            }
}

// Sum of the slices' partial structure factors, in slice order.
__global__ __launch_bounds__(kBlock) void sum_q_kernel(const double2* __restrict__ partial, int slices, int nk,
                                                       double2* __restrict__ q_out) {
    const int k = blockIdx.x * kBlock + threadIdx.x;
    if (k >= nk) return;
    double2 s = partial[k];
#pragma unroll 8
    for (int i = 1; i < slices; ++i) {
        const double2 v = partial[static_cast<size_t>(i) * static_cast<size_t>(nk) + static_cast<size_t>(k)];
        s.x += v.x;
        s.y += v.y;
    }
    q_out[k] = s;
}

// All pairs i < j (Change::everything, energy.h:1290-1299).  Block (x, y) pairs the
// particles i of tile x (one per thread) with those of run y of `len` particles; j is the
// same for every lane, so its coordinates come through scalar loads.  kCut: every pair
// energy is exactly zero beyond a distance, and `range2` lies just above its square; a wave
// whose 64 pairs are all farther goes on after the rounded distance.
// One block per tile over all later particles (79 blocks of up to 20000 steps, one wave
// per SIMD) took 5848 us at N = 20000 with the pair energy cut at 12 A, now 178 us; 4096
// waters with a group cutoff took 12528 us, now 521.
template <bool kGroups, bool kCut>
__global__ __launch_bounds__(kBlock) void all_pairs_kernel(const double4* __restrict__ pos,
                                                            const uint32_t* __restrict__ meta, int n,
                                                            const DevPair* __restrict__ pairs_g, int ntypes,
                                                            const DevCoulomb* __restrict__ coul_g, Box box,
                                                            GroupTable groups, int len, double range2,
                                                            double* __restrict__ partials) {
    __shared__ DevPair s_pairs[kMaxTypes * kMaxTypes];
    __shared__ DevCoulomb s_coul;
    __shared__ double s_red[kBlock / 64];
    const int part = static_cast<int>(blockIdx.y * gridDim.x + blockIdx.x);
    const int i0 = static_cast<int>(blockIdx.x) * kBlock, jb = static_cast<int>(blockIdx.y) * len;
    const int je = min(n, jb + len);
    if (je <= i0 + 1) { // no j of this run is behind an i of this tile
        if (threadIdx.x == 0) partials[part] = 0.0;
        return;
    }
    for (int i = threadIdx.x; i < ntypes * ntypes; i += kBlock) s_pairs[i] = pairs_g[i];
    lds_copy(s_coul, coul_g, static_cast<int>(threadIdx.x), kBlock);
    const int i = i0 + static_cast<int>(threadIdx.x);
    const double4 pi = pos[min(i, n - 1)];
    const uint32_t mi = meta[min(i, n - 1)];
    const int ti = static_cast<int>(mi & 0xffu), gi = static_cast<int>(mi >> 8);
    __syncthreads();
    const double inv[3] = {1.0 / box.L[0], 1.0 / box.L[1], 1.0 / box.L[2]};
    double acc = 0.0;
#pragma unroll 2
    for (int j = max(jb, i0 + 1); j < je; ++j) {
        const double4 pj = pos[j];
        if (kCut && near_dist2(box, inv, pi.x, pi.y, pi.z, pj.x, pj.y, pj.z) >= range2) continue;
        if (j <= i || i >= n) continue;
        const double r2 = dist2(box, pi.x, pi.y, pi.z, pj.x, pj.y, pj.z);
        const uint32_t mj = meta[j];
        if (kGroups) {
            const int gj = static_cast<int>(mj >> 8);
            if (gi == gj) {
                if (groups.flags[gi] & 2) continue; // rigid: no internal pairs
                if (pair_excluded(groups.excl_off, groups.excl, i, j)) continue;
            } else if (groups.g2g2 && (groups.flags[gi] & 1) && (groups.flags[gj] & 1)) {
                const double* a = groups.cm + 3 * gi;
                const double* b = groups.cm + 3 * gj;
                if (!(dist2(box, a[0], a[1], a[2], b[0], b[1], b[2]) <
                      g2g_cutoff2(groups.g2g2, groups.nmol, groups.flags[gi], groups.flags[gj])))
                    continue;
            }
        }
        const DevPair& p = s_pairs[ti * ntypes + static_cast<int>(mj & 0xffu)];
        acc += pair_energy(p, s_coul, pi.w, pj.w, r2);
    }
    const double s = block_sum<kBlock>(acc, s_red);
    if (threadIdx.x == 0) partials[part] = s;
}

// Sum of `count` partials in a fixed order (one block).
__global__ __launch_bounds__(kBlock) void sum_partials_kernel(const double* __restrict__ partials, int count,
                                                               double* __restrict__ out) {
    __shared__ double s_red[kBlock / 64];
    double acc = 0.0;
#pragma unroll 4
    for (int b = threadIdx.x; b < count; b += kBlock) acc += partials[b];
    const double s = block_sum<kBlock>(acc, s_red);
    if (threadIdx.x == 0) *out = s;
}

// Plain streaming copy of a known byte count; its HBM counter readings calibrate
// the FETCH_SIZE / WRITE_SIZE scale of the profiles.
// Sum of all intra-molecular bond energies (Bonded::energy on Change::everything,
// energy.cpp:1047-1066); one partial per block.
__global__ __launch_bounds__(kBlock) void bond_total_kernel(const double4* __restrict__ pos,
                                                             const DevBondPair* __restrict__ bonds, int nb, Box box,
                                                             double* __restrict__ partials) {
    __shared__ double s_red[kBlock / 64];
    double acc = 0.0;
    for (int e = blockIdx.x * kBlock + threadIdx.x; e < nb; e += gridDim.x * kBlock) {
        const DevBondPair B = bonds[e];
        const double4 a = pos[B.i], b = pos[B.j];
        const double x = B.req - sqrt(dist2(box, a.x, a.y, a.z, b.x, b.y, b.z));
        acc += B.half_k * x * x;
    }
    const double s = block_sum<kBlock>(acc, s_red);
    if (threadIdx.x == 0) partials[blockIdx.x] = s;
}

__global__ __launch_bounds__(kBlock) void copy_probe_kernel(const double4* __restrict__ src, double4* __restrict__ dst,
                                                            long long n) {
    for (long long i = blockIdx.x * static_cast<long long>(kBlock) + threadIdx.x; i < n;
         i += static_cast<long long>(gridDim.x) * kBlock)
        dst[i] = src[i];
}

} // namespace

double copy_probe(long long bytes, int repeats) {
    const long long n = bytes / static_cast<long long>(sizeof(double4));
    if (n <= 0 || repeats <= 0) throw std::runtime_error("copy_probe: bad size");
    double4 *src = nullptr, *dst = nullptr;
    check_hip(hipMalloc(&src, sizeof(double4) * n), "hipMalloc probe");
    check_hip(hipMalloc(&dst, sizeof(double4) * n), "hipMalloc probe");
    check_hip(hipMemset(src, 0, sizeof(double4) * n), "memset probe");
    hipEvent_t a, b;
    check_hip(hipEventCreate(&a), "event");
    check_hip(hipEventCreate(&b), "event");
    hipLaunchKernelGGL(copy_probe_kernel, dim3(2048), dim3(kBlock), 0, nullptr, src, dst, n);
    check_hip(hipEventRecord(a, nullptr), "event");
    for (int r = 0; r < repeats; ++r) hipLaunchKernelGGL(copy_probe_kernel, dim3(2048), dim3(kBlock), 0, nullptr, src, dst, n);
    check_hip(hipEventRecord(b, nullptr), "event");
    check_hip(hipEventSynchronize(b), "event sync");
    float ms = 0;
    check_hip(hipEventElapsedTime(&ms, a, b), "elapsed");
    (void)hipEventDestroy(a);
    (void)hipEventDestroy(b);
    (void)hipFree(src);
    (void)hipFree(dst);
    return ms / repeats;
}

// ==============================================================================
Engine::Engine(const std::string& config_json) : model_(Model::from_json(config_json)) {
    int ndev = 0;
    check_hip(hipGetDeviceCount(&ndev), "hipGetDeviceCount");
    if (ndev < 1) throw std::runtime_error("no HIP device visible: the GPU engine needs an MI355X");
    check_hip(hipGetDevice(&device_), "hipGetDevice");
    hipDeviceProp_t prop;
    check_hip(hipGetDeviceProperties(&prop, device_), "hipGetDeviceProperties");
    num_cu_ = prop.multiProcessorCount;
    check_hip(hipStreamCreateWithFlags(&stream_, hipStreamNonBlocking), "hipStreamCreate");
    if (model_.ntypes > kMaxTypes) throw std::runtime_error("too many atom types for the GPU engine");
    max_blocks_ = 4096;
    check_hip(hipMalloc(&d_partials_, sizeof(double2) * max_blocks_), "hipMalloc partials");
    check_hip(hipMalloc(&d_ticket_, sizeof(unsigned)), "hipMalloc ticket");
    check_hip(hipMemset(d_ticket_, 0, sizeof(unsigned)), "hipMemset ticket");
    check_hip(hipHostMalloc(&h_result_, sizeof(DeltaResult), hipHostMallocCoherent), "hipHostMalloc result");
    std::memset(h_result_, 0, sizeof(DeltaResult));
    check_hip(hipMalloc(&d_moved_, sizeof(MovedParticle) * kMaxMoved), "hipMalloc moved");
    upload_potentials();
}

Engine::~Engine() {
    if (stream_) (void)hipStreamSynchronize(stream_);
    for (auto e : ev_pool_) (void)hipEventDestroy(e);
    (void)hipFree(d_pos_);
    (void)hipFree(d_meta_);
    (void)hipFree(d_pairs_);
    (void)hipFree(d_coul_);
    (void)hipFree(d_kn_);
    (void)hipFree(d_qcol_);
    (void)hipFree(d_ak_);
    (void)hipFree(d_q_acc_);
    (void)hipFree(d_q_trial_);
    (void)hipFree(d_partials_);
    (void)hipFree(d_ticket_);
    (void)hipFree(d_moved_);
    (void)hipFree(cells_.count);
    (void)hipFree(cells_.members);
    (void)hipFree(cells_.cell_of);
    (void)hipFree(cells_.overflow);
    (void)hipFree(d_gflags_);
    (void)hipFree(d_gcm_);
    (void)hipFree(d_g2g_);
    (void)hipFree(d_bond_off_);
    (void)hipFree(d_bond_);
    (void)hipFree(d_bond_all_);
    (void)hipFree(d_excl_off_);
    (void)hipFree(d_excl_);
    if (h_result_) (void)hipHostFree(h_result_);
    if (stream_) (void)hipStreamDestroy(stream_);
}

void Engine::upload_potentials() {
    const int nt = model_.ntypes;
    h_pairs_.assign(static_cast<size_t>(nt * nt), DevPair{});
    for (int i = 0; i < nt * nt; ++i) {
        const PairParam& p = model_.pairs[static_cast<size_t>(i)];
        h_pairs_[static_cast<size_t>(i)] = DevPair{p.lj_s2, p.lj_e4, p.wca_s2, p.wca_e4, p.hs_s2, p.coulomb, 0, 0, 0.0};
    }
    std::memset(&h_coul_, 0, sizeof(h_coul_));
    if (model_.splined) {
        // one table per unordered type pair
        std::vector<int> slot(static_cast<size_t>(nt * nt), -1);
        int ns = 0;
        for (int a = 0; a < nt; ++a)
            for (int b = 0; b <= a; ++b) {
                if (ns == kSplMaxTables)
                    throw std::runtime_error("nonbonded_splined: at most " + std::to_string(kSplMaxTables) +
                                             " type-pair tables on the device (four atom types)");
                const SplinedPairCfg& s = model_.spl[static_cast<size_t>(a * nt + b)];
                const int n = static_cast<int>(s.table.knots.size());
                if (n < 2 || n > kSplMaxKnots)
                    throw std::runtime_error("nonbonded_splined: a table has " + std::to_string(n) +
                                             " knots; the device holds at most " + std::to_string(kSplMaxKnots));
                DevSplineTable& T = h_coul_.spl[ns];
                T.rmin2 = s.rmin2;
                T.rmax2 = s.rmax2;
                T.n = n;
                T.hs = s.hardsphere ? 1 : 0;
                std::fill(T.knots, T.knots + kSplMaxKnots + 4, s.table.knots.back());
                std::copy(s.table.knots.begin(), s.table.knots.end(), T.knots);
                std::copy(s.table.coeff.begin(), s.table.coeff.end(), T.coeff);
                T.x0 = s.table.knots.front();
                const double span = s.table.knots.back() - T.x0;
                T.inv_w = kSplBuckets / span;
                for (int k = 0; k <= kSplBuckets; ++k) {
                    // a little below the bucket's edge, so that the knot before the first one
                    // found lies below every r2 that rounds into the bucket
                    const double x = T.x0 + k / T.inv_w - 1e-9 * span;
                    T.bucket[k] = static_cast<unsigned char>(
                        std::lower_bound(s.table.knots.begin(), s.table.knots.end(), x) - s.table.knots.begin());
                }
                // lower_bound(x) for x in bucket k lies in [bucket[k], bucket[k+1]] (one more
                // for rounding of the bucket edges); the search starts one knot early
                int steps = 1;
                for (int k = 0; k < kSplBuckets; ++k) {
                    const int start = std::max(0, static_cast<int>(T.bucket[k]) - 1);
                    steps = std::max(steps, std::min(n, static_cast<int>(T.bucket[k + 1]) + 1) - start + 1);
                }
                T.steps = steps;
                slot[static_cast<size_t>(a * nt + b)] = slot[static_cast<size_t>(b * nt + a)] = ns++;
            }
        h_coul_.nspl = ns;
        for (int i = 0; i < nt * nt; ++i) h_pairs_[static_cast<size_t>(i)].spl = slot[static_cast<size_t>(i)];
    }
    const CoulombModel& c = model_.coulomb;
    h_coul_.scheme = c.scheme;
    h_coul_.splined = c.splined ? 1 : 0;
    h_coul_.lB = c.lB;
    h_coul_.rc = c.rc;
    h_coul_.rc_inv = c.rc_inv;
    h_coul_.alpha = c.alpha;
    if (c.splined && (c.scheme == kCoulEwald || c.scheme == kCoulFanourgakis)) {
        if (static_cast<int>(c.S.knots.size()) > kMaxKnots) throw std::runtime_error("spline has too many knots");
        h_coul_.nknots = static_cast<int>(c.S.knots.size());
        std::fill(h_coul_.knots, h_coul_.knots + kMaxKnots + 4, c.S.knots.back());
        std::copy(c.S.knots.begin(), c.S.knots.end(), h_coul_.knots);
        std::copy(c.S.coeff.begin(), c.S.coeff.end(), h_coul_.coeff);
        for (int b = 0; b <= kSplineBuckets; ++b) {
            const double x = static_cast<double>(b) / kSplineBuckets;
            h_coul_.bucket[b] = static_cast<unsigned short>(
                std::lower_bound(c.S.knots.begin(), c.S.knots.end(), x) - c.S.knots.begin());
        }
        // lower_bound(x) for x in bucket b lies in [bucket[b], bucket[b+1]]; the search
        // starts one knot early and gets one extra step for FP32 rounding of the knots
        int steps = 1;
        for (int b = 0; b < kSplineBuckets; ++b) {
            const int start = std::max(0, static_cast<int>(h_coul_.bucket[b]) - 1);
            steps = std::max(steps, static_cast<int>(h_coul_.bucket[b + 1]) - start + 1);
        }
        h_coul_.spline_steps = steps;
    }
    check_hip(hipMalloc(&d_pairs_, sizeof(DevPair) * h_pairs_.size()), "hipMalloc pairs");
    check_hip(hipMalloc(&d_coul_, sizeof(DevCoulomb)), "hipMalloc coulomb");
    check_hip(hipMemcpy(d_pairs_, h_pairs_.data(), sizeof(DevPair) * h_pairs_.size(), hipMemcpyHostToDevice), "copy pairs");
    check_hip(hipMemcpy(d_coul_, &h_coul_, sizeof(DevCoulomb), hipMemcpyHostToDevice), "copy coulomb");
}

void Engine::set_particles(int n, const double* xyz, const double* charge, const int* atom_id) {
    if (n <= 0) throw std::runtime_error("set_particles: n must be positive");
    n_ = n;
    h_xyz_.assign(xyz, xyz + 3 * static_cast<size_t>(n));
    h_q_.assign(charge, charge + n);
    h_type_.assign(atom_id, atom_id + n);
    for (int t : h_type_)
        if (t < 0 || t >= model_.ntypes) throw std::runtime_error("set_particles: atom id out of range");
    h_gid_.assign(static_cast<size_t>(n), 0);
}

void Engine::set_groups(int ng, const int* begin, const int* size, const int* molid, const double* mass_center) {
    if (n_ == 0) throw std::runtime_error("set_groups: call set_particles first");
    if (ng <= 0 || ng >= (1 << 24)) throw std::runtime_error("set_groups: bad number of groups");
    g_begin_.assign(begin, begin + ng);
    g_size_.assign(size, size + ng);
    g_molid_.assign(molid, molid + ng);
    g_cm_.assign(3 * static_cast<size_t>(ng), 0.0);
    if (mass_center) g_cm_.assign(mass_center, mass_center + 3 * static_cast<size_t>(ng));
    int expect = 0;
    any_molecular_ = false;
    for (int g = 0; g < ng; ++g) {
        if (g_begin_[g] != expect) throw std::runtime_error("set_groups: groups must tile the particles in order");
        if (g_size_[g] < 0 || g_size_[g] > n_ - expect)
            throw std::runtime_error("set_groups: group extends past the last particle");
        if (g_molid_[g] < 0 || g_molid_[g] >= static_cast<int>(model_.molecules.size()))
            throw std::runtime_error("set_groups: molecule id out of range");
        for (int i = 0; i < g_size_[g]; ++i) h_gid_[static_cast<size_t>(g_begin_[g] + i)] = g;
        expect += g_size_[g];
        const auto& mol = model_.molecules[static_cast<size_t>(g_molid_[g])];
        if (!mol.atomic) any_molecular_ = true;
    }
    if (expect != n_) throw std::runtime_error("set_groups: groups must cover all particles");
    if (!mass_center)
        for (int g = 0; g < ng; ++g)
            if (!model_.molecules[static_cast<size_t>(g_molid_[g])].atomic && g_size_[g] > 0)
                group_mass_center_host(g, &g_cm_[static_cast<size_t>(3 * g)]);
}

// Geometry::weightedCenter with masses (geometry.h:505-525): shift by minus the first
// atom, wrap, mass-weighted mean, shift back, wrap.
void Engine::group_mass_center_host(int g, double* cm) const {
    const int b = g_begin_[static_cast<size_t>(g)];
    const double shift[3] = {-h_xyz_[3 * b], -h_xyz_[3 * b + 1], -h_xyz_[3 * b + 2]};
    auto wrap = [&](double& x, int d) {
        const double L = model_.box[d];
        if (std::fabs(x) > 0.5 * L) {
            const double t = x / L;
            x -= L * static_cast<double>(static_cast<int>(t > 0.0 ? t + 0.5 : t - 0.5));
        }
    };
    double c[3] = {0, 0, 0}, wsum = 0;
    for (int k = 0; k < g_size_[static_cast<size_t>(g)]; ++k) {
        const int i = b + k;
        const double w = model_.atoms[static_cast<size_t>(h_type_[static_cast<size_t>(i)])].mw;
        for (int d = 0; d < 3; ++d) {
            double x = h_xyz_[3 * i + d] + shift[d];
            wrap(x, d);
            c[d] += w * x;
        }
        wsum += w;
    }
    for (int d = 0; d < 3; ++d) {
        double x = c[d] / wsum - shift[d];
        wrap(x, d);
        cm[d] = x;
    }
}

void Engine::stage_mass_center(int group, const double* cm) {
    if (group < 0 || group >= static_cast<int>(g_begin_.size())) throw std::runtime_error("stage_mass_center: group out of range");
    staged_cm_group_ = group;
    for (int d = 0; d < 3; ++d) staged_cm_[d] = cm[d];
}

// Group flags, mass centres and the bond tables on the device.
void Engine::build_group_tables() {
    const int ng = static_cast<int>(g_begin_.size());
    std::vector<int> flags(static_cast<size_t>(ng));
    for (int g = 0; g < ng; ++g) {
        const MoleculeCfg& mol = model_.molecules[static_cast<size_t>(g_molid_[static_cast<size_t>(g)])];
        flags[static_cast<size_t>(g)] = (mol.atomic ? 0 : 1) | (mol.rigid ? 2 : 0) | (g_molid_[static_cast<size_t>(g)] << 8);
    }
    (void)hipFree(d_g2g_);
    d_g2g_ = nullptr;
    if (model_.has_g2g()) {
        check_hip(hipMalloc(&d_g2g_, sizeof(double) * model_.g2g2.size()), "hipMalloc g2g cutoffs");
        check_hip(hipMemcpy(d_g2g_, model_.g2g2.data(), sizeof(double) * model_.g2g2.size(), hipMemcpyHostToDevice),
                  "copy g2g cutoffs");
    }
    (void)hipFree(d_gflags_);
    (void)hipFree(d_gcm_);
    check_hip(hipMalloc(&d_gflags_, sizeof(int) * std::max(1, ng)), "hipMalloc group flags");
    check_hip(hipMalloc(&d_gcm_, sizeof(double) * 3 * std::max(1, ng)), "hipMalloc group centres");
    check_hip(hipMemcpy(d_gflags_, flags.data(), sizeof(int) * ng, hipMemcpyHostToDevice), "copy group flags");
    check_hip(hipMemcpy(d_gcm_, g_cm_.data(), sizeof(double) * 3 * ng, hipMemcpyHostToDevice), "copy group centres");
    // bonds (Bonded::updateGroupBonds, energy.cpp:974-984: molecule bonds shifted to absolute indices)
    std::vector<std::vector<DevBond>> per(static_cast<size_t>(n_));
    std::vector<DevBondPair> flat;
    if (model_.bonded_term >= 0) {
        for (int g = 0; g < ng; ++g) {
            const MoleculeCfg& mol = model_.molecules[static_cast<size_t>(g_molid_[static_cast<size_t>(g)])];
            const int b0 = g_begin_[static_cast<size_t>(g)], sz = g_size_[static_cast<size_t>(g)];
            for (const BondCfg& bd : mol.bonds) {
                if (bd.i >= sz || bd.j >= sz) throw std::runtime_error("bonded index out of range for group size");
                per[static_cast<size_t>(b0 + bd.i)].push_back(DevBond{b0 + bd.j, 0, bd.half_k, bd.req});
                per[static_cast<size_t>(b0 + bd.j)].push_back(DevBond{b0 + bd.i, 0, bd.half_k, bd.req});
                flat.push_back(DevBondPair{b0 + bd.i, b0 + bd.j, bd.half_k, bd.req});
            }
        }
    }
    // exclusions (MoleculeData::isPairExcluded): per-particle sorted absolute partners
    std::vector<std::vector<int>> ex(static_cast<size_t>(n_));
    bool any_excl = false;
    for (int g = 0; g < ng; ++g) {
        const MoleculeCfg& mol = model_.molecules[static_cast<size_t>(g_molid_[static_cast<size_t>(g)])];
        if (mol.atomic) continue;
        const int b0 = g_begin_[static_cast<size_t>(g)], sz = g_size_[static_cast<size_t>(g)];
        for (auto [i, j] : mol.excluded) {
            if (i >= sz || j >= sz) continue; // pairs beyond the group's atoms do not apply
            ex[static_cast<size_t>(b0 + i)].push_back(b0 + j);
            ex[static_cast<size_t>(b0 + j)].push_back(b0 + i);
            any_excl = true;
        }
    }
    (void)hipFree(d_excl_off_);
    (void)hipFree(d_excl_);
    d_excl_off_ = d_excl_ = nullptr;
    if (any_excl) {
        std::vector<int> eoff(static_cast<size_t>(n_) + 1, 0), elist;
        for (int i = 0; i < n_; ++i) {
            auto& v = ex[static_cast<size_t>(i)];
            std::sort(v.begin(), v.end());
            elist.insert(elist.end(), v.begin(), v.end());
            eoff[static_cast<size_t>(i) + 1] = static_cast<int>(elist.size());
        }
        check_hip(hipMalloc(&d_excl_off_, sizeof(int) * eoff.size()), "hipMalloc exclusion offsets");
        check_hip(hipMalloc(&d_excl_, sizeof(int) * elist.size()), "hipMalloc exclusions");
        check_hip(hipMemcpy(d_excl_off_, eoff.data(), sizeof(int) * eoff.size(), hipMemcpyHostToDevice), "copy exclusions");
        check_hip(hipMemcpy(d_excl_, elist.data(), sizeof(int) * elist.size(), hipMemcpyHostToDevice), "copy exclusions");
    }
    std::vector<int> off(static_cast<size_t>(n_) + 1, 0);
    std::vector<DevBond> list;
    for (int i = 0; i < n_; ++i) {
        off[static_cast<size_t>(i) + 1] = off[static_cast<size_t>(i)] + static_cast<int>(per[static_cast<size_t>(i)].size());
        list.insert(list.end(), per[static_cast<size_t>(i)].begin(), per[static_cast<size_t>(i)].end());
    }
    nbonds_ = static_cast<int>(flat.size());
    (void)hipFree(d_bond_off_);
    (void)hipFree(d_bond_);
    (void)hipFree(d_bond_all_);
    check_hip(hipMalloc(&d_bond_off_, sizeof(int) * off.size()), "hipMalloc bond offsets");
    check_hip(hipMalloc(&d_bond_, sizeof(DevBond) * std::max<size_t>(1, list.size())), "hipMalloc bonds");
    check_hip(hipMalloc(&d_bond_all_, sizeof(DevBondPair) * std::max<size_t>(1, flat.size())), "hipMalloc bond list");
    check_hip(hipMemcpy(d_bond_off_, off.data(), sizeof(int) * off.size(), hipMemcpyHostToDevice), "copy bond offsets");
    if (!list.empty())
        check_hip(hipMemcpy(d_bond_, list.data(), sizeof(DevBond) * list.size(), hipMemcpyHostToDevice), "copy bonds");
    if (!flat.empty())
        check_hip(hipMemcpy(d_bond_all_, flat.data(), sizeof(DevBondPair) * flat.size(), hipMemcpyHostToDevice),
                  "copy bond list");
}

void Engine::build_kvectors() {
    // PolicyIonIon::updateBox (energy.cpp:133-186): n_x >= 0, |n|^2 <= n_c^2, n != 0.
    const EwaldModel& e = model_.ewald;
    const int nc = static_cast<int>(std::ceil(e.n_cutoff));
    if (nc > 127) throw std::runtime_error("ncutoff too large");
    const double maxL = std::max(model_.box[0], std::max(model_.box[1], model_.box[2]));
    const double k2zero = 0.1 * std::pow(2 * kPi / maxL, 2);
    const double nc2 = e.n_cutoff * e.n_cutoff;
    std::vector<int> kn;
    std::vector<double> ak;
    for (int nx = 0; nx <= nc; nx++)
        for (int ny = -nc; ny <= nc; ny++)
            for (int nz = -nc; nz <= nc; nz++) {
                const double kx = 2 * kPi * (double(nx) / model_.box[0]);
                const double ky = 2 * kPi * (double(ny) / model_.box[1]);
                const double kz = 2 * kPi * (double(nz) / model_.box[2]);
                const double k2 = kx * kx + ky * ky + kz * kz;
                if (k2 < k2zero) continue;
                if (e.spherical_sum && (double(nx * nx) + double(ny * ny) + double(nz * nz)) / nc2 > 1) continue;
                kn.push_back((nx & 0xff) | ((ny & 0xff) << 8) | ((nz & 0xff) << 16));
                ak.push_back((nx > 0 ? 2.0 : 1.0) * std::exp(-k2 / (4 * e.alpha * e.alpha)) / k2);
            }
    nk_ = static_cast<int>(kn.size());
    // the (nx, ny) columns of the list: each a run of k-vectors with nz ascending
    std::vector<QColumn> cols;
    for (int k = 0; k < nk_; ++k) {
        const int nx = static_cast<signed char>(kn[static_cast<size_t>(k)] & 0xff);
        const int ny = static_cast<signed char>((kn[static_cast<size_t>(k)] >> 8) & 0xff);
        const int nz = static_cast<signed char>((kn[static_cast<size_t>(k)] >> 16) & 0xff);
        if (cols.empty() || cols.back().nx != nx || cols.back().ny != ny)
            cols.push_back(QColumn{static_cast<short>(nx), static_cast<short>(ny), k, nz, nz});
        cols.back().nzmax = nz;
    }
    std::stable_sort(cols.begin(), cols.end(), [](const QColumn& a, const QColumn& b) { return a.nzmax > b.nzmax; });
    ncol_ = static_cast<int>(cols.size());
    check_hip(hipMalloc(&d_qcol_, sizeof(QColumn) * std::max(1, ncol_)), "hipMalloc k columns");
    if (ncol_ > 0)
        check_hip(hipMemcpy(d_qcol_, cols.data(), sizeof(QColumn) * cols.size(), hipMemcpyHostToDevice), "copy k columns");
    check_hip(hipMalloc(&d_kn_, sizeof(int) * std::max(1, nk_)), "hipMalloc kn");
    check_hip(hipMalloc(&d_ak_, sizeof(double) * std::max(1, nk_)), "hipMalloc ak");
    check_hip(hipMalloc(&d_q_acc_, sizeof(double2) * std::max(1, nk_)), "hipMalloc q");
    check_hip(hipMalloc(&d_q_trial_, sizeof(double2) * std::max(1, nk_)), "hipMalloc q trial");
    if (nk_ > 0) {
        check_hip(hipMemcpy(d_kn_, kn.data(), sizeof(int) * nk_, hipMemcpyHostToDevice), "copy kn");
        check_hip(hipMemcpy(d_ak_, ak.data(), sizeof(double) * nk_, hipMemcpyHostToDevice), "copy ak");
    }
}

static Box make_box(const Model& m) {
    Box b;
    for (int d = 0; d < 3; ++d) {
        b.L[d] = m.box[d];
        b.half[d] = 0.5 * m.box[d];
    }
    return b;
}

// Full Q(k) from the positions into `out`; complete when it returns.
void Engine::full_q(double2* out) {
    if (nk_ == 0) return;
    const Box box = make_box(model_);
    const int ncut = static_cast<int>(std::ceil(model_.ewald.n_cutoff));
    // two column tiles per wave once one would take a second block of columns (a block's
    // table sincos then serve twice the columns)
    const int ct = ncol_ > kQCols ? 2 : 1;
    const int col_blocks = (ncol_ + kQCols * ct - 1) / (kQCols * ct);
    const int z_blocks = (2 * (ncut + 1) + 16 * kQTiles - 1) / (16 * kQTiles);
    const size_t row = sizeof(double2) * 3 * static_cast<size_t>(ncut + 1);
    int chunk = kQChunk;
    while (chunk > 4 && chunk * row > 40 * 1024) chunk /= 2;
    // slices of the particles: one block per CU, or as many as there are chunks or as fit
    // 24 MB of partial sums
    int slices = std::max(1, num_cu_ / (col_blocks * z_blocks));
    slices = std::min({slices, (n_ + chunk - 1) / chunk,
                       std::max(1, static_cast<int>((24u << 20) / (sizeof(double2) * static_cast<size_t>(nk_))))});
    int slice = (n_ + slices - 1) / slices;
    slice = (slice + chunk - 1) / chunk * chunk;
    slices = (n_ + slice - 1) / slice;
    double2* part = out;
    if (slices > 1) check_hip(hipMalloc(&part, sizeof(double2) * static_cast<size_t>(slices) * static_cast<size_t>(nk_)), "hipMalloc partial Q");
    // the pad takes the reads past the last table row (see full_q_kernel)
    const size_t lds = chunk * row + sizeof(double) * 16 * kQTiles * static_cast<size_t>(z_blocks);
    const dim3 grid(static_cast<unsigned>(col_blocks), static_cast<unsigned>(slices), static_cast<unsigned>(z_blocks));
    hipLaunchKernelGGL(ct == 2 ? full_q_kernel<2> : full_q_kernel<1>, grid, dim3(kQThreads), lds, stream_, d_pos_, n_,
                       d_qcol_, ncol_, ncut, chunk, slice, nk_, box, part);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess && slices > 1) {
        hipLaunchKernelGGL(sum_q_kernel, dim3((nk_ + kBlock - 1) / kBlock), dim3(kBlock), 0, stream_, part, slices, nk_, out);
        e = hipGetLastError();
    }
    const hipError_t done = hipStreamSynchronize(stream_);
    if (part != out) (void)hipFree(part);
    check_hip(e, "full_q_kernel");
    check_hip(done, "full Q");
}

void Engine::set_cell_capacity(int cap) {
    if (cap < 0) throw std::runtime_error("cell capacity must be >= 0");
    cell_capacity_ = cap;
}

void Engine::set_cell_divisions(int d) {
    if (d < 1 || d > 2) throw std::runtime_error("cell divisions: 1 or 2");
    if (d_pos_ != nullptr) throw std::runtime_error("cell divisions must be set before init");
    cell_divisions_ = d;
}

void Engine::regrid(int d) {
    if (d < 1 || d > 2) throw std::runtime_error("cell divisions: 1 or 2");
    cell_divisions_ = d; // the next reset_positions builds the grid
}

// Distance beyond which no pair of atoms interacts: the pair potentials' range, or with
// cutoff_g2g in a system made only of rigid molecules the largest group cutoff plus the
// two largest distances of an atom from its group's mass centre (GroupCutoff::cut drops
// every pair of groups whose centres are farther apart).
double Engine::interaction_range() const {
    double range = model_.pair_range;
    if (!model_.has_g2g() || g_begin_.empty()) return range;
    double rmax = 0.0;
    for (size_t g = 0; g < g_begin_.size(); ++g) {
        const MoleculeCfg& mol = model_.molecules[static_cast<size_t>(g_molid_[g])];
        if (mol.atomic || !mol.rigid) return range;
        for (int k = 0; k < g_size_[g]; ++k) {
            const int i = g_begin_[g] + k;
            double r2 = 0.0;
            for (int d = 0; d < 3; ++d) {
                double x = h_xyz_[3 * static_cast<size_t>(i) + d] - g_cm_[3 * g + d];
                x -= model_.box[d] * std::round(x / model_.box[d]);
                r2 += x * x;
            }
            rmax = std::max(rmax, std::sqrt(r2));
        }
    }
    double c2 = 0.0;
    for (double v : model_.g2g2) c2 = std::max(c2, v);
    // 1e-6 A above the bound: rigid rotations keep the atom distances up to rounding
    return std::min(range, std::sqrt(c2) + 2.0 * rmax + 1e-6);
}

bool Engine::rigid_reach(double* reach, double* sure) const {
    if (g_begin_.empty()) return false;
    double rmax = 0.0, cmin = kInf, cmax = 0.0;
    for (size_t g = 0; g < g_begin_.size(); ++g) {
        const MoleculeCfg& mol = model_.molecules[static_cast<size_t>(g_molid_[g])];
        if (mol.atomic || !mol.rigid) return false;
        for (int k = 0; k < g_size_[g]; ++k) {
            const int i = g_begin_[g] + k;
            double r2 = 0.0;
            for (int d = 0; d < 3; ++d) {
                double x = h_xyz_[3 * static_cast<size_t>(i) + d] - g_cm_[3 * g + d];
                x -= model_.box[d] * std::round(x / model_.box[d]);
                r2 += x * x;
            }
            rmax = std::max(rmax, std::sqrt(r2));
        }
    }
    for (double v : model_.g2g2) {
        cmin = std::min(cmin, std::sqrt(v));
        cmax = std::max(cmax, std::sqrt(v));
    }
    // 1e-5 A for rounding of rotated atoms; 5e-6 of the cutoff for 32-bit centre distances
    *reach = model_.pair_range + 2.0 * rmax + 1e-5;
    *reach *= 1.0 + 1e-6;
    *sure = kInf;
    if (model_.has_g2g()) {
        *reach = std::min(*reach, cmax * (1.0 + 5e-6));
        *sure = cmin * (1.0 - 5e-6);
    }
    return std::isfinite(*reach);
}

void Engine::build_cell_list() {
    cells_.enabled = false;
    const double range = interaction_range();
    cell_range_ = range;
    if (!(range > 0) || !std::isfinite(range)) return;
    int nc[3];
    // cells of at least range / r with a (2r+1)^3 stencil; the finer grid needs 2r+1
    // cells per side, else the 27-cell grid is used
    int r = cell_divisions_;
    for (int d = 0; d < 3; ++d)
        if (std::floor(model_.box[d] * r / range) < 2 * r + 1) r = 1;
    for (int d = 0; d < 3; ++d) {
        if (range > 0.5 * model_.box[d]) return;
        nc[d] = static_cast<int>(std::floor(model_.box[d] * r / range));
        if (nc[d] < 2 * r + 1) return;
    }
    cells_.radius = r;
    const long ncell = static_cast<long>(nc[0]) * nc[1] * nc[2];
    if (ncell > (1L << 24)) return;
    std::vector<int> count(static_cast<size_t>(ncell), 0), cell_of(static_cast<size_t>(n_));
    auto coord = [&](double x, int d) {
        int c = static_cast<int>(std::floor((x + 0.5 * model_.box[d]) * (nc[d] / model_.box[d])));
        c %= nc[d];
        if (c < 0) c += nc[d];
        return c;
    };
    for (int i = 0; i < n_; ++i) {
        const int c = (coord(h_xyz_[3 * i + 2], 2) * nc[1] + coord(h_xyz_[3 * i + 1], 1)) * nc[0] + coord(h_xyz_[3 * i], 0);
        cell_of[static_cast<size_t>(i)] = c;
        count[static_cast<size_t>(c)]++;
    }
    const int maxcount = *std::max_element(count.begin(), count.end());
    const double mean = static_cast<double>(n_) / static_cast<double>(ncell);
    int cap = std::max(maxcount * 2, static_cast<int>(4 * mean + 32));
    cap = (cap + 7) & ~7;
    if (cell_capacity_ > 0) {
        if (cell_capacity_ < maxcount) throw std::runtime_error("cell capacity below the fullest initial cell");
        cap = cell_capacity_;
    }
    std::vector<int> members(static_cast<size_t>(ncell * cap), -1);
    std::fill(count.begin(), count.end(), 0);
    for (int i = 0; i < n_; ++i) {
        const int c = cell_of[static_cast<size_t>(i)];
        members[static_cast<size_t>(c) * cap + count[static_cast<size_t>(c)]++] = i;
    }
    cells_.enabled = true;
    cells_.cap = cap;
    for (int d = 0; d < 3; ++d) {
        cells_.nc[d] = nc[d];
        cells_.inv_cell[d] = nc[d] / model_.box[d];
    }
    check_hip(hipMalloc(&cells_.count, sizeof(int) * ncell), "hipMalloc cells");
    check_hip(hipMalloc(&cells_.members, sizeof(int) * ncell * cap), "hipMalloc cells");
    check_hip(hipMalloc(&cells_.cell_of, sizeof(int) * n_), "hipMalloc cells");
    check_hip(hipMalloc(&cells_.overflow, sizeof(int)), "hipMalloc cells");
    check_hip(hipMemcpy(cells_.count, count.data(), sizeof(int) * ncell, hipMemcpyHostToDevice), "copy cells");
    check_hip(hipMemcpy(cells_.members, members.data(), sizeof(int) * ncell * cap, hipMemcpyHostToDevice), "copy cells");
    check_hip(hipMemcpy(cells_.cell_of, cell_of.data(), sizeof(int) * n_, hipMemcpyHostToDevice), "copy cells");
    check_hip(hipMemset(cells_.overflow, 0, sizeof(int)), "memset cells");
}

void Engine::init() {
    if (n_ == 0 || g_begin_.empty()) throw std::runtime_error("init: particles and groups must be set");
    // device particle arrays
    std::vector<double4> p(static_cast<size_t>(n_));
    std::vector<uint32_t> meta(static_cast<size_t>(n_));
    for (int i = 0; i < n_; ++i) {
        p[static_cast<size_t>(i)] = make_double4(h_xyz_[3 * i], h_xyz_[3 * i + 1], h_xyz_[3 * i + 2], h_q_[static_cast<size_t>(i)]);
        meta[static_cast<size_t>(i)] = static_cast<uint32_t>(h_type_[static_cast<size_t>(i)]) |
                                       (static_cast<uint32_t>(h_gid_[static_cast<size_t>(i)]) << 8);
    }
    (void)hipFree(d_pos_);
    (void)hipFree(d_meta_);
    check_hip(hipMalloc(&d_pos_, sizeof(double4) * n_), "hipMalloc pos");
    check_hip(hipMalloc(&d_meta_, sizeof(uint32_t) * n_), "hipMalloc meta");
    check_hip(hipMemcpy(d_pos_, p.data(), sizeof(double4) * n_, hipMemcpyHostToDevice), "copy pos");
    check_hip(hipMemcpy(d_meta_, meta.data(), sizeof(uint32_t) * n_, hipMemcpyHostToDevice), "copy meta");
    if (model_.ewald.present) {
        build_kvectors();
        full_q(d_q_acc_);
    }
    for (int d = 0; d < 3; ++d) {
        dipole_[d] = 0;
        for (int i = 0; i < n_; ++i) dipole_[d] += h_xyz_[3 * i + d] * h_q_[static_cast<size_t>(i)];
    }
    build_cell_list();
    build_group_tables();
}

void Engine::stage_trial(int m, const int* idx, const double* xyz) {
    if (m < 0 || m > kMaxMoved) throw std::runtime_error("stage_trial: too many moved particles");
    staged_.resize(static_cast<size_t>(m));
    for (int a = 0; a < m; ++a) {
        const int i = idx[a];
        if (i < 0 || i >= n_) throw std::runtime_error("stage_trial: particle index out of range");
        MovedParticle& M = staged_[static_cast<size_t>(a)];
        M.idx = i;
        M.type = h_type_[static_cast<size_t>(i)];
        M.gid = h_gid_[static_cast<size_t>(i)];
        M.pad = 0;
        M.newp = make_double4(xyz[3 * a], xyz[3 * a + 1], xyz[3 * a + 2], h_q_[static_cast<size_t>(i)]);
        M.oldp = make_double4(h_xyz_[3 * i], h_xyz_[3 * i + 1], h_xyz_[3 * i + 2], h_q_[static_cast<size_t>(i)]);
    }
}

double Engine::self_energy_of(int idx) const {
    const double q = h_q_[static_cast<size_t>(idx)];
    return model_.coulomb.self_prefactor * q * q;
}

double Engine::surface_energy(const double* dip) const {
    const EwaldModel& e = model_.ewald;
    if (e.const_inf < 0.5) return 0.0;
    const double V = model_.box[0] * model_.box[1] * model_.box[2];
    const double m2 = dip[0] * dip[0] + dip[1] * dip[1] + dip[2] * dip[2];
    return e.const_inf * 2.0 * kPi / ((2.0 * e.epss + 1.0) * V) * m2 * e.lB;
}

void Engine::set_timing(bool on) {
    timing_ = on;
    ev_pairs_.clear();
}

void Engine::timing(double* total_ms, long* launches) {
    check_hip(hipStreamSynchronize(stream_), "timing sync");
    double t = 0;
    for (auto& pr : ev_pairs_) {
        float ms = 0;
        check_hip(hipEventElapsedTime(&ms, ev_pool_[static_cast<size_t>(pr.first)], ev_pool_[static_cast<size_t>(pr.second)]), "event elapsed");
        t += ms;
    }
    *total_ms = t;
    *launches = static_cast<long>(ev_pairs_.size());
}

void Engine::launch_delta(const MoveArgs& args, int ewald_blocks, bool bond_block) {
    const Box box = make_box(model_);
    GroupTable gt{d_gflags_, d_gcm_, d_g2g_, static_cast<int>(model_.molecules.size()), d_excl_off_, d_excl_};
    CellArgs ca{cells_.count, cells_.members, cells_.nc[0], cells_.nc[1], cells_.nc[2], cells_.cap,
                cells_.inv_cell[0], cells_.inv_cell[1], cells_.inv_cell[2]};
    const int ncut = model_.ewald.present ? static_cast<int>(std::ceil(model_.ewald.n_cutoff)) : 0;
    PairSplit split{1, 1, args.m, kBlock, h_coul_.nspl, std::max(1, std::min(args.m, kPhaseTableMoved))};
    const size_t table = sizeof(double2) * 6 * static_cast<size_t>(2 * ncut + 1); // one moved particle's
    while (split.chunk > 1 && split.chunk * table > 16 * 1024) --split.chunk;
    if (cells_.enabled) {
        // as many lanes per cell as it holds particles on average (a power of two)
        const double mean = static_cast<double>(n_) / (static_cast<double>(cells_.nc[0]) * cells_.nc[1] * cells_.nc[2]);
        split.lanes = 4;
        while (split.lanes < 64 && split.lanes < mean) split.lanes *= 2;
        split.blocks = std::min((args.m * 54 * split.lanes + kBlock - 1) / kBlock, 256);
    } else {
        // one particle per thread, then runs of at least two moved atoms while CUs are free
        split.j_blocks = std::max(1, std::min((n_ + kBlock - 1) / kBlock, 2 * num_cu_));
        const int runs = std::max(1, std::min((args.m + 1) / 2, 2 * num_cu_ / split.j_blocks));
        split.a_run = std::max(1, (args.m + runs - 1) / runs);
        split.blocks = split.j_blocks * std::max(1, (args.m + split.a_run - 1) / split.a_run);
    }
    const int ewald_end = split.blocks + ewald_blocks;
    const int grid = ewald_end + (bond_block ? 1 : 0);
    if (grid > max_blocks_) throw std::runtime_error("too many blocks");
    const size_t lds = nk_ > 0 ? static_cast<size_t>(split.chunk) * table : 0;
    const double V = model_.box[0] * model_.box[1] * model_.box[2];
    const double pref = model_.ewald.present ? 2 * kPi * model_.ewald.lB / V : 0.0;
    // reference order: 2*pi*energy*lB/V (energy.cpp:530); the prefactor is applied to
    // the sum, a difference in the last bit at most.
    ++seq_;
    int e0 = -1, e1 = -1;
    if (timing_) {
        while (ev_pool_.size() < ev_pairs_.size() * 2 + 2) {
            hipEvent_t e;
            check_hip(hipEventCreate(&e), "hipEventCreate");
            ev_pool_.push_back(e);
        }
        e0 = static_cast<int>(ev_pairs_.size() * 2);
        e1 = e0 + 1;
        check_hip(hipEventRecord(ev_pool_[static_cast<size_t>(e0)], stream_), "event record");
    }
    // mass centres of the moved group (group cutoff between molecular groups)
    double cn[3] = {0, 0, 0}, co[3] = {0, 0, 0};
    if (args.change_group >= 0) {
        for (int d = 0; d < 3; ++d) co[d] = cn[d] = g_cm_[static_cast<size_t>(3 * args.change_group + d)];
        if (staged_cm_group_ == args.change_group)
            for (int d = 0; d < 3; ++d) cn[d] = staged_cm_[d];
    }
    if (cells_.enabled && cells_.radius != 1)
        throw std::runtime_error("the per-move path walks 27-cell stencils (cell divisions 1)");
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(grid), dim3(kBlock), lds, stream_, d_pos_, d_meta_, n_, d_pairs_,
                           model_.ntypes, d_coul_, box, gt, ca, args, split, d_kn_, d_ak_, d_q_acc_, d_q_trial_,
                           nk_, ncut, reinterpret_cast<double*>(d_partials_), d_ticket_, h_result_, seq_, pref, cn[0], cn[1], cn[2], co[0], co[1],
                           co[2], ewald_end, d_bond_off_, d_bond_);
    };
    if (any_molecular_) {
        if (cells_.enabled) go(delta_kernel<true, true>);
        else go(delta_kernel<true, false>);
    } else {
        if (cells_.enabled) go(delta_kernel<false, true>);
        else go(delta_kernel<false, false>);
    }
    check_hip(hipGetLastError(), "delta_kernel launch");
    if (timing_) {
        check_hip(hipEventRecord(ev_pool_[static_cast<size_t>(e1)], stream_), "event record");
        ev_pairs_.emplace_back(e0, e1);
    }
    ++launches_;
}

// Wait for the result of launch seq_: the kernel's last block writes it to host memory with
// the launch's number behind it, so the host need not wait for the end of the kernel and its
// completion signal.  Work enqueued afterwards still follows the kernel on the stream.  A
// result that does not come within 20 ms is left to the stream's synchronisation, which
// reports a launch or device error.
void Engine::wait_result() {
    const auto start = std::chrono::steady_clock::now();
    for (unsigned spins = 1; __atomic_load_n(&h_result_->seq, __ATOMIC_ACQUIRE) != seq_; ++spins) {
        if ((spins & 0xfffu) != 0 || std::chrono::steady_clock::now() - start < std::chrono::milliseconds(20)) continue;
        check_hip(hipStreamSynchronize(stream_), "delta sync");
        return;
    }
}

void Engine::delta(const std::vector<int>& groups, const std::vector<char>& all, const std::vector<char>& internal,
                   const std::vector<std::vector<int>>& rel, double* e_new, double* e_old) {
    if (d_pos_ == nullptr) throw std::runtime_error("delta: engine not initialised");
    if (groups.empty()) throw std::runtime_error("delta: empty change");
    // Moved set of the pair loop (GroupPairing::accumulate, energy.h:1447-1475) and of
    // the Ewald update (energy.cpp:219-247) for this Change.
    std::vector<int> moved;
    const bool single = groups.size() == 1;
    for (size_t g = 0; g < groups.size(); ++g) {
        const int gi = groups[g];
        if (gi < 0 || gi >= static_cast<int>(g_begin_.size())) throw std::runtime_error("delta: group index out of range");
        const bool whole = !single || all[g] || rel[g].empty();
        if (!single && !all[g] && !rel[g].empty() && static_cast<int>(rel[g].size()) != g_size_[static_cast<size_t>(gi)])
            throw std::runtime_error("delta: partial moves of several groups are not supported");
        if (whole) {
            if (!all[g] && rel[g].empty()) throw std::runtime_error("delta: a group change without indices is not supported");
            for (int i = 0; i < g_size_[static_cast<size_t>(gi)]; ++i) moved.push_back(g_begin_[static_cast<size_t>(gi)] + i);
        } else {
            for (int r : rel[g]) {
                if (r < 0 || r >= g_size_[static_cast<size_t>(gi)]) throw std::runtime_error("delta: relative index out of range");
                moved.push_back(g_begin_[static_cast<size_t>(gi)] + r);
            }
        }
    }
    if (!single && model_.has_g2g())
        for (int gi : groups)
            if (!model_.molecules[static_cast<size_t>(g_molid_[static_cast<size_t>(gi)])].atomic)
                throw std::runtime_error("delta: changes of several molecular groups with cutoff_g2g are not supported");
    std::sort(moved.begin(), moved.end());
    if (std::adjacent_find(moved.begin(), moved.end()) != moved.end()) throw std::runtime_error("delta: duplicate moved particle");
    if (static_cast<int>(moved.size()) > kMaxMoved) throw std::runtime_error("delta: too many moved particles");
    // coordinates: staged trial coordinates where given, accepted ones otherwise
    std::vector<MovedParticle> mv(moved.size());
    for (size_t a = 0; a < moved.size(); ++a) {
        const int i = moved[a];
        MovedParticle M;
        M.idx = i;
        M.type = h_type_[static_cast<size_t>(i)];
        M.gid = h_gid_[static_cast<size_t>(i)];
        M.pad = 0;
        M.oldp = make_double4(h_xyz_[3 * i], h_xyz_[3 * i + 1], h_xyz_[3 * i + 2], h_q_[static_cast<size_t>(i)]);
        M.newp = M.oldp;
        for (const auto& s : staged_)
            if (s.idx == i) M.newp = s.newp;
        mv[a] = M;
    }
    MoveArgs args{};
    args.m = static_cast<int>(mv.size());
    args.change_group = single ? groups[0] : -1;
    args.internal = single ? (internal[0] ? 1 : 0) : 0;
    if (args.m <= kMaxInlineMoved) {
        for (int a = 0; a < args.m; ++a) args.inl[a] = mv[static_cast<size_t>(a)];
        args.ext = nullptr;
    } else {
        check_hip(hipMemcpyAsync(d_moved_, mv.data(), sizeof(MovedParticle) * mv.size(), hipMemcpyHostToDevice, stream_),
                  "copy moved");
        args.ext = d_moved_;
    }
    int ewald_blocks = 0;
    if (nk_ > 0) ewald_blocks = std::max(1, std::min((nk_ + 2 * kBlock - 1) / (2 * kBlock), 2 * num_cu_));
    if (single && any_molecular_ && model_.has_g2g() &&
        !model_.molecules[static_cast<size_t>(g_molid_[static_cast<size_t>(groups[0])])].atomic &&
        staged_cm_group_ != groups[0])
        throw std::runtime_error("delta: stage the trial mass centre of a moved molecular group when cutoff_g2g is set");
    launch_delta(args, ewald_blocks, nbonds_ > 0 && model_.bonded_term >= 0);
    wait_result();
    const DeltaResult* r = h_result_;
    if (r->seq != seq_) throw std::runtime_error("delta: result sequence mismatch");
    // dipole of the trial state (surface term, energy.cpp:466-482)
    for (int d = 0; d < 3; ++d) dipole_trial_[d] = dipole_[d];
    for (const auto& M : mv) {
        dipole_trial_[0] += M.newp.w * M.newp.x - M.oldp.w * M.oldp.x;
        dipole_trial_[1] += M.newp.w * M.newp.y - M.oldp.w * M.oldp.y;
        dipole_trial_[2] += M.newp.w * M.newp.z - M.oldp.w * M.oldp.z;
    }
    // Hamiltonian::energy order and early break (energy.cpp:1227-1241)
    double self = 0;
    if (model_.has_self_term) {
        for (size_t g = 0; g < groups.size(); ++g) {
            const int gi = groups[g];
            if (all[g]) {
                for (int i = 0; i < g_size_[static_cast<size_t>(gi)]; ++i) self += self_energy_of(g_begin_[static_cast<size_t>(gi)] + i);
            } else {
                for (int r2 : rel[g]) self += self_energy_of(g_begin_[static_cast<size_t>(gi)] + r2);
            }
        }
    }
    auto fill = [&](double* out, double pair, double rec, double bond, const double* dip) {
        bool stop = false;
        for (size_t t = 0; t < model_.term_names.size(); ++t) {
            const std::string& name = model_.term_names[t];
            double v = 0.0;
            if (name == "selfenergy") v = self;
            else if (name == "nonbonded") v = pair;
            else if (name == "ewald") v = surface_energy(dip) + rec;
            else if (name == "bonded") v = bond;
            out[t] = stop ? 0.0 : v;
            if (!stop && (v >= model_.maximum_allowed_energy || std::isnan(v))) stop = true;
        }
    };
    fill(e_new, r->pair_new, r->rec_new, r->bond_new, dipole_trial_);
    fill(e_old, r->pair_old, r->rec_old, r->bond_old, dipole_);
    pending_moved_ = mv;
    pending_cm_group_ = (single && staged_cm_group_ == groups[0]) ? staged_cm_group_ : -1;
    for (int d = 0; d < 3; ++d) pending_cm_[d] = staged_cm_[d];
    pending_ = true;
}

void Engine::sync(bool accept) {
    if (!pending_) return;
    if (accept) {
        MoveArgs args{};
        args.m = static_cast<int>(pending_moved_.size());
        if (args.m <= kMaxInlineMoved) {
            for (int a = 0; a < args.m; ++a) args.inl[a] = pending_moved_[static_cast<size_t>(a)];
        } else {
            check_hip(hipMemcpyAsync(d_moved_, pending_moved_.data(), sizeof(MovedParticle) * pending_moved_.size(),
                                     hipMemcpyHostToDevice, stream_), "copy moved");
            args.ext = d_moved_;
        }
        CellArgs ca{cells_.count, cells_.members, cells_.nc[0], cells_.nc[1], cells_.nc[2], cells_.cap,
                    cells_.inv_cell[0], cells_.inv_cell[1], cells_.inv_cell[2]};
        hipLaunchKernelGGL(commit_kernel, dim3(1), dim3(64), 0, stream_, d_pos_, args, ca, cells_.cell_of,
                           cells_.overflow, make_box(model_), cells_.enabled ? 1 : 0, d_gcm_, pending_cm_group_, pending_cm_[0],
                           pending_cm_[1], pending_cm_[2]);
        check_hip(hipGetLastError(), "commit_kernel");
        for (const auto& M : pending_moved_) {
            h_xyz_[3 * M.idx] = M.newp.x;
            h_xyz_[3 * M.idx + 1] = M.newp.y;
            h_xyz_[3 * M.idx + 2] = M.newp.z;
        }
        std::swap(d_q_acc_, d_q_trial_);
        for (int d = 0; d < 3; ++d) dipole_[d] = dipole_trial_[d];
        if (pending_cm_group_ >= 0)
            for (int d = 0; d < 3; ++d) g_cm_[static_cast<size_t>(3 * pending_cm_group_ + d)] = pending_cm_[d];
    }
    pending_ = false;
    pending_cm_group_ = -1;
    staged_cm_group_ = -1;
    staged_.clear();
}

double Engine::reciprocal_energy_host(const std::vector<double2>& q) const {
    std::vector<double> ak(static_cast<size_t>(nk_));
    check_hip(hipMemcpy(ak.data(), d_ak_, sizeof(double) * nk_, hipMemcpyDeviceToHost), "copy ak");
    double e = 0;
    for (int k = 0; k < nk_; ++k) e += ak[static_cast<size_t>(k)] * (q[static_cast<size_t>(k)].x * q[static_cast<size_t>(k)].x + q[static_cast<size_t>(k)].y * q[static_cast<size_t>(k)].y);
    const double V = model_.box[0] * model_.box[1] * model_.box[2];
    return 2 * kPi * e * model_.ewald.lB / V;
}

void Engine::total_energy(double* terms) {
    check_hip(hipStreamSynchronize(stream_), "sync");
    int cells_overflow = 0;
    if (cells_.enabled) {
        check_hip(hipMemcpy(&cells_overflow, cells_.overflow, sizeof(int), hipMemcpyDeviceToHost), "copy overflow");
        if (cells_overflow) throw std::runtime_error("cell list overflow: a cell exceeded its capacity");
    }
    double self = 0;
    if (model_.has_self_term) {
        for (size_t g = 0; g < g_begin_.size(); ++g) {
            double gs = 0;
            for (int i = 0; i < g_size_[g]; ++i) gs += self_energy_of(g_begin_[g] + i);
            self += gs;
        }
    }
    // nonbonded: all pairs (GroupPairing::all, energy.h:1290-1299).  The runs of j are cut
    // shorter, down to 16, until there are about eight blocks per CU
    const int tiles = (n_ + kBlock - 1) / kBlock;
    int len = kBlock;
    while (len > 16 && static_cast<long long>(tiles) * ((n_ + len - 1) / len) < 16LL * num_cu_) len /= 2;
    while (static_cast<long long>(tiles) * ((n_ + len - 1) / len) > (1LL << 17)) len *= 2;
    const int runs = (n_ + len - 1) / len;
    const int blocks = tiles * runs;
    // pairs from the range on add exactly zero; 1e-9 above its square for rounding
    const double range = model_.pair_range;
    const double range2 = std::isfinite(range) ? range * range * (1.0 + 1e-9) : kInf;
    const int bond_blocks = nbonds_ > 0 ? std::min(64, (nbonds_ + kBlock - 1) / kBlock) : 0;
    double* d_part = nullptr; // pair partials, bond partials, pair sum, bond sum
    check_hip(hipMalloc(&d_part, sizeof(double) * (static_cast<size_t>(blocks + bond_blocks) + 2)), "hipMalloc partials");
    double* d_sum = d_part + blocks + bond_blocks;
    double sums[2] = {0.0, 0.0};
    try {
        GroupTable gt{d_gflags_, d_gcm_, d_g2g_, static_cast<int>(model_.molecules.size()), d_excl_off_, d_excl_};
        const auto kernel = any_molecular_ ? (range2 < kInf ? all_pairs_kernel<true, true> : all_pairs_kernel<true, false>)
                                           : (range2 < kInf ? all_pairs_kernel<false, true> : all_pairs_kernel<false, false>);
        hipLaunchKernelGGL(kernel,
                           dim3(static_cast<unsigned>(tiles), static_cast<unsigned>(runs)), dim3(kBlock), 0, stream_,
                           d_pos_, d_meta_, n_, d_pairs_, model_.ntypes, d_coul_, make_box(model_), gt, len, range2, d_part);
        check_hip(hipGetLastError(), "all_pairs_kernel");
        hipLaunchKernelGGL(sum_partials_kernel, dim3(1), dim3(kBlock), 0, stream_, d_part, blocks, d_sum);
        check_hip(hipGetLastError(), "sum_partials_kernel");
        if (bond_blocks > 0) {
            hipLaunchKernelGGL(bond_total_kernel, dim3(bond_blocks), dim3(kBlock), 0, stream_, d_pos_, d_bond_all_,
                               nbonds_, make_box(model_), d_part + blocks);
            check_hip(hipGetLastError(), "bond_total_kernel");
            hipLaunchKernelGGL(sum_partials_kernel, dim3(1), dim3(kBlock), 0, stream_, d_part + blocks, bond_blocks,
                               d_sum + 1);
            check_hip(hipGetLastError(), "sum_partials_kernel");
        }
        check_hip(hipMemcpyAsync(sums, d_sum, sizeof(double) * (bond_blocks > 0 ? 2 : 1), hipMemcpyDeviceToHost, stream_),
                  "copy sums");
        check_hip(hipStreamSynchronize(stream_), "sync");
    } catch (...) {
        (void)hipStreamSynchronize(stream_);
        (void)hipFree(d_part);
        throw;
    }
    (void)hipFree(d_part);
    const double pair = sums[0], bond = sums[1];
    double ewald = 0;
    if (model_.ewald.present) {
        std::vector<double2> q(static_cast<size_t>(nk_));
        check_hip(hipMemcpy(q.data(), d_q_acc_, sizeof(double2) * nk_, hipMemcpyDeviceToHost), "copy q");
        ewald = surface_energy(dipole_) + reciprocal_energy_host(q);
    }
    bool stop = false;
    for (size_t t = 0; t < model_.term_names.size(); ++t) {
        const std::string& name = model_.term_names[t];
        double v = 0.0;
        if (name == "selfenergy") v = self;
        else if (name == "nonbonded") v = pair;
        else if (name == "ewald") v = ewald;
        else if (name == "bonded") v = bond;
        terms[t] = stop ? 0.0 : v;
        if (!stop && (v >= model_.maximum_allowed_energy || std::isnan(v))) stop = true;
    }
}

void Engine::check_q(double* max_abs_dq, double* rel_rec) {
    *max_abs_dq = 0;
    *rel_rec = 0;
    if (!model_.ewald.present) return;
    double2* d_tmp = nullptr;
    check_hip(hipMalloc(&d_tmp, sizeof(double2) * nk_), "hipMalloc q tmp");
    full_q(d_tmp);
    std::vector<double2> qf(static_cast<size_t>(nk_)), qr(static_cast<size_t>(nk_));
    check_hip(hipMemcpyAsync(qf.data(), d_tmp, sizeof(double2) * nk_, hipMemcpyDeviceToHost, stream_), "copy");
    check_hip(hipMemcpyAsync(qr.data(), d_q_acc_, sizeof(double2) * nk_, hipMemcpyDeviceToHost, stream_), "copy");
    check_hip(hipStreamSynchronize(stream_), "sync");
    (void)hipFree(d_tmp);
    double mx = 0;
    for (int k = 0; k < nk_; ++k)
        mx = std::max(mx, std::max(std::fabs(qf[static_cast<size_t>(k)].x - qr[static_cast<size_t>(k)].x),
                                   std::fabs(qf[static_cast<size_t>(k)].y - qr[static_cast<size_t>(k)].y)));
    const double ef = reciprocal_energy_host(qf), er = reciprocal_energy_host(qr);
    *max_abs_dq = mx;
    *rel_rec = (er - ef) / (std::fabs(ef) > 0 ? std::fabs(ef) : 1.0);
}

void Engine::get_positions(double* xyz) const { std::copy(h_xyz_.begin(), h_xyz_.end(), xyz); }

void Engine::reset_positions(const double* xyz, const double* mass_center) {
    if (!d_pos_) throw std::runtime_error("reset_positions: engine not initialised");
    if (pending_) throw std::runtime_error("reset_positions: a move is pending (sync first)");
    check_hip(hipStreamSynchronize(stream_), "sync");
    h_xyz_.assign(xyz, xyz + 3 * static_cast<size_t>(n_));
    std::vector<double4> p(static_cast<size_t>(n_));
    for (int i = 0; i < n_; ++i)
        p[static_cast<size_t>(i)] = make_double4(h_xyz_[3 * i], h_xyz_[3 * i + 1], h_xyz_[3 * i + 2], h_q_[static_cast<size_t>(i)]);
    check_hip(hipMemcpy(d_pos_, p.data(), sizeof(double4) * n_, hipMemcpyHostToDevice), "copy pos");
    const int ng = static_cast<int>(g_begin_.size());
    if (mass_center) g_cm_.assign(mass_center, mass_center + 3 * static_cast<size_t>(ng));
    else
        for (int g = 0; g < ng; ++g)
            if (!model_.molecules[static_cast<size_t>(g_molid_[static_cast<size_t>(g)])].atomic && g_size_[static_cast<size_t>(g)] > 0)
                group_mass_center_host(g, &g_cm_[static_cast<size_t>(3 * g)]);
    check_hip(hipMemcpy(d_gcm_, g_cm_.data(), sizeof(double) * 3 * ng, hipMemcpyHostToDevice), "copy group centres");
    for (int d = 0; d < 3; ++d) {
        dipole_[d] = 0;
        for (int i = 0; i < n_; ++i) dipole_[d] += h_xyz_[3 * i + d] * h_q_[static_cast<size_t>(i)];
    }
    if (model_.ewald.present) {
        full_q(d_q_acc_);
    }
    (void)hipFree(cells_.count);
    (void)hipFree(cells_.members);
    (void)hipFree(cells_.cell_of);
    (void)hipFree(cells_.overflow);
    cells_ = CellList{};
    cell_capacity_ = 0; // a fixed capacity applies to the first build only
    build_cell_list();
}

void Engine::refresh_host_positions() {
    std::vector<double4> p(static_cast<size_t>(n_));
    check_hip(hipStreamSynchronize(stream_), "sync");
    check_hip(hipMemcpy(p.data(), d_pos_, sizeof(double4) * n_, hipMemcpyDeviceToHost), "copy pos");
    for (int i = 0; i < n_; ++i) {
        h_xyz_[3 * i] = p[static_cast<size_t>(i)].x;
        h_xyz_[3 * i + 1] = p[static_cast<size_t>(i)].y;
        h_xyz_[3 * i + 2] = p[static_cast<size_t>(i)].z;
    }
    for (int d = 0; d < 3; ++d) {
        dipole_[d] = 0;
        for (int i = 0; i < n_; ++i) dipole_[d] += h_xyz_[3 * i + d] * h_q_[static_cast<size_t>(i)];
    }
}

} // namespace fmc
