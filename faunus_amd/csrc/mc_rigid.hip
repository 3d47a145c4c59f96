// Device-resident Metropolis for systems of small rigid molecules (water): every group is a
// rigid molecule and every move a translate+rotate (move.cpp:1618-1689), one workgroup per
// replica.  Proposals, energies and decisions are those of mc_general_kernel; the pair sum
// goes over molecules instead of a cell list of atoms.
//
// The mass centres of all molecules stay in LDS as 32-bit fixed-point words (12 bytes each),
// so a move finds the molecules within reach of the moved one's new and old centre by testing
// every centre (4096 waters: 8 per thread, about 0.5 us) with no dependent load, compacts
// them into one list in molecule order and deals the (molecule, atom) items of the list over
// all threads.  mc_general_kernel walked 2 x 125 cells of atoms: three times as many candidates,
// of which 14 % passed the group cutoff, each after a search of its cell in a prefix sum and a
// chain of dependent loads (member, its group, the group's flags, centre and cutoff), and its
// commit edited the cell lists in one thread.
//
// A move takes three barriers: phase tables and candidate counts, the list, the reduction.
// Every wave computes the trial coordinates and the decision for itself.  The k-vectors
// +-nz of a column are summed together from one set of products.
// Per move, mc_general_kernel -> here: 4096 waters, FP32 pairs, group cutoff (8 replicas) 79.5 ->
// 9.2 us; 1728 waters, FP64, splined and cut (4 replicas) 60.6 -> 14.0 us.  What is left is the
// chain of a move's phases, each a few LDS or L2 latencies long at two waves per SIMD, and the
// LDS reads of the pair energies.  1024 threads spill (36 us per move), and so does the form for
// more than two k-vector pairs per thread (K above about 1900): 101 VGPRs in FP64, 173 in FP32; 100
// moves of 4 x 1000 waters with K = 3796 take 1.6 ms there against 7.7 (FP64) on the general kernel.
//
// The LDS holds 16 bytes per molecule beside its tables: about 4900 molecules with FP32 pairs and
// 5900 in FP64 (three atoms, ncut = 9); larger systems, molecules of more than 8 atoms and a cell
// capacity fixed by the caller keep the general kernel (rigid_route, set_rigid_fields).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <stdexcept>

#include "device_math.hpp"
#include "mc_batch.hpp"
#include "mc_common.hpp"
#include "mc_moves.hpp"

namespace fmc {
namespace {

constexpr int kRigidThreads = 512;
constexpr int kRigidWaves = kRigidThreads / 64;
constexpr int kRigidAtoms = 8;         // atoms per molecule, at most
constexpr int kRigidRounds = 16;       // molecules per thread, at most (bits of the pass mask / 2)
constexpr int kRigidEntries = 5;       // k-vector pairs +-nz per thread, at most
constexpr unsigned kListState = 1u << 13, kListCheck = 1u << 14; // list entry: molecule | state | check the cut
static_assert(kRigidThreads * kRigidRounds <= (1 << 13), "a molecule index fits a list entry");

// One state of the moved molecule: atoms, their fixed-point copies and the mass centre.
struct RigidTrial {
    double4 at[2][kRigidAtoms]; // new, old
    FixPos fix[2][kRigidAtoms];
    double centre[2][3];
    int type[kRigidAtoms];
};

// Running values of a replica that only thread 0 keeps.
struct RigidTotals {
    double energy, sum_du, e_sum, e_sum2;
    unsigned long long accepted, e_samples;
};

// Byte offsets of the dynamic LDS.
struct RigidLds {
    size_t pairs, pairs_f, phase, centre, list, total;
};

__host__ __device__ inline RigidLds rigid_lds(int ntypes, int ncut, int ngroups, int nk, bool f32) {
    RigidLds l;
    const size_t nt2 = static_cast<size_t>(ntypes) * static_cast<size_t>(ntypes);
    l.pairs = 0;
    l.pairs_f = l.pairs + nt2 * sizeof(DevPair);
    l.phase = l.pairs_f + (f32 ? nt2 * sizeof(DevPairF) : 0);
    l.centre = l.phase + sizeof(double2) * 6 * kRigidAtoms * static_cast<size_t>(ncut + 1);
    l.list = l.centre + sizeof(uint32_t) * 3 * static_cast<size_t>((ngroups + 3) & ~3);
    const size_t end = l.list + sizeof(unsigned short) * 2 * static_cast<size_t>(ngroups);
    // the k-vectors with nz >= 0 are gathered over the centres and the list at the start
    l.total = end > l.centre + sizeof(int) * static_cast<size_t>(nk) ? end : l.centre + sizeof(int) * static_cast<size_t>(nk);
    return l;
}

template <int kEnt, bool kF32>
__global__ __launch_bounds__(kRigidThreads) void mc_rigid_kernel(ReplicaState* __restrict__ states,
                                                                 const long long* __restrict__ moves,
                                                                 TraceEntry* __restrict__ trace, int trace_cap,
                                                                 ReplicaMap map) {
    constexpr int kT = kRigidThreads;
    const int rep = map.first + map.id[blockIdx.x];
    ReplicaState& S = states[rep];
    const long long M = moves[rep];
    if (M <= 0 || S.error) return;
    __shared__ float4 s_stab[kF32 ? kSTable : 1];
    __shared__ DevCoulomb s_coul;
    __shared__ double s_gk[kMaxGk];
    __shared__ double s_dpa[kMaxTypes];
    __shared__ MoveKindDev s_kinds[kMaxKinds];
    __shared__ MoveDraw s_draw[2][kDraw];
    __shared__ RigidTrial s_trial[2]; // by move parity: a wave may start the next move while another commits
    __shared__ double s_red[3][kRigidWaves];
    __shared__ int s_count[kRigidWaves];
    __shared__ RigidTotals s_tot;
    __shared__ double s_dip[2][3]; // dipole sum before the move (by move parity)
    __shared__ unsigned s_later[kRigidWaves][4 * 64]; // per wave, pairs left to the FP64 coordinates: atom j | state | moved atom
    extern __shared__ __align__(16) unsigned char s_dyn[];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int nk = S.nk, ncut = S.ncut, nt = S.ntypes, ng = S.ngroups;
    const int w = ncut + 1;
    const RigidLds at = rigid_lds(nt, ncut, ng, nk, kF32);
    DevPair* s_pairs = reinterpret_cast<DevPair*>(s_dyn + at.pairs);
    DevPairF* s_pairs_f = reinterpret_cast<DevPairF*>(s_dyn + at.pairs_f);
    double2* s_phase = reinterpret_cast<double2*>(s_dyn + at.phase); // [atom][state][axis][n >= 0]
    uint32_t* s_cx = reinterpret_cast<uint32_t*>(s_dyn + at.centre);
    const int pitch = (ng + 3) & ~3;
    uint32_t *s_cy = s_cx + pitch, *s_cz = s_cy + pitch;
    unsigned short* s_list = reinterpret_cast<unsigned short*>(s_dyn + at.list);
    const double L = S.L, half = S.half, inv = S.inv;

    for (int i = tid; i < nt * nt; i += kT) {
        s_pairs[i] = S.pairs[i];
        if (kF32) s_pairs_f[i] = to_f32(S.pairs[i]);
    }
    lds_copy(s_coul, S.coul, tid, kT);
    for (int i = tid; i < nt; i += kT) s_dpa[i] = S.dp_atom[i];
    for (int i = tid; i < S.nkinds; i += kT) s_kinds[i] = S.kinds[i];
    for (int i = tid; i <= ncut * ncut && i < kMaxGk; i += kT) s_gk[i] = S.gk[i];
    if (kF32 && S.stab)
        for (int i = tid; i < kSTable; i += kT) s_stab[i] = S.stab[i];

    // this thread's k-vectors: consecutive ones of those with nz >= 0, each with its -nz
    // partner (a column holds nz ascending without gaps, except nz = 0 at nx = ny = 0)
    int kp[kEnt];                // index of the +nz k-vector, -1 for none
    int nx[kEnt], ny[kEnt], nz[kEnt]; // ny without its sign (sy)
    double ak[kEnt], sy[kEnt];
    double2 qp[kEnt], qm[kEnt];
    {
        int* s_ent = reinterpret_cast<int*>(s_dyn + at.centre);
        const int run = (nk + kT - 1) / kT, b = min(nk, tid * run), e = min(nk, b + run);
        int cnt = 0, total = 0;
        for (int k = b; k < e; ++k) cnt += unpack_n(S.kn[k], 2) >= 0 ? 1 : 0;
        int pos = block_exclusive_scan<kT>(cnt, s_count, &total);
        for (int k = b; k < e; ++k)
            if (unpack_n(S.kn[k], 2) >= 0) s_ent[pos++] = k;
        __syncthreads();
        const int per = (total + kT - 1) / kT;
#pragma unroll
        for (int s = 0; s < kEnt; ++s) {
            const int i = tid * per + s;
            kp[s] = s < per && i < total ? s_ent[i] : -1;
            nx[s] = ny[s] = nz[s] = 0;
            ak[s] = 0.0;
            sy[s] = 1.0;
            qp[s] = qm[s] = make_double2(0.0, 0.0);
            if (kp[s] < 0) continue;
            const int packed = S.kn[kp[s]];
            nx[s] = unpack_n(packed, 0);
            ny[s] = unpack_n(packed, 1);
            nz[s] = unpack_n(packed, 2);
            ak[s] = (nx[s] > 0 ? 2.0 : 1.0) * s_gk[nx[s] * nx[s] + ny[s] * ny[s] + nz[s] * nz[s]];
            qp[s] = S.q[kp[s]];
            if (nz[s] > 0) qm[s] = S.q[kp[s] - 2 * nz[s] + (nx[s] == 0 && ny[s] == 0 ? 1 : 0)];
            if (ny[s] < 0) {
                ny[s] = -ny[s];
                sy[s] = -1.0;
            }
        }
        __syncthreads();
    }
    double* __restrict__ gcm = S.gcm;
    const double to_fix = kFix * inv;
    for (int h = tid; h < ng; h += kT) {
        s_cx[h] = fixed_coord(gcm[3 * h], to_fix);
        s_cy[h] = fixed_coord(gcm[3 * h + 1], to_fix);
        s_cz[h] = fixed_coord(gcm[3 * h + 2], to_fix);
    }

    const CoulF cf = coul_f32(s_coul);
    const bool splined = s_coul.nspl > 0;
    const CoulF plain{cf.scheme, cf.lB, cf.rc, cf.rc_inv, nullptr}; // without tables
    double4* __restrict__ pos = S.pos;
    FixPos* __restrict__ pos32 = S.pos32;
    const uint32_t* __restrict__ meta = S.meta;
    const float hf = static_cast<float>(L * kFixInv);
    const float reach2 = static_cast<float>(S.reach2), sure2 = static_cast<float>(S.sure2);
    const unsigned long long move0 = S.moves;
    const double beta = S.beta, pref = S.rec_prefactor, surf = S.surf;
    if (tid == 0) {
        s_tot = RigidTotals{S.energy, S.sum_du, S.e_sum, S.e_sum2, S.accepted, S.e_samples};
        for (int d = 0; d < 3; ++d) s_dip[0][d] = S.dip[d];
    }
    const uint32_t replica = static_cast<uint32_t>(S.replica_id);
    const unsigned long long seed = S.seed;
    const Box box{{L, L, L}, {half, half, half}};
    const int terms = S.terms, gmax = S.rigid;
    const bool even = S.rigid_even != 0;
    const int* __restrict__ gbegin = S.gbegin;
    const long long sample_every = S.sample_every;
    const float per_item = 1.0f / static_cast<float>(gmax);

    auto draw = [&](long long t) { // the draws of moves t .. t + kDraw - 1
        if (tid < kDraw)
            draw_move(s_draw[(t / kDraw) & 1][tid], move0 + static_cast<unsigned long long>(t + tid), replica, seed,
                      s_kinds, S.nkinds, S.total_weight, S.kind_groups, gbegin, S.gsize, S.pivot_bonds, meta, s_dpa, nullptr);
    };
    draw(0);
    __syncthreads();

    // the moved molecule's accepted coordinates (atom `lane`) and centre, loaded one move ahead
    double4 p_old = make_double4(0.0, 0.0, 0.0, 0.0);
    int p_type = 0;
    double c_old[3] = {0.0, 0.0, 0.0};
    auto load_molecule = [&](const MoveDraw& D) {
        const int i = min(D.mlo + lane, max(D.mhi - 1, D.mlo));
        p_old = pos[i];
        p_type = static_cast<int>(meta[i] & 0xffu);
        const int g = max(D.group, 0);
        for (int d = 0; d < 3; ++d) c_old[d] = gcm[3 * g + d];
    };
    load_molecule(s_draw[0][0]);
    int g_prev = -1; // the molecule the last move displaced, and its new centre
    uint32_t prev_x = 0, prev_y = 0, prev_z = 0;

    for (long long t = 0; t < M; ++t) {
        const unsigned long long mvi = move0 + static_cast<unsigned long long>(t);
        const MoveDraw& D = s_draw[(t / kDraw) & 1][t % kDraw];
        RigidTrial& R = s_trial[t & 1];
        const int m = D.mhi - D.mlo, g = D.group, first = D.mlo;
        // ---- trial coordinates, by every wave (all write the same values)
        const bool translate = (D.flags & 1) != 0, rotate = (D.flags & 2) != 0;
        double c_new[3] = {c_old[0], c_old[1], c_old[2]};
        if (translate)
            for (int d = 0; d < 3; ++d) c_new[d] = wrap(c_new[d] + D.dir[d], L, half, inv);
        double4 p_new = p_old;
        {
            double x = p_old.x, y = p_old.y, z = p_old.z;
            if (translate) { // Group::translate (group.cpp:115-123)
                x = wrap(x + D.dir[0], L, half, inv);
                y = wrap(y + D.dir[1], L, half, inv);
                z = wrap(z + D.dir[2], L, half, inv);
            }
            if (rotate) { // Geometry::rotate about the mass centre (geometry.h:613-626)
                x = wrap(x - c_new[0], L, half, inv);
                y = wrap(y - c_new[1], L, half, inv);
                z = wrap(z - c_new[2], L, half, inv);
                const double rx = D.R[0] * x + D.R[1] * y + D.R[2] * z;
                const double ry = D.R[3] * x + D.R[4] * y + D.R[5] * z;
                const double rz = D.R[6] * x + D.R[7] * y + D.R[8] * z;
                x = wrap(rx + c_new[0], L, half, inv);
                y = wrap(ry + c_new[1], L, half, inv);
                z = wrap(rz + c_new[2], L, half, inv);
            }
            p_new = make_double4(x, y, z, p_old.w);
        }
        if (lane < m) {
            R.at[0][lane] = p_new;
            R.at[1][lane] = p_old;
            if (kF32) {
                R.fix[0][lane] = fixed_pos(p_new.x, p_new.y, p_new.z, p_new.w, inv);
                R.fix[1][lane] = fixed_pos(p_old.x, p_old.y, p_old.z, p_old.w, inv);
            }
            R.type[lane] = p_type;
        }
        if (lane == 0)
            for (int d = 0; d < 3; ++d) {
                R.centre[0][d] = c_new[d];
                R.centre[1][d] = c_old[d];
            }
        __builtin_amdgcn_wave_barrier(); // this wave's own writes are in order

        // ---- molecules within reach of the new or old centre (the cut is checked exactly
        // later where the fixed-point distance does not settle it)
        const uint32_t nfx = fixed_coord(c_new[0], to_fix), nfy = fixed_coord(c_new[1], to_fix),
                       nfz = fixed_coord(c_new[2], to_fix);
        const uint32_t ofx = fixed_coord(c_old[0], to_fix), ofy = fixed_coord(c_old[1], to_fix),
                       ofz = fixed_coord(c_old[2], to_fix);
        unsigned pass = 0, check = 0; // bits 2 r (new), 2 r + 1 (old) of molecule tid + r kT
        int upto = 0;                 // list entries of this wave's lanes up to this one
        if (m > 0) {
            for (int r0 = 0; r0 * kT < ng; r0 += 4) {
                uint32_t x[4], y[4], z[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int h = min((r0 + r) * kT + tid, ng - 1);
                    x[r] = s_cx[h];
                    y[r] = s_cy[h];
                    z[r] = s_cz[h];
                }
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int h = (r0 + r) * kT + tid, bit = 2 * (r0 + r);
                    const bool moved = h == g_prev;
                    const uint32_t hx = moved ? prev_x : x[r], hy = moved ? prev_y : y[r], hz = moved ? prev_z : z[r];
                    const float ax = static_cast<float>(static_cast<int>(nfx - hx)) * hf,
                                ay = static_cast<float>(static_cast<int>(nfy - hy)) * hf,
                                az = static_cast<float>(static_cast<int>(nfz - hz)) * hf;
                    const float bx = static_cast<float>(static_cast<int>(ofx - hx)) * hf,
                                by = static_cast<float>(static_cast<int>(ofy - hy)) * hf,
                                bz = static_cast<float>(static_cast<int>(ofz - hz)) * hf;
                    const float a2 = ax * ax + ay * ay + az * az, b2 = bx * bx + by * by + bz * bz;
                    const bool in = h < ng && h != g;
                    pass |= ((in && a2 < reach2 ? 1u : 0u) | (in && b2 < reach2 ? 2u : 0u)) << bit;
                    check |= ((a2 >= sure2 ? 1u : 0u) | (b2 >= sure2 ? 2u : 0u)) << bit;
                }
            }
            upto = wave_scan(__popc(pass));
            if (lane == 63) s_count[wave] = upto;
            // ---- Ewald phase tables e^{i k_a(n) r_a}, n >= 0
            for (int e = tid; e < m * 6 * w; e += kT) {
                const int nn = e % w, q = e / w, axis = q % 3, st = (q / 3) & 1, a = q / 6;
                const double4 A = R.at[st][a];
                s_phase[e] = axis_phase(nn, axis == 0 ? A.x : (axis == 1 ? A.y : A.z), inv);
            }
        }
        // the last move of a draw block draws the next one (its buffer was last read before
        // the previous move's barriers)
        if ((t + 1) % kDraw == 0 && t + 1 < M) draw(t + 1);
        __syncthreads();

        // ---- the list (by wave, lane, molecule and state); and the next move's molecule (all
        // earlier commits were issued before the barrier above; this move's is taken below)
        int W = 0;
        if (m > 0) {
            int at = upto - __popc(pass);
#pragma unroll
            for (int v = 0; v < kRigidWaves; ++v) {
                const int c = s_count[v];
                at += v < wave ? c : 0;
                W += c;
            }
            for (; pass != 0; pass &= pass - 1) {
                const int b = __builtin_ctz(pass);
                s_list[at++] = static_cast<unsigned short>(static_cast<unsigned>((b >> 1) * kT + tid) | ((b & 1) ? kListState : 0u) |
                                                           (((check >> b) & 1u) ? kListCheck : 0u));
            }
        }
        const MoveDraw& N = s_draw[((t + 1) / kDraw) & 1][(t + 1) % kDraw];
        const bool again = t + 1 < M;
        if (again) load_molecule(N);
        lds_barrier(); // those loads stay in flight

        double e_new = 0.0, e_old = 0.0, de = 0.0;
        double2 dp[kEnt], dm[kEnt];
#pragma unroll
        for (int s = 0; s < kEnt; ++s) dp[s] = dm[s] = make_double2(0.0, 0.0);
        if (m > 0) {
            const int items = W * gmax;
            unsigned entry = 0;
            int jj;
            uint32_t mj;
            FixPos pf;
            double4 pj;
            mj = 0;
            auto load_item = [&](int w0) {
                jj = -1;
                if (w0 < items) {
                    const int k = static_cast<int>((static_cast<float>(w0) + 0.5f) * per_item), b = w0 - k * gmax;
                    entry = s_list[k];
                    const int h = static_cast<int>(entry & (kListState - 1u));
                    const int hb = even ? h * gmax : gbegin[h];
                    if (even || b < S.gsize[h]) jj = hb + b;
                }
                if (jj >= 0) {
                    mj = meta[jj];
                    if (kF32) pf = pos32[jj];
                    else pj = pos[jj];
                }
            };
            // pairs left to the FP64 coordinates (FP32: hot pairs; FP64: pairs inside their table's
            // first knot, common in water with eps_r = 1) are queued, and the wave evaluates 64 of
            // them side by side
            int queued = 0;
            auto sum_queue = [&]() {
                __builtin_amdgcn_wave_barrier();
                for (int i = lane; i < queued; i += 64) {
                    const unsigned x = s_later[wave][i];
                    const int j = static_cast<int>(x >> 4), st = (x >> 3) & 1u, a = static_cast<int>(x & 7u);
                    const double4 q = pos[j], A = R.at[st][a];
                    const DevPair& p = s_pairs[R.type[a] * nt + static_cast<int>(meta[j] & 0xffu)];
                    const double r2 = dist2(box, A.x, A.y, A.z, q.x, q.y, q.z);
                    const double u = kF32 ? pair_energy_t(p, s_coul, A.w, q.w, r2, terms) : pair_energy_exact(p, s_coul, A.w, q.w, r2);
                    if (st == 0) e_new += u;
                    else e_old += u;
                }
                __builtin_amdgcn_wave_barrier();
                queued = 0;
            };
            auto sum_item = [&]() {
                const int st = (entry & kListState) ? 1 : 0;
                if (jj >= 0 && (entry & kListCheck)) { // GroupCutoff::cut (energy.h:761-768) in FP64
                    const int h = static_cast<int>(entry & (kListState - 1u));
                    const double r2 = dist2(box, R.centre[st][0], R.centre[st][1], R.centre[st][2], gcm[3 * h],
                                            gcm[3 * h + 1], gcm[3 * h + 2]);
                    if (!(r2 < g2g_cutoff2(S.g2g2, S.nmol, S.gflags[g], S.gflags[h]))) jj = -1;
                }
                const int tj = static_cast<int>(mj & 0xffu);
                // three moved atoms at a time, side by side: the chains of LDS reads of one pair
                // energy overlap with the others'
                for (int a0 = 0; a0 < m; a0 += 3) {
                    unsigned later = 0;
                    if (jj >= 0) {
                        double e = 0.0;
#pragma unroll
                        for (int v = 0; v < 3; ++v) {
                            const int a = min(a0 + v, m - 1);
                            const bool ok = a0 + v < m;
                            const int pt = R.type[a] * nt + tj;
                            double u;
                            bool skip = false; // left to the queue
                            if (kF32) {
                                const FixPos A = R.fix[st][a];
                                const float r2 = dist2_fix(A, pf, hf);
                                float uf;
                                if (splined) {
                                    bool below;
                                    uf = static_cast<float>(splined_pair_select(s_coul.spl[s_pairs_f[pt].spl],
                                                                                static_cast<double>(r2), below));
                                    skip = r2 < s_pairs_f[pt].hot_r2;
                                    if (below) uf = pair_energy_ft(s_pairs_f[pt], cf, s_stab, terms, A.q, pf.q, r2, skip);
                                } else {
                                    uf = pair_energy_ft(s_pairs_f[pt], plain, s_stab, terms, A.q, pf.q, r2, skip);
                                }
                                u = static_cast<double>(uf);
                            } else {
                                const double4 A = R.at[st][a];
                                const double r2 = dist2(box, A.x, A.y, A.z, pj.x, pj.y, pj.z);
                                u = splined ? splined_pair_select(s_coul.spl[s_pairs[pt].spl], r2, skip)
                                            : pair_energy_exact(s_pairs[pt], s_coul, A.w, pj.w, r2);
                            }
                            e += ok && !skip ? u : 0.0;
                            later |= ok && skip ? 1u << a : 0u;
                        }
                        if (st == 0) e_new += e;
                        else e_old += e;
                    }
                    const int count = __popc(later), end = wave_scan(count);
                    int at = queued + end - count;
                    for (; later != 0; later &= later - 1)
                        s_later[wave][at++] = (static_cast<unsigned>(jj) << 4) | (st ? 8u : 0u) |
                                              static_cast<unsigned>(__builtin_ctz(later));
                    queued += __builtin_amdgcn_readlane(end, 63);
                    if (queued >= 64) sum_queue();
                }
            };
            load_item(tid);

            // ---- Ewald: dQ(k) = sum_a q_a (e^{ik.r_new} - e^{ik.r_old}) for +-nz, while the
            // first items' loads are in flight
            for (int a = 0; a < m; ++a) {
                const double qa = R.at[0][a].w;
#pragma unroll
                for (int st = 0; st < 2; ++st) {
                    const double2* tb = s_phase + (2 * a + st) * 3 * w;
                    const double sq = st == 0 ? qa : -qa;
#pragma unroll
                    for (int s = 0; s < kEnt; ++s) {
                        const double2 X = tb[nx[s]], Y = tb[w + ny[s]], Z = tb[2 * w + nz[s]];
                        const double yi = sy[s] * Y.y;
                        const double re = sq * (X.x * Y.x - X.y * yi), im = sq * (X.x * yi + X.y * Y.x);
                        const double rc = re * Z.x, is = im * Z.y, rs = re * Z.y, ic = im * Z.x;
                        dp[s].x += rc - is;
                        dp[s].y += rs + ic;
                        dm[s].x += rc + is;
                        dm[s].y += ic - rs;
                    }
                }
            }
#pragma unroll
            for (int s = 0; s < kEnt; ++s) { // unused entries and the partner of nz = 0 have weight zero
                const double x = 2.0 * (qp[s].x * dp[s].x + qp[s].y * dp[s].y) + (dp[s].x * dp[s].x + dp[s].y * dp[s].y);
                const double y = 2.0 * (qm[s].x * dm[s].x + qm[s].y * dm[s].y) + (dm[s].x * dm[s].x + dm[s].y * dm[s].y);
                de += ak[s] * (nz[s] > 0 ? x + y : x);
            }

            sum_item();
            for (int w0 = kT; w0 < items; w0 += kT) {
                load_item(w0 + tid);
                sum_item();
            }
            if (queued > 0) sum_queue();
        }

        // ---- reduction in a fixed order; every thread takes the decision
        {
            const double a = wave_sum(e_new), b = wave_sum(e_old), c = wave_sum(de);
            if (lane == 0) {
                s_red[0][wave] = a;
                s_red[1][wave] = b;
                s_red[2][wave] = c;
            }
        }
        lds_barrier();
        bool acc = true;
        double du = 0.0, mx = 0.0, my = 0.0, mz = 0.0;
        if (m > 0) {
            double v0 = 0.0, v1 = 0.0, v2 = 0.0;
#pragma unroll
            for (int v = 0; v < kRigidWaves; ++v) {
                v0 += s_red[0][v];
                v1 += s_red[1][v];
                v2 += s_red[2][v];
            }
            // the surface term enters with the reciprocal one (Ewald::energy, energy.cpp:581-587)
            double dsurf = 0.0;
            if (surf != 0.0) {
                const double dip0 = s_dip[t & 1][0], dip1 = s_dip[t & 1][1], dip2 = s_dip[t & 1][2];
                mx = dip0;
                my = dip1;
                mz = dip2;
                for (int a = 0; a < m; ++a) {
                    const double4 A = R.at[0][a], B = R.at[1][a];
                    mx += A.w * (A.x - B.x);
                    my += A.w * (A.y - B.y);
                    mz += A.w * (A.z - B.z);
                }
                dsurf = surf * ((mx * mx + my * my + mz * mz) - (dip0 * dip0 + dip1 * dip1 + dip2 * dip2));
            }
            du = energy_change(v0, v1, pref * v2 + dsurf);
            acc = metropolis_log(beta * du, D.accept_u, D.neg_log_u);
        }
        if (tid == 0) {
            if (trace && t < trace_cap) {
                TraceEntry& T = trace[static_cast<size_t>(rep) * trace_cap + t];
                T.index = m > 0 ? first : -1;
                T.accepted = acc ? 1 : 0;
                T.du = du;
                T.x = m > 0 ? R.at[0][0].x : 0.0;
                T.y = m > 0 ? R.at[0][0].y : 0.0;
                T.z = m > 0 ? R.at[0][0].z : 0.0;
            }
            if (acc) {
                ++s_tot.accepted;
                if (m > 0) {
                    s_tot.energy += du;
                    s_tot.sum_du += du;
                }
            }
            if (sample_every > 0 && isfinite(s_tot.energy) &&
                (mvi + 1ull) % static_cast<unsigned long long>(sample_every) == 0ull) {
                s_tot.e_sum += s_tot.energy;
                s_tot.e_sum2 += s_tot.energy * s_tot.energy;
                ++s_tot.e_samples;
            }
            if (surf != 0.0) {
                const bool take = acc && m > 0;
                s_dip[(t + 1) & 1][0] = take ? mx : s_dip[t & 1][0];
                s_dip[(t + 1) & 1][1] = take ? my : s_dip[t & 1][1];
                s_dip[(t + 1) & 1][2] = take ? mz : s_dip[t & 1][2];
            }
        }
        g_prev = -1;
        if (acc && m > 0) {
            if (wave == 0) {
                if (lane < m) {
                    pos[first + lane] = R.at[0][lane];
                    if (kF32) pos32[first + lane] = R.fix[0][lane];
                }
                if (lane == 0) {
                    if (translate) {
                        for (int d = 0; d < 3; ++d) gcm[3 * g + d] = R.centre[0][d];
                    }
                    s_cx[g] = nfx;
                    s_cy[g] = nfy;
                    s_cz[g] = nfz;
                }
            }
            // the centre table is read by faster waves before it is written: they take these
            g_prev = g;
            prev_x = nfx;
            prev_y = nfy;
            prev_z = nfz;
#pragma unroll
            for (int s = 0; s < kEnt; ++s) {
                qp[s].x += dp[s].x;
                qp[s].y += dp[s].y;
                qm[s].x += dm[s].x;
                qm[s].y += dm[s].y;
            }
        }
        // the next move's molecule was loaded before this commit
        if (again && g_prev >= 0 && N.group == g_prev) {
            if (lane < m) p_old = R.at[0][lane];
            for (int d = 0; d < 3; ++d) c_old[d] = R.centre[0][d];
        }
    }

#pragma unroll
    for (int s = 0; s < kEnt; ++s) {
        if (kp[s] < 0) continue;
        S.q[kp[s]] = qp[s];
        if (nz[s] > 0) S.q[kp[s] - 2 * nz[s] + (nx[s] == 0 && ny[s] == 0 ? 1 : 0)] = qm[s];
    }
    if (tid == 0) {
        S.moves = move0 + static_cast<unsigned long long>(M);
        S.accepted = s_tot.accepted;
        S.energy = s_tot.energy;
        S.sum_du = s_tot.sum_du;
        for (int d = 0; d < 3; ++d) S.dip[d] = surf != 0.0 ? s_dip[M & 1][d] : S.dip[d];
        S.e_samples = s_tot.e_samples;
        S.e_sum = s_tot.e_sum;
        S.e_sum2 = s_tot.e_sum2;
    }
}

using RigidKernel = void (*)(ReplicaState*, const long long*, TraceEntry*, int, ReplicaMap);

RigidKernel rigid_kernel(int entries, bool f32) {
    if (entries <= 2) return f32 ? mc_rigid_kernel<2, true> : mc_rigid_kernel<2, false>;
    return f32 ? mc_rigid_kernel<kRigidEntries, true> : mc_rigid_kernel<kRigidEntries, false>;
}

// k-vectors with nz >= 0 of a replica, at most.
int rigid_entries(const ReplicaState& s) {
    const int columns = 2 * s.ncut * s.ncut + 3 * s.ncut + 1; // (nx, ny) of a box around the disc
    const int e = std::min(s.nk, (s.nk + columns) / 2 + 1);
    return (e + kRigidThreads - 1) / kRigidThreads;
}

// Dynamic LDS such a kernel may take: what its static LDS leaves of the CU's 160 KB.
size_t rigid_lds_limit(RigidKernel fn) {
    hipFuncAttributes attr;
    check_hip(hipFuncGetAttributes(&attr, reinterpret_cast<const void*>(fn)), "hipFuncGetAttributes");
    const size_t limit = 160 * 1024 - attr.sharedSizeBytes;
    check_hip(hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize,
                                  static_cast<int>(limit)),
              "hipFuncSetAttribute");
    return limit;
}

size_t rigid_limit(int entries, bool f32) {
    static const size_t limits[4] = {rigid_lds_limit(rigid_kernel(1, false)), rigid_lds_limit(rigid_kernel(1, true)),
                                     rigid_lds_limit(rigid_kernel(kRigidEntries, false)),
                                     rigid_lds_limit(rigid_kernel(kRigidEntries, true))};
    return limits[(entries <= 2 ? 0 : 2) + (f32 ? 1 : 0)];
}

size_t rigid_bytes(const ReplicaState& s, bool f32) { return rigid_lds(s.ntypes, s.ncut, s.ngroups, s.nk, f32).total; }

} // namespace

void set_rigid_fields(const Engine& e, ReplicaState& s, const std::vector<MoveKindSpec>& kinds) {
    s.rigid = s.rigid_even = 0;
    s.ngroups = static_cast<int>(e.group_size().size());
    s.reach2 = s.sure2 = 0.0;
    double reach = 0.0, sure = 0.0;
    if (!e.rigid_reach(&reach, &sure)) return;
    // a capacity fixed by the caller asks for the cell list and its overflow error
    if (e.cell_capacity_fixed()) return;
    for (const MoveKindSpec& k : kinds)
        if (k.kind != 1) return;
    int lo = 1 << 30, hi = 0;
    for (int v : e.group_size()) {
        lo = std::min(lo, v);
        hi = std::max(hi, v);
    }
    // larger molecules and larger systems than the kernel's tables hold keep the general one
    if (hi < 1 || hi > kRigidAtoms || s.ngroups > kRigidThreads * kRigidRounds) return;
    if (s.nk > 8 * kRigidThreads || rigid_entries(s) > kRigidEntries) return; // the general kernel's limit
    s.rigid = hi;
    s.rigid_even = lo == hi ? 1 : 0;
    s.reach2 = reach * reach;
    s.sure2 = sure * sure;
}

bool rigid_route(const ReplicaState& s, bool f32) {
    return s.rigid > 0 && s.parts <= 1 && rigid_bytes(s, f32) <= rigid_limit(rigid_entries(s), f32);
}

void launch_rigid(const ReplicaState* h_states, const std::vector<int>& ids, const ReplicaMap& map, ReplicaState* d_states,
                  const long long* d_moves, bool f32, TraceEntry* trace, int trace_cap, hipStream_t stream) {
    int entries = 1;
    size_t lds = 0;
    for (int r : ids) {
        entries = std::max(entries, rigid_entries(h_states[r]));
        lds = std::max(lds, rigid_bytes(h_states[r], f32));
    }
    (void)rigid_limit(entries, f32); // sets the kernels' attributes
    hipLaunchKernelGGL(rigid_kernel(entries, f32), dim3(static_cast<unsigned>(ids.size())), dim3(kRigidThreads), lds, stream,
                       d_states, d_moves, trace, trace_cap, map);
    check_hip(hipGetLastError(), "mc_rigid_kernel launch");
}

} // namespace fmc
