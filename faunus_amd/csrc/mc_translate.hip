// Device-resident Metropolis of single-particle translations (montecarlo.cpp:139-227,
// move.cpp:225-293), one workgroup per replica, for replicas with few k-vectors per thread.
// The energies and decisions are those of mc_advance_kernel (which keeps the systems with more
// than 8 k-vectors per thread); a move costs less:
//
//   - two barriers (three with a cell list): every thread reduces and decides for itself, so
//     nothing is broadcast; the threshold -log(u) is drawn with the proposal;
//   - the k-vectors +-nz of a column are summed together from one set of products, and the
//     dQ of the sum stays in registers for the commit (it was computed again);
//   - the next particle is loaded a move ahead, and the moved particle's new position reaches
//     the next move's pair row from registers, not through memory;
//   - with a cell list, each cell's members go to a group of lanes of the list's mean
//     occupancy, and the commit's cells are searched by a wave while the others sum.
//
// A pass of the salt ladder up to N = 8571 (48 replicas, FP32 pairs) 23.3 -> 19.2 ms against
// mc_advance_kernel, of the one at N = 1203 (8 replicas, FP64) 5.55 -> 4.38 ms, of 800 moves of 200
// ions with a 27-cell list (FP64) 6.03 -> 3.55 ms.  What is left at N = 8571 is the pair row (VALU
// issue at two waves per SIMD); at small N the chain of the move's phases.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <mutex>
#include <stdexcept>
#include <utility>
#include <vector>

#include "device_math.hpp"
#include "mc_batch.hpp"
#include "mc_common.hpp"
#include "mc_ladder.hpp"
#include "philox.hpp"

namespace fmc {
namespace {

// Running values of a replica that only thread 0 keeps.
struct TranslateTotals {
    double energy, sum_du, e_sum, e_sum2;
    unsigned long long accepted, e_samples;
};

// Two waves per SIMD, so at most 256 VGPRs: with 256 threads two workgroups share a CU, whose
// 160 KB of LDS hold both also in the FP32 form (73.2 KB static and at most 8 KB of k-vectors each;
// with 512 threads, one per CU, A_k is staged in 8 KB more for the set-up).
template <int kThreads, int kEnt, bool kCells, bool kF32>
__global__ __launch_bounds__(kThreads, 2) void mc_translate_kernel(ReplicaState* __restrict__ states,
                                                                const long long* __restrict__ moves,
                                                                TraceEntry* __restrict__ trace, int trace_cap,
                                                                const LadderRun* __restrict__ ladders, ReplicaMap map) {
    constexpr int kWaves = kThreads / 64;
    const int rep = map.first + map.id[blockIdx.x];
    ReplicaState& S = states[rep];
    const long long M = moves[rep];
    // free-running ladders: every replica takes part in its ladder's barriers, also one
    // with no moves or an error
    const int n_iv = ladders != nullptr ? ladders->intervals[rep] : 1;
    if (ladders == nullptr && (M <= 0 || S.error)) return;
    __shared__ DevPair s_pairs[kMaxTypes * kMaxTypes];
    __shared__ DevPairF s_pairs_f[kF32 ? kMaxTypes * kMaxTypes : 1];
    __shared__ float4 s_stab[kF32 ? kSTable : 1];
    __shared__ DevCoulomb s_coul;
    __shared__ double s_dp[kMaxTypes];
    __shared__ double s_gk[kThreads > 256 ? kMaxGk : 1];
    __shared__ double s_red[3][kWaves];
    __shared__ int s_scan[kWaves];
    __shared__ int s_nhot[2]; // hot pairs queued (FP32 form), by move parity
    __shared__ int s_stop;    // a full cell stopped the chain
    __shared__ int2 s_hot[kF32 ? kHotCap : 1];
    __shared__ Proposal s_prop[2][64]; // proposals drawn one per lane, two blocks
    __shared__ double s_nlu[2][64];    // -log of their acceptance deviates
    __shared__ double s_dip[2][3];     // dipole sum before the move (by move parity)
    __shared__ TranslateTotals s_tot;
    extern __shared__ double2 s_phase[]; // [state][axis][n >= 0]; first the k-vectors with nz >= 0

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int n = S.n, nk = S.nk, ncut = S.ncut, nt = S.ntypes;
    const int w = ncut + 1;
    const double L = S.L, half = S.half, inv = S.inv;
    for (int i = tid; i < nt * nt; i += kThreads) {
        s_pairs[i] = S.pairs[i];
        if (kF32) s_pairs_f[i] = to_f32(S.pairs[i]);
    }
    lds_copy(s_coul, S.coul, tid, kThreads);
    for (int i = tid; i < nt; i += kThreads) s_dp[i] = S.dp_type[i];
    if (kThreads > 256)
        for (int i = tid; i <= ncut * ncut && i < kMaxGk; i += kThreads) s_gk[i] = S.gk[i];
    if (kF32 && S.stab)
        for (int i = tid; i < kSTable; i += kThreads) s_stab[i] = S.stab[i];
    if (tid == 0) {
        s_tot = TranslateTotals{S.energy, S.sum_du, S.e_sum, S.e_sum2, S.accepted, S.e_samples};
        for (int d = 0; d < 3; ++d) s_dip[0][d] = S.dip[d];
        s_nhot[0] = s_nhot[1] = s_stop = 0;
    }

    // this thread's k-vectors: consecutive ones of those with nz >= 0, each with its -nz
    // partner (a column holds nz ascending without gaps, except nz = 0 at nx = ny = 0)
    int kp[kEnt], nx[kEnt], ny[kEnt], nz[kEnt]; // ny without its sign (sy)
    double ak[kEnt], sy[kEnt];
    double2 qp[kEnt], qm[kEnt];
    {
        int* s_ent = reinterpret_cast<int*>(s_phase);
        const int run = (nk + kThreads - 1) / kThreads, b = min(nk, tid * run), e = min(nk, b + run);
        int cnt = 0, total = 0;
        for (int k = b; k < e; ++k) cnt += unpack_n(S.kn[k], 2) >= 0 ? 1 : 0;
        int at = block_exclusive_scan<kThreads>(cnt, s_scan, &total);
        for (int k = b; k < e; ++k)
            if (unpack_n(S.kn[k], 2) >= 0) s_ent[at++] = k;
        __syncthreads();
        const int per = (total + kThreads - 1) / kThreads;
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
            const int n2 = nx[s] * nx[s] + ny[s] * ny[s] + nz[s] * nz[s];
            ak[s] = (nx[s] > 0 ? 2.0 : 1.0) * (kThreads > 256 ? s_gk[n2] : S.gk[n2]);
            qp[s] = S.q[kp[s]];
            if (nz[s] > 0) qm[s] = S.q[kp[s] - 2 * nz[s] + (nx[s] == 0 && ny[s] == 0 ? 1 : 0)];
            if (ny[s] < 0) {
                ny[s] = -ny[s];
                sy[s] = -1.0;
            }
        }
        __syncthreads();
    }

    const CoulF cf = coul_f32(s_coul);
    const int form = pair_form(s_coul, S.terms, kF32);
    double4* __restrict__ pos = S.pos;
    FixPos* __restrict__ pos32 = S.pos32;
    const uint32_t* __restrict__ meta = S.meta;
    const float hf = static_cast<float>(L * kFixInv);
    unsigned long long move0 = S.moves;
    double beta = S.beta;
    const double pref = S.rec_prefactor, surf = S.surf;
    const int replica = S.replica_id, terms = S.terms;
    const unsigned long long seed = S.seed;
    const long long sample_every = S.sample_every;
    const Box box{{L, L, L}, {half, half, half}};
    const double inv_cell = S.inv_cell;
    const int nc = S.nc0; // a cubic grid
    const int cap = S.cap;
    int* __restrict__ cell_count = S.cell_count;
    int* __restrict__ cell_members = S.cell_members;
    int* __restrict__ cell_of = S.cell_of;
    // lanes per cell of the stencils: the mean occupancy, a power of two, at most what gives
    // each of the 54 cells a group of its own at once
    int cell_shift = 0; // log2 of the lanes
    if (kCells) {
        const int mean = n / (nc * nc * nc);
        while ((1 << cell_shift) < mean && (54 << (cell_shift + 1)) <= kThreads) ++cell_shift;
    }
    const int cell_lanes = 1 << cell_shift;
    auto cell_at = [&](double x, double y, double z) {
        return (cell_of_coord(z, half, inv_cell, nc) * nc + cell_of_coord(y, half, inv_cell, nc)) * nc +
               cell_of_coord(x, half, inv_cell, nc);
    };
    long long dip_at = 0; // parity of s_dip and s_nhot over all intervals

    for (int iv = 0; iv < n_iv; ++iv) {
        const long long Mi = (M > 0 && !S.error) ? M : 0;
        long long t_done = Mi; // moves decided in this interval
        auto draw = [&](long long t) { // the proposals of moves t .. t + 63
            if (tid < 64) {
                const int b = static_cast<int>((t / 64) & 1);
                s_prop[b][tid] = make_proposal(seed, static_cast<uint32_t>(replica),
                                               move0 + static_cast<unsigned long long>(t + tid), n);
                s_nlu[b][tid] = -log(s_prop[b][tid].accept_u);
            }
        };
        double4 po = make_double4(0.0, 0.0, 0.0, 0.0); // the moved particle, loaded one move ahead
        int ti = 0, cold = 0, cnew = 0; // its type, and its cell before and after the move (the latter: last wave)
        if (Mi > 0) {
            draw(0);
            __syncthreads();
            po = pos[s_prop[0][0].index];
            ti = static_cast<int>(meta[s_prop[0][0].index] & 0xffu);
            if (kCells) cold = cell_of[s_prop[0][0].index];
        }
        // the particle the last move displaced (its store may be under way)
        int moved = -1;
        double4 moved_at = po;
        FixPos moved_fix{0u, 0u, 0u, 0.0f};
        for (long long t = 0; t < Mi; ++t, ++dip_at) {
            const Proposal P = s_prop[(t / 64) & 1][t & 63];
            const int i = P.index;
            const double scale = s_dp[ti] * P.length_u;
            const double nx_ = wrap(po.x + P.dir[0] * scale, L, half, inv);
            const double ny_ = wrap(po.y + P.dir[1] * scale, L, half, inv);
            const double nz_ = wrap(po.z + P.dir[2] * scale, L, half, inv);
            int* nhot = &s_nhot[dip_at & 1];

            // Ewald phase tables e^{i k_a(n) r_a}, n >= 0, new (st = 0) and old (st = 1), by the last threads
            for (int e = kThreads - 1 - tid; e < 6 * w; e += kThreads) {
                const int nn = e % w, axis = (e / w) % 3, st = e / (3 * w);
                const double x = st == 0 ? (axis == 0 ? nx_ : (axis == 1 ? ny_ : nz_))
                                         : (axis == 0 ? po.x : (axis == 1 ? po.y : po.z));
                s_phase[e] = axis_phase(nn, x, inv);
            }

            // nonbonded pair sums of the moved particle in the new and old position
            double e_new = 0.0, e_old = 0.0;
            FixPos fa{}, fb{};
            if (kF32) {
                fa = fixed_pos(nx_, ny_, nz_, po.w, inv);
                fb = fixed_pos(po.x, po.y, po.z, po.w, inv);
            }
            if (!kCells) {
                with_form(form, [&](auto f) __attribute__((always_inline)) {
                    if (kF32)
                        pair_row_f32<kThreads, f()>(pos32, meta, 0, n, i, -1, true, s_pairs_f + ti * nt, cf, s_stab, terms, hf,
                                                    fa, fb, nhot, s_hot, 0, e_new, e_old, moved, moved_fix);
                    else
                        pair_row_f64<kThreads, f()>(pos, meta, 0, n, i, -1, true, s_pairs + ti * nt, s_coul, terms, box, nx_,
                                                    ny_, nz_, po.x, po.y, po.z, po.w, e_new, e_old, moved, moved_at);
                });
            } else {
                // 27-cell stencils around the new (st = 0) and old (st = 1) position
                with_form(form, [&](auto f) __attribute__((always_inline)) {
                    for (int combo = tid >> cell_shift; combo < 54; combo += kThreads >> cell_shift) {
                        const int st = combo / 27, c = combo % 27;
                        const double px = st == 0 ? nx_ : po.x, py = st == 0 ? ny_ : po.y, pz = st == 0 ? nz_ : po.z;
                        int cx = cell_of_coord(px, half, inv_cell, nc) + (c % 3) - 1;
                        int cy = cell_of_coord(py, half, inv_cell, nc) + ((c / 3) % 3) - 1;
                        int cz = cell_of_coord(pz, half, inv_cell, nc) + (c / 9) - 1;
                        cx += cx < 0 ? nc : (cx >= nc ? -nc : 0);
                        cy += cy < 0 ? nc : (cy >= nc ? -nc : 0);
                        cz += cz < 0 ? nc : (cz >= nc ? -nc : 0);
                        const int cell = (cz * nc + cy) * nc + cx;
                        const int cnt = cell_count[cell];
                        constexpr int kU = 2;
                        for (int k0 = tid & (cell_lanes - 1); k0 < cnt; k0 += cell_lanes * kU) {
                            int j[kU];
                            uint32_t mj[kU];
                            double4 pj[kU];
                            FixPos pf[kU];
#pragma unroll
                            for (int u = 0; u < kU; ++u)
                                j[u] = cell_members[cell * cap + min(k0 + u * cell_lanes, cnt - 1)];
#pragma unroll
                            for (int u = 0; u < kU; ++u) {
                                mj[u] = meta[j[u]];
                                if (kF32) pf[u] = pos32[j[u]];
                                else pj[u] = pos[j[u]];
                            }
#pragma unroll
                            for (int u = 0; u < kU; ++u) {
                                const bool ok = k0 + u * cell_lanes < cnt && j[u] != i;
                                const int pt = ti * nt + static_cast<int>(mj[u] & 0xffu);
                                double e;
                                if (kF32) {
                                    const FixPos A = st == 0 ? fa : fb;
                                    bool hot;
                                    const float uf = pair_f32<f()>(s_pairs_f[pt], cf, s_stab, terms, A.q, pf[u].q,
                                                                   dist2_fix(A, pf[u], hf), hot);
                                    e = (ok && hot && push_hot(nhot, s_hot, j[u], st)) ? 0.0 : static_cast<double>(uf);
                                } else {
                                    const double r2 = dist2(box, px, py, pz, pj[u].x, pj[u].y, pj[u].z);
                                    e = f() == kFormAny ? pair_energy(s_pairs[pt], s_coul, po.w, pj[u].w, r2)
                                                        : pair_f64<f()>(s_pairs[pt], s_coul, po.w, pj[u].w, r2, terms);
                                }
                                if (st == 0) e_new += ok ? e : 0.0;
                                else e_old += ok ? e : 0.0;
                            }
                        }
                    }
                });
            }
            // the last move of a block of proposals draws the next block
            if ((t & 63) == 63 && t + 1 < Mi) draw(t + 1);
            __syncthreads(); // phase tables, hot-pair queue, next proposals; earlier commits are in memory

            // the next move's particle
            const bool again = t + 1 < Mi;
            const int i1 = s_prop[((t + 1) / 64) & 1][(t + 1) & 63].index;
            double4 po1 = po;
            int ti1 = ti, cold1 = 0;
            if (again) {
                po1 = pos[i1];
                ti1 = static_cast<int>(meta[i1] & 0xffu);
                if (kCells) cold1 = cell_of[i1];
            }
            if (kF32) {
                // hot pairs in FP64 from the FP64 coordinates
                const int nh = min(*nhot, kHotCap);
                for (int h = tid; h < nh; h += kThreads) {
                    const int2 e = s_hot[h];
                    const double4 pj = !kCells && e.x == moved ? moved_at : pos[e.x];
                    const int tj = static_cast<int>(meta[e.x] & 0xffu);
                    const bool nw = (e.y & 1) == 0;
                    const double u = pair_energy_t(s_pairs[ti * nt + tj], s_coul, po.w, pj.w,
                                                   dist2(box, nw ? nx_ : po.x, nw ? ny_ : po.y, nw ? nz_ : po.z, pj.x, pj.y, pj.z),
                                                   terms);
                    if (nw) e_new += u;
                    else e_old += u;
                }
                if (tid == 0) s_nhot[(dip_at + 1) & 1] = 0; // read by every thread before the last reduction
            }
            // the commit's cells (last wave): counts, the moved particle's slot, the last member
            int nold = 0, nnew = 0, slot = -1, last_member = 0;
            if (kCells && wave == kWaves - 1) {
                cnew = cell_at(nx_, ny_, nz_);
                if (cold != cnew) {
                    nold = cell_count[cold];
                    nnew = cell_count[cnew];
                    for (int k = 0; k < nold && slot < 0; k += 64) {
                        const unsigned long long found =
                            __ballot(k + lane < nold && cell_members[cold * cap + min(k + lane, nold - 1)] == i);
                        if (found) slot = k + __builtin_ctzll(found);
                    }
                    last_member = cell_members[cold * cap + nold - 1];
                }
            }

            // Ewald: dE = sum_k A_k (2 Re(conj(Q) dQ) + |dQ|^2) over this thread's k-vectors
            double de = 0.0;
            double2 dqp[kEnt], dqm[kEnt];
#pragma unroll
            for (int s = 0; s < kEnt; ++s) {
                double re[2], im[2], zc[2], zs[2];
#pragma unroll
                for (int st = 0; st < 2; ++st) {
                    const double2* tb = s_phase + st * 3 * w;
                    const double2 X = tb[nx[s]], Y = tb[w + ny[s]], Z = tb[2 * w + nz[s]];
                    const double yi = sy[s] * Y.y;
                    re[st] = X.x * Y.x - X.y * yi;
                    im[st] = X.x * yi + X.y * Y.x;
                    zc[st] = Z.x;
                    zs[st] = Z.y;
                }
                const double rc = re[0] * zc[0] - re[1] * zc[1], is = im[0] * zs[0] - im[1] * zs[1];
                const double rs = re[0] * zs[0] - re[1] * zs[1], ic = im[0] * zc[0] - im[1] * zc[1];
                dqp[s] = make_double2(po.w * (rc - is), po.w * (rs + ic));
                dqm[s] = make_double2(po.w * (rc + is), po.w * (ic - rs));
                // unused entries and the partner of nz = 0 have weight zero
                const double x = 2.0 * (qp[s].x * dqp[s].x + qp[s].y * dqp[s].y) + (dqp[s].x * dqp[s].x + dqp[s].y * dqp[s].y);
                const double y = 2.0 * (qm[s].x * dqm[s].x + qm[s].y * dqm[s].y) + (dqm[s].x * dqm[s].x + dqm[s].y * dqm[s].y);
                de += ak[s] * (nz[s] > 0 ? x + y : x);
            }

            // reduction in a fixed order; every thread takes the decision
            {
                const double a = wave_sum(e_new), b = wave_sum(e_old), c = wave_sum(de);
                if (lane == 0) {
                    s_red[0][wave] = a;
                    s_red[1][wave] = b;
                    s_red[2][wave] = c;
                }
            }
            lds_barrier(); // the next particle's loads stay in flight
            double v0 = 0.0, v1 = 0.0, v2 = 0.0;
#pragma unroll
            for (int v = 0; v < kWaves; ++v) {
                v0 += s_red[0][v];
                v1 += s_red[1][v];
                v2 += s_red[2][v];
            }
            // the surface term enters with the reciprocal one (Ewald::energy, energy.cpp:581-587)
            double dsurf = 0.0, mx = 0.0, my = 0.0, mz = 0.0;
            if (surf != 0.0) {
                const double d0 = s_dip[dip_at & 1][0], d1 = s_dip[dip_at & 1][1], d2 = s_dip[dip_at & 1][2];
                mx = d0 + po.w * (nx_ - po.x);
                my = d1 + po.w * (ny_ - po.y);
                mz = d2 + po.w * (nz_ - po.z);
                dsurf = surf * ((mx * mx + my * my + mz * mz) - (d0 * d0 + d1 * d1 + d2 * d2));
            }
            const double du = energy_change(v0, v1, pref * v2 + dsurf);
            const bool acc = metropolis_log(beta * du, P.accept_u, s_nlu[(t / 64) & 1][t & 63]);
            if (tid == 0) {
                if (trace && t < trace_cap) {
                    TraceEntry& T = trace[static_cast<size_t>(rep) * trace_cap + t];
                    T.index = i;
                    T.accepted = acc ? 1 : 0;
                    T.du = du;
                    T.x = nx_;
                    T.y = ny_;
                    T.z = nz_;
                }
                if (acc) {
                    s_tot.energy += du;
                    s_tot.sum_du += du;
                    ++s_tot.accepted;
                }
                if (sample_every > 0 && isfinite(s_tot.energy) &&
                    (move0 + static_cast<unsigned long long>(t) + 1ull) % static_cast<unsigned long long>(sample_every) == 0ull) {
                    s_tot.e_sum += s_tot.energy;
                    s_tot.e_sum2 += s_tot.energy * s_tot.energy;
                    ++s_tot.e_samples;
                }
                if (surf != 0.0) {
                    s_dip[(dip_at + 1) & 1][0] = acc ? mx : s_dip[dip_at & 1][0];
                    s_dip[(dip_at + 1) & 1][1] = acc ? my : s_dip[dip_at & 1][1];
                    s_dip[(dip_at + 1) & 1][2] = acc ? mz : s_dip[dip_at & 1][2];
                }
            }
            moved = -1;
            if (acc) {
                moved = i;
                moved_at = make_double4(nx_, ny_, nz_, po.w);
                moved_fix = fa;
                if (wave == kWaves - 1 && lane == 0) {
                    pos[i] = moved_at;
                    if (kF32) pos32[i] = fa;
                    if (kCells && cnew != cold) {
                        if (nnew >= cap) {
                            // full cell: the lists are left as they are and the chain stops
                            // after this move
                            S.error = 1;
                            s_stop = 1;
                        } else {
                            if (slot >= 0) cell_members[cold * cap + slot] = last_member;
                            cell_count[cold] = nold - 1;
                            cell_members[cnew * cap + nnew] = i;
                            cell_count[cnew] = nnew + 1;
                            cell_of[i] = cnew;
                        }
                    }
                }
#pragma unroll
                for (int s = 0; s < kEnt; ++s) {
                    qp[s].x += dqp[s].x;
                    qp[s].y += dqp[s].y;
                    qm[s].x += dqm[s].x;
                    qm[s].y += dqm[s].y;
                }
            }
            po = again && i1 == moved ? moved_at : po1;
            ti = ti1;
            if (kCells) {
                cold = i1 == moved ? cnew : cold1; // (last wave's)
                __syncthreads(); // the commit, before the next move walks the lists
                if (s_stop) {
                    t_done = t + 1;
                    ++dip_at;
                    break;
                }
            }
        }

        __syncthreads();
        if (tid == 0) {
            S.moves = move0 + static_cast<unsigned long long>(t_done);
            S.accepted = s_tot.accepted;
            S.energy = s_tot.energy;
            S.sum_du = s_tot.sum_du;
            if (surf != 0.0)
                for (int d = 0; d < 3; ++d) S.dip[d] = s_dip[dip_at & 1][d];
            S.e_samples = s_tot.e_samples;
            S.e_sum = s_tot.e_sum;
            S.e_sum2 = s_tot.e_sum2;
            if (ladders != nullptr) {
                ladder_barrier(*ladders, rep, states, S, iv, beta);
                s_red[0][0] = beta;
            }
        }
        move0 += static_cast<unsigned long long>(t_done);
        __syncthreads(); // the interval's state and error are written before the next interval reads them
        if (ladders != nullptr) beta = s_red[0][0];
        __syncthreads();
    }

#pragma unroll
    for (int s = 0; s < kEnt; ++s) {
        if (kp[s] < 0) continue;
        S.q[kp[s]] = qp[s];
        if (nz[s] > 0) S.q[kp[s] - 2 * nz[s] + (nx[s] == 0 && ny[s] == 0 ? 1 : 0)] = qm[s];
    }
}

using TranslateKernel = void (*)(ReplicaState*, const long long*, TraceEntry*, int, const LadderRun*, ReplicaMap);

template <int kThreads> TranslateKernel select_translate(int entries, bool cells, bool f32) {
    if (entries <= 2) {
        if (cells) return f32 ? mc_translate_kernel<kThreads, 2, true, true> : mc_translate_kernel<kThreads, 2, true, false>;
        return f32 ? mc_translate_kernel<kThreads, 2, false, true> : mc_translate_kernel<kThreads, 2, false, false>;
    }
    if (cells) return f32 ? mc_translate_kernel<kThreads, 5, true, true> : mc_translate_kernel<kThreads, 5, true, false>;
    return f32 ? mc_translate_kernel<kThreads, 5, false, true> : mc_translate_kernel<kThreads, 5, false, false>;
}

// Dynamic LDS a kernel may take: what its static LDS leaves of the CU's 160 KB (set once).
size_t translate_lds_limit(const void* fn) {
    static std::mutex mutex;
    static std::vector<std::pair<const void*, size_t>> done;
    const std::lock_guard<std::mutex> lock(mutex);
    for (const auto& d : done)
        if (d.first == fn) return d.second;
    hipFuncAttributes attr;
    check_hip(hipFuncGetAttributes(&attr, fn), "hipFuncGetAttributes");
    const size_t limit = 160 * 1024 - attr.sharedSizeBytes;
    check_hip(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(limit)),
              "hipFuncSetAttribute");
    done.emplace_back(fn, limit);
    return limit;
}

} // namespace

void launch_translate(const ReplicaState* h_states, const std::vector<int>& ids, const ReplicaMap& map, int threads,
                      ReplicaState* d_states, const long long* d_moves, bool f32, TraceEntry* trace, int trace_cap,
                      hipStream_t stream, const LadderRun* ladders) {
    const int count = static_cast<int>(ids.size());
    const bool cells = h_states[ids[0]].cells != 0;
    int entries = 1;
    size_t lds = 0;
    for (int r : ids) {
        const ReplicaState& s = h_states[r];
        // k-vectors with nz >= 0, at most: half of those in columns without nz = 0, plus the columns
        const int columns = 2 * s.ncut * s.ncut + 3 * s.ncut + 1;
        const int e = std::min(s.nk, (s.nk + columns) / 2 + 1);
        entries = std::max(entries, (e + threads - 1) / threads);
        lds = std::max({lds, sizeof(double2) * 6 * static_cast<size_t>(s.ncut + 1), sizeof(int) * static_cast<size_t>(s.nk)});
    }
    if (entries > 5) throw std::runtime_error("too many k-vectors per thread for the translation kernel");
    const TranslateKernel fn =
        threads == 512 ? select_translate<512>(entries, cells, f32) : select_translate<256>(entries, cells, f32);
    if (lds > translate_lds_limit(reinterpret_cast<const void*>(fn)))
        throw std::runtime_error("k-vector table too large for LDS");
    if (ladders == nullptr) {
        hipLaunchKernelGGL(fn, dim3(static_cast<unsigned>(count)), dim3(static_cast<unsigned>(threads)), lds, stream, d_states,
                           d_moves, trace, trace_cap, ladders, map);
        check_hip(hipGetLastError(), "mc_translate_kernel launch");
        return;
    }
    // ladders wait for each other: every workgroup must be resident at once
    int dev = 0, per_cu = 0;
    hipDeviceProp_t prop;
    check_hip(hipGetDevice(&dev), "hipGetDevice");
    check_hip(hipGetDeviceProperties(&prop, dev), "hipGetDeviceProperties");
    check_hip(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void*>(fn), threads, lds),
              "occupancy");
    if (per_cu * prop.multiProcessorCount < count)
        throw std::runtime_error("run_ladders: the replicas cannot all be resident at once");
    ReplicaMap by_value = map;
    void* args[] = {&d_states, &d_moves, &trace, &trace_cap, &ladders, &by_value};
    check_hip(hipLaunchCooperativeKernel(reinterpret_cast<const void*>(fn), dim3(static_cast<unsigned>(count)),
                                         dim3(static_cast<unsigned>(threads)), args, static_cast<unsigned>(lds), stream),
              "mc_translate_kernel cooperative launch");
}

} // namespace fmc
