// Device-resident Metropolis of single-particle translations for replicas with more than 8
// k-vectors per thread (mc_translate_kernel takes the others): the kernel and its launch, in
// two sources, since the form for up to 32 k-vectors per thread and the one for up to 68 are
// compiled with different flags (see the Makefile).
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <stdexcept>

#include "device_math.hpp"
#include "mc_batch.hpp"
#include "mc_common.hpp"
#include "mc_ladder.hpp"
#include "philox.hpp"

namespace fmc {
namespace {

constexpr int kAdvanceThreads = 256;

template <int kMaxKPT, bool kCells, bool kF32>
__global__ __launch_bounds__(kAdvanceThreads) void mc_advance_kernel(ReplicaState* __restrict__ states,
                                                               const long long* __restrict__ moves,
                                                               TraceEntry* __restrict__ trace, int trace_cap,
                                                               const LadderRun* __restrict__ ladders, ReplicaMap map) {
    constexpr int kThreads = kAdvanceThreads;
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
    __shared__ double s_gk[kMaxGk];
    __shared__ double s_red[3][kThreads / 64];
    __shared__ int s_accept;
    __shared__ int s_nhot;                        // hot pairs queued this move (FP32 form)
    __shared__ int2 s_hot[kF32 ? kHotCap : 1];
    __shared__ Proposal s_prop[64]; // the next 64 proposals, drawn one per lane of wave 0
    extern __shared__ int s_dyn[]; // kn[nk] followed by the phase tables (double2)

    const int tid = threadIdx.x;
    const int n = S.n, nk = S.nk, ncut = S.ncut, nt = S.ntypes;
    const int width = 2 * ncut + 1;
    const int kpt = (nk + kThreads - 1) / kThreads;
    const double L = S.L, half = S.half, inv = S.inv;
    int* s_kn = s_dyn;
    double2* s_phase = reinterpret_cast<double2*>(s_dyn + ((nk + 3) & ~3));

    for (int i = tid; i < nt * nt; i += kThreads) {
        s_pairs[i] = S.pairs[i];
        if (kF32) {
            const DevPair& p = S.pairs[i];
            s_pairs_f[i] = to_f32(p);
        }
    }
    lds_copy(s_coul, S.coul, tid, kThreads);
    for (int i = tid; i < nt; i += kThreads) s_dp[i] = S.dp_type[i];
    for (int i = tid; i <= ncut * ncut && i < kMaxGk; i += kThreads) s_gk[i] = S.gk[i];
    for (int k = tid; k < nk; k += kThreads) s_kn[k] = S.kn[k];
    __syncthreads();
    if (kF32) {
        if (S.stab)
            for (int i = tid; i < kSTable; i += kThreads) s_stab[i] = S.stab[i];
    }
    const CoulF cf = coul_f32(s_coul);
    const int form = pair_form(s_coul, S.terms, kF32);

    // this thread's chunk of k-vectors and their running structure factors
    const int k0 = tid * kpt;
    double2 q[kMaxKPT];
#pragma unroll
    for (int s = 0; s < kMaxKPT; ++s) q[s] = (s < kpt && k0 + s < nk) ? S.q[k0 + s] : make_double2(0.0, 0.0);

    double4* __restrict__ pos = S.pos;
    FixPos* __restrict__ pos32 = S.pos32;
    const uint32_t* __restrict__ meta = S.meta;
    const float hf = static_cast<float>(L * kFixInv);
    unsigned long long move0 = S.moves;
    double beta = S.beta; // thread 0's (a ladder swap changes it between intervals)
    const double pref = S.rec_prefactor;
    const double surf = S.surf;
    double dip0 = S.dip[0], dip1 = S.dip[1], dip2 = S.dip[2]; // thread 0's running dipole
    double energy = S.energy, sum_du = S.sum_du;
    unsigned long long accepted = S.accepted;
    const int replica = S.replica_id;
    const unsigned long long seed = S.seed;
    const long long sample_every = S.sample_every;
    unsigned long long e_samples = S.e_samples;
    double e_sum = S.e_sum, e_sum2 = S.e_sum2;
    if (tid == 0) s_nhot = 0;
    __syncthreads();

    for (int iv = 0; iv < n_iv; ++iv) {
    const long long Mi = (M > 0 && !S.error) ? M : 0;
    long long t_done = Mi; // moves decided in this interval
    for (long long t = 0; t < Mi; ++t) {
        if ((t & 63) == 0) {
            // the previous proposals were last read before this move's barriers; the
            // Philox blocks and sin/cos of 64 moves overlap instead of forming one serial
            // chain per move
            if (tid < 64)
                s_prop[tid] = make_proposal(seed, static_cast<uint32_t>(replica),
                                            move0 + static_cast<unsigned long long>(t + tid), n);
            __syncthreads();
        }
        const Proposal P = s_prop[t & 63];
        const int i = P.index;
        const double4 po = pos[i];
        const int ti = static_cast<int>(meta[i] & 0xffu);
        const double dp = s_dp[ti];
        const double scale = dp * P.length_u;
        const double nx_ = wrap(po.x + P.dir[0] * scale, L, half, inv);
        const double ny_ = wrap(po.y + P.dir[1] * scale, L, half, inv);
        const double nz_ = wrap(po.z + P.dir[2] * scale, L, half, inv);

        // Ewald phase tables e^{i k_a(n) r_a}, n in [-ncut, ncut], new (st=0) and old (st=1)
        for (int e = tid; e < 6 * width; e += kThreads) {
            const int nn = e % width - ncut;
            const int axis = (e / width) % 3;
            const int st = e / (3 * width);
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
                if (kF32) {
                    pair_row_f32<kThreads, f()>(pos32, meta, 0, n, i, -1, true, s_pairs_f + ti * nt, cf, s_stab, S.terms, hf,
                                                fa, fb, &s_nhot, s_hot, 0, e_new, e_old);
                } else {
                    const Box b{{L, L, L}, {half, half, half}};
                    pair_row_f64<kThreads, f()>(pos, meta, 0, n, i, -1, true, s_pairs + ti * nt, s_coul, S.terms, b, nx_,
                                                ny_, nz_, po.x, po.y, po.z, po.w, e_new, e_old);
                }
            });
        } else {
            // 27-cell stencils around the new (st=0) and old (st=1) position
            const int lanes_per = kThreads / 54 > 0 ? kThreads / 54 : 1;
            const int combo = tid / lanes_per;
            const int slot0 = tid % lanes_per;
            if (combo < 54) {
                const int st = combo / 27, c = combo % 27;
                const double px = st == 0 ? nx_ : po.x, py = st == 0 ? ny_ : po.y, pz = st == 0 ? nz_ : po.z;
                const int cx = (cell_of_coord(px, half, S.inv_cell, S.nc0) + (c % 3) - 1 + S.nc0) % S.nc0;
                const int cy = (cell_of_coord(py, half, S.inv_cell, S.nc1) + ((c / 3) % 3) - 1 + S.nc1) % S.nc1;
                const int cz = (cell_of_coord(pz, half, S.inv_cell, S.nc2) + (c / 9) - 1 + S.nc2) % S.nc2;
                const int cell = (cz * S.nc1 + cy) * S.nc0 + cx;
                const int cnt = S.cell_count[cell];
                for (int k = slot0; k < cnt; k += lanes_per) {
                    const int j = S.cell_members[cell * S.cap + k];
                    if (j == i) continue;
                    const int tj = static_cast<int>(meta[j] & 0xffu);
                    double u;
                    if (kF32) {
                        const FixPos pj = pos32[j];
                        const FixPos& A = st == 0 ? fa : fb;
                        bool hot;
                        const float uf = pair_energy_ft(s_pairs_f[ti * nt + tj], cf, s_stab, S.terms, A.q, pj.q,
                                                        dist2_fix(A, pj, hf), hot);
                        u = (hot && push_hot(&s_nhot, s_hot, j, st)) ? 0.0 : static_cast<double>(uf);
                    } else {
                        const double4 pj = pos[j];
                        Box b{{L, L, L}, {half, half, half}};
                        u = pair_energy(s_pairs[ti * nt + tj], s_coul, po.w, pj.w, dist2(b, px, py, pz, pj.x, pj.y, pj.z));
                    }
                    if (st == 0) e_new += u;
                    else e_old += u;
                }
            }
        }
        __syncthreads(); // phase tables complete (and the hot-pair queue)
        if (kF32) {
            // hot pairs in FP64 from the FP64 coordinates
            const Box b{{L, L, L}, {half, half, half}};
            const int nh = min(s_nhot, kHotCap);
            for (int h = tid; h < nh; h += kThreads) {
                const int2 e = s_hot[h];
                const double4 pj = pos[e.x];
                const int tj = static_cast<int>(meta[e.x] & 0xffu);
                const bool nw = (e.y & 1) == 0;
                const double u = pair_energy_t(s_pairs[ti * nt + tj], s_coul, po.w, pj.w,
                                               dist2(b, nw ? nx_ : po.x, nw ? ny_ : po.y, nw ? nz_ : po.z, pj.x, pj.y, pj.z),
                                               S.terms);
                if (nw) e_new += u;
                else e_old += u;
            }
        }

        // Ewald: dE = sum_k A_k (2 Re(conj(Q) dQ) + |dQ|^2) over this thread's k-vectors
        double de = 0.0;
        {
            int prev_col = -1;
            double2 exy_n = make_double2(1.0, 0.0), exy_o = make_double2(1.0, 0.0);
            const double qi = po.w;
#pragma unroll
            for (int s = 0; s < kMaxKPT; ++s) {
                const int k = k0 + s;
                if (s < kpt && k < nk) {
                    const int packed = s_kn[k];
                    const int nx = unpack_n(packed, 0), ny = unpack_n(packed, 1), nz = unpack_n(packed, 2);
                    const int col = packed & 0xffff;
                    if (col != prev_col) {
                        const double2 xn = s_phase[nx + ncut], yn = s_phase[width + ny + ncut];
                        const double2 xo = s_phase[3 * width + nx + ncut], yo = s_phase[4 * width + ny + ncut];
                        exy_n = make_double2(xn.x * yn.x - xn.y * yn.y, xn.x * yn.y + xn.y * yn.x);
                        exy_o = make_double2(xo.x * yo.x - xo.y * yo.y, xo.x * yo.y + xo.y * yo.x);
                        prev_col = col;
                    }
                    const double2 zn = s_phase[2 * width + nz + ncut], zo = s_phase[5 * width + nz + ncut];
                    const double en_re = exy_n.x * zn.x - exy_n.y * zn.y, en_im = exy_n.x * zn.y + exy_n.y * zn.x;
                    const double eo_re = exy_o.x * zo.x - exy_o.y * zo.y, eo_im = exy_o.x * zo.y + exy_o.y * zo.x;
                    const double dre = qi * (en_re - eo_re), dim = qi * (en_im - eo_im);
                    const int n2 = nx * nx + ny * ny + nz * nz;
                    const double A = (nx > 0 ? 2.0 : 1.0) * s_gk[n2];
                    de += A * (2.0 * (q[s].x * dre + q[s].y * dim) + (dre * dre + dim * dim));
                }
            }
        }

        // block reduction (fixed order) and the acceptance test on thread 0
        {
            const double a = wave_sum(e_new), b = wave_sum(e_old), c = wave_sum(de);
            if ((tid & 63) == 0) {
                s_red[0][tid >> 6] = a;
                s_red[1][tid >> 6] = b;
                s_red[2][tid >> 6] = c;
            }
        }
        __syncthreads();
        if (tid == 0) {
            double a = 0.0, b = 0.0, c = 0.0;
            for (int w = 0; w < kThreads / 64; ++w) {
                a += s_red[0][w];
                b += s_red[1][w];
                c += s_red[2][w];
            }
            // the surface term enters with the reciprocal one (Ewald::energy, energy.cpp:581-587)
            double dsurf = 0.0, mx = dip0, my = dip1, mz = dip2;
            if (surf != 0.0) {
                mx += po.w * (nx_ - po.x);
                my += po.w * (ny_ - po.y);
                mz += po.w * (nz_ - po.z);
                dsurf = surf * ((mx * mx + my * my + mz * mz) - (dip0 * dip0 + dip1 * dip1 + dip2 * dip2));
            }
            const double du = energy_change(a, b, pref * c + dsurf);
            const bool acc = metropolis(beta * du, P.accept_u);
            if (acc) {
                dip0 = mx;
                dip1 = my;
                dip2 = mz;
            }
            s_accept = acc ? 1 : 0;
            if (kF32) s_nhot = 0; // every thread has read the queue before the reduction
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
                energy += du;
                sum_du += du;
                ++accepted;
                pos[i] = make_double4(nx_, ny_, nz_, po.w);
                if (kF32) pos32[i] = fa;
                if (kCells) {
                    const int cxn = cell_of_coord(nx_, half, S.inv_cell, S.nc0);
                    const int cyn = cell_of_coord(ny_, half, S.inv_cell, S.nc1);
                    const int czn = cell_of_coord(nz_, half, S.inv_cell, S.nc2);
                    const int cnew = (czn * S.nc1 + cyn) * S.nc0 + cxn;
                    const int cold = S.cell_of[i];
                    if (cnew != cold) {
                        const int nn = S.cell_count[cnew];
                        if (nn >= S.cap) {
                            // full cell: the lists are left as they are and the chain stops
                            // after this move
                            S.error = 1;
                        } else {
                            const int nold = S.cell_count[cold];
                            for (int kk = 0; kk < nold; ++kk)
                                if (S.cell_members[cold * S.cap + kk] == i) {
                                    S.cell_members[cold * S.cap + kk] = S.cell_members[cold * S.cap + nold - 1];
                                    break;
                                }
                            S.cell_count[cold] = nold - 1;
                            S.cell_members[cnew * S.cap + nn] = i;
                            S.cell_count[cnew] = nn + 1;
                            S.cell_of[i] = cnew;
                        }
                    }
                }
            }
            if (sample_every > 0 && isfinite(energy) &&
                (move0 + static_cast<unsigned long long>(t) + 1ull) % static_cast<unsigned long long>(sample_every) == 0ull) {
                e_sum += energy;
                e_sum2 += energy * energy;
                ++e_samples;
            }
        }
        __syncthreads();
        if (s_accept) {
            // Q += dQ for this thread's k-vectors (phase tables still hold this move)
            int prev_col = -1;
            double2 exy_n = make_double2(1.0, 0.0), exy_o = make_double2(1.0, 0.0);
            const double qi = po.w;
#pragma unroll
            for (int s = 0; s < kMaxKPT; ++s) {
                const int k = k0 + s;
                if (s < kpt && k < nk) {
                    const int packed = s_kn[k];
                    const int nx = unpack_n(packed, 0), ny = unpack_n(packed, 1), nz = unpack_n(packed, 2);
                    const int col = packed & 0xffff;
                    if (col != prev_col) {
                        const double2 xn = s_phase[nx + ncut], yn = s_phase[width + ny + ncut];
                        const double2 xo = s_phase[3 * width + nx + ncut], yo = s_phase[4 * width + ny + ncut];
                        exy_n = make_double2(xn.x * yn.x - xn.y * yn.y, xn.x * yn.y + xn.y * yn.x);
                        exy_o = make_double2(xo.x * yo.x - xo.y * yo.y, xo.x * yo.y + xo.y * yo.x);
                        prev_col = col;
                    }
                    const double2 zn = s_phase[2 * width + nz + ncut], zo = s_phase[5 * width + nz + ncut];
                    const double en_re = exy_n.x * zn.x - exy_n.y * zn.y, en_im = exy_n.x * zn.y + exy_n.y * zn.x;
                    const double eo_re = exy_o.x * zo.x - exy_o.y * zo.y, eo_im = exy_o.x * zo.y + exy_o.y * zo.x;
                    q[s].x += qi * (en_re - eo_re);
                    q[s].y += qi * (en_im - eo_im);
                }
            }
        }
        if (S.error) {
            t_done = t + 1;
            break;
        }
        __syncthreads(); // phase tables and the accepted position are consumed before the next move
    }

    if (tid == 0) {
        S.moves = move0 + static_cast<unsigned long long>(t_done);
        S.accepted = accepted;
        S.energy = energy;
        S.sum_du = sum_du;
        S.dip[0] = dip0;
        S.dip[1] = dip1;
        S.dip[2] = dip2;
        S.e_samples = e_samples;
        S.e_sum = e_sum;
        S.e_sum2 = e_sum2;
        if (ladders != nullptr) ladder_barrier(*ladders, rep, states, S, iv, beta);
    }
    move0 += static_cast<unsigned long long>(t_done);
    __syncthreads(); // the interval's state and error are written before the next interval reads them
    }

#pragma unroll
    for (int s = 0; s < kMaxKPT; ++s)
        if (s < kpt && k0 + s < nk) S.q[k0 + s] = q[s];
}

template <int kMaxKPT, bool kCells, bool kF32>
void launch_advance(int grid, size_t lds, hipStream_t st, ReplicaState* s, const long long* m, TraceEntry* tr, int cap,
                    const LadderRun* lr, ReplicaMap map) {
    constexpr int kThreads = kAdvanceThreads;
    auto fn = mc_advance_kernel<kMaxKPT, kCells, kF32>;
    // dynamic LDS: what the static LDS leaves of the CU's 160 KB, at most 96 KB (set once)
    static size_t limit = 0;
    if (limit == 0) {
        hipFuncAttributes attr;
        check_hip(hipFuncGetAttributes(&attr, reinterpret_cast<const void*>(fn)), "hipFuncGetAttributes");
        limit = std::min<size_t>(96 * 1024, 160 * 1024 - attr.sharedSizeBytes);
        check_hip(hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize,
                                      static_cast<int>(limit)),
                  "hipFuncSetAttribute");
    }
    if (lds > limit) throw std::runtime_error("k-vector table too large for LDS");
    if (lr == nullptr) {
        hipLaunchKernelGGL(fn, dim3(grid), dim3(kThreads), lds, st, s, m, tr, cap, lr, map);
        return;
    }
    // ladders wait for each other: every workgroup must be resident at once
    int dev = 0, per_cu = 0;
    hipDeviceProp_t prop;
    check_hip(hipGetDevice(&dev), "hipGetDevice");
    check_hip(hipGetDeviceProperties(&prop, dev), "hipGetDeviceProperties");
    check_hip(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void*>(fn), kThreads, lds),
              "occupancy");
    if (per_cu * prop.multiProcessorCount < grid)
        throw std::runtime_error("run_ladders: the replicas cannot all be resident at once");
    void* args[] = {&s, &m, &tr, &cap, &lr, &map};
    check_hip(hipLaunchCooperativeKernel(reinterpret_cast<const void*>(fn), dim3(grid), dim3(kThreads), args,
                                         static_cast<unsigned>(lds), st),
              "mc_advance_kernel cooperative launch");
}

} // namespace

// The forms for 33 to 68 k-vectors per thread, but for FP32 without a cell list.
void launch_wide(bool cells, bool f32, int grid, size_t lds, hipStream_t st, ReplicaState* s, const long long* m,
                 TraceEntry* tr, int cap, const LadderRun* lr, const ReplicaMap& map);

} // namespace fmc
