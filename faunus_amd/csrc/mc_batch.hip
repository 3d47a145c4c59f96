// Batches of replicas advanced on the device: one workgroup advances one replica through
// many trial moves (the reference's MetropolisMonteCarlo::sweep/performMove loop,
// montecarlo.cpp:139-227, with AtomicTranslateRotate proposals, move.cpp:225-293),
// computing the nonbonded pair dU and the Ewald reciprocal dU in the same pass
// (mc_translate.hip, mc_advance.hpp; move sets: mc_general.hip, mc_rigid.hip).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <stdexcept>

#include "device_math.hpp"
#include "mc_advance.hpp"
#include "mc_batch.hpp"
#include "mc_common.hpp"
#include "mc_ladder.hpp"
#include "philox.hpp"

namespace fmc {
namespace {

// Replica exchange along each ladder (odd/even neighbour pairs by round parity):
// accept with min(1, exp((beta_a - beta_b)(U_a - U_b))), energies at T_ref; swaps the
// beta labels (ParallelTempering semantics, move.cpp:844-965, without moving data).
// With round_counter non-null (one block holding every ladder, as in a captured
// interval), the round is read from that device counter, which the block then
// advances, so that each replay of the interval takes the next round.
__global__ void ladder_swap_kernel(ReplicaState* states, const int* ladder_begin, const int* ladder_size,
                                   int* rung_slot, int nladders, unsigned long long seed, unsigned long long round,
                                   unsigned long long* counters, unsigned long long* round_counter) {
    const int l = blockIdx.x * blockDim.x + threadIdx.x;
    if (round_counter) {
        round = *round_counter;
        __syncthreads();
        if (threadIdx.x == 0) *round_counter = round + 1ull;
    }
    if (l >= nladders) return;
    swap_ladder_rungs(states, ladder_begin[l], ladder_size[l], rung_slot, l, seed, round, counters);
}

constexpr int kRdfList = 2048;

// Pair-distance histogram of one configuration (AtomRDF::_sample, analysis.cpp:1556-1600):
// types a != b: every (a, b) pair; a == b: pairs i < j.  r = |minimum-image distance|,
// bin floor(r / dr) as Equidistant2DTable::to_bin (equidistant_table.h:32-39), bins >= nbins
// dropped.  Block (x, y): one j per thread from `ids` (the particles of type b, `nb` of
// them), against the i of type a in run y of `len` particles, whose coordinates are the
// same for every lane (scalar loads).  Pairs beyond the last bin (range2: 1e-9 above its
// squared edge) stop at the rounded distance; counts go to an LDS histogram, then once
// per block to the global one.  Up to kRdfList particles, where the
// list's copy to the device takes longer than the lanes it saves, every particle has a thread
// (kList false): N = 200 37 -> 29 us a call, N = 4000 74 us against 59 with the list.  N = 20000, 240 bins of 0.1 A: 717 us with one i per block
// (every block read all positions), now 125 us.
template <bool kList>
__global__ __launch_bounds__(256) void rdf_kernel(const double4* __restrict__ pos, const uint32_t* __restrict__ meta,
                                                  int n, int ta, int tb, double L, double half, double inv_dr,
                                                  double range2, int nbins, int len, const int* __restrict__ ids, int nb,
                                                  unsigned long long* __restrict__ counts) {
    extern __shared__ unsigned int s_hist[];
    for (int b = threadIdx.x; b < nbins; b += blockDim.x) s_hist[b] = 0u;
    const int t = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x);
    int j = -1;
    if (t < nb) j = kList ? ids[t] : (static_cast<int>(meta[t] & 0xffu) == tb ? t : -1);
    const double4 pj = pos[max(j, 0)];
    const Box box{{L, L, L}, {half, half, half}};
    const double inv[3] = {1.0 / L, 1.0 / L, 1.0 / L};
    __syncthreads();
    const int ie = min(n, len * (static_cast<int>(blockIdx.y) + 1));
    for (int i = len * static_cast<int>(blockIdx.y); i < ie; ++i) {
        if (static_cast<int>(meta[i] & 0xffu) != ta) continue; // uniform over the block
        const double4 pi = pos[i];
        if (near_dist2(box, inv, pi.x, pi.y, pi.z, pj.x, pj.y, pj.z) >= range2) continue;
        if (j < 0 || (ta == tb && j <= i)) continue;
        const double dx = min_image(pi.x - pj.x, L, half);
        const double dy = min_image(pi.y - pj.y, L, half);
        const double dz = min_image(pi.z - pj.z, L, half);
        // x^2 + y^2 + z^2 rounded term by term, as the reference's norm
        const double r = sqrt(__dadd_rn(__dadd_rn(__dmul_rn(dx, dx), __dmul_rn(dy, dy)), __dmul_rn(dz, dz)));
        const double x = floor(__dmul_rn(r, inv_dr));
        if (x < static_cast<double>(nbins)) atomicAdd(&s_hist[static_cast<int>(x)], 1u);
    }
    __syncthreads();
    for (int b = threadIdx.x; b < nbins; b += blockDim.x)
        if (s_hist[b]) atomicAdd(&counts[b], static_cast<unsigned long long>(s_hist[b]));
}

} // namespace

// ==============================================================================
Batch::Batch(int precision_fp32) : fp32_(precision_fp32) {
    check_hip(hipStreamCreateWithFlags(&stream_, hipStreamNonBlocking), "hipStreamCreate");
    check_hip(hipEventCreate(&ev0_), "hipEventCreate");
    check_hip(hipEventCreate(&ev1_), "hipEventCreate");
}

SideBySide::~SideBySide() {
    for (int k = 0; k < kStreams; ++k) {
        if (streams_[k]) (void)hipStreamDestroy(streams_[k]);
        if (done_[k]) (void)hipEventDestroy(done_[k]);
    }
    if (forked_) (void)hipEventDestroy(forked_);
}

// The first `side` streams wait for all that was enqueued on `main`.
void SideBySide::fork(hipStream_t main, int side) {
    if (!forked_) check_hip(hipEventCreateWithFlags(&forked_, hipEventDisableTiming), "hipEventCreate");
    for (int k = 0; k < side; ++k) {
        if (!streams_[k]) check_hip(hipStreamCreateWithFlags(&streams_[k], hipStreamNonBlocking), "hipStreamCreate");
        if (!done_[k]) check_hip(hipEventCreateWithFlags(&done_[k], hipEventDisableTiming), "hipEventCreate");
    }
    check_hip(hipEventRecord(forked_, main), "fork streams");
    for (int k = 0; k < side; ++k) check_hip(hipStreamWaitEvent(streams_[k], forked_, 0), "fork streams");
}

// `main` waits for them; the first error, after all have been joined as far as possible.
hipError_t SideBySide::join(hipStream_t main, int side) {
    hipError_t first = hipSuccess;
    for (int k = 0; k < side; ++k) {
        hipError_t e = hipEventRecord(done_[k], streams_[k]);
        if (e == hipSuccess) e = hipStreamWaitEvent(main, done_[k], 0);
        if (first == hipSuccess) first = e;
    }
    return first;
}

Batch::~Batch() {
    if (stream_) (void)hipStreamSynchronize(stream_);
    if (graph_) (void)hipGraphExecDestroy(graph_);
    for (auto p : graph_owned_) (void)hipFree(p);
    for (auto p : owned_) (void)hipFree(p);
    (void)hipFree(d_states_);
    (void)hipFree(d_moves_);
    (void)hipFree(d_trace_);
    (void)hipFree(split_slots_);
    (void)hipFree(split_priv_);
    (void)hipFree(pipe_slots_);
    (void)hipFree(split_err_);
    (void)hipFree(d_map_);
    if (ev0_) (void)hipEventDestroy(ev0_);
    if (ev1_) (void)hipEventDestroy(ev1_);
    if (stream_) (void)hipStreamDestroy(stream_);
}


namespace {
template <class T> T* upload(const std::vector<T>& v, std::vector<void*>& owned, const char* what) {
    T* d = nullptr;
    check_hip(hipMalloc(&d, sizeof(T) * std::max<size_t>(1, v.size())), what);
    owned.push_back(d);
    if (!v.empty()) check_hip(hipMemcpy(d, v.data(), sizeof(T) * v.size(), hipMemcpyHostToDevice), what);
    return d;
}
} // namespace

// S(q) and dS/dq of the engine's Coulomb model: the Andrea spline (value and the
// derivative of its interval polynomial) or the exact function.
static void short_range_and_slope(const DevCoulomb& c, double q, double* s, double* ds) {
    if (c.splined) {
        const int n = c.nknots;
        const int lo = static_cast<int>(std::lower_bound(c.knots, c.knots + n, q) - c.knots);
        int pos = std::min(std::max(lo - 1, 0), n - 2);
        const double* k = c.coeff + 6 * pos;
        const double z = q - c.knots[pos];
        *s = ((((k[5] * z + k[4]) * z + k[3]) * z + k[2]) * z + k[1]) * z + k[0];
        *ds = (((5 * k[5] * z + 4 * k[4]) * z + 3 * k[3]) * z + 2 * k[2]) * z + k[1];
    } else if (c.scheme == kCoulEwald) {
        const double a = c.alpha * c.rc;
        *s = std::erfc(a * q);
        *ds = -2.0 * a / std::sqrt(kPi) * std::exp(-a * a * q * q);
    } else {
        const double q5 = q * q * q * q * q;
        *s = 1.0 - 1.75 * q + 5.25 * q5 - 7.0 * q5 * q + 2.5 * q5 * q * q;
        *ds = -1.75 + 26.25 * q * q * q * q - 42.0 * q5 + 17.5 * q5 * q;
    }
}

// Cubic Hermite coefficients (in the local coordinate of each interval) of S(q).
static std::vector<float4> short_range_table(const DevCoulomb& c) {
    std::vector<float4> t(static_cast<size_t>(kSTable));
    const double h = 1.0 / kSTable;
    for (int i = 0; i < kSTable; ++i) {
        double f0, d0, f1, d1;
        short_range_and_slope(c, i * h, &f0, &d0);
        short_range_and_slope(c, (i + 1) * h, &f1, &d1);
        const double c2 = 3.0 * (f1 - f0) - h * (2.0 * d0 + d1);
        const double c3 = 2.0 * (f0 - f1) + h * (d0 + d1);
        t[static_cast<size_t>(i)] = make_float4(static_cast<float>(f0), static_cast<float>(h * d0),
                                                static_cast<float>(c2), static_cast<float>(c3));
    }
    return t;
}

namespace {
// One pair energy per thread in both device forms: the FP64 one (pair_energy) and the
// FP32-pair form of the device-resident kernels (pair_energy_ft with its S(q) table, and
// the FP64 re-evaluation of hot pairs), at the same distance.
__global__ void pair_probe_kernel(const DevPair* __restrict__ pairs, const DevCoulomb* __restrict__ coul,
                                  const float4* __restrict__ stab, int nt, int terms, int ta, int tb, double qa, double qb,
                                  int n, const double* __restrict__ r2, double* __restrict__ u64,
                                  double* __restrict__ u32) {
    const int i = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x);
    if (i >= n) return;
    const DevPair& p = pairs[ta * nt + tb];
    u64[i] = pair_energy(p, *coul, qa, qb, r2[i]);
    const DevPairF pf = to_f32(p);
    const CoulF cf = coul_f32(*coul);
    bool hot;
    const float uf = pair_energy_ft(pf, cf, stab, terms, static_cast<float>(qa), static_cast<float>(qb),
                                    static_cast<float>(r2[i]), hot);
    u32[i] = hot ? pair_energy_t(p, *coul, qa, qb, r2[i], terms) : static_cast<double>(uf);
}
} // namespace

void pair_probe(Engine& e, int ta, int tb, double qa, double qb, int n, const double* r2, double* u64, double* u32) {
    const int nt = e.model().ntypes;
    if (ta < 0 || tb < 0 || ta >= nt || tb >= nt) throw std::runtime_error("pair probe: bad atom type");
    if (n < 0 || n > (1 << 24)) throw std::runtime_error("pair probe: 0 to 2^24 distances");
    if (n == 0) return;
    std::vector<void*> owned;
    try {
        const DevCoulomb& dc = e.dev_coulomb();
        const float4* stab = (dc.scheme == kCoulEwald || dc.scheme == kCoulFanourgakis)
                                 ? upload(short_range_table(dc), owned, "upload S(q) table")
                                 : nullptr;
        int terms = 0;
        for (const DevPair& p : e.dev_pairs()) {
            if (p.lj_e4 != 0.0) terms |= kTermLJ;
            if (p.wca_e4 != 0.0) terms |= kTermWCA;
            if (p.hs_s2 > 0.0) terms |= kTermHS;
        }
        const std::vector<double> x(r2, r2 + n);
        const double* d_r2 = upload(x, owned, "upload r2");
        double* d_out = upload(std::vector<double>(2 * static_cast<size_t>(n), 0.0), owned, "probe output");
        hipLaunchKernelGGL(pair_probe_kernel, dim3((n + 255) / 256), dim3(256), 0, e.stream(), e.d_pairs(), e.d_coul(),
                           stab, nt, terms, ta, tb, qa, qb, n, d_r2, d_out, d_out + n);
        check_hip(hipGetLastError(), "pair_probe_kernel");
        check_hip(hipStreamSynchronize(e.stream()), "pair probe");
        check_hip(hipMemcpy(u64, d_out, sizeof(double) * n, hipMemcpyDeviceToHost), "copy probe");
        check_hip(hipMemcpy(u32, d_out + n, sizeof(double) * n, hipMemcpyDeviceToHost), "copy probe");
    } catch (...) {
        for (void* p : owned) (void)hipFree(p);
        throw;
    }
    for (void* p : owned) (void)hipFree(p);
}

// The dipole sum q r over the engine's particles (positions as stored).
static void replica_dipole(Engine& e, double* dip) {
    const int n = e.num_particles();
    std::vector<double> xyz(3 * static_cast<size_t>(n));
    e.get_positions(xyz.data());
    const auto& q = e.host_charges();
    dip[0] = dip[1] = dip[2] = 0.0;
    for (int i = 0; i < n; ++i)
        for (int d = 0; d < 3; ++d) dip[d] += xyz[3 * static_cast<size_t>(i) + d] * q[static_cast<size_t>(i)];
}

ReplicaState make_replica_state(Engine& e, bool fp32, unsigned long long seed, int stream_id, double beta, int ladder,
                                std::vector<void*>& owned, const std::vector<MoveKindSpec>* kinds) {
    const Model& m = e.model();
    const int n = e.num_particles();
    if (!(m.box[0] == m.box[1] && m.box[1] == m.box[2])) throw std::runtime_error("device MC needs a cubic box");
    ReplicaState s{};
    s.n = n;
    s.nk = e.num_kvectors();
    s.ncut = m.ewald.present ? static_cast<int>(std::ceil(m.ewald.n_cutoff)) : 0;
    if (s.ncut * s.ncut >= kMaxGk) throw std::runtime_error("ncutoff too large for the device MC (max 32)");
    if (m.ewald.present && !m.ewald.spherical_sum) throw std::runtime_error("device MC needs spherical_sum: true");
    if (!kinds)
        for (const auto& mol : m.molecules)
            if (!mol.atomic) throw std::runtime_error("device MC handles atomic groups (single-particle translations)");
    // Hamiltonian::energy stops summing a state's terms at the first one >= maxenergy
    // (energy.cpp:1227-1241); the device kernels form dU as one difference, so a finite
    // maxenergy is left to the per-move path
    if (std::isfinite(m.maximum_allowed_energy))
        throw std::runtime_error("device MC: maxenergy is supported by the per-move path only");
    s.ntypes = m.ntypes;
    s.L = m.box[0];
    s.half = 0.5 * m.box[0];
    s.inv = 1.0 / m.box[0];
    s.rec_prefactor = m.ewald.present ? 2 * kPi * m.ewald.lB / (m.box[0] * m.box[1] * m.box[2]) : 0.0;
    s.pos = e.d_pos();
    s.meta = e.d_meta();
    s.q = e.d_q_acc();
    s.kn = e.d_kn();
    s.pairs = e.d_pairs();
    s.coul = e.d_coul();
    CellList& cl = e.cells();
    s.cells = cl.enabled ? 1 : 0;
    if (cl.enabled) {
        if (!(cl.nc[0] == cl.nc[1] && cl.nc[1] == cl.nc[2])) throw std::runtime_error("cubic cell grid expected");
        s.nc0 = cl.nc[0];
        s.nc1 = cl.nc[1];
        s.nc2 = cl.nc[2];
        s.cap = cl.cap;
        s.inv_cell = cl.inv_cell[0];
        s.cell_count = cl.count;
        s.cell_members = cl.members;
        s.cell_of = cl.cell_of;
    }
    // A_k as a function of |n|^2 for a cubic box (the n_x>0 factor 2 is applied in the kernel)
    std::vector<double> gk(static_cast<size_t>(kMaxGk), 0.0);
    if (m.ewald.present) {
        const double kb = 2 * kPi / m.box[0];
        for (int n2 = 1; n2 <= s.ncut * s.ncut; ++n2) {
            const double k2 = kb * kb * n2;
            gk[static_cast<size_t>(n2)] = std::exp(-k2 / (4 * m.ewald.alpha * m.ewald.alpha)) / k2;
        }
    }
    double* d_gk = nullptr;
    check_hip(hipMalloc(&d_gk, sizeof(double) * kMaxGk), "hipMalloc gk");
    owned.push_back(d_gk);
    check_hip(hipMemcpy(d_gk, gk.data(), sizeof(double) * kMaxGk, hipMemcpyHostToDevice), "copy gk");
    s.gk = d_gk;
    std::vector<double> dpt(static_cast<size_t>(m.ntypes));
    for (int t = 0; t < m.ntypes; ++t) dpt[static_cast<size_t>(t)] = m.atoms[static_cast<size_t>(t)].dp;
    double* d_dp = nullptr;
    check_hip(hipMalloc(&d_dp, sizeof(double) * m.ntypes), "hipMalloc dp");
    owned.push_back(d_dp);
    check_hip(hipMemcpy(d_dp, dpt.data(), sizeof(double) * m.ntypes, hipMemcpyHostToDevice), "copy dp");
    s.dp_type = d_dp;
    FixPos* d_p32 = nullptr;
    if (fp32) {
        std::vector<double> xyz(3 * static_cast<size_t>(n));
        e.get_positions(xyz.data());
        const std::vector<FixPos> p32 = fixed_positions(xyz.data(), e.host_charges(), n, s.inv);
        check_hip(hipMalloc(&d_p32, sizeof(FixPos) * n), "hipMalloc pos32");
        owned.push_back(d_p32);
        check_hip(hipMemcpy(d_p32, p32.data(), sizeof(FixPos) * n, hipMemcpyHostToDevice), "copy pos32");
    }
    s.pos32 = d_p32;
    s.parts = 1;
    s.gslots = nullptr;
    s.sample_every = 0;
    s.e_samples = 0;
    s.e_sum = s.e_sum2 = 0.0;
    s.pair_range = e.cells().enabled ? e.cell_range() : e.model().pair_range;
    // surface term (PolicyIonIon::surfaceEnergy, energy.cpp:466-482): the prefactor and
    // the dipole sum, kept up to date by the kernels
    s.surf = 0.0;
    s.dip[0] = s.dip[1] = s.dip[2] = 0.0;
    if (m.ewald.present && m.ewald.const_inf > 0.5) {
        const double V = m.box[0] * m.box[1] * m.box[2];
        s.surf = m.ewald.const_inf * 2.0 * kPi / ((2.0 * m.ewald.epss + 1.0) * V) * m.ewald.lB;
        replica_dipole(e, s.dip);
    }
    s.cell_radius = e.cell_radius();
    s.threads = 0;
    const DevCoulomb& dc = e.dev_coulomb();
    if (fp32 && (dc.scheme == kCoulEwald || dc.scheme == kCoulFanourgakis)) s.stab = upload(short_range_table(dc), owned, "upload S(q) table");
    s.terms = 0;
    for (const DevPair& p : e.dev_pairs()) {
        if (p.lj_e4 != 0.0) s.terms |= kTermLJ;
        if (p.wca_e4 != 0.0) s.terms |= kTermWCA;
        if (p.hs_s2 > 0.0) s.terms |= kTermHS;
    }
    s.seed = seed;
    s.replica_id = stream_id;
    s.ladder = ladder;
    s.beta = beta;
    if (kinds) {
        if (kinds->empty()) throw std::runtime_error("empty move set");
        const auto& gb = e.group_begin();
        const auto& gs = e.group_size();
        const auto& gm = e.group_molid();
        std::vector<MoveKindDev> kd;
        std::vector<int> kgroups;
        std::vector<int2> pbonds;
        unsigned long long cum = 0;
        int max_moved = 1;
        std::vector<int> kind_of_molid(m.molecules.size(), -1);
        for (const MoveKindSpec& k : *kinds) {
            if (k.kind < 0 || k.kind > 2) throw std::runtime_error("unknown move kind");
            if (k.molid < 0 || k.molid >= static_cast<int>(m.molecules.size())) throw std::runtime_error("move molid out of range");
            // translate+rotate keeps the mass centre by translation only: its molecule
            // type must not also be changed internally by the other kinds
            int& seen = kind_of_molid[static_cast<size_t>(k.molid)];
            if (seen >= 0 && ((seen == 1) != (k.kind == 1)))
                throw std::runtime_error("a molecule type moved by translate+rotate takes no atom or pivot moves");
            seen = k.kind;
            MoveKindDev d{};
            d.kind = k.kind;
            d.group_first = static_cast<int>(kgroups.size());
            for (size_t g = 0; g < gm.size(); ++g)
                if (gm[g] == k.molid) {
                    kgroups.push_back(static_cast<int>(g));
                    if (k.kind != 0) max_moved = std::max(max_moved, gs[g]);
                }
            d.group_count = static_cast<int>(kgroups.size()) - d.group_first;
            if (d.group_count == 0) throw std::runtime_error("move kind without groups");
            const MoleculeCfg& mol = m.molecules[static_cast<size_t>(k.molid)];
            if (k.kind == 1 && mol.atomic) throw std::runtime_error("translate+rotate needs a molecular group");
            if (k.kind == 2) {
                if (mol.atomic) throw std::runtime_error("pivot needs a molecular group");
                d.bond_first = static_cast<int>(pbonds.size());
                for (const BondCfg& b : mol.bonds) pbonds.push_back(make_int2(b.i, b.j));
                d.bond_count = static_cast<int>(pbonds.size()) - d.bond_first;
            }
            cum += k.weight;
            d.cum = cum;
            d.dp = k.dp;
            d.dprot = k.dprot;
            kd.push_back(d);
        }
        if (cum == 0 || cum > 0xffffffffull) throw std::runtime_error("move weights must sum to 1..2^32-1");
        if (max_moved > kGeneralMaxMoved) throw std::runtime_error("molecule too large for the device MC");
        std::vector<double> dpa(static_cast<size_t>(m.ntypes));
        for (int t = 0; t < m.ntypes; ++t)
            dpa[static_cast<size_t>(t)] = m.atoms[static_cast<size_t>(t)].has_dp ? m.atoms[static_cast<size_t>(t)].dp : -1.0;
        s.nkinds = static_cast<int>(kd.size());
        s.max_moved = max_moved;
        s.total_weight = cum;
        s.kinds = upload(kd, owned, "upload move kinds");
        s.kind_groups = upload(kgroups, owned, "upload kind groups");
        s.pivot_bonds = upload(pbonds, owned, "upload pivot bonds");
        s.gbegin = upload(gb, owned, "upload group begin");
        s.gsize = upload(gs, owned, "upload group size");
        s.gflags = e.d_group_flags();
        s.gcm = e.d_mass_centers();
        s.dp_atom = upload(dpa, owned, "upload atom dp");
        const bool bonded = m.bonded_term >= 0 && e.num_bonds() > 0;
        s.bond_off = bonded ? e.d_bond_offsets() : nullptr;
        s.bonds = bonded ? e.d_bonds() : nullptr;
        s.excl_off = e.d_exclusion_offsets();
        s.excl = e.d_exclusions();
        s.nmol = static_cast<int>(m.molecules.size());
        s.g2g2 = e.d_g2g_cutoffs();
        std::vector<double> mw(static_cast<size_t>(m.ntypes));
        for (int t = 0; t < m.ntypes; ++t) mw[static_cast<size_t>(t)] = m.atoms[static_cast<size_t>(t)].mw;
        s.mw = upload(mw, owned, "upload atom masses");
        set_rigid_fields(e, s, *kinds);
    }
    std::vector<double> terms(static_cast<size_t>(e.num_terms()));
    e.total_energy(terms.data());
    double u0 = 0;
    for (double v : terms) u0 += v;
    s.energy = u0;
    return s;
}

// Replicas with at most 8 k-vectors per thread run mc_translate_kernel, the others
// mc_advance_kernel: a function of the replica alone.
bool translate_route(const ReplicaState& s) { return s.nk <= 8 * advance_threads(s); }

// 512 threads where they hold the k-vectors at 8 per thread, except with a cell list of so few
// members that 256 threads take one each and so few k-vectors that 256 threads hold them at 8:
// there a smaller workgroup's barriers are cheaper (400 moves of 1000 Na/Cl, 2.9 members per cell:
// 2.52 against 2.68 ms; of 1600 ions, 4.7: 2.12 against 2.26), while 800 moves of 200 ions (7.4) take
// 4.12 against 3.59 ms and 400 of 3000 Na/Cl with K = 2900 4.04 against 2.69.
int advance_threads(const ReplicaState& s) {
    if (s.threads) return s.threads;
    if (s.nk > 8 * 512) return 256;
    if (!s.cells || s.nk > 8 * 256) return 512;
    return 54LL * s.n > 256LL * s.nc0 * s.nc1 * s.nc2 ? 512 : 256;
}

void launch_advance(const ReplicaState* h_states, int count, ReplicaState* d_states, const long long* d_moves, bool f32,
                    TraceEntry* trace, int trace_cap, hipStream_t stream, SideBySide& side, const LadderRun* ladders) {
    // workgroup size and kernel of each replica, functions of the replica alone (so that its
    // arithmetic does not depend on the others) unless its batch set one size (the tuner, or
    // Batch::finalize for more cell-list replicas than CUs); the replicas of a ladder launch with
    // cell lists take 256 threads, and the kernel for any K, when they do not agree
    std::vector<int> threads(static_cast<size_t>(count));
    std::vector<char> translate(static_cast<size_t>(count));
    bool same = true, cells = true, all = true;
    for (int r = 0; r < count; ++r) {
        const ReplicaState& s = h_states[r];
        if (s.cells != h_states[0].cells) throw std::runtime_error("replicas of one launch must agree on the cell list");
        threads[static_cast<size_t>(r)] = advance_threads(s);
        same = same && threads[static_cast<size_t>(r)] == threads[0];
        cells = cells && s.cells != 0;
    }
    if (ladders != nullptr && !same) {
        if (!cells) throw std::runtime_error("run_ladders: every replica must take the same workgroup size");
        std::fill(threads.begin(), threads.end(), 256);
    }
    if (ladders != nullptr && count > ReplicaMap::kMax)
        throw std::runtime_error("run_ladders: the replicas cannot all be resident at once");
    for (int r = 0; r < count; ++r) {
        const int kpt = (h_states[r].nk + threads[static_cast<size_t>(r)] - 1) / threads[static_cast<size_t>(r)];
        if (kpt > 68) throw std::runtime_error("too many k-vectors per replica for the device MC (max 68 per thread)");
        translate[static_cast<size_t>(r)] = kpt <= 8 ? 1 : 0;
        all = all && kpt <= 8;
    }
    if (ladders != nullptr && !all) std::fill(translate.begin(), translate.end(), 0);
    auto table_bytes = [&](const std::vector<int>& ids) {
        int nk = 0, width = 0;
        for (int r : ids) {
            nk = std::max(nk, h_states[r].nk);
            width = std::max(width, 2 * h_states[r].ncut + 1);
        }
        return sizeof(int) * static_cast<size_t>((nk + 3) & ~3) + sizeof(double2) * 6 * static_cast<size_t>(width);
    };
    for (int r = 0; r < count; ++r)
        if (table_bytes({r}) > 96 * 1024) throw std::runtime_error("k-vector table too large for LDS");
    const auto route = [&](int r) { return 2 * threads[static_cast<size_t>(r)] + translate[static_cast<size_t>(r)]; };
    side.run(launches_by_route(count, route), stream, [&](const RouteLaunch& l, hipStream_t on) {
        const size_t first = static_cast<size_t>(l.ids[0]);
        if (translate[first]) {
            launch_translate(h_states, l.ids, l.map, threads[first], d_states, d_moves, f32, trace, trace_cap, on, ladders);
            return;
        }
        int kpt = 0;
        for (int r : l.ids) kpt = std::max(kpt, (h_states[r].nk + 255) / 256);
        const int grid = static_cast<int>(l.ids.size());
        const size_t lds = table_bytes(l.ids);
        const auto go = [&](auto launch) { launch(grid, lds, on, d_states, d_moves, trace, trace_cap, ladders, l.map); };
        if (kpt > 32 && (cells || !f32))
            launch_wide(cells, f32, grid, lds, on, d_states, d_moves, trace, trace_cap, ladders, l.map);
        else if (kpt > 32) go(launch_advance<68, false, true>);
        else if (cells) go(f32 ? launch_advance<32, true, true> : launch_advance<32, true, false>);
        else go(f32 ? launch_advance<32, false, true> : launch_advance<32, false, false>);
        check_hip(hipGetLastError(), "mc_advance_kernel launch");
    });
}

int Batch::add_replica(const std::string& config_json, int n, const double* xyz, const double* charge, const int* ids,
                       int ngroups, const int* gbegin, const int* gsize, const int* gmolid, double beta,
                       unsigned long long seed, int ladder, const std::vector<MoveKindSpec>* kinds) {
    if (finalized_) throw std::runtime_error("batch already finalized");
    const int general = kinds ? 1 : 0;
    if (general_ >= 0 && general_ != general)
        throw std::runtime_error("a batch holds either translate-only replicas or replicas with move sets");
    auto e = std::make_unique<Engine>(config_json);
    e->set_particles(n, xyz, charge, ids);
    e->set_groups(ngroups, gbegin, gsize, gmolid, nullptr);
    e->set_cell_divisions(cell_divisions_);
    e->set_cell_capacity(cell_capacity_);
    e->init();
    if (!general && e->cell_list_enabled() && e->cell_radius() != 1)
        throw std::runtime_error("the finer cell grid is walked by the general move-set kernel only");
    ReplicaState s = make_replica_state(*e, fp32_ != 0, seed, static_cast<int>(engines_.size()), beta, ladder, owned_,
                                        kinds);
    general_ = general;
    h_states_.push_back(s);
    kinds_.push_back(kinds ? *kinds : std::vector<MoveKindSpec>());
    engines_.push_back(std::move(e));
    return s.replica_id;
}

void Batch::set_cell_capacity(int cap) {
    if (cap < 0) throw std::runtime_error("cell capacity must be >= 0");
    cell_capacity_ = cap;
}

void Batch::set_cell_divisions(int d) {
    if (d < 1 || d > 2) throw std::runtime_error("cell divisions: 1 or 2");
    if (!engines_.empty()) throw std::runtime_error("set the cell divisions before adding replicas");
    cell_divisions_ = d;
}

int Batch::threads_for(int r) const {
    if (threads_override_) return threads_override_;
    const ReplicaState& s = h_states_[static_cast<size_t>(r)];
    (void)s;
    return 256;
}

void Batch::finalize() {
    if (engines_.empty()) throw std::runtime_error("empty batch");
    const int threads = threads_for(0);
    for (int r = 0; r < size(); ++r) {
        if (threads_for(r) != threads) throw std::runtime_error("replicas of one batch must share the workgroup size");
        ReplicaState& s = h_states_[static_cast<size_t>(r)];
        s.kpt = (s.nk + threads - 1) / threads;
        if (s.kpt > 68) throw std::runtime_error("too many k-vectors per replica for the device MC (max 68 per thread)");
        if (s.cells != h_states_[0].cells) throw std::runtime_error("replicas must agree on the cell list");
    }
    // More replicas with a cell list than CUs: 256 threads for those whose k-vectors they hold at
    // 8 per thread.  Two such workgroups share a CU (of 512 threads one fills it), so up to two
    // per CU run at once and as one free-running launch; one size for all of the batch's launches,
    // which must agree bit for bit.  200 moves of 512 x 200 ions: FP64
    // 1.94 -> 1.30 ms, FP32 1.67 -> 1.02.
    int dev = 0, cus = 0;
    check_hip(hipGetDevice(&dev), "hipGetDevice");
    check_hip(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev), "hipDeviceGetAttribute");
    if (general_ == 0 && size() > cus)
        for (ReplicaState& s : h_states_)
            if (s.cells && s.nk <= 8 * 256) s.threads = 256;
    check_hip(hipMalloc(&d_states_, sizeof(ReplicaState) * size()), "hipMalloc states");
    check_hip(hipMemcpy(d_states_, h_states_.data(), sizeof(ReplicaState) * size(), hipMemcpyHostToDevice), "copy states");
    check_hip(hipMalloc(&d_moves_, sizeof(long long) * size()), "hipMalloc moves");
    finalized_ = true;
}

void Batch::run(const std::vector<long long>& moves, bool trace, int trace_cap) {
    if (!finalized_) finalize();
    if (static_cast<int>(moves.size()) != size()) throw std::runtime_error("run: one move count per replica");
    check_hip(hipMemcpyAsync(d_moves_, moves.data(), sizeof(long long) * size(), hipMemcpyHostToDevice, stream_), "copy moves");
    if (trace) {
        if (trace_cap > trace_cap_) {
            (void)hipFree(d_trace_);
            check_hip(hipMalloc(&d_trace_, sizeof(TraceEntry) * static_cast<size_t>(trace_cap) * size()), "hipMalloc trace");
            trace_cap_ = trace_cap;
        }
    }
    if (threads_for(0) != 256) throw std::runtime_error("unsupported workgroup size");
    TraceEntry* tr = trace ? d_trace_ : nullptr;
    const int cap = trace ? trace_cap : 0;
    time_begin();
    if (general_ == 1) {
        // one workgroup per replica, also for replicas that earlier ran split
        std::vector<ReplicaState> one(h_states_);
        for (auto& s : one) s.parts = 1;
        launch_general(one.data(), size(), d_states_, d_moves_, fp32_ != 0, tr, cap, stream_, side_);
    }
    else launch_advance(h_states_.data(), size(), d_states_, d_moves_, fp32_ != 0, tr, cap, stream_, side_);
    time_end();
}

void Batch::sample_energy(long long every) {
    if (every < 0) throw std::runtime_error("sample_energy: interval >= 0");
    if (!finalized_) finalize();
    check_hip(hipStreamSynchronize(stream_), "batch sync");
    std::vector<ReplicaState> cur(static_cast<size_t>(size()));
    check_hip(hipMemcpy(cur.data(), d_states_, sizeof(ReplicaState) * size(), hipMemcpyDeviceToHost), "copy states");
    for (int r = 0; r < size(); ++r) {
        for (ReplicaState* s : {&cur[static_cast<size_t>(r)], &h_states_[static_cast<size_t>(r)]}) {
            s->sample_every = every;
            s->e_samples = 0;
            s->e_sum = s->e_sum2 = 0.0;
        }
    }
    check_hip(hipMemcpy(d_states_, cur.data(), sizeof(ReplicaState) * size(), hipMemcpyHostToDevice), "copy states");
}

void Batch::rdf(int r, int type_a, int type_b, double dr, int nbins, unsigned long long* counts) {
    if (r < 0 || r >= size()) throw std::runtime_error("replica index out of range");
    if (!(dr > 0.0)) throw std::runtime_error("rdf: dr must be positive");
    if (nbins < 1 || nbins > 8192) throw std::runtime_error("rdf: 1 to 8192 bins");
    const ReplicaState& h = h_states_[static_cast<size_t>(r)];
    if (type_a < 0 || type_b < 0 || type_a >= h.ntypes || type_b >= h.ntypes) throw std::runtime_error("rdf: bad atom type");
    if (!finalized_) finalize();
    // the particles of type b, then the counts, in one allocation
    std::vector<int> ids;
    const auto& types = engines_[static_cast<size_t>(r)]->host_types();
    for (int j = 0; j < h.n; ++j)
        if (types[static_cast<size_t>(j)] == type_b) ids.push_back(j);
    if (ids.empty()) return;
    if (h.n <= kRdfList) ids.clear();
    const int nb = ids.empty() ? h.n : static_cast<int>(ids.size());
    const size_t head = (sizeof(int) * ids.size() + 7) & ~static_cast<size_t>(7);
    unsigned char* d = nullptr;
    check_hip(hipMalloc(&d, head + sizeof(unsigned long long) * static_cast<size_t>(nbins)), "hipMalloc rdf");
    unsigned long long* d_counts = reinterpret_cast<unsigned long long*>(d + head);
    std::vector<unsigned long long> part(static_cast<size_t>(nbins));
    try {
        if (!ids.empty())
            check_hip(hipMemcpyAsync(d, ids.data(), sizeof(int) * ids.size(), hipMemcpyHostToDevice, stream_), "copy rdf ids");
        check_hip(hipMemsetAsync(d_counts, 0, sizeof(unsigned long long) * static_cast<size_t>(nbins), stream_),
                  "clear rdf");
        const int tiles = (nb + 255) / 256;
        // about 2048 blocks, each with at least 32 i for its histogram's clear and flush (fewer,
        // down to 4, where that leaves CUs without a block)
        const int least = std::max(4, std::min(32, static_cast<int>(static_cast<long long>(h.n) * tiles / 256)));
        const int runs = std::max(1, std::min((h.n + least - 1) / least, 2048 / tiles));
        const int len = (h.n + runs - 1) / runs;
        const double edge = static_cast<double>(nbins) * dr;
        hipLaunchKernelGGL(ids.empty() ? rdf_kernel<false> : rdf_kernel<true>, dim3(static_cast<unsigned>(tiles), static_cast<unsigned>((h.n + len - 1) / len)),
                           dim3(256), sizeof(unsigned int) * static_cast<size_t>(nbins), stream_, h.pos, h.meta, h.n, type_a,
                           type_b, h.L, h.half, 1.0 / dr, edge * edge * (1.0 + 1e-9), nbins, len,
                           reinterpret_cast<const int*>(d), nb, d_counts);
        check_hip(hipGetLastError(), "rdf_kernel launch");
        check_hip(hipMemcpyAsync(part.data(), d_counts, sizeof(unsigned long long) * static_cast<size_t>(nbins),
                                 hipMemcpyDeviceToHost, stream_),
                  "copy rdf");
        check_hip(hipStreamSynchronize(stream_), "rdf sync");
    } catch (...) {
        (void)hipStreamSynchronize(stream_);
        (void)hipFree(d);
        throw;
    }
    check_hip(hipFree(d), "hipFree rdf");
    for (int b = 0; b < nbins; ++b) counts[b] += part[static_cast<size_t>(b)];
}

void Batch::time_begin() {
    if (timing_) check_hip(hipEventRecord(ev0_, stream_), "event");
}

void Batch::time_end() {
    if (!timing_) return;
    check_hip(hipEventRecord(ev1_, stream_), "event");
    ev_pending_ = true;
}

// Waits for the batch's stream; the duration of the last timed launch is read once.
void Batch::sync() {
    check_hip(hipStreamSynchronize(stream_), "batch sync");
    if (ev_pending_) {
        float ms = 0;
        ev_pending_ = false;
        check_hip(hipEventElapsedTime(&ms, ev0_, ev1_), "event elapsed");
        last_ms_ = ms;
    }
}

void Batch::swap_ladders(unsigned long long seed, unsigned long long round) {
    // ladders: replicas with equal ladder id, ordered by decreasing beta at creation
    if (!finalized_) finalize();
    std::vector<int> lb, ls, slots;
    std::vector<int> ids;
    for (auto& s : h_states_) ids.push_back(s.ladder);
    std::vector<int> uniq = ids;
    std::sort(uniq.begin(), uniq.end());
    uniq.erase(std::unique(uniq.begin(), uniq.end()), uniq.end());
    sync();
    std::vector<ReplicaState> cur(static_cast<size_t>(size()));
    check_hip(hipMemcpy(cur.data(), d_states_, sizeof(ReplicaState) * size(), hipMemcpyDeviceToHost), "copy states");
    for (int lid : uniq) {
        if (lid < 0) continue;
        std::vector<int> members;
        for (int r = 0; r < size(); ++r)
            if (cur[static_cast<size_t>(r)].ladder == lid) members.push_back(r);
        std::sort(members.begin(), members.end(), [&](int a, int b) { return cur[static_cast<size_t>(a)].beta > cur[static_cast<size_t>(b)].beta; });
        lb.push_back(static_cast<int>(slots.size()));
        ls.push_back(static_cast<int>(members.size()));
        slots.insert(slots.end(), members.begin(), members.end());
    }
    if (lb.empty()) return;
    int *d_lb = nullptr, *d_ls = nullptr, *d_slots = nullptr;
    unsigned long long* d_cnt = nullptr;
    check_hip(hipMalloc(&d_lb, sizeof(int) * lb.size()), "hipMalloc");
    check_hip(hipMalloc(&d_ls, sizeof(int) * ls.size()), "hipMalloc");
    check_hip(hipMalloc(&d_slots, sizeof(int) * slots.size()), "hipMalloc");
    check_hip(hipMalloc(&d_cnt, sizeof(unsigned long long) * 2), "hipMalloc");
    check_hip(hipMemcpy(d_lb, lb.data(), sizeof(int) * lb.size(), hipMemcpyHostToDevice), "copy");
    check_hip(hipMemcpy(d_ls, ls.data(), sizeof(int) * ls.size(), hipMemcpyHostToDevice), "copy");
    check_hip(hipMemcpy(d_slots, slots.data(), sizeof(int) * slots.size(), hipMemcpyHostToDevice), "copy");
    check_hip(hipMemset(d_cnt, 0, sizeof(unsigned long long) * 2), "memset");
    const int nl = static_cast<int>(lb.size());
    hipLaunchKernelGGL(ladder_swap_kernel, dim3((nl + 63) / 64), dim3(64), 0, stream_, d_states_, d_lb, d_ls, d_slots, nl,
                       seed, round, d_cnt, static_cast<unsigned long long*>(nullptr));
    check_hip(hipGetLastError(), "ladder_swap_kernel");
    unsigned long long cnt[2] = {0, 0};
    check_hip(hipMemcpyAsync(cnt, d_cnt, sizeof(cnt), hipMemcpyDeviceToHost, stream_), "copy");
    check_hip(hipStreamSynchronize(stream_), "sync");
    swaps_att_ += static_cast<long long>(cnt[0]);
    swaps_acc_ += static_cast<long long>(cnt[1]);
    (void)hipFree(d_lb);
    (void)hipFree(d_ls);
    (void)hipFree(d_slots);
    (void)hipFree(d_cnt);
}

void Batch::get_replica_state(int r, double* xyz, double* mass_center, unsigned long long* moves,
                              unsigned long long* accepted) {
    const ReplicaState s = state(r);
    positions(r, xyz);
    Engine& e = *engines_[static_cast<size_t>(r)];
    if (mass_center) {
        const size_t ng = e.group_begin().size();
        check_hip(hipMemcpy(mass_center, e.d_mass_centers(), sizeof(double) * 3 * ng, hipMemcpyDeviceToHost),
                  "copy mass centres");
    }
    if (moves) *moves = s.moves;
    if (accepted) *accepted = s.accepted;
}

void Batch::set_replica_state(int r, const double* xyz, const double* mass_center, unsigned long long moves,
                              unsigned long long accepted) {
    ReplicaState cur = state(r); // finalizes and waits for the stream
    Engine& e = *engines_[static_cast<size_t>(r)];
    e.reset_positions(xyz, mass_center);
    const CellList& cl = e.cells();
    ReplicaState& h = h_states_[static_cast<size_t>(r)];
    for (ReplicaState* s : {&cur, &h}) {
        if (s->cells != (cl.enabled ? 1 : 0)) throw std::runtime_error("set_replica_state: cell list changed kind");
        if (cl.enabled) {
            s->nc0 = cl.nc[0];
            s->nc1 = cl.nc[1];
            s->nc2 = cl.nc[2];
            s->inv_cell = cl.inv_cell[0];
            s->cell_radius = cl.radius;
            s->cap = cl.cap;
            s->cell_count = cl.count;
            s->cell_members = cl.members;
            s->cell_of = cl.cell_of;
        }
    }
    const auto& kinds = kinds_[static_cast<size_t>(r)];
    if (!kinds.empty()) {
        set_rigid_fields(e, cur, kinds);
        set_rigid_fields(e, h, kinds);
    }
    if (cur.surf != 0.0) {
        replica_dipole(e, cur.dip);
        for (int d = 0; d < 3; ++d) h.dip[d] = cur.dip[d];
    }
    if (cur.pos32) {
        const int n = e.num_particles();
        std::vector<double> now(3 * static_cast<size_t>(n));
        e.get_positions(now.data());
        const std::vector<FixPos> p32 = fixed_positions(now.data(), e.host_charges(), n, cur.inv);
        check_hip(hipMemcpy(cur.pos32, p32.data(), sizeof(FixPos) * n, hipMemcpyHostToDevice), "copy pos32");
    }
    std::vector<double> terms(static_cast<size_t>(e.num_terms()));
    e.total_energy(terms.data());
    double u = 0.0;
    for (double v : terms) u += v;
    cur.energy = u;
    cur.moves = moves;
    cur.accepted = accepted;
    cur.sum_du = 0.0;
    cur.error = 0;
    check_hip(hipMemcpy(d_states_ + r, &cur, sizeof(ReplicaState), hipMemcpyHostToDevice), "copy state");
}

// One replica-exchange interval as a HIP graph: the persistent launch that advances
// replica r by moves[r] moves and one odd/even round of neighbour swaps on every ladder
// (ParallelTempering, move.cpp:844-965), the round taken from a device counter so that
// replays alternate the pairings.  Ladders, their rung order and the counters live on
// the device from here on.
void Batch::capture_interval(const std::vector<long long>& moves, unsigned long long seed, unsigned long long round0) {
    if (!finalized_) finalize();
    if (static_cast<int>(moves.size()) != size()) throw std::runtime_error("capture_interval: one move count per replica");
    for (const auto& s : h_states_)
        if (s.parts > 1) throw std::runtime_error("capture_interval: replicas shared by several workgroups are not captured");
    sync();
    // ladders: replicas with equal ladder id >= 0, rungs ordered by decreasing beta
    std::vector<ReplicaState> cur(static_cast<size_t>(size()));
    check_hip(hipMemcpy(cur.data(), d_states_, sizeof(ReplicaState) * size(), hipMemcpyDeviceToHost), "copy states");
    std::vector<int> ids;
    for (const auto& s : cur) ids.push_back(s.ladder);
    std::sort(ids.begin(), ids.end());
    ids.erase(std::unique(ids.begin(), ids.end()), ids.end());
    std::vector<int> lb, ls, slots;
    for (int lid : ids) {
        if (lid < 0) continue;
        std::vector<int> members;
        for (int r = 0; r < size(); ++r)
            if (cur[static_cast<size_t>(r)].ladder == lid) members.push_back(r);
        std::sort(members.begin(), members.end(),
                  [&](int a, int b) { return cur[static_cast<size_t>(a)].beta > cur[static_cast<size_t>(b)].beta; });
        lb.push_back(static_cast<int>(slots.size()));
        ls.push_back(static_cast<int>(members.size()));
        slots.insert(slots.end(), members.begin(), members.end());
    }
    const int nl = static_cast<int>(lb.size());
    if (nl > 1024) throw std::runtime_error("capture_interval: at most 1024 ladders");
    if (graph_) {
        (void)hipGraphExecDestroy(graph_);
        graph_ = nullptr;
    }
    for (void* p : graph_owned_) (void)hipFree(p);
    graph_owned_.clear();
    auto dev_copy = [&](const std::vector<int>& v) {
        int* d = nullptr;
        check_hip(hipMalloc(&d, sizeof(int) * std::max<size_t>(1, v.size())), "hipMalloc ladders");
        graph_owned_.push_back(d);
        if (!v.empty()) check_hip(hipMemcpy(d, v.data(), sizeof(int) * v.size(), hipMemcpyHostToDevice), "copy ladders");
        return d;
    };
    int* d_lb = dev_copy(lb);
    int* d_ls = dev_copy(ls);
    int* d_rung = dev_copy(slots);
    unsigned long long* d_cnt = nullptr;
    check_hip(hipMalloc(&d_cnt, sizeof(unsigned long long) * 3), "hipMalloc swap counters");
    graph_owned_.push_back(d_cnt);
    const unsigned long long init[3] = {0ull, 0ull, round0};
    check_hip(hipMemcpy(d_cnt, init, sizeof(init), hipMemcpyHostToDevice), "copy swap counters");
    graph_counters_ = d_cnt;
    check_hip(hipMemcpy(d_moves_, moves.data(), sizeof(long long) * size(), hipMemcpyHostToDevice), "copy moves");
    // one launch outside the capture sets the kernels' attributes (not a stream operation)
    const std::vector<long long> zero(static_cast<size_t>(size()), 0);
    check_hip(hipMemcpy(d_moves_, zero.data(), sizeof(long long) * size(), hipMemcpyHostToDevice), "copy moves");
    if (general_ == 1) launch_general(h_states_.data(), size(), d_states_, d_moves_, fp32_ != 0, nullptr, 0, stream_, side_);
    else launch_advance(h_states_.data(), size(), d_states_, d_moves_, fp32_ != 0, nullptr, 0, stream_, side_);
    check_hip(hipStreamSynchronize(stream_), "attribute run");
    check_hip(hipMemcpy(d_moves_, moves.data(), sizeof(long long) * size(), hipMemcpyHostToDevice), "copy moves");
    hipGraph_t g = nullptr;
    check_hip(hipStreamBeginCapture(stream_, hipStreamCaptureModeThreadLocal), "hipStreamBeginCapture");
    try {
        if (general_ == 1) launch_general(h_states_.data(), size(), d_states_, d_moves_, fp32_ != 0, nullptr, 0, stream_, side_);
        else launch_advance(h_states_.data(), size(), d_states_, d_moves_, fp32_ != 0, nullptr, 0, stream_, side_);
        if (nl > 0) {
            hipLaunchKernelGGL(ladder_swap_kernel, dim3(1), dim3(((nl + 63) / 64) * 64), 0, stream_, d_states_, d_lb, d_ls,
                               d_rung, nl, seed, 0ull, d_cnt, d_cnt + 2);
            check_hip(hipGetLastError(), "ladder_swap_kernel");
        }
    } catch (...) {
        (void)hipStreamEndCapture(stream_, &g);
        if (g) (void)hipGraphDestroy(g);
        throw;
    }
    check_hip(hipStreamEndCapture(stream_, &g), "hipStreamEndCapture");
    const hipError_t ie = hipGraphInstantiate(&graph_, g, nullptr, nullptr, 0);
    (void)hipGraphDestroy(g);
    check_hip(ie, "hipGraphInstantiate");
}

// Free-running ladders: intervals[r] swap intervals of moves[r] moves per replica in one
// cooperative launch of the translate-only kernel.  After each interval the replicas of a
// ladder meet at a barrier in HBM and the last to arrive runs that ladder's round of swaps
// (round0 + interval, the same rule and deviates as the captured interval), so a ladder
// waits only for its own rungs: ladders of different sizes and interval counts share the
// device without a device-wide barrier per interval.  The rungs of a ladder share its
// interval count; replicas outside ladders just run their intervals.
void Batch::run_ladders(const std::vector<long long>& moves, const std::vector<int>& intervals, unsigned long long seed,
                        unsigned long long round0) {
    if (!finalized_) finalize();
    const int n = size();
    if (static_cast<int>(moves.size()) != n || static_cast<int>(intervals.size()) != n)
        throw std::runtime_error("run_ladders: one move count and one interval count per replica");
    if (general_ == 1) throw std::runtime_error("run_ladders: translate-only replicas");
    for (int r = 0; r < n; ++r) {
        if (intervals[static_cast<size_t>(r)] < 0) throw std::runtime_error("run_ladders: interval counts >= 0");
        if (h_states_[static_cast<size_t>(r)].parts > 1)
            throw std::runtime_error("run_ladders: replicas shared by several workgroups");
    }
    sync();
    std::vector<ReplicaState> cur(static_cast<size_t>(n));
    check_hip(hipMemcpy(cur.data(), d_states_, sizeof(ReplicaState) * n, hipMemcpyDeviceToHost), "copy states");
    // ladders as in capture_interval: ids >= 0 in increasing order, rungs by decreasing beta
    std::vector<int> ids;
    for (const auto& s : cur) ids.push_back(s.ladder);
    std::sort(ids.begin(), ids.end());
    ids.erase(std::unique(ids.begin(), ids.end()), ids.end());
    std::vector<int> lb, ls, slots, ladder_of(static_cast<size_t>(n), -1);
    for (int lid : ids) {
        if (lid < 0) continue;
        std::vector<int> members;
        for (int r = 0; r < n; ++r)
            if (cur[static_cast<size_t>(r)].ladder == lid) members.push_back(r);
        std::sort(members.begin(), members.end(),
                  [&](int a, int b) { return cur[static_cast<size_t>(a)].beta > cur[static_cast<size_t>(b)].beta; });
        for (int r : members) {
            if (intervals[static_cast<size_t>(r)] != intervals[static_cast<size_t>(members[0])])
                throw std::runtime_error("run_ladders: the rungs of a ladder must share the interval count");
            ladder_of[static_cast<size_t>(r)] = static_cast<int>(lb.size());
        }
        lb.push_back(static_cast<int>(slots.size()));
        ls.push_back(static_cast<int>(members.size()));
        slots.insert(slots.end(), members.begin(), members.end());
    }
    const size_t nl = lb.size();
    // one allocation: counters (2 x u64), then intervals, ladder_of, begin, size, rung_slot,
    // arrive, gen (ints); arrive and gen start at zero
    std::vector<int> words;
    words.insert(words.end(), intervals.begin(), intervals.end());
    words.insert(words.end(), ladder_of.begin(), ladder_of.end());
    words.insert(words.end(), lb.begin(), lb.end());
    words.insert(words.end(), ls.begin(), ls.end());
    words.insert(words.end(), slots.begin(), slots.end());
    words.insert(words.end(), 2 * nl, 0);
    // the descriptor first, then the counters (2 x u64), then the words
    const size_t head = (sizeof(LadderRun) + 15) & ~static_cast<size_t>(15);
    const size_t bytes = head + 16 + sizeof(int) * words.size();
    std::vector<unsigned char> host(bytes, 0);
    unsigned char* d = nullptr;
    check_hip(hipMalloc(&d, bytes), "hipMalloc ladders");
    try {
        int* w = reinterpret_cast<int*>(d + head + 16);
        LadderRun lr{};
        lr.intervals = w;
        lr.ladder_of = w + n;
        lr.begin = w + 2 * n;
        lr.size = w + 2 * n + nl;
        lr.rung_slot = w + 2 * n + 2 * nl;
        lr.arrive = reinterpret_cast<unsigned*>(w + 2 * n + 2 * nl + slots.size());
        lr.gen = lr.arrive + nl;
        lr.counters = reinterpret_cast<unsigned long long*>(d + head);
        lr.seed = seed;
        lr.round0 = round0;
        lr.spin_limit = 1LL << 26;
        std::memcpy(host.data(), &lr, sizeof(lr));
        std::memcpy(host.data() + head + 16, words.data(), sizeof(int) * words.size());
        check_hip(hipMemcpy(d_moves_, moves.data(), sizeof(long long) * n, hipMemcpyHostToDevice), "copy moves");
        check_hip(hipMemcpy(d, host.data(), bytes, hipMemcpyHostToDevice), "copy ladders");
        time_begin();
        launch_advance(h_states_.data(), n, d_states_, d_moves_, fp32_ != 0, nullptr, 0, stream_, side_,
                       reinterpret_cast<const LadderRun*>(d));
        time_end();
        unsigned long long cnt[2] = {0, 0};
        check_hip(hipMemcpyAsync(cnt, d + head, sizeof(cnt), hipMemcpyDeviceToHost, stream_), "copy swap counters");
        sync();
        swaps_att_ += static_cast<long long>(cnt[0]);
        swaps_acc_ += static_cast<long long>(cnt[1]);
    } catch (...) {
        (void)hipStreamSynchronize(stream_);
        (void)hipFree(d);
        throw;
    }
    check_hip(hipFree(d), "hipFree ladders");
}

void Batch::replay(int count) {
    if (!graph_) throw std::runtime_error("replay: no interval captured");
    if (count < 0) throw std::runtime_error("replay: count >= 0");
    time_begin();
    for (int i = 0; i < count; ++i) check_hip(hipGraphLaunch(graph_, stream_), "hipGraphLaunch");
    time_end();
}

// Tile autotuner: times each candidate launch shape of this batch on a short run and
// keeps the fastest for the whole batch (one shape per batch keeps every replica in one
// persistent launch).  Translate-only replicas: workgroups of 256 or 512 threads (K/256
// or K/512 k-vectors per thread; 512 holds at most 8 per thread, so K <= 4096).
// Move-set replicas with a cell list: cells of at least the pair range (27-cell stencils)
// or half of it (125 smaller cells); replicas on mc_rigid_kernel do not walk them, so for a
// batch of these the candidates time the same kernel and either choice is as good.  Every candidate runs `trial` moves per replica from
// checkpoints that are restored afterwards, so the chains continue from their states
// before tuning (Q(k) and the running energy rebuilt from the positions).
std::vector<TuneCandidate> Batch::autotune(long long trial) {
    if (trial < 1) throw std::runtime_error("autotune: trial moves >= 1");
    if (!finalized_) finalize();
    for (const auto& s : h_states_)
        if (s.parts > 1) throw std::runtime_error("autotune: replicas shared by several workgroups");
    sync();
    struct Checkpoint {
        std::vector<double> xyz, cm;
        unsigned long long moves = 0, accepted = 0;
    };
    std::vector<Checkpoint> ck(static_cast<size_t>(size()));
    for (int r = 0; r < size(); ++r) {
        Checkpoint& c = ck[static_cast<size_t>(r)];
        c.xyz.resize(3 * static_cast<size_t>(engines_[static_cast<size_t>(r)]->num_particles()));
        c.cm.resize(3 * engines_[static_cast<size_t>(r)]->group_begin().size());
        get_replica_state(r, c.xyz.data(), c.cm.data(), &c.moves, &c.accepted);
    }
    std::vector<int> cands;
    if (general_ == 1) {
        bool cells = false;
        for (const auto& s : h_states_) cells = cells || s.cells;
        if (!cells) return {};
        cands = {1, 2};
    } else {
        cands = {256};
        bool fits512 = true;
        for (const auto& s : h_states_) fits512 = fits512 && (s.nk + 511) / 512 <= 8;
        if (fits512) cands.push_back(512);
    }
    auto apply = [&](int c) {
        for (int r = 0; r < size(); ++r) {
            if (general_ == 1) engines_[static_cast<size_t>(r)]->regrid(c);
            else h_states_[static_cast<size_t>(r)].threads = c;
        }
    };
    auto restore = [&]() {
        for (int r = 0; r < size(); ++r) {
            const Checkpoint& c = ck[static_cast<size_t>(r)];
            set_replica_state(r, c.xyz.data(), c.cm.data(), c.moves, c.accepted);
        }
    };
    const bool timing = timing_;
    timing_ = true;
    std::vector<TuneCandidate> out;
    try {
        for (int c : cands) {
            apply(c);
            if (general_ == 1) restore(); // the new grid
            run(std::vector<long long>(static_cast<size_t>(size()), trial), false, 0);
            sync();
            out.push_back(TuneCandidate{c, last_ms_ * 1e3 / (static_cast<double>(trial) * size())});
            restore();
        }
    } catch (...) {
        timing_ = timing;
        throw;
    }
    timing_ = timing;
    const auto best = std::min_element(out.begin(), out.end(),
                                       [](const TuneCandidate& a, const TuneCandidate& b) { return a.us_per_move < b.us_per_move; });
    apply(best->value);
    restore();
    tuned_ = best->value;
    return out;
}

void Batch::swap_counts(long long* attempted, long long* accepted) {
    sync();
    long long a = swaps_att_, b = swaps_acc_;
    if (graph_counters_) {
        unsigned long long c[2] = {0, 0};
        check_hip(hipMemcpy(c, graph_counters_, sizeof(c), hipMemcpyDeviceToHost), "copy swap counters");
        a += static_cast<long long>(c[0]);
        b += static_cast<long long>(c[1]);
    }
    *attempted = a;
    *accepted = b;
}

int Batch::kernel_of(int r) {
    if (r < 0 || r >= size()) throw std::runtime_error("replica index out of range");
    if (!finalized_) finalize(); // which may choose the workgroup size
    ReplicaState s = h_states_[static_cast<size_t>(r)];
    s.parts = 1; // as in run()
    if (general_ != 1) return translate_route(s) ? 0 : 1;
    return rigid_route(s, fp32_ != 0) ? 4 : (s.cells ? 3 : 2);
}

ReplicaState Batch::state(int r) {
    if (r < 0 || r >= size()) throw std::runtime_error("replica index out of range");
    if (!finalized_) finalize();
    sync();
    ReplicaState s;
    check_hip(hipMemcpy(&s, d_states_ + r, sizeof(ReplicaState), hipMemcpyDeviceToHost), "copy state");
    return s;
}

void Batch::positions(int r, double* xyz) {
    if (r < 0 || r >= size()) throw std::runtime_error("replica index out of range");
    sync();
    Engine& e = *engines_[static_cast<size_t>(r)];
    e.refresh_host_positions();
    e.get_positions(xyz);
}

std::vector<TraceEntry> Batch::trace(int r, int count) {
    if (r < 0 || r >= size() || count < 0) throw std::runtime_error("trace: replica index or count out of range");
    sync();
    std::vector<TraceEntry> t(static_cast<size_t>(count));
    if (!d_trace_ || count > trace_cap_) throw std::runtime_error("trace not recorded");
    check_hip(hipMemcpy(t.data(), d_trace_ + static_cast<size_t>(r) * trace_cap_, sizeof(TraceEntry) * count,
                        hipMemcpyDeviceToHost), "copy trace");
    return t;
}

} // namespace fmc
