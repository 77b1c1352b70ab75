// The launch behind the pair kernel: workgroups of terms (exceptions
// nonbonded.rs:995-1036, harmonic bonds and angles) first, then workgroups that
// add the slot-ordered pair sums to the atoms.
//
// Terms: the tile's atoms are staged in LDS once, each wave evaluates terms of
// one kind (a wave that mixes them runs the kinds one after another), the forces
// are summed per atom in LDS and leave with one add per atom component.  Bound:
// latency (a chain of two loads, an FP64 erf or acos, two barriers): 4.8 us for
// 23,550 atoms of water, 23 for 300,000.  As two launches, a molecule's terms on eight
// lanes that ran the kinds one after another, they took 13 us at 23,550 atoms and the gap
// between them, 11 us of a step.
#include <algorithm>
#include <climits>

#include "fold.h"
#include "terms.h"

namespace ommhip {

namespace {

__device__ __forceinline__ void add_raw(long long* p, long long v) {
    atomicAdd(reinterpret_cast<unsigned long long*>(p), (unsigned long long)v);
}
__device__ __forceinline__ void add_raw(double* p, double v) { unsafeAtomicAdd(p, v); }

// An atom's sum over a tile's terms in LDS.  Mixed form: each value is cut into
// multiples of 2^20 kJ/mol/nm (hardly ever any), steps of the accumulator and
// fractions at 2^-20 of a step, summed as integers (at most 3 x TERM_THREADS of
// each: below 2^53, 2^62 and 2^31).  So the atom's force is rounded and checked once,
// not term by term, and the order of the adds does not matter.
template <class A>
struct LdsForce;
template <>
struct LdsForce<long long> {
    long long large[3][TERM_THREADS], steps[3][TERM_THREADS];
    int parts[3][TERM_THREADS];
    static __device__ __forceinline__ void add_to(long long* p, long long v) {
        atomicAdd(reinterpret_cast<unsigned long long*>(p), (unsigned long long)v);
    }
    __device__ __forceinline__ void clear(int c, int i) {
        large[c][i] = steps[c][i] = 0;
        parts[c][i] = 0;
    }
    __device__ __forceinline__ void add(int c, int i, double v, unsigned* status) {
        const double l = trunc(v * (1.0 / 1048576.0));
        if (l != 0.0) {
            if (!(fabs(l) < 4398046511104.0)) {  // 2^42, or not a number
                (void)to_fixed(v, FORCE_SCALE, status);
                return;
            }
            add_to(&large[c][i], (long long)l);
            v -= l * 1048576.0;
        }
        const long long whole = (long long)(v * FORCE_SCALE);
        add_to(&steps[c][i], whole);
        atomicAdd(&parts[c][i], (int)rint((v * FORCE_SCALE - (double)whole) * 1048576.0));
    }
    __device__ __forceinline__ long long total(int c, int i, unsigned* status) const {
        const long long s = steps[c][i] + ((parts[c][i] + 524288) >> 20), l = large[c][i];
        if (l == 0) return s;
        const double v = (double)l * 1048576.0 + (double)s * (1.0 / FORCE_SCALE);
        if (!(fabs(v * FORCE_SCALE) < 9.0e18)) return to_fixed(v, FORCE_SCALE, status);
        return s + l * (1ll << 52);
    }
};
template <>
struct LdsForce<double> {
    double sum[3][TERM_THREADS];
    __device__ __forceinline__ void clear(int c, int i) { sum[c][i] = 0.0; }
    __device__ __forceinline__ void add(int c, int i, double v, unsigned*) { atomicAdd(&sum[c][i], v); }
    __device__ __forceinline__ double total(int c, int i, unsigned*) const { return sum[c][i]; }
};

// The pair sums are added atomically, because the mesh may add into the same
// accumulator from another stream meanwhile.
template <class A>
__global__ __launch_bounds__(TERM_THREADS) void k_fold(int ntiles, const Term* __restrict__ terms,
                                                       const int* __restrict__ tile_atoms,
                                                       const int* __restrict__ tile_sys,
                                                       const double* __restrict__ c6, TermParams P,
                                                       const double* __restrict__ charge,
                                                       const double* __restrict__ pos,
                                                       const SysInfo* __restrict__ sys,
                                                       const int* __restrict__ sorted_atom, int nslots, A* fslot,
                                                       A* force, A* energy, int* order_a, int* order_b,
                                                       unsigned* status) {
    __shared__ double s_pos[3][TERM_THREADS], s_q[TERM_THREADS];
    __shared__ LdsForce<A> s_f;
    __shared__ double s_e[TERM_THREADS / 64];
    __shared__ int s_kind[TERM_THREADS / 64];
    const int t = threadIdx.x;
    if ((int)blockIdx.x >= ntiles) {
        const int s = ((int)blockIdx.x - ntiles) * TERM_THREADS + t;
        if (s >= nslots) return;
        const int a = sorted_atom[s];
        if (order_a) order_a[s] = a;
        if (order_b) order_b[s] = a;
        for (int c = 0; c < 3; ++c) {
            const A v = fslot[(size_t)c * nslots + s];
            if (v != (A)0) {
                if (a >= 0) add_raw(force + 3 * (size_t)a + c, v);
                fslot[(size_t)c * nslots + s] = (A)0;
            }
        }
        return;
    }
    const size_t place = (size_t)blockIdx.x * TERM_THREADS + t;
    const int a = tile_atoms[place], a0 = max(a, 0);
    const Term term = terms[place];
    const double c6_term = c6 ? c6[place] : 0.0;
    const int si = tile_sys[blockIdx.x];
    const double px = pos[3 * (size_t)a0], py = pos[3 * (size_t)a0 + 1], pz = pos[3 * (size_t)a0 + 2];
    const double q = charge[a0];
    s_pos[0][t] = px;
    s_pos[1][t] = py;
    s_pos[2][t] = pz;
    s_q[t] = q;
    for (int c = 0; c < 3; ++c) s_f.clear(c, t);
    __syncthreads();
    const int kind = term.kind_atoms >> 24;
    const int i = term.kind_atoms & 255, j = (term.kind_atoms >> 8) & 255, k = (term.kind_atoms >> 16) & 255;
    double e = 0.0;
    if (kind != TERM_NONE) {
        const double pi[3] = {s_pos[0][i], s_pos[1][i], s_pos[2][i]};
        const double pj[3] = {s_pos[0][j], s_pos[1][j], s_pos[2][j]};
        double fi[3], fk[3];
        if (kind == TERM_ANGLE) {
            const double pk[3] = {s_pos[0][k], s_pos[1][k], s_pos[2][k]};
            e = angle_xyz(pi, pj, pk, term.p[0], term.p[1], fi, fk);
            for (int c = 0; c < 3; ++c) {
                s_f.add(c, k, fk[c], status);
                fk[c] += fi[c];
            }
        } else {
            if (kind == TERM_BOND)
                e = bond_xyz(pi, pj, term.p[0], term.p[1], fi);
            else
                e = exception_xyz(pi, pj, term.p[0], term.p[1], term.p[2], s_q[i], s_q[j], sys[si].box, P.use_pbc,
                                  P.screened, P.alpha, c6_term, P.lj_alpha, fi);
            for (int c = 0; c < 3; ++c) fk[c] = fi[c];
        }
        for (int c = 0; c < 3; ++c) {
            s_f.add(c, i, fi[c], status);
            s_f.add(c, j, -fk[c], status);
        }
    }
    __syncthreads();
    if (a >= 0)
        for (int c = 0; c < 3; ++c) {
            const A v = s_f.total(c, t, status);
            if (v != (A)0) add_raw(force + 3 * (size_t)a + c, v);
        }
    if (energy) {
        // A wave's terms are of its first lane's kind; one add per kind and
        // workgroup (they meet on one address).
        const double sum = wave_sum(e);
        if ((t & 63) == 0) {
            s_e[t >> 6] = sum;
            s_kind[t >> 6] = kind;
        }
        __syncthreads();
        if (t < 3) {
            const int of = t == 0 ? TERM_EXCEPTION : (t == 1 ? TERM_BOND : TERM_ANGLE);
            double total = 0.0;
            for (int w = 0; w < TERM_THREADS / 64; ++w) total += s_kind[w] == of ? s_e[w] : 0.0;
            const int slot = t == 0 ? E_EXCEPT : (t == 1 ? E_BOND : E_ANGLE);
            if (total != 0.0) acc_add(energy + (size_t)si * E_SLOTS + slot, total, ENERGY_SCALE, status);
        }
    }
}

}  // namespace

void TermTiles::build(const std::vector<int>& e1, const std::vector<int>& e2, const std::vector<int>& b1,
                      const std::vector<int>& b2, const std::vector<double>& bp, const std::vector<int>& a1,
                      const std::vector<int>& a2, const std::vector<int>& a3, const std::vector<double>& ap,
                      const std::vector<int>& atom_sys, hipStream_t s) {
    // In the order of each term's lowest atom, tiles closed when a term's kind
    // has no place left, the atoms are full or the system changes.
    struct Item {
        int low, kind, index;
    };
    std::vector<Item> items;
    items.reserve(e1.size() + b1.size() + a1.size());
    host.reserve(2 * items.capacity());
    for (size_t k = 0; k < e1.size(); ++k) items.push_back({std::min(e1[k], e2[k]), TERM_EXCEPTION, (int)k});
    for (size_t k = 0; k < b1.size(); ++k) items.push_back({std::min(b1[k], b2[k]), TERM_BOND, (int)k});
    for (size_t k = 0; k < a1.size(); ++k)
        items.push_back({std::min(a1[k], std::min(a2[k], a3[k])), TERM_ANGLE, (int)k});
    std::stable_sort(items.begin(), items.end(), [](const Item& x, const Item& y) { return x.low < y.low; });
    constexpr int WAVES = TERM_THREADS / 64;
    std::vector<int> tile_atoms, tile_sys;
    std::vector<int> at(atom_sys.size(), -1), tile_of(atom_sys.size(), -1);  // place in the last tile that has the atom
    host.clear();
    place.assign(e1.size(), -1);
    ntiles = 0;
    std::vector<Term> kinds[4];
    std::vector<int> exc_index;
    int natoms = 0;
    auto waves = [&](int extra) {
        int n = 0;
        for (int kd = 1; kd < 4; ++kd) n += ((int)kinds[kd].size() + (kd == extra ? 1 : 0) + 63) / 64;
        return n;
    };
    auto close = [&] {
        if (natoms == 0) return;
        const size_t first = host.size();
        for (int kd = 1; kd < 4; ++kd) {
            if (kd == TERM_EXCEPTION)
                for (size_t k = 0; k < exc_index.size(); ++k) place[exc_index[k]] = (int)(host.size() + k);
            host.insert(host.end(), kinds[kd].begin(), kinds[kd].end());
            host.resize(first + (host.size() - first + 63) / 64 * 64);
            kinds[kd].clear();
        }
        exc_index.clear();
        host.resize(first + TERM_THREADS);
        tile_atoms.resize(first + TERM_THREADS, -1);
        natoms = 0;
        ++ntiles;
    };
    for (const Item& it : items) {
        int a[3], n = 2;
        double p[2] = {0.0, 0.0};
        if (it.kind == TERM_EXCEPTION) {
            a[0] = e1[it.index];
            a[1] = e2[it.index];
        } else if (it.kind == TERM_BOND) {
            a[0] = b1[it.index];
            a[1] = b2[it.index];
        } else {
            a[0] = a1[it.index];
            a[1] = a2[it.index];
            a[2] = a3[it.index];
            n = 3;
        }
        const std::vector<double>* src = it.kind == TERM_BOND ? &bp : (it.kind == TERM_ANGLE ? &ap : nullptr);
        if (src)
            for (int c = 0; c < 2; ++c) p[c] = (*src)[2 * (size_t)it.index + c];
        int fresh = 0;
        for (int c = 0; c < n; ++c)
            if (tile_of[a[c]] != ntiles) ++fresh;
        if (natoms > 0 && (waves(it.kind) > WAVES || natoms + fresh > TERM_THREADS ||
                           tile_sys.back() != atom_sys[a[0]]))
            close();
        if (natoms == 0) tile_sys.push_back(atom_sys[a[0]]);
        Term term = {};
        term.p[0] = p[0];
        term.p[1] = p[1];
        term.kind_atoms = it.kind << 24;
        for (int c = 0; c < n; ++c) {
            if (tile_of[a[c]] != ntiles) {
                tile_of[a[c]] = ntiles;
                at[a[c]] = natoms++;
                tile_atoms.push_back(a[c]);
            }
            term.kind_atoms |= at[a[c]] << (8 * c);
        }
        if (it.kind == TERM_EXCEPTION) exc_index.push_back(it.index);
        kinds[it.kind].push_back(term);
    }
    close();
    if (ntiles == 0) return;
    atoms.upload(tile_atoms, s);
    sys.upload(tile_sys, s);
}

void TermTiles::set_exceptions(const std::vector<double>& qq, const std::vector<double>& sig,
                               const std::vector<double>& eps, const std::vector<double>& c6_by_exception,
                               hipStream_t s) {
    if (ntiles == 0) return;
    for (size_t k = 0; k < place.size(); ++k) {
        Term& term = host[place[k]];
        term.p[0] = qq[k];
        term.p[1] = sig[k];
        term.p[2] = eps[k];
    }
    terms.upload(host, s);
    if (!c6_by_exception.empty()) {
        std::vector<double> by_place(host.size(), 0.0);
        for (size_t k = 0; k < place.size(); ++k) by_place[place[k]] = c6_by_exception[k];
        c6.upload(by_place, s);
    }
}

void launch_fold(bool mixed, const NlistDev& nl, bool slots, const TermTiles* terms, const TermParams& prm,
                 const double* charge, const double* pos, const SysInfo* sys_dev, long long* force_fx, double* force_d,
                 long long* energy_fx, double* energy_d, unsigned* status, hipStream_t s, int* order_a, int* order_b) {
    const int ntiles = terms ? terms->ntiles : 0, nslots = slots ? nl.nslots : 0;
    const int blocks = ntiles + (nslots + TERM_THREADS - 1) / TERM_THREADS;
    if (blocks == 0) return;
    auto go = [&](auto* fslot, auto* force, auto* energy) {
        using A = std::remove_pointer_t<decltype(force)>;
        hipLaunchKernelGGL(k_fold<A>, dim3(blocks), dim3(TERM_THREADS), 0, s, ntiles, ntiles ? terms->terms.p : nullptr,
                           ntiles ? terms->atoms.p : nullptr, ntiles ? terms->sys.p : nullptr,
                           ntiles && prm.lj_alpha > 0.0 ? terms->c6.p : nullptr, prm, charge, pos, sys_dev,
                           nl.sorted_atom.p, nslots, fslot, force, energy, order_a, order_b, status);
    };
    if (mixed) go(nl.fslot_fx.p, force_fx, energy_fx);
    else go(nl.fslot_d.p, force_d, energy_d);
    OMM_HIP(hipGetLastError());
}

}  // namespace ommhip
