// Direct-space LJ + Ewald-screened Coulomb over the tile list
// (nonbonded.rs:842-924).
//
// One wave64 per task = (cluster of 8 i-atoms, up to tpt consecutive tiles
// of 64 entries of the cluster's list); the loads of the next tiles are in
// flight while a tile is evaluated.  Lane l owns i-atom l%8 and the group of entries
// 8*(l/8) .. 8*(l/8)+7; in step k (0..7) it pairs with entry 8*(l/8) + (l%8 ^ k),
// so every entry is touched by exactly one lane per step.  j-data sit in LDS
// (read-only); the j-force accumulators travel with their entry between the
// lanes of a group through DPP permutations (lane ^ 1, ^ 3, ^ 7), so no lane
// writes LDS inside the loop and no LDS instruction moves them.  Positions are FP64 in HBM; each task converts them to
// FP32 offsets from the i-block's FP64 centre, so deltas carry ~1e-7 nm
// absolute error instead of the ~5e-7 nm of absolute FP32 coordinates.
// Near-cutoff pairs (|r^2 - rc^2| < 1e-5 rc^2) are re-decided in FP64 with
// the reference's exact arithmetic, which makes the pair set bit-exact.
//
// Energies of the mixed form: k_pair_energy evaluates each pair in FP64 from
// FP64 offsets, beside the FP32 forces.  The Coulomb classes of a water box (O-O,
// O-H, H-H) are each ~1e6 kJ/mol and cancel to ~1e2-1e3, so any
// distance-dependent FP32 rounding bias would survive in the sum; FP64 pair
// energies remove it.  The MD step does not request energies and never pays
// for this.
#include <climits>
#include <type_traits>

#include "fmath.h"
#include "pairs.h"
#include "terms.h"

namespace ommhip {

namespace {

template <class R>
struct alignas(4 * sizeof(R)) Q4 {
    R x, y, z, w;
};
template <class R>
struct alignas(2 * sizeof(R)) Q2 {
    R x, y;
};

// The reference's cutoff decision for the pair (a, b): delta = x_j - x_i with
// i < j, reduced-triclinic minimum image, r^2 = dx dx + dy dy + dz dz, no FMA.
// Inlined: a call would make the compiler wait for every load in flight
// (the next tile's prefetch) before the band loop of each tile.
__device__ __forceinline__ bool within_cutoff_exact(const double* __restrict__ pos, int a, int b, const Box& bx,
                                                 int periodic, double cutoff2) {
#pragma clang fp contract(off)
    int i = min(a, b), j = max(a, b);
    double d[3] = {pos[3 * j] - pos[3 * i], pos[3 * j + 1] - pos[3 * i + 1], pos[3 * j + 2] - pos[3 * i + 2]};
    if (periodic) min_image_exact(d, bx.v);
    double r2 = d[0] * d[0];
    r2 = r2 + d[1] * d[1];
    r2 = r2 + d[2] * d[2];
    return r2 < cutoff2;
}

// The reference's LJ switch (nonbonded.rs:887-899): S(t) = 1 + t^3 (-10 + t (15 - 6 t))
// and dS/dr for t = (r - r_switch) / (r_cut - r_switch), applied past r_switch.
template <class R>
__device__ __forceinline__ void lj_switch(R r, const PairParams& P, R& s, R& ds) {
    const R inv_width = (R)P.inv_switch_width;
    const R t = (r - (R)P.switch_distance) * inv_width;
    s = (R)1 + t * t * t * ((R)-10 + t * ((R)15 - (R)6 * t));
    ds = (R)-30 * t * t * ((R)1 - t) * ((R)1 - t) * inv_width;
}

// FP64 energy of one pair (nonbonded.rs:1203-1214, 1219-1273) at squared distance r2.
template <int KIND>
__device__ __forceinline__ double pair_energy_fp64(double r2, double sig, double eps4, double ss, double qq,
                                                   const PairParams& P) {
    constexpr int ELEC = KIND & ELEC_MASK;
    // Straight-line: nearly every wave holds pairs with and without LJ and
    // charge, whose terms vanish by their factors eps4 and qq.
    using M = PairF64;
    const double inv_r = M::rsqrt(r2);
    const double r = r2 * inv_r;
    double e = 0.0;
    {
        const double s2 = sig * sig * (inv_r * inv_r);
        const double s6 = s2 * s2 * s2;
        e = eps4 * (s6 * s6 - s6);
        if (KIND & PAIR_LJPME) {
            // nonbonded.rs:875-886: + the reciprocal dispersion of the pair,
            // minus both terms at the cutoff.  C6 = 4 sqrt(eps_i eps_j)
            // (sigma_i sigma_j)^3 = eps4 (4 ss)^3 with ss = (sigma_i/2)(sigma_j/2).
            const double c6 = eps4 * 64.0 * ss * ss * ss, rc2 = P.cutoff * P.cutoff, a = P.lj_alpha;
            double dd;
            const double sc2 = sig * sig / rc2, sc6 = sc2 * sc2 * sc2;
            e += disp_recip_pair(c6, r2, a, &dd) - (eps4 * (sc6 * sc6 - sc6) + disp_recip_pair(c6, rc2, a, &dd));
        }
        if ((KIND & PAIR_SWITCH) && r > P.switch_distance) {
            double sw, dsw;
            lj_switch<double>(r, P, sw, dsw);
            e *= sw;
        }
    }
    if (ELEC == ELEC_EWALD) {
        double ec, ex;
        M::erfc_exp(P.alpha * r, ec, ex);
        e += qq * ec * inv_r;
    } else if (ELEC == ELEC_REACTION_FIELD) {
        e += qq * (inv_r + P.krf * r2 - P.crf);
    } else {
        e += qq * inv_r;
    }
    return e;
}

// Lane permutations by DPP inside each row of 16 lanes: quad_perm [1,0,3,2]
// is lane ^ 1, quad_perm [3,2,1,0] is lane ^ 3, row_half_mirror is lane ^ 7
// (each group of 8 reversed), row_ror:8 is lane ^ 8.
constexpr int DPP_XOR1 = 0xB1, DPP_XOR3 = 0x1B, DPP_XOR7 = 0x141, DPP_XOR8 = 0x128;

// Every control used here reads a lane of the same row, so no lane falls
// back to an old value and the move needs none.
template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xF, 0xF, false));
}
template <int CTRL>
__device__ __forceinline__ double dpp(double v) {
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xF, 0xF, false);
    return __hiloint2double(hi, lo);
}

// The j-force accumulators move from step k to step k + 1: lane l takes the
// accumulator of lane l ^ (k ^ (k + 1)) of its group of 8.
template <int K, class R>
__device__ __forceinline__ void rotate_j(R& gx, R& gy, R& gz) {
    constexpr int m = K ^ (K + 1);
    constexpr int ctrl = m == 1 ? DPP_XOR1 : (m == 3 ? DPP_XOR3 : DPP_XOR7);
    gx = dpp<ctrl>(gx);
    gy = dpp<ctrl>(gy);
    gz = dpp<ctrl>(gz);
}

// Raw data of one tile entry as loaded from HBM, before it is staged in LDS.
template <class R>
struct EntryRaw {
    double x = 0, y = 0, z = 0;
    R q = 0, s = 0, e = 0;
};

// Loads the data of atom a >= 0 with no branch: the entries past the end of
// a list load some real atom's data and are masked when their tile is staged,
// so the loads of a tile never wait on a branch's merge.
template <class R>
__device__ __forceinline__ void load_entry(const int a, const double* __restrict__ pos, const R* __restrict__ qk,
                                           const R* __restrict__ sh, const R* __restrict__ e2, EntryRaw<R>& r) {
    r.x = pos[3 * a];
    r.y = pos[3 * a + 1];
    r.z = pos[3 * a + 2];
    r.q = qk[a];
    r.s = sh[a];
    r.e = e2[a];
}

// Valid entries of the lane's group for i-atom `is` (slot): present, not
// excluded, and after the i-atom where they are of its own cluster (entries
// before the cluster's first slot come from blocks the cluster takes
// cyclically).  il: the i-atom's index in the cluster.
__device__ __forceinline__ unsigned valid_entries(const int* js, const unsigned char* ex, int is, int il) {
    const int4* g4 = reinterpret_cast<const int4*>(js);
    const int4 lo = g4[0], hi = g4[1];
    const int jv[CLUSTER] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
    const int cfirst = is & ~(CLUSTER - 1);
    unsigned vmask = 0;
#pragma unroll
    for (int s8 = 0; s8 < CLUSTER; ++s8)
        if (jv[s8] != INT_MAX && (jv[s8] > is || jv[s8] < cfirst)) vmask |= 1u << s8;
    // Bit il of each of the group's eight exclusion bytes, gathered into bits
    // 0-7: each byte's bit il moves to the byte's bit 0, and a multiply by
    // 2^0 + 2^7 + 2^14 + 2^21 carries the bits of bytes 0-3 (positions 0, 8, 16,
    // 24) to positions 21-24 without collisions.
    const unsigned long long xb = *reinterpret_cast<const unsigned long long*>(ex);
    const unsigned long long sel = (xb >> il) & 0x0101010101010101ull;
    const unsigned lo4 = (((unsigned)sel * 0x00204081u) >> 21) & 0xFu;
    const unsigned hi4 = (((unsigned)(sel >> 32) * 0x00204081u) >> 21) & 0xFu;
    return vmask & ~(lo4 | (hi4 << 4));
}

// Sum over the eight groups (lanes l, l ^ 8, l ^ 16, ...).
__device__ __forceinline__ double group_sum(double v) {
    for (int o = CLUSTER; o < 64; o <<= 1) v += __shfl_xor(v, o, 64);
    return v;
}
// Likewise, by register permutations: a swap of the odd rows (or the upper half) with a
// copy's even rows (lower half) leaves the two partners' values in the two results.
__device__ __forceinline__ long long group_sum(long long v) {
    v += __double_as_longlong(dpp<DPP_XOR8>(__longlong_as_double(v)));
    auto joined = [](unsigned lo, unsigned hi) { return (long long)(((unsigned long long)hi << 32) | lo); };
    {
        const unsigned lo = (unsigned)v, hi = (unsigned)((unsigned long long)v >> 32);
        const auto l = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
        const auto h = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
        v = joined(l[0], h[0]) + joined(l[1], h[1]);
    }
    const unsigned lo = (unsigned)v, hi = (unsigned)((unsigned long long)v >> 32);
    const auto l = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
    const auto h = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
    return joined(l[0], h[0]) + joined(l[1], h[1]);
}
// A lane's force on its i-atom over a task.  Mixed form: each tile's FP32 sum is
// rounded to multiples of 2^-32, the accumulators' step, which are added as
// integers, so the total does not depend on how many tiles a task holds.  Adding
// 1.5 x 2^20, where FP64 has that step, leaves the multiple in the low bits.
// Components of 2^19 kJ/mol/nm and more, which are rare, are multiples of 2^-4 and
// are added in FP64, exactly while sums stay below 2^49.
struct FixedForce {
    static constexpr double STEP = 1572864.0;  // 1.5 x 2^20
    static constexpr float LARGE = 524288.0f;  // 2^19
    long long sum[3] = {0, 0, 0};
    double large[3] = {0, 0, 0};
    static __device__ __forceinline__ long long steps(float f) {
        return __double_as_longlong((double)f + STEP) - __double_as_longlong(STEP);
    }
    __device__ __forceinline__ void add(float fx, float fy, float fz) {
        const float f[3] = {fx, fy, fz};
        // The absolute sum bounds each component and is NaN where one of them is.
        if (__ballot(!(fabsf(fx) + fabsf(fy) + fabsf(fz) < LARGE)) == 0ull) {
#pragma unroll
            for (int c = 0; c < 3; ++c) sum[c] += steps(f[c]);
            return;
        }
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const bool small = fabsf(f[c]) < LARGE;
            sum[c] += steps(small ? f[c] : 0.0f);
            large[c] += small ? 0.0 : (double)f[c];
        }
    }
    __device__ __forceinline__ void totals(long long t[3], unsigned* status) const {
        for (int c = 0; c < 3; ++c) t[c] = group_sum(sum[c]);  // below 2^56
        if (__ballot(large[0] != 0.0 || large[1] != 0.0 || large[2] != 0.0) == 0ull) return;
        // The range is that of the whole task's force.
        for (int c = 0; c < 3; ++c) {
            const double l = group_sum(large[c]);
            if (fabs(l * FORCE_SCALE + (double)t[c]) < 9.0e18) t[c] += (long long)(l * FORCE_SCALE);
            else t[c] = to_fixed(l + (double)t[c] * (1.0 / FORCE_SCALE), FORCE_SCALE, status);
        }
    }
};
struct PlainForce {
    double x[3] = {0, 0, 0};
    __device__ __forceinline__ void add(double fx, double fy, double fz) {
        x[0] += fx;
        x[1] += fy;
        x[2] += fz;
    }
    __device__ __forceinline__ void totals(double t[3], unsigned*) const {
        for (int c = 0; c < 3; ++c) t[c] = group_sum(x[c]);
    }
};
__device__ __forceinline__ void add_total(long long* p, long long v) {
    if (v) atomicAdd(reinterpret_cast<unsigned long long*>(p), (unsigned long long)v);
}
__device__ __forceinline__ void add_total(double* p, double v) {
    if (v != 0.0) unsafeAtomicAdd(p, v);
}

// FP64 forces with energies beside a mesh: one wave per SIMD, though the registers
// allow two, so that the mesh's kernels find room beside them (9,000 atoms, a call
// of energy and forces 481 us with two, 430 with one; the kernel alone 64 either way).
constexpr int pair_waves_per_simd(int kind, bool energy) {
    return energy && (kind & ELEC_MASK) == ELEC_EWALD ? 1 : 8;
}

template <class R, class A, int KIND, bool STATS, bool ENERGY>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(1, pair_waves_per_simd(KIND, ENERGY)))) void k_pairs(const double* __restrict__ pos, const R* __restrict__ qk,
                                              const R* __restrict__ sh, const R* __restrict__ e2,
                                              const int* __restrict__ sorted_atom,
                                              const unsigned char* __restrict__ clist_ex,
                                              const double* __restrict__ center,
                                              const int* __restrict__ minimg, const int2* __restrict__ clist,
                                              const int* __restrict__ ccount, const int* __restrict__ tasks,
                                              const int* __restrict__ ntasks, const int* __restrict__ block_sys,
                                              const SysInfo* __restrict__ sys, PairParams P, int tpt, A* fslot, A* energy,
                                              unsigned* status, unsigned long long* stats, int* list_flag,
                                              int nflags) {
    using M = Math<R>;
    constexpr int ELEC = KIND & ELEC_MASK;
    constexpr bool SWITCH = (KIND & PAIR_SWITCH) != 0;
    constexpr bool LJPME = (KIND & PAIR_LJPME) != 0;
    static_assert(!ENERGY || sizeof(R) == 8, "the mixed form's energies: k_pair_energy");
    __shared__ Q4<R> s_pq[JTILE];
    __shared__ Q2<R> s_se[JTILE];
    __shared__ __align__(16) int s_js[JTILE];
    __shared__ int s_ja[JTILE];
    __shared__ __align__(8) unsigned char s_ex[JTILE];  // exclusion bits of each entry (bit k: i-atom k)

    const int lane = threadIdx.x;
    const int grp = lane / CLUSTER;  // the lane's group of 8 tile entries
    const int il = lane % CLUSTER;   // the lane's i-atom in the cluster
    const double cutoff2 = P.cutoff * P.cutoff;
    const double band = sizeof(R) == 4 ? 1e-5 : 1e-12;
    const R rc2_lo = (R)(cutoff2 * (1.0 - band));
    const R rc2_hi = (R)(cutoff2 * (1.0 + band));
    const R alpha = (R)P.alpha;
    const R two_a_sqrtpi = (R)(2.0 * P.alpha / sqrt(PI));
    const R krf = (R)P.krf, crf = (R)P.crf;
    const R lj_a2 = (R)(P.lj_alpha * P.lj_alpha);
    // This kernel runs after every list build and before the next integrator,
    // so it serves the rebuild requests.
    if (blockIdx.x == 0)
        for (int i = threadIdx.x; i < nflags; i += blockDim.x) list_flag[i] = 0;

    const int total = ntasks[0];
    for (int t = blockIdx.x; t < total; t += gridDim.x) {
        const int task = tasks[t];
        const int C = task >> 8;
        const int first = task & 255;
        const int I = C / CPB;
        const int count = ccount[C];
        const int ntile = min(tpt, (count + JTILE - 1) / JTILE - first);
        const int sidx = block_sys[I];
        const Box& bx = sys[sidx].box;
        const double c0 = center[3 * I], c1 = center[3 * I + 1], c2 = center[3 * I + 2];
        const int2* list = clist + (size_t)C * P.cap + (size_t)first * JTILE;
        const unsigned char* list_ex = clist_ex + (size_t)C * P.cap + (size_t)first * JTILE;
        const int nentries = count - first * JTILE;
        // Entry e of tile tl is live when tl < ntile and e < nentries.  Every
        // lane loads some real entry of the list (the last one past its end)
        // and the liveness is applied when the tile is staged, so no load
        // sits behind a branch.
        const int last = max(nentries - 1, 0);
        auto live = [&](int tl) { return tl < ntile && tl * JTILE + lane < nentries; };
        auto entry = [&](int tl) { return list[min(tl * JTILE + lane, last)]; };
        auto entry_ex = [&](int tl) -> unsigned { return list_ex[min(tl * JTILE + lane, last)]; };
        // The task waits for two rounds of loads before its first tile: the
        // i-atom's slot with the first two tiles' entries, then the i-atom's
        // data with tile 0's coordinates and parameters.
        const int is = C * CLUSTER + il;
        const int ia = sorted_atom[is];  // -1 in the padding of a system's last block
        // Software pipeline: the entries of tile k + 2 and the coordinates of
        // tile k + 1 are in flight while tile k is evaluated.
        int2 e0 = entry(0), e1 = entry(1);
        unsigned x0 = entry_ex(0), x1 = entry_ex(1);
        const int ia0 = max(ia, 0);
        const double pxi = pos[3 * ia0], pyi = pos[3 * ia0 + 1], pzi = pos[3 * ia0 + 2];
        const R qi_raw = qk[ia0], si_raw = sh[ia0], ei_raw = e2[ia0];
        EntryRaw<R> r0;
        load_entry<R>(max(e0.y, 0), pos, qk, sh, e2, r0);

        R xi = 0, yi = 0, zi = 0, qi = 0, si = 0, ei = 0;
        if (ia >= 0) {
            double d[3] = {pxi - c0, pyi - c1, pzi - c2};
            if (P.periodic) wrap_nearest(d, bx);
            xi = (R)d[0];
            yi = (R)d[1];
            zi = (R)d[2];
            qi = qi_raw;
            si = si_raw;
            ei = ei_raw;
        }
        // The pair steps read the i-atom's parameters inside divergent
        // branches, where the compiler cannot prove an earlier wait and
        // would wait for every load in flight, the next tile's prefetch
        // included, in each step.  Reading them here once, on every path,
        // completes their loads before the tiles start.
        asm volatile("" ::"v"(qi), "v"(si), "v"(ei));
        const bool mi = P.periodic && minimg[I];
        R bv[9], ib0 = 0, ib4 = 0, ib8 = 0;
        if (mi) {
            for (int k = 0; k < 9; ++k) bv[k] = (R)bx.v[k];
            ib0 = (R)(1.0 / bx.v[0]);
            ib4 = (R)(1.0 / bx.v[4]);
            ib8 = (R)(1.0 / bx.v[8]);
        }

        using Force = typename std::conditional<sizeof(R) == 4, FixedForce, PlainForce>::type;
        Force ftot;
        double eacc = 0.0;
        unsigned long long npair = 0, hsum = 0;
        for (int k = 0; k < ntile; ++k) {
            const int2 e2n = entry(k + 2);
            const unsigned x2n = entry_ex(k + 2);
            EntryRaw<R> r1;
            load_entry<R>(max(e1.y, 0), pos, qk, sh, e2, r1);

            // Stage tile k in LDS as offsets from the block centre.
            {
                if (!live(k)) {
                    e0 = make_int2(INT_MAX, -1);
                    x0 = 0u;
                }
                Q4<R> pq = {0, 0, 0, 0};
                Q2<R> se = {0, 0};
                if (e0.y >= 0) {
                    double d[3] = {r0.x - c0, r0.y - c1, r0.z - c2};
                    if (P.periodic) wrap_nearest(d, bx);
                    pq = {(R)d[0], (R)d[1], (R)d[2], r0.q};
                    se = {r0.s, r0.e};
                }
                s_pq[lane] = pq;
                s_se[lane] = se;
                s_js[lane] = e0.x;
                s_ja[lane] = e0.y;
                s_ex[lane] = (unsigned char)x0;
            }
            __syncthreads();

            unsigned vmask = 0;
            if (ia >= 0) vmask = valid_entries(s_js + grp * CLUSTER, s_ex + grp * CLUSTER, is, il);

            R fx = 0, fy = 0, fz = 0;
            R gx = 0, gy = 0, gz = 0;
            // Offset of the entry at pj from the lane's i-atom, with the FP32
            // minimum image when MI (the block is near half the box).
            auto delta = [&](const Q4<R>& pj, R& dx, R& dy, R& dz, auto MI) {
                dx = pj.x - xi;
                dy = pj.y - yi;
                dz = pj.z - zi;
                if (decltype(MI)::value) {
                    R s = M::round(dz * ib8);
                    dx -= s * bv[6];
                    dy -= s * bv[7];
                    dz -= s * bv[8];
                    s = M::round(dy * ib4);
                    dx -= s * bv[3];
                    dy -= s * bv[4];
                    s = M::round(dx * ib0);
                    dx -= s * bv[0];
                }
            };
            // F/r of a pair at squared distance r2 with the entry's charge qj
            // and LJ parameters sj; e receives the pair's working-precision energy.
            auto pair_fe = [&](const R qj, const Q2<R> sj, const R r2, R& e) -> R {
                const R inv_r = M::rsqrt(r2);
                const R inv_r2 = inv_r * inv_r;
                // Lennard-Jones with Lorentz-Berthelot combination (nonbonded.rs:869-874, 1203-1214).
                const R sig = si + sj.x;
                const R eps4 = ei * sj.y;
                const R s2 = sig * sig * inv_r2;
                const R s6 = s2 * s2 * s2;
                const R s12 = s6 * s6;
                e = eps4 * (s12 - s6);
                R f = eps4 * ((R)6 * s6 - (R)12 * s12) * inv_r2;
                if (LJPME) {
                    // nonbonded.rs:875-886 with C6 = eps4 (4 (sigma_i/2)(sigma_j/2))^3.
                    // Closed form (no small-x series: x = alpha^2 r^2 < 0.01 needs
                    // r < 0.1/alpha, far inside any non-excluded pair's LJ core).
                    const R ss = si * sj.x;
                    const R c6 = eps4 * (R)64 * ss * ss * ss;
                    const R x = lj_a2 * r2;
                    const R ex = M::exp_neg(x);
                    const R poly = (R)1 + x * ((R)1 + (R)0.5 * x);
                    const R c6r6 = c6 * inv_r2 * inv_r2 * inv_r2;
                    f -= (R)6 * c6r6 * inv_r2 * ((R)1 - ex * (poly + x * x * x * (R)(1.0 / 6.0)));
                    if (ENERGY) {
                        const R rc2 = (R)(P.cutoff * P.cutoff);
                        const R sc2 = sig * sig / rc2, sc6 = sc2 * sc2 * sc2;
                        const R xc = lj_a2 * rc2;
                        const R shift = eps4 * (sc6 * sc6 - sc6) +
                                        c6 / (rc2 * rc2 * rc2) *
                                            ((R)1 - M::exp_neg(xc) * ((R)1 + xc * ((R)1 + (R)0.5 * xc)));
                        e += c6r6 * ((R)1 - ex * poly) - shift;
                    }
                }
                if (SWITCH) {
                    // Inside the switching distance t = 0 gives S = 1 and
                    // dS/dr = 0 exactly, so no branch is needed.
                    const R r = M::max(r2 * inv_r, (R)P.switch_distance);
                    R sw, dsw;
                    lj_switch<R>(r, P, sw, dsw);
                    f = sw * f + e * dsw * inv_r;
                    e *= sw;
                }
                const R qq = qi * qj;
                if (ELEC == ELEC_EWALD) {
                    // screened_coulomb (nonbonded.rs:1263-1273)
                    const R r = r2 * inv_r;
                    R erfc_v, ex2;
                    M::erfc_exp(alpha * r, erfc_v, ex2);
                    const R ec = qq * erfc_v * inv_r;
                    e += ec;
                    f -= (ec + qq * two_a_sqrtpi * ex2) * inv_r2;
                } else if (ELEC == ELEC_REACTION_FIELD) {
                    // reaction_field (nonbonded.rs:1233-1250)
                    e += qq * (inv_r + krf * r2 - crf);
                    f += qq * ((R)2 * krf - inv_r * inv_r2);
                } else {
                    // coulomb_pair (nonbonded.rs:1219-1226)
                    const R ec = qq * inv_r;
                    e += ec;
                    f -= ec * inv_r2;
                }
                return f;
            };
            // Step k: lane (grp, il) pairs i-atom il with entry grp * 8 + (il ^ k);
            // each entry meets every i-atom of the cluster once over the 8 steps.
            // Pairs whose FP32 r^2 falls in the band around the cutoff are only
            // marked here and decided in FP64 after the steps.  Every lane
            // evaluates its slot whether or not it holds an accepted pair: a
            // wave nearly always holds one in each step, so a branch would skip
            // nothing, and straight-line steps let the compiler issue the next
            // step's LDS reads early.  A rejected slot's r^2 is replaced by 1
            // (away from the singularity at 0) and its force selected to zero.
            // The minimum-image choice is made once per tile, outside the
            // steps, so the eight steps form one straight block.
            // Energies are selected and the statistics' pairs marked and counted
            // afterwards: behind a branch in each step the FP64 forms needed up to 284
            // registers, the rest beyond 256 in accumulation registers.
            unsigned near = 0, taken = 0;
            auto pair_step = [&](const int k, auto MI) {
                const int s8 = il ^ k;
                const int slot = grp * CLUSTER + s8;
                const Q4<R> pj = s_pq[slot];
                const Q2<R> sj = s_se[slot];
                R dx, dy, dz;
                delta(pj, dx, dy, dz, MI);
                const R r2 = dx * dx + dy * dy + dz * dz;
                const bool valid = (vmask >> s8) & 1u;
                const bool in = valid && (!P.use_cutoff || r2 < rc2_lo);
                if (valid && !in && r2 < rc2_hi) near |= 1u << s8;
                R e;
                R f = pair_fe(pj.w, sj, in ? r2 : (R)1, e);
                f = in ? f : (R)0;
                if (ENERGY) eacc += in ? (double)e : 0.0;
                if (STATS) taken |= in ? 1u << s8 : 0u;
                fx += f * dx;
                fy += f * dy;
                fz += f * dz;
                gx -= f * dx;
                gy -= f * dy;
                gz -= f * dz;
            };
            auto eight_steps = [&](auto MI) {
                pair_step(0, MI);
                rotate_j<0>(gx, gy, gz);
                pair_step(1, MI);
                rotate_j<1>(gx, gy, gz);
                pair_step(2, MI);
                rotate_j<2>(gx, gy, gz);
                pair_step(3, MI);
                rotate_j<3>(gx, gy, gz);
                pair_step(4, MI);
                rotate_j<4>(gx, gy, gz);
                pair_step(5, MI);
                rotate_j<5>(gx, gy, gz);
                pair_step(6, MI);
                rotate_j<6>(gx, gy, gz);
                pair_step(7, MI);
            };
            if (mi) eight_steps(std::true_type{});
            else eight_steps(std::false_type{});
            // The cutoff band: the reference's FP64 decision (rare pairs; their
            // j-forces go straight to the slot-ordered accumulator).
            while (__ballot(near != 0u)) {
                if (near) {
                    const int s8 = __ffs(near) - 1;
                    near &= near - 1u;
                    const int slot = grp * CLUSTER + s8;
                    if (within_cutoff_exact(pos, ia, s_ja[slot], bx, P.periodic, cutoff2)) {
                        const Q4<R> pj = s_pq[slot];
                        R dx, dy, dz, e;
                        if (mi) delta(pj, dx, dy, dz, std::true_type{});
                        else delta(pj, dx, dy, dz, std::false_type{});
                        const R f = pair_fe(pj.w, s_se[slot], dx * dx + dy * dy + dz * dz, e);
                        if (ENERGY) eacc += (double)e;
                        if (STATS) taken |= 1u << s8;
                        fx += f * dx;
                        fy += f * dy;
                        fz += f * dz;
                        const int js = s_js[slot];
                        acc_add(fslot + js, (double)(-f * dx), FORCE_SCALE, status);
                        acc_add(fslot + P.nslots + js, (double)(-f * dy), FORCE_SCALE, status);
                        acc_add(fslot + 2 * P.nslots + js, (double)(-f * dz), FORCE_SCALE, status);
                    }
                }
            }
            if (STATS)
                for (; taken; taken &= taken - 1u) {
                    const int ja = s_ja[grp * CLUSTER + __ffs(taken) - 1];
                    ++npair;
                    hsum += pair_key(min(ia, ja), max(ia, ja));
                }
            // After step 7 the lane holds the accumulator of entry grp * 8 + (il ^ 7).
            const int jmine = grp * CLUSTER + (il ^ (CLUSTER - 1));
            if (s_ja[jmine] >= 0) {
                const int js = s_js[jmine];
                acc_add(fslot + js, (double)gx, FORCE_SCALE, status);
                acc_add(fslot + P.nslots + js, (double)gy, FORCE_SCALE, status);
                acc_add(fslot + 2 * P.nslots + js, (double)gz, FORCE_SCALE, status);
            }
            ftot.add(fx, fy, fz);
            __syncthreads();
            e0 = e1;
            e1 = e2n;
            x0 = x1;
            x1 = x2n;
            r0 = r1;
        }
        // i-forces: the eight groups' sums, in a fixed order.
        A ft[3];
        ftot.totals(ft, status);
        if (grp == 0 && ia >= 0) {
            add_total(fslot + is, ft[0]);
            add_total(fslot + P.nslots + is, ft[1]);
            add_total(fslot + 2 * P.nslots + is, ft[2]);
        }
        if (ENERGY) {
            double etot = wave_sum(eacc);
            if (lane == 0) acc_add(energy + sidx * E_SLOTS + E_DIRECT, etot, ENERGY_SCALE, status);
        }
        if (STATS) {
            npair = wave_sum_u64(npair);
            hsum = wave_sum_u64(hsum);
            if (lane == 0) {
                atomicAdd(stats + 2 * sidx, npair);
                atomicAdd(stats + 2 * sidx + 1, hsum);
            }
        }
    }
}

// Pair energies of the mixed form in FP64, over the pair kernel's tasks and
// pair set: FP64 offsets and parameters, the cutoff decided as the pair kernel
// decides it (exactly, near the cutoff).  A kernel of its own: within the pair
// kernel the FP64 values took its registers to one or two waves per SIMD.
// Waves loop over tasks; each tile's sum is rounded to fixed point and added, so
// neither the tasks' size nor their order changes the total.  Adds to one energy
// serialise (12 ns each: one per task was 60 us at 9,000 atoms), so few waves
// are launched and a workgroup adds once when its waves saw one system.
// Bound: FP64 issue.  36% of a tile's slots are in range: they are lined up in
// LDS first and evaluated 64 at a time (every slot evaluated: 9,000 atoms 27.7 us,
// so 24.1; 23,550 62.6 and 55.2; 300,000 869 and 733).  Pair forces and energies
// together, in one kernel and now in two: 58 -> 18 us at 900 atoms, 91 -> 44 at
// 9,000, 132 -> 98 at 23,550.
constexpr int ENERGY_WAVES = 4;           // waves per workgroup
constexpr int ENERGY_WORKGROUPS = 768;    // at most: three waves per SIMD of the chip

template <int KIND>
__global__ __launch_bounds__(64 * ENERGY_WAVES) void k_pair_energy(
    const double* __restrict__ pos, const double* __restrict__ qk, const double* __restrict__ sh,
    const double* __restrict__ e2, const int* __restrict__ sorted_atom, const unsigned char* __restrict__ clist_ex,
    const double* __restrict__ center, const int* __restrict__ minimg, const int2* __restrict__ clist,
    const int* __restrict__ ccount, const int* __restrict__ tasks, const int* __restrict__ ntasks,
    const int* __restrict__ block_sys, const SysInfo* __restrict__ sys, PairParams P, int tpt, long long* energy,
    unsigned* status) {
    __shared__ Q4<double> s_pw[ENERGY_WAVES][JTILE];
    __shared__ Q2<double> s_sew[ENERGY_WAVES][JTILE];
    __shared__ __align__(16) int s_jsw[ENERGY_WAVES][JTILE];
    __shared__ int s_jaw[ENERGY_WAVES][JTILE];
    __shared__ __align__(8) unsigned char s_exw[ENERGY_WAVES][JTILE];
    __shared__ long long s_sum[ENERGY_WAVES];
    __shared__ int s_of[ENERGY_WAVES];
    constexpr int RING = 128, RING_VALUES = (KIND & PAIR_LJPME) != 0 ? 5 : 4;
    __shared__ double s_ring[ENERGY_WAVES][RING_VALUES][RING];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    double(*ring)[RING] = s_ring[wave];
    Q4<double>* s_p = s_pw[wave];
    Q2<double>* s_se = s_sew[wave];
    int *s_js = s_jsw[wave], *s_ja = s_jaw[wave];
    unsigned char* s_ex = s_exw[wave];
    const int lane = threadIdx.x & 63, grp = lane / CLUSTER, il = lane % CLUSTER;
    const unsigned long long below = (1ull << lane) - 1ull;
    const double cutoff2 = P.cutoff * P.cutoff;
    const double rc2_lo = cutoff2 * (1.0 - 1e-12), rc2_hi = cutoff2 * (1.0 + 1e-12);
    long long esum = 0;  // lane 0: fixed-point energy of system esys
    int esys = -1;
    const int total = ntasks[0];
    for (int t = blockIdx.x * ENERGY_WAVES + wave; t < total; t += gridDim.x * ENERGY_WAVES) {
        const int task = tasks[t], C = task >> 8, first = task & 255, I = C / CPB;
        const int count = ccount[C];
        const int ntile = min(tpt, (count + JTILE - 1) / JTILE - first);
        const int sidx = block_sys[I];
        const Box& bx = sys[sidx].box;
        const double c0 = center[3 * I], c1 = center[3 * I + 1], c2 = center[3 * I + 2];
        const int2* list = clist + (size_t)C * P.cap + (size_t)first * JTILE;
        const unsigned char* list_ex = clist_ex + (size_t)C * P.cap + (size_t)first * JTILE;
        const int nentries = count - first * JTILE, last = max(nentries - 1, 0);
        auto entry = [&](int tl) { return list[min(tl * JTILE + lane, last)]; };
        auto entry_ex = [&](int tl) -> unsigned { return list_ex[min(tl * JTILE + lane, last)]; };
        const int is = C * CLUSTER + il;
        const int ia = sorted_atom[is], ia0 = max(ia, 0);
        int2 e0 = entry(0);
        unsigned x0 = entry_ex(0);
        double di[3] = {pos[3 * ia0] - c0, pos[3 * ia0 + 1] - c1, pos[3 * ia0 + 2] - c2};
        const double qi = qk[ia0], si = sh[ia0], ei = e2[ia0];
        if (P.periodic) wrap_nearest(di, bx);
        const bool mi = P.periodic && minimg[I];
        if (sidx != esys) {
            if (lane == 0 && esys >= 0) add_total(energy + esys * E_SLOTS + E_DIRECT, esum);
            esum = 0;
            esys = sidx;
        }
        for (int k = 0; k < ntile; ++k) {
            EntryRaw<double> r0;
            load_entry<double>(max(e0.y, 0), pos, qk, sh, e2, r0);
            const int2 e1 = entry(k + 1);
            const unsigned x1 = entry_ex(k + 1);
            const bool live = k * JTILE + lane < nentries;
            double d[3] = {r0.x - c0, r0.y - c1, r0.z - c2};
            if (P.periodic) wrap_nearest(d, bx);
            s_p[lane] = {d[0], d[1], d[2], r0.q};
            s_se[lane] = {r0.s, r0.e};
            s_js[lane] = live && e0.y >= 0 ? e0.x : INT_MAX;
            s_ja[lane] = e0.y;
            s_ex[lane] = (unsigned char)x0;
            wave_lds_fence();
            const unsigned present = valid_entries(s_js + grp * CLUSTER, s_ex + grp * CLUSTER, is, il);
            const unsigned vmask = ia >= 0 ? present : 0u;
            double eacc = 0.0;
            // The tile's pairs in range are lined up in a ring, 64 evaluated at
            // a time; the last turn evaluates the rest.
            int head = 0, waiting = 0;
#pragma unroll 1
            for (int s8 = 0; s8 <= CLUSTER; ++s8) {
                if (s8 < CLUSTER) {
                    const int slot = grp * CLUSTER + s8;
                    const Q4<double> pj = s_p[slot];
                    double dd[3] = {pj.x - di[0], pj.y - di[1], pj.z - di[2]};
                    if (mi) wrap_nearest(dd, bx);
                    const double r2 = dd[0] * dd[0] + dd[1] * dd[1] + dd[2] * dd[2];
                    const bool valid = (vmask >> s8) & 1u;
                    bool in = valid && (!P.use_cutoff || r2 < rc2_lo);
                    if (valid && !in && r2 < rc2_hi)
                        in = within_cutoff_exact(pos, ia, s_ja[slot], bx, P.periodic, cutoff2);
                    const unsigned long long m = __ballot(in);
                    if (in) {
                        const Q2<double> sj = s_se[slot];
                        const int at = (head + waiting + __popcll(m & below)) & (RING - 1);
                        ring[0][at] = r2;
                        ring[1][at] = si + sj.x;
                        ring[2][at] = ei * sj.y;
                        ring[3][at] = qi * pj.w;
                        if constexpr ((KIND & PAIR_LJPME) != 0) ring[4][at] = si * sj.x;
                    }
                    waiting += __popcll(m);
                    wave_lds_fence();
                    if (waiting < 64) continue;
                } else if (waiting == 0) {
                    break;
                }
                // A lane without a pair evaluates the last one.
                const int at = (head + min(lane, waiting - 1)) & (RING - 1);
                const double ss = (KIND & PAIR_LJPME) != 0 ? ring[RING_VALUES - 1][at] : 0.0;
                const double e = pair_energy_fp64<KIND>(ring[0][at], ring[1][at], ring[2][at], ss, ring[3][at], P);
                eacc += lane < waiting ? e : 0.0;
                const int taken = min(waiting, 64);
                head += taken;
                waiting -= taken;
                wave_lds_fence();
            }
            const double et = wave_sum(eacc);
            esum += to_fixed_nearest(et, ENERGY_SCALE, status);
            wave_lds_fence();
            e0 = e1;
            x0 = x1;
        }
    }
    if (lane == 0) {
        s_sum[wave] = esum;
        s_of[wave] = esys;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        // Waves 0, 1, ... took the first tasks: an idle wave follows a busy one.
        for (int w = 0; w < ENERGY_WAVES && s_of[w] >= 0;) {
            long long sum = 0;
            const int of = s_of[w];
            for (; w < ENERGY_WAVES && s_of[w] == of; ++w) sum += s_sum[w];
            add_total(energy + of * E_SLOTS + E_DIRECT, sum);
        }
    }
}

template <class A>
A* slot_buffer(const NlistDev& nl);
template <>
long long* slot_buffer<long long>(const NlistDev& nl) {
    return nl.fslot_fx.p;
}
template <>
double* slot_buffer<double>(const NlistDev& nl) {
    return nl.fslot_d.p;
}

template <class R, class A, int ELEC, bool STATS, bool ENERGY>
void launch_one(const NlistDev& nl, const PairParams& p, const R* qk, const R* sh, const R* e2,
                const ParticleDev& part, const double* pos, const SysInfo* sys_dev, A* energy,
                unsigned* status, unsigned long long* stats, int grid,
                hipStream_t s) {
    constexpr bool MIXED = sizeof(R) == 4;
    hipLaunchKernelGGL((k_pairs<R, A, ELEC, STATS, ENERGY && !MIXED>), dim3(grid), dim3(64), 0, s, pos, qk, sh, e2,
                       nl.sorted_atom.p, nl.clist_ex.p, nl.block_center.p, nl.block_minimg.p, nl.clist.p, nl.ccount.p,
                       nl.tasks.p, nl.ntasks.p, nl.block_sys.p, sys_dev, p, nl.tpt, slot_buffer<A>(nl), energy, status,
                       stats, nl.flag.p, nl.nsys + 1);
    if constexpr (ENERGY && MIXED)
        hipLaunchKernelGGL((k_pair_energy<ELEC>), dim3(std::min((grid + ENERGY_WAVES - 1) / ENERGY_WAVES, ENERGY_WORKGROUPS)),
                           dim3(64 * ENERGY_WAVES), 0, s, pos, part.qk_d.p,
                           part.sh_d.p, part.e2_d.p, nl.sorted_atom.p, nl.clist_ex.p, nl.block_center.p,
                           nl.block_minimg.p, nl.clist.p, nl.ccount.p, nl.tasks.p, nl.ntasks.p, nl.block_sys.p,
                           sys_dev, p, nl.tpt, energy, status);
}

template <class R, class A, int ELEC>
void launch_pairs_t(bool stats_on, bool energy_on, const NlistDev& nl, const PairParams& p, const R* qk, const R* sh,
                    const R* e2, const ParticleDev& part, const double* pos, const SysInfo* sys_dev, A* energy,
                    unsigned* status, unsigned long long* stats, int grid,
                    hipStream_t s) {
    if (stats_on)
        launch_one<R, A, ELEC, true, false>(nl, p, qk, sh, e2, part, pos, sys_dev, energy, status, stats, grid, s);
    else if (energy_on)
        launch_one<R, A, ELEC, false, true>(nl, p, qk, sh, e2, part, pos, sys_dev, energy, status, stats, grid, s);
    else
        launch_one<R, A, ELEC, false, false>(nl, p, qk, sh, e2, part, pos, sys_dev, energy, status, stats, grid, s);
}

}  // namespace

namespace {
// Pair kernel variants: the electrostatics kind, plus PAIR_SWITCH when the LJ
// switching function is on (a separate kernel, so the common case carries
// none of its arithmetic).
template <class R, class A>
void dispatch_kind(int kind, bool st, bool energy_on, const NlistDev& nl, const PairParams& p, const R* qk,
                   const R* sh, const R* e2, const ParticleDev& part, const double* pos, const SysInfo* sys_dev,
                   A* energy, unsigned* status, unsigned long long* stats, int grid, hipStream_t s) {
    switch (kind) {
        case ELEC_EWALD:
            launch_pairs_t<R, A, ELEC_EWALD>(st, energy_on, nl, p, qk, sh, e2, part, pos, sys_dev, energy, status,
                                             stats, grid, s);
            break;
        case ELEC_REACTION_FIELD:
            launch_pairs_t<R, A, ELEC_REACTION_FIELD>(st, energy_on, nl, p, qk, sh, e2, part, pos, sys_dev, energy, status, stats, grid, s);
            break;
        case ELEC_COULOMB:
            launch_pairs_t<R, A, ELEC_COULOMB>(st, energy_on, nl, p, qk, sh, e2, part, pos, sys_dev, energy,
                                               status, stats, grid, s);
            break;
        case ELEC_EWALD | PAIR_SWITCH:
            launch_pairs_t<R, A, ELEC_EWALD | PAIR_SWITCH>(st, energy_on, nl, p, qk, sh, e2, part, pos, sys_dev, energy, status, stats, grid, s);
            break;
        case ELEC_REACTION_FIELD | PAIR_SWITCH:
            launch_pairs_t<R, A, ELEC_REACTION_FIELD | PAIR_SWITCH>(st, energy_on, nl, p, qk, sh, e2, part, pos,
                                                                    sys_dev, energy, status, stats, grid, s);
            break;
        case ELEC_EWALD | PAIR_LJPME:
            launch_pairs_t<R, A, ELEC_EWALD | PAIR_LJPME>(st, energy_on, nl, p, qk, sh, e2, part, pos, sys_dev, energy, status, stats, grid, s);
            break;
        default:
            throw Error(OMM_ERR_INVALID, "no pair kernel for this electrostatics / switching combination");
    }
}
}  // namespace

void launch_pairs(bool mixed, bool energy_on, const NlistDev& nl, const PairParams& p, const ParticleDev& part,
                  const double* pos, const SysInfo* sys_dev, long long* energy_fx, double* energy_d, unsigned* status, unsigned long long* stats, int grid, hipStream_t s) {
    const bool st = stats != nullptr;
    const int kind = p.elec | (p.switching ? PAIR_SWITCH : 0) | (p.ljpme ? PAIR_LJPME : 0);
    if (mixed)
        dispatch_kind<float, long long>(kind, st, energy_on, nl, p, part.qk.p, part.sh.p, part.e2.p, part, pos,
                                        sys_dev, energy_fx, status, stats, grid, s);
    else
        dispatch_kind<double, double>(kind, st, energy_on, nl, p, part.qk_d.p, part.sh_d.p, part.e2_d.p, part, pos,
                                      sys_dev, energy_d, status, stats, grid, s);
    OMM_HIP(hipGetLastError());
}

}  // namespace ommhip
