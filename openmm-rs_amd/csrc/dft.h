// The mesh's transforms on the matrix cores (systems of dft_system): each 1D
// transform is a dense product with the DFT matrix (v_mfma_f32_16x16x4_f32 or
// v_mfma_f64_16x16x4_f64, FP32 or FP64 throughout), so any length, prime or
// not, takes one pass over LDS without stages.
//
// Three launches transform, convolve and transform back.  The unit of work is
// a tile of DFT_COLS complex columns (kz values), 16 matrix columns: the real
// parts then the imaginary parts.
//   k_dft_zy: one workgroup per (x, tile): the plane's z transforms for the
//             tile's kz, then its y transforms;
//   k_dft_x : one workgroup per (ky, tile): forward x, influence, inverse x;
//   k_dft_yz: one workgroup per (x, 16 rows y): the inverse y transforms of
//             those rows, then their z transforms to real values.
// A plane is split over workgroups by output columns (or rows), which repeats
// reads of the plane (from L2) but no arithmetic, and gives 220 workgroups per
// pass at 55^3 where one per plane left most of the chip idle.  The half
// spectrum is kept as [tile][ky][x][16], so the x pass reads and writes
// contiguous runs.
//
// Bound: launch and load latency up to about 64 points per axis (three
// launches of 4-7 us at 55^3, 0.3 of it matrix-core issue), matrix-core issue
// and LDS reads above.  Transforms and convolution, FP32, serial launches,
// before (staged passes) and with these passes: 19^3 25 -> 15 us, 55^3 31 ->
// 22, 109^3 268 -> 81, 116^3 147 -> 102.
//
// FP32 accuracy (StepSum), relative RMS error of the mesh forces of water boxes
// with staged passes and with these: 37^3 8.50e-6, 8.23e-6; 55^3 1.31e-5, 1.32e-5;
// 96^3 1.31e-5, 1.32e-5; 116^3 1.56e-5, 1.55e-5; 120^3 1.92e-5, 1.91e-5 (10 to 24
// boxes each, 1% of scatter; the splines and the gather make up most of it).
// On 120 x 12 x 12 points, where the transforms show: 1.65e-6 and 1.47e-6.
#pragma once

#include "fmath.h"
#include "pme.h"

namespace ommhip {

template <class R>
struct Cx {
    R x, y;
};

// x / d and x mod d for 0 <= x < 2^20 and 1 <= d: a single-precision estimate
// of the quotient corrected by one step either way.
__device__ __forceinline__ int div_small(int x, int d, float inv_d) {
    int q = (int)((float)x * inv_d);
    if (q * d > x) --q;
    else if ((q + 1) * d <= x) ++q;
    return q;
}
__device__ __forceinline__ int mod_small(int x, int d, float inv_d) { return x - div_small(x, d, inv_d) * d; }

__device__ __forceinline__ double grid_real(long long v) { return (double)v * (1.0 / GRID_SCALE); }
__device__ __forceinline__ double grid_real(double v) { return v; }

// Influence function of the reciprocal convolution (pme.rs:332-372) at point
// (kx, ky, kz) of the half spectrum; zero at the origin except for the
// dispersion mesh.
//
// Dispersion mesh (pme.rs:358-362): I(k) = -pi^1.5 / (3 V B(k))
// (2 pi^3 sqrt(pi) erfc(b) k^3 + e^{-b^2} (alpha^3 - 2 alpha pi^2 k^2)),
// b = pi k / alpha, with the k = 0 term kept.
//
// The FP32 mesh serves force-only evaluations: the influence function in FP32
// (exp2 of the hardware), no energy.  The FP64 meshes evaluate it in FP64.
//
// The half spectrum stands for each point k and its mirror -k.  The reference
// sums the influence over the full grid and keeps the real part of the inverse
// transform, which is the half spectrum weighted by the mean influence of k
// and its mirror.  The mirror's frequency is -m on every axis except at a
// Nyquist index (2 k = n), where it is m itself; in a triclinic box |k|^2 then
// differs between the two, so those points take the mean of both influences.
template <class R>
struct Influence {
    const R *mod_x, *mod_y, *mod_z;
    int nx, ny, nz;
    bool tric, disp;
    R recip[9];
    // Coulomb: pref e^{-rate k^2} / (k^2 B), rate in units of ln 2 for FP32.
    R rate, pref;
    double dpref, dc1, dc2, da3, pi_a;
    static constexpr bool F32 = sizeof(R) == 4;

    __device__ __forceinline__ Influence(const SysInfo& S, const R* __restrict__ moduli) {
        mod_x = moduli + S.moduli_off[0];
        mod_y = moduli + S.moduli_off[1];
        mod_z = moduli + S.moduli_off[2];
        nx = S.grid[0];
        ny = S.grid[1];
        nz = S.grid[2];
        const Box& b = S.box;
        tric = b.triclinic != 0;
        disp = S.dispersion != 0;
        for (int k = 0; k < 9; ++k) recip[k] = (R)b.recip[k];
        const double pi2_a2 = PI * PI / (S.alpha * S.alpha);
        rate = F32 ? (R)(pi2_a2 * 1.4426950408889634) : (R)pi2_a2;
        pref = (R)(ONE_4PI_EPS0 / (PI * b.volume));
        dpref = -PI * sqrt(PI) / (3.0 * b.volume);
        dc1 = 2.0 * PI * PI * PI * sqrt(PI);
        da3 = S.alpha * S.alpha * S.alpha;
        dc2 = 2.0 * S.alpha * PI * PI;
        pi_a = PI / S.alpha;
    }
    __device__ __forceinline__ R at(R ax, R ay, R az, R mod) const {
        R k2 = 0;
        for (int a = 0; a < 3; ++a) {
            const R kv = ax * recip[a] + ay * recip[3 + a] + az * recip[6 + a];
            k2 += kv * kv;
        }
        if constexpr (F32) {
            if (disp) {
                const float kk = __builtin_sqrtf(k2);
                float ec, ex;
                Math<float>::erfc_exp((float)pi_a * kk, ec, ex);
                return (float)dpref * ((float)dc1 * ec * kk * k2 + ex * ((float)da3 - (float)dc2 * k2)) / mod;
            }
            return pref * __builtin_amdgcn_exp2f(-rate * k2) / (k2 * mod);
        } else {
            if (disp) {
                const double kk = sqrt(k2), bb = pi_a * kk;
                return dpref / mod * (dc1 * erfc(bb) * kk * k2 + exp(-bb * bb) * (da3 - dc2 * k2));
            }
            return pref * exp(-rate * k2) / (k2 * mod);
        }
    }
    __device__ __forceinline__ R operator()(int kx, int y, int kz) const {
        if (kx == 0 && y == 0 && kz == 0 && !disp) return (R)0;
        const R mx = (R)(kx < (nx + 1) / 2 ? kx : kx - nx);
        const R my = (R)(y < (ny + 1) / 2 ? y : y - ny);
        const R mz = (R)(kz < (nz + 1) / 2 ? kz : kz - nz);
        const R mod = mod_x[kx] * mod_y[y] * mod_z[kz];
        const R infl = at(mx, my, mz, mod);
        // Mirror signs: the mirror's frequency is -m except at a Nyquist index.
        if (!(tric && (2 * kx == nx || 2 * y == ny || 2 * kz == nz))) return infl;
        const int sx = 2 * kx == nx ? 1 : -1, sy = 2 * y == ny ? 1 : -1, sz = 2 * kz == nz ? 1 : -1;
        return (R)0.5 * (infl + at(-sx * mx, -sy * my, -sz * mz, mod));
    }
};

// Waves per workgroup (a template argument W): four, or eight where an axis has
// more than 64 points (more than four blocks of 16 rows).
constexpr int DFT_WAVES = 4, DFT_WAVES_WIDE = 8;
constexpr int DFT_W = 2 * DFT_COLS;  // matrix columns of a tile

// The system of this workgroup (si), its shape, and the workgroup's index in it.
#define DFT_LOCATE                                                    \
    int si = 0, local = blockIdx.x;                                   \
    MeshShape S = one;                                                \
    if (nsys > 1) {                                                   \
        si = find_sys(off, nsys, blockIdx.x);                         \
        local -= off[si];                                             \
        S = MeshShape::of(sys[si]);                                   \
    }

// A 16x16 block of the product in the accumulator registers of a wave: lane l
// holds column l % 16 of rows row(l, 0 .. 3); operands: lane l supplies
// A[l % 16][l / 16] and B[l / 16][l % 16] of each 16x4 by 4x16 step.
template <class R>
struct Mat;
template <>
struct Mat<float> {
    typedef float V4 __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ V4 mac(float a, float b, V4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int lane, int r) { return 4 * (lane >> 4) + r; }
};
template <>
struct Mat<double> {
    typedef double V4 __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ V4 mac(double a, double b, V4 c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int lane, int r) { return 4 * r + (lane >> 4); }
};

// The products step through their inner index four at a time, in pairs of
// steps whose LDS operands are loaded while the pair before them multiplies.
__host__ __device__ inline int round8(int n) { return (n + 7) & ~7; }

// Sum of the pairs of steps.  FP32: each pair is summed by itself and then added
// to the others, so that the rounding error of n terms grows as that of 8 + n/8
// (one chain had 2.5e-6 on the 120 points above).  The pair added is the one
// before the last, whose products are done.  FP64: one chain.
template <class R>
struct StepSum {
    using V4 = typename Mat<R>::V4;
    static constexpr bool BLOCKED = sizeof(R) == 4;
    V4 sum = {0, 0, 0, 0}, last = {0, 0, 0, 0};
    __device__ __forceinline__ V4 start() const {
        const V4 zero = {0, 0, 0, 0};
        return BLOCKED ? zero : last;
    }
    __device__ __forceinline__ void add(V4 pair) {
        if (BLOCKED) sum += last;
        last = pair;
    }
    __device__ __forceinline__ V4 total() const { return BLOCKED ? sum + last : last; }
};

// Rows row0 .. row0 + 15 of the complex DFT of one tile held in LDS as
// b[round8(n)][16] with zeros past row n.  roots[m] = e^{-2 pi i m / n}; sgn =
// +1 for the forward transform, -1 for the inverse.  With w = wr + i wi,
//   [Re | Im] of w (zr + i zi) = wr [zr | zi] + wi [-zi | zr],
// so both products accumulate into the same block.
template <class R>
__device__ __forceinline__ typename Mat<R>::V4 dft_rows(const R* b, int n, int row0, const Cx<R>* roots, R sgn) {
    const int lane = threadIdx.x & 63, c = lane & 15, kq = lane >> 4;
    const int row = row0 + c < n ? row0 + c : 0;  // rows past n are not stored
    const float inv_n = 1.0f / (float)n;
    int idx = mod_small(row * kq, n, inv_n);
    const int step = mod_small(4 * row, n, inv_n);
    const R* p = b + kq * DFT_W + c;
    const R* q = b + kq * DFT_W + (c ^ DFT_COLS);
    const R s = c < DFT_COLS ? -sgn : sgn;
    StepSum<R> total;
    Cx<R> w[2];
    R v[2], u[2];
    auto load = [&](int k) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            w[h] = roots[idx];
            v[h] = p[DFT_W * (k + 4 * h)];
            u[h] = q[DFT_W * (k + 4 * h)];
            idx += step;
            if (idx >= n) idx -= n;
        }
    };
    load(0);
    const int end = round8(n);
    for (int k = 8;; k += 8) {
        const Cx<R> w0 = w[0], w1 = w[1];
        const R v0 = v[0], v1 = v[1], u0 = s * u[0], u1 = s * u[1];
        if (k < end) load(k);
        typename Mat<R>::V4 acc = total.start();
        acc = Mat<R>::mac(w0.x, v0, acc);
        acc = Mat<R>::mac(w0.y, u0, acc);
        acc = Mat<R>::mac(w1.x, v1, acc);
        acc = Mat<R>::mac(w1.y, u1, acc);
        total.add(acc);
        if (k >= end) break;
    }
    return total.total();
}

// Every load of a workgroup is issued without a branch (indices past the end
// read the last element and are masked when stored to LDS): behind a branch the
// compiler waits for each load before the next.

// The roots of two axes (DFT_MAX at most each) into LDS, one load per thread.
template <class R>
__device__ __forceinline__ void load_roots(Cx<R>* a, int na, const Cx<R>* __restrict__ ra, Cx<R>* b, int nb,
                                           const Cx<R>* __restrict__ rb) {
    static_assert(64 * DFT_WAVES == 2 * DFT_MAX, "128 threads per axis");
    const int t = threadIdx.x & (DFT_MAX - 1);
    const bool first = threadIdx.x < DFT_MAX;
    const int n = first ? na : (threadIdx.x < 2 * DFT_MAX ? nb : 1);
    const Cx<R> v = (first ? ra : rb)[min(t, n - 1)];
    if (t < n && threadIdx.x < 2 * DFT_MAX) (first ? a : b)[t] = v;
}

// LDS layout in elements of R.
struct DftLds {
    static __host__ __device__ size_t stage_stride(int nz) { return (size_t)round8(nz) + 1; }
    static __host__ __device__ size_t zy(int ny, int nz, int waves) {
        return 2 * (size_t)(ny + nz) + (size_t)DFT_W * round8(ny) + waves * 16 * stage_stride(nz);
    }
    static __host__ __device__ size_t x(int nx) { return 2 * (size_t)nx + 2 * (size_t)DFT_W * round8(nx); }
    static __host__ __device__ size_t yz(int ny, int nz, int tiles, int waves) {
        return 2 * (size_t)(ny + nz) + waves * (size_t)DFT_W * round8(ny) + 16 * ((size_t)DFT_W * tiles + 1);
    }
};

template <int W, class R, class G>
__global__ __launch_bounds__(64 * W) void k_dft_zy(const int* __restrict__ off, int nsys,
                                                        const SysInfo* __restrict__ sys,
                                                        const G* __restrict__ qgrid, R* __restrict__ cgrid,
                                                        const Cx<R>* __restrict__ roots_all, MeshShape one, int* clear,
                                                        int nclear) {
    extern __shared__ unsigned char smem_raw[];
    // Clears the spread's bin counts, as the staged first pass does.
    if (clear)
        for (int i = blockIdx.x * (64 * W) + threadIdx.x; i < nclear; i += gridDim.x * (64 * W)) clear[i] = 0;
    DFT_LOCATE
    const int nx = S.grid[0], ny = S.grid[1], nz = S.grid[2];
    const int ntile = dft_tiles(S.nzh);
    const int x = local / ntile, tile = local - x * ntile;
    Cx<R>* rz = reinterpret_cast<Cx<R>*>(smem_raw);
    Cx<R>* ry = rz + nz;
    R* z = reinterpret_cast<R*>(ry + ny);
    const int zs = (int)DftLds::stage_stride(nz), nzp = round8(nz), nyp = round8(ny);
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, c = lane & 15, kq = lane >> 4;
    R* stage = z + DFT_W * nyp + wave * 16 * zs;
    load_roots(rz, nz, roots_all + S.roots_off[2], ry, ny, roots_all + S.roots_off[1]);
    const G* q = qgrid + S.qgrid_off + (size_t)x * ny * nz;
    const float inv_nz = 1.0f / (float)nz;
    const int kz = mod_small(tile * DFT_COLS + (c & (DFT_COLS - 1)), nz, inv_nz);
    const int step = mod_small(4 * kz, nz, inv_nz);
    bool roots_ready = false;
    for (int y0 = 16 * wave; y0 < nyp || !roots_ready; y0 += 16 * W) {
        for (int e = lane; e < nzp && y0 < nyp; e += 64) {
            G v[16];
            const G* qe = q + min(e, nz - 1);
#pragma unroll
            for (int r = 0; r < 16; ++r) v[r] = qe[min(y0 + r, ny - 1) * nz];
#pragma unroll
            for (int r = 0; r < 16; ++r) stage[r * zs + e] = e < nz && y0 + r < ny ? (R)grid_real(v[r]) : (R)0;
        }
        if (!roots_ready) {
            __syncthreads();
            roots_ready = true;
        } else {
            wave_lds_fence();
        }
        if (y0 >= nyp) break;
        // Column c < 8: sum_z q cos(2 pi z kz / nz), else its imaginary part.
        const R* w = reinterpret_cast<const R*>(rz) + (c >= DFT_COLS ? 1 : 0);
        StepSum<R> total;
        int idx = mod_small(kq * kz, nz, inv_nz);
        const R* a = stage + c * zs + kq;
        R av[2], wv[2];
        auto load = [&](int k) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                av[h] = a[k + 4 * h];
                wv[h] = w[2 * idx];
                idx += step;
                if (idx >= nz) idx -= nz;
            }
        };
        load(0);
        for (int k = 8;; k += 8) {
            const R a0 = av[0], a1 = av[1], w0 = wv[0], w1 = wv[1];
            if (k < nzp) load(k);
            typename Mat<R>::V4 acc = total.start();
            acc = Mat<R>::mac(a0, w0, acc);
            acc = Mat<R>::mac(a1, w1, acc);
            total.add(acc);
            if (k >= nzp) break;
        }
        const typename Mat<R>::V4 acc = total.total();
        for (int r = 0; r < 4; ++r) {
            const int y = y0 + Mat<R>::row(lane, r);
            if (y < nyp) z[y * DFT_W + c] = acc[r];  // rows past ny are zero
        }
        wave_lds_fence();
    }
    __syncthreads();
    R* out = cgrid + 2 * S.cgrid_off + ((size_t)tile * ny * nx + x) * DFT_W + c;
    for (int k0 = 16 * wave; k0 < ny; k0 += 16 * W) {
        const typename Mat<R>::V4 acc = dft_rows<R>(z, ny, k0, ry, (R)1);
        for (int r = 0; r < 4; ++r) {
            const int ky = k0 + Mat<R>::row(lane, r);
            if (ky < ny) out[(size_t)ky * nx * DFT_W] = acc[r];
        }
    }
}

template <int W, class R, class G, class A>
__global__ __launch_bounds__(64 * W) void k_dft_x(const int* __restrict__ off, int nsys,
                                                       const SysInfo* __restrict__ sys, G* __restrict__ qgrid,
                                                       R* __restrict__ cgrid, const Cx<R>* __restrict__ roots_all,
                                                       const R* __restrict__ moduli_all, MeshShape one, A* energy,
                                                       unsigned* status) {
    extern __shared__ unsigned char smem_raw[];
    DFT_LOCATE
    const int nx = S.grid[0], ny = S.grid[1], nz = S.grid[2], nzh = S.nzh;
    const int tile = local / ny, ky = local - tile * ny;  // local = tile * ny + ky
    Cx<R>* rx = reinterpret_cast<Cx<R>*>(smem_raw);
    const int nxp = round8(nx);
    R* s = reinterpret_cast<R*>(rx + nx);
    R* t = s + DFT_W * nxp;
    R* line = cgrid + 2 * S.cgrid_off + (size_t)local * nx * DFT_W;
    {
        const Cx<R> w = roots_all[S.roots_off[0] + min((int)threadIdx.x, nx - 1)];
        for (int i0 = threadIdx.x; i0 < DFT_W * nxp; i0 += 4 * (64 * W)) {
            R v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) v[u] = line[min(i0 + u * (64 * W), DFT_W * nx - 1)];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int i = i0 + u * (64 * W);
                if (i < DFT_W * nxp) s[i] = i < DFT_W * nx ? v[u] : (R)0;
            }
        }
        if (threadIdx.x < nx) rx[threadIdx.x] = w;
    }
    // The charge grid is zero between runs: this pass, after every read of it,
    // clears the system's points, an equal share per workgroup.
    {
        const int plane = nx * nz, share = (plane + dft_tiles(nzh) - 1) / dft_tiles(nzh);
        G* g = qgrid + S.qgrid_off + ky * plane;
        for (int i = tile * share + threadIdx.x; i < min(plane, (tile + 1) * share); i += (64 * W)) g[i] = (G)0;
    }
    __syncthreads();
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, c = lane & 15;
    const int kz = tile * DFT_COLS + (c & (DFT_COLS - 1));
    const Influence<R> I(sys[si], moduli_all);
    constexpr bool ENERGY = sizeof(R) == 8;
    __shared__ double s_e[DFT_MAX / 16];  // energy of each block of 16 rows
    for (int k0 = 16 * wave; k0 < nxp; k0 += 16 * W) {
        double eacc = 0.0;
        const typename Mat<R>::V4 acc = dft_rows<R>(s, nx, k0, rx, (R)1);
        // The real and the imaginary column of a point share its influence:
        // each of the two lanes evaluates half of the rows.
        R mine[2], infl[4];
        const bool im = c >= DFT_COLS;
        for (int h = 0; h < 2; ++h) {
            const int kx = k0 + Mat<R>::row(lane, (im ? 2 : 0) + h);
            mine[h] = kx < nx && kz < nzh ? I(kx, ky, kz) : (R)0;
        }
        for (int h = 0; h < 2; ++h) {
            const R other = __shfl_xor(mine[h], DFT_COLS, 64);
            infl[h] = im ? other : mine[h];
            infl[2 + h] = im ? mine[h] : other;
        }
        for (int r = 0; r < 4; ++r) {
            const int kx = k0 + Mat<R>::row(lane, r);
            // Rows past nx hold a repeated row; their influence is zero.
            const R v = kx < nx ? acc[r] : (R)0;
            if (ENERGY) {
                const double wz = (kz == 0 || 2 * kz == nz) ? 1.0 : 2.0;
                eacc += wz * 0.5 * (double)infl[r] * ((double)v * v);
            }
            if (kx < nxp) t[kx * DFT_W + c] = v * infl[r];
        }
        if (ENERGY) {
            const double et = wave_sum(eacc);
            if (lane == 0) s_e[k0 >> 4] = et;
        }
    }
    __syncthreads();
    if (ENERGY && threadIdx.x == 0) {
        // One add per workgroup (the adds to one address serialise), summed in
        // an order that does not depend on W.
        double et = 0.0;
        for (int k = 0; 16 * k < nxp; ++k) et += s_e[k];
        acc_add(energy + si * E_SLOTS + E_RECIP, et, ENERGY_SCALE, status);
    }
    for (int x0 = 16 * wave; x0 < nx; x0 += 16 * W) {
        const typename Mat<R>::V4 acc = dft_rows<R>(t, nx, x0, rx, (R)-1);
        for (int r = 0; r < 4; ++r) {
            const int x = x0 + Mat<R>::row(lane, r);
            if (x < nx) line[x * DFT_W + c] = acc[r];
        }
    }
}

template <int W, class R>
__global__ __launch_bounds__(64 * W) void k_dft_yz(const int* __restrict__ off, int nsys,
                                                        const SysInfo* __restrict__ sys, const R* __restrict__ cgrid,
                                                        R* __restrict__ phi, const Cx<R>* __restrict__ roots_all,
                                                        MeshShape one) {
    extern __shared__ unsigned char smem_raw[];
    DFT_LOCATE
    const int nx = S.grid[0], ny = S.grid[1], nz = S.grid[2], nzh = S.nzh;
    const int ntile = dft_tiles(nzh), nrow = (ny + 15) / 16;
    const int x = local / nrow, y0 = 16 * (local - x * nrow);
    const int nyp = round8(ny);
    Cx<R>* rz = reinterpret_cast<Cx<R>*>(smem_raw);
    Cx<R>* ry = rz + nz;
    R* v = reinterpret_cast<R*>(ry + ny);
    const int vs = DFT_W * ntile + 1;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, c = lane & 15, kq = lane >> 4;
    R* stage = v + 16 * vs + wave * DFT_W * nyp;
    load_roots(rz, nz, roots_all + S.roots_off[2], ry, ny, roots_all + S.roots_off[1]);
    const R* in = cgrid + 2 * S.cgrid_off + (size_t)x * DFT_W;
    bool roots_ready = false;
    for (int tile = wave; tile < ntile || !roots_ready; tile += W) {
        if (tile < ntile) {
            const R* p = in + (size_t)tile * ny * nx * DFT_W;
            constexpr int AT_ONCE = 8;  // loads in flight
            for (int e0 = lane; e0 < DFT_W * nyp; e0 += 64 * AT_ONCE) {
                R t[AT_ONCE];
#pragma unroll
                for (int u = 0; u < AT_ONCE; ++u) {
                    const int ky = (e0 + 64 * u) / DFT_W;
                    t[u] = p[min(ky, ny - 1) * nx * DFT_W + c];
                }
#pragma unroll
                for (int u = 0; u < AT_ONCE; ++u) {
                    const int e = e0 + 64 * u;
                    if (e < DFT_W * nyp) stage[e] = e < DFT_W * ny ? t[u] : (R)0;
                }
            }
        }
        if (!roots_ready) {
            __syncthreads();
            roots_ready = true;
        } else {
            wave_lds_fence();
        }
        if (tile >= ntile) break;
        const typename Mat<R>::V4 acc = dft_rows<R>(stage, ny, y0, ry, (R)-1);
        for (int r = 0; r < 4; ++r) v[Mat<R>::row(lane, r) * vs + tile * DFT_W + c] = acc[r];
        wave_lds_fence();
    }
    __syncthreads();
    const float inv_nz = 1.0f / (float)nz;
    // phi(z) = sum over the full spectrum's kz of Re(V e^{2 pi i z kz / nz}):
    // kz = 0 and the Nyquist column once, the others twice (their mirrors).
    for (int z0 = 16 * wave; z0 < nz; z0 += 16 * W) {
        const int z = z0 + c < nz ? z0 + c : 0;
        int idx = mod_small(z * kq, nz, inv_nz);
        const int step = mod_small(4 * z, nz, inv_nz);
        StepSum<R> total;
        const R* a = v + c * vs + kq;
        Cx<R> w[2];
        R re[2], im[2];
        auto load = [&](int g) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int kz = g * DFT_COLS + 4 * h + kq;
                const R cw = kz >= nzh ? (R)0 : (kz == 0 || 2 * kz == nz ? (R)1 : (R)2);
                w[h] = rz[idx];
                re[h] = cw * a[g * DFT_W + 4 * h];
                im[h] = cw * a[g * DFT_W + DFT_COLS + 4 * h];
                idx += step;
                if (idx >= nz) idx -= nz;
            }
        };
        load(0);
        for (int g = 1;; ++g) {
            const Cx<R> w0 = w[0], w1 = w[1];
            const R r0 = re[0], r1 = re[1], i0 = im[0], i1 = im[1];
            if (g < ntile) load(g);
            typename Mat<R>::V4 acc = total.start();
            acc = Mat<R>::mac(r0, w0.x, acc);
            acc = Mat<R>::mac(i0, w0.y, acc);
            acc = Mat<R>::mac(r1, w1.x, acc);
            acc = Mat<R>::mac(i1, w1.y, acc);
            total.add(acc);
            if (g >= ntile) break;
        }
        const typename Mat<R>::V4 acc = total.total();
        for (int r = 0; r < 4; ++r) {
            const int y = y0 + Mat<R>::row(lane, r);
            if (y < ny && z0 + c < nz) phi[S.qgrid_off + ((size_t)x * ny + y) * nz + z0 + c] = acc[r];
        }
    }
}

}  // namespace ommhip
