// The charge-mesh derivatives of PmeCache::charge_derivatives (pme.rs:88-138)
// for callers that cannot allocate device memory (code under HIP graph
// capture, tight serving loops): inputs and outputs are the caller's device
// buffers, every launch goes to the caller's stream, and the only other memory
// is the file-scope `scratch` array below, one FP64 complex grid of at most
// NM_MAX_POINTS points per device, held until the process ends.
//
// The mesh is the reference's algorithm: spread of the charges with order-5
// B-splines, forward transform along z, y and x (direct DFTs, roots from
// sincospi), the influence function with the B-spline moduli (pme.rs:239-259
// and 332-372, k = 0 cleared), the unnormalised inverse transform, and the
// potential at each listed particle's stencil added to its derivative.  All
// FP64, on the half spectrum kz <= nz/2.
//
// Four launches, each bound by its latency: spread, z and y lines of an x plane
// by one workgroup; the x lines, the influence function and the x lines back by
// groups of columns; y and z lines of a plane back; the potentials.  As ten
// launches over the full complex grid a call of 900 particles took 47.5 us, now 23.
//
// Plane x of the scratch array holds the half spectrum of that plane, ny rows of
// nzh complex values, or its ny rows of nz real ones (charges, potential).
#include <hip/hip_runtime.h>

#include <cmath>
#include <mutex>

#include "../../include/ommhip.h"
#include "plane_spread.h"
#include "spline.h"

namespace ommhip {
namespace {

constexpr int NM_MAX_EDGE = 64;
constexpr long long NM_MAX_POINTS = (long long)NM_MAX_EDGE * NM_MAX_EDGE * NM_MAX_EDGE;
constexpr int NM_MAX_DEVICES = 64;

}  // namespace
}  // namespace ommhip

// One grid per device: 64^3 FP64 complex values, 4 MiB.
static __device__ __align__(256) double2 scratch[ommhip::NM_MAX_POINTS];

namespace ommhip {
namespace {

std::mutex g_scratch_mutex;
double2* g_scratch[NM_MAX_DEVICES] = {};

// The device address of `scratch` on the current device, looked up once per
// device (each device holds its own copy of the array at its own address).
double2* scratch_ptr() {
    int dev = 0;
    OMM_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= NM_MAX_DEVICES) throw Error(OMM_ERR_DEVICE, "device index out of range");
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch[dev]) {
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            throw Error(OMM_ERR_DEVICE, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
        g_scratch[dev] = static_cast<double2*>(p);
    }
    return g_scratch[dev];
}

struct NmGrid {
    int n[3], nzh;
    __host__ __device__ size_t plane() const { return (size_t)n[1] * nzh; }  // complex values of a plane
};
constexpr int NM_HALF = NM_MAX_EDGE / 2 + 1, NM_PER = (NM_MAX_EDGE * NM_HALF + CHARGE_PLANE_THREADS - 1) / CHARGE_PLANE_THREADS;
static_assert(NM_MAX_EDGE * NM_MAX_EDGE <= PLANE_POINTS, "a plane of the largest grid");
static_assert((long long)NM_MAX_EDGE * NM_MAX_EDGE * NM_HALF <= NM_MAX_POINTS, "the half spectrum fits");

__global__ void k_nm_clear(double2* g, size_t count) {
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < count; i += (size_t)gridDim.x * blockDim.x)
        g[i] = make_double2(0.0, 0.0);
}

// Spread (pme.rs:315-330) of more than PLANE_CHARGES particles: five threads per
// particle, one per x plane of its stencil; uncharged particles do not spread.
__global__ void k_nm_spread(int n, const double* __restrict__ pos, const double* __restrict__ charge, Box b,
                            NmGrid G, double2* g) {
    const long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x;
    if (t >= 5LL * n) return;
    const int a = (int)(t / 5), ix = (int)(t - 5LL * a);
    const double q = charge[a];
    if (q == 0.0) return;
    int base[3];
    double w[3][5], dw[3][5];
    stencil<double>(pos + 3 * (size_t)a, b, G.n, base, w, dw);
    const int gx = (base[0] + ix) % G.n[0];
    const double wx = pick(w[0], ix);
    double* plane = reinterpret_cast<double*>(g + gx * G.plane());
    for (int iy = 0; iy < 5; ++iy) {
        double* row = plane + (base[1] + iy) % G.n[1] * G.n[2];
        for (int iz = 0; iz < 5; ++iz) atomicAdd(&row[(base[2] + iz) % G.n[2]], q * wx * w[1][iy] * w[2][iz]);
    }
}

// e^{-2 pi i k / n} for k < n.
__device__ __forceinline__ void nm_roots(double2* root, int n) {
    if ((int)threadIdx.x < n) {
        double s, c;
        sincospi(2.0 * threadIdx.x / n, &s, &c);
        root[threadIdx.x] = make_double2(c, -s);
    }
}

// Plane x: its charges, then the z lines (real to half spectrum) and the y lines.
// SPREAD: from the particles; otherwise the plane's charges are in the array.
template <bool SPREAD>
__global__ __launch_bounds__(CHARGE_PLANE_THREADS) void k_nm_forward(int n, const double* __restrict__ pos,
                                                              const double* __restrict__ charge, Box b, NmGrid G,
                                                              double2* g) {
    __shared__ double2 s_c[NM_MAX_EDGE * NM_HALF], s_rz[NM_MAX_EDGE], s_ry[NM_MAX_EDGE];
    double* s_r = reinterpret_cast<double*>(s_c);
    const int t = threadIdx.x, ny = G.n[1], nz = G.n[2], nzh = G.nzh;
    double2* plane = g + blockIdx.x * G.plane();
    nm_roots(s_rz, nz);
    nm_roots(s_ry, ny);
    if constexpr (SPREAD) {
        spread_plane(blockIdx.x, n, pos, charge, b, G.n, s_r);
    } else {
        for (int i = t; i < ny * nz; i += CHARGE_PLANE_THREADS) s_r[i] = reinterpret_cast<const double*>(plane)[i];
        __syncthreads();
    }
    double2 v[NM_PER];
#pragma unroll
    for (int k = 0; k < NM_PER; ++k) {
        const int i = t + k * CHARGE_PLANE_THREADS;
        if (i >= ny * nzh) break;
        const int y = i / nzh, kz = i - y * nzh;
        const double* line = s_r + y * nz;
        double re = 0.0, im = 0.0;
        int at = 0;
        for (int z = 0; z < nz; ++z) {
            const double2 w = s_rz[at];
            re += line[z] * w.x;
            im += line[z] * w.y;
            at += kz;
            if (at >= nz) at -= nz;
        }
        v[k] = make_double2(re, im);
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NM_PER; ++k) {
        const int i = t + k * CHARGE_PLANE_THREADS;
        if (i < ny * nzh) s_c[i] = v[k];
    }
    __syncthreads();
    for (int i = t; i < ny * nzh; i += CHARGE_PLANE_THREADS) {
        const int ky = i / nzh, kz = i - ky * nzh;
        double re = 0.0, im = 0.0;
        int at = 0;
        for (int y = 0; y < ny; ++y) {
            const double2 w = s_ry[at], c = s_c[y * nzh + kz];
            re += c.x * w.x - c.y * w.y;
            im += c.x * w.y + c.y * w.x;
            at += ky;
            if (at >= ny) at -= ny;
        }
        plane[i] = make_double2(re, im);
    }
}

// Plane x back: the y lines, then the z lines from the half spectrum.
__global__ __launch_bounds__(CHARGE_PLANE_THREADS) void k_nm_backward(NmGrid G, double2* g) {
    __shared__ double2 s_c[NM_MAX_EDGE * NM_HALF], s_rz[NM_MAX_EDGE], s_ry[NM_MAX_EDGE];
    const int t = threadIdx.x, ny = G.n[1], nz = G.n[2], nzh = G.nzh;
    double2* plane = g + blockIdx.x * G.plane();
    nm_roots(s_rz, nz);
    nm_roots(s_ry, ny);
    for (int i = t; i < ny * nzh; i += CHARGE_PLANE_THREADS) s_c[i] = plane[i];
    __syncthreads();
    double2 v[NM_PER];
#pragma unroll
    for (int k = 0; k < NM_PER; ++k) {
        const int i = t + k * CHARGE_PLANE_THREADS;
        if (i >= ny * nzh) break;
        const int y = i / nzh, kz = i - y * nzh;
        double re = 0.0, im = 0.0;
        int at = 0;
        for (int ky = 0; ky < ny; ++ky) {
            const double2 w = s_ry[at], c = s_c[ky * nzh + kz];
            re += c.x * w.x + c.y * w.y;
            im += c.y * w.x - c.x * w.y;
            at += y;
            if (at >= ny) at -= ny;
        }
        v[k] = make_double2(re, im);
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NM_PER; ++k) {
        const int i = t + k * CHARGE_PLANE_THREADS;
        if (i < ny * nzh) s_c[i] = v[k];
    }
    __syncthreads();
    double* phi = reinterpret_cast<double*>(plane);
    for (int i = t; i < ny * nz; i += CHARGE_PLANE_THREADS) {
        const int y = i / nz, z = i - y * nz;
        const double2* line = s_c + y * nzh;
        double sum = 0.0;
        int at = z;
        for (int kz = 1; kz < (nz + 1) / 2; ++kz) {
            const double2 w = s_rz[at], c = line[kz];
            sum += c.x * w.x + c.y * w.y;
            at += z;
            if (at >= nz) at -= nz;
        }
        sum = 2.0 * sum + line[0].x;
        if (nz % 2 == 0) sum += z % 2 == 0 ? line[nz / 2].x : -line[nz / 2].x;
        phi[i] = sum;
    }
}

// |sum_i M5(i+1) e^{2 pi i k i / n}|^2 (pme.rs:239-259) before the
// replacement of near-zero values.
__device__ double nm_modulus_raw(int k, int n) {
    const double m5[4] = {1.0 / 24.0, 11.0 / 24.0, 11.0 / 24.0, 1.0 / 24.0};
    double re = 0.0, im = 0.0;
    for (int i = 0; i < 4; ++i) {
        double s, c;
        sincospi(2.0 * (double)((long long)k * i % n) / n, &s, &c);
        re += m5[i] * c;
        im += m5[i] * s;
    }
    return re * re + im * im;
}

__device__ double nm_modulus(int k, int n) {
    const double v = nm_modulus_raw(k, n);
    if (v >= 1e-7) return v;
    return 0.5 * (nm_modulus_raw((k + n - 1) % n, n) + nm_modulus_raw((k + 1) % n, n));
}

// The x lines of NM_COLS columns (ky, kz), times the influence function
// (pme.rs:332-372, k = 0 cleared), and back.
constexpr int NM_COLS = 4;

__global__ __launch_bounds__(NM_COLS* NM_MAX_EDGE) void k_nm_convolve(NmGrid G, Box b, double alpha, double2* g) {
    __shared__ double2 s_c[NM_MAX_EDGE][NM_COLS], s_root[NM_MAX_EDGE];
    __shared__ double s_mx[NM_MAX_EDGE], s_my[NM_COLS], s_mz[NM_COLS];
    const int t = threadIdx.x, c = t % NM_COLS, x = t / NM_COLS, nx = G.n[0];
    const int columns = (int)G.plane(), column = blockIdx.x * NM_COLS + c;
    const bool mine = x < nx && column < columns;
    const int ky = min(column, columns - 1) / G.nzh, kz = min(column, columns - 1) - ky * G.nzh;
    nm_roots(s_root, nx);
    if (t < nx) s_mx[t] = nm_modulus(t, nx);
    else if (x == NM_MAX_EDGE - 1) s_my[c] = nm_modulus(ky, G.n[1]);
    if (x == NM_MAX_EDGE - 2) s_mz[c] = nm_modulus(kz, G.n[2]);
    if (mine) s_c[x][c] = g[x * G.plane() + column];
    __syncthreads();
    double2 v = make_double2(0.0, 0.0);
    if (mine) {
        int at = 0;
        for (int k = 0; k < nx; ++k) {
            const double2 w = s_root[at], u = s_c[k][c];
            v.x += u.x * w.x - u.y * w.y;
            v.y += u.x * w.y + u.y * w.x;
            at += x;
            if (at >= nx) at -= nx;
        }
        const double m[3] = {(double)(x < (nx + 1) / 2 ? x : x - nx),
                             (double)(ky < (G.n[1] + 1) / 2 ? ky : ky - G.n[1]),
                             (double)(kz < (G.n[2] + 1) / 2 ? kz : kz - G.n[2])};
        const double mod = s_mx[x] * s_my[c] * s_mz[c];
        const double pi2_a2 = PI * PI / (alpha * alpha), pref = ONE_4PI_EPS0 / (PI * b.volume);
        auto influence = [&](double m0, double m1, double m2) {
            double k2 = 0.0;
            for (int a = 0; a < 3; ++a) {
                const double kv = m0 * b.recip[a] + m1 * b.recip[3 + a] + m2 * b.recip[6 + a];
                k2 += kv * kv;
            }
            return pref * exp(-pi2_a2 * k2) / (k2 * mod);
        };
        double infl = x == 0 && column == 0 ? 0.0 : influence(m[0], m[1], m[2]);
        // The point -k of the full grid has the index -n/2 as well where k has
        // it; the real part of the inverse takes the mean of the two.
        if (2 * x == nx || 2 * ky == G.n[1] || 2 * kz == G.n[2])
            infl = 0.5 * (infl + influence(2 * x == nx ? -m[0] : m[0], 2 * ky == G.n[1] ? -m[1] : m[1],
                                           2 * kz == G.n[2] ? -m[2] : m[2]));
        v.x *= infl;
        v.y *= infl;
    }
    __syncthreads();
    if (mine) s_c[x][c] = v;
    __syncthreads();
    if (!mine) return;
    v = make_double2(0.0, 0.0);
    int at = 0;
    for (int k = 0; k < nx; ++k) {
        const double2 w = s_root[at], u = s_c[k][c];
        v.x += u.x * w.x + u.y * w.y;
        v.y += u.y * w.x - u.x * w.y;
        at += x;
        if (at >= nx) at -= nx;
    }
    g[x * G.plane() + column] = v;
}

// derivatives[k] += the potential at the stencil of particle atoms[k]
// (pme.rs:117-137); an index outside [0, n) gives NaN.
// Eight lanes per listed particle.
__global__ __launch_bounds__(256) void k_nm_potential(int count, const int* __restrict__ atoms, int n,
                                                      const double* __restrict__ pos, Box b, NmGrid G,
                                                      const double2* __restrict__ g, double* out) {
    const int k = (blockIdx.x * blockDim.x + threadIdx.x) / 8;
    if (k >= count) return;  // all eight lanes
    const int a = atoms[k];
    if (a < 0 || a >= n) {
        if ((threadIdx.x & 7) == 0) out[k] = __longlong_as_double(0x7ff8000000000000ll);
        return;
    }
    const double v = potential_at(pos + 3 * (size_t)a, b, G.n, reinterpret_cast<const double*>(g), 2 * G.plane());
    if ((threadIdx.x & 7) == 0) out[k] += v;
}

}  // namespace
}  // namespace ommhip

using ommhip::Error;

extern "C" omm_status omm_pme_charge_derivatives_noalloc(int32_t num_particles, const double* pos,
                                                         const double* charges, const double* box, double alpha,
                                                         const int32_t grid[3], const int32_t* indices, int32_t count,
                                                         double* derivatives, void* stream) {
    return ommhip::guarded([&]() -> omm_status {
        using namespace ommhip;
        if (num_particles < 0 || count < 0) throw Error(OMM_ERR_INVALID, "negative particle or index count");
        if (!box || !grid) throw Error(OMM_ERR_INVALID, "null box or grid");
        if (num_particles > 0 && (!pos || !charges)) throw Error(OMM_ERR_INVALID, "null positions or charges");
        if (count > 0 && (!indices || !derivatives)) throw Error(OMM_ERR_INVALID, "null indices or derivatives");
        if (!(std::isfinite(alpha) && alpha > 0.0)) throw Error(OMM_ERR_INVALID, "alpha must be positive and finite");
        for (int a = 0; a < 3; ++a)
            if (grid[a] < 5 || grid[a] > NM_MAX_EDGE)
                throw Error(OMM_ERR_INVALID, "grid dimensions must lie in [5, 64] for the allocation-free mesh");
        validate_box(box);
        if (count == 0) return OMM_OK;
        const Box b = make_box(box);
        const NmGrid G{{grid[0], grid[1], grid[2]}, grid[2] / 2 + 1};
        hipStream_t s = static_cast<hipStream_t>(stream);
        double2* g = scratch_ptr();
        if (num_particles <= PLANE_CHARGES) {
            hipLaunchKernelGGL(k_nm_forward<true>, dim3(grid[0]), dim3(CHARGE_PLANE_THREADS), 0, s, num_particles, pos,
                               charges, b, G, g);
        } else {
            hipLaunchKernelGGL(k_nm_clear, dim3(1024), dim3(256), 0, s, g, grid[0] * G.plane());
            hipLaunchKernelGGL(k_nm_spread, dim3((unsigned)((5LL * num_particles + 255) / 256)), dim3(256), 0, s,
                               num_particles, pos, charges, b, G, g);
            hipLaunchKernelGGL(k_nm_forward<false>, dim3(grid[0]), dim3(CHARGE_PLANE_THREADS), 0, s, num_particles, pos,
                               charges, b, G, g);
        }
        hipLaunchKernelGGL(k_nm_convolve, dim3((unsigned)((G.plane() + NM_COLS - 1) / NM_COLS)),
                           dim3(NM_COLS * NM_MAX_EDGE), 0, s, G, b, alpha, g);
        hipLaunchKernelGGL(k_nm_backward, dim3(grid[0]), dim3(CHARGE_PLANE_THREADS), 0, s, G, g);
        hipLaunchKernelGGL(k_nm_potential, dim3((unsigned)((count + 31) / 32)), dim3(256), 0, s, count, indices,
                           num_particles, pos, b, G, g, derivatives);
        OMM_HIP(hipGetLastError());
        return OMM_OK;
    });
}
