// Spread of charges in no spatial order on an FP64 grid, one workgroup per x
// plane: the workgroup lists the charges whose stencils meet its plane, then
// sums their 25 points each in LDS.  No device atomics (125 a charge, each on a
// cache line of its own, bound the spread by charge: 3,000 charges 22 us), at the
// price of every workgroup reading every position: 3,000 charges 8 us.
#pragma once

#include "spline.h"

namespace ommhip {

constexpr int CHARGE_PLANE_THREADS = 1024;
constexpr int PLANE_POINTS = 6144;   // points of the largest plane
// Every plane reads every position, so the planes pay up to a product of planes and
// charges: by planes and by tiles, whole calls in microseconds, 16,000 charges on 30
// planes 134, 199; 60,000 on 64 363, 401; 60,000 on 512 (3.1e7) 576, 611; 32,000 on
// 1,000 (3.2e7) 357, 363; but 60,000 on 1,000 (6e7) 507, 488.
constexpr long long PLANE_WORK = 40000000;
constexpr bool planes_pay(int planes, int charges) { return (long long)planes * charges <= PLANE_WORK; }
// Charges of the allocation-free mesh (at most 64 planes), which has no tiles to change to.
constexpr int PLANE_CHARGES = 65536;

// s_plane[y * dims[2] + z] receives plane x (all threads of the workgroup call;
// they may read it on return).
__device__ __forceinline__ void spread_plane(int x, int n, const double* __restrict__ pos,
                                             const double* __restrict__ charge, const Box& b, const int dims[3],
                                             double* s_plane) {
    constexpr int BATCH = 4 * CHARGE_PLANE_THREADS;
    __shared__ unsigned short s_list[BATCH];
    __shared__ int s_count;
    const int t = threadIdx.x;
    for (int i = t; i < dims[1] * dims[2]; i += CHARGE_PLANE_THREADS) s_plane[i] = 0.0;
    for (int first = 0; first < n; first += BATCH) {
        if (t == 0) s_count = 0;
        __syncthreads();
#pragma unroll
        for (int k = 0; k < BATCH; k += CHARGE_PLANE_THREADS) {
            const int a = first + k + t, a0 = min(a, n - 1);
            const double p[3] = {pos[3 * (size_t)a0], pos[3 * (size_t)a0 + 1], pos[3 * (size_t)a0 + 2]};
            int ix = x - stencil_base(p, b, 0, dims[0]);
            if (ix < 0) ix += dims[0];
            if (a < n && ix < 5 && charge[a0] != 0.0) s_list[atomicAdd(&s_count, 1)] = (unsigned short)(k + t);
        }
        __syncthreads();
        const int count = s_count;
        for (int i = t; i < count; i += CHARGE_PLANE_THREADS) {
            const size_t a = (size_t)first + s_list[i];
            const double p[3] = {pos[3 * a], pos[3 * a + 1], pos[3 * a + 2]}, q = charge[a];
            int idx[3];
            double w[3][5], dw[3][5];
            stencil<double>(p, b, dims, idx, w, dw);
            int ix = x - idx[0];
            if (ix < 0) ix += dims[0];
            const double wx = pick(w[0], ix);
#pragma unroll
            for (int iy = 0; iy < 5; ++iy) {
                int y = idx[1] + iy;
                if (y >= dims[1]) y -= dims[1];
                const double qw = q * wx * w[1][iy];
#pragma unroll
                for (int iz = 0; iz < 5; ++iz) {
                    int z = idx[2] + iz;
                    if (z >= dims[2]) z -= dims[2];
                    atomicAdd(s_plane + y * dims[2] + z, qw * w[2][iz]);
                }
            }
        }
        __syncthreads();
    }
    if (n <= 0) __syncthreads();
}

// sum_p phi_p w_x w_y w_z at the stencil of the position p, by eight consecutive
// lanes (lane j < 5 takes the x plane j); every one of them has the sum.
__device__ __forceinline__ double potential_at(const double* __restrict__ p, const Box& b, const int dims[3],
                                               const double* __restrict__ phi, size_t plane_stride) {
    const int j = threadIdx.x & 7;
    const double x[3] = {p[0], p[1], p[2]};
    int idx[3];
    double w[3][5], dw[3][5];
    stencil<double>(x, b, dims, idx, w, dw);
    int gx = idx[0] + min(j, 4);
    if (gx >= dims[0]) gx -= dims[0];
    const double* plane = phi + (size_t)gx * plane_stride;
    double sum = 0.0;
#pragma unroll
    for (int iy = 0; iy < 5; ++iy) {
        int y = idx[1] + iy;
        if (y >= dims[1]) y -= dims[1];
        double r = 0.0;
#pragma unroll
        for (int iz = 0; iz < 5; ++iz) {
            int z = idx[2] + iz;
            if (z >= dims[2]) z -= dims[2];
            r += plane[(size_t)y * dims[2] + z] * w[2][iz];
        }
        sum += r * w[1][iy];
    }
    sum = j < 5 ? sum * pick(w[0], j) : 0.0;
    for (int o = 1; o < 8; o <<= 1) sum += __shfl_xor(sum, o, 64);
    return sum;
}

}  // namespace ommhip
