// Smooth PME on the device: B-spline spread into a fixed-point (mixed) or
// FP64 (plain) grid, a real-to-complex 3D FFT as three passes of batched 1D
// mixed-radix Stockham transforms held in LDS, the reciprocal convolution and
// its energy fused into the x pass (forward x, multiply, inverse x in one
// kernel), the inverse passes and the force gather.
//
// The reference transforms the full complex grid (pme.rs:271-303) and sums the
// energy over all of it (pme.rs:339-372); for a real charge grid S(-k) =
// conj(S(k)) and the influence function is even, so the half spectrum
// kz <= nz/2 with weights 1 (kz = 0, nz/2) and 2 (otherwise) carries the same
// sum.  Any grid size is supported: radices are the prime factors of n (8 and
// 4 preferred), each stage a direct DFT of its radix.
#include <climits>
#include <cmath>
#include <complex>
#include <type_traits>

#include "dft.h"
#include "fmath.h"
#include "pme.h"
#include "plane_spread.h"
#include "spline.h"

namespace ommhip {

namespace {

constexpr int FFT_THREADS = 256;

// Spread without atomics on the grid.  The grid of every system is cut into tiles
// of ptile = 8 or 6 points per axis (the last tile of an axis takes the
// remainder, so tile widths lie in [4, 11]; smaller tiles give small grids
// more workgroups).  Each step, k_pme_bin computes every charged atom's
// stencil (base point and weights, stored per atom) and appends the atom to
// the bin of the tile holding its base point.  An atom's 5-point stencil then
// only reaches its own tile and the next one along each axis, so the points
// of tile T receive contributions from the bins of T and of the tiles before
// it: at most 8 bins.  k_spread_tiles runs one workgroup per tile, sums those
// contributions in LDS (fixed point: the order of the adds does not matter)
// and writes every point of the tile with plain stores.  Each point has one
// owner, and the whole grid is overwritten.
constexpr int TILE_MAX = 11;
constexpr int SPREAD_THREADS = 256;
constexpr int SPREAD_MIN_TILES = 1024;  // smaller tile edges until a batch has this many tiles

__device__ __forceinline__ int tile_of(int i, int tiles, int edge) { return min(i / edge, tiles - 1); }

// Tiles along an axis of n points for edge e: widths e ... (last) in [4, 11].
inline int tiles_for(int n, int e) { return e == 8 ? std::max(1, (n + 4) / 8) : std::max(1, n / e); }

// Atoms are visited in the neighbour list's sorted order, so the lanes of a
// wave mostly fall into one or two tiles, or (order == nullptr) in atom
// order, which lets the spread start before a list build has placed the
// atoms; each distinct tile of a wave takes one atomic for all of its lanes
// (contended device-scope atomics serialise).  The bins' order never changes
// a result: the spread's fixed-point sums are order-independent.
template <class R>
__global__ void k_pme_bin(int nslots, const int* __restrict__ order, const double* __restrict__ pos,
                          const double* __restrict__ charge, const int* __restrict__ atom_sys,
                          const SysInfo* __restrict__ sys, int* st_idx, R* st_w, int* bin_count, int* bins,
                          int bin_cap, unsigned* status) {
    const int slot = blockIdx.x * blockDim.x + threadIdx.x;
    const int lane = threadIdx.x & 63;
    const int a = slot < nslots ? (order ? order[slot] : slot) : -1;
    const double q = a >= 0 ? charge[a] : 0.0;
    int tile = -1;
    if (q != 0.0) {  // uncharged atoms do not spread (pme.rs:315-330)
        const SysInfo& S = sys[atom_sys[a]];
        int idx[3];
        R w[3][5], dw[3][5];
        stencil<R>(pos + 3 * a, S.box, S.grid, idx, w, dw);
        for (int d = 0; d < 3; ++d) st_idx[4 * a + d] = idx[d];
        for (int d = 0; d < 3; ++d)
            for (int k = 0; k < 5; ++k) st_w[16 * a + 5 * d + k] = w[d][k];
        tile = S.tile_off +
               (tile_of(idx[0], S.tiles[0], S.ptile) * S.tiles[1] + tile_of(idx[1], S.tiles[1], S.ptile)) *
                   S.tiles[2] +
               tile_of(idx[2], S.tiles[2], S.ptile);
    }
    unsigned long long pending = __ballot(tile >= 0);
    while (pending) {
        const int leader = __ffsll((long long)pending) - 1;
        const int t = __shfl(tile, leader, 64);
        const unsigned long long group = __ballot(tile == t);
        int base = 0;
        if (lane == leader) base = atomicAdd(&bin_count[t], __popcll(group));
        base = __shfl(base, leader, 64);
        if (tile == t) {
            const int p = base + __popcll(group & ((1ull << lane) - 1ull));
            if (p < bin_cap) bins[(size_t)t * bin_cap + p] = a;
            else atomicOr(status, ST_BIN_OVERFLOW);
        }
        pending &= ~group;
    }
}

__device__ __forceinline__ void lds_add(unsigned long long* p, long long v) {
    if (v) atomicAdd(p, (unsigned long long)v);
}
__device__ __forceinline__ void lds_add(double* p, double v) {
    if (v != 0.0) atomicAdd(p, v);
}

// FP32 spread into the fixed-point grid: the contributions of one staged
// round of SPREAD_THREADS atoms are summed as int32 at 2^-24 and added to the
// int64 tile sums at the end of the round.  A contribution q w is at most
// |q| 0.2153 (the largest 3-D weight of the order-5 spline is (115/192)^3),
// so a round's sum stays below 2^31 / 2^24 = 128 whenever |q| <= 2 for every
// atom (SPREAD32_MAX_CHARGE); otherwise the int64 path is used throughout.
constexpr double SPREAD32_SCALE = 16777216.0;  // 2^24
constexpr double SPREAD32_MAX_CHARGE = 2.0;

template <class R, class G>
__global__ __launch_bounds__(SPREAD_THREADS) void k_spread_tiles(const int* __restrict__ tile_off, int nsys,
                                                                 const SysInfo* __restrict__ sys,
                                                                 const int* __restrict__ st_idx,
                                                                 const R* __restrict__ st_w,
                                                                 const double* __restrict__ charge,
                                                                 const int* __restrict__ bin_count,
                                                                 const int* __restrict__ bins, int bin_cap, G* grid,
                                                                 int small_charges, unsigned* status) {
    constexpr bool FIXED = sizeof(G) == sizeof(long long) && G(0.5) == G(0);  // int64 grid
    using Acc = typename std::conditional<FIXED, unsigned long long, double>::type;
    constexpr bool I32 = FIXED && sizeof(R) == 4;
    const bool use32 = I32 && small_charges;
    __shared__ Acc s_acc[TILE_MAX * TILE_MAX * TILE_MAX];
    __shared__ int s_acc32[I32 ? TILE_MAX * TILE_MAX * TILE_MAX : 1];
    __shared__ int s_src[8], s_pre[9];
    __shared__ int s_idx[3][SPREAD_THREADS];
    __shared__ R s_w[15][SPREAD_THREADS];
    __shared__ double s_q[SPREAD_THREADS];
    const int si = find_sys(tile_off, nsys, blockIdx.x);
    const SysInfo& S = sys[si];
    const int T0 = S.tiles[0], T1 = S.tiles[1], T2 = S.tiles[2];
    const int local = blockIdx.x - S.tile_off;
    const int tz = local % T2, txy = local / T2;
    const int ty = txy % T1, tx = txy / T1;
    const int tcoord[3] = {tx, ty, tz}, tiles[3] = {T0, T1, T2};
    int lo[3], wid[3];
    for (int d = 0; d < 3; ++d) {
        lo[d] = tcoord[d] * S.ptile;
        wid[d] = (tcoord[d] == tiles[d] - 1 ? S.grid[d] : lo[d] + S.ptile) - lo[d];
    }
    const int npts = wid[0] * wid[1] * wid[2];
    for (int i = threadIdx.x; i < npts; i += SPREAD_THREADS) {
        s_acc[i] = (Acc)0;
        if (I32) s_acc32[i] = 0;
    }
    if (threadIdx.x == 0) {
        // Source bins: this tile and the previous one along each axis
        // (periodic), without repeats when an axis has one or two tiles.
        int nsrc = 0;
        for (int dx = -1; dx <= 0; ++dx)
            for (int dy = -1; dy <= 0; ++dy)
                for (int dz = -1; dz <= 0; ++dz) {
                    if ((dx && T0 == 1) || (dy && T1 == 1) || (dz && T2 == 1)) continue;
                    const int sx = (tx + dx + T0) % T0, sy = (ty + dy + T1) % T1, sz = (tz + dz + T2) % T2;
                    s_src[nsrc++] = S.tile_off + (sx * T1 + sy) * T2 + sz;
                }
        s_pre[0] = 0;
        for (int b = 0; b < nsrc; ++b) s_pre[b + 1] = s_pre[b] + min(bin_count[s_src[b]], bin_cap);
        for (int b = nsrc; b < 8; ++b) s_pre[b + 1] = s_pre[b];
    }
    __syncthreads();
    // Source atoms are staged in LDS, SPREAD_THREADS at a time, with one
    // independent load chain per thread; the work items are then (staged
    // atom, x plane of its stencil), five per atom, so atoms that reach only
    // a corner of the tile do not hold up the others.
    const int natoms_src = s_pre[8];
    for (int base = 0; base < natoms_src; base += SPREAD_THREADS) {
        const int k = base + threadIdx.x;
        if (k < natoms_src) {
            int b = 0;
            while (s_pre[b + 1] <= k) ++b;
            const int a = bins[(size_t)s_src[b] * bin_cap + (k - s_pre[b])];
            for (int d = 0; d < 3; ++d) s_idx[d][threadIdx.x] = st_idx[4 * a + d];
            for (int j = 0; j < 15; ++j) s_w[j][threadIdx.x] = st_w[16 * (size_t)a + j];
            s_q[threadIdx.x] = charge[a];
        }
        __syncthreads();
        const int cnt = min(SPREAD_THREADS, natoms_src - base);
        for (int item = threadIdx.x; item < 5 * cnt; item += SPREAD_THREADS) {
            const int m = item / 5, ix = item - 5 * m;
            int px = s_idx[0][m] + ix;
            if (px >= S.grid[0]) px -= S.grid[0];
            const int lx = px - lo[0];
            if (lx < 0 || lx >= wid[0]) continue;
            const double q = s_q[m];
            int loc[2][5];
            for (int d = 0; d < 2; ++d) {
                const int n = S.grid[d + 1];
                int p = s_idx[d + 1][m];
                for (int j = 0; j < 5; ++j) {
                    const int l = p - lo[d + 1];
                    loc[d][j] = (l >= 0 && l < wid[d + 1]) ? l : -1;
                    if (++p == n) p = 0;
                }
            }
            const R wx = s_w[ix][m];
            if (I32 && use32) {
                const float qx = (float)(q * SPREAD32_SCALE) * (float)wx;
                for (int iy = 0; iy < 5; ++iy) {
                    if (loc[0][iy] < 0) continue;
                    const float qxy = qx * (float)s_w[5 + iy][m];
                    int* row = s_acc32 + (lx * wid[1] + loc[0][iy]) * wid[2];
                    for (int iz = 0; iz < 5; ++iz) {
                        if (loc[1][iz] < 0) continue;
                        const int v = __float2int_rn(qxy * (float)s_w[10 + iz][m]);
                        if (v) atomicAdd(row + loc[1][iz], v);
                    }
                }
                continue;
            }
            for (int iy = 0; iy < 5; ++iy) {
                if (loc[0][iy] < 0) continue;
                const R wxy = wx * s_w[5 + iy][m];
                Acc* row = s_acc + (lx * wid[1] + loc[0][iy]) * wid[2];
                for (int iz = 0; iz < 5; ++iz) {
                    if (loc[1][iz] < 0) continue;
                    const double c = q * (double)(wxy * s_w[10 + iz][m]);
                    if (FIXED) lds_add(row + loc[1][iz], (long long)to_fixed(c, GRID_SCALE, status));
                    else lds_add(row + loc[1][iz], c);
                }
            }
        }
        __syncthreads();
        if (I32 && use32) {
            // Fold the round's int32 sums into the int64 tile sums (2^-24 -> 2^-40).
            for (int i = threadIdx.x; i < npts; i += SPREAD_THREADS) {
                s_acc[i] += (Acc)((long long)s_acc32[i] * 65536ll);
                s_acc32[i] = 0;
            }
            __syncthreads();
        }
    }
    G* g = grid + S.qgrid_off;
    const int ny = S.grid[1], nz = S.grid[2];
    for (int i = threadIdx.x; i < npts; i += SPREAD_THREADS) {
        const int lz = i % wid[2], r = i / wid[2];
        const int ly = r % wid[1], lx = r / wid[1];
        g[((size_t)(lo[0] + lx) * ny + (lo[1] + ly)) * nz + lo[2] + lz] = (G)s_acc[i];
    }
}

// Atom-owned spread (the autotuner's alternative to the tile-owned one): chunks
// of PME_CHUNK sorted slots, whose stencils lie in a small box of the grid.
// The contributions are summed in the box in LDS and the box is added to the
// grid with one device atomic per non-zero point; a chunk whose box does not
// fit SPREAD_BOX_BYTES adds every contribution to the grid.  Each contribution
// is the tile-owned spread's value, and integer sums do not depend on their
// order, so on a fixed-point grid both spreads write the same bits (FP64 grids
// sum in a varying order either way).  The grid is zero at the launch (the
// transform after the previous spread cleared every point).
//
// One workgroup per chunk; three waves take the splines and the box along one
// axis each, then its four waves hold the same atoms, one per lane, with their
// weights in registers, and share the stencil's 25 rows.  Bound:
// latency at small systems, the device atomics of the box (27 points per atom at
// 100 atoms/nm^3; a compute unit issues one in 1.5 ns) at large ones.  Before, with
// the weights in LDS and a thread per row of an atom's stencil, and now: FP32
// stencils 900 atoms 18 -> 9 us, 300,000 91 -> 75; 9,000 on an FP64 grid, by tiles
// before, 50 -> 9.  Four chunks per workgroup in one box add a third fewer points
// and take twice as long below 60,000 atoms (36 us against 16 at 23,550).
constexpr int SPREAD_BOX_BYTES = 32768;
constexpr int ATOM_SPREAD_WAVES = 4, ATOM_SPREAD_THREADS = 64 * ATOM_SPREAD_WAVES;
// Smaller groups where that gives idle compute units work (chunks: time with 64,
// 32 and 16 slots per workgroup, us).  FP32 stencils, 15: 16, 10, 9; 141: 13, 10, 10;
// 235: 13, 11, 11; 368: 14, 13, 18; 469: 14, 16, 19; 938: 24, 27, 35.  FP64 ones, 282: 16,
// 12, 18; 368: 16, 14, 19; 469: 19, 17, 21; 563: 17, 24, 27.
constexpr int SPREAD_16_CHUNKS = 192, SPREAD_32_CHUNKS = 256, SPREAD_32_CHUNKS_F64 = 512;
static_assert(PME_CHUNK == 64, "a wave of the atom-owned spread holds a chunk");

// Extrema over each N consecutive lanes.
template <int N>
__device__ __forceinline__ int group_min(int v) {
    for (int o = N / 2; o >= 1; o >>= 1) v = min(v, __shfl_xor(v, o, 64));
    return v;
}
template <int N>
__device__ __forceinline__ int group_max(int v) {
    for (int o = N / 2; o >= 1; o >>= 1) v = max(v, __shfl_xor(v, o, 64));
    return v;
}
// r reduced to (-n/2, n/2], for r in (-n, n).
__device__ __forceinline__ int nearest_offset(int r, int n) {
    if (r > n / 2) return r - n;
    return r <= -(n - n / 2) ? r + n : r;
}
// i reduced to [0, n), for i in [-n, 3n) (a box is at most n + 4 points long).
__device__ __forceinline__ int wrap_near(int i, int n) {
    if (i < 0) i += n;
    if (i >= n) i -= n;
    return i >= n ? i - n : i;
}
__device__ __forceinline__ void grid_add(long long* p, unsigned long long v) {
    atomicAdd(reinterpret_cast<unsigned long long*>(p), v);
}
__device__ __forceinline__ void grid_add(double* p, double v) { unsafeAtomicAdd(p, v); }

// A contribution q w to a grid of G: an int at 2^-24 (I32), or an Acc.
template <class R, class G, bool I32>
struct SpreadSum {
    static constexpr bool FIXED = sizeof(G) == sizeof(long long) && G(0.5) == G(0);  // int64 grid
    using Acc = typename std::conditional<FIXED, unsigned long long, double>::type;
    using Box = typename std::conditional<I32, int, Acc>::type;  // a sum over one chunk
    static __device__ __forceinline__ Box value(double q, R wx, R wy, R wz, unsigned* status) {
        if constexpr (I32) {
            const float qx = (float)(q * SPREAD32_SCALE) * (float)wx;
            const float qxy = qx * (float)wy;
            return __float2int_rn(qxy * (float)wz);
        } else {
            const R wxy = wx * wy;
            const double c = q * (double)(wxy * wz);
            if constexpr (FIXED) return (Acc)to_fixed(c, GRID_SCALE, status);
            else return c;
        }
    }
    static __device__ __forceinline__ void to_grid(G* p, Box v) {
        if constexpr (I32) grid_add(p, (unsigned long long)((long long)v * 65536ll));
        else grid_add(p, v);
    }
};

// Adds one row of an atom's stencil to the grid directly.
template <class R, class G, bool I32>
__device__ __forceinline__ void spread_row_direct(double q, R wx, R wy, const R wz[5], G* row, int gz0, int nz,
                                                  unsigned* status) {
    using Sum = SpreadSum<R, G, I32>;
#pragma unroll
    for (int iz = 0; iz < 5; ++iz) {
        int gz = gz0 + iz;
        if (gz >= nz) gz -= nz;
        const typename Sum::Box v = Sum::value(q, wx, wy, wz[iz], status);
        if (v != (typename Sum::Box)0) Sum::to_grid(row + gz, v);
    }
}

// ATOMS slots per workgroup: lane k of every ATOMS lanes holds slot k, and the
// groups of ATOMS lanes share the rows.
template <class R, class G, bool I32, int ATOMS>
__global__ __launch_bounds__(ATOM_SPREAD_THREADS) void k_spread_atoms(const int* __restrict__ chunk_off, int nsys,
                                                                      const int* __restrict__ order,
                                                                      const double* __restrict__ pos,
                                                                      const double* __restrict__ charge,
                                                                      const SysInfo* __restrict__ sys, G* grid,
                                                                      unsigned* status) {
    using Sum = SpreadSum<R, G, I32>;
    using Box = typename Sum::Box;
    constexpr int PARTS = PME_CHUNK / ATOMS, GROUPS = ATOM_SPREAD_THREADS / ATOMS;
    // The box (int32 sums at 2^-24: at most PME_CHUNK contributions of
    // |q| w <= 2 x 0.2153 per point stay below 2^31).
    __shared__ Box box[SPREAD_BOX_BYTES / sizeof(Box)];
    __shared__ R s_w[3][5][ATOMS];
    __shared__ int s_idx[3][ATOMS], s_at[3][ATOMS], s_org[3], s_ext[3];
    const int t = threadIdx.x, k = t & (ATOMS - 1), group = t / ATOMS;
    const int chunk = blockIdx.x / PARTS;
    int si = 0, local = chunk;
    if (nsys > 1) {
        si = find_sys(chunk_off, nsys, chunk);
        local -= chunk_off[si];
    }
    const SysInfo& S = sys[si];
    const int slot = S.slot_off + local * PME_CHUNK + (blockIdx.x & (PARTS - 1)) * ATOMS + k;
    const int end = S.slot_off + S.nblocks * IBLOCK;
    const int listed = order[min(slot, end - 1)];
    const int a = slot < end ? listed : -1, a0 = max(a, 0);
    const double charge_a = charge[a0];
    const double p[3] = {pos[3 * (size_t)a0], pos[3 * (size_t)a0 + 1], pos[3 * (size_t)a0 + 2]};
    const int n[3] = {S.grid[0], S.grid[1], S.grid[2]};
    const double q = a >= 0 ? charge_a : 0.0;
    const bool on = q != 0.0;  // uncharged atoms do not spread (pme.rs:315-330)
    const unsigned long long live = __ballot(on);
    if (!live) return;  // the same in all four waves
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6), lead = __ffsll((long long)live) - 1;
    if (wave < 3) {
        // One axis per wave: the splines, and the box's origin and extent from
        // the offsets from the first charged atom, nearest images.
        R wd[5], dw[5];
        const int i = stencil_axis<R>(p, S.box, wave, n[wave], wd, dw);
        const int first = __shfl(i, lead, 64);
        const int r = nearest_offset(i - first, n[wave]);
        const int lo = group_min<ATOMS>(on ? r : INT_MAX), hi = group_max<ATOMS>(on ? r : INT_MIN);
        if (t % 64 < ATOMS) {
            s_at[wave][k] = r - lo;
            s_idx[wave][k] = i;
#pragma unroll
            for (int j = 0; j < 5; ++j) s_w[wave][j][k] = wd[j];
        }
        if (t % 64 == 0) {
            s_org[wave] = wrap_near(first + lo, n[wave]);
            s_ext[wave] = hi - lo + 5;
        }
    }
    __syncthreads();
    int idx[3], org[3], ext[3], at[3];
    R w[3][5];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        idx[d] = s_idx[d][k];
        at[d] = s_at[d][k];
        org[d] = s_org[d];
        ext[d] = s_ext[d];
#pragma unroll
        for (int j = 0; j < 5; ++j) w[d][j] = s_w[d][j][k];
    }
    G* g = grid + S.qgrid_off;
    const int e1 = ext[1], e2 = ext[2], vol = ext[0] * e1 * e2;
    if (vol > SPREAD_BOX_BYTES / (int)sizeof(Box)) {
        if (!on) return;
        for (int r = group; r < 25; r += GROUPS) {
            const int ix = r / 5, iy = r - 5 * ix;
            int gx = idx[0] + ix, gy = idx[1] + iy;
            if (gx >= n[0]) gx -= n[0];
            if (gy >= n[1]) gy -= n[1];
            spread_row_direct<R, G, I32>(q, pick(w[0], ix), pick(w[1], iy), w[2],
                                         g + ((size_t)gx * n[1] + gy) * n[2], idx[2], n[2], status);
        }
        return;
    }
    for (int i = t; i < vol; i += ATOM_SPREAD_THREADS) box[i] = (Box)0;
    __syncthreads();
    if (on) {
        const int base = (at[0] * e1 + at[1]) * e2 + at[2];
        for (int r = group; r < 25; r += GROUPS) {
            const int ix = r / 5, iy = r - 5 * ix;
            const R wx = pick(w[0], ix), wy = pick(w[1], iy);
            Box* row = box + base + (ix * e1 + iy) * e2;
#pragma unroll
            for (int iz = 0; iz < 5; ++iz) {
                const Box v = Sum::value(q, wx, wy, w[2][iz], status);
                if (v != (Box)0) atomicAdd(row + iz, v);
            }
        }
    }
    __syncthreads();
    // Sixteen threads per row of the box.
    const float inv_e1 = 1.0f / (float)e1;
    for (int row = t >> 4; row < ext[0] * e1; row += ATOM_SPREAD_THREADS / 16) {
        const int lx = div_small(row, e1, inv_e1), ly = row - lx * e1;
        G* grow = g + ((size_t)wrap_near(org[0] + lx, n[0]) * n[1] + wrap_near(org[1] + ly, n[1])) * n[2];
        for (int lz = t & 15; lz < e2; lz += 16) {
            const Box v = box[row * e2 + lz];
            if (v != (Box)0) Sum::to_grid(grow + wrap_near(org[2] + lz, n[2]), v);
        }
    }
}

// Atoms in no spatial order: five threads per atom (one per x plane of the
// stencil), every contribution added to the grid.
template <class R, class G, bool I32>
__global__ __launch_bounds__(256) void k_spread_direct(int natoms, const double* __restrict__ pos,
                                                       const double* __restrict__ charge,
                                                       const int* __restrict__ atom_sys,
                                                       const SysInfo* __restrict__ sys, G* grid,
                                                       unsigned* status) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    const int a = t / 5, ix = t - 5 * a;
    if (a >= natoms) return;
    const double q = charge[a];
    if (q == 0.0) return;  // pme.rs:315-330
    const SysInfo& S = sys[atom_sys[a]];
    int idx[3];
    R w[3][5], dw[3][5];
    stencil<R>(pos + 3 * (size_t)a, S.box, S.grid, idx, w, dw);
    const R wx = pick(w[0], ix);
    int gx = idx[0] + ix;
    if (gx >= S.grid[0]) gx -= S.grid[0];
#pragma unroll
    for (int iy = 0; iy < 5; ++iy) {
        int gy = idx[1] + iy;
        if (gy >= S.grid[1]) gy -= S.grid[1];
        spread_row_direct<R, G, I32>(q, wx, w[1][iy], w[2], grid + S.qgrid_off + ((size_t)gx * S.grid[1] + gy) * S.grid[2],
                                     idx[2], S.grid[2], status);
    }
}

// One system's charges in no spatial order (a mesh of charges alone).
__global__ __launch_bounds__(CHARGE_PLANE_THREADS) void k_spread_planes(int natoms, const double* __restrict__ pos,
                                                                 const double* __restrict__ charge,
                                                                 const SysInfo* __restrict__ sys, double* grid) {
    __shared__ double s_plane[PLANE_POINTS];
    const SysInfo& S = sys[0];
    spread_plane(blockIdx.x, natoms, pos, charge, S.box, S.grid, s_plane);
    const int points = S.grid[1] * S.grid[2];
    double* out = grid + S.qgrid_off + (size_t)blockIdx.x * points;
    for (int i = threadIdx.x; i < points; i += CHARGE_PLANE_THREADS) out[i] = s_plane[i];
}

// Gather with five threads per atom, one per z of the stencil, so that five
// lanes read a row's consecutive points together (one per x plane touches five
// times as many cache lines, which bounds the kernel); atoms in the spatially
// sorted order.  The first three waves take the splines of one axis each, the
// five partial gradients are combined in LDS.  300,000 atoms 45 -> 38 us, 900
// atoms 5.0 -> 4.0 (with a plane and the whole stencil per thread before).
constexpr int GATHER_ATOMS = PME_CHUNK;

template <class R, class A>
__global__ __launch_bounds__(GATHER_ATOMS * 5) void k_gather5(const int* __restrict__ chunk_off, int nsys,
                                                              const int* __restrict__ order,
                                                              const double* __restrict__ pos,
                                                              const double* __restrict__ charge,
                                                              const SysInfo* __restrict__ sys,
                                                              const R* __restrict__ phi, A* force, unsigned* status) {
    __shared__ R s_w[3][5][GATHER_ATOMS], s_dw[3][5][GATHER_ATOMS], s_g[3][5][GATHER_ATOMS];
    __shared__ int s_idx[3][GATHER_ATOMS], s_atom[GATHER_ATOMS];
    __shared__ double s_q[GATHER_ATOMS];
    int si = 0, local = blockIdx.x;
    if (nsys > 1) {
        si = find_sys(chunk_off, nsys, blockIdx.x);
        local -= chunk_off[si];
    }
    const SysInfo& S = sys[si];
    const Box& b = S.box;
    const int nx = S.grid[0], ny = S.grid[1], nz = S.grid[2];
    phi += S.qgrid_off;
    const int t = threadIdx.x;
    if (t < 3 * GATHER_ATOMS) {
        const int k = t & (GATHER_ATOMS - 1), d = __builtin_amdgcn_readfirstlane(t / GATHER_ATOMS);
        const int slot = S.slot_off + local * GATHER_ATOMS + k, end = S.slot_off + S.nblocks * IBLOCK;
        const int listed = order[min(slot, end - 1)];
        const int a = slot < end ? listed : -1, a0 = max(a, 0);
        const double p[3] = {pos[3 * (size_t)a0], pos[3 * (size_t)a0 + 1], pos[3 * (size_t)a0 + 2]};
        if (d == 0) {
            const double qa = charge[a0];
            s_atom[k] = a0;
            s_q[k] = a >= 0 ? qa : 0.0;
        }
        R w[5], dw[5];
        s_idx[d][k] = stencil_axis<R>(p, b, d, S.grid[d], w, dw);
#pragma unroll
        for (int j = 0; j < 5; ++j) {
            s_w[d][j][k] = w[j];
            s_dw[d][j][k] = dw[j];
        }
    }
    __syncthreads();
    const int k = t / 5, iz = t - k * 5;
    const double q = s_q[k];
    if (q != 0.0) {
        R wy[5], dwy[5];
        int row[5];
#pragma unroll
        for (int iy = 0; iy < 5; ++iy) {
            wy[iy] = s_w[1][iy][k];
            dwy[iy] = s_dw[1][iy][k];
            int gy = s_idx[1][k] + iy;
            if (gy >= ny) gy -= ny;
            row[iy] = gy * nz;
        }
        int gz = s_idx[2][k] + iz;
        if (gz >= nz) gz -= nz;
        const int gx0 = s_idx[0][k];
        const R* column = phi + gz;
        R s00 = 0, s10 = 0, s01 = 0;  // sums of phi w_x w_y, phi w'_x w_y, phi w_x w'_y
#pragma unroll
        for (int ix = 0; ix < 5; ++ix) {
            int gx = gx0 + ix;
            if (gx >= nx) gx -= nx;
            const R* plane = column + (size_t)gx * ny * nz;
            const R wx = s_w[0][ix][k], dwx = s_dw[0][ix][k];
            R r0 = 0, r1 = 0;
#pragma unroll
            for (int iy = 0; iy < 5; ++iy) {
                const R v = plane[row[iy]];
                r0 += v * wy[iy];
                r1 += v * dwy[iy];
            }
            s00 += wx * r0;
            s10 += dwx * r0;
            s01 += wx * r1;
        }
        const R wz = s_w[2][iz][k], dwz = s_dw[2][iz][k];
        s_g[0][iz][k] = s10 * wz;
        s_g[1][iz][k] = s01 * wz;
        s_g[2][iz][k] = s00 * dwz;
    }
    __syncthreads();
    if (iz < 3 && q != 0.0) {
        R G[3] = {0, 0, 0};
        for (int d = 0; d < 3; ++d)
            for (int m = 0; m < 5; ++m) G[d] += s_g[d][m][k];
        // pme.rs:417-422
        const double s = (double)G[0] * nx * b.recip[0 * 3 + iz] + (double)G[1] * ny * b.recip[1 * 3 + iz] +
                         (double)G[2] * nz * b.recip[2 * 3 + iz];
        acc_add(force + 3 * (size_t)s_atom[k] + iz, -q * s, FORCE_SCALE, status);
    }
}

enum : int { MODE_Z_R2C = 0, MODE_Y_FWD = 1, MODE_X_CONV = 2, MODE_Y_INV = 3, MODE_Z_C2R = 4 };

// Batched Stockham FFT of `lines` lines of length n held line-major in a/b,
// T threads per line.  A stage of radix R is a direct DFT per output:
// out[(j - k) R + k + q Ns] = sum_r in[j + r m] W_n^{r (k n/(Ns R) + q m)},
// m = n/R, output index o = q m + j, k = j mod Ns.  The exponent base
// k n/(Ns R) + q m stays below n, so the root index wraps with one conditional
// subtraction.  Each output is computed by one thread in a fixed order, so
// the result does not depend on T or on how lines are grouped.
__device__ __forceinline__ float fused(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double fused(double a, double b, double c) { return __builtin_fma(a, b, c); }

template <class R>
__device__ Cx<R>* fft_lds(Cx<R>* a, Cx<R>* b, int n, const int* radices, const Cx<R>* roots, bool inverse, int T) {
    const int li = threadIdx.x / T, t = threadIdx.x - li * T;
    const R sgn = inverse ? (R)-1 : (R)1;
    int Ns = 1;
    for (int s = 0; s < MAX_STAGES && radices[s]; ++s) {
        const int Rr = radices[s];
        const int m = n / Rr;
        const int step = n / (Ns * Rr);
        const Cx<R>* in = a + li * n;
        Cx<R>* out = b + li * n;
        const float inv_ns = 1.0f / (float)Ns;
        const float inv_m = 1.0f / (float)m;
        for (int o = t; o < n; o += T) {
            const int q = div_small(o, m, inv_m);
            const int j = o - q * m;
            const int k = j - div_small(j, Ns, inv_ns) * Ns;
            const int base = k * step + q * m;
            R ax = 0, ay = 0;
            int idx = 0;
            for (int r = 0; r < Rr; ++r) {
                const Cx<R> w = roots[idx];
                const R wy = sgn * w.y;
                const Cx<R> v = in[j + r * m];
                // Explicit fused multiply-adds: every kernel that inlines
                // this routine rounds the same way.
                ax = fused(v.x, w.x, fused(-v.y, wy, ax));
                ay = fused(v.x, wy, fused(v.y, w.x, ay));
                idx += base;
                if (idx >= n) idx -= n;
            }
            out[(j - k) * Rr + k + q * Ns] = Cx<R>{ax, ay};
        }
        __syncthreads();
        Cx<R>* tmp = a;
        a = b;
        b = tmp;
        Ns *= Rr;
    }
    return a;
}

// The z passes transform two real lines y = 2p, 2p + 1 of an x plane at once
// as the complex line a + i b (the last line alone when ny is odd).  From
// Z = FFT(a + i b) at k and at (n - k) mod n, the half spectra are
//   A = (Z_k + conj(Z_{n-k})) / 2,  B = (Z_k - conj(Z_{n-k})) / (2i);
// the inverse transforms A_full + i B_full (each rebuilt from its half by
// Hermitian symmetry) and reads a and b as the real and imaginary parts.
// Every kernel pairs the lines the same way and calls the same routines, so
// the plane and line passes keep giving the same bits.
template <class R>
__device__ __forceinline__ void unpack_pair(Cx<R> U, Cx<R> W, Cx<R>& A, Cx<R>& B) {
    A = Cx<R>{(R)0.5 * (U.x + W.x), (R)0.5 * (U.y - W.y)};
    B = Cx<R>{(R)0.5 * (U.y + W.y), (R)0.5 * (W.x - U.x)};
}
template <class R>
__device__ __forceinline__ Cx<R> pack_pair(Cx<R> A, Cx<R> B) {
    return Cx<R>{A.x - B.y, A.y + B.x};
}
// Element el of the full spectrum of a real line from its half h[0 .. nz/2].
template <class R>
__device__ __forceinline__ Cx<R> hermitian_at(const Cx<R>* h, int el, int nz, int nzh) {
    if (el < nzh) return h[el];
    const Cx<R> v = h[nz - el];
    return Cx<R>{v.x, -v.y};
}

template <class R, class G, class A, int MODE>
__global__ __launch_bounds__(FFT_THREADS) void k_fft(const int* __restrict__ blk_off, int nsys,
                                                     const SysInfo* __restrict__ sys, G* __restrict__ qgrid,
                                                     Cx<R>* cgrid, R* phi, const Cx<R>* __restrict__ roots_all,
                                                     const R* __restrict__ moduli_all, A* energy, unsigned* status,
                                                     int* clear, int nclear) {
    extern __shared__ unsigned char smem_raw[];
    // The first pass also clears the spread's bin counts (every spread
    // workgroup is done by now), so no fill kernel opens the next spread.
    if (MODE == MODE_Z_R2C && clear)
        for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < nclear; i += gridDim.x * blockDim.x) clear[i] = 0;
    const bool zmode = MODE == MODE_Z_R2C || MODE == MODE_Z_C2R;
    const bool ymode = MODE == MODE_Y_FWD || MODE == MODE_Y_INV;
    const int axis = zmode ? 2 : (ymode ? 1 : 0);
    const int si = find_sys(blk_off, nsys, blockIdx.x);
    const SysInfo& S = sys[si];
    const int nx = S.grid[0], ny = S.grid[1], nz = S.grid[2], nzh = S.nzh;
    const int n = S.grid[axis];
    const int LINES = S.fft_lines[sizeof(R) == 8 ? 1 : 0][axis];
    const int T = FFT_THREADS / LINES;
    const int nyp = (ny + 1) / 2;  // z passes: line pairs per x plane
    const int nlines = zmode ? nx * nyp : (ymode ? nx * nzh : ny * nzh);
    const int line0 = (blockIdx.x - blk_off[si]) * LINES;
    qgrid += S.qgrid_off;
    phi += S.qgrid_off;
    cgrid += S.cgrid_off;

    Cx<R>* bufA = reinterpret_cast<Cx<R>*>(smem_raw);
    Cx<R>* bufB = bufA + LINES * n;
    Cx<R>* roots = bufB + LINES * n;
    __shared__ int s_radix[MAX_STAGES];
    if (threadIdx.x < MAX_STAGES) s_radix[threadIdx.x] = S.radix[axis][threadIdx.x];
    for (int i = threadIdx.x; i < n; i += FFT_THREADS) roots[i] = roots_all[S.roots_off[axis] + i];

    // Load.
    for (int e = threadIdx.x; e < LINES * n; e += FFT_THREADS) {
        int li, el;
        if (zmode) {
            li = e / n;
            el = e - li * n;
        } else {
            li = e % LINES;
            el = e / LINES;
        }
        const int L = line0 + li;
        Cx<R> v = {0, 0};
        if (L < nlines) {
            if (zmode) {
                const int x = L / nyp, y = 2 * (L - x * nyp);
                const size_t row = (size_t)x * ny + y;
                if (MODE == MODE_Z_R2C) {
                    // The grid is zero between runs: each point is cleared as
                    // it is read.
                    G& g0 = qgrid[row * nz + el];
                    v.x = (R)grid_real(g0);
                    g0 = (G)0;
                    if (y + 1 < ny) {
                        G& g1 = qgrid[(row + 1) * nz + el];
                        v.y = (R)grid_real(g1);
                        g1 = (G)0;
                    }
                } else {
                    const Cx<R> a = hermitian_at(cgrid + row * nzh, el, nz, nzh);
                    const Cx<R> b = y + 1 < ny ? hermitian_at(cgrid + (row + 1) * nzh, el, nz, nzh) : Cx<R>{0, 0};
                    v = pack_pair(a, b);
                }
            } else if (ymode) {
                const int x = L / nzh, kz = L - x * nzh;
                v = cgrid[((size_t)x * ny + el) * nzh + kz];
            } else {
                const int y = L / nzh, kz = L - y * nzh;
                v = cgrid[((size_t)el * ny + y) * nzh + kz];
            }
        }
        bufA[li * n + el] = v;
    }
    __syncthreads();
    const int* rad = s_radix;
    const bool inverse_first = MODE == MODE_Y_INV || MODE == MODE_Z_C2R;
    Cx<R>* res = fft_lds<R>(bufA, bufB, n, rad, roots, inverse_first, T);

    if (MODE == MODE_X_CONV) {
        // Reciprocal convolution and energy (pme.rs:332-372) on the half spectrum.
        constexpr bool F32 = sizeof(R) == 4;
        const Influence<R> I(S, moduli_all);
        double eacc = 0.0;
        for (int e = threadIdx.x; e < LINES * n; e += FFT_THREADS) {
            const int li = e % LINES, kx = e / LINES;
            const int L = line0 + li;
            if (L >= nlines) continue;
            const int y = L / nzh, kz = L - y * nzh;
            Cx<R>& v = res[li * n + kx];
            const R infl = I(kx, y, kz);
            if (!F32) {
                const double wz = (kz == 0 || 2 * kz == nz) ? 1.0 : 2.0;
                eacc += wz * 0.5 * (double)infl * ((double)v.x * v.x + (double)v.y * v.y);
            }
            v.x *= infl;
            v.y *= infl;
        }
        if (!F32) {
            double et = wave_sum(eacc);
            if ((threadIdx.x & 63) == 0) acc_add(energy + si * E_SLOTS + E_RECIP, et, ENERGY_SCALE, status);
        }
        __syncthreads();
        Cx<R>* other = res == bufA ? bufB : bufA;
        res = fft_lds<R>(res, other, n, rad, roots, true, T);
    }

    // Store.
    if (MODE == MODE_Z_R2C) {
        for (int e = threadIdx.x; e < LINES * nzh; e += FFT_THREADS) {
            const int li = e / nzh, el = e - li * nzh;
            const int L = line0 + li;
            if (L >= nlines) continue;
            const int x = L / nyp, y = 2 * (L - x * nyp);
            Cx<R> a, b;
            unpack_pair(res[li * n + el], res[li * n + (el ? n - el : 0)], a, b);
            Cx<R>* row = cgrid + ((size_t)x * ny + y) * nzh;
            row[el] = a;
            if (y + 1 < ny) row[nzh + el] = b;
        }
        return;
    }
    for (int e = threadIdx.x; e < LINES * n; e += FFT_THREADS) {
        int li, el;
        if (zmode) {
            li = e / n;
            el = e - li * n;
        } else {
            li = e % LINES;
            el = e / LINES;
        }
        const int L = line0 + li;
        if (L >= nlines) continue;
        const Cx<R> v = res[li * n + el];
        if (MODE == MODE_Z_C2R) {
            const int x = L / nyp, y = 2 * (L - x * nyp);
            const size_t row = (size_t)x * ny + y;
            phi[row * nz + el] = v.x;
            if (y + 1 < ny) phi[(row + 1) * nz + el] = v.y;
        } else if (ymode) {
            const int x = L / nzh, kz = L - x * nzh;
            cgrid[((size_t)x * ny + el) * nzh + kz] = v;
        } else {
            const int y = L / nzh, kz = L - y * nzh;
            cgrid[((size_t)el * ny + y) * nzh + kz] = v;
        }
    }
}

// Plane passes: one workgroup per x plane of a system transforms the plane
// along z and along y in LDS.  Forward (DIR 0): pairs of real z lines to their
// half spectra (kept as P[kz][y]), then y lines, stored as cgrid[x][ky][kz].
// Inverse (DIR 1): y lines of the half spectrum, then pairs of z lines rebuilt
// from it by Hermitian symmetry and transformed to real values.  Every line
// goes through fft_lds (and the pair packing) with the data the corresponding
// line pass would load, so the results are the same bits as the five-pass
// form.
//
// LDS (complex elements): roots along z [nz] and y [ny], P and Q
// [lyp x ny] (lyp = nzh rounded up to a multiple of the y lines per call),
// and the ping-pong buffers of lz z-line pairs [2 x lz x nz], which share
// the one of P and Q that does not hold live data when they fit in it.
constexpr int PLANE_THREADS = 1024;
constexpr size_t PLANE_LDS_MAX = 160 * 1024 - 256;  // gfx950 LDS per workgroup, less the static arrays

struct PlaneLayout {
    int lyp;
    size_t pq;      // elements of P (and of Q)
    bool z_shared;  // the z buffers fit in the free one of P and Q
    size_t elems;   // total complex elements
};

__host__ __device__ inline PlaneLayout plane_layout(int ny, int nz, int nzh, int lz, int ly) {
    PlaneLayout L;
    L.lyp = (nzh + ly - 1) / ly * ly;
    L.pq = (size_t)L.lyp * ny;
    const size_t zb = 2 * (size_t)lz * nz;
    L.z_shared = zb <= L.pq;
    L.elems = (size_t)nz + ny + 2 * L.pq + (L.z_shared ? 0 : zb);
    return L;
}

template <class R, class G, int DIR>
__global__ __launch_bounds__(PLANE_THREADS) void k_fft_plane(const int* __restrict__ plane_off, int nsys,
                                                            const SysInfo* __restrict__ sys, G* __restrict__ qgrid,
                                                            Cx<R>* cgrid, R* phi,
                                                            const Cx<R>* __restrict__ roots_all, int* clear,
                                                            int nclear) {
    extern __shared__ unsigned char smem_raw[];
    __shared__ int s_rz[MAX_STAGES], s_ry[MAX_STAGES];
    // The forward pass also clears the spread's bin counts (every spread
    // workgroup is done by now), as the first line pass does.
    if (DIR == 0 && clear)
        for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < nclear; i += gridDim.x * blockDim.x) clear[i] = 0;
    const int si = find_sys(plane_off, nsys, blockIdx.x);
    const SysInfo& S = sys[si];
    const int ny = S.grid[1], nz = S.grid[2], nzh = S.nzh;
    const int x = blockIdx.x - plane_off[si];
    constexpr int prec = sizeof(R) == 8 ? 1 : 0;
    const int lz = S.plane_lines[prec][0], ly = S.plane_lines[prec][1];
    const int nyp = (ny + 1) / 2;  // z line pairs
    const PlaneLayout L = plane_layout(ny, nz, nzh, lz, ly);
    Cx<R>* rz = reinterpret_cast<Cx<R>*>(smem_raw);
    Cx<R>* ry = rz + nz;
    Cx<R>* P = ry + ny;
    Cx<R>* Q = P + L.pq;
    Cx<R>* extra = Q + L.pq;
    if (threadIdx.x < MAX_STAGES) {
        s_rz[threadIdx.x] = S.radix[2][threadIdx.x];
        s_ry[threadIdx.x] = S.radix[1][threadIdx.x];
    }
    for (int i = threadIdx.x; i < nz; i += PLANE_THREADS) rz[i] = roots_all[S.roots_off[2] + i];
    for (int i = threadIdx.x; i < ny; i += PLANE_THREADS) ry[i] = roots_all[S.roots_off[1] + i];
    qgrid += S.qgrid_off + (size_t)x * ny * nz;
    phi += S.qgrid_off + (size_t)x * ny * nz;
    cgrid += S.cgrid_off + (size_t)x * ny * nzh;
    const int Tz = PLANE_THREADS / lz, Ty = PLANE_THREADS / ly;

    if (DIR == 0) {
        Cx<R>* Z = L.z_shared ? Q : extra;
        __syncthreads();  // roots and radices
        for (int p0 = 0; p0 < nyp; p0 += lz) {
            // Line pairs (y, y + 1) = (2p, 2p + 1), as the line passes pair them.
            for (int e = threadIdx.x; e < lz * nz; e += PLANE_THREADS) {
                const int li = e / nz, el = e - li * nz;
                const int y = 2 * (p0 + li);
                Cx<R> v = {0, 0};
                if (y < ny) {
                    G& g0 = qgrid[(size_t)y * nz + el];  // cleared as read
                    v.x = (R)grid_real(g0);
                    g0 = (G)0;
                    if (y + 1 < ny) {
                        G& g1 = qgrid[(size_t)(y + 1) * nz + el];
                        v.y = (R)grid_real(g1);
                        g1 = (G)0;
                    }
                }
                Z[e] = v;
            }
            __syncthreads();
            const Cx<R>* res = fft_lds<R>(Z, Z + (size_t)lz * nz, nz, s_rz, rz, false, Tz);
            for (int e = threadIdx.x; e < lz * nzh; e += PLANE_THREADS) {
                const int li = e / nzh, kz = e - li * nzh;
                const int y = 2 * (p0 + li);
                if (y < ny) {
                    Cx<R> a, b;
                    unpack_pair(res[(size_t)li * nz + kz], res[(size_t)li * nz + (kz ? nz - kz : 0)], a, b);
                    P[(size_t)kz * ny + y] = a;
                    if (y + 1 < ny) P[(size_t)kz * ny + y + 1] = b;
                }
            }
            __syncthreads();
        }
        const Cx<R>* res = P;
        for (int k0 = 0; k0 < L.lyp; k0 += ly)
            res = fft_lds<R>(P + (size_t)k0 * ny, Q + (size_t)k0 * ny, ny, s_ry, ry, false, Ty) - (size_t)k0 * ny;
        for (int e = threadIdx.x; e < ny * nzh; e += PLANE_THREADS) {
            const int ky = e / nzh, kz = e - ky * nzh;
            cgrid[e] = res[(size_t)kz * ny + ky];
        }
    } else {
        for (int e = threadIdx.x; e < ny * nzh; e += PLANE_THREADS) {
            const int ky = e / nzh, kz = e - ky * nzh;
            P[(size_t)kz * ny + ky] = cgrid[e];
        }
        __syncthreads();
        const Cx<R>* res = P;
        for (int k0 = 0; k0 < L.lyp; k0 += ly)
            res = fft_lds<R>(P + (size_t)k0 * ny, Q + (size_t)k0 * ny, ny, s_ry, ry, true, Ty) - (size_t)k0 * ny;
        Cx<R>* Z = L.z_shared ? (res == P ? Q : P) : extra;
        // The half spectrum of line y at kz is res[kz][y].
        auto half_at = [&](int y, int el) {
            if (el < nzh) return res[(size_t)el * ny + y];
            const Cx<R> v = res[(size_t)(nz - el) * ny + y];
            return Cx<R>{v.x, -v.y};
        };
        for (int p0 = 0; p0 < nyp; p0 += lz) {
            for (int e = threadIdx.x; e < lz * nz; e += PLANE_THREADS) {
                const int li = e / nz, el = e - li * nz;
                const int y = 2 * (p0 + li);
                Cx<R> v = {0, 0};
                if (y < ny) v = pack_pair(half_at(y, el), y + 1 < ny ? half_at(y + 1, el) : Cx<R>{0, 0});
                Z[e] = v;
            }
            __syncthreads();
            const Cx<R>* out = fft_lds<R>(Z, Z + (size_t)lz * nz, nz, s_rz, rz, true, Tz);
            for (int e = threadIdx.x; e < lz * nz; e += PLANE_THREADS) {
                const int li = e / nz, el = e - li * nz;
                const int y = 2 * (p0 + li);
                if (y < ny) {
                    phi[(size_t)y * nz + el] = out[e].x;
                    if (y + 1 < ny) phi[(size_t)(y + 1) * nz + el] = out[e].y;
                }
            }
            __syncthreads();
        }
    }
}

std::vector<int> factorize(int n) {
    std::vector<int> r;
    while (n % 8 == 0) {
        r.push_back(8);
        n /= 8;
    }
    while (n % 4 == 0) {
        r.push_back(4);
        n /= 4;
    }
    while (n % 2 == 0) {
        r.push_back(2);
        n /= 2;
    }
    for (int p = 3; p * p <= n; p += 2)
        while (n % p == 0) {
            r.push_back(p);
            n /= p;
        }
    if (n > 1) r.push_back(n);
    return r;
}

// Most lines per workgroup whose two LDS buffers fit in 60 KB (at most 16).
int max_lines(int n, size_t csize) {
    int lines = 16;
    while (lines > 1 && (2 * (size_t)lines * n + n) * csize > 60000) lines >>= 1;
    return lines;
}

template <class R, class G, class A, int MODE>
void launch_fft(const PmeDev& pm, const SysInfo* sys, G* qgrid, Cx<R>* cgrid, R* phi, const R* roots, const R* moduli,
                A* energy, unsigned* status, hipStream_t s, int* clear = nullptr, int nclear = 0) {
    const int prec = sizeof(R) == 8 ? 1 : 0;
    const bool zmode = MODE == MODE_Z_R2C || MODE == MODE_Z_C2R;
    const bool ymode = MODE == MODE_Y_FWD || MODE == MODE_Y_INV;
    const int axis = zmode ? 2 : (ymode ? 1 : 0);
    hipLaunchKernelGGL((k_fft<R, G, A, MODE>), dim3(pm.fft_blocks[prec][MODE]), dim3(FFT_THREADS),
                       pm.fft_shmem[prec][axis], s, pm.fft_off[prec][MODE].p, pm.nsys, sys, qgrid, cgrid, phi,
                       reinterpret_cast<const Cx<R>*>(roots), moduli, energy, status, clear, nclear);
}

template <class R, class G, int DIR>
void launch_plane(const PmeDev& pm, const SysInfo* sys, G* qgrid, Cx<R>* cgrid, R* phi, const R* roots,
                  hipStream_t s, int* clear = nullptr, int nclear = 0) {
    constexpr int prec = sizeof(R) == 8 ? 1 : 0;
    hipLaunchKernelGGL((k_fft_plane<R, G, DIR>), dim3(pm.plane_blocks[prec]), dim3(PLANE_THREADS), pm.plane_shmem[prec], s,
                       pm.plane_off[prec].p, pm.nsys, sys, qgrid, cgrid, phi, reinterpret_cast<const Cx<R>*>(roots), clear,
                       nclear);
}

// The matrix-core passes over the systems that take them.
template <int W, class R, class G, class A>
void launch_dft_w(const PmeDev& pm, const SysInfo* sys, G* qgrid, R* cgrid, R* phi, const Cx<R>* roots,
                  const R* moduli, A* energy, unsigned* status, hipStream_t s, int* clear, int nclear) {
    constexpr int prec = sizeof(R) == 8 ? 1 : 0;
    const dim3 wg(64 * W);
    hipLaunchKernelGGL((k_dft_zy<W, R, G>), dim3(pm.dft_blocks[prec][0]), wg, pm.dft_shmem[prec][0], s, pm.dft_off[prec][0].p,
                       pm.nsys, sys, qgrid, cgrid, roots, pm.shape, clear, nclear);
    hipLaunchKernelGGL((k_dft_x<W, R, G, A>), dim3(pm.dft_blocks[prec][1]), wg, pm.dft_shmem[prec][1], s, pm.dft_off[prec][1].p,
                       pm.nsys, sys, qgrid, cgrid, roots, moduli, pm.shape, energy, status);
    hipLaunchKernelGGL((k_dft_yz<W, R>), dim3(pm.dft_blocks[prec][2]), wg, pm.dft_shmem[prec][2], s, pm.dft_off[prec][2].p,
                       pm.nsys, sys, cgrid, phi, roots, pm.shape);
}

template <class R, class G, class A>
void launch_dft(const PmeDev& pm, const SysInfo* sys, G* qgrid, R* cgrid, R* phi, const R* roots_r, const R* moduli,
                A* energy, unsigned* status, hipStream_t s, int* clear, int nclear) {
    const Cx<R>* roots = reinterpret_cast<const Cx<R>*>(roots_r);
    constexpr int prec = sizeof(R) == 8 ? 1 : 0;
    if (pm.dft_wide[prec])
        launch_dft_w<DFT_WAVES_WIDE, R, G, A>(pm, sys, qgrid, cgrid, phi, roots, moduli, energy, status, s, clear,
                                              nclear);
    else
        launch_dft_w<DFT_WAVES, R, G, A>(pm, sys, qgrid, cgrid, phi, roots, moduli, energy, status, s, clear, nclear);
}

template <class R>
R* pme_weights(PmeDev& pm);
template <>
float* pme_weights<float>(PmeDev& pm) {
    return pm.st_wf.p;
}
template <>
double* pme_weights<double>(PmeDev& pm) {
    return pm.st_wd.p;
}

template <class R, class G, bool I32>
void launch_spread_atoms(const PmeDev& pm, const NlistDev& nl, const int* order, const double* pos,
                         const double* charge, const SysInfo* sys, G* qgrid, unsigned* status, hipStream_t s) {
    auto chunks = [&](auto kernel, int atoms) {
        hipLaunchKernelGGL(kernel, dim3(nl.nchunks * (PME_CHUNK / atoms)), dim3(ATOM_SPREAD_THREADS), 0, s,
                           nl.chunk_off.p, pm.nsys, order, pos, charge, sys, qgrid, status);
    };
    if (!order)
        hipLaunchKernelGGL((k_spread_direct<R, G, I32>), dim3((5 * pm.natoms + 255) / 256), dim3(256), 0, s, pm.natoms,
                           pos, charge, pm.atom_sys, sys, qgrid, status);
    else if (nl.nchunks < SPREAD_16_CHUNKS)
        chunks(k_spread_atoms<R, G, I32, 16>, 16);
    else if (nl.nchunks < (sizeof(R) == 8 ? SPREAD_32_CHUNKS_F64 : SPREAD_32_CHUNKS))
        chunks(k_spread_atoms<R, G, I32, 32>, 32);
    else
        chunks(k_spread_atoms<R, G, I32, 64>, 64);
}

// Atoms in no order spread by planes where those pay, else by tiles: chunks of them
// fit no box, and each atom then adds to 125 points of the grid, which only few
// atoms do sooner (reciprocal-only calls, by chunks and by tiles: 9,000 atoms 132, 150
// us; 23,550 272, 216; 90,000 1,004, 684; charges on 100^3 points: 8,000 320, 334;
// 16,000 392, 366).
constexpr int UNORDERED_CHUNKS = 12000;
template <class G>
bool by_planes(const PmeDev& pm) {
    return std::is_same<G, double>::value && pm.charges_only && pm.plane_points <= PLANE_POINTS &&
           planes_pay(pm.planes, pm.natoms);
}
bool by_tiles(const PmeDev& pm) { return !pm.spread_atoms || (pm.unordered && pm.natoms > UNORDERED_CHUNKS); }

template <class R, class G, class A>
void run_t(PmeDev& pm, const NlistDev& nl, bool atom_order, const double* pos, const double* charge,
           const SysInfo* sys, G* qgrid,
           R* cgrid, R* phi, const R* roots, const R* moduli, A* force, A* energy, unsigned* status, int phases,
           hipStream_t s) {
    // Bin counts and the charge grid are zero between runs: set so at
    // allocation, and cleared by the first FFT pass after each spread (the
    // grid point by point as the pass reads it), or by fills when a run
    // spreads without transforming.
    const bool own_order = pme_order_ready(pm, nl);
    const int* own = own_order ? pm.order.p + (size_t)pm.order_sel * nl.nslots : nullptr;
    if (phases & PME_SPREAD) {
        const int* order = atom_order ? own : nl.sorted_atom.p;
        const int small = pm.max_charge <= SPREAD32_MAX_CHARGE ? 1 : 0;
        if (by_planes<G>(pm)) {
            if constexpr (std::is_same<G, double>::value)
                hipLaunchKernelGGL(k_spread_planes, dim3(pm.planes), dim3(CHARGE_PLANE_THREADS), 0, s, pm.natoms, pos,
                                   charge, sys, qgrid);
        } else if (!by_tiles(pm)) {
            constexpr bool I32 = sizeof(R) == 4 && SpreadSum<R, G, false>::FIXED;
            if (I32 && small) launch_spread_atoms<R, G, I32>(pm, nl, order, pos, charge, sys, qgrid, status, s);
            else launch_spread_atoms<R, G, false>(pm, nl, order, pos, charge, sys, qgrid, status, s);
        } else {
            R* st_w = pme_weights<R>(pm);
            const int nitems = order ? nl.nslots : pm.natoms;
            hipLaunchKernelGGL((k_pme_bin<R>), dim3((nitems + 255) / 256), dim3(256), 0, s, nitems, order, pos,
                               charge, pm.atom_sys, sys, pm.st_idx.p, st_w, pm.bin_count.p, pm.bins.p, pm.bin_cap,
                               status);
            hipLaunchKernelGGL((k_spread_tiles<R, G>), dim3(pm.ntiles), dim3(SPREAD_THREADS), 0, s, pm.tile_off.p,
                               pm.nsys, sys, pm.st_idx.p, st_w, charge, pm.bin_count.p, pm.bins.p, pm.bin_cap,
                               qgrid, small, status);
            if (!(phases & PME_FFT)) fill_async<int>(pm.bin_count.p, (size_t)pm.ntiles, 0, s);
        }
        if (!(phases & PME_FFT)) fill_async<G>(qgrid, (size_t)pm.qpoints, (G)0, s);
    }
    if (phases & PME_FFT) {
        Cx<R>* cg = reinterpret_cast<Cx<R>*>(cgrid);
        int* clear = (phases & PME_SPREAD) && !by_planes<G>(pm) && by_tiles(pm) ? pm.bin_count.p : nullptr;
        constexpr int prec = sizeof(R) == 8 ? 1 : 0;
        if (pm.dft_blocks[prec][0] > 0) {
            launch_dft<R, G, A>(pm, sys, qgrid, cgrid, phi, roots, moduli, energy, status, s, clear, pm.ntiles);
            clear = nullptr;
        }
        if (pm.plane_blocks[prec] == 0) {
            // Every system takes the matrix-core passes.
        } else if (pm.plane[prec]) {
            launch_plane<R, G, 0>(pm, sys, qgrid, cg, phi, roots, s, clear, pm.ntiles);
            launch_fft<R, G, A, MODE_X_CONV>(pm, sys, qgrid, cg, phi, roots, moduli, energy, status, s);
            launch_plane<R, G, 1>(pm, sys, qgrid, cg, phi, roots, s);
        } else {
            launch_fft<R, G, A, MODE_Z_R2C>(pm, sys, qgrid, cg, phi, roots, moduli, energy, status, s, clear,
                                            pm.ntiles);
            launch_fft<R, G, A, MODE_Y_FWD>(pm, sys, qgrid, cg, phi, roots, moduli, energy, status, s);
            launch_fft<R, G, A, MODE_X_CONV>(pm, sys, qgrid, cg, phi, roots, moduli, energy, status, s);
            launch_fft<R, G, A, MODE_Y_INV>(pm, sys, qgrid, cg, phi, roots, moduli, energy, status, s);
            launch_fft<R, G, A, MODE_Z_C2R>(pm, sys, qgrid, cg, phi, roots, moduli, energy, status, s);
        }
    }
    if (phases & PME_GATHER) {
        // With atom_order the gather follows the same order as the spread:
        // it may then run while a list build rewrites nl.sorted_atom.
        const int* order = atom_order && own_order ? own : nl.sorted_atom.p;
        hipLaunchKernelGGL((k_gather5<R, A>), dim3(nl.nchunks), dim3(GATHER_ATOMS * 5), 0, s, nl.chunk_off.p, pm.nsys,
                           order, pos, charge, sys, phi, force, status);
    }
    OMM_HIP(hipGetLastError());
}

// The mesh potential at the stencil of each listed atom of system 0,
// sum_p phi_p w_x w_y w_z (PmeCache::charge_derivatives, pme.rs:117-137: the
// derivative of the mesh energy with respect to that atom's charge), from the
// FP64 potential of the last FP64 transform.  Eight lanes per listed atom: one
// thread per atom waits for 125 loads a row at a time (1,000 atoms 19.5 us).
__global__ __launch_bounds__(256) void k_mesh_potential(int count, const int* __restrict__ atoms,
                                                        const double* __restrict__ pos,
                                                        const SysInfo* __restrict__ sys,
                                                        const double* __restrict__ phi, double* out) {
    const int k = (blockIdx.x * blockDim.x + threadIdx.x) / 8;
    const SysInfo& S = sys[0];
    const double v = potential_at(pos + 3 * (size_t)atoms[min(k, count - 1)], S.box, S.grid, phi,
                                  (size_t)S.grid[1] * S.grid[2]);
    if (k < count && (threadIdx.x & 7) == 0) out[k] = v;
}

}  // namespace

void pme_potential_at(const PmeDev& pm, const SysInfo* sys_dev, const double* pos, const int* atoms, int count,
                      double* out, hipStream_t s) {
    if (count <= 0) return;
    hipLaunchKernelGGL(k_mesh_potential, dim3((count + 31) / 32), dim3(256), 0, s, count, atoms, pos, sys_dev,
                       pm.phi_d.p, out);
    OMM_HIP(hipGetLastError());
}

std::vector<double> bspline_moduli(int n) {
    // Order-5 spline at integer points: M5(1..4) = 1/24, 11/24, 11/24, 1/24
    // (the weights of a zero fractional coordinate).
    const double w[5] = {1.0 / 24.0, 11.0 / 24.0, 11.0 / 24.0, 1.0 / 24.0, 0.0};
    std::vector<double> values(n);
    for (int k = 0; k < n; ++k) {
        double re = 0.0, im = 0.0;
        for (int i = 0; i < 5; ++i) {
            double t = 2.0 * PI * (double)k * (double)i / (double)n;
            re += w[i] * std::cos(t);
            im += w[i] * std::sin(t);
        }
        values[k] = re * re + im * im;
    }
    for (int k = 0; k < n; ++k)
        if (values[k] < 1e-7) values[k] = 0.5 * (values[(k + n - 1) % n] + values[(k + 1) % n]);
    return values;
}

void pm_set_bin_cap(PmeDev& pm, int cap) {
    pm.bin_cap = cap;
    pm.bins.alloc((size_t)pm.ntiles * cap);
}

void pme_grow_bins(PmeDev& pm) { pm_set_bin_cap(pm, 2 * pm.bin_cap); }

namespace {
// Both halves of each given order.
__global__ void k_copy_order(int n, const int* __restrict__ src, int* a, int* b) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const int v = src[k];
    if (a) a[k] = a[n + k] = v;
    if (b) b[k] = b[n + k] = v;
}
}  // namespace

void pme_follow_order(PmeDev& pm, PmeDev* other, const NlistDev& nl, hipStream_t s) {
    const size_t n2 = 2 * (size_t)nl.nslots;
    int* a = nl.nslots > 0 && pm.order.n == n2 ? pm.order.p : nullptr;
    int* b = nl.nslots > 0 && other && other->order.n == n2 ? other->order.p : nullptr;
    if (!a && !b) return;
    hipLaunchKernelGGL(k_copy_order, dim3((nl.nslots + 255) / 256), dim3(256), 0, s, nl.nslots, nl.sorted_atom.p, a,
                       b);
    OMM_HIP(hipGetLastError());
    if (a) pm.order_gen = nl.generation;
    if (b) other->order_gen = nl.generation;
}

bool pme_order_ready(const PmeDev& pm, const NlistDev& nl) {
    return nl.nslots > 0 && pm.order_gen == nl.generation && pm.order.n == 2 * (size_t)nl.nslots;
}

int* pme_next_order(PmeDev& pm, const NlistDev& nl) {
    pm.order_sel ^= 1;
    return pm.order.p + (size_t)pm.order_sel * nl.nslots;
}

void pme_take_order(PmeDev& pm, const NlistDev& nl, hipStream_t s) {
    if (nl.nslots == 0 || nl.sorted_atom.n < (size_t)nl.nslots) return;
    if (pm.order.n != 2 * (size_t)nl.nslots) pm.order.alloc(2 * (size_t)nl.nslots);
    pm.order_gen = -1;  // pme_follow_order sets it
    pme_follow_order(pm, nullptr, nl, s);
}

namespace {
const int PASS_AXIS[5] = {2, 1, 0, 1, 2};  // MODE_Z_R2C, Y_FWD, X_CONV, Y_INV, Z_C2R

int fft_nlines(const SysInfo& S, int a) {
    // z passes: pairs of real lines, (ny + 1) / 2 per x plane.
    return a == 0 ? S.grid[1] * S.nzh : (a == 1 ? S.grid[0] * S.nzh : S.grid[0] * ((S.grid[1] + 1) / 2));
}
}  // namespace

namespace {
// Workgroup tables and LDS of the matrix-core passes.
void dft_setup(PmeDev& pm, const std::vector<SysInfo>& sys, hipStream_t s) {
    pm.shape = MeshShape::of(sys[0]);
    for (int prec = 0; prec < 2; ++prec) {
        pm.dft_wide[prec] = false;
        for (const SysInfo& S : sys)
            for (int a = 0; a < 3; ++a)
                if (dft_system(S, prec) && S.grid[a] > 16 * DFT_WAVES) pm.dft_wide[prec] = true;
        const int waves = pm.dft_wide[prec] ? DFT_WAVES_WIDE : DFT_WAVES;
        std::vector<int> off[3];
        size_t lds[3] = {0, 0, 0};
        for (int k = 0; k < 3; ++k) off[k].assign(1, 0);
        for (const SysInfo& S : sys) {
            const bool on = dft_system(S, prec);
            const int nx = S.grid[0], ny = S.grid[1], nz = S.grid[2], tiles = dft_tiles(S.nzh);
            const int blocks[3] = {nx * tiles, ny * tiles, nx * ((ny + 15) / 16)};
            const size_t need[3] = {DftLds::zy(ny, nz, waves), DftLds::x(nx), DftLds::yz(ny, nz, tiles, waves)};
            for (int k = 0; k < 3; ++k) {
                off[k].push_back(off[k].back() + (on ? blocks[k] : 0));
                if (on) lds[k] = std::max(lds[k], need[k]);
            }
        }
        for (int k = 0; k < 3; ++k) {
            if (pm.nsys > 1) pm.dft_off[prec][k].upload(off[k], s);  // a lone system's workgroups start at 0
            pm.dft_blocks[prec][k] = off[k].back();
            pm.dft_shmem[prec][k] = lds[k] * (prec ? sizeof(double) : sizeof(float));
        }
    }
    // Dynamic LDS above 64 KB per workgroup.
    auto allow = [&](const void* f, int prec, int k) {
        if (pm.dft_shmem[prec][k] > 64 * 1024)
            OMM_HIP(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)PLANE_LDS_MAX));
    };
    allow((const void*)&k_dft_zy<DFT_WAVES_WIDE, float, long long>, 0, 0);
    allow((const void*)&k_dft_zy<DFT_WAVES_WIDE, double, long long>, 1, 0);
    allow((const void*)&k_dft_zy<DFT_WAVES_WIDE, double, double>, 1, 0);
    allow((const void*)&k_dft_yz<DFT_WAVES_WIDE, float>, 0, 2);
    allow((const void*)&k_dft_yz<DFT_WAVES_WIDE, double>, 1, 2);
}
}  // namespace

int pme_set_fft_lines(PmeDev& pm, std::vector<SysInfo>& sys, int prec, int cap, hipStream_t s) {
    const size_t csize = prec ? 2 * sizeof(double) : 2 * sizeof(float);
    if (cap <= 0) {
        // The most lines that fit in LDS, lowered for the whole batch until
        // every pass has ~2048 workgroups (8 per CU) or two lines each.
        for (cap = 16;; cap >>= 1) {
            long long fewest = LLONG_MAX;
            for (int k = 0; k < 5; ++k) {
                long long blocks = 0;
                for (const SysInfo& S : sys) {
                    const int a = PASS_AXIS[k];
                    const int l = std::min(cap, max_lines(S.grid[a], csize));
                    blocks += (fft_nlines(S, a) + l - 1) / l;
                }
                fewest = std::min(fewest, blocks);
            }
            if (fewest >= 2048 || cap <= 2) break;
        }
    }
    std::vector<int> off[5];
    for (int k = 0; k < 5; ++k) off[k].assign(1, 0);
    for (int a = 0; a < 3; ++a) pm.fft_shmem[prec][a] = 0;
    for (SysInfo& S : sys) {
        for (int a = 0; a < 3; ++a) {
            S.fft_lines[prec][a] = std::min(cap, max_lines(S.grid[a], csize));
            pm.fft_shmem[prec][a] =
                std::max(pm.fft_shmem[prec][a], (2 * (size_t)S.fft_lines[prec][a] * S.grid[a] + S.grid[a]) * csize);
        }
        for (int k = 0; k < 5; ++k) {
            const int l = S.fft_lines[prec][PASS_AXIS[k]];
            const int blocks = (fft_nlines(S, PASS_AXIS[k]) + l - 1) / l;
            off[k].push_back(off[k].back() + (dft_system(S, prec) ? 0 : blocks));
        }
    }
    for (int k = 0; k < 5; ++k) {
        pm.fft_off[prec][k].upload(off[k], s);
        pm.fft_blocks[prec][k] = off[k].back();
    }
    pm.fft_cap[prec] = cap;
    return cap;
}

bool pme_set_fft_plane(PmeDev& pm, std::vector<SysInfo>& sys, int prec, int use) {
    const size_t csize = prec ? 2 * sizeof(double) : 2 * sizeof(float);
    size_t shmem = 0;
    bool ok = use != 0 && !sys.empty();
    for (SysInfo& S : sys) {
        if (!ok) break;
        const int ny = S.grid[1], nz = S.grid[2], nzh = S.nzh;
        // y lines per call: all of the half spectrum's lines when the threads
        // of a line stay at most ny, fewer calls otherwise; z line pairs per call:
        // as many as fit, down to the fewest that keep the threads of a line
        // at most nz.
        auto pow2_at_least = [](int v) {
            int p = 1;
            while (p < v) p <<= 1;
            return p;
        };
        const int ly = std::min(PLANE_THREADS, std::max(pow2_at_least(nzh), pow2_at_least((PLANE_THREADS + ny - 1) / ny)));
        const int lz_min = std::min(PLANE_THREADS, pow2_at_least((PLANE_THREADS + nz - 1) / nz));
        int lz = std::min(PLANE_THREADS, std::max(lz_min, pow2_at_least((ny + 1) / 2)));
        while (lz > lz_min && plane_layout(ny, nz, nzh, lz, ly).elems * csize > PLANE_LDS_MAX) lz >>= 1;
        const size_t bytes = plane_layout(ny, nz, nzh, lz, ly).elems * csize;
        if (bytes > PLANE_LDS_MAX) {
            ok = false;
            break;
        }
        S.plane_lines[prec][0] = lz;
        S.plane_lines[prec][1] = ly;
        shmem = std::max(shmem, bytes);
    }
    pm.plane[prec] = ok;
    pm.plane_shmem[prec] = ok ? shmem : 0;
    return ok;
}

int pme_set_spread_edge(PmeDev& pm, std::vector<SysInfo>& sys, int edge, hipStream_t s) {
    if (edge <= 0) {
        edge = 8;
        for (int e : {8, 6}) {
            long long total = 0;
            for (const SysInfo& S : sys)
                total += (long long)tiles_for(S.grid[0], e) * tiles_for(S.grid[1], e) * tiles_for(S.grid[2], e);
            edge = e;
            if (total >= SPREAD_MIN_TILES) break;
        }
    }
    std::vector<int> toff{0};
    int bin_cap = 64;
    for (SysInfo& S : sys) {
        S.ptile = edge;
        for (int a = 0; a < 3; ++a) S.tiles[a] = tiles_for(S.grid[a], edge);
        S.tile_off = toff.back();
        const int nt = S.tiles[0] * S.tiles[1] * S.tiles[2];
        toff.push_back(toff.back() + nt);
        // Twice the atoms of the largest tile at the system's mean density
        // (the last tile of an axis is up to twice as wide as the others).
        double largest = 1.0;
        for (int a = 0; a < 3; ++a) {
            const int last = S.grid[a] - (S.tiles[a] - 1) * edge;
            largest *= (double)std::max(last, std::min(edge, S.grid[a])) / (double)S.grid[a];
        }
        bin_cap = std::max(bin_cap, (int)(2.0 * largest * S.n) + 64);
    }
    pm.ntiles = toff.back();
    pm.tile_off.upload(toff, s);
    pm.bin_count.alloc((size_t)pm.ntiles);
    fill_async<int>(pm.bin_count.p, (size_t)pm.ntiles, 0, s);
    pm_set_bin_cap(pm, bin_cap);
    pm.spread_edge = edge;
    return edge;
}

void pme_setup(PmeDev& pm, std::vector<SysInfo>& sys, int natoms, const int* atom_sys, bool mixed, hipStream_t s) {
    const int nsys = (int)sys.size();
    pm.nsys = nsys;
    pm.natoms = natoms;
    pm.atom_sys = atom_sys;
    // Until an autotuner chooses: atom-owned (9,000 atoms with FP64 stencils, 9 us
    // against 50 for the tiles).
    pm.spread_atoms = true;
    pm.planes = nsys == 1 ? sys[0].grid[0] : 0;
    pm.plane_points = nsys == 1 ? sys[0].grid[1] * sys[0].grid[2] : INT_MAX;
    std::vector<double> roots, moduli;
    long long qpts = 0, cpts = 0;
    for (int si = 0; si < nsys; ++si) {
        SysInfo& S = sys[si];
        for (int a = 0; a < 3; ++a)
            if (S.grid[a] < 5 || S.grid[a] > 1024)
                throw Error(OMM_ERR_INVALID, "PME grid dimensions must be in [5, 1024]");
        S.nzh = S.grid[2] / 2 + 1;
        S.qgrid_off = qpts;
        S.cgrid_off = cpts;
        qpts += (long long)S.grid[0] * S.grid[1] * S.grid[2];
        // The matrix-core passes pad kz to whole tiles.
        cpts += (long long)S.grid[0] * S.grid[1] * (dft_system(S, 0) || dft_system(S, 1) ? DFT_COLS * dft_tiles(S.nzh) : S.nzh);
        for (int a = 0; a < 3; ++a) {
            const int n = S.grid[a];
            std::vector<int> f = factorize(n);
            if ((int)f.size() >= MAX_STAGES) throw Error(OMM_ERR_INVALID, "PME grid dimension has too many factors");
            for (int k = 0; k < MAX_STAGES; ++k) S.radix[a][k] = k < (int)f.size() ? f[k] : 0;
            S.roots_off[a] = (int)(roots.size() / 2);
            for (int m = 0; m < n; ++m) {
                double t = -2.0 * PI * (double)m / (double)n;
                roots.push_back(std::cos(t));
                roots.push_back(std::sin(t));
            }
            S.moduli_off[a] = (int)moduli.size();
            auto mod = bspline_moduli(n);
            moduli.insert(moduli.end(), mod.begin(), mod.end());
        }
    }
    pm.qpoints = qpts;
    pm.cpoints = cpts;
    // Default grouping: the largest line cap with ~2048 workgroups per FFT
    // pass, and the largest spread tile edge with SPREAD_MIN_TILES tiles.
    pme_set_fft_lines(pm, sys, 0, 0, s);
    pme_set_fft_lines(pm, sys, 1, 0, s);
    {
        for (int prec = 0; prec < 2; ++prec) {
            std::vector<int> poff{0};
            for (const SysInfo& S : sys) poff.push_back(poff.back() + (dft_system(S, prec) ? 0 : S.grid[0]));
            pm.plane_off[prec].upload(poff, s);
            pm.plane_blocks[prec] = poff.back();
        }
        // Dynamic LDS above 64 KB per workgroup.
        const int lds = (int)PLANE_LDS_MAX;
        OMM_HIP(hipFuncSetAttribute((const void*)&k_fft_plane<float, long long, 0>,
                                    hipFuncAttributeMaxDynamicSharedMemorySize, lds));
        OMM_HIP(hipFuncSetAttribute((const void*)&k_fft_plane<float, long long, 1>,
                                    hipFuncAttributeMaxDynamicSharedMemorySize, lds));
        OMM_HIP(hipFuncSetAttribute((const void*)&k_fft_plane<double, long long, 0>,
                                    hipFuncAttributeMaxDynamicSharedMemorySize, lds));
        OMM_HIP(hipFuncSetAttribute((const void*)&k_fft_plane<double, long long, 1>,
                                    hipFuncAttributeMaxDynamicSharedMemorySize, lds));
        OMM_HIP(hipFuncSetAttribute((const void*)&k_fft_plane<double, double, 0>,
                                    hipFuncAttributeMaxDynamicSharedMemorySize, lds));
        OMM_HIP(hipFuncSetAttribute((const void*)&k_fft_plane<double, double, 1>,
                                    hipFuncAttributeMaxDynamicSharedMemorySize, lds));
        for (int prec = 0; prec < 2; ++prec) pme_set_fft_plane(pm, sys, prec, -1);
    }
    dft_setup(pm, sys, s);
    pme_set_spread_edge(pm, sys, 0, s);
    pm.st_idx.alloc(4 * (size_t)pm.natoms);
    if (mixed) pm.st_wf.alloc(16 * (size_t)pm.natoms);
    pm.st_wd.alloc(16 * (size_t)pm.natoms);
    pm.roots_d.upload(roots, s);
    pm.moduli_d.upload(moduli, s);
    pm.cgrid_d.alloc(2 * (size_t)cpts);
    pm.phi_d.alloc((size_t)qpts);
    if (mixed) {
        std::vector<float> rf(roots.begin(), roots.end()), mf(moduli.begin(), moduli.end());
        pm.roots_f.upload(rf, s);
        pm.moduli_f.upload(mf, s);
        pm.qgrid_fx.alloc((size_t)qpts);
        fill_async<long long>(pm.qgrid_fx.p, (size_t)qpts, 0ll, s);
        pm.cgrid_f.alloc(2 * (size_t)cpts);
        pm.phi_f.alloc((size_t)qpts);
    } else {
        pm.qgrid_d.alloc((size_t)qpts);
        fill_async<double>(pm.qgrid_d.p, (size_t)qpts, 0.0, s);
    }
    OMM_HIP(hipStreamSynchronize(s));
}

void pme_run(PmeDev& pm, int mode, const NlistDev& nl, const double* pos, const double* charge,
             const SysInfo* sys_dev, long long* force_fx, double* force_d, long long* energy_fx, double* energy_d,
             unsigned* status, hipStream_t s, int phases, bool atom_order) {
    if (mode == MESH_F32)
        run_t<float, long long, long long>(pm, nl, atom_order, pos, charge, sys_dev, pm.qgrid_fx.p, pm.cgrid_f.p, pm.phi_f.p,
                                           pm.roots_f.p, pm.moduli_f.p, force_fx, energy_fx, status, phases, s);
    else if (mode == MESH_F64_FIXED)
        run_t<double, long long, long long>(pm, nl, atom_order, pos, charge, sys_dev, pm.qgrid_fx.p, pm.cgrid_d.p, pm.phi_d.p,
                                            pm.roots_d.p, pm.moduli_d.p, force_fx, energy_fx, status, phases, s);
    else
        run_t<double, double, double>(pm, nl, atom_order, pos, charge, sys_dev, pm.qgrid_d.p, pm.cgrid_d.p, pm.phi_d.p,
                                      pm.roots_d.p, pm.moduli_d.p, force_d, energy_d, status, phases, s);
}

}  // namespace ommhip
