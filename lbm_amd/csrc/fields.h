// Transfer of per-cell values between the storage order of the device (layout.h: rows along ax0) and
// the reference's order (i fastest, ghost layers included), as the C ABI's arrays have it.
//
// Both sides are bound by memory, and one of them is strided for any plain thread-per-cell kernel:
// with j contiguous, 64 lanes along i read 64 different rows of every population.  A block therefore
// takes a tile of kTile cells, TI along i and TA along the storage axis, walks it once in each order
// and turns it in LDS, so that both sides move whole segments (TA = 32: 128 bytes of 4-byte values
// per row and population; TI = 8: 32 bytes of a field or 8 cells of a population record).  A row
// of the tile is padded by one value, which spreads the column accesses over the banks.  With i
// contiguous no turn is needed: the tile is 64 cells along i.  Measured on MI355X, one call each,
// D3Q27 FP32 384x192x128 with j contiguous, thread-per-cell kernels -> these: moments out
// 1718 -> 370 us, equilibrium start 3872 -> 854 us; D3Q19 FP32 192x96x96: record in 1029 -> 186 us.
// Averages, forcing fields and the adjoint's gradient, which the host turned one cell at a time (180,
// 114 and about 15 ms at these sizes), take 20 to 300 us here.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>
#include <type_traits>

#include "layout.h"

namespace lbm {

constexpr int kTile = 256;   // cells of a tile, threads of a block

struct TileShape {
    int li, la;   // log2 of the cells along i and along the storage axis a
    int axa, axb; // the axes of a and of the tile's plane
    int pad;      // LDS values between rows of the tile
};

inline TileShape tile_shape(const Layout& L) {
    if (L.ax0 == 0) return {6, 2, 1, 2, 0};
    return {3, 5, L.ax0, 3 - L.ax0, 1};
}
inline dim3 tile_grid(const Layout& L, const TileShape& T) {
    return dim3((L.nx + 2 + (1 << T.li) - 1) >> T.li, (L.n(T.axa) + 2 + (1 << T.la) - 1) >> T.la, L.n(T.axb) + 2);
}

// The tile of this block: first cell and what of it lies in the padded grid.
struct Tile {
    int i0, a0, b, ni, na;
    __device__ Tile(const Layout& L, const TileShape& T) {
        i0 = blockIdx.x << T.li;
        a0 = blockIdx.y << T.la;
        b = blockIdx.z;
        const int mi = L.nx + 2 - i0, ma = L.n(T.axa) + 2 - a0;
        ni = mi < (1 << T.li) ? mi : 1 << T.li;
        na = ma < (1 << T.la) ? ma : 1 << T.la;
    }
    // cell of this thread in storage order; false outside the grid
    __device__ bool cell(const TileShape& T, int& il, int& al) const {
        const int t = threadIdx.x;
        if (T.pad) {
            al = t & ((1 << T.la) - 1);
            il = t >> T.la;
        } else {
            il = t & ((1 << T.li) - 1);
            al = t >> T.li;
        }
        return il < ni && al < na;
    }
    __device__ void ijk(const TileShape& T, int il, int al, int x[3]) const {
        x[0] = i0 + il;
        x[T.axa] = a0 + al;
        x[T.axb] = b;
    }
};

// Element of the reference's cell arrays.
__device__ __forceinline__ size_t ref_cell(const Layout& L, const int x[3]) {
    return ((size_t)x[2] * (L.ny + 2) + x[1]) * (L.nx + 2) + x[0];
}

// Tile elements in the reference's order: calls f(place in LDS, element in memory) for every value of
// the tile, consecutive threads on consecutive values.  AOS: NV values per cell; otherwise NV arrays
// plane elements apart.  CLAMP: a ghost cell stands for the interior cell next to it.
template <int NV, bool AOS, bool CLAMP, class F>
__device__ __forceinline__ void tile_ref(const Layout& L, const TileShape& T, const Tile& t, size_t plane, F f) {
    constexpr int N = AOS ? NV : 1;   // values of a cell next to each other
    const int row = N << T.li;
    for (int e = threadIdx.x; e < NV * kTile; e += kTile) {
        const int v = AOS ? 0 : e >> 8;
        const int w = AOS ? e : e & (kTile - 1);
        const int al = (w / N) >> T.li;
        const int r = w - al * row;
        if (al >= t.na || r >= t.ni * N) continue;
        int x[3];
        t.ijk(T, 0, al, x);
        size_t g;
        if (CLAMP) {
            x[0] += r;
            const int n[3] = {L.nx, L.ny, L.nz};
#pragma unroll
            for (int d = 0; d < 3; ++d) x[d] = x[d] < 1 ? 1 : x[d] > n[d] ? n[d] : x[d];
            g = ref_cell(L, x);
        } else {
            g = ref_cell(L, x) * N + r;
        }
        f(v * (kTile + (T.pad << T.la)) + al * (row + T.pad) + r, (size_t)v * plane + g);
    }
}
// Place in LDS of value v of cell (il, al).
template <int NV, bool AOS>
__device__ __forceinline__ int tile_place(const TileShape& T, int il, int al, int v) {
    if (AOS) return al * ((NV << T.li) + T.pad) + il * NV + v;
    return v * (kTile + (T.pad << T.la)) + al * ((1 << T.li) + T.pad) + il;
}
template <int NV, bool AOS>
constexpr int kTileValues = AOS ? NV * kTile + 32 : NV * (kTile + 32);

// f(i, j, k, v): the NV values of a cell.
template <int NV, bool AOS, typename H, class F>
__global__ void __launch_bounds__(kTile) cells_out_kernel(const Layout L, const TileShape T, const F f, H* __restrict__ out,
                                                          size_t plane) {
    __shared__ H sm[kTileValues<NV, AOS>];
    const Tile t(L, T);
    int il, al;
    if (t.cell(T, il, al)) {
        int x[3];
        t.ijk(T, il, al, x);
        H v[NV];
        f(L, x[0], x[1], x[2], v);
#pragma unroll
        for (int q = 0; q < NV; ++q) sm[tile_place<NV, AOS>(T, il, al, q)] = v[q];
    }
    __syncthreads();
    tile_ref<NV, AOS, false>(L, T, t, plane, [&](int s, size_t g) { out[g] = sm[s]; });
}

// f(i, j, k, v) takes the NV values of a cell.
template <int NV, bool AOS, bool CLAMP, typename H, class F>
__global__ void __launch_bounds__(kTile) cells_in_kernel(const Layout L, const TileShape T, const F f,
                                                         const H* __restrict__ in, size_t plane) {
    __shared__ H sm[kTileValues<NV, AOS>];
    const Tile t(L, T);
    tile_ref<NV, AOS, CLAMP>(L, T, t, plane, [&](int s, size_t g) { sm[s] = in[g]; });
    __syncthreads();
    int il, al;
    if (!t.cell(T, il, al)) return;
    int x[3];
    t.ijk(T, il, al, x);
    H v[NV];
#pragma unroll
    for (int q = 0; q < NV; ++q) v[q] = sm[tile_place<NV, AOS>(T, il, al, q)];
    f(L, x[0], x[1], x[2], v);
}

template <int NV, bool AOS, typename H, class F>
hipError_t cells_out(const Layout& L, const F& f, H* out, hipStream_t s) {
    const TileShape T = tile_shape(L);
    const size_t plane = (size_t)(L.nx + 2) * (L.ny + 2) * (L.nz + 2);
    hipLaunchKernelGGL((cells_out_kernel<NV, AOS, H, F>), tile_grid(L, T), dim3(kTile), 0, s, L, T, f, out, plane);
    return hipGetLastError();
}
template <int NV, bool AOS, bool CLAMP, typename H, class F>
hipError_t cells_in(const Layout& L, const F& f, const H* in, hipStream_t s) {
    const TileShape T = tile_shape(L);
    const size_t plane = (size_t)(L.nx + 2) * (L.ny + 2) * (L.nz + 2);
    hipLaunchKernelGGL((cells_in_kernel<NV, AOS, CLAMP, H, F>), tile_grid(L, T), dim3(kTile), 0, s, L, T, f, in, plane);
    return hipGetLastError();
}

// Whether a cell of the padded grid is a fluid or solid cell of the interior.
__device__ __forceinline__ bool interior_cell(const Layout& L, int i, int j, int k) {
    return i >= 1 && i <= L.nx && j >= 1 && j <= L.ny && k >= 1 && k <= L.nz;
}

// Time averages and turbulence intensity from the six sums (src/m_averaging_full_kernelfin.F90:46-60),
// zero in ghost cells.  The means are quotients in FP64 rounded to R, as are the mean squares; the
// variances are differences of those in R, not contracted.
template <typename S>
struct AveragesOut {
    using R = std::conditional_t<sizeof(S) == 4, float, double>;   // a tangent value's own part
    const S* avg;
    double count;
    template <typename H>
    __device__ void operator()(const Layout& L, int i, int j, int k, H (&o)[4]) const {
#pragma clang fp contract(off)
        o[0] = o[1] = o[2] = o[3] = H(0);
        if (!interior_cell(L, i, j, k)) return;
        const size_t c = (size_t)L.cidx(i, j, k);
        const size_t P = (size_t)L.cplane;
        double t = 0.0;
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            const R m = (R)((double)avg[q * P + c] / count);
            const R m2 = (R)((double)avg[(3 + q) * P + c] / count);
            const R var = m2 - m * m;
            t += var > R(0) ? (double)var : 0.0;
            o[q] = (H)m;
        }
        const R third = (R)t / R(3);
        o[3] = (H)::sqrt(third > R(0) ? third : R(0));   // lbm::sqrt is the tangent type's
    }
};

// Reference-order reals (NV per cell) into NV per-cell arrays of the compute type.
template <int NV, typename R>
struct CellsIn {
    R* to[NV];
    template <typename H>
    __device__ void operator()(const Layout& L, int i, int j, int k, const H (&v)[NV]) const {
        const int c = L.cidx(i, j, k);
#pragma unroll
        for (int q = 0; q < NV; ++q) to[q][c] = (R)v[q];
    }
};

// The adjoint's force gradient, zero in ghost cells.
struct GradientOut {
    const double* g;
    __device__ void operator()(const Layout& L, int i, int j, int k, double (&o)[3]) const {
        const bool in = interior_cell(L, i, j, k);
        const size_t c = (size_t)L.cidx(i, j, k);
#pragma unroll
        for (int q = 0; q < 3; ++q) o[q] = in ? g[q * (size_t)L.cplane + c] : 0.0;
    }
};

}  // namespace lbm
