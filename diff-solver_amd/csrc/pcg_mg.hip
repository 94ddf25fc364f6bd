// pcg_mg.hip — conjugate gradients preconditioned by an aggregation multigrid V-cycle
// (DS_CG_MULTIGRID): the same pressure system as the Jacobi forms (the reference solves it with
// Jacobi-preconditioned CG, solvers/smoke/operators.cu), to the same FP64 stopping test on the true
// residual, in about ten iterations instead of about a thousand at 128^3.
//
// Hierarchy: each coarser level aggregates 2 x 2 x 2 cells of the finer one (an odd extent leaves
// a last aggregate one cell wide; an extent of 1 stays 1). The prolongation P copies a coarse value
// to the aggregate's cells and the restriction is its transpose (the cells' sum), so the coarse
// operator A_c = P^T A P sums the fine couplings over the aggregates: a 7-point operator again, held
// as its diagonal and the per-axis couplings to the + neighbour, built once per context on the host
// from the connectivity code (periodic wraps included). The coarsest level (at most kMgDense cells)
// is solved exactly with its inverse (FP64 Cholesky on the host, applied in FP64); a grid of at most
// kMgCoarsest cells is its own coarsest level.
//
// V-cycle (symmetric, so a valid CG preconditioner): on every level two Jacobi sweeps from zero
// weighted as the second Chebyshev polynomial on [0.45, 2] (D^-1 A has its spectrum in [0, 2]; the
// lower end is where the smoother hands over to the coarse level), the residual restricted, the
// coarse correction scaled by 1.9 (piecewise-constant aggregation under-corrects smooth errors:
// its coarse operator is about twice too stiff), the two sweeps again in the reverse order. An FP64
// CPU model (random and smooth right-hand sides, 64^3 to 128^3, with and without solids) needs 7 to
// 10 iterations to 1e-6 this way; with the equal weights of 0.9, one sweep on the coarser levels and
// corrections of 1.8 and 1.5 that this file used before, 11 to 17; Jacobi-PCG 1015 at 128^3.
//
// The outer loop is textbook PCG with two reductions per iteration. Level 0 costs three kernels per
// iteration, each staging its brick of cells and the halo that its chain of stencils needs in LDS:
//   direction   p = z + beta p_old, <p, A p>                                         (halo 1)
//   down        x += alpha p, r -= alpha A p, ||r||^2; both sweeps; restriction      (halo 3 of p)
//   post        prolongation, both sweeps, <r, z>                                    (halo 2)
// The halo's values are recomputed instead of exchanged. A coarser level of more than kMgBottomCells
// costs two kernels of the same build; the levels below run in one workgroup that keeps them in LDS
// (a 16^3 grid fills one CU, and a launch costs more than its sweeps). Every scalar comes from FP64
// per-block partials that each consumer block reduces in the same order, so the iteration is
// deterministic. Every kernel returns at once after the stopping test has fired.
// Measured (128^3, kernel trace): 8 launches and about 110 us an iteration, 9 iterations from x0 = 0,
// where thirteen launches took 108 us and 19 iterations; 64^3: 6 launches, 40 us, 8 iterations against
// 11, 50 us, 12; 256^3: 620 us, 11 iterations against 720 us, 24.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <bit>
#include <cmath>
#include <cstdint>
#include <type_traits>
#include <utility>
#include <vector>

#include "context.hpp"

namespace ds {

namespace {

// 1 / (centre -+ half width cos(pi / 4)) of [0.45, 2]: the roots of the second Chebyshev polynomial.
constexpr float kCheb[2]{0.564013325f, 1.477121796f};
constexpr float kOver = 1.9f;   // scale of the prolonged coarse correction
constexpr uint32_t kMgDotThreads = 512;
// Boxes of level 0 and of a coarser level by its cells. The lines lie where the two sides are within 5 % of
// each other (steps, us): large 545 and medium 502 at 64^3, 708 and 702 at 80 x 80 x 81, 720 and 740 at
// 81 x 81 x 82, 735 and 757 at 90 x 70 x 110, 963 and 910 at 100^3, 1005 and 995 at 102^3; medium 420 and small 424
// at 40^3, 426 and 432 at 41 x 40 x 40, 433 and 437 at 48^3; a coarser level's large and small at 65600 cells 731 and
// 702, at 131072 844 and 818, at 175616 1105 and 1076.
constexpr uint32_t kMgLargeCells = 1u << 19, kMgMediumCells = 1u << 16;
constexpr uint32_t kMgCoarseLarge = 1u << 17;

// 1 / d for a level-0 diagonal count (the hardware reciprocal: every use of a cell's value is the
// same, so the smoother stays symmetric). Counts of 0 (not an unknown) give 1; the values they scale
// are 0 there.
__device__ __forceinline__ float mg_dinv(uint32_t d) { return __builtin_amdgcn_rcpf((float)max(d, 1u)); }

// A box of cells handled by a workgroup of T threads. With a halo of H cells its planes are
// X(H) x Y(H) points, Z(H) of them. A thread owns one column (x, y) of the halo-2 planes for the whole
// kernel and walks z: coordinates, wraps and bounds of x and y are formed once per box, those of z are
// uniform, and a column's own values and its z neighbours stay in registers; LDS serves the four
// neighbours in the plane. (One thread per tile element, decoding each, took 3.5 times the
// instructions and 63 instead of 32 us for the down kernel at 128^3.)
template <int BX_, int BY_, int BZ_, int T_>
struct Box {
    static constexpr int BX = BX_, BY = BY_, BZ = BZ_, T = T_;
    template <int H>
    static constexpr int X = BX + 2 * H;
    template <int H>
    static constexpr int Y = BY + 2 * H;
    template <int H>
    static constexpr int Z = BZ + 2 * H;
    template <int H>
    static constexpr int P = X<H> * Y<H>;
    static_assert(T % 64 == 0 && T >= P<2>, "one column per thread");
    struct Grid {   // the boxes that cover a level
        uint32_t nx, ny, count;
    };
    static __host__ __device__ Grid grid(const MgLevel& L) {
        const uint32_t nx = (uint32_t)(L.nx + BX - 1) / BX, ny = (uint32_t)(L.ny + BY - 1) / BY;
        return Grid{nx, ny, nx * ny * ((uint32_t)(L.nz + BZ - 1) / BZ)};
    }
    static __device__ __forceinline__ void origin(const Grid& g, uint32_t b, int& x, int& y, int& z) {
        const uint32_t r = b / g.nx;
        x = (int)(b - r * g.nx) * BX;
        const uint32_t q = r / g.ny;
        y = (int)(r - q * g.ny) * BY;
        z = (int)q * BZ;
    }
};
// Level 0 (large, medium, small grids) and the coarser levels (large, small). 32 x 8 x 8 keeps the
// halo's share of the work low (2.5 times the cells with a halo of 2); smaller boxes fill the 256 CUs
// of a small grid.
using BoxL = Box<32, 8, 8, 448>;
using BoxM = Box<16, 8, 4, 256>;
using BoxS = Box<16, 4, 4, 192>;
using BoxC = Box<16, 8, 8, 256>;
using BoxD = Box<8, 8, 4, 192>;
// Large grids of a few cells along x or z, level 0 and coarser. In a box of 32 x 8 x 8 the kernels load
// and sweep 12 planes for one plane of cells, and 36 columns for one along x. Steps with it, with these
// boxes, and with kernels of one thread per cell: 1024 x 1024 x 1 2257, 1490, 2135 us; 2 x 1024 x 1024
// 6735, 2198, 2928; 3 x 1024 x 1024 7254, 3118, 4066; 6 x 1024 x 1024 8039, 4386, 6855; 512 x 512 x 2
// 977, 789, 1442. (Thin along x: 4 x 32 x 8 3124, 8 x 16 x 8 3352, 4 x 64 x 4 3068 us at 2 x 1024 x 1024.)
// Along y the cubic box does: 1024 x 2 x 1024 2350 against 2638 us.
using BoxLX = Box<2, 64, 8, 448>;
using BoxLZ = Box<32, 16, 2, 768>;
using BoxCX = Box<2, 32, 8, 256>;
using BoxCZ = Box<16, 16, 2, 448>;

// Column (x, y) of a level, wrapped along the periodic axes: its offset in a plane, and whether it
// lies in the grid and is the thread's to handle (the offset is 0 when not).
struct Column {
    uint32_t at;
    bool in;
};
__device__ __forceinline__ Column mg_column(const MgLevel& L, uint32_t per, int x, int y, bool mine = true) {
    if (per & 1u) x = wrapi(x, L.nx);
    if (per & 2u) y = wrapi(y, L.ny);
    Column c;
    c.in = mine && (unsigned)x < (unsigned)L.nx && (unsigned)y < (unsigned)L.ny;
    c.at = c.in ? (uint32_t)x + __umul24((uint32_t)y, (uint32_t)L.nx) : 0u;
    return c;
}
// N consecutive planes of a level from z0 on (uniform over the workgroup), wrapped along a periodic
// axis: first elements, and the set that lies in the grid (offset 0 else). Formed once per box: the
// scalar unit's instructions bound these kernels when every access formed its own.
template <int N>
struct Planes {
    uint32_t at[N], in;
};
template <int N>
__device__ __forceinline__ Planes<N> mg_planes(const MgLevel& L, uint32_t per, int z0) {
    Planes<N> p;
    p.in = 0u;
    const uint32_t stride = (uint32_t)L.nx * (uint32_t)L.ny;
#pragma unroll
    for (int k = 0; k < N; ++k) {
        int z = z0 + k;
        if (per & 4u) z = wrapi(z, L.nz);
        const bool in = (unsigned)z < (unsigned)L.nz;
        p.at[k] = in ? (uint32_t)z * stride : 0u;
        p.in |= in ? 1u << k : 0u;
    }
    return p;
}
// Element i of v. The byte offset stays a 32-bit register beside a uniform base (a level has at most
// 2^30 cells of 4 bytes).
template <typename V>
__device__ __forceinline__ V& mg_at(V* v, uint32_t i) {
    return *reinterpret_cast<V*>(reinterpret_cast<std::conditional_t<std::is_const_v<V>, const char, char>*>(v) + i * (uint32_t)sizeof(V));
}
template <typename V, int N>
__device__ __forceinline__ V mg_load(const V* __restrict__ v, const Planes<N>& p, int k, const Column& c) {
    const V l = mg_at(v, c.at + p.at[k]);
    return (p.in >> k & 1u) && c.in ? l : (V)0;
}

struct Pair2 {   // double-buffered vector: iteration k's value is p[k & 1]
    float* p[2];
};

// The aggregates' values over N planes of a column, from plane z0 (even) of the finer level on (nz its
// planes): one aggregate serves two planes unless a periodic axis wraps in between.
template <int N>
__device__ __forceinline__ void mg_load_coarse(const MgLevel& C, uint32_t per, int z0, int nz, const float* __restrict__ e, const Column& cc,
                                               float (&v)[N]) {
    const uint32_t stride = (uint32_t)C.nx * (uint32_t)C.ny;
#pragma unroll
    for (int k = 0; k < N; ++k) {
        if ((k & 1) == 0 || (per & 4u)) {
            int z = z0 + k;
            if (per & 4u) z = wrapi(z, nz);
            const bool in = (unsigned)z < (unsigned)nz;
            const float l = mg_at(e, cc.at + (in ? (uint32_t)(z >> 1) * stride : 0u));
            v[k] = in && cc.in ? l : 0.0f;
        } else {
            v[k] = v[k - 1];
        }
    }
}

// The end of a solve's queue finds status->stop set and every kernel returns. The test stands behind
// the kernel's first loads, which do not depend on it (the host passes the iteration index), so that
// its latency hides behind theirs; the barrier keeps the compiler from moving them below the branch.
__device__ __forceinline__ bool mg_stopped(uint32_t stop) {
    asm volatile("" ::: "memory");
    return stop != 0u;
}

// A producer's per-block partial sums: the loads, issued before the kernel's others, and their sum
// over the workgroup of T threads in a fixed order.
template <int T>
struct Partials {
    static constexpr int N = ((int)kPcgMaxBlocks + T - 1) / T;
    double v[N];
    __device__ __forceinline__ Partials(const double* __restrict__ parts, uint32_t count) {
#pragma unroll
        for (int m = 0; m < N; ++m) {
            const uint32_t i = threadIdx.x + (uint32_t)(m * T);
            v[m] = i < count ? parts[i] : 0.0;
        }
    }
    __device__ __forceinline__ double sum(double* lds) const {
        double s[1]{v[0]};
#pragma unroll
        for (int m = 1; m < N; ++m) s[0] += v[m];
        block_sum<1>(s, lds);
        return s[0];
    }
};

// In-plane neighbours of LDS element i of planes X wide.
template <int X>
__device__ __forceinline__ float mg_plane_sum(const float* v, int i) {
    return (v[i - 1] + v[i + 1]) + (v[i - X] + v[i + X]);
}

// Level 0 on the way down, with the PCG update of the iteration fused in front (Update): alpha =
// rz / <p, A p>; x += alpha p; r' = r - alpha A p, partials of ||r'||^2 (r is double-buffered: the
// neighbouring boxes read the old one). The solution pair (hi + lo, about 48 bits) takes alpha p in
// FP64 and A p is formed in FP64 from p, exactly as the direction kernel forms it, so the recursive
// residual follows the true one to FP32 rounding of r itself: with the near-null mode of the matrix
// the solution is some 10^3 ||b|| large, and an FP32 increment (or an FP32 A p) would leave a gap of
// about 1e-4 ||b|| between them after the first, largest steps.
// Then (Smooth) the two sweeps from zero for A x = r' and the restriction of r' - A x to level 1.
template <typename B, bool Update, bool Smooth>
__global__ __launch_bounds__(B::T) void mg_down0_kernel(MgLevel L, MgLevel C, uint32_t per, Pair2 r, Pair2 p, float* __restrict__ xh,
                                                        float* __restrict__ xl, float* __restrict__ x, float* __restrict__ rc,
                                                        double* __restrict__ partials, const double* __restrict__ hist,
                                                        const PcgStatus* status, uint32_t k) {
    constexpr int X3 = B::template X<3>, X2 = B::template X<2>, X1 = B::template X<1>;
    constexpr int P3 = B::template P<3>, P2 = B::template P<2>, P1 = B::template P<1>;
    constexpr int Z3 = B::template Z<3>, Z2 = B::template Z<2>, Z1 = B::template Z<1>;
    constexpr int kPasses = (P3 + B::T - 1) / B::T;
    __shared__ float sp[P3 * Z3];   // p, then the first sweep's iterate, then the residual's z pairs
    __shared__ float sx[P1 * Z1];
    __shared__ double lds[kMaxWaves];
    const uint32_t stop = status->stop;
    const Partials<B::T> pq(partials + kPartPQ * kPcgMaxBlocks, Update ? gridDim.x : 0u);
    const double rz = Update ? hist[2 * k] : 0.0;
    const float* __restrict__ r_in = r.p[k & 1u];
    float* __restrict__ r_out = r.p[(k + 1u) & 1u];
    const float* __restrict__ pk = p.p[k & 1u];
    const int t = (int)threadIdx.x;
    const uint32_t lb = xcd_block();
    const typename B::Grid grid = B::grid(L);
    const uint32_t first = (uint32_t)((uint64_t)grid.count * lb / gridDim.x), last = (uint32_t)((uint64_t)grid.count * (lb + 1u) / gridDim.x);
    const int cy = t / X2, cx = t - cy * X2;   // column in the halo-2 planes
    const bool mine2 = t < P2;
    const bool mine1 = mine2 && cx >= 1 && cx < X2 - 1 && cy >= 1 && cy < B::template Y<2> - 1;
    const bool mine0 = mine2 && cx >= 2 && cx < X2 - 2 && cy >= 2 && cy < B::template Y<2> - 2;
    const int i3 = (cy + 1) * X3 + cx + 1, i1 = (cy - 1) * X1 + cx - 1;   // the column's element in a plane
    double alpha = 0.0, rr = 0.0;
    if (first == last && stop) return;   // (no boxes here)
    for (uint32_t b = first; b < last; ++b) {
        int x0, y0, z0;
        B::origin(grid, b, x0, y0, z0);
        const Planes<Z3> pl3 = mg_planes<Z3>(L, per, z0 - 3);
        if (Update) {
#pragma unroll
            for (int s = 0; s < kPasses; ++s) {
                const int e = s * B::T + t;
                const int ey = e / X3, ex = e - ey * X3;
                const Column c = mg_column(L, per, x0 - 3 + ex, y0 - 3 + ey);
                if (e < P3) {
#pragma unroll
                    for (int z = 0; z < Z3; ++z) sp[z * P3 + e] = mg_load(pk, pl3, z, c);
                }
            }
        }
        const Column c = mg_column(L, per, x0 - 2 + cx, y0 - 2 + cy, mine2);
        float rv[Z2];
        uint32_t dv[Z2];
#pragma unroll
        for (int z = 0; z < Z2; ++z) {
            rv[z] = mg_load(r_in, pl3, z + 1, c);
            dv[z] = mg_load(L.code, pl3, z + 1, c);
        }
        if (b == first) {
            if (mg_stopped(stop)) return;
            if (Update) alpha = rz / pq.sum(lds);
        }
        const bool own = mine0 && x0 - 2 + cx < L.nx && y0 - 2 + cy < L.ny;   // the box's own cells (not wrapped ones)
        if (Update) {
            __syncthreads();
            if (mine2) {
                double lo = (double)sp[i3], mid = (double)sp[P3 + i3];
#pragma unroll
                for (int z = 0; z < Z2; ++z) {
                    const float* pl = sp + (z + 1) * P3;
                    const double hi = (double)pl[P3 + i3];
                    const double around = ((double)pl[i3 - 1] + (double)pl[i3 + 1]) + ((double)pl[i3 - X3] + (double)pl[i3 + X3]) + (lo + hi);
                    const double q = (double)dv[z] * mid - around;
                    const float rn = dv[z] ? (float)__fma_rn(-alpha, q, (double)rv[z]) : 0.0f;
                    rv[z] = rn;
                    if (z >= 2 && z < Z2 - 2) {
                        const uint32_t i = c.at + pl3.at[z + 1];
                        if (own && z0 - 2 + z < L.nz) {
                            mg_at(r_out, i) = rn;
                            rr = __fma_rn((double)rn, (double)rn, rr);
                            if (dv[z]) {
                                float &h = mg_at(xh, i), &l = mg_at(xl, i);
                                const double xv = __fma_rn(alpha, mid, (double)h + (double)l);
                                const float hi32 = (float)xv;
                                h = hi32;
                                l = (float)(xv - (double)hi32);
                            }
                        }
                    }
                    lo = mid;
                    mid = hi;
                }
            }
            __syncthreads();   // p is done with
        }
        if (Smooth) {
            // first sweep, x1 = w D^-1 r, into LDS (planes P2)
            if (mine2) {
#pragma unroll
                for (int z = 0; z < Z2; ++z) sp[z * P2 + t] = kCheb[0] * mg_dinv(dv[z]) * rv[z];
            }
            __syncthreads();
            float x2[Z1];
            if (mine1) {
                float lo = sp[t], mid = sp[P2 + t];
#pragma unroll
                for (int z = 0; z < Z1; ++z) {
                    const float hi = sp[(z + 2) * P2 + t];
                    const uint32_t d = dv[z + 1];
                    const float sum = mg_plane_sum<X2>(sp + (z + 1) * P2, t) + (lo + hi);
                    const float res = rv[z + 1] - __fmaf_rn((float)d, mid, -sum);
                    x2[z] = d ? __fmaf_rn(kCheb[1] * mg_dinv(d), res, mid) : 0.0f;
                    sx[z * P1 + i1] = x2[z];
                    lo = mid;
                    mid = hi;
                }
            }
            __syncthreads();
            // x stored, the residual's sums over z pairs into LDS
            if (mine0) {
#pragma unroll
                for (int z = 0; z < B::BZ; z += 2) {
                    float pair = 0.0f;
#pragma unroll
                    for (int m = z; m < z + 2; ++m) {
                        const bool in = own && z0 + m < L.nz;
                        if (in) mg_at(x, c.at + pl3.at[m + 3]) = x2[m + 1];
                        const uint32_t d = dv[m + 2];
                        const float sum = mg_plane_sum<X1>(sx + (m + 1) * P1, i1) + (x2[m] + x2[m + 2]);
                        const float res = rv[m + 2] - __fmaf_rn((float)d, x2[m + 1], -sum);
                        // (beyond an odd extent a periodic axis wraps: not a cell of this aggregate)
                        pair += d && in ? res : 0.0f;
                    }
                    sp[(z / 2) * (B::BX * B::BY) + (cy - 2) * B::BX + cx - 2] = pair;
                }
            }
            __syncthreads();
            constexpr int CX = B::BX / 2, CY = B::BY / 2;
            for (int I = t; I < CX * CY * (B::BZ / 2); I += B::T) {
                const int lx = I % CX, ly = I / CX % CY, lz = I / (CX * CY);
                const float* v = sp + lz * (B::BX * B::BY) + 2 * ly * B::BX + 2 * lx;
                const int gX = (x0 >> 1) + lx, gY = (y0 >> 1) + ly, gZ = (z0 >> 1) + lz;
                if (gX < C.nx && gY < C.ny && gZ < C.nz)
                    rc[lattice_index(gX, gY, gZ, C.nx, C.ny)] = (v[0] + v[1]) + (v[B::BX] + v[B::BX + 1]);
            }
            __syncthreads();   // the next box reuses the tiles
        }
    }
    if (Update) {
        double v[1]{rr};
        block_sum<1>(v, lds);
        if (t == 0) partials[kPartRR * kPcgMaxBlocks + lb] = v[0];
    }
}

// Level 0 on the way up: xc = x + over P e (x the pre-smoothed iterate), the two sweeps in the
// reverse order, z, partials of <r, z>.
template <typename B>
__global__ __launch_bounds__(B::T) void mg_post0_kernel(MgLevel L, MgLevel C, uint32_t per, Pair2 r, const float* __restrict__ x,
                                                        const float* __restrict__ e_c, float* __restrict__ z_out, double* __restrict__ partials,
                                                        const PcgStatus* status, uint32_t k) {
    constexpr int X2 = B::template X<2>, X1 = B::template X<1>, P2 = B::template P<2>, P1 = B::template P<1>;
    constexpr int Z2 = B::template Z<2>, Z1 = B::template Z<1>;
    __shared__ float sx[P2 * Z2];
    __shared__ float sy[P1 * Z1];
    __shared__ double lds[kMaxWaves];
    const uint32_t stop = status->stop;
    const float* __restrict__ rk = r.p[k & 1u];
    const int t = (int)threadIdx.x;
    const uint32_t lb = xcd_block();
    const typename B::Grid grid = B::grid(L);
    const uint32_t first = (uint32_t)((uint64_t)grid.count * lb / gridDim.x), last = (uint32_t)((uint64_t)grid.count * (lb + 1u) / gridDim.x);
    const int cy = t / X2, cx = t - cy * X2;
    const bool mine2 = t < P2;
    const bool mine1 = mine2 && cx >= 1 && cx < X2 - 1 && cy >= 1 && cy < B::template Y<2> - 1;
    const bool mine0 = mine2 && cx >= 2 && cx < X2 - 2 && cy >= 2 && cy < B::template Y<2> - 2;
    const int i1 = (cy - 1) * X1 + cx - 1;
    double rz = 0.0;
    if (first == last && stop) return;
    for (uint32_t b = first; b < last; ++b) {
        int x0, y0, z0;
        B::origin(grid, b, x0, y0, z0);
        const Column c = mg_column(L, per, x0 - 2 + cx, y0 - 2 + cy, mine2);
        const uint32_t gy = c.at / (uint32_t)L.nx, gx = c.at - gy * (uint32_t)L.nx;
        const Column cc{(gx >> 1) + __umul24(gy >> 1, (uint32_t)C.nx), c.in};   // the column's aggregate
        const Planes<Z2> pl2 = mg_planes<Z2>(L, per, z0 - 2);
        float xv[Z2], rv[Z1];
        uint32_t dv[Z2];
#pragma unroll
        for (int z = 0; z < Z2; ++z) {
            dv[z] = mg_load(L.code, pl2, z, c);
            xv[z] = mg_load(x, pl2, z, c);
        }
        float ev[Z2];
        mg_load_coarse<Z2>(C, per, z0 - 2, L.nz, e_c, cc, ev);
#pragma unroll
        for (int z = 0; z < Z2; ++z) xv[z] = dv[z] ? __fmaf_rn(kOver, ev[z], xv[z]) : 0.0f;
#pragma unroll
        for (int z = 0; z < Z1; ++z) rv[z] = mg_load(rk, pl2, z + 1, c);
        if (b == first && mg_stopped(stop)) return;
        if (mine2) {
#pragma unroll
            for (int z = 0; z < Z2; ++z) sx[z * P2 + t] = xv[z];
        }
        __syncthreads();
        float y[Z1];
        if (mine1) {
#pragma unroll
            for (int z = 0; z < Z1; ++z) {
                const uint32_t d = dv[z + 1];
                const float sum = mg_plane_sum<X2>(sx + (z + 1) * P2, t) + (xv[z] + xv[z + 2]);
                const float res = rv[z] - __fmaf_rn((float)d, xv[z + 1], -sum);
                y[z] = d ? __fmaf_rn(kCheb[1] * mg_dinv(d), res, xv[z + 1]) : 0.0f;
                sy[z * P1 + i1] = y[z];
            }
        }
        __syncthreads();
        if (mine0 && x0 - 2 + cx < L.nx && y0 - 2 + cy < L.ny) {
#pragma unroll
            for (int z = 0; z < B::BZ; ++z) {
                const uint32_t d = dv[z + 2];
                const float ri = rv[z + 1];
                const float sum = mg_plane_sum<X1>(sy + (z + 1) * P1, i1) + (y[z] + y[z + 2]);
                const float res = ri - __fmaf_rn((float)d, y[z + 1], -sum);
                const float zi = d ? __fmaf_rn(kCheb[0] * mg_dinv(d), res, y[z + 1]) : 0.0f;
                if (z0 + z < L.nz) {
                    mg_at(z_out, c.at + pl2.at[z + 2]) = zi;
                    rz = __fma_rn((double)ri, (double)zi, rz);
                }
            }
        }
        __syncthreads();
    }
    double v[1]{rz};
    block_sum<1>(v, lds);
    if (t == 0) partials[kPartRZ * kPcgMaxBlocks + lb] = v[0];
}

// PCG direction of iteration k: beta = rz_k / rz_{k-1} (RZ partials of the V-cycle), p = z + beta p_old
// (p = z when k = 0), partials of <p, A p> with A p in FP64 (exact, as the update forms it).
template <typename B>
__global__ __launch_bounds__(B::T) void mg_direction_kernel(MgLevel L, uint32_t per, const float* __restrict__ z_in, Pair2 p,
                                                            double* __restrict__ partials, double* __restrict__ hist,
                                                            const PcgStatus* status, uint32_t k) {
    constexpr int X1 = B::template X<1>, P1 = B::template P<1>, Z1 = B::template Z<1>;
    __shared__ float sp[P1 * Z1];
    __shared__ double lds[kMaxWaves];
    const uint32_t stop = status->stop;
    const Partials<B::T> rz(partials + kPartRZ * kPcgMaxBlocks, gridDim.x);
    const double rz_old = k > 0u ? hist[2 * (k - 1u)] : 1.0;
    float* __restrict__ p_new = p.p[k & 1u];
    const float* __restrict__ p_old = p.p[(k + 1u) & 1u];
    const int t = (int)threadIdx.x;
    const uint32_t lb = xcd_block();
    const typename B::Grid grid = B::grid(L);
    const uint32_t first = (uint32_t)((uint64_t)grid.count * lb / gridDim.x), last = (uint32_t)((uint64_t)grid.count * (lb + 1u) / gridDim.x);
    const int cy = t / X1, cx = t - cy * X1;
    const bool mine1 = t < P1;
    const bool mine0 = mine1 && cx >= 1 && cx < X1 - 1 && cy >= 1 && cy < B::template Y<1> - 1;
    float beta = 0.0f;
    double pq = 0.0;
    if (first == last && stop) return;
    for (uint32_t b = first; b < last; ++b) {
        int x0, y0, z0;
        B::origin(grid, b, x0, y0, z0);
        const Column c = mg_column(L, per, x0 - 1 + cx, y0 - 1 + cy, mine1);
        const Planes<Z1> pl1 = mg_planes<Z1>(L, per, z0 - 1);
        float zv[Z1], pv[Z1];
        uint32_t dv[B::BZ];
#pragma unroll
        for (int z = 0; z < Z1; ++z) {
            zv[z] = mg_load(z_in, pl1, z, c);
            pv[z] = k > 0u ? mg_load(p_old, pl1, z, c) : 0.0f;
        }
#pragma unroll
        for (int z = 0; z < B::BZ; ++z) dv[z] = mg_load(L.code, pl1, z + 1, c);
        if (b == first) {
            if (mg_stopped(stop)) return;
            const double rz_new = rz.sum(lds);
            if (b == 0 && t == 0) hist[2 * k] = rz_new;   // the block of the first box
            beta = k > 0u ? (float)(rz_new / rz_old) : 0.0f;
        }
#pragma unroll
        for (int z = 0; z < Z1; ++z) {
            zv[z] = k > 0u ? __fmaf_rn(beta, pv[z], zv[z]) : zv[z];
            if (mine1) sp[z * P1 + t] = zv[z];
        }
        __syncthreads();
        if (mine0 && x0 - 1 + cx < L.nx && y0 - 1 + cy < L.ny) {
#pragma unroll
            for (int z = 0; z < B::BZ; ++z) {
                const float* pl = sp + (z + 1) * P1;
                const double pi = (double)zv[z + 1];   // 0 off the unknowns
                const double around = ((double)pl[t - 1] + (double)pl[t + 1]) + ((double)pl[t - X1] + (double)pl[t + X1]) +
                                      ((double)zv[z] + (double)zv[z + 2]);
                if (z0 + z < L.nz) {
                    mg_at(p_new, c.at + pl1.at[z + 1]) = zv[z + 1];
                    pq = __fma_rn(pi, (double)dv[z] * pi - around, pq);
                }
            }
        }
        __syncthreads();
    }
    double v[1]{pq};
    block_sum<1>(v, lds);
    if (t == 0) partials[kPartPQ * kPcgMaxBlocks + lb] = v[0];
}

// A row of a coarser level's operator: the + couplings are the cell's own, the - couplings the
// - neighbours' (along z the previous plane's).
struct CoarseRow {
    float diag, xp, xm, yp, ym, zp;
};
struct CoarseColumn {   // a column and its - neighbours along x and y
    Column c, xm, ym;
};
__device__ __forceinline__ CoarseColumn mg_coarse_column(const MgLevel& L, uint32_t per, int x, int y, bool mine) {
    CoarseColumn k{mg_column(L, per, x, y, mine), mg_column(L, per, x - 1, y), mg_column(L, per, x, y - 1)};
    k.xm.in = k.xm.in && k.c.in;
    k.ym.in = k.ym.in && k.c.in;
    return k;
}
template <int N>
__device__ __forceinline__ CoarseRow mg_row(const MgLevel& L, const Planes<N>& p, int z, const CoarseColumn& k) {
    return CoarseRow{mg_load(L.diag, p, z, k.c),  mg_load(L.wp[0], p, z, k.c),  mg_load(L.wp[0], p, z, k.xm),
                     mg_load(L.wp[1], p, z, k.c), mg_load(L.wp[1], p, z, k.ym), mg_load(L.wp[2], p, z, k.c)};
}
// (A v)_i: v's plane in LDS at pl (element i), its z neighbours lo, mid, hi; zm: the - z coupling.
template <int X>
__device__ __forceinline__ float mg_coarse_apply(const CoarseRow& w, float zm, const float* pl, int i, float lo, float mid, float hi) {
    float s = w.diag * mid;
    s = __fmaf_rn(w.xp, pl[i + 1], s);
    s = __fmaf_rn(w.xm, pl[i - 1], s);
    s = __fmaf_rn(w.yp, pl[i + X], s);
    s = __fmaf_rn(w.ym, pl[i - X], s);
    s = __fmaf_rn(w.zp, hi, s);
    return __fmaf_rn(zm, lo, s);
}

// A coarser level on the way down: both sweeps from zero, x stored, r - A x restricted.
template <typename B>
__global__ __launch_bounds__(B::T) void mg_down_kernel(MgLevel L, MgLevel C, uint32_t per, const float* __restrict__ r,
                                                       float* __restrict__ x, float* __restrict__ rc, const PcgStatus* status) {
    constexpr int X2 = B::template X<2>, X1 = B::template X<1>, P2 = B::template P<2>, P1 = B::template P<1>;
    constexpr int Z2 = B::template Z<2>, Z1 = B::template Z<1>;
    __shared__ float s1[P2 * Z2], sx[P1 * Z1];
    const uint32_t stop = status->stop;
    const int t = (int)threadIdx.x;
    const typename B::Grid grid = B::grid(L);
    const uint32_t b = xcd_block();
    if (b >= grid.count) return;
    const int cy = t / X2, cx = t - cy * X2;
    const bool mine2 = t < P2;
    const bool mine1 = mine2 && cx >= 1 && cx < X2 - 1 && cy >= 1 && cy < B::template Y<2> - 1;
    const bool mine0 = mine2 && cx >= 2 && cx < X2 - 2 && cy >= 2 && cy < B::template Y<2> - 2;
    const int i1 = (cy - 1) * X1 + cx - 1;
    int x0, y0, z0;
    B::origin(grid, b, x0, y0, z0);
    const CoarseColumn k = mg_coarse_column(L, per, x0 - 2 + cx, y0 - 2 + cy, mine2);
    const Planes<Z2> pl2 = mg_planes<Z2>(L, per, z0 - 2);
    float rv[Z2], iv[Z2], x1[Z2];
#pragma unroll
    for (int z = 0; z < Z2; ++z) {
        rv[z] = mg_load(r, pl2, z, k.c);
        iv[z] = mg_load(L.idiag, pl2, z, k.c);
    }
    CoarseRow w[Z1];
    const float zm0 = mg_load(L.wp[2], pl2, 0, k.c);
#pragma unroll
    for (int z = 0; z < Z1; ++z) w[z] = mg_row(L, pl2, z + 1, k);
    if (mg_stopped(stop)) return;
#pragma unroll
    for (int z = 0; z < Z2; ++z) {
        x1[z] = kCheb[0] * iv[z] * rv[z];   // 0 off the unknowns (1 / diag is 0 there)
        if (mine2) s1[z * P2 + t] = x1[z];
    }
    __syncthreads();
    float x2[Z1];
    if (mine1) {
#pragma unroll
        for (int z = 0; z < Z1; ++z) {
            const float ax = mg_coarse_apply<X2>(w[z], z ? w[z ? z - 1 : 0].zp : zm0, s1 + (z + 1) * P2, t, x1[z], x1[z + 1], x1[z + 2]);
            x2[z] = __fmaf_rn(kCheb[1] * iv[z + 1], rv[z + 1] - ax, x1[z + 1]);
            sx[z * P1 + i1] = x2[z];
        }
    }
    __syncthreads();
    if (mine0) {
        const bool own = x0 - 2 + cx < L.nx && y0 - 2 + cy < L.ny;
#pragma unroll
        for (int z = 0; z < B::BZ; z += 2) {
            float pair = 0.0f;
#pragma unroll
            for (int m = z; m < z + 2; ++m) {
                const bool in = own && z0 + m < L.nz;
                if (in) mg_at(x, k.c.at + pl2.at[m + 2]) = x2[m + 1];
                const float ax = mg_coarse_apply<X1>(w[m + 1], w[m].zp, sx + (m + 1) * P1, i1, x2[m], x2[m + 1], x2[m + 2]);
                pair += in && iv[m + 2] > 0.0f ? rv[m + 2] - ax : 0.0f;
            }
            s1[(z / 2) * (B::BX * B::BY) + (cy - 2) * B::BX + cx - 2] = pair;   // (every read of s1 is behind the barrier)
        }
    }
    __syncthreads();
    constexpr int CX = B::BX / 2, CY = B::BY / 2;
    for (int I = t; I < CX * CY * (B::BZ / 2); I += B::T) {
        const int lx = I % CX, ly = I / CX % CY, lz = I / (CX * CY);
        const float* v = s1 + lz * (B::BX * B::BY) + 2 * ly * B::BX + 2 * lx;
        const int gX = (x0 >> 1) + lx, gY = (y0 >> 1) + ly, gZ = (z0 >> 1) + lz;
        if (gX < C.nx && gY < C.ny && gZ < C.nz) rc[lattice_index(gX, gY, gZ, C.nx, C.ny)] = (v[0] + v[1]) + (v[B::BX] + v[B::BX + 1]);
    }
}

// A coarser level on the way up: xc = x + over P e, the two sweeps in the reverse order.
template <typename B>
__global__ __launch_bounds__(B::T) void mg_up_kernel(MgLevel L, MgLevel C, uint32_t per, const float* __restrict__ r,
                                                     const float* __restrict__ x, const float* __restrict__ e_c, float* __restrict__ z_out,
                                                     const PcgStatus* status) {
    constexpr int X2 = B::template X<2>, X1 = B::template X<1>, P2 = B::template P<2>, P1 = B::template P<1>;
    constexpr int Z2 = B::template Z<2>, Z1 = B::template Z<1>;
    __shared__ float sx[P2 * Z2], sy[P1 * Z1];
    const uint32_t stop = status->stop;
    const int t = (int)threadIdx.x;
    const typename B::Grid grid = B::grid(L);
    const uint32_t b = xcd_block();
    if (b >= grid.count) return;
    const int cy = t / X2, cx = t - cy * X2;
    const bool mine2 = t < P2;
    const bool mine1 = mine2 && cx >= 1 && cx < X2 - 1 && cy >= 1 && cy < B::template Y<2> - 1;
    const bool mine0 = mine2 && cx >= 2 && cx < X2 - 2 && cy >= 2 && cy < B::template Y<2> - 2;
    const int i1 = (cy - 1) * X1 + cx - 1;
    int x0, y0, z0;
    B::origin(grid, b, x0, y0, z0);
    const CoarseColumn k = mg_coarse_column(L, per, x0 - 2 + cx, y0 - 2 + cy, mine2);
    const uint32_t gy = k.c.at / (uint32_t)L.nx, gx = k.c.at - gy * (uint32_t)L.nx;
    const Column cc{(gx >> 1) + __umul24(gy >> 1, (uint32_t)C.nx), k.c.in};
    const Planes<Z2> pl2 = mg_planes<Z2>(L, per, z0 - 2);
    float xv[Z2], iv[Z2], ev[Z2], rv[Z1];
#pragma unroll
    for (int z = 0; z < Z2; ++z) {
        iv[z] = mg_load(L.idiag, pl2, z, k.c);
        xv[z] = mg_load(x, pl2, z, k.c);
    }
    mg_load_coarse<Z2>(C, per, z0 - 2, L.nz, e_c, cc, ev);
    CoarseRow w[Z1];
    const float zm0 = mg_load(L.wp[2], pl2, 0, k.c);
#pragma unroll
    for (int z = 0; z < Z1; ++z) {
        w[z] = mg_row(L, pl2, z + 1, k);
        rv[z] = mg_load(r, pl2, z + 1, k.c);
    }
    if (mg_stopped(stop)) return;
#pragma unroll
    for (int z = 0; z < Z2; ++z) xv[z] = iv[z] > 0.0f ? __fmaf_rn(kOver, ev[z], xv[z]) : 0.0f;
    if (mine2) {
#pragma unroll
        for (int z = 0; z < Z2; ++z) sx[z * P2 + t] = xv[z];
    }
    __syncthreads();
    float y[Z1];
    if (mine1) {
#pragma unroll
        for (int z = 0; z < Z1; ++z) {
            const float ax = mg_coarse_apply<X2>(w[z], z ? w[z ? z - 1 : 0].zp : zm0, sx + (z + 1) * P2, t, xv[z], xv[z + 1], xv[z + 2]);
            y[z] = __fmaf_rn(kCheb[1] * iv[z + 1], rv[z] - ax, xv[z + 1]);
            sy[z * P1 + i1] = y[z];
        }
    }
    __syncthreads();
    if (mine0 && x0 - 2 + cx < L.nx && y0 - 2 + cy < L.ny) {
#pragma unroll
        for (int z = 0; z < B::BZ; ++z) {
            const float ax = mg_coarse_apply<X1>(w[z + 1], w[z].zp, sy + (z + 1) * P1, i1, y[z], y[z + 1], y[z + 2]);
            if (z0 + z < L.nz) mg_at(z_out, k.c.at + pl2.at[z + 2]) = __fmaf_rn(kCheb[0] * iv[z + 2], rv[z + 1] - ax, y[z + 1]);
        }
    }
}

// ---- the levels that one workgroup handles ------------------------------------------------------

// A cell of such a level, as the host lays it out (kBottomWords arrays of n words per level): its row
// of the operator, its neighbours' indices (two per word, in the order -x, +x, -y, ...), its
// aggregate's index on the next level; and for cell I of the next level its first child's index with
// a bit per existing child (-1: not used). One CU runs this kernel, and the instructions to form
// these in place took most of its time.
struct BottomCell {
    float diag, idiag, w[6];
    uint32_t nb[3], parent;
};
__device__ __forceinline__ BottomCell mg_bottom_cell(const uint32_t* __restrict__ words, uint32_t n, uint32_t i) {
    BottomCell c;
    c.diag = __uint_as_float(words[i]);
    c.idiag = __uint_as_float(words[n + i]);
#pragma unroll
    for (int k = 0; k < 6; ++k) c.w[k] = __uint_as_float(words[(2 + k) * n + i]);
#pragma unroll
    for (int k = 0; k < 3; ++k) c.nb[k] = words[(8 + k) * n + i];
    c.parent = words[11 * n + i];
    return c;
}
__device__ __forceinline__ float mg_bottom_apply(const BottomCell& c, const float* v, float own) {
    float s = c.diag * own;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        s = __fmaf_rn(c.w[2 * a], v[c.nb[a] & 0xffffu], s);
        s = __fmaf_rn(c.w[2 * a + 1], v[c.nb[a] >> 16], s);
    }
    return s;
}

// The stopping test of an iteration (or of the initial residual), then the V-cycle of the levels of
// at most kMgBottomCells cells in one workgroup: vectors in LDS, the rows of the first two levels in
// registers, and the coarsest level's inverse (n x n, FP64, n <= kMgDense) spread over the threads.
// Levels: how many (the last is the dense one; 0: only the test).
// k: updates applied so far. mode: bit 1 the first test of a solve (||b||^2 from its partials, the
// initial residual kept), bit 2 the guess is rejected when its residual exceeds ||b||, bit 3 when it
// is not finite. A rejection stops the solve: the host, which reads the status once at its end, runs
// it again without the guess.
constexpr int kBottomThreads = 1024;
constexpr int kBottomWords = 13;
template <int Levels>
__global__ __launch_bounds__(kBottomThreads) void mg_bottom_kernel(MgBottom B, const float* __restrict__ r,
                                                                   float* __restrict__ out, const double* __restrict__ partials,
                                                                   uint32_t blocks, PcgStatus* status, double tol2, uint32_t mode, uint32_t k) {
    constexpr int T = kBottomThreads, last = Levels - 1;
    __shared__ float vr[Levels ? kMgBottomLds : 1], vx[Levels ? kMgBottomLds : 1], vy[Levels ? kMgBottomLds : 1];
    __shared__ double lds[(T / 64) * kMgDense];
    const uint32_t stopped = status->stop;
    const uint32_t t = threadIdx.x;
    const double bb0 = status->bb;
    const bool opening = mode & 2u;
    const Partials<T> rr_parts(partials + kPartRR * kPcgMaxBlocks, blocks);
    const Partials<T> bb_parts(partials + kPartBB * kPcgMaxBlocks, opening ? blocks : 0u);
    // everything the cycle reads from memory, up front
    BottomCell c0[4], c1[2];
    double inv[4];
    if constexpr (last >= 0) {
        for (uint32_t i = t; i < B.n[0]; i += T) vr[i] = r[i];
        const uint32_t n = B.n[last];
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            const uint32_t j = (t >> 6) + 16u * m;
            inv[m] = (t & 63u) < n && j < n ? B.dense[j * n + (t & 63u)] : 0.0;
        }
    }
    if constexpr (last >= 1) {
#pragma unroll
        for (int m = 0; m < 4; ++m)
            if (t + m * T < B.n[0]) c0[m] = mg_bottom_cell(B.words[0], B.n[0], t + m * T);
    }
    if constexpr (last >= 2) {
#pragma unroll
        for (int m = 0; m < 2; ++m)
            if (t + m * T < B.n[1]) c1[m] = mg_bottom_cell(B.words[1], B.n[1], t + m * T);
    }
    if (mg_stopped(stopped)) return;
    double red[2]{rr_parts.v[0], bb_parts.v[0]};
    static_assert(Partials<T>::N == 1, "one partial per thread");
    block_sum<2>(red, lds);
    const double rr = red[0], bb = opening ? red[1] : bb0;
    const bool finite = isfinite(rr);
    const bool rejected = ((mode & 4u) && !(finite && rr <= bb)) || ((mode & 8u) && !finite);
    const bool stop = rejected || !(rr > tol2 * bb);
    if (t == 0) {
        status->k = k;
        status->rr = rr;
        status->iterations = k;
        if (opening) {
            status->bb = bb;
            status->rr0 = rr;
        }
        if (rejected) status->rejected = 1u;
        if (stop) status->stop = 1u;
    }
    if (stop) return;
    if constexpr (last >= 0) {
        // f(row, cell) over the cells of level l
        auto cells = [&]<int l>(auto&& f) {
            if constexpr (l == 0) {
#pragma unroll
                for (int m = 0; m < 4; ++m)
                    if (t + m * T < B.n[0]) f(c0[m], t + m * T);
            } else if constexpr (l == 1) {
#pragma unroll
                for (int m = 0; m < 2; ++m)
                    if (t + m * T < B.n[1]) f(c1[m], t + m * T);
            } else {
                for (uint32_t i = t; i < B.n[l]; i += T) f(mg_bottom_cell(B.words[l], B.n[l], i), i);
            }
        };
        auto down = [&]<int l>() {
            float *rl = vr + B.off[l], *xl = vx + B.off[l], *yl = vy + B.off[l];
            cells.template operator()<l>([&](const BottomCell& c, uint32_t i) { xl[i] = kCheb[0] * c.idiag * rl[i]; });
            __syncthreads();
            cells.template operator()<l>([&](const BottomCell& c, uint32_t i) {
                const float v = xl[i];
                yl[i] = __fmaf_rn(kCheb[1] * c.idiag, rl[i] - mg_bottom_apply(c, xl, v), v);
            });
            __syncthreads();
            cells.template operator()<l>(
                [&](const BottomCell& c, uint32_t i) { xl[i] = c.idiag > 0.0f ? rl[i] - mg_bottom_apply(c, yl, yl[i]) : 0.0f; });
            __syncthreads();
            float* rn = vr + B.off[l + 1];
            const uint32_t sy = B.nx[l], sz = B.nxy[l];
            for (uint32_t I = t; I < B.n[l + 1]; I += T) {
                const uint32_t w = B.words[l][12u * B.n[l] + I], i = w & 0xffffu;
                float s = 0.0f;
#pragma unroll
                for (int ch = 0; ch < 8; ++ch) {
                    const bool in = w >> (16 + ch) & 1u;
                    const float v = xl[in ? i + (ch & 1) + (ch >> 1 & 1) * sy + (ch >> 2) * sz : 0u];
                    s += in ? v : 0.0f;
                }
                rn[I] = s;
            }
            __syncthreads();
        };
        auto up = [&]<int l>() {
            float *rl = vr + B.off[l], *xl = vx + B.off[l], *yl = vy + B.off[l];
            const float* e = vx + B.off[l + 1];
            cells.template operator()<l>([&](const BottomCell& c, uint32_t i) { yl[i] = c.idiag > 0.0f ? __fmaf_rn(kOver, e[c.parent], yl[i]) : 0.0f; });
            __syncthreads();
            cells.template operator()<l>([&](const BottomCell& c, uint32_t i) {
                const float v = yl[i];
                xl[i] = __fmaf_rn(kCheb[1] * c.idiag, rl[i] - mg_bottom_apply(c, yl, v), v);
            });
            __syncthreads();
            float* res = l == 0 ? out : yl;
            cells.template operator()<l>([&](const BottomCell& c, uint32_t i) {
                const float v = xl[i];
                res[i] = __fmaf_rn(kCheb[0] * c.idiag, rl[i] - mg_bottom_apply(c, xl, v), v);
            });
            if (l > 0) {
                __syncthreads();
                for (uint32_t i = t; i < B.n[l]; i += T) xl[i] = yl[i];
                __syncthreads();
            }
        };
        __syncthreads();
        [&]<int... l>(std::integer_sequence<int, l...>) { (down.template operator()<l>(), ...); }(std::make_integer_sequence<int, last>{});
        {   // coarsest: e = A^-1 r; thread t sums columns t / 64 + 16 m of row t % 64
            const uint32_t n = B.n[last], row = t & 63u, part = t >> 6;
            const float* rl = vr + B.off[last];
            double s = 0.0;
#pragma unroll
            for (int m = 0; m < 4; ++m) s = __fma_rn(inv[m], (double)rl[min(part + 16u * m, n - 1u)], s);
            lds[part * kMgDense + row] = s;
            __syncthreads();
            if (t < n) {
                double e = 0.0;
#pragma unroll
                for (int m = 0; m < T / 64; ++m) e += lds[m * kMgDense + t];
                if (last == 0) out[t] = (float)e;
                else vx[B.off[last] + t] = (float)e;
            }
            __syncthreads();
        }
        [&]<int... l>(std::integer_sequence<int, l...>) { (up.template operator()<last - 1 - l>(), ...); }(std::make_integer_sequence<int, last>{});
    }
}

// A grid of at most kMgCoarsest cells: z = A^-1 r in FP64, one block per row of the inverse.
__global__ __launch_bounds__(kBlock) void mg_dense_kernel(uint32_t n, const double* __restrict__ inv, Pair2 rp, float* __restrict__ x,
                                                          const PcgStatus* status, uint32_t k) {
    __shared__ double lds[kMaxWaves];
    if (status->stop) return;
    const float* __restrict__ r = rp.p[k & 1u];
    const uint32_t I = blockIdx.x;
    double s = 0.0;
    for (uint32_t j = threadIdx.x; j < n; j += blockDim.x) s = __fma_rn(inv[(size_t)I * n + j], (double)r[j], s);
    double v[1]{s};
    block_sum<1>(v, lds);
    if (threadIdx.x == 0) x[I] = (float)v[0];
}

// Partials of <r, z> on such a grid.
__global__ __launch_bounds__(kMgDotThreads) void mg_dot_kernel(uint32_t n, Pair2 rp, const float* __restrict__ z, double* __restrict__ partials,
                                                               const PcgStatus* status, uint32_t k) {
    __shared__ double lds[kMaxWaves];
    if (status->stop) return;
    const float* __restrict__ r = rp.p[k & 1u];
    double rz = 0.0;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) rz = __fma_rn((double)r[i], (double)z[i], rz);
    double v[1]{rz};
    block_sum<1>(v, lds);
    if (threadIdx.x == 0) partials[kPartRZ * kPcgMaxBlocks + blockIdx.x] = v[0];
}

// ---- hierarchy (host) ------------------------------------------------------------------------

struct HostLevel {
    int nx = 0, ny = 0, nz = 0;
    std::vector<double> diag;    // A_ii
    std::vector<double> wp[3];   // coupling to the + neighbour per axis (wrapped on a periodic axis)
    size_t cells() const { return (size_t)nx * ny * nz; }
};

// Index of the + neighbour of (x, y, z) along a, or SIZE_MAX outside a non-periodic axis.
size_t plus_neighbour(const HostLevel& L, const bool per[3], int x, int y, int z, int a) {
    int q[3]{x, y, z};
    const int e[3]{L.nx, L.ny, L.nz};
    if (++q[a] >= e[a]) {
        if (!per[a]) return SIZE_MAX;
        q[a] = 0;
    }
    return (size_t)q[0] + (size_t)L.nx * ((size_t)q[1] + (size_t)L.ny * (size_t)q[2]);
}

// Galerkin operator P^T A P of the 2 x 2 x 2 aggregation of level f. Each + edge (i, j) of weight w
// adds 2 w to the aggregate's diagonal when i and j share an aggregate (the edge's two off-diagonal
// entries), else w to the + coupling of i's aggregate along the edge's axis (a periodic wrap of the
// fine level is a wrap of the coarse level too).
HostLevel coarsen(const HostLevel& f, const bool per[3]) {
    HostLevel c;
    c.nx = (f.nx + 1) / 2;
    c.ny = (f.ny + 1) / 2;
    c.nz = (f.nz + 1) / 2;
    const size_t nc = c.cells();
    c.diag.assign(nc, 0.0);
    for (auto& w : c.wp) w.assign(nc, 0.0);
    auto agg = [&](size_t j) {
        const size_t x = j % (size_t)f.nx, t = j / (size_t)f.nx;
        const size_t y = t % (size_t)f.ny, z = t / (size_t)f.ny;
        return x / 2 + (size_t)c.nx * (y / 2 + (size_t)c.ny * (z / 2));
    };
    for (int z = 0; z < f.nz; ++z)
        for (int y = 0; y < f.ny; ++y)
            for (int x = 0; x < f.nx; ++x) {
                const size_t i = (size_t)x + (size_t)f.nx * ((size_t)y + (size_t)f.ny * (size_t)z);
                const size_t I = (size_t)(x / 2) + (size_t)c.nx * ((size_t)(y / 2) + (size_t)c.ny * (size_t)(z / 2));
                c.diag[I] += f.diag[i];
                for (int a = 0; a < 3; ++a) {
                    const double w = f.wp[a][i];
                    if (w == 0.0) continue;
                    const size_t j = plus_neighbour(f, per, x, y, z, a);
                    if (j == SIZE_MAX) continue;
                    if (agg(j) == I) c.diag[I] += 2.0 * w;
                    else c.wp[a][I] += w;
                }
            }
    return c;
}

// The words of level f for the single-workgroup kernel (BottomCell; c: the next level).
std::vector<uint32_t> bottom_words(const HostLevel& f, const HostLevel& c, const bool per[3]) {
    const size_t n = f.cells();
    std::vector<uint32_t> out(kBottomWords * n, 0u);
    auto bits = [](double v) { return std::bit_cast<uint32_t>((float)v); };
    for (int z = 0; z < f.nz; ++z)
        for (int y = 0; y < f.ny; ++y)
            for (int x = 0; x < f.nx; ++x) {
                const size_t i = (size_t)x + (size_t)f.nx * ((size_t)y + (size_t)f.ny * (size_t)z);
                const bool live = f.diag[i] > 0.0;
                out[i] = bits(f.diag[i]);
                out[n + i] = bits(live ? 1.0 / f.diag[i] : 0.0);
                for (int a = 0; a < 3; ++a) {
                    int q[3]{x, y, z};
                    const int e[3]{f.nx, f.ny, f.nz};
                    const size_t hi = plus_neighbour(f, per, x, y, z, a);
                    size_t lo = SIZE_MAX;
                    if (q[a] > 0 || per[a]) {
                        q[a] = q[a] > 0 ? q[a] - 1 : e[a] - 1;
                        lo = (size_t)q[0] + (size_t)f.nx * ((size_t)q[1] + (size_t)f.ny * (size_t)q[2]);
                    }
                    out[(2 + 2 * a) * n + i] = bits(lo == SIZE_MAX ? 0.0 : f.wp[a][lo]);
                    out[(3 + 2 * a) * n + i] = bits(hi == SIZE_MAX ? 0.0 : f.wp[a][i]);
                    out[(8 + a) * n + i] = (uint32_t)(lo == SIZE_MAX ? i : lo) | (uint32_t)(hi == SIZE_MAX ? i : hi) << 16;
                }
                const size_t I = (size_t)(x / 2) + (size_t)c.nx * ((size_t)(y / 2) + (size_t)c.ny * (size_t)(z / 2));
                out[11 * n + i] = (uint32_t)I;
                if (!(x & 1) && !(y & 1) && !(z & 1)) {
                    uint32_t w = (uint32_t)i;
                    for (int k = 0; k < 8; ++k)
                        if (x + (k & 1) < f.nx && y + (k >> 1 & 1) < f.ny && z + (k >> 2) < f.nz) w |= 1u << (16 + k);
                    out[12 * n + I] = w;
                }
            }
    return out;
}

// Inverse of level L's operator over its unknowns (diag > 0), FP64 Cholesky, as a symmetric
// n x n matrix with zero rows and columns off the unknowns.
std::vector<double> dense_inverse(const HostLevel& L, const bool per[3]) {
    const size_t n = L.cells();
    std::vector<int64_t> pos(n, -1);
    std::vector<size_t> unk;
    for (size_t i = 0; i < n; ++i)
        if (L.diag[i] > 0.0) {
            pos[i] = (int64_t)unk.size();
            unk.push_back(i);
        }
    const size_t m = unk.size();
    std::vector<double> A(m * m, 0.0);
    for (int z = 0; z < L.nz; ++z)
        for (int y = 0; y < L.ny; ++y)
            for (int x = 0; x < L.nx; ++x) {
                const size_t i = (size_t)x + (size_t)L.nx * ((size_t)y + (size_t)L.ny * (size_t)z);
                if (pos[i] < 0) continue;
                const size_t pi = (size_t)pos[i];
                A[pi * m + pi] += L.diag[i];
                for (int a = 0; a < 3; ++a) {
                    const double w = L.wp[a][i];
                    if (w == 0.0) continue;
                    const size_t j = plus_neighbour(L, per, x, y, z, a);
                    if (j == SIZE_MAX || pos[j] < 0) continue;
                    const size_t pj = (size_t)pos[j];
                    A[pi * m + pj] += w;
                    A[pj * m + pi] += w;
                }
            }
    // A = G G^T, G lower triangular (in place)
    for (size_t j = 0; j < m; ++j) {
        double s = A[j * m + j];
        for (size_t k = 0; k < j; ++k) s -= A[j * m + k] * A[j * m + k];
        if (!(s > 0.0)) throw Failure{DS_ERROR_RUNTIME, "multigrid: the coarsest operator is not positive definite"};
        const double d = std::sqrt(s);
        A[j * m + j] = d;
        for (size_t i = j + 1; i < m; ++i) {
            double t = A[i * m + j];
            for (size_t k = 0; k < j; ++k) t -= A[i * m + k] * A[j * m + k];
            A[i * m + j] = t / d;
        }
    }
    // column c of A^-1: G y = e_c, then G^T x = y
    std::vector<double> inv(m * m);
    std::vector<double> col(m);
    for (size_t c = 0; c < m; ++c) {
        for (size_t i = 0; i < m; ++i) {
            double t = i == c ? 1.0 : 0.0;
            for (size_t k = 0; k < i; ++k) t -= A[i * m + k] * col[k];
            col[i] = t / A[i * m + i];
        }
        for (size_t i = m; i-- > 0;) {
            double t = col[i];
            for (size_t k = i + 1; k < m; ++k) t -= A[k * m + i] * col[k];
            col[i] = t / A[i * m + i];
        }
        for (size_t i = 0; i < m; ++i) inv[i * m + c] = col[i];
    }
    std::vector<double> out(n * n, 0.0);
    for (size_t a = 0; a < m; ++a)
        for (size_t b = 0; b < m; ++b) out[unk[a] * n + unk[b]] = 0.5 * (inv[a * m + b] + inv[b * m + a]);
    return out;
}

// Points of a level with halos of 2 that boxes of type B load and sweep.
template <typename B>
uint64_t box_points(const MgLevel& L) {
    return (uint64_t)B::grid(L).count * (uint64_t)(B::template P<2> * B::template Z<2>);
}

// The box type of level l: by the number of cells, but a thin one on a large grid where it has less
// than two thirds of the points (from 11 cells along x or 3 along z on it does not).
MgBox choose_box(const MgLevel& L, int l) {
    auto thin = [&]<typename N, typename X, typename Z>() {
        const uint64_t x = box_points<X>(L), z = box_points<Z>(L);
        if (3 * std::min(x, z) >= 2 * box_points<N>(L)) return kMgBoxLarge;
        return x < z ? kMgBoxThinX : kMgBoxThinZ;
    };
    if (l > 0) return L.n < kMgCoarseLarge ? kMgBoxSmall : thin.template operator()<BoxC, BoxCX, BoxCZ>();
    if (L.n < kMgMediumCells) return kMgBoxSmall;
    if (L.n < kMgLargeCells) return kMgBoxMedium;
    return thin.template operator()<BoxL, BoxLX, BoxLZ>();
}

}  // namespace

void mg_prepare(ds_context* c, const std::vector<uint8_t>& code) {
    MgWork& w = c->mg;
    const Geo& g = c->geo;
    require(code.size() >= (size_t)g.n, "multigrid: code shorter than the grid");
    // The levels' axes: the grid's, those of one cell last. The cells lie in memory the same way, so a
    // grid of 1 x ny x nz is one of ny x nz x 1, which the boxes fit better (1 x 1024 x 1024: 1490 us a
    // step against 2189 with boxes thin along x).
    int ext[3]{g.nx, g.ny, g.nz};
    bool per[3]{c->pressure_periodic[0], c->pressure_periodic[1], c->pressure_periodic[2]};
    for (int pass = 0; pass < 2; ++pass)
        for (int a = 0; a < 2; ++a)
            if (ext[a] == 1) {
                std::swap(ext[a], ext[a + 1]);
                std::swap(per[a], per[a + 1]);
            }
    w.per = (per[0] ? 1u : 0u) | (per[1] ? 2u : 0u) | (per[2] ? 4u : 0u);
    // level 0 as diagonal + couplings: A_ii = code_i, -1 between neighbouring unknowns (on an
    // extent-1 periodic axis a cell neighbours itself twice, as in the matrix-vector product)
    std::vector<HostLevel> levels(1);
    {
        HostLevel& f = levels[0];
        f.nx = ext[0];
        f.ny = ext[1];
        f.nz = ext[2];
        const size_t n = f.cells();
        f.diag.resize(n);
        for (auto& v : f.wp) v.assign(n, 0.0);
        for (int z = 0; z < f.nz; ++z)
            for (int y = 0; y < f.ny; ++y)
                for (int x = 0; x < f.nx; ++x) {
                    const size_t i = (size_t)x + (size_t)f.nx * ((size_t)y + (size_t)f.ny * (size_t)z);
                    f.diag[i] = (double)code[i];
                    if (!code[i]) continue;
                    for (int a = 0; a < 3; ++a) {
                        const size_t j = plus_neighbour(f, per, x, y, z, a);
                        if (j != SIZE_MAX && code[j]) f.wp[a][i] = -1.0;
                    }
                }
    }
    // a grid of at most kMgCoarsest cells is solved directly; else down to kMgDense cells
    const bool direct = levels[0].cells() <= kMgCoarsest;
    while (!direct && levels.back().cells() > kMgDense) {
        if ((int)levels.size() == kMgMaxLevels) throw Failure{DS_ERROR_UNSUPPORTED, "multigrid: too many levels"};
        HostLevel next = coarsen(levels.back(), per);
        levels.push_back(std::move(next));
    }
    w.levels = (int)levels.size();
    // the levels one workgroup handles, from bottom_first on: they are laid out below
    w.bottom_first = direct ? 1 : w.levels - 1;
    while (!direct && w.bottom_first > 1 && levels[w.bottom_first - 1].cells() <= kMgBottomCells) --w.bottom_first;
    for (int l = 0; l < w.levels; ++l) {
        const HostLevel& H = levels[l];
        MgLevel& L = w.lv[l];
        L.nx = H.nx;
        L.ny = H.ny;
        L.nz = H.nz;
        L.n = (uint32_t)H.cells();
        L.code = l == 0 ? c->code : nullptr;
        L.diag = nullptr;
        L.idiag = nullptr;
        for (int a = 0; a < 3; ++a) L.wp[a] = nullptr;
        if (l > 0 && l < w.bottom_first) {
            std::vector<float> buf(L.n);
            auto put = [&](const std::vector<double>& v) {
                for (uint32_t i = 0; i < L.n; ++i) buf[i] = (float)v[i];
                float* d = device_alloc<float>(c, L.n);
                DS_HIP(hipMemcpy(d, buf.data(), L.n * sizeof(float), hipMemcpyHostToDevice));
                return d;
            };
            L.diag = put(H.diag);
            std::vector<double> inv(L.n);
            for (uint32_t i = 0; i < L.n; ++i) inv[i] = H.diag[i] > 0.0 ? 1.0 / H.diag[i] : 0.0;
            L.idiag = put(inv);
            for (int a = 0; a < 3; ++a) L.wp[a] = put(H.wp[a]);
        }
        if (!direct && l <= w.bottom_first) {
            // right-hand side, pre-smoothed iterate, result
            const bool used[3]{l > 0, l < w.bottom_first, l > 0};
            for (int k = 0; k < 3; ++k)
                if (used[k]) {
                    w.vec[l][k] = device_alloc<float>(c, L.n);
                    fill_zero(c, w.vec[l][k], L.n);
                }
        }
    }
    const std::vector<double> inv = dense_inverse(levels.back(), per);
    w.dense = device_alloc<double>(c, inv.size());
    DS_HIP(hipMemcpy(w.dense, inv.data(), inv.size() * sizeof(double), hipMemcpyHostToDevice));
    w.z = device_alloc<float>(c, g.n);
    fill_zero(c, w.z, g.n);
    MgBottom& bt = w.bottom;
    uint32_t off = 0;
    for (int l = w.bottom_first; l < w.levels; ++l) {
        require(bt.count < (uint32_t)kMgBottomLevels, "multigrid: too many coarse levels");
        bt.n[bt.count] = w.lv[l].n;
        bt.nx[bt.count] = (uint32_t)w.lv[l].nx;
        bt.nxy[bt.count] = (uint32_t)w.lv[l].nx * (uint32_t)w.lv[l].ny;
        bt.words[bt.count] = nullptr;
        if (l + 1 < w.levels) {
            const std::vector<uint32_t> words = bottom_words(levels[l], levels[l + 1], per);
            uint32_t* d = device_alloc<uint32_t>(c, words.size());
            DS_HIP(hipMemcpy(d, words.data(), words.size() * sizeof(uint32_t), hipMemcpyHostToDevice));
            bt.words[bt.count] = d;
        }
        bt.off[bt.count++] = off;
        off += w.lv[l].n;
    }
    require(off <= kMgBottomLds, "multigrid: the coarse levels do not fit one workgroup");
    bt.dense = w.dense;
    for (int l = 0; l < w.levels; ++l) w.box[l] = choose_box(w.lv[l], l);
}

namespace {

Pair2 residuals(const ds_context* c) { return Pair2{{c->pcg.r, c->pcg.r_alt}}; }
Pair2 directions(const ds_context* c) { return Pair2{{c->pcg.p[0], c->pcg.p[1]}}; }

// Runs f with the box type of the context's level 0, or of its coarser level l.
template <typename F>
void with_box(const ds_context* c, F&& f) {
    switch (c->mg.box[0]) {
        case kMgBoxSmall: return f.template operator()<BoxS>();
        case kMgBoxMedium: return f.template operator()<BoxM>();
        case kMgBoxThinX: return f.template operator()<BoxLX>();
        case kMgBoxThinZ: return f.template operator()<BoxLZ>();
        default: return f.template operator()<BoxL>();
    }
}

template <typename F>
void with_coarse_box(const ds_context* c, int l, F&& f) {
    switch (c->mg.box[l]) {
        case kMgBoxSmall: return f.template operator()<BoxD>();
        case kMgBoxThinX: return f.template operator()<BoxCX>();
        case kMgBoxThinZ: return f.template operator()<BoxCZ>();
        default: return f.template operator()<BoxC>();
    }
}

void launch_bottom(const MgBottom& B, const float* r, float* out, const double* partials, uint32_t blocks, PcgStatus* st,
                   double tol2, uint32_t mode, uint32_t k, hipStream_t s) {
    auto launch = [&]<int N>() { mg_bottom_kernel<N><<<1, kBottomThreads, 0, s>>>(B, r, out, partials, blocks, st, tol2, mode, k); };
    switch (B.count) {
        case 0: return launch.template operator()<0>();
        case 1: return launch.template operator()<1>();
        case 2: return launch.template operator()<2>();
        case 3: return launch.template operator()<3>();
        case 4: return launch.template operator()<4>();
        default: return launch.template operator()<5>();
    }
}

// Level 0's down kernel, the coarser levels, level 0's post kernel: the V-cycle of the residual that
// iteration k leaves (advance: after its direction kernel; else of the residual of index k as it stands).
void launch_cycle(ds_context* c, uint32_t k, bool advance, float* xh, float* xl, double tol2, uint32_t mode) {
    const uint32_t after = k + (advance ? 1u : 0u);
    MgWork& w = c->mg;
    PcgWork& pw = c->pcg;
    hipStream_t s = c->stream;
    PcgStatus* st = pw.status;
    const uint32_t per = w.per;
    const Pair2 r = residuals(c), p = directions(c);
    const bool direct = w.levels == 1;
    const MgLevel &L0 = w.lv[0], &L1 = w.lv[direct ? 0 : 1];
    with_box(c, [&]<typename B>() {
        if (direct && advance) mg_down0_kernel<B, true, false><<<pw.blocks, B::T, 0, s>>>(L0, L1, per, r, p, xh, xl, nullptr, nullptr, pw.partials, pw.hist, st, k);
        else if (advance) mg_down0_kernel<B, true, true><<<pw.blocks, B::T, 0, s>>>(L0, L1, per, r, p, xh, xl, w.vec[0][1], w.vec[1][0], pw.partials, pw.hist, st, k);
        else if (!direct) mg_down0_kernel<B, false, true><<<pw.blocks, B::T, 0, s>>>(L0, L1, per, r, p, xh, xl, w.vec[0][1], w.vec[1][0], pw.partials, pw.hist, st, k);
    });
    const int bf = w.bottom_first;
    for (int l = 1; l < bf; ++l)
        with_coarse_box(c, l, [&]<typename B>() {
            mg_down_kernel<B><<<(B::grid(w.lv[l]).count + 7u) & ~7u, B::T, 0, s>>>(w.lv[l], w.lv[l + 1], per, w.vec[l][0], w.vec[l][1], w.vec[l + 1][0],
                                                                                 st);
        });
    launch_bottom(w.bottom, direct ? nullptr : w.vec[bf][0], direct ? nullptr : w.vec[bf][2], pw.partials, pw.blocks, st, tol2,
                  mode, after, s);
    for (int l = bf - 1; l >= 1; --l)
        with_coarse_box(c, l, [&]<typename B>() {
            mg_up_kernel<B><<<(B::grid(w.lv[l]).count + 7u) & ~7u, B::T, 0, s>>>(w.lv[l], w.lv[l + 1], per, w.vec[l][0], w.vec[l][1], w.vec[l + 1][2],
                                                                               w.vec[l][2], st);
        });
    if (direct) {
        mg_dense_kernel<<<L0.n, kBlock, 0, s>>>(L0.n, w.dense, r, w.z, st, after);
        mg_dot_kernel<<<pw.blocks, kMgDotThreads, 0, s>>>(L0.n, r, w.z, pw.partials, st, after);
    } else {
        with_box(c, [&]<typename B>() {
            mg_post0_kernel<B><<<pw.blocks, B::T, 0, s>>>(L0, L1, per, r, w.vec[0][1], w.vec[1][2], w.z, pw.partials, st, after);
        });
    }
    check_launch("multigrid V-cycle");
}

__global__ void mg_set_iteration_kernel(PcgStatus* status, uint32_t k) {
    if (threadIdx.x == 0) {
        status->k = k;
        status->stop = 0u;
    }
}

}  // namespace

uint32_t mg_blocks(const ds_context* c) {
    uint32_t n = 8;
    with_box(c, [&]<typename B>() { n = B::grid(c->mg.lv[0]).count; });
    return std::min<uint32_t>(kPcgMaxBlocks, (n + 7u) & ~7u);
}

void mg_start(ds_context* c, uint32_t k, double tol2, uint32_t first, uint32_t reject) {
    launch_cycle(c, k, false, nullptr, nullptr, tol2, (first ? 2u : 0u) | (reject << 2));
}

void mg_set_iteration(ds_context* c, uint32_t k) {
    mg_set_iteration_kernel<<<1, 64, 0, c->stream>>>(c->pcg.status, k);
    check_launch("mg_set_iteration_kernel");
}

// Eight direct launches at 128^3, six at 64^3: the host queues them faster (2.9 us each) than the GPU
// runs them. (Replayed as a graph per iteration they cost about 8 us more at each graph's edge:
// simulate at 64^3, 20 steps, 9.59 against 9.03 ms.)
void mg_iteration(ds_context* c, uint32_t k, float* xh, float* xl, double tol2) {
    PcgWork& pw = c->pcg;
    with_box(c, [&]<typename B>() {
        mg_direction_kernel<B><<<pw.blocks, B::T, 0, c->stream>>>(c->mg.lv[0], c->mg.per, c->mg.z, directions(c), pw.partials, pw.hist,
                                                                 pw.status, k);
    });
    launch_cycle(c, k, true, xh, xl, tol2, 0u);
}

}  // namespace ds

