// rbgs.hip — the reference's own pressure solve on gfx950 (DS_PROJECTION_RBGS): red-black
// Gauss-Seidel from p = 0 for `pressure_iterations` sweeps of each colour (projection_forward,
// solvers/smoke/operators.cu:1004-1013; rbgs_kernel, :885-902), its unrolled reverse
// (projection_vjp, :1020-1031; rbgs_reverse_kernel, :935-955) and its tangent (projection_jvp,
// :1015-1018: the same sweeps with the fixed boundary values zeroed).
//
// A sweep updates one colour, so one launch covers only that colour's cells (x advances by 2
// within a row); the forward sweeps run two iterations to a launch in boxes with a halo
// (rbgs_box_kernel). The reverse of a sweep of colour P scatters p_bar[i] / diag_i (i of colour P) to
// i's connected neighbours, adds it to rhs_bar[i] and clears p_bar[i]; here it is a gather: the
// neighbours (colour 1 - P) read p_bar[i] / diag_i, and the clearing and the rhs_bar update of
// colour P are deferred into the next launch, which runs over colour P. So each launch writes
// only its own colour: no atomics, deterministic, 2 * pressure_iterations + 1 launches.
//
// A periodic axis with an odd cell count puts cells of one colour side by side across the seam;
// the reference's kernel then reads a neighbour that the same launch writes, and so does this one.
#include <hip/hip_runtime.h>

#include <utility>

#include "context.hpp"
#include "kernels.hpp"
#include "rhs.hpp"

namespace ds {

namespace {

// pressure_neighbor (operators.cu:852-873): the neighbour of (x, y, z) along dimension d in
// direction dir: a connected fluid cell (index j), or a fixed-value face (value), or neither.
__device__ __forceinline__ void rbgs_neighbour(const Geo& g, const SBound& b, const uint8_t* __restrict__ mask, int x, int y, int z, int d,
                                               int dir, uint32_t& j, bool& connected, bool& fixed, float& fixed_value) {
    int c[3]{x, y, z};
    c[d] += dir;
    const int size = dim_size(g, d);
    connected = false;
    fixed = false;
    if (c[d] < 0 || c[d] >= size) {
        if (b.modes[2 * d] == 2u && b.modes[2 * d + 1] == 2u) {
            c[d] = c[d] < 0 ? c[d] + size : c[d] - size;
        } else {
            const int face = 2 * d + (dir > 0 ? 1 : 0);
            fixed = b.modes[face] == 0u;
            fixed_value = b.values[face];
            return;
        }
    }
    j = cidx(g, c[0], c[1], c[2]);
    connected = mask[j] == 0;
}

// Diagonal of every cell (connected neighbours + fixed faces), 0 for solids, the anchor and cells
// with no neighbour: the cells the sweeps leave alone.
__global__ __launch_bounds__(256) void rbgs_diag_kernel(Geo g, const SBound* __restrict__ bp, const uint8_t* __restrict__ mask,
                                                        uint32_t anchor, uint8_t* __restrict__ diag) {
    const uint32_t i = xcd_block() * blockDim.x + threadIdx.x;
    if (i >= g.n) return;
    if (mask[i] != 0 || i == anchor) {
        diag[i] = 0;
        return;
    }
    int x, y, z;
    decode_cell(g, i, x, y, z);
    uint32_t count = 0;
#pragma unroll
    for (int d = 0; d < 3; ++d)
#pragma unroll
        for (int dir = -1; dir <= 1; dir += 2) {
            uint32_t j;
            bool connected, fixed;
            float fv;
            rbgs_neighbour(g, *bp, mask, x, y, z, d, dir, j, connected, fixed, fv);
            count += (connected || fixed) ? 1u : 0u;
        }
    diag[i] = (uint8_t)count;
}

// Cell (x, y, z) of colour `parity` handled by thread t of a colour launch: rows of (nx + 1) / 2.
__device__ __forceinline__ bool colour_cell(const Geo& g, uint32_t t, uint32_t parity, int& x, int& y, int& z) {
    const uint32_t half = ((uint32_t)g.nx + 1u) / 2u;
    const uint32_t row = t / half;
    const uint32_t k = t - row * half;
    y = (int)(row % (uint32_t)g.ny);
    z = (int)(row / (uint32_t)g.ny);
    if (z >= g.nz) return false;
    x = (int)(2u * k + ((parity + (uint32_t)y + (uint32_t)z) & 1u));
    return x < g.nx;
}

// Right-hand side of the sweeps: b = -h^2 div(u) / dt on fluid non-anchor cells, 0 elsewhere
// (pressure_rhs_kernel, operators.cu:875-883); with Adjoint, the projection reverse as a gather
// (project_velocity_reverse_kernel, operators.cu:922-933) on fluid cells. Also zeroes x.
template <int Kind>
__global__ __launch_bounds__(256) void rbgs_rhs_kernel(Geo g, const uint8_t* __restrict__ mask, uint32_t anchor, RhsIn in,
                                                       float* __restrict__ b, float* __restrict__ x0, float* __restrict__ x1) {
    const uint32_t i = xcd_block() * blockDim.x + threadIdx.x;
    if (i >= g.n) return;
    x0[i] = 0.0f;
    x1[i] = 0.0f;
    const bool skip = mask[i] != 0 || (Kind != kRhsAdjoint && i == anchor);
    if (skip) {
        b[i] = 0.0f;
        return;
    }
    int x, y, z;
    decode_cell(g, i, x, y, z);
    b[i] = cell_rhs<Kind>(g, in, mask, nullptr, i, x, y, z);
}

// rbgs_kernel (operators.cu:885-902) over the cells of one colour.
__global__ __launch_bounds__(256) void rbgs_sweep_kernel(Geo g, const SBound* __restrict__ bp, const uint8_t* __restrict__ mask,
                                                         const uint8_t* __restrict__ diag, const float* __restrict__ rhs, float* p,
                                                         uint32_t parity) {
    int x, y, z;
    if (!colour_cell(g, blockIdx.x * blockDim.x + threadIdx.x, parity, x, y, z)) return;
    const uint32_t i = cidx(g, x, y, z);
    const uint32_t d = diag[i];
    if (d == 0u) return;
    float sum = rhs[i];
#pragma unroll
    for (int dim = 0; dim < 3; ++dim)
#pragma unroll
        for (int dir = -1; dir <= 1; dir += 2) {
            uint32_t j;
            bool connected, fixed;
            float fv = 0.0f;
            rbgs_neighbour(g, *bp, mask, x, y, z, dim, dir, j, connected, fixed, fv);
            if (connected) sum += p[j];
            else if (fixed) sum += fv;
        }
    p[i] = sum / (float)d;
}

// `iterations` <= S red-black iterations (a red and a black sweep each) in one launch. A workgroup
// loads a box and 2 S cells around it; every sweep shrinks what is up to date by one cell, so after
// the last one the box is, and it is written to the other buffer (p_in is still read by others).
//
// Thread (k, j) holds two cells of row j, x = 2k and 2k + 1 (one less in odd rows), on every plane of
// the box: p, rhs and the diagonal in registers. So shifted, the first cell has the colour of its
// plane's parity in every row, and which cell a sweep updates is known at compile time. The partner
// and the neighbours along z are the thread's own registers, the other three come from LDS (one array
// for the first cells, one for the second: consecutive lanes on consecutive words). A box starts at
// even coordinates, so the parity of the local coordinates is the colour; a periodic axis of odd
// extent has no such colouring.
//
// A cell outside the domain holds what a sweep adds for it, the face's fixed value or 0, and a solid
// one holds 0; neither is updated. So the sum is the six neighbours in the order of
// rbgs_sweep_kernel, without tests: the same values (a zero can have the other sign).
//
// Bound by the loads of the halo (4 1/2 times the box, in lines of 128 bytes) and the latency of a
// workgroup's load, sweep and store phases. At 128 x 192 x 128, us per iteration: a launch per colour
// 35.4 (seven mask tests and loads, an index division and a rounded division per cell); boxes of
// 32 x 16 x 8, two iterations a launch, 11.7 (23.5 a launch: 14.1 without the paired loads, 18.7
// with the selects of unshifted rows and the full division); one iteration a launch: 32 x 16 x 8
// 19.2, 64 x 8 x 8 16.0, 64 x 16 x 8 17.8, 128 x 8 x 8 18.8; two: 64 x 16 x 8 15.2, 32 x 16 x 16
// 19.8, 32 x 24 x 8 16.0; three, 32 x 16 x 8: 21.3. Small grids (two steps of 160 iterations): 24^3
// 3707 -> 1245 us, 64^3 3472 -> 1352, 96 x 100 x 75 5535 -> 2152.
template <int S_, int X_, int Y_, int Z_>
struct SweepBox {
    static constexpr int S = S_, X = X_, Y = Y_, Z = Z_, H = 2 * S_;   // iterations, box, halo
    static constexpr int K = X / 2 + H + 1, RY = Y + 2 * H, RZ = Z + 2 * H, P = K * RY;
    static constexpr int T = (P + 63) / 64 * 64;
};

// Index of coordinate v along an axis of n cells, or -1 outside, where `value` becomes what a sweep adds.
__device__ __forceinline__ int sweep_coord(const SBound& b, int d, int v, int n, float& value) {
    if ((unsigned)v < (unsigned)n) return v;
    if (b.modes[2 * d] == 2u && b.modes[2 * d + 1] == 2u) return wrapi(v, n);
    const int face = 2 * d + (v < 0 ? 0 : 1);
    value = b.modes[face] == 0u ? b.values[face] : 0.0f;
    return -1;
}

// sum / d, rounded to nearest, for d = 1 .. 6: the reciprocal of such a d is the nearest FP32 number,
// so one corrected step gives the nearest quotient (Markstein 1990; tiny results, below 2^-100, can
// be one unit off); the fix-up is for zeros, infinities and NaN. d = 0 gives what the caller drops.
__device__ __forceinline__ float divide_small(float sum, float d) {
    const float rd = __builtin_amdgcn_rcpf(d);
    const float q = sum * rd;
    return __builtin_amdgcn_div_fixupf(__fmaf_rn(__fmaf_rn(-d, q, sum), rd, q), d, sum);
}

// g, bp: the grid and its boundary with the axes in the boxes' order (box_axes).
// Wide: the thread's two cells in one load; x is not periodic then and nx >= 2 (a pair that has one
// cell outside reads the pair next to it).
template <typename B, bool Wide>
__global__ __launch_bounds__(B::T) void rbgs_box_kernel(Geo g, const SBound* __restrict__ bp, const uint8_t* __restrict__ diag,
                                                        const float* __restrict__ rhs, const float* __restrict__ p_in,
                                                        float* __restrict__ p_out, uint32_t ntx, uint32_t nty, uint32_t boxes, int ex, int ey,
                                                        int ez, int iterations) {
    constexpr int H = B::H, K = B::K, RY = B::RY, RZ = B::RZ, P = B::P, Pad = K + 2;
    __shared__ float s[2][RZ * P + 2 * Pad];
    const uint32_t b = xcd_block();
    if (b >= boxes) return;
    const int bx = (int)(b % ntx), by = (int)(b / ntx % nty), bz = (int)(b / ntx / nty);
    const int t = (int)threadIdx.x, j = t / K, k = t - j * K, odd = j & 1;
    const bool active = j < RY;
    const int x = bx * ex - H + 2 * k - odd, y = by * ey - H + j, z0 = bz * ez - H;
    float out[2]{}, out_y = 0.0f;
    const int iy = sweep_coord(*bp, 1, y, g.ny, out_y);
    const int ix[2]{sweep_coord(*bp, 0, x, g.nx, out[0]), sweep_coord(*bp, 0, x + 1, g.nx, out[1])};
    bool in[2];
    uint32_t at[2], keep[2];   // keep: 0 where there is nothing to update, or a neighbour is not loaded
#pragma unroll
    for (int f = 0; f < 2; ++f) {
        in[f] = active && iy >= 0 && ix[f] >= 0;
        if (iy < 0) out[f] = out_y;
        at[f] = in[f] ? (uint32_t)iy * (uint32_t)g.nx + (uint32_t)ix[f] : 0u;
        keep[f] = in[f] && j != 0 && j != RY - 1 && k != (f == 0 ? 0 : K - 1) ? 7u : 0u;
    }
    const uint32_t pair = in[0] || in[1] ? (uint32_t)iy * (uint32_t)g.nx + (uint32_t)min(max(x, 0), g.nx - 2) : 0u;
    const bool first_high = x == g.nx - 1, second_low = x == -1;
    const uint32_t plane = (uint32_t)g.nx * (uint32_t)g.ny;
    float p[2][RZ], r[2][RZ];
    uint32_t d[2][(RZ + 3) / 4]{};
    float out_z[2]{};
    const bool wraps = sweep_coord(*bp, 2, -1, g.nz, out_z[0]) >= 0;
    (void)sweep_coord(*bp, 2, g.nz, g.nz, out_z[1]);
    int wz = wraps ? wrapi(z0, g.nz) : 0;
#pragma unroll
    for (int z = 0; z < RZ; ++z) {
        const bool inside = wraps || (unsigned)(z0 + z) < (unsigned)g.nz;
        const float outside = z0 + z < 0 ? out_z[0] : out_z[1];
        const size_t base = (size_t)(wraps ? wz : min(max(z0 + z, 0), g.nz - 1)) * plane;
        wz = wz + 1 == g.nz ? 0 : wz + 1;
        float pv[2], rv[2];
        uint32_t dv[2];
        if constexpr (Wide) {
            uint16_t dw;
            __builtin_memcpy(pv, p_in + base + pair, sizeof pv);
            __builtin_memcpy(rv, rhs + base + pair, sizeof rv);
            __builtin_memcpy(&dw, diag + base + pair, sizeof dw);
            dv[0] = first_high ? dw >> 8 : dw;   // (the bits above are masked below)
            dv[1] = second_low ? dw : dw >> 8;
            const float p0 = pv[0], r0 = rv[0];
            pv[0] = first_high ? pv[1] : pv[0], rv[0] = first_high ? rv[1] : rv[0];
            pv[1] = second_low ? p0 : pv[1], rv[1] = second_low ? r0 : rv[1];
        } else {
#pragma unroll
            for (int f = 0; f < 2; ++f) pv[f] = p_in[base + at[f]], rv[f] = rhs[base + at[f]], dv[f] = diag[base + at[f]];
        }
#pragma unroll
        for (int f = 0; f < 2; ++f) {
            r[f][z] = rv[f];
            p[f][z] = in[f] && inside ? pv[f] : inside ? out[f] : outside;
            d[f][z / 4] |= (dv[f] & (inside ? keep[f] : 0u)) << (8 * (z % 4));
        }
    }
    if (active) {
#pragma unroll
        for (int z = 1; z < RZ - 1; ++z) s[(z + 1) & 1][Pad + z * P + t] = p[(z + 1) & 1][z];   // the black cells
    }
    __syncthreads();
    // sweep N of the launch, of colour N & 1: the planes that are not up to date any more are left out
    auto sweep = [&]<int N>() {
        constexpr int C = N & 1;
        if (active) {
#pragma unroll
            for (int z = N + 1; z < RZ - 1 - N; ++z) {
                const int f = (z + C) & 1;
                const float* o = &s[1 - f][Pad + z * P + t];
                const float* row = o + f - odd;
                float sum = r[f][z] + (f == 0 ? o[-1] : p[0][z]);
                sum += f == 0 ? p[1][z] : o[1];
                sum += row[-K];
                sum += row[K];
                sum += p[f][z - 1];
                sum += p[f][z + 1];
                const float dz = (float)((d[f][z / 4] >> (8 * (z % 4))) & 255u);
                p[f][z] = dz != 0.0f ? divide_small(sum, dz) : p[f][z];
                s[f][Pad + z * P + t] = p[f][z];
            }
        }
        __syncthreads();
    };
    [&]<int... It>(std::integer_sequence<int, It...>) {
        ((It < iterations ? (sweep.template operator()<2 * It>(), sweep.template operator()<2 * It + 1>()) : void()), ...);
    }(std::make_integer_sequence<int, B::S>{});
    if (j < H || j >= H + ey) return;
    const int lx = 2 * k - odd;
#pragma unroll
    for (int f = 0; f < 2; ++f) {
        if (!in[f] || lx + f < H || lx + f >= H + ex || y >= g.ny || x + f >= g.nx) continue;   // (not a periodic image)
#pragma unroll
        for (int z = H; z < RZ - H; ++z)
            if (z < H + ez && z0 + z < g.nz) p_out[(size_t)(z0 + z) * plane + at[f]] = p[f][z];
    }
}

// One launch of the reverse over the cells of colour `parity`: with Finish, the deferred second
// half of the previous reverse sweep (that colour's rhs_bar += p_bar / diag, p_bar = 0); with
// Gather, the first half of the next one (p_bar += sum over connected neighbours of p_bar / diag).
// links: how often a cell is its own neighbour, twice per periodic axis of one cell. A sweep reads the
// cell's old value that often, so its reverse leaves that share in p_bar instead of 0.
template <bool Finish, bool Gather>
__global__ __launch_bounds__(256) void rbgs_reverse_kernel(Geo g, const SBound* __restrict__ bp, const uint8_t* __restrict__ mask,
                                                           const uint8_t* __restrict__ diag, float* pbar, float* __restrict__ rbar,
                                                           uint32_t parity, uint32_t links) {
    int x, y, z;
    if (!colour_cell(g, blockIdx.x * blockDim.x + threadIdx.x, parity, x, y, z)) return;
    const uint32_t i = cidx(g, x, y, z);
    float own = pbar[i];
    if (Finish) {
        const uint32_t d = diag[i];
        if (d != 0u) {
            own /= (float)d;
            rbar[i] += own;
            own = links ? own * (float)links : 0.0f;
        }
    }
    if (Gather && mask[i] == 0) {
        float s = 0.0f;
#pragma unroll
        for (int dim = 0; dim < 3; ++dim)
#pragma unroll
            for (int dir = -1; dir <= 1; dir += 2) {
                uint32_t j;
                bool connected, fixed;
                float fv;
                rbgs_neighbour(g, *bp, mask, x, y, z, dim, dir, j, connected, fixed, fv);
                if (connected && j != i) {
                    const uint32_t dj = diag[j];
                    if (dj != 0u) s += pbar[j] / (float)dj;
                }
            }
        own += s;
    }
    pbar[i] = own;
}

template <typename B>
uint64_t box_count(const Geo& g) {
    auto count = [](int n, int most) { return ((uint64_t)n + (uint64_t)most - 1) / (uint64_t)most; };
    return count(g.nx, B::X) * count(g.ny, B::Y) * count(g.nz, B::Z);
}

// Cells that the boxes of type B load, their halos among them.
template <typename B>
uint64_t box_points(const Geo& g) {
    return box_count<B>(g) * (uint64_t)(2 * B::P * B::RZ);
}

// The grid with the axes in the order of the boxes: those of one cell last. The cells lie in memory the
// same way, so a grid of 1 x ny x nz is swept as ny x nz x 1 (the sum's order follows; colours are the
// same). of: the grid's axes.
Geo box_axes(const Geo& g, int (&of)[3]) {
    Geo b = g;   // (the boxes use its cells and extents only)
    int* const extents[3]{&b.nx, &b.ny, &b.nz};
    for (int a = 0; a < 3; ++a) of[a] = a;
    for (int pass = 0; pass < 2; ++pass)
        for (int a = 0; a < 2; ++a)
            if (*extents[a] == 1) {
                std::swap(*extents[a], *extents[a + 1]);
                std::swap(of[a], of[a + 1]);
            }
    return b;
}

// One launch of rbgs_box_kernel; boxes of equal even extents that cover the grid.
template <typename B>
void launch_boxes(ds_context* c, const Geo& g, bool periodic_x, const SBound* bp, const float* b, const float* p_in, float* p_out,
                  uint32_t iterations) {
    auto split = [](int n, int most, uint32_t& count) {
        count = ((uint32_t)n + (uint32_t)most - 1) / (uint32_t)most;
        return (int)((((uint32_t)n + count - 1) / count + 1u) & ~1u);
    };
    uint32_t cx, cy, cz;
    const int ex = split(g.nx, B::X, cx), ey = split(g.ny, B::Y, cy), ez = split(g.nz, B::Z, cz);
    const uint32_t boxes = cx * cy * cz, blocks = (boxes + 7u) & ~7u;
    auto launch = [&](auto kernel) {
        kernel<<<blocks, B::T, 0, c->stream>>>(g, bp, c->rbgs_diag, b, p_in, p_out, cx, cy, boxes, ex, ey, ez, (int)iterations);
    };
    if (!periodic_x && g.nx >= 2) launch(rbgs_box_kernel<B, true>);
    else launch(rbgs_box_kernel<B, false>);
}

uint32_t colour_blocks(const Geo& g) {
    const uint64_t threads = (uint64_t)(((uint32_t)g.nx + 1u) / 2u) * (uint64_t)g.ny * (uint64_t)g.nz;
    return (uint32_t)((threads + kBlock - 1) / kBlock);
}

}  // namespace

void rbgs_prepare(ds_context* c) {
    rbgs_diag_kernel<<<xcd_blocks_for(c->geo.n), kBlock, 0, c->stream>>>(c->geo, c->d_pb, c->mask, (uint32_t)c->anchor, c->rbgs_diag);
    check_launch("rbgs_diag_kernel");
    // the pressure boundary and its zeroed form for the boxes
    int of[3];
    (void)box_axes(c->geo, of);
    SBound host[2]{c->pb, c->pb_zero};
    for (int a = 0; a < 3; ++a)
        for (int f = 0; f < 2; ++f) {
            host[0].modes[2 * a + f] = host[1].modes[2 * a + f] = c->pb.modes[2 * of[a] + f];
            host[0].values[2 * a + f] = c->pb.values[2 * of[a] + f];
        }
    SBound* const bounds = device_alloc<SBound>(c, 2);
    DS_HIP(hipMemcpy(bounds, host, sizeof host, hipMemcpyHostToDevice));
    c->d_rbgs_pb = bounds;
}

// Forward (kind 1) or tangent (kind 3): p = RBGS(rhs of u) from 0, into xh (xl = 0). Adjoint
// (kind 2): xh = rhs_bar of the unrolled reverse for the projection reverse of u (+ extra), xl = 0.
ds_solve_info rbgs_solve_kind(ds_context* c, int kind, const float* const u[3], const float* const extra[3], float* xh, float* xl) {
    const Geo& g = c->geo;
    RhsIn in{};
    for (int a = 0; a < 3; ++a) {
        in.u[a] = u[a];
        in.extra[a] = extra ? extra[a] : nullptr;
    }
    float* b = c->pcg.b;
    const uint32_t G = xcd_blocks_for(g.n);
    const uint32_t anchor = (uint32_t)c->anchor;
    if (kind == kRhsAdjoint) rbgs_rhs_kernel<kRhsAdjoint><<<G, kBlock, 0, c->stream>>>(g, c->mask, anchor, in, b, xh, xl);
    else rbgs_rhs_kernel<kRhsForward><<<G, kBlock, 0, c->stream>>>(g, c->mask, anchor, in, b, xh, xl);
    check_launch("rbgs_rhs_kernel");
    const uint32_t iterations = c->config.pressure_iterations;
    const uint32_t CB = colour_blocks(g);
    if (kind != kRhsAdjoint) {
        const SBound* bp = kind == kRhsTangent ? c->d_pb_zero : c->d_pb;
        const bool coloured = (!c->pressure_periodic[0] || g.nx % 2 == 0) && (!c->pressure_periodic[1] || g.ny % 2 == 0) &&
                              (!c->pressure_periodic[2] || g.nz % 2 == 0);
        // boxes wherever the colouring holds: the launches of one colour remain for a periodic axis of
        // odd extent, where a sweep reads a neighbour that it writes itself
        if (coloured && iterations > 0) {
            int of[3];
            const Geo gb = box_axes(g, of);
            const SBound* const boxes_bp = kind == kRhsTangent ? c->d_rbgs_pb + 1 : c->d_rbgs_pb;
            auto sweeps = [&]<typename B>() {
                const uint32_t launches = (iterations + B::S - 1) / B::S;
                float* from = launches % 2 ? xl : xh;   // both are zero; the last launch writes xh
                for (uint32_t l = 0, done = 0; l < launches; ++l, done += B::S) {
                    float* to = from == xh ? xl : xh;
                    launch_boxes<B>(c, gb, c->pressure_periodic[of[0]], boxes_bp, b, from, to, std::min<uint32_t>(B::S, iterations - done));
                    from = to;
                }
            };
            // A small grid is bound by the latency of one workgroup, so its boxes are flat while they
            // are at most one for each of the 256 CUs: 64^3 (256 flat boxes, 64 deep ones), two steps of
            // 160 iterations, 1352 against 1929 us, 24^3 1245 against 1750; beyond that the halo
            // decides: 96 x 100 x 75 (798 flat boxes, 210 deep ones) 2788 against 2152 us.
            // On a grid of a few cells along z or x Deep sweeps mostly cells outside it; a thin box is taken
            // where it has less than two thirds of Deep's points (up to 2 cells along z, 8 along x). Steps of
            // 80 iterations with Deep, with the thin box, and with a launch per colour: 1024 x 1024 x 1 1529,
            // 1098, 2002 us; 512 x 512 x 2 604, 452, 1112; 2 x 1024 x 1024 6647, 2449, 2943 (4 x 64 x 8: 3481);
            // 4 x 1024 x 1024 7056, 2484, 5168 (8 x 32 x 8: 4359); 6 x 1024 x 1024 7415, 4405, 7923. With axes of
            // one cell last: 1 x 1024 x 1024 6051 -> 1101, 1024 x 1 x 1024 2876 -> 1094. Along y Deep does:
            // 1024 x 2 x 1024 3046 against 3193.
            // Along x only beyond one deep box for each CU: 4 x 256 x 256 (512 of them) 663, 522; 7 x 128 x 256 (256)
            // 503, 515; 8 x 128 x 128 (128) 483, 492.
            using Flat = SweepBox<2, 32, 16, 2>;
            using Deep = SweepBox<2, 32, 16, 8>;
            using Thin2 = SweepBox<2, 2, 64, 8>;
            using Thin4 = SweepBox<2, 4, 64, 8>;
            const uint64_t deep = box_points<Deep>(gb);
            auto thin = [&]<typename B>() { return 3 * box_points<B>(gb) < 2 * deep; };
            if (box_count<Flat>(gb) <= 256u || thin.template operator()<Flat>()) sweeps.template operator()<Flat>();
            else if (box_count<Deep>(gb) <= 256u) sweeps.template operator()<Deep>();
            else if (gb.nx <= 2) sweeps.template operator()<Thin2>();
            else if (thin.template operator()<Thin4>()) sweeps.template operator()<Thin4>();
            else sweeps.template operator()<Deep>();
            fill_zero(c, xl, g.n);
        } else for (uint32_t it = 0; it < iterations; ++it) {
            rbgs_sweep_kernel<<<CB, kBlock, 0, c->stream>>>(g, bp, c->mask, c->rbgs_diag, b, xh, 0u);
            rbgs_sweep_kernel<<<CB, kBlock, 0, c->stream>>>(g, bp, c->mask, c->rbgs_diag, b, xh, 1u);
        }
        check_launch("rbgs_sweep_kernel");
    } else if (iterations > 0) {
        // b holds p_bar; xh accumulates rhs_bar. Reverse order of the sweeps: colour 1, then 0, ...
        const int extents[3]{g.nx, g.ny, g.nz};
        uint32_t links = 0;
        for (int a = 0; a < 3; ++a) links += c->pressure_periodic[a] && extents[a] == 1 ? 2u : 0u;
        rbgs_reverse_kernel<false, true><<<CB, kBlock, 0, c->stream>>>(g, c->d_pb, c->mask, c->rbgs_diag, b, xh, 0u, links);
        for (uint32_t k = 1; k < 2 * iterations; ++k)
            rbgs_reverse_kernel<true, true><<<CB, kBlock, 0, c->stream>>>(g, c->d_pb, c->mask, c->rbgs_diag, b, xh, k & 1u, links);
        rbgs_reverse_kernel<true, false><<<CB, kBlock, 0, c->stream>>>(g, c->d_pb, c->mask, c->rbgs_diag, b, xh, 0u, links);
        check_launch("rbgs_reverse_kernel");
    }
    ds_solve_info si{};
    si.iterations = iterations;
    si.converged = 1;
    return si;
}

}  // namespace ds
