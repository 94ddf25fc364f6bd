// device.hpp — gfx950 device helpers of the smoke solver: grid geometry, boundary-aware loads,
// trilinear sampling and its transpose, RK2 backtrace, wave64 FP64 reductions.
//
// The discretisation restates solvers/smoke/operators.cu:32-284 (Xayah-Graphics/diff-solver) in
// FP32: indexing x + nx*(y + ny*z), face extents n_a + 1 on the own axis, boundary loads
// (fixed-value faces return their value, periodic wraps, otherwise clamp), trilinear sampling
// with its analytic gradient, and the RK2 midpoint backtrace with box clamp and solid bisection.
// Indices are 32-bit (grids up to 1024^3); divisions by runtime extents use multiply-high.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace ds {

constexpr int kBlock = 256;
constexpr int kWave = 64;

// Division by a runtime constant d >= 1 with a 32-bit multiply-high (round-up method):
// q = (umulhi(n, m) + n) >> s, valid for every 32-bit n.
struct FastDiv {
    uint32_t d, m, s;
};

inline FastDiv make_fastdiv(uint32_t d) {
    FastDiv f{d, 0u, 0u};
    uint32_t s = 0;
    while ((1ull << s) < d) ++s;
    f.s = s;
    f.m = (uint32_t)(((1ull << 32) * ((1ull << s) - d)) / d + 1ull);
    return f;
}

__device__ __forceinline__ uint32_t fdiv(uint32_t n, const FastDiv& f) {
    const uint64_t t = (uint64_t)__umulhi(n, f.m) + n;
    return (uint32_t)(t >> f.s);
}

// Geometry passed by value to every kernel (Grid, cuda_types.h:13-19, plus derived sizes).
struct Geo {
    int nx, ny, nz;
    float h, inv_h, dt;
    uint32_t h_pow2;       // 1 when h is a power of two: p / h is then exactly p * inv_h
    uint32_t n;            // cells
    uint32_t nf[3];        // faces per axis
    uint32_t foff[4];      // offsets of axis 0/1/2 in the concatenated face index space, total
    FastDiv cx, cy;        // cell decode: divide by nx, ny
    FastDiv fx[3], fy[3];  // face decode per axis: divide by extent x, extent y
};

struct VBound {   // VelocityBoundaryData, cuda_types.h:26-29
    uint32_t modes[6];
    float values[18];
};
struct SBound {   // ScalarBoundaryData, cuda_types.h:21-24
    uint32_t modes[6];
    float values[6];
};

__device__ __forceinline__ int ext(const Geo& g, int axis, int dim) {
    const int base = dim == 0 ? g.nx : dim == 1 ? g.ny : g.nz;
    return base + (axis == dim ? 1 : 0);
}
__device__ __forceinline__ int dim_size(const Geo& g, int dim) { return dim == 0 ? g.nx : dim == 1 ? g.ny : g.nz; }
__device__ __forceinline__ uint32_t cidx(const Geo& g, int x, int y, int z) {
    return (uint32_t)x + (uint32_t)g.nx * ((uint32_t)y + (uint32_t)g.ny * (uint32_t)z);
}
__device__ __forceinline__ uint32_t fidx(const Geo& g, int axis, int x, int y, int z) {
    return (uint32_t)x + (uint32_t)ext(g, axis, 0) * ((uint32_t)y + (uint32_t)ext(g, axis, 1) * (uint32_t)z);
}
__device__ __forceinline__ void decode_cell(const Geo& g, uint32_t i, int& x, int& y, int& z) {
    const uint32_t t = fdiv(i, g.cx);
    x = (int)(i - t * (uint32_t)g.nx);
    const uint32_t u = fdiv(t, g.cy);
    y = (int)(t - u * (uint32_t)g.ny);
    z = (int)u;
}
// Local face index of axis A -> (x, y, z).
template <int A>
__device__ __forceinline__ void decode_face_axis(const Geo& g, uint32_t local, int& x, int& y, int& z) {
    const uint32_t ex = (uint32_t)ext(g, A, 0), ey = (uint32_t)ext(g, A, 1);
    const uint32_t t = fdiv(local, g.fx[A]);
    x = (int)(local - t * ex);
    const uint32_t u = fdiv(t, g.fy[A]);
    y = (int)(t - u * ey);
    z = (int)u;
}

// Runs body.template operator()<A>(local) for the axis A owning concatenated face index f
// (blocks straddle at most one axis boundary, so the branch is uniform in almost every wave).
template <typename Body>
__device__ __forceinline__ void for_face(const Geo& g, uint32_t f, Body&& body) {
    if (f < g.foff[1]) body.template operator()<0>(f);
    else if (f < g.foff[2]) body.template operator()<1>(f - g.foff[1]);
    else body.template operator()<2>(f - g.foff[2]);
}

// Workgroups are dispatched round-robin over the 8 XCDs (block b runs on XCD b % 8). Remapping
// gives each XCD a contiguous range of logical blocks, so the neighbour reuse of a stencil or
// a gather stays in that XCD's L2. The grid must be a multiple of 8.
__device__ __forceinline__ uint32_t xcd_block() {
    const uint32_t b = blockIdx.x, G = gridDim.x;
    return (b & 7u) * (G >> 3) + (b >> 3);
}

__device__ __forceinline__ bool vperiodic(const VBound& b, int d) { return b.modes[2 * d] == 3u && b.modes[2 * d + 1] == 3u; }
__device__ __forceinline__ bool speriodic(const SBound& b, int d) { return b.modes[2 * d] == 2u && b.modes[2 * d + 1] == 2u; }
// v modulo p for a coordinate that is at most one period outside [0, p) in almost every case.
__device__ __forceinline__ int wrapi(int v, int p) {
    int r = v < 0 ? v + p : v >= p ? v - p : v;
    if ((unsigned)r >= (unsigned)p) {
        r = v % p;
        r = r < 0 ? r + p : r;
    }
    return r;
}

// One axis of a trilinear stencil whose lower corner is at coordinate c0, on a lattice of `size`
// points: the stored coordinates of its two corners (periodic: modulo `period`, the cell count;
// else clamped), and whether each corner lies beyond a face whose value is fixed, with the value.
// The bounds are tested per axis, not per corner, and without divisions: a wave that holds one
// domain-edge cell runs this for all its lanes (the rows of a grid end in every second wave at 128^3),
// so the boundary path's instructions bound the trace kernels. With this form, the fixed stencils of
// the start point (start_velocity) and paired loads: velocity / scalar reverse 277 / 448 -> 159 / 207
// us (per axis at 128^3), velocity / scalar tangent 608 / 258 -> 180 / 79 us (96^3), forward velocity
// 133 -> 53 us (90 x 70 x 110, solids) and 1241 -> 756 us (256^3).
struct AxisStencil {
    int i[2];
    bool fixed[2];
    float value[2];
};
__device__ __forceinline__ AxisStencil axis_stencil(int c0, int size, bool periodic, int period, bool fix_lo, bool fix_hi, float lo,
                                                    float hi) {
    AxisStencil s;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const int c = c0 + k;
        const bool below = c < 0, above = c >= size;
        s.fixed[k] = (below && fix_lo) || (above && fix_hi);
        s.value[k] = below ? lo : hi;
        s.i[k] = periodic ? wrapi(c, period) : min(max(c, 0), size - 1);
    }
    return s;
}

// load_scalar's rule for axis d (operators.cu:115-121, scatter skip at :212).
template <int D>
__device__ __forceinline__ AxisStencil scalar_axis(const Geo& g, int c0, const SBound& b) {
    const int n = dim_size(g, D);
    return axis_stencil(c0, n, speriodic(b, D), n, b.modes[2 * D] == 0u, b.modes[2 * D + 1] == 0u, b.values[2 * D], b.values[2 * D + 1]);
}
// load_face's rule for the faces of axis A along axis D (operators.cu:105-113,125-132, scatter skip
// at :230-237). The axes are template parameters so that every boundary-array index is a
// compile-time constant (a runtime index into a by-value kernel argument would move it to scratch).
template <int A, int D>
__device__ __forceinline__ AxisStencil face_axis(const Geo& g, int c0, const VBound& b) {
    const uint32_t ml = b.modes[2 * D], mh = b.modes[2 * D + 1];
    return axis_stencil(c0, ext(g, A, D), vperiodic(b, D), dim_size(g, D), ml == 0u || (ml == 2u && A == D), mh == 0u || (mh == 2u && A == D),
                        b.values[3 * (2 * D) + A], b.values[3 * (2 * D + 1) + A]);
}

// Index x + ex (y + ey z) of a lattice whose extents are at most 1025: the partial products fit the
// 24-bit multiply, which runs at the full rate (the 32-bit one at a quarter of it).
__device__ __forceinline__ uint32_t lattice_index(int x, int y, int z, int ex, int ey) {
    return (uint32_t)x + __umul24((uint32_t)ex, (uint32_t)y + __umul24((uint32_t)ey, (uint32_t)z));
}

struct Corner8 {   // the 2x2x2 trilinear stencil: base cell and fractional offsets
    int x0, y0, z0;
    float tx, ty, tz;
};

// p / h: grid coordinates divide by h as the reference does (operators.cu:137-139,167-172); with a
// cell size that is not a power of two, p * (1/h) can round to the other side of a cell boundary.
// For a power of two the product is the same number and skips the division sequence (the branch
// is uniform: g is a kernel argument).
__device__ __forceinline__ float over_h(const Geo& g, float p) { return g.h_pow2 ? p * g.inv_h : p / g.h; }

__device__ __forceinline__ Corner8 corners(const Geo& g, float px, float py, float pz, float ox, float oy, float oz) {
    const float gx = over_h(g, px) - ox, gy = over_h(g, py) - oy, gz = over_h(g, pz) - oz;
    Corner8 c;
    const float fx = floorf(gx), fy = floorf(gy), fz = floorf(gz);
    // A non-finite or huge position (a diverged solve upstream) must not reach the index
    // arithmetic: clamped to +-2^24 cells (NaN to the lower bound) before the conversion, the
    // corner lies far outside the domain, fails every interior test without overflowing (x0 + 1
    // stays representable) and takes the boundary-mapped loads; finite positions within 2^24
    // cells of the domain are unchanged.
    constexpr float kFar = 16777216.0f;
    c.x0 = (int)__builtin_amdgcn_fmed3f(fx, -kFar, kFar);
    c.y0 = (int)__builtin_amdgcn_fmed3f(fy, -kFar, kFar);
    c.z0 = (int)__builtin_amdgcn_fmed3f(fz, -kFar, kFar);
    c.tx = gx - fx;
    c.ty = gy - fy;
    c.tz = gz - fz;
    return c;
}

struct Sample {
    float value, gx, gy, gz;
};

// Trilinear value and analytic gradient of 8 corner values (operators.cu:150-163).
template <bool Grad>
__device__ __forceinline__ Sample trilerp(const float v[8], const Corner8& c, float inv_h) {
    const float wx0 = 1.0f - c.tx, wx1 = c.tx, wy0 = 1.0f - c.ty, wy1 = c.ty, wz0 = 1.0f - c.tz, wz1 = c.tz;
    // v index: dx + 2*dy + 4*dz
    Sample s;
    s.value = wz0 * (wy0 * (wx0 * v[0] + wx1 * v[1]) + wy1 * (wx0 * v[2] + wx1 * v[3])) +
              wz1 * (wy0 * (wx0 * v[4] + wx1 * v[5]) + wy1 * (wx0 * v[6] + wx1 * v[7]));
    if (Grad) {
        s.gx = (wz0 * (wy0 * (v[1] - v[0]) + wy1 * (v[3] - v[2])) + wz1 * (wy0 * (v[5] - v[4]) + wy1 * (v[7] - v[6]))) * inv_h;
        s.gy = (wz0 * (wx0 * (v[2] - v[0]) + wx1 * (v[3] - v[1])) + wz1 * (wx0 * (v[6] - v[4]) + wx1 * (v[7] - v[5]))) * inv_h;
        s.gz = (wy0 * (wx0 * (v[4] - v[0]) + wx1 * (v[5] - v[1])) + wy1 * (wx0 * (v[6] - v[2]) + wx1 * (v[7] - v[3]))) * inv_h;
    } else {
        s.gx = s.gy = s.gz = 0.0f;
    }
    return s;
}

// True when all 8 corners of a face stencil are in range and map to themselves. A periodic
// axis maps its own-axis face n to face 0 (wrap with period n, operators.cu:109-111), so the
// fast path stops one face earlier there.
template <int A>
__device__ __forceinline__ bool face_interior(const Geo& g, const Corner8& c, const VBound& b) {
    const int lx = A == 0 && !vperiodic(b, 0) ? g.nx + 1 : g.nx;
    const int ly = A == 1 && !vperiodic(b, 1) ? g.ny + 1 : g.ny;
    const int lz = A == 2 && !vperiodic(b, 2) ? g.nz + 1 : g.nz;
    return c.x0 >= 0 && c.x0 + 1 < lx && c.y0 >= 0 && c.y0 + 1 < ly && c.z0 >= 0 && c.z0 + 1 < lz;
}

// The 8 corner values of an interior stencil: four loads of two neighbours along x (4-byte aligned)
// from one address per row pair.
struct __attribute__((packed, aligned(4))) Pair {
    float a, b;
};
__device__ __forceinline__ void load8(const float* __restrict__ v, uint32_t base, uint32_t sy, uint32_t sz, float vals[8]) {
    const float* p = v + base;
    const Pair q0 = *reinterpret_cast<const Pair*>(p), q1 = *reinterpret_cast<const Pair*>(p + sy);
    const Pair q2 = *reinterpret_cast<const Pair*>(p + sz), q3 = *reinterpret_cast<const Pair*>(p + (size_t)(sz + sy));
    vals[0] = q0.a;
    vals[1] = q0.b;
    vals[2] = q1.a;
    vals[3] = q1.b;
    vals[4] = q2.a;
    vals[5] = q2.b;
    vals[6] = q3.a;
    vals[7] = q3.b;
}
// The 8 corner values of a stencil that touches a boundary; x decides a corner's fixed value before
// y, y before z.
__device__ __forceinline__ void load8_boundary(const float* __restrict__ v, const AxisStencil& ax, const AxisStencil& ay,
                                               const AxisStencil& az, int ex, int ey, float vals[8]) {
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const int dx = k & 1, dy = (k >> 1) & 1, dz = k >> 2;
        const float l = v[lattice_index(ax.i[dx], ay.i[dy], az.i[dz], ex, ey)];
        vals[k] = ax.fixed[dx] ? ax.value[dx] : ay.fixed[dy] ? ay.value[dy] : az.fixed[dz] ? az.value[dz] : l;
    }
}

// sample_face (operators.cu:166-194) with an interior fast path.
template <int A, bool Grad>
__device__ __forceinline__ Sample sample_face(const float* __restrict__ v, float px, float py, float pz, const Geo& g,
                                              const VBound& b) {
    const Corner8 c = corners(g, px, py, pz, A == 0 ? 0.0f : 0.5f, A == 1 ? 0.0f : 0.5f, A == 2 ? 0.0f : 0.5f);
    const int ex = ext(g, A, 0), ey = ext(g, A, 1);
    float vals[8];
    if (face_interior<A>(g, c, b))
        load8(v, lattice_index(c.x0, c.y0, c.z0, ex, ey), (uint32_t)ex, (uint32_t)ex * (uint32_t)ey, vals);
    else
        load8_boundary(v, face_axis<A, 0>(g, c.x0, b), face_axis<A, 1>(g, c.y0, b), face_axis<A, 2>(g, c.z0, b), ex, ey, vals);
    return trilerp<Grad>(vals, c, g.inv_h);
}

// sample_scalar (operators.cu:136-164) with an interior fast path.
template <bool Grad>
__device__ __forceinline__ Sample sample_scalar(const float* __restrict__ v, float px, float py, float pz, const Geo& g,
                                                const SBound& b) {
    const Corner8 c = corners(g, px, py, pz, 0.5f, 0.5f, 0.5f);
    float vals[8];
    if (c.x0 >= 0 && c.x0 + 1 < g.nx && c.y0 >= 0 && c.y0 + 1 < g.ny && c.z0 >= 0 && c.z0 + 1 < g.nz)
        load8(v, lattice_index(c.x0, c.y0, c.z0, g.nx, g.ny), (uint32_t)g.nx, (uint32_t)g.nx * (uint32_t)g.ny, vals);
    else
        load8_boundary(v, scalar_axis<0>(g, c.x0, b), scalar_axis<1>(g, c.y0, b), scalar_axis<2>(g, c.z0, b), g.nx, g.ny, vals);
    return trilerp<Grad>(vals, c, g.inv_h);
}

// The adds of one trilinear stencil's transpose (operators.cu:196-240) into array W of a sink: the
// corners' weights times adj, on a lattice of extents ex, ey. `interior`: every corner is a stored
// point (at c.x0 .. c.x0 + 1 and so on); else the axes' stencils give the points and the skipped
// corners. A sink may take a whole interior stencil at once (Sink::window8: true when all eight
// points lie in its window); it is not offered non-finite adjoints, whose product with a zero weight
// would not be 0.
template <int W, typename Sink, typename Axes>
__device__ __forceinline__ void scatter8(const Sink& sink, const Corner8& c, float adj, int ex, int ey, bool interior, Axes&& axes) {
    const float w[2][3] = {{1.0f - c.tx, 1.0f - c.ty, 1.0f - c.tz}, {c.tx, c.ty, c.tz}};
    float a[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) a[k] = w[k & 1][0] * w[(k >> 1) & 1][1] * w[k >> 2][2];
    if (interior && fabsf(adj) < __builtin_inff() && sink.template window8<W>(c.x0, c.y0, c.z0, adj, a)) return;
    AxisStencil ax, ay, az;
    axes(ax, ay, az);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const int dx = k & 1, dy = (k >> 1) & 1, dz = k >> 2;
        if (ax.fixed[dx] || ay.fixed[dy] || az.fixed[dz] || a[k] == 0.0f) continue;
        const int x = ax.i[dx], y = ay.i[dy], z = az.i[dz];
        sink.template add<W>(x, y, z, lattice_index(x, y, z, ex, ey), adj * a[k]);
    }
}

// scatter_face (operators.cu:217-240): transpose of sample_face's value.
template <int A, typename Sink>
__device__ __forceinline__ void scatter_face_to(const Sink& sink, float px, float py, float pz, float adj, const Geo& g, const VBound& b) {
    if (adj == 0.0f) return;
    const Corner8 c = corners(g, px, py, pz, A == 0 ? 0.0f : 0.5f, A == 1 ? 0.0f : 0.5f, A == 2 ? 0.0f : 0.5f);
    scatter8<A>(sink, c, adj, ext(g, A, 0), ext(g, A, 1), face_interior<A>(g, c, b), [&](AxisStencil& ax, AxisStencil& ay, AxisStencil& az) {
        ax = face_axis<A, 0>(g, c.x0, b);
        ay = face_axis<A, 1>(g, c.y0, b);
        az = face_axis<A, 2>(g, c.z0, b);
    });
}

// scatter_scalar (operators.cu:196-215): transpose of sample_scalar's value, into the sink's array W.
template <int W, typename Sink>
__device__ __forceinline__ void scatter_scalar_to(const Sink& sink, float px, float py, float pz, float adj, const Geo& g,
                                                  const SBound& b) {
    if (adj == 0.0f) return;
    const Corner8 c = corners(g, px, py, pz, 0.5f, 0.5f, 0.5f);
    const bool interior = c.x0 >= 0 && c.x0 + 1 < g.nx && c.y0 >= 0 && c.y0 + 1 < g.ny && c.z0 >= 0 && c.z0 + 1 < g.nz;
    scatter8<W>(sink, c, adj, g.nx, g.ny, interior, [&](AxisStencil& ax, AxisStencil& ay, AxisStencil& az) {
        ax = scalar_axis<0>(g, c.x0, b);
        ay = scalar_axis<1>(g, c.y0, b);
        az = scalar_axis<2>(g, c.z0, b);
    });
}

struct Vel3 {
    const float* __restrict__ u[3];
};

// solid_at, operators.cu:246-254 (mask: u8 per cell, 1 = solid).
__device__ __forceinline__ bool solid_at(float px, float py, float pz, const uint8_t* __restrict__ mask, const Geo& g,
                                         const VBound& b) {
    if (vperiodic(b, 0)) { const float L = g.nx * g.h; px -= floorf(px / L) * L; }
    if (vperiodic(b, 1)) { const float L = g.ny * g.h; py -= floorf(py / L) * L; }
    if (vperiodic(b, 2)) { const float L = g.nz * g.h; pz -= floorf(pz / L) * L; }
    // clamped as floats, so a non-finite position maps to a cell of the domain (NaN to 0)
    const int x = (int)fminf(fmaxf(floorf(over_h(g, px)), 0.0f), (float)(g.nx - 1));
    const int y = (int)fminf(fmaxf(floorf(over_h(g, py)), 0.0f), (float)(g.ny - 1));
    const int z = (int)fminf(fmaxf(floorf(over_h(g, pz)), 0.0f), (float)(g.nz - 1));
    return mask[cidx(g, x, y, z)] != 0;
}

struct TraceOut {
    float px, py, pz;   // end point
    float dx, dy, dz;   // derivative scale per axis (0 when clamped, bisection fraction when bisected)
    float mx, my, mz;   // midpoint
};

// Component B of the velocity at a lattice point: face (x, y, z) of axis L, or the centre of cell
// (x, y, z) for L = 3. The trilinear stencil is fixed there: along an axis where the two lattices
// agree one point (weight 1), else the two around it (1/2 each); so 1, 2 or 4 loads instead of 8.
// Order of the sums: x inside y inside z, as trilerp.
template <int L, int B>
struct StartStencil {
    // axis d of B's stencil has two points when exactly one of L and B is staggered along d
    static constexpr bool two(int d) { return (L == d) != (B == d); }
    // lower point's offset: a face of axis L sits between cells c - 1 and c, a cell between faces c and c + 1
    static constexpr int lower(int d) { return L == d && B != d ? -1 : 0; }
};
template <int L, int B, int D>
__device__ __forceinline__ AxisStencil start_axis(const Geo& g, int c, const VBound& b) {
    return face_axis<B, D>(g, c + StartStencil<L, B>::lower(D), b);
}
template <int L, int B>
__device__ __forceinline__ float start_velocity(const float* __restrict__ v, int x, int y, int z, const Geo& g, const VBound& b) {
    using S = StartStencil<L, B>;
    const AxisStencil ax = start_axis<L, B, 0>(g, x, b), ay = start_axis<L, B, 1>(g, y, b), az = start_axis<L, B, 2>(g, z, b);
    const int ex = ext(g, B, 0), ey = ext(g, B, 1);
    float sz[2];
#pragma unroll
    for (int dz = 0; dz <= (S::two(2) ? 1 : 0); ++dz) {
        float sy[2];
#pragma unroll
        for (int dy = 0; dy <= (S::two(1) ? 1 : 0); ++dy) {
            float sx[2];
#pragma unroll
            for (int dx = 0; dx <= (S::two(0) ? 1 : 0); ++dx) {
                const float l = v[lattice_index(ax.i[dx], ay.i[dy], az.i[dz], ex, ey)];
                sx[dx] = ax.fixed[dx] ? ax.value[dx] : ay.fixed[dy] ? ay.value[dy] : az.fixed[dz] ? az.value[dz] : l;
            }
            sy[dy] = S::two(0) ? 0.5f * sx[0] + 0.5f * sx[1] : sx[0];
        }
        sz[dz] = S::two(1) ? 0.5f * sy[0] + 0.5f * sy[1] : sy[0];
    }
    return S::two(2) ? 0.5f * sz[0] + 0.5f * sz[1] : sz[0];
}
// Transpose of start_velocity into array B of a sink.
template <int L, int B, typename Sink>
__device__ __forceinline__ void scatter_start(const Sink& sink, int x, int y, int z, float adj, const Geo& g, const VBound& b) {
    if (adj == 0.0f) return;
    using S = StartStencil<L, B>;
    const AxisStencil ax = start_axis<L, B, 0>(g, x, b), ay = start_axis<L, B, 1>(g, y, b), az = start_axis<L, B, 2>(g, z, b);
    const float a = adj * ((S::two(0) ? 0.5f : 1.0f) * (S::two(1) ? 0.5f : 1.0f) * (S::two(2) ? 0.5f : 1.0f));
#pragma unroll
    for (int dz = 0; dz <= (S::two(2) ? 1 : 0); ++dz)
#pragma unroll
        for (int dy = 0; dy <= (S::two(1) ? 1 : 0); ++dy)
#pragma unroll
            for (int dx = 0; dx <= (S::two(0) ? 1 : 0); ++dx) {
                if (ax.fixed[dx] || ay.fixed[dy] || az.fixed[dz]) continue;
                const int px = ax.i[dx], py = ay.i[dy], pz = az.i[dz];
                sink.template add<B>(px, py, pz, lattice_index(px, py, pz, ext(g, B, 0), ext(g, B, 1)), a);
            }
}

// Position of a lattice point (a face of axis L, or a cell centre for L = 3).
struct Pos {
    float x, y, z;
};
template <int L>
__device__ __forceinline__ Pos start_position(const Geo& g, int x, int y, int z) {
    return Pos{(x + (L == 0 ? 0.0f : 0.5f)) * g.h, (y + (L == 1 ? 0.0f : 0.5f)) * g.h, (z + (L == 2 ? 0.0f : 0.5f)) * g.h};
}

// trace_rk2, operators.cu:256-276, from face (x, y, z) of axis L (a cell centre for L = 3).
// has_solids = false skips the mask lookup (no colliders).
// MidGrad: also return the three velocity samples at the midpoint with their gradients in mid
// (the reverse and tangent sweeps need them; the values are the ones the trace uses).
template <int L, bool HasSolids, bool MidGrad = false>
__device__ __forceinline__ TraceOut trace_rk2(int x, int y, int z, const Vel3& u, const uint8_t* __restrict__ mask,
                                              const Geo& g, const VBound& b, Sample* mid = nullptr) {
    TraceOut t;
    const Pos start = start_position<L>(g, x, y, z);
    const float sx = start.x, sy = start.y, sz = start.z;
    const float v0x = start_velocity<L, 0>(u.u[0], x, y, z, g, b);
    const float v0y = start_velocity<L, 1>(u.u[1], x, y, z, g, b);
    const float v0z = start_velocity<L, 2>(u.u[2], x, y, z, g, b);
    t.mx = sx - 0.5f * g.dt * v0x;
    t.my = sy - 0.5f * g.dt * v0y;
    t.mz = sz - 0.5f * g.dt * v0z;
    const Sample m0 = sample_face<0, MidGrad>(u.u[0], t.mx, t.my, t.mz, g, b);
    const Sample m1 = sample_face<1, MidGrad>(u.u[1], t.mx, t.my, t.mz, g, b);
    const Sample m2 = sample_face<2, MidGrad>(u.u[2], t.mx, t.my, t.mz, g, b);
    if (MidGrad) {
        mid[0] = m0;
        mid[1] = m1;
        mid[2] = m2;
    }
    const float v1x = m0.value, v1y = m1.value, v1z = m2.value;
    float rx = sx - g.dt * v1x, ry = sy - g.dt * v1y, rz = sz - g.dt * v1z;
    t.dx = t.dy = t.dz = 1.0f;
    const float Lx = g.nx * g.h, Ly = g.ny * g.h, Lz = g.nz * g.h;
    if (!vperiodic(b, 0) && (rx < 0.0f || rx > Lx)) { rx = fminf(fmaxf(rx, 0.0f), Lx); t.dx = 0.0f; }
    if (!vperiodic(b, 1) && (ry < 0.0f || ry > Ly)) { ry = fminf(fmaxf(ry, 0.0f), Ly); t.dy = 0.0f; }
    if (!vperiodic(b, 2) && (rz < 0.0f || rz > Lz)) { rz = fminf(fmaxf(rz, 0.0f), Lz); t.dz = 0.0f; }
    if (HasSolids && solid_at(rx, ry, rz, mask, g, b)) {
        float lo = 0.0f, hi = 1.0f;
        for (int it = 0; it < 8; ++it) {
            const float f = 0.5f * (lo + hi);
            if (solid_at(sx + f * (rx - sx), sy + f * (ry - sy), sz + f * (rz - sz), mask, g, b)) hi = f;
            else lo = f;
        }
        rx = sx + lo * (rx - sx);
        ry = sy + lo * (ry - sy);
        rz = sz + lo * (rz - sz);
        t.dx *= lo;
        t.dy *= lo;
        t.dz *= lo;
    }
    t.px = rx;
    t.py = ry;
    t.pz = rz;
    return t;
}

// ---- reductions: FP64 sums over a block of up to 1024 threads (wave64 shuffles, then LDS) ---
constexpr int kMaxWaves = 16;

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// Sums N values per thread over the block; every thread receives the totals in a fixed order.
// lds: N * kMaxWaves doubles.
template <int N>
__device__ __forceinline__ void block_sum(double (&v)[N], double* lds) {
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int waves = (int)(blockDim.x >> 6);
#pragma unroll
    for (int k = 0; k < N; ++k) v[k] = wave_sum(v[k]);
    __syncthreads();   // lds may still be read by a previous call
    if (lane == 0)
#pragma unroll
        for (int k = 0; k < N; ++k) lds[k * kMaxWaves + wid] = v[k];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < N; ++k) {
        double s = 0.0;
        for (int w = 0; w < waves; ++w) s += lds[k * kMaxWaves + w];
        v[k] = s;
    }
}

// Deterministic sum of `count` partials (same order in every block): returns the total to all
// threads. Used by a consumer kernel to finish the reduction its producer left per block.
template <int N>
__device__ __forceinline__ void reduce_partials(const double* const (&parts)[N], uint32_t count, double (&out)[N], double* lds) {
    double v[N];
#pragma unroll
    for (int k = 0; k < N; ++k) v[k] = 0.0;
    for (uint32_t i = threadIdx.x; i < count; i += blockDim.x)
#pragma unroll
        for (int k = 0; k < N; ++k) v[k] += parts[k][i];
    block_sum<N>(v, lds);
#pragma unroll
    for (int k = 0; k < N; ++k) out[k] = v[k];
}

}  // namespace ds
