// adjoint.hip — reverse (VJP) operators of the smoke step on gfx950 (solvers/smoke/operators.cu:
// 297-302, 326-337, 366-379, 415-439, 483-497, 537-561, 922-969).
//
// Adjoint fields are FP32. Scatters that follow a data-dependent trace (the transposes of the
// trilinear samples) use hardware FP32 atomics; every transpose with a fixed stencil is
// rewritten as a gather so that it needs no atomics: the projection reverse (p_bar per cell),
// the divergence reverse and the constraint transpose (one face kernel), and the integration
// reverse (force adjoint per cell, fused with the buoyancy and source reverses). Parameter
// adjoints are FP64 block partials reduced in a fixed order.
#include <hip/hip_runtime.h>

#include <cmath>

#include "context.hpp"
#include "kernels.hpp"
#include "vorticity.hpp"

namespace ds {

namespace {

// Adds of a whole interior stencil into an LDS window of X x Y x Z doubles when its 8 points lie in
// it, its lower corner at window coordinates (lx, ly, lz): one address, constant offsets.
template <int X, int Y, int Z>
__device__ __forceinline__ bool window_add8(double* win, int lx, int ly, int lz, float adj, const float (&a)[8]) {
    if ((unsigned)lx >= (unsigned)(X - 1) || (unsigned)ly >= (unsigned)(Y - 1) || (unsigned)lz >= (unsigned)(Z - 1)) return false;
    double* p = win + (lz * Y + ly) * X + lx;
#pragma unroll
    for (int k = 0; k < 8; ++k)
        __hip_atomic_fetch_add(p + ((k >> 2) * Y + ((k >> 1) & 1)) * X + (k & 1), (double)(adj * a[k]), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_WORKGROUP);
    return true;
}

// Reverse of trace_rk2 + final sample (operators.cu:422-438 / 544-560) from lattice point (x, y, z)
// of L: given the adjoint of the trace end point (v1x, v1y, v1z) = -deriv * dt * grad(sample) *
// out_adj, scatter through the midpoint and start samples of the velocity; mid: the velocity samples
// at the midpoint with their gradients (from trace_rk2<.., true>).
template <int L, typename Sink>
__device__ __forceinline__ void trace_reverse(const Geo& g, const VBound& b, const Sink& sink, int x, int y, int z, const TraceOut& t,
                                              const Sample (&mid)[3], float v1x, float v1y, float v1z) {
    const Sample& m0 = mid[0];
    const Sample& m1 = mid[1];
    const Sample& m2 = mid[2];
    scatter_face_to<0>(sink, t.mx, t.my, t.mz, v1x, g, b);
    scatter_face_to<1>(sink, t.mx, t.my, t.mz, v1y, g, b);
    scatter_face_to<2>(sink, t.mx, t.my, t.mz, v1z, g, b);
    const float mx = m0.gx * v1x + m1.gx * v1y + m2.gx * v1z;
    const float my = m0.gy * v1x + m1.gy * v1y + m2.gy * v1z;
    const float mz = m0.gz * v1x + m1.gz * v1y + m2.gz * v1z;
    const float s = -0.5f * g.dt;
    scatter_start<L, 0>(sink, x, y, z, s * mx, g, b);
    scatter_start<L, 1>(sink, x, y, z, s * my, g, b);
    scatter_start<L, 2>(sink, x, y, z, s * mz, g, b);
}

constexpr int kVjpThreads = 512;   // of both advection reverses

// advect_scalar_vjp_kernel (operators.cu:537-561) for NF fields that share one trace: the
// velocity adjoint of both fields is summed before it is scattered (the map is linear). A block
// owns a kSvBX x kSvBY x kSvBZ brick of cells and privatises its scatters as the velocity reverse
// does: the NF fields' and the three velocity components' adds that land in a window around the
// brick (halo kSvHalo) are LDS atomics, the rest (long traces, periodic wraps) global atomics; the
// windows are flushed once. The windows hold FP64: see kVjpThreads.
constexpr int kSvBX = 32, kSvBY = 8, kSvBZ = 2, kSvHalo = 1;
constexpr int kSwX = kSvBX + 2 * kSvHalo + 1, kSwY = kSvBY + 2 * kSvHalo + 1, kSwZ = kSvBZ + 2 * kSvHalo + 1;
constexpr int kSw = kSwX * kSwY * kSwZ;   // per target array: velocity components 0-2, fields 3-4

struct ScalarBrickSink {
    double* win;       // LDS, 5 * kSw
    int ox, oy, oz;    // coordinates of window element (0, 0, 0)
    F3 va;
    float* s0;
    float* s1;
    template <int W>
    __device__ __forceinline__ void add(int x, int y, int z, uint32_t i, float value) const {
        const unsigned lx = (unsigned)(x - ox), ly = (unsigned)(y - oy), lz = (unsigned)(z - oz);
        if (lx < (unsigned)kSwX && ly < (unsigned)kSwY && lz < (unsigned)kSwZ)
            __hip_atomic_fetch_add(win + W * kSw + ((int)lz * kSwY + (int)ly) * kSwX + (int)lx, (double)value, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_WORKGROUP);
        else
            atomicAdd((W < 3 ? va.p[W < 3 ? W : 0] : W == 3 ? s0 : s1) + i, value);
    }
    template <int W>
    __device__ __forceinline__ bool window8(int x, int y, int z, float adj, const float (&a)[8]) const {
        return window_add8<kSwX, kSwY, kSwZ>(win + W * kSw, x - ox, y - oy, z - oz, adj, a);
    }
};

// One cell per thread; 4 waves per SIMD (registers capped at 128, the rest spilled), the most two
// blocks' 77 KB of LDS allow: the dependent gathers of the trace want waves more than registers.
template <int NF, bool HasSolids>
__global__ __launch_bounds__(kVjpThreads) __attribute__((amdgpu_waves_per_eu(4))) void advect_scalar_vjp_kernel(Geo g, const VBound* __restrict__ vbp, const SBound* __restrict__ sb0p,
                                                                const SBound* __restrict__ sb1p, const uint8_t* __restrict__ mask,
                                                                const float* __restrict__ src0, const float* __restrict__ src1, Vel3 u,
                                                                const float* __restrict__ oa0, const float* __restrict__ oa1,
                                                                float* src_adj0, float* src_adj1, F3 va) {
    static_assert(kSvBX * kSvBY * kSvBZ == kVjpThreads, "one cell of the brick per thread");
    __shared__ double win[5 * kSw];
    const VBound& vb = *vbp;
    const SBound& sb0 = *sb0p;
    const SBound& sb1 = *sb1p;
    const uint32_t nbx = (uint32_t)(g.nx + kSvBX - 1) / kSvBX, nby = (uint32_t)(g.ny + kSvBY - 1) / kSvBY;
    const uint32_t bricks = nbx * nby * (uint32_t)((g.nz + kSvBZ - 1) / kSvBZ);
    const uint32_t lb = xcd_block();
    if (lb >= bricks) return;   // padding blocks of the XCD-rounded grid (whole block)
    const int x0 = (int)(lb % nbx) * kSvBX, y0 = (int)((lb / nbx) % nby) * kSvBY, z0 = (int)(lb / (nbx * nby)) * kSvBZ;
    for (int k = threadIdx.x; k < 5 * kSw; k += blockDim.x) win[k] = 0.0;
    __syncthreads();
    const ScalarBrickSink sink{win, x0 - kSvHalo, y0 - kSvHalo, z0 - kSvHalo, va, src_adj0, NF == 2 ? src_adj1 : src_adj0};
    const int x = x0 + (int)(threadIdx.x % kSvBX), y = y0 + (int)(threadIdx.x / kSvBX) % kSvBY,
              z = z0 + (int)threadIdx.x / (kSvBX * kSvBY);
    auto cell = [&] {
        if (x >= g.nx || y >= g.ny || z >= g.nz) return;
        const uint32_t i = cidx(g, x, y, z);
        if (HasSolids && mask[i] != 0) return;
        const float a0 = oa0[i];
        const float a1 = NF == 2 ? oa1[i] : 0.0f;
        if (a0 == 0.0f && a1 == 0.0f) return;
        Sample mid[3];
        const TraceOut t = trace_rk2<3, HasSolids, true>(x, y, z, u, mask, g, vb, mid);
        const Sample s0 = sample_scalar<true>(src0, t.px, t.py, t.pz, g, sb0);
        scatter_scalar_to<3>(sink, t.px, t.py, t.pz, a0, g, sb0);
        float gx = s0.gx * a0, gy = s0.gy * a0, gz = s0.gz * a0;
        if (NF == 2) {
            const Sample s1 = sample_scalar<true>(src1, t.px, t.py, t.pz, g, sb1);
            scatter_scalar_to<4>(sink, t.px, t.py, t.pz, a1, g, sb1);
            gx += s1.gx * a1;
            gy += s1.gy * a1;
            gz += s1.gz * a1;
        }
        const float v1x = -(t.dx * g.dt) * gx, v1y = -(t.dy * g.dt) * gy, v1z = -(t.dz * g.dt) * gz;
        trace_reverse<3>(g, vb, sink, x, y, z, t, mid, v1x, v1y, v1z);
    };
    cell();
    __syncthreads();
    for (int k = threadIdx.x; k < 5 * kSw; k += blockDim.x) {
        const float v = (float)win[k];
        if (v == 0.0f) continue;
        const int W = k / kSw, r = k - W * kSw;
        const int wx = x0 - kSvHalo + r % kSwX, wy = y0 - kSvHalo + (r / kSwX) % kSwY, wz = z0 - kSvHalo + r / (kSwX * kSwY);
        // only in-range targets receive window adds; the test keeps the flush in bounds regardless
        if (W < 3) {
            if (wx < 0 || wy < 0 || wz < 0 || wx >= ext(g, W, 0) || wy >= ext(g, W, 1) || wz >= ext(g, W, 2)) continue;
            float* dst = W == 0 ? va.p[0] : W == 1 ? va.p[1] : va.p[2];
            atomicAdd(dst + fidx(g, W, wx, wy, wz), v);
        } else {
            if (wx < 0 || wy < 0 || wz < 0 || wx >= g.nx || wy >= g.ny || wz >= g.nz) continue;
            atomicAdd((W == 3 ? src_adj0 : src_adj1) + cidx(g, wx, wy, wz), v);
        }
    }
}

// advect_velocity_vjp_kernel (operators.cu:415-439) for the faces of axis A, with its scatters
// privatised per block: a block owns a kVjpBX x kVjpBY x kVjpBZ brick of A-faces, whose traces
// move a few cells at most, so their 56 scatters per face land in a small box around the brick.
// Scatters inside the box (brick plus a halo of kVjpHalo faces, each component) are LDS atomics;
// those outside it (long traces, periodic wraps) stay global atomics. The box is flushed once.
//
// The windows hold FP64. An LDS FP32 add serialises its lanes (193 cycles per wave and CU, measured
// with conflict-free addresses; the integer add takes 5.5, the FP64 add 9.3), and these scatters
// bound both reverse kernels: with FP64 windows the velocity reverse of one axis went from 455 to
// 230-310 us and the scalar reverse from 685 to 448 us at 128^3, with sums that no longer round
// per add. The windows are twice as large, so blocks of 512 threads (not 256) share one: two blocks
// and 4 waves per SIMD per CU, as with FP32.
constexpr int kVjpBX = 32, kVjpBY = 8, kVjpBZ = 4, kVjpHalo = 1;
constexpr int kVjpPlanes = kVjpThreads / (kVjpBX * kVjpBY);   // brick planes handled at once
constexpr int kWinX = kVjpBX + 2 * kVjpHalo + 1, kWinY = kVjpBY + 2 * kVjpHalo + 1, kWinZ = kVjpBZ + 2 * kVjpHalo + 1;
constexpr int kWin = kWinX * kWinY * kWinZ;   // per component

struct WindowSink {
    double* win;       // LDS, 3 * kWin
    int ox, oy, oz;    // face coordinates of window element (0, 0, 0)
    F3 va;
    template <int B>
    __device__ __forceinline__ void add(int x, int y, int z, uint32_t i, float value) const {
        const unsigned lx = (unsigned)(x - ox), ly = (unsigned)(y - oy), lz = (unsigned)(z - oz);
        // workgroup scope for the LDS add: it keeps the two atomics distinct (merged into one
        // atomic on a selected pointer they would both become flat atomics)
        if (lx < (unsigned)kWinX && ly < (unsigned)kWinY && lz < (unsigned)kWinZ)
            __hip_atomic_fetch_add(win + B * kWin + ((int)lz * kWinY + (int)ly) * kWinX + (int)lx, (double)value, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_WORKGROUP);
        else
            atomicAdd(va.p[B] + i, value);
    }
    template <int B>
    __device__ __forceinline__ bool window8(int x, int y, int z, float adj, const float (&a)[8]) const {
        return window_add8<kWinX, kWinY, kWinZ>(win + B * kWin, x - ox, y - oy, z - oz, adj, a);
    }
};

__device__ __forceinline__ uint32_t vjp_bricks(const Geo& g, int A, int& nbx, int& nby) {
    nbx = (ext(g, A, 0) + kVjpBX - 1) / kVjpBX;
    nby = (ext(g, A, 1) + kVjpBY - 1) / kVjpBY;
    return (uint32_t)nbx * nby * ((ext(g, A, 2) + kVjpBZ - 1) / kVjpBZ);
}

// 4 waves per SIMD (registers capped at 128, the rest spilled), the most two blocks' 65 KB windows allow.
template <int A, bool HasSolids>
__global__ __launch_bounds__(kVjpThreads) __attribute__((amdgpu_waves_per_eu(4))) void advect_velocity_vjp_kernel(Geo g, const VBound* __restrict__ bp, const uint8_t* __restrict__ mask,
                                                                  Vel3 u, const float* __restrict__ oa, F3 va) {
    __shared__ double win[3 * kWin];
    const VBound& b = *bp;
    int nbx, nby;
    const uint32_t bricks = vjp_bricks(g, A, nbx, nby);
    const uint32_t lb = xcd_block();
    if (lb >= bricks) return;   // padding blocks of the XCD-rounded grid (whole block)
    const int x0 = (int)(lb % (uint32_t)nbx) * kVjpBX;
    const int y0 = (int)((lb / (uint32_t)nbx) % (uint32_t)nby) * kVjpBY;
    const int z0 = (int)(lb / ((uint32_t)nbx * nby)) * kVjpBZ;
    for (int i = threadIdx.x; i < 3 * kWin; i += blockDim.x) win[i] = 0.0;
    __syncthreads();
    const WindowSink sink{win, x0 - kVjpHalo, y0 - kVjpHalo, z0 - kVjpHalo, va};
    const int ex = ext(g, A, 0), ey = ext(g, A, 1), ez = ext(g, A, 2);
    const int x = x0 + (int)(threadIdx.x % kVjpBX), y = y0 + (int)(threadIdx.x / kVjpBX) % kVjpBY;
    for (int f = (int)threadIdx.x / (kVjpBX * kVjpBY); f < kVjpBZ; f += kVjpPlanes) {
        const int z = z0 + f;
        if (x >= ex || y >= ey || z >= ez) continue;
        const uint32_t fi = fidx(g, A, x, y, z);
        const float a = oa[fi];
        if (a == 0.0f) continue;
        Sample mid[3];
        const TraceOut t = trace_rk2<A, HasSolids, true>(x, y, z, u, mask, g, b, mid);
        const Sample s = sample_face<A, true>(u.u[A], t.px, t.py, t.pz, g, b);
        scatter_face_to<A>(sink, t.px, t.py, t.pz, a, g, b);
        trace_reverse<A>(g, b, sink, x, y, z, t, mid, -(t.dx * g.dt) * (s.gx * a), -(t.dy * g.dt) * (s.gy * a), -(t.dz * g.dt) * (s.gz * a));
    }
    __syncthreads();
    for (int i = threadIdx.x; i < 3 * kWin; i += blockDim.x) {
        const float v = (float)win[i];
        if (v == 0.0f) continue;
        const int B = i / kWin, r = i - B * kWin;
        const int wx = x0 - kVjpHalo + r % kWinX, wy = y0 - kVjpHalo + (r / kWinX) % kWinY, wz = z0 - kVjpHalo + r / (kWinX * kWinY);
        // only in-range faces receive window adds; the test keeps the flush in bounds regardless
        if (wx < 0 || wy < 0 || wz < 0 || wx >= ext(g, B, 0) || wy >= ext(g, B, 1) || wz >= ext(g, B, 2)) continue;
        float* dst = B == 0 ? va.p[0] : B == 1 ? va.p[1] : va.p[2];
        atomicAdd(dst + fidx(g, B, wx, wy, wz), v);
    }
}

// constrained_boundary, operators.cu:452-458
template <int A>
__device__ __forceinline__ bool constrained_boundary(const Geo& g, const VBound& b, int coord) {
    const int n_a = dim_size(g, A);
    if (coord != 0 && coord != n_a) return false;
    const uint32_t mode = coord == n_a ? b.modes[2 * A + 1] : b.modes[2 * A];
    return mode == 0u || mode == 2u;
}

// Adjoint of the advected velocity at one face from the projected-velocity adjoint and lambda
// (projection reverse + pressure_rhs_reverse as a gather, operators.cu:922-933,957-969):
//   adj = u_bar(f) - (h/dt) * (lambda(c0) - lambda(c1)), lambda = 0 off the unknowns.
struct ProjAdjIn {
    const float* ua[3];
    const float* extra[3];
    const float* lh;
    const float* ll;
};

template <int A>
__device__ __forceinline__ float projected_face_adjoint(const Geo& g, const ProjAdjIn& in, int x, int y, int z, uint32_t local) {
    float a = in.ua[A][local];
    if (in.extra[A]) a += in.extra[A][local];
    const int coord = A == 0 ? x : A == 1 ? y : z;
    const int n_a = dim_size(g, A);
    float l0 = 0.0f, l1 = 0.0f;
    if (coord > 0) {
        const uint32_t c0 = cidx(g, x - (A == 0), y - (A == 1), z - (A == 2));
        l0 = in.lh[c0] + in.ll[c0];
    }
    if (coord < n_a) {
        const uint32_t c1 = cidx(g, x, y, z);
        l1 = in.lh[c1] + in.ll[c1];
    }
    return a - g.h * (l0 - l1) / g.dt;
}

// Projection reverse with the constraint transpose fused (constrain_velocity_vjp_kernel,
// operators.cu:483-497, as a gather): constrained, solid-adjacent and periodic-duplicate faces
// receive 0; face 0 of a periodic axis also receives its duplicate's adjoint.
// Constrain = false: out += projected adjoint (the per-operator projection VJP).
template <bool Constrain>
__global__ __launch_bounds__(256) void projection_vjp_face_kernel(Geo g, const VBound* __restrict__ bp, const uint8_t* __restrict__ mask,
                                                                  uint32_t has_solids, ProjAdjIn in, F3 out) {
    const VBound& b = *bp;
    const uint32_t fi = xcd_block() * blockDim.x + threadIdx.x;
    if (fi >= g.foff[3]) return;
    for_face(g, fi, [&]<int A>(uint32_t local) {
        int x, y, z;
        decode_face_axis<A>(g, local, x, y, z);
        if (!Constrain) {
            out.p[A][local] += projected_face_adjoint<A>(g, in, x, y, z, local);
            return;
        }
        const int coord = A == 0 ? x : A == 1 ? y : z;
        const int n_a = dim_size(g, A);
        const bool per = vperiodic(b, A);
        float a = 0.0f;
        if (!(constrained_boundary<A>(g, b, coord) || (has_solids && adjacent_solid<A>(g, mask, x, y, z)) || (per && coord == n_a)))
            a = projected_face_adjoint<A>(g, in, x, y, z, local);
        if (per && coord == 0) {   // (also where a solid beyond this face, but not beyond its duplicate, constrains it)
            const int dx = A == 0 ? n_a : x, dy = A == 1 ? n_a : y, dz = A == 2 ? n_a : z;
            if (!(has_solids && adjacent_solid<A>(g, mask, dx, dy, dz)))
                a += projected_face_adjoint<A>(g, in, dx, dy, dz, fidx(g, A, dx, dy, dz));
        }
        out.p[A][local] = a;
    });
}

// constrain_velocity_vjp_kernel (operators.cu:483-497) as a gather: out += C^T in.
__global__ __launch_bounds__(256) void constrain_vjp_kernel(Geo g, const VBound* __restrict__ bp, const uint8_t* __restrict__ mask,
                                                            uint32_t has_solids, CF3 in, F3 out) {
    const VBound& b = *bp;
    const uint32_t fi = xcd_block() * blockDim.x + threadIdx.x;
    if (fi >= g.foff[3]) return;
    for_face(g, fi, [&]<int A>(uint32_t local) {
        int x, y, z;
        decode_face_axis<A>(g, local, x, y, z);
        const int coord = A == 0 ? x : A == 1 ? y : z;
        const int n_a = dim_size(g, A);
        const bool per = vperiodic(b, A);
        float a = 0.0f;
        if (!(constrained_boundary<A>(g, b, coord) || (has_solids && adjacent_solid<A>(g, mask, x, y, z)) || (per && coord == n_a)))
            a = in.p[A][local];
        if (per && coord == 0) {
            const int dx = A == 0 ? n_a : x, dy = A == 1 ? n_a : y, dz = A == 2 ? n_a : z;
            if (!(has_solids && adjacent_solid<A>(g, mask, dx, dy, dz))) a += in.p[A][fidx(g, A, dx, dy, dz)];
        }
        out.p[A][local] += a;
    });
}

// out += in over the concatenated faces (the velocity pass-through of integrate_vjp_kernel,
// operators.cu:370, and accumulate_kernel, operators.cu:292-295).
__global__ __launch_bounds__(256) void face_accumulate_kernel(Geo g, CF3 in, F3 out) {
    const uint32_t fi = xcd_block() * blockDim.x + threadIdx.x;
    if (fi >= g.foff[3]) return;
    for_face(g, fi, [&]<int A>(uint32_t local) { out.p[A][local] += in.p[A][local]; });
}

__global__ __launch_bounds__(256) void cell_accumulate_kernel(uint32_t n, const float* __restrict__ in, float* __restrict__ out) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] += in[i];
}

// Integration reverse (force part), buoyancy reverse (operators.cu:326-337) and source reverse
// (operators.cu:297-302) fused per fluid cell. Parameter adjoints: FP64 block partials.
// Vort: the confinement force reverse runs on the same force adjoint (vorticity_force_reverse +
// the per-cell part of normal_reverse, operators.cu:781-812), writing vort.ga / vort.t (zeros in
// solids) and the confinement adjoint as partial set 3; the vorticity fields in vort.in come
// from the curl pass over the step's input velocity.
struct VortReverse {
    VortFields in;
    F3 ga, t;
};

template <bool Vort>
__global__ __launch_bounds__(256) void force_source_vjp_kernel(Geo g, const uint8_t* __restrict__ mask, CF3 forced_adj,
                                                               const float* __restrict__ rho_s, const float* __restrict__ t_s,
                                                               const float* __restrict__ rho_s_adj, const float* __restrict__ t_s_adj,
                                                               Params prm, F3 e_adj, float* __restrict__ prev_rho,
                                                               float* __restrict__ prev_t, float* __restrict__ s_rho_adj,
                                                               float* __restrict__ s_t_adj, VortReverse vort, double* __restrict__ partials) {
    constexpr int kParts = Vort ? 4 : 3;
    __shared__ double lds[kParts * kMaxWaves];
    const uint32_t lb = xcd_block();
    uint32_t chunk = (g.n + gridDim.x - 1) / gridDim.x;
    chunk = (chunk + 255u) & ~255u;
    const uint32_t start = min(g.n, lb * chunk), end = min(g.n, start + chunk);
    const float amb = *prm.ambient, ar = *prm.alpha_rho, at = *prm.alpha_t;
    const float scale = Vort ? *prm.confinement * g.h : 0.0f;
    double p_amb = 0.0, p_ar = 0.0, p_at = 0.0, p_conf = 0.0;
    for (uint32_t i = start + threadIdx.x; i < end; i += blockDim.x) {
        if (mask[i] != 0) {
            if constexpr (Vort) {
#pragma unroll
                for (int a = 0; a < 3; ++a) vort.ga.p[a][i] = vort.t.p[a][i] = 0.0f;
            }
            continue;
        }
        int x, y, z;
        decode_cell(g, i, x, y, z);
        float f[3];
        force_gather(g, mask, forced_adj, i, x, y, z, f);
        if constexpr (Vort) {
            float ga[3], t[3];
            p_conf += confinement_reverse_at(g, vort.in, i, x, y, z, scale, f, ga, t);
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                vort.ga.p[a][i] = ga[a];
                vort.t.p[a][i] = t[a];
            }
        }
        if (e_adj.p[0]) {
            e_adj.p[0][i] += f[0];
            e_adj.p[1][i] += f[1];
            e_adj.p[2][i] += f[2];
        }
        const float rsa = (rho_s_adj ? rho_s_adj[i] : 0.0f) + ar * f[1];
        const float tsa = (t_s_adj ? t_s_adj[i] : 0.0f) + at * f[1];
        p_amb += -(double)at * f[1];
        p_ar += (double)rho_s[i] * f[1];
        p_at += (double)(t_s[i] - amb) * f[1];
        prev_rho[i] += rsa;
        prev_t[i] += tsa;
        if (s_rho_adj) s_rho_adj[i] += g.dt * rsa;
        if (s_t_adj) s_t_adj[i] += g.dt * tsa;
    }
    double v[kParts];
    v[0] = p_amb;
    v[1] = p_ar;
    v[2] = p_at;
    if constexpr (Vort) v[3] = p_conf;
    block_sum<kParts>(v, lds);
    if (threadIdx.x == 0 && partials) {
#pragma unroll
        for (int k = 0; k < kParts; ++k) partials[k * gridDim.x + lb] = v[k];
    }
}

// buoyancy_vjp_kernel (operators.cu:326-337) with FP64 block partials for the parameters.
__global__ __launch_bounds__(256) void buoyancy_vjp_kernel(Geo g, const uint8_t* __restrict__ mask, const float* __restrict__ rho,
                                                           const float* __restrict__ T, Params prm, CF3 fa, float* __restrict__ rho_adj,
                                                           float* __restrict__ t_adj, F3 e_adj, double* __restrict__ partials) {
    __shared__ double lds[3 * kMaxWaves];
    const uint32_t lb = xcd_block();
    uint32_t chunk = (g.n + gridDim.x - 1) / gridDim.x;
    chunk = (chunk + 255u) & ~255u;
    const uint32_t start = min(g.n, lb * chunk), end = min(g.n, start + chunk);
    const float amb = *prm.ambient, ar = *prm.alpha_rho, at = *prm.alpha_t;
    double p_amb = 0.0, p_ar = 0.0, p_at = 0.0;
    for (uint32_t i = start + threadIdx.x; i < end; i += blockDim.x) {
        if (mask[i] != 0) continue;
        const float fy = fa.p[1][i];
        if (e_adj.p[0]) {
            e_adj.p[0][i] += fa.p[0][i];
            e_adj.p[1][i] += fy;
            e_adj.p[2][i] += fa.p[2][i];
        }
        rho_adj[i] += ar * fy;
        t_adj[i] += at * fy;
        p_amb += -(double)at * fy;
        p_ar += (double)rho[i] * fy;
        p_at += (double)(T[i] - amb) * fy;
    }
    double v[3]{p_amb, p_ar, p_at};
    block_sum<3>(v, lds);
    if (threadIdx.x == 0) {
        partials[0 * gridDim.x + lb] = v[0];
        partials[1 * gridDim.x + lb] = v[1];
        partials[2 * gridDim.x + lb] = v[2];
    }
}

// One block: param_adj[k] += sum of the partials of parameter k (fixed order), for the K first
// parameters (ambient, density buoyancy, temperature buoyancy, confinement).
struct ParamOut {
    double* p[4];
};
template <int K>
__global__ __launch_bounds__(256) void param_finalize_kernel(const double* __restrict__ partials, uint32_t G, ParamOut out) {
    __shared__ double lds[K * kMaxWaves];
    const double* parts[K];
#pragma unroll
    for (int k = 0; k < K; ++k) parts[k] = partials + (size_t)k * G;
    double red[K];
    reduce_partials<K>(parts, G, red, lds);
    if (threadIdx.x == 0) {
#pragma unroll
        for (int k = 0; k < K; ++k)
            if (out.p[k]) *out.p[k] += red[k];
    }
}

ParamOut param_out(const ds_parameter_adjoint* a) {
    return ParamOut{{a->ambient_temperature, a->density_buoyancy, a->temperature_buoyancy, a->vorticity_confinement}};
}

// source_vjp_kernel, operators.cu:297-302
__global__ __launch_bounds__(256) void source_vjp_kernel(Geo g, const uint8_t* __restrict__ mask, const float* __restrict__ oa,
                                                         float* __restrict__ sa, float* __restrict__ srca) {
    const uint32_t i = xcd_block() * blockDim.x + threadIdx.x;
    if (i >= g.n || mask[i] != 0) return;
    sa[i] += oa[i];
    if (srca) srca[i] += g.dt * oa[i];
}

// Force part of integrate_vjp_kernel as a gather (per-operator entry point).
__global__ __launch_bounds__(256) void integrate_force_vjp_kernel(Geo g, const uint8_t* __restrict__ mask, CF3 fa, F3 force_adj) {
    const uint32_t i = xcd_block() * blockDim.x + threadIdx.x;
    if (i >= g.n || mask[i] != 0) return;
    int x, y, z;
    decode_cell(g, i, x, y, z);
    float f[3];
    force_gather(g, mask, fa, i, x, y, z, f);
    force_adj.p[0][i] += f[0];
    force_adj.p[1][i] += f[1];
    force_adj.p[2][i] += f[2];
}

}  // namespace

void launch_advect_scalar_vjp(ds_context* c, int nf, int first_field, const float* src0, const float* src1, CF3 u, const float* oa0,
                              const float* oa1, float* sa0, float* sa1, F3 va) {
    const Vel3 v{{u.p[0], u.p[1], u.p[2]}};
    const Geo& g = c->geo;
    const uint64_t bricks = (uint64_t)((g.nx + kSvBX - 1) / kSvBX) * ((g.ny + kSvBY - 1) / kSvBY) * ((g.nz + kSvBZ - 1) / kSvBZ);
    const uint32_t G = (uint32_t)((bricks + 7) & ~7ull);
    if (nf == 2) {
        if (c->has_solids)
            advect_scalar_vjp_kernel<2, true><<<G, kVjpThreads, 0, c->stream>>>(c->geo, c->d_vb, c->d_db, c->d_tb, c->mask, src0, src1, v, oa0, oa1, sa0,
                                                                          sa1, va);
        else
            advect_scalar_vjp_kernel<2, false><<<G, kVjpThreads, 0, c->stream>>>(c->geo, c->d_vb, c->d_db, c->d_tb, c->mask, src0, src1, v, oa0, oa1,
                                                                           sa0, sa1, va);
    } else {
        const SBound* b0 = first_field == 0 ? c->d_db : c->d_tb;
        if (c->has_solids)
            advect_scalar_vjp_kernel<1, true><<<G, kVjpThreads, 0, c->stream>>>(c->geo, c->d_vb, b0, b0, c->mask, src0, src0, v, oa0, oa0, sa0, sa0,
                                                                          va);
        else
            advect_scalar_vjp_kernel<1, false><<<G, kVjpThreads, 0, c->stream>>>(c->geo, c->d_vb, b0, b0, c->mask, src0, src0, v, oa0, oa0, sa0,
                                                                           sa0, va);
    }
    check_launch("advect_scalar_vjp_kernel");
}

void launch_advect_velocity_vjp(ds_context* c, CF3 u, CF3 oa, F3 va) {
    const Vel3 v{{u.p[0], u.p[1], u.p[2]}};
    const Geo& g = c->geo;
    // profiling: every sample_every-th call has each axis launch bracketed by HIP events
    Profiler& prof = c->profiler;
    const bool sample = prof.every && (prof.launches[6] / 3) % prof.every == 0 && prof.used + 6 <= 6000;
    auto launch = [&]<int A>() {
        const int e[3]{g.nx + (A == 0), g.ny + (A == 1), g.nz + (A == 2)};   // face extents of axis A
        const uint64_t bricks = (uint64_t)((e[0] + kVjpBX - 1) / kVjpBX) * ((e[1] + kVjpBY - 1) / kVjpBY) * ((e[2] + kVjpBZ - 1) / kVjpBZ);
        const uint32_t G = (uint32_t)((bricks + 7) & ~7ull);
        hipEvent_t e0 = sample ? prof.take() : nullptr, e1 = sample ? prof.take() : nullptr;
        if (e0) DS_HIP(hipEventRecord(e0, c->stream));
        if (c->has_solids) advect_velocity_vjp_kernel<A, true><<<G, kVjpThreads, 0, c->stream>>>(g, c->d_vb, c->mask, v, oa.p[A], va);
        else advect_velocity_vjp_kernel<A, false><<<G, kVjpThreads, 0, c->stream>>>(g, c->d_vb, c->mask, v, oa.p[A], va);
        if (e0 && e1) {
            DS_HIP(hipEventRecord(e1, c->stream));
            prof.recs.push_back({6, e0, e1});
        }
        if (prof.every) prof.launches[6]++;
    };
    launch.template operator()<0>();
    launch.template operator()<1>();
    launch.template operator()<2>();
    check_launch("advect_velocity_vjp_kernel");
}

void launch_projection_vjp_faces(ds_context* c, const float* const ua[3], const float* const extra[3], const float* lh, const float* ll,
                                 F3 out, bool constrain) {
    ProjAdjIn in{};
    for (int a = 0; a < 3; ++a) {
        in.ua[a] = ua[a];
        in.extra[a] = extra ? extra[a] : nullptr;
    }
    in.lh = lh;
    in.ll = ll;
    const uint32_t G = xcd_blocks_for(c->geo.foff[3]);
    if (constrain)
        projection_vjp_face_kernel<true><<<G, kBlock, 0, c->stream>>>(c->geo, c->d_vb, c->mask, c->has_solids ? 1u : 0u, in, out);
    else
        projection_vjp_face_kernel<false><<<G, kBlock, 0, c->stream>>>(c->geo, c->d_vb, c->mask, c->has_solids ? 1u : 0u, in, out);
    check_launch("projection_vjp_face_kernel");
}

void launch_face_accumulate(ds_context* c, CF3 in, F3 out) {
    face_accumulate_kernel<<<xcd_blocks_for(c->geo.foff[3]), kBlock, 0, c->stream>>>(c->geo, in, out);
    check_launch("face_accumulate_kernel");
}

void launch_cell_accumulate(ds_context* c, const float* in, float* out) {
    cell_accumulate_kernel<<<blocks_for(c->geo.n), kBlock, 0, c->stream>>>(c->geo.n, in, out);
    check_launch("cell_accumulate_kernel");
}

void launch_force_source_vjp(ds_context* c, CF3 forced_adj, const float* rho_s, const float* t_s, const float* rho_s_adj,
                             const float* t_s_adj, const Params& prm, F3 e_adj, float* prev_rho, float* prev_t, float* s_rho_adj,
                             float* s_t_adj, const ds_parameter_adjoint* param_adj) {
    if (c->vorticity) {
        require(prm.confinement != nullptr, "parameters: vorticity_confinement must be a device pointer with confinement on");
        const VortReverse vr{VortFields{{c->vort_w[0], c->vort_w[1], c->vort_w[2]}, c->vort_mag},
                             F3{{c->vort_ga[0], c->vort_ga[1], c->vort_ga[2]}}, F3{{c->vort_t[0], c->vort_t[1], c->vort_t[2]}}};
        force_source_vjp_kernel<true><<<kForceBlocks, kBlock, 0, c->stream>>>(c->geo, c->mask, forced_adj, rho_s, t_s, rho_s_adj, t_s_adj,
                                                                            prm, e_adj, prev_rho, prev_t, s_rho_adj, s_t_adj, vr,
                                                                            c->param_partials);
    } else {
        force_source_vjp_kernel<false><<<kForceBlocks, kBlock, 0, c->stream>>>(c->geo, c->mask, forced_adj, rho_s, t_s, rho_s_adj, t_s_adj,
                                                                             prm, e_adj, prev_rho, prev_t, s_rho_adj, s_t_adj, VortReverse{},
                                                                             c->param_partials);
    }
    check_launch("force_source_vjp_kernel");
    if (param_adj) {
        if (c->vorticity) param_finalize_kernel<4><<<1, kBlock, 0, c->stream>>>(c->param_partials, kForceBlocks, param_out(param_adj));
        else param_finalize_kernel<3><<<1, kBlock, 0, c->stream>>>(c->param_partials, kForceBlocks, param_out(param_adj));
        check_launch("param_finalize_kernel");
    }
}

}  // namespace ds

using namespace ds;

namespace {
bool need_differentiable(ds_context* c, const char* name) {
    if (c->mode != DS_MODE_DIFFERENTIABLE) {
        set_error(std::string(name) + ": the context was not created in differentiable mode");
        return false;
    }
    return true;
}
}  // namespace

extern "C" {

ds_status ds_source_vjp(ds_context* c, const float* out_adj, float* state_adj, float* source_adj) {
    if (!c || !out_adj || !state_adj) {
        set_error("ds_source_vjp: null argument");
        return DS_ERROR_INVALID_ARGUMENT;
    }
    return guard([&] {
        source_vjp_kernel<<<xcd_blocks_for(c->geo.n), kBlock, 0, c->stream>>>(c->geo, c->mask, out_adj, state_adj, source_adj);
        check_launch("source_vjp_kernel");
    });
}

ds_status ds_buoyancy_vjp(ds_context* c, const float* density, const float* temperature, const ds_parameters* params,
                          float* const force_adj[3], float* density_adj, float* temperature_adj, float* e_adj[3],
                          const ds_parameter_adjoint* param_adj) {
    if (!c || !density || !temperature || !force_adj || !density_adj || !temperature_adj) {
        set_error("ds_buoyancy_vjp: null argument");
        return DS_ERROR_INVALID_ARGUMENT;
    }
    if (!need_differentiable(c, "ds_buoyancy_vjp")) return DS_ERROR_INVALID_ARGUMENT;
    return guard([&] {
        const Params prm = params_of(params);
        F3 ea{{e_adj ? e_adj[0] : nullptr, e_adj ? e_adj[1] : nullptr, e_adj ? e_adj[2] : nullptr}};
        buoyancy_vjp_kernel<<<kPcgBlocks, kBlock, 0, c->stream>>>(c->geo, c->mask, density, temperature, prm,
                                                                  CF3{{force_adj[0], force_adj[1], force_adj[2]}}, density_adj,
                                                                  temperature_adj, ea, c->param_partials);
        check_launch("buoyancy_vjp_kernel");
        if (param_adj) {
            ParamOut out = param_out(param_adj);
            out.p[3] = nullptr;
            param_finalize_kernel<3><<<1, kBlock, 0, c->stream>>>(c->param_partials, kPcgBlocks, out);
            check_launch("param_finalize_kernel");
        }
    });
}

ds_status ds_integrate_velocity_vjp(ds_context* c, float* const out_adj[3], float* velocity_adj[3], float* force_adj[3]) {
    if (!c || !out_adj || !velocity_adj) {
        set_error("ds_integrate_velocity_vjp: null argument");
        return DS_ERROR_INVALID_ARGUMENT;
    }
    return guard([&] {
        const CF3 oa{{out_adj[0], out_adj[1], out_adj[2]}};
        launch_face_accumulate(c, oa, F3{{velocity_adj[0], velocity_adj[1], velocity_adj[2]}});
        if (force_adj) {
            integrate_force_vjp_kernel<<<xcd_blocks_for(c->geo.n), kBlock, 0, c->stream>>>(c->geo, c->mask, oa,
                                                                                           F3{{force_adj[0], force_adj[1], force_adj[2]}});
            check_launch("integrate_force_vjp_kernel");
        }
    });
}

ds_status ds_advect_velocity_vjp(ds_context* c, float* const velocity[3], float* const out_adj[3], float* velocity_adj[3]) {
    if (!c || !velocity || !out_adj || !velocity_adj) {
        set_error("ds_advect_velocity_vjp: null argument");
        return DS_ERROR_INVALID_ARGUMENT;
    }
    return guard([&] {
        launch_advect_velocity_vjp(c, CF3{{velocity[0], velocity[1], velocity[2]}}, CF3{{out_adj[0], out_adj[1], out_adj[2]}},
                                   F3{{velocity_adj[0], velocity_adj[1], velocity_adj[2]}});
    });
}

ds_status ds_constrain_velocity_vjp(ds_context* c, float* const out_adj[3], float* velocity_adj[3]) {
    if (!c || !out_adj || !velocity_adj) {
        set_error("ds_constrain_velocity_vjp: null argument");
        return DS_ERROR_INVALID_ARGUMENT;
    }
    return guard([&] {
        constrain_vjp_kernel<<<xcd_blocks_for(c->geo.foff[3]), kBlock, 0, c->stream>>>(
            c->geo, c->d_vb, c->mask, c->has_solids ? 1u : 0u, CF3{{out_adj[0], out_adj[1], out_adj[2]}},
            F3{{velocity_adj[0], velocity_adj[1], velocity_adj[2]}});
        check_launch("constrain_vjp_kernel");
    });
}

ds_status ds_advect_scalar_vjp(ds_context* c, uint32_t field, const float* source, float* const velocity[3], const float* out_adj,
                               float* source_adj, float* velocity_adj[3]) {
    if (!c || !source || !velocity || !out_adj || !source_adj || !velocity_adj || field > 1u) {
        set_error("ds_advect_scalar_vjp: invalid argument");
        return DS_ERROR_INVALID_ARGUMENT;
    }
    return guard([&] {
        launch_advect_scalar_vjp(c, 1, (int)field, source, source, CF3{{velocity[0], velocity[1], velocity[2]}}, out_adj, out_adj,
                                 source_adj, source_adj, F3{{velocity_adj[0], velocity_adj[1], velocity_adj[2]}});
    });
}

ds_status ds_projection_vjp(ds_context* c, float* const out_adj[3], float* velocity_adj[3], ds_solve_info* info) {
    if (!c || !out_adj || !velocity_adj) {
        set_error("ds_projection_vjp: null argument");
        return DS_ERROR_INVALID_ARGUMENT;
    }
    if (!need_differentiable(c, "ds_projection_vjp")) return DS_ERROR_INVALID_ARGUMENT;
    ds_solve_info si{};
    const ds_status st = guard([&] {
        const float* ua[3]{out_adj[0], out_adj[1], out_adj[2]};
        si = pcg_solve_kind(c, 2, ua, nullptr, c->lambda_hi, c->lambda_lo, nullptr, nullptr, c->tolerance, c->max_iterations);
        c->lambda_valid = true;
        launch_projection_vjp_faces(c, ua, nullptr, c->lambda_hi, c->lambda_lo, F3{{velocity_adj[0], velocity_adj[1], velocity_adj[2]}},
                                    false);
    });
    if (info) *info = si;
    if (st != DS_OK) return st;
    if (!si.converged) {
        set_error("ds_projection_vjp: adjoint pressure solve did not converge");
        return std::isfinite(si.final_residual) ? DS_ERROR_NOT_CONVERGED : DS_ERROR_NON_FINITE;
    }
    return DS_OK;
}

}  // extern "C"
