// mgf_device.h — device-side arithmetic of the MAC-grid step for gfx950.
//
// Every routine here reproduces one reference operation with the same
// operation order and one rounding per written float operation (the
// library is compiled with -ffp-contract=off); the BLAS axpy of the
// back-trace is one explicit fused multiply-add (__builtin_fmaf).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <cmath>

#define MGF_UNKNOWN 3.40282346638528859812e+38f   /* FLT_MAX, MMathExtra.h:58 */
#define MGF_FLT_EPSILON 1.19209290e-07f          /* FLT_EPSILON, MMathExtra.h:55 */

namespace mgf {

struct GridDev {
    int nx, ny, nz;
    float ox, oy, oz;
    float hx, hy, hz;
    // 1/h per axis and whether every spacing is a power of two whose
    // reciprocal is a normal float (set by set_recip)
    float rhx = 0, rhy = 0, rhz = 0;
    int pow2 = 0;
    int path = 0;   // which instance of the samplers serves the grid (kPath*)
    // 1/d of the index decodes' divisors (cells: nx, nx ny; u faces: nx + 1,
    // (nx + 1) ny; v faces: nx, nx (ny + 1); w faces as cells), set by set_recip
    double r_nx = 0, r_nxy = 0, r_nx1 = 0, r_nx1y = 0, r_nxy1 = 0;
};

// Division by a spacing h = 2^k and multiplication by 2^-k round the same
// real number once, so they give the same float (overflow, underflow, zero
// signs and NaN included) while the multiplication avoids the correctly
// rounded division's instruction sequence.  Other spacings divide.
enum : int { kPathAny = 0, kPathPow2 = 1, kPathRecip = 2 };

// The samplers' instances (sample_vel_t and the like):
//   kPathAny    any grid: one load a corner, true divisions
//   kPathPow2   multiplications by 2^-k, two corners a load, 32-bit offsets
//   kPathRecip  the same with the quotients of div_path (spacings that are no
//               powers of two)
// The two fast ones need rows of two values, extents and plane sizes within
// 24-bit products and byte offsets within 32 bits; kPathRecip also spacings
// far from the ends of the exponent range (div_path).
inline int sample_path(const GridDev& g) {
    const double ex = double(g.nx) + 1.0, ey = double(g.ny) + 1.0, ez = double(g.nz) + 1.0;
    if (g.nx < 2 || ex * ey >= 16777216.0 || ez >= 16777216.0 || ex * ey * ez >= 1073741824.0) return kPathAny;
    if (g.pow2) return kPathPow2;
    auto mid = [](float h) { return h >= 9.5367431640625e-07f && h <= 1048576.0f; };   // 2^-20 .. 2^20
    return mid(g.hx) && mid(g.hy) && mid(g.hz) ? kPathRecip : kPathAny;
}

inline void set_recip(GridDev& g) {
    auto p2 = [](float h, float& r) {
        int e = 0;
        const float m = std::frexp(h, &e);
        r = 1.0f / h;
        return h > 0.0f && m == 0.5f && std::isnormal(h) && std::isnormal(r);
    };
    const bool a = p2(g.hx, g.rhx), b = p2(g.hy, g.rhy), c = p2(g.hz, g.rhz);
    g.pow2 = (a && b && c) ? 1 : 0;
    const double nx = double(g.nx), ny = double(g.ny);
    g.r_nx = 1.0 / nx;
    g.r_nxy = 1.0 / (nx * ny);
    g.r_nx1 = 1.0 / (nx + 1.0);
    g.r_nx1y = 1.0 / ((nx + 1.0) * ny);
    g.r_nxy1 = 1.0 / (nx * (ny + 1.0));
    g.path = sample_path(g);
}

// a / d for a < 2^32, d >= 1, from rd = 1/d in FP64: a * rd is within one of
// the quotient and is corrected once, so the quotient is exact (the integer
// divide's instruction sequence avoided).
__device__ __forceinline__ uint32_t udiv_rd(uint32_t a, uint32_t d, double rd) {
    uint32_t q = uint32_t(double(a) * rd);
    const uint32_t r = a - q * d;
    if (int32_t(r) < 0) --q;
    else if (r >= d) ++q;
    return q;
}

// (x, y, z) of index i in an ex x ey x .. array: rex = 1/ex, rexy = 1/(ex ey).
__device__ __forceinline__ void decode3(uint32_t i, uint32_t ex, uint32_t ey, double rex, double rexy, int& x,
                                        int& y, int& z) {
    const uint32_t exy = ex * ey;
    const uint32_t zz = udiv_rd(i, exy, rexy);
    const uint32_t rem = i - zz * exy;
    const uint32_t yy = udiv_rd(rem, ex, rex);
    x = int(rem - yy * ex);
    y = int(yy);
    z = int(zz);
}

__device__ __forceinline__ float div_h(float x, float h, float rh, int pow2) {
    return pow2 ? x * rh : x / h;
}

// limitIndex (MPhysics/EulerMathTool.cu:16-27).
__device__ __forceinline__ int clampi(int i, int n) {
    return i < 0 ? 0 : (i > n - 1 ? n - 1 : i);
}

// transIndex2LinearWithOffset (MPhysics/EulerMathTool.cu:63-73).
__device__ __forceinline__ uint32_t lin3(int x, int y, int z, int nx, int ny, int nz) {
    x = clampi(x, nx);
    y = clampi(y, ny);
    z = clampi(z, nz);
    return (uint32_t(z) * uint32_t(ny) + uint32_t(y)) * uint32_t(nx) + uint32_t(x);
}

// floorCUDA (MPhysics/EulerMathTool.cu:93-103): truncate, minus one when the
// input is negative.  The conversion saturates at +-2^24 and maps NaN to 0
// (points that far out clamp to the grid edge either way).
__device__ __forceinline__ int floor_ref(float v) {
    int t;
    if (!(v == v)) t = 0;
    else if (v >= 16777216.0f) t = 16777216;
    else if (v <= -16777216.0f) t = -16777216;
    else t = int(v);
    return v >= 0.0f ? t : t - 1;
}

// Trilinear gather on a cell-centred grid (extents nx,ny,nz, origin o,
// spacing h): sampleCellCenteredScalarFieldTrilerp
// (MPhysics/FieldMathTool.cu:52-104).
__device__ __forceinline__ float trilerp(const float* __restrict__ f, int nx, int ny, int nz,
                                         float ox, float oy, float oz, const GridDev& g,
                                         float px, float py, float pz) {
    const float hx = g.hx, hy = g.hy, hz = g.hz;
    const float rx = px - ox - hx / 2;
    const float ry = py - oy - hy / 2;
    const float rz = pz - oz - hz / 2;
    const int ix = floor_ref(div_h(rx, hx, g.rhx, g.pow2));
    const int iy = floor_ref(div_h(ry, hy, g.rhy, g.pow2));
    const int iz = floor_ref(div_h(rz, hz, g.rhz, g.pow2));
    const float fx = div_h(rx - float(ix) * hx, hx, g.rhx, g.pow2);
    const float fy = div_h(ry - float(iy) * hy, hy, g.rhy, g.pow2);
    const float fz = div_h(rz - float(iz) * hz, hz, g.rhz, g.pow2);
    const int x0 = clampi(ix, nx), x1 = clampi(ix + 1, nx);
    const int y0 = clampi(iy, ny), y1 = clampi(iy + 1, ny);
    const int z0 = clampi(iz, nz), z1 = clampi(iz + 1, nz);
    const uint32_t sy = uint32_t(nx), sz = uint32_t(nx) * uint32_t(ny);
    const uint32_t r00 = uint32_t(z0) * sz + uint32_t(y0) * sy;
    const uint32_t r01 = uint32_t(z0) * sz + uint32_t(y1) * sy;
    const uint32_t r10 = uint32_t(z1) * sz + uint32_t(y0) * sy;
    const uint32_t r11 = uint32_t(z1) * sz + uint32_t(y1) * sy;
    const float dbl = f[r00 + x0], dbr = f[r00 + x1];
    const float ubl = f[r01 + x0], ubr = f[r01 + x1];
    const float dfl = f[r10 + x0], dfr = f[r10 + x1];
    const float ufl = f[r11 + x0], ufr = f[r11 + x1];
    return dbl * (1 - fx) * (1 - fy) * (1 - fz) +
           dbr * fx * (1 - fy) * (1 - fz) +
           ubl * (1 - fx) * fy * (1 - fz) +
           ubr * fx * fy * (1 - fz) +
           dfl * (1 - fx) * (1 - fy) * fz +
           dfr * fx * (1 - fy) * fz +
           ufl * (1 - fx) * fy * fz +
           ufr * fx * fy * fz;
}

// Component c of a face-centred field: a cell-centred grid one layer longer on
// axis c with the origin moved by -h/2 on that axis
// (MPhysics/FieldMathTool.cu:783-892).
__device__ __forceinline__ float sample_comp(const float* __restrict__ f, int c, const GridDev& g,
                                             float px, float py, float pz) {
    if (c == 0) return trilerp(f, g.nx + 1, g.ny, g.nz, g.ox - g.hx / 2, g.oy, g.oz, g, px, py, pz);
    if (c == 1) return trilerp(f, g.nx, g.ny + 1, g.nz, g.ox, g.oy - g.hy / 2, g.oz, g, px, py, pz);
    return trilerp(f, g.nx, g.ny, g.nz + 1, g.ox, g.oy, g.oz - g.hz / 2, g, px, py, pz);
}

struct Vel {
    const float* __restrict__ u;
    const float* __restrict__ v;
    const float* __restrict__ w;
};

__device__ __forceinline__ void sample_vel(const Vel& V, const GridDev& g, float px, float py,
                                           float pz, float& a, float& b, float& c) {
    a = sample_comp(V.u, 0, g, px, py, pz);
    b = sample_comp(V.v, 1, g, px, py, pz);
    c = sample_comp(V.w, 2, g, px, py, pz);
}

// ---------------------------------------------------------------------------
// The same samples for the grids of sample_path's fast instances, bit for bit.
// A sample is bound by its vector instructions, not by its loads: the general
// form spends them on branches around each conversion and division, on the
// same axis worked out again for each component and on eight 64-bit addresses.
// Here an axis' index and fraction are formed once for the components that
// share its origin, without a branch, and the two corners of a row are one
// load.  258^3 faces,
// first order, powers of two: 625 -> 487 us; 152 x 63 x 99, third order,
// h = 1/50: 128 -> 70 us (first-order bytes alone: 90 us and 5 us).

// x / h with the rounding of the division.  kPathRecip: q0 = x RN(1/h) is
// within two units of the quotient, q1 = q0 + (x - q0 h) RN(1/h) within one,
// and one more such step rounds correctly (Markstein, IBM J. Res. Dev. 34(1),
// 1990: a faithful quotient, its exact residual and the rounded reciprocal).
// The residuals are exact while nothing nears underflow or overflow: callers
// pass |x| < 2^22 h (axis_t's check; NaN fails it) and x that is zero or at
// least 2^-46: x is a position minus an origin minus h/2, and such a
// difference with h >= 2^-20 is a multiple of 2^-46 where it is small.  Nor is
// x ever -0, which this would turn into +0.
template <int kPath>
__device__ __forceinline__ float div_path(float x, float h, float rh) {
    if (kPath == kPathPow2) return x * rh;
    if (kPath == kPathAny) return x / h;
    const float q0 = x * rh;
    const float q1 = __builtin_fmaf(__builtin_fmaf(-q0, h, x), rh, q0);
    return __builtin_fmaf(__builtin_fmaf(-q1, h, x), rh, q1);
}

// floor_ref without branches: the conversion instruction itself saturates and
// takes NaN to 0 (the language leaves both undefined, hence the instruction).
__device__ __forceinline__ int floor_sat(float v) {
    int t;
    asm("v_cvt_i32_f32 %0, %1" : "=v"(t) : "v"(v));
    t = t < -16777216 ? -16777216 : (t > 16777216 ? 16777216 : t);
    return v >= 0.0f ? t : t - 1;
}

// i limited to 0 .. top
__device__ __forceinline__ uint32_t limit(int i, int top) {
    int t;
    asm("v_med3_i32 %0, %1, 0, %2" : "=v"(t) : "v"(i), "v"(top));
    return uint32_t(t);
}

// a * b for factors below 2^24
__device__ __forceinline__ uint32_t mul24(uint32_t a, uint32_t b) { return (a & 0xffffffu) * (b & 0xffffffu); }

struct Axis {
    int i;      // floor of the coordinate, not limited
    float f;    // fraction
};

template <int kPath>
__device__ __forceinline__ Axis axis_t(float p, float o, float h, float rh, bool& ok) {
    const float r = p - o - h / 2;
    if (kPath == kPathRecip) ok = ok && fabsf(r) < h * 4194304.0f;
    Axis a;
    a.i = floor_sat(div_path<kPath>(r, h, rh));
    a.f = div_path<kPath>(r - float(a.i) * h, h, rh);
    return a;
}

// trilerp's sum over an ex x ey x ez field (ex >= 2) at the axes' indices
__device__ __forceinline__ float gather_t(const float* __restrict__ f, int ex, int ey, int ez, Axis ax, Axis ay,
                                          Axis az) {
    typedef float Pair __attribute__((ext_vector_type(2), aligned(4)));
    const uint32_t xb = limit(ax.i, ex - 2);
    const uint32_t y0 = mul24(limit(ay.i, ey - 1), uint32_t(ex)), y1 = mul24(limit(ay.i + 1, ey - 1), uint32_t(ex));
    const uint32_t exy = uint32_t(ex) * uint32_t(ey);
    const uint32_t z0 = mul24(limit(az.i, ez - 1), exy) + xb, z1 = mul24(limit(az.i + 1, ez - 1), exy) + xb;
    const char* b = reinterpret_cast<const char*>(f);
    const Pair a00 = *reinterpret_cast<const Pair*>(b + (z0 + y0) * 4u);
    const Pair a01 = *reinterpret_cast<const Pair*>(b + (z0 + y1) * 4u);
    const Pair a10 = *reinterpret_cast<const Pair*>(b + (z1 + y0) * 4u);
    const Pair a11 = *reinterpret_cast<const Pair*>(b + (z1 + y1) * 4u);
    // beyond an end both corners are the end's value
    const bool lo = ax.i < 0, hi = ax.i > ex - 2;
    const float dbl = hi ? a00.y : a00.x, dbr = lo ? a00.x : a00.y;
    const float ubl = hi ? a01.y : a01.x, ubr = lo ? a01.x : a01.y;
    const float dfl = hi ? a10.y : a10.x, dfr = lo ? a10.x : a10.y;
    const float ufl = hi ? a11.y : a11.x, ufr = lo ? a11.x : a11.y;
    const float fx = ax.f, fy = ay.f, fz = az.f;
    return dbl * (1 - fx) * (1 - fy) * (1 - fz) +
           dbr * fx * (1 - fy) * (1 - fz) +
           ubl * (1 - fx) * fy * (1 - fz) +
           ubr * fx * fy * (1 - fz) +
           dfl * (1 - fx) * (1 - fy) * fz +
           dfr * fx * (1 - fy) * fz +
           ufl * (1 - fx) * fy * fz +
           ufr * fx * fy * fz;
}

template <int kPath>
__device__ __forceinline__ void sample_vel_t(const Vel& V, const GridDev& g, float px, float py, float pz, float& a,
                                             float& b, float& c) {
    if (kPath == kPathAny) {
        sample_vel(V, g, px, py, pz, a, b, c);
        return;
    }
    const float fx = g.ox - g.hx / 2, fy = g.oy - g.hy / 2, fz = g.oz - g.hz / 2;
    bool ok = true;
    Axis xf = axis_t<kPath>(px, fx, g.hx, g.rhx, ok), xc = axis_t<kPath>(px, g.ox, g.hx, g.rhx, ok);
    Axis yf = axis_t<kPath>(py, fy, g.hy, g.rhy, ok), yc = axis_t<kPath>(py, g.oy, g.hy, g.rhy, ok);
    Axis zf = axis_t<kPath>(pz, fz, g.hz, g.rhz, ok), zc = axis_t<kPath>(pz, g.oz, g.hz, g.rhz, ok);
    if (kPath == kPathRecip && !ok) {
        xf = axis_t<kPathAny>(px, fx, g.hx, g.rhx, ok); xc = axis_t<kPathAny>(px, g.ox, g.hx, g.rhx, ok);
        yf = axis_t<kPathAny>(py, fy, g.hy, g.rhy, ok); yc = axis_t<kPathAny>(py, g.oy, g.hy, g.rhy, ok);
        zf = axis_t<kPathAny>(pz, fz, g.hz, g.rhz, ok); zc = axis_t<kPathAny>(pz, g.oz, g.hz, g.rhz, ok);
    }
    a = gather_t(V.u, g.nx + 1, g.ny, g.nz, xf, yc, zc);
    b = gather_t(V.v, g.nx, g.ny + 1, g.nz, xc, yf, zc);
    c = gather_t(V.w, g.nx, g.ny, g.nz + 1, xc, yc, zf);
}

__device__ __forceinline__ void sample_vel_any(const Vel& V, const GridDev& g, float px, float py, float pz, float& a,
                                               float& b, float& c) {
    if (g.path == kPathPow2) sample_vel_t<kPathPow2>(V, g, px, py, pz, a, b, c);
    else if (g.path == kPathRecip) sample_vel_t<kPathRecip>(V, g, px, py, pz, a, b, c);
    else sample_vel(V, g, px, py, pz, a, b, c);
}

// trilerp of one field or, for the axes of one point, of several: the axes
// of a cell-centred field (c = 3) or of a face component c
struct Point {
    Axis x, y, z;
    int ex, ey, ez;
};

template <int kPath>
__device__ __forceinline__ Point point_t(const GridDev& g, int c, float px, float py, float pz) {
    const float ox = c == 0 ? g.ox - g.hx / 2 : g.ox;
    const float oy = c == 1 ? g.oy - g.hy / 2 : g.oy;
    const float oz = c == 2 ? g.oz - g.hz / 2 : g.oz;
    bool ok = true;
    Point P;
    P.x = axis_t<kPath>(px, ox, g.hx, g.rhx, ok);
    P.y = axis_t<kPath>(py, oy, g.hy, g.rhy, ok);
    P.z = axis_t<kPath>(pz, oz, g.hz, g.rhz, ok);
    if (kPath == kPathRecip && !ok) {
        P.x = axis_t<kPathAny>(px, ox, g.hx, g.rhx, ok);
        P.y = axis_t<kPathAny>(py, oy, g.hy, g.rhy, ok);
        P.z = axis_t<kPathAny>(pz, oz, g.hz, g.rhz, ok);
    }
    P.ex = g.nx + (c == 0); P.ey = g.ny + (c == 1); P.ez = g.nz + (c == 2);
    return P;
}

// plusAlphaX's early return: |alpha| < FLT_EPSILON skips the update.
__device__ __forceinline__ bool axpy_on(float a) { return !(fabsf(a) < MGF_FLT_EPSILON); }

// CSemiLagrangian::backTrace for one point (MPhysics/SemiLagrangian.cpp:
// 188-347).  `coef` holds the host-computed axpy factors:
// [0] -dt  [1] -0.5*dt  [2] -0.75*dt  [3] -(2/9)dt  [4] -(3/9)dt  [5] -(4/9)dt.
struct RkCoef {
    float c[6];
};

template <int kPath>
__device__ __forceinline__ void backtrace(const Vel& V, const GridDev& g, int order,
                                          const RkCoef& k, float& px, float& py, float& pz) {
    const float x0 = px, y0 = py, z0 = pz;
    float v1x, v1y, v1z;
    sample_vel_t<kPath>(V, g, x0, y0, z0, v1x, v1y, v1z);
    if (order == 1) {
        if (axpy_on(k.c[0])) {
            px = __builtin_fmaf(k.c[0], v1x, x0);
            py = __builtin_fmaf(k.c[0], v1y, y0);
            pz = __builtin_fmaf(k.c[0], v1z, z0);
        }
        return;
    }
    float mx = x0, my = y0, mz = z0;
    if (axpy_on(k.c[1])) {
        mx = __builtin_fmaf(k.c[1], v1x, x0);
        my = __builtin_fmaf(k.c[1], v1y, y0);
        mz = __builtin_fmaf(k.c[1], v1z, z0);
    }
    float v2x, v2y, v2z;
    sample_vel_t<kPath>(V, g, mx, my, mz, v2x, v2y, v2z);
    if (order == 2) {
        if (axpy_on(k.c[0])) {
            px = __builtin_fmaf(k.c[0], v2x, x0);
            py = __builtin_fmaf(k.c[0], v2y, y0);
            pz = __builtin_fmaf(k.c[0], v2z, z0);
        }
        return;
    }
    float tx = x0, ty = y0, tz = z0;
    if (axpy_on(k.c[2])) {
        tx = __builtin_fmaf(k.c[2], v2x, x0);
        ty = __builtin_fmaf(k.c[2], v2y, y0);
        tz = __builtin_fmaf(k.c[2], v2z, z0);
    }
    float v3x, v3y, v3z;
    sample_vel_t<kPath>(V, g, tx, ty, tz, v3x, v3y, v3z);
    float ox = x0, oy = y0, oz = z0;
    if (axpy_on(k.c[3])) {
        ox = __builtin_fmaf(k.c[3], v1x, ox);
        oy = __builtin_fmaf(k.c[3], v1y, oy);
        oz = __builtin_fmaf(k.c[3], v1z, oz);
    }
    if (axpy_on(k.c[4])) {
        ox = __builtin_fmaf(k.c[4], v2x, ox);
        oy = __builtin_fmaf(k.c[4], v2y, oy);
        oz = __builtin_fmaf(k.c[4], v2z, oz);
    }
    if (axpy_on(k.c[5])) {
        ox = __builtin_fmaf(k.c[5], v3x, ox);
        oy = __builtin_fmaf(k.c[5], v3y, oy);
        oz = __builtin_fmaf(k.c[5], v3z, oz);
    }
    px = ox;
    py = oy;
    pz = oz;
}

// Face position of component c at (x,y,z) and cell-centre position
// (MPhysics/SemiLagrangian.cpp:47-97).
__device__ __forceinline__ float cpos(int k, float h, float o) { return (k + 0.5f) * h + o; }
__device__ __forceinline__ float fpos(int k, float h, float o) { return float(k) * h + o; }

// ---------------------------------------------------------------------------
// Markers: 0 air, 1 fluid, 2 solid (MPhysics/EulerSolverTool.cu:30-56).
enum : uint8_t { kAir = 0, kFluid = 1, kSolid = 2 };

// One row of the pressure matrix recomputed from the markers
// (buildPressureMatrixA, MPhysics/EulerSolverTool.cu:58-126): diagonal and the
// three "+" couplings; scale s = dt/(rho*h^2).  The diagonal is accumulated in
// the reference's order so it is bitwise the stored value.
struct Row {
    float d, ax, ay, az;
};

template <class M>
__device__ __forceinline__ Row matrix_row(const M& mk, int x, int y, int z, int nx, int ny, int nz,
                                          float sx, float sy, float sz) {
    Row r{0.f, 0.f, 0.f, 0.f};
    if (mk(x, y, z) != kFluid) {
        r.d = 1.0f;
        return r;
    }
    if (x > 0 && mk(x - 1, y, z) != kSolid) r.d += sx;
    if (x + 1 < nx) {
        const uint8_t m = mk(x + 1, y, z);
        if (m != kSolid) {
            r.d += sx;
            if (m == kFluid) r.ax -= sx;
        }
    }
    if (y > 0 && mk(x, y - 1, z) != kSolid) r.d += sy;
    if (y + 1 < ny) {
        const uint8_t m = mk(x, y + 1, z);
        if (m != kSolid) {
            r.d += sy;
            if (m == kFluid) r.ay -= sy;
        }
    }
    if (z > 0 && mk(x, y, z - 1) != kSolid) r.d += sz;
    if (z + 1 < nz) {
        const uint8_t m = mk(x, y, z + 1);
        if (m != kSolid) {
            r.d += sz;
            if (m == kFluid) r.az -= sz;
        }
    }
    return r;
}

// "+d" coupling of cell (x,y,z) toward its +d neighbour, which is what the
// reference reads from the neighbour's slot for the -d term.
__device__ __forceinline__ float plus_coupling(uint8_t mc, uint8_t mn, float s) {
    return (mc == kFluid && mn == kFluid) ? -s : 0.0f;
}

}  // namespace mgf
